"""The double-precision rollout with pair_eps 0 and next to it: no pair of the scene
is closer than 1e-4 except two particles in one place (and each particle with
itself), whose terms vanish with r = 0, so every pair_eps below gives the same
bits, forward and backward, with one lane and a lane pair per particle."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from parity_util import dev, say  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


@pytest.mark.parametrize("lanes", [1, 2])
@pytest.mark.parametrize("together", [False, True])
@pytest.mark.parametrize("eps", [0.0, 1e-38, 1e-20])
def test_small_pair_eps_equal_bits(fluid, scene, eps, together, lanes):
    x0 = scene.jittered_lattice((11, 10, 9), (0.3, 0.5, 0.3), 0.0045, 0.1, seed=3)
    if together:
        x0[500] = x0[400]
    n = len(x0)
    say(f"double rollout, pair_eps {eps}, two particles in one place: {together}, {lanes} lanes")
    outs = []
    for e in (1e-12, eps):
        ctx = fluid.Context("cuda:0", pair_eps=e)
        ctx.set_tuning(256, 0, 0, lanes)
        x = dev(x0).double()
        v = torch.zeros_like(x)
        rho = torch.zeros(n, dtype=torch.float64, device="cuda:0")
        token = ctx.rollout_forward(x, v, rho, 2, 2)
        xb = torch.linspace(-1, 1, 3 * n, dtype=torch.float64, device="cuda:0").reshape(n, 3)
        vb = xb.flip(0) * 1e-3
        ctx.rollout_backward(xb, vb, token)
        outs.append([t.cpu().numpy() for t in (x, v, rho, xb, vb)])
    for a, b in zip(*outs):
        assert np.isfinite(a).all()
        np.testing.assert_array_equal(a, b)
