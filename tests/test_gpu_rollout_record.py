"""fluid.rollout with and without a gradient to come, in turn on one context: a
forward that autograd differentiates records its last segment, another one does
not; states and gradients equal a fresh context's, bit for bit."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from parity_util import dev, say  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def run(fluid, ctx, x0, how, every):
    """(states, gradients or ()) of four steps."""
    v0 = torch.zeros_like(x0)
    if how == "grad" or how == "grad of v":
        x, v = x0.clone().requires_grad_(how == "grad"), v0.requires_grad_(True)
        wrt = [x, v] if how == "grad" else [v]
        out = fluid.rollout(ctx, x, v, 4, every)
        w = torch.linspace(-1, 1, x0.numel(), dtype=x0.dtype, device=x0.device).reshape(x0.shape)
        grads = torch.autograd.grad([out[0], out[1]], wrt, [w, 1e-3 * w])
        return [*(o.detach() for o in out), *grads]
    if how == "no_grad":
        with torch.no_grad():
            return list(fluid.rollout(ctx, x0.clone().requires_grad_(True), v0, 4, every))
    if how == "inference":
        with torch.inference_mode():
            return list(fluid.rollout(ctx, x0, v0, 4, every))
    return list(fluid.rollout(ctx, x0, v0, 4, every))  # no input asks for one


@pytest.mark.parametrize("double", [False, True])
@pytest.mark.parametrize("every", [2, 10])
def test_rollouts_with_and_without_gradients(fluid, scene, double, every):
    say(f"rollouts with and without gradients in turn, {'f64' if double else 'f32'}, checkpoint {every}")
    ctx = fluid.Context("cuda:0")
    order = ["grad", "no_grad", "grad", "plain", "inference", "grad of v", "grad", "no_grad", "grad"]
    for seed, how in enumerate(order):
        x0 = dev(scene.jittered_lattice((20, 15, 10), (0.3, 0.5, 0.3), 0.0042, 0.1, seed=seed))
        x0 = x0.double() if double else x0
        got = run(fluid, ctx, x0, how, every)
        want = run(fluid, fluid.Context("cuda:0"), x0, how, every)
        assert len(got) == len(want) and all(g.requires_grad is False for g in got)
        for a, b in zip(got, want):
            np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy())
