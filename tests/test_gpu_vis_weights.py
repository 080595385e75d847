"""The fused viscosity solve with the weights kept over its iterations (lane
pairs) against the form that forms them again in each (one lane per particle):
the same bits, for list lengths around a chunk of the list, staged and plain
lists, lists that do not fit their reservation, and coincident particles."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from parity_util import dev, say  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def inputs(scene, name):
    if name == "lines":  # rows of 1 to about 20 neighbors, some coincident
        x = np.full((700, 3), 0.5, np.float32)
        for k in range(14):
            x[50 * k:50 * k + 50, 0] = 0.1 + 0.0125 / (0.7 + 0.7 * k) * np.arange(50)
            x[50 * k:50 * k + 50, 1] = 0.1 + 0.05 * k
        x[101] = x[100]
        return x
    if name == "blob":
        return scene.gaussian_blobs(1, 6000, 0.012, seed=7)
    n = int(name)
    side = int(np.ceil(n ** (1 / 3) - 1e-9))
    return scene.jittered_lattice((side,) * 3, (0.3, 0.4, 0.3), 0.005, 0.1, seed=n, count=n)


@pytest.mark.parametrize("iterations", [1, 2, 5])
@pytest.mark.parametrize("kw", [{}, {"stage_min_particles": 1}, {"list_slots": 4}],
                         ids=["plain", "staged", "short reservation"])
@pytest.mark.parametrize("name", ["1", "63", "65", "20000", "lines", "blob"])
def test_kept_weights_equal_formed_weights(fluid, scene, name, kw, iterations):
    x = inputs(scene, name)
    n = len(x)
    say(f"viscosity weights kept, {name}: {n} particles, {iterations} iterations, {kw}")
    v = (0.5 * (scene.uniform01(5, 3 * n).reshape(n, 3) - 0.5)).astype(np.float32)
    outs = []
    for lanes in (1, 2):
        ctx = fluid.Context("cuda:0", flags=fluid._capi.PBF_FLAG_VISCOSITY, viscosity_iterations=iterations, **kw)
        ctx.set_tuning(256, kw.get("stage_min_particles", 0), 0, lanes)
        xd, vd, rho = dev(x), dev(v), torch.zeros(n, dtype=torch.float32, device="cuda:0")
        for _ in range(2):
            ctx.step(xd, vd, rho)
        torch.cuda.synchronize()
        assert ctx.stats()["pass_lanes"] == lanes
        outs.append([t.cpu().numpy().view(np.uint32) for t in (xd, vd, rho)])
    for a, b in zip(*outs):
        np.testing.assert_array_equal(a, b)
