"""The lane-pair passes at the sizes and list lengths where another form of them
runs: 163,841 to 196,608 particles (six waves per SIMD, the second chunk of a list
not read ahead) and lists of more than 384 slots (workgroups of 256). One lane per
particle gives the same bits, for plain lists, staged ones and waves without a
list, with and without the viscosity solve."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from parity_util import dev, say  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


@pytest.mark.parametrize("flags", [0, 1])
@pytest.mark.parametrize("kw", [{"stage_min_particles": -1}, {"stage_min_particles": 1},
                                {"stage_min_particles": -1, "list_slots": 64}],
                         ids=["plain", "staged", "some waves without a list"])
@pytest.mark.parametrize("n, spacing", [(163840, 0.005), (163841, 0.005), (180001, 0.0042), (196608, 0.005),
                                        (196609, 0.005), (20000, 0.0026), (170000, 0.0028)])
def test_lane_pair_equals_one_lane(fluid, scene, n, spacing, kw, flags):
    side = int(np.ceil(n ** (1 / 3) - 1e-9))
    x = scene.jittered_lattice((side,) * 3, (0.25, 0.3, 0.25), spacing, 0.1, seed=n, count=n)
    v = (0.05 * (scene.uniform01(6, 3 * n).reshape(n, 3) - 0.5)).astype(np.float32)
    say(f"lane pair against one lane, {n} particles, spacing {spacing}, {kw}, flags {flags}")
    outs = []
    for lanes in (1, 2, 0):
        ctx = fluid.Context("cuda:0", flags=flags, **kw)
        if lanes:
            ctx.set_tuning(256, kw["stage_min_particles"], 0, lanes)
        xd, vd, rho = dev(x), dev(v), torch.zeros(n, dtype=torch.float32, device="cuda:0")
        for _ in range(2):  # the second call has its lists as long as it needs
            ctx.step(xd, vd, rho)
            torch.cuda.synchronize()
        if lanes:
            assert ctx.stats()["pass_lanes"] == lanes
        outs.append([t.cpu().numpy().view(np.uint32) for t in (xd, vd, rho)])
    for other in outs[1:]:
        for a, b in zip(outs[0], other):
            np.testing.assert_array_equal(a, b)
