"""The sort of a small scene in one workgroup where its particles are not a compact
block: thousands of them outside the grid, or all over the scene box. A batch of
the scene and an empty one takes the general sort; both give the same bits over
two steps (caller's order and cell order) and the same lists. A step takes no more
than three times (outside the grid) or twice (scattered) the time of a block of as
many particles, which has far more pairs; comparing the out-of-grid particles with
each other took 20 times it, a search of the keys for every cell four times."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from parity_util import dev, say  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def block(scene, n, spacing=0.005):
    side = int(np.ceil(n ** (1 / 3) - 1e-9))
    return scene.jittered_lattice((side,) * 3, (0.2, 0.3, 0.2), spacing, 0.1, seed=n, count=n)


def shuffled(x):
    return np.ascontiguousarray(x[np.random.default_rng(3).permutation(len(x))])


def inputs(scene, name):
    kind, n = name.rsplit(" ", 1)
    x = block(scene, int(n))
    if kind == "all out":
        x += np.float32(3)
    elif kind == "one in":
        x[1:] += np.float32(3)
    elif kind == "half out":
        x[: len(x) // 2] += np.float32(3)
    elif kind == "few out, wide":  # a window of more cells than buckets
        x[::9] += np.float32(3)
        x[1::300] = scene.uniform01(5, 3 * len(x[1::300])).reshape(-1, 3)
    return shuffled(x)


NAMES = ["all out 1", "all out 64", "all out 2049", "all out 4096", "one in 4096", "half out 33", "half out 4096",
         "few out, wide 4000"]


@pytest.mark.parametrize("name", NAMES)
def test_small_sort_equals_the_general_one(fluid, scene, name):
    x = inputs(scene, name)
    n = len(x)
    say(f"sort of a small scene: {name}")
    v = (0.05 * (scene.uniform01(6, 3 * n).reshape(n, 3) - 0.5)).astype(np.float32)
    outs = []
    for batch in (False, True):
        ctx = fluid.Context("cuda:0", stage_min_particles=-1)
        got = []
        for steps in (1, 2):
            xd, vd, rho = dev(x), dev(v), torch.zeros(n, dtype=torch.float32, device="cuda:0")
            if batch:
                ctx.batch_step(xd, vd, torch.tensor([0, n, n], dtype=torch.int32, device="cuda:0"), rho, steps)
            else:
                ctx.step(xd, vd, rho, steps)
            nl = ctx.step_neighbors(n)
            got += [t.cpu().numpy().view(np.uint32) for t in (xd, vd, rho, nl.index, nl.elements)]
        st = ctx.stats()
        outs.append(got + [(st["neighbor_pairs"], st["candidates"], st["out_of_grid"], st["nonfinite"])])
    for a, b in zip(*outs):
        np.testing.assert_array_equal(a, b)


def step_time(fluid, x, h=0.0125):
    """A step's time in us: the best of five runs of ten."""
    ctx = fluid.Context("cuda:0", smoothing_length=h)
    x0 = dev(x)
    xd, vd = x0.clone(), torch.zeros_like(x0)
    best = float("inf")
    for _ in range(6):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        for _ in range(10):
            xd.copy_(x0)
            vd.zero_()
            ctx.step(xd, vd)
        b.record()
        torch.cuda.synchronize()
        best = min(best, 100 * a.elapsed_time(b))
    return best


def test_out_of_grid_particles_are_not_compared(fluid, scene):
    base, out = step_time(fluid, block(scene, 4096)), step_time(fluid, inputs(scene, "all out 4096"))
    say(f"a step of 4,096 particles: in a block {base:.0f} us, out of the grid {out:.0f} us")
    assert out < 3 * base


@pytest.mark.parametrize("n, h", [(1, 0.0125), (1000, 0.006), (4096, 0.0125), (4096, 0.006), (4096, 0.0041)])
def test_scattered_scene(fluid, scene, n, h):
    """A window of up to 28 million cells, most of them empty, whose starts come from
    the sorted keys."""
    x = scene.uniform01(4, 3 * n).reshape(-1, 3).astype(np.float32)
    lists = []
    for batch in (False, True):
        ctx = fluid.Context("cuda:0", smoothing_length=h, stage_min_particles=-1)
        xd, vd = dev(x), torch.zeros((n, 3), dtype=torch.float32, device="cuda:0")
        if batch:
            ctx.batch_step(xd, vd, torch.tensor([0, n, n], dtype=torch.int32, device="cuda:0"))
        else:
            ctx.step(xd, vd)
        nl = ctx.step_neighbors(n)
        lists.append([t.cpu().numpy() for t in (xd, vd, nl.index, nl.elements)])
    for a, b in zip(*lists):
        np.testing.assert_array_equal(a, b)
    if h >= 0.006:
        base, wide = step_time(fluid, block(scene, n), h), step_time(fluid, x, h)
        say(f"a step of {n} particles, h {h}: in a block {base:.0f} us, scattered {wide:.0f} us")
        assert wide < 2 * base
