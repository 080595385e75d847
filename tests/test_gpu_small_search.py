"""The neighbor pass with several lanes per particle (small unstaged searches)
against the one with one lane per particle, which staged lists select: one step
gives the same bits (x, v, density) and the exported lists hold the same
elements in the same order, at the sizes and shapes where the cooperative
kernel's rounds, list pieces and workgroups begin and end, and where it keeps
bit masks or none of both. Every call goes through the C ABI."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from parity_util import dev, say  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def line(n, spacing):
    """n particles on a line along x: one run holds nearly all candidates."""
    x = np.full((n, 3), 0.5, np.float32)
    x[:, 0] = 0.1 + spacing * np.arange(n)
    return x


def scenes(scene):
    lat = scene.jittered_lattice
    return {
        "1": lat((1, 1, 1), (0.3, 0.5, 0.3), 0.005, 0.1, seed=1),
        "63": lat((7, 3, 3), (0.3, 0.5, 0.3), 0.005, 0.1, seed=2),
        "65": lat((13, 5, 1), (0.3, 0.5, 0.3), 0.005, 0.1, seed=3),
        "4096": lat((16, 16, 16), (0.3, 0.5, 0.3), 0.005, 0.1, seed=4),
        "rows of 8 to 56 candidates": np.concatenate([line(400, s) for s in (0.002, 0.0008, 0.0007, 0.0006)]
                                                     + [line(100, 0.0003) + np.float32(0.2)]),
        "rows of over 128 entries": lat((14, 13, 11), (0.3, 0.5, 0.3), 0.0028, 0.1, seed=33),
        "blob": scene.gaussian_blobs(1, 6000, 0.012, seed=7),
        "out of the grid": lat((20, 16, 20), (-0.04, 0.5, 0.3), 0.005, 0.1, seed=8),
        "65536": lat((64, 32, 32), (0.3, 0.5, 0.3), 0.005, 0.1, seed=5),
    }


NAMES = ["1", "63", "65", "4096", "rows of 8 to 56 candidates", "rows of over 128 entries", "blob", "out of the grid",
         "65536"]


@pytest.mark.parametrize("reserve", [{}, {"list_slots": 4}, {"list_slots": 4, "mask_words": 512}])
@pytest.mark.parametrize("name", NAMES)
def test_several_lanes_equal_one(fluid, scene, name, reserve):
    x = scenes(scene)[name]
    n = len(x)
    say(f"neighbor pass with several lanes per particle, {name}: {n} particles, {reserve}")
    v = (0.05 * (scene.uniform01(5, 3 * n).reshape(n, 3) - 0.5)).astype(np.float32)
    outs = []
    for smin in (-1, 1):  # never / always staged
        ctx = fluid.Context("cuda:0", stage_min_particles=smin, **reserve)
        for _ in range(2):  # the second call has its reservations as long as it needs
            xd, vd, rho = dev(x), dev(v), torch.zeros(n, dtype=torch.float32, device="cuda:0")
            ctx.step(xd, vd, rho)
            torch.cuda.synchronize()
        nl = ctx.step_neighbors(n)
        st = ctx.stats()
        outs.append([t.cpu().numpy() for t in (xd, vd, rho, nl.index, nl.elements)]
                    + [(st["neighbor_pairs"], st["candidates"], st["out_of_grid"])])
    for a, b in zip(*outs):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("n", [1000, 40000])
def test_lists_after_a_replayed_step(fluid, scene, n):
    """step_neighbors exports the search of a step that a replayed graph ran
    after an earlier export (the row starts are kept between the exports)."""
    say(f"lists of a replayed step, {n} particles")
    side = int(np.ceil(n ** (1 / 3)))
    far, near = (scene.jittered_lattice((side,) * 3, (0.2, 0.3, 0.2), d, 0.1, seed=2, count=n)
                 for d in (0.007, 0.005))
    ctx = fluid.Context("cuda:0")
    x, v = dev(near), dev(np.zeros_like(near))
    ctx.step(x, v)  # reservations for the longer lists
    torch.cuda.synchronize()
    ctx.stats()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, capture_error_mode="relaxed"):
        ctx.step(x, v)
    for start in (far, near, far):
        x.copy_(dev(start))
        v.zero_()
        graph.replay()
        got = ctx.step_neighbors(n)
        one = fluid.Context("cuda:0")
        xd, vd = dev(start), dev(np.zeros_like(start))
        one.step(xd, vd)
        want = one.step_neighbors(n)
        torch.cuda.synchronize()
        for a, b in ((x, xd), (got.index, want.index), (got.elements, want.elements)):
            np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy())
