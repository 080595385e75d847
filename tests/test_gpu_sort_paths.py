"""The sort's forms against each other: one workgroup (one scene, at most 4,096
particles), the bounds pass whose last block makes the window (one scene, at
most 262,144) and the separate windows kernel. A batch of the scene and an empty
one takes the general form; both give the same bits over two steps (caller's
order and cell order) and the same lists. Every call goes through the C ABI."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from parity_util import dev, say  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def lattice(scene, n, origin=(0.2, 0.3, 0.2)):
    side = int(np.ceil(n ** (1 / 3) - 1e-9))
    return scene.jittered_lattice((side, side, side), origin, 0.005, 0.1, seed=n, count=n)


def inputs(scene, name):
    if name.startswith("lattice"):
        return lattice(scene, int(name.split()[1]))
    if name == "wide window":  # more cells than buckets, many of them in one bucket
        x = np.concatenate([lattice(scene, 3000), scene.uniform01(3, 3 * 900).reshape(-1, 3).astype(np.float32)])
        return np.ascontiguousarray(x[np.random.default_rng(1).permutation(len(x))])
    if name == "scattered":
        return scene.uniform01(4, 3 * 4096).reshape(-1, 3).astype(np.float32)
    if name == "dense cells":  # cells of several hundred particles
        return scene.gaussian_blobs(1, 4000, 0.012, seed=5)
    x = lattice(scene, 3500, (-0.08, 0.5, 0.3))  # partly outside the grid
    if name == "not finite":
        x[::97] = np.nan
        x[5] = np.inf
    return x


@pytest.mark.parametrize("name", ["lattice 1", "lattice 64", "lattice 1023", "lattice 1025", "lattice 4096",
                                  "lattice 4097", "lattice 262144", "lattice 262145", "wide window", "scattered",
                                  "dense cells", "out of the grid", "not finite"])
def test_one_scene_equals_batch_with_an_empty_scene(fluid, scene, name):
    x = inputs(scene, name)
    n = len(x)
    say(f"sort of one scene against a batch with an empty scene: {name}, {n} particles")
    v = (0.05 * (scene.uniform01(6, 3 * n).reshape(n, 3) - 0.5)).astype(np.float32)
    outs = []
    for batch in (False, True):
        ctx = fluid.Context("cuda:0", stage_min_particles=-1)
        got = []
        for steps in (1, 2):
            xd, vd, rho = dev(x), dev(v), torch.zeros(n, dtype=torch.float32, device="cuda:0")
            if batch:
                off = torch.tensor([0, n, n], dtype=torch.int32, device="cuda:0")
                ctx.batch_step(xd, vd, off, rho, steps)
            else:
                ctx.step(xd, vd, rho, steps)
            nl = ctx.step_neighbors(n)
            got += [t.cpu().numpy().view(np.uint32) for t in (xd, vd, rho)] + [nl.index.cpu().numpy(),
                                                                              nl.elements.cpu().numpy()]
        st = ctx.stats()
        outs.append(got + [(st["neighbor_pairs"], st["candidates"], st["out_of_grid"], st["nonfinite"])])
    for a, b in zip(*outs):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("sizes", [(700, 400, 3000), (1, 0, 2, 1020, 1, 5, 1023, 1024, 1025, 90), tuple(range(1, 90))])
def test_scenes_that_share_blocks(fluid, scene, sizes):
    """Scenes that begin and end inside the bounds pass's blocks of 1,024
    particles, few and many of them in one block, each equal to its own run."""
    say(f"scenes that share bounds blocks: {len(sizes)} scenes, {sum(sizes)} particles")
    xs = [lattice(scene, k, (0.2, 0.3, 0.2) if s % 3 else (-0.035, 0.3, 0.2)) if k else np.zeros((0, 3), np.float32)
          for s, k in enumerate(sizes)]
    off = torch.from_numpy(np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)).cuda()
    x = dev(np.concatenate(xs))
    v = torch.zeros_like(x)
    ctx = fluid.Context("cuda:0")
    ctx.batch_step(x, v, off, None, 2)
    one = fluid.Context("cuda:0")
    start = 0
    for p in xs:
        if len(p):
            xd, vd = dev(p), dev(np.zeros_like(p))
            one.step(xd, vd, None, 2)
            for a, b in ((x, xd), (v, vd)):
                np.testing.assert_array_equal(a[start:start + len(p)].cpu().numpy(), b.cpu().numpy())
        start += len(p)
