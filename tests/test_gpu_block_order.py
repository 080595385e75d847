"""The passes' block order: a batch of 262,144 particles and more whose neighbor
pairs are spread unevenly over its eighths goes to the chip in chunks, a scene
below that size in contiguous eighths. Each scene of an uneven batch ends on the
same bits as its own run, forward (the plain step, and the step with the
viscosity solve) and backward (a rollout's gradients)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from parity_util import dev, say  # noqa: E402


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def scenes(scene, order):
    side = 61
    even = scene.jittered_lattice((side,) * 3, (0.2, 0.3, 0.2), 0.005, 0.1, seed=1)  # 226,981 of 80 neighbors
    dense = scene.gaussian_blobs(1, 40013, 0.03, seed=5)  # about 280 neighbors on average
    out = [dense, even] if order == "dense first" else [even, dense]
    assert sum(map(len, out)) >= 1 << 18 > max(map(len, out))
    return [(x, (0.05 * (scene.uniform01(6, 3 * len(x)).reshape(-1, 3) - 0.5)).astype(np.float32)) for x in out]


def even_scene():
    i = np.indices((65,) * 3).reshape(3, -1).T
    x = (0.2 + 0.0051 * i).astype(np.float32)
    assert len(x) >= 1 << 18
    return x


def run(fluid, parts, kind):
    """x, v (and rho, or the gradients) of the scenes as one batch; of one scene, alone."""
    off = np.concatenate([[0], np.cumsum([len(x) for x, _ in parts])]).astype(np.int32)
    off_d = torch.from_numpy(off).cuda() if len(parts) > 1 else None
    x, v = (dev(np.concatenate(a)) for a in zip(*parts))
    n = int(off[-1])
    if kind == "gradients":
        ctx = fluid.Context("cuda:0", iterations=2)
        ctx.rollout_forward(x, v, None, 2, 1, off_d)
        xb, vb = torch.ones_like(x), torch.full_like(v, 0.5)
        ctx.rollout_backward(xb, vb)
        out = (x, v, xb, vb)
    else:
        rho = torch.zeros(n, dtype=torch.float32, device="cuda:0")
        ctx = fluid.Context("cuda:0", flags=fluid._capi.PBF_FLAG_VISCOSITY if kind == "viscosity" else 0)
        if kind == "after an even search":  # the context expects another one
            e = dev(even_scene())
            ctx.step(e, torch.zeros_like(e))
            torch.cuda.synchronize()
        if off_d is None:
            ctx.step(x, v, rho, 3)
        else:
            ctx.batch_step(x, v, off_d, rho, 3)
        out = (x, v, rho)
    out = [t.cpu().numpy().view(np.uint32) for t in out]
    return [[t[a:b] for t in out] for a, b in zip(off[:-1], off[1:])]


@pytest.mark.parametrize("order", ["dense first", "dense last"])
@pytest.mark.parametrize("kind", ["plain", "viscosity", "gradients", "after an even search"])
def test_uneven_batch_equals_its_scenes(fluid, scene, kind, order):
    parts = scenes(scene, order)
    say(f"uneven batch of {sum(len(x) for x, _ in parts)} particles, {kind}, {order}")
    for got, part in zip(run(fluid, parts, kind), parts):
        for a, b in zip(got, run(fluid, [part], kind)[0]):
            np.testing.assert_array_equal(a, b)
