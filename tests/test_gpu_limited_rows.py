"""Limited rows (NeighborQuery::queryNeighborFixed) at the row lengths where the
kernel changes its way: few places are extracted one by one, many ranked, and a
row of more than 120 neighbors drops keys between its list chunks. Clusters of
every such size, each within h of itself and far from the others, on a coarse grid
of positions, so that many distances tie and the ids decide. Whole numbers: exact."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from parity_util import dev, say  # noqa: E402

SIZES = (1, 2, 7, 8, 9, 15, 28, 31, 56, 63, 64, 65, 76, 77, 78, 112, 119, 120, 121, 126, 127, 128, 129, 136, 137, 184,
         185, 192, 193, 257, 420)
LIMITS = (1, 2, 3, 4, 8, 9, 11, 12, 16, 17, 18, 19, 31, 32)


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


@pytest.mark.parametrize("storage", ["list", "staged", "masks"])
@pytest.mark.parametrize("shuffled", [False, True])
@pytest.mark.parametrize("spacings", [2.5, 1.2])  # 1.2: a new context's first query runs one lane per particle
def test_limits_and_row_lengths(fluid, storage, shuffled, spacings):
    say(f"limited rows of {LIMITS}, rows of {SIZES}, {storage}, {spacings} spacings in h")
    rng = np.random.default_rng(5)
    parts = []
    for k, m in enumerate(SIZES):
        at = np.array([0.1 + 0.12 * (k % 6), 0.3, 0.1 + 0.12 * (k // 6)])
        parts.append(at + rng.integers(0, 5, (m, 3)) * 2.0 ** -10)  # 4 sqrt(3) / 1024 < h
    x = np.concatenate(parts).astype(np.float32)
    if shuffled:
        x = np.ascontiguousarray(x[rng.permutation(len(x))])
    n = len(x)
    opts = dict(sampling_distance=0.0125 / spacings, list_slots=4 if storage == "masks" else 448)
    if storage == "staged":
        opts["stage_min_particles"] = 1
    ctx = fluid.Context("cuda:0", **opts)
    xd = dev(x)
    f = np.float32
    near, order = [], []
    for i in range(n):
        d = (x[i] - x).astype(f)
        r = np.sqrt((d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2])
        ids = np.flatnonzero(r < f(0.0125))
        near.append(len(ids))
        order.append(ids[np.lexsort((ids, r[ids]))])
    assert sorted(set(near)) == sorted(SIZES)
    for limit in LIMITS:
        if spacings < 1.4:
            ctx = fluid.Context("cuda:0", **opts)
        nl = ctx.neighbor_query_fixed(xd, limit)
        counts, el = nl.index.cpu().numpy(), nl.elements.cpu().numpy().reshape(n, limit)
        np.testing.assert_array_equal(counts, np.minimum(near, limit))
        want = np.full((n, limit), -1, np.int32)
        for i in range(n):
            want[i, :counts[i]] = order[i][:limit]
        np.testing.assert_array_equal(el, want)


@pytest.mark.parametrize("n", [65535, 65536])
def test_one_lane_and_eight_agree(fluid, scene, n):
    """Four places (one lane per particle from 65,536 particles on) are the first four of
    five (eight lanes)."""
    say(f"limited rows of 4 and 5, {n} particles")
    x = scene.jittered_lattice((64, 32, 32), (0.2, 0.3, 0.2), 0.005, 0.1, seed=3)[:n]
    ctx = fluid.Context("cuda:0")
    rows = [ctx.neighbor_query_fixed(dev(x), k).elements.cpu().numpy().reshape(n, k) for k in (4, 5)]
    np.testing.assert_array_equal(rows[0], rows[1][:, :4])
    assert (rows[0] >= 0).all()
