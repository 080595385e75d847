"""The passes over lists of few neighbors per row (a mean of at most 7: one lane
per row) around that line, against double-precision numpy with the bars of
test_gpu_csr_rows.py, and against four lanes per row where the order of the sums
is the same."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from parity_util import RHO_REL, V_ABS, X_ABS, dev, rel_err, say  # noqa: E402
from test_gpu_csr_rows import block, need_gpu, rows_of, scatter, to_list  # noqa: E402,F401

LINE = 7


@pytest.mark.parametrize("mass", [False, True])
@pytest.mark.parametrize("form", ["both_ways", "one_way", "few_long_rows", "empty"])
def test_constrain_short_rows(fluid, scene, form, mass):
    x, a = block(scene)
    n = len(x)
    rng = np.random.default_rng(17)
    v = (0.05 * rng.standard_normal((n, 3))).astype(np.float32)
    keep = np.triu(rng.random((n, n)) < 0.06, 1)
    if form == "both_ways":
        a = a * (keep | keep.T)
    elif form == "one_way":
        a = a * keep
    elif form == "few_long_rows":  # 0 entries in most rows, up to a hundred in some
        a[np.setdiff1d(np.arange(n), np.arange(5, n, 19))] = 0
    else:
        a = np.zeros_like(a)
    assert a.sum() <= LINE * n
    say(f"DensityPBD::constrain over a {form} list{' with masses' if mass else ''}: {n} rows of "
        f"{a.sum(1).min()}..{a.sum(1).max()} entries, {a.sum() / n:.2f} in the mean")
    minv = (0.5 + rng.random(n)).astype(np.float32) if mass else None
    # a low rest density: lambda is active in rows of a few entries too
    ctx = fluid.Context("cuda:0", iterations=3, lambda_rest=100.0)
    st = ctx.stats()
    p = dict(ctx.params(), cw=st["density_factor"] * st["particle_mass"] * 15.0 / (np.pi * float(np.float32(0.0125)) ** 3))
    want, single = (scatter(f, p, x, v, a, 3, minv) for f in (np.float64, np.float32))
    xd, vd, rho = dev(x), dev(v), torch.zeros(n, dtype=torch.float32, device="cuda:0")
    nl = to_list(fluid, rows_of(a, rng))
    if mass:
        ctx.pbd_constrain_mass(xd, vd, nl, dev(minv), rho)
    else:
        ctx.pbd_constrain(xd, vd, nl, rho)
    assert form == "empty" or np.abs(want[0] - x).max() > 1e-5
    got, ref = rho.cpu().numpy(), want[2]
    some = ref > 0
    off = [np.abs(g - w).max() for g, w in zip((xd.cpu().numpy(), vd.cpu().numpy()), want)]
    off32 = [np.abs(g - w).max() for g, w in zip(single[:2], want[:2])]
    off.append(rel_err(got[some], ref[some]).max() if some.any() else 0.0)
    off32.append(rel_err(single[2][some], ref[some]).max() if some.any() else 0.0)
    say(f"from double (x, v, rho): GPU {off}, single precision {off32}")
    assert all(o <= max(bar, 2 * o32) for o, o32, bar in zip(off, off32, (X_ABS, V_ABS, RHO_REL)))
    assert (got[~some] == 0).all()


@pytest.mark.parametrize("n", [1, 63, 300, 5000])
def test_line_between_one_and_four_lanes(fluid, scene, n):
    """7 n entries, and one more in the last row: the density's terms are added in the
    row's order either way, so the other rows' densities are the same bits; the
    viscosity's sums are the lanes' (each within 16 roundings of the other's)."""
    say(f"lists of 7 n and 7 n + 1 entries, {n} rows")
    rng = np.random.default_rng(n)
    side = int(np.ceil(n ** (1 / 3)))
    x = scene.jittered_lattice((side, side, side), (0.3, 0.3, 0.3), 0.0042, 0.1, seed=5)[:n]
    v = rng.standard_normal((n, 3)).astype(np.float32)
    cuts = np.sort(rng.integers(0, LINE * n + 1, n - 1))
    lengths = np.diff(np.concatenate([[0], cuts, [LINE * n]]))
    rows = [np.clip(i + rng.integers(-3, 4, k), 0, n - 1) for i, k in enumerate(lengths)]
    ctx = fluid.Context("cuda:0", viscosity_iterations=1)
    rhos, vs = [], []
    for extra in (0, 1):
        rows[-1] = np.concatenate([rows[-1], np.full(extra, n - 1)])
        nl = to_list(fluid, rows)
        assert nl.elements.numel() == LINE * n + extra
        rho, vd = torch.zeros(n, dtype=torch.float32, device="cuda:0"), dev(v)
        ctx.density(dev(x), nl, rho)
        ctx.viscosity(dev(x), vd, nl)
        rhos.append(rho.cpu().numpy())
        vs.append(vd.cpu().numpy())
    np.testing.assert_array_equal(rhos[0][:-1].view(np.uint32), rhos[1][:-1].view(np.uint32))
    assert np.abs(vs[0][:-1] - vs[1][:-1]).max(initial=0.0) <= 16 * 2.0 ** -24 * np.abs(v).max()
