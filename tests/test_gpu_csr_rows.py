"""The passes over neighbor lists by row (several lanes per row) at the row
lengths where their groups begin and end, against double-precision numpy.

DensityPBD::constrain takes any list: one with every pair listed both ways runs
without atomics, every other one as the reference's pairwise scatter. Each form
is held against a literal scatter in double (dp_ij to i, -dp_ij to j for every
listed pair, K_ComputeDisplacement, DensityPBD.cu:135-179) with the bars of the
step parity: 1e-6 m, 1e-3 m/s and 1e-5 of the density, or twice what the same
scatter in single precision is from it. The limited rows and the list export are whole numbers: exact.
Every call goes through the C ABI."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from parity_util import RHO_REL, V_ABS, X_ABS, dev, rel_err, say  # noqa: E402

H = np.float64(np.float32(0.0125))


@pytest.fixture(scope="module", autouse=True)
def need_gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def block(scene, seed=31):
    """A compressed block (lambda is active) and its neighbor matrix."""
    x = scene.jittered_lattice((9, 8, 7), (0.3, 0.5, 0.3), 0.0042, 0.1, seed=seed)
    d = x[:, None, :].astype(np.float64) - x[None, :, :].astype(np.float64)
    return x, ((d ** 2).sum(-1) < H * H).astype(np.int64)


def rows_of(a, rng):
    """The multiset matrix a (a_ij: how often row i lists j) as rows in random order."""
    out = []
    for r in a:
        row = np.repeat(np.arange(len(r)), r)
        rng.shuffle(row)
        out.append(row)
    return out


def to_list(fluid, rows):
    index = np.concatenate([[0], np.cumsum([len(r) for r in rows])])[:-1].astype(np.int32)
    el = np.concatenate(rows).astype(np.int32)
    return fluid.NeighborList(torch.from_numpy(index).cuda(), torch.from_numpy(el).cuda())


def scatter(f, p, x, v, a, iterations, minv=None):
    """K rounds over the multiset matrix a in the type f, as the reference's scatter."""
    a = a.astype(f)
    h, eps, rest = f(p["smoothing_length"]), f(p["lambda_eps"]), f(p["lambda_rest"])
    cw = f(p["cw"])
    cg = f(-45.0 / (np.pi * H ** 3))
    minv = np.ones(len(x), f) if minv is None else minv.astype(f)
    q = x.astype(f)
    rho = None
    for _ in range(iterations):
        d = q[:, None, :] - q[None, :, :]
        r = np.sqrt((d ** 2).sum(-1))
        t = np.clip(f(1) - r / h, f(0), None)
        rho = cw * (a * t ** 3).sum(1)
        far = r > f(p["pair_eps"])
        g = np.where(far, cg * t * t / np.where(far, r, f(1)), f(0))[:, :, None] * d
        G = (a[:, :, None] * g).sum(1)
        S = (a * (g ** 2).sum(-1) * minv[None, :]).sum(1) + (G ** 2).sum(1) * minv
        lam = np.minimum(f(0), -(rho - rest) / (S + eps))
        dp = f(p["corr_scale"]) * (lam[:, None] + lam[None, :])[:, :, None] * g * a[:, :, None]
        q = q + (dp.sum(1) - dp.sum(0)) * minv[:, None]
    return q, v.astype(f) + (q - x.astype(f)) / f(p["dt"]), rho


@pytest.mark.parametrize("mass", [False, True])
@pytest.mark.parametrize("form", ["both_ways", "one_sided", "one_missing", "double_both_ways", "double_one_way",
                                  "empty_rows"])
def test_constrain_list_forms(fluid, scene, form, mass):
    x, a = block(scene)
    n = len(x)
    rng = np.random.default_rng(7)
    v = (0.05 * rng.standard_normal((n, 3))).astype(np.float32)
    if form == "one_sided":
        a = a * (rng.random((n, n)) < 0.7)
    elif form == "one_missing":
        a[200, np.flatnonzero(a[200])[-1]] = 0
    elif form == "double_both_ways":
        twice = np.triu(rng.random((n, n)) < 0.1, 1)
        a = a * (1 + (twice | twice.T))
    elif form == "double_one_way":
        # as many entries above the diagonal as below it, but not pair by pair
        i, j = np.argwhere(np.triu(a, 1))[:: len(a)][:2].T
        a[i[0], j[0]] += 1
        a[j[1], i[1]] += 1
    elif form == "empty_rows":
        gone = rng.permutation(n)[:64]
        a[gone] = 0
        a[:, gone] = 0
    say(f"DensityPBD::constrain over a {form} list{' with masses' if mass else ''}: {n} rows of "
        f"{a.sum(1).min()}..{a.sum(1).max()} entries")
    minv = (0.5 + rng.random(n)).astype(np.float32) if mass else None
    ctx = fluid.Context("cuda:0", iterations=3)
    st = ctx.stats()
    p = dict(ctx.params(), cw=st["density_factor"] * st["particle_mass"] * 15.0 / (np.pi * H ** 3))
    want, single = (scatter(f, p, x, v, a, 3, minv) for f in (np.float64, np.float32))
    xd, vd, rho = dev(x), dev(v), torch.zeros(n, dtype=torch.float32, device="cuda:0")
    nl = to_list(fluid, rows_of(a, rng))
    if mass:
        ctx.pbd_constrain_mass(xd, vd, nl, dev(minv), rho)
    else:
        ctx.pbd_constrain(xd, vd, nl, rho)
    assert np.abs(want[0] - x).max() > 1e-5  # the constraint moves particles
    got, ref = rho.cpu().numpy(), want[2]
    some = ref > 0
    off = [np.abs(g - w).max() for g, w in zip((xd.cpu().numpy(), vd.cpu().numpy()), want)]
    off32 = [np.abs(g - w).max() for g, w in zip(single[:2], want[:2])]
    off.append(rel_err(got[some], ref[some]).max())
    off32.append(rel_err(single[2][some], ref[some]).max())
    say(f"from double (x, v, rho): GPU {off}, single precision {off32}")
    assert all(o <= max(bar, 2 * o32) for o, o32, bar in zip(off, off32, (X_ABS, V_ABS, RHO_REL)))
    assert (got[~some] == 0).all()


def test_density_and_viscosity_row_lengths(fluid, scene):
    """Rows of every length from 0 to 70: one lane, part of a group, several groups.
    t = 1 - r/h cancels: its error is absolute, a few ulps of 1 (reciprocal
    square root 2, products and the difference 1 each: at most 8 * 2^-24), which
    enters each term as 3 t^2 dt; the sums' own rounding is within RHO_REL."""
    say("SummationDensity and ImplicitViscosity over rows of 0..70 entries")
    x, a = block(scene)
    n = len(x)
    rng = np.random.default_rng(9)
    v = rng.standard_normal((n, 3)).astype(np.float32)
    rows = [rng.integers(0, n, k % 71) for k in range(n)]
    ctx = fluid.Context("cuda:0", viscosity_iterations=1)
    st = ctx.stats()
    p = ctx.params()
    nl = to_list(fluid, rows)
    rho, vd = torch.zeros(n, dtype=torch.float32, device="cuda:0"), dev(v)
    ctx.density(dev(x), nl, rho)
    ctx.viscosity(dev(x), vd, nl)
    b = p["dt"] * p["viscosity"] / H
    for i, row in enumerate(rows):
        r = np.sqrt(((x[i].astype(np.float64) - x[row]) ** 2).sum(1))
        t = np.clip(1 - r / H, 0, None)
        cw = st["density_factor"] * st["particle_mass"] * 15 / (np.pi * H ** 3)
        want = cw * (t ** 3).sum()
        assert abs(float(rho[i]) - want) <= RHO_REL * want + cw * (3 * t * t * 8 * 2.0 ** -24).sum()
        w = t * (r > p["pair_eps"])
        if w.sum() > 0:
            mean = (w[:, None] * v[row]).sum(0) / w.sum()
            assert np.abs(vd[i].cpu().numpy() - (v[i] + mean * b) / (1 + b)).max() <= 1e-5


@pytest.mark.parametrize("storage, spacing", [("list", 0.0061), ("list", 0.0028), ("staged", 0.0061),
                                              ("staged", 0.0028), ("masks", 0.0061), ("masks", 0.0028),
                                              ("index32", 0.005)])
def test_limited_rows_and_export(fluid, scene, storage, spacing):
    """Limited rows of 1, 20 and 32 and the exported list, over rows of up to 45
    (spacing 0.0061), 81 (0.005; a slab whose cell planes hold 41k particles, so
    that waves keep 32-bit lists) and over 300 neighbors (0.0028, several
    rounds), against a search over all particles."""
    if storage == "index32":
        x = scene.jittered_lattice((128, 128, 8), (0.18, 0.18, 0.4), spacing, 0.1, seed=6)
    else:
        x = scene.jittered_lattice((14, 13, 11), (0.3, 0.5, 0.3), spacing, 0.1, seed=33)
        x = np.ascontiguousarray(x[np.random.default_rng(11).permutation(len(x))])
    n = len(x)
    opts = {"staged": dict(stage_min_particles=1), "masks": dict(list_slots=4)}.get(storage, {})
    ctx = fluid.Context("cuda:0", **opts)
    xd = dev(x)
    for _ in range(2):  # the second search has lists as long as it needs
        nl = ctx.neighbor_query(xd)
        torch.cuda.synchronize()
    got = nl.rows()
    limits = (1, 20, 32)
    fixed = [(r.elements.cpu().numpy(), r.index.cpu().numpy())
             for r in (ctx.neighbor_query_fixed(xd, k) for k in limits)]
    f = np.float32
    longest = 0
    for i in range(0, n, max(1, n // 400)):
        d = (x[i] - x).astype(f)
        r = np.sqrt((d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2])
        near = np.flatnonzero(r < f(0.0125))
        longest = max(longest, len(near))
        np.testing.assert_array_equal(np.sort(got[i]), near)
        order = near[np.lexsort((near, r[near]))]
        for k, (el, counts) in zip(limits, fixed):
            assert counts[i] == min(k, len(near))
            np.testing.assert_array_equal(el[k * i:k * i + counts[i]], order[:k])
            assert (el[k * i + counts[i]:k * (i + 1)] == -1).all()
    say(f"limited rows and export, {storage}, spacing {spacing}: {n} particles, rows of up to {longest}")
    assert longest > (128 if spacing < 0.005 else 32)


def test_viscosity_workgroup_sizes(fluid, scene):
    """65,536 rows (workgroups of 64 threads) and the same with one isolated
    particle more (256): the same bits for the rows they share."""
    say("viscosity over 65,536 and 65,537 rows")
    x = scene.jittered_lattice((64, 32, 32), (0.2, 0.3, 0.2), 0.005, 0.1, seed=3)
    n = len(x)
    v = (0.5 * (scene.uniform01(4, 3 * n).reshape(n, 3) - 0.5)).astype(np.float32)
    outs = []
    for extra in (0, 1):
        xa = np.concatenate([x, np.full((extra, 3), 0.9, np.float32)])
        va = np.concatenate([v, np.zeros((extra, 3), np.float32)])
        ctx = fluid.Context("cuda:0")
        xd, vd = dev(xa), dev(va)
        ctx.viscosity(xd, vd, ctx.neighbor_query(xd))
        outs.append(vd.cpu().numpy()[:n].view(np.uint32))
    np.testing.assert_array_equal(*outs)
