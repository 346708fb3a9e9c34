"""Small accumulates and sorts at the edges of their tiles: the input-order
disc kernel in tiles of 64 and of 256, the cell-ordered kernels with segments
of one to five tiles, and sorts of 512- and 2048-item tiles."""
import numpy as np
import pytest

from tests.test_gpu_parity import big, block_rel_eof, block_rel_sl, disc_halo, f32, relmax  # noqa: F401
from oracle import bfe_oracle as O

pytestmark = pytest.mark.gpu

# a term carries at most about six float32 roundings (3.6e-7 of itself, random
# signs), a group of 16 three more of its sum; blocks are compared at their
# largest coefficient
TOL = 2e-6


@pytest.fixture(scope="module")
def particles():
    return [f32(*p) for p in disc_halo(4 * 64 * 1024 + 1, 77)]


@pytest.mark.parametrize("omin", [1 << 40, 1], ids=["input", "cells"])
@pytest.mark.parametrize("n", [1, 15, 17, 63, 64, 65, 255, 257, 511, 513, 1300, 65535, 65536, 65537])
def test_accumulate_edges(big, particles, n, omin):  # noqa: F811
    s, slo, eo = big
    d, h = [[a[:n] for a in p] for p in particles]
    rc, rs = O.eof_accumulate(eo, *d)
    ref = O.sl_accumulate(slo, *h)
    s.set_tuning("order_min", omin)
    c, sn = (v.cpu().numpy() for v in s.eof_accumulate(*d))
    g = s.sl_accumulate(*h).cpu().numpy()
    s.set_tuning("order_min", 65536)
    assert block_rel_eof(c, rc) <= TOL and block_rel_eof(sn[1:], rs[1:]) <= TOL
    assert block_rel_sl(g, ref, slo.lmax) <= TOL


@pytest.mark.parametrize("n", [2, 511, 512, 513, 1025, 262143, 262144, 262145])
def test_sort_edges(big, particles, n):  # noqa: F811
    """Evaluation in cell order writes every point once, with the input-order bits."""
    import torch
    s, _, _ = big
    d, h = particles
    s.set_field(*s.eof_accumulate(*d), s.sl_accumulate(*h))
    x, y, z = (np.concatenate([a[:n // 2], b[:n - n // 2]]) for a, b in zip(d[:3], h[:3]))
    out = []
    for omin in (1, 1 << 40):
        s.set_tuning("order_min", omin)
        out.append(s.field_forces(x, y, z, rotpos=0.1))
    s.set_tuning("order_min", 65536)
    for a, b in zip(*out):
        assert (a is None and b is None) or torch.equal(a, b)


@pytest.mark.parametrize("omin", [1 << 40, 1], ids=["input", "cells"])
@pytest.mark.parametrize("nsnap", [2, 127, 128, 129, 257])
def test_batch_pieces_edges(nsnap, omin):
    """Batches around the 128 snapshots of a table chunk, with empty snapshots
    and snapshots at the edges of a segment and a tile: every snapshot as its
    own call (another segment plan regroups the float32 sums), every point's
    bits as in its own field."""
    import torch
    from exptool_amd.bfe import BFESystem
    from exptool_amd.utils import workloads as W
    st, et = W.disc_halo_tables(seed=2, n_eof_sample=4000, lmax_s=10, nmax_s=8,
                                eof=dict(mmax=3, norder=6, numx=24, numy=16),
                                sl=dict(lmax=3, nmax=6, numr=200))
    s = BFESystem(sl=st, eof=et)
    rng = np.random.default_rng(nsnap)
    counts = rng.choice([0, 1, 63, 64, 65, 255, 256, 257, 511, 512, 513, 1500], nsnap)
    counts[:2] = (0, 513)
    d, h = W.disc_halo_particles(int(counts.sum()), int(counts.sum()), seed=8)
    d, h = ([torch.tensor(np.asarray(a, np.float32), device="cuda") for a in p] for p in (d, h))
    s.set_tuning("order_min", omin)
    c, sn = s.eof_accumulate_batch(*d, counts)
    hl = s.sl_accumulate_batch(*h, counts)
    s.set_field_batch(c, sn, hl)
    f = s.field_forces_batch(*h[:3], counts, rotpos=0.3)
    o = np.concatenate([[0], np.cumsum(counts)])
    for q in sorted({0, 1, 2 % nsnap, nsnap // 2, nsnap - 2, nsnap - 1}):
        a, b = int(o[q]), int(o[q + 1])
        cq, sq = (v.cpu().numpy() for v in s.eof_accumulate(*(v[a:b] for v in d)))
        hq = s.sl_accumulate(*(v[a:b] for v in h)).cpu().numpy()
        assert block_rel_eof(c[q].cpu().numpy(), cq) <= TOL
        assert block_rel_eof(sn[q].cpu().numpy()[1:], sq[1:]) <= TOL
        assert block_rel_sl(hl[q].cpu().numpy(), hq, 3) <= TOL
        if b > a:
            s.set_field(c[q], sn[q], hl[q])
            for u, v in zip(f, s.field_forces(*(v[a:b] for v in h[:3]), rotpos=0.3)):
                assert torch.equal(u[a:b], v)


@pytest.mark.parametrize("nset", [1, 2, 5, 6, 7, 13])
@pytest.mark.parametrize("lmax,mmax,numr,numx,numy", [(0, 0, 4, 8, 6), (3, 3, 5, 9, 6), (6, 4, 201, 20, 15),
                                                      (9, 8, 64, 31, 17)])
def test_folds_of_a_batch_equal_single_folds(nset, lmax, mmax, numr, numx, numy):
    """Batch folds (several sets a block) and the two folds of one field in one
    launch, at sizes that leave remainders of the node and row groups: every
    point's bits as with the separate single folds of the point evaluators'
    kernels (per-set fields), and the field of the oracle."""
    import torch
    from exptool_amd.bfe import BFESystem
    from exptool_amd.utils import workloads as W
    st, et = W.disc_halo_tables(seed=2, n_eof_sample=3000, lmax_s=10, nmax_s=8,
                                eof=dict(mmax=mmax, norder=5, numx=numx, numy=numy),
                                sl=dict(lmax=lmax, nmax=7, numr=numr))
    s = BFESystem(sl=st, eof=et)
    d, h = W.disc_halo_particles(64 * nset, 64 * nset, seed=3)
    d, h = ([torch.tensor(np.asarray(a, np.float32), device="cuda") for a in p] for p in (d, h))
    counts = [64] * nset
    c, sn = s.eof_accumulate_batch(*d, counts)
    hl = s.sl_accumulate_batch(*h, counts)
    s.set_field_batch(c, sn, hl)
    f = s.field_forces_batch(*d[:3], counts)
    for q in range(nset):
        s.set_field(c[q], sn[q], hl[q])
        for u, v in zip(f, s.field_forces(*(v[64 * q:64 * q + 64] for v in d[:3]))):
            assert torch.equal(u[64 * q:64 * q + 64], v)
    slo = O.SLTable(st["lmax"], st["nmax"], st["numr"], st["cmap"], st["rmin"], st["rmax"], st["scale"],
                    st["ev"], st["ef"], st["xi"], st["p0"], st["d0"])
    eo = O.EOFTable(et["mmax"], et["norder"], et["numx"], et["numy"], et["cmap"], et["rmin"], et["rmax"],
                    et["ascale"], et["hscale"], et["potC"], et["rforceC"], et["zforceC"], et["potS"],
                    et["rforceS"], et["zforceS"], et["densC"], et["densS"])
    F = O.FieldSpec(eo, c[-1].cpu().numpy(), sn[-1].cpu().numpy(), slo, hl[-1].cpu().numpy())
    x, y, z = (v[-64:].cpu().numpy().astype(np.float64) for v in d[:3])
    for u, r in zip(f, O.total_force(F, x, y, z)):
        assert relmax(u[-64:].cpu().numpy(), r) <= 1e-5    # the field's bound, per output


@pytest.mark.parametrize("lmax,nmax,mmax,norder", [(2, 5, 2, 5), (6, 9, 6, 21), (6, 20, 8, 33)])
@pytest.mark.parametrize("nd,nh", [(1, 1), (64, 65), (1300, 3), (0, 70), (70, 0), (5000, 4097)])
def test_small_dump_in_one_stream(nd, nh, lmax, nmax, mmax, norder):
    """forces_disc_halo of few particles (both accumulates, reductions and folds
    in one launch each): the coefficients of the oracle, and the bits of the
    separate freeze and evaluation with them."""
    import torch
    from exptool_amd.bfe import BFESystem
    from exptool_amd.utils import workloads as W
    st, et = W.disc_halo_tables(seed=2, n_eof_sample=3000, lmax_s=10, nmax_s=max(8, norder),
                                eof=dict(mmax=mmax, norder=norder, numx=20, numy=12),
                                sl=dict(lmax=lmax, nmax=nmax, numr=150))
    s = BFESystem(sl=st, eof=et)
    d, h = (f32(*p) for p in W.disc_halo_particles(max(nd, 1), max(nh, 1), seed=5))
    d, h = [a[:nd] for a in d], [a[:nh] for a in h]
    slo = O.SLTable(st["lmax"], st["nmax"], st["numr"], st["cmap"], st["rmin"], st["rmax"], st["scale"],
                    st["ev"], st["ef"], st["xi"], st["p0"], st["d0"])
    eo = O.EOFTable(et["mmax"], et["norder"], et["numx"], et["numy"], et["cmap"], et["rmin"], et["rmax"],
                    et["ascale"], et["hscale"], et["potC"], et["rforceC"], et["zforceC"], et["potS"],
                    et["rforceS"], et["zforceS"], et["densC"], et["densS"])
    out = s.forces_disc_halo(d, h, rotpos=0.2)
    c, sn, g = out["cos"], out["sin"], out["coef"]
    if nd:
        rc, rs = O.eof_accumulate(eo, *d)
        assert block_rel_eof(c.cpu().numpy(), rc) <= TOL
        assert block_rel_eof(sn.cpu().numpy()[1:], rs[1:]) <= TOL
    assert not nd or torch.all(sn[0] == 0)
    if nh:
        assert block_rel_sl(g.cpu().numpy(), O.sl_accumulate(slo, *h), lmax) <= TOL
    s.set_field(c, sn, g)
    ref = s.field_forces(*(np.concatenate([a, b]) for a, b in zip(d[:3], h[:3])), rotpos=0.2)
    for k, v in zip(("fx", "fy", "fz", "pot"), ref):
        assert torch.equal(out[k], v), k


@pytest.mark.parametrize("density", [False, True])
@pytest.mark.parametrize("lmax,mmax,numr,numx,numy", [(0, 0, 4, 8, 6), (6, 6, 201, 20, 15), (9, 16, 64, 31, 17)])
def test_point_forms_by_cells_equal_whole_folds(lmax, mmax, numr, numx, numy, density):
    """The point evaluators' fold of the points' own cells against the
    whole-table folds: the same bits, in the first, last and middle cells, past
    the tables, at r = 0, at NaN, with truncations, masks and options."""
    import torch
    from exptool_amd.bfe import BFESystem
    from exptool_amd.utils import workloads as W
    st, et = W.disc_halo_tables(seed=2, n_eof_sample=3000, lmax_s=16, nmax_s=8,
                                eof=dict(mmax=mmax, norder=7, numx=numx, numy=numy),
                                sl=dict(lmax=lmax, nmax=7, numr=numr))
    s = BFESystem(sl=st, eof=et)
    d, h = W.disc_halo_particles(500, 500, seed=3)
    c, sn = s.eof_accumulate(*d)
    hl = s.sl_accumulate(*h)
    g = np.random.default_rng(5)
    r = np.concatenate([[0.0, 1e-9, 1e-3, 1e6, np.nan, 1.0], 10 ** g.uniform(-3, 2, 95)])
    z = np.concatenate([[0.0, 1e-9, -30.0, 1e6, 0.5, np.nan], g.normal(0, 0.5, 95)])
    t = np.concatenate([[1.0, -1.0, 0.0, np.nan, 0.3, 0.1], g.uniform(-1, 1, 95)])
    ph = g.uniform(-4, 4, r.size)
    runs = [lambda n: s.sl_eval_sph(r[:n], t[:n], ph[:n], hl, density=density),
            lambda n: s.sl_eval_sph(r[:n], t[:n], ph[:n], hl, lmax_use=2, nmax_use=3, no_odd=True,
                                    density=density, edge=True),
            lambda n: s.sl_eval_sph(r[:n], t[:n], ph[:n], hl, density=density, cos_l=True),
            lambda n: s.eof_eval_cyl(r[:n], z[:n], ph[:n], c, sn, density=density),
            lambda n: s.eof_eval_cyl(r[:n], z[:n], ph[:n], c, sn, mmax_use=2, nmax_use=3, no_odd=True,
                                     compat_mask=True, density=density)]
    for run in runs:
        for n in (0, 1, r.size):
            out = []
            for pb in (0, 512):
                s.set_tuning("point_blocks", pb)
                out.append(run(n))
            assert torch.equal(torch.nan_to_num(out[0], nan=7.5), torch.nan_to_num(out[1], nan=7.5))


@pytest.mark.parametrize("comp", [False, True])
@pytest.mark.parametrize("nd,nh", [(1, 1), (255, 257), (2048, 2049), (4099, 300), (3, 5000)])
def test_dump_evaluated_in_the_accumulate_orders(big, particles, nd, nh, comp):  # noqa: F811
    """Both accumulates in cell order: the evaluation takes their two orders (and
    the deposits read masses by index).  Coefficients as the separate calls'
    within the float32 sums, field bits as the separate evaluation's; with one
    side in input order the points are ordered together."""
    import torch
    s, _, _ = big
    d, h = ([torch.tensor(a[:n], dtype=torch.float32, device="cuda") for a in p]
            for p, n in zip(particles, (nd, nh)))
    for omin in (1, min(nd, nh) + 1):
        s.set_tuning("order_min", omin)
        s.set_tuning("split_eval_max", 0)
        out = s.forces_disc_halo(d, h, rotpos=0.2, components=comp)
        c, sn = s.eof_accumulate(*d)
        hl = s.sl_accumulate(*h)
        s.set_tuning("order_min", 1 << 40)
        s.set_field(out["cos"], out["sin"], out["coef"])
        ref = s.field_forces(*(torch.cat([a, b]) for a, b in zip(d[:3], h[:3])), rotpos=0.2,
                             components=comp)
        s.set_tuning("order_min", 65536)
        s.set_tuning("split_eval_max", 131072)
        assert block_rel_eof(out["cos"].cpu().numpy(), c.cpu().numpy()) <= TOL
        assert block_rel_eof(out["sin"].cpu().numpy()[1:], sn.cpu().numpy()[1:]) <= TOL
        assert block_rel_sl(out["coef"].cpu().numpy(), hl.cpu().numpy(), 6) <= TOL
        for k, v in zip(("fx", "fy", "fz", "pot", "comp"), ref):
            assert torch.equal(out[k], v), k
