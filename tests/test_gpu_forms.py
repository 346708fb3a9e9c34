"""The forms a fold or an evaluation chooses between give the same bits per point: whole
calls against the same points in slices that take another build or form."""
import numpy as np
import pytest

from tests.test_gpu_split import _points, _same, system  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ordered", [False, True])
def test_three_and_four_wave_builds_agree(system, ordered):  # noqa: F811
    """589 824 points and more take the four-wave build, slices of them the
    three-wave one; ragged last block."""
    import torch
    p = _points(589_824 + 77, 8)
    system.set_tuning("split_eval_max", 0)
    system.set_tuning("order_min", 1 if ordered else 1 << 40)
    whole = system.field_forces(*p.unbind(0), rotpos=0.4)
    parts = [system.field_forces(*q.contiguous().unbind(0), rotpos=0.4) for q in p.split(200_001, dim=1)]
    system.set_tuning("split_eval_max", 131072)
    system.set_tuning("order_min", 65536)
    for k, a in enumerate(whole):
        _same(a, torch.cat([q[k] for q in parts]))


@pytest.mark.parametrize("n", [16_384, 16_385, 49_153, 65_537, 98_305, 131_072])
def test_default_form_agrees_with_input_order(system, n):  # noqa: F811
    """The default choice on either side of its lines, and the fused call of n
    particles in its own field, against one lane a point in input order."""
    import torch
    p = _points(n, n + 3)
    d, h = ([a.contiguous() for a in q.unbind(0)] for q in p.split((n + 1) // 2, dim=1))
    for q in (d, h):
        q.append(torch.full_like(q[0], 1.0 / n))
    got = [system.field_forces(*p.unbind(0), rotpos=0.4, components=True)]
    kept = system._field_keep
    out = system.forces_disc_halo(d, h, rotpos=0.4, components=True)
    got.append([out[k] for k in ("fx", "fy", "fz", "pot", "comp")])
    system.set_tuning("split_eval_max", 0)
    system.set_tuning("order_min", 1 << 40)
    ref = [system.field_forces(*p.unbind(0), rotpos=0.4, components=True)]
    system.set_field(*kept)
    ref.insert(0, system.field_forces(*p.unbind(0), rotpos=0.4, components=True))
    system.set_tuning("split_eval_max", 131072)
    system.set_tuning("order_min", 65536)
    for a, b in zip(got, ref):
        for u, v in zip(a, b):
            _same(u, v)


@pytest.mark.parametrize("nd,nh", [(9001, 2500), (9001, 9001), (9001, 9000), (2500, 9001), (5001, 0)])
def test_fused_forces_of_a_halo_in_input_order(system, nd, nh):  # noqa: F811
    """The fused call with the disc in cell order and a halo that is not (few
    particles, or the matrix-product form), one side as large as the other or not:
    the coefficients of the accumulates and the forces in input order, every time."""
    import torch
    p = _points(nd + nh, 5)
    m = torch.linspace(0.5, 1.5, nd + nh, dtype=torch.float32, device="cuda") / (nd + nh)
    d, h = ([q[k].contiguous() for q in (*p.unbind(0), m)] for k in (slice(0, nd), slice(nd, None)))
    system.set_tuning("split_eval_max", 0)
    try:
        for path in (0, 1):
            if path and system.sl["lmax"] > 7:
                continue
            system.set_tuning("sl_acc_path", path)
            for _ in range(3):
                system.set_tuning("order_min", 5000)
                out = system.forces_disc_halo(d, h, rotpos=0.4, components=True)
                acc = system.accumulate_disc_halo(d, h)
                for a, b in zip((out["cos"], out["sin"], out["coef"]), acc):
                    _same(a, b)
                system.set_tuning("order_min", 1 << 40)
                ref = system.field_forces(*p.unbind(0), rotpos=0.4, components=True)
                for k, v in zip(("fx", "fy", "fz", "pot", "comp"), ref):
                    _same(out[k], v)
    finally:
        system.set_tuning("sl_acc_path", 0)
        system.set_tuning("split_eval_max", 131072)
        system.set_tuning("order_min", 65536)


@pytest.mark.parametrize("n", [32_769, 40_003])
def test_halo_sums_of_two_and_three_blocks_a_unit(n):
    """A halo in input order of more than 512 tiles, with the device to itself and
    beside a disc: the same segments, the same bits."""
    import torch
    from exptool_amd.bfe import BFESystem
    from exptool_amd.utils import workloads as W
    st, et = W.disc_halo_tables(seed=2, n_eof_sample=4000, lmax_s=10, nmax_s=8,
                                eof=dict(mmax=2, norder=4, numx=32, numy=16), sl=dict(lmax=8, nmax=12, numr=300))
    s = BFESystem(sl=st, eof=et)
    p = _points(n, 9)
    m = torch.linspace(0.5, 1.5, n, dtype=torch.float32, device="cuda") / n
    h = [q.contiguous() for q in (*p.unbind(0), m)]
    s.set_tuning("order_min", 1 << 40)
    alone = s.sl_accumulate(*h)
    _same(alone, s.accumulate_disc_halo([q[:70] for q in h], h)[2])


@pytest.mark.parametrize("density", [False, True])
@pytest.mark.parametrize("lmax,numr", [(3, 1638), (3, 1639), (9, 601), (16, 108)])
def test_sl_fold_of_one_and_two_nodes(lmax, numr, density):
    """Whole-table SL folds on either side of the line (32 768 lanes), odd and even
    numr, against the points' own cells: the same bits in every part of the table."""
    import torch
    from exptool_amd.basis import tablegen
    from exptool_amd.bfe import BFESystem
    s = BFESystem(sl=tablegen.make_sl_tables(lmax=lmax, nmax=5, numr=numr, rmin=1e-3, rmax=50.0, cmap=1, scale=1.0))
    g = np.random.default_rng(lmax)
    r = np.concatenate([[0.0, 1e-9, 1e-3, 49.9, 1e6], 10 ** g.uniform(-3, 1.7, 400)])
    t, ph = g.uniform(-1, 1, r.size), g.uniform(-4, 4, r.size)
    c = g.normal(size=((lmax + 1) ** 2, 5))
    out = []
    for pb in (0, 512):
        s.set_tuning("point_blocks", pb)
        out.append(s.sl_eval_sph(r, t, ph, c, density=density))
    assert torch.equal(out[0], out[1])
