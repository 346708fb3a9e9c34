"""The split-block evaluation (64 points per block, eight waves sharing the
orders) against the one-lane kernels it replaces at small counts: the same
bits for the field, the leapfrog (one and per-orbit step sizes, rotating
field, energies, records) and RK4, at block edges and for orders with and
without a compile-time instance (lmax 6, mmax 6; others)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

OFF, ON = 0, 1 << 40


@pytest.fixture(scope="module", params=[(6, 6), (4, 3), (9, 8), (0, 0)], ids=lambda p: f"l{p[0]}m{p[1]}")
def system(request):
    import torch
    from exptool_amd.bfe import BFESystem
    from exptool_amd.utils import workloads as W
    lmax, mmax = request.param
    st, et = W.disc_halo_tables(seed=2, n_eof_sample=4000, lmax_s=10, nmax_s=8,
                                eof=dict(mmax=mmax, norder=6, numx=48, numy=32),
                                sl=dict(lmax=lmax, nmax=6, numr=300))
    s = BFESystem(sl=st, eof=et)
    d, h = W.disc_halo_particles(3000, 3000, seed=4)
    s.set_field(*s.eof_accumulate(*d), s.sl_accumulate(*h))
    return s


def _points(n, seed):
    import torch
    from exptool_amd.utils import workloads as W
    d, h = W.disc_halo_particles(max(n, 2), max(n, 2), seed=seed)
    p = np.stack([np.concatenate([a[:(n + 1) // 2], b[:n // 2]]) for a, b in zip(d[:3], h[:3])])
    if n > 4:
        p[:, 1] = 0.0                  # the origin, the axis, past the grid's edges
        p[:, 2] = (0.0, 0.0, 0.7)
        p[:, 3] = (60.0, 3.0, -25.0)
    return torch.tensor(p, dtype=torch.float32, device="cuda").contiguous()


def _same(a, b):
    import torch
    assert (a is None) == (b is None)
    if a is not None:
        assert a.shape == b.shape and torch.equal(torch.nan_to_num(a, nan=7.5), torch.nan_to_num(b, nan=7.5))


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000, 2049])
def test_split_field_equals_one_lane(system, n):
    p = _points(n, n)
    out = []
    for m in (OFF, ON):
        system.set_tuning("split_eval_max", m)
        out.append(system.field_forces(*p.unbind(0), rotpos=0.4, components=True))
    system.set_tuning("split_eval_max", 131072)
    for a, b in zip(*out):
        _same(a, b)


@pytest.mark.parametrize("n", [1, 64, 65, 2500])
def test_split_orbits_equal_one_lane(system, n):
    import torch
    p = _points(n, n + 1)
    v = 0.3 * torch.randn(3, n, generator=torch.Generator("cuda").manual_seed(n), device="cuda")
    start = torch.cat([p, v])
    dtv = 1e-3 * (1.0 + torch.rand(n, generator=torch.Generator("cuda").manual_seed(3), device="cuda",
                                   dtype=torch.float64))
    runs = (lambda s: system.leapfrog(s, dt=1e-3, nsteps=23, record_every=4),
            lambda s: system.leapfrog(s, dt=1e-3, nsteps=23, energy_every=5, rotfreq=0.05),
            lambda s: system.leapfrog(s, dt=dtv, nsteps=12, rotfreq=0.1, energy_every=4, record_every=3),
            lambda s: dict(traj=system.rk4(s, dt=4e-3, nsteps=7, omegab=0.3, record_every=2)))
    for run in runs:
        res = []
        for m in (OFF, ON):
            system.set_tuning("split_max", m)
            st = start.clone()
            res.append((st, run(list(st.unbind(0)))))
        system.set_tuning("split_max", 36864)
        _same(res[0][0], res[1][0])
        for k in res[0][1]:
            _same(res[0][1][k], res[1][1][k])
