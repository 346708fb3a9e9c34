"""Launch shapes of the conservative surrogate against each other: the same bits
per point whatever number of waves a block and of tiles a wave, ragged last waves
included."""
import pytest

from tests.test_gpu_mlp import _pts, field  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def surrogate(field):  # noqa: F811
    import numpy as np
    from exptool_amd.surrogate.mlp import MLPField
    m = MLPField(field, seed=4, conservative=True)
    m.set_base(np.array([2, 1.3, 0.6, 0.2, -0.4, 1.7, 0.3, 9.0, 4.0, -0.05]))
    m.set_scaling([0.3, 1, 1, 1], [-1.0, 0.0, 0.0, 0.0])
    m.upload()
    yield m
    m.set_mode(False)
    m.set_base(None)


@pytest.mark.parametrize("n", [1, 17, 16_385, 32_769, 65_537, 98_305 + 6, 131_072 + 17, 300_000])
def test_inference_shapes_agree(surrogate, n):
    """A call against its points in calls of at most 16 384, which take four waves
    a block and one tile a wave."""
    import torch
    x, y, z = (torch.tensor(v, device="cuda") for v in _pts(n, n))
    whole = surrogate.forward(x, y, z)
    parts = [surrogate.forward(*(v[k:k + 16_000].contiguous() for v in (x, y, z))) for k in range(0, n, 16_000)]
    assert torch.isfinite(whole).all() and torch.equal(whole, torch.cat(parts, dim=1))


@pytest.mark.parametrize("n", [1, 65, 129, 16_385, 40_007])
def test_orbit_shapes_agree(surrogate, n):
    """Orbits in one call against calls of at most 16 000 (four waves a block): state,
    drift and fallbacks the same bits, the summed energies to float64 rounding."""
    import torch
    x, y, z = (torch.tensor(v, device="cuda") for v in _pts(n, n + 5))
    g = torch.Generator("cuda").manual_seed(n)
    start = torch.cat([torch.stack([x, y, z]), 0.3 * torch.randn(3, n, generator=g, device="cuda")])
    start[:3, ::7] *= 6.0                       # some outside the domain
    whole = start.clone()
    r = surrogate.leapfrog(list(whole.unbind(0)), dt=1e-2, nsteps=20, rotfreq=0.05, energy_every=8, check_period=0)
    got, energy = [], 0.0
    for k in range(0, n, 16_000):
        st = start[:, k:k + 16_000].contiguous()
        q = surrogate.leapfrog(list(st.unbind(0)), dt=1e-2, nsteps=20, rotfreq=0.05, energy_every=8, check_period=0)
        got.append((st, q["drift"], q["fallback"]))
        energy = energy + q["energy"]
    assert torch.equal(whole, torch.cat([v[0] for v in got], dim=1))
    assert torch.equal(r["drift"], torch.cat([v[1] for v in got]))
    assert torch.equal(r["fallback"], torch.cat([v[2] for v in got]))
    assert torch.allclose(r["energy"], energy, rtol=1e-12, atol=0.0)
