"""Gradients of W0, b0..b3, W4 and b4: products and sums over points in float64.

Sixteen points at one place in one wave, all of weight 0 but three, of weights 1,
2^-12 and -1: the large contributions all but cancel.  A point alone (the
others of weight 0) gives its own contribution: to a bias a float32 value as it
is, so the three runs' values sum exactly in float64; to W0 the same times the
point's float32 feature; to W4, which no matrix product precedes, contributions
of weights 1 and -1 are exact opposites and the middle point's run is the whole
sum.  In float64 the kernel's sums leave 2^-53 of the large terms, 2^-41 of the
result; float32 sums or products would leave 2^-24 of the large terms, 2^-12 of
the result.  Tolerance: the result's own float32 rounding either way (2^-23)."""
import numpy as np
import pytest

from oracle import mlp_oracle as MO
from tests.test_gpu_mlp import field  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", range(6))
def test_small_gradients_sum_in_float64(field, seed):  # noqa: F811
    import torch
    from exptool_amd.surrogate.mlp import MLPField
    m = MLPField(field, seed=5)
    g = np.random.default_rng(seed)
    x, y, z = (np.full(16, v, np.float32) for v in (3.1, -1.7, 0.23))
    t = torch.tensor(np.repeat(g.normal(size=(4, 1)), 16, axis=1).astype(np.float32), device="cuda")
    p = g.permutation(16)[:3]
    w = np.zeros((4, 16), np.float32)
    for k, v in enumerate((1.0, 2.0 ** -12, -1.0)):
        w[0, p[k]] = w[1 + k, p[k]] = v
    got, *alone = (m.gradient(x, y, z, t, torch.tensor(v, device="cuda"))[0].cpu().numpy().astype(np.float64)
                   for v in w)

    def block(v, name):
        o, s = MO.OFF[name]
        return v[o:o + s]

    want = {b: sum(block(v, b) for v in alone) for b in ("b0", "b1", "b2", "b3", "b4")}
    sxy = np.float32(m.cfg[0])
    for d, v in enumerate((x, y)):
        want["W0", d] = want["b0"] * np.float64(v[0] / sxy)
    want["W4"] = block(alone[1], "W4")
    for name, b in want.items():
        a = block(got, "W0").reshape(-1, 3)[:, name[1]] if isinstance(name, tuple) else block(got, name)
        assert np.any(b != 0) and np.all(np.abs(a - b) <= 2.0 ** -23 * np.abs(b)), (name, np.max(np.abs(a - b) / np.abs(b)))
