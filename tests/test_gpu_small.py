"""Small accumulates and sorts at the edges of their tiles: the input-order
disc kernel in tiles of 64 and of 256, the cell-ordered kernels with segments
of one to five tiles, and sorts of 512- and 2048-item tiles."""
import numpy as np
import pytest

from tests.test_gpu_parity import big, block_rel_eof, block_rel_sl, disc_halo, f32  # noqa: F401
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
