"""The forms an evaluation chooses between give the same bits per point: whole
calls against the same points in slices that take another build or form."""
import pytest

from tests.test_gpu_split import _points, _same, system  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ordered", [False, True])
def test_three_and_four_wave_builds_agree(system, ordered):  # noqa: F811
    """524 288 points and more take the four-wave build, slices of them the
    three-wave one; ragged last block."""
    import torch
    p = _points(524_288 + 77, 8)
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
