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
