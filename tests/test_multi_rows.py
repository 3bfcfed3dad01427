"""Rows per multi task of the row kernel (several short rows per wavefront):
one pass of a wavefront's slots unless the tasks fill the chip all the same or
end long before the others."""
import numpy as np
import pytest

import spmm_amd as S

SLOTS, FILL = 8, 16384  # slots at N = 32 fp32 (8 lanes per row); kMultiTasks


def _groups(n_short, n_other=0, other_len=100, n=32, slots=SLOTS):
    lens = np.concatenate([np.full(n_other, other_len), np.full(n_short, 3), np.zeros(5, int)])
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    a = S.CSR(len(lens), 1, rowptr, np.zeros(rowptr[-1], np.int32), np.zeros(rowptr[-1], np.float32), S.TCA_F32)
    tasks, _, _, geo = S.plan_row_tasks(a, n, S.TCA_F32)
    assert 64 // geo["lanes_per_row"] == slots and geo["multi_max"] < other_len <= geo["row_len"]
    multi = tasks[(tasks[:, 3] == 1) & (tasks[:, 2] > 0)]
    assert multi[:, 1].sum() == n_short and (tasks[:, 3] == 0).sum() == n_other
    assert (multi[:-1, 1] == multi[0, 1]).all()
    return int(multi[0, 1])


@pytest.mark.parametrize("n_short,n_other,passes", [
    (300, 0, 1), (20000, 9000, 1),
    (SLOTS * FILL * 2 - SLOTS, 0, 1), (SLOTS * FILL * 2, 0, 2), (SLOTS * FILL * 4, 0, 4), (SLOTS * FILL * 6, 0, 4),
    (1000, FILL - 1, 1), (1000, FILL, 4),               # others enough for the chip
    (SLOTS * FILL // 8, FILL, 4), (SLOTS * FILL // 8 + SLOTS, FILL, 1)])  # and eight times the short rows' tasks
def test_passes(n_short, n_other, passes):
    assert _groups(n_short, n_other) == passes * SLOTS


@pytest.mark.parametrize("n,slots,enough", [(64, 4, FILL // 4), (128, 2, FILL // 16)])
def test_fewer_slots_need_fewer_tasks(n, slots, enough):
    for k, passes in ((2 * enough - 1, 1), (2 * enough, 2), (4 * enough, 4)):
        assert _groups(slots * k, n=n, slots=slots) == passes * slots
