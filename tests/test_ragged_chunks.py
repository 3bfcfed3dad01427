"""Rows of B that whole vectors do not divide.  Column chunks when they are read
in place: one chunk (two of a small B's wide rows) unless every row of B is
gathered many times; aligned widths keep theirs.  Vectors that divide the width
where every row is short."""
import numpy as np
import pytest

import spmm_amd as S

REUSE = 128  # kRaggedChunkReuse


def _chunks(k, nnz, n, dtype):
    rowptr = np.array([0, nnz // 2, nnz], np.int32)
    a = S.CSR(2, k, rowptr, np.zeros(nnz, np.int32), np.zeros(nnz, np.float32), S.TCA_F32)
    return S.plan_row_tasks(a, n, dtype)[3]["col_chunks"]


@pytest.mark.parametrize("k,nnz,n,dtype,chunks", [
    (100000, 1000000, 63, S.TCA_F32, 1), (100000, 1000000, 64, S.TCA_F32, 2),
    (100000, 1000000, 126, S.TCA_F16, 1), (100000, 1000000, 128, S.TCA_F16, 2),
    (100000, 1000000, 127, S.TCA_F32, 1), (100000, 1000000, 128, S.TCA_F32, 4),
    (10000, 100000, 255, S.TCA_F32, 2), (100000, 1000000, 255, S.TCA_F32, 1),  # 10 MB and 100 MB
    (100000, 1000000, 333, S.TCA_F32, 2),                                      # 84 vectors: two wavefronts' widths
    (20000, 20000 * REUSE - 1, 111, S.TCA_F32, 1), (20000, 20000 * REUSE, 111, S.TCA_F32, 2)])
def test_chunks(k, nnz, n, dtype, chunks):
    assert _chunks(k, nnz, n, dtype) == chunks


def test_a_copy_keeps_the_aligned_chunks():
    """10M nonzeros on 300,000 rows of B: copied to an aligned pitch."""
    assert _chunks(300000, 10000000, 127, S.TCA_F16) == _chunks(300000, 10000000, 128, S.TCA_F16) == 2


@pytest.mark.parametrize("m,k,per_row,longest,n,dtype,elems", [
    (1000, 2048, 48, 0, 33, S.TCA_F16, 1), (1000, 2048, 48, 0, 34, S.TCA_BF16, 2),
    (1000, 2049, 48, 0, 33, S.TCA_F16, 8), (1000, 2048, 49, 0, 33, S.TCA_F16, 8),  # columns, average
    (1000, 1000, 20, 52, 47, S.TCA_F16, 1), (1000, 1000, 20, 53, 47, S.TCA_F16, 8),  # longest row
    (1000, 1000, 20, 0, 63, S.TCA_F16, 1), (1000, 1000, 20, 0, 65, S.TCA_F16, 8),  # a wavefront's width
    (1000, 1000, 20, 0, 126, S.TCA_F16, 2), (1000, 1000, 20, 0, 130, S.TCA_F16, 8),
    (1000, 1000, 6, 0, 47, S.TCA_F32, 4),
    (1000, 1000, 20, 0, 48, S.TCA_F16, 8)])
def test_short_rows_keep_dividing_vectors(m, k, per_row, longest, n, dtype, elems):
    lens = np.full(m, per_row)
    lens[7] = max(longest, per_row)
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    a = S.CSR(m, k, rowptr, np.zeros(rowptr[-1], np.int32), np.zeros(rowptr[-1], np.float32), S.TCA_F32)
    assert S.plan_row_tasks(a, n, dtype)[3]["elems_per_lane"] == elems
