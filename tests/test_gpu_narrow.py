"""Row kernel with 16 slots and more (rows of B up to four vectors wide): chunk
remainders of its spans, and short rows on either side of the limit up to
which slots walk rows of their own."""
import numpy as np
import pytest

from conftest import exact_dense, exact_values
from oracle import oracle
from test_gpu_parity import run_gpu

import spmm_amd as S

pytestmark = pytest.mark.gpu

# one chunk of 128, 256 and 512 nonzeros less one, whole, and one more; quarters and segments
LENS = [0, 1, 3, 4, 5, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 0, 1023, 1024, 1025, 2100, 4500]


def _matrix(rng, lens, k, dtype):
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    colidx = np.concatenate([np.sort(rng.choice(k, n, replace=False)) for n in lens]).astype(np.int32)
    return S.CSR(len(lens), k, rowptr, colidx, S.to_storage(exact_values(rng, len(colidx)), dtype), dtype)


@pytest.mark.parametrize("dtype", [S.TCA_F32, S.TCA_F16, S.TCA_BF16])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 6, 8, 12, 16, 24, 32])
def test_exact_span_remainders(torch_cuda, dtype, n):
    rng = np.random.default_rng(n)
    a = _matrix(rng, LENS, 4600, dtype)
    b = S.to_storage(exact_dense(rng, (4600, n)), dtype)
    with S.Plan(a, n, S.TCA_PLAN_NO_MFMA | S.TCA_PLAN_NO_PANELS) as plan:
        got = run_gpu(torch_cuda, a, b, plan=plan)
    assert np.array_equal(got, oracle.csr_spmm(a.rowptr, a.colidx, a.values_f32(), S.from_storage(b, dtype)))


@pytest.mark.parametrize("rows", [40, 5000, 12000, 30000])
@pytest.mark.parametrize("n", [1, 8, 16])
def test_exact_short_rows(torch_cuda, rows, n):
    """The limit follows the number of rows (4, 8, 20 and 32 here); rows of every
    length around it, host and GPU plans alike."""
    torch = torch_cuda
    rng = np.random.default_rng(rows + n)
    lens = rng.integers(0, 40, rows).tolist()
    a = _matrix(rng, lens, 64, S.TCA_F16)
    b = S.to_storage(exact_dense(rng, (64, n)), S.TCA_F16)
    want = oracle.csr_spmm(a.rowptr, a.colidx, a.values_f32(), S.from_storage(b, S.TCA_F16))
    flags = S.TCA_PLAN_NO_MFMA
    with S.Plan(a, n, flags) as plan:
        assert np.array_equal(run_gpu(torch, a, b, plan=plan), want)
        tasks = plan.export_rows()[0]
    limit = min(32, max(4, min(rows, a.nnz // 8) // 600))
    multi = tasks[tasks[:, 3] == 1]
    assert multi[:, 2].max() == max(x for x in lens if x <= limit)
    rp, ci = torch.from_numpy(a.rowptr).to("cuda:0"), torch.from_numpy(a.colidx).to("cuda:0")
    with S.Plan.from_device(rp, ci, rows, 64, a.nnz, n, S.TCA_F16, flags) as plan:
        assert np.array_equal(plan.export_rows()[0], tasks)


def test_non_finite_b_at_narrow_widths(torch_cuda):
    """Lanes without a nonzero add nothing, whatever B holds."""
    rng = np.random.default_rng(2)
    a = _matrix(rng, LENS, 4600, S.TCA_F16)
    b = exact_dense(rng, (4600, 8))
    b[0] = np.inf
    with S.Plan(a, 8, S.TCA_PLAN_NO_MFMA | S.TCA_PLAN_NO_PANELS) as plan:
        got = run_gpu(torch_cuda, a, S.to_storage(b, S.TCA_F16), plan=plan)
    hit = np.array([a.rowptr[r] < a.rowptr[r + 1] and a.colidx[a.rowptr[r]] == 0 for r in range(a.nrow)])
    assert np.array_equal(np.isfinite(got).all(axis=1), ~hit)
