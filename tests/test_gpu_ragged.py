"""Widths that the row kernel's 16-byte vectors do not divide (RowPlan::ragged):
every tail, every kind of task, operands at any element, nothing read into the
product or written past a row's end."""
import numpy as np
import pytest

from conftest import exact_dense, exact_values
from oracle import oracle

import spmm_amd as S

pytestmark = pytest.mark.gpu

TORCH = {S.TCA_F16: "float16", S.TCA_BF16: "bfloat16", S.TCA_F32: "float32"}
# short rows (several per wavefront), medium, workgroup-shared and segmented ones;
# empty rows alone, in a run, first and last
LENS = [0, 1, 2, 5, 0, 0, 0, 9, 31, 64, 65, 200, 0, 300, 700, 1030, 0, 1500, 3000, 4100] + [3] * 70 + [0] * 130 + [1, 0]


def _matrix(rng, lens, k, dtype):
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    colidx = np.concatenate([np.sort(rng.choice(k, n, replace=False)) for n in lens]).astype(np.int32)
    return S.CSR(len(lens), k, rowptr, colidx, S.to_storage(exact_values(rng, len(colidx)), dtype), dtype)


def _run(torch, a, b, flags=S.TCA_PLAN_NO_PANELS, shift=0):
    """C (guarded on both sides) of a plan whose B starts `shift` elements into its
    buffer, with NaN before and after it."""
    dt = getattr(torch, TORCH[a.dtype])
    n = b.shape[1]
    buf = torch.full((b.size + shift + 8,), float("nan"), dtype=dt, device="cuda:0")
    buf[shift:shift + b.size] = torch.from_numpy(b.ravel()).to("cuda:0").to(dt)
    val = torch.from_numpy(a.values_f32()).to("cuda:0").to(dt)
    c = torch.full((a.nrow * n + 128,), -7.0, device="cuda:0")
    with S.Plan(a, n, flags) as plan:
        info = plan.info()
        plan.run(val, buf[shift:], c[64:64 + a.nrow * n])
        torch.cuda.synchronize()
    out = c.cpu().numpy()
    assert (out[:64] == -7).all() and (out[64 + a.nrow * n:] == -7).all()
    return out[64:64 + a.nrow * n].reshape(a.nrow, n), info


@pytest.mark.parametrize("dtype,n", [(S.TCA_F32, n) for n in (17, 18, 19, 21, 33, 47, 63, 65, 127, 255, 257, 1023)] +
                         [(S.TCA_F16, n) for n in (33, 34, 35, 37, 38, 39, 47, 63, 65, 130, 333, 511, 1023)] +
                         [(S.TCA_BF16, n) for n in (41, 127, 514)])
def test_every_tail_and_task(torch_cuda, dtype, n):
    print(f"ragged dtype={dtype} n={n}", flush=True)
    rng = np.random.default_rng(n)
    a = _matrix(rng, LENS, 4200, dtype)
    b = exact_dense(rng, (4200, n))
    got, info = _run(torch_cuda, a, b, S.TCA_PLAN_NO_PANELS | S.TCA_PLAN_NO_MFMA)
    assert info["elems_per_lane"] == (4 if dtype == S.TCA_F32 else 8) and n % info["elems_per_lane"]
    assert np.array_equal(got, oracle.csr_spmm(a.rowptr, a.colidx, a.values_f32(), b))


@pytest.mark.parametrize("dtype,n", [(S.TCA_F32, 47), (S.TCA_F16, 333), (S.TCA_F16, 46), (S.TCA_BF16, 39)])
def test_column_chunks_and_b_at_any_element(torch_cuda, monkeypatch, dtype, n):
    """Chunks that end inside a row's vectors, B no more aligned than the widest
    vector dividing N (one element for odd N)."""
    rng = np.random.default_rng(n + 1)
    a = _matrix(rng, LENS, 4200, dtype)
    b = exact_dense(rng, (4200, n))
    want = oracle.csr_spmm(a.rowptr, a.colidx, a.values_f32(), b)
    for slices in ("1", "2", "3"):
        monkeypatch.setenv("TCA_SLICES", slices)
        got, _ = _run(torch_cuda, a, b, S.TCA_PLAN_NO_PANELS | S.TCA_PLAN_NO_MFMA, shift=2 if n % 2 == 0 else 1)
        assert np.array_equal(got, want), slices


@pytest.mark.parametrize("dtype,n", [(S.TCA_F32, 47), (S.TCA_F16, 47)])
def test_non_finite_b_reaches_only_its_rows(torch_cuda, dtype, n):
    rng = np.random.default_rng(5)
    a = _matrix(rng, LENS, 4200, dtype)
    b = exact_dense(rng, (4200, n))
    b[0], b[-1] = np.inf, np.nan
    got, _ = _run(torch_cuda, a, b, S.TCA_PLAN_NO_PANELS | S.TCA_PLAN_NO_MFMA)
    touched = np.zeros(a.nrow, bool)
    for r in range(a.nrow):
        cols = a.colidx[a.rowptr[r]:a.rowptr[r + 1]]
        touched[r] = len(cols) > 0 and (cols[0] == 0 or cols[-1] == 4199)
    assert np.array_equal(~np.isfinite(got).all(axis=1), touched)
    b[0] = b[-1] = 0.0
    want = oracle.csr_spmm(a.rowptr, a.colidx, a.values_f32(), b)
    assert np.array_equal(got[~touched], want[~touched])
