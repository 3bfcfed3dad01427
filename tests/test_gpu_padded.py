"""Ragged widths whose plan copies B to an aligned pitch first (padded_pitch):
the same bits as in place for every kind of task, tail and chunking, B at any
element, nothing read past B's end; the rule's sides; graph replays."""
import numpy as np
import pytest

from conftest import exact_dense
from oracle import oracle
from test_gpu_ragged import LENS, TORCH, _matrix, _run

import spmm_amd as S

pytestmark = pytest.mark.gpu

FLAGS = S.TCA_PLAN_NO_PANELS | S.TCA_PLAN_NO_MFMA


def _copies(a, n, flags=FLAGS):
    with S.Plan(a, n, flags) as plan:
        return "pack" in plan.phases()


@pytest.mark.parametrize("dtype,n", [(S.TCA_F32, n) for n in (17, 31, 47, 126, 127, 255, 1023)] +
                         [(S.TCA_F16, n) for n in (33, 34, 47, 63, 127, 333, 511)] + [(S.TCA_BF16, n) for n in (41, 1023)])
def test_same_bits_as_in_place(torch_cuda, monkeypatch, dtype, n):
    print(f"padded dtype={dtype} n={n}", flush=True)
    rng = np.random.default_rng(n)
    a = _matrix(rng, LENS, 4200, dtype)
    b = exact_dense(rng, (4200, n))
    b[0, :5], b[-1, -3:] = np.inf, np.nan  # reach only the rows that hold columns 0 and 4199
    for slices in ("1", "2", "3"):
        monkeypatch.setenv("TCA_SLICES", slices)
        monkeypatch.setenv("TCA_PAD", "0")
        assert not _copies(a, n)
        want, _ = _run(torch_cuda, a, b, FLAGS, shift=n % 2)
        monkeypatch.setenv("TCA_PAD", "1")
        assert _copies(a, n)
        got, _ = _run(torch_cuda, a, b, FLAGS, shift=n % 2)
        assert np.array_equal(got, want, equal_nan=True), slices
    b[~np.isfinite(b)] = 0.0
    got, _ = _run(torch_cuda, a, b, FLAGS)
    assert np.array_equal(got, oracle.csr_spmm(a.rowptr, a.colidx, a.values_f32(), b))


@pytest.mark.parametrize("m,k,per_row,n,dtype,copies", [
    (3000, 2000, 160, 333, S.TCA_F16, True),    # odd 16-bit rows, gathered 240 times
    (3000, 2000, 160, 334, S.TCA_F16, False),   # dword-aligned ones off the lines gain nothing
    (3000, 2000, 160, 333, S.TCA_F32, False),
    (3000, 2000, 160, 127, S.TCA_F32, False),   # fp32 within the L2s neither
    (60000, 60000, 40, 127, S.TCA_F32, True),   # behind them, in whole lines
    (3000, 60000, 40, 127, S.TCA_F32, False),   # a row of B gathered twice
    (3000, 2000, 160, 336, S.TCA_F16, False)])  # whole vectors
def test_rule(torch_cuda, m, k, per_row, n, dtype, copies):
    rng = np.random.default_rng(m + n)
    rowptr = (np.arange(m + 1) * per_row).astype(np.int32)
    start = rng.integers(0, k // per_row, (m, per_row))
    colidx = (start + np.arange(per_row) * (k // per_row)).astype(np.int32).ravel()
    a = S.CSR(m, k, rowptr, colidx, S.to_storage(rng.choice([-1.0, 1.0], len(colidx)), dtype), dtype)
    assert _copies(a, n) == copies
    assert not _copies(a, n, FLAGS | S.TCA_PLAN_NO_SCRATCH)
    if copies:
        b = exact_dense(rng, (k, n))
        got, _ = _run(torch_cuda, a, b, FLAGS)
        rows = rng.choice(m, 200, replace=False)
        dense = a.values_f32().reshape(m, per_row)[rows, :, None] * b[colidx.reshape(m, per_row)[rows]]
        assert np.array_equal(got[rows], dense.sum(1, dtype=np.float64).astype(np.float32))


def test_graph_replays(torch_cuda, monkeypatch):
    torch = torch_cuda
    monkeypatch.setenv("TCA_PAD", "1")
    rng = np.random.default_rng(3)
    a = _matrix(rng, LENS, 4200, S.TCA_F16)
    n = 47
    val = torch.from_numpy(a.values_f32()).to("cuda:0").half()
    b = torch.empty((4200, n), dtype=torch.float16, device="cuda:0")
    c, e = (torch.empty((a.nrow, n), device="cuda:0") for _ in range(2))
    with S.Plan(a, n, FLAGS) as plan:
        s = torch.cuda.Stream()
        b.copy_(torch.from_numpy(exact_dense(rng, (4200, n))))
        torch.cuda.synchronize()
        plan.run(val, b, c, stream=s.cuda_stream)
        s.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            plan.run(val, b, c, stream=s.cuda_stream)
        for _ in range(4):  # a new B each time
            b.copy_(torch.from_numpy(exact_dense(rng, (4200, n))))
            c.fill_(-1.0)
            g.replay()
            torch.cuda.synchronize()
            plan.run(val, b, e)
            torch.cuda.synchronize()
            assert torch.equal(c, e)


def test_copy_is_reported(torch_cuda, monkeypatch):
    """b_copy_bytes: rows at the copy's pitch (whole vectors, whole lines where
    that adds little), none for plans that read B in place or keep no scratch;
    every plan of a matrix reports its own."""
    rng = np.random.default_rng(6)
    a = _matrix(rng, LENS, 4200, S.TCA_F16)

    def copied(n, flags=FLAGS):
        with S.Plan(a, n, flags) as plan:
            assert ("pack" in plan.phases()) == (plan.info()["b_copy_bytes"] > 0)
            return plan.info()["b_copy_bytes"]

    monkeypatch.setenv("TCA_PAD", "1")
    assert copied(47) == 4200 * 48 * 2 and copied(127) == 4200 * 128 * 2 and copied(48) == 0
    assert copied(47, FLAGS | S.TCA_PLAN_NO_SCRATCH) == 0
    monkeypatch.setenv("TCA_PAD", "0")
    assert copied(47) == 0
