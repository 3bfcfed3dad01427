"""GPU parity of the 2:4 sparse-MFMA kernel (tca_spmm_24) against the CPU
oracle on the pruned matrix: bit-exact on exact-arithmetic inputs, within
the reference verdict and a 1e-3 relative bar elsewhere; fp16 / bf16, K not
a multiple of 64, ragged M and N, rows without entries."""
import numpy as np
import pytest

from conftest import exact_dense, exact_values
from oracle import oracle
from test_gpu_parity import _dev, assert_parity

import spmm_amd as S

pytestmark = pytest.mark.gpu


def _pruned(rng, m, k, p, dtype, exact=True):
    a, _ = S.gen_bernoulli(m, k, p, seed=int(rng.integers(1 << 30)), dtype=dtype)
    v = exact_values(rng, a.nnz) if exact else (rng.standard_normal(a.nnz) * 0.02).astype(np.float32)
    v[v == 0] = 0.5
    a = S.CSR(a.nrow, a.ncol, a.rowptr, a.colidx, S.to_storage(v, dtype), dtype)
    return S.prune_24(a)


def _run(torch, a, b):
    vals, meta = S.csr_to_24(a)
    n = b.shape[1]
    c = torch.full((a.nrow, n), float("nan"), dtype=torch.float32, device="cuda:0")
    print(f"2:4 M={a.nrow} K={a.ncol} N={n} nnz={a.nnz}", flush=True)
    S.spmm_24(_dev(torch, vals), _dev(torch, meta), a.nrow, a.ncol, n, a.dtype, _dev(torch, b), c)
    torch.cuda.synchronize()
    return c.cpu().numpy()


@pytest.mark.parametrize("dtype", [S.TCA_F16, S.TCA_BF16])
def test_spmm_24_exact_bit_equal(torch_cuda, dtype):
    rng = np.random.default_rng(31 + dtype)
    for m, k, p in [(64, 64, 0.5), (100, 200, 0.3), (17, 1000, 0.05), (256, 130, 0.9), (1, 64, 1.0)]:
        a = _pruned(rng, m, k, p, dtype)
        for n in (8, 64, 256, 264):
            b = S.to_storage(exact_dense(rng, (k, n)), dtype)
            got = _run(torch_cuda, a, b)
            want = oracle.csr_spmm(a.rowptr, a.colidx, a.values_f32(), S.from_storage(b, dtype))
            assert np.array_equal(got, want), (m, k, p, n, np.abs(got - want).max())


def test_spmm_24_random_values_within_tolerance(torch_cuda):
    rng = np.random.default_rng(47)
    a = _pruned(rng, 2048, 2048, 0.4, S.TCA_F16, exact=False)
    b = S.to_storage(rng.uniform(-1, 1, (2048, 512)).astype(np.float32), S.TCA_F16)
    got = _run(torch_cuda, a, b)
    assert_parity(a, b, got, "2:4 2048x2048")


@pytest.mark.parametrize("m,n", [(1, 8), (287, 16), (15, 1000), (17, 72), (300, 1000), (600, 1000), (640, 1024),
                                 (1100, 1000), (1281, 904)])
@pytest.mark.parametrize("k", [1, 63, 64, 65, 129, 448, 1000])
def test_spmm_24_every_tile(torch_cuda, m, n, k):
    """Sizes that take each tile height (16, 32, 64 and 128 rows), with partial
    row and column tiles, whole and half last step pairs, fewer pairs than
    wavefronts and index windows that end inside a row."""
    rng = np.random.default_rng(m * 7 + k)
    a = _pruned(rng, m, k, 0.2, S.TCA_BF16 if k % 2 else S.TCA_F16)
    b = S.to_storage(exact_dense(rng, (k, n)), a.dtype)
    got = _run(torch_cuda, a, b)
    want = oracle.csr_spmm(a.rowptr, a.colidx, a.values_f32(), S.from_storage(b, a.dtype))
    assert np.array_equal(got, want), np.abs(got - want).max()


@pytest.mark.parametrize("k", [64, 320, 1000])
@pytest.mark.parametrize("shift", [1, 2])
def test_spmm_24_index_words_at_any_halfword(torch_cuda, k, shift):
    """Index words that start 2 or 4 bytes into their buffer; NaN rows of B past
    K and a NaN row of A after the last one stay out of the product."""
    torch = torch_cuda
    rng = np.random.default_rng(k + shift)
    m, n = 50, 72
    a = _pruned(rng, m, k, 0.4, S.TCA_F16)
    vals, meta = S.csr_to_24(a)
    b = S.to_storage(exact_dense(rng, (k, n)), S.TCA_F16)
    buf = torch.zeros(meta.size + shift, dtype=torch.int16, device="cuda:0")
    buf[shift:] = torch.from_numpy(meta.ravel().view(np.int16)).to("cuda:0")
    nan = np.full((70, n), np.nan, np.float16)
    bd = _dev(torch, np.concatenate([b, nan]))
    vd = _dev(torch, np.concatenate([vals, np.full((1, vals.shape[1]), 0x7e00, np.uint16)]))
    c = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda:0")
    print(f"2:4 K={k} shift={shift}", flush=True)
    S.spmm_24(vd, buf[shift:], m, k, n, S.TCA_F16, bd, c)
    torch.cuda.synchronize()
    want = oracle.csr_spmm(a.rowptr, a.colidx, a.values_f32(), S.from_storage(b, S.TCA_F16))
    assert np.array_equal(c.cpu().numpy(), want)


@pytest.mark.parametrize("m,k,n", [(5901, 60, 512), (5901, 256, 504),           # one wavefront, 64 rows
                                   (5901, 257, 512), (2950, 700, 1000),         # two, 128 rows
                                   (5901, 250, 1016), (8321, 61, 520), (4200, 900, 1024),  # one, 128 rows
                                   (4096, 129, 512), (4097, 193, 512)])         # tallest tiles on 256 CUs, one more
def test_spmm_24_more_tiles_than_cus(torch_cuda, m, k, n):
    rng = np.random.default_rng(m + k)
    a = _pruned(rng, m, k, 0.4, S.TCA_BF16 if k % 2 else S.TCA_F16)
    b = S.to_storage(exact_dense(rng, (k, n)), a.dtype)
    print(f"2:4 {m} x {k} x {n}", flush=True)
    got = _run(torch_cuda, a, b)
    want = oracle.csr_spmm(a.rowptr, a.colidx, a.values_f32(), S.from_storage(b, a.dtype))
    assert np.array_equal(got, want)
