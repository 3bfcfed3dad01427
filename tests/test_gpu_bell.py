"""GPU parity of the Blocked-ELL MFMA kernel (tca_bell_spmm) against the CPU
oracle: bit-exact on exact-arithmetic inputs, within the reference verdict
and a 1e-3 relative bar elsewhere, for block sizes 32 and 64, fp16 / bf16,
ragged M, K and N, block rows without blocks and long block lists."""
import numpy as np
import pytest

from conftest import exact_dense, exact_values
from oracle import oracle
from test_gpu_parity import _dev, assert_parity

import spmm_amd as S

pytestmark = pytest.mark.gpu


def _csr(rng, m, k, p, dtype, exact=True, empty_rows=()):
    mask = rng.random((m, k)) < p
    for r in empty_rows:
        mask[r] = False
    lens = mask.sum(axis=1)
    rowptr = np.zeros(m + 1, np.int32)
    np.cumsum(lens, out=rowptr[1:])
    colidx = np.nonzero(mask)[1].astype(np.int32)
    nnz = int(rowptr[-1])
    v = exact_values(rng, nnz) if exact else (rng.standard_normal(nnz) * 0.02).astype(np.float32)
    v[v == 0] = 0.5
    return S.CSR(m, k, rowptr, colidx, S.to_storage(v, dtype), dtype)


def _run(torch, a, b, bs):
    colind, vals = S.csr_to_bell(a, bs)
    n = b.shape[1]
    dc = _dev(torch, colind)
    dv = _dev(torch, vals)
    db = _dev(torch, b)
    c = torch.full((a.nrow, n), float("nan"), dtype=torch.float32, device="cuda:0")
    print(f"bell M={a.nrow} K={a.ncol} N={n} bs={bs} ell_blocks={colind.shape[1]} nnz={a.nnz}", flush=True)
    S.bell_spmm(dc, dv, a.nrow, a.ncol, n, bs, a.dtype, db, c)
    torch.cuda.synchronize()
    return c.cpu().numpy()


@pytest.mark.parametrize("bs", [32, 64])
@pytest.mark.parametrize("dtype", [S.TCA_F16, S.TCA_BF16])
def test_bell_exact_bit_equal(torch_cuda, dtype, bs):
    rng = np.random.default_rng(5 + dtype + bs)
    for m, k, p in [(128, 256, 0.02), (100, 70, 0.1), (257, 1000, 0.005), (64, 64, 0.6), (33, 5, 0.3)]:
        a = _csr(rng, m, k, p, dtype, empty_rows=range(0, m, 7))
        for n in (8, 64, 256, 264, 512):
            b = S.to_storage(exact_dense(rng, (k, n)), dtype)
            got = _run(torch_cuda, a, b, bs)
            want = oracle.csr_spmm(a.rowptr, a.colidx, a.values_f32(), S.from_storage(b, dtype))
            assert np.array_equal(got, want), (m, k, p, n, bs, np.abs(got - want).max())


@pytest.mark.parametrize("bs", [32, 64])
def test_bell_random_values_within_tolerance(torch_cuda, bs):
    rng = np.random.default_rng(17 + bs)
    a = _csr(rng, 2048, 2048, 0.01, S.TCA_F16, exact=False)
    b = S.to_storage(rng.uniform(-1, 1, (2048, 256)).astype(np.float32), S.TCA_F16)
    got = _run(torch_cuda, a, b, bs)
    assert_parity(a, b, got, f"bell bs={bs}")


def test_bell_block_row_without_blocks_is_zero(torch_cuda):
    rng = np.random.default_rng(3)
    a = _csr(rng, 96, 128, 0.1, S.TCA_F16, empty_rows=range(32, 64))
    b = S.to_storage(exact_dense(rng, (128, 64)), S.TCA_F16)
    got = _run(torch_cuda, a, b, 32)
    assert np.all(got[32:64] == 0.0)
    assert np.array_equal(got, oracle.csr_spmm(a.rowptr, a.colidx, a.values_f32(), S.from_storage(b, S.TCA_F16)))


def _blocks(rng, lists, k, bs, dtype, pad_nan=False):
    """Blocked-ELL arrays with the given block columns per block row, and the dense A."""
    eb = max((len(x) for x in lists), default=0) + (1 if pad_nan else 0)
    colind = np.full((len(lists), eb), -1, np.int32)
    vals = np.zeros((len(lists) * bs, eb * bs), np.float32)
    dense = np.zeros((len(lists) * bs, (k + bs - 1) // bs * bs))
    if pad_nan:
        vals[:] = np.nan
    for i, cols in enumerate(lists):
        for e, c in enumerate(cols):
            colind[i, e] = c
            v = exact_values(rng, bs * bs).reshape(bs, bs) * (rng.random((bs, bs)) < 0.1)
            vals[i * bs:(i + 1) * bs, e * bs:(e + 1) * bs] = v
            if c * bs < k:
                dense[i * bs:(i + 1) * bs, c * bs:(c + 1) * bs] = v
    return colind, S.to_storage(vals, dtype), dense[:, :k]


@pytest.mark.parametrize("bs", [32, 64])
@pytest.mark.parametrize("n,brows", [(8, 3), (72, 150), (520, 60), (1000, 40)])
def test_bell_list_lengths(torch_cuda, bs, n, brows):
    """Every count of wavefronts per tile (by workgroups: up to 256, 512, more)
    over empty, odd and even lists, shorter and longer than the wavefronts, and
    lists of more than 64 blocks; NaN in the padding blocks, a block column past
    K, K that ends inside a block, M inside the last block row."""
    torch = torch_cuda
    rng = np.random.default_rng(brows + bs)
    k = 70 * bs - 5
    lens = [0, 1, 2, 3, 4, 7, 16, 17]
    lists = [np.sort(rng.choice(70, lens[i % len(lens)], replace=False)) for i in range(brows)]
    lists[1], lists[2] = np.arange(70), np.arange(65)
    lists[0] = np.array([3, 69, 70 + 5, 2 ** 30])
    colind, vals, dense = _blocks(rng, lists, k, bs, S.TCA_BF16, pad_nan=True)
    m = brows * bs - 3
    b = exact_dense(rng, (k, n))
    c = torch.full((m, n), float("nan"), dtype=torch.float32, device="cuda:0")
    print(f"bell lists bs={bs} n={n} brows={brows}", flush=True)
    db = _dev(torch, S.to_storage(np.concatenate([b, np.full((64, n), np.nan, np.float32)]), S.TCA_BF16))
    dc, dv = _dev(torch, colind), _dev(torch, vals)
    S.bell_spmm(dc, dv, m, k, n, bs, S.TCA_BF16, db, c)
    torch.cuda.synchronize()
    want = (dense[:m] @ b.astype(np.float64)).astype(np.float32)
    assert np.array_equal(c.cpu().numpy(), want)


@pytest.mark.parametrize("bs,n,brows", [(32, 1000, 130), (64, 520, 230), (32, 1000, 128)])
def test_bell_one_wavefront_per_tile(torch_cuda, bs, n, brows):
    """The same over more than 2048 workgroups (and just 2048) with long lists."""
    test_bell_list_lengths(torch_cuda, bs, n, brows)
