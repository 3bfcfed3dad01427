"""The sampled product of the backward pass (tca_sddmm) at the widths, row
lengths and alignments where its split of the nonzeros, its piece columns and
its partial-sum exchange can go wrong."""
import numpy as np
import pytest

from conftest import exact_dense

import spmm_amd as S

pytestmark = pytest.mark.gpu

TORCH = {S.TCA_F16: "float16", S.TCA_BF16: "bfloat16", S.TCA_F32: "float32"}


def _pattern(rng, lens, k):
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    colidx = np.concatenate([np.sort(rng.choice(k, n, replace=False)) for n in lens] + [np.zeros(0, np.int64)])
    return rowptr, colidx.astype(np.int32)


def _run(torch, dtype, lens, k, n, rng, shift=0):
    """out[j] and its exact value; B, G and out start `shift` elements into their buffers."""
    rowptr, colidx = _pattern(rng, lens, k)
    m, nnz = len(lens), len(colidx)
    a = S.CSR(m, k, rowptr, colidx, S.to_storage(np.ones(nnz, np.float32), dtype), dtype)
    g, b = exact_dense(rng, (m, n)), exact_dense(rng, (k, n))
    dt = getattr(torch, TORCH[dtype])

    def dev(x, t):
        buf = torch.zeros(x.size + shift, dtype=t, device="cuda:0")
        buf[shift:] = torch.from_numpy(x.ravel()).to("cuda:0").to(t)
        return buf[shift:]

    out = torch.full((nnz + shift + 1,), -1.0, device="cuda:0")
    gd, bd = dev(g, torch.float32), dev(b, dt)
    with S.Plan(a, n) as plan:
        S.call("tca_sddmm", plan._p, S._addr(gd), S._addr(bd), S._addr(out[shift:]), None)
        torch.cuda.synchronize()
    got = out.cpu().numpy()
    rows = np.repeat(np.arange(m), lens)
    want = (g[rows].astype(np.float64) * b[colidx]).sum(1).astype(np.float32)
    assert (got[:shift] == -1).all() and got[nnz + shift] == -1  # nothing written beside out
    return got[shift:nnz + shift], want


@pytest.mark.parametrize("dtype", [S.TCA_F32, S.TCA_F16, S.TCA_BF16])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 8, 9, 12, 16, 20, 31, 32, 33, 47, 64, 65, 128, 333, 520])
def test_exact_widths(torch_cuda, dtype, n):
    """Every count of pieces and tail of the last piece; rows that start inside
    a slot, fill several batches, are empty (first, last and in runs)."""
    print(f"sddmm dtype={dtype} n={n}", flush=True)
    rng = np.random.default_rng(100 + n)
    lens = [0, 0, 3, 1, 64, 8, 8, 200, 0, 0, 0, 1, 7, 9, 130, 0]
    got, want = _run(torch_cuda, dtype, lens, 220, n, rng)
    assert np.array_equal(got, want), n


@pytest.mark.parametrize("nnz", [1, 2, 63, 64, 65, 255, 256, 257])
def test_exact_ends(torch_cuda, nnz):
    """One row whose nonzeros end in, at and after a batch and a workgroup."""
    got, want = _run(torch_cuda, S.TCA_F32, [nnz], 300, 24, np.random.default_rng(nnz))
    assert np.array_equal(got, want)


@pytest.mark.parametrize("dtype,n", [(S.TCA_F32, 47), (S.TCA_F16, 47), (S.TCA_BF16, 64), (S.TCA_F32, 2)])
def test_operands_at_any_element(torch_cuda, dtype, n):
    """G, B and out need no more than their element's alignment."""
    got, want = _run(torch_cuda, dtype, [5, 0, 70, 1, 1, 40], 90, n, np.random.default_rng(n), shift=1)
    assert np.array_equal(got, want)


def test_many_rows_and_a_hub(torch_cuda):
    """More than 64^2 rows (three search steps), most of them empty, beside a
    row of 30,000; spans of several batches per wavefront."""
    rng = np.random.default_rng(9)
    lens = rng.integers(0, 3, 70000) * 20
    lens[[0, 40000]] = 0, 30000
    got, want = _run(torch_cuda, S.TCA_F32, lens.tolist(), 40000, 8, rng)
    assert len(want) > 2 * 64 * 16384 * 0.6
    assert np.array_equal(got, want)


def test_non_finite_rows_stay_in_their_products(torch_cuda):
    """An infinite or NaN row of B reaches only the nonzeros of its column, at a
    width whose last piece overlaps the one before it."""
    torch = torch_cuda
    rng = np.random.default_rng(3)
    rowptr, colidx = _pattern(rng, [20, 9, 33], 40)
    a = S.CSR(3, 40, rowptr, colidx, np.ones(62, np.float32), S.TCA_F32)
    g = torch.from_numpy(exact_dense(rng, (3, 45))).to("cuda:0")
    b = torch.from_numpy(exact_dense(rng, (40, 45))).to("cuda:0")
    b[7, 41], b[8] = float("inf"), float("nan")
    out = torch.empty(62, device="cuda:0")
    with S.Plan(a, 45) as plan:
        S.call("tca_sddmm", plan._p, S._addr(g), S._addr(b), S._addr(out), None)
        torch.cuda.synchronize()
    rows = torch.from_numpy(np.repeat(np.arange(3), np.diff(rowptr))).to("cuda:0")
    want = (g[rows].double() * b[torch.from_numpy(colidx).long().to("cuda:0")].double()).sum(1).float()
    assert torch.equal(torch.isfinite(out), torch.isfinite(want))
    assert torch.equal(torch.nan_to_num(out, 1.0, 2.0, 3.0), torch.nan_to_num(want, 1.0, 2.0, 3.0))
