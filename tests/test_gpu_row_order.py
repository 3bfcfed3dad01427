"""The one-launch row order of small structures planned on the GPU: plans equal
to the host planner's at the ends of its tiles and of its range, with rows in
its shared bin (511 nonzeros and more) and with more of them than it ranks;
invalid structures are refused before the order is used."""
import numpy as np
import pytest

import spmm_amd as S

pytestmark = pytest.mark.gpu

FLAGS = S.TCA_PLAN_NO_MFMA | S.TCA_PLAN_NO_PANELS


def _csr(rng, lens, k, dtype=S.TCA_F32):
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    starts = rng.integers(0, k - np.asarray(lens) + 1)
    colidx = np.concatenate([np.arange(s, s + n) for s, n in zip(starts, lens)] + [np.zeros(0)]).astype(np.int32)
    return S.CSR(len(lens), k, rowptr, colidx, S.to_storage(np.zeros(len(colidx), np.float32), dtype),
                 dtype)


def _same(torch, a, n=32):
    with S.Plan(a, n, FLAGS) as host:
        want, order = host.export_rows(), host.export_order()
    rp = torch.from_numpy(a.rowptr).to("cuda:0")
    ci = torch.from_numpy(a.colidx if a.nnz else np.zeros(1, np.int32)).to("cuda:0")
    with S.Plan.from_device(rp, ci, a.nrow, a.ncol, a.nnz, n, a.dtype, FLAGS) as dev:
        got, got_order = dev.export_rows(), dev.export_order()
    for x, y in zip(want, got):
        assert np.array_equal(x, y)
    assert np.array_equal(order, got_order)


@pytest.mark.parametrize("m", [1, 63, 64, 65, 1023, 1024, 1025, 9000, 65535, 65536, 65537])
def test_order_equals_the_host_planners(torch_cuda, m):
    rng = np.random.default_rng(m)
    lens = rng.integers(0, 9, m)
    lens[rng.integers(0, m, min(m, 5))] = [0, 509, 510, 511, 900][:min(m, 5)]
    _same(torch_cuda, _csr(rng, lens, 1000))


def test_all_rows_alike_or_empty(torch_cuda):
    rng = np.random.default_rng(1)
    for lens in (np.zeros(300, int), np.full(300, 7), np.full(70, 600)):
        _same(torch_cuda, _csr(rng, lens, 700))


@pytest.mark.parametrize("n_long", [2047, 2048, 2049, 2500])
def test_many_long_rows(torch_cuda, n_long):
    """Up to 2048 rows of the shared bin are ranked in place, more are sorted the
    general way."""
    rng = np.random.default_rng(n_long)
    lens = np.concatenate([rng.integers(510, 530, n_long - 3), [5000, 5000, 4999], rng.integers(0, 4, 2000)])
    lens[:n_long - 3] = np.maximum(lens[:n_long - 3], 510)
    rng.shuffle(lens)
    lens[lens == 510] = 511
    _same(torch_cuda, _csr(rng, lens, 5100))


@pytest.mark.parametrize("longest,elems", [(20, 1), (26, 8)])
def test_vectors_by_the_longest_row(torch_cuda, longest, elems):
    """The longest row, which decides the vectors of short-row plans, is found on
    the GPU as on the host, in the first rows and in the last."""
    rng = np.random.default_rng(longest)
    for m, at in ((3, 2), (70, 0), (5000, 4999), (70000, 66000)):
        lens = rng.integers(4, 7, m)
        lens[at] = longest
        a = _csr(rng, lens, 1000, S.TCA_F16)
        if m > 3:
            with S.Plan(a, 47, FLAGS) as plan:
                assert plan.info()["elems_per_lane"] == elems
        _same(torch_cuda, a, 47)


@pytest.mark.parametrize("m,per_row", [(40000, 12), (40000, 13), (70000, 7), (70000, 20), (300000, 2), (600000, 1)])
def test_arrays_together_and_apart(torch_cuda, m, per_row):
    """Structure, temporaries and tables below 2 MiB in one allocation and above
    it in one each: plans and products equal to the host planner's."""
    torch = torch_cuda
    rng = np.random.default_rng(m + per_row)
    a = _csr(rng, rng.integers(max(per_row - 2, 0), per_row + 3, m), 5000)
    _same(torch, a)
    val = torch.from_numpy(rng.choice(np.float32([-1, 1]), a.nnz)).to("cuda:0")
    b = torch.from_numpy(rng.integers(-9, 9, (5000, 32)).astype(np.float32)).to("cuda:0")
    rp, ci = torch.from_numpy(a.rowptr).to("cuda:0"), torch.from_numpy(a.colidx).to("cuda:0")
    c = torch.full((2, m, 32), -1.0, device="cuda:0")
    with S.Plan(a, 32, FLAGS) as host, S.Plan.from_device(rp, ci, m, 5000, a.nnz, 32, S.TCA_F32, FLAGS) as dev:
        host.run(val, b, c[0])
        dev.run(val, b, c[1])
        torch.cuda.synchronize()
    assert torch.equal(c[0], c[1])


@pytest.mark.parametrize("where", ["rows", "columns", "range"])
def test_invalid_structures_are_refused(torch_cuda, where):
    torch = torch_cuda
    rng = np.random.default_rng(4)
    a = _csr(rng, rng.integers(1, 9, 500), 100)
    rp, ci = a.rowptr.copy(), a.colidx.copy()
    if where == "rows":
        rp[200] = rp[199] - 3
    elif where == "columns":
        ci[rp[100]] = 99 if rp[101] - rp[100] > 1 else 100
    else:
        ci[-1] = 100
    with pytest.raises(S.TcaError):
        S.Plan.from_device(torch.from_numpy(rp).to("cuda:0"), torch.from_numpy(ci).to("cuda:0"), 500, 100, a.nnz, 32,
                           S.TCA_F32, FLAGS)
