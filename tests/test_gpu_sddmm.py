"""The sampled product of the backward pass (tca_sddmm) at the widths, row
lengths and alignments where its split of the nonzeros, its piece columns and
its partial-sum exchange can go wrong."""
import ctypes

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


def _run(torch, dtype, lens, k, n, rng, shift=0, flags=S.TCA_PLAN_DEFAULT, info=None):
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
    with S.Plan(a, n, flags) as plan:
        if info is not None:
            info.update(plan.info())
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


@pytest.mark.parametrize("dtype,n", [(S.TCA_F32, 60), (S.TCA_F32, 61), (S.TCA_F32, 64), (S.TCA_F32, 255), (S.TCA_F32, 257),
                                     (S.TCA_F16, 121), (S.TCA_F16, 128), (S.TCA_BF16, 333), (S.TCA_BF16, 520)])
def test_wavefront_per_nonzero_and_batches(torch_cuda, dtype, n):
    """The most nonzeros that take a wavefront each (16 pieces of 16 bytes a row
    and more: 256 per piece) and one more, which go in batches."""
    pieces = -(-n // (4 if dtype == S.TCA_F32 else 8))
    for nnz in (256 * pieces, 256 * pieces + 1):
        print(f"sddmm dtype={dtype} n={n} nnz={nnz}", flush=True)
        rng = np.random.default_rng(nnz)
        lens = [0, 1, 0, 3, 64, 0, 200] * 8
        lens += [500] * ((nnz - sum(lens)) // 500)
        lens += [nnz - sum(lens), 0]
        got, want = _run(torch_cuda, dtype, lens, 700, n, rng, shift=n % 2)
        assert len(want) == nnz and np.array_equal(got, want)


def test_wavefront_per_nonzero_keeps_non_finite_rows_apart(torch_cuda):
    """Its last piece overlaps the one before: an infinity there counts once."""
    torch = torch_cuda
    rng = np.random.default_rng(8)
    rowptr, colidx = _pattern(rng, [20, 9, 33], 40)
    a = S.CSR(3, 40, rowptr, colidx, np.ones(62, np.float32), S.TCA_F32)
    g = torch.from_numpy(exact_dense(rng, (3, 1025)) + 2).to("cuda:0")
    b = torch.from_numpy(exact_dense(rng, (40, 1025))).to("cuda:0")
    b[7, 1023], b[8] = float("inf"), float("nan")
    out = torch.empty(62, device="cuda:0")
    with S.Plan(a, 1025) as plan:
        S.call("tca_sddmm", plan._p, S._addr(g), S._addr(b), S._addr(out), None)
        torch.cuda.synchronize()
    rows = torch.from_numpy(np.repeat(np.arange(3), np.diff(rowptr))).to("cuda:0")
    want = (g[rows].double() * b[torch.from_numpy(colidx).long().to("cuda:0")].double()).sum(1).float()
    assert torch.equal(torch.isfinite(out), torch.isfinite(want))
    assert torch.equal(torch.nan_to_num(out, 1.0, 2.0, 3.0), torch.nan_to_num(want, 1.0, 2.0, 3.0))


PANEL_SHAPES = [(S.TCA_F32, 32), (S.TCA_F32, 64), (S.TCA_F32, 128), (S.TCA_F16, 64), (S.TCA_F16, 128), (S.TCA_BF16, 64),
                (S.TCA_BF16, 128)]


def _graph_lens(rng):
    """Rows of a power law, some empty, one in every column."""
    lens = np.minimum(3000, (4 / rng.random(900) ** 0.8).astype(int))
    lens[rng.integers(0, 900, 60)] = 0
    lens[17] = 3000
    return lens.tolist()


@pytest.mark.parametrize("window", ["0", "1"])
@pytest.mark.parametrize("dtype,n", PANEL_SHAPES)
def test_panels_exact(torch_cuda, monkeypatch, dtype, n, window):
    """The panel form (every geometry of one column chunk, run data where they lie
    or through windows, panels split into several units)."""
    monkeypatch.setenv("TCA_PANEL_WINDOW", window)
    monkeypatch.setenv("TCA_PANEL_UNIT", "900")
    print(f"panel sddmm dtype={dtype} n={n} window={window}", flush=True)
    rng = np.random.default_rng(n)
    info = {}
    got, want = _run(torch_cuda, dtype, _graph_lens(rng), 3000, n, rng, flags=S.TCA_PLAN_FORCE_PANELS | S.TCA_PLAN_NO_MFMA,
                     info=info)
    assert info["nnz_panels"] == len(want) and info["n_panel_units"] > info["n_panels"]
    assert np.array_equal(got, want)


@pytest.mark.parametrize("dtype,n", [(S.TCA_F32, 128), (S.TCA_BF16, 128)])
def test_panels_and_other_rows(torch_cuda, monkeypatch, dtype, n):
    """Some rows in panels, the others gathered, each nonzero written once."""
    monkeypatch.setenv("TCA_PANEL_MIN_REUSE", "1.5")
    monkeypatch.setenv("TCA_PANEL_MIN_NNZ", "1")
    rng = np.random.default_rng(n + 7)
    info = {}
    got, want = _run(torch_cuda, dtype, _graph_lens(rng) + [2] * 700, 3000, n, rng, flags=S.TCA_PLAN_NO_MFMA, info=info)
    assert 0 < info["nnz_panels"] < len(want)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("dtype,n", [(S.TCA_F32, 64), (S.TCA_F32, 128), (S.TCA_F16, 128), (S.TCA_BF16, 128)])
def test_every_task_beside_panels(torch_cuda, monkeypatch, dtype, n):
    """Panels keep a band of like rows; short rows in groups, medium rows, quarters
    and segments of long rows are left to the row kernel's list."""
    monkeypatch.setenv("TCA_PANEL_MIN_REUSE", "2")
    monkeypatch.setenv("TCA_PANEL_MIN_NNZ", "1")
    rng = np.random.default_rng(n + 1)
    k = 60000
    lens = [9000, 4000, 1500, 700, 300] + rng.integers(0, 40, 187).tolist() + [0, 1, 2, 3] * 200
    band = np.arange(40)
    # the longest rows share little with the 600 rows of 35 that share 40 columns
    cols = [np.sort(rng.choice(np.arange(40, k), x, replace=False)) for x in lens]
    lens2 = [35] * 600
    cols += [np.sort(rng.choice(band, 35, replace=False)) for _ in lens2]
    lens = lens + lens2
    rowptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    colidx = np.concatenate(cols).astype(np.int32)
    a = S.CSR(len(lens), k, rowptr, colidx, S.to_storage(np.ones(len(colidx), np.float32), dtype), dtype)
    g, b = exact_dense(rng, (len(lens), n)), exact_dense(rng, (k, n))
    gd = torch_cuda.from_numpy(g).to("cuda:0")
    bd = torch_cuda.from_numpy(b).to("cuda:0").to(getattr(torch_cuda, TORCH[dtype]))
    out = torch_cuda.full((len(colidx),), -1.0, device="cuda:0")
    with S.Plan(a, n, S.TCA_PLAN_NO_MFMA) as plan:
        info = plan.info()
        S.call("tca_sddmm", plan._p, S._addr(gd), S._addr(bd), S._addr(out), None)
        torch_cuda.cuda.synchronize()
    print(f"tasks beside panels dtype={dtype} n={n}: {info['rows_panels']} of {len(lens)} rows in panels", flush=True)
    rows = np.repeat(np.arange(len(lens)), lens)
    want = (g[rows].astype(np.float64) * b[colidx]).sum(1).astype(np.float32)
    assert 0 < info["rows_panels"] < len(lens) and info["n_long_rows"] > 0 and info["n_wide_tasks"] > 0
    assert np.array_equal(out.cpu().numpy(), want)


def _graph_kernels(torch, call):
    """Kernel nodes of the graph that `call(stream)` is captured into."""
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(g, stream=s):
        call(s.cuda_stream)
    hip = ctypes.CDLL(None)  # the runtime is loaded for all
    graph, n = ctypes.c_void_p(g.raw_cuda_graph()), ctypes.c_size_t(0)
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(graph, nodes, ctypes.byref(n)) == 0
    kinds = []
    for node in nodes:
        kind = ctypes.c_int(-1)
        assert hip.hipGraphNodeGetType(ctypes.c_void_p(node), ctypes.byref(kind)) == 0
        kinds.append(kind.value)
    return kinds.count(0)  # hipGraphNodeTypeKernel


@pytest.mark.parametrize("on_device", [False, True])
@pytest.mark.parametrize("dtype", [S.TCA_F32, S.TCA_F16, S.TCA_BF16])
def test_each_nonzero_computed_once(torch_cuda, monkeypatch, dtype, on_device):
    """One kernel when every nonzero is in panels, with empty rows (the row
    kernel's list only clears) and without any (it has no list); one when
    there are no panels; two when rows lie beside them."""
    torch = torch_cuda
    monkeypatch.setenv("TCA_PANEL_MIN_REUSE", "1.5")
    monkeypatch.setenv("TCA_PANEL_MIN_NNZ", "1")
    n, k = 128, 600
    band = [120] * 400
    rng = np.random.default_rng(5)
    for lens, flags, panels, kernels in ((band, S.TCA_PLAN_FORCE_PANELS, 400, 1),
                                         (band + [0] * 9, S.TCA_PLAN_FORCE_PANELS, 400, 1),
                                         (band, S.TCA_PLAN_NO_PANELS, 0, 1),
                                         (band + [2] * 300, S.TCA_PLAN_DEFAULT, None, 2)):
        rowptr, colidx = _pattern(rng, lens, k)
        m, nnz = len(lens), len(colidx)
        flags |= S.TCA_PLAN_NO_MFMA
        if on_device:
            rp, ci = torch.from_numpy(rowptr).to("cuda:0"), torch.from_numpy(colidx).to("cuda:0")
            plan = S.Plan.from_device(rp, ci, m, k, nnz, n, dtype, flags)
        else:
            plan = S.Plan(S.CSR(m, k, rowptr, colidx, S.to_storage(np.ones(nnz, np.float32), dtype), dtype), n, flags)
        g, b = exact_dense(rng, (m, n)), exact_dense(rng, (k, n))
        gd = torch.from_numpy(g).to("cuda:0")
        bd = torch.from_numpy(b).to("cuda:0").to(getattr(torch, TORCH[dtype]))
        out = torch.full((nnz,), -1.0, device="cuda:0")
        with plan:
            info = plan.info()
            if panels is None:
                assert 0 < info["nnz_panels"] < nnz
            else:
                assert info["rows_panels"] == panels and (info["n_row_tasks"] == 0) == (panels == m)
            run = lambda s: S.call("tca_sddmm", plan._p, S._addr(gd), S._addr(bd), S._addr(out), s)
            run(None)
            torch.cuda.synchronize()
            got = out.cpu().numpy()
            count = _graph_kernels(torch, run)
        rows = np.repeat(np.arange(m), lens)
        assert np.array_equal(got, (g[rows].astype(np.float64) * b[colidx]).sum(1).astype(np.float32))
        assert count == kernels, (len(lens), flags)


@pytest.mark.parametrize("n,shift", [(256, 0), (128, 1)])
def test_panels_that_gather(torch_cuda, n, shift):
    """Plans with two column chunks, and B off 16 bytes, keep to the gathering form."""
    rng = np.random.default_rng(n)
    info = {}
    got, want = _run(torch_cuda, S.TCA_F32, _graph_lens(rng), 3000, n, rng, shift=shift,
                     flags=S.TCA_PLAN_FORCE_PANELS, info=info)
    assert info["n_panels"] > 0
    assert np.array_equal(got, want)


def test_panels_keep_non_finite_rows_apart(torch_cuda):
    """Infinite rows of G and NaN rows of B reach only their own products."""
    torch = torch_cuda
    rng = np.random.default_rng(12)
    lens = _graph_lens(rng)
    rowptr, colidx = _pattern(rng, lens, 3000)
    a = S.CSR(len(lens), 3000, rowptr, colidx, np.ones(len(colidx), np.float32), S.TCA_F32)
    g = torch.from_numpy(exact_dense(rng, (len(lens), 128))).to("cuda:0")
    b = torch.from_numpy(exact_dense(rng, (3000, 128))).to("cuda:0")
    g[17], b[8], b[2999] = float("inf"), float("nan"), float("nan")
    out = torch.empty(len(colidx), device="cuda:0")
    with S.Plan(a, 128, S.TCA_PLAN_FORCE_PANELS) as plan:
        S.call("tca_sddmm", plan._p, S._addr(g), S._addr(b), S._addr(out), None)
        torch.cuda.synchronize()
    rows = np.repeat(np.arange(len(lens)), lens)
    bad = torch.from_numpy((rows == 17) | (colidx == 8) | (colidx == 2999)).to("cuda:0")
    assert torch.equal(~torch.isfinite(out), bad)
