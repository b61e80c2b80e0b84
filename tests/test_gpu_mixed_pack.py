"""The first layer without a scatter: the gather alone, from the rows where
they lie and from rows packed into a workspace, over widths around the packed
layout's edges, with rows in several device caches, in host memory, missing
and refused, against the oracle."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _table(nc, F, rng, refused):
    """Rows in two device caches, in host memory and missing; (source, X as it
    is read, what to keep)."""
    from tcc_amd import swtcf
    from tcc_amd.hostmem import PinnedArray

    X = rng.standard_normal((nc, F)).astype(np.float32)
    kind = rng.integers(0, 4, nc)  # 0, 1: device caches; 2: host; 3: none
    cap = nc
    csm = np.full(nc, -1, np.int32)
    caches = []
    for d in range(2):
        ids = np.flatnonzero(kind == d)
        csm[ids] = d * cap + np.arange(ids.size)
        caches.append(torch.from_numpy(np.ascontiguousarray(X[ids])).cuda())
    host = PinnedArray((nc, F))
    order = rng.permutation(nc)
    host.array[order] = X  # row j lies at order[j]
    ids = np.where(kind == 3, -1, order).astype(np.int32)
    seen = X.copy()
    seen[kind == 3] = 0.0
    csm[7] = 2 * cap + 5
    if refused:  # one cache entry past the table
        j = int(np.flatnonzero((kind == 0) & (np.arange(nc) != 7))[0])
        csm[j] = 2 * cap + 1
        seen[j] = 0.0
    ptrs = torch.tensor([c.data_ptr() for c in caches], dtype=torch.int64, device="cuda")
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    src = swtcf.feature_source(torch.from_numpy(ids).cuda(), torch.from_numpy(csm).cuda(), ptrs, cap, host.device_ptr,
                               nc * F, device_error=err)
    return src, seen, err, (caches, host)


@pytest.mark.parametrize("refused", [False, True])
@pytest.mark.parametrize("F", [17, 63, 64, 100, 129, 256, 257, 300, 602])
def test_mixed_without_scatter(gpu, oracle, F, refused):
    from tcc_amd import _lib, swtcf
    from tcc_amd.gcn import _EMPTY_BCSC

    nr, nc, nnz = 203, 150, 9000
    rng = np.random.default_rng(F)
    key = np.sort(rng.choice(nr * nc, size=nnz, replace=False))
    key = key[(key // nc < 40) | (key // nc >= 70)]  # rows without an entry, and windows
    key = key[key % nc != 7]  # a column that no row uses: its entry is not looked at
    dst, col = (key // nc).astype(np.uint32), (key % nc).astype(np.uint32)
    src, seen, err, keep = _table(nc, F, rng, refused)
    A = swtcf.coo_to_bcsr(torch.from_numpy(dst.view(np.int32)).cuda(), torch.from_numpy(col.view(np.int32)).cuda(), None,
                          nr, nc)
    rowptr = np.zeros(nr + 1, np.int64)
    np.cumsum(np.bincount(dst, minlength=nr), out=rowptr[1:])
    want = oracle.csr_spmm(rowptr, col, None, seen, use_tf32=True)
    L = _lib.lib()
    args = (ctypes.byref(A.view), ctypes.byref(_EMPTY_BCSC.view), ctypes.byref(src.struct))
    # what packing takes; the query names it only for tables where packing pays
    need = L.tcc_tf32_packed_bytes(nc, F) + 16 + 4 * ((nc + 31) // 32)
    assert L.tcc_spmm_cnic_forward_mixed_workspace_bytes(*args, F) == 0
    rows = (A.view.num_rowWindows + 1) * 8
    for ws_bytes in (0, need - 1, need):
        ws = torch.full((need + 64,), 255, dtype=torch.uint8, device="cuda")
        denseC = torch.full((rows, F), float("nan"), device="cuda")
        err.zero_()
        _lib.check(L.tcc_spmm_cnic_forward_mixed_ws(*args, denseC.data_ptr(), F, ws.data_ptr() if ws_bytes else None,
                                                    ws_bytes, torch.cuda.current_stream().cuda_stream))
        got = denseC.cpu().numpy()
        # fp32 sums of at most 150 TF32 products a row
        assert np.linalg.norm(got[:nr] - want) <= 150 * 2.0**-24 * np.linalg.norm(want), ws_bytes
        assert not got[nr:].any()
        assert int(err.item()) == (7 if refused else 0)
        assert int((ws[need:] != 255).sum()) == 0
    del keep


def test_mixed_workspace_only_where_it_applies(gpu):
    """A workspace for a table of 128 MiB whose rows are gathered 16 times
    each, and none beside a scatter, for packed tables, smaller ones or rows
    gathered too seldom; a launch on another stream packs on that stream."""
    from tcc_amd import gcn, graphs, swtcf, _lib

    n, F = 70_000, 480  # 134.4 MB
    rows, cols = graphs.rmat_graph(n, 2_000_000, 3, device="cuda")
    X = torch.randn((n, F), generator=torch.Generator().manual_seed(3))
    L = _lib.lib()

    def need(table, g, F=F):
        b = g.bcsc if g.bcsc is not None else gcn._EMPTY_BCSC
        return L.tcc_spmm_cnic_forward_mixed_workspace_bytes(ctypes.byref(g.bcsr.view), ctypes.byref(b.view),
                                                             ctypes.byref(table.source.struct), F)

    hot = gcn.FeatureTable(X, cols, hot_fraction=1.0)
    g = gcn.LayerGraph(rows, cols, n, n, hot_src=hot.hot)
    assert need(hot, g) == L.tcc_tf32_packed_bytes(n, F) + 16 + 4 * ((n + 31) // 32)
    assert need(hot, g, F=479) == 0  # 134,120,000 bytes
    half = gcn.FeatureTable(X, cols, hot_fraction=0.5)
    assert need(half, gcn.LayerGraph(rows, cols, n, n, hot_src=half.hot)) == 0
    assert need(gcn.FeatureTable(X, cols, hot_fraction=1.0, packed=True), g) == 0
    assert need(hot, gcn.LayerGraph(rows[::8], cols[::8], n, n, hot_src=hot.hot)) == 0
    # every partial sum of whole numbers is exact: any order gives one result
    hot.cache.random_(-3, 4, generator=torch.Generator(device="cuda").manual_seed(4))
    out = torch.empty(((g.bcsr.view.num_rowWindows + 1) * 8, F), device="cuda")
    direct = torch.empty_like(out)
    _lib.check(L.tcc_spmm_cnic_forward_mixed(ctypes.byref(g.bcsr.view), ctypes.byref(gcn._EMPTY_BCSC.view),
                                             ctypes.byref(hot.source.struct), direct.data_ptr(), F,
                                             torch.cuda.current_stream().cuda_stream))
    assert torch.equal(g.aggregate(F, source=hot.source), direct[:n])
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    for _ in range(3):  # a freed workspace goes to that stream's next call
        swtcf.spmm_cnic_forward_mixed(g.bcsr, gcn._EMPTY_BCSC, hot.source, out, F, stream=s)
    s.synchronize()
    assert torch.equal(out, direct)


@pytest.mark.parametrize("F", [449, 450, 452])
@pytest.mark.parametrize("rows", [18_000, 20_000])
def test_mixed_stored_and_added(gpu, rows, F):
    """Both routes of the unpacked first layer without a scatter, at their line
    of 32 MiB: whole numbers, so that every order of the sums gives one result."""
    from tcc_amd import gcn, graphs, swtcf

    n = 20_000
    r, c = graphs.rmat_graph(n, 200_000, 5, device="cuda")
    keep = (r < rows) & (r // 8 % 5 != 2)  # windows without an entry
    r, c = r[keep], c[keep]
    X = torch.randint(-3, 4, (n, F), generator=torch.Generator().manual_seed(F)).float()
    table = gcn.FeatureTable(X, c, hot_fraction=1.0)
    g = gcn.LayerGraph(r, c, rows, n, hot_src=table.hot, backward_bcsc=gcn._EMPTY_BCSC)
    assert (g.bcsr.view.num_rowWindows * 32 * F >= 32 << 20) == (rows == 20_000)
    want = torch.zeros(rows, F, dtype=torch.float64, device="cuda").index_add_(0, r, X.cuda().double()[c])
    out = torch.full(((g.bcsr.view.num_rowWindows + 1) * 8, F), float("nan"), device="cuda")
    swtcf.spmm_cnic_forward_mixed(g.bcsr, gcn._EMPTY_BCSC, table.source, out, F)
    assert torch.equal(out[:rows].double(), want) and not out[rows:].any()


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("columns", [1_048_575, 1_048_577, 2_450_000, 8_388_608, 8_388_609])
def test_packed_columns_of_every_slice(gpu, columns, shift):
    """The columns in use, marked in LDS by one to eight slices of 1,048,576
    columns and past those in memory, from block arrays aligned to 16 and to 4
    bytes: whole numbers from a workspace of other bytes, against the rows where
    they lie and a float64 product."""
    from tcc_amd import _lib, gcn, swtcf

    nr, F = 700, 17
    g = torch.Generator(device="cuda").manual_seed(columns)
    # both sides of every slice's start
    edge = torch.tensor(list(range(1_048_576, columns, 1_048_576)), dtype=torch.int64, device="cuda")
    c = torch.cat([torch.randint(0, columns, (20_000,), generator=g, device="cuda"), edge, edge - 1,
                   torch.tensor([0, columns - 1], device="cuda")])
    key = torch.unique(torch.randint(0, nr, (c.numel(),), generator=g, device="cuda") * columns + c)
    r, c = key // columns, key % columns
    X = torch.randint(-3, 4, (columns, F), generator=g, device="cuda").float()
    csm = torch.arange(columns, dtype=torch.int32, device="cuda")
    none = torch.full((columns,), -1, dtype=torch.int32, device="cuda")
    ptrs = torch.tensor([X.data_ptr()], dtype=torch.int64, device="cuda")
    src = swtcf.feature_source(none, csm, ptrs, columns, 0, 0)
    A = swtcf.coo_to_bcsr(r.int(), c.int(), None, nr, columns)
    idx = torch.as_tensor(A.to_host()["sparseA2B"].view(np.int32)).cuda()
    moved = torch.empty(idx.numel() + 1, dtype=torch.int32, device="cuda")[shift:]
    moved[: idx.numel()].copy_(idx)
    v = _lib.BCSR.from_buffer_copy(A.view)
    v.sparseA2B = moved.data_ptr()
    L = _lib.lib()
    need = L.tcc_tf32_packed_bytes(columns, F) + 16 + 4 * ((columns + 31) // 32)
    ws = torch.full((need,), 255, dtype=torch.uint8, device="cuda")
    out = torch.full(((v.num_rowWindows + 1) * 8, F), float("nan"), device="cuda")
    direct = torch.full_like(out, float("nan"))
    stream = torch.cuda.current_stream().cuda_stream
    args = (ctypes.byref(v), ctypes.byref(gcn._EMPTY_BCSC.view), ctypes.byref(src.struct))
    _lib.check(L.tcc_spmm_cnic_forward_mixed_ws(*args, direct.data_ptr(), F, None, 0, stream))
    _lib.check(L.tcc_spmm_cnic_forward_mixed_ws(*args, out.data_ptr(), F, ws.data_ptr(), need, stream))
    want = torch.zeros(nr, F, dtype=torch.float64, device="cuda").index_add_(0, r, X.double()[c])
    assert torch.equal(out[:nr].double(), want) and torch.equal(direct, out)
