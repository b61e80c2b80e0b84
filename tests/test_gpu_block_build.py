"""BCSR and BCSC construction where its routes meet: grouped and shuffled
COOs, runs of empty windows, windows around the sizes that one wave sorts
(64 to 1024 edges), long windows over one and over several 128K slices,
windows too long for one workgroup, keys of more than 32 bits, every degree,
phases, single edges; bit for bit against the oracle."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _u32(a):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.int32)).cuda()


def _rows(spec, nc, rng):
    """Edges of a list of (row, number of columns)."""
    dst, src = [], []
    for r, k in spec:
        dst.append(np.full(k, r))
        src.append(np.sort(rng.choice(nc, size=k, replace=False)))
    return np.concatenate(dst).astype(np.uint32), np.concatenate(src).astype(np.uint32)


def _random(nr, nc, nnz, rng):
    key = np.sort(rng.choice(nr * nc, size=nnz, replace=False))
    return (key // nc).astype(np.uint32), (key % nc).astype(np.uint32)


def _case(name, rng):
    """(rows, cols, dst, src), in (row, column) order."""
    if name == "one_edge":
        return 1, 1, np.array([0], np.uint32), np.array([0], np.uint32)
    if name == "last_corner":
        return 900, 700, np.array([899], np.uint32), np.array([699], np.uint32)
    if name == "empty_runs":  # long runs of empty windows, at the ends too
        nr, nc = 40_000, 3000
        return (nr, nc, *_rows([(r, 5) for r in (1700, 1701, 9000, 9001, 9007, 30_001)], nc, rng))
    if name == "sort_sizes":  # windows of 2^k - 1, 2^k and 2^k + 1 edges between short ones
        nc, spec = 9000, [(0, 3)]
        for k in range(5, 12):
            for d in (-1, 0, 1):
                a = (1 << k) // 3  # spread over three rows, columns shared
                spec += [(8 * len(spec) + r, m) for r, m in ((1, a), (4, a), (7, (1 << k) - 2 * a + d))]
        nr = max(r for r, _ in spec) + 1
        return (nr, nc, *_rows(spec, nc, rng))
    if name == "long":  # windows over several slices of 128K columns, hub sources too
        nr, nc = 64, 300_000
        spec = [(r, 4000 + 100 * r) for r in range(8)] + [(9, 1), (20, 20_000), (63, 2500)]
        return (nr, nc, *_rows(spec, nc, rng))
    if name == "slices":  # long windows that leave slices without edges, rows too
        nc, spec = 900_000, [(r, 700) for r in range(8)] + [(12, 3000)]
        dst, src = _rows(spec, 100_000, rng)
        src = src + 150_000 * (src % 6)
        o = np.lexsort((src, dst))
        return 900_000, nc, np.where(dst == 12, 899_999, dst).astype(np.uint32)[o], src[o]
    if name in ("hub_row", "hub_column"):  # 10 slices of a window with 480K edges: the whole COO is sorted
        spec = [(0, 30), (5, 400_000), (6, 80_000), (9, 1500), (30, 4)]
        dst, src = _rows(spec, 1_200_000, rng)
        if name == "hub_row":
            return 64, 1_200_000, dst, src
        o = np.lexsort((dst, src))
        return 1_200_000, 64, src[o], dst[o]
    if name == "wide":  # keys of more than 32 bits
        nc = 600_000_000
        spec = [(0, 40), (8, 200), (17, 700), (25, 1000), (33, 1500), (41, 2100)]
        key = [np.sort(rng.integers(0, nc, 2 * k)) for _, k in spec]
        key = [np.unique(x)[:k] for x, (_, k) in zip(key, spec)]
        return (48, nc, np.concatenate([np.full(x.size, r) for x, (r, _) in zip(key, spec)]).astype(np.uint32),
                np.concatenate(key).astype(np.uint32))
    if name == "dense":  # every degree up to 8, long windows both ways
        return (1100, 1000, *_random(1100, 1000, 500_000, rng))
    return (2600, 2300, *_random(2600, 2300, 30_000, rng))


def _same(got, want, values):
    for k, v in want.items():
        if k == "data":
            if values:
                assert np.array_equal(got["data"], v), k
            else:
                assert got["data"] is None
        elif isinstance(v, np.ndarray):
            assert np.array_equal(got[k], v), k
        else:
            assert got[k] == v, k


@pytest.mark.parametrize("values", [False, True])
@pytest.mark.parametrize("name", ["one_edge", "last_corner", "empty_runs", "sort_sizes", "long", "slices", "wide",
                                  "hub_row", "hub_column", "dense", "sparse"])
def test_block_build_bit_exact(gpu, oracle, name, values):
    from tcc_amd import swtcf

    rng = np.random.default_rng(len(name))
    nr, nc, dst, src = _case(name, rng)
    val = rng.standard_normal(dst.size).astype(np.float32) if values else None
    rowptr = np.zeros(nr + 1, np.int64)
    np.cumsum(np.bincount(dst, minlength=nr), out=rowptr[1:])
    o = np.lexsort((dst, src))
    want_r = oracle.bcsr_build(nr, nc, rowptr, src, val)
    want_c = None
    if name != "wide":
        colptr = np.zeros(nc + 1, np.int64)
        np.cumsum(np.bincount(src, minlength=nc), out=colptr[1:])
        want_c = oracle.bcsc_build(nr, nc, colptr, dst[o], None if val is None else val[o])
    for order in (np.arange(dst.size), rng.permutation(dst.size), o):
        args = (_u32(dst[order]), _u32(src[order]), None if val is None else torch.from_numpy(val[order]).cuda())
        _same(swtcf.coo_to_bcsr(*args, nr, nc).to_host(), want_r, values)
        if want_c is not None:
            _same(swtcf.coo_to_bcsc(*args, nr, nc).to_host(), want_c, values)


@pytest.mark.parametrize("phases", [2, 3, 7])
@pytest.mark.parametrize("name", ["sort_sizes", "long", "hub_row", "dense", "sparse"])
def test_phased_build_is_the_slices_stacked(gpu, oracle, name, phases):
    from tcc_amd import swtcf

    rng = np.random.default_rng(phases)
    nr, nc, dst, src = _case(name, rng)
    W = (nr + 7) // 8
    r2 = (src.astype(np.int64) * phases // nc) * 8 * W + dst  # row of the stacked matrix
    o = np.lexsort((src, r2))
    rowptr = np.zeros(8 * W * phases + 1, np.int64)
    np.cumsum(np.bincount(r2, minlength=8 * W * phases), out=rowptr[1:])
    want = oracle.bcsr_build(8 * W * phases, nc, rowptr, src[o], None)
    got = swtcf.coo_to_bcsr(_u32(dst), _u32(src), None, nr, nc, phases=phases).to_host()
    for k in ("rowWindowOffset", "tcOffset", "sparseA2B", "tcLocalBit"):
        assert np.array_equal(got[k], want[k]), k


@pytest.mark.parametrize("columns,hub", [(5000, 2500), (200_000, 2500), (1_200_000, 480_000)])
def test_duplicates_and_ranges(gpu, oracle, columns, hub):
    """A repeated edge is refused for a BCSR wherever its window is built; a
    BCSC takes it (up to degree 8) as another degree, its bit set once."""
    from tcc_amd import _lib, swtcf

    rng = np.random.default_rng(9)
    dst, src = _rows([(3, 40), (17, hub), (18, 30), (31, 2)], columns, rng)
    for at in (0, 41, hub + 60):  # in a short window, a long one and the last
        d = np.insert(dst, at, dst[at])
        s = np.insert(src, at, src[at])
        for p in (np.arange(d.size), rng.permutation(d.size)):
            with pytest.raises(_lib.TccError, match="duplicate"):
                swtcf.coo_to_bcsr(_u32(d[p]), _u32(s[p]), None, 32, columns)
            B = swtcf.coo_to_bcsc(_u32(d[p]), _u32(s[p]), None, 32, columns).to_host()
            assert int(sum(bin(int(b)).count("1") for b in B["tcLocalBit"])) == dst.size
            assert B["nnz"] == d.size
    bad = dst.copy()
    bad[100] = 32
    with pytest.raises(_lib.TccError, match="out of range"):
        swtcf.coo_to_bcsr(_u32(bad), _u32(src), None, 32, columns)
    with pytest.raises(_lib.TccError):
        swtcf.coo_to_bcsc(_u32(bad), _u32(src), None, 32, columns)
    with pytest.raises(_lib.TccError, match="out of range"):
        swtcf.coo_to_bcsr(_u32(dst), _u32(src), None, 32, int(src.max()), phases=2)


def test_builds_from_several_threads_and_streams(gpu, oracle):
    """Kept memory goes from one build to the next: four threads on streams of
    their own build and release different matrices at the same time, with a
    release of everything kept in between."""
    import threading

    from tcc_amd import _lib, swtcf

    cases, errors = [], []
    for k in range(4):
        rng = np.random.default_rng(100 + k)
        nr, nc = 700 + 311 * k, 900 + 17 * k
        dst, src = _random(nr, nc, 9000 + 4000 * k, rng)
        p = rng.permutation(dst.size)
        rowptr = np.zeros(nr + 1, np.int64)
        np.cumsum(np.bincount(dst, minlength=nr), out=rowptr[1:])
        colptr = np.zeros(nc + 1, np.int64)
        np.cumsum(np.bincount(src, minlength=nc), out=colptr[1:])
        o = np.lexsort((dst, src))
        cases.append((nr, nc, _u32(dst[p]), _u32(src[p]), oracle.bcsr_build(nr, nc, rowptr, src, None),
                      oracle.bcsc_build(nr, nc, colptr, dst[o], None)))
    torch.cuda.synchronize()

    def work(k):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for i in range(12):
                    nr, nc, d, s, want_r, want_c = cases[(k + i) % 4]
                    A, B = swtcf.coo_to_bcsr(d, s, None, nr, nc), swtcf.coo_to_bcsc(d, s, None, nr, nc)
                    if i == 5:
                        _lib.check(_lib.lib().tcc_swtcf_release_plans())
                    _same(A.to_host(), want_r, False)
                    _same(B.to_host(), want_c, False)
                    A.release()
                    B.release()
        except Exception as e:  # shown by the main thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


def test_one_row_joined_to_every_column(gpu):
    """A window is no longer one workgroup's work however long it is: 2M edges
    of one row or column, and 2M elsewhere, take within a few times what 4M
    spread edges take (from 20 times it on, were that window built by one
    workgroup)."""
    import time

    from tcc_amd import swtcf

    n = 2_000_000
    g = torch.Generator(device="cuda").manual_seed(1)

    def seconds(build, hub, swap):
        r = torch.randint(0, n, (2 * n,), generator=g, device="cuda")
        if hub:
            r[:n] = n // 2
        c = torch.cat([torch.arange(n, device="cuda"), torch.randint(0, n, (n,), generator=g, device="cuda")])
        key = torch.unique(r * n + c)
        r, c = (key // n).int(), (key % n).int()
        if swap:
            r, c = c, r
        best = float("inf")
        for _ in range(4):
            torch.cuda.synchronize()
            t = time.perf_counter()
            build(r, c, None, n, n)
            torch.cuda.synchronize()
            best = min(best, time.perf_counter() - t)
        return best

    for build, swap in ((swtcf.coo_to_bcsr, False), (swtcf.coo_to_bcsc, True)):
        spread, hub = seconds(build, False, swap), seconds(build, True, swap)
        print(f"spread {spread * 1e3:.2f} ms, with a hub {hub * 1e3:.2f} ms")
        assert hub < 8 * spread


@pytest.mark.parametrize("values", [False, True])
@pytest.mark.parametrize("deg", [250, 800])
def test_arrays_take_what_their_blocks_need(gpu, deg, values):
    """A kept matrix holds its blocks, not what its edges could fill: 8 rows a
    window that share their columns give an eighth of those blocks."""
    from tcc_amd import _lib, swtcf

    n = 64_000
    g = torch.Generator(device="cuda").manual_seed(2)
    start = torch.randint(0, n - 8 * deg, (n // 8,), generator=g, device="cuda").repeat_interleave(8 * deg)
    k = torch.arange(n // 8, device="cuda").repeat_interleave(8 * deg)
    r = 8 * k + torch.arange(8, device="cuda").repeat_interleave(deg).repeat(n // 8)
    c = start + torch.arange(deg, device="cuda").repeat(n)
    val = torch.arange(r.numel(), device="cuda").float() if values else None
    for build, a, b in ((swtcf.coo_to_bcsr, r, c), (swtcf.coo_to_bcsc, c, r)):
        a, b = a.int(), b.int()
        torch.cuda.synchronize()
        _lib.check(_lib.lib().tcc_release_kept_memory())
        free = torch.cuda.mem_get_info()[0]
        A = build(a, b, val, n, n)
        _lib.check(_lib.lib().tcc_release_kept_memory())
        held = free - torch.cuda.mem_get_info()[0]
        blocks = A.view.num_TCBlocks
        assert blocks <= r.numel() // 48
        # 44 bytes a block, the window offsets, and the allocation's granularity
        assert held <= 44 * blocks + 4 * (n // 8 + 1) + (4 * r.numel() if values else 0) + (8 << 20), (held, blocks)
        # whole numbers: every order of the sums gives one result
        X = torch.ones(n, 1, device="cuda")
        if build is swtcf.coo_to_bcsr and not values:
            assert torch.equal(swtcf.bcsr_spmm(A, X)[:n, 0], torch.full((n,), float(deg), device="cuda"))
        if build is swtcf.coo_to_bcsr and values:
            H = A.to_host()
            assert np.array_equal(np.sort(H["data"]), val.cpu().numpy())
        A.release()
