"""Kernel variants at the sizes where their tiles end, against the FP64 oracle."""
import numpy as np
import pytest

from conftest import say
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [2, 3, 15, 16, 17, 63, 64, 65, 131])
@pytest.mark.parametrize("n", [65, 700])
def test_weighted_values_bitwise(ctx, n, t):
    """Edge weights and the FP64 recheck over series whose runs of 16 (bulk) and
    64 (short lists) time points end early, at odd lengths and aligned ones."""
    from pagani_amd import synth
    x = synth.bold(31 + t, n, t, 5)
    z64, _ = O.zscore(x)
    thr = 0.9 if t < 10 else 0.3
    for prec in (0, 1):
        say(f"weighted values n={n} t={t} prec={prec}")
        info = ctx.corr_build(x, n, t, thr, weighted=True, prec=prec)
        row, col, val = ctx.corr_csr(n, info.nnz, True)
        orow, ocol, oval = O.corr_csr_r(z64, thr, True)
        np.testing.assert_array_equal(row, orow)
        np.testing.assert_array_equal(col, ocol)
        np.testing.assert_array_equal(val.view(np.uint32), oval.view(np.uint32))


# chunked copies of the series just up to 20 MiB (values in one launch) and just
# beyond (slices of four chunks with partial sums), the last chunk and slice ragged
@pytest.mark.parametrize("n,t", [(2600, 1000), (2601, 1000), (2600, 1009), (9600, 270)])
def test_weighted_values_in_slices(ctx, n, t):
    from pagani_amd import synth
    x = synth.bold(n + t, n, t, 7)
    z64, _ = O.zscore(x)
    rows = np.unique(np.concatenate([[0, n - 1], np.random.default_rng(n).integers(0, n, 150)])).astype(np.int32)
    want = O.corr_rows_r(z64, 0.4, rows, True)
    for prec in (0, 1):
        say(f"weighted values in slices n={n} t={t} prec={prec}")
        info = ctx.corr_build(x, n, t, 0.4, weighted=True, prec=prec)
        row, col, val = ctx.corr_csr(n, info.nnz, True)
        for i, (ocol, oval) in zip(rows, want):
            np.testing.assert_array_equal(col[row[i]:row[i + 1]], ocol)
            np.testing.assert_array_equal(val[row[i]:row[i + 1]].view(np.uint32), oval.view(np.uint32))
        # the other direction of every entry carries the same weight
        src = np.repeat(np.arange(n, dtype=np.int64), np.diff(row))
        back = np.argsort(col.astype(np.int64) * n + src)
        np.testing.assert_array_equal(val[back].view(np.uint32), val.view(np.uint32))


# buckets of 16 rows beyond the 12,288 entries kept in registers, the last wave
# of their entries with 1 to 63 lanes (bucket lengths vary with the rows)
@pytest.mark.parametrize("n", [801, 1537, 2999, 4500])
def test_dense_buckets(ctx, n):
    from pagani_amd import synth
    x = synth.bold(n, n, 40, 6)
    z64, _ = O.zscore(x)
    for thr in (-0.9, -0.05):
        say(f"dense buckets n={n} thr={thr}")
        info = ctx.corr_build(x, n, 40, thr)
        row, col, _ = ctx.corr_csr(n, info.nnz)
        orow, ocol, _ = O.corr_csr_r(z64, thr, False)
        np.testing.assert_array_equal(row, orow)
        np.testing.assert_array_equal(col, ocol)


def _graph(n, m, seed, hub=0):
    """Random network of about m edges plus a vertex joined to `hub` others
    that are themselves a ring, as sorted symmetric CSR with weights."""
    rng = np.random.default_rng(seed)
    a, b = rng.integers(0, n, m), rng.integers(0, n, m)
    if hub:
        h = rng.permutation(n - 1)[:hub] + 1
        a = np.concatenate([a, np.zeros(hub, np.int64), h])
        b = np.concatenate([b, h, np.roll(h, 1)])
    lo, hi = np.minimum(a, b), np.maximum(a, b)
    key = np.unique(lo[lo != hi] * np.int64(n) + hi[lo != hi])
    lo, hi = key // n, key % n
    w = rng.uniform(0.05, 1.0, key.size).astype(np.float32)
    both = np.concatenate([key, hi * n + lo])
    order = np.argsort(both)
    row = np.zeros(n + 1, np.int32)
    row[1:] = np.cumsum(np.bincount(both[order] // n, minlength=n))
    return row, (both[order] % n).astype(np.int32), np.concatenate([w, w])[order]


# 8,191 / 8,192: the splitting epilogue, the band-free one; copies of 200 series
# put 560,000 pairs at one r, more than the candidate list's first size (thr
# 1.0), and a tenth of all pairs past the segments' first size (thr 0.02)
@pytest.mark.parametrize("n,copies,thr", [(8191, 0, 0.5), (8192, 0, 0.5), (8193, 0, 1.0), (8449, 0, 0.7),
                                          (15000, 200, 1.0), (9001, 0, 0.02)])
@pytest.mark.parametrize("weighted", [False, True])
def test_r_threshold_forms(ctx, n, copies, thr, weighted):
    from pagani_amd import synth
    x = synth.bold(n, copies or n, 24, 7)
    if copies:
        assert x.shape == (24, copies)
        x = np.ascontiguousarray(x[:, np.arange(n) % copies])
    z64, _ = O.zscore(x)
    say(f"r threshold n={n} copies={copies} thr={thr} weighted={weighted}")
    orow, ocol, oval = O.corr_csr_r(z64, thr, weighted)
    for _ in range(2):
        info = ctx.corr_build(x, n, 24, thr, weighted=weighted)
        row, col, val = ctx.corr_csr(n, info.nnz, weighted)
        np.testing.assert_array_equal(row, orow)
        np.testing.assert_array_equal(col, ocol)
        if weighted:
            np.testing.assert_array_equal(val.view(np.uint32), oval.view(np.uint32))


# 65,534 / 65,535 / 65,536: the last 16-bit lists, the first 32-bit ones
@pytest.mark.parametrize("n,m,hub", [(2, 3, 0), (3, 9, 0), (63, 700, 0), (64, 1500, 20), (257, 12000, 256),
                                     (5000, 60000, 1500), (65534, 150000, 1023), (65535, 150000, 1024),
                                     (65536, 150000, 1025)])
def test_clustering_lists(ctx, n, m, hub):
    """Triangles, binary and weighted clustering over the packed upper lists:
    lists that end inside a group, hubs around the 1,024 factors held in LDS."""
    row, col, val = _graph(n, m, n + m, hub)
    say(f"clustering lists n={n} nnz={col.size} hub={hub}")
    np.testing.assert_array_equal(ctx.triangles(row, col), O.triangles(row, col))
    cp, mean = ctx.cp_binary(row, col)
    ocp, omean = O.cp_binary(row, col)
    np.testing.assert_array_equal(cp.view(np.uint32), ocp.view(np.uint32))
    assert abs(mean - omean) <= 1e-12 * max(abs(omean), 1e-300)
    for kind in (1, 2):
        for mode in (0, 1):
            say(f"weighted kind={kind} mode={mode}")
            c, mw = ctx.cp_weighted(row, col, val, kind, mode)
            oc, omw = O.cp_weighted(row, col, val, kind, mode)
            np.testing.assert_allclose(c, oc, rtol=1e-12, atol=0)
            assert abs(mw - omw) <= 1e-12 * max(abs(omw), 1e-300)


# two work-groups a CU, one, and the largest n whose bitmap and prefixes fit
# (127 factors beside them): hubs below and above the factors held in LDS
@pytest.mark.parametrize("n", [300000, 610304, 638976])
@pytest.mark.parametrize("hub", [100, 3000])
def test_weighted_clustering_of_large_networks(ctx, n, hub):
    row, col, val = _graph(n, 2 * n, n + hub, hub)
    for kind in (1, 2):
        say(f"weighted clustering n={n} hub={hub} kind={kind}")
        c, mean = ctx.cp_weighted(row, col, val, kind, 0)
        oc, omean = O.cp_weighted(row, col, val, kind, 0)
        np.testing.assert_allclose(c, oc, rtol=1e-12, atol=0)
        assert abs(mean - omean) <= 1e-12 * max(abs(omean), 1e-300)


def test_clustering_zero_and_negative_weights(ctx):
    """Zero weights close no triangle; a negative product has no real root."""
    row, col, val = _graph(300, 9000, 5)
    for kind in (1, 2):
        v = val.copy()
        # both directions of an edge keep one weight: drawn by the pair
        src = np.repeat(np.arange(300), np.diff(row))
        pick = (np.minimum(src, col) * 300 + np.maximum(src, col)) % 11
        v[pick == 0] = 0.0
        if kind == 2:
            v[pick == 1] *= -1.0
        say(f"zero and negative weights kind={kind}")
        c, _ = ctx.cp_weighted(row, col, v, kind, 0)
        oc, _ = O.cp_weighted(row, col, v, kind, 0)
        np.testing.assert_array_equal(np.isnan(c), np.isnan(oc))
        ok = ~np.isnan(oc)
        np.testing.assert_allclose(c[ok], oc[ok], rtol=1e-12, atol=0)


# sparse networks, whose vector is gathered: rows that end inside a batch of 64
# entries, a hub row of several
@pytest.mark.parametrize("n,m,hub", [(5, 7, 0), (300, 9000, 299), (16384, 60000, 700), (16385, 60000, 700),
                                     (33000, 90000, 2000)])
@pytest.mark.parametrize("weighted", [False, True])
def test_segmented_spmv(ctx, n, m, hub, weighted):
    """Eigenvector centrality and modularity (both stops) over the segmented
    SpMV: iteration counts and labels equal to the oracle's."""
    row, col, val = _graph(n, m, 3 * n + m, hub)
    v = val if weighted else None
    say(f"segmented spmv n={n} nnz={col.size} weighted={weighted}")
    vh, av, lam, it = ctx.eigenvector_centrality(row, col, v)
    ovh, oav, olam, oit = O.ec(row, col, v)
    assert it == oit
    np.testing.assert_allclose(vh, ovh, rtol=1e-9, atol=1e-12)
    np.testing.assert_allclose(av, oav, rtol=1e-9, atol=1e-12 * max(1.0, abs(olam)))
    assert abs(lam - olam) <= 1e-9 * abs(olam)


def _core_network(n, core, deg, seed):
    """A clique of `core` vertices in a sparse random network: a leading
    eigenvalue far from the rest, so that a power iteration ends soon."""
    rng = np.random.default_rng(seed)
    m = n * deg // 2
    k = rng.choice(n, core, replace=False).astype(np.int64)
    i, j = np.triu_indices(core, 1)
    a, b = np.concatenate([rng.integers(0, n, m), k[i]]), np.concatenate([rng.integers(0, n, m), k[j]])
    lo, hi = np.minimum(a, b), np.maximum(a, b)
    key = np.unique(lo[lo != hi] * np.int64(n) + hi[lo != hi])
    lo, hi = key // n, key % n
    w = rng.uniform(0.5, 1.0, key.size).astype(np.float32)
    both = np.concatenate([key, hi * n + lo])
    order = np.argsort(both, kind="stable")
    row = np.zeros(n + 1, np.int32)
    row[1:] = np.cumsum(np.bincount(both[order] // n, minlength=n))
    return row, (both[order] % n).astype(np.int32), np.concatenate([w, w])[order]


# 1,024 rows per work-group: more of them than 256 CUs hold at once, so that
# some start while the launch's first one has already found the stop
@pytest.mark.parametrize("n", [262144, 300003, 600001])
@pytest.mark.parametrize("weighted", [False, True])
def test_centrality_in_many_rounds_of_blocks(ctx, n, weighted):
    row, col, val = _core_network(n, 150, 4, n)
    v = val if weighted else None
    say(f"centrality rounds n={n} nnz={col.size} weighted={weighted}")
    ovh, oav, olam, oit = O.ec(row, col, v)
    assert oit < 100
    for _ in range(3):
        vh, av, lam, it = ctx.eigenvector_centrality(row, col, v)
        assert it == oit
        np.testing.assert_allclose(vh, ovh, rtol=1e-9, atol=1e-12)
        np.testing.assert_allclose(av, oav, rtol=1e-9, atol=1e-12 * max(1.0, abs(olam)))
        assert abs(lam - olam) <= 1e-9 * abs(olam)


# one (short and full), two and three staged 16,384-entry vector segments with
# rows that end inside a group; a hub row longer than a batch of 256 entries
STAGED = [(700, 120000, 600), (16384, 900000, 700), (16385, 1700000, 700), (33000, 2600000, 2000)]


@pytest.mark.parametrize("n,m,hub", STAGED)
@pytest.mark.parametrize("weighted", [False, True])
def test_staged_spmv(ctx, n, m, hub, weighted):
    row, col, val = _graph(n, m, 3 * n + m, hub)
    v = val if weighted else None
    say(f"staged spmv n={n} nnz={col.size} weighted={weighted}")
    # 3,000 entries per work-group and segment: the gathered form's limit
    assert col.size >= 3000 * -(-n // max(16, -(-n // 256))) * -(-n // 16384)
    vh, av, lam, it = ctx.eigenvector_centrality(row, col, v)
    ovh, oav, olam, oit = O.ec(row, col, v)
    assert it == oit
    np.testing.assert_allclose(vh, ovh, rtol=1e-9, atol=1e-12)
    np.testing.assert_allclose(av, oav, rtol=1e-9, atol=1e-12 * max(1.0, abs(olam)))
    assert abs(lam - olam) <= 1e-9 * abs(olam)
    for cap in (2, 40):  # vector stop at the cap: no division of noise by a gap
        got = ctx.modularity(row, col, v, 0, stop=0, max_iter=cap, max_depth=1)
        want = O.modularity(row, col, v, 0, stop=0, max_iter=cap, max_depth=1)
        assert abs(got[2] - want[2]) <= 1e-9 * max(1.0, abs(want[2]))
        np.testing.assert_allclose(got[3], want[3], rtol=1e-7, atol=1e-9)


@pytest.mark.parametrize("weighted", [False, True])
def test_power_iterations_on_millions_of_vertices(ctx, weighted):
    """Rows times vector segments beyond 2^31: the layout of a sparse network
    grows with its entries and rows only."""
    n = 6_000_000
    row, col, val = _core_network(n, 300, 2, 17)
    v = val if weighted else None
    say(f"power iterations n={n} nnz={col.size} weighted={weighted}")
    vh, av, lam, it = ctx.eigenvector_centrality(row, col, v)
    ovh, oav, olam, oit = O.ec(row, col, v)
    assert it == oit
    np.testing.assert_allclose(vh, ovh, rtol=1e-9, atol=1e-12)
    np.testing.assert_allclose(av, oav, rtol=1e-9, atol=1e-12 * max(1.0, abs(olam)))
    assert abs(lam - olam) <= 1e-9 * abs(olam)
    got = ctx.modularity(row, col, v, 0, stop=1, max_iter=64, max_depth=1)
    want = O.modularity(row, col, v, 0, stop=1, max_iter=64, max_depth=1)
    assert abs(got[2] - want[2]) <= 1e-9 * max(1.0, abs(want[2]))
    np.testing.assert_allclose(got[3], want[3], rtol=1e-7, atol=1e-9)
    clear = np.abs(want[3]) > 2e-9  # a vertex's side is its entry's sign
    np.testing.assert_array_equal(got[0][clear], want[0][clear])


@pytest.mark.parametrize("n,m,hub", [(300, 9000, 299), (16385, 60000, 700), (33000, 90000, 2000)])
@pytest.mark.parametrize("stop", [0, 1])
@pytest.mark.parametrize("weighted", [False, True])
def test_segmented_modularity(ctx, n, m, hub, stop, weighted):
    """One and two bisection levels over segmented groups; with the vector stop
    the pass ends at the iteration cap (1, 2 and 40), where the launch that
    stops is not the one after a test."""
    row, col, val = _graph(n, m, 5 * n + m, hub)
    v = val if weighted else None
    for cap in ((1, 2, 40) if stop == 0 else (10000,)):
        say(f"segmented modularity n={n} stop={stop} weighted={weighted} cap={cap}")
        got = ctx.modularity(row, col, v, 0, stop=stop, max_iter=cap, max_depth=2)
        want = O.modularity(row, col, v, 0, stop=stop, max_iter=cap, max_depth=2)
        np.testing.assert_array_equal(got[0], want[0])
        assert abs(got[1] - want[1]) <= 1e-9
        assert abs(got[2] - want[2]) <= 1e-9 * max(1.0, abs(want[2]))
        np.testing.assert_allclose(got[3], want[3], rtol=1e-7, atol=1e-9)
        assert got[4] == want[4]


# one to four 4,096-source chunks (a work-group's waves of one chunk mark found
# sources together up to three); work-groups whose last round of 256 vertices is
# whole (512, 4,096) or ragged, whose last wave is past the end (4,501, 9,003)
@pytest.mark.parametrize("n,m,tail", [(70, 200, 10), (512, 3000, 20), (4096, 30000, 3), (4500, 40000, 300),
                                      (4501, 20000, 30), (9003, 30000, 40), (12301, 40000, 5)])
def test_efficiency_components_and_tails(ctx, n, m, tail):
    """A random part, a chain hanging off it (sources that stay active for many
    levels), a separate triangle and isolated vertices."""
    rng = np.random.default_rng(n)
    core = n - tail - 8
    a, b = rng.integers(0, core, m), rng.integers(0, core, m)
    c = np.arange(core, core + tail)
    t = core + tail
    a = np.concatenate([a, [0], c[:-1], [t, t + 1, t + 2]])
    b = np.concatenate([b, [c[0]], c[1:], [t + 1, t + 2, t]])
    perm = rng.permutation(n)  # t + 3 .. n - 1 stay isolated
    a, b = perm[a], perm[b]
    lo, hi = np.minimum(a, b), np.maximum(a, b)
    key = np.unique(lo[lo != hi] * np.int64(n) + hi[lo != hi])
    lo, hi = key // n, key % n
    both = np.sort(np.concatenate([key, hi * n + lo]))
    row = np.zeros(n + 1, np.int32)
    row[1:] = np.cumsum(np.bincount(both // n, minlength=n))
    col = (both % n).astype(np.int32)
    say(f"efficiency components n={n} tail={tail}")
    e, lp, iso, unc = ctx.bfs_efficiency(row, col)
    oe, olp, oiso, ounc = O.bfs_efficiency(row, col)
    np.testing.assert_array_equal(e.view(np.uint32), oe.view(np.uint32))
    assert abs(lp - olp) <= 1e-12 * abs(olp) and (iso, unc) == (oiso, ounc)


# bitmap of the edges (n^2 / 16 bytes up to 64 MB or 48 per edge), the hash
# beyond; a hub row
@pytest.mark.parametrize("n,m,hub", [(31, 200, 0), (32, 300, 0), (33, 200, 20), (2000, 30000, 1500),
                                     (32000, 100000, 1500), (40000, 100000, 1500)])
@pytest.mark.parametrize("weighted", [False, True])
def test_rewire_paths(ctx, n, m, hub, weighted):
    from helpers import check_rewired
    row, col, val = _graph(n, m, 7 * n + m, hub)
    v = val if weighted else None
    say(f"rewire paths n={n} nnz={col.size} weighted={weighted}")
    oc, ov, sw = ctx.rewire(row, col, v, seed=9)
    check_rewired(row, col, v, oc, ov)
    oc2, ov2, sw2 = ctx.rewire(row, col, v, seed=9)
    assert sw == sw2 and np.array_equal(oc, oc2) and (v is None or np.array_equal(ov, ov2))
    # an entry without its mirror is refused on either path
    bad = col.copy()
    bad[row[1] - 1] = bad[row[1] - 1] + 1 if bad[row[1] - 1] + 1 < n else 1
    if not np.array_equal(bad, col):
        import pagani_amd
        with pytest.raises(pagani_amd.PgError) as ex:
            ctx.rewire(row, bad, v, seed=9)
        assert ex.value.status == 4


# 325,632: the last n whose rows the counting sort takes; beyond, rows are filled
# and sorted one by one, those above 1,024 entries by a bitmap
@pytest.mark.parametrize("n", [325632, 325633, 326000])
@pytest.mark.parametrize("hub", [0, 1024, 1025, 5000])
@pytest.mark.parametrize("weighted", [False, True])
def test_rewire_beyond_the_counting_sort(ctx, n, hub, weighted):
    from helpers import check_rewired
    row, col, val = _graph(n, 400000, n + hub, hub)
    v = val if weighted else None
    say(f"rewire rows n={n} hub={hub} nnz={col.size} weighted={weighted}")
    if hub:
        assert np.diff(row).max() >= hub
    oc, ov, sw = ctx.rewire(row, col, v, seed=5)
    check_rewired(row, col, v, oc, ov)
    assert sw > 0.9 * col.size


def _ladder(stages, width):
    """Layers of `width` vertices, every layer joined to the next: width^k
    shortest paths over k layers."""
    edges = [(0, 1 + j) for j in range(width)]
    for k in range(stages - 1):
        a, b = 1 + k * width, 1 + (k + 1) * width
        edges += [(a + i, b + j) for i in range(width) for j in range(width)]
    return 1 + stages * width, edges


# path counts below, at and above 2^32 (16^8): the last stay in 32 bits, the
# others run again in 64, with more groups of sources behind them
@pytest.mark.parametrize("stages,width", [(7, 16), (9, 16), (10, 16), (40, 2)])
def test_bc_path_counts_beyond_32_bits(ctx, stages, width, monkeypatch):
    from helpers import csr_from_edges
    n, edges = _ladder(stages, width)
    row, col, _ = csr_from_edges(n, edges)
    monkeypatch.setenv("PAGANI_BC_BATCHES", "1")
    say(f"bc ladder stages={stages} width={width} n={n}")
    bc = ctx.bc(row, col)
    obc = O.bc(row, col, np.arange(n, dtype=np.int32))
    np.testing.assert_allclose(bc, obc, rtol=1e-9, atol=1e-9)
    src = np.arange(0, n, 2, dtype=np.int32)
    np.testing.assert_array_equal(ctx.bfs(row, col, src), np.stack([O.bfs(row, col, int(s)) for s in src]))


FAILING = """
import ctypes as C, os, sys
mem = C.CDLL({mem!r}, mode=os.RTLD_GLOBAL)
sys.modules["torch"] = None  # ROCm's own runtime, so that hipMalloc is the test's
for p in ({root!r}, {pkg!r}):
    sys.path.insert(0, p)
import numpy as np
import pagani_amd
from pagani_amd import synth

def build(ctx, x, prec, sparsity):
    info = ctx.corr_build(x, x.shape[1], x.shape[0], 5.0 if sparsity else 0.2, sparsity=sparsity, weighted=True, prec=prec)
    return ctx.corr_csr(x.shape[1], info.nnz, True)

x = synth.bold(7, 1500, 101, 6)
for prec in (0, 1):
    for sparsity in (False, True):
        with pagani_amd.Context(0) as ctx:
            want = build(ctx, x, prec, sparsity)
        spared, made, nth = 0, 0, 0
        while made >= nth:
            nth += 1
            print("prec", prec, "sparsity", sparsity, "request", nth, flush=True)
            with pagani_amd.Context(0) as ctx:
                mem.malloc_fails(nth)
                try:
                    got = build(ctx, x, prec, sparsity)
                except pagani_amd.PgError as e:
                    assert e.status == 2, e
                    got = None
                made = mem.malloc_requests()
                mem.malloc_fails(0)
                if got is None:  # and the context still works
                    got = build(ctx, x, prec, sparsity)
                elif made >= nth:
                    spared += 1
                for a, b in zip(got, want):
                    assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), nth
        assert spared >= 2, spared
"""


def test_weighted_builds_without_room_for_the_lists(tmp_path):
    """Each allocation of a weighted build's first call refused in turn: the
    weights summed in the scatter are those of the lists, bit for bit."""
    import os
    import subprocess
    import sys
    here = os.path.dirname(os.path.abspath(__file__))
    root = os.path.dirname(here)
    mem = str(tmp_path / "libmallocfails.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", os.path.join(here, "hip_malloc_fails.cpp"), "-ldl", "-o", mem],
                   check=True)
    src = FAILING.format(mem=mem, root=root, pkg=os.path.join(root, "pagani-toolkit_amd"))
    say("weighted builds with one refused allocation each")
    r = subprocess.run([sys.executable, "-c", src], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:] + r.stdout[-500:]
