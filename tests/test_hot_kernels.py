"""Sizes at which the counting kernels change tile, table or schedule, against
the oracle: on the CPU through the stand-in runtime of tests/emu (under
AddressSanitizer) and on the GPU.  Counts are whole numbers and must be equal."""
import math
import os
import subprocess

import numpy as np
import pytest

import oracle
import subgraphmatchgpu_amd as sme
from conftest import ROOT, clique

EMU_DIR = os.path.join(ROOT, "tests", "emu")


@pytest.fixture(scope="module")
def emu(tmp_path_factory):
    """Counts through the CPU build: (graph, query) -> (count, levels)."""
    subprocess.run(["make", "-C", EMU_DIR, "-s", "all"], check=True)
    path = str(tmp_path_factory.mktemp("hot") / "g.bin")

    def go(g, q, vb=0, ve=None, cl=3, bounds=None, budget=1 << 30, hub=None, **env):
        sme.write_bin(path, g)
        e = dict(os.environ, ASAN_OPTIONS="detect_leaks=0", **{k: str(v) for k, v in env.items()})
        if bounds is not None:
            e["BUCKETS"] = ",".join(map(str, bounds))
        cmd = [os.path.join(EMU_DIR, "emu_driver"), path, "6", str(q), str(cl), "1", str(vb),
               str(g.n if ve is None else ve), str(budget)] + ([str(hub)] if hub else [])
        r = subprocess.run(cmd, capture_output=True, text=True, env=e, timeout=600)
        assert r.returncode == 0, r.stderr[-3000:]
        parts = r.stdout.split()
        out = int(parts[0].split("=")[1]), [int(x) for x in parts[1].split("=")[1].split(",")]
        if bounds is not None:
            return out + ([int(x) for x in r.stdout.split("buckets=")[1].split(",")],)
        return out

    return go


@pytest.fixture(scope="module")
def dev():
    d = sme.Device(0, budget_bytes=2 << 30)
    yield d
    d.close()


def on_gpu(dev, g, q, vb=0, ve=None, cl=3):
    print(f"case q={q} cl={cl} n={g.n} nnz={g.nnz} [{vb},{ve})", flush=True)
    dg = dev.upload(g)
    r = dev.count(dg, sme.Plan(q, compress_level=cl), vb, ve)
    dg.release()
    return r.count, r.levels


def union(*graphs):
    """Disjoint union, ids in order."""
    rp, cols, n = [np.zeros(1, dtype=np.uint64)], [], 0
    for g in graphs:
        rp.append(g.row_ptrs[1:] + rp[-1][-1])
        cols.append(g.cols + np.uint32(n))
        n += g.n
    return sme.Graph(np.concatenate(rp), np.concatenate(cols).astype(np.uint32))


# upper neighbourhoods of 0 .. 66 (63 and 64 fill a wave, 65 leaves it), alone and beside one another
def small_graphs(n):
    """Cliques whose upper neighbourhoods straddle 64, then sparse vertices up to n of them."""
    dense = union(clique(66), clique(3), sme.gen_er(90, 1500, seed=3))
    return union(dense, sme.gen_er(n - dense.n, 2 * n, seed=n)) if n > dense.n else dense


@pytest.mark.parametrize("q", [0, 3, 7, 11])
def test_emu_small_neighbourhoods(emu, q):
    """One start vertex per wave step (few start vertices)."""
    g = small_graphs(0)
    want = oracle.light_count(g.row_ptrs, g.cols, q, 3)
    assert emu(g, q) == (want[0], want[1])
    bounds = [0, 1, 2, 65, 70, g.n]
    want = [oracle.light_count(g.row_ptrs, g.cols, q, 3, v_begin=a, v_end=b)[0] for a, b in zip(bounds, bounds[1:])]
    assert emu(g, q, bounds=bounds)[2] == want


def test_emu_small_neighbourhood_groups(emu):
    """Four start vertices per wave step, the last step part full."""
    g = small_graphs(16387)
    want = oracle.light_count(g.row_ptrs, g.cols, 3, 3)
    assert emu(g, 3) == (want[0], want[1])


@pytest.mark.gpu
@pytest.mark.parametrize("n", [0, 16384, 16385, 16390])
@pytest.mark.parametrize("q", [0, 3, 7])
def test_small_neighbourhoods(dev, n, q):
    g = small_graphs(n)
    want = oracle.light_count(g.row_ptrs, g.cols, q, 3)
    assert on_gpu(dev, g, q) == (want[0], want[1])
    vb, ve = 7, g.n - 3
    want = oracle.light_count(g.row_ptrs, g.cols, q, 3, v_begin=vb, v_end=ve)
    assert on_gpu(dev, g, q, vb, ve) == (want[0], want[1])


def fan(n, d, stride, extra, seed):
    """Vertex 0 joined to every stride-th vertex up to d of them, plus random edges among those: one
    upper neighbourhood of d vertices spanning about d * stride ids."""
    rng = np.random.default_rng(seed)
    ends = np.arange(1, 1 + d) * stride
    adj = [[] for _ in range(n)]
    pairs = {(0, int(e)) for e in ends}
    for a, b in rng.integers(0, d, size=(extra, 2)):
        if a != b:
            pairs.add((int(ends[min(a, b)]), int(ends[max(a, b)])))
    for a, b in pairs:
        adj[a].append(b)
        adj[b].append(a)
    return sme.from_adjacency(adj)


# (d, stride): the row table takes d <= 4,096 and a span below 65,536 ids, the hash (tables for d <= 512
# and d <= 4,096) wider spans, the search longer lists; 256 rows per part
ROW_SHAPES = [(65, 1), (255, 1), (256, 2), (257, 1), (1024, 1), (1025, 1), (90, 728), (90, 729), (90, 737),
              (513, 150), (4096, 1), (4100, 1)]


@pytest.mark.parametrize("d,stride", [(257, 1), (90, 728), (90, 737), (1025, 1)])
def test_emu_row_shapes(emu, d, stride):
    g = fan(d * stride + 2, d, stride, 3 * d, d)
    for q in (0, 3):
        want = oracle.light_count(g.row_ptrs, g.cols, q, 3)
        assert emu(g, q) == (want[0], want[1])
    bounds = [0, 1, g.n // 2, g.n]
    want = [oracle.light_count(g.row_ptrs, g.cols, 0, 3, v_begin=a, v_end=b)[0] for a, b in zip(bounds, bounds[1:])]
    assert emu(g, 0, bounds=bounds)[2] == want


@pytest.mark.gpu
@pytest.mark.parametrize("d,stride", ROW_SHAPES)
def test_row_shapes(dev, d, stride):
    g = fan(d * stride + 2, d, stride, 12 * d, d + stride)
    for q in (0, 2, 3, 7):
        want = oracle.light_count(g.row_ptrs, g.cols, q, 3)
        assert on_gpu(dev, g, q) == (want[0], want[1])
    bounds = [0, 1, g.n // 2, g.n]
    dg = dev.upload(g)
    for q in (0, 3):
        want = [oracle.light_count(g.row_ptrs, g.cols, q, 3, v_begin=a, v_end=b)[0] for a, b in zip(bounds, bounds[1:])]
        assert dev.count_buckets(dg, sme.Plan(q), bounds)[0].tolist() == want
    dg.release()


def hub_and_sparse(n, d, m, seed):
    """A vertex of degree d spread over [0, n) on top of G(n, m)."""
    g = sme.gen_er(n, m, seed=seed)
    src = np.repeat(np.arange(n), np.diff(g.row_ptrs.astype(np.int64)))
    hub = n // 3
    ends = np.unique(np.linspace(0, n - 1, d).astype(np.int64))
    ends = ends[ends != hub]
    a = np.concatenate([src, np.full(ends.size, hub), ends])
    b = np.concatenate([g.cols.astype(np.int64), ends, np.full(ends.size, hub)])
    key = np.unique(a * n + b)
    rp = np.searchsorted(key, np.arange(n + 1) * n).astype(np.uint64)
    return sme.Graph(rp, (key % n).astype(np.uint32))


def one_way(g):
    """The same lists without the mirror of every third entry."""
    src = np.repeat(np.arange(g.n), np.diff(g.row_ptrs.astype(np.int64)))
    keep = np.arange(g.nnz) % 3 != 0
    rp = np.concatenate([[0], np.cumsum(np.bincount(src[keep], minlength=g.n))]).astype(np.uint64)
    return sme.Graph(rp, g.cols[keep])


# byte counters over a span (one pass, two passes), hash beyond two spans, 16,384-id and 65,536-id
# tiles (one and two), start vertices with over 64 middles or 4,096 list entries, and a graph whose
# entries have no mirrors (level engine)
def wedge_graphs(small):
    out = {"rmat7": sme.gen_rmat(7, 6, seed=3), "span": sme.gen_er(4500, 9000, seed=2),
           "one_way": one_way(sme.gen_rmat(7, 6, seed=4)), "k12": clique(12)}
    if small:
        return out
    return dict(out, k66=clique(66), rmat12=sme.gen_rmat(12, 16, seed=5), hash=sme.gen_er(16384, 60000, seed=6),
                tile=hub_and_sparse(16385, 5000, 60000, 7), tiles=hub_and_sparse(65537, 12000, 100000, 8),
                two_tiles=hub_and_sparse(70001, 3000, 300000, 9))


@pytest.mark.parametrize("name", list(wedge_graphs(True)))
@pytest.mark.parametrize("q", [1, 4])
def test_emu_wedges(emu, name, q):
    g = wedge_graphs(True)[name]
    for cl in (0, 3):
        want = oracle.light_count(g.row_ptrs, g.cols, q, cl)
        assert emu(g, q, cl=cl) == (want[0], want[1])
    vb, ve = g.n // 5, g.n // 2
    want = oracle.light_count(g.row_ptrs, g.cols, q, 3, v_begin=vb, v_end=ve)
    assert emu(g, q, vb, ve) == (want[0], want[1])
    bounds = [1, 2, g.n // 3, g.n // 3, g.n]
    want = [oracle.light_count(g.row_ptrs, g.cols, q, 3, v_begin=a, v_end=b)[0] for a, b in zip(bounds, bounds[1:])]
    assert emu(g, q, bounds=bounds)[2] == want


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(wedge_graphs(False)))
@pytest.mark.parametrize("q", [1, 4])
def test_wedges(dev, name, q):
    g = wedge_graphs(False)[name]
    for cl in range(4):
        want = oracle.light_count(g.row_ptrs, g.cols, q, cl)
        assert on_gpu(dev, g, q, cl=cl) == (want[0], want[1])
    vb, ve = g.n // 5, g.n // 2
    want = oracle.light_count(g.row_ptrs, g.cols, q, 3, v_begin=vb, v_end=ve)
    assert on_gpu(dev, g, q, vb, ve) == (want[0], want[1])
    bounds = [1, 2, g.n // 3, g.n // 3, g.n]
    dg = dev.upload(g)
    got = dev.count_buckets(dg, sme.Plan(q), bounds)[0].tolist()
    dg.release()
    assert got == [oracle.light_count(g.row_ptrs, g.cols, q, 3, v_begin=a, v_end=b)[0] for a, b in zip(bounds, bounds[1:])]


# row sizes at which the packed count changes: 32, 64, 128 members per wave, 512 per workgroup,
# longer rows unpacked (vertex 0 of a clique of n has n - 1 upper neighbours, its first row n - 2)
@pytest.mark.parametrize("q,n", [(7, 67), (7, 131), (11, 70)])
def test_emu_packed_rows(emu, q, n):
    g = union(clique(n) if n < 100 else sme.gen_er(n, n * n // 3, seed=n), sme.gen_er(70, 1200, seed=5))
    want = oracle.light_count(g.row_ptrs, g.cols, q, 3)
    assert emu(g, q) == (want[0], want[1])


@pytest.mark.gpu
@pytest.mark.parametrize("q,n,p", [(7, 98, 1.0), (7, 131, 1.0), (7, 132, 0.9), (7, 300, 0.5), (7, 600, 0.97), (11, 131, 0.6),
                                   (11, 200, 0.7), (7, 900, 0.2)])
def test_packed_rows(dev, q, n, p):
    m = int(p * n * (n - 1) / 2)
    g = clique(n) if p == 1.0 else sme.gen_er(n, m, seed=n)
    cut = max(0, n - 128) if p > 0.9 and n > 500 else 0  # (keeps the oracle's share small)
    want = oracle.light_count(g.row_ptrs, g.cols, q, 3, v_begin=cut)
    got = on_gpu(dev, g, q, cut)
    assert got == (want[0], want[1])
    # the level engine, which the oracle is too slow to stand in for on the dense ones
    dg = dev.upload(g)
    a = dev.count(dg, sme.Plan(q))
    dev.set_tuning(super_chunks=4, clique_level_engine=1)
    b = dev.count(dg, sme.Plan(q))
    dev.set_tuning(super_chunks=4)
    bounds = [0, 1, n // 3, n]
    buckets = dev.count_buckets(dg, sme.Plan(q), bounds)[0]
    dg.release()
    assert (a.count, a.levels) == (b.count, b.levels)
    assert int(buckets.sum()) == a.count


# path runs: bitmaps of 8,192 ids, 32,768 ids and none; a hub whose list is over 16 times the shared one
@pytest.mark.gpu
@pytest.mark.parametrize("n", [8192, 8193, 32768, 32769])
@pytest.mark.parametrize("q", [6, 8])
def test_path_runs(dev, q, n):
    tail = sme.gen_rmat(8, 12, seed=n)
    g = union(hub_and_sparse(n - tail.n, 1500, 6 * n, n), tail)
    assert g.n == n
    want = oracle.light_count(g.row_ptrs, g.cols, q, 3)
    assert want[0] and on_gpu(dev, g, q) == (want[0], want[1])
    bounds = [0, 9, n // 2, n - tail.n, n]
    dg = dev.upload(g)
    got = dev.count_buckets(dg, sme.Plan(q), bounds)[0].tolist()
    dg.release()
    assert got == [oracle.light_count(g.row_ptrs, g.cols, q, 3, v_begin=a, v_end=b)[0] for a, b in zip(bounds, bounds[1:])]


@pytest.mark.parametrize("q", [6, 8])
def test_emu_path_runs(emu, q):
    g = union(hub_and_sparse(400, 90, 700, 3), sme.gen_rmat(5, 8, seed=2))
    for self_loop in (False, True):
        if self_loop:  # the != conditions then count
            src = np.repeat(np.arange(g.n), np.diff(g.row_ptrs.astype(np.int64)))
            key = np.unique(np.concatenate([src * g.n + g.cols, np.arange(0, g.n, 7) * (g.n + 1)]))
            g = sme.Graph(np.searchsorted(key, np.arange(g.n + 1) * g.n).astype(np.uint64),
                          (key % g.n).astype(np.uint32))
        want = oracle.light_count(g.row_ptrs, g.cols, q, 3)
        assert emu(g, q) == (want[0], want[1])


@pytest.mark.gpu
def test_small_calls_in_a_row(dev):
    """Calls whose kernel hands its sums to the host itself, among others that copy theirs, keep apart."""
    gs = [sme.gen_er(n, 3 * n, seed=n) for n in (5, 64, 300, 1000)] + [small_graphs(0)]
    up = [(g, dev.upload(g)) for g in gs]
    want = {(i, q): oracle.light_count(g.row_ptrs, g.cols, q, 3) for i, (g, _) in enumerate(up) for q in (0, 1, 3, 7)}
    for k in range(200):
        i, q = k % len(up), (0, 3, 1, 0, 7)[k % 4]
        r = dev.count(up[i][1], sme.Plan(q))
        assert (r.count, r.levels) == (want[i, q][0], want[i, q][1]), (k, i, q)
    for _, dg in up:
        dg.release()


# upper neighbourhoods at the classes of the dense 4-clique count: 128, 256, 384 and 512 rows, beyond
@pytest.mark.gpu
@pytest.mark.parametrize("d", [65, 127, 128, 129, 256, 257, 384, 385, 512, 513])
def test_dense_rows(dev, d):
    rng = np.random.default_rng(d)
    inner = sme.gen_er(d, min(d * (d - 1) // 2, 14 * d), seed=d)
    first = clique(2)  # vertex 0 below all of them
    src = np.repeat(np.arange(d), np.diff(inner.row_ptrs.astype(np.int64))) + 1
    key = np.unique(np.concatenate([src * (d + 1) + inner.cols + 1, np.arange(1, d + 1),
                                    np.arange(1, d + 1) * (d + 1)]))
    g = sme.Graph(np.searchsorted(key, np.arange(d + 2) * (d + 1)).astype(np.uint64), (key % (d + 1)).astype(np.uint32))
    g = union(g, first, sme.gen_er(150, 6000 + int(rng.integers(50)), seed=d))
    want = oracle.light_count(g.row_ptrs, g.cols, 3, 3)
    assert on_gpu(dev, g, 3) == (want[0], want[1])
    bounds = [0, 1, d // 2, g.n]
    dg = dev.upload(g)
    got = dev.count_buckets(dg, sme.Plan(3), bounds)[0].tolist()
    dg.release()
    assert got == [oracle.light_count(g.row_ptrs, g.cols, 3, 3, v_begin=a, v_end=b)[0] for a, b in zip(bounds, bounds[1:])]


def test_emu_middle_edges(emu):
    """Per-edge counts on the degree-ranked copy: rows from the table, middle edges per u."""
    g = union(sme.gen_er(150, 7000, seed=3), clique(70), sme.gen_rmat(6, 6, seed=2))
    want = oracle.light_count(g.row_ptrs, g.cols, 2, 3)
    assert emu(g, 2, RANK=1) == (want[0], want[1])
    assert emu(g, 4, RANK=1, NOLEVELS=1)[0] == oracle.light_count(g.row_ptrs, g.cols, 4, 3)[0]


# spans and lengths at which u's list leaves the middle pass (1,024 entries, 65,536 ids)
@pytest.mark.gpu
@pytest.mark.parametrize("d,stride", [(300, 1), (300, 230), (1100, 1), (80, 900)])
def test_middle_edges(d, stride):
    g = union(fan(d * stride + 2, d, stride, 30 * d, d), sme.gen_er(400, 24000, seed=d), clique(90))
    ranked = sme.Device(0, budget_bytes=2 << 30)
    ranked.set_rank_order(True)
    dg = ranked.upload(g)
    for q in (2, 4):
        want = oracle.light_count(g.row_ptrs, g.cols, q, 3)
        print(f"case q={q} d={d} stride={stride}", flush=True)
        if q == 2:
            r = ranked.count(dg, sme.Plan(q))
            assert (r.count, r.levels) == (want[0], want[1])
        else:
            assert ranked.count_only(dg, sme.Plan(q)).count == want[0]
    ranked.close()


# graphs that list an edge in one direction only: the passes over edges rely on mirrors and leave
# them to the level engine, with level outputs or without
ONE_WAY = [(7, 6, 4), (6, 8, 3), (8, 5, 9)]


@pytest.mark.parametrize("scale,ef,seed", ONE_WAY[:2])
def test_emu_one_way_edges(emu, scale, ef, seed):
    g = one_way(sme.gen_rmat(scale, ef, seed=seed))
    for q in (2, 4):
        want = oracle.light_count(g.row_ptrs, g.cols, q, 3)
        assert emu(g, q) == (want[0], want[1])
        assert emu(g, q, NOLEVELS=1)[0] == want[0]


@pytest.mark.gpu
@pytest.mark.parametrize("scale,ef,seed", ONE_WAY)
def test_one_way_edges(dev, scale, ef, seed):
    g = one_way(sme.gen_rmat(scale, ef, seed=seed))
    dg = dev.upload(g)
    for q in range(9):
        want = oracle.light_count(g.row_ptrs, g.cols, q, 3)
        r = dev.count(dg, sme.Plan(q))
        assert (r.count, r.levels) == (want[0], want[1]), q
        assert dev.count_only(dg, sme.Plan(q)).count == want[0], q
    dg.release()


@pytest.mark.parametrize("scale,ef,seed", ONE_WAY[:2])
def test_emu_one_way_edges_keep_their_ids(emu, scale, ef, seed):
    """The ids decide which of a one-way graph's edges a count follows: not on the ranked copy."""
    g = one_way(sme.gen_rmat(scale, ef, seed=seed))
    for q in (0, 3, 7):
        want = oracle.light_count(g.row_ptrs, g.cols, q, 3)
        assert emu(g, q, RANK=1) == (want[0], want[1])
    for q in (1, 2, 4, 6, 8):
        assert emu(g, q, RANK=1, NOLEVELS=1)[0] == oracle.light_count(g.row_ptrs, g.cols, q, 3)[0]


@pytest.mark.gpu
@pytest.mark.parametrize("scale,ef,seed", ONE_WAY)
def test_one_way_edges_keep_their_ids(scale, ef, seed):
    g = one_way(sme.gen_rmat(scale, ef, seed=seed))
    d = sme.Device(0, budget_bytes=1 << 30)
    d.set_rank_order(True)
    dg = d.upload(g)
    for q in range(9):
        want = oracle.light_count(g.row_ptrs, g.cols, q, 3)
        r = d.count(dg, sme.Plan(q))
        assert (r.count, r.levels) == (want[0], want[1]), q
        assert d.count_only(dg, sme.Plan(q)).count == want[0], q
    d.close()


def test_emu_rows_of_nine_tenths_of_the_memory(emu, tmp_path):
    """5-clique: vertex 0's rows (500 x 8 words) take four fifths of a 40 KB budget, which they may:
    one batch of rows and no run of the level engine."""
    g = fan(502, 500, 1, 3000, 8)
    want = oracle.light_count(g.row_ptrs, g.cols, 7, 3)
    assert emu(g, 7, budget=40_000) == (want[0], want[1])
    path = str(tmp_path / "g.bin")
    sme.write_bin(path, g)
    r = subprocess.run([os.path.join(EMU_DIR, "emu_driver"), path, "6", "7", "3", "1", "0", str(g.n), "40000"],
                       capture_output=True, text=True, env=dict(os.environ, ASAN_OPTIONS="detect_leaks=0"), timeout=600)
    assert r.stdout.split()[2] == "batches=1"


def slots_used(d, call):
    """Kernel slots that a call times."""
    d.profile(True)
    d.profile_reset()
    call()
    used = {k for k, v in d.profile_read().items() if v["launches"]}
    d.profile(False)
    return used


# a house over start vertices with a few neighbours each, spread over several tiles of ids (and, for
# the largest degree, enough of them): the level engine; over a hub alone: the tiles
@pytest.mark.gpu
@pytest.mark.parametrize("n,d,m,tiles", [(70001, 1000, 140000, False), (60000, 1000, 120000, False),
                                         (300000, 3000, 600000, False), (70001, 3000, 1100000, True)])
def test_house_over_sparse_ids(dev, n, d, m, tiles):
    g = hub_and_sparse(n, d, m, n)
    dg = dev.upload(g)
    plan, hub = sme.Plan(4), n // 3
    got = {}
    assert ("house_wedge" in slots_used(dev, lambda: got.update(r=dev.count(dg, plan)))) == tiles
    dev.set_tuning(super_chunks=4, census_level_engine=1)
    want = dev.count(dg, plan)
    dev.set_tuning(super_chunks=4)
    assert (got["r"].count, got["r"].levels) == (want.count, want.levels)
    assert "house_wedge" in slots_used(dev, lambda: got.update(h=dev.count(dg, plan, hub - 2, hub + 1)))
    want = oracle.light_count(g.row_ptrs, g.cols, 4, 3, v_begin=hub - 2, v_end=hub + 1)
    assert (got["h"].count, got["h"].levels) == (want[0], want[1])
    dg.release()


# lists walked for few (edge, further neighbour) pairs: hubs above all their neighbours (level
# engine), below them (tiles)
@pytest.mark.gpu
@pytest.mark.parametrize("n,hubs,share,m,low,tiles", [(9000, 1, 1.0, 9000, False, False), (60000, 1, 1.0, 60000, False, False),
                                                      (9000, 1, 1.0, 9000, True, True), (70000, 2, 0.4, 70000, False, False),
                                                      (30000, 3, 0.7, 60000, False, True)])
def test_house_under_long_lists(dev, n, hubs, share, m, low, tiles):
    g = hubs_over(n, hubs, share, m, n)
    if low:  # ids in reverse
        src = np.repeat(np.arange(n), np.diff(g.row_ptrs.astype(np.int64)))
        key = np.sort((n - 1 - src) * n + (n - 1 - g.cols.astype(np.int64)))
        g = sme.Graph(np.searchsorted(key, np.arange(n + 1) * n).astype(np.uint64), (key % n).astype(np.uint32))
    dg = dev.upload(g)
    got = {}
    assert ("house_wedge" in slots_used(dev, lambda: got.update(r=dev.count(dg, sme.Plan(4))))) == tiles
    dev.set_tuning(super_chunks=4, census_level_engine=1)
    want = dev.count(dg, sme.Plan(4))
    dev.set_tuning(super_chunks=4)
    assert (got["r"].count, got["r"].levels) == (want.count, want.levels)
    dg.release()


@pytest.mark.gpu
def test_square_over_sparse_ids(dev):
    """Many start vertices just above the light kernel's limits, 13 tiles of ids: the level engine
    takes over what the light kernel has begun; a few of them keep the tiles."""
    g = sme.gen_er(800_000, 9_600_000, seed=4)
    dg = dev.upload(g)
    plan = sme.Plan(1)
    for vb, ve, tiles in ((0, g.n, False), (0, 1000, False), (0, 200, True), (500_000, 500_100, True)):
        got = {}
        bounds = [vb, vb + 3, (vb + ve) // 2, ve]
        used = slots_used(dev, lambda: got.update(r=dev.count(dg, plan, vb, ve)))
        assert used == {"house_wedge"} if tiles else "house_wedge" in used and len(used) > 1
        buckets = dev.count_buckets(dg, plan, bounds)
        dev.set_tuning(super_chunks=4, census_level_engine=1)
        want, each = dev.count(dg, plan, vb, ve), dev.count_buckets(dg, plan, bounds)
        dev.set_tuning(super_chunks=4)
        assert (got["r"].count, got["r"].levels) == (want.count, want.levels)
        assert (buckets[0].tolist(), buckets[1].count, buckets[1].levels) == (each[0].tolist(), want.count, want.levels)
    dg.release()


@pytest.mark.gpu
@pytest.mark.parametrize("n,m,groups", [(1_700_000, 20_400_000, True), (1_200_000, 14_400_000, False)])
def test_house_apexes_over_sparse_ids(n, m, groups):
    """26 tiles of ids and apexes just above the hash's limit: dense arrays, in groups; 19: the tiles."""
    g = sme.gen_er(n, m, seed=6)
    d = sme.Device(0, budget_bytes=16 << 30)
    dg = d.upload(g)
    r = d.count_only(dg, sme.Plan(4))
    assert (r.batches > 1) == groups
    d.set_tuning(super_chunks=4, census_level_engine=1)
    assert r.count == d.count_only(dg, sme.Plan(4)).count
    d.close()


def hubs_over(n, hubs, share, m, seed):
    """The last `hubs` vertices joined to a share of all, on top of m random edges: long lists that
    many runs of one or two short ones share."""
    rng = np.random.default_rng(seed)
    a, b = [rng.integers(0, n, m)], [rng.integers(0, n, m)]
    for h in range(hubs):
        ends = rng.choice(n, size=int(share * n), replace=False)
        a.append(np.full(ends.size, n - 1 - h))
        b.append(ends)
    a, b = np.concatenate(a), np.concatenate(b)
    a, b = a[a != b], b[a != b]
    key = np.unique(np.concatenate([a * n + b, b * n + a]))
    return sme.Graph(np.searchsorted(key, np.arange(n + 1) * n).astype(np.uint64), (key % n).astype(np.uint32))


@pytest.mark.parametrize("q", [6, 8])
def test_emu_path_runs_under_long_lists(emu, q):
    g = hubs_over(900, 2, 0.6, 700, 3)
    want = oracle.light_count(g.row_ptrs, g.cols, q, 3)
    assert emu(g, q) == (want[0], want[1])
    bounds = [0, 9, 450, 899, 900]
    want = [oracle.light_count(g.row_ptrs, g.cols, q, 3, v_begin=a, v_end=b)[0] for a, b in zip(bounds, bounds[1:])]
    assert emu(g, q, bounds=bounds)[2] == want


@pytest.mark.gpu
@pytest.mark.parametrize("n,hubs,share,m", [(8192, 1, 1.0, 8192), (32768, 2, 0.5, 8192), (32768, 1, 1.0, 65536)])
def test_path_runs_under_long_lists(dev, n, hubs, share, m):
    """Runs of few short lists are searched; reading the shared lists for each took 3 to 10 times
    as long as the item schedule, which a setting asks for."""
    g = hubs_over(n, hubs, share, m, n + hubs)
    dg = dev.upload(g)
    for q in (6, 8):
        want = oracle.light_count(g.row_ptrs, g.cols, q, 3)
        r = dev.count(dg, sme.Plan(q))
        assert (r.count, r.levels) == (want[0], want[1])
        bounds = [0, 9, n // 2, n]
        got = dev.count_buckets(dg, sme.Plan(q), bounds)[0].tolist()
        assert got == [oracle.light_count(g.row_ptrs, g.cols, q, 3, v_begin=a, v_end=b)[0]
                       for a, b in zip(bounds, bounds[1:])]
    dg.release()


# dense 4-clique classes of up to 128 rows, 256 (alone or below larger ones) and 512, of fewer and of
# more vertices than fill them: (upper neighbourhoods, copies)
@pytest.mark.gpu
@pytest.mark.parametrize("shapes", [[(100, 3)], [(200, 3)], [(100, 5), (200, 4), (300, 1)], [(200, 130), (300, 2)],
                                    [(300, 130), (500, 2)], [(500, 129), (600, 2)], [(260, 5)]])
def test_dense_classes(dev, shapes):
    g = union(*[fan(d + 1, d, 1, 25 * d, 1000 * d + k) for d, copies in shapes for k in range(copies)])
    want = oracle.light_count(g.row_ptrs, g.cols, 3, 3)
    assert want[0] and on_gpu(dev, g, 3) == (want[0], want[1])
    bounds = [0, 1, g.n // 3, g.n]
    dg = dev.upload(g)
    got = dev.count_buckets(dg, sme.Plan(3), bounds)[0].tolist()
    dg.release()
    assert got == [oracle.light_count(g.row_ptrs, g.cols, 3, 3, v_begin=a, v_end=b)[0] for a, b in zip(bounds, bounds[1:])]


@pytest.mark.gpu
def test_served_house_keeps_its_memory():
    """What a house pass held at its peak is a quarter of what it has to be allowed: the passes
    after the first take as long as it does (the level engine needs over a second)."""
    g = sme.gen_rmat(16, 8, seed=5)
    srv = sme.Server(g, mem_cap_bytes=160 << 20, slots=2, min_reserve_bytes=1 << 20)
    want = None
    for k in range(4):
        count, ms = srv.wait(srv.submit(4, 1, g.n))
        print(f"pass {k}: {ms:.1f} ms", flush=True)
        assert want in (None, count)
        want = count
        assert ms < 300
    ids = [srv.submit(4, a, b) for a, b in ((1, 30000), (20000, 65536), (1, g.n))]
    got = [srv.wait(i) for i in ids]
    assert got[2][0] == want and max(ms for _, ms in got) < 300
    srv.close()


def broad_hubs(low, hubs, m, first, seed):
    """Hubs joined to every one of `low` vertices, on top of G(low, m) among those; the hubs hold the
    first ids or the last.  With its houses and 4-cycles, in closed form."""
    s = sme.gen_er(low, m, seed=seed)
    deg = np.diff(s.row_ptrs.astype(np.int64))
    src = np.repeat(np.arange(low), deg)
    cols = s.cols.astype(np.int64)
    lists = [set(cols[int(s.row_ptrs[v]):int(s.row_ptrs[v + 1])].tolist()) for v in range(low)]
    # 4-cycles: tr A^4 = sum of squared common-neighbour counts = 8 C4 + 2 sum d^2 - sum d
    common = {}
    for v in range(low):
        for a in lists[v]:
            for b in lists[v]:
                common[a, b] = common.get((a, b), 0) + 1
    sums = sum(common.values()), sum(x * x for x in common.values())
    trace = hubs * hubs * low * low + 2 * hubs * sums[0] + sums[1]            # two low vertices
    trace += 2 * hubs * int((deg ** 2).sum()) + hubs * hubs * low * low      # a hub and a low one, two hubs
    d = np.concatenate([deg + hubs, np.full(hubs, low)])
    squares, rest = divmod(trace - 2 * int((d ** 2).sum()) + int(d.sum()), 8)
    assert rest == 0
    # houses: sum over edges of t p - 2 t (t - 1), t triangles and p = A^3 - d(u) - d(v) + 1 4-cycles on it
    houses = 0
    for u, v in zip(src.tolist(), cols.tolist()):
        if u < v:
            t = len(lists[u] & lists[v]) + hubs
            # neighbours x of u, each with its common neighbours with v
            walks = sum(len(lists[x] & lists[v]) + hubs for x in lists[u]) + hubs * int(deg[v])
            houses += t * (walks - int(deg[u] + deg[v]) - 2 * hubs + 1) - 2 * t * (t - 1)
    for v in range(low):  # the edge (hub, v): t = deg(v); x over the low vertices or the neighbours of v
        t = int(deg[v])
        walks = sum(len(lists[x]) for x in lists[v]) + hubs * low  # A^3(v, h) = sum over x in N(v) of common(x, h)
        houses += hubs * (t * (walks - (t + hubs) - low + 1) - 2 * t * (t - 1))
    ids = np.arange(low) + (hubs if first else 0)
    hub_ids = np.arange(hubs) + (0 if first else low)
    n = low + hubs
    a = np.concatenate([ids[src], np.repeat(hub_ids, low), np.tile(ids, hubs)])
    b = np.concatenate([ids[cols], np.tile(ids, hubs), np.repeat(hub_ids, low)])
    key = np.sort(a * n + b)
    g = sme.Graph(np.searchsorted(key, np.arange(n + 1) * n).astype(np.uint64), (key % n).astype(np.uint32))
    return g, houses, squares


def test_broad_hubs_closed_forms():
    for first in (True, False):
        g, houses, squares = broad_hubs(40, 2, 70, first, 3)
        assert oracle.light_count(g.row_ptrs, g.cols, 4, 3)[0] == houses
        assert oracle.light_count(g.row_ptrs, g.cols, 1, 3)[0] == squares


# apexes and start vertices with more neighbours than 16-bit counters hold: dense arrays, here in one
# group and in two; the level engine for the 4-cycle
@pytest.mark.gpu
@pytest.mark.parametrize("budget,groups", [(1 << 30, 1), (6 << 20, 2)])
@pytest.mark.parametrize("ranked", [False, True])
def test_apexes_over_65535_neighbours(budget, groups, ranked):
    g, houses, squares = broad_hubs(65600, 3, 20000, False, 5)
    d = sme.Device(0, budget_bytes=budget)
    d.set_rank_order(ranked)
    dg = d.upload(g)
    r = d.count_only(dg, sme.Plan(4))
    assert r.count == houses and r.batches == 1 + groups
    assert d.count_only(dg, sme.Plan(1)).count == squares
    d.close()


@pytest.mark.gpu
def test_start_vertices_over_65535_neighbours(dev):
    g, _, squares = broad_hubs(65600, 3, 20000, True, 6)
    dg = dev.upload(g)
    assert dev.count(dg, sme.Plan(1)).count == squares
    vb, ve = 3, 40000  # (the hubs are not among the start vertices, but the graph has them)
    want = oracle.light_count(g.row_ptrs, g.cols, 1, 3, v_begin=vb, v_end=ve)
    r = dev.count(dg, sme.Plan(1), vb, ve)
    assert (r.count, r.levels) == (want[0], want[1])
    dg.release()


# lists of which a wave streams 1,024 entries at a time, just below, at and above one and two such steps
@pytest.mark.gpu
@pytest.mark.parametrize("degree", [1000, 1023, 1024, 1025, 2047, 2048, 2049, 9000])
def test_path_runs_over_long_lists(dev, degree):
    n = 9216
    low = np.zeros(0, dtype=np.int64)
    a, b = [low], [low]
    for h, step in ((n - 1, 1), (n - 2, 2), (n - 3, 3)):  # (the hubs' lists have ends in common)
        ends = (np.arange(degree) * step) % (n - 3)
        a.append(np.full(degree, h))
        b.append(ends)
    # the hubs among themselves, and what each path adds
    a += [np.array([n - 1, n - 1, n - 2]), np.arange(0, 6000, 2)]
    b += [np.array([n - 2, n - 3, n - 3]), np.arange(1, 6001, 2)]
    a, b = np.concatenate(a), np.concatenate(b)
    key = np.unique(np.concatenate([a * n + b, b * n + a]))
    g = sme.Graph(np.searchsorted(key, np.arange(n + 1) * n).astype(np.uint64), (key % n).astype(np.uint32))
    for q in (2, 6, 8):
        for vb, ve in ((0, n), (n - 3, n)):
            want = oracle.light_count(g.row_ptrs, g.cols, q, 3, v_begin=vb, v_end=ve)
            assert on_gpu(dev, g, q, vb, ve) == (want[0], want[1])


# rows of few vertices (64 a workgroup) and of as many as fill the chip (256), in one part and two
@pytest.mark.gpu
@pytest.mark.parametrize("d,copies", [(65, 1), (257, 7), (256, 2), (66, 504), (66, 512), (257, 248), (257, 256), (66, 2048), (257, 1024)])
def test_row_parts(dev, d, copies):
    g = union(*[fan(d + 1, d, 1, 6 * d, 100 * copies + k) for k in range(min(copies, 8))] * (-(-copies // 8)))
    assert g.n >= copies * (d + 1)
    for q in (0, 2, 3, 7):
        want = oracle.light_count(g.row_ptrs, g.cols, q, 3)
        assert want[0] and on_gpu(dev, g, q) == (want[0], want[1])
    dg = dev.upload(g)
    assert dev.count_only(dg, sme.Plan(4)).count == oracle.light_count(g.row_ptrs, g.cols, 4, 3)[0]
    dg.release()


# cliques whose first rows have as many members as a wave, a workgroup of either size and neither packs,
# and one more; no kernel is launched for rows that cannot be there
@pytest.mark.gpu
@pytest.mark.parametrize("n,q", [(n, 7) for n in (66, 129, 130, 131, 257, 258, 259, 513, 514, 515)] +
                                [(n, 11) for n in (66, 129, 130, 131, 258)])
def test_clique_rows_by_size(dev, n, q):
    k = 5 if q == 7 else 6
    count, levels = on_gpu(dev, clique(n), q)
    assert count == math.comb(n, k) == levels[-1]
    assert sorted(set(levels)) == sorted({math.comb(n, j) for j in range(1, k + 1)})
