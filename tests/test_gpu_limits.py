"""Builds, cleans and host calls at the limits of their buffers, lists and
counters.  Labels, answers and counts are integers: every comparison is exact."""
import os
import subprocess
import sys
import time

import numpy as np
import pytest

import gpu4hophl_code_amd as H
import oracle_lib as O
from test_gpu_parity import csr_of, same_labels
from test_gpu_variants import ragged

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heavy", ["1", "512", "65536"])
def test_lists_that_run_out_inside_an_expansion(monkeypatch, heavy):
    """Candidate lists far below a round's candidates, so that workgroups of
    the expansion set the batch's stop flag while others of the same launch
    start, with every frontier group in heavy pieces, some and none: the
    oracle's labels after the batches have been rolled back and run again."""
    monkeypatch.setenv("HSDL_LIST_INIT", "64")
    monkeypatch.setenv("HSDL_HEAVY_PAIRS", heavy)
    for n, K, wmax, batch in ((3000, 4, 100, 64), (1200, 5, 30000, 16), (700, 3, 9, 0)):
        print(f"[lists run out] n={n} K={K} batch={batch} heavy={heavy}", flush=True)
        g = ragged(n, n + K, wmax, 16)
        same_labels(H.hop_constrained_two_hop_labels_generation(g, K, hub_batch=batch),
                    O.kround(csr_of(g), K).arrays())


@pytest.mark.parametrize("pad", [0, 5000])
def test_clean_of_chains_over_many_rounds(pad):
    """Lists whose labels each fall through the one before, if that one is
    kept: at K = 15 the decisions run along chains of 15, over windows that
    different waves take, so a list needs several rounds of the clean's second
    pass.  Chains of every length side by side in 2,000 lists, with and without
    hubs between them that push the list out of LDS: the oracle's clean."""
    K = 15
    rng = np.random.default_rng(pad + 1)
    lists = [[(0, 0, 0)]]
    # hub x: a label through hub x - 1, so that a kept (x - 1, h, d) removes (x, h + 1, d + 1)
    lists += [[(x - 1, 1, 1), (x, 0, 0)] for x in range(1, 400 + pad)]
    for v in range(2000 if not pad else 300):
        x, rows = 0, []
        while x < 380:
            for i in range(int(rng.integers(1, K + 1))):
                # now and then a distance too small to fall
                rows.append((x, i + 1, 40 + i - 3 * int(rng.random() < 0.05)))
                x += 1
            x += int(rng.integers(1, 4))
        rows = [r for r in rows if r[0] < 400]
        if v % 3 == 0:
            rows += [(400 + u, 1 + u % K, 1 + u % 7) for u in range(pad)]
        lists.append(rows + [(len(lists), 0, 0)])
    off = np.concatenate([[0], np.cumsum([len(x) for x in lists])])
    hub, hop, dist = np.array([e for x in lists for e in x]).T
    hub, hop, dist = hub.astype(np.uint32), hop.astype(np.uint8), dist.astype(np.int32)
    n = len(lists)
    want = O.clean(O.labels_from_arrays(n, off.astype(np.int64), hub, hop, dist))
    print(f"[chains] n={n} labels={len(hub)} kept={want.total()}", flush=True)
    assert want.total() < len(hub) - n
    idx = H.Index.from_labels(n, K, off.astype(np.uint64), hub, hop, dist)
    idx.clean()
    same_labels(idx, want.arrays())


@pytest.mark.parametrize("n", [9001, 20000, 70000])
def test_row_slots_count_each_scan_once(monkeypatch, n):
    """Stars: the centre has every other vertex as a candidate, so a row item's
    candidates fill the LDS list several times over and its slots are loaded
    again for each further piece.  prune_row_slots counts a scan of a slot once:
    the rows of n slots of the centre's batch, in the one round with candidates."""
    monkeypatch.setenv("HSDL_PRUNE_ROWS", "2")
    u = np.zeros(n - 1, np.uint32)
    v = np.arange(1, n, dtype=np.uint32)
    g = H.Graph.from_edges(n, u, v, np.full(n - 1, 3, np.int32))
    for K in (1, 3):
        print(f"[row slots] n={n} K={K}", flush=True)
        idx = H.hop_constrained_two_hop_labels_generation(g, K, hub_batch=64)
        same_labels(idx, O.kround(csr_of(g), K).arrays())
        assert idx.stats()["prune_row_slots"] == 64 * n


def test_a_retried_batch_counts_its_landmark_tests_once(monkeypatch):
    """A batch whose landmark tests reject nothing ends the test from 4,096
    tests on.  Hubs 16..31 of this graph make 2,880 of them, in a round whose
    candidates outgrow 2,048 list entries: run again with larger lists the batch
    still counts 2,880, so the later hubs, where landmarks reject most pairs,
    open as many candidates as without the retry."""
    monkeypatch.setenv("HSDL_HEAVY_PAIRS", "65536")
    edges, n = [], 32
    for x in range(16, 32):  # 60 neighbours each, three more behind each of those
        for _ in range(60):
            y, n = n, n + 1
            edges.append((x, y, 5))
            for _ in range(3):
                edges.append((y, n, 5))
                n += 1
    rng = np.random.default_rng(8)
    late = np.arange(n, n + 180)  # next to hubs 0..7, and among themselves far apart
    n += 180
    edges += [(x, y, 1) for x in range(8) for y in late]
    edges += [(x, y, 50) for x, y in rng.choice(late, (800, 2)) if x != y]
    u, v, w = np.array(edges).T
    g = H.Graph.from_edges(n, u.astype(np.uint32), v.astype(np.uint32), w.astype(np.int32))
    want = O.kround(csr_of(g), 2).arrays()
    cands = []
    for lists in (None, "2048"):
        if lists:
            monkeypatch.setenv("HSDL_LIST_INIT", lists)
        print(f"[retried batch] n={n} lists={lists}", flush=True)
        idx = H.hop_constrained_two_hop_labels_generation(g, 2, hub_batch=16)
        same_labels(idx, want)
        cands.append(idx.stats()["candidates"])
    assert cands[0] == cands[1]


@pytest.mark.parametrize("mb", [1400, 1520, 1700])
def test_growing_batches_leave_the_budget_to_the_pool(mb):
    """Builds within budgets that hold the labels as long as the candidate lists
    stay small: batches that grow eightfold outgrow the lists, and lists
    grown for them would leave the label pool no room to grow in.  The labels of
    a build without such a limit."""
    K = 5
    g = H.Graph.rmat(15, 16, 7, 1, 40000)
    want = H.hop_constrained_two_hop_labels_generation(g, K, hbm_budget=60 << 30).labels()
    g = H.Graph.rmat(15, 16, 7, 1, 40000)  # another handle: nothing kept from the first build
    print(f"[tight budget] {mb} MB", flush=True)
    idx = H.hop_constrained_two_hop_labels_generation(g, K, hbm_budget=mb << 20,
                                                      pool_init_labels=4 * len(want[1]))
    same_labels(idx, want)


@pytest.mark.parametrize("scale,K,batch,group,budget", [
    (14, 5, 64, True, 260762640), (14, 2, 1, False, 176436256), (13, 1, 16, False, 163329296)])
def test_least_budgets(monkeypatch, scale, K, batch, group, budget):
    """The least budgets of builds whose buffers never grow, as the per-vertex
    state, slots, lists, pool and tile arena of a 256-CU device add up to: any
    further array per vertex would refuse them."""
    monkeypatch.setenv("HSDL_LIST_INIT", "2000000")
    monkeypatch.setenv("HSDL_HEAVY_CAP", "4096")
    g = H.Graph.rmat(scale, 8, 7, 1, 100)
    hubs = np.arange(0, g.n, 3, dtype=np.uint32) if group else None
    print(f"[least budget] scale={scale} K={K} batch={batch} group={group}", flush=True)
    idx = H.hop_constrained_two_hop_labels_generation(g, K, hbm_budget=budget, hubs=hubs,
                                                      pool_init_labels=400 * g.n, hub_batch=batch)
    if not group:
        same_labels(idx, O.kround(csr_of(g), K).arrays())


@pytest.mark.parametrize("stream32", ["1", "0"])
def test_pool_that_runs_out_between_vertices(monkeypatch, stream32):
    """A pool that takes some vertices' longer segments and not others', so that
    part of a round's labels is written before the batch is rolled back and run
    again: the oracle's labels."""
    monkeypatch.setenv("HSDL_STREAM32", stream32)
    for n, K, batch, extra in ((3000, 4, 64, 40), (3000, 4, 700, 3000), (1300, 5, 0, 9)):
        print(f"[pool] n={n} K={K} batch={batch} extra={extra} stream32={stream32}", flush=True)
        g = ragged(n, n + K, 60, 16)
        same_labels(H.hop_constrained_two_hop_labels_generation(
            g, K, hub_batch=batch, pool_init_labels=16 * n + extra),
            O.kround(csr_of(g), K).arrays())


def skewed(rng, n, short, longs, size, K, far):
    """n - longs lists of up to `short` even hubs, then `longs` lists of `size`
    odd ones: pairs of a long list's labels find no partner in its heads' lists,
    but for its few even hubs.  far: distances fall with the hop, so that no pair
    passes the clean's distance bound; else nearly all do."""
    lists, base = [], n - longs
    for v in range(n):
        if v < base:
            u = np.sort(rng.choice((v + 1) // 2, min(v // 2, short), replace=False)) * 2
            u = u[u < v]
            hop, dist = rng.integers(1, K + 1, len(u)), rng.integers(1, 10, len(u))
        else:
            odd = rng.choice(base // 2, size, replace=False) * 2 + 1
            u = np.unique(np.concatenate([odd, rng.choice(base // 2, 5) * 2]))
            hop = rng.integers(1, K + 1, len(u))
            dist = 1000 * (K - hop) + 500 + rng.integers(0, 400, len(u)) if far else \
                rng.integers(5, 60, len(u))
        lists.append((np.append(u, v), np.append(hop, 0), np.append(dist, 0)))
    off = np.concatenate([[0], np.cumsum([len(x[0]) for x in lists])]).astype(np.uint64)
    hub, hop, dist = (np.concatenate([x[i] for x in lists]) for i in range(3))
    return off, hub.astype(np.uint32), hop.astype(np.uint8), dist.astype(np.int32)


@pytest.mark.parametrize("stream32,piece", [("1", None), ("0", None), ("1", "9000")])
@pytest.mark.parametrize("far", [False, True])
def test_clean_leaves_costly_lists_to_the_tiles(monkeypatch, stream32, piece, far):
    """Lists whose pairs are too many for the clean's pair form go on to the
    tiles: from a wave's lists and from a workgroup's (past 1,024 labels), from
    32-bit and 8-byte copies, whole and sliced, beside lists that stay: the
    oracle's clean."""
    monkeypatch.setenv("HSDL_CLEAN_PAIRS", "2")
    monkeypatch.setenv("HSDL_STREAM32", stream32)
    if piece:
        monkeypatch.setenv("HSDL_CLEAN_SLICE", piece)
    rng = np.random.default_rng(12)
    for n, short, longs, size, K in ((5000, 20, 12, 1900, 5), (5000, 20, 40, 1000, 5), (17000, 10, 3, 8300, 4),
                                     (2000, 9, 200, 300, 15)):
        a = skewed(rng, n, short, longs, size, K, far)
        want = O.clean(O.labels_from_arrays(n, a[0].astype(np.int64), *a[1:]))
        print(f"[skewed clean] n={n} size={size} far={far} kept={want.total()} of {len(a[1])}",
              flush=True)
        idx = H.Index.from_labels(n, K, *a)
        idx.clean()
        same_labels(idx, want.arrays())


def test_clean_of_a_few_long_lists_is_not_quadratic():
    """Four lists of 60,000 labels whose heads have twenty each: 0.34 s by pairs
    alone, a twentieth of that where they go on to the tiles."""
    a = skewed(np.random.default_rng(3), 140000, 20, 4, 60000, 5, False)
    sec = []
    for _ in range(3):
        idx = H.Index.from_labels(140000, 5, *a)
        idx.clean()
        sec.append(idx.stats()["t_clean_s"])
    print(f"[long lists] {sec}", flush=True)
    assert min(sec) < 0.1


def mixed_lists(rng, n, sizes, K, top):
    """n - len(sizes) lists of up to 20 hubs, then one of each of `sizes`."""
    base, rows = n - len(sizes), []
    for v in range(n):
        m = min(v, int(rng.integers(0, 21))) if v < base else sizes[v - base]
        u = np.sort(rng.choice(min(v, base), m, replace=False)) if m else np.zeros(0, int)
        rows.append((np.append(u, v), np.append(rng.integers(1, K + 1, m), 0),
                     np.append(rng.integers(1, top, m), 0)))
    off = np.concatenate([[0], np.cumsum([len(x[0]) for x in rows])]).astype(np.uint64)
    hub, hop, dist = (np.concatenate([x[i] for x in rows]) for i in range(3))
    return off, hub.astype(np.uint32), hop.astype(np.uint8), dist.astype(np.int32)


@pytest.mark.parametrize("team", ["0", "6000"])
@pytest.mark.parametrize("q32,slots", [("1", "1024"), ("1", "2048"), ("0", "1024")])
def test_query_of_lists_far_above_the_mean(monkeypatch, q32, slots, team):
    """A few long lists among many short ones: parts that fill the table to the
    last slot and outgrow it (answered from the 8-byte labels, in pieces), and
    lists past 8,192 labels that a short one searches, beside every other pair
    of lengths, a wave, four and eight waves per query: the oracle's answers."""
    monkeypatch.setenv("HSDL_QUERY32", q32)
    monkeypatch.setenv("HSDL_QUERY_SLOTS", slots)
    monkeypatch.setenv("HSDL_QUERY_TEAM", team)
    rng = np.random.default_rng(41)
    n, K = 20000, 5
    sizes = [128, 129, 510, 514, 1023, 1030, 2600, 5200, 8191, 8193, 8200, 12000, 12000]
    a = mixed_lists(rng, n, sizes, K, 2000)
    want = O.labels_from_arrays(n, a[0].astype(np.int64), *a[1:])
    idx = H.Index.from_labels(n, K, *a)
    s, t = rng.integers(0, n, (2, 6000))
    s[:4000] = n - len(sizes) + rng.integers(0, len(sizes), 4000)
    t[2000:4000] = n - len(sizes) + rng.integers(0, len(sizes), 2000)
    s, t = s.astype(np.uint32), t.astype(np.uint32)
    swap = rng.random(6000) < 0.5
    s, t = np.where(swap, t, s), np.where(swap, s, t)
    k = rng.integers(-1, K + 3, 6000).astype(np.int8)
    ans = O.query(want, s, t, k)
    for m in (6000, 1000, 1):
        print(f"[long lists] q32={q32} slots={slots} team={team} queries={m}", flush=True)
        o = 1500
        sl = slice(0, m) if m > 1000 else slice(o, o + m)
        assert np.array_equal(idx.query(s[sl], t[sl], k[sl]), ans[sl])


def test_queries_of_a_short_and_a_long_list_are_quick():
    """100,000 queries of a list of at most 20 labels and one of 60,000: 0.2 ms
    with their copies, and 5 ms where all of the long list is read."""
    rng = np.random.default_rng(6)
    n, nq = 70000, 100000
    idx = H.Index.from_labels(n, 5, *mixed_lists(rng, n, [60000] * 16, 5, 2000))
    s, t = rng.integers(100, 60000, nq).astype(np.uint32), rng.integers(n - 16, n, nq).astype(np.uint32)
    k = rng.integers(2, 6, nq).astype(np.int8)
    sec = []
    for _ in range(6):
        t0 = time.perf_counter()
        idx.query(s, t, k)
        sec.append(time.perf_counter() - t0)
    print(f"[short and long] {sec}", flush=True)
    assert min(sec) < 2e-3


@pytest.mark.parametrize("n,K,ef", [(6000, 4, 16), (3000, 5, 4), (300, 15, 3)])
def test_query_forms_by_call_size(n, K, ef):
    """Calls on both sides of every line of the choice between the query copy
    and the 8-byte labels, and between a wave, four and eight waves per query:
    the oracle's answers, in one call and over the same requests in another."""
    g = ragged(n, n, 1000, ef)
    want = O.kround(csr_of(g), K)
    idx = H.hop_constrained_two_hop_labels_generation(g, K)
    mean = idx.label_count() // n
    line = int(3 * 2 ** 30 / mean ** 2)
    rng = np.random.default_rng(n)
    sizes = {1, 2, 63, 64, 65, 1023, 1024, 1025, 2047, 2048, 2049, mean ** 2 // 4, mean ** 2 // 4 + 1,
             line, line + 1, 150001}
    most = 150001
    s, t = rng.integers(0, n, (2, most)).astype(np.uint32)
    t[:50] = s[:50]
    k = rng.integers(-1, K + 3, most).astype(np.int8)
    ans = O.query(want, s, t, k)
    for m in sorted(x for x in sizes if 0 < x <= most):
        print(f"[form] n={n} mean={mean} queries={m}", flush=True)
        assert np.array_equal(idx.query(s[:m], t[:m], k[:m]), ans[:m])


@pytest.mark.parametrize("q32", ["0", "1"])
@pytest.mark.parametrize("n", [900, 6000])
def test_team_requests_in_chunks(monkeypatch, q32, n):
    """A workgroup takes consecutive queries: one, several, 64 and more than 64
    each, with a remainder at the call's end, queries without a join among
    them: the oracle's answers, through host arrays, without allocation and
    served."""
    monkeypatch.setenv("HSDL_QUERY32", q32)
    monkeypatch.setenv("HSDL_QUERY_TEAM", "10000000")
    g = ragged(n, n, 100, 8)
    want = O.kround(csr_of(g), 3)
    idx = H.hop_constrained_two_hop_labels_generation(g, 3)
    rng = np.random.default_rng(n)
    most = 250007
    s, t = rng.integers(0, n, (2, most)).astype(np.uint32)
    t[::7] = s[::7]
    k = rng.integers(-1, 5, most).astype(np.int8)
    ans = O.query(want, s, t, k)
    for m in (1, 1023, 1025, 2047, 2049, 4097, 10001, 131071, 131073, most):
        print(f"[team chunks] n={n} q32={q32} queries={m}", flush=True)
        assert np.array_equal(idx.query(s[:m], t[:m], k[:m]), ans[:m])
        assert np.array_equal(idx.query_noalloc(s[:m], t[:m], k[:m]), ans[:m])
    srv = H.Server(idx, max_batch=5003, max_wait_us=50, inflight=3)
    got, _ = srv.replay(s, t, k, np.arange(most, dtype=np.uint64) * 5)
    srv.close()
    assert np.array_equal(got, ans)


@pytest.mark.parametrize("deg", [1000, 2600, 9000])
def test_paths_between_short_and_long_lists(deg):
    """A few vertices of the lowest ranks next to very many others: their lists
    span several staged pieces of 512 labels, or are searched by the other's
    where that is far shorter (past 2,048 labels); weights 1..2, so that equal
    sums meet on both sides of a piece's end: the oracle's edges."""
    n, last = 12000, 6
    rng = np.random.default_rng(deg)
    base = n - last
    u = [np.full(deg, x) for x in range(base, n)]
    v = [rng.choice(base, deg, replace=False) for _ in range(last)]
    y = rng.integers(0, base, (2, 3 * n))
    y = y[:, y[0] != y[1]]
    u, v = np.concatenate(u + [y[0]]), np.concatenate(v + [y[1]])
    g = H.Graph.from_edges(n, u.astype(np.uint32), v.astype(np.uint32),
                           rng.integers(1, 3, len(u)).astype(np.int32))
    idx = H.hop_constrained_two_hop_labels_generation(g, 2, parents=True)
    want = O.kround(csr_of(g), 2)
    lens = np.diff(np.asarray(want.arrays()[0]).astype(np.int64))
    print(f"[paths] deg={deg} longest={lens.max()} mean={lens.mean():.0f}", flush=True)
    assert lens.max() > 1024 and lens[-last:].min() > deg
    short = np.argsort(lens)[:80]
    assert deg < 2000 or lens[-last:].min() > 64 * lens[short].max()
    s, t = rng.integers(0, n, (2, 3000)).astype(np.uint32)
    s[:1800] = base + rng.integers(0, last, 1800)
    t[:900] = rng.choice(short, 900)
    t[900:1800] = base + rng.integers(0, last, 900)
    swap = rng.random(3000) < 0.5
    s, t = np.where(swap, t, s), np.where(swap, s, t)
    k = rng.integers(0, 4, 3000).astype(np.int8)
    edges, counts = idx.paths(s, t, k, cap=3)
    wedges, wcounts = O.paths(want, s, t, k.astype(np.int32), 3)
    assert np.array_equal(counts.astype(np.int32), wcounts)
    assert np.array_equal(edges.astype(np.int32), wedges)


@pytest.mark.parametrize("cap", [1, 7, 31, 32, 33, 70])
def test_path_rows_of_every_width(cap):
    """Paths of up to 30 edges (K = 15 on a path) into rows below, at and past the 64
    words that a wave stores at once, cut at the row's end: the oracle's rows."""
    n, K = 61, 15
    at = np.argsort(np.abs(np.arange(n) - n // 2), kind="stable")  # the middle ranks first
    ids = np.argsort(at).astype(np.uint32)
    g = H.Graph.from_edges(n, ids[:-1], ids[1:], np.full(n - 1, 2, np.int32))
    idx = H.hop_constrained_two_hop_labels_generation(g, K, parents=True)
    want = O.kround(csr_of(g), K)
    s, t = (x.ravel().astype(np.uint32) for x in np.meshgrid(np.arange(n), np.arange(n)))
    k = np.full(n * n, 40, np.int8)
    edges, counts = idx.paths(s, t, k, cap=cap)
    wedges, wcounts = O.paths(want, s, t, k.astype(np.int32), cap)
    print(f"[path rows] cap={cap} longest={wcounts.max()}", flush=True)
    assert wcounts.max() == 30
    assert np.array_equal(counts.astype(np.int32), wcounts)
    assert np.array_equal(edges.astype(np.int32), wedges)


FIRST_CALLS = """
import sys, time
import numpy as np
import gpu4hophl_code_amd as H
g = H.Graph.rmat(12, 8, 1, 1, 100)
n = g.info()[0]
idx = H.hop_constrained_two_hop_labels_generation(g, 4, parents=True)
rng = np.random.default_rng(1)
s, t = rng.integers(0, n, (2, 1 << 18)).astype(np.uint32)
k = rng.integers(1, 5, 1 << 18).astype(np.int8)
t0 = time.perf_counter()
idx.paths(s[:1024], t[:1024], k[:1024], cap=4)
idx.paths(s, t, k, cap=4)
print(1e3 * (time.perf_counter() - t0))
"""


def test_first_host_calls_of_a_process():
    """A small and a large path call, the first of their process: 5 ms together, and 16
    with a second stream and the process's first asynchronous copy in them."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    ms = []
    for _ in range(3):
        out = subprocess.run([sys.executable, "-c", FIRST_CALLS], cwd=root, timeout=100,
                             capture_output=True, text=True)
        assert out.returncode == 0, out.stderr[-2000:]
        ms.append(float(out.stdout.split()[-1]))
        print(f"[first calls] {ms[-1]:.2f} ms", flush=True)
    assert min(ms) < 11


@pytest.fixture(scope="module")
def room_driver(tmp_path_factory):
    """tests/clean_room_driver.cpp, and label sets with redundant labels: short lists, and
    short lists with long ones that leave the pair form (tiles beside its copy)."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    tmp = tmp_path_factory.mktemp("room")
    exe, lib = str(tmp / "driver"), os.path.join(root, "gpu4hophl_code_amd")
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", os.path.join(root, "include"),
                           os.path.join(root, "tests", "clean_room_driver.cpp"), "-o", exe,
                           "-rdynamic", "-L", lib, "-lhsdl", "-ldl", f"-Wl,-rpath,{lib}"])
    dumps = []
    for sizes in ([], [9000, 12000]):
        a = mixed_lists(np.random.default_rng(8), 30000, sizes, 5, 300)
        dumps.append(str(tmp / f"labels{len(sizes)}.bin"))
        H.Index.from_labels(30000, 5, *a).save(dumps[-1])
    return exe, dumps


@pytest.mark.parametrize("what", ["room", "refused"])
@pytest.mark.parametrize("longer", [0, 1])
def test_clean_where_memory_is_short(room_driver, what, longer):
    """A clean takes no more device memory than its least form (tiles over the index's own
    labels) has to have: with exactly that much it gives the labels that it
    gives with all there is.  Each allocation of a clean refused in turn: the same labels, or
    the documented refusal, the index as it was and the next clean right."""
    exe, dumps = room_driver
    out = subprocess.run([exe, dumps[longer], "5", what], timeout=110, capture_output=True, text=True)
    print(out.stdout, flush=True)
    assert out.returncode == 0 and f"{what} done" in out.stdout, out.stderr[-2000:]


def test_build_after_one_that_passed_its_deadline():
    """A build that ends between batches leaves its buffers to the graph's next build,
    with a batch's re-sort still queued: the next build's labels are another handle's."""
    g, other = (H.Graph.rmat(15, 16, 5, 1, 100) for _ in range(2))
    want = H.hop_constrained_two_hop_labels_generation(other, 4).labels()
    for batch in (3000, 0, 700):
        with pytest.raises(H.HSDLError) as e:
            H.hop_constrained_two_hop_labels_generation(g, 4, hub_batch=batch, deadline_s=1e-6)
        assert e.value.code == -5
        same_labels(H.hop_constrained_two_hop_labels_generation(g, 4), want)


@pytest.fixture(scope="module")
def long_lists():
    """Vertices of the lowest ranks next to 450 to 6,500 others: lists that grow past what
    the re-sort holds in registers (1,024 labels, 512 of 8 bytes) and its LDS slices."""
    degs = [450, 540, 900, 1100, 1340, 1420, 3000, 4000, 4300, 6500]
    n = 8000
    base = n - len(degs)
    rng = np.random.default_rng(17)
    u = [np.full(d, base + i) for i, d in enumerate(degs)]
    v = [rng.choice(base, d, replace=False) for d in degs]
    y = rng.integers(0, base, (2, 2 * n))
    y = y[:, y[0] != y[1]]
    u, v = np.concatenate(u + [y[0]]), np.concatenate(v + [y[1]])
    g = H.Graph.from_edges(n, u.astype(np.uint32), v.astype(np.uint32),
                           rng.integers(1, 30, len(u)).astype(np.int32))
    return g, O.kround(csr_of(g), 3).arrays()


@pytest.mark.parametrize("stream32,held,default", [("1", 1024, 4080), ("0", 512, 1360)])
@pytest.mark.parametrize("lds,piece", [(None, None), ("0", None), ("700", None), ("0", "2000"),
                                       ("700", "2000"), ("1300", "64")])
def test_resort_of_long_lists(monkeypatch, long_lists, stream32, held, default, lds, piece):
    """Lists around the re-sort's register limit, its LDS slice and its slice in memory:
    scattered in LDS, in memory, or left unsorted past a capped slice, in 32- and
    8-byte labels, over batches that add to lists sorted before: the oracle's labels."""
    monkeypatch.setenv("HSDL_STREAM32", stream32)
    monkeypatch.setenv("HSDL_RESORT_DIV", "8")
    if lds:
        monkeypatch.setenv("HSDL_SORT_LDS", lds)
    if piece:
        monkeypatch.setenv("HSDL_SORT_SLICE", piece)
    g, want = long_lists
    lens = np.diff(np.asarray(want[0]).astype(np.int64))
    in_lds = int(lds or default)
    most = max(in_lds, int(piece or lens.max()))
    print(f"[re-sort] stream32={stream32} lds={lds} slice={piece} "
          f"held={(lens <= held).sum()} lds={((lens > held) & (lens <= in_lds)).sum()} "
          f"memory={((lens > max(held, in_lds)) & (lens <= most)).sum()} "
          f"unsorted={(lens > max(held, most)).sum()}", flush=True)
    assert (lens > max(held, most)).any() if piece else (lens > max(held, in_lds)).any()
    assert in_lds <= held or ((lens > held) & (lens <= in_lds)).any()
    for batch in (600, 0):
        same_labels(H.hop_constrained_two_hop_labels_generation(g, 3, hub_batch=batch), want)


def test_query_copy_of_lists_of_every_length():
    """The query copy holds lists of up to 1,024 labels in a wave's registers, 64 at a time,
    and reads longer ones twice: empty lists, lists around every 64th length up to
    1,100 and far longer ones, with hops up to 15, queried through the copy: the oracle's
    answers."""
    rng = np.random.default_rng(5)
    lens = sorted({0, 1, 2, 62, 63, 64, 1022, 1023, 1024, 1025, 1100, 3000, 5001} |
                  {64 * i + d for i in range(1, 17) for d in (-1, 0, 1)})
    base, K = 6000, 15
    rows = [(np.zeros(0, int),) * 3 for _ in range(base)]  # no labels, not even their own
    for m in lens:
        u = np.sort(rng.choice(base, m, replace=False))
        rows.append((u, rng.integers(1, K + 1, m), rng.integers(1, 900, m)))
    n = len(rows)
    off = np.concatenate([[0], np.cumsum([len(x[0]) for x in rows])]).astype(np.uint64)
    hub, hop, dist = (np.concatenate([x[i] for x in rows]) for i in range(3))
    a = (off, hub.astype(np.uint32), hop.astype(np.uint8), dist.astype(np.int32))
    want = O.labels_from_arrays(n, off.astype(np.int64), *a[1:])
    idx = H.Index.from_labels(n, K, *a)
    s, t = (x.ravel().astype(np.uint32) for x in np.meshgrid(np.arange(base, n), np.arange(base, n)))
    for kk in (1, 2, 7, 16, 30):
        k = np.full(len(s), kk, np.int8)
        print(f"[copy] lists={n - base} queries={len(s)} k={kk}", flush=True)
        os.environ["HSDL_QUERY32"] = "1"
        try:
            got = idx.query(s, t, k)
        finally:
            del os.environ["HSDL_QUERY32"]
        assert np.array_equal(got, O.query(want, s, t, k))


def test_builds_on_several_threads():
    """Eight threads build, clean, query and extract paths on graphs of their own at the
    same time, with the kept buffers released in between: no call is refused for what
    another thread does, and all answers are the oracle's."""
    from concurrent.futures import ThreadPoolExecutor
    sets = []
    for i in range(4):
        n, K = 700 + 400 * i, 3 + i % 3
        c = csr_of(ragged(n, 50 + i, 50))
        red = O.kround_gid(c, K, (np.arange(n) % 3).astype(np.int32))
        sets.append((n, K, O.kround(c, K), red, O.clean(red)))

    def work(j):
        n, K, want, red, cleaned = sets[j % 4]
        rng = np.random.default_rng(j)
        g = ragged(n, 50 + j % 4, 50)
        for r in range(6):
            idx = H.hop_constrained_two_hop_labels_generation(g, K, parents=True)
            same_labels(idx, want.arrays())
            s, t = rng.integers(0, n, (2, 3000)).astype(np.uint32)
            k = rng.integers(0, K + 3, 3000).astype(np.int8)
            assert np.array_equal(idx.query(s, t, k), O.query(want, s, t, k))
            edges, counts = idx.paths(s, t, k, cap=K)
            wedges, wcounts = O.paths(want, s, t, k.astype(np.int32), K)
            assert np.array_equal(counts.astype(np.int32), wcounts)
            assert np.array_equal(edges.astype(np.int32), wedges)
            off, hub, hop, dist = red.arrays()
            idx = H.Index.from_labels(n, K, off.astype(np.uint64), hub.astype(np.uint32),
                                      hop.astype(np.uint8), dist.astype(np.int32))
            same_labels(H.hop_constrained_clean_L(idx), cleaned.arrays())
            if r == 3:
                H.release_scratch()
        return True

    with ThreadPoolExecutor(8) as pool:
        assert all(pool.map(work, range(16)))
