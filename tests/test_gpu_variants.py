"""Kernel variants that a size, a type or an option selects, at the edges of
their ranges, against the oracle.  Integer work: every comparison is exact."""
import numpy as np
import pytest

import gpu4hophl_code_amd as H
import oracle_lib as O
from test_gpu_parity import csr_of, same_labels

pytestmark = pytest.mark.gpu


def ragged(n, seed, wmax, ef=8):
    """The n top-ranked vertices of an R-MAT graph, renamed by degree."""
    g = H.Graph.rmat(max(1, (n - 1).bit_length()), ef, seed, 1, wmax)
    off, col, w = g.csr()
    row = np.repeat(np.arange(len(off) - 1, dtype=np.uint32), np.diff(off.astype(np.int64)))
    keep = (row < col) & (col < n)
    g = H.Graph.from_edges(n, row[keep], col[keep], w[keep])
    g.reorder_by_degree()
    return g


@pytest.mark.parametrize("landmarks", ["0", "8", "24", "64"])
@pytest.mark.parametrize("rows", ["0", "2"])
def test_landmark_test_keeps_the_labels(monkeypatch, landmarks, rows):
    """Candidates are tested against the first hubs' rows before the prune
    searches (rows of 2 to 64 chunks by K and the landmark count, by lists
    and by rows): the labels are the oracle's, for whole builds, batches that
    end inside and past the landmarks, groups (landmarks are the group's own
    hubs) and 8-byte labels."""
    monkeypatch.setenv("HSDL_LANDMARKS", landmarks)
    monkeypatch.setenv("HSDL_PRUNE_ROWS", rows)
    for n, K, wmax in ((1500, 4, 100), (1031, 2, 3), (700, 9, 2), (2049, 5, 13000), (90, 3, 9)):
        g = ragged(n, n, wmax)
        c = csr_of(g)
        want = O.kround(c, K).arrays()
        for batch in (0, 7, 65):
            print(f"[landmarks] n={n} K={K} hubs={landmarks} rows={rows} batch={batch}", flush=True)
            same_labels(H.hop_constrained_two_hop_labels_generation(g, K, hub_batch=batch), want)
        hubs = np.arange(1, n, 3, dtype=np.uint32)
        gid = np.ones(n, np.uint32)
        gid[hubs] = 0
        got = H.hop_constrained_two_hop_labels_generation(g, K, hubs=hubs, hub_batch=40)
        ref = O.kround_gid(c, K, gid).arrays()
        keep = np.isin(ref[1], hubs)
        for x, y in zip(got.labels()[1:], ref[1:]):
            assert np.array_equal(x, np.asarray(y)[keep])
    monkeypatch.setenv("HSDL_STREAM32", "0")
    g = ragged(1500, 4, 100)
    same_labels(H.hop_constrained_two_hop_labels_generation(g, 4), O.kround(csr_of(g), 4).arrays())


@pytest.mark.parametrize("rows,density", [("0", "32"), ("1", "32"), ("2", "32"), ("2", "1")])
def test_prune_tiles_by_hub_id(monkeypatch, rows, density):
    """Tiles addressed by hub id (values while the hub range is small, then
    row indexes, then hashes: 21,001 vertices pass through all three in a
    build, at a different hub in each round) and row items whose candidates
    fill the list several times (dense rounds) or leave steps empty: the
    oracle's labels, with K at both ends of a 3-bit hop field."""
    monkeypatch.setenv("HSDL_PRUNE_ROWS", rows)
    monkeypatch.setenv("HSDL_ROW_DENSITY", density)
    for n, K, wmax, batch, lm in ((21001, 3, 50, 0, "16"), (21001, 3, 50, 1000, "0"),
                                  (1025, 7, 4, 0, "0"), (4100, 4, 100, 3, "16"),
                                  (9000, 3, 20000, 4096, "0")):
        monkeypatch.setenv("HSDL_LANDMARKS", lm)
        print(f"[tiles] n={n} K={K} batch={batch} rows={rows} landmarks={lm}", flush=True)
        g = ragged(n, n + K, wmax)
        same_labels(H.hop_constrained_two_hop_labels_generation(g, K, hub_batch=batch),
                    O.kround(csr_of(g), K).arrays())


@pytest.mark.parametrize("heavy,piece", [("1", "64"), ("1", "65536"), ("40", "300"), ("65536", "1")])
def test_expansion_shapes(monkeypatch, heavy, piece):
    """Frontier groups as pieces of a workgroup (every group, in pieces of an
    edge and of all edges; groups of one label to a few hundred, so 1 to 64
    lanes share an edge) and by waves (chunks of one group and more), with the
    hub's landmark chunks held in registers (few hops) and read per pair (many,
    or several chunks per hop): the oracle's labels."""
    monkeypatch.setenv("HSDL_HEAVY_PAIRS", heavy)
    monkeypatch.setenv("HSDL_PIECE_PAIRS", piece)
    for n, K, wmax, lm in ((2500, 4, 100, "8"), (700, 7, 3, "8"), (1500, 4, 20, "24"),
                           (300, 3, 30000, "8"), (65, 2, 5, "8")):
        monkeypatch.setenv("HSDL_LANDMARKS", lm)
        print(f"[expansion] n={n} K={K} landmarks={lm} heavy={heavy} piece={piece}", flush=True)
        g = ragged(n, n + K, wmax, 16)
        for batch in (0, 33):
            same_labels(H.hop_constrained_two_hop_labels_generation(g, K, hub_batch=batch),
                        O.kround(csr_of(g), K).arrays())
    g = H.Graph.grid(37, 41, 5, 1, 300)
    same_labels(H.hop_constrained_two_hop_labels_generation(g, 6), O.kround(csr_of(g), 6).arrays())


@pytest.mark.parametrize("items,cands", [("1", "64"), ("1", "3"), ("300", "64"), ("0", "32")])
@pytest.mark.parametrize("stream32", ["1", "0"])
def test_prune_wave_items(monkeypatch, items, cands, stream32):
    """Hubs with few candidates and a short list take a wave each (from the
    first such hub, from the 300th, never), beside hubs that do not; batches
    whose workgroups accept more labels than their staging holds, 16- and
    32-bit tile values, tiles of few slots, lists read whole, and a group's
    hubs: the oracle's labels."""
    monkeypatch.setenv("HSDL_WAVE_ITEMS", items)
    monkeypatch.setenv("HSDL_WAVE_CANDS", cands)
    monkeypatch.setenv("HSDL_STREAM32", stream32)
    monkeypatch.setenv("HSDL_PRUNE_ROWS", "0")
    monkeypatch.setenv("HSDL_LANDMARKS", "0")

    def check(g, K, **kw):
        c = csr_of(g)
        print(f"[wave items] n={c.n} K={K} {kw} items={items} cands={cands} s32={stream32}",
              flush=True)
        same_labels(H.hop_constrained_two_hop_labels_generation(g, K, **kw),
                    O.kround(c, K).arrays())

    for n, K, wmax, ef in ((2500, 4, 100, 8), (2500, 3, 30000, 4), (700, 7, 3, 4), (300, 15, 20, 2)):
        g = ragged(n, n + K, wmax, ef)
        check(g, K)
        check(g, K, hub_batch=n)
        check(g, K, hub_batch=n, lds_tile_slots=64)
    g = H.Graph.grid(61, 67, 3, 1, 300)
    check(g, 8, hub_batch=2000)
    check(H.Graph.grid(31, 67, 3, 1, 300), 15, hub_batch=2000)
    monkeypatch.setenv("HSDL_HOP_ZONES", "0")
    check(g, 5, hub_batch=2000)
    monkeypatch.delenv("HSDL_HOP_ZONES")
    n, K = 2400, 4
    g = ragged(n, 5, 50)
    hubs = np.arange(1, n, 3, dtype=np.uint32)
    gid = np.ones(n, np.uint32)
    gid[hubs] = 0
    got = H.hop_constrained_two_hop_labels_generation(g, K, hubs=hubs, hub_batch=800)
    ref = O.kround_gid(csr_of(g), K, gid).arrays()
    keep = np.isin(ref[1], hubs)
    for x, y in zip(got.labels()[1:], ref[1:]):
        assert np.array_equal(x, np.asarray(y)[keep])


@pytest.mark.parametrize("team", ["0", "6000"])
@pytest.mark.parametrize("q32,slots", [("1", "1024"), ("1", "64"), ("0", "1024")])
def test_query_forms(monkeypatch, q32, slots, team):
    """Queries from the hop-ordered 32-bit copy (parts that fit the table, and
    with 64 slots parts hashed in many pieces) and from the 8-byte labels (lists
    of one piece of 512 labels and of several), a wave or a workgroup of
    four (6,000 queries) or eight waves (1,000 and one) per query: every k from 0 past K, on a
    graph of long lists, short lists at K = 15, a group's index (vertices
    without their self label) and an imported set with hubs ranked below their
    vertex: the oracle's answers."""
    monkeypatch.setenv("HSDL_QUERY32", q32)
    monkeypatch.setenv("HSDL_QUERY_SLOTS", slots)
    monkeypatch.setenv("HSDL_QUERY_TEAM", team)
    rng = np.random.default_rng(17)

    def check(name, idx, want, n, K):
        print(f"[query] {name} q32={q32} slots={slots} team={team}", flush=True)
        s, t = rng.integers(0, n, (2, 6000)).astype(np.uint32)
        t[:50] = s[:50]
        k = rng.integers(-1, K + 3, 6000).astype(np.int8)
        ans = O.query(want, s, t, k)
        for m in (6000, 1000, 1):
            assert np.array_equal(idx.query(s[:m], t[:m], k[:m]), ans[:m])

    def imported(off, hub, hop, dist, K):
        o = O.labels_from_arrays(len(off) - 1, off, hub, hop, dist)
        return H.Index.from_labels(len(off) - 1, K, off, hub, hop, dist), o

    for n, K, wmax, ef in ((6000, 4, 1000, 16), (400, 15, 2, 4), (33, 3, 5, 2)):
        g = ragged(n, n, wmax, ef)
        want = O.kround(csr_of(g), K)
        check(f"n={n}", H.hop_constrained_two_hop_labels_generation(g, K), want, n, K)
    hubs = np.arange(0, 6000, 2, dtype=np.uint32)
    g = ragged(6000, 6000, 1000, 16)
    idx = H.hop_constrained_two_hop_labels_generation(g, 4, hubs=hubs)
    check("group", idx, O.labels_from_arrays(6000, *idx.labels()), 6000, 4)
    # vertex v also holds, for some of its labels (u, h, d), the mirrored label at u
    off, hub, hop, dist = idx.labels()
    v = np.repeat(np.arange(6000), np.diff(off.astype(np.int64)))
    pick = (rng.random(len(v)) < 0.2) & (hop > 0)
    rows = np.concatenate([np.stack([v, hub, hop, dist], 1),
                           np.stack([hub[pick], v[pick], hop[pick], dist[pick]], 1)]).astype(np.int64)
    rows = rows[np.lexsort((rows[:, 2], rows[:, 1], rows[:, 0]))]
    off = np.zeros(6001, np.uint64)
    off[1:] = np.cumsum(np.bincount(rows[:, 0], minlength=6000))
    idx, want = imported(off, rows[:, 1].astype(np.uint32), rows[:, 2].astype(np.uint8),
                         rows[:, 3].astype(np.int32), 4)
    check("hubs below", idx, want, 6000, 4)


def test_paths_over_pieces():
    """Paths where a list spans several staged pieces of 512 labels, runs of a
    hub cut by a piece's end, ties (weights 1..2), and lists far shorter than
    the other side's: the oracle's edges."""
    rng = np.random.default_rng(3)
    for n, K, wmax, ef in ((6000, 4, 2, 16), (4000, 5, 1000, 16), (300, 9, 2, 4)):
        g = ragged(n, n, wmax, ef)
        print(f"[paths] n={n} K={K}", flush=True)
        idx = H.hop_constrained_two_hop_labels_generation(g, K, parents=True)
        want = O.kround(csr_of(g), K)
        s, t = rng.integers(0, n, (2, 4000)).astype(np.uint32)
        s[:1000] = np.arange(1000) % 40
        k = rng.integers(0, K + 2, 4000).astype(np.int8)
        edges, counts = idx.paths(s, t, k, cap=K + 1)
        wedges, wcounts = O.paths(want, s, t, k.astype(np.int32), K + 1)
        assert np.array_equal(counts.astype(np.int32), wcounts)
        assert np.array_equal(edges.astype(np.int32), wedges)


def test_host_calls_in_parts():
    """Host-array queries and paths that end at, before and past a staging
    slot's part and span several, paths whose cap exceeds a slot, and calls from
    six threads at once on one index (more than the pool keeps), with the pool
    released in between: the oracle's answers."""
    from concurrent.futures import ThreadPoolExecutor
    g = ragged(500, 3, 9)
    want = O.kround(csr_of(g), 4)
    idx = H.hop_constrained_two_hop_labels_generation(g, 4, parents=True)
    s, t = (x.ravel().astype(np.uint32) for x in np.meshgrid(np.arange(500), np.arange(500)))
    k = (np.arange(250000) % 6).astype(np.int8)
    ans = O.query(want, s, t, k)
    edges, counts = O.paths(want, s, t, k.astype(np.int32), 5)

    def query(n, at):
        i = (np.arange(n) + at) % 250000
        return np.array_equal(idx.query(s[i], t[i], k[i]), ans[i])

    def paths(n, at):
        i = (np.arange(n) + at) % 250000
        e, c = idx.paths(s[i], t[i], k[i], cap=5)
        return np.array_equal(c, counts[i]) and np.array_equal(e, edges[i])

    part = 1 << 18
    for n in (1, part - 1, part, part + 1, 3 * part + 5):
        print(f"[parts] queries {n}", flush=True)
        assert query(n, n)
    part = ((4 << 20) - 64) // 53 & ~3
    for n in (part, part + 1, 3 * part - 1):
        print(f"[parts] paths {n}", flush=True)
        assert paths(n, n)
    e, c = idx.paths(s[:3], t[:3], k[:3], cap=600000)
    assert np.array_equal(c, counts[:3]) and np.array_equal(e[:, :5], edges[:3]) and not e[:, 5:].any()
    for _ in range(2):
        with ThreadPoolExecutor(6) as pool:
            jobs = [pool.submit(query, 300001, 7 * i) for i in range(6)]
            jobs += [pool.submit(paths, 90001, 11 * i) for i in range(6)]
            assert all(j.result() for j in jobs)
        H.release_scratch()


@pytest.mark.parametrize("pairs,stream32,piece", [("0", "1", None), ("0", "0", None), ("1", "1", None),
                                                  ("2", "1", None), ("2", "0", None),
                                                  ("2", "1", "3000"), ("2", "0", "1")])
def test_clean_forms(monkeypatch, pairs, stream32, piece):
    """The clean's first pass over tiles, over label pairs and as the mean list
    length chooses, from 32-bit and 8-byte lists, whole and in slices down to
    one list: redundant sets of short and of long lists (past 2,048 labels, a
    workgroup each), hubs ranked below their vertex, empty lists, K = 1 and
    15, and sets that lose nothing: the oracle's clean."""
    monkeypatch.setenv("HSDL_CLEAN_PAIRS", pairs)
    monkeypatch.setenv("HSDL_STREAM32", stream32)
    if piece:
        monkeypatch.setenv("HSDL_CLEAN_SLICE", piece)
    rng = np.random.default_rng(29)

    def check(name, K, off, hub, hop, dist):
        print(f"[clean] {name} pairs={pairs} stream32={stream32} slice={piece}", flush=True)
        off = np.asarray(off, np.uint64)
        n = len(off) - 1
        want = O.clean(O.labels_from_arrays(n, off.astype(np.int64), hub, hop, dist))
        idx = H.Index.from_labels(n, K, off, hub, hop, dist)
        idx.clean()
        same_labels(idx, want.arrays())
        return want.total()

    for n, K, wmax, group in ((900, 4, 50, 32), (500, 15, 3, 64), (300, 2, 30000, 9), (65, 1, 5, 7),
                              (3500, 3, 1000, 3000)):
        off, hub, hop, dist = O.kround_grouped(csr_of(ragged(n, n + K, wmax)), K, group).arrays()
        check(f"groups n={n} K={K}", K, off, hub, hop, dist)
    # some labels (u, h, d) of v also at u as (v, h, d); every third list empty
    off, hub, hop, dist = O.kround(csr_of(ragged(1200, 8, 40)), 4).arrays()
    v = np.repeat(np.arange(1200), np.diff(np.asarray(off).astype(np.int64)))
    rows = np.stack([v, hub, hop, dist], 1).astype(np.int64)
    pick = (rng.random(len(v)) < 0.3) & (rows[:, 2] > 0)
    rows = np.concatenate([rows, rows[pick][:, [1, 0, 2, 3]]])
    rows = rows[rows[:, 0] % 3 > 0]
    rows = rows[np.lexsort((rows[:, 2], rows[:, 1], rows[:, 0]))]
    off = np.concatenate([[0], np.cumsum(np.bincount(rows[:, 0], minlength=1200))])
    check("hubs below", 4, off, rows[:, 1].astype(np.uint32), rows[:, 2].astype(np.uint8),
          rows[:, 3].astype(np.int32))
    # lists of 2,047, 2,048, 2,049 and 4,500 labels over hubs that share ten
    # first hubs; the last ones' hop-2 labels fall through them now and then
    W, U = 10, 4600
    lists = [[(x, 0, 0)] for x in range(W)]
    lists += [[(w, 1, int(rng.integers(1, 50))) for w in range(W)] + [(u, 0, 0)]
              for u in range(W, W + U)]
    for i, (size, top) in enumerate(((2047, 3), (2048, 120), (2049, 3), (4500, 3), (4500, 120))):
        a = [(w, 1, int(rng.integers(top, 50 + top))) for w in range(W)]
        a += [(u, 2, int(rng.integers(1, top))) for u in range(W, size - 1)]
        lists.append(a + [(W + U + i, 0, 0)])
    off = np.concatenate([[0], np.cumsum([len(x) for x in lists])])
    hub, hop, dist = np.array([e for x in lists for e in x]).T
    check("long", 3, off, hub.astype(np.uint32), hop.astype(np.uint8), dist.astype(np.int32))


@pytest.mark.parametrize("n,K,top", [(40, 2, 3), (130, 3, 4), (130, 3, 12), (90, 15, 6)])
def test_clean_decides_chains_in_rounds(n, K, top):
    """Lists over all hubs with random hops and small distances: most labels
    fall, many through labels that fall themselves, so a round of the clean's
    second pass leaves labels open for the next: the oracle's clean, and a clean
    of the result changes nothing that the oracle's does not."""
    rng = np.random.default_rng(n + K + top)
    offs, rows = [0], []
    for v in range(n):
        for u in range(v):
            for h in sorted(set(rng.integers(1, K + 1, 2).tolist())):
                rows.append((u, h, int(rng.integers(1, top)) + (K - h) * (top > 8)))
        rows.append((v, 0, 0))
        offs.append(len(rows))
    hub, hop, dist = np.array(rows).T
    off = np.array(offs, np.uint64)
    arrays = (off, hub.astype(np.uint32), hop.astype(np.uint8), dist.astype(np.int32))
    for turn in range(2):
        print(f"[rounds] n={n} K={K} top={top} turn={turn} labels={len(arrays[1])}", flush=True)
        want = O.clean(O.labels_from_arrays(n, np.asarray(arrays[0]).astype(np.int64), *arrays[1:]))
        idx = H.Index.from_labels(n, K, *arrays)
        idx.clean()
        same_labels(idx, want.arrays())
        arrays = idx.labels()
