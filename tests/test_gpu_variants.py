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
