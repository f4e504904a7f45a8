"""Builds, cleans and host calls at the limits of their buffers, lists and
counters.  Labels, answers and counts are integers: every comparison is exact."""
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
