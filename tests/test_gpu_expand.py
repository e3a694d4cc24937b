"""The queued expansion (a wave filters several chunks of work items and
queues the survivors) at its edges, against the CPU oracle, bit for bit."""

import numpy as np
import pytest

from helpers import assert_same_results

pytestmark = pytest.mark.gpu

VOCAB = 700


def _search(ft, po, K, beam, env, monkeypatch, batch=2, lmin=2):
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    toks, offs = ft.synth_keys(60000, VOCAB, lmin, 4, 0.8, 7)
    t = ft.Trie()
    t.build_arrays(toks, offs)
    T = 4
    t.init_tbs_gpu(batch, max_num_topk=2049, max_num_outpos=T, max_num_out_beams=beam,
                   max_num_out_tokens=beam * T, max_num_inter_beams=beam * T)
    o = po.OracleTrie.from_keys(toks=toks, offs=offs)
    rng = np.random.default_rng(K)
    ids = np.array([[np.sort(rng.choice(max(VOCAB, K), K, replace=False)) for _ in range(T)]
                    for _ in range(batch)]).astype(np.uint32)
    lp = (-rng.integers(1, 33, (batch, T, K)) * 0.125).astype(np.float32)  # ties; -4 is dropped
    beams = [[beam, beam, beam, beam - 1]] * batch
    for early in (False, True):
        print("K", K, env, "early", early, flush=True)
        got = ft.bs_tbs_gpu(t, batch, beams, ids, lp, -4.0, -11.0, 1.0, early)
        for r in range(batch):
            want = o.tbs(beams[r], ids[r], lp[r], -4.0, -11.0, 1.0, early)
            assert_same_results((got[0][r], got[1][r]), want, f"K {K} {env} request {r}")


# A wave has more than four chunks: one workgroup a request (solo steps) or two
# (shared); children scanned, looked up with and without fingerprint words, or
# both kinds in one step (K = 64: nodes of up to 128 children are scanned);
# rows around a wave, and the longest that is hashed and one more.
@pytest.mark.parametrize("wgs", ["1", "2"])
@pytest.mark.parametrize("K,scan_mult,fp_max",
                         [(63, "2", "16"), (64, "2", "16"), (65, "2", "0"), (500, "0", "16"),
                          (500, "0", "0"), (500, "2", "16"), (2048, "0", "16"),
                          (2048, "2", "16"), (2049, "0", "16")])
def test_queued_items(ft, po, monkeypatch, K, scan_mult, fp_max, wgs):
    _search(ft, po, K, 300, dict(FT_WGS=wgs, FT_SHARE_MIN="0", FT_WIDE_MIN="2",
                                 FT_SCAN_MULT=scan_mult, FT_FP_MAX_LOG2=fp_max), monkeypatch)


# The longest beams and rows of the lean instantiation, one more of either, and
# the general instantiation at a size of the lean one.
@pytest.mark.parametrize("beam,K,lean", [(1024, 500, "1"), (1025, 500, "1"), (300, 1024, "1"),
                                         (300, 1025, "1"), (300, 500, "0")])
def test_lean_limits(ft, po, monkeypatch, beam, K, lean):
    _search(ft, po, K, beam, dict(FT_WGS="2", FT_WIDE_MIN="2", FT_SCAN_MULT="0", FT_LEAN=lean),
            monkeypatch)


# A shared step's cut: one that lets far too few pushes through, about enough,
# and most (the first two end in a second round when under `beam` pushes reach
# it); tables all open (keys of 3 tokens or more at step 1) and closing keys.
@pytest.mark.parametrize("lmin", [2, 3])
@pytest.mark.parametrize("fp_max", ["0", "16"])
@pytest.mark.parametrize("pairs", ["1", "12", "200"])
def test_cut_steps(ft, po, monkeypatch, pairs, fp_max, lmin):
    _search(ft, po, 500, 300, dict(FT_WGS="3", FT_WIDE_MIN="2", FT_SCAN_MULT="0",
                                   FT_FP_MAX_LOG2=fp_max, FT_CUT_PAIRS=pairs), monkeypatch,
            lmin=lmin)


def test_cut_with_taken_over_slices(ft, po, monkeypatch):
    _search(ft, po, 500, 300, dict(FT_WGS="3", FT_WIDE_MIN="2", FT_SCAN_MULT="0",
                                   FT_CUT_PAIRS="1", FT_TEST_NO_CLAIMS="1"), monkeypatch, lmin=3)
