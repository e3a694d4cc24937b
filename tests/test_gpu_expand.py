"""The lean instantiation's expansion -- steps whose items are queued (a wave
filters its chunks and queues the survivors), and their cuts -- at its edges,
against the CPU oracle, bit for bit.  FT_TEST_STEP_KINDS has the last word of a
step's counters say how the step was expanded."""

import numpy as np
import pytest

from helpers import assert_same_results

pytestmark = pytest.mark.gpu

VOCAB = 700
T = 4
QUEUED, CUT, TWICE = 1, 2, 4


def _synth(ft, lmin=2):
    return ft.synth_keys(60000, VOCAB, lmin, T, 0.8, 7)


def _arrays(keys):
    return (np.concatenate(keys).astype(np.uint32),
            np.concatenate([[0], np.cumsum([len(k) for k in keys])]).astype(np.uint64))


def _part_open(ft, share):
    """Keys of which those below a `share` of the first tokens have at least
    three tokens (no child of such a node closes a key at step 1)."""
    rng = np.random.default_rng(11)
    keys = [rng.integers(0, VOCAB, n) for n in rng.integers(2, T + 1, 60000)]
    for k in keys:
        if k[0] < share * VOCAB and len(k) < 3:
            k[0] = VOCAB - 1
    return _arrays(keys)


def _wide_and_narrow(ft):
    """Half of 600 first tokens have 300 children, the others 100."""
    rng = np.random.default_rng(12)
    return _arrays([np.array([a, b, rng.integers(0, 600)]) for a in range(600)
                    for b in rng.choice(600, 300 if a < 300 else 100, replace=False)])


class _Case:
    """One trie, one context, one batch: rows with ties, some below the
    threshold."""

    def __init__(self, ft, po, monkeypatch, K, beam, env, keys=None, batch=2, shuffled=False,
                 vocab=VOCAB):
        for k, v in dict(env, FT_TEST_STEP_KINDS="1").items():
            monkeypatch.setenv(k, v)
        toks, offs = keys if keys is not None else _synth(ft)
        self.ft, self.batch, self.what = ft, batch, f"K {K} beam {beam} {env}"
        self.t = ft.Trie()
        self.t.build_arrays(toks, offs)
        self.t.init_tbs_gpu(batch, max_num_topk=2049, max_num_outpos=T, max_num_out_beams=beam,
                            max_num_out_tokens=beam * T, max_num_inter_beams=beam * T)
        self.o = po.OracleTrie.from_keys(toks=toks, offs=offs)
        rng = np.random.default_rng(K)
        rows = [[rng.choice(max(vocab, K), K, replace=False) for _ in range(T)]
                for _ in range(batch)]
        self.ids = np.array(rows).astype(np.uint32)
        if not shuffled:
            self.ids.sort(axis=2)
        self.lp = (-rng.integers(1, 33, (batch, T, K)) * 0.125).astype(np.float32)
        self.beams = np.array([[beam] * (T - 1) + [beam - 1]] * batch, dtype=np.uint32)

    def check(self):
        """Streamed (both exit rules) and staged searches against the oracle;
        returns the staged steps' counters [batch][T][10]."""
        ft, B = self.ft, self.batch
        for early in (False, True):
            print(self.what, "early", early, flush=True)
            want = [self.o.tbs(self.beams[r].tolist(), self.ids[r], self.lp[r], -4.0, -11.0, 1.0,
                               early) for r in range(B)]
            got = ft.bs_tbs_gpu(self.t, B, self.beams.tolist(), self.ids, self.lp, -4.0, -11.0,
                                1.0, early)
            for r in range(B):
                assert_same_results((got[0][r], got[1][r]), want[r], f"{self.what} request {r}")
        steps = self.steps(early)
        for r in range(B):
            assert_same_results(self.staged[r], want[r], f"{self.what} staged request {r}")
        return steps

    def steps(self, early=False):
        ft = self.ft
        ft.stage(self.t, self.beams, self.ids, self.lp, -4.0, -11.0, 1.0, early)
        ft.launch(self.t, 0, self.batch)
        counts, norms, lengths, tokens, timing = ft.fetch(self.t)
        self.staged = [([tokens[r, i, :lengths[r, i]].tolist() for i in range(counts[r])],
                        norms[r, :counts[r]].copy()) for r in range(self.batch)]
        return timing["step_stats"].copy()


def _kinds(steps, t):
    return [int(x) for x in steps[:, t, 9]]


# Queued steps of one workgroup a request (solo) and two (shared); children
# scanned, looked up with and without fingerprint words, or both kinds of
# parents; rows around a wave, and the longest of the instantiation.
@pytest.mark.parametrize("wgs", ["1", "2"])
@pytest.mark.parametrize("K,scan_mult,fp_max", [(500, "0", "16"), (500, "0", "0"),
                                                (500, "2", "16"), (1023, "2", "16"),
                                                (1024, "0", "16"), (1024, "0", "0")])
def test_queued_items(ft, po, monkeypatch, K, scan_mult, fp_max, wgs):
    steps = _Case(ft, po, monkeypatch, K, 300,
                  dict(FT_WGS=wgs, FT_SHARE_MIN="0", FT_WIDE_MIN="2", FT_SCAN_MULT=scan_mult,
                       FT_FP_MAX_LOG2=fp_max, FT_CUT_PAIRS="0")).check()
    assert _kinds(steps, 1) == [QUEUED] * 2


@pytest.mark.parametrize("K,scan_mult,fp_max", [(63, "2", "16"), (64, "2", "16"), (64, "0", "0"),
                                                (65, "0", "16"), (65, "2", "0")])
def test_queued_short_rows(ft, po, monkeypatch, K, scan_mult, fp_max):
    rng = np.random.default_rng(13)
    keys = _arrays([rng.integers(0, 150, n) for n in rng.integers(3, 5, 400000)])
    steps = _Case(ft, po, monkeypatch, K, 1000,
                  dict(FT_WGS="1", FT_WIDE_MIN="2", FT_SCAN_MULT=scan_mult,
                       FT_FP_MAX_LOG2=fp_max), keys=keys, vocab=150).check()
    assert _kinds(steps, 2) == [QUEUED] * 2


# Rows longer than the lean instantiation's, on the general one: the longest
# that is hashed and one more.
@pytest.mark.parametrize("wgs", ["1", "2"])
@pytest.mark.parametrize("K,scan_mult", [(2048, "0"), (2048, "2"), (2049, "0")])
def test_long_rows(ft, po, monkeypatch, K, scan_mult, wgs):
    _Case(ft, po, monkeypatch, K, 300, dict(FT_WGS=wgs, FT_SHARE_MIN="0", FT_WIDE_MIN="2",
                                            FT_SCAN_MULT=scan_mult)).check()


# The longest beams and rows of the lean instantiation, one more of either, and
# the general instantiation at a size of the lean one (whose step_stats keep
# the wait, nothing for a solo step).
@pytest.mark.parametrize("beam,K,lean", [(1024, 500, "1"), (1025, 500, "1"), (300, 1024, "1"),
                                         (300, 1025, "1"), (300, 500, "0")])
def test_lean_limits(ft, po, monkeypatch, beam, K, lean):
    steps = _Case(ft, po, monkeypatch, K, beam,
                  dict(FT_WGS="1", FT_WIDE_MIN="2", FT_SCAN_MULT="0", FT_LEAN=lean)).check()
    expect = QUEUED if lean == "1" and beam <= 1024 and K <= 1024 else 0
    assert _kinds(steps, 1) == [expect] * 2


# A shared step's cut: far too few pushes reach it (a second round), or enough;
# every parent's table open (keys of three tokens or more), or half of them
# (the others feed `selected` too); tables with and without fingerprint words.
@pytest.mark.parametrize("share", [1.0, 0.5])
@pytest.mark.parametrize("fp_max", ["0", "16"])
@pytest.mark.parametrize("pairs,kind", [("1", QUEUED | CUT | TWICE), ("50", QUEUED | CUT),
                                        ("200", QUEUED | CUT)])
def test_cut_steps(ft, po, monkeypatch, pairs, kind, fp_max, share):
    if share < 1.0 and pairs == "200":
        pairs = "150"  # (as many proposals as can be skipped)
    steps = _Case(ft, po, monkeypatch, 500, 300,
                  dict(FT_WGS="3", FT_WIDE_MIN="2", FT_SCAN_MULT="0", FT_FP_MAX_LOG2=fp_max,
                       FT_CUT_PAIRS=pairs), keys=_part_open(ft, share)).check()
    assert _kinds(steps, 1) == [kind] * 2
    if share < 1.0:
        assert steps[:, 1, 3].min() > 0  # pushes into `selected` beside the cut


# Few parents can skip lookups: the cut is taken when the sampled pairs above
# it are found to have children, and left when they promise too few.
@pytest.mark.parametrize("pairs,kind", [("1", QUEUED), ("50", QUEUED | CUT)])
def test_cut_looked_up(ft, po, monkeypatch, pairs, kind):
    steps = _Case(ft, po, monkeypatch, 500, 300,
                  dict(FT_WGS="3", FT_WIDE_MIN="2", FT_SCAN_MULT="0", FT_CUT_PAIRS=pairs),
                  keys=_part_open(ft, 0.25)).check()
    assert _kinds(steps, 1) == [kind] * 2


def test_cut_with_taken_over_slices(ft, po, monkeypatch):
    steps = _Case(ft, po, monkeypatch, 500, 300,
                  dict(FT_WGS="3", FT_WIDE_MIN="2", FT_SCAN_MULT="0", FT_CUT_PAIRS="1",
                       FT_TEST_NO_CLAIMS="1"), keys=_synth(ft, 3)).check()
    assert _kinds(steps, 1) == [QUEUED | CUT | TWICE] * 2


# Rows sorted on the device: the caller's indices break the ties of steps with
# a cut and of second rounds.
@pytest.mark.parametrize("wgs", ["2", "3"])
@pytest.mark.parametrize("pairs,kind", [("1", QUEUED | CUT | TWICE), ("50", QUEUED | CUT)])
def test_cut_shuffled_rows(ft, po, monkeypatch, pairs, kind, wgs):
    steps = _Case(ft, po, monkeypatch, 500, 300,
                  dict(FT_WGS=wgs, FT_WIDE_MIN="2", FT_SCAN_MULT="0", FT_CUT_PAIRS=pairs,
                       FT_SORT_MIN="0"), keys=_synth(ft, 3), shuffled=True).check()
    assert _kinds(steps, 1) == [kind] * 2


# The counters of a step with a cut: the same in every run, children scanned
# counted once, pushes below the cut left out, or made in the second round.
@pytest.mark.parametrize("pairs", ["1", "10"])
def test_cut_counters(ft, po, monkeypatch, pairs):
    def steps(pairs):
        c = _Case(ft, po, monkeypatch, 200, 200,
                  dict(FT_WGS="2", FT_WIDE_MIN="2", FT_SCAN_MULT="1", FT_CUT_PAIRS=pairs),
                  keys=_wide_and_narrow(ft), batch=4, vocab=600)
        return [c.check()] + [c.steps(True) for _ in range(6)]

    runs, (whole, *_) = steps(pairs), steps("0")
    counters = [0, 1, 2, 3, 6, 7]
    for s in runs[1:]:
        assert np.array_equal(s[:, :, counters], runs[0][:, :, counters])
    assert _kinds(whole, 1) == [QUEUED] * 4 and whole[:, 1, 6].min() > 0
    assert np.array_equal(runs[0][:, 1, 6], whole[:, 1, 6])
    kinds = _kinds(runs[0], 1)
    assert all(k & CUT for k in kinds) and any(k & TWICE for k in kinds) == (pairs == "1")
    for k, cut, all_ in zip(kinds, runs[0][:, 1, 2], whole[:, 1, 2]):
        assert cut == all_ if k & TWICE else 200 <= cut < all_
