"""Rows in no token order, sorted on the device in front of the search:
against the CPU oracle, bit for bit (ranks of the caller's proposals break
the ties that quantised logps make)."""

import ctypes

import numpy as np
import pytest

from cabi import Batch, check, load
from helpers import assert_same_results

pytestmark = pytest.mark.gpu

VOCAB = 8192


@pytest.fixture(scope="module")
def trie(ft, po):
    toks, offs = ft.synth_keys(30000, VOCAB, 2, 5, 0.6, 3)
    t = ft.Trie()
    t.build_arrays(toks, offs)
    with pytest.MonkeyPatch.context() as m:  # the small rows on the device too
        m.setenv("FT_SORT_MIN", "0")
        t.init_tbs_gpu(4, max_num_topk=4097, max_num_outpos=4, max_num_out_beams=48,
                       max_num_out_tokens=48 * 4, max_num_inter_beams=4096)
    return t, po.OracleTrie.from_keys(toks=toks, offs=offs)


def _rows(rng, B, T, K, high):
    ids = np.stack([[rng.choice(high, K, replace=False) for _ in range(T)] for _ in range(B)])
    lp = (-rng.integers(1, 9, (B, T, K)) * 0.5).astype(np.float32)
    return ids.astype(np.uint32), lp


# the sorts' edges: a wave, a workgroup of 256 and of 1024 pairs, four pairs a
# thread, one more than the device sorts, and powers of two on either side
@pytest.mark.parametrize("K", [2, 3, 63, 64, 65, 128, 255, 256, 257, 777, 1023, 1024, 1025, 2048,
                               2049, 4095, 4096, 4097])
def test_sorted_on_device(ft, trie, K):
    t, o = trie
    rng = np.random.default_rng(K)
    B, T = 3, 4
    print("K", K, flush=True)
    ids, lp = _rows(rng, B, T, K, max(VOCAB, K))
    ids[0].sort(axis=1)  # a request whose rows are in order, among the others
    beams = [[int(b) for b in rng.integers(1, 48, T)] for _ in range(B)]
    for early in (False, True):
        got = ft.bs_tbs_gpu(t, B, beams, ids, lp, -4.0, -40.0, 5.0, early)
        for r in range(B):
            want = o.tbs(beams[r], ids[r], lp[r], -4.0, -40.0, 5.0, early)
            assert_same_results((got[0][r], got[1][r]), want, f"K {K} early {early} request {r}")


def test_order_lost_later(ft, trie):
    """Only a later row is out of order: the packing thread sorts it."""
    t, o = trie
    ids, lp = _rows(np.random.default_rng(1), 1, 4, 100, VOCAB)
    ids[0, :2].sort(axis=1)
    got = ft.bs_tbs_gpu(t, 1, [[20] * 4], ids, lp, -4.0, -40.0, 1.0, False)
    assert_same_results((got[0][0], got[1][0]),
                        o.tbs([20] * 4, ids[0], lp[0], -4.0, -40.0, 1.0, False))


@pytest.mark.parametrize("K", [5, 300, 1500])
def test_bad_rows_are_refused(ft, trie, K):
    t, o = trie
    ids, lp = _rows(np.random.default_rng(K), 3, 4, K, VOCAB)
    ids[:, 0, :2] = ids[:, 0, 1::-1] if ids[0, 0, 0] < ids[0, 0, 1] else ids[:, 0, :2]
    args = (-4.0, -40.0, 1.0, False)
    beams = [[20] * 4] * 3
    twice = ids.copy()
    twice[1, 3, K - 1] = twice[1, 3, 0]
    with pytest.raises(RuntimeError, match=f"request 1: duplicate token id {twice[1, 3, 0]} "
                                           "in topk row 3"):
        ft.bs_tbs_gpu(t, 3, beams, twice, lp, *args)
    nan = lp.copy()
    nan[2, 1, 0] = np.nan
    with pytest.raises(RuntimeError, match="request 2: topk_logp holds NaN"):
        ft.bs_tbs_gpu(t, 3, beams, ids, nan, *args)
    with pytest.raises(RuntimeError, match="request 1: duplicate"):  # the first bad request
        ft.bs_tbs_gpu(t, 3, beams, twice, nan, *args)
    got = ft.bs_tbs_gpu(t, 3, beams, ids, lp, *args)  # and the context goes on
    for r in range(3):
        assert_same_results((got[0][r], got[1][r]), o.tbs([20] * 4, ids[r], lp[r], *args))


# Which batches are sorted on the device: those with enough proposals out of
# order for their ordered rest.  Every other is launched before its rows are
# packed, so that a pause of the packing thread is part of the kernel's time.
@pytest.mark.parametrize("B,K,n_out,device",
                         [(16, 300, 0, False), (16, 300, 1, False), (16, 300, 2, False),
                          (16, 300, 3, True), (16, 300, 16, True),
                          (1, 511, 1, False), (1, 512, 1, True),
                          (3, 4096, 1, True), (3, 4097, 3, False)])
def test_which_batches(ft, po, monkeypatch, B, K, n_out, device):
    monkeypatch.setenv("FT_PACK_DELAY_US", "20000")
    toks, offs = ft.synth_keys(30000, VOCAB, 2, 5, 0.6, 3)
    t = ft.Trie()
    t.build_arrays(toks, offs)
    image = np.array(t.image(), dtype=np.uint8)
    o = po.OracleTrie.from_keys(toks=toks, offs=offs)
    rng = np.random.default_rng(K + n_out)
    ids, lp = _rows(rng, B, 4, K, VOCAB)
    at = set(range(0, B, max(1, B // max(1, n_out)))[:n_out])
    for r in range(B):
        if r not in at:
            ids[r].sort(axis=1)
        else:
            ids[r, 0, :2] = np.sort(ids[r, 0, :2])[::-1]
    beams = np.full((B, 4), 20, dtype=np.uint32)
    lib = load()
    ctx = ctypes.c_void_p()
    check(lib, lib.ft_create(image.ctypes.data, image.nbytes, 0, ctypes.byref(ctx)))
    try:
        check(lib, lib.ft_reserve(ctx, B, K, 4, 20, 80, 4096))
        batch = Batch(beams, ids, lp, -4.0, -40.0, 5.0, False, 20)
        timing = (ctypes.c_double * 8)()
        print("B", B, "K", K, "out of order", n_out, flush=True)
        check(lib, lib.ft_search(ctx, batch.reqs, B, batch.res, ctypes.byref(timing)))
        assert (timing[0] < 15.0) == device, timing[0]
        for r in range(B):
            assert_same_results(batch.results(r), o.tbs(list(beams[r]), ids[r], lp[r], -4.0, -40.0,
                                                        5.0, False), f"request {r}")
    finally:
        lib.ft_destroy(ctx)
