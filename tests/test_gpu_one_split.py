"""The scan that merges by itself (one split covers the sequence, no merge launch): the sizes where it can go wrong --
single rows, page and chunk edges, fewer positions than winners, empty sequences, ties at the cut that fill more than one
wavefront's rank list, corrections at the edge of its LDS -- against the oracle, and against the same call cut into splits
of 256 positions, which takes the merge kernel."""
import ctypes as C

import numpy as np
import pytest
import torch

from tests.helpers import make_case, to_device
from tests.test_gpu_fused import check_against_oracle, run_fused

pytestmark = pytest.mark.gpu

SCALE = 128 ** -0.5


def _plan(scheme_id, gs, B, Hq, Hkv, S, K):
    from jetfire_amd import _lib
    out = [C.c_int() for _ in range(4)]
    _lib.check(_lib.load().jf_fused_plan(scheme_id, gs, B, Hq, Hkv, S, K, *[C.byref(o) for o in out]))
    return [o.value for o in out]


def _one_split(scheme_id, gs, B, Hq, Hkv, S, K, split_len):
    """Whether the call merges by itself when its splits are `split_len` positions long."""
    from jetfire_amd import _lib
    out = C.c_int(-1)
    _lib.check(_lib.debug_hook("jf_debug_split_len")(split_len))
    try:
        _lib.check(_lib.debug_hook("jf_debug_one_split")(0, scheme_id, gs, B, Hq, Hkv, S, K, C.byref(out)))
    finally:
        _lib.check(_lib.debug_hook("jf_debug_split_len")(0))
    return out.value


def _both(scheme, c, d, S, K):
    """The call with one split, which merges by itself, and with splits of 256 positions and the merge launch."""
    from jetfire_amd import _lib, ops
    res = []
    for split in (-(-S // 256) * 256, 256):
        assert _one_split(ops.FUSED_SCHEMES[scheme], c["gs"], c["B"], c["Hq"], c["Hkv"], S, K, split) == (split >= S)
        _lib.check(_lib.debug_hook("jf_debug_split_len")(split))
        try:
            res.append([t.clone() for t in run_fused(scheme, c, d, S, K)])
        finally:
            _lib.check(_lib.debug_hook("jf_debug_split_len")(0))
    return res


@pytest.mark.parametrize("scheme,kb,vb,gs,G,S,lens,K", [
    ("k4v4", 4, 4, 128, 4, 1, [1], 32),
    ("k4v4", 4, 4, 128, 4, 257, [257, 0, 256, 17], 64),
    ("k3v2", 3, 2, 64, 4, 1024, [1024, 1023, 63, 65], 256),
    ("k3v2", 3, 2, 64, 4, 2040, [2040, 1, 0], 512),
    ("k3v2", 3, 2, 64, 8, 1111, [1111, 700], 128),
    ("k3v2", 3, 2, 64, 8, 512, [512, 100], 128),
    ("k2v2", 2, 2, 64, 1, 3900, [3900, 16], 2048),
    ("k3v3", 3, 3, 64, 2, 1500, [1500, 64], 256),
    ("k3v3", 3, 3, 128, 7, 800, [800, 799], 64),
    ("b4v4", 4, 4, 64, 4, 900, [900, 450], 128),
    ("a2v4", 2, 4, 128, 16, 400, [400, 33], 64),
])
def test_one_split_matches_oracle_and_merge(scheme, kb, vb, gs, G, S, lens, K):
    Hkv = 2 if G < 16 else 1
    c = make_case(91, len(lens), G * Hkv, Hkv, S, kb, vb, gs, lens=lens, k_asym=scheme.startswith("a"))
    d = to_device(c)
    one, cut = _both(scheme, c, d, S, K)
    check_against_oracle(scheme, c, S, K, one)
    # same winners; the sums differ by the order of fp32 additions over the splits (and, over the winners, of at most
    # 2048 terms of one sign pattern): 3e-6, the bound both hold against the oracle
    assert torch.equal(one[4], cut[4]) and torch.equal(one[1], cut[1])
    for a, b in ((one[0], cut[0]), (one[2], cut[2]), (one[3], cut[3])):
        assert float((a - b).abs().max()) <= 6e-6


@pytest.mark.parametrize("levels", [1, 3, 40])
@pytest.mark.parametrize("S,K", [(300, 64), (300, 256), (1500, 256)])
def test_one_split_ties(levels, S, K):
    """Key rows copied from a few distinct ones: the cut bucket holds fewer members than a rank list (levels 40), more
    (levels 3: hundreds of equal scores; 1: all of them, more than top_k and its slack).  Lowest positions win."""
    c = make_case(92, 2, 8, 2, S, 4, 4, 128, lens=[S, S - 37])
    d = to_device(c)
    kd, ks, bt = d["kd"].clone(), d["ks"].clone(), d["bt"]
    pos = torch.arange(S, device="cuda")
    for b in range(2):
        slot = bt[b, pos // 16] * 16 + pos % 16
        src = slot[pos % levels]
        kd[:, slot], ks[:, slot] = d["kd"][:, src], d["ks"][:, src]
    d["kd"], d["ks"] = kd, ks
    one, cut = _both("k4v4", c, d, S, K)
    assert torch.equal(one[4], cut[4]) and torch.equal(one[1], cut[1])
    scores = one[7].cpu().numpy()
    for b, n in enumerate((S, S - 37)):
        for h in range(8):
            want = np.sort(np.lexsort((np.arange(n), -scores[b, h, :n]))[:K])
            got = one[4][b, h].cpu().numpy()
            assert np.array_equal(got[:len(want)], want) and (got[len(want):] == -1).all()


def test_plan_takes_one_split_for_short_and_many_sequences():
    assert _plan(44, 128, 1, 32, 8, 777, 64)[1] == 1 and _one_split(44, 128, 1, 32, 8, 777, 64, 0)
    assert _plan(32, 64, 32, 32, 8, 2048, 256)[1] == 1 and _one_split(32, 64, 32, 32, 8, 2048, 256, 0)
    assert _plan(44, 128, 1, 32, 8, 4096, 64)[1] > 1


def _crowded(d, c, S, kind):
    """Scores that put far more positions in the bucket of the cut than a rank list holds."""
    kd, ks, bt = d["kd"].clone(), d["ks"].clone(), d["bt"]
    pos = torch.arange(S, device="cuda")
    for b in range(bt.size(0)):
        slot = bt[b, pos // 16] * 16 + pos % 16
        if kind == "outlier":      # one key row three hundred times the others: the buckets of every head are that much wider
            ks[:, slot[S // 3]] *= 300
        elif kind == "levels":     # eight distinct rows: eight scores, each shared by an eighth of the positions
            src = slot[pos % 8]
            kd[:, slot], ks[:, slot] = d["kd"][:, src], d["ks"][:, src]
        elif kind == "infinite":   # scores of both signs' infinity: no finite range, everything in one bucket
            ks[:, slot[5]] = float("inf")
        elif kind == "nan":        # a finite range, and scores without a place in it
            ks[:, slot[[5, S // 2]]] = float("nan")
    d["kd"], d["ks"] = kd, ks


@pytest.mark.parametrize("kind", ["outlier", "levels", "plain", "infinite", "nan"])
@pytest.mark.parametrize("scheme,kb,vb,gs,G,S,K", [
    ("k2v2", 2, 2, 64, 1, 3900, 2048),
    ("k4v4", 4, 4, 128, 2, 2048, 512),
    ("k4v4", 4, 4, 128, 4, 777, 64),
    ("k3v2", 3, 2, 64, 4, 2048, 256),
    ("k3v2", 3, 2, 64, 7, 1000, 128),
    ("k3v2", 3, 2, 64, 8, 512, 128),
    ("k3v3", 3, 3, 64, 16, 256, 32),
])
def test_one_split_selects_from_a_crowded_bucket(scheme, kb, vb, gs, G, S, K, kind):
    Hkv, lens = 2, [S, S - S // 5]
    c = make_case(94, 2, G * Hkv, Hkv, S, kb, vb, gs, lens=lens)
    d = to_device(c)
    _crowded(d, c, S, kind)
    one, cut = _both(scheme, c, d, S, K)
    assert torch.equal(one[4], cut[4]) and torch.equal(one[1], cut[1])
    scores = one[7].cpu().numpy()
    for b, n in enumerate(lens):
        for h in range(G * Hkv):
            # the order of the kernels' keys: NaNs with the sign bit below everything, the others above
            u = scores[b, h, :n].view(np.uint32)
            key = np.where(u >> 31, ~u, u | np.uint32(1 << 31)).astype(np.int64)
            want = np.sort(np.lexsort((np.arange(n), -key))[:K])
            got = one[4][b, h].cpu().numpy()
            assert np.array_equal(got[:len(want)], want) and (got[len(want):] == -1).all()


def _winners_by_key(scores, n, K):
    """Positions of the K largest of scores[:n] in the order of the kernels' keys, ties to the lowest position."""
    u = scores[:n].view(np.uint32)
    key = np.where(u >> 31, ~u, u | np.uint32(1 << 31)).astype(np.int64)
    return np.sort(np.lexsort((np.arange(n), -key))[:K])


# a head's finite scores this close together have no finite number of buckets per unit: 254.99 / range overflows
NARROW = 254.99 / float(np.finfo(np.float32).max)


@pytest.mark.parametrize("scheme,kb,vb,gs,G,S,K", [
    ("k3v2", 3, 2, 64, 4, 1024, 512),      # more winners than one of the head's four segments has positions
    ("k3v2", 3, 2, 64, 8, 1000, 128),
    ("k2v2", 2, 2, 64, 1, 3900, 2048),
    ("b4v4", 4, 4, 64, 4, 900, 64),
])
def test_one_split_scores_within_a_range_too_narrow_for_buckets(scheme, kb, vb, gs, G, S, K):
    Hkv, lens = 2, [S, S - S // 5]
    c = make_case(97, 2, G * Hkv, Hkv, S, kb, vb, gs, lens=lens)
    d = to_device(c)
    d["ks"] = (d["ks"].float() * 2.0 ** -122).to(torch.bfloat16)
    one, cut = _both(scheme, c, d, S, K)
    scores = one[7].cpu().numpy()
    narrow = 0
    for b, n in enumerate(lens):
        for h in range(G * Hkv):
            s = scores[b, h, :n]
            narrow += 0 < float(s.max()) - float(s.min()) < NARROW
            want, got = _winners_by_key(s, n, K), one[4][b, h].cpu().numpy()
            assert np.array_equal(got[:len(want)], want) and (got[len(want):] == -1).all(), (b, h)
    assert narrow > 0
    assert torch.equal(one[4], cut[4]) and torch.equal(one[1], cut[1])
    for a, b in ((one[0], cut[0]), (one[2], cut[2]), (one[3], cut[3])):
        assert float((a - b).abs().max()) <= 6e-6


@pytest.mark.parametrize("width", [1e-40, 1e-37, 4e-37, 7e-37, 8e-37])
@pytest.mark.parametrize("Hq,S,K", [(4, 2048, 1024), (4, 777, 64), (2, 1000, 512), (1, 3900, 2048)])
def test_selection_from_given_scores_within_a_range_too_narrow_for_buckets(Hq, S, K, width):
    from jetfire_amd import _lib, ops
    rng = np.random.default_rng(98)
    lens = np.array([S, S - 100], np.int32)
    scores = (rng.random((2, Hq, S)) - rng.choice([0.0, 0.5, 1.0], (2, Hq, 1))).astype(np.float32) * np.float32(width)
    table = torch.randperm(2 * ((S + 15) // 16)).reshape(2, -1).cuda()
    got = []
    for split in (-(-S // 256) * 256, 256):
        _lib.check(_lib.debug_hook("jf_debug_split_len")(split))
        try:
            got.append(ops._topk(torch.from_numpy(scores).cuda(), table, torch.from_numpy(lens).cuda(), S, Hq, 16, K, True, "topk"))
        finally:
            _lib.check(_lib.debug_hook("jf_debug_split_len")(0))
    for b, n in enumerate(lens):
        for h in range(Hq):
            want = _winners_by_key(scores[b, h], n, K)
            for idx, slots, _, _ in got:
                i = idx[b, h].cpu().numpy()
                assert np.array_equal(i[:len(want)], want) and (i[len(want):] == -1).all(), (b, h)
                pos = idx[b, h, :len(want)]
                assert torch.equal(slots[b, h, :len(want)], table[b, pos // 16] * 16 + pos % 16)


@pytest.mark.parametrize("kind", ["outlier", "levels", "plain"])
@pytest.mark.parametrize("scheme,kb,vb,gs,B,Hkv,G,S,K,other", [
    ("k2v2", 2, 2, 64, 16, 8, 1, 3900, 2048, 256),
    ("k2v2", 2, 2, 64, 16, 8, 1, 3900, 1024, 2048),
    ("k4v4", 4, 4, 128, 32, 8, 4, 1024, 512, 256),
    ("k3v2", 3, 2, 64, 16, 4, 8, 1000, 256, 256),
])
def test_one_split_is_no_slower_than_the_merge_launch(scheme, kb, vb, gs, B, Hkv, G, S, K, other, kind):
    """Bounded work per member of the cut bucket: ranking each against the whole list took two to seventeen times the
    merge launch's time here, and the exact selection by one wavefront per head, where the list was too short for the
    bucket, twice that of the longest splits with a launch (`other`: their length)."""
    from jetfire_amd import _lib, ops
    c = make_case(95, B, G * Hkv, Hkv, S, kb, vb, gs)
    d = to_device(c)
    _crowded(d, c, S, kind)
    times = []
    for split in (-(-S // 256) * 256, other):
        assert _one_split(ops.FUSED_SCHEMES[scheme], gs, B, G * Hkv, Hkv, S, K, split) == (split > other)
        _lib.check(_lib.debug_hook("jf_debug_split_len")(split))
        try:
            best = float("inf")
            for _ in range(6):
                e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                torch.cuda.synchronize()
                e0.record()
                for _ in range(10):
                    run_fused(scheme, c, d, S, K)
                e1.record()
                e1.synchronize()
                best = min(best, e0.elapsed_time(e1))
            times.append(best)
        finally:
            _lib.check(_lib.debug_hook("jf_debug_split_len")(0))
    assert times[0] <= 1.5 * times[1], times


@pytest.mark.parametrize("G,S,K,filled", [(2, 300, 512, "first"), (8, 600, 128, "holes"), (4, 700, 256, "last"),
                                          (7, 290, 32, "holes"), (2, 400, 64, "none"), (1, 300, 1024, "ascending")])
def test_stage_b_goes_over_the_entries_that_name_positions(G, S, K, filled):
    """Stage B alone, merging in the scan: given lists that end early, have holes, or name positions past the end."""
    from jetfire_amd import _lib, ops
    Hkv = 2
    c = make_case(96, 2, G * Hkv, Hkv, S, 3, 3, 64, lens=[S, S - 40])
    d = to_device(c)
    sc = ops.int3_qk_scores(d["q"], d["kd"], d["ks"], d["bt"], d["lens"], S, G * Hkv, Hkv, 16, SCALE)
    idx = torch.full((2, G * Hkv, K), -1, dtype=torch.int64, device="cuda")
    n = min(K, S)
    if filled in ("first", "ascending"):
        idx[..., :n] = torch.arange(n, device="cuda") if filled == "ascending" else torch.randperm(S, device="cuda")[:n]
    elif filled == "holes":
        idx[..., ::3] = torch.arange(0, K, 3, device="cuda")
        idx[..., 1::3] = S + 5
    elif filled == "last":
        idx[..., -1] = S // 2
    res = []
    for split in (-(-S // 256) * 256, 256):
        assert _one_split(33, 64, 2, G * Hkv, Hkv, S, K, split) == (split > 256)
        _lib.check(_lib.debug_hook("jf_debug_split_len")(split))
        try:
            res.append([t.clone() for t in ops.int3_softmax_v_with_pre_corr_wvs2(sc, d["vd"], d["vs"], d["bt"], d["lens"], idx,
                                                                                  S, G * Hkv, Hkv, 16, K)])
        finally:
            _lib.check(_lib.debug_hook("jf_debug_split_len")(0))
    for a, b in zip(*res):      # (the bound of the comparison above)
        assert float((a - b).abs().max()) <= 6e-6
