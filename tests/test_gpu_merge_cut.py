"""The merge kernel's threshold search at the sizes of its three paths: a cut bucket of at most 16 members (ranked in
registers), of up to 1024 (a list in LDS), of more (bisection), with ties across the cut (and once without), in both
shapes of the kernel (1024 threads; 256 threads for more rows than compute units); and with the winners in few of the lists."""
import numpy as np
import pytest
import torch

from tests.helpers import make_case, to_device
from tests.test_gpu_fused import check_against_oracle, run_fused

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [1, 40])
@pytest.mark.parametrize("K,copies", [(32, 10), (32, 12), (32, 14), (32, 15), (32, 17), (64, 40), (64, 45), (64, 58),
                                      (64, 64), (64, 65), (64, 500), (64, 1100)])
def test_equal_scores_around_the_cut(B, K, copies):
    from jetfire_amd import _lib
    S, Hq, Hkv = 2048, 8, 1
    c = make_case(93, 1, Hq, Hkv, S, 4, 4, 128, lens=[S])
    if B > 1:      # the same sequence B times: the same pages, the same queries
        for key in ("q", "bt", "lens"):
            c[key] = np.repeat(c[key], B, axis=0)
        c["B"] = B
    d = to_device(c)
    base = run_fused("k4v4", c, d, S, 32)
    # `copies` positions get the key row of the 20th best position of head 0: one bucket of equal scores at the cut
    order = torch.argsort(base[7][0, 0], descending=True, stable=True)
    src, dst = int(order[20]), torch.sort(order[200:200 + copies]).values
    bt = d["bt"][0]
    slot = lambda t: bt[t // 16] * 16 + t % 16
    d["kd"], d["ks"] = d["kd"].clone(), d["ks"].clone()
    d["kd"][:, slot(dst)] = d["kd"][:, slot(torch.tensor([src], device="cuda"))]
    d["ks"][:, slot(dst)] = d["ks"][:, slot(torch.tensor([src], device="cuda"))]
    _lib.check(_lib.debug_hook("jf_debug_split_len")(256))
    try:
        out = run_fused("k4v4", c, d, S, K)
    finally:
        _lib.check(_lib.debug_hook("jf_debug_split_len")(0))
    scores, idx = out[7].cpu().numpy(), out[4].cpu().numpy()
    # (head 0: twenty better positions, the copied one and its copies; the tie lies across the cut from K - 20 copies on)
    ranked = np.sort(scores[0, 0])[::-1]
    assert (ranked[K - 1] == ranked[K]) == (copies >= K - 20)
    for b in (0, B - 1):
        for h in range(Hq):
            want = np.sort(np.lexsort((np.arange(S), -scores[b, h]))[:K])
            assert np.array_equal(idx[b, h], want), (b, h)


@pytest.mark.parametrize("B", [1, 40])
@pytest.mark.parametrize("split_len", [256, 512])
@pytest.mark.parametrize("order", ["falling", "rising", "infinite"])
@pytest.mark.parametrize("K", [32, 64, 256, 512, 1024, 2048, 4096])
def test_winners_crowd_into_few_lists(B, split_len, order, K):
    """The merge bounds the K-th largest score by the splits' own cuts: positions sorted by head 0's scores put all of its
    winners into one list (or two, or all of each), whose cut lies above everything the other lists hold; an infinite
    score leaves no range to cut into buckets; corrections beyond a split's length, and beyond the sequence's."""
    from jetfire_amd import _lib
    S, Hq, Hkv = 2045, 8, 1
    c = make_case(94, 1, Hq, Hkv, S, 4, 4, 128, lens=[S])
    if B > 1:
        for key in ("q", "bt", "lens"):
            c[key] = np.repeat(c[key], B, axis=0)
        c["B"] = B
    d = to_device(c)
    base = run_fused("k4v4", c, d, S, 32)
    pos = torch.arange(S, device="cuda")
    slot = d["bt"][0][pos // 16] * 16 + pos % 16
    by_score = torch.argsort(base[7][0, 0], descending=order != "rising", stable=True)
    if order == "infinite":
        d["ks"] = d["ks"].clone()
        d["ks"][:, slot[by_score[700]]] = float("inf")
    else:
        d["kd"], d["ks"] = d["kd"].clone(), d["ks"].clone()
        d["kd"][:, slot], d["ks"][:, slot] = d["kd"][:, slot[by_score]], d["ks"][:, slot[by_score]]
    _lib.check(_lib.debug_hook("jf_debug_split_len")(split_len))
    try:
        out = run_fused("k4v4", c, d, S, K)
    finally:
        _lib.check(_lib.debug_hook("jf_debug_split_len")(0))
    scores, idx = out[7].cpu().numpy(), out[4].cpu().numpy()
    assert not np.isnan(scores).any()
    for b in (0, B - 1):
        for h in range(Hq):
            want = np.full(K, -1)
            n = min(K, S)
            want[:n] = np.sort(np.lexsort((np.arange(S), -scores[b, h, :S]))[:n])
            assert np.array_equal(idx[b, h], want), (b, h)


@pytest.mark.parametrize("order", ["falling", "rising", "infinite", "nan"])
@pytest.mark.parametrize("S,K,split_len,first,final", [
    (20000, 64, 256, 1280, 1024),         # two stages, lists longer than the correction: each part bounded by its largest cut
    (40000, 2048, 256, 10240, 8192),      # lists shorter than it (the smallest cut); parts of the 32-candidate shape
    (40000, 2048, 2048, 10240, 8192),     # ... lists as long as it
    (65536, 4096, 256, 16384, 16384),     # 256 lists; winners in dynamic LDS in both stages
    (33100, 8192, 256, 0, 33280),         # one stage, 130 lists, candidates beyond the registers
])
def test_winners_crowd_into_few_lists_of_two_stages(S, K, split_len, first, final, order):
    """The first stage hands the second a lower bound with every part's list, and the shapes of 32 candidates per thread look
    up a winner's position when it is known: the same orders of scores as above, and scores that are NaN."""
    import ctypes as C
    from jetfire_amd import _lib
    Hq, Hkv = 8, 1
    c = make_case(97, 1, Hq, Hkv, S, 4, 4, 128, lens=[S])
    d = to_device(c)
    base = run_fused("k4v4", c, d, S, 32)
    pos = torch.arange(S, device="cuda")
    slot = d["bt"][0][pos // 16] * 16 + pos % 16
    by_score = torch.argsort(base[7][0, 0], descending=order != "rising", stable=True)
    d["kd"], d["ks"] = d["kd"].clone(), d["ks"].clone()
    if order in ("infinite", "nan"):
        d["ks"][:, slot[by_score[[700, S // 2]]]] = float("inf" if order == "infinite" else "nan")
    else:
        d["kd"][:, slot], d["ks"][:, slot] = d["kd"][:, slot[by_score]], d["ks"][:, slot[by_score]]
    L, ns, cap, parts = [C.c_int() for _ in range(4)]
    _lib.check(_lib.debug_hook("jf_debug_split_len")(split_len))
    try:
        _lib.check(_lib.load().jf_fused_plan(44, 128, 1, Hq, Hkv, S, K, *[C.byref(x) for x in (L, ns, cap, parts)]))
        out = run_fused("k4v4", c, d, S, K)
    finally:
        _lib.check(_lib.debug_hook("jf_debug_split_len")(0))
    if parts.value > 1:
        assert (-(-ns.value // parts.value) * cap.value, parts.value * K) == (first, final)
    else:
        assert (0, ns.value * cap.value) == (first, final)
    scores, idx, slots = out[7].cpu().numpy(), out[4].cpu().numpy(), out[1].cpu().numpy()
    for h in range(Hq):
        # the order of the kernels' keys: NaNs with the sign bit below everything, the others above
        u = scores[0, h].view(np.uint32)
        key = np.where(u >> 31, ~u, u | np.uint32(1 << 31)).astype(np.int64)
        want = np.sort(np.lexsort((np.arange(S), -key))[:K])
        assert np.array_equal(idx[0, h], want), h
        assert np.array_equal(slots[0, h], slot.cpu().numpy()[want]), h


@pytest.mark.parametrize("scheme,kb,vb,gs,S,K", [
    ("k4v4", 4, 4, 128, 33100, 64),       # 130 splits, the third group of 64; two stages
    ("k3v2", 3, 2, 64, 50000, 8192),      # 196 splits, the fourth; one stage
    ("k3v2", 3, 2, 64, 65536, 256),       # 256 splits, the most there are
])
def test_up_to_256_splits_match_the_oracle(scheme, kb, vb, gs, S, K):
    """The merge keeps the splits' statistics in the lanes, 64 splits at a time: all four groups of them, and sequences that
    end in the third, the second and the first, behind which the splits are empty."""
    from jetfire_amd import _lib
    c = make_case(98, 4, 2, 1, S, kb, vb, gs, lens=[S, 129 * 256, 100 * 256 + 7, 300])
    d = to_device(c)
    _lib.check(_lib.debug_hook("jf_debug_split_len")(256))
    try:
        out = [t.clone() for t in run_fused(scheme, c, d, S, K)]
    finally:
        _lib.check(_lib.debug_hook("jf_debug_split_len")(0))
    check_against_oracle(scheme, c, S, K, out)


@pytest.mark.parametrize("G,copies,split_len", [
    (4, 1, 256), (8, 1, 256),     # a merge launch, 1024 threads
    (8, 3, 256), (4, 12, 256),    # ... 256 threads, all roles at once and one at a time
    (1, 1, 768), (4, 1, 768), (8, 1, 768),     # the scan that merges by itself: sixteen wavefronts per head to one
])
@pytest.mark.parametrize("scheme,kb,vb,gs", [("k3v2", 3, 2, 64), ("k3v3", 3, 3, 64), ("k4v4", 4, 4, 128), ("b4v4", 4, 4, 64)])
def test_sums_over_the_winners_at_the_edges_of_their_batches(scheme, kb, vb, gs, G, copies, split_len):
    """Value rows are gathered in full batches and a short one behind them: as many winners as positions, around every
    multiple a batch can have."""
    from jetfire_amd import _lib
    lens = [1, 7, 9, 31, 33, 64, 65, 127, 129, 192, 255, 256, 257, 320, 383, 385, 449, 511, 512, 600] * copies
    c = make_case(99, len(lens), G, 1, 600, kb, vb, gs, lens=lens)
    d = to_device(c)
    _lib.check(_lib.debug_hook("jf_debug_split_len")(split_len))
    try:
        out = [t.clone() for t in run_fused(scheme, c, d, 600, 512)]
    finally:
        _lib.check(_lib.debug_hook("jf_debug_split_len")(0))
    check_against_oracle(scheme, c, 600, 512, out)


def test_five_rows_of_the_light_shape_share_a_compute_unit():
    """What the light shape is for (many rows, few candidates each): its registers and LDS leave room for five
    workgroups per compute unit."""
    import ctypes as C

    from jetfire_amd import _lib
    n = C.c_int(0)
    _lib.check(_lib.debug_hook("jf_debug_light_merge_per_cu")(C.byref(n)))
    assert n.value >= 5
