"""The merge kernel's threshold search at the sizes of its three paths: a cut bucket of at most 16 members (ranked in
registers), of up to 1024 (a list in LDS), of more (bisection), with ties across the cut (and once without), in both
shapes of the kernel (1024 threads; 256 threads for more rows than compute units); and with the winners in few of the lists."""
import numpy as np
import pytest
import torch

from tests.helpers import make_case, to_device
from tests.test_gpu_fused import run_fused

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


def test_five_rows_of_the_light_shape_share_a_compute_unit():
    """What the light shape is for (many rows, few candidates each): its registers and LDS leave room for five
    workgroups per compute unit."""
    import ctypes as C

    from jetfire_amd import _lib
    n = C.c_int(0)
    _lib.check(_lib.debug_hook("jf_debug_light_merge_per_cu")(C.byref(n)))
    assert n.value >= 5
