"""A head whose scores are infinite or NaN leaves the other heads of its kv-head alone: their outputs are the bits of the same
call without it."""
import numpy as np
import pytest
import torch

from tests.helpers import make_case, to_device
from tests.test_gpu_fused import run_fused

pytestmark = pytest.mark.gpu

SCALE = 128 ** -0.5


def _same_elsewhere(good, bad, heads):
    keep = [h for h in range(good[0].size(1)) if h not in heads]
    for a, b in zip(good, bad):
        a, b = a[:, keep].contiguous(), b[:, keep].contiguous()
        assert torch.equal(a.view(torch.int32), b.view(torch.int32)), (a.shape, int((a != b).sum()))


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
@pytest.mark.parametrize("G,heads", [(1, [0]), (2, [0]), (3, [0]), (4, [0]), (4, [2]), (4, [0, 1, 2]), (8, [0, 4])])
@pytest.mark.parametrize("scheme,vb,split_len", [("k4v4", 4, 1024), ("k4v4", 4, 256), ("k4v2", 2, 512), ("k4v3", 3, 1024)])
def test_query_with_an_element_that_is_no_number(scheme, vb, split_len, G, heads, value):
    from jetfire_amd import _lib
    S, Hkv, K = 1000, 2, 64
    c = make_case(111, 2, G * Hkv, Hkv, S, 4, vb, 128, lens=[S, 300])
    d = to_device(c)
    _lib.check(_lib.debug_hook("jf_debug_split_len")(split_len))
    try:
        good = [t.clone() for t in run_fused(scheme, c, d, S, K)]
        d["q"][:, heads, 5] = value
        bad = [t.clone() for t in run_fused(scheme, c, d, S, K)]
    finally:
        _lib.check(_lib.debug_hook("jf_debug_split_len")(0))
    _same_elsewhere(good, bad, heads)


@pytest.mark.parametrize("kind", ["infinite", "nan", "nowhere"])
@pytest.mark.parametrize("bits,gs", [(2, 64), (2, 128), (3, 64), (4, 64), (4, 128)])
@pytest.mark.parametrize("G,heads,split_len", [(4, [0], 1024), (4, [0], 256), (4, [1], 1024), (8, [0, 4], 512), (2, [0], 1024)])
def test_given_scores_that_are_no_numbers(bits, gs, G, heads, split_len, kind):
    from jetfire_amd import _lib, ops
    S, Hkv, K = 700, 2, 64
    c = make_case(112, 2, G * Hkv, Hkv, S, 3, bits, gs, lens=[S, 300])
    d = to_device(c)
    scores = torch.from_numpy(np.random.default_rng(113).standard_normal((2, G * Hkv, S)).astype(np.float32)).cuda()
    idx = torch.arange(K, device="cuda").expand(2, G * Hkv, K).contiguous()
    stage_b = {2: ops.int2_softmax_v_with_pre_corr_wvs2, 3: ops.int3_softmax_v_with_pre_corr_wvs2,
               4: ops.int4_softmax_v_with_pre_corr_wvs2_scores}[bits]
    _lib.check(_lib.debug_hook("jf_debug_split_len")(split_len))
    try:
        good = [t.clone() for t in stage_b(scores, d["vd"], d["vs"], d["bt"], d["lens"], idx, S, G * Hkv, Hkv, 16, K)]
        if kind == "nowhere":
            scores[:, heads] = float("-inf")
        else:
            scores[:, heads, 77] = float("inf" if kind == "infinite" else "nan")
        bad = [t.clone() for t in stage_b(scores, d["vd"], d["vs"], d["bt"], d["lens"], idx, S, G * Hkv, Hkv, 16, K)]
    finally:
        _lib.check(_lib.debug_hook("jf_debug_split_len")(0))
    _same_elsewhere(good, bad, heads)
