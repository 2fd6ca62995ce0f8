"""Sums over the winners' value rows, 64 at a time with 30-bit weights: rows whose scales lie far apart or are negative, a large
weight whose codes are zero, an infinite scale or a NaN among them, and one in a slot that only padding names; in the scan that
merges by itself and the shapes of the merge."""
import numpy as np
import pytest
import torch

from oracle import jetfire_oracle as O
from tests.helpers import bits_to_bf16, make_case, to_device
from tests.test_gpu_fused import run_fused

pytestmark = pytest.mark.gpu


def _bits(x):
    return O.f32_to_bf16_bits(np.asarray(x, np.float32))


@pytest.mark.parametrize("kind", ["range", "signed", "zero", "infinite", "nan", "unused"])
@pytest.mark.parametrize("copies,split_len,K", [(1, 768, 64), (1, 768, 256), (1, 256, 64), (1, 256, 512), (20, 256, 256), (20, 256, 512)])
@pytest.mark.parametrize("scheme,kb,vb,gs", [("k3v2", 3, 2, 64), ("k3v2", 3, 2, 128), ("k3v3", 3, 3, 64), ("k4v4", 4, 4, 128), ("b4v4", 4, 4, 64)])
def test_scales_of_any_size(scheme, kb, vb, gs, copies, split_len, K, kind):
    from jetfire_amd import _lib
    S, G, Hkv = 700, 8, 2
    lens = [S, 70] * copies
    c = make_case(101, len(lens), G * Hkv, Hkv, S, kb, vb, gs, lens=lens, extra_blocks=1)
    c["bt"] = (np.random.default_rng(5).permutation(c["bt"].size) + 1).reshape(c["bt"].shape).astype(np.int64)  # (block 0: nobody's)
    d = to_device(c)
    _lib.check(_lib.debug_hook("jf_debug_split_len")(split_len))
    try:
        if kind == "signed":
            vs = O.bf16_bits_to_f32(c["vs"])
            c["vs"] = _bits(np.where(np.random.default_rng(7).random(vs.shape) < 0.4, -vs, vs))
        elif kind == "zero":        # one weight 2^16 times the others', in channels to which it adds nothing
            out = [t.cpu().numpy() for t in run_fused(scheme, c, d, S, K)]
            vs = O.bf16_bits_to_f32(c["vs"])
            for hkv in range(Hkv):
                slot = int(out[1][0, hkv * G, 5])
                vs[hkv, slot] *= 2.0 ** 16
                c["vd"][hkv, slot] = O.pack_codes(np.full(128, O.offset(vb)), vb)
            c["vs"] = _bits(vs)
            d["vd"] = torch.from_numpy(c["vd"]).cuda()
        elif kind != "range":
            out = [t.cpu().numpy() for t in run_fused(scheme, c, d, S, K)]
            bad = np.float32(np.nan if kind == "nan" else np.inf)
            slot = 0 if kind == "unused" else int(out[1][0, 0, 5])
            c["vs"][0, slot, -1] = _bits([bad])[0]
        else:
            vs = O.bf16_bits_to_f32(c["vs"])
            c["vs"] = _bits(vs * np.exp2(np.random.default_rng(6).integers(-20, 21, vs.shape)).astype(np.float32))
        d["vs"] = bits_to_bf16(c["vs"]).cuda()
        out = [t.cpu().numpy() for t in run_fused(scheme, c, d, S, K)]
    finally:
        _lib.check(_lib.debug_hook("jf_debug_split_len")(0))
    _, slots, o_old, W, idx, m, iz, scores = out
    codes = O.decode_codes(c["vd"], vb).astype(np.float64) - O.offset(vb)
    vs = O.bf16_bits_to_f32(c["vs"]).astype(np.float64)
    for b in range(2):      # (the others are further copies)
        for hq in range(G * Hkv):
            won = idx[b, hq] >= 0
            p = np.exp(scores[b, hq, idx[b, hq][won]].astype(np.float64) - m[b, hq]) * iz[b, hq]
            sl = slots[b, hq][won]
            for g in range(128 // gs):
                w = p * vs[hq // G, sl, g]
                got = o_old[b, hq, g * gs:(g + 1) * gs]
                if not np.isfinite(w).all():
                    assert not np.isfinite(got).any(), (b, hq, g)
                    continue
                v = codes[hq // G, sl, g * gs:(g + 1) * gs]
                # the weights' own fp32 error (scores, exponential, products): 4e-6 of the sum of magnitudes; half a unit of 30
                # bits of the largest of 64 for each code, and a unit where the sums of the limbs are joined
                tol = 4e-6 * (np.abs(w[:, None] * v)).sum(0)
                for i in range(0, len(w), 64):
                    tol += 2.0 ** (np.frexp(np.abs(w[i:i + 64]).max())[1] - 31) * (np.abs(v[i:i + 64]).sum(0) + 2)
                assert (np.abs(got - (w[:, None] * v).sum(0)) <= tol).all(), (b, hq, g)
            assert abs(W[b, hq] - p.sum()) <= 4e-6 * max(1.0, p.sum())


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("G,K", [(4, 32), (4, 64), (1, 256), (8, 32), (4, 256)])     # code by code, and 64 at a time
@pytest.mark.parametrize("scheme,kb,vb,gs", [("k3v2", 3, 2, 64), ("k3v3", 3, 3, 64), ("k4v4", 4, 4, 128), ("b4v4", 4, 4, 64)])
def test_scale_of_the_slot_that_stands_in_for_no_winner(scheme, kb, vb, gs, G, K, bad):
    """Fewer winners than the correction is wide, and Stage B with lists that have holes: entries without a position read slot 0,
    which is nobody's, and whose scale makes no difference."""
    from jetfire_amd import _lib, ops
    S, Hkv = 700, 2
    c = make_case(105, 3, G * Hkv, Hkv, S, kb, vb, gs, lens=[S, 9, 33], extra_blocks=1)
    c["bt"] = (np.random.default_rng(5).permutation(c["bt"].size) + 1).reshape(c["bt"].shape).astype(np.int64)
    d = to_device(c)
    idx = torch.arange(K, device="cuda").expand(3, G * Hkv, K).clone()
    idx[..., 1::3] = -1
    stage_b = {2: ops.int2_softmax_v_with_pre_corr_wvs2, 3: ops.int3_softmax_v_with_pre_corr_wvs2,
               4: ops.int4_softmax_v_with_pre_corr_wvs2_scores}[vb]
    res = []
    for scale in (1.0, bad):
        d["vs"][:, 0] = scale
        for split in (768, 256):
            _lib.check(_lib.debug_hook("jf_debug_split_len")(split))
            try:
                full = run_fused(scheme, c, d, S, K)
                res.append([t.clone() for t in list(full) + list(stage_b(full[7], d["vd"], d["vs"], d["bt"], d["lens"], idx, S, G * Hkv, Hkv, 16, K))])
            finally:
                _lib.check(_lib.debug_hook("jf_debug_split_len")(0))
    for plain, odd in ((res[0], res[2]), (res[1], res[3])):
        for a, b in zip(plain, odd):
            assert torch.equal(a, b), a.shape


@pytest.mark.parametrize("Hq,Hkv,S,lens,K", [(8, 2, 700, [700, 70], 64), (8, 1, 2000, [2000, 1999], 512), (32, 8, 300, [300] * 10, 256)])
def test_negative_scales_in_the_int8_tiles_form(Hq, Hkv, S, lens, K):
    """The form whose o_hat takes scales of either sign: o_old_unnorm does too."""
    from jetfire_amd import ops
    c = make_case(104, len(lens), Hq, Hkv, S, 4, 4, 128, lens=lens)
    vs = O.bf16_bits_to_f32(c["vs"])
    c["vs"] = _bits(np.where(np.random.default_rng(8).random(vs.shape) < 0.4, -vs, vs))
    d = to_device(c)
    sc = O.scores_int8_model(c["q"], c["kd"], c["ks"], c["bt"], c["lens"], S, Hq, Hkv, 16, 128 ** -0.5)
    idx, _ = O.topk_select(sc, c["lens"], c["bt"], S, K)
    m, iz = O.softmax_stats(sc, c["lens"], S)
    got = ops.int8tc_softmax_v_with_pre_corr_reg_stats(
        torch.from_numpy(sc).cuda(), torch.from_numpy(m).cuda(), torch.from_numpy(iz).cuda(), d["vd"], d["vs"], d["bt"], d["lens"],
        torch.from_numpy(idx).cuda(), S, Hq, Hkv, 16, K)
    want = O.softmax_v_int8_tiles(sc, m, iz, c["vd"], c["vs"], c["bt"], c["lens"], idx, S, Hq, Hkv, 16)
    # o_hat: a weight at half a quantum may round either way (a quantum is the tile's largest weight over 127); the others as there
    quantum = float((np.exp(sc - m[..., None]) * iz[..., None]).max()) * float(np.abs(vs).max()) / 127 * 8
    for g, w, tol in zip(got, want, (3e-6 + 2 * quantum, 3e-6, 3e-6)):
        np.testing.assert_allclose(g.cpu().numpy(), w, atol=tol, rtol=2e-5)


@pytest.mark.parametrize("code", ["lowest", "highest"])
@pytest.mark.parametrize("G", [1, 4, 8])
@pytest.mark.parametrize("scheme,kb,vb,gs", [("k3v2", 3, 2, 64), ("k3v3", 3, 3, 64), ("k4v4", 4, 4, 128), ("b4v4", 4, 4, 64)])
def test_longest_splits_of_equal_weights_and_codes(scheme, kb, vb, gs, G, code):
    """Equal scores and scales that are powers of two: every weight is the largest and its two lower limbs are -128 each, every
    code the largest there is, so the accumulator sums of the longest split reach the end of their range."""
    from jetfire_amd import _lib
    S, Hkv, K = 8192, 2, 64
    c = make_case(102, 1, G * Hkv, Hkv, S, kb, vb, gs, lens=[S])
    top = (1 << vb) - 1 if code == "highest" else 0
    c["q"] = np.zeros_like(c["q"])
    c["vd"] = np.broadcast_to(O.pack_codes(np.full(128, top), vb), c["vd"].shape).copy()
    c["vs"] = np.full_like(c["vs"], _bits([0.25])[0])
    d = to_device(c)
    _lib.check(_lib.debug_hook("jf_debug_split_len")(4096 if G <= 4 else 2048))
    try:
        out = [t.cpu().numpy() for t in run_fused(scheme, c, d, S, K)]
    finally:
        _lib.check(_lib.debug_hook("jf_debug_split_len")(0))
    value = 0.25 * (top - O.offset(vb))
    assert np.abs(out[0] - value).max() <= 3e-6 * abs(value)
    assert np.abs(out[2] - value * K / S).max() <= 3e-6 * abs(value) * K / S
    assert np.array_equal(out[4][0], np.broadcast_to(np.arange(K), out[4][0].shape))


@pytest.mark.parametrize("scheme,kb,vb,gs,S,K,split_len", [
    ("k3v2", 3, 2, 64, 700, 64, 256), ("k4v4", 4, 4, 128, 700, 256, 256), ("b4v4", 4, 4, 64, 1500, 512, 768),    # 256 threads a row
    ("k3v3", 3, 3, 64, 1200, 512, 512),                                                # ... with two turns of winners at once
    ("k3v2", 3, 2, 64, 2040, 1024, 256), ("k4v4", 4, 4, 128, 1111, 1024, 512),         # 512 threads
    ("k3v2", 3, 2, 64, 8192, 2048, 2048), ("k3v3", 3, 3, 128, 6000, 64, 256),          # ... as many candidates as they hold; few winners
    ("k4v4", 4, 4, 128, 9000, 2048, 2048),                                             # beyond: 32 candidates per thread
])
def test_shapes_of_the_merge_give_the_same_bits(scheme, kb, vb, gs, S, K, split_len):
    """More rows than compute units, whose merge has fewer wavefronts per row, and the same rows a few at a time."""
    from jetfire_amd import _lib, ops
    G, Hkv, B = 8, 4, 10            # 320 rows, and 96 or fewer
    c = make_case(103, B, G * Hkv, Hkv, S, kb, vb, gs, lens=[max(1, S - 97 * b * b) for b in range(B)])
    d = to_device(c)
    _lib.check(_lib.debug_hook("jf_debug_split_len")(split_len))
    try:
        whole = [t.clone() for t in run_fused(scheme, c, d, S, K)]
        for lo in range(0, B, 3):
            at = slice(lo, min(B, lo + 3))
            part = ops.fused_attn_topk(scheme, d["q"][at].contiguous(), d["kd"], d["ks"], d["vd"], d["vs"], d["bt"][at].contiguous(),
                                       d["lens"][at].contiguous(), S, G * Hkv, Hkv, 16, K, 128 ** -0.5, return_scores=True,
                                       return_stats=True)
            for a, b in zip(whole, part):
                assert torch.equal(a[at], b)
    finally:
        _lib.check(_lib.debug_hook("jf_debug_split_len")(0))
