"""The int8-tile-quantised Stage B (jf_softmax_v_int8_tiles) where its tiles can go wrong: single positions, tiles and
pages cut by the eight ranges, every head-set size, unused pages of the table, a value tensor that starts at a dword."""
import numpy as np
import pytest
import torch

from oracle import jetfire_oracle as O
from tests.helpers import make_case, to_device

pytestmark = pytest.mark.gpu


def _either_way(sc, m, iz, c, S, Hq, Hkv):
    """Per element of o_hat, the sum of quantum * |code| over the weights whose quotient is a half to within 4e-6 of its
    size: the weight is an exponential of up to 20, whose argument's last bit is 20 * 2^-24 of it, times two factors.
    And the share of such weights among all."""
    codes = np.abs(O.decode_codes(c["vd"], 4).astype(np.int64) - 8)
    vs = O.bf16_bits_to_f32(c["vs"])[..., 0]
    slots = O.slots_from_block_table(c["bt"], S, 16)
    extra, near, total = np.zeros((c["B"], Hq, 128), np.float32), 0, 0
    chunk = (S + 7) // 8
    for b in range(c["B"]):
        n = int(c["lens"][b])
        for h in range(Hq):
            hk = h // (Hq // Hkv)
            pv = np.exp(sc[b, h, :n].astype(np.float64) - m[b, h]) * iz[b, h] * vs[hk, slots[b, :n]]
            for s0 in range(0, n, chunk):
                for t in range(s0 // 16 * 16, min(s0 + chunk, n), 32):
                    at = slice(max(t, s0), min(t + 32, s0 + chunk, n))
                    rs = np.abs(pv[at]).max() / 127
                    if rs > 0:
                        q = np.abs(pv[at]) / rs
                        half = np.abs(q - np.floor(q) - 0.5) <= 4e-6 * q
                        near, total = near + int(half.sum()), total + len(q)
                        extra[b, h] += rs * codes[hk, slots[b, at]][half].sum(axis=0)
    return extra, near / max(1, total)


@pytest.mark.parametrize("Hq,Hkv,S,lens,K", [
    (4, 4, 1, [1], 32),
    (6, 2, 31, [31, 0, 5], 32),
    (8, 2, 130, [130, 129, 17], 64),
    (7, 1, 777, [777, 300], 128),
    (16, 2, 2000, [2000, 1999, 64], 256),
    (16, 1, 2600, [2600, 33], 64),
    (12, 1, 5000, [5000, 4097], 64),
    (8, 2, 9000, [9000, 100, 8999], 4096),      # wider than the merge kernel takes: the combine kernel
])
@pytest.mark.parametrize("shifted", [False, True])
def test_int8_tiles_match_the_tile_model(Hq, Hkv, S, lens, K, shifted):
    from jetfire_amd import ops
    c = make_case(17, len(lens), Hq, Hkv, S, 4, 4, 128, lens=lens, extra_blocks=3)
    d = to_device(c)
    sc = O.scores_int8_model(c["q"], c["kd"], c["ks"], c["bt"], c["lens"], S, Hq, Hkv, 16, 128 ** -0.5)
    idx, _ = O.topk_select(sc, c["lens"], c["bt"], S, K)
    m, iz = O.softmax_stats(sc, c["lens"], S)
    vd = d["vd"]
    if shifted:      # the same bytes four further on: rows no longer start at 16-byte boundaries
        store = torch.empty(vd.numel() + 4, dtype=torch.uint8, device="cuda")
        vd = store[4:].view(vd.shape).copy_(vd)
    got = ops.int8tc_softmax_v_with_pre_corr_reg_stats(
        torch.from_numpy(sc).cuda(), torch.from_numpy(m).cuda(), torch.from_numpy(iz).cuda(), vd, d["vs"], d["bt"], d["lens"],
        torch.from_numpy(idx).cuda(), S, Hq, Hkv, 16, K)
    want = O.softmax_v_int8_tiles(sc, m, iz, c["vd"], c["vs"], c["bt"], c["lens"], idx, S, Hq, Hkv, 16)
    # 3e-6, the bound of the other tests of this form, and what the weights may add whose quotient lies within the
    # exponential's error of a half: those, and only those, may round either way, by one quantum times their code
    may_differ, share = _either_way(sc, m, iz, c, S, Hq, Hkv)
    assert share <= 1e-3
    for i, (g, w) in enumerate(zip(got, want)):
        diff = np.abs(g.cpu().numpy() - w) - 2e-5 * np.abs(w)
        assert (diff <= 3e-6 + (may_differ if i == 0 else 0)).all()
