"""The int8-tile-quantised Stage B (jf_softmax_v_int8_tiles) where its tiles can go wrong: single positions, tiles and
pages cut by the eight ranges, every head-set size, unused pages of the table, a value tensor that starts at a dword."""
import numpy as np
import pytest
import torch

from oracle import jetfire_oracle as O
from tests.helpers import make_case, to_device

pytestmark = pytest.mark.gpu


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
    # 3e-6, the bound of the other tests of this form.  A weight whose quotient lies within the exponential's last bits
    # of a half may round either way: one quantum (at most iz * max scale / 127) times a code (at most 8) in one row's
    # elements.  Two of those per row, in at most one element of fifty.
    quantum = iz[..., None] * float(d["vs"].float().max()) / 127 * 8
    for i, (g, w) in enumerate(zip(got, want)):
        diff = np.abs(g.cpu().numpy() - w) - 2e-5 * np.abs(w)
        if i == 0:
            assert (diff <= 3e-6 + 2 * quantum).all() and (diff > 3e-6).mean() <= 0.02
        else:
            assert diff.max() <= 3e-6
