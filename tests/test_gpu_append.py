"""The one-launch append (jf_append_rows) through the cache store against the oracle's quantiser: cache bytes, scales,
filled marks and the host mirror, at token counts around the 16-token blocks."""
import numpy as np
import pytest
import torch

from oracle import jetfire_oracle as O
from tests.helpers import bf16_tensor, bf16_to_bits, bf16_to_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kb,vb,asym,gs", [(3, 2, False, 64), (4, 4, False, 128), (2, 3, True, 64), (2, 4, False, 32)])
@pytest.mark.parametrize("T", [1, 15, 16, 17, 130])
def test_store_append_matches_the_oracle(T, kb, vb, asym, gs):
    from jetfire_amd.adapter.cache_store import JetFireInt4CacheStore
    H, nblk = 3, (T + 15) // 16 + 2
    rng = np.random.default_rng(T * 10 + kb)
    store = JetFireInt4CacheStore(num_kv_heads=H, head_dim=128, group_size=gs, num_blocks=nblk, block_size=16, device="cuda",
                                  k_nbits=kb, v_nbits=vb, k_asymmetric=asym)
    x = [O.bf16_round(rng.standard_normal((T, H, 128)).astype(np.float32)) for _ in range(2)]
    slots = rng.permutation(nblk * 16)[:T].astype(np.int64)
    if T > 1:
        slots[T // 2] = -1                       # padding
    if T > 16:
        slots[3] = nblk * 16 + 5                 # outside the cache: skipped like padding
    live = (slots >= 0) & (slots < nblk * 16)
    # (values as every second row of a wider tensor: the strides of a fused QKV projection)
    wide = torch.stack([bf16_tensor(x[1])] * 2, dim=2).cuda()
    store.write_slots(key=bf16_tensor(x[0]).cuda(), value=wide[:, :, 1], slot_mapping=torch.from_numpy(slots).cuda())
    store.flush_pending_writes()
    torch.cuda.synchronize()
    filled = np.zeros(nblk * 16, bool)
    filled[slots[live]] = True
    assert np.array_equal(store.slot_filled.cpu().numpy(), filled)
    quant = [O.quantize_and_pack_asym(x[0], gs, kb) if asym else O.quantize_and_pack(x[0], gs, kb), O.quantize_and_pack(x[1], gs, vb)]
    for q, data, scales, shadow, rows in ((quant[0], store.k_data, store.k_scales, store.k_shadow, x[0]),
                                          (quant[1], store.v_data, store.v_scales, store.v_shadow, x[1])):
        want = np.zeros(data.shape, np.uint8)
        want[:, slots[live]] = q[0][live].transpose(1, 0, 2)
        assert np.array_equal(data.cpu().numpy(), want)
        want_s = np.zeros(scales.shape, np.uint16)
        want_s[:, slots[live]] = q[1][live].transpose(1, 0, 2)
        assert np.array_equal(bf16_to_bits(scales), want_s)
        mirror = np.zeros(shadow.shape, np.float32)
        mirror[:, slots[live]] = rows[live].transpose(1, 0, 2)
        assert np.array_equal(bf16_to_f32(shadow), mirror)
    if asym:
        want_z = np.zeros(store.k_zp.shape, np.uint16)
        want_z[:, slots[live]] = quant[0][2][live].transpose(1, 0, 2)
        assert np.array_equal(bf16_to_bits(store.k_zp), want_z)


def test_store_append_of_unaligned_rows_takes_the_separate_operators():
    from jetfire_amd.adapter.cache_store import JetFireInt4CacheStore
    rng = np.random.default_rng(5)
    a, b = (JetFireInt4CacheStore(num_kv_heads=2, head_dim=128, group_size=64, num_blocks=4, block_size=16, device="cuda",
                                  k_nbits=3, v_nbits=2) for _ in range(2))
    k, v = (bf16_tensor(O.bf16_round(rng.standard_normal((20, 2, 128)).astype(np.float32))).cuda() for _ in range(2))
    slots = torch.arange(40, 60, device="cuda")
    shifted = torch.empty(20 * 2 * 128 + 2, dtype=torch.bfloat16, device="cuda")[2:].view(20, 2, 128)   # 4-byte aligned rows
    shifted.copy_(k)
    a.write_slots(key=shifted, value=v, slot_mapping=slots)
    b.write_slots(key=k, value=v, slot_mapping=slots)
    torch.cuda.synchronize()
    for x, y in ((a.k_data, b.k_data), (a.k_scales, b.k_scales), (a.v_data, b.v_data), (a.v_scales, b.v_scales),
                 (a.slot_filled, b.slot_filled), (a.k_shadow, b.k_shadow), (a.v_shadow, b.v_shadow)):
        assert torch.equal(x, y)


@pytest.mark.parametrize("kb,vb,asym,gs", [(3, 2, False, 64), (4, 4, False, 128), (2, 3, True, 64), (2, 4, False, 32)])
@pytest.mark.parametrize("aligned", [True, False])
def test_slots_beyond_the_cache_are_skipped_by_every_writer(aligned, kb, vb, asym, gs):
    """The same call does the same whatever the alignment of its token rows: slots past the end of the cache (and of its
    filled marks and shadow) are dropped like padding.  `store` appends them among valid ones, `want` without them."""
    from jetfire_amd import ops
    from jetfire_amd.adapter.cache_store import JetFireInt4CacheStore
    H, nblk, T = 2, 4, 40
    rng = np.random.default_rng(kb * 10 + vb)
    store, want = (JetFireInt4CacheStore(num_kv_heads=H, head_dim=128, group_size=gs, num_blocks=nblk, block_size=16,
                                         device="cuda", k_nbits=kb, v_nbits=vb, k_asymmetric=asym) for _ in range(2))
    x = [bf16_tensor(O.bf16_round(rng.standard_normal((T, H, 128)).astype(np.float32))).cuda() for _ in range(2)]
    slots = rng.permutation(nblk * 16)[:T].astype(np.int64)
    slots[[0, 7, 16, 31]] = [nblk * 16, nblk * 16 + 3, 2**32 + 5, -1]
    keep = torch.from_numpy(np.flatnonzero((slots >= 0) & (slots < nblk * 16))).cuda()
    slots = torch.from_numpy(slots).cuda()
    rows = list(x)
    if not aligned:      # rows that start at dwords (asymmetric keys have no writer for those: the values only)
        for i in range(1 if asym else 0, 2):
            rows[i] = torch.empty(T * H * 128 + 2, dtype=torch.bfloat16, device="cuda")[2:].view(T, H, 128).copy_(x[i])
    store.write_slots(key=rows[0], value=rows[1], slot_mapping=slots)
    want.write_slots(key=x[0][keep], value=x[1][keep], slot_mapping=slots[keep])
    torch.cuda.synchronize()
    names = ["k_data", "k_scales", "v_data", "v_scales", "slot_filled", "k_shadow", "v_shadow"] + (["k_zp"] if asym else [])
    for name in names:
        assert torch.equal(getattr(store, name), getattr(want, name)), name
    # the writers called one by one, on caches that are the front part of larger ones
    for name, tok, bits in (("fused_quant_write_int2_sym", rows[1], 2), ("fused_quant_write_int3_sym", rows[1], 3),
                            ("fused_quant_write_int4_sym", rows[1], 4)):
        data = torch.zeros(H, nblk * 32, 16 * bits, dtype=torch.uint8, device="cuda")
        scales = torch.zeros(H, nblk * 32, 128 // gs, dtype=torch.bfloat16, device="cuda")
        getattr(ops, name)(tok, slots, data[:, :nblk * 16], scales[:, :nblk * 16], gs)
        assert not data[:, nblk * 16:].any() and not scales[:, nblk * 16:].any()
        assert torch.equal(scales[0, :nblk * 16, 0] != 0, want.slot_filled)


def test_append_refuses_zero_points_whose_groups_do_not_lie_side_by_side():
    """The kernel stores a row's zero-points next to each other, as the separate writer checks they are."""
    from jetfire_amd import ops
    T, H, S = 4, 2, 32
    tok = torch.zeros(T, H, 128, dtype=torch.bfloat16, device="cuda")
    data = [torch.zeros(H, S, 32, dtype=torch.uint8, device="cuda") for _ in range(2)]
    scales = [torch.zeros(H, S, 2, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    zp = torch.zeros(H, S, 4, dtype=torch.bfloat16, device="cuda")[:, :, ::2]
    slots = torch.arange(T, device="cuda")
    for call in (lambda: ops.append_rows(tok, tok, slots, data[0], scales[0], zp, data[1], scales[1], 64, 2, 2),
                 lambda: ops.fused_quant_write_int2_asym(tok, slots, data[0], scales[0], zp, 64)):
        with pytest.raises(RuntimeError):
            call()
