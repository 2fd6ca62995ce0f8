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
