// Sixteen-lane row quantisers shared by the quantise-on-append kernels (quant_write.hip, shadow_write.hip): lane l of
// sixteen holds channels 8l .. 8l+7 of one (token, kv-head) row, group maxima are DPP reductions inside the 16-lane
// row, and the packed row leaves as dword stores that are contiguous across the lanes.
#pragma once
#include "common.h"

namespace jf {
namespace {

struct RowDst {
  uint8_t* data;            // cache base
  int64_t data_stride_h;    // bytes
  int64_t data_stride_slot; // bytes
  uint16_t* scale;
  int64_t scale_stride_h;   // elements
  int64_t scale_stride_slot;
};
struct RowSrc {
  const uint16_t* x;
  int64_t stride_t, stride_h;  // elements
};

template <int CTRL>
__device__ inline uint32_t dpp_u32(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ inline float dpp_f32(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}

__device__ inline void widen8(const uint4& raw, float (&x)[8]) {
  x[0] = bf16_to_f32((uint16_t)(raw.x & 0xffffu)); x[1] = bf16_to_f32((uint16_t)(raw.x >> 16));
  x[2] = bf16_to_f32((uint16_t)(raw.y & 0xffffu)); x[3] = bf16_to_f32((uint16_t)(raw.y >> 16));
  x[4] = bf16_to_f32((uint16_t)(raw.z & 0xffffu)); x[5] = bf16_to_f32((uint16_t)(raw.z >> 16));
  x[6] = bf16_to_f32((uint16_t)(raw.w & 0xffffu)); x[7] = bf16_to_f32((uint16_t)(raw.w >> 16));
}

// Symmetric INT2 / INT3 / INT4.  `slot` is the row of kv-head h; rows that are not `live` take part in the cross-lane
// steps and store nothing.  (Per-thread products are 32 x 32 -> 64 multiply-adds: the launchers take these functions only
// when the strides fit 32 bits.)
template <int NBITS>
__device__ inline void quant16_row(const uint4& raw, const RowDst& d, int h, uint32_t slot, bool live, int l16, int group_size) {
  constexpr int QMAX = (1 << (NBITS - 1)) - 1;
  constexpr int OFF = 1 << (NBITS - 1);
  float x[8];
  widen8(raw, x);
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) amax = fmaxf(amax, fabsf(x[i]));
  // all-reduce over the lanes of one scale group: 4, 8 or 16 lanes
  amax = fmaxf(amax, dpp_f32<0xB1>(amax));   // quad_perm [1,0,3,2]
  amax = fmaxf(amax, dpp_f32<0x4E>(amax));   // quad_perm [2,3,0,1]
  if (group_size >= 64) amax = fmaxf(amax, dpp_f32<0x141>(amax));   // row_half_mirror: lane i <-> 7 - i
  if (group_size >= 128) amax = fmaxf(amax, dpp_f32<0x140>(amax));  // row_mirror: lane i <-> 15 - i
  // scale = bf16(max(amax / QMAX, 1e-8)).  amax is a bf16 value M * 2^e with an 8-bit M, so the exact quotient by 3
  // or 7 is either an 8-bit value itself or has a binary tail of k/3 (k/7) of the unit it is cut at: at least 1/6
  // (1/14) of a bf16 ulp away from every bf16 rounding boundary.  The product with the fp32 reciprocal is within one
  // fp32 ulp of the quotient, i.e. rounds to the same bf16 value as the correctly rounded division (the floor 1e-8
  // is not within an fp32 ulp of a boundary either); checked for every mantissa by the tests.
  constexpr float RQ = 1.0f / (float)QMAX;
  const float sraw = fmaxf(amax * RQ, 1e-8f);
  const uint16_t sb = f32_to_bf16(sraw);
  const float sf = bf16_to_f32(sb);
  // code = clamp(rint(x / sf)).  x and sf are bf16 values (8 significant bits each), so the exact quotient is
  // either exactly a half-integer or at least 1/2040 away from one (for |q| >= 1/2): rint of the fp32-rounded
  // quotient equals rint of ANY value within a few ulp of the exact quotient, provided exact half-integers come
  // out exact.  q0 = x * rcp(sf) is within 2 ulp; one correction with the exact residual r = x - sf * q0 (an
  // fma) gives the exact quotient up to ~2^-45 relative, which rounds to the half-integer itself in a tie.
  // One reciprocal per lane replaces eight correctly rounded divisions.  The clamp comes before the rounding (the
  // bounds are integers: same result), and the rounding is the addition of 2^23 + OFF: the sum lies in
  // [2^23 + 1, 2^23 + 2 OFF - 1], where floats are the integers, so the addition rounds to nearest-even like rint
  // and leaves code = rint(q) + OFF in the low bits of the sum's pattern 0x4B000000 | code.  The pattern's own bits
  // start at bit 24: the packing below shifts and merges the patterns as they are and only ever keeps bits that
  // the codes alone reach.
  const float ry = __builtin_amdgcn_rcpf(sf);
  uint32_t c[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float q0 = x[i] * ry;
    const float q = __builtin_fmaf(__builtin_fmaf(-sf, q0, x[i]), ry, q0);
    const float qc = fminf(fmaxf(q, (float)-QMAX), (float)QMAX);
    c[i] = __builtin_bit_cast(uint32_t, qc + (8388608.0f + (float)OFF));
  }
  const uint64_t so = (uint64_t)slot;
  uint8_t* drow = d.data + (int64_t)h * d.data_stride_h + so * (uint32_t)d.data_stride_slot;
  uint16_t* srow = d.scale + (int64_t)h * d.scale_stride_h + so * (uint32_t)d.scale_stride_slot;
  const int lpg = group_size >> 3;  // lanes per scale group: 4, 8 or 16
  const int lpg_shift = (group_size >= 128) ? 4 : ((group_size >= 64) ? 3 : 2);
  if (live && (l16 & (lpg - 1)) == 0) srow[l16 >> lpg_shift] = sb;
  if (NBITS == 4) {
    // byte j of the lane's dword = (c[2j] << 4) | c[2j+1]: the low byte of each merged pair (v_perm_b32 gathers them)
    const uint32_t p0 = (c[0] << 4) | c[1], p1 = (c[2] << 4) | c[3], p2 = (c[4] << 4) | c[5], p3 = (c[6] << 4) | c[7];
    const uint32_t v = __builtin_amdgcn_perm(p1, p0, 0x0c0c0400u) | __builtin_amdgcn_perm(p3, p2, 0x04000c0cu);
    if (live) reinterpret_cast<uint32_t*>(drow)[l16] = v;
  } else if (NBITS == 2) {
    // the lane's 8 codes are two bytes, four codes each MSB first (the low bytes of the two merged quadruples);
    // lane pairs share a dword
    const uint32_t pa = (c[0] << 6) | (c[1] << 4) | (c[2] << 2) | c[3], pb = (c[4] << 6) | (c[5] << 4) | (c[6] << 2) | c[7];
    const uint32_t hw = __builtin_amdgcn_perm(pb, pa, 0x0c0c0400u);
    const uint32_t nb = dpp_u32<0xB1>(hw);  // neighbour inside the lane pair
    if (live && (l16 & 1) == 0) reinterpret_cast<uint32_t*>(drow)[l16 >> 1] = hw | (nb << 16);
  } else {
    // INT3 planar: the lane's 8 codes are the 24-bit word l16, MSB first (bits 0..23 of w; what lies above is the
    // patterns' own bits and is never extracted); plane p holds byte p of every word.
    // Lane (4j + p), p < 3, assembles dword j of plane p from the four words of its quad.
    const uint32_t w = (c[0] << 21) | (c[1] << 18) | (c[2] << 15) | (c[3] << 12) | (c[4] << 9) | (c[5] << 6) | (c[6] << 3) | c[7];
    const uint32_t w0 = dpp_u32<0x00>(w), w1 = dpp_u32<0x55>(w), w2 = dpp_u32<0xAA>(w), w3 = dpp_u32<0xFF>(w);  // quad broadcasts
    const int pl = l16 & 3;
    const int sh = 16 - 8 * pl;
    const uint32_t v = ((w0 >> sh) & 255u) | (((w1 >> sh) & 255u) << 8) | (((w2 >> sh) & 255u) << 16) | (((w3 >> sh) & 255u) << 24);
    if (live && pl < 3) reinterpret_cast<uint32_t*>(drow)[4 * pl + (l16 >> 2)] = v;
  }
}

// Asymmetric INT2 keys over the full codebook (jetfire_vllm/kernels/intN_pack.py:110-169,
// fused_quant_write.py:85-133): per group scale = bf16(max((xmax - xmin) / 3, 1e-8)),
// zp = bf16(xmin + 2 * scale_f32), code = clamp(rint((x - zp) / scale), -2, 1) + 2.  The divisions are IEEE divisions:
// the numerator x - zp is not a bf16 value, so the reciprocal shortcut of the symmetric kernel does not apply.
__device__ inline void quant16_row_int2_asym(const uint4& raw, const RowDst& d, uint16_t* zp_out, int64_t zp_stride_h,
                                             int64_t zp_stride_slot, int h, int64_t slot, bool live, int l16, int group_size) {
  float x[8];
  widen8(raw, x);
  float xmax = x[0], xmin = x[0];
#pragma unroll
  for (int i = 1; i < 8; ++i) {
    xmax = fmaxf(xmax, x[i]);
    xmin = fminf(xmin, x[i]);
  }
  xmax = fmaxf(xmax, dpp_f32<0xB1>(xmax)); xmin = fminf(xmin, dpp_f32<0xB1>(xmin));
  xmax = fmaxf(xmax, dpp_f32<0x4E>(xmax)); xmin = fminf(xmin, dpp_f32<0x4E>(xmin));
  if (group_size >= 64) { xmax = fmaxf(xmax, dpp_f32<0x141>(xmax)); xmin = fminf(xmin, dpp_f32<0x141>(xmin)); }
  if (group_size >= 128) { xmax = fmaxf(xmax, dpp_f32<0x140>(xmax)); xmin = fminf(xmin, dpp_f32<0x140>(xmin)); }
  const float sraw = fmaxf((xmax - xmin) / 3.0f, 1e-8f);
  const float zraw = xmin + 2.0f * sraw;
  const uint16_t sb = f32_to_bf16(sraw), zb = f32_to_bf16(zraw);
  const float sf = bf16_to_f32(sb), zf = bf16_to_f32(zb);
  uint32_t c[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) c[i] = (uint32_t)((int)fminf(fmaxf(rintf((x[i] - zf) / sf), -2.0f), 1.0f) + 2);
  const int64_t so = (int64_t)slot;
  uint8_t* drow = d.data + (int64_t)h * d.data_stride_h + so * d.data_stride_slot;
  const int lpg = group_size >> 3;
  if (live && (l16 & (lpg - 1)) == 0) {
    d.scale[(int64_t)h * d.scale_stride_h + so * d.scale_stride_slot + l16 / lpg] = sb;
    zp_out[(int64_t)h * zp_stride_h + so * zp_stride_slot + l16 / lpg] = zb;
  }
  const uint32_t hw = ((c[0] << 6) | (c[1] << 4) | (c[2] << 2) | c[3]) | (((c[4] << 6) | (c[5] << 4) | (c[6] << 2) | c[7]) << 8);
  const uint32_t nb = dpp_u32<0xB1>(hw);
  if (live && (l16 & 1) == 0) reinterpret_cast<uint32_t*>(drow)[l16 >> 1] = hw | (nb << 16);
}

inline bool rows_16b_aligned(const void* x, int64_t stride_t, int64_t stride_h) {
  return ((uintptr_t)x & 15) == 0 && stride_t % 8 == 0 && stride_h % 8 == 0;
}
// what quant16_row multiplies per thread with 32-bit operands
inline bool strides_fit_32(int64_t x_stride_t, int64_t data_stride_slot, int64_t scale_stride_slot) {
  const int64_t lim = (int64_t)1 << 32;
  return x_stride_t >= 0 && x_stride_t < lim && data_stride_slot >= 0 && data_stride_slot < lim &&
         scale_stride_slot >= 0 && scale_stride_slot < lim;
}

}  // namespace
}  // namespace jf
