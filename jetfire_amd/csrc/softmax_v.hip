// Stage B in its split form: consumes an fp32 score tensor and produces o_hat, o_old_unnorm, W.
//
//   w_s   = exp(score_s - m) * inv_z                (jetfire_vllm/csrc/int4_softmax_v.cu:162-176)
//   ws    = w_s * f32(v_scale[s, group(d)])         (jetfire_vllm/csrc/int2_softmax_v.cu:681-694)
//   o_hat[d] = sum_s fma(ws, code[s, d] - offset)   (:696-706), positions in ascending order
//   o_old_unnorm / W: the same sums over the top-k positions only (:738-788)
//
// Three launches: row statistics (only when the caller has none), a split-S weighted-V pass in which
// one workgroup owns a (sequence, kv-head, S-range) and serves all G query heads from one read of V,
// and a combine pass that adds the split partials in ascending order (deterministic, no atomics) and
// does the top-k pre-correction.
#include "common.h"

namespace jf {
namespace {

constexpr int SV_THREADS = 128;

__device__ inline float block_max_128(float v, float* red) {
  v = wave_max(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return fmaxf(red[0], red[1]);
}
__device__ inline float block_sum_128(float v, float* red) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return red[0] + red[1];
}

__global__ __launch_bounds__(SV_THREADS) void softmax_stats_kernel(const float* __restrict__ scores,
                                                                   const int32_t* __restrict__ seq_lens,
                                                                   float* __restrict__ m_out, float* __restrict__ iz_out,
                                                                   int max_S, int H_q) {
  __shared__ float red[2];
  const int b = blockIdx.x, hq = blockIdx.y, tid = threadIdx.x;
  const size_t bh = (size_t)b * H_q + hq;
  const int n = max(0, min(max_S, seq_lens[b]));
  const float* row = scores + bh * (size_t)max_S;
  float lm = -INFINITY;
  for (int i = tid; i < n; i += SV_THREADS) lm = fmaxf(lm, row[i]);
  float m = block_max_128(lm, red);
  if (!isfinite(m)) m = 0.0f;
  float ls = 0.0f;
  for (int i = tid; i < n; i += SV_THREADS) ls += __expf(row[i] - m);
  const float z = block_sum_128(ls, red);
  if (tid == 0) {
    m_out[bh] = m;
    iz_out[bh] = (z > 0.0f) ? (1.0f / z) : 0.0f;
  }
}

template <int NBITS>
__device__ inline int v_code(const uint8_t* row, int d) {
  if (NBITS == 2) return (int)((row[d >> 2] >> ((3 - (d & 3)) * 2)) & 3) - 2;
  if (NBITS == 3) {  // planar: codes 8w .. 8w+7 are the 24-bit word whose bytes sit at w, 16 + w, 32 + w (MSB first)
    const int w = d >> 3;
    const uint32_t word = ((uint32_t)row[w] << 16) | ((uint32_t)row[16 + w] << 8) | (uint32_t)row[32 + w];
    return (int)((word >> (21 - 3 * (d & 7))) & 7u) - 4;
  }
  return (int)((row[d >> 1] >> ((1 - (d & 1)) * 4)) & 15) - 8;
}

// grid (n_splits, H_kv, B); thread = output channel d; acc[g] for the G query heads of this kv-head.
template <int NBITS, int G, int NG>
__global__ __launch_bounds__(SV_THREADS) void weighted_v_split_kernel(
    const float* __restrict__ scores, const float* __restrict__ softmax_m, const float* __restrict__ softmax_inv_z,
    const uint8_t* __restrict__ v_data, const uint16_t* __restrict__ v_scales, const int64_t* __restrict__ block_table,
    const int32_t* __restrict__ seq_lens, float* __restrict__ partial, int H_q, int H_kv, int max_S, int max_blocks,
    int64_t num_slots, int chunk, int n_splits, int ga) {
  // ga: the query heads that belong to a kv-head; G is ga rounded up to a kernel size, the heads past ga carry no weight
  constexpr int P = D * NBITS / 8;
  __shared__ __align__(16) uint8_t vbuf[BS * P];
  __shared__ float wsbuf[G][BS][NG];
  const int split = blockIdx.x, hkv = blockIdx.y, b = blockIdx.z, tid = threadIdx.x;
  const int S = max(0, min(max_S, seq_lens[b]));
  const int s0 = split * chunk, s1 = min(s0 + chunk, S);
  float acc[G];
#pragma unroll
  for (int g = 0; g < G; ++g) acc[g] = 0.0f;
  const int grp = (NG == 1) ? 0 : (tid / (D / NG));
  const uint8_t* vbase = v_data + (size_t)hkv * num_slots * P;
  const uint16_t* sbase = v_scales + (size_t)hkv * num_slots * NG;
  const int64_t* bt = block_table + (size_t)b * max_blocks;
  for (int p0 = s0; p0 < s1; p0 += BS) {  // chunk is a multiple of BS, so pages are aligned
    const int64_t base_slot = bt[p0 / BS] * BS;
    __syncthreads();
    {
      constexpr int NDW = BS * P / 4;  // dwords of a page (128, 192 or 256)
      const uint32_t* src = reinterpret_cast<const uint32_t*>(vbase + base_slot * P);
#pragma unroll
      for (int i = 0; i < (NDW + SV_THREADS - 1) / SV_THREADS; ++i)
        if (NDW % SV_THREADS == 0 || tid + i * SV_THREADS < NDW)
          reinterpret_cast<uint32_t*>(vbuf)[tid + i * SV_THREADS] = src[tid + i * SV_THREADS];
    }
    for (int i = tid; i < G * BS; i += SV_THREADS) {
      const int g = i / BS, j = i % BS;
      const int p = p0 + j;
      const size_t bh = (size_t)b * H_q + (size_t)hkv * ga + g;
      const bool live = p < s1 && g < ga;
      float w = 0.0f;
      if (live) w = __expf(scores[bh * (size_t)max_S + p] - softmax_m[bh]) * softmax_inv_z[bh];
#pragma unroll
      for (int k = 0; k < NG; ++k)
        wsbuf[g][j][k] = live ? w * bf16_to_f32(sbase[(size_t)(base_slot + j) * NG + k]) : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < BS; ++j) {
      const float c = (float)v_code<NBITS>(vbuf + j * P, tid);
#pragma unroll
      for (int g = 0; g < G; ++g) acc[g] = __builtin_fmaf(wsbuf[g][j][grp], c, acc[g]);
    }
  }
#pragma unroll
  for (int g = 0; g < G; ++g)
    if (g < ga) partial[(((size_t)b * H_q + (size_t)hkv * ga + g) * n_splits + split) * D + tid] = acc[g];
}

// INT4 values with int8-quantised weights, the arithmetic of the reference's register-MMA Stage B
// (jetfire_vllm/csrc/int8tc_softmax_v_fused.cu:1049-1052 split geometry, :1178 tile origin, :1203-1236 weight
// quantisation, :1298-1311 accumulation): the sequence is cut into TQ_SPLITS ranges of ceil(max_S / TQ_SPLITS)
// positions; a range is walked in tiles of two pages that start at the page holding its first position; per tile
// and query head
//     pv_t = exp(score_t - m) * inv_z * f32(v_scale_t)   (0 outside the range)
//     rs   = max_t |pv_t| / 127,  pq_t = clamp(rint(pv_t * (1 / rs)), -127, 127)   (rs == 0: pq = 0)
//     o_hat[d] += f32(sum_t pq_t * (nibble_t,d - 8)) * rs
// with an exact int32 sum per tile and an fp32 running sum over the tiles in ascending order.
// grid (TQ_SPLITS * sub_count, H_kv, B).  A range's tiles are dealt out in runs to `sub_count` workgroups and inside a
// run to four wavefronts (the tiles themselves, and with them every quantisation step, stay those of the reference's
// eight ranges; only the association of the fp32 sum over tiles changes, at the 1e-7 level).
// A wavefront takes two tiles (64 positions) at a time on v_mfma_i32_16x16x64_i8, contracting over the positions: lane =
// token quantises the heads' weights and stores one 16-byte row whose byte 4h + t is head h's weight if the token lies
// in tile t and 0 otherwise, so accumulator register t of lane 16h + c is tile t's exact sum for head h and column c;
// the -8 of the codes enters as the C operand (the weights against a tile of eights, negated).  V rows are fetched with
// 16-byte loads consecutive inside a page, one step ahead, staged in wavefront-private LDS with swapped quarters and
// transposed by ds_read_b64_tr_b4.  B 4, 32 / 8 heads, 8192 to 16384 positions: 12 - 14 us = 2.9 TB/s of rows, scales
// and scores (a thread per channel with scalar products took 30.7 us); a wavefront's chain of load, exponential, two
// divisions per head, LDS turn-around and MFMA bounds it, not the memory.
__device__ inline void wave_lds_order() {  // a wavefront's earlier LDS accesses before its later ones
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
constexpr int TQ_SPLITS = 8;
constexpr int TQ_TILE = 2 * BS;
constexpr int TQ_WAVES = 4;
typedef int tq_v2i __attribute__((ext_vector_type(2)));
typedef int tq_v4i __attribute__((ext_vector_type(4)));
typedef tq_v4i tq_row __attribute__((aligned(4)));  // 16 bytes of a packed row (the tensor may start at any dword)
template <int NSET>
__global__ __launch_bounds__(TQ_WAVES * 64) void tile_quantised_v_split_kernel(
    const float* __restrict__ scores, const float* __restrict__ softmax_m, const float* __restrict__ softmax_inv_z,
    const uint8_t* __restrict__ v_data, const uint16_t* __restrict__ v_scales, const int64_t* __restrict__ block_table,
    const int32_t* __restrict__ seq_lens, float* __restrict__ partial, int H_q, int H_kv, int max_S, int max_blocks,
    int64_t num_slots, int sub_count, int ga) {
  constexpr int P = D / 2, G = NSET * 4;
  constexpr int VST = 64 * P, WST = NSET * 64 * 16;
  __shared__ __align__(16) uint8_t stage[TQ_WAVES][VST + WST];
  const int range = blockIdx.x / sub_count, sub = blockIdx.x % sub_count;
  const int hkv = blockIdx.y, b = blockIdx.z, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int S = max(0, min(max_S, seq_lens[b]));
  const int len = (max_S + TQ_SPLITS - 1) / TQ_SPLITS;
  const int s_start = range * len, s_end = min(s_start + len, S);
  const uint8_t* vbase = v_data + (size_t)hkv * num_slots * P;
  const uint16_t* sbase = v_scales + (size_t)hkv * num_slots;
  const int64_t* bt = block_table + (size_t)b * max_blocks;
  const size_t head0 = (size_t)b * H_q + (size_t)hkv * ga;
  const int t_first = (s_start / BS) * BS;
  const int n_pairs = (s_end > t_first) ? (s_end - t_first + 2 * TQ_TILE - 1) / (2 * TQ_TILE) : 0;  // pairs of tiles
  const int per_sub = (n_pairs + sub_count - 1) / sub_count;
  const int p_end = min(n_pairs, (sub + 1) * per_sub);
  uint8_t* vst = stage[wave];
  uint8_t* wl = vst + VST;
  float m[G], iz[G];
#pragma unroll
  for (int h = 0; h < G; ++h) {
    m[h] = softmax_m[head0 + min(h, ga - 1)];
    iz[h] = softmax_inv_z[head0 + min(h, ga - 1)];
  }
  // everything a pair of tiles needs from memory; a page past the table or the sequence contributes zero weights and
  // its rows are not read
  struct Fetch {
    tq_v4i row[4];
    float sc[G];
    uint32_t vs;
    bool live;
  };
  auto fetch = [&](int pair) -> Fetch {
    Fetch f;
    const int t0 = t_first + pair * 2 * TQ_TILE;
    int64_t slot0[4];
#pragma unroll
    for (int pg = 0; pg < 4; ++pg) {
      const int blk = t0 / BS + pg;
      const int64_t e = (blk < max_blocks && blk * BS < s_end) ? bt[blk] : -1;
      slot0[pg] = (e >= 0 && (e + 1) * BS <= num_slots) ? e * BS : -1;
    }
#pragma unroll
    for (int pg = 0; pg < 4; ++pg) {
      f.row[pg] = (tq_v4i){0, 0, 0, 0};
      if (slot0[pg] >= 0) f.row[pg] = *reinterpret_cast<const tq_row*>(vbase + slot0[pg] * P + 16 * lane);  // (uniform)
    }
    const int pg = lane >> 4, pos = t0 + lane;
    const int64_t s0 = pg == 0 ? slot0[0] : pg == 1 ? slot0[1] : pg == 2 ? slot0[2] : slot0[3];
    f.live = pos >= s_start && pos < s_end && s0 >= 0;
    f.vs = f.live ? sbase[s0 + (lane & 15)] : 0;
#pragma unroll
    for (int h = 0; h < G; ++h) f.sc[h] = f.live ? scores[(head0 + min(h, ga - 1)) * (size_t)max_S + pos] : 0.f;
    return f;
  };
  const int r16 = lane & 15, kb4 = lane >> 4;
  const int tr_tok = (((r16 >> 1) & 3) << 1) | ((r16 >> 3) & 1);
  const uint8_t* wrow = wl + (kb4 * 16 + tr_tok) * 16 + (r16 & 1) * 8;
  const uint8_t* vrow = vst + lane * P;
  const int vx = 16 * ((lane >> 2) & 3);
  const tq_v4i minus8 = {(int)0xf8f8f8f8, (int)0xf8f8f8f8, (int)0xf8f8f8f8, (int)0xf8f8f8f8};
  float acc[NSET][8];
#pragma unroll
  for (int s = 0; s < NSET; ++s)
#pragma unroll
    for (int t = 0; t < 8; ++t) acc[s][t] = 0.f;
  int pair = sub * per_sub + wave;
  Fetch nxt = {};
  if (pair < p_end) nxt = fetch(pair);
  for (; pair < p_end; pair += TQ_WAVES) {
    const Fetch cur = nxt;
    if (pair + TQ_WAVES < p_end) nxt = fetch(pair + TQ_WAVES);
#pragma unroll
    for (int pg = 0; pg < 4; ++pg) {  // row 16 pg + lane / 4, quarter lane % 4
      const int row = 16 * pg + (lane >> 2);
      *reinterpret_cast<tq_v4i*>(vst + row * P + (((lane & 3) ^ ((row >> 2) & 3)) * 16)) = cur.row[pg];
    }
    const float vs = bf16_to_f32((uint16_t)cur.vs);
    const int shift = (lane >> 5) * 8;  // byte of the token's tile
    float rs[NSET][2];
#pragma unroll
    for (int s = 0; s < NSET; ++s) {
      tq_v4i row;
      float r0 = 0.f, r1 = 0.f;
#pragma unroll
      for (int hh = 0; hh < 4; ++hh) {
        const int h = s * 4 + hh;
        float pv = 0.0f;
        if (cur.live && h < ga) {
          const float pr = __expf(cur.sc[h] - m[h]) * iz[h];
          pv = pr * vs;
        }
        float a = fabsf(pv);  // maximum over the 32 tokens of the tile
        a = fmaxf(a, __builtin_bit_cast(float, dpp_mov<0xb1, 0xf>(0, __builtin_bit_cast(int, a))));   // lane ^ 1
        a = fmaxf(a, __builtin_bit_cast(float, dpp_mov<0x4e, 0xf>(0, __builtin_bit_cast(int, a))));   // lane ^ 2
        a = fmaxf(a, __builtin_bit_cast(float, dpp_mov<0x141, 0xf>(0, __builtin_bit_cast(int, a))));  // mirrored in 8 lanes
        a = fmaxf(a, __builtin_bit_cast(float, dpp_mov<0x140, 0xf>(0, __builtin_bit_cast(int, a))));  // mirrored in 16 lanes
        a = fmaxf(a, __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, a), 0x401F)));  // lane ^ 16
        const float row_scale = a / 127.0f;
        const float inv_scale = (row_scale > 0.0f) ? (1.0f / row_scale) : 0.0f;
        int qv = (int)rintf(pv * inv_scale);
        qv = max(-127, min(127, qv));
        row[hh] = (qv & 0xff) << shift;
        const float lo = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, row_scale), 0));
        const float hi = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, row_scale), 32));
        r0 = (kb4 == hh) ? lo : r0;
        r1 = (kb4 == hh) ? hi : r1;
      }
      rs[s][0] = r0;
      rs[s][1] = r1;
      *reinterpret_cast<tq_v4i*>(wl + (s * 64 + lane) * 16) = row;
    }
    wave_lds_order();
    tq_v4i A[NSET], C[NSET];
#pragma unroll
    for (int s = 0; s < NSET; ++s) {
      const uint8_t* src = wrow + s * 1024;
      const tq_v2i x0 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) tq_v2i*)(src));
      const tq_v2i x1 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) tq_v2i*)(src + 128));
      A[s] = (tq_v4i){x0[0], x0[1], x1[0], x1[1]};
      C[s] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[s], minus8, (tq_v4i){0, 0, 0, 0}, 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const tq_v2i x = __builtin_amdgcn_ds_read_tr4_b64_v2i32((__attribute__((address_space(3))) tq_v2i*)(vrow + ((8 * t) ^ vx)));
      const uint32_t x0 = (uint32_t)x[0], x1 = (uint32_t)x[1];
      const tq_v4i Bv = {(int)(x0 & 0x0f0f0f0fu), (int)((x0 >> 4) & 0x0f0f0f0fu),
                         (int)(x1 & 0x0f0f0f0fu), (int)((x1 >> 4) & 0x0f0f0f0fu)};
#pragma unroll
      for (int s = 0; s < NSET; ++s) {
        const tq_v4i dot = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[s], Bv, C[s], 0, 0, 0);
        acc[s][t] = __builtin_fmaf((float)dot[0], rs[s][0], acc[s][t]);
        acc[s][t] = __builtin_fmaf((float)dot[1], rs[s][1], acc[s][t]);
      }
    }
    wave_lds_order();
  }
  // the wavefronts' sums, in wavefront order: one head set at a time through LDS
  float* red = reinterpret_cast<float*>(&stage[0][0]);  // [TQ_WAVES][8][64]
  static_assert(sizeof(stage) >= TQ_WAVES * 8 * 64 * 4, "the final sums fit the staging areas");
#pragma unroll
  for (int s = 0; s < NSET; ++s) {
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 8; ++t) red[(wave * 8 + t) * 64 + lane] = acc[s][t];
    __syncthreads();
    for (int i = tid; i < 8 * 64; i += TQ_WAVES * 64) {
      float o = 0.f;
#pragma unroll
      for (int w = 0; w < TQ_WAVES; ++w) o += red[w * 512 + i];
      const int t = i >> 6, h = s * 4 + ((i >> 4) & 3), c = i & 15;
      const int d = t * 16 + 2 * (c >> 1) + (1 - (c & 1));
      if (h < ga) partial[((head0 + h) * (size_t)(TQ_SPLITS * sub_count) + blockIdx.x) * D + d] = o;
    }
  }
}

// grid (B, H_q); adds split partials in order, then the top-k pre-correction.
template <int NBITS, int NG>
__global__ __launch_bounds__(SV_THREADS) void combine_precorr_kernel(
    const float* __restrict__ partial, const float* __restrict__ scores, const float* __restrict__ softmax_m,
    const float* __restrict__ softmax_inv_z, const uint8_t* __restrict__ v_data, const uint16_t* __restrict__ v_scales,
    const int64_t* __restrict__ block_table, const int32_t* __restrict__ seq_lens, const int64_t* __restrict__ topk_idx,
    float* __restrict__ o_hat, float* __restrict__ o_old, float* __restrict__ W_out, int H_q, int H_kv, int max_S,
    int max_blocks, int64_t num_slots, int n_splits, int K) {
  constexpr int P = D * NBITS / 8;
  constexpr int STEP = 128;
  __shared__ int64_t slot_buf[STEP];
  __shared__ float ws_buf[STEP][NG];
  __shared__ float w_buf[STEP];
  const int b = blockIdx.x, hq = blockIdx.y, tid = threadIdx.x;
  const size_t bh = (size_t)b * H_q + hq;
  const int hkv = hq / (H_q / H_kv);
  float acc = 0.0f;
  for (int s0 = 0; s0 < n_splits; s0 += 8) {  // eight loads in flight, the sum keeps its order
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = (s0 + u < n_splits) ? partial[(bh * n_splits + s0 + u) * D + tid] : 0.0f;
#pragma unroll
    for (int u = 0; u < 8; ++u) acc += v[u];
  }
  o_hat[bh * D + tid] = acc;
  if (topk_idx == nullptr) return;
  const int S = max(0, min(max_S, seq_lens[b]));
  const int grp = (NG == 1) ? 0 : (tid / (D / NG));
  const uint8_t* vbase = v_data + (size_t)hkv * num_slots * P;
  const uint16_t* sbase = v_scales + (size_t)hkv * num_slots * NG;
  const int64_t* bt = block_table + (size_t)b * max_blocks;
  const float m = softmax_m[bh], iz = softmax_inv_z[bh];
  float acc_old = 0.0f, acc_w = 0.0f;
  for (int k0 = 0; k0 < K; k0 += STEP) {
    __syncthreads();
    {
      const int kk = k0 + tid;
      int64_t slot = -1;
      float w = 0.0f;
      if (kk < K) {
        const int64_t pos = topk_idx[bh * (size_t)K + kk];
        if (pos >= 0 && pos < S) {
          const int64_t blk = bt[pos / BS];
          if (blk >= 0) {
            slot = blk * BS + pos % BS;
            w = __expf(scores[bh * (size_t)max_S + pos] - m) * iz;
          }
        }
      }
      slot_buf[tid] = slot;
      w_buf[tid] = w;
#pragma unroll
      for (int g = 0; g < NG; ++g) ws_buf[tid][g] = (slot >= 0) ? w * bf16_to_f32(sbase[(size_t)slot * NG + g]) : 0.0f;
    }
    __syncthreads();
    const int kend = min(STEP, K - k0);
    for (int j = 0; j < kend; ++j) {
      const int64_t slot = slot_buf[j];
      if (slot < 0) continue;
      const float c = (float)v_code<NBITS>(vbase + slot * P, tid);
      acc_old = __builtin_fmaf(ws_buf[j][grp], c, acc_old);
      acc_w += w_buf[j];
    }
  }
  o_old[bh * D + tid] = acc_old;
  if (tid == 0) W_out[bh] = acc_w;
}

inline int sv_splits(int B, int H_kv, int max_S) {
  const int units = B * H_kv;
  int want = (2048 + units - 1) / units;
  const int max_by_len = (max_S + 63) / 64;
  want = want < 1 ? 1 : want;
  want = want > max_by_len ? max_by_len : want;
  return want < 1 ? 1 : want;
}

}  // namespace
}  // namespace jf

using namespace jf;

extern "C" size_t jf_softmax_v_workspace_bytes(int B, int H_q, int max_S) {
  if (B <= 0 || H_q <= 0) return 256;
  // partials for the largest split count any H_kv can produce, plus the two statistics rows
  size_t max_splits = (size_t)((max_S + 63) / 64 < 2048 ? (max_S + 63) / 64 : 2048);
  if (max_splits < (size_t)TQ_SPLITS) max_splits = TQ_SPLITS;  // the tile-quantised form always uses TQ_SPLITS ranges
  return ((size_t)B * H_q * max_splits * D + 2 * (size_t)B * H_q) * sizeof(float) + 256;
}

extern "C" int jf_softmax_v_pre_corr(const float* scores, const float* softmax_m, const float* softmax_inv_z,
                                     const uint8_t* v_data, const uint16_t* v_scales, const int64_t* block_table,
                                     const int32_t* seq_lens, const int64_t* topk_idx, int B, int H_q, int H_kv,
                                     int max_S, int max_blocks, int64_t num_slots, int block_size, int top_k,
                                     int v_nbits, int n_scale_groups, float* o_hat, float* o_old_unnorm, float* W,
                                     void* workspace, size_t workspace_bytes, void* stream) {
  JF_CHECK_ARG(B >= 0 && H_q > 0 && H_kv > 0 && max_S >= 0 && H_q % H_kv == 0, "softmax_v: bad shape");
  const int G = H_q / H_kv;
  JF_CHECK_ARG(G >= 1 && G <= 16, "softmax_v: GQA group %d not in 1..16", G);
  JF_CHECK_ARG(block_size == 16, "wvs2 only supports block_size=16");
  JF_CHECK_ARG(v_nbits == 2 || v_nbits == 3 || v_nbits == 4, "softmax_v: v_nbits must be 2, 3 or 4 (got %d)", v_nbits);
  JF_CHECK_ARG(n_scale_groups == 1 || n_scale_groups == 2, "wvs2 requires num_groups=1 or 2 (got %d)", n_scale_groups);
  JF_CHECK_ARG((int64_t)max_blocks * block_size >= max_S, "softmax_v: block_table does not cover max_S");
  JF_CHECK_ARG((softmax_m == nullptr) == (softmax_inv_z == nullptr), "softmax_v: softmax_m and softmax_inv_z go together");
  JF_CHECK_ARG(topk_idx == nullptr || top_k > 0, "softmax_v: top_k must be positive");
  if (B == 0) return JF_OK;
  JF_CHECK_ARG(scores && v_data && v_scales && block_table && seq_lens && o_hat, "softmax_v: null pointer");
  JF_CHECK_ARG(topk_idx == nullptr || (o_old_unnorm && W), "softmax_v: o_old_unnorm / W required with topk_idx");
  JF_CHECK_ARG(workspace && workspace_bytes >= jf_softmax_v_workspace_bytes(B, H_q, max_S),
               "softmax_v: workspace too small (%zu < %zu)", workspace_bytes, jf_softmax_v_workspace_bytes(B, H_q, max_S));
  hipStream_t st = (hipStream_t)stream;
  const int n_splits = sv_splits(B, H_kv, max_S);
  int chunk = (max_S + n_splits - 1) / n_splits;
  chunk = (chunk + BS - 1) / BS * BS;
  if (chunk < BS) chunk = BS;
  float* partial = reinterpret_cast<float*>(workspace);
  float* m_ws = partial + (size_t)B * H_q * n_splits * D;
  float* iz_ws = m_ws + (size_t)B * H_q;
  if (softmax_m == nullptr) {
    hipLaunchKernelGGL(softmax_stats_kernel, dim3(B, H_q), dim3(SV_THREADS), 0, st, scores, seq_lens, m_ws, iz_ws, max_S, H_q);
    JF_CHECK_LAUNCH();
    softmax_m = m_ws;
    softmax_inv_z = iz_ws;
  }
  dim3 grid(n_splits, H_kv, B), block(SV_THREADS);
#define JF_SV_LAUNCH(NB, NGC)                                                                                           \
  JF_DISPATCH_G2(G, {                                                                                                    \
    hipLaunchKernelGGL((weighted_v_split_kernel<NB, GG, NGC>), grid, block, 0, st, scores, softmax_m, softmax_inv_z,     \
                       v_data, v_scales, block_table, seq_lens, partial, H_q, H_kv, max_S, max_blocks, num_slots, chunk, \
                       n_splits, G);                                                                                     \
  });                                                                                                                    \
  JF_CHECK_LAUNCH();                                                                                                     \
  hipLaunchKernelGGL((combine_precorr_kernel<NB, NGC>), dim3(B, H_q), block, 0, st, partial, scores, softmax_m,          \
                     softmax_inv_z, v_data, v_scales, block_table, seq_lens, topk_idx, o_hat, o_old_unnorm, W, H_q, H_kv, \
                     max_S, max_blocks, num_slots, n_splits, top_k);                                                     \
  JF_CHECK_LAUNCH();
#define JF_DISPATCH_G2(G, ...)                               \
  switch ((G) <= 2 ? (G) : ((G) <= 4 ? 4 : ((G) <= 8 ? 8 : 16))) {  /* the next kernel size; the kernels take G itself too */ \
    case 1: { constexpr int GG = 1; __VA_ARGS__; } break;    \
    case 2: { constexpr int GG = 2; __VA_ARGS__; } break;    \
    case 4: { constexpr int GG = 4; __VA_ARGS__; } break;    \
    case 8: { constexpr int GG = 8; __VA_ARGS__; } break;    \
    default: { constexpr int GG = 16; __VA_ARGS__; } break;  \
  }
  if (v_nbits == 2 && n_scale_groups == 1) { JF_SV_LAUNCH(2, 1) }
  else if (v_nbits == 2) { JF_SV_LAUNCH(2, 2) }
  else if (v_nbits == 3 && n_scale_groups == 1) { JF_SV_LAUNCH(3, 1) }
  else if (v_nbits == 3) { JF_SV_LAUNCH(3, 2) }
  else if (n_scale_groups == 1) { JF_SV_LAUNCH(4, 1) }
  else { JF_SV_LAUNCH(4, 2) }
  return JF_OK;
}

extern "C" int jf_softmax_v_int8_tiles(const float* scores, const float* softmax_m, const float* softmax_inv_z,
                                       const uint8_t* v_data, const uint16_t* v_scales, const int64_t* block_table,
                                       const int32_t* seq_lens, const int64_t* topk_idx, int B, int H_q, int H_kv,
                                       int max_S, int max_blocks, int64_t num_slots, int block_size, int top_k,
                                       float* o_hat, float* o_old_unnorm, float* W, void* workspace,
                                       size_t workspace_bytes, void* stream) {
  JF_CHECK_ARG(B >= 0 && H_q > 0 && H_kv > 0 && max_S >= 0 && H_q % H_kv == 0, "int8tc_softmax_v: bad shape");
  const int G = H_q / H_kv;
  JF_CHECK_ARG(G >= 1 && G <= 16, "int8tc_softmax_v requires H_q/H_kv in 1..16 (got %d)", G);
  JF_CHECK_ARG(block_size == 16, "int8tc_softmax_v only supports block_size=16");
  JF_CHECK_ARG((int64_t)max_blocks * block_size >= max_S, "int8tc_softmax_v: block_table does not cover max_S");
  JF_CHECK_ARG(topk_idx == nullptr || top_k > 0, "int8tc_softmax_v: top_k must be positive");
  if (B == 0) return JF_OK;
  JF_CHECK_ARG(scores && softmax_m && softmax_inv_z && v_data && v_scales && block_table && seq_lens && o_hat,
               "int8tc_softmax_v: null pointer (the Stage-A statistics are required)");
  JF_CHECK_ARG(topk_idx == nullptr || (o_old_unnorm && W), "int8tc_softmax_v: o_old_unnorm / W required with topk_idx");
  JF_CHECK_ARG(workspace && workspace_bytes >= jf_softmax_v_workspace_bytes(B, H_q, max_S) &&
                   workspace_bytes >= (size_t)B * H_q * TQ_SPLITS * D * sizeof(float),
               "int8tc_softmax_v: workspace too small");
  hipStream_t st = (hipStream_t)stream;
  float* partial = reinterpret_cast<float*>(workspace);
  // A range is cut into `sub_count` runs (at most sixteen): enough workgroups of four wavefronts for four per CU, and
  // at least two pairs of tiles per wavefront (8 * sub_count <= max_S / 64 partial rows: inside the workspace, which
  // holds max(8, max_S / 64))
  const int pairs_per_range = ((max_S + TQ_SPLITS - 1) / TQ_SPLITS + 2 * TQ_TILE - 1) / (2 * TQ_TILE) + 1;
  const int want = (4 * device_cus() + TQ_SPLITS * H_kv * B - 1) / (TQ_SPLITS * H_kv * B);
  int sub_count = pairs_per_range / (2 * TQ_WAVES);
  sub_count = sub_count < want ? sub_count : want;
  sub_count = sub_count < 1 ? 1 : (sub_count > 16 ? 16 : sub_count);
  while (sub_count > 1 && (size_t)TQ_SPLITS * sub_count > (size_t)(max_S + 63) / 64) --sub_count;
  const dim3 grid(TQ_SPLITS * sub_count, H_kv, B);
#define JF_TQ_LAUNCH(NSET)                                                                                              \
  hipLaunchKernelGGL((tile_quantised_v_split_kernel<NSET>), grid, dim3(TQ_WAVES * 64), 0, st, scores, softmax_m,        \
                     softmax_inv_z, v_data, v_scales, block_table, seq_lens, partial, H_q, H_kv, max_S, max_blocks,     \
                     num_slots, sub_count, G)
  if (G <= 4) JF_TQ_LAUNCH(1);
  else if (G <= 8) JF_TQ_LAUNCH(2);
  else JF_TQ_LAUNCH(4);
#undef JF_TQ_LAUNCH
  JF_CHECK_LAUNCH();
  // the sum of the partials and the pre-correction terms run on the merge kernel of the fused step where its limits
  // allow (the same formula, p_j = exp(score_j - m) * inv_z with the caller's statistics), else in the combine kernel
  if (topk_idx != nullptr && top_k <= 2048 && num_slots <= (1ll << 26) && ((uintptr_t)v_data & 3) == 0)
    return precorr_int4_given_stats(scores, softmax_m, softmax_inv_z, v_data, v_scales, block_table, seq_lens, topk_idx, B,
                                    H_q, H_kv, max_S, max_blocks, num_slots, top_k, partial, TQ_SPLITS * sub_count, o_hat,
                                    o_old_unnorm, W, stream);
  hipLaunchKernelGGL((combine_precorr_kernel<4, 1>), dim3(B, H_q), dim3(SV_THREADS), 0, st, partial, scores, softmax_m,
                     softmax_inv_z, v_data, v_scales, block_table, seq_lens, topk_idx, o_hat, o_old_unnorm, W, H_q, H_kv,
                     max_S, max_blocks, num_slots, TQ_SPLITS * sub_count, top_k);
  JF_CHECK_LAUNCH();
  return JF_OK;
}
