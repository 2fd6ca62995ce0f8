// Fused decode scan + top-k for gfx950: one pass over the packed K and V of every (sequence, kv-head),
// no (B, H_q, S) score tensor in HBM.
//
// Launch 1, fused_scan_kernel, grid (H_kv, n_splits, B), 16 wavefronts per workgroup (8 where the register
// budget does not allow 1024 threads).  A workgroup owns L consecutive positions of one (sequence, kv-head)
// and all G query heads of that kv-head.  The page table of the split is read once into LDS.  Key and value
// rows are fetched in 64-position chunks with 16-byte loads whose lane addresses are consecutive inside a
// page, two chunks per wavefront in flight, staged in wavefront-private LDS and read back in the layout the
// arithmetic wants; barriers order LDS traffic only, so prefetched rows stay in flight across them.
//   phase A  Q.K^T on v_mfma_i32_16x16x64_i8, tokens on the N side, rows = (head, limb or block):
//            INT3 keys: the bf16 query as exact 23-bit fixed point in three int8 limbs, codes spread from the
//                       byte planes with shift/mask on dwords, a second contraction with the indicator of
//                       codes +-3 reproduces the reference's bf16 rounding of the dequantised key.
//            INT2 keys: the same limbs against the four-codes-per-byte rows; no second contraction, every
//                       dequantised INT2 key is exact in bf16.
//            INT4 keys: int8-quantised Q, exact nibble codes, one accumulator row per 32-channel block, the
//                       reference's fp32 rescale order (bit-equal to the split-form kernel).
//            scores[G][L] -> LDS (fp32), running max / min per head.
//   phase B  P.V on the same MFMA.  p = exp(s - m_split) is known exactly because phase A is complete, so
//            w = p * v_scale is converted to 23-bit fixed point once (fma with 2^23), the four bytes of the
//            converted word are the A-operand rows (head, limb 0..2 and the constant exponent byte), and the
//            int32 accumulators live for the whole split: every product is exact.  V codes are transposed by
//            ds_read_b64_tr_b4, weight rows by ds_read_b64_tr_b8.
//            The same pass drops every score into one of 256 linear buckets per (head, segment).
//   phase C  one wavefront per (head, segment): from the bucket histograms the smallest bucket range that holds
//            the split's top min(K, n) scores and fits the candidate buffer (every wavefront of a head finds it
//            itself); its positions are emitted as (key, position) in ascending position, sixteen consecutive
//            scores per lane and block.  Heavily tied scores fall back to a radix select.
//   sum of the wavefronts' integer accumulators with LDS integer atomics (issued along the emission's
//   comparisons), exact int64 recombination -> partial o.
// Launch 2, fused_merge_kernel, grid (G, H_kv, B) (ahead of it, with many candidates per row, a first stage of it on grid
// (B, H_q, parts)): selects the global top-k among the candidates (ties to the lower position, ascending output), merges
// the split partials
//   M = max m_i, l = sum l_i e^{m_i-M}, o_hat = sum o_i e^{m_i-M} / l
// (the split-KV combine of jetfire_vllm/csrc/fused_decode_wmma.cu:1226-1253), and computes the
// pre-correction terms o_old_unnorm, W over the winners (jetfire_vllm/csrc/int2_softmax_v.cu:738-788).
// Where one split covers the sequence (short contexts, large batches) launch 1 does both (template argument ONE).
// Both kernels take a template argument MODE: the whole step, or one stage alone (Stage A: scores written out,
// top-k, statistics; Stage B: scores and winners given, value stream; selection alone), for callers that keep the
// reference's separate operators.
//
// This header holds the kernels, the launch planner and the launcher; it is included by the translation units that
// instantiate them (fused_scan.hip and the stage-wise forms), each for its own set of template arguments.
#pragma once
#include "common.h"

#include <atomic>
#include <type_traits>
#include <mutex>
#include <utility>
#include <vector>

namespace jf {

#ifdef JF_DEBUG_HOOKS
// Process-wide measurement / test switches shared by those translation units (defined in fused_scan.hip),
// reachable from the debug entry points of jetfire_amd_debug.h; a library built without JF_DEBUG_HOOKS has none of
// them.  The event list has its own lock, the two scalars are atomics (a launch reads each once).
// Optional measurement hook: when armed, every fused_scan_kernel launch is bracketed by a pair of HIP
// events on its own stream, so a benchmark can read the kernel's device time without a profiler.
struct ScanProfile {
  std::vector<hipEvent_t> ev;
  int used = 0;
  std::atomic<bool> armed{false};
};
extern ScanProfile g_prof;
extern std::mutex g_prof_mu;
extern std::atomic<long long*> g_phase_clock;
extern std::atomic<int> g_force_split_len;  // test / measurement aid: overrides the planner's split length when positive
constexpr bool kDebugHooks = true;
// clock of the phase stamps: the wavefront's own cycle counter, or (JF_STAMP_WALL_CLOCK) the constant 100 MHz counter
// that every XCD shares, for comparing workgroups on different XCDs (their cycle counters run at different rates)
#ifdef JF_STAMP_WALL_CLOCK
#define JF_CLK() ((long long)wall_clock64())
#else
#define JF_CLK() clock64()
#endif
#else
#define JF_CLK() 0ll
constexpr bool kDebugHooks = false;
#endif
// The one-pass scan kernels are instantiated in five translation units (fused_full_*.hip), one per family of
// schemes, and five more for the form for short splits (fused_short_*.hip: the same files with JF_SHORT_FORM), so that they
// compile side by side; `params` points to the launcher's FusedParams.
#define JF_SCAN_FAMILY(F)                                                                        \
  int launch_full_scan_##F(int scheme, int G, int NG, const void* params, void* stream);         \
  int launch_short_scan_##F(int scheme, int G, int NG, const void* params, void* stream);
JF_SCAN_FAMILY(a)  // K3V2, K4V4, K3V4, K4V2
JF_SCAN_FAMILY(b)  // K2V2, K2V3, K2V4
JF_SCAN_FAMILY(c)  // K3V3, K4V3
JF_SCAN_FAMILY(d)  // A2V2, A2V3, A2V4
JF_SCAN_FAMILY(e)  // B4V2, B4V3, B4V4
#undef JF_SCAN_FAMILY
#ifdef JF_SHORT_FORM
#define JF_SCAN_ENTRY(F) launch_short_scan_##F
constexpr bool kShortForm = true;
#else
#define JF_SCAN_ENTRY(F) launch_full_scan_##F
constexpr bool kShortForm = false;
#endif

namespace {

typedef int v2i __attribute__((ext_vector_type(2)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v3i __attribute__((ext_vector_type(3)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));

// Forms of the step (template argument MODE of both kernels):
//   FS_FULL     Stage A + Stage B + top-k in one pass (keys and values streamed once, scores never in HBM)
//   FS_STAGE_A  Stage A alone: scores (optionally written out), top-k, softmax statistics; no value stream
//   FS_STAGE_B  Stage B alone: scores and winners are inputs; value stream, o_hat and the pre-correction terms
//   FS_TOPK     selection alone: scores are an input; top-k, slots and softmax statistics (scan kernel only; its
//               merge is the FS_STAGE_A one)
constexpr int FS_FULL = 0, FS_STAGE_A = 1, FS_STAGE_B = 2, FS_TOPK = 3;

constexpr int FS_MAX_TOPK = 8192;      // widest correction
constexpr int FS_LDS_TOPK = 2048;      // winners the merge kernel keeps in static LDS; wider ones go to dynamic LDS
constexpr long long FS_MAX_SLOTS = 1ll << 26;  // slots per kv-head tensor: 64-byte rows, 32-bit row offsets (4 GB)
constexpr int FS_CAND_SLACK = 256;     // extra candidate slots per (row, split): room for the whole cut bucket

struct FusedParams {
  const uint16_t* q;
  const uint8_t* k_data;
  const uint16_t* k_scales;
  const uint16_t* k_zp;  // asymmetric INT2 keys only: zero-points, shaped like k_scales
  const uint8_t* v_data;
  const uint16_t* v_scales;
  const int64_t* block_table;
  const int32_t* seq_lens;
  int B, H_q, H_kv, max_S, max_blocks;
  int one_split;  // (host) the scan merges by itself: n_splits == 1 and one_split_merges
  int g_act;  // query heads per kv-head (H_q / H_kv); the kernel's G is this rounded up to 1, 2, 4, 8 or 16
  int64_t num_slots;
  float attn_scale;
  int top_k;
  int L, n_splits, Kc;
  float* scores;  // optional (B, H_q, max_S)
  const float* scores_in;  // FS_STAGE_B: the scores (B, H_q, max_S)
  const float* stats_m;    // FS_STAGE_B merge, optional: softmax statistics (B, H_q) that replace the ones derived
  const float* stats_iz;   //   from the split partials (which are then already normalised; part_m, part_l NULL)
  int scores_only;         // FS_STAGE_A: stop after writing `scores`
  float* part_m;  // (B, H_q, NS)
  float* part_l;  // (B, H_q, NS)
  float* part_o;  // (B, H_q, NS, D)
  uint32_t* cand_key;  // (B, H_q, NS, Kc)
  int32_t* cand_idx;   // (B, H_q, NS, Kc)
  float* cand_edge;    // (B, H_q, NS) about the smallest score of the list: where it holds top_k, that many lie no lower
  // two-stage merge (long contexts): `mg_parts` workgroups per row first reduce `mg_spp` consecutive
  // candidate lists each to the row's top_k among them; the final merge then reads those lists
  int mg_parts, mg_spp;
  uint32_t* key2;      // (B, H_q, mg_parts, top_k)
  int32_t* idx2;       // (B, H_q, mg_parts, top_k)
  float* edge2;        // (B, H_q, mg_parts)
  // merge outputs
  int64_t* topk_idx;
  int64_t* topk_slots;
  float* o_hat;
  float* o_old;
  float* W;
  float* softmax_m;
  float* softmax_inv_z;
  // optional merge epilogue: out = bf16(fma(W, o_new, o_hat) - o_old_unnorm), both (B, H_q, D) bf16
  const uint16_t* blend_o_new;
  uint16_t* blend_out;
  long long* phase_clock;  // optional: 10 s_memtime stamps per scan workgroup, 8 per merge workgroup (measurement aid)
};

// What the merge kernel takes (its first loads depend on the first block: one round trip for the arguments).
struct MergeParams {
  const uint32_t* list_key;  // (B, H_q, lists, list_cap) candidate lists: the scan's or, in the final of two stages, the first stage's
  const int32_t* list_idx;   // (B, H_q, lists, list_cap)
  const float* list_edge;    // (B, H_q, lists)
  const float* part_m;       // (B, H_q, n_splits); NULL (Stage B, given statistics): part_o is already normalised
  const float* part_l;
  const float* part_o;
  const int64_t* block_table;
  const int32_t* seq_lens;
  const uint16_t* blend_o_new;
  int H_q, g_act, n_splits, lists, list_cap, list_len, top_k, max_blocks, max_S, mg_spp, mg_parts;
  int64_t num_slots;
  const uint8_t* v_data;
  const uint16_t* v_scales;
  const float* scores_in;  // FS_STAGE_B
  const float* stats_m;
  const float* stats_iz;
  int64_t* topk_idx;
  int64_t* topk_slots;
  float* o_hat;
  float* o_old;
  float* W;
  float* softmax_m;
  float* softmax_inv_z;
  uint16_t* blend_out;
  uint32_t* out_key;  // first stage: (B, H_q, mg_parts, top_k), and (B, H_q, mg_parts)
  int32_t* out_idx;
  float* out_edge;
  long long* phase_clock;
};

// The merge of one scan (`first`: its first stage) as the kernel takes it.
inline MergeParams merge_params(const FusedParams& p, bool first) {
  MergeParams m = {};
  const bool staged = !first && p.mg_parts > 1;
  m.list_key = staged ? p.key2 : p.cand_key;
  m.list_idx = staged ? p.idx2 : p.cand_idx;
  m.list_edge = staged ? p.edge2 : p.cand_edge;
  m.lists = staged ? p.mg_parts : p.n_splits;
  m.list_cap = staged ? p.top_k : p.Kc;
  m.list_len = staged ? p.mg_spp * p.L : p.L;
  m.part_m = p.part_m; m.part_l = p.part_l; m.part_o = p.part_o;
  m.block_table = p.block_table; m.seq_lens = p.seq_lens; m.blend_o_new = p.blend_o_new;
  m.H_q = p.H_q; m.g_act = p.g_act; m.n_splits = p.n_splits; m.top_k = p.top_k; m.max_blocks = p.max_blocks;
  m.max_S = p.max_S; m.mg_spp = p.mg_spp; m.mg_parts = p.mg_parts; m.num_slots = p.num_slots;
  m.v_data = p.v_data; m.v_scales = p.v_scales; m.scores_in = p.scores_in; m.stats_m = p.stats_m; m.stats_iz = p.stats_iz;
  m.topk_idx = p.topk_idx; m.topk_slots = p.topk_slots; m.o_hat = p.o_hat; m.o_old = p.o_old; m.W = p.W;
  m.softmax_m = p.softmax_m; m.softmax_inv_z = p.softmax_inv_z; m.blend_out = p.blend_out;
  m.out_key = p.key2; m.out_idx = p.idx2; m.out_edge = p.edge2;
  m.phase_clock = p.phase_clock ? p.phase_clock + (size_t)p.B * p.H_kv * p.n_splits * 10 : nullptr;
  return m;
}

// Phase-A constants of the INT3 path, built once per workgroup in LDS.
template <int NSET>
struct K3Prep {
  int8_t aop[NSET][16][4][2][16];  // A operand bytes: [set][row = 4*head + limb][k-block][MFMA][byte]
  int sq4[NSET * 4][2];            // code offset * sum of the fixed-point query over the scale group (WIDE_SUM: the sum)
  float qsc[NSET * 4][2];          // 2^(e-22) * attn_scale of the (head, group)
  float amax_w[NSET * 8];          // per 64-channel half row: |q| maximum, fixed-point sum, exponent
  int sum_w[NSET * 8];
  int exp_w[NSET * 8];
};

// Phase-A constants of the INT4 path: the int8-quantised query rows as MFMA A operand.  Row 4*head + kk holds
// the head's values of 32-channel block kk and zeros elsewhere, so one accumulator register per block.
template <int NSET>
struct QInt8F {
  int8_t aop[NSET][16][4][2][16];  // [set][row = 4*head + block][k-block][MFMA][byte]
  float qs[NSET * 4][4];           // query scale of (head, block)
  int sum8[NSET * 4][4];           // 8 * sum of the int8 query over the block (the codes carry an offset of 8)
};

// LDS carve-up shared by the kernel and its launcher.
//   sc     [G][L] fp32 scores of the split
//   sbase  [L/16] first slot of every 16-position page
//   aux    phase A: query constants (K3Prep / QInt8F) and the rounding tables of the bf16-model INT4 keys; afterwards:
//          selection histograms [G][SEG][256].  With those keys it lies in front of sc instead of behind sbase, so that a
//          look-up's address is the index plus a constant the instruction carries
//   stage  one private staging area per wavefront: key rows in phase A, V rows + weight rows in phase B
// After phase B the staging area holds the sum of the wavefronts' P.V accumulators.
template <int SCHEME, int G, int NG>
struct ScanLds {
  // SCHEME = 10 * key bits + value bits (key digit 1: asymmetric INT2; 5: INT4 with the bf16 model): the key side (staging, query constants, phase A) and the value side
  // (staging, phase B) are chosen independently
  static constexpr bool K3 = (SCHEME / 10 == 3);
  static constexpr bool KA = (SCHEME / 10 == 1);        // INT2 keys with a zero-point per group (four levels)
  static constexpr bool K2 = (SCHEME / 10 == 2) || KA;  // four codes per byte
  static constexpr bool KB4 = (SCHEME / 10 == 5);       // INT4 keys scored with the bf16 model (any group size)
  static constexpr bool KLIMB = K2 || K3 || KB4;  // keys with the bf16 model: fixed-point query limbs against integer codes
  static constexpr bool V2 = (SCHEME % 10 == 2);
  static constexpr bool V3 = (SCHEME % 10 == 3);
  static_assert((KLIMB || SCHEME / 10 == 4) && (V2 || V3 || SCHEME % 10 == 4), "keys and values are INT2, INT3 or INT4");
  static constexpr int NSET = (G + 3) / 4;
  // wavefronts per workgroup: sixteen where the register budget allows (128 VGPRs at 1024 threads), else eight
  static constexpr int NW = (G <= 4) ? 16 : 8;
  static constexpr int NT = NW * 64;
  static constexpr int LMAX = NW * 256;  // four 64-position chunks per wavefront
  // emission segments per head (one wavefront each)
  static constexpr int SEG = (NW / G >= 4) ? 4 : ((NW / G >= 2) ? 2 : 1);
  static constexpr int KP = K2 ? 32 : (K3 ? 48 : 64);
  static constexpr int KROW = K2 ? 40 : (K3 ? 48 : 80);  // LDS pitch of a staged key row (INT2, INT4: padded against bank conflicts)
  static constexpr int VP = V2 ? 32 : (V3 ? 48 : 64);
  // LDS pitch of a staged V row.  INT2 rows (32 bytes) are padded so that 16 consecutive rows hit 16 distinct
  // bank pairs; INT4 rows (64 bytes) keep their pitch and swap their 16-byte quarters instead (quarter q of row r
  // sits at q ^ ((r >> 2) & 3)), which has the same effect without the padding bytes.  INT3 rows (48 bytes: 16
  // consecutive rows already hit distinct bank pairs) swap the 8-byte halves of every plane in rows 16..31 and
  // 48..63, so that the two 16-row groups one 8-byte read serves in a cycle do not meet either.
  static constexpr bool VSWZ = !(V2 || V3);
  static constexpr int VROW = (VSWZ || V3) ? VP : VP + 8;
  static constexpr int VST = 64 * VROW;
  static constexpr int WL = NG * NSET * 64 * 16;  // per (group, set): one 16-byte weight row per token
  static constexpr int KST = 64 * KROW;
  static constexpr int WAVE_STAGE = (VST + WL > KST) ? (VST + WL) : KST;
  // INT3 / symmetric INT2 keys: the scale word of a token is loaded once (lane = token) and turned into the floats
  // phase A multiplies by -- the group scales and the rounding coefficients -- in a table behind the staged key rows,
  // 8 * NG bytes per token, instead of by every one of the four lanes that handle the token's heads
  static constexpr int SCT = 8 * NG;
  static constexpr bool SPREP = (K3 || (K2 && !KA)) && (WAVE_STAGE >= KST + 64 * SCT);
  static constexpr int ACC_REGS = 8 + NG;                   // v4i accumulators per set: 8 channel tiles + NG weight sums
  // sum of the wavefronts' accumulators: two ints per (set, accumulator register, lane) and one per (set, tile, column), in the staging
  // area (dead after phase B), followed by what the emission needs per wavefront
  static constexpr int XACC = NSET * (ACC_REGS * 2 * 64 + 8 * 16) * 4;
  static constexpr int PREP = KLIMB ? (int)sizeof(K3Prep<NSET>) : (int)sizeof(QInt8F<NSET>);
  // selection histograms: 32-bit counters, or (any INT4 side, where the staging areas are larger and LDS is
  // tighter) two 16-bit counters per word: a (head, segment) histogram counts at most LMAX / SEG <= 4096 positions
  static constexpr bool H16 = !(KLIMB && V2);
  static constexpr int HIST = G * SEG * 256 * (H16 ? 2 : 4);
  // Rounding tables: 128 entries of 16 bytes, then 128 of four.  In LDS of their own they cost the format the splits of 4096
  // positions: 4 x 32768 positions, 8 kv-heads, G = 4, top-k 256, B4V4 in one group took 16 splits of 2048 instead of 8 and
  // two rounds of workgroups, per layer 52.5 us, now 40.1 (B4V3 in 64-channel groups 55.5 / 42.4; 1 x 131072, top-k 512, B4V4
  // in one group 62.5 / 48.0).
  static constexpr int RND_AT = (PREP + 15) & ~15, RND = KB4 ? 128 * (16 + 4) : 0;
  static constexpr int AUX = ((RND_AT + RND > HIST ? RND_AT + RND : HIST) + 15) & ~15;
  static constexpr int SC_AT = KB4 ? AUX : 0;
  __host__ __device__ static constexpr int stage_bytes() { return NW * WAVE_STAGE; }
  // per wavefront behind it: the candidates of a block of 1024 positions, or the exact selection's histogram
  static constexpr int EMIT = 2048;
  static_assert(NW * WAVE_STAGE >= XACC + NW * EMIT, "the staging area must hold the accumulator sums and the selection scratch");
  __host__ __device__ static constexpr size_t per_position() { return (size_t)G * 4; }
  __host__ __device__ static size_t aux_offset(int L) { return (per_position() * L + (size_t)(L / 16) * 4 + 15) & ~(size_t)15; }
  __host__ __device__ static size_t total(int L) {
    return aux_offset(L) + AUX + stage_bytes() + 64;
  }
};

// LDS behind the staging area of a scan workgroup that holds the whole sequence and merges by itself (ONE): per head
// the members of the cut bucket, the winners' positions, slots and weights, o_hat and a few words.
template <int G, int SEG>
struct ScanTail {
  static constexpr int MEM = 64;  // members of the cut bucket that are selected from a list, one per lane
  static constexpr int RANK = 24;  // up to here against each other, beyond by bits
  static constexpr int INTS = ((3 + SEG + 3) * G * 4 + 15) & ~15;
  __host__ __device__ static constexpr size_t bytes(int top_k, int kc) {
    return INTS + (size_t)G * (D * 4 + 8 * (size_t)top_k + 8 * MEM + 2 * (size_t)kc);
  }
};

__device__ inline float key_to_score(uint32_t key) {
  const uint32_t u = (key & 0x80000000u) ? (key & 0x7fffffffu) : ~key;
  return __builtin_bit_cast(float, u);
}

// Narrows `active` to the lanes that hold the `need`-th largest of the active lanes' words (need: 1 .. their number, uniform;
// afterwards its place among those equal lanes).  One ballot per bit from the highest in which the words differ, the rest on
// the scalar unit, until one lane is left: about 1 us whatever the number of words.  (Comparing every word with every other
// one, as a loop over scalars, costs five vector instructions per word in each of the workgroup's wavefronts: 2 us at 60.)
__device__ inline void nth_largest(uint32_t word, unsigned long long& active, int& need) {
  if (active == 0ull) return;
  const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)word, __ffsll((long long)active) - 1);
  const bool in = (active >> (threadIdx.x & 63)) & 1ull;
  const uint32_t differ = (uint32_t)__builtin_amdgcn_readfirstlane((int)wave_max_u(in ? word ^ first : 0u));
  if (differ == 0u) return;
  for (int b = 31 - __clz((int)differ); b >= 0 && (active & (active - 1)) != 0ull; --b) {
    const unsigned long long ones = __builtin_amdgcn_ballot_w64(((word >> b) & 1u) != 0u) & active;
    const int c = __popcll(ones);
    if (need <= c || ones == active) {
      active = ones;
    } else {
      need -= c;
      active &= ~ones;
    }
  }
}

// Orders this wavefront's earlier LDS writes before its later LDS reads (the LDS pipe executes one
// wavefront's instructions in order; this only stops the compiler from moving them).
__device__ inline void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Workgroup barrier that orders LDS traffic only: unlike __syncthreads() it does not wait for global loads
// that are still in flight (the prefetched key / value rows), which no other wavefront consumes.
__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// A copy the compiler cannot see through: the source register is dead afterwards, so a load issued next can
// write it directly instead of a temporary that is moved into place (after a wait) at the end of the block.
__device__ inline uint32_t reg_copy(uint32_t v) {
  uint32_t r;
  asm volatile("v_mov_b32 %0, %1" : "=v"(r) : "v"(v));
  return r;
}

// (hi * 256 + mid) * 256 + lo as two v_lshl_add_u32.  Written as plain shifts and adds the compiler re-associates
// it into two shifts and a three-operand add, one instruction more, in the innermost loop of the key stream; the
// empty statement makes the intermediate opaque.  (The instructions themselves stay the compiler's: it alone knows
// how long after an MFMA its results may be read.)
__device__ inline int join_limbs(int hi, int mid, int lo) {
  int t = (hi << 8) + mid;
  asm("" : "+v"(t));
  return (t << 8) + lo;
}

// s_setprio takes an immediate; `p` is a compile-time constant after unrolling
__device__ inline void set_wave_prio(int p) {
  if (p >= 3) __builtin_amdgcn_s_setprio(3);
  else if (p == 2) __builtin_amdgcn_s_setprio(2);
  else if (p == 1) __builtin_amdgcn_s_setprio(1);
  else __builtin_amdgcn_s_setprio(0);
}

__device__ inline float uniform_f(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}

// |x| as an integer of the same order; zero for a NaN, which takes no part in a maximum
__device__ inline uint32_t abs_bits(float x) { return (x == x) ? __builtin_bit_cast(uint32_t, x) & 0x7fffffffu : 0u; }
// Reductions over each half of a wavefront (32 lanes), the result in every lane of the half: DPP row shifts and the first
// row broadcast.  (Five shuffles through the LDS crossbar, one after the other, take some 600 cycles.)
__device__ inline uint32_t half_max_u(uint32_t v) {
  JF_DPP_ROW_REDUCE(v, op_umax, uint32_t, 0u);
  v = op_umax(v, (uint32_t)dpp_mov<0x142, 0xa>(0, (int)v));
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)v, 31), hi = (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
  return (threadIdx.x & 32) ? hi : lo;
}
__device__ inline int half_sum_i(int v) {
  JF_DPP_ROW_REDUCE(v, op_iadd, int, 0);
  v += dpp_mov<0x142, 0xa>(0, v);
  const int lo = __builtin_amdgcn_readlane(v, 31), hi = __builtin_amdgcn_readlane(v, 63);
  return (threadIdx.x & 32) ? hi : lo;
}

// Range-checked loads through a buffer descriptor (raw, the offsets in bytes): past its end a load returns zero, and the
// scalar base and offset take the place of 64-bit vector address arithmetic.
__device__ inline __amdgpu_buffer_rsrc_t buffer_of(const void* base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00020000);
}
__device__ inline int buffer_i32(__amdgpu_buffer_rsrc_t r, int voffset, int soffset) {
  return (int)__builtin_amdgcn_raw_buffer_load_b32(r, voffset, soffset, 0);
}
__device__ inline v4i buffer_i32x4(__amdgpu_buffer_rsrc_t r, int voffset, int soffset) {
  return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(r, voffset, soffset, 0));
}
__device__ inline float buffer_f32(__amdgpu_buffer_rsrc_t r, int voffset, int soffset) {
  return __builtin_bit_cast(float, buffer_i32(r, voffset, soffset));
}

// The streams' steps must be part of the kernel: as calls (the compiler's choice for some instantiations) they keep every
// captured array in scratch memory, at three times the run time.
#define JF_INLINE __attribute__((always_inline))

// Value codes as MFMA B operands.  64 packed V rows lie in LDS (`stash_row`, or the value stream's own stores to the same
// places), and transposed reads hand every lane 16 tokens of a channel or two, which are spread to one code per byte.  Tile t,
// column c of the products is channel `channel(t, c)`.
template <int VBITS, int NG>
struct VTiles {
  static constexpr bool V2 = VBITS == 2, V3 = VBITS == 3;
  static constexpr int VP = D * VBITS / 8;
  // LDS pitch of a staged V row.  INT2 rows (32 bytes) are padded so that 16 consecutive rows hit 16 distinct
  // bank pairs; INT4 rows (64 bytes) keep their pitch and swap their 16-byte quarters instead (quarter q of row r
  // sits at q ^ ((r >> 2) & 3)), which has the same effect without the padding bytes.  INT3 rows (48 bytes: 16
  // consecutive rows already hit distinct bank pairs) swap the 8-byte halves of every plane in rows 16..31 and
  // 48..63, so that the two 16-row groups one 8-byte read serves in a cycle do not meet either.
  static constexpr bool VSWZ = !(V2 || V3);
  static constexpr int VROW = (VSWZ || V3) ? VP : VP + 8;
  static constexpr int VST = 64 * VROW;
  static constexpr int OFFSET = V2 ? 2 : (V3 ? 4 : 8);  // of the codes
  // even INT2 tiles hold four times their codes
  static constexpr int times(int tile) { return V2 && !(tile & 1) ? 4 : 1; }
  static __device__ inline int channel(int tile, int col) {
    if (V2) return (tile >> 1) * 32 + (col >> 1) * 4 + ((col & 1) ? 0 : 2) + (tile & 1);
    // tile = 4 * (64-channel half) + code within the lane's four; odd columns hold codes 0..3
    if (V3) return (tile >> 2) * 64 + (col >> 1) * 8 + ((col & 1) ? 0 : 4) + (tile & 3);
    return tile * 16 + 2 * (col >> 1) + (1 - (col & 1));
  }
  // piece i (16 bytes) of row `row` to its place
  static __device__ inline void stash_piece(uint8_t* vst, int row, int i, const v4u& x) {
    uint8_t* dst = vst + row * VROW;
    if constexpr (VSWZ) {
      *reinterpret_cast<v4u*>(dst + ((i ^ ((row >> 2) & 3)) * 16)) = x;
    } else {
      const int first = V3 ? 8 * ((row >> 4) & 1) : 0;  // (INT3: first half's place)
      *reinterpret_cast<v2u*>(dst + 16 * i + first) = (v2u){x[0], x[1]};
      *reinterpret_cast<v2u*>(dst + 16 * i + (8 - first)) = (v2u){x[2], x[3]};
    }
  }
  // calls f(tile, scale group, operand) for the eight tiles of 16 channels
  template <class F>
  static __device__ JF_INLINE void spread(const uint8_t* vst, int lane, F&& f) {
    // the nibble spread of a transposed V dword yields tokens 0,2,4,6 | 1,3,5,7 | 8,10,12,14 | 9,11,13,15 of the
    // lane group's 16 tokens: token r sits in byte (r&8) | ((r&1)<<2) | ((r>>1)&3)
    const uint8_t* vrow = vst + lane * VROW;
    spread_from(vrow, lane, f, std::make_integer_sequence<int, V2 ? 4 : (V3 ? 2 : 8)>{});
  }
  template <class F, int... Q>
  static __device__ JF_INLINE void spread_from(const uint8_t* vrow, int lane, F&& f, std::integer_sequence<int, Q...>) {
    (step<Q>(vrow, lane, f), ...);
  }
  template <int Q, class F>
  static __device__ JF_INLINE void step(const uint8_t* vrow, int lane, F&& f) {
    if constexpr (V2) {
      const v2i x = __builtin_amdgcn_ds_read_tr4_b64_v2i32((__attribute__((address_space(3))) v2i*)(vrow + 8 * Q));
      const uint32_t x0 = (uint32_t)x[0], x1 = (uint32_t)x[1], y0 = x0 >> 4, y1 = x1 >> 4;
      // the upper code of every nibble stays where it is: tile 2 * Q accumulates 4 * code (undone where the sums are read)
      const v4i Ba = {(int)(x0 & 0x0c0c0c0cu), (int)(y0 & 0x0c0c0c0cu), (int)(x1 & 0x0c0c0c0cu), (int)(y1 & 0x0c0c0c0cu)};
      const v4i Bb = {(int)(x0 & 0x03030303u), (int)(y0 & 0x03030303u), (int)(x1 & 0x03030303u), (int)(y1 & 0x03030303u)};
      const int g = (NG == 1) ? 0 : (Q >> 1);
      f(std::integral_constant<int, 2 * Q>{}, g, Ba);
      f(std::integral_constant<int, 2 * Q + 1>{}, g, Bb);
    } else if constexpr (V3) {
      // Planar INT3: bytes j of the three 16-byte planes form the 24-bit word of channels 8j .. 8j+7, code i at
      // bits 23-3i .. 21-3i.  A transposed read of one plane's 8-byte half hands lane c the nibble c of 16 tokens:
      // odd lanes the high nibbles of byte c >> 1, even lanes the low ones.  With one exchange inside the lane
      // pair (the odd lane needs its partner's plane-0 nibble, the even lane its partner's plane-2 nibble) the odd
      // lane holds what codes 0..3 of the word are made of and the even lane what codes 4..7 are made of, in the
      // same three positions: a = [c0 c0 c0 c1], b = [c1 c1 c2 c2], c = [c2 c3 c3 c3] (msb first).
      const bool odd = (lane & 1) != 0;
      const int hsw = 8 * ((lane >> 4) & 1);  // rows 16..31, 48..63 keep their plane halves swapped
      const uint8_t* src = vrow + (Q ? 8 - hsw : hsw);
      const v2i x0 = __builtin_amdgcn_ds_read_tr4_b64_v2i32((__attribute__((address_space(3))) v2i*)(src));
      const v2i x1 = __builtin_amdgcn_ds_read_tr4_b64_v2i32((__attribute__((address_space(3))) v2i*)(src + 16));
      const v2i x2 = __builtin_amdgcn_ds_read_tr4_b64_v2i32((__attribute__((address_space(3))) v2i*)(src + 32));
      v4i Bc[4];
#pragma unroll
      for (int hw = 0; hw < 2; ++hw) {  // tokens 0..7 and 8..15 of the lane group, one nibble each
        const int send = odd ? x2[hw] : x0[hw];
        const uint32_t b = (uint32_t)dpp_mov<0xb1, 0xf>(0, send);  // quad_perm [1,0,3,2]: the pair partner's value
        const uint32_t a = (uint32_t)(odd ? x0[hw] : x1[hw]), c = (uint32_t)(odd ? x1[hw] : x2[hw]);
        // per nibble (bit 3 of the two middle codes is cleared by the byte masks below)
        const uint32_t n1 = ((b >> 2) & 0x33333333u) | ((a << 2) & ~0x33333333u);
        const uint32_t n2 = ((c >> 3) & 0x11111111u) | ((b << 1) & ~0x11111111u);
        Bc[0][2 * hw] = (int)((a >> 1) & 0x07070707u);
        Bc[0][2 * hw + 1] = (int)((a >> 5) & 0x07070707u);
        Bc[1][2 * hw] = (int)(n1 & 0x07070707u);
        Bc[1][2 * hw + 1] = (int)((n1 >> 4) & 0x07070707u);
        Bc[2][2 * hw] = (int)(n2 & 0x07070707u);
        Bc[2][2 * hw + 1] = (int)((n2 >> 4) & 0x07070707u);
        Bc[3][2 * hw] = (int)(c & 0x07070707u);
        Bc[3][2 * hw + 1] = (int)((c >> 4) & 0x07070707u);
      }
      const int g = (NG == 1) ? 0 : Q;
      f(std::integral_constant<int, 4 * Q>{}, g, Bc[0]);
      f(std::integral_constant<int, 4 * Q + 1>{}, g, Bc[1]);
      f(std::integral_constant<int, 4 * Q + 2>{}, g, Bc[2]);
      f(std::integral_constant<int, 4 * Q + 3>{}, g, Bc[3]);
    } else {
      const int vx = 16 * ((lane >> 2) & 3);  // quarter swap of this lane's row
      const v2i x = __builtin_amdgcn_ds_read_tr4_b64_v2i32((__attribute__((address_space(3))) v2i*)(vrow + ((8 * Q) ^ vx)));
      const uint32_t x0 = (uint32_t)x[0], x1 = (uint32_t)x[1];
      const v4i Bv = {(int)(x0 & 0x0f0f0f0fu), (int)((x0 >> 4) & 0x0f0f0f0fu),
                      (int)(x1 & 0x0f0f0f0fu), (int)((x1 >> 4) & 0x0f0f0f0fu)};
      f(std::integral_constant<int, Q>{}, (NG == 1) ? 0 : (Q >> 2), Bv);
    }
  }
};

// Byte j of an A operand is token tr8_token of the lane group's 16: what pairs a transposed read of 16-byte rows with the
// byte order of VTiles' operands (the lane pair (2j, 2j+1) supplies the two halves of the row that must land in byte j).
__device__ inline int tr8_token(int lane) { return (((lane >> 1) & 3) << 1) | ((lane >> 3) & 1); }

// Pre-correction terms over the winners' packed V rows where a wavefront has 64 winners of a head at a time (one per lane): the
// contraction of phase B on v_mfma_i32_16x16x64_i8, with one head's weights in four rows of the operand.  The weights are held
// to 30 bits of the largest among the 64 (a float times a power of two is exact, 30 bits are what four signed digits of eight
// take without an overflow), so a weight 2^-6 of the largest keeps all its bits; the products are exact, and each of the
// 64-winner sums is rounded once.  (24 bits were off by up to three times what sums code by code in fp32 are where one score
// stands out.)
// What a conversion and a multiply-add per code take instead, per
// layer: 32 sequences x 2048 positions, K3V2, top-k 256 25.2 us, this 24.1; K4V4 26.6 / 25.5; 32 x 1900, K3V2, 512 28.9 / 26.8;
// 16 x 1024, K4V4, 512 21.7 / 19.3; 32 x 500, eight heads, K3V2, 256 22.1 / 20.5.
template <int VBITS, int NG>
struct WinnerSums {
  using Tiles = VTiles<VBITS, NG>;
  static constexpr int PIECES = Tiles::VP / 16;
  static constexpr int STAGE = Tiles::VST + 1024;  // LDS per wavefront: the rows, and a 16-byte weight row per winner
  struct Rows {
    v4u r[PIECES];
    uint32_t s;  // scale word
    float w;     // weight, zero for no winner
  };
  // winners first .. first + 63 of n; slots (-1: none) and weights of the head's winners in LDS.  The lanes of a row lie side by
  // side: a lane per row touched sixty-four
  // lines with every load (32 sequences x 2048 positions, K4V4, top-k 256 27.3 us per layer, 25.8 with this).
  static __device__ JF_INLINE Rows fetch(const uint8_t* vbase, const uint8_t* vsbase, const int* slots, const float* weights, int first, int n, int lane) {
    Rows x;
    int slot[PIECES];
#pragma unroll
    for (int i = 0; i < PIECES; ++i) slot[i] = slots[min(first + (1024 * i + 16 * lane) / Tiles::VP, n - 1)];
    const int own = min(first + lane, n - 1);
    const int mine = slots[own];
    const float w = weights[own];
    const bool valid = first + lane < n && mine >= 0;
    x.w = valid ? w : 0.f;
    const uint32_t sl = (uint32_t)max(mine, 0);
    if (NG == 2) x.s = *reinterpret_cast<const uint32_t*>(vsbase + (size_t)(sl * 4u));
    else x.s = (uint32_t) * reinterpret_cast<const uint16_t*>(vsbase + (size_t)(sl * 2u));
    if (!valid) x.s = 0u;  // (whatever scale that slot has)
#pragma unroll
    for (int i = 0; i < PIECES; ++i)
      x.r[i] = *reinterpret_cast<const v4u*>(vbase + (size_t)((uint32_t)max(slot[i], 0) * (uint32_t)Tiles::VP + (uint32_t)(1024 * i + 16 * lane) % Tiles::VP));
    return x;
  }
  // channel of o[i] in `add`
  static __device__ inline int channel(int lane, int i) { return Tiles::channel(2 * (lane >> 4) + i, lane & 15); }
  // o[0], o[1] += the sums of two channels per lane.  A weight row holds the limbs four times, once for each lane group of the
  // products (the first two take the first scale group's, the others the second's).  Tiles 2q and 2q + 1 are multiplied with the
  // rows of lane group q alone, so two accumulators hold all eight and every lane has two channels.
  static __device__ JF_INLINE void add(const Rows& x, uint8_t* st, int lane, float (&o)[2]) {
    uint8_t* wl = st + Tiles::VST;
    float top[NG];
    int E[NG];
    uint32_t limbs[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      const float v = x.w * bf16_to_f32((uint16_t)(g ? x.s >> 16 : x.s & 0xffffu));
      const uint32_t most = wave_max_u(__builtin_bit_cast(uint32_t, v) & 0x7fffffffu);
      top[g] = uniform_f(__builtin_bit_cast(float, most));
      int e = 0;
      float f;
      if (isfinite(top[g])) {  // (uniform)
        if (top[g] > 0.f) (void)frexpf(top[g], &e);  // top = f * 2^e, f in [0.5, 1)
        f = ldexpf(v, 30 - e);
      } else {  // an infinite weight or a NaN: it alone counts, and `top` becomes the sums' factor
        f = (__builtin_bit_cast(uint32_t, v) & 0x7fffffffu) == most ? copysignf(1.f, v) : 0.f;
      }
      E[g] = 30 - e;
      limbs[g] = ((uint32_t)(int)rintf(f) + 0x808080u) ^ 0x808080u;
    }
    *reinterpret_cast<v4u*>(wl + lane * 16) = (v4u){limbs[0], limbs[0], limbs[NG - 1], limbs[NG - 1]};
#pragma unroll
    for (int i = 0; i < PIECES; ++i) Tiles::stash_piece(st, (1024 * i + 16 * lane) / Tiles::VP, (1024 * i + 16 * lane) % Tiles::VP / 16, x.r[i]);
    wave_lds_fence();
    const uint8_t* wrow = wl + ((lane >> 4) * 16 + tr8_token(lane)) * 16 + (lane & 1) * 8;
    const v2i x0 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i*)(wrow));
    const v2i x1 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i*)(wrow + 128));
    const v4i A = {x0[0], x0[1], x1[0], x1[1]}, zero = {0, 0, 0, 0}, ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
    const v4i sw = __builtin_amdgcn_mfma_i32_16x16x64_i8(A, ones, zero, 0, 0, 0);
    v4i acc[2] = {zero, zero};
    Tiles::spread(st, lane, [&](auto tile, int, const v4i& B) JF_INLINE {
      constexpr int t = decltype(tile)::value;
      const bool own = ((lane & 15) >> 2) == t / 2;  // (lane: a row of the operand)
      v4i Aq;
#pragma unroll
      for (int c = 0; c < 4; ++c) Aq[c] = own ? A[c] : 0;
      acc[t & 1] = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aq, B, acc[t & 1], 0, 0, 0);
    });
    const int lo = Tiles::OFFSET * (sw[0] + (sw[1] << 8)), hi = Tiles::OFFSET * (sw[2] + (sw[3] << 8));
    const bool upper = (lane & 32) != 0;
    const float factor = upper ? top[NG - 1] : top[0];
    const int e = upper ? E[NG - 1] : E[0];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      constexpr int m[2] = {Tiles::times(0), Tiles::times(1)};
      const v4i a = acc[i];
      // (floats hold both: `high` is below 2^24, `low` below 1.004 * 2^24, where it may be rounded to an even number)
      const float low = (float)(a[0] + (a[1] << 8) - m[i] * lo), high = (float)(a[2] + (a[3] << 8) - m[i] * hi);
      const float sum = __builtin_fmaf(high, 65536.f, low) * (m[i] == 4 ? 0.25f : 1.f);
      o[i] += isfinite(factor) ? ldexpf(sum, -e) : sum * factor;
    }
    wave_lds_fence();
  }
};

// The same terms code by code, for few winners of a scan that merges by itself: DW lanes per row, lane dwi holds dword dwi of it
// (INT2, INT4) or two bytes of each of the three planes (INT3) = CPD codes; a wavefront instruction covers WPI rows.
template <int VBITS>
struct PreCorr {
  static constexpr int VP = D * VBITS / 8;
  static constexpr int DW = (VBITS == 3) ? 8 : VP / 4;
  static constexpr int CPD = (VBITS == 3) ? 16 : 32 / VBITS;
  static constexpr int WPI = 64 / DW;
  // INT3: all rows of a batch are requested before the first is used.  Left to itself the compiler requests a row or two and
  // waits: 19 sequences x 16 heads over 4 kv-heads, 4955 positions, K4V3, top-k 512 38.4 us, 36.3 with this.  (The others' one
  // load per row goes ahead anyway, and holding all of them costs registers: 28 x 32 heads over 4 kv-heads, 887 positions,
  // INT4 in 64-channel groups, top-k 512 33.2 us, 37.0 with this.)
  static constexpr bool ALL_AHEAD = VBITS == 3;
  // what a lane requests of a row: its dword, or (INT3) bytes 2*dwi, 2*dwi+1 of every plane
  struct Row {
    uint32_t w[VBITS == 3 ? 3 : 1];
  };
  static __device__ inline Row fetch(const uint8_t* vbase, uint32_t slot, int dwi) {
    Row x;
    if constexpr (VBITS == 3) {
      const uint8_t* row = vbase + (size_t)(slot * (uint32_t)VP) + dwi * 2;
#pragma unroll
      for (int i = 0; i < 3; ++i) x.w[i] = *reinterpret_cast<const uint16_t*>(row + 16 * i);
    } else {
      x.w[0] = *reinterpret_cast<const uint32_t*>(vbase + (size_t)(slot * (uint32_t)VP) + dwi * 4);
    }
    return x;
  }
  // acc[c] += ws * (code c - offset).  Byte `byte` of the dword holds its codes MSB first; channel of code c in the
  // dword = dwi*CPD + c.  code - offset is the code with its top bit flipped, read as a two's complement field.  INT4
  // and INT2: the field goes to the top of a nibble, and one conversion with a byte select turns the nibble into a
  // sixteenth (INT2: a quarter) of its value; the factor, a power of two, sits in the weight, so every product is the
  // same number.  Two instructions per code; the bit-field extract, conversion and multiply-add of the INT3 words
  // take three, and with 256 winners for each of a workgroup's four heads the multiply-adds fill the vector ALU.
  static __device__ inline void add(const Row& row, float ws, float (&acc)[CPD]) {
    const uint32_t word = row.w[0];
    if constexpr (VBITS == 3) {  // the 24-bit words of two 8-code groups
      const uint32_t h0 = row.w[0], h1 = row.w[1], h2 = row.w[2];
      const uint32_t wa = ((h0 & 0xffu) << 16) | ((h1 & 0xffu) << 8) | (h2 & 0xffu);
      const uint32_t wb = ((h0 >> 8) << 16) | ((h1 >> 8) << 8) | (h2 >> 8);
      const uint32_t xa = wa ^ 0x00924924u, xb = wb ^ 0x00924924u;
#pragma unroll
      for (int c = 0; c < CPD; ++c) {
        const int sh = 21 - 3 * (c & 7);
        const int code = (int)((c >= 8 ? xb : xa) << (32 - VBITS - sh)) >> (32 - VBITS);
        acc[c] = __builtin_fmaf(ws, (float)code, acc[c]);
      }
    } else if constexpr (VBITS == 4) {  // even codes: high nibbles
      const float w = ws * 16.f;
      const uint32_t x = word ^ 0x88888888u, xh = x >> 4;
      add_bytes<0, 2>(xh, w, acc);
      add_bytes<1, 2>(x, w, acc);
    } else {
      const float w = ws * 4.f;
      const uint32_t x = word ^ 0xaaaaaaaau;
      add_bytes<0, 4>((x >> 4) & 0x0c0c0c0cu, w, acc);
      add_bytes<1, 4>((x >> 2) & 0x0c0c0c0cu, w, acc);
      add_bytes<2, 4>(x & 0x0c0c0c0cu, w, acc);
      add_bytes<3, 4>((x << 2) & 0x0c0c0c0cu, w, acc);
    }
  }
  // the low nibbles of the four bytes belong to codes FIRST, FIRST + STEP, ...
  template <int FIRST, int STEP>
  static __device__ inline void add_bytes(uint32_t x, float w, float (&acc)[CPD]) {
    float f0, f1, f2, f3;
    asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_0" : "=v"(f0) : "v"(x));
    asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_1" : "=v"(f1) : "v"(x));
    asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_2" : "=v"(f2) : "v"(x));
    asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_3" : "=v"(f3) : "v"(x));
    acc[FIRST] = __builtin_fmaf(w, f0, acc[FIRST]);
    acc[FIRST + STEP] = __builtin_fmaf(w, f1, acc[FIRST + STEP]);
    acc[FIRST + 2 * STEP] = __builtin_fmaf(w, f2, acc[FIRST + 2 * STEP]);
    acc[FIRST + 3 * STEP] = __builtin_fmaf(w, f3, acc[FIRST + 3 * STEP]);
  }
  // Sums over the WPI rows of a wavefront instruction (lanes with equal dwi): every exchange step halves the channels
  // a lane is responsible for (the lane whose offset bit is clear keeps the lower half), so after log2(WPI) steps
  // every lane holds the sums of two channels, acc[0] and acc[1]; -> the first of them.
  static __device__ inline int reduce(float (&acc)[CPD], int lane) {
    int chan = (lane % DW) * CPD;
    auto halve = [&](auto off_c, auto n_c) {
      constexpr int OFF = decltype(off_c)::value, N = decltype(n_c)::value;
      const bool upper = (lane & OFF) != 0;
#pragma unroll
      for (int i = 0; i < N / 2; ++i) {
        if constexpr (OFF == 32) {  // one half-wave swap serves both directions
          const auto sw = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, acc[i]), __builtin_bit_cast(uint32_t, acc[i + N / 2]), false, false);
          acc[i] = __builtin_bit_cast(float, (uint32_t)sw[0]) + __builtin_bit_cast(float, (uint32_t)sw[1]);
        } else {
          const float keep = upper ? acc[i + N / 2] : acc[i];
          const int send = __builtin_bit_cast(int, upper ? acc[i] : acc[i + N / 2]);
          // lane ^ 8: rotation by 8 inside the 16-lane row; lane ^ 16: swizzle inside 32 lanes
          const int recv = (OFF == 8) ? dpp_mov<0x128, 0xf>(0, send) : __builtin_amdgcn_ds_swizzle(send, 0x401F);
          acc[i] = keep + __builtin_bit_cast(float, recv);
        }
      }
      chan += upper ? N / 2 : 0;
    };
    static_assert(DW == 8 || DW == 16, "eight or sixteen lanes per V row");
    if constexpr (DW == 8) {
      halve(std::integral_constant<int, 8>{}, std::integral_constant<int, CPD>{});
      halve(std::integral_constant<int, 16>{}, std::integral_constant<int, CPD / 2>{});
      halve(std::integral_constant<int, 32>{}, std::integral_constant<int, CPD / 4>{});
    } else {
      halve(std::integral_constant<int, 16>{}, std::integral_constant<int, CPD>{});
      halve(std::integral_constant<int, 32>{}, std::integral_constant<int, CPD / 2>{});
    }
    static_assert(CPD / WPI == 2, "two channels per lane after the exchange");
    return chan;
  }
};

// ---------------------------------------------------------------------------------------------------
// ONE: the split is the whole sequence (n_splits == 1), so this workgroup holds everything the merge kernel would
// fetch: it selects the winners, forms the pre-correction terms and writes the step's outputs itself, and no merge is
// launched.  A merge launch costs 9 - 10 us whatever it merges (its loads are first touches, its intervals a chain of
// barriers), 18 us at 1024 rows; the same steps from LDS, four wavefronts per head, cost 4 to 8 us at the end of the
// scan.  Per layer, MI355X, graph replay, when it was made: 32 sequences x 2048 positions, K3V2, 8 kv-heads, top-k 256 37.5 -> 26.7
// us (22.8 since its winners are marked in place and summed on the matrix cores); 32 x 464, K3V4, 4 kv-heads, top-k 64 30.1 -> 19.4;
// 7 x 311, K4V4, 8 kv-heads, G = 2 20.7 -> 16.5.
//
// SHORT: at most one chunk per wavefront (splits of up to NW * 64 positions).  Its V rows are requested along with the key
// rows; the form for longer splits requests V rows with the last two of four key chunks, which a short split never
// reaches, so that it would wait for them from a standing start.  Wavefronts without a chunk request no keys: sixteen
// wavefronts' loads are issued one after the other, some twelve cycles each, before the query set-up's barrier.  Per layer:
// 4 x 8100 positions, B4V4 in 64-channel groups (splits of 1024) 28.0 -> 26.4 us; 1 x 4096, K4V4 (256) 18.3 -> 17.5.
// (Two chunks per wavefront, all four requested at once: 2 to 4 % slower on 32 x 2048.  One form for all lengths that puts
// V rows into the key buffers at run time: the compiler's waits, counted for the shorter path, cost long splits 2 %.)
template <int MODE, int SCHEME, int G, int NG, bool ONE = false, bool SHORT = false>
__global__ __launch_bounds__((ScanLds<SCHEME, G, NG>::NT)) void fused_scan_kernel(FusedParams p) {
  using Lds = ScanLds<SCHEME, G, NG>;
  constexpr bool HAS_K = (MODE == FS_FULL || MODE == FS_STAGE_A);  // key stream and phase A
  constexpr bool HAS_V = (MODE == FS_FULL || MODE == FS_STAGE_B);  // value stream and the P.V part of phase B
  constexpr bool HAS_TOPK = (MODE != FS_STAGE_B);                  // histograms and phase C
  constexpr bool K3 = Lds::K3, KLIMB = Lds::KLIMB, KA = Lds::KA, KB4 = Lds::KB4;
  // INT4 keys over 128 channels in one group: their sums reach 128 * 2^22 * 8 = 2^32 and are put together in two parts
  constexpr bool WIDE_SUM = KB4 && NG == 1;
  constexpr bool V2 = Lds::V2, V3 = Lds::V3;
  // What the outputs and the winners' rows are addressed by follows from the thread's number; the compiler forms it ahead of phase B,
  // and where the value rows in flight leave no registers for it (16 wavefronts, 128 registers) it waits for a chunk of them to put
  // that into scratch memory.  Behind phase B those kernels take the number as a value of its own, for the winners' rows (TIGHT) and
  // for all outputs (TIGHTER): the ones that spilled.  Forming it anew costs the others, which have the registers, 1 to 4 %.
  // Per layer, 32 sequences x 8 kv-heads: K3V3 in two groups, 3900 positions, top-k 256, one head each 29.7 us, with this 28.2; 1900
  // positions, four heads 28.4 / 25.1; A2V2 in two groups, 3900, 128, one head 35.6 / 34.3.
  constexpr bool TIGHT = ONE && !SHORT && Lds::NW == 16 &&
                         (V3 ? !(G == 1 && NG == 1 && (K3 || KA)) : NG == 2 && (KA || (!V2 && G == 4)));
  constexpr bool TIGHTER = (TIGHT && (KA ? NG == 2 : (G > 1 && (G == 4 || NG == 2)))) || (!ONE && !SHORT && V3 && G == 4);
  constexpr int NSET = Lds::NSET;
  constexpr int SEG = Lds::SEG;
  constexpr int KP = Lds::KP;
  constexpr int KROW = Lds::KROW;
  constexpr int VP = Lds::VP;
  constexpr int VROW = Lds::VROW;
  using Tiles = VTiles<SCHEME % 10, NG>;
  constexpr int VOFF = Tiles::OFFSET;  // code offset of the V format
  static_assert(VROW == Tiles::VROW, "one layout of the staged V rows");
  constexpr int NTILE = 8;          // 8 MFMA column tiles of 16 channels
  constexpr int AR = Lds::ACC_REGS;
  constexpr float LOG2E = 1.44269504088896340736f;
  constexpr int NW = Lds::NW, NT = Lds::NT;
  static_assert(!SHORT || MODE == FS_FULL, "the stage-wise forms have no short variant");
  constexpr int MAXIT = SHORT ? 1 : Lds::LMAX / 64 / NW;  // chunks per wavefront

  extern __shared__ __align__(16) uint8_t smem[];
  const int L = p.L;
  float* sc = reinterpret_cast<float*>(smem + Lds::SC_AT);                     // [G][L]
  int* sbase = reinterpret_cast<int*>(smem + Lds::SC_AT + (size_t)G * L * 4);  // [L/16] first slot of each page
  uint8_t* aux = (Lds::SC_AT != 0) ? smem : smem + Lds::aux_offset(L);
  uint8_t* stage = smem + Lds::aux_offset(L) + Lds::AUX;
  int* hist = reinterpret_cast<int*>(aux);  // [G][SEG][256], valid after phase A
  __shared__ float red_f[NW][2 * G];
  __shared__ uint32_t vmax_sh[NW][2];
  __shared__ float m_sh[G], bin_a_sh[G], bin_b_sh[G], lsum_sh[NW][G];
  __shared__ int e_sh[2];
  // Rounding of bf16(c s) for s = 1 + m/128.  INT3: the coefficient 256 * (bf16(3 s) - 3 s) / s.  INT4 (bf16 model): the
  // byte tables the roundings are looked up in and what they are multiples of, 256 / (128 s) (see phase A).
  // At a place known when this is compiled, so that a look-up's address is the index plus a constant the instruction carries.
  __shared__ float eps_k3[K3 ? 128 : 1];
  v4u* const rnd_sh = reinterpret_cast<v4u*>(smem + Lds::RND_AT);
  float* const eps_sh = KB4 ? reinterpret_cast<float*>(smem + Lds::RND_AT + 128 * 16) : eps_k3;
  __shared__ unsigned long long tmax_sh;
  if (threadIdx.x == 0) tmax_sh = 0ull;

  // kv-head fastest: workgroups go to the eight XCDs in turn, and the heads of one (sequence, split) have equal work.
  // With the split fastest an XCD got the same split (mod 8) of every sequence: in a batch of different lengths the
  // early splits, which all sequences have, on some XCDs and the late, mostly empty ones on others.  Per layer, graph
  // replay: 16 sequences of 983 .. 16384 positions, K4V4 63.7 -> 62.2 us (with splits of 1024: 125 -> 96); equal
  // lengths gain too, 4 x 32768 K3V2 37.0 -> 36.3, 131072 K4V4 49.7 -> 48.6.
  const int hkv = blockIdx.x, split = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: keeps wave-derived addresses in SGPRs
  const int S = max(0, min(p.max_S, p.seq_lens[b]));
  const int s0 = split * L;
  const int s1 = min(s0 + L, S);
  const int n = max(0, s1 - s0);
  const int s_cover = min(s0 + L, p.max_S);
  const int n_cover = max(0, s_cover - s0);
  const int64_t* bt = p.block_table + (size_t)b * p.max_blocks;
  // GA query heads belong to this kv-head; the template's G may be larger (the next of 1, 2, 4, 8, 16): the heads
  // past GA are zero query rows whose arithmetic runs along and whose results are never stored
  const int GA = p.g_act;
  const size_t head0 = (size_t)b * p.H_q + (size_t)hkv * GA;
  const size_t part_base = head0 * p.n_splits + split;  // + h * n_splits
  const uint8_t* kbase = p.k_data + (size_t)hkv * p.num_slots * KP;
  const uint8_t* vbase = p.v_data + (size_t)hkv * p.num_slots * VP;
  const uint8_t* vsbase = reinterpret_cast<const uint8_t*>(p.v_scales + (size_t)hkv * p.num_slots * NG);

  long long* clk = (kDebugHooks && p.phase_clock) ? p.phase_clock + (((size_t)b * p.H_kv + hkv) * p.n_splits + split) * 10 : nullptr;
  if (clk && tid == 0) clk[0] = JF_CLK();

  // The page-table entry and the query elements of this thread do not depend on the sequence length: they
  // are requested first, so their latency runs in parallel with the load of seq_lens[b] instead of after it.
  const int nch_cover = (n_cover + 63) >> 6;
  // (both unconditional, on clamped indices: under a condition the compiler waits for each load inside its branch,
  // one cold miss after the other)
  const int64_t bt_mine = bt[min((s0 >> 4) + tid, p.max_blocks - 1)];  // LMAX / 16 <= NT: one entry per thread covers the split
  constexpr int QN = NSET * 4 * D;               // elements of the padded query block (whole head sets)
  constexpr int QPT = (QN + NT - 1) / NT;
  uint16_t qraw[QPT];
#pragma unroll
  for (int it = 0; it < QPT; ++it) qraw[it] = HAS_K ? p.q[head0 * D + min(it * NT + tid, GA * D - 1)] : (uint16_t)0;
  auto q_elem = [&](int it) -> float { return (it * NT + tid < GA * D) ? bf16_to_f32(qraw[it]) : 0.f; };

  if (n == 0) {  // nothing valid in this split: padding scores, empty partials
    if (p.scores)
      for (int i = tid; i < GA * n_cover; i += NT)
        p.scores[(head0 + i / n_cover) * (size_t)p.max_S + s0 + (i % n_cover)] = -INFINITY;
    if constexpr (MODE == FS_STAGE_A)
      if (p.scores_only) return;
    if constexpr (ONE) {  // no winners, zero sums
      for (int i = tid; HAS_TOPK && i < GA * p.top_k; i += NT) {
        p.topk_idx[head0 * p.top_k + i] = -1;
        p.topk_slots[head0 * p.top_k + i] = -1;
      }
      for (int i = tid; HAS_V && i < GA * D; i += NT) {
        p.o_hat[head0 * D + i] = 0.f;
        p.o_old[head0 * D + i] = 0.f;
        if (MODE == FS_FULL && p.blend_out)
          p.blend_out[head0 * D + i] = f32_to_bf16(__builtin_fmaf(0.f, bf16_to_f32(p.blend_o_new[head0 * D + i]), 0.f) - 0.f);
      }
      if (tid < GA) {
        if (HAS_V) p.W[head0 + tid] = 0.f;
        if (p.softmax_m) {
          p.softmax_m[head0 + tid] = 0.f;
          p.softmax_inv_z[head0 + tid] = 0.f;
        }
      }
      return;
    }
    for (int i = tid; i < GA * D; i += NT) p.part_o[(part_base + (size_t)(i / D) * p.n_splits) * D + (i % D)] = 0.f;
    if (tid < GA) {
      p.part_m[part_base + (size_t)tid * p.n_splits] = -INFINITY;
      p.part_l[part_base + (size_t)tid * p.n_splits] = 0.f;
      p.cand_edge[part_base + (size_t)tid * p.n_splits] = -INFINITY;
    }
    // unused candidate slots hold key 0 (no score maps to it); a list's length is a multiple of 4
    for (int h = wave / (NW / 4); HAS_TOPK && h < GA; h += 4) {
      uint32_t* ck = p.cand_key + (part_base + (size_t)h * p.n_splits) * p.Kc;
      for (int i = (wave % (NW / 4) * 64 + lane) * 4; i < p.Kc; i += NW / 4 * 256) *reinterpret_cast<v4u*>(ck + i) = (v4u){0u, 0u, 0u, 0u};
    }
    return;
  }

  // A candidate list with room for all of the split's positions takes them all, in place: no selection buckets, no cut, no
  // compaction.  1 x 4096 positions, K4V4, top-k 64 (splits of 256), per layer 17.4 -> 15.5 us.  (Short splits only: the
  // test in the value stream costs the long ones, which have room for all of them in the widest corrections only, 0.8 %.)
  const bool take_all = SHORT && !ONE && n <= p.Kc;  // (uniform)

  // Page table of the split: one entry per 16 positions of every 64-token chunk that is touched.  Table
  // entries past the last valid position may hold anything: those pages read slot 0 instead, so every row
  // address formed below is in bounds (those rows' scores are masked to -inf, their softmax weights are
  // exactly zero).
  const int nch = (n + 63) >> 6;
  if (tid < nch_cover * 4) sbase[tid] = (tid <= ((n - 1) >> 4)) ? (int)(bt_mine * BS) : 0;
  lds_barrier();

  // ---- key stream, set-up.  A chunk is 64 consecutive positions = 4 pages; its rows are fetched with
  // 16-byte loads whose lane addresses are consecutive inside a page, staged in this wavefront's LDS area
  // in position order, and read back in the layout the arithmetic wants.
  uint8_t* kst = stage + wave * Lds::WAVE_STAGE;
  constexpr int KLD = KP / 16;  // 16-byte loads per lane and chunk
  uint32_t kl_page[KLD], kl_off[KLD], kl_lds[KLD];
#pragma unroll
  for (int i = 0; i < KLD; ++i) {
    const int o = 1024 * i + 16 * lane;  // byte offset inside the chunk's 64 rows
    kl_page[i] = (uint32_t)(o / (16 * KP));
    kl_off[i] = (uint32_t)(o % (16 * KP));
    kl_lds[i] = (uint32_t)((o / KP) * KROW + (o % KP));
  }
  const uint8_t* ksb = reinterpret_cast<const uint8_t*>(p.k_scales + (size_t)hkv * p.num_slots * (KLIMB ? NG : 1));
  const uint8_t* kzb = KA ? reinterpret_cast<const uint8_t*>(p.k_zp + (size_t)hkv * p.num_slots * NG) : nullptr;
  constexpr bool SPREP = HAS_K && Lds::SPREP;
  // one scale word per lane (lane = token of the chunk), handed to the lanes that work on the token through the table
  // (SPREP) or a lane permutation; the asymmetric keys load scales and zero-points per page
  constexpr bool SL = HAS_K && !KA;
  struct KBuf {
    v4u r[KLD];
    uint32_t s[SL ? 1 : 4];   // scale words: of the lane's token (SL), or of token t16 of each of the four pages
    uint32_t z[KA ? 4 : 1];  // zero-points of the asymmetric keys, packed like the scales
  };
  const int t16 = lane & 15, lg = lane >> 4;
  constexpr int KNG = KLIMB ? NG : 1;  // key scales per row
  auto issue_k = [&](int chunk) -> KBuf {
    KBuf kbuf;
    // (the scales first: they are copied out of the buffer one chunk earlier than the rows are, and loads return in order)
    if constexpr (SL) {
      const int tl = chunk * 64 + lane;
      const uint32_t slot = (uint32_t)(sbase[tl >> 4] + (tl & 15));
      if (KNG == 2) kbuf.s[0] = *reinterpret_cast<const uint32_t*>(ksb + (size_t)(slot * 4u));
      else kbuf.s[0] = (uint32_t) * reinterpret_cast<const uint16_t*>(ksb + (size_t)(slot * 2u));
    }
#pragma unroll
    for (int j = 0; j < (SL ? 0 : 4); ++j) {
      const int sb = __builtin_amdgcn_readfirstlane(sbase[chunk * 4 + j]);  // first slot of the page (uniform)
      const uint8_t* srow = ksb + (size_t)sb * (KNG * 2) + t16 * (KNG * 2);
      if (KNG == 2) kbuf.s[SL ? 0 : j] = *reinterpret_cast<const uint32_t*>(srow);
      else kbuf.s[SL ? 0 : j] = *reinterpret_cast<const uint16_t*>(srow);
      if constexpr (KA) {
        const uint8_t* zrow = kzb + (size_t)sb * (KNG * 2) + t16 * (KNG * 2);
        if (KNG == 2) kbuf.z[j] = *reinterpret_cast<const uint32_t*>(zrow);
        else kbuf.z[j] = *reinterpret_cast<const uint16_t*>(zrow);
      }
    }
#pragma unroll
    for (int i = 0; i < KLD; ++i) {
      const uint32_t sb = (uint32_t)sbase[chunk * 4 + kl_page[i]];
      // (streaming hint: a key row is read exactly once; measured 0.6 - 2 us per launch against plain loads.  The
      // value rows keep the default policy: the merge kernel gathers the winners' rows again.)
      kbuf.r[i] = __builtin_nontemporal_load(reinterpret_cast<const v4u*>(kbase + (size_t)(sb * (uint32_t)KP + kl_off[i])));
    }
    return kbuf;
  };
  // the scale word of token t16 of page j
  auto scale_word = [&](const uint32_t (&Sx)[4], int j) -> uint32_t {
    if constexpr (SL) return (uint32_t)__builtin_amdgcn_ds_bpermute(4 * (16 * j + t16), (int)Sx[0]);
    else return Sx[j];
  };
  auto stash_k = [&](const KBuf& kbuf) {
#pragma unroll
    for (int i = 0; i < KLD; ++i) *reinterpret_cast<v4u*>(kst + kl_lds[i]) = kbuf.r[i];
  };
  // first two chunks of this wavefront and the V scales of the split start now, before the query set-up
  KBuf Ka = {}, Kb = {};
  // (every wavefront requests, chunk or not: the number of loads in flight at each later wait is then the same on every
  // path, and the compiler's waits leave the younger loads in flight)
  if constexpr (HAS_K && !SHORT) Ka = issue_k(min(wave, nch_cover - 1));
  constexpr int VSPT = MAXIT;  // one word per thread and step
  // (positions past the split's end read the scale of its last row again: straight-line code whose loads leave
  // together, and the only use of these values is their maximum)
  uint32_t vsw[VSPT];
#pragma unroll
  for (int i = 0; i < VSPT; ++i) vsw[i] = 0u;
  auto request_vs = [&]() {
    uint32_t vs_slot[VSPT];
#pragma unroll
    for (int i = 0; i < VSPT; ++i) {
      const int t = min(tid + i * NT, n - 1);
      vs_slot[i] = (uint32_t)(sbase[t >> 4] + (t & 15));
    }
#pragma unroll
    for (int i = 0; i < VSPT; ++i) {
      if (NG == 2) vsw[i] = *reinterpret_cast<const uint32_t*>(vsbase + (size_t)(vs_slot[i] * 4u));
      else vsw[i] = (uint32_t) * reinterpret_cast<const uint16_t*>(vsbase + (size_t)(vs_slot[i] * 2u));
    }
  };
  if constexpr (SHORT) {
    if (wave < nch_cover) {  // (a wavefront without a chunk requests nothing: its loads would only be in the others' way)
      Ka = issue_k(wave);
      request_vs();
    }
  } else if constexpr (HAS_V) {
    request_vs();
  }
  if constexpr (!HAS_K) {
    // the scores are an input: no query constants
  } else if constexpr (KLIMB) {
    // Query rows -> 23-bit fixed point per (head, scale group), three balanced int8 limbs, written in the
    // byte order of the MFMA A operand.  One element per thread; group statistics by wavefront reductions.
    K3Prep<NSET>* prep = reinterpret_cast<K3Prep<NSET>*>(aux);
    // (the rounding table is built by two wavefronts that have no query rows to prepare, where there are such)
    constexpr int EPS_T0 = (QN / 64 <= NW - 2) ? NT - 128 : 0;
    if ((K3 || KB4) && tid >= EPS_T0 && tid < EPS_T0 + 128) {
      const int m = tid - EPS_T0;
      const float sm = 1.0f + (float)m * (1.0f / 128.0f);
      if constexpr (KB4) {
        // in units of 1/128 a rounding is a whole number of at most 4
        auto rounding = [&](float c) -> int { return (int)(128.0f * (bf16_to_f32(f32_to_bf16(c * sm)) - c * sm)); };
        const int r3 = rounding(3.f), r5 = rounding(5.f), r7 = rounding(7.f);
        auto bytes = [](int b0, int b1, int b2, int b3) -> uint32_t {
          return (uint32_t)(b0 & 255) | ((uint32_t)(b1 & 255) << 8) | ((uint32_t)(b2 & 255) << 16) | ((uint32_t)b3 << 24);
        };
        // first the codes 0..7, then -8..-1; each entry less what the other table's look-up yields for the same code
        const int n1 = -r7 + (r3 < 0 ? 1 : 0), n2 = -2 * r3 + (r5 < -1 ? 1 : 0), n3 = -r5 + (r7 < -1 ? 1 : 0), n5 = 1 - r3;
        rnd_sh[m] = (v4u){bytes(n1 < 0 ? 1 : 0, n3 < 0 ? 1 : 0, n5 < 0 ? 1 : 0, r3), bytes(0, r5 + 1, 2 * r3 + 1, r7 + 1),
                          bytes(0, n1, n2, n3), bytes(0, n5, 1, 1)};
        eps_sh[m] = 2.0f / sm;
      } else {
        const float t = 3.0f * sm;  // exact in fp32
        eps_sh[m] = 256.0f * ((bf16_to_f32(f32_to_bf16(t)) - t) / sm);
      }
    }
    // stores the three limbs of element (h, d) in the byte order of the MFMA A operand
    auto put_limbs = [&](int h, int d, int qf) {
      const int l0 = (int)(int8_t)(qf & 255);
      const int r1 = (qf - l0) >> 8;
      const int l1 = (int)(int8_t)(r1 & 255);
      const int l2 = (r1 - l1) >> 8;
      const int set = h >> 2, hh = h & 3;
      // A lane of phase A spreads the 32 channels 32*lg .. 32*lg+31 of its token into two 16-byte operands u = 0, 1
      // (dword e, byte b).  INT3 (plane spread): channel 8b + 4u + e; INT2 (four codes per byte): channel 16u + 4b + e;
      // INT4 (nibble spread of the lane's four dwords): channel 16u + 8(e >> 1) + 2b + (e & 1).
      // With two scale groups MFMA g covers group g only (see the lane swap in phase A).
      const int u = K3 ? ((d >> 2) & 1) : ((d >> 4) & 1);
      const int mi = (NG == 2) ? (d >> 6) : u;
      const int kb = (NG == 2) ? (((d >> 5) & 1) + 2 * u) : (d >> 5);
      const int by = KB4 ? (4 * (2 * ((d >> 3) & 1) + (d & 1)) + ((d >> 1) & 3))
                         : (4 * (d & 3) + (K3 ? ((d >> 3) & 3) : ((d >> 2) & 3)));
      prep->aop[set][4 * hh + 0][kb][mi][by] = (int8_t)l0;
      prep->aop[set][4 * hh + 1][kb][mi][by] = (int8_t)l1;
      prep->aop[set][4 * hh + 2][kb][mi][by] = (int8_t)l2;
      prep->aop[set][4 * hh + 3][kb][mi][by] = 0;
    };
    // the codes are used unsigned: offset 8 (INT4), 4 (INT3) or 2 (INT2); WIDE_SUM keeps the query's sum itself
    constexpr int CODE_OFF4 = KB4 ? (WIDE_SUM ? 1 : 8) : (K3 ? 4 : 2);
    if constexpr (NG == 2) {
      // a wavefront's 64 elements are one scale group of one head: its statistics never leave the wavefront
#pragma unroll
      for (int it = 0; it < QPT; ++it) {
        const int c = it * NW + wave;  // 64-channel half row of this wavefront
        if (c * 64 >= QN) continue;    // uniform per wavefront
        const int i = it * NT + tid, h = i >> 7, d = i & 127;
        const float x = q_elem(it);
        const float amax = __builtin_bit_cast(float, wave_max_u(abs_bits(x)));
        int e = 0;
        if (amax > 0.f && isfinite(amax)) (void)frexpf(amax, &e);  // amax = f * 2^e, f in [0.5, 1)
        const int qf = (int)rintf(ldexpf(x, 22 - e));
        const int sum = wave_sum_i(qf);
        put_limbs(h, d, qf);
        if (lane == 0) {
          prep->sq4[h][c & 1] = CODE_OFF4 * sum;
          prep->qsc[h][c & 1] = ldexpf(p.attn_scale, e - 22);
        }
      }
    } else {
#pragma unroll
      for (int it = 0; it < QPT; ++it) {
        const int c = it * NW + wave;  // 64-channel half row of this wavefront
        if (c * 64 < QN) {             // uniform per wavefront
          const float am = __builtin_bit_cast(float, wave_max_u(abs_bits(q_elem(it))));
          if (lane == 0) prep->amax_w[c] = am;
        }
      }
      lds_barrier();
#pragma unroll
      for (int it = 0; it < QPT; ++it) {
        const int i = it * NT + tid, h = i >> 7, d = i & 127;
        const float x = q_elem(it);
        const int c = it * NW + wave;
        if (c * 64 >= QN) continue;
        const float amax = fmaxf(prep->amax_w[c & ~1], prep->amax_w[c | 1]);
        int e = 0;
        if (amax > 0.f && isfinite(amax)) (void)frexpf(amax, &e);  // amax = f * 2^e, f in [0.5, 1)
        const int qf = (int)rintf(ldexpf(x, 22 - e));
        const int s = wave_sum_i(qf);
        if (lane == 0) {
          prep->sum_w[c] = s;
          prep->exp_w[c] = e;
        }
        put_limbs(h, d, qf);
      }
      lds_barrier();
      if (tid < NSET * 4) {
        const int h = tid;
        prep->sq4[h][0] = CODE_OFF4 * (prep->sum_w[2 * h] + prep->sum_w[2 * h + 1]);
        prep->qsc[h][0] = ldexpf(p.attn_scale, prep->exp_w[2 * h] - 22);
      }
    }
  } else {
    // int8 quantisation of the query rows per 32 channels (int8tc_qk_scores.cu:250-290), one element per thread;
    // heads past G are zero rows
    QInt8F<NSET>* qsh = reinterpret_cast<QInt8F<NSET>*>(aux);
#pragma unroll
    for (int it = 0; it < QPT; ++it) {
      const int i = it * NT + tid;
      if (i < QN) {  // uniform per wavefront: QN is a multiple of 64
        const int h = i >> 7, d = i & 127, kk = d >> 5;
        const float x = q_elem(it);
        const float a = __builtin_bit_cast(float, half_max_u(abs_bits(x)));
        const float sq = fmaxf(a / 127.0f, 1e-12f);
        const float inv = 1.0f / sq;
        const int v = max(-128, min(127, (int)rintf(x * inv)));
        const int sv = half_sum_i(v);
        // channel d sits in MFMA d>>6, k-block (d>>4)&3; inside the k-block's 16 bytes the nibble spread of two
        // packed dwords yields: even channels of bytes 0-3, odd channels of bytes 0-3, then the same for bytes 4-7
        const int set = h >> 2, hh = h & 3, mi = d >> 6, kb = (d >> 4) & 3;
        const int j2 = (d & 15) >> 1, odd = d & 1;
        const int by = (j2 >> 2) * 8 + odd * 4 + (j2 & 3);
#pragma unroll
        for (int r = 0; r < 4; ++r) qsh->aop[set][4 * hh + r][kb][mi][by] = (r == kk) ? (int8_t)v : (int8_t)0;
        if ((lane & 31) == 0) {
          qsh->qs[h][kk] = sq;
          qsh->sum8[h][kk] = 8 * sv;
        }
      }
    }
  }
  lds_barrier();
  if constexpr (HAS_K && !SHORT) Kb = issue_k(min(wave + NW, nch_cover - 1));
  if (clk && tid == 0) clk[7] = JF_CLK();

  // ---- V stream, set-up (same scheme as the key stream)
  uint8_t* vst = stage + wave * Lds::WAVE_STAGE;  // [64][VROW], this wavefront only
  uint8_t* wl = vst + Lds::VST;                   // [NG][NSET][64 tokens][16]
  constexpr int VLD = VP / 16;
  uint32_t vl_page[VLD], vl_off[VLD], vl_lds[VLD];
#pragma unroll
  for (int i = 0; i < VLD; ++i) {
    const int o = 1024 * i + 16 * lane;
    vl_page[i] = (uint32_t)(o / (16 * VP));
    vl_off[i] = (uint32_t)(o % (16 * VP));
    const int row = o / VP, q16 = (o % VP) / 16;
    vl_lds[i] = Lds::VSWZ ? (uint32_t)(row * VROW + ((q16 ^ ((row >> 2) & 3)) * 16))
                          : (uint32_t)(row * VROW + (o % VP) + (V3 ? 8 * ((row >> 4) & 1) : 0));  // (INT3: first half's place)
  }
  // (the V scales of a chunk are not fetched again: position chunk * 64 + lane of step `it` is tid + it * NT, whose
  // scale word this thread has held in vsw[it] since the set-up)
  struct VBuf {
    v4u r[VLD];
  };
  auto issue_v = [&](int chunk) -> VBuf {
    VBuf vbuf;
    // (SHORT, a chunk the wavefront does not have: all lanes read one place)
    const uint32_t lm = (!SHORT || chunk < nch) ? 0xffffffffu : 0u;
    if constexpr (SHORT) chunk = (lm != 0u) ? chunk : 0;
#pragma unroll
    for (int i = 0; i < VLD; ++i) {
      const uint32_t sb = (uint32_t)sbase[chunk * 4 + (vl_page[i] & lm)];
      vbuf.r[i] = *reinterpret_cast<const v4u*>(vbase + (size_t)(sb * (uint32_t)VP + (vl_off[i] & lm)));
    }
    return vbuf;
  };
  // the first two V chunks are requested while the last key chunks are being worked on
  VBuf Va = {}, Vb = {};
  bool va_requested = SHORT, vb_requested = SHORT;  // (uniform per wavefront)
  auto prefetch_v = [&](int it) {
    if constexpr (MODE == FS_FULL && !SHORT) {
      if (it == MAXIT - 2) {
        Va = issue_v(min(wave, nch - 1));
        va_requested = true;
      }
      if (it == MAXIT - 1) {
        Vb = issue_v(min(wave + NW, nch - 1));
        vb_requested = true;
      }
    }
  };
  if constexpr (SHORT) Va = issue_v(wave);
  if constexpr (MODE == FS_STAGE_B) {  // nothing to wait for: the value stream starts at once
    Va = issue_v(min(wave, nch - 1));
    Vb = issue_v(min(wave + NW, nch - 1));
  }


  // A chunk the sequence ends in (0 < n_local < 64 valid rows; uniform): the staged rows past the end and their
  // scale words become copies of the last valid row, so the stream's arithmetic runs without a validity select per
  // score (a copy of a valid score changes neither extremum), and `mask_tail` afterwards stores -inf over what those
  // positions produced.  A chunk past the end (n_local <= 0) is not worked through at all.
  auto clone_last_row = [&](int n_local, uint32_t (&Sx)[4], uint32_t (&Zx)[4]) JF_INLINE {
    const int last = n_local - 1, jl = last >> 4;
    if constexpr (SL) {  // one scale word per lane (= token): Sx[0]
      const uint32_t sl = (uint32_t)__builtin_amdgcn_readlane((int)Sx[0], last);
      Sx[0] = (lane >= n_local) ? sl : Sx[0];
    } else {
      uint32_t sl = Sx[0], zl = Zx[0];
#pragma unroll
      for (int j = 1; j < 4; ++j) {
        sl = (jl == j) ? Sx[j] : sl;
        zl = (jl == j) ? Zx[j] : zl;
      }
      sl = (uint32_t)__builtin_amdgcn_readlane((int)sl, last & 15);
      zl = (uint32_t)__builtin_amdgcn_readlane((int)zl, last & 15);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool past = 16 * j + (lane & 15) >= n_local;
        Sx[j] = past ? sl : Sx[j];
        Zx[j] = past ? zl : Zx[j];
      }
    }
    constexpr int RDW = KP / 4;  // dwords per staged row
    const uint8_t* src = kst + last * KROW;
    for (int i = lane; i < (64 - n_local) * RDW; i += 64) {
      const int r = n_local + i / RDW, dw = i % RDW;
      *reinterpret_cast<uint32_t*>(kst + r * KROW + 4 * dw) = *reinterpret_cast<const uint32_t*>(src + 4 * dw);
    }
    wave_lds_fence();
  };
  auto mask_tail = [&](int chunk, int n_local) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int tl = 16 * j + (lane & 15);
      if (tl >= n_local) {
#pragma unroll
        for (int set = 0; set < NSET; ++set) {
          const int h = set * 4 + (lane >> 4);
          if ((G % 4 == 0) || h < G) sc[h * L + chunk * 64 + tl] = -INFINITY;
        }
      }
    }
  };

  // ------------------------------------------------------------------ phase A
  if constexpr (!HAS_K) {
    // the split's scores come from the caller's (B, H_q, max_S) tensor: -> LDS, running maximum per head;
    // positions past the sequence (and the rest of the last chunk) become -inf
#pragma unroll
    for (int h = 0; h < G; ++h) {
      const float* srow = p.scores_in + (head0 + min(h, GA - 1)) * (size_t)p.max_S + s0;  // (past GA: a copy, unused)
      float mx = -INFINITY, mn = INFINITY;
      for (int t = tid; t < nch * 64; t += NT) {
        const float v = (t < n) ? srow[t] : -INFINITY;
        sc[h * L + t] = v;
        mx = fmaxf(mx, v);
        mn = fminf(mn, (t < n) ? v : INFINITY);
      }
      mx = wave_max(mx);
      mn = -wave_max(-mn);
      if (lane == 0) {
        red_f[wave][h] = mx;
        red_f[wave][G + h] = mn;  // (the minimum shapes the selection buckets)
      }
    }
  } else if constexpr (KLIMB) {
    // INT2 keys: the same scheme without the second contraction: (code - 2) * scale is exact in bf16 for every code,
    // so the reference's rounding (int2_qk_scores.cu:66-79) changes nothing; the codes sit four to a byte, MSB first.
    // INT3 keys on v_mfma_i32_16x16x64_i8.  The bf16 query row is held exactly as a 23-bit fixed-point number
    // per (head, scale group), split into three balanced int8 limbs that sit in different A-operand rows
    // (row = 4*head + limb), so one MFMA yields the three integer partial sums of a (token, head) in the
    // registers of one lane.  K codes are spread from the three byte planes to one byte per code with
    // shift/mask on whole dwords (4 codes per VALU operation) and used unsigned; the -4 offset is removed with
    // the per-row constant 4*sum(q).  Lane (token, k-block lg) holds channels 32*lg .. 32*lg+31, i.e. lanes
    // 0-31 hold scale group 0 and lanes 32-63 group 1; one v_permlane32_swap per dword regroups them so that
    // each MFMA contracts over exactly one scale group.  The reference rounds every dequantised key to bf16
    // (int3_qk_scores.cu:90-99); only codes +-3 are inexact, so that rounding is reproduced by a second
    // contraction with the indicator (+1 for code 7, -1 for code 1, byte LUT through v_perm_b32) weighted by
    // eps = (bf16(3s) - 3s) / s, which depends on the 7 mantissa bits of the scale only (128-entry table).
    const K3Prep<NSET>* prep = reinterpret_cast<const K3Prep<NSET>*>(aux);
    v4i Aop[NSET][2];
    int sq4[NSET][NG];
    float qsc[NSET][NG];
#pragma unroll
    for (int set = 0; set < NSET; ++set) {
#pragma unroll
      for (int mi = 0; mi < 2; ++mi) Aop[set][mi] = *reinterpret_cast<const v4i*>(&prep->aop[set][t16][lg][mi][0]);
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        sq4[set][g] = prep->sq4[set * 4 + lg][g];
        qsc[set][g] = prep->qsc[set * 4 + lg][g];
      }
    }
    // this lane's plane dwords (INT2: its 8 bytes, INT4: its 16 bytes) of token t16 of a page
    const uint8_t* krd = kst + t16 * KROW + lg * (K3 ? 4 : (KB4 ? 16 : 8));
    float mxl[NSET], mnl[NSET];
#pragma unroll
    for (int set = 0; set < NSET; ++set) {
      mxl[set] = -INFINITY;
      mnl[set] = INFINITY;
    }
    float sumq[NSET][NG];  // fixed-point sum of the query over the scale group (asymmetric keys)
#pragma unroll
    for (int set = 0; set < NSET; ++set)
#pragma unroll
      for (int g = 0; g < NG; ++g) sumq[set][g] = (float)(sq4[set][g] / 2);
    (void)sumq;
    // (the offset term -sq4 of the limb-0 sum enters as the accumulator's initial value: exact, and one subtraction
    // per token, head and group less)
    v4i Cin[NSET][NG];
#pragma unroll
    for (int set = 0; set < NSET; ++set)
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        if constexpr (WIDE_SUM) {  // 8 sum(q) = 256 * (sum(q) >> 5) + 8 * (sum(q) & 31), the parts to two limbs
          Cin[set][g] = (v4i){-8 * (sq4[set][g] & 31), -(sq4[set][g] >> 5), 0, 0};
        } else {
          Cin[set][g] = (v4i){-sq4[set][g], 0, 0, 0};
        }
      }
    auto body = [&](int chunk, const uint32_t (&Sx)[4], const uint32_t (&Zx)[4]) JF_INLINE {
      (void)Zx;
      // all LDS reads of the chunk first (plane dwords of the four pages, rounding coefficients), then arithmetic
      uint32_t Pj[4][3];
      float sgj[4][NG], egj[4][NG];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint8_t* rp = krd + j * 16 * KROW;
        if constexpr (K3) {
          Pj[j][0] = *reinterpret_cast<const uint32_t*>(rp);
          Pj[j][1] = *reinterpret_cast<const uint32_t*>(rp + 16);
          Pj[j][2] = *reinterpret_cast<const uint32_t*>(rp + 32);
        } else if constexpr (KB4) {  // (read where they are used: the registers are the tighter resource)
        } else {
          const v2u x = *reinterpret_cast<const v2u*>(rp);
          Pj[j][0] = x[0];
          Pj[j][1] = x[1];
          Pj[j][2] = 0u;
        }
        if constexpr (SPREP) {  // the token's entry of the table the wavefront has just written
          const uint8_t* sp = kst + Lds::KST + (16 * j + t16) * Lds::SCT;
          if (NG == 2) {
            const v4f x = *reinterpret_cast<const v4f*>(sp);
            sgj[j][0] = x[0];
            sgj[j][NG - 1] = x[1];
            egj[j][0] = x[2];
            egj[j][NG - 1] = x[3];
          } else {
            const v2f x = *reinterpret_cast<const v2f*>(sp);
            sgj[j][0] = x[0];
            egj[j][0] = x[1];
          }
        } else if constexpr (!KB4) {
          const uint32_t sw = scale_word(Sx, j);
          sgj[j][0] = bf16_to_f32((uint16_t)(sw & 0xffffu));
          egj[j][0] = K3 ? eps_sh[sw & 0x7fu] : 0.f;
          if (NG == 2) {
            sgj[j][NG - 1] = bf16_to_f32((uint16_t)(sw >> 16));
            egj[j][NG - 1] = K3 ? eps_sh[(sw >> 16) & 0x7fu] : 0.f;
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v4i Bc[2], Br[2];
        v4u X = {0u, 0u, 0u, 0u};
        if constexpr (KB4) {
          // (one page at a time, the scheduler would otherwise hold the operands of all four and spill)
          __builtin_amdgcn_sched_barrier(0);
          X = *reinterpret_cast<const v4u*>(krd + j * 16 * KROW);
        } else {
#pragma unroll
          for (int i = 0; i < 3; ++i) X[i] = Pj[j][i];
        }
        const uint32_t P0 = X[0], P1 = X[1], P2 = X[2];
        if constexpr (KB4) {  // two codes per byte, the even channel in the high nibble
          const uint32_t P3 = X[3];
          Bc[0] = (v4i){(int)((P0 >> 4) & 0x0f0f0f0fu), (int)(P0 & 0x0f0f0f0fu), (int)((P1 >> 4) & 0x0f0f0f0fu), (int)(P1 & 0x0f0f0f0fu)};
          Bc[1] = (v4i){(int)((P2 >> 4) & 0x0f0f0f0fu), (int)(P2 & 0x0f0f0f0fu), (int)((P3 >> 4) & 0x0f0f0f0fu), (int)(P3 & 0x0f0f0f0fu)};
        } else if constexpr (K3) {
          Bc[0][0] = (int)((P0 >> 5) & 0x07070707u);
          Bc[0][1] = (int)((P0 >> 2) & 0x07070707u);
          Bc[0][2] = (int)(((P0 << 1) & 0x06060606u) | ((P1 >> 7) & 0x01010101u));
          Bc[0][3] = (int)((P1 >> 4) & 0x07070707u);
          Bc[1][0] = (int)((P1 >> 1) & 0x07070707u);
          Bc[1][1] = (int)(((P1 << 2) & 0x04040404u) | ((P2 >> 6) & 0x03030303u));
          Bc[1][2] = (int)((P2 >> 3) & 0x07070707u);
          Bc[1][3] = (int)(P2 & 0x07070707u);
        } else {  // four codes per byte, MSB first: dword e of operand u holds code e of each of the four bytes
          (void)P2;
          Bc[0] = (v4i){(int)((P0 >> 6) & 0x03030303u), (int)((P0 >> 4) & 0x03030303u), (int)((P0 >> 2) & 0x03030303u), (int)(P0 & 0x03030303u)};
          Bc[1] = (v4i){(int)((P1 >> 6) & 0x03030303u), (int)((P1 >> 4) & 0x03030303u), (int)((P1 >> 2) & 0x03030303u), (int)(P1 & 0x03030303u)};
        }
        if (NG == 2) {
          // Bc[0] <- lanes 0-31 keep their first half, lanes 32-63 receive the second half of lane-32;
          // Bc[1] <- lanes 0-31 receive the first half of lane+32, lanes 32-63 keep their second half
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const auto sw = __builtin_amdgcn_permlane32_swap((uint32_t)Bc[0][e], (uint32_t)Bc[1][e], false, false);
            Bc[0][e] = (int)sw[0];
            Bc[1][e] = (int)sw[1];
          }
        }
        if constexpr (KB4) {
          // khat = bf16((u - 8) s) for the unsigned nibble u and s = 2^e (1 + m/128) is (c + r_c(m) / (128 + m)) s, c = u - 8,
          // with whole numbers r_c, |r_c| <= 4, that depend on the scale's mantissa alone: zero but for c = +-3, 5, 7 (and
          // +-6 = 2 * +-3), and odd in c.  So next to the code contraction there is one with the bytes r_c, each the sum of two
          // byte look-ups in tables of the lane's token: one that is right for the codes >= 0 (selector u ^ 8 = c) and one for
          // the codes < 0 (selector u = c + 8).  Selectors 8..15 of v_perm_b32 are not table entries but constants (8..11 the
          // signs of bytes 1, 3, 5, 7, 12 zero, 13..15 minus one); the tables hold what makes the two sums come out, and the
          // matrix cores, which are idle mostly, do the adding: three vector instructions per dword.
          // (Three contractions with the signed indicators of +-3, +-5 and +-7 from constant tables, each with its own
          // coefficient per token, took seven and the scan's phase A 12.5 k cycles instead of 8.6 k: 4 x 8100 positions,
          // B4V4 in 64-channel groups, per layer 25.8 -> 24.2 us.  Scores are off the 64-bit ones by 4.9e-8, 5.2e-8 before.)
          const uint32_t sw = scale_word(Sx, j);
          const int tok = chunk * 64 + 16 * j + t16;
          float acc_s[NSET][NG];
#pragma unroll
          for (int set = 0; set < NSET; ++set)
#pragma unroll
            for (int g = 0; g < NG; ++g) {
              v4i Dc;
              if (NG == 2) {
                Dc = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][g], Bc[g], Cin[set][g], 0, 0, 0);
              } else {
                Dc = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][0], Bc[0], Cin[set][0], 0, 0, 0);
                Dc = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][1], Bc[1], Dc, 0, 0, 0);
              }
              // (WIDE_SUM: the upper limbs' part is at most 2^24 in size and a whole number, so the one rounding is that of
              // the sum, as where it fits 32 bits)
              acc_s[set][g] = WIDE_SUM ? __builtin_fmaf((float)((Dc[2] << 8) + Dc[1]), 256.0f, (float)Dc[0])
                                       : (float)join_limbs(Dc[2], Dc[1], Dc[0]);
            }
          v4i Bp[2], Bn[2];
          v4u rnd[NG];
          float unit[NG];
#pragma unroll
          for (int g = 0; g < NG; ++g) {
            const uint32_t m = ((g == 0) ? sw : (sw >> 16)) & 0x7fu;
            rnd[g] = rnd_sh[m];
            unit[g] = eps_sh[m];
          }
#pragma unroll
          for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const v4u r = rnd[(NG == 2) ? u : 0];
              Bp[u][e] = (int)__builtin_amdgcn_perm(r[1], r[0], (uint32_t)(Bc[u][e] ^ 0x08080808));
              Bn[u][e] = (int)__builtin_amdgcn_perm(r[3], r[2], (uint32_t)Bc[u][e]);
            }
#pragma unroll
          for (int set = 0; set < NSET; ++set)
#pragma unroll
            for (int g = 0; g < NG; ++g) {
              const v4i zero = {0, 0, 0, 0};
              v4i Dr;
              if (NG == 2) {
                Dr = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][g], Bp[g], zero, 0, 0, 0);
                Dr = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][g], Bn[g], Dr, 0, 0, 0);
              } else {
                Dr = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][0], Bp[0], zero, 0, 0, 0);
                Dr = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][1], Bp[1], Dr, 0, 0, 0);
                Dr = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][0], Bn[0], Dr, 0, 0, 0);
                Dr = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][1], Bn[1], Dr, 0, 0, 0);
              }
              acc_s[set][g] = __builtin_fmaf(unit[g], (float)((Dr[2] << 8) + Dr[1]), acc_s[set][g]);
            }
#pragma unroll
          for (int set = 0; set < NSET; ++set) {
            float score = 0.f;
#pragma unroll
            for (int g = 0; g < NG; ++g)
              score = __builtin_fmaf(acc_s[set][g], bf16_to_f32((uint16_t)((g == 0) ? (sw & 0xffffu) : (sw >> 16))) * qsc[set][g], score);
            const int h = set * 4 + lg;
            if ((G % 4 == 0) || h < G) {
              sc[h * L + tok] = score;
              mxl[set] = fmaxf(mxl[set], score);
              mnl[set] = fminf(mnl[set], score);
            }
          }
          continue;
        }
        if constexpr (KA) {
          // Four levels per group: khat(code) = bf16(fma(code - 2, scale, zp)) (int2_qk_scores.cu:66-79) is any function
          // of the code's two bits b1 b0, so with the indicator bytes x0 = b0, x1 = b1, x01 = b0 & b1
          //   khat = v0 + (v1 - v0) x0 + (v2 - v0) x1 + (v3 - v2 - v1 + v0) x01,   v_c = khat(c),
          // and q . khat is four exact fixed-point sums (the query's own, and the three contractions with the
          // indicators) combined in fp32 with coefficients that are exact differences of bf16 values.
          v4i X0[2], X1[2], X01[2];
#pragma unroll
          for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const uint32_t c = (uint32_t)Bc[u][e];
              const uint32_t b0 = c & 0x01010101u, b1 = (c >> 1) & 0x01010101u;
              X0[u][e] = (int)b0;
              X1[u][e] = (int)b1;
              X01[u][e] = (int)(b0 & b1);
            }
          float coef[NG][4];
#pragma unroll
          for (int g = 0; g < NG; ++g) {
            const float sc_g = sgj[j][g];
            const float zp_g = bf16_to_f32((uint16_t)((g == 0) ? (Zx[j] & 0xffffu) : (Zx[j] >> 16)));
            float v[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) v[c] = bf16_to_f32(f32_to_bf16(__builtin_fmaf((float)(c - 2), sc_g, zp_g)));
            coef[g][0] = v[0];
            coef[g][1] = v[1] - v[0];
            coef[g][2] = v[2] - v[0];
            coef[g][3] = (v[3] - v[2]) - (v[1] - v[0]);
          }
          const int tok = chunk * 64 + 16 * j + t16;
#pragma unroll
          for (int set = 0; set < NSET; ++set) {
            const v4i zero = {0, 0, 0, 0};
            float score = 0.f;
#pragma unroll
            for (int g = 0; g < NG; ++g) {
              v4i D0, D1, D01;
              if (NG == 2) {
                D0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][g], X0[g], zero, 0, 0, 0);
                D1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][g], X1[g], zero, 0, 0, 0);
                D01 = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][g], X01[g], zero, 0, 0, 0);
              } else {
                D0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][0], X0[0], zero, 0, 0, 0);
                D0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][1], X0[1], D0, 0, 0, 0);
                D1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][0], X1[0], zero, 0, 0, 0);
                D1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][1], X1[1], D1, 0, 0, 0);
                D01 = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][0], X01[0], zero, 0, 0, 0);
                D01 = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][1], X01[1], D01, 0, 0, 0);
              }
              const float s0f = (float)join_limbs(D0[2], D0[1], D0[0]);
              const float s1f = (float)join_limbs(D1[2], D1[1], D1[0]);
              const float s01f = (float)join_limbs(D01[2], D01[1], D01[0]);
              float v = coef[g][0] * sumq[set][g];
              v = __builtin_fmaf(coef[g][1], s0f, v);
              v = __builtin_fmaf(coef[g][2], s1f, v);
              v = __builtin_fmaf(coef[g][3], s01f, v);
              score = __builtin_fmaf(v, qsc[set][g], score);
            }
            const int h = set * 4 + lg;
            if ((G % 4 == 0) || h < G) {
              sc[h * L + tok] = score;
              mxl[set] = fmaxf(mxl[set], score);
              mnl[set] = fminf(mnl[set], score);
            }
          }
          continue;
        }
        if constexpr (K3) {
#pragma unroll
          for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              Br[u][e] = (int)__builtin_amdgcn_perm(0x01000000u, 0x0000ff00u, (uint32_t)Bc[u][e]);
        }
        // per-token scales (both groups) and the rounding coefficient
        float sg[NG], eg[NG];
#pragma unroll
        for (int g = 0; g < NG; ++g) {
          sg[g] = sgj[j][g];
          eg[g] = egj[j][g];
        }
        const int tok = chunk * 64 + 16 * j + t16;
        if constexpr (NG == 2 && NSET >= 2) {
          // Two head sets: with two wavefronts per SIMD little else hides the wait for an MFMA's results, so all of a
          // token group's products are issued first and read afterwards.
          const v4i zero = {0, 0, 0, 0};
          v4i Dc_all[NSET][NG], Dr_all[NSET][NG];
#pragma unroll
          for (int set = 0; set < NSET; ++set)
#pragma unroll
            for (int g = 0; g < NG; ++g) {
              Dc_all[set][g] = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][g], Bc[g], Cin[set][g], 0, 0, 0);
              Dr_all[set][g] = K3 ? __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][g], Br[g], zero, 0, 0, 0) : zero;
            }
#pragma unroll
          for (int set = 0; set < NSET; ++set) {
            float score = 0.f;
#pragma unroll
            for (int g = 0; g < NG; ++g) {
              const int xc = join_limbs(Dc_all[set][g][2], Dc_all[set][g][1], Dc_all[set][g][0]);
              float v = (float)xc;
              if constexpr (K3) v = __builtin_fmaf(eg[g], (float)((Dr_all[set][g][2] << 8) + Dr_all[set][g][1]), v);
              score = __builtin_fmaf(v, sg[g] * qsc[set][g], score);
            }
            const int h = set * 4 + lg;
            if ((G % 4 == 0) || h < G) {
              sc[h * L + tok] = score;
              mxl[set] = fmaxf(mxl[set], score);
              mnl[set] = fminf(mnl[set], score);
            }
          }
          continue;
        }
#pragma unroll
        for (int set = 0; set < NSET; ++set) {
          float score = 0.f;
          const v4i zero = {0, 0, 0, 0};
          if (NG == 2) {
#pragma unroll
            for (int g = 0; g < NG; ++g) {
              const v4i Dc = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][g], Bc[g], Cin[set][g], 0, 0, 0);
              const int xc = join_limbs(Dc[2], Dc[1], Dc[0]);
              float v = (float)xc;
              if constexpr (K3) {
                const v4i Dr = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][g], Br[g], zero, 0, 0, 0);
                const int xr = (Dr[2] << 8) + Dr[1];
                v = __builtin_fmaf(eg[g], (float)xr, v);
              }
              score = __builtin_fmaf(v, sg[g] * qsc[set][g], score);
            }
          } else {
            v4i Dc = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][0], Bc[0], Cin[set][0], 0, 0, 0);
            Dc = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][1], Bc[1], Dc, 0, 0, 0);
            const int xc = join_limbs(Dc[2], Dc[1], Dc[0]);
            float v = (float)xc;
            if constexpr (K3) {
              v4i Dr = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][0], Br[0], zero, 0, 0, 0);
              Dr = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][1], Br[1], Dr, 0, 0, 0);
              const int xr = (Dr[2] << 8) + Dr[1];
              v = __builtin_fmaf(eg[0], (float)xr, v);
            }
            score = __builtin_fmaf(v, sg[0] * qsc[set][0], score);
          }
          const int h = set * 4 + lg;
          if ((G % 4 == 0) || h < G) {
            sc[h * L + tok] = score;
            mxl[set] = fmaxf(mxl[set], score);
            mnl[set] = fminf(mnl[set], score);
          }
        }
      }
    };
    // at most Lds::LMAX / 64 / NW chunks per wavefront: straight-line code, so that the wait for a chunk's
    // loads leaves the loads of the following chunks in flight
    // (step it + 1 sits inside step it's block, and the chunk two ahead is requested unconditionally, clamped: no
    // two paths with different numbers of loads in flight meet before a wait)
    auto key_step = [&](auto self, auto it_tag) JF_INLINE -> void {
      constexpr int it = decltype(it_tag)::value;
      const int chunk = wave + it * NW;
      prefetch_v(it);
      if (chunk < nch_cover) {
        set_wave_prio(3 - it);  // wavefronts that are behind get the issue slots first
        KBuf& cur = (it & 1) ? Kb : Ka;
        stash_k(cur);
        wave_lds_fence();
        uint32_t Sc[4] = {0u, 0u, 0u, 0u}, Zc[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (!SL || j == 0) Sc[j] = reg_copy(cur.s[SL ? 0 : j]);
          Zc[j] = KA ? reg_copy(cur.z[KA ? j : 0]) : 0u;
        }
        if constexpr (it + 2 < MAXIT) cur = issue_k(min(chunk + 2 * NW, nch_cover - 1));
        const int n_local = n - chunk * 64;  // (uniform)
        if (n_local > 0) {
          if (n_local < 64) clone_last_row(n_local, Sc, Zc);
          if constexpr (SPREP) {  // lane = token: scales and rounding coefficients of the chunk -> table
            const uint32_t sw = Sc[0];
            uint8_t* sp = kst + Lds::KST + lane * Lds::SCT;
            const float s0f = bf16_to_f32((uint16_t)(sw & 0xffffu));
            const float e0f = K3 ? eps_sh[sw & 0x7fu] : 0.f;
            if (NG == 2) {
              const float s1f = bf16_to_f32((uint16_t)(sw >> 16));
              const float e1f = K3 ? eps_sh[(sw >> 16) & 0x7fu] : 0.f;
              *reinterpret_cast<v4f*>(sp) = (v4f){s0f, s1f, e0f, e1f};
            } else {
              *reinterpret_cast<v2f*>(sp) = (v2f){s0f, e0f};
            }
            wave_lds_fence();
          }
          body(chunk, Sc, Zc);
        }
        if (n_local < 64) mask_tail(chunk, n_local);
        wave_lds_fence();
        if constexpr (it + 1 < MAXIT) self(self, std::integral_constant<int, it + 1>{});
      }
    };
    key_step(key_step, std::integral_constant<int, 0>{});
    // lanes of 16-lane row lg hold the running extrema of head set*4 + lg: reduce inside the rows (lane 15 of
    // a row ends up with the row's result) and publish them
#pragma unroll
    for (int set = 0; set < NSET; ++set) {
      float a = mxl[set], c = -mnl[set];
      JF_DPP_ROW_REDUCE(a, op_fmax, float, -INFINITY);
      JF_DPP_ROW_REDUCE(c, op_fmax, float, -INFINITY);
      const int h = set * 4 + lg;
      if (t16 == 15 && h < G) {
        red_f[wave][h] = a;
        red_f[wave][G + h] = -c;
      }
    }
  } else {
    // INT4 keys, int8-Q model on v_mfma_i32_16x16x64_i8: exact nibble codes (offset 8 removed through the
    // per-block constant), int32 block sums, the reference's four-term fp32 rescale in its order
    // (int8tc_qk_scores.cu:455-468).  Lane (token, k-block lg) spreads the 16 channels 64*m + 16*lg .. +15 of
    // both 64-channel spans m; its accumulator registers are the four 32-channel blocks of head lg.
    const QInt8F<NSET>* qsh = reinterpret_cast<const QInt8F<NSET>*>(aux);
    v4i Aop[NSET][2];
    v4i nsum8[NSET];  // minus the block sums: the accumulators' initial values
    float qs[NSET][4];
#pragma unroll
    for (int set = 0; set < NSET; ++set) {
#pragma unroll
      for (int mi = 0; mi < 2; ++mi) Aop[set][mi] = *reinterpret_cast<const v4i*>(&qsh->aop[set][t16][lg][mi][0]);
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        nsum8[set][kk] = -qsh->sum8[set * 4 + lg][kk];
        qs[set][kk] = qsh->qs[set * 4 + lg][kk];
      }
    }
    const uint8_t* krd = kst + t16 * KROW + lg * 8;
    float mxl[NSET], mnl[NSET];
#pragma unroll
    for (int set = 0; set < NSET; ++set) {
      mxl[set] = -INFINITY;
      mnl[set] = INFINITY;
    }
    auto body = [&](int chunk, const uint32_t (&Sx)[4]) JF_INLINE {
      v2u Xj[4][2];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint8_t* rp = krd + j * 16 * KROW;
        Xj[j][0] = *reinterpret_cast<const v2u*>(rp);
        Xj[j][1] = *reinterpret_cast<const v2u*>(rp + 32);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v4i Bm[2];
#pragma unroll
        for (int mi = 0; mi < 2; ++mi) {
          const uint32_t x0 = Xj[j][mi][0], x1 = Xj[j][mi][1];
          Bm[mi] = (v4i){(int)((x0 >> 4) & 0x0f0f0f0fu), (int)(x0 & 0x0f0f0f0fu), (int)((x1 >> 4) & 0x0f0f0f0fu), (int)(x1 & 0x0f0f0f0fu)};
        }
        const float ks = bf16_to_f32((uint16_t)scale_word(Sx, j));
        const int tok = chunk * 64 + 16 * j + t16;
#pragma unroll
        for (int set = 0; set < NSET; ++set) {
          // (the -8 * sum of the block's query values, the codes being used unsigned, enters as the accumulator's
          // initial value: exact, and four subtractions per token and head less)
          v4i Dq = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][0], Bm[0], nsum8[set], 0, 0, 0);
          Dq = __builtin_amdgcn_mfma_i32_16x16x64_i8(Aop[set][1], Bm[1], Dq, 0, 0, 0);
          float sacc = (float)Dq[0] * qs[set][0];
#pragma unroll
          for (int kk = 1; kk < 4; ++kk) sacc = __builtin_fmaf((float)Dq[kk], qs[set][kk], sacc);
          const float a = __fmul_rn(__fmul_rn(sacc, ks), p.attn_scale);
          const int h = set * 4 + lg;
          if ((G % 4 == 0) || h < G) {
            sc[h * L + tok] = a;
            mxl[set] = fmaxf(mxl[set], a);
            mnl[set] = fminf(mnl[set], a);
          }
        }
      }
    };
    auto key_step = [&](auto self, auto it_tag) JF_INLINE -> void {  // (nested, as for the other key formats)
      constexpr int it = decltype(it_tag)::value;
      const int chunk = wave + it * NW;
      prefetch_v(it);
      if (chunk < nch_cover) {
        set_wave_prio(3 - it);
        KBuf& cur = (it & 1) ? Kb : Ka;
        stash_k(cur);
        wave_lds_fence();
        uint32_t Sc[4] = {0u, 0u, 0u, 0u}, Zc[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int j = 0; j < (SL ? 1 : 4); ++j) Sc[j] = reg_copy(cur.s[SL ? 0 : j]);
        if constexpr (it + 2 < MAXIT) cur = issue_k(min(chunk + 2 * NW, nch_cover - 1));
        const int n_local = n - chunk * 64;  // (uniform)
        if (n_local > 0) {
          if (n_local < 64) clone_last_row(n_local, Sc, Zc);
          body(chunk, Sc);
        }
        if (n_local < 64) mask_tail(chunk, n_local);
        wave_lds_fence();
        if constexpr (it + 1 < MAXIT) self(self, std::integral_constant<int, it + 1>{});
      }
    };
    key_step(key_step, std::integral_constant<int, 0>{});
#pragma unroll
    for (int set = 0; set < NSET; ++set) {
      float a = mxl[set], c = -mnl[set];
      JF_DPP_ROW_REDUCE(a, op_fmax, float, -INFINITY);
      JF_DPP_ROW_REDUCE(c, op_fmax, float, -INFINITY);
      const int h = set * 4 + lg;
      if (t16 == 15 && h < G) {
        red_f[wave][h] = a;
        red_f[wave][G + h] = -c;
      }
    }
  }

  if (clk && tid == 0) clk[9] = JF_CLK();  // wavefront 0 finished its chunks
  if (clk && lane == 0) atomicMax(&tmax_sh, (unsigned long long)JF_CLK());
  __builtin_amdgcn_s_setprio(0);
  // split extrema per head; fixed-point exponent of the V scales; selection buckets
  if constexpr (HAS_V) {
    uint32_t vm0 = 0u, vm1 = 0u;
#pragma unroll
    for (int i = 0; i < VSPT; ++i) {
      vm0 = max(vm0, vsw[i] & 0x7fffu);
      vm1 = max(vm1, (vsw[i] >> 16) & 0x7fffu);
    }
    vm0 = wave_max_u(vm0);
    vm1 = wave_max_u(vm1);
    if (lane == 0) {
      vmax_sh[wave][0] = vm0;
      vmax_sh[wave][1] = vm1;
    }
  }
  lds_barrier();  // phase A complete: the query constants are dead, their space becomes the histograms
  if (clk && tid == 0) { clk[8] = JF_CLK(); clk[5] = (long long)tmax_sh; }
  if (p.scores)  // validation output
    for (int i = tid; i < GA * n_cover; i += NT) {
      const int h = i / n_cover, t = i - h * n_cover;
      p.scores[(head0 + h) * (size_t)p.max_S + s0 + t] = sc[h * L + t];
    }
  if constexpr (MODE == FS_STAGE_A)
    if (p.scores_only) return;
  if constexpr (HAS_TOPK)
    if (!take_all)
      for (int i = tid; i < Lds::HIST / 4; i += NT) hist[i] = 0;
  if (tid < G) {
    float m = red_f[0][tid], lo = red_f[0][G + tid];
    if constexpr (ONE) reinterpret_cast<int*>(stage + Lds::stage_bytes() + 64)[tid] = 0;  // (tl_put, see below)
#pragma unroll
    for (int w = 1; w < NW; ++w) {
      m = fmaxf(m, red_f[w][tid]);
      lo = fminf(lo, red_f[w][G + tid]);
    }
    m_sh[tid] = m;
    // bucket of a score: min(255, (m - s) * 255 / (m - lo)), bucket 0 = largest; monotone in s.  No slope where the range has no
    // width or no end, or is so narrow (below 7.5e-37) that its slope has none: all scores in bucket 0.
    const float range = m - lo, slope = 254.99f / range;
    const float iw = (range > 0.f && isfinite(range) && isfinite(slope)) ? slope : 0.f;
    bin_a_sh[tid] = -iw;
    bin_b_sh[tid] = isfinite(m) ? m * iw : 0.f;
  }
  if (HAS_V && tid >= 64 && tid < 64 + NG) {
    const int g = tid - 64;
    uint32_t vb = vmax_sh[0][g];
#pragma unroll
    for (int w = 1; w < NW; ++w) vb = max(vb, vmax_sh[w][g]);
    const float v = bf16_to_f32((uint16_t)vb);
    int e = 0;
    if (v > 0.f && isfinite(v)) (void)frexpf(v, &e);  // v = f * 2^e, f in [0.5, 1)
    e_sh[g] = 23 - e;                                 // v * 2^E in [2^22, 2^23): the weights use all 23 mantissa bits
  }
  lds_barrier();
  if (clk && tid == 0) clk[1] = JF_CLK();

  // ------------------------------------------------------------------ phase B: P.V on v_mfma_i32_16x16x64_i8
  // p = exp(s - m_split) is known exactly because phase A is complete, so w = p * v_scale is converted to
  // 23-bit fixed point once (fma with 2^23: p <= 1 and the largest V scale below 2^e keep the sum below 2^24, where
  // floats are integers); its three bytes, the lower two balanced around zero, are rows (limb, head) of
  // the A operand.  Lane = token stores the four heads' converted words as one 16-byte row per scale group (head-major;
  // the word's top byte is the constant 75 and becomes a constant row), and ds_read_b64_tr_b8 turns 8 token rows into the per-row byte runs the MFMA
  // wants.  V codes are staged packed in wavefront-private LDS and transposed by ds_read_b64_tr_b4 (16
  // tokens of one channel pair per lane), then spread.  sum_t w_t*(code - off) = sum_t w_t*code - off*sum_t w_t:
  // the constant row gives 75 * sum_t code (needed because the limbs are balanced), a ones B tile gives sum_t w_t.
  // Every accumulation is an exact integer.  The same pass drops every score into one of 256 linear buckets
  // per (head, half of the split) for the candidate selection.
  int E[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) E[g] = HAS_V ? __builtin_amdgcn_readfirstlane(e_sh[g]) : 0;
  v4i acc[NSET][NTILE], accw[NSET][NG];
#pragma unroll
  for (int set = 0; set < NSET; ++set) {
#pragma unroll
    for (int t = 0; t < NTILE; ++t) acc[set][t] = (v4i){0, 0, 0, 0};
#pragma unroll
    for (int g = 0; g < NG; ++g) accw[set][g] = (v4i){0, 0, 0, 0};
  }
  float lsum[G], nml[G], bin_a[G], bin_b[G];
#pragma unroll
  for (int h = 0; h < G; ++h) {
    lsum[h] = 0.f;
    nml[h] = uniform_f(-(m_sh[h] * LOG2E));
    bin_a[h] = uniform_f(bin_a_sh[h]);
    bin_b[h] = uniform_f(bin_b_sh[h]);
  }
  // The bucket of a score is fma(s, a, b) clamped to [0, 255] with a and b uniform: an instruction takes one scalar
  // operand only, and left alone the compiler copies b (and 255.0, and the increment) into a vector register again
  // for every head of every chunk.  Copies it cannot see through stay in their registers through the stream.
  float bin_bv[G], clamp_hi = 255.f;
#pragma unroll
  for (int h = 0; h < G; ++h) {
    bin_bv[h] = bin_b[h];
    asm volatile("" : "+v"(bin_bv[h]));
  }
  asm volatile("" : "+v"(clamp_hi));
  v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};  // all-ones B tile of the weight sums (kept, like the above)
  asm volatile("" : "+v"(ones));
  const int r16 = lane & 15, kb4 = lane >> 4;
  // transposed weight read: 16-lane group kb4 fetches the rows of tokens 16*kb4 .. +15; the lane pair (2j, 2j+1)
  // supplies the two halves of the row that must land in byte j, i.e. of the token whose byte position in the
  // V operand (see below) is j
  const int tr_tok = tr8_token(lane);
  const uint8_t* wrow = wl + (kb4 * 16 + tr_tok) * 16 + (r16 & 1) * 8;
  const int seg_chunks = L / 64 / SEG;  // chunks per emission segment
  auto body_v = [&](int chunk, uint32_t vsw) JF_INLINE {
    const int t = chunk * 64 + lane;
    float vsf[NG];
    vsf[0] = ldexpf(bf16_to_f32((uint16_t)(vsw & 0xffffu)), E[0]);
    if (NG == 2) vsf[NG - 1] = ldexpf(bf16_to_f32((uint16_t)(vsw >> 16)), E[NG - 1]);
    int* hb = hist + ((SEG == 1) ? 0 : (chunk / seg_chunks) * (Lds::H16 ? 128 : 256));
    const bool tv = t < n;
    const int inc = tv ? 1 : 0;
    (void)inc;
    uint32_t bits[NSET * 4][NG];
#pragma unroll
    for (int h = 0; h < NSET * 4; ++h) {
      if (h < G) {
        const float s = sc[h * L + t];
        // masked positions hold -inf: their weight is exactly zero
        const float pw = __builtin_amdgcn_exp2f(__builtin_fmaf(s, LOG2E, nml[h]));
        lsum[h] += pw;
        // A weight that is a NaN (an infinite or NaN score) is the sum's affair, which makes the head's outputs what they are.  Here
        // it counts zero: converted, it would change the word's top byte, which the other heads of the set take their code sums from.
        const float pv = fmaxf(pw, 0.f);
#pragma unroll
        for (int g = 0; g < NG; ++g) bits[h][g] = __builtin_bit_cast(uint32_t, __builtin_fmaf(pv, vsf[g], 8388608.0f));
        if (HAS_TOPK && !take_all) {
          // (positions past the end add zero instead of branching around the add: their score is -inf or, with a
          // degenerate range, gives a NaN, and either clamps to a bucket inside the table)
          const uint32_t bin = (uint32_t)__builtin_amdgcn_fmed3f(__builtin_fmaf(s, bin_a[h], bin_bv[h]), 0.f, clamp_hi);
          if (Lds::H16) atomicAdd(hb + ((h * (SEG * 256) + (int)bin) >> 1), inc << ((bin & 1u) << 4));
          else atomicAdd(hb + h * (SEG * 256) + (int)bin, inc);
        }
      } else {
#pragma unroll
        for (int g = 0; g < NG; ++g) bits[h][g] = 0x4b000000u;
      }
    }
    if constexpr (!HAS_V) return;  // Stage A alone: the weights' sums and the selection buckets were all
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int set = 0; set < NSET; ++set) {
        // one 16-byte row per token: byte 4h + l = limb l of head h (limbs 0 and 1 balanced around zero, limb 2 < 128),
        // byte 4h + 3 = 75, the exponent byte of the fixed-point conversion, which serves as the constant row that
        // yields the code sums
        v4i row;
#pragma unroll
        for (int hh = 0; hh < 4; ++hh) row[hh] = (int)(bits[set * 4 + hh][g] ^ 0x00008080u);
        *reinterpret_cast<v4i*>(wl + ((g * NSET + set) * 64 + lane) * 16) = row;
      }
    wave_lds_fence();
    v4i A[NG][NSET];
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int set = 0; set < NSET; ++set) {
        const uint8_t* src = wrow + (g * NSET + set) * 1024;
        const v2i x0 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i*)(src));
        const v2i x1 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i*)(src + 128));
        A[g][set] = (v4i){x0[0], x0[1], x1[0], x1[1]};
      }
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int set = 0; set < NSET; ++set)
        accw[set][g] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[g][set], ones, accw[set][g], 0, 0, 0);
    Tiles::spread(vst, lane, [&](auto tile, int g, const v4i& Bv) JF_INLINE {
#pragma unroll
      for (int set = 0; set < NSET; ++set)
        acc[set][decltype(tile)::value] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[g][set], Bv, acc[set][decltype(tile)::value], 0, 0, 0);
    });
    wave_lds_fence();
  };
  auto stash_v = [&](const VBuf& vbuf) {
#pragma unroll
    for (int i = 0; i < VLD; ++i) {
      if (Lds::VSWZ) {
        *reinterpret_cast<v4u*>(vst + vl_lds[i]) = vbuf.r[i];  // 16-byte aligned with the unpadded pitch
      } else {
        *reinterpret_cast<v2u*>(vst + vl_lds[i]) = (v2u){vbuf.r[i][0], vbuf.r[i][1]};
        *reinterpret_cast<v2u*>(vst + (V3 ? (vl_lds[i] ^ 8u) : (vl_lds[i] + 8u))) = (v2u){vbuf.r[i][2], vbuf.r[i][3]};
      }
    }
  };
  if constexpr (MODE == FS_FULL) {  // (wavefronts that left the key stream before its last two steps)
    if (!va_requested) Va = issue_v(min(wave, nch - 1));
    if (!vb_requested) Vb = issue_v(min(wave + NW, nch - 1));
  }
  auto value_step = [&](auto self, auto it_tag) JF_INLINE -> void {  // (nested like the key stream's steps)
    constexpr int it = decltype(it_tag)::value;
    const int chunk = wave + it * NW;
    if (chunk < nch) {
      set_wave_prio(3 - it);
      uint32_t vw = 0u;
      if constexpr (HAS_V) {
        VBuf& cur = (it & 1) ? Vb : Va;
        stash_v(cur);
        static_assert(VSPT == MAXIT, "one V scale word per thread and step");
        vw = vsw[it];
        if constexpr (it + 2 < MAXIT) cur = issue_v(min(chunk + 2 * NW, nch - 1));
      }
      body_v(chunk, vw);
      if constexpr (it + 1 < MAXIT) self(self, std::integral_constant<int, it + 1>{});
    }
  };
  value_step(value_step, std::integral_constant<int, 0>{});
  __builtin_amdgcn_s_setprio(0);
#pragma unroll
  for (int h = 0; h < G; ++h) {
    const float ls = wave_sum(lsum[h]);
    if (lane == 0) lsum_sh[wave][h] = ls;  // summed in wavefront order below: run-to-run deterministic
  }
  if constexpr (HAS_V) {
    // The accumulator sums below live at the start of the staging area: each wavefront clears what lies in its own
    // part (it is done with it), so the array is zero behind the barrier.
    const int z0 = wave * Lds::WAVE_STAGE;
    const int z1 = min(z0 + Lds::WAVE_STAGE, Lds::XACC);
    for (int o = z0 + lane * 16; o < z1; o += 1024) *reinterpret_cast<v4i*>(stage + o) = (v4i){0, 0, 0, 0};
  }
  lds_barrier();
  if (clk && tid == 0) clk[2] = JF_CLK();

  // ---- sum of the integer accumulators over the wavefronts: LDS integer atomics into one array at the start of
  // the staging area (cleared before the barrier above), read by `combine` after the candidates have been emitted.
  // Integer sums: exact and independent of the order.  The atomics return nothing, so a wavefront issues them a few
  // at a time along the comparisons of its first emission blocks: they drain in the LDS pipe while the vector ALU
  // works.
  // D layout: row r of a tile sits in lane 16*(r>>2) + column, register r&3; row 4*head + l is limb l for l < 3 and
  // the constant row (75 * sum of codes) for l = 3.  The two lower limbs go in as one number, 256 * limb 1 + limb 0 (at most
  // 4096 * 128 * 257 * 15 in size: 31 bits), and the constant rows, which are the same for every head, from the first lane group
  // alone.  Item j = 2 * (register i of set i / AR) + {0: lower limbs, 1: limb 2} lies at xacc[j * 64 + lane], the constant row of
  // tile t of set s behind all items, at [(s * 8 + t) * 16 + column].
  int* xacc = reinterpret_cast<int*>(stage);
  // ONE: what the in-kernel merge keeps behind the staging area (see ScanTail)
  using Tail = ScanTail<G, SEG>;
  const int Kcap = p.Kc;
  [[maybe_unused]] const int K = p.top_k;
  uint8_t* tail = stage + Lds::stage_bytes() + 64;
  [[maybe_unused]] int* tl_put = reinterpret_cast<int*>(tail);              // [G] members put into the head's list
  [[maybe_unused]] int* tl_mem = tl_put + G;                                // [G] members of the cut bucket
  [[maybe_unused]] int* tl_nout = tl_mem + G;                               // [G] winners (Stage B); the selection's words
  [[maybe_unused]] int* tl_segc = tl_nout + G;                              // [G][SEG] winners per wavefront
  [[maybe_unused]] float* tl_m = reinterpret_cast<float*>(tl_segc + G * SEG);  // [G] softmax maximum, 1 / sum, e^{m - M}
  [[maybe_unused]] float* tl_iz = tl_m + G;
  [[maybe_unused]] float* tl_coef = tl_iz + G;
  [[maybe_unused]] float* tl_ohat = reinterpret_cast<float*>(tail + Tail::INTS);          // [G][D]
  [[maybe_unused]] int* tl_wslot = reinterpret_cast<int*>(tl_ohat + G * D);               // [G][top_k] paged slot of a winner
  [[maybe_unused]] float* tl_ww = reinterpret_cast<float*>(tl_wslot + (size_t)G * K);     // [G][top_k] its softmax weight
  // [G][MEM] members of the cut bucket, as rank words
  [[maybe_unused]] unsigned long long* tl_mlist = reinterpret_cast<unsigned long long*>(tl_ww + (size_t)G * K);
  [[maybe_unused]] uint16_t* tl_list = reinterpret_cast<uint16_t*>(tl_mlist + G * Tail::MEM);  // [G][Kcap] the winners' positions, ascending
  if constexpr (ONE) {
    if (tid < G) {
      float l = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) l += lsum_sh[w][tid];
      const float pm = m_sh[tid], M = isfinite(pm) ? pm : 0.f;
      const float coef = (pm == -INFINITY) ? 0.f : __expf(pm - M);
      l *= coef;
      tl_m[tid] = M;
      tl_coef[tid] = coef;
      tl_iz[tid] = (l > 0.f) ? 1.0f / l : 0.f;
    }
  }
  constexpr int ACC_ITEMS = NSET * AR * 2, ACC_HALF = NSET * AR;
  // (uniform) this wavefront's sums are on their way (or it had no chunk: a short split occupies a few wavefronts only)
  bool acc_issued = wave >= nch;
  auto add_acc_range = [&](const int first, const int last) {  // (constants once the caller's loop is unrolled)
#pragma unroll
    for (int j = 0; j < ACC_ITEMS; ++j) {
      if (j < first || j >= last) continue;
      const int i = j >> 1, set = i / AR, r = i % AR;
      const v4i v = (r < NTILE) ? acc[set][r < NTILE ? r : 0] : accw[set][r >= NTILE ? r - NTILE : 0];
      atomicAdd(xacc + j * 64 + lane, (j & 1) ? v[2] : v[0] + (v[1] << 8));
    }
    if (last == ACC_ITEMS && lane < 16) {
#pragma unroll
      for (int set = 0; set < NSET; ++set)
#pragma unroll
        for (int t = 0; t < NTILE; ++t) atomicAdd(xacc + ACC_ITEMS * 64 + (set * NTILE + t) * 16 + lane, acc[set][t][3]);
    }
  };
  [[maybe_unused]] float* late_o_hat = nullptr;  // ONE: see below
  auto combine = [&](int set) {
    // thread -> (tile, head, column)
    int first = tid;
    if constexpr (TIGHTER) asm volatile("" : "+v"(first));
    for (int i = first; i < 4 * D; i += NT) {
      const int col = i & 15, hh = (i >> 4) & 3, tile = i >> 6;
      const int h = set * 4 + hh;
      if (h >= GA) continue;
      const int d = Tiles::channel(tile, col);
      const int g = (NG == 1) ? 0 : (d / (D / NG));
      const int* ta = xacc + ((set * AR + tile) * 2) * 64 + 16 * hh + col;
      const int* wa = xacc + ((set * AR + NTILE + g) * 2) * 64 + 16 * hh;    // weight sums: any column of the all-ones tile
      int lo = ta[0], i2 = ta[64], cs = xacc[ACC_ITEMS * 64 + (set * NTILE + tile) * 16 + col] / 75;
      if (V2 && !(tile & 1)) {  // even INT2 tiles hold four times their sums (exact multiples)
        lo >>= 2;
        i2 >>= 2;
        cs >>= 2;
      }
      const long long wsum = (long long)wa[64] * 65536ll + (long long)wa[0] + 32896ll * 64ll * (long long)nch;
      const long long tot = (long long)i2 * 65536ll + (long long)lo + 32896ll * (long long)cs - (long long)VOFF * wsum;
      const float o = (float)ldexp((double)tot, -E[g]);
      if constexpr (ONE) {
        const float o_hat = __builtin_fmaf(o, tl_coef[h], 0.f) * tl_iz[h];
        late_o_hat[(head0 + h) * D + d] = o_hat;
        tl_ohat[h * D + d] = o_hat;
      } else {
        p.part_o[(part_base + (size_t)h * p.n_splits) * D + d] = o;
      }
    }
  };

  // ------------------------------------------------------------------ phase C: candidates of the split
  // The merge kernel needs a superset of the split's top Kt = min(top_k, n) scores per head that fits the
  // candidate buffer (Kcap entries), in ascending position.  From the histograms: the smallest bucket index
  // `cut` with count(bucket <= cut) >= Kt.  If that count fits, every position whose bucket is <= cut is
  // emitted, one wavefront per (head, segment of the split), each segment starting where the counts of the segments
  // before it end.  Otherwise (heavily tied scores) one wavefront falls back to an exact radix select over the keys.
  const int Kt = min(p.top_k, n);
  // Blocks of 1024 positions, 16 consecutive ones per lane: the lane's candidates are consecutive in the output,
  // so a block costs one comparison per position, one wavefront scan of the lanes' counts, and a loop over the
  // few set bits of every lane.  The lane reads its four 16-byte quads starting at quad (lane >> 2) & 3 (the
  // four lanes that share a bank group then read different banks) and rotates its bit mask back afterwards.
  const int rot4 = ((lane >> 2) & 3) * 4;
  // -> bit i: position t0 + 16 * lane + i lies before `thr` in the buckets; ONE: `sure`, likewise before `thr_lo`
  auto block_mask = [&](const float* lp, float ba, float bb, float thr, float thr_lo, int nvalid, auto acc_tag, uint32_t& sure) JF_INLINE -> uint32_t {
    constexpr int ACCSEL = decltype(acc_tag)::value;  // accumulator sums issued along the comparisons: -1 none, 0 / 1 a half, 2 all
    constexpr int A_LO = (ACCSEL == 1) ? ACC_HALF : 0;
    constexpr int A_HI = (ACCSEL < 0) ? 0 : ((ACCSEL == 0) ? ACC_HALF : ACC_ITEMS);
    constexpr int PER = (A_HI - A_LO + 15) / 16;      // a few behind every comparison: the LDS queue never fills
    v4f x[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) x[q] = *reinterpret_cast<const v4f*>(lp + ((4 * q + rot4) & 15));
    uint32_t ge = 0u, ge_lo = 0u;  // bit 4q + e set: element e of quad register q falls behind the cut (not emitted)
#pragma unroll
    for (int bi = 15; bi >= 0; --bi) {
      // ge = 2 * ge + [value >= thr]: the comparison's lane mask is the carry of one add
      const float v = __builtin_fmaf(x[bi >> 2][bi & 3], ba, bb);
      const unsigned long long c = __builtin_amdgcn_ballot_w64(v >= thr);
      // (the two wait states between a vector instruction's scalar result and a vector instruction that reads it
      // are the compiler's job everywhere else; it does not look inside an asm statement)
      asm("s_nop 1\n\tv_addc_co_u32_e64 %0, vcc, %1, %1, %2" : "=v"(ge) : "v"(ge), "s"(c) : "vcc");
      if constexpr (ONE) {
        const unsigned long long c_lo = __builtin_amdgcn_ballot_w64(v >= thr_lo);
        asm("s_nop 1\n\tv_addc_co_u32_e64 %0, vcc, %1, %1, %2" : "=v"(ge_lo) : "v"(ge_lo), "s"(c_lo) : "vcc");
        __builtin_amdgcn_sched_barrier(0);  // (all lane masks together do not fit the scalar registers)
      }
      if constexpr (HAS_V && PER > 0) {
        const int lo = A_LO + (15 - bi) * PER;
        if (lo < A_HI) {
          add_acc_range(lo, (lo + PER < A_HI) ? lo + PER : A_HI);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    // register bit b is position (b + rot4) mod 16 of the lane's run
    auto in_order = [&](uint32_t m) -> uint32_t {
      m = ~m & 0xffffu;
      m |= m << 16;
      return (m >> (16 - rot4)) & ((1u << nvalid) - 1u);
    };
    if constexpr (ONE) sure = in_order(ge_lo);
    return in_order(ge);
  };
  // The cut of a head's histograms: the bucket, the positions up to and with it, those before it, and in the segments before
  // `seg` those up to and with it and those before it.  Every wavefront of a head searches it for itself (same histograms, same
  // result): no exchange, no barrier between the search and the emission.
  struct Cut {
    bool found;
    int cut, tot, above_cut, before_me, before_above;
  };
  auto find_cut = [&](int h, int seg) JF_INLINE -> Cut {
    const int* h0 = hist + h * (SEG * 256) / (Lds::H16 ? 2 : 1);
    // lane l owns buckets 4l .. 4l+3 (ascending bucket = descending score) of every segment's histogram
    int cs[SEG][4];
#pragma unroll
    for (int sg = 0; sg < SEG; ++sg) {
      if (Lds::H16) {
        const uint32_t w0 = (uint32_t)h0[sg * 128 + 2 * lane], w1 = (uint32_t)h0[sg * 128 + 2 * lane + 1];
        cs[sg][0] = (int)(w0 & 0xffffu);
        cs[sg][1] = (int)(w0 >> 16);
        cs[sg][2] = (int)(w1 & 0xffffu);
        cs[sg][3] = (int)(w1 >> 16);
      } else {
        const v4i x = *reinterpret_cast<const v4i*>(h0 + sg * 256 + 4 * lane);
#pragma unroll
        for (int u = 0; u < 4; ++u) cs[sg][u] = x[u];
      }
    }
    // pk[u]: the bucket's count over all segments in the low half, over the segments before this wavefront's in the high half (each
    // sum <= 4096)
    int c[4] = {0, 0, 0, 0}, cum[4] = {0, 0, 0, 0}, pk[4];
#pragma unroll
    for (int sg = 0; sg < SEG; ++sg) {
      if (sg == seg) {  // (uniform)
#pragma unroll
        for (int u = 0; u < 4; ++u) cum[u] = c[u];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) c[u] += cs[sg][u];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) pk[u] = c[u] | (cum[u] << 16);
    const int packed = (pk[0] + pk[1]) + (pk[2] + pk[3]);
    const int incl = wave_incl_scan_i(packed);
    // the first lane whose inclusive total reaches Kt holds the cut bucket; every lane finds the bucket that would be the cut were
    // it that lane
    const unsigned long long who = __builtin_amdgcn_ballot_w64((incl & 0xffff) >= Kt);
    const int r_1 = incl - packed, r0 = r_1 + pk[0], r1 = r0 + pk[1], r2 = r1 + pk[2];  // sums up to the bucket
    const bool t0 = (r0 & 0xffff) < Kt, t1 = (r1 & 0xffff) < Kt, t2 = (r2 & 0xffff) < Kt;
    const int with = t2 ? incl : (t1 ? r2 : (t0 ? r1 : r0)), without = t2 ? r2 : (t1 ? r1 : (t0 ? r0 : r_1));
    const int bucket = 4 * lane + (t0 ? 1 : 0) + (t1 ? 1 : 0) + (t2 ? 1 : 0);
    const bool found = who != 0ull;
    const int src = found ? __ffsll((long long)who) - 1 : 63;
    const uint32_t upto = (uint32_t)__builtin_amdgcn_readlane(with, src), before = (uint32_t)__builtin_amdgcn_readlane(without, src);
    return {found, __builtin_amdgcn_readlane(bucket, src), (int)(upto & 0xffffu), (int)(before & 0xffffu), (int)(upto >> 16), (int)(before >> 16)};
  };
  for (int hs = wave; HAS_TOPK && !ONE && hs < G * SEG; hs += NW) {
    const int h = hs / SEG, seg = hs % SEG;
    if (h >= GA) continue;
    if (SHORT && take_all) {
      const float* srow = sc + h * L;
      uint32_t* ck = p.cand_key + (part_base + (size_t)h * p.n_splits) * Kcap;
      int32_t* ci = p.cand_idx + (part_base + (size_t)h * p.n_splits) * Kcap;
      for (int t = (seg * 64 + lane) * 4; t < Kcap; t += SEG * 256) {  // (the list's length is a multiple of 4, at most L)
        const v4f x = *reinterpret_cast<const v4f*>(srow + t);
        v4u key;
        v4i pos;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          key[u] = (t + u < n) ? score_key(x[u]) : 0u;  // unused slots hold key 0
          pos[u] = s0 + t + u;
        }
        *reinterpret_cast<v4u*>(ck + t) = key;
        *reinterpret_cast<v4i*>(ci + t) = pos;
      }
      if (seg == 0) {  // the smallest score
        float lo = -red_f[lane & (NW - 1)][G + h];
        JF_DPP_ROW_REDUCE(lo, op_fmax, float, -INFINITY);
        if (lane == 15) p.cand_edge[part_base + (size_t)h * p.n_splits] = -lo;
      }
      continue;
    }
    const float ba = uniform_f(bin_a_sh[h]);
    float bb = uniform_f(bin_b_sh[h]);
    asm volatile("" : "+v"(bb));  // (kept in a vector register: the multiply-add takes one scalar operand only)
    const Cut c = find_cut(h, seg);
    const bool ok = c.found && c.tot <= Kcap;
    const int cut = c.cut, tot = c.tot, before_me = c.before_me;
    if (clk && tid == 0) clk[6] = JF_CLK();
    const float* srow = sc + h * L;
    uint32_t* ck = p.cand_key + (part_base + (size_t)h * p.n_splits) * Kcap;
    int32_t* ci = p.cand_idx + (part_base + (size_t)h * p.n_splits) * Kcap;
    if (ok) {
      // bucket(s) <= cut  <=>  not (s * ba + bb >= cut + 1): the bucket is the floor of that value clamped to
      // [0, 255]; with cut = 255 every position qualifies
      const float thr = uniform_f((cut >= 255) ? INFINITY : (float)(cut + 1));
      const int tb = seg * (L / SEG);
      const int te = min(n, (seg + 1) * (L / SEG));
      // the emitted total is at most Kcap by construction of the cut
      int count = __builtin_amdgcn_readfirstlane(before_me);
      // unused slots hold key 0 (no score maps to it); the planned total is known, so the head's wavefronts
      // share the padding and its stores leave before the emission's
      const int etot = min(Kcap, tot);
      for (int i = etot + seg * 64 + lane; i < Kcap; i += SEG * 64) ck[i] = 0u;
      // A block's candidates go to a list in the wavefront's own LDS first, then out one per lane: stored from the loop over a
      // lane's set bits, keys and positions took a dozen partly filled stores each instead of two or three.  Per layer: 32 sequences x 3000
      // positions, K4V4, top-k 2048 94.8 us, this 84.4; 1 x 65536, eight heads, K3V2, 512 40.9 / 37.1; 16 x 4096, K3V2, 1024 45.4 / 42.1;
      // 4 x 32768, eight heads, 256 31.8 / 31.6.
      uint16_t* cl = reinterpret_cast<uint16_t*>(stage + Lds::XACC + wave * Lds::EMIT);
      auto emit_block = [&](int t0, auto acc_tag) JF_INLINE {
        const int lt = t0 + 16 * lane;                    // first position of this lane
        const float* lp = srow + lt;
        uint32_t none;
        uint32_t mask = block_mask(lp, ba, bb, thr, 0.f, max(0, min(16, te - lt)), acc_tag, none);
        const int mine = __popc(mask);
        const int incl = wave_incl_scan_i(mine);
        const int start = count;
        int at = incl - mine;
        count += __builtin_amdgcn_readlane(incl, 63);
        while (mask != 0u) {
          cl[at++] = (uint16_t)(lt + __ffs((int)mask) - 1);
          mask &= mask - 1u;
        }
        wave_lds_fence();
        for (int r = start + lane; r < min(count, Kcap); r += 64) {  // (the bound only matters for non-finite scores)
          const int t = cl[r - start];
          ck[r] = score_key(srow[t]);
          ci[r] = s0 + t;
        }
        wave_lds_fence();
      };
      if constexpr (SHORT) {
        // Segments of at most 256 positions (512 beyond four heads): one position per lane, 64 at a time; all scores first,
        // then the sums' atomics, which would otherwise be ahead of them in the LDS queue.  (Sixteen positions per lane,
        // as below, leave a segment of 256 to sixteen lanes.)
        constexpr int STEPS = Lds::NT / SEG / 64;
        float x[STEPS];
#pragma unroll
        for (int i = 0; i < STEPS; ++i) x[i] = srow[min(tb + 64 * i + lane, L - 1)];
        if (HAS_V && !acc_issued) {
          add_acc_range(0, ACC_ITEMS);
          acc_issued = true;
        }
#pragma unroll
        for (int i = 0; i < STEPS; ++i) {
          if (tb + 64 * i < te) {
            const int t = tb + 64 * i + lane;
            const bool emit = t < te && !(__builtin_fmaf(x[i], ba, bb) >= thr);
            const unsigned long long em = __builtin_amdgcn_ballot_w64(emit);
            const uint32_t o = (uint32_t)(count + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(em >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)em, 0u)));
            count += __popcll(em);
            if (emit && o < (uint32_t)Kcap) {  // the bound only matters for non-finite scores
              ck[o] = score_key(x[i]);
              ci[o] = s0 + t;
            }
          }
        }
      }
      constexpr std::integral_constant<int, -1> plain{};
      int t0 = SHORT ? te : tb;
      if (!SHORT && HAS_V && !acc_issued && te > tb) {  // the first block (or the first two) of this wavefront carry the sums
        if (te - tb > 1024) {
          emit_block(tb, std::integral_constant<int, 0>{});
          emit_block(tb + 1024, std::integral_constant<int, 1>{});
          t0 = tb + 2048;
        } else {
          emit_block(tb, std::integral_constant<int, 2>{});
          t0 = tb + 1024;
        }
        acc_issued = true;
      }
      for (; t0 < te; t0 += 1024) emit_block(t0, plain);
      if (seg == SEG - 1) {
        // the lower edge of the cut bucket (a degenerate range: one bucket, the largest score)
        if (lane == 0) p.cand_edge[part_base + (size_t)h * p.n_splits] = (ba < 0.f) ? (bb - (float)(cut + 1)) * __builtin_amdgcn_rcpf(-ba) : m_sh[h];
        for (int i = count + lane; i < etot; i += 64) ck[i] = 0u;  // (only if a segment emitted less than planned)
      }
    } else if (seg == 0) {
      // exact fallback: 8-bit radix select over the order-preserving keys (bits shared by every key skipped),
      // then the keys above the K-th and the lowest-position ties that fill the quota
      int* rh = reinterpret_cast<int*>(stage + Lds::XACC + wave * Lds::EMIT);
      uint32_t T = 0;
      int quota = 0;
      uint32_t kmin = 0xffffffffu, kmax = 0u;
      for (int t = lane; t < n; t += 64) {
        const uint32_t k = score_key(srow[t]);
        kmin = min(kmin, k);
        kmax = max(kmax, k);
      }
      kmin = wave_min_u(kmin);
      kmax = wave_max_u(kmax);
      const uint32_t diff = kmin ^ kmax;
      if (diff == 0u) {  // every key equal: the lowest positions win
        T = kmax;
        quota = Kt;
      } else {
        int bits_left = 32 - __clz((int)diff);  // number of low bits that vary
        uint32_t prefix = (bits_left == 32) ? 0u : (kmax >> bits_left);
        int k_rem = Kt;
        while (bits_left > 0) {
          const int nb = min(8, bits_left);
          const int shift = bits_left - nb;
          const uint32_t dmask = (1u << nb) - 1u;
          for (int i = lane; i < 256; i += 64) rh[i] = 0;
          const bool first = (bits_left == 32);
          const int hi_shift = first ? 0 : bits_left;
          for (int t0 = 0; t0 < n; t0 += 64) {
            const int t = t0 + lane;
            const uint32_t k = (t < n) ? score_key(srow[t]) : 0u;
            const bool inpre = (t < n) && (first || ((k >> hi_shift) == prefix));
            if (inpre) atomicAdd(&rh[(int)((k >> shift) & dmask)], 1);
          }
          // lane l owns bins 255-4l .. 252-4l (descending), so a prefix scan over lanes counts the bins above
          const int c3 = rh[255 - 4 * lane], c2 = rh[254 - 4 * lane], c1 = rh[253 - 4 * lane], c0 = rh[252 - 4 * lane];
          const int mine = c0 + c1 + c2 + c3;
          const int e3 = wave_incl_scan_i(mine) - mine;  // keys in bins above 255-4l
          const int e2 = e3 + c3, e1 = e2 + c2, e0 = e1 + c1;
          int cut = -1, above = 0;
          if (e3 < k_rem && k_rem <= e3 + c3) { cut = 255 - 4 * lane; above = e3; }
          else if (e2 < k_rem && k_rem <= e2 + c2) { cut = 254 - 4 * lane; above = e2; }
          else if (e1 < k_rem && k_rem <= e1 + c1) { cut = 253 - 4 * lane; above = e1; }
          else if (e0 < k_rem && k_rem <= e0 + c0) { cut = 252 - 4 * lane; above = e0; }
          const unsigned long long who = __ballot(cut >= 0);
          const int src = __ffsll((long long)who) - 1;
          cut = __builtin_amdgcn_readlane(cut, src);
          above = __builtin_amdgcn_readlane(above, src);
          prefix = (prefix << nb) | (uint32_t)cut;
          k_rem -= above;
          bits_left = shift;
        }
        T = prefix;
        quota = k_rem;
      }
      int count = 0, base_tie = 0;
      for (int t0 = 0; t0 < n; t0 += 64) {
        const int t = t0 + lane;
        const uint32_t k = (t < n) ? score_key(srow[t]) : 0u;
        const bool above = (t < n) && (k > T), tie = (t < n) && (k == T);
        const unsigned long long ma = __ballot(above), mt = __ballot(tie);
        const int pa = count + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(ma >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)ma, 0u));
        const int pt = base_tie + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mt >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mt, 0u));
        if (above || (tie && pt < quota)) {
          const int pos = pa + min(pt, quota);
          if (pos < Kcap) {
            ck[pos] = k;
            ci[pos] = s0 + t;
          }
        }
        count += __popcll(ma);
        base_tie += __popcll(mt);
      }
      count += min(base_tie, quota);
      if (lane == 0) p.cand_edge[part_base + (size_t)h * p.n_splits] = key_to_score(T);
      for (int i = count + lane; i < Kcap; i += 64) ck[i] = 0u;
    }
  }
  // ONE: the workgroup holds all scores, so the winners are marked where they stand.  The positions whose bucket lies before the
  // cut bucket win; of the cut bucket's members the `need` largest (ties: the lowest positions).  A wavefront has the positions
  // of its (head, segment) in two masks per lane and puts its members, a dozen per head, into the head's list; where the
  // segments' winners go follows from the histograms and that list, so behind one barrier every wavefront finds the last
  // winner and writes its own.  A list of candidates as the merge kernel takes it, gone over once for the members, once for the
  // winners and once for their outputs with a barrier each, took longer, per layer: 1 x 777 positions, K4V4, top-k 64 15.1 us, now
  // 14.1; 20 x 1000, K3V2, 128 17.9 / 17.2; 32 x 1900, K3V2, 512 29.5 / 28.8; 32 x 2048, K4V4, 256 26.8 / 26.6.
  // (rank word: key over inverted position, 32 + 12 bits, so that the larger word is the earlier winner)
  constexpr int NHS = (G * SEG + NW - 1) / NW;  // (head, segment) pairs per wavefront
  static_assert(Lds::LMAX <= 4096 && Lds::LMAX / SEG <= 2048, "a position takes twelve bits, a lane's share of a segment 32");
  constexpr int STEPS = SHORT ? NT / SEG / 64 : 1;
  static_assert(!SHORT || STEPS <= 32, "one bit a step");
  [[maybe_unused]] uint32_t sure[NHS], memb[NHS];  // SHORT: bit i is position 64 i + lane of the segment; else 1024 (i / 16) + 16 lane + i % 16
  [[maybe_unused]] int need[NHS], members[NHS], before[NHS];  // winners among the head's members, members, sure winners in the segments before
  [[maybe_unused]] auto rank_word = [](uint32_t key, int pos) { return ((unsigned long long)key << 12) | (uint32_t)(4095 - pos); };
  [[maybe_unused]] auto place_of = [&](int i) -> int { return SHORT ? 64 * i + lane : (i >> 4) * 1024 + 16 * lane + (i & 15); };
  if constexpr (ONE && HAS_TOPK) {
#pragma unroll
    for (int it = 0; it < NHS; ++it) {
      const int hs = wave + it * NW, h = hs / SEG, seg = hs % SEG;
      sure[it] = memb[it] = 0u;
      need[it] = members[it] = before[it] = 0;
      if (hs >= G * SEG || h >= GA) continue;
      const float ba = uniform_f(bin_a_sh[h]);
      float bb = uniform_f(bin_b_sh[h]);
      asm volatile("" : "+v"(bb));
      const Cut c = find_cut(h, seg);
      const float lw = lsum_sh[min(lane, NW - 1)][h];
      if (clk && tid == 0) clk[6] = JF_CLK();
      const bool all = Kt == n;  // every position wins
      // No range to cut into buckets, or a NaN among the scores (its sum of weights is one too), whose place in the order of the
      // keys the buckets do not know: all positions are members.
      const bool exact = !all && (!c.found || !(ba < 0.f) || __builtin_amdgcn_ballot_w64(lw != lw) != 0ull);
      const int tb = seg * (L / SEG), te = min(n, tb + L / SEG);
      need[it] = all ? 0 : (exact ? Kt : Kt - c.above_cut);
      members[it] = all ? 0 : (exact ? n : c.tot - c.above_cut);
      before[it] = all ? tb : (exact ? 0 : c.before_above);
      // bucket(s) <= cut  <=>  not (s * ba + bb >= cut + 1): the bucket is the floor of that value clamped to [0, 255]
      const float thr = uniform_f((all || exact || c.cut >= 255) ? INFINITY : (float)(c.cut + 1));
      const float thr_lo = uniform_f((c.cut == 0) ? -INFINITY : (float)c.cut);
      const float* srow = sc + h * L;
      uint32_t upto = 0u, lower = 0u;
      if constexpr (SHORT) {
        float x[STEPS];
#pragma unroll
        for (int i = 0; i < STEPS; ++i) x[i] = srow[min(tb + 64 * i + lane, L - 1)];
        if (HAS_V && !acc_issued) {
          add_acc_range(0, ACC_ITEMS);
          acc_issued = true;
        }
#pragma unroll
        for (int i = 0; i < STEPS; ++i) {
          const float v = __builtin_fmaf(x[i], ba, bb);
          const bool in = tb + 64 * i + lane < te;
          upto |= (in && !(v >= thr) ? 1u : 0u) << i;
          lower |= (in && !(v >= thr_lo) ? 1u : 0u) << i;
        }
      } else {
        auto block = [&](int t0, auto acc_tag) JF_INLINE {
          const int lt = t0 + 16 * lane;
          uint32_t lo;
          const uint32_t m = block_mask(srow + lt, ba, bb, thr, thr_lo, max(0, min(16, te - lt)), acc_tag, lo);
          const int at = (t0 > tb) ? 16 : 0;
          upto |= m << at;
          lower |= lo << at;
        };
        constexpr std::integral_constant<int, -1> plain{};
        if (HAS_V && !acc_issued && te > tb) {
          if (te - tb > 1024) {
            block(tb, std::integral_constant<int, 0>{});
            block(tb + 1024, std::integral_constant<int, 1>{});
          } else {
            block(tb, std::integral_constant<int, 2>{});
          }
          acc_issued = true;
        } else {
          if (te > tb) block(tb, plain);
          if (te > tb + 1024) block(tb + 1024, plain);
        }
      }
      sure[it] = all ? upto : (exact ? 0u : upto & lower);
      memb[it] = all ? 0u : upto & ~sure[it];
      if (seg == 0 && lane == 0) tl_mem[h] = members[it];
      if (members[it] <= Tail::MEM) {  // (uniform)
        uint32_t m = memb[it];
        while (m != 0u) {
          const int pos = tb + place_of(__ffs((int)m) - 1);
          m &= m - 1u;
          const int k = atomicAdd(&tl_put[h], 1);
          if (k < Tail::MEM) tl_mlist[h * Tail::MEM + k] = rank_word(score_key(srow[pos]), pos);
        }
      }
    }
  }
  if (clk && tid == 0) clk[3] = JF_CLK();

  if constexpr (HAS_V) {  // whatever the emission did not carry (no batch of this wavefront, a short split, the exact selection)
    if (!acc_issued) add_acc_range(0, ACC_ITEMS);
  }
  // ONE: the outputs' addresses are read from the argument block again here (the compiler keeps what it has read, and with the
  // streams' own values the scalar registers do not hold it: some twenty of them went to vector lanes), all together ahead of
  // the barrier: read where each is used they were waited for one after the other (20 x 1000 positions, K3V2, top-k 128
  // 17.4 us per layer, all together 17.35).
  struct {
    int64_t *topk_idx, *topk_slots;
    float *o_hat, *o_old, *W, *softmax_m, *softmax_inv_z;
    const uint16_t* blend_o_new;
    uint16_t* blend_out;
    int64_t num_slots;
  } late = {};
  if constexpr (ONE) {
    auto args = (const __attribute__((address_space(4))) FusedParams*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(args));
    late = {args->topk_idx, args->topk_slots, args->o_hat, args->o_old, args->W, args->softmax_m, args->softmax_inv_z,
            args->blend_o_new, args->blend_out, args->num_slots};
    asm volatile("" : "+s"(late.topk_idx), "+s"(late.topk_slots), "+s"(late.o_hat), "+s"(late.o_old), "+s"(late.W),
                      "+s"(late.softmax_m), "+s"(late.softmax_inv_z), "+s"(late.blend_o_new), "+s"(late.blend_out), "+s"(late.num_slots));
    late_o_hat = late.o_hat;
  }
  if constexpr (HAS_V || ONE) lds_barrier();
  if constexpr (ONE) {
    int late_tid = tid, late_lane = lane;
    if constexpr (TIGHTER) {
      asm volatile("" : "+v"(late_tid));
      late_lane = late_tid & 63;
    }
    const int tid = late_tid, lane = late_lane;
    if (late.softmax_m && tid < GA) {
      late.softmax_m[head0 + tid] = tl_m[tid];
      late.softmax_inv_z[head0 + tid] = tl_iz[tid];
    }
    if constexpr (HAS_V) {
#pragma unroll
      for (int set = 0; set < NSET; ++set) combine(set);
    }
    // what the blend takes is requested here; behind the last barrier its first touch was waited for (20 x 1000 positions, K3V2,
    // top-k 128 18.2 us per layer, 17.9 with this; 32 x 2048, K4V4, 256 27.0 / 26.75)
    constexpr int OPT = (G * D + NT - 1) / NT;  // outputs per thread
    [[maybe_unused]] uint16_t o_new[OPT];
    if constexpr (MODE == FS_FULL) {
#pragma unroll
      for (int it = 0; it < OPT; ++it)  // (no blend: any readable address)
        o_new[it] = *(late.blend_o_new ? late.blend_o_new + head0 * D + min(it * NT + tid, GA * D - 1) : p.q + head0 * D);
    }
    if constexpr (HAS_TOPK) {
      // More members than a rank list holds: the buckets are linear between the smallest and the largest score, so one
      // outlying score (an attention sink) makes them wide, a correction of thousands puts hundreds of positions in
      // one, and equal scores share one.  Radix select over the rank words, eight bits a pass from the highest bit in
      // which a head's members differ: the head's wavefronts count the digits of their members, each finds the digit of
      // the last winner, and the head is done when the members left are as many as the winners left.  At most six
      // passes (the words are distinct), two or three where scores differ.  Ranking each such member against the whole
      // list, as this did at first, took 67 us per layer for 32 sequences x 2048 positions, K3V2, 8 kv-heads, top-k 256
      // and one score at 40 sigma (this: 29.5, no outlier: 24.9, splits of 256 with a merge launch: 103), and 1055 us
      // for 16 x 3900, K2V2, one head per kv-head, top-k 2048 and no outlier at all (31.6; 81).
      unsigned long long last[NHS] = {};  // the last winner among the head's members
      int ahead[NHS] = {};                // members that win in the segments before
      auto pair_of = [&](int it, int& h, int& seg) -> bool {  // (false: nothing for this wavefront)
        const int hs = wave + it * NW;
        h = hs / SEG;
        seg = hs % SEG;
        return hs < G * SEG && h < GA;
      };
      const int any_mem = tl_mem[min(lane, G - 1)];  // (the same in every wavefront)
      const unsigned long long crowded = __builtin_amdgcn_ballot_w64(lane < GA && any_mem > Tail::MEM);
      if (__builtin_expect(crowded != 0ull, 0)) {
        if constexpr (HAS_V) lds_barrier();  // (the sums in the staging area have been read)
        // per head the digit counts, the smallest and the largest member's key
        int* rh = reinterpret_cast<int*>(stage);
        uint32_t* ends = reinterpret_cast<uint32_t*>(rh + G * 256);
        static_assert(NW * Lds::WAVE_STAGE >= G * (256 * 4 + 8), "the digit counts lie in the staging area");
        auto for_members = [&](int it, int h, int seg, auto&& f) {  // four scores per lane in flight
          const int tb = seg * (L / SEG);
          const float* srow = sc + h * L;
#pragma unroll 1  // (unrolled, its lane masks spill)
          for (int i0 = 0; i0 < (SHORT ? STEPS : 32); i0 += 4) {
            float x[4];
            int pos[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              pos[u] = min(tb + place_of(i0 + u), n - 1);
              x[u] = srow[pos[u]];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
              if ((memb[it] >> (i0 + u)) & 1u) f(i0 + u, rank_word(score_key(x[u]), pos[u]));
          }
        };
        for (int i = tid; i < G * 256; i += NT) rh[i] = 0;
        if (tid < 2 * G) ends[tid] = (tid & 1) ? 0u : 0xffffffffu;
        if (tid < G) tl_nout[tid] = 0;
        lds_barrier();
#pragma unroll
        for (int it = 0; it < NHS; ++it) {
          int h, seg;
          if (!pair_of(it, h, seg) || !((crowded >> h) & 1ull)) continue;
          uint32_t kmin = 0xffffffffu, kmax = 0u;
          for_members(it, h, seg, [&](int, unsigned long long w) { kmin = min(kmin, (uint32_t)(w >> 12)); kmax = max(kmax, (uint32_t)(w >> 12)); });
          kmin = wave_min_u(kmin);
          kmax = wave_max_u(kmax);
          if (lane == 0) {
            atomicMin(&ends[2 * h], kmin);
            atomicMax(&ends[2 * h + 1], kmax);
          }
        }
        lds_barrier();
        int bits[NHS], want[NHS], left[NHS];
        unsigned long long top[NHS];  // members in the running have these bits above the lowest `bits` ones
#pragma unroll
        for (int it = 0; it < NHS; ++it) {
          int h, seg;
          bits[it] = want[it] = left[it] = 0;
          top[it] = 0ull;
          if (!pair_of(it, h, seg) || !((crowded >> h) & 1ull)) continue;
          const uint32_t kmin = __builtin_amdgcn_readfirstlane(ends[2 * h]), kmax = __builtin_amdgcn_readfirstlane(ends[2 * h + 1]);
          bits[it] = 12 + ((kmin == kmax) ? 0 : 32 - __clz((int)(kmin ^ kmax)));
          top[it] = rank_word(kmax, 0) >> bits[it];
          want[it] = need[it];
          left[it] = members[it];
        }
        for (int pass = 0; pass < 6; ++pass) {
#pragma unroll
          for (int it = 0; it < NHS; ++it) {
            int h, seg;
            if (!pair_of(it, h, seg) || left[it] == want[it]) continue;
            const int shift = max(0, bits[it] - 8);
            for_members(it, h, seg, [&](int, unsigned long long w) {
              if ((w >> bits[it]) == top[it]) atomicAdd(&rh[h * 256 + (int)((w >> shift) & ((1u << (bits[it] - shift)) - 1u))], 1);
            });
          }
          lds_barrier();
#pragma unroll
          for (int it = 0; it < NHS; ++it) {
            int h, seg;
            if (!pair_of(it, h, seg)) continue;
            if (left[it] != want[it]) {
              // lane l owns the digits 255 - 4l .. 252 - 4l: a scan over the lanes counts from the largest digit down
              const v4i c = *reinterpret_cast<const v4i*>(rh + h * 256 + 252 - 4 * lane);
              const int mine = (c[0] + c[1]) + (c[2] + c[3]);
              int above = wave_incl_scan_i(mine) - mine, digit = -1, count = 0, less = 0;
#pragma unroll
              for (int u = 3; u >= 0; --u) {
                if (above < want[it] && want[it] <= above + c[u]) {
                  digit = 252 - 4 * lane + u;
                  count = c[u];
                  less = above;
                }
                above += c[u];
              }
              const unsigned long long who = __builtin_amdgcn_ballot_w64(digit >= 0);
              const int src = (who != 0ull) ? __ffsll((long long)who) - 1 : 0;
              const int shift = max(0, bits[it] - 8);
              top[it] = (top[it] << (bits[it] - shift)) | (uint32_t)__builtin_amdgcn_readlane(digit, src);
              want[it] -= __builtin_amdgcn_readlane(less, src);
              left[it] = __builtin_amdgcn_readlane(count, src);
              bits[it] = shift;
            }
            if (seg == 0 && lane == 0) tl_nout[h] = left[it] - want[it];
          }
          lds_barrier();
          if (__builtin_amdgcn_ballot_w64(lane < GA && tl_nout[min(lane, G - 1)] != 0) == 0ull) break;
          for (int i = tid; i < G * 256; i += NT) rh[i] = 0;
          lds_barrier();
        }
        // the members that win join the sure winners; how many every segment has goes through LDS
#pragma unroll
        for (int it = 0; it < NHS; ++it) {
          int h, seg;
          if (!pair_of(it, h, seg) || !((crowded >> h) & 1ull)) continue;
          last[it] = top[it] << bits[it];
          const uint32_t alone = sure[it];
          for_members(it, h, seg, [&](int i, unsigned long long w) { sure[it] |= (w >= last[it] ? 1u : 0u) << i; });
          const int won = wave_sum_i(__popc(sure[it]) - __popc(alone));
          if (lane == 0) tl_segc[h * SEG + seg] = won;
        }
        lds_barrier();
#pragma unroll
        for (int it = 0; it < NHS; ++it) {
          int h, seg;
          if (!pair_of(it, h, seg) || !((crowded >> h) & 1ull)) continue;
#pragma unroll
          for (int sg = 0; sg < SEG; ++sg) ahead[it] += (sg < seg) ? tl_segc[h * SEG + sg] : 0;
        }
      }
#pragma unroll
      for (int it = 0; it < NHS; ++it) {
        int h, seg;
        if (!pair_of(it, h, seg)) continue;
        const int tb = seg * (L / SEG), m = members[it];
        const float* srow = sc + h * L;
        // a short list: every wavefront of the head finds the last winner itself, one member per lane (no exchange): few
        // members are ranked against each other as scalars (40 ns per member), more by bits (1 us)
        if (m > 0 && m <= Tail::MEM) {
          const unsigned long long own = (lane < m) ? tl_mlist[h * Tail::MEM + lane] : 0ull;
          unsigned long long held;
          if (m <= Tail::RANK) {
            int rank = 0;
            for (int k = 0; k < m; ++k) {
              const unsigned long long o = ((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(own >> 32), k) << 32) |
                                           (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)own, k);
              rank += (o > own) ? 1 : 0;
            }
            held = __builtin_amdgcn_ballot_w64(lane < m && rank == need[it] - 1);
          } else {
            held = (m < 64) ? (1ull << m) - 1ull : ~0ull;
            int place = need[it];
            nth_largest((uint32_t)(own >> 12), held, place);   // the key,
            nth_largest((uint32_t)own & 4095u, held, place);   // and among equal ones the position
          }
          const int src = (held != 0ull) ? __ffsll((long long)held) - 1 : 0;
          last[it] = ((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(own >> 32), src) << 32) |
                     (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)own, src);
          ahead[it] = __popcll(__builtin_amdgcn_ballot_w64(lane < m && own >= last[it] && 4095 - (int)((uint32_t)own & 4095u) < tb));
          uint32_t mm = memb[it];
          while (mm != 0u) {
            const int i = __ffs((int)mm) - 1, pos = tb + place_of(i);
            mm &= mm - 1u;
            sure[it] |= (rank_word(score_key(srow[pos]), pos) >= last[it] ? 1u : 0u) << i;
          }
        }
        // this wavefront's winners in position order
        uint16_t* cl = tl_list + h * Kcap;
        const int base = before[it] + ahead[it];
        int count = base;
        if constexpr (SHORT) {
#pragma unroll
          for (int i = 0; i < STEPS; ++i) {
            const bool win = ((sure[it] >> i) & 1u) != 0u;
            const unsigned long long mw = __builtin_amdgcn_ballot_w64(win);
            const int r = count + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mw >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mw, 0u));
            count += __popcll(mw);
            if (win && r < Kt) cl[r] = (uint16_t)(tb + 64 * i + lane);
          }
        } else {
#pragma unroll
          for (int blk = 0; blk < Lds::LMAX / SEG / 1024; ++blk) {
            uint32_t w = (sure[it] >> (16 * blk)) & 0xffffu;
            const int mine = __popc(w), incl = wave_incl_scan_i(mine);
            int r = count + incl - mine;
            count += __builtin_amdgcn_readlane(incl, 63);
            while (w != 0u) {
              if (r < Kt) cl[r] = (uint16_t)(tb + 1024 * blk + 16 * lane + __ffs((int)w) - 1);
              ++r;
              w &= w - 1u;
            }
          }
        }
        wave_lds_fence();
        // outputs, and slot and weight for the pre-correction, one winner per lane
        int64_t* out_idx = late.topk_idx + (head0 + h) * (size_t)K;
        int64_t* out_slot = late.topk_slots + (head0 + h) * (size_t)K;
        const float M = tl_m[h], iz = tl_iz[h];
        for (int r = base + lane; r < min(count, Kt); r += 64) {
          const int pos = min((int)cl[r], n - 1);
          const int slot = sbase[pos >> 4] + (pos & 15);
          out_idx[r] = pos;
          out_slot[r] = slot;
          if constexpr (HAS_V) {
            tl_wslot[h * K + r] = (slot >= 0 && slot < late.num_slots) ? slot : -1;
            tl_ww[h * K + r] = __expf(srow[pos] - M) * iz;
          }
        }
        for (int r = Kt + seg * 64 + lane; r < K; r += SEG * 64) {
          out_idx[r] = -1;
          out_slot[r] = -1;
        }
      }
    } else {  // Stage B alone: the winners are given (or none)
      const int n_out = late.topk_idx ? K : 0;
      if (tid < G) tl_nout[tid] = 0;
      lds_barrier();
      for (int i = tid; i < GA * n_out; i += NT) {
        const int h = i / K;
        const int64_t pos = late.topk_idx[head0 * K + i];
        const bool valid = pos >= 0 && pos < n;
        const int slot = valid ? sbase[(int)pos >> 4] + ((int)pos & 15) : -1;
        tl_wslot[i] = (slot >= 0 && slot < late.num_slots) ? slot : -1;
        tl_ww[i] = valid ? __expf(sc[h * L + (int)pos] - tl_m[h]) * tl_iz[h] : 0.f;
        // A head's list ends with its last entry that names a position (the padding of a short sequence is not gone
        // over: 1024 entries for eight heads over 16 positions took 50 us).  K >= 32: 32 lanes hold entries of one head.
        const uint32_t named = (uint32_t)(__builtin_amdgcn_ballot_w64(valid) >> (lane & 32));
        if (valid && (named >> (lane & 31)) == 1u) atomicMax(&tl_nout[h], i - h * K + 1);
      }
    }
    if constexpr (HAS_V) {
      lds_barrier();
      // ---- pre-correction over the winners
      // WPH wavefronts per head (more heads than wavefronts: one after the other), which take its winners 64 at a time in turn
      using Sums = WinnerSums<SCHEME % 10, NG>;
      constexpr int WPH = (NW >= G) ? NW / G : 1;
      // a wavefront's staging area: the rows of 64 winners; then (more heads than wavefronts: behind them) the head's sums
      constexpr int RES_AT = (G > NW) ? Sums::STAGE : 0, RES = (D + 4) * 4;
      static_assert(Lds::WAVE_STAGE >= Sums::STAGE && Lds::WAVE_STAGE >= RES_AT + (G + NW - 1) / NW * RES, "the sums lie in the staging area");
      static_assert(Lds::WAVE_STAGE % 16 == 0, "16-byte rows");
      uint8_t* st = stage + wave * Lds::WAVE_STAGE;
      if constexpr (TIGHT) asm volatile("" : "+v"(late_lane));
      for (int hw = wave; hw < GA * WPH; hw += NW) {
        const int lane = late_lane;
        const int h = hw / WPH, part = hw % WPH, n_out = HAS_TOPK ? Kt : __builtin_amdgcn_readfirstlane(tl_nout[h]);
        const int* slots = tl_wslot + h * K;
        const float* weights = tl_ww + h * K;
        float* res = reinterpret_cast<float*>(st + RES_AT + hw / NW * RES);
        float wsum = 0.f;
        if (K <= 16 * WPH) {  // (the correction's width, not the winners': Stage B is given a list of that length)
          // Few winners: code by code, WPI rows per wavefront instruction, four requests per lane at a time; a shorter chain than
          // the staged rows'.  1 x 777 positions, K4V4, top-k 64 14.35 us per layer, 14.8 the other way; 16 x 2048, K3V2, 64 20.6 /
          // 21.7.  (With up to half as many 20 x 1000, K3V2, 128 17.4 us, 17.6 the other way; 24 x 500, G = 8, 32 15.6 / 15.8.)
          using Pre = PreCorr<SCHEME % 10>;
          const int dwi = lane % Pre::DW, w_in = lane / Pre::DW;
          const int g_of_lane = (NG == 1) ? 0 : ((dwi * Pre::CPD) / (D / NG));
          float acc[Pre::CPD];
#pragma unroll
          for (int c = 0; c < Pre::CPD; ++c) acc[c] = 0.f;
          auto gather = [&](int first, auto count) JF_INLINE {  // `count` rows per lane from winner `first` on
            constexpr int NU = decltype(count)::value;
            typename Pre::Row row[NU];
            uint16_t sb[NU];
            int slot[NU];
            float wv[NU];
            // (all look-ups ahead of all rows: one round trip to LDS instead of one for each row's request)
#pragma unroll
            for (int u = 0; u < NU; ++u) {
              const int k = first + (u * WPH + part) * Pre::WPI + w_in, kc = min(k, n_out - 1);
              const int named = slots[kc];
              wv[u] = weights[kc];
              slot[u] = (k < n_out) ? named : -1;
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < NU; ++u) {
              wv[u] = (slot[u] >= 0) ? wv[u] : 0.f;
              const uint32_t sl = (uint32_t)max(slot[u], 0);
              row[u] = Pre::fetch(vbase, sl, dwi);
              sb[u] = *reinterpret_cast<const uint16_t*>(vsbase + (size_t)(sl * (uint32_t)(NG * 2)) + g_of_lane * 2);
            }
            if constexpr (Pre::ALL_AHEAD) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < NU; ++u) {
              Pre::add(row[u], slot[u] >= 0 ? wv[u] * bf16_to_f32(sb[u]) : 0.f, acc);  // (whatever scale slot 0 has)
              if (dwi == 0) wsum += wv[u];
            }
          };
          constexpr int ROWS = WPH * Pre::WPI;  // winners per row of every lane
          int first = 0;
          for (; n_out - first > 2 * ROWS; first += 4 * ROWS) gather(first, std::integral_constant<int, 4>{});
          if (first < n_out) gather(first, std::integral_constant<int, 2>{});
          const int chan = Pre::reduce(acc, lane);
          res[chan] = acc[0];
          res[chan + 1] = acc[1];
        } else {
          float o[2] = {};
          int first = part * 64;
          if (first < n_out) {
            typename Sums::Rows x = Sums::fetch(vbase, vsbase, slots, weights, first, n_out, lane);
            for (;;) {
              const bool more = first + WPH * 64 < n_out;  // (uniform)
              typename Sums::Rows next = x;
              if (more) next = Sums::fetch(vbase, vsbase, slots, weights, first + WPH * 64, n_out, lane);
              wsum += x.w;
              Sums::add(x, st, lane, o);
              if (!more) break;
              x = next;
              first += WPH * 64;
            }
          }
#pragma unroll
          for (int i = 0; i < 2; ++i) res[Sums::channel(lane, i)] = o[i];
        }
        wsum = wave_sum(wsum);
        if (lane == 0) res[D] = wsum;
      }
      lds_barrier();
#pragma unroll
      for (int it = 0; it < OPT; ++it) {
        const int i = it * NT + tid, h = i >> 7, d = i & 127;
        if (i >= GA * D) break;
        float o = 0.f, wt = 0.f;
#pragma unroll
        for (int w = 0; w < WPH; ++w) {
          const int hw = h * WPH + w;
          const float* res = reinterpret_cast<const float*>(stage + hw % NW * Lds::WAVE_STAGE + RES_AT + hw / NW * RES);
          o += res[d];
          wt += res[D];
        }
        late.o_old[(head0 + h) * D + d] = o;
        if (d == 0) late.W[head0 + h] = wt;
        if (MODE == FS_FULL && late.blend_out) {
          const size_t at = (head0 + h) * D + d;
          late.blend_out[at] = f32_to_bf16(__builtin_fmaf(wt, bf16_to_f32(o_new[it]), tl_ohat[h * D + d]) - o);
        }
      }
    }
    if (clk && tid == 0) clk[4] = JF_CLK();
    return;
  }
  float lfin = 0.f;
  if (tid < G) {
#pragma unroll
    for (int w = 0; w < NW; ++w) lfin += lsum_sh[w][tid];
  }
#pragma unroll
  for (int set = 0; set < NSET; ++set)
    if constexpr (HAS_V) combine(set);
  if (tid < GA) {
    p.part_m[part_base + (size_t)tid * p.n_splits] = m_sh[tid];
    p.part_l[part_base + (size_t)tid * p.n_splits] = lfin;
  }
  if (clk && tid == 0) clk[4] = JF_CLK();
}

// Reductions over one value per wavefront (at most sixteen, in LDS): lane w of the first 16-lane row takes
// wavefront w's value, the row reduces on the DPP network and the result is read from lane 15 -- a handful of
// instructions instead of a loop over the sixteen entries in every thread.  Integer and min/max only: the result
// does not depend on the order.
template <int NWV>
__device__ inline uint32_t waves_max_u(const uint32_t* arr, int lane) {
  uint32_t v = (lane < NWV) ? arr[lane] : 0u;
  JF_DPP_ROW_REDUCE(v, op_umax, uint32_t, 0u);
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 15);
}
template <int NWV>
__device__ inline uint32_t waves_min_u(const uint32_t* arr, int lane) {
  uint32_t v = (lane < NWV) ? arr[lane] : 0xffffffffu;
  JF_DPP_ROW_REDUCE(v, op_umin, uint32_t, 0xffffffffu);
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 15);
}
// sum of the entries before wavefront `wave` (uniform) and of all entries
template <int NWV>
__device__ inline void waves_prefix_i(const int* arr, int lane, int wave, int* before, int* all) {
  const int own = (lane < NWV) ? arr[lane] : 0;
  int v = own;
  JF_DPP_ROW_REDUCE(v, op_iadd, int, 0);  // inclusive scan inside the row
  *before = __builtin_amdgcn_readlane(v - own, wave);
  *all = __builtin_amdgcn_readlane(v, 15);
}

// ---------------------------------------------------------------------------------------------------
constexpr int MG_MAX_SPLITS = 256;
constexpr int MG_BINS = 512;       // linear score buckets of the threshold search (32 candidates per thread: twice as many); the last one holds all that lies below
constexpr int MG_LIST = 1024;      // members of the cut bucket resolved by rank counting
constexpr int MG_RANK = 16;        // up to here all pairs at once in every wavefront, beyond over the list in LDS
constexpr int MG_BT_LDS = 4096;    // block-table entries cached in LDS (65536 positions)
constexpr int MG_LIGHT_THREADS = 256, MG_LIGHT_REGK = 16, MG_LIGHT_TOPK = 512;  // the light shape of the merge
constexpr int MG_MEDIUM_THREADS = 512, MG_MEDIUM_REGK = 16;                     // the medium one

// Launch 2: one workgroup per (sequence, query head).
//   1. split statistics -> M, l, o_hat; a lower bound of the K-th largest score from the splits' own cuts
//   2. the K-th largest candidate: the candidates are dropped into MG_BINS linear score buckets between that bound and
//      the largest score, a scan finds the bucket that holds the K-th largest, and the few members of that bucket are
//      ranked against each other (a bisection over the key range covers the case of more than MG_LIST members)
//   3. ordered compaction of the winners (candidates are stored in position order, so ties resolve to the lower
//      position and the output is ascending)
//   4. slots, softmax weights, and the pre-correction terms over the winners' V rows.
// The first MG_REGK * MG_THREADS candidates stay in registers from a single load; anything beyond that is
// re-read from global memory in every pass.
// Shapes: 1024 threads x 8 register-resident candidates each (up to 8192 candidates, the common case), 1024 x 32 beyond, and
// 512 x 16 and 256 x 16 where there are more rows than CUs.
//
// What bounds it is neither memory nor launch: run a second time over warm caches the same workgroup takes as long.  It
// is the length of the chain every wavefront goes through, some 900 instructions and a dozen round trips to LDS, which
// four wavefronts per SIMD share.  So: the arguments come in one block, first the ones the first loads need (scattered
// over the scan's they were four dependent scalar loads); the loads are range-checked buffer loads, 16 bytes of candidates
// each, instead of clamped and masked ones; every wavefront reduces the splits' statistics for itself (lane = split); the
// range of the buckets comes with the lists instead of from a pass over the candidates; few members of the cut bucket are
// ranked all pairs at once, in every wavefront.  Six barriers instead of twelve.  Per layer, graph replay, before / now:
// 1 x 4096 positions, K4V4, top-k 64 20.5 / 18.3 us; 4 x 8100, B4V4 30.3 / 28.9; 4 x 32768, K3V2 36.1 / 35.0;
// the same with G = 8 33.4 / 32.3; 1 x 131072, K4V4, top-k 512 (two stages) 49.3 / 48.0.
// Lane masks are short-lived: no comparison of the candidates is made twice in a form the compiler could recognise (an unused
// slot's bucket lies behind all others instead of a second test of its key; the bounds of the second pass are opaque; counts
// are taken at once).  Kept from one pass to the next the masks took 93 scalar registers in the first stage, which with the
// trap handler's 16 leaves one workgroup per CU instead of two, and 190 spilled words in the shape of 32 candidates.  First
// stage, 1024 / 1664 workgroups of 7000 candidates, top-k 1024 35.9 -> 22.5, 55.0 -> 33.7 us; 32-candidate shape, 16 / 512 /
// 1376 rows 22.2 -> 15.6, 80.9 -> 67.6, 257 -> 223 us.
// PARTIAL = true is the first stage of the two-stage merge: blockIdx.z selects a run of mg_spp candidate
// lists, steps 2 and 3 run on those alone and the winners (still in position order) are written out as one
// new candidate list; the final merge (PARTIAL = false, mg_parts > 1) reads these lists instead of the
// scan's.  The top K of a union is the top K of the parts' top K's, ties included: a candidate that a part
// drops is beaten by K candidates of that part.
// (Stage B alone keeps no candidates: registers for two workgroups per CU.  One more than the 64 that allows, INT3 values, and 512 rows (16
// sequences x 4096 positions, top-k 256) took 27.6 us per layer, 24.5 with the bound.)
template <int MODE, int VBITS, int NG, int MG_THREADS, int MG_REGK, bool PARTIAL, bool WIDE = false, int PER_CU = 1>
__global__ __launch_bounds__(MG_THREADS, PER_CU == 4 ? 4 : (MODE == FS_STAGE_B ? 2 : 1) * MG_THREADS / 256) void fused_merge_kernel(MergeParams p) {
  static_assert(!(PARTIAL && MODE == FS_STAGE_B), "Stage B alone selects nothing");
  constexpr int MG_WAVES = MG_THREADS / 64;
  // PER_CU = 4, light shape: four workgroups per CU are all there are, and a wavefront has registers for the rows of both its turns
  constexpr bool AHEAD = PER_CU == 4;
  // The floating-point sums (o_hat over the splits, the pre-correction terms over the winners) are organised
  // as if eight thread groups of 128 and eight wavefronts were at work, whatever MG_THREADS is: a smaller
  // workgroup takes several of those roles one after the other, so every shape of this kernel adds the same
  // numbers in the same order and the results do not depend on which shape the launcher picks.
  constexpr int VGRP = 8;
  static_assert(MG_THREADS % D == 0 && VGRP % (MG_THREADS / D) == 0 && (MG_WAVES >= VGRP || VGRP % MG_WAVES == 0), "whole roles per thread group / wavefront");
  // the light shape (many rows per launch, few candidates per row) trades table sizes for workgroups per CU
  constexpr int MG_BT = (MG_THREADS > MG_LIGHT_THREADS) ? MG_BT_LDS : 1024;  // block-table entries cached in LDS
  constexpr int MG_WIN = (MG_THREADS > MG_LIGHT_THREADS) ? FS_LDS_TOPK : 512;  // widest correction of this shape (WIDE: any)
  // (the shape of 32 candidates per thread meets wide corrections, whose cut lies where the scores are densest: twice the buckets)
  constexpr int BINS = (MG_REGK > 16) ? 2 * MG_BINS : MG_BINS;
  // The sums over the winners need a staging area; what the selection needs lies in the same place (a barrier lies between).  Side by
  // side the two took the 1024-thread shape longer to start than they saved: 16 sequences x 4096 positions, K3V2, top-k 1024 46.6 us
  // per layer, this 46.0; 1 x 131072, K4V4, 512 46.4 / 46.05.
  using Sums = WinnerSums<VBITS, NG>;
  constexpr bool HAS_SUMS = !PARTIAL && MODE != FS_STAGE_A;
  constexpr int SUM_WAVES = MG_WAVES < VGRP ? MG_WAVES : VGRP;
  constexpr int EARLY = (BINS + MG_LIST + MG_BT + VGRP * D) * 4, AREAS = (AHEAD && VBITS < 4) ? 2 : 1,  // one for each turn (INT4 rows: that would be three workgroups per CU)
                STAGED = HAS_SUMS ? AREAS * SUM_WAVES * Sums::STAGE : 0;
  __shared__ __align__(16) uint8_t pool[!HAS_SUMS ? 16 : (EARLY > STAGED ? EARLY : STAGED)];
  __shared__ __align__(16) int hist_s[HAS_SUMS ? 1 : BINS];
  __shared__ uint32_t lkey_s[HAS_SUMS ? 1 : MG_LIST];
  __shared__ int bt_s[HAS_SUMS ? 1 : MG_BT];
  __shared__ float red_s[HAS_SUMS ? 1 : VGRP][D];
  int* const hist = HAS_SUMS ? reinterpret_cast<int*>(pool) : hist_s;
  uint32_t* const lkey = HAS_SUMS ? reinterpret_cast<uint32_t*>(pool) + BINS : lkey_s;
  int* const bt_sh = HAS_SUMS ? reinterpret_cast<int*>(pool) + BINS + MG_LIST : bt_s;
  float (*const red_sh)[D] = HAS_SUMS ? reinterpret_cast<float (*)[D]>(pool + (BINS + MG_LIST + MG_BT) * 4) : red_s;
  __shared__ int lpos[MG_RANK];  // candidate number of the first members
  // winners: key and position while they are selected; the thread that turns winner r into its softmax weight and
  // paged slot overwrites the two entries in place (weight bits over the key, slot over the position)
  // (WIDE, corrections beyond FS_LDS_TOPK: the two arrays are the launch's dynamic LDS, top_k entries each)
  __shared__ uint32_t win_key_s[WIDE ? 1 : MG_WIN];
  __shared__ int win_idx_s[WIDE ? 1 : MG_WIN];
  extern __shared__ __align__(16) uint32_t win_dyn[];
  uint32_t* const win_key = WIDE ? win_dyn : win_key_s;
  int* const win_idx = WIDE ? reinterpret_cast<int*>(win_dyn + p.top_k) : win_idx_s;
  __shared__ float sum_sh[HAS_SUMS ? SUM_WAVES : 1][D];
  __shared__ float ohat_sh[D];
  __shared__ float w_sh[VGRP];
  __shared__ uint32_t wred_u[MG_WAVES], wred_k[MG_WAVES];
  __shared__ int wred_i[MG_WAVES], wred_j[MG_WAVES];
  __shared__ int lcount_sh, quota_sh;
  __shared__ uint32_t tau_sh;

  // (first stage: x = sequence, y = query head, z = part; else x = head of the group, y = kv-head, z = sequence)
  const int b = PARTIAL ? blockIdx.x : blockIdx.z, hkv = PARTIAL ? 0 : blockIdx.y, tid = threadIdx.x, lane = tid & 63;
  const int hq = PARTIAL ? blockIdx.y : hkv * p.g_act + blockIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const size_t bh = (size_t)b * p.H_q + hq;
  const int NS = p.n_splits, K = p.top_k, Kc = p.list_cap, LL = p.list_len;
  // candidate lists of this workgroup: NL lists of capacity Kc, each over LL positions
  const int part = PARTIAL ? (int)blockIdx.z : 0;
  const int l0 = PARTIAL ? part * p.mg_spp : 0;
  // (Stage B alone: the winners are an input, there are no candidate lists)
  constexpr bool HAS_LISTS = (MODE != FS_STAGE_B);
  const int NL = !HAS_LISTS ? 0 : (PARTIAL ? min(p.mg_spp, p.lists - l0) : p.lists);
  const size_t list0 = bh * p.lists + l0, split0 = bh * NS + l0;
  const uint32_t* ck = p.list_key + list0 * Kc;
  const int32_t* ci = p.list_idx + list0 * Kc;
  const float* ce = p.list_edge + list0;
  const int64_t* bt = p.block_table + (size_t)b * p.max_blocks;
  const int flat = NL * Kc;
  const int nblk_lds = min(p.max_blocks, MG_BT);

  long long* mclk = (kDebugHooks && p.phase_clock && !PARTIAL) ? p.phase_clock + bh * 8 : nullptr;
  if (mclk && tid == 0) mclk[0] = JF_CLK();

  // ---- everything that does not depend on anything else is requested first, in the order of its use: one round trip
  // of first touches (what other XCDs wrote) instead of one after the other.  Buffer loads: past the end of what the
  // descriptor covers they return zero, so neither clamps nor masks are needed.
  // (given statistics, jf_softmax_v_int8_tiles: the partial rows are already normalised and come without maxima and
  // sums)
  const bool has_parts = MODE != FS_STAGE_B || p.part_m != nullptr;
  constexpr int SPL = MG_MAX_SPLITS / 64;  // splits per lane
  const int NV = PARTIAL ? NL : NS;        // splits whose statistics are read
  float pm[SPL], pl[SPL], pe[SPL];
  // (a vector load: a wait for the kernel's arguments would wait for any scalar load that is under way)
  const int len_mine = buffer_i32(buffer_of(p.seq_lens + b, 4), 0, 0);
  const auto rm = buffer_of(p.part_m + split0, has_parts ? NV * 4 : 0), rl = buffer_of(p.part_l + split0, has_parts ? NV * 4 : 0);
  const auto re = buffer_of(ce, NL * 4);
  const bool many = NV > 64;  // (uniform) more splits than lanes
#pragma unroll
  for (int i = 0; i < SPL; ++i) pm[i] = pl[i] = pe[i] = 0.f;
  auto request_split = [&](int i) {
    pm[i] = buffer_f32(rm, lane * 4, i * 256);
    if constexpr (HAS_LISTS) pe[i] = buffer_f32(re, lane * 4, i * 256);
    pl[i] = buffer_f32(rl, lane * 4, i * 256);
  };
  request_split(0);
  if (many) {
#pragma unroll
    for (int i = 1; i < SPL; ++i) request_split(i);
  }
  // The first MG_REGK * MG_THREADS candidates live in registers: wavefront w holds `per` x 64 consecutive ones, 256 per group
  // of four registers, of which lane l has the four at 4 l (one 16-byte load).  Slots past a list's end hold key 0 (written
  // by the producer).
  static_assert(MG_REGK % 4 == 0, "register candidates come in groups of four");
  constexpr int NGRP = MG_REGK / 4;
  constexpr bool LAZY = MG_REGK > 16;  // the positions of the winners are fetched when they are known
  const int per = min((flat + 4 * MG_THREADS - 1) / (4 * MG_THREADS), NGRP) * 4;  // registers in use (uniform)
  const int f0 = wave * per * 64;  // number of this wavefront's first candidate
  auto f_of = [&](int r) -> int { return f0 + (r >> 2) * 256 + lane * 4 + (r & 3); };
  const auto rk = buffer_of(ck, flat * 4), ri = buffer_of(ci, flat * 4);
  uint32_t kreg[MG_REGK];
  int ireg[LAZY ? 1 : MG_REGK];
#pragma unroll
  for (int g = 0; g < NGRP; ++g) {
    v4i x = {0, 0, 0, 0};
    if (HAS_LISTS && (g == 0 || 4 * g < per)) x = buffer_i32x4(rk, lane * 16, (f0 + g * 256) * 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) kreg[4 * g + j] = (uint32_t)x[j];
  }
  if constexpr (!LAZY) {
#pragma unroll
    for (int g = 0; g < NGRP; ++g) {
      v4i x = {0, 0, 0, 0};
      if (HAS_LISTS && (g == 0 || 4 * g < per)) x = buffer_i32x4(ri, lane * 16, (f0 + g * 256) * 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) ireg[4 * g + j] = x[j];
    }
  }
  // o_hat: the thread groups of 128 take the splits round-robin (first terms requested now)
  constexpr int PO_PRE = 2, PO_GRP = MG_THREADS / D;
  const int q4 = wave / (D / 64);
  const auto ro = buffer_of(p.part_o + bh * NS * D, NS * D * 4);
  float po[PO_PRE];
#pragma unroll
  for (int i = 0; i < PO_PRE; ++i) {
    po[i] = 0.f;
    if constexpr (MODE != FS_STAGE_A && !PARTIAL) po[i] = buffer_f32(ro, (tid & (D - 1)) * 4, (q4 + VGRP * i) * (D * 4));
  }
  // page-table entries for the table in LDS (the low half of the 64-bit entry only)
  constexpr int BTPT = (MG_BT + MG_THREADS - 1) / MG_THREADS;
  int bt_mine[BTPT];
  const auto rb = buffer_of(bt, nblk_lds * 8);
#pragma unroll
  for (int i = 0; i < BTPT; ++i) bt_mine[i] = 0;
  if constexpr (!PARTIAL) {
    bt_mine[0] = buffer_i32(rb, tid * 8, 0);
    if (nblk_lds > MG_THREADS) {  // (uniform)
#pragma unroll
      for (int i = 1; i < BTPT; ++i) bt_mine[i] = buffer_i32(rb, tid * 8, i * MG_THREADS * 8);
    }
  }
  uint16_t blend_raw = 0;
  if constexpr (MODE == FS_FULL && !PARTIAL)  // (no blend: any readable address)
    blend_raw = *(p.blend_o_new ? p.blend_o_new + bh * D + (tid & (D - 1)) : reinterpret_cast<const uint16_t*>(ck));
  for (int i = tid; i < BINS; i += MG_THREADS) hist[i] = 0;
  if (tid == 0) lcount_sh = 0;
  lds_barrier();

  // positions the lists stand for; not more than K of them: every candidate wins
  const int S = max(0, min(p.max_S, __builtin_amdgcn_readfirstlane(len_mine))) - l0 * LL;
  const bool take_all = (PARTIAL ? min(S, NL * LL) : S) <= K;  // (uniform)
  // ---- interval 1: the statistics, in every wavefront; the candidates drop into the buckets
  // The K-th largest score is no smaller than the cut of any list that stands for at least K positions (K of its own
  // lie above), nor than the smallest of all cuts.
  // (reduced as order-preserving integers, 0 below every score: one instruction a step)
  const bool whole = LL >= K;  // (uniform) lists of K positions: their largest cut; else the smallest cut
  const uint32_t flip = whole ? 0u : 0xffffffffu;
  uint32_t m_key = 0u, e_key = 0u;
  auto take_split = [&](int i) {
    const int s = lane + 64 * i;
    pm[i] = (s < NV && has_parts) ? pm[i] : -INFINITY;
    m_key = max(m_key, score_key(pm[i]));
    const int n_list = S - s * LL;  // (a list past the end of the sequence: not above zero)
    const uint32_t e = score_key(pe[i]) ^ flip;
    e_key = max(e_key, (s < NL && n_list >= (whole ? K : 1)) ? e : 0u);
  };
  take_split(0);
  if (many) {
#pragma unroll
    for (int i = 1; i < SPL; ++i) take_split(i);
  }
  m_key = wave_max_u(m_key);
  e_key = wave_max_u(e_key) ^ flip;
  float M = key_to_score(m_key);
  const float hi = M, lo = key_to_score(e_key);
  if (!isfinite(M)) M = 0.f;
  float coef[SPL], lsum = 0.f;
#pragma unroll
  for (int i = 0; i < SPL; ++i) coef[i] = 0.f;
  auto weigh_split = [&](int i) {
    coef[i] = (pm[i] == -INFINITY) ? 0.f : __expf(pm[i] - M);
    lsum += wave_sum(pl[i] * coef[i]);  // fixed reduction tree: deterministic
    if (!has_parts) coef[i] = 1.f;
  };
  weigh_split(0);
  if (many) {
#pragma unroll
    for (int i = 1; i < SPL; ++i) weigh_split(i);
  }
  // (bucket 0 = largest scores; the last one, for what lies below `lo`, is not counted)
  const float range = hi - lo;
  const float iw = ((float)BINS - 1.5f) * __builtin_amdgcn_rcpf(range);
  const float bb = hi * iw;
  // No usable range (all cuts at the largest score, infinite scores), or a NaN among the scores, whose place in the order
  // of the keys the buckets do not know (its split's sum of weights is a NaN too): bisection over the keys.
  const bool exact = !take_all && !(range > 0.f && isfinite(range) && isfinite(iw) && isfinite(bb) && lsum == lsum);  // (uniform)
  // (an unused slot's key 0 stands for a NaN, which the minimum turns into the last bucket)
  auto bin_of = [&](uint32_t k) -> int {
    return (int)__builtin_fmaxf(__builtin_fminf(__builtin_fmaf(key_to_score(k), -iw, bb), (float)(BINS - 1)), 0.f);
  };
  // key of candidate f in pass-over-all-candidates loops: registers first, global memory beyond
  const int rounds = (flat + MG_THREADS - 1) / MG_THREADS;
  auto key_of = [&](int r) -> uint32_t {
    const int f = r * MG_THREADS + tid;
    return (f < flat) ? ck[f] : 0u;
  };
  int bin[MG_REGK];
#pragma unroll
  for (int r = 0; r < MG_REGK; ++r) bin[r] = BINS;  // (unused slots, behind all buckets: a winner's or a member's bin says it all)
  if constexpr (HAS_LISTS) {
    if (take_all) {
#pragma unroll
      for (int r = 0; r < MG_REGK; ++r) bin[r] = (kreg[r] != 0u) ? 0 : BINS;
    } else if (!exact) {
#pragma unroll
      for (int g = 0; g < NGRP; ++g)
        if (g == 0 || 4 * g < per) {
#pragma unroll
          for (int r = 4 * g; r < 4 * g + 4; ++r) {
            bin[r] = (kreg[r] != 0u) ? bin_of(kreg[r]) : BINS;
            if (bin[r] < BINS - 1) atomicAdd(&hist[bin[r]], 1);
          }
        }
      for (int r = MG_REGK; r < rounds; ++r) {
        const uint32_t k = key_of(r);
        if (k != 0u) {
          const int c = bin_of(k);
          if (c < BINS - 1) atomicAdd(&hist[c], 1);
        }
      }
    }
  }
  if constexpr (!PARTIAL) {
    bt_sh[tid] = bt_mine[0];
    if (nblk_lds > MG_THREADS) {
#pragma unroll
      for (int i = 1; i < BTPT; ++i) bt_sh[tid + i * MG_THREADS] = bt_mine[i];
    }
  }
  if constexpr (!PARTIAL && MODE != FS_STAGE_A) {
    // o_hat: group vg of the eight takes every eighth split, then a fixed-order sum (after the next barrier)
    auto coef_of = [&](int sp) -> float {  // (sp is uniform)
      float c = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, coef[0]), sp & 63));
      if (!many) return c;
#pragma unroll
      for (int i = 1; i < SPL; ++i)
        if (sp / 64 == i) c = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, coef[i]), sp & 63));
      return c;
    };
    const int d4 = (tid & (D - 1)) * 4;
#pragma unroll
    for (int v = 0; v < VGRP / PO_GRP; ++v) {
      const int vg = q4 + v * PO_GRP;
      float o = 0.f;
#pragma unroll
      for (int i = 0; i < PO_PRE; ++i) {
        const int sp = vg + VGRP * i;
        if (sp < NS) o = __builtin_fmaf((v == 0) ? po[i] : buffer_f32(ro, d4, sp * (D * 4)), coef_of(sp), o);
      }
      // the remaining splits eight at a time: the loads of a batch are in flight together, the sum keeps its order
      constexpr int PO_B = 8;
      for (int sp0 = vg + VGRP * PO_PRE; sp0 < NS; sp0 += VGRP * PO_B) {
        float w[PO_B];
#pragma unroll
        for (int u = 0; u < PO_B; ++u) w[u] = buffer_f32(ro, d4, (sp0 + VGRP * u) * (D * 4));
#pragma unroll
        for (int u = 0; u < PO_B; ++u)
          if (sp0 + VGRP * u < NS) o = __builtin_fmaf(w[u], coef_of(sp0 + VGRP * u), o);
      }
      red_sh[vg][tid & (D - 1)] = o;
    }
  }
  if (mclk && tid == 0) mclk[6] = JF_CLK();
  lds_barrier();
  if (mclk && tid == 0) mclk[7] = JF_CLK();
  int n_out = 0;
  float edge = whole ? -INFINITY : lo;  // PARTIAL: no winner scores less
  if constexpr (HAS_LISTS) {
    // ---- interval 2, in every wavefront: the bucket of the K-th largest; the wavefront's candidates before it, and the
    // list of that bucket's members
    int cut = 1, need = 0;  // (every candidate wins: they are in bucket 0)
    if (!take_all && !exact) {
      constexpr int BPL = BINS / 64;  // lane l owns buckets BPL * l .. (ascending bucket = descending score)
      static_assert(BPL % 4 == 0, "16-byte reads");
      int mine = 0;
#pragma unroll
      for (int u = 0; u < BPL; u += 4) {
        const v4i x = *reinterpret_cast<const v4i*>(hist + BPL * lane + u);
        mine += (x[0] + x[1]) + (x[2] + x[3]);
      }
      const int incl = wave_incl_scan_i(mine);
      const unsigned long long who = __builtin_amdgcn_ballot_w64(incl >= K);
      cut = BINS - 1;
      int above = __builtin_amdgcn_readlane(incl, 63);
      if (who != 0ull) {
        const int src = __ffsll((long long)who) - 1;
        // the buckets of that lane, one per lane
        const int own = (lane < BPL) ? hist[BPL * src + lane] : 0;
        int run = own;
        JF_DPP_ROW_REDUCE(run, op_iadd, int, 0);  // inclusive scan inside the row
        run += __builtin_amdgcn_readlane(incl - mine, src);
        const int u = __ffsll((long long)__builtin_amdgcn_ballot_w64(run >= K)) - 1;  // (the lane's total reaches K)
        static_assert(BPL <= 16, "one row");
        cut = BPL * src + u;
        above = __builtin_amdgcn_readlane(run - own, u);
      }
      need = K - above;  // so many of the cut bucket's members belong to the top K
    }
    int n_above = 0;
    bool has_members = false;  // (uniform)
    auto list_member = [&](uint32_t key, int f) {
      const int i = atomicAdd(&lcount_sh, 1);
      if (i < MG_LIST) lkey[i] = key;
      if (i < MG_RANK) lpos[i] = f;
    };
    if (!exact) {
#pragma unroll
      for (int g = 0; g < NGRP; ++g)
        if (g == 0 || 4 * g < per) {
#pragma unroll
          for (int r = 4 * g; r < 4 * g + 4; ++r) {
            n_above += __popcll(__builtin_amdgcn_ballot_w64(bin[r] < cut));
            const bool member = bin[r] == cut;
            if (__builtin_amdgcn_ballot_w64(member) != 0ull) {
              has_members = true;
              if (member) list_member(kreg[r], f_of(r));
            }
          }
        }
      if (!take_all) {
        for (int r = MG_REGK; r < rounds; ++r) {
          const uint32_t k = key_of(r);
          if (k != 0u && bin_of(k) == cut) list_member(k, r * MG_THREADS + tid);
        }
      }
    }
    if (lane == 0) wred_i[wave] = n_above;
    lds_barrier();
    if (mclk && tid == 0) mclk[1] = JF_CLK();
    const int m = __builtin_amdgcn_readfirstlane(lcount_sh);
    if (!exact && m <= MG_RANK && rounds <= MG_REGK) {
      // ---- interval 3: the last winner among the members (larger key first, then lower position), then every winner
      // stores its key and position at its place
      uint32_t tk = 0u;
      int tf = -1, own_f = 0;
      unsigned long long won = 0ull;  // members that win (bit = place in the list)
      if (m > 0) {  // (uniform) all pairs: lane (i, j) compares member 4 * step + i with member j
        const int j = lane & 15, i = lane >> 4;
        const bool vj = j < m;
        const uint32_t kj = vj ? lkey[j] : 0u;
        const int fj = vj ? lpos[j] : 0x7fffffff;
        uint32_t ki[MG_RANK / 4];
        int fi[MG_RANK / 4], sel = 0;
#pragma unroll
        for (int st = 0; st < MG_RANK / 4; ++st) {
          ki[st] = lkey[4 * st + i];
          fi[st] = lpos[4 * st + i];
        }
        own_f = fj;
#pragma unroll
        for (int st = 0; st < MG_RANK / 4; ++st) {
          if (4 * st < m) {
            const unsigned long long gt = __builtin_amdgcn_ballot_w64(vj && (kj > ki[st] || (kj == ki[st] && fj < fi[st])));
            const int rank = __popc((uint32_t)(gt >> (16 * i)) & 0xffffu);
            const unsigned long long hit = __builtin_amdgcn_ballot_w64(4 * st + i < m && rank == need - 1);
            if (hit != 0ull) sel = 4 * st + (__ffsll((long long)hit) - 1) / 16;
          }
        }
        tk = (uint32_t)__builtin_amdgcn_readlane((int)kj, sel);
        tf = __builtin_amdgcn_readlane(fj, sel);
        won = __builtin_amdgcn_ballot_w64(lane < 16 && vj && (kj > tk || (kj == tk && fj <= tf)));
      }
      int before, all;
      waves_prefix_i<MG_WAVES>(wred_i, lane, wave, &before, &all);
      int place = before + __popcll(won & __builtin_amdgcn_ballot_w64(own_f < f0));
      n_out = min(K, all + __popcll(won));
#pragma unroll
      for (int g = 0; g < NGRP; ++g)
        if (g == 0 || 4 * g < per) {
          bool win[4];
          int mine = 0;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int r = 4 * g + j;
            win[j] = bin[r] < cut;
            if (has_members)  // (uniform)
              win[j] = win[j] || (bin[r] == cut && (kreg[r] > tk || (kreg[r] == tk && f_of(r) <= tf)));
            mine += win[j] ? 1 : 0;
          }
          const int incl = wave_incl_scan_i(mine);
          int at = place + incl - mine;
          place += __builtin_amdgcn_readlane(incl, 63);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int r = 4 * g + j;
            if (win[j]) {
              if (at < K) {
                win_key[at] = kreg[r];
                win_idx[at] = LAZY ? f_of(r) : ireg[LAZY ? 0 : r];
              }
              ++at;
            }
          }
        }
      if (PARTIAL && !take_all) edge = key_to_score(tk);
    } else {
      // ---- the general case: tau = the K-th largest key, `quota` of the keys equal to it win
      uint32_t tau = 0u;
      int quota = 0;
      if (take_all) {
        quota = 0;
      } else if (!exact && m <= MG_LIST) {
        // rank counting: the member with fewer than `need` larger members and at least `need` members >= it
        for (int i = tid; i < m; i += MG_THREADS) {
          const uint32_t k = lkey[i];
          int gt = 0, ge = 0;
          for (int j = 0; j < m; ++j) {
            const uint32_t o = lkey[j];
            gt += (o > k) ? 1 : 0;
            ge += (o >= k) ? 1 : 0;
          }
          if (gt < need && need <= ge) {  // every thread that gets here writes the same pair
            tau_sh = k;
            quota_sh = need - gt;
          }
        }
        lds_barrier();
        tau = tau_sh;
        quota = quota_sh;
      } else {
        // bisection over the key range: largest x with count(key >= x) >= K
        uint32_t kmin = 0xffffffffu, kmax = 0u;
#pragma unroll
        for (int r = 0; r < MG_REGK; ++r)
          if (kreg[r] != 0u) { kmin = min(kmin, kreg[r]); kmax = max(kmax, kreg[r]); }
        for (int r = MG_REGK; r < rounds; ++r) {
          const uint32_t k = key_of(r);
          if (k != 0u) { kmin = min(kmin, k); kmax = max(kmax, k); }
        }
        kmin = wave_min_u(kmin);
        kmax = wave_max_u(kmax);
        if (lane == 0) { wred_u[wave] = kmin; wred_k[wave] = kmax; }
        lds_barrier();
        kmin = waves_min_u<MG_WAVES>(wred_u, lane);
        kmax = waves_max_u<MG_WAVES>(wred_k, lane);
        // number of candidates with key >= x (x > 0), identical in every thread
        auto count_ge = [&](uint32_t x) -> int {
          int c = 0;
#pragma unroll
          for (int r = 0; r < MG_REGK; ++r)
            if (r < per) c += __popcll(__builtin_amdgcn_ballot_w64(kreg[r] >= x));
          for (int r = MG_REGK; r < rounds; ++r) c += __popcll(__builtin_amdgcn_ballot_w64(key_of(r) >= x));
          lds_barrier();
          if (lane == 0) wred_i[wave] = c;
          lds_barrier();
          int before, t;
          waves_prefix_i<MG_WAVES>(wred_i, lane, 0, &before, &t);
          return t;
        };
        uint32_t lo_k = kmin, hi_k = kmax;  // invariant: count_ge(lo_k) >= K
        while (lo_k < hi_k) {
          const uint32_t mid = lo_k + (hi_k - lo_k + 1u) / 2u;
          if (count_ge(mid) >= K) lo_k = mid;
          else hi_k = mid - 1u;
        }
        tau = lo_k;
        quota = K - ((tau == 0xffffffffu) ? 0 : count_ge(tau + 1u));
      }
      // ordered compaction: winners (key above tau) and ties of every wavefront, then its own, register by register
      // (unused slots have key 0: never above, and equal to tau only where every candidate wins, with a quota of none)
      if (!take_all) tau = max(tau, 1u);
      auto is_above = [&](uint32_t key) { return key > tau; };
      auto is_tie = [&](uint32_t key) { return key == tau; };
      int na = 0, nt = 0;
#pragma unroll
      for (int r = 0; r < MG_REGK; ++r) {
        na += __popcll(__builtin_amdgcn_ballot_w64(is_above(kreg[r])));
        nt += __popcll(__builtin_amdgcn_ballot_w64(is_tie(kreg[r])));
        asm volatile("" : "+s"(na), "+s"(nt));  // (counted at once: all masks together do not fit the scalar registers)
      }
      // (a bound the compiler takes for a new one: it would otherwise carry the lane masks of all these comparisons across the
      // barrier, four scalar registers per candidate register)
      asm volatile("" : "+v"(tau));
      lds_barrier();  // (wred_i has been read)
      if (lane == 0) {
        wred_i[wave] = na;
        wred_j[wave] = nt;
      }
      lds_barrier();
      int base_above, base_tie, all_above, all_tie;
      waves_prefix_i<MG_WAVES>(wred_i, lane, wave, &base_above, &all_above);
      waves_prefix_i<MG_WAVES>(wred_j, lane, wave, &base_tie, &all_tie);
      auto store = [&](uint32_t key, int pa, int pt, auto position) {  // pa, pt: winners above and ties before this one
        if (is_above(key) || (is_tie(key) && pt < quota)) {
          const int at = pa + min(pt, quota);
          if (at < K) {
            win_key[at] = key;
            win_idx[at] = position();
          }
        }
      };
#pragma unroll
      for (int g = 0; g < NGRP; ++g)
        if (4 * g < per) {
          int c = 0;  // low half: winners above, high half: ties (at most 256 of a wavefront's group)
#pragma unroll
          for (int r = 4 * g; r < 4 * g + 4; ++r) c += (is_above(kreg[r]) ? 1 : 0) + (is_tie(kreg[r]) ? 0x10000 : 0);
          const int incl = wave_incl_scan_i(c), last = __builtin_amdgcn_readlane(incl, 63);
          int pa = base_above + ((incl - c) & 0xffff), pt = base_tie + ((incl - c) >> 16);
#pragma unroll
          for (int r = 4 * g; r < 4 * g + 4; ++r) {
            store(kreg[r], pa, pt, [&]() { return LAZY ? f_of(r) : ireg[LAZY ? 0 : r]; });
            pa += is_above(kreg[r]) ? 1 : 0;
            pt += is_tie(kreg[r]) ? 1 : 0;
          }
          base_above += last & 0xffff;
          base_tie += last >> 16;
        }
      for (int r = MG_REGK; r < rounds; ++r) {  // candidates beyond the register-resident ones, one round at a time
        const int f = r * MG_THREADS + tid;
        const uint32_t key = key_of(r);
        const unsigned long long ma = __builtin_amdgcn_ballot_w64(is_above(key)), mt = __builtin_amdgcn_ballot_w64(is_tie(key));
        lds_barrier();
        if (lane == 0) {
          wred_i[wave] = __popcll(ma);
          wred_j[wave] = __popcll(mt);
        }
        lds_barrier();
        int ba, bt_, ra, rt;
        waves_prefix_i<MG_WAVES>(wred_i, lane, wave, &ba, &ra);
        waves_prefix_i<MG_WAVES>(wred_j, lane, wave, &bt_, &rt);
        const int pa = all_above + ba + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(ma >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)ma, 0u));
        const int pt = all_tie + bt_ + (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mt >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mt, 0u));
        store(key, pa, pt, [&]() { return LAZY ? f : ci[f]; });
        all_above += ra;
        all_tie += rt;
      }
      n_out = min(K, all_above + min(all_tie, quota));
      if (PARTIAL && !take_all) edge = key_to_score(tau);
    }
  } else {
    // the winners are given (ascending positions, -1 padded, possibly none at all): their keys come from the
    // caller's score tensor
    n_out = p.topk_idx ? K : 0;
    for (int r = tid; r < n_out; r += MG_THREADS) {
      const int64_t pos = p.topk_idx[bh * (size_t)K + r];
      const bool ok = pos >= 0 && pos < S;
      win_idx[r] = ok ? (int)pos : -1;
      win_key[r] = ok ? score_key(p.scores_in[bh * (size_t)p.max_S + pos]) : 0u;
    }
  }
  if (mclk && tid == 0) mclk[2] = JF_CLK();
  lds_barrier();
  if (mclk && tid == 0) mclk[3] = JF_CLK();
  constexpr bool BATCHED = LAZY && HAS_LISTS && WIDE, LOOK_UP = LAZY && HAS_LISTS && !WIDE;
  if constexpr (BATCHED) {
    // the winners' positions, every thread those of the winners it goes on with, four requests in flight (one after the
    // other, in the loops below, 8192 winners' slots and weights took 11.4 k cycles instead of 6.5 k; up to 2048 winners, two
    // per thread, are quicker looked up there)
    constexpr int PB = 4;
    for (int r = tid; r < n_out; r += PB * MG_THREADS) {
      int pos[PB];
#pragma unroll
      for (int u = 0; u < PB; ++u) pos[u] = buffer_i32(ri, win_idx[(r + u * MG_THREADS < n_out) ? r + u * MG_THREADS : r] * 4, 0);
#pragma unroll
      for (int u = 0; u < PB; ++u)
        if (r + u * MG_THREADS < n_out) win_idx[r + u * MG_THREADS] = pos[u];
    }
  }
  if (PARTIAL) {  // the winners become one candidate list of the final merge
    const size_t at = (bh * p.mg_parts + part) * (size_t)K;
    for (int r = tid; r < K; r += MG_THREADS) {
      p.out_key[at + r] = (r < n_out) ? win_key[r] : 0u;  // unused slots: key 0
      if (r < n_out) p.out_idx[at + r] = LOOK_UP ? ci[win_idx[r]] : win_idx[r];
    }
    if (tid == 0) p.out_edge[bh * p.mg_parts + part] = edge;
    return;
  }

  float inv_z = (lsum > 0.f) ? 1.0f / lsum : 0.f;
  if (!PARTIAL && tid == 0 && p.softmax_m) {
    p.softmax_m[bh] = M;
    p.softmax_inv_z[bh] = inv_z;
  }
  if constexpr (MODE == FS_STAGE_B) {
    if (p.stats_m) {  // (uniform) the caller's statistics
      M = p.stats_m[bh];
      inv_z = p.stats_iz[bh];
    }
  }
  // one thread per winner: position, paged slot, softmax weight
  int64_t* out_idx = p.topk_idx + bh * (size_t)K;
  int64_t* out_slot = p.topk_slots + bh * (size_t)K;
  for (int r = tid; r < K; r += MG_THREADS) {
    int64_t position = -1, slot = -1;
    int wslot = -1;
    float ww = 0.f;
    if (r < n_out && win_idx[r] >= 0) {
      position = LOOK_UP ? ci[win_idx[r]] : win_idx[r];
      const int blk = (int)(position / BS);
      if (blk < p.max_blocks) slot = (int64_t)((blk < nblk_lds) ? (int64_t)bt_sh[blk] : bt[blk]) * BS + (position % BS);
      wslot = (slot >= 0 && slot < p.num_slots) ? (int)slot : -1;
      ww = __expf(key_to_score(win_key[r]) - M) * inv_z;
    }
    if constexpr (MODE != FS_STAGE_B) {
      out_idx[r] = position;
      out_slot[r] = slot;
    }
    win_idx[r] = wslot;
    win_key[r] = __builtin_bit_cast(uint32_t, ww);
  }
  if constexpr (MODE == FS_STAGE_A) return;  // Stage A alone ends with the winners and the statistics
  if constexpr (!PARTIAL && MODE != FS_STAGE_A) {  // o_hat, by the last two wavefronts while the first ones look after the winners
    const int d = tid - (MG_THREADS - D);
    if (d >= 0) {
      float o8[VGRP];
#pragma unroll
      for (int q = 0; q < VGRP; ++q) o8[q] = red_sh[q][d];
#pragma unroll
      for (int n = VGRP / 2; n >= 1; n /= 2) {  // fixed order
#pragma unroll
        for (int q = 0; q < n; ++q) o8[q] += o8[q + n];
      }
      const float o2 = has_parts ? o8[0] * inv_z : o8[0];
      p.o_hat[bh * D + d] = o2;
      ohat_sh[d] = o2;
    }
  }
  lds_barrier();
  if (mclk && tid == 0) mclk[4] = JF_CLK();

  // ---- pre-correction over the winners, 64 at a time on the matrix cores, in eight groups whatever MG_THREADS is (four
  // wavefronts: two groups each, added as the first step of the sum over eight would).  What a conversion and a multiply-add per
  // code in all wavefronts took instead, per layer: 32 sequences x 3000 positions, K4V4, top-k 2048 100.5 us, this 95.0; 32 x 3000,
  // K3V2, 1024 66.4 / 64.1; 24 x 2500, eight heads, K3V2, 512 72.7 / 69.7; 32 x 6000, K3V2, 256 58.8 / 56.8; 12 x 8192, K4V4, 64
  // 33.4 / 31.6; 16 of 983 .. 16384, K4V4, 256 60.2 / 59.1; 4 x 32768, K3V2, 256 34.4 / 34.2.
  if constexpr (HAS_SUMS) {
    const uint8_t* vbase = p.v_data + (size_t)hkv * p.num_slots * Sums::Tiles::VP;
    const uint8_t* vsbase = reinterpret_cast<const uint8_t*>(p.v_scales + (size_t)hkv * p.num_slots * NG);
    if (wave < SUM_WAVES) {
      uint8_t* st = pool + wave * Sums::STAGE;
      auto fetch = [&](int first) JF_INLINE { return Sums::fetch(vbase, vsbase, win_idx, reinterpret_cast<const float*>(win_key), first, n_out, lane); };
      float sum[2] = {}, wsum = 0.f;
      if constexpr (AHEAD) {  // (at most 512 winners: two turns of 64)
        static_assert(VGRP == 2 * SUM_WAVES && MG_WIN <= VGRP * 64, "a turn for each of two groups");
        const int second = (wave + SUM_WAVES) * 64;
        if (wave * 64 < n_out) {
          const typename Sums::Rows x = fetch(wave * 64), y = fetch(min(second, n_out - 1));
          __builtin_amdgcn_sched_barrier(0);
          Sums::add(x, st, lane, sum);
          wsum = wave_sum(x.w);
          if (second < n_out) {  // (uniform)
            float o[2] = {};
            Sums::add(y, st + (AREAS - 1) * SUM_WAVES * Sums::STAGE, lane, o);
            sum[0] += o[0];
            sum[1] += o[1];
            wsum += wave_sum(y.w);
          }
        }
      } else {
#pragma unroll 1
        for (int vg = wave; vg < VGRP; vg += SUM_WAVES) {
          float o[2] = {}, ws = 0.f;
#pragma unroll 1
          for (int first = vg * 64; first < n_out; first += VGRP * 64) {
            const typename Sums::Rows x = fetch(first);
            ws += x.w;
            Sums::add(x, st, lane, o);
          }
          sum[0] += o[0];
          sum[1] += o[1];
          wsum += wave_sum(ws);
        }
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) sum_sh[wave][Sums::channel(lane, i)] = sum[i];
      if (lane == 0) w_sh[wave] = wsum;
    }
    lds_barrier();
    if (tid < D) {
      float o8[SUM_WAVES], w8[SUM_WAVES];
#pragma unroll
      for (int q = 0; q < SUM_WAVES; ++q) {
        o8[q] = sum_sh[q][tid];
        w8[q] = w_sh[q];
      }
#pragma unroll
      for (int n = SUM_WAVES / 2; n >= 1; n /= 2) {  // fixed order
#pragma unroll
        for (int q = 0; q < n; ++q) {
          o8[q] += o8[q + n];
          w8[q] += w8[q + n];
        }
      }
      const float o = o8[0], wt = w8[0];  // (the same wt in every thread)
      p.o_old[bh * D + tid] = o;
      if (tid == 0) p.W[bh] = wt;
      // the blend of jetfire_vllm/csrc/blend.cu:202-226 for callers that hold o_new already
      if (MODE == FS_FULL && p.blend_out) p.blend_out[bh * D + tid] = f32_to_bf16(__builtin_fmaf(wt, bf16_to_f32(blend_raw), ohat_sh[tid]) - o);
    }
  }
  if (mclk && tid == 0) mclk[5] = JF_CLK();
}

constexpr size_t LDS_BUDGET_2WG = 80 * 1024 - 512;    // two workgroups per CU (160 KB LDS)
constexpr size_t LDS_BUDGET_1WG = 160 * 1024 - 1024;

// LDS a scan workgroup has left for what grows with the split: the scores, the page table (and, with one split, ScanTail)
template <int SCHEME, int G, int NG>
long lds_room_for() {
  using Lds = ScanLds<SCHEME, G, NG>;
  const size_t budget = (G <= 4 && Lds::NW == 8) ? LDS_BUDGET_2WG : LDS_BUDGET_1WG;
  const size_t fixed = Lds::AUX + Lds::stage_bytes() + 64 + 832 + (Lds::K3 ? 512 : 0);  // + static LDS of the kernel (INT3: incl. the rounding table)
  return (long)budget - (long)fixed;
}

inline long lds_room(int scheme, int G, int NG) {
#define JF_ROOM_CASE(SCH, GG, NGG) if (scheme == SCH && G == GG && NG == NGG) return lds_room_for<SCH, GG, NGG>()
  JF_ROOM_CASE(JF_SCHEME_K3V2, 1, 1); JF_ROOM_CASE(JF_SCHEME_K3V2, 2, 1); JF_ROOM_CASE(JF_SCHEME_K3V2, 4, 1);
  JF_ROOM_CASE(JF_SCHEME_K3V2, 8, 1); JF_ROOM_CASE(JF_SCHEME_K3V2, 16, 1);
  JF_ROOM_CASE(JF_SCHEME_K3V2, 1, 2); JF_ROOM_CASE(JF_SCHEME_K3V2, 2, 2); JF_ROOM_CASE(JF_SCHEME_K3V2, 4, 2);
  JF_ROOM_CASE(JF_SCHEME_K3V2, 8, 2); JF_ROOM_CASE(JF_SCHEME_K3V2, 16, 2);
  JF_ROOM_CASE(JF_SCHEME_K4V4, 1, 1); JF_ROOM_CASE(JF_SCHEME_K4V4, 2, 1); JF_ROOM_CASE(JF_SCHEME_K4V4, 4, 1);
  JF_ROOM_CASE(JF_SCHEME_K4V4, 8, 1); JF_ROOM_CASE(JF_SCHEME_K4V4, 16, 1);
  JF_ROOM_CASE(JF_SCHEME_K3V4, 1, 1); JF_ROOM_CASE(JF_SCHEME_K3V4, 2, 1); JF_ROOM_CASE(JF_SCHEME_K3V4, 4, 1);
  JF_ROOM_CASE(JF_SCHEME_K3V4, 8, 1); JF_ROOM_CASE(JF_SCHEME_K3V4, 16, 1);
  JF_ROOM_CASE(JF_SCHEME_K4V2, 1, 1); JF_ROOM_CASE(JF_SCHEME_K4V2, 2, 1); JF_ROOM_CASE(JF_SCHEME_K4V2, 4, 1);
  JF_ROOM_CASE(JF_SCHEME_K4V2, 8, 1); JF_ROOM_CASE(JF_SCHEME_K4V2, 16, 1);
  JF_ROOM_CASE(JF_SCHEME_K2V2, 1, 1); JF_ROOM_CASE(JF_SCHEME_K2V2, 2, 1); JF_ROOM_CASE(JF_SCHEME_K2V2, 4, 1);
  JF_ROOM_CASE(JF_SCHEME_K2V2, 8, 1); JF_ROOM_CASE(JF_SCHEME_K2V2, 16, 1);
  JF_ROOM_CASE(JF_SCHEME_K2V2, 1, 2); JF_ROOM_CASE(JF_SCHEME_K2V2, 2, 2); JF_ROOM_CASE(JF_SCHEME_K2V2, 4, 2);
  JF_ROOM_CASE(JF_SCHEME_K2V2, 8, 2); JF_ROOM_CASE(JF_SCHEME_K2V2, 16, 2);
  JF_ROOM_CASE(JF_SCHEME_K2V4, 1, 1); JF_ROOM_CASE(JF_SCHEME_K2V4, 2, 1); JF_ROOM_CASE(JF_SCHEME_K2V4, 4, 1);
  JF_ROOM_CASE(JF_SCHEME_K2V4, 8, 1); JF_ROOM_CASE(JF_SCHEME_K2V4, 16, 1);
#define JF_ROOM_ALL_G(SCH, NGG)                                                                      \
  JF_ROOM_CASE(SCH, 1, NGG); JF_ROOM_CASE(SCH, 2, NGG); JF_ROOM_CASE(SCH, 4, NGG); JF_ROOM_CASE(SCH, 8, NGG); \
  JF_ROOM_CASE(SCH, 16, NGG)
  JF_ROOM_ALL_G(JF_SCHEME_K2V3, 1); JF_ROOM_ALL_G(JF_SCHEME_K2V3, 2);
  JF_ROOM_ALL_G(JF_SCHEME_K3V3, 1); JF_ROOM_ALL_G(JF_SCHEME_K3V3, 2);
  JF_ROOM_ALL_G(JF_SCHEME_K4V3, 1);
  JF_ROOM_ALL_G(JF_SCHEME_A2V2, 1); JF_ROOM_ALL_G(JF_SCHEME_A2V2, 2);
  JF_ROOM_ALL_G(JF_SCHEME_A2V3, 1); JF_ROOM_ALL_G(JF_SCHEME_A2V3, 2);
  JF_ROOM_ALL_G(JF_SCHEME_A2V4, 1);
  JF_ROOM_ALL_G(JF_SCHEME_K3V4, 2); JF_ROOM_ALL_G(JF_SCHEME_K2V4, 2); JF_ROOM_ALL_G(JF_SCHEME_A2V4, 2);
  JF_ROOM_ALL_G(JF_SCHEME_B4V2, 1); JF_ROOM_ALL_G(JF_SCHEME_B4V2, 2); JF_ROOM_ALL_G(JF_SCHEME_B4V3, 1);
  JF_ROOM_ALL_G(JF_SCHEME_B4V3, 2); JF_ROOM_ALL_G(JF_SCHEME_B4V4, 1); JF_ROOM_ALL_G(JF_SCHEME_B4V4, 2);
#undef JF_ROOM_ALL_G
#undef JF_ROOM_CASE
  return 0;
}

// Longest split: what fits LDS (scores and one page-table entry per 16 positions), at most four chunks per wavefront.
inline int split_len_max(int scheme, int G, int NG) {
  long lm = lds_room(scheme, G, NG) / (4 * G + 1) / 256 * 256;
  const long cap = (G <= 4 ? 16 : 8) * 256;
  if (lm > cap) lm = cap;
  return lm < 256 ? 256 : (int)lm;
}

inline size_t scan_tail_bytes(int G, int top_k, int kc) {
  return G == 1 ? ScanTail<1, 4>::bytes(top_k, kc) : G == 2 ? ScanTail<2, 4>::bytes(top_k, kc) :
         G == 4 ? ScanTail<4, 4>::bytes(top_k, kc) : G == 8 ? ScanTail<8, 1>::bytes(top_k, kc) :
                  ScanTail<16, 1>::bytes(top_k, kc);
}

// Whether a scan whose single split of L positions covers the sequence can merge by itself: its tables fit the LDS
// that is left, and so does the list of winners (kc counts their most and more).
inline bool one_split_fits(int scheme, int G, int NG, int L, int top_k, int kc) {
  return (long)((4 * G + 1) * (long)L + (long)scan_tail_bytes(G, top_k, kc)) <= lds_room(scheme, G, NG);
}

// Estimated microseconds of the merge (fitted on MI355X): a fixed part per launch plus a part proportional to
// the candidates one workgroup visits.
constexpr double kMergeFixed = 8.5, kPartialFixed = 7.5, kPerCand = 0.0004, kPerCandBig = 0.001;
constexpr int MG_REG_CANDS = 8192;  // candidates the common merge shape keeps in registers
inline double merge_pass_us(double fixed, long cands) {
  return cands <= MG_REG_CANDS ? fixed + kPerCand * (double)cands : fixed + 1.5 + kPerCandBig * (double)cands;
}
// One stage of the shape that keeps 32 candidates per thread, against two stages at the same split length, 36 shapes of 9472 to
// 30720 candidates, 16 to 256 rows, per layer: up to 16384 candidates 1.5 - 9 us shorter, around 22000 as long, 2.4 us longer at
// 30720 (rows 16; with 64 rows and more it is the shorter way throughout, which the estimate, by the candidates alone, leaves
// out).  3 x 28076 positions, 8 kv-heads, G = 4, K3V2, top-k
// 1024 (12800 candidates, 96 rows) 47.9 -> 42.4 us; 2 x 61876, K4V4, top-k 512 (12288, 64) 45.1 -> 42.6; 1 x 131072, K4V4, top-k
// 512 (24576, 32) stays at two, 46.1 against 47.2.
constexpr double kOneStageFixed = 11.6, kOneStagePerCand = 0.00032;
inline double merge_one_stage_us(long cands) {
  return cands > MG_REG_CANDS && cands <= 4 * MG_REG_CANDS ? kOneStageFixed + kOneStagePerCand * (double)cands
                                                           : merge_pass_us(kMergeFixed, cands);
}

// Two-stage merge when one workgroup per row would face more than MG_REG_CANDS candidates: the number of
// parts (at most MG_REG_CANDS / top_k, so that the final merge keeps its candidates in registers, and at least
// two lists per part) with the smallest estimated time, which is returned.  parts == 1: single stage.
inline double merge_plan(int rows, int ns, int kc, int top_k, int* parts_out, int* spp_out) {
  *parts_out = 1;
  *spp_out = ns;
  double best = merge_one_stage_us((long)ns * kc);
  if ((long long)ns * kc <= MG_REG_CANDS || ns < 4) return best;
  // (wide corrections run the 32-register shape throughout: its 32768 candidates bound the final merge)
  int cap = (top_k > FS_LDS_TOPK ? 4 * MG_REG_CANDS : MG_REG_CANDS) / top_k;
  if (cap > ns / 2) cap = ns / 2;
  for (int parts = 2; parts <= cap; ++parts) {
    const int spp = (ns + parts - 1) / parts;
    if ((ns + spp - 1) / spp != parts) continue;  // the same spp as a smaller number of parts
    const long wgs = (long)(rows > 0 ? rows : 1) * parts;
    const double rounds = (double)((wgs + 511) / 512);  // two workgroups per CU
    const double us = kPartialFixed + rounds * (merge_pass_us(kPartialFixed, (long)spp * kc) - kPartialFixed) +
                      merge_pass_us(kMergeFixed, (long)parts * top_k);
    if (us < best) {
      best = us;
      *parts_out = parts;
      *spp_out = spp;
    }
  }
  return best;
}

// Estimated microseconds of the merge launches: the above, the slots and pre-correction of the winners, and what a launch
// of more rows than CUs takes (16 us at 512 rows, 18 at 1024).
inline double merge_us(int rows, int max_S, int ns, int kc, int top_k) {
  constexpr double kManyRows = 5.0, kPerRowBeyond = 0.005;
  const int winners = top_k < max_S ? top_k : max_S, cus = device_cus();
  int parts, spp;
  double us = merge_plan(rows, ns, kc, top_k, &parts, &spp);
  if (winners > 256) us += 1.5 * ((double)winners / 256.0 - 1.0);
  if (rows > cus) us += kManyRows + kPerRowBeyond * (double)(rows - cus);
  return us;
}

// Estimated microseconds by which a scan workgroup gets longer when it merges by itself.  The sums over the winners'
// value rows bound it: a wavefront takes 64 rows of one head at a time, the heads of the kv-head share the workgroup's
// wavefronts (more heads than wavefronts: one after the other), and all wavefronts of a SIMD share its vector ALU.
// Measured against the merge launch at the same split length, up to 256 rows: 64-row batches per wavefront 1 / 2 / 4 with
// sixteen wavefronts 3 us faster / equal / 4 us slower, 1 / 2 / 4 / 8 with eight wavefronts 4 and 2 us faster, 2 and up to 10
// slower; with more rows the launch takes longer and the workgroups here do not.  (Both ways' sums have moved to the matrix cores
// since; over 450 random shapes, each timed in every split length from a graph, the planner's choice is 2.0 % off the best one's time
// in the mean.)
inline double one_split_us(int G, int units, int max_S, int top_k) {
  constexpr double kFixed = 1.4, kPerBatch = 0.25;
  const int nw = G <= 4 ? 16 : 8, per_head = nw >= G ? nw / G : 1, winners = top_k < max_S ? top_k : max_S;
  const int batches = (winners + 64 * per_head - 1) / (64 * per_head) * ((G + nw - 1) / nw), cus = device_cus();
  return (kFixed + kPerBatch * nw * batches) * (double)((units + cus - 1) / cus);
}

// Whether a scan of one split merges by itself: it can (one_split_fits), and that is estimated to be the shorter way
// (selection alone always is: 64 heads over 4 kv-heads, 190 positions, top-k 128 17.4 us, with the launch 20.8).  The same
// for the whole step and Stage B alone, whose sums over the winners are then the same numbers.
inline bool one_split_merges(int mode, int scheme, int G, int NG, int B, int H_q, int H_kv, int max_S, int L, int top_k,
                             int kc) {
  return one_split_fits(scheme, G, NG, L, top_k, kc) &&
         (mode == FS_STAGE_A || mode == FS_TOPK ||
          one_split_us(G, B * H_kv, max_S, top_k) <= merge_us(B * H_q, max_S, 1, kc, top_k));
}

inline int padded_group(int g) { return g <= 2 ? g : (g <= 4 ? 4 : (g <= 8 ? 8 : 16)); }

// (One plan for the whole step and for either stage alone, so that their sums over the splits are the same numbers.)
inline void fused_plan(int scheme, int NG, int B, int H_q, int H_kv, int max_S, int top_k, int* L_out, int* ns_out,
                       int* kc_out) {
  const int G = padded_group(H_q / H_kv);
  const int units = B * H_kv > 0 ? B * H_kv : 1;
  const int rows = B * H_q > 0 ? B * H_q : 1;
  // One scan workgroup is resident per CU (256 CUs).  Among the split lengths that fit LDS pick the one with
  // the smallest estimated time of scan + merge.  The constants are microseconds fitted to measurements on
  // MI355X: a scan workgroup costs a fixed part plus a part proportional to the 64-position chunks each of
  // its wavefronts works through; a last, partly filled round of workgroups runs faster than a full one; the
  // merge costs a fixed part per launch plus a part proportional to the candidates one workgroup visits.
  const int lmax = split_len_max(scheme, G, NG);
  const int nw = (G <= 4) ? 16 : 8;
  const int kCUs = device_cus();
  constexpr double kScanFixed = 8.5;
  // one chunk per wavefront, all wavefronts; the mixed schemes are priced like the wider one
  const double per_chunk = (scheme == JF_SCHEME_K3V2 || scheme == JF_SCHEME_K2V2) ? 5.9 : 6.6;  // (INT3 values, asymmetric keys: as INT4)
  // What one chunk per wavefront costs in an almost empty round, against a full one.  One split for the whole sequence
  // means few workgroups with several chunks each, and the INT4 keys of the bf16 model then take 4.7 - 5.5 us a chunk
  // where the others take 1.5 - 3: 3 sequences x 8 kv-heads, 1679 positions, G = 4, top-k 32 in one split 26.6 us, in
  // splits of 256 22.3.  (Between several split lengths the higher figure changed no choice for the better.)
  // Asymmetric keys with two scale groups (three contractions per group) lie between: 4 sequences x 4 kv-heads, 1181
  // positions, A2V2, G = 2, top-k 1024 in one split 28.9 us, in splits of 256 25.5; 4 x 1, 1262 positions, A2V4 24.4 / 22.6.
  // (With one group, or at 0.8, as many shapes lost as gained.)
  const double lone_split = scheme / 10 == 5 ? 0.8 : (scheme / 10 == 1 && NG == 2) ? 0.65 : 0.5;
  // These keys, more than 256 winners, a sequence that two splits in the short form hold: one split for all of it takes that
  // much longer against those than the figures say.  28 sequences x 4 kv-heads, 1361 positions, G = 4, B4V4 in 64-channel
  // groups, top-k 512 in one split 32.2 us, in two of 768 30.0 (256 winners 26.9 / 26.5, 64 22.8 / 24.9).  Of 1600 random
  // shapes 21 are cut otherwise, 20 of them for the better, by up to 20 %, one 1.3 % slower; charged whatever the number of
  // winners a dozen lose 8 to 22 %.
  const double lone_wide = (scheme / 10 == 5 && top_k > 256 && max_S <= 2 * 64 * nw) ? 3.5 : 0.0;
  int L = 256;
  double best = -1.0;
  for (int cand = 256; cand <= lmax; cand += 256) {
    const long nsp = (max_S + cand - 1) / cand > 0 ? (max_S + cand - 1) / cand : 1;
    if (nsp > MG_MAX_SPLITS && cand < lmax) continue;
    const long nwg = nsp * units;
    const long full = nwg / kCUs, rem = nwg % kCUs;
    const double stream = per_chunk * (double)cand / (64.0 * nw);
    double cost = (double)full * (kScanFixed + stream);
    const double lone = nsp == 1 ? lone_split : 0.5;
    if (rem > 0) cost += kScanFixed + stream * (lone + (1.0 - lone) * (double)rem / kCUs);
    const int kc = (top_k + FS_CAND_SLACK) < cand ? (top_k + FS_CAND_SLACK) : cand;
    if (nsp == 1 && one_split_merges(FS_FULL, scheme, G, NG, B, H_q, H_kv, max_S, cand, top_k, kc))
      cost += one_split_us(G, units, max_S, top_k) + (cand > 64 * nw ? lone_wide : 0.0);
    else
      cost += merge_us(rows, max_S, (int)nsp, kc, top_k);
    if (best < 0.0 || cost <= best) {
      best = cost;
      L = cand;
    }
    if (cand >= max_S) break;
  }
#ifdef JF_DEBUG_HOOKS
  if (const int forced = g_force_split_len.load(std::memory_order_relaxed); forced > 0) {
    L = (forced + 255) / 256 * 256;
    if (L > lmax) L = lmax;
    while ((max_S + L - 1) / L > MG_MAX_SPLITS && L < lmax) L += 256;
  }
#endif
  int ns = (max_S + L - 1) / L;
  if (ns < 1) ns = 1;
  *L_out = L;
  *ns_out = ns;
  const int cap = top_k + FS_CAND_SLACK;  // the split may emit a superset of its top-k (see phase C)
  *kc_out = cap < L ? cap : L;
}

struct WsLayout {
  size_t off_m, off_l, off_o, off_key, off_idx, off_edge, off_key2, off_idx2, off_edge2, total;
};
inline WsLayout ws_layout(int B, int H_q, int ns, int kc, int parts, int top_k) {
  WsLayout w;
  const size_t rows = (size_t)B * H_q;
  size_t o = 0;
  auto take = [&](size_t bytes) { size_t r = o; o += (bytes + 255) / 256 * 256; return r; };
  w.off_m = take(rows * ns * 4);
  w.off_l = take(rows * ns * 4);
  w.off_o = take(rows * ns * D * 4);
  w.off_key = take(rows * ns * kc * 4);
  w.off_idx = take(rows * ns * kc * 4);
  w.off_edge = take(rows * ns * 4);
  w.off_key2 = w.off_idx2 = w.off_edge2 = 0;
  if (parts > 1) {
    w.off_key2 = take(rows * parts * top_k * 4);
    w.off_idx2 = take(rows * parts * top_k * 4);
    w.off_edge2 = take(rows * parts * 4);
  }
  w.total = o + 256;
  return w;
}

template <int MODE, int SCHEME, int G, int NG, bool SHORT = false>
int launch_scan(const FusedParams& p, hipStream_t st) {
  using Lds = ScanLds<SCHEME, G, NG>;
  const bool one = p.one_split != 0;
  const size_t smem = Lds::total(p.L) + (one ? ScanTail<G, Lds::SEG>::bytes(p.top_k, p.Kc) : 0);
  auto kern = one ? fused_scan_kernel<MODE, SCHEME, G, NG, true, SHORT> : fused_scan_kernel<MODE, SCHEME, G, NG, false, SHORT>;
  // per instantiation: raise the dynamic-LDS limit only when it grows (launches may come from several threads)
  static std::mutex attr_mu;
  static size_t attr_smem[2] = {0, 0};
  {
    std::lock_guard<std::mutex> lock(attr_mu);
    if (smem > attr_smem[one]) {
      JF_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
      attr_smem[one] = smem;
    }
  }
#ifdef JF_DEBUG_HOOKS
  std::unique_lock<std::mutex> plock(g_prof_mu, std::defer_lock);
  bool prof = false;
  if (g_prof.armed) {  // (read without the lock: arming happens-before the launches a benchmark times)
    plock.lock();
    prof = g_prof.armed && g_prof.used + 2 <= (int)g_prof.ev.size();
    if (!prof) plock.unlock();
  }
  if (prof) JF_CHECK_HIP(hipEventRecord(g_prof.ev[g_prof.used], st));
#endif
  hipLaunchKernelGGL(kern, dim3(p.H_kv, p.n_splits, p.B), dim3(ScanLds<SCHEME, G, NG>::NT), smem, st, p);
  JF_CHECK_LAUNCH();
#ifdef JF_DEBUG_HOOKS
  if (prof) {
    JF_CHECK_HIP(hipEventRecord(g_prof.ev[g_prof.used + 1], st));
    g_prof.used += 2;
  }
#endif
  return JF_OK;
}

// One scheme of the one-pass form: the GQA group picks the instantiation (of this translation unit's form).
template <int SCHEME, int NG>
int launch_full_by_group(int G, const void* params, void* stream) {
  const FusedParams& p = *static_cast<const FusedParams*>(params);
  hipStream_t st = (hipStream_t)stream;
  switch (G) {
    case 1: return launch_scan<FS_FULL, SCHEME, 1, NG, kShortForm>(p, st);
    case 2: return launch_scan<FS_FULL, SCHEME, 2, NG, kShortForm>(p, st);
    case 4: return launch_scan<FS_FULL, SCHEME, 4, NG, kShortForm>(p, st);
    case 8: return launch_scan<FS_FULL, SCHEME, 8, NG, kShortForm>(p, st);
    default: return launch_scan<FS_FULL, SCHEME, 16, NG, kShortForm>(p, st);
  }
}

inline bool scheme_has_zp(int scheme) {  // asymmetric INT2 keys
  return scheme == JF_SCHEME_A2V2 || scheme == JF_SCHEME_A2V3 || scheme == JF_SCHEME_A2V4;
}
inline bool known_scheme(int scheme) {
  return scheme == JF_SCHEME_K3V2 || scheme == JF_SCHEME_K4V4 || scheme == JF_SCHEME_K3V4 || scheme == JF_SCHEME_K4V2 ||
         scheme == JF_SCHEME_K2V2 || scheme == JF_SCHEME_K2V4 || scheme == JF_SCHEME_K2V3 || scheme == JF_SCHEME_K3V3 ||
         scheme == JF_SCHEME_K4V3 || scheme_has_zp(scheme) || scheme == JF_SCHEME_B4V2 || scheme == JF_SCHEME_B4V3 ||
         scheme == JF_SCHEME_B4V4;
}
// scale groups per row: every scheme but those with INT4 keys (int8-Q model: one key scale per row) may use
// 64-channel groups
inline bool scheme_any_group(int scheme) { return known_scheme(scheme) && scheme / 10 != 4; }
inline int scheme_ng(int scheme, int group_size) { return scheme_any_group(scheme) ? D / group_size : 1; }


// A merge kernel whose winners live in dynamic LDS (corrections wider than FS_LDS_TOPK): 8 bytes per winner; the
// dynamic-LDS limit of the instantiation is raised once.
template <void (*KERN)(MergeParams)>
int launch_wide_merge(dim3 grid, const MergeParams& p, hipStream_t st) {
  static std::mutex mu;
  static bool raised = false;
  {
    std::lock_guard<std::mutex> lock(mu);
    if (!raised) {
      JF_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(KERN), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       FS_MAX_TOPK * 8));
      raised = true;
    }
  }
  hipLaunchKernelGGL(KERN, grid, dim3(1024), (size_t)p.top_k * 8, st, p);
  return JF_OK;
}

// The whole step on caller-provided workspace memory; every public entry point of the fused forms ends here.
// MODE FS_FULL: all arguments as in jf_fused_scan_topk.  FS_STAGE_A: the value side, o_hat, o_old_unnorm, W are
// unused; top_k == 0 asks for the scores alone (then nothing but `scores` is written and no workspace is needed).
// FS_STAGE_B: q and the key side are unused, `scores_in` and `topk_idx` are inputs (topk_idx may be NULL: o_hat only,
// zeros for the pre-correction terms), topk_slots is unused.
template <int MODE>
static int fused_run(int scheme, int group_size, const uint16_t* q, const uint8_t* k_data,
                     const uint16_t* k_scales, const uint16_t* k_zp, const uint8_t* v_data, const uint16_t* v_scales,
                     const int64_t* block_table, const int32_t* seq_lens, int B, int H_q, int H_kv,
                     int max_S, int max_blocks, int64_t num_slots, int block_size, float attn_scale,
                     int top_k, int64_t* topk_idx, int64_t* topk_slots, float* o_hat,
                     float* o_old_unnorm, float* W, float* softmax_m, float* softmax_inv_z, float* scores,
                     const float* scores_in, const uint16_t* blend_o_new, uint16_t* blend_out, void* workspace,
                     size_t workspace_bytes, void* stream) {
  JF_CHECK_ARG(known_scheme(scheme), "fused_scan: unknown scheme %d", scheme);
  JF_CHECK_ARG(MODE == FS_FULL || scheme == JF_SCHEME_K3V2 || scheme == JF_SCHEME_K4V4 ||
                   (MODE == FS_STAGE_A && (scheme == JF_SCHEME_K2V2 || scheme == JF_SCHEME_A2V2 || scheme == JF_SCHEME_B4V2)) ||
                   (MODE == FS_STAGE_B && (scheme == JF_SCHEME_K3V3 || scheme == JF_SCHEME_K3V4)),
               "fused_scan: the stage-wise forms take the K3V2 or K4V4 side formats (Stage A also K2V2 and A2V2, Stage B also K3V3)");
  JF_CHECK_ARG(!(MODE == FS_FULL || MODE == FS_STAGE_A) || scheme_has_zp(scheme) == (k_zp != nullptr) || B == 0,
               "fused_scan: zero-points go with the asymmetric INT2 key formats, and only with them");
  constexpr bool HAS_K = (MODE == FS_FULL || MODE == FS_STAGE_A), HAS_V = (MODE == FS_FULL || MODE == FS_STAGE_B);
  JF_CHECK_ARG(MODE != FS_TOPK || scheme == JF_SCHEME_K4V4, "fused_scan: the selection-only form uses the K4V4 layout");
  JF_CHECK_ARG((blend_o_new == nullptr) == (blend_out == nullptr), "fused_scan: o_new and out go together");
  JF_CHECK_ARG(B >= 0 && H_q > 0 && H_kv > 0 && max_S >= 0 && H_q % H_kv == 0, "fused_scan: bad shape");
  const int g_act = H_q / H_kv;
  JF_CHECK_ARG(g_act >= 1 && g_act <= 16, "fused_scan: GQA group %d not in 1..16", g_act);
  const int G = padded_group(g_act);  // the kernels come for 1, 2, 4, 8 and 16 query heads per kv-head
  JF_CHECK_ARG(block_size == 16, "fused_scan only supports block_size=16");
  JF_CHECK_ARG(group_size == 64 || group_size == 128, "fused_scan: group_size must be 64 or 128 (got %d)", group_size);
  JF_CHECK_ARG(scheme_any_group(scheme) || group_size == 128,
               "fused_scan: the INT4 sides (int8-Q keys, INT4 values) need group_size 128");
  const bool scores_only = (MODE == FS_STAGE_A) && top_k == 0;
  if (scores_only) top_k = 32;  // (any valid width: the plan depends on it, the kernel stops before using it)
  JF_CHECK_ARG(is_pow2(top_k) && top_k >= 32 && top_k <= FS_MAX_TOPK,
               "fused_scan: unsupported top_k=%d (supported: the powers of two from 32 to 8192)", top_k);
  JF_CHECK_ARG(max_S <= 262144, "fused_scan: max_S=%d exceeds supported limit (262144)", max_S);
  JF_CHECK_ARG((int64_t)max_blocks * block_size >= max_S, "fused_scan: block_table does not cover max_S");
  // (a row's byte offset inside one kv-head's tensor is formed in 32 bits: rows of at most 64 bytes)
  JF_CHECK_ARG(num_slots > 0 && num_slots <= FS_MAX_SLOTS, "fused_scan: num_slots out of range (at most 2^26: row offsets are 32-bit)");
  JF_CHECK_ARG((softmax_m == nullptr) == (softmax_inv_z == nullptr), "fused_scan: softmax_m and softmax_inv_z go together");
  if (B == 0) return JF_OK;
  JF_CHECK_ARG(block_table && seq_lens, "fused_scan: null input");
  if (HAS_K) {
    JF_CHECK_ARG(q && k_data && k_scales, "fused_scan: null input");
    JF_CHECK_ARG(((uintptr_t)k_data & 15) == 0 && ((uintptr_t)q & 15) == 0, "fused_scan: q and k_data must be 16-byte aligned");
    JF_CHECK_ARG(((uintptr_t)k_scales & 3) == 0 && ((uintptr_t)k_zp & 3) == 0, "fused_scan: k_scales and k_zp must be 4-byte aligned");
  }
  if (MODE != FS_STAGE_B) JF_CHECK_ARG(scores_only ? scores != nullptr : (topk_idx && topk_slots), "fused_scan: null output");
  if (HAS_V) {
    JF_CHECK_ARG(v_data && v_scales, "fused_scan: null input");
    JF_CHECK_ARG(((uintptr_t)v_data & 15) == 0 && ((uintptr_t)v_scales & 3) == 0,
                 "fused_scan: v_data must be 16-byte aligned, v_scales 4-byte aligned");
    JF_CHECK_ARG(o_hat && o_old_unnorm && W, "fused_scan: null output");
  }
  if (!HAS_K) JF_CHECK_ARG(scores_in != nullptr, "fused_scan: null scores");
  const int NGv = scheme_ng(scheme, group_size);
  FusedParams p;
  p.q = q; p.k_data = k_data; p.k_scales = k_scales; p.k_zp = k_zp; p.v_data = v_data; p.v_scales = v_scales;
  p.block_table = block_table; p.seq_lens = seq_lens;
  p.B = B; p.H_q = H_q; p.H_kv = H_kv; p.max_S = max_S; p.max_blocks = max_blocks; p.num_slots = num_slots;
  p.g_act = g_act;
  p.attn_scale = attn_scale; p.top_k = top_k;
  fused_plan(scheme, NGv, B, H_q, H_kv, max_S, top_k, &p.L, &p.n_splits, &p.Kc);
  JF_CHECK_ARG(p.n_splits <= MG_MAX_SPLITS, "fused_scan: too many splits (%d > %d)", p.n_splits, MG_MAX_SPLITS);
  merge_plan(B * H_q, p.n_splits, p.Kc, top_k, &p.mg_parts, &p.mg_spp);
  if (MODE == FS_STAGE_B) { p.mg_parts = 1; p.mg_spp = p.n_splits; }
  p.one_split = !scores_only && p.n_splits == 1 &&
                one_split_merges(MODE, scheme, G, NGv, B, H_q, H_kv, max_S, p.L, top_k, p.Kc);
  const WsLayout wl = ws_layout(B, H_q, p.n_splits, p.Kc, p.mg_parts, top_k);
  if (!scores_only) {
    JF_CHECK_ARG(workspace && workspace_bytes >= wl.total, "fused_scan: workspace too small (%zu < %zu)", workspace_bytes, wl.total);
    JF_CHECK_ARG(((uintptr_t)workspace & 255) == 0, "fused_scan: workspace must be 256-byte aligned");
  }
  uint8_t* ws = reinterpret_cast<uint8_t*>(workspace);
  p.scores = HAS_K ? scores : nullptr;
  p.scores_in = scores_in;
  p.stats_m = p.stats_iz = nullptr;
  p.scores_only = scores_only ? 1 : 0;
  p.part_m = reinterpret_cast<float*>(ws + wl.off_m);
  p.part_l = reinterpret_cast<float*>(ws + wl.off_l);
  p.part_o = reinterpret_cast<float*>(ws + wl.off_o);
  p.cand_key = reinterpret_cast<uint32_t*>(ws + wl.off_key);
  p.cand_idx = reinterpret_cast<int32_t*>(ws + wl.off_idx);
  p.cand_edge = reinterpret_cast<float*>(ws + wl.off_edge);
  p.key2 = reinterpret_cast<uint32_t*>(ws + wl.off_key2);
  p.idx2 = reinterpret_cast<int32_t*>(ws + wl.off_idx2);
  p.edge2 = reinterpret_cast<float*>(ws + wl.off_edge2);
  p.topk_idx = topk_idx; p.topk_slots = topk_slots; p.o_hat = o_hat; p.o_old = o_old_unnorm; p.W = W;
  p.softmax_m = softmax_m; p.softmax_inv_z = softmax_inv_z;
  p.blend_o_new = blend_o_new; p.blend_out = blend_out;
#ifdef JF_DEBUG_HOOKS
  p.phase_clock = g_phase_clock.load(std::memory_order_relaxed);
#else
  p.phase_clock = nullptr;
#endif
  hipStream_t st = (hipStream_t)stream;
  int rc = JF_OK;
#define JF_FUSED_CASE(SCH, GG, NGG) rc = launch_scan<MODE, SCH, GG, NGG>(p, st)
#define JF_FUSED_BY_G(SCH, NGG)                        \
  switch (G) {                                         \
    case 1: JF_FUSED_CASE(SCH, 1, NGG); break;         \
    case 2: JF_FUSED_CASE(SCH, 2, NGG); break;         \
    case 4: JF_FUSED_CASE(SCH, 4, NGG); break;         \
    case 8: JF_FUSED_CASE(SCH, 8, NGG); break;         \
    default: JF_FUSED_CASE(SCH, 16, NGG); break;       \
  }
  if constexpr (MODE == FS_FULL) {  // (instantiated elsewhere, by family)
    // One chunk of 64 positions per wavefront at most (see SHORT).  It is the split's length that counts, not the sequence's:
    // the emission's segments are parts of L, and the form works through 64 positions per wavefront of each.
    const bool is_short = p.L <= 64 * (G <= 4 ? 16 : 8);
#define JF_SCAN_OF(F) rc = is_short ? launch_short_scan_##F(scheme, G, NGv, &p, stream) : launch_full_scan_##F(scheme, G, NGv, &p, stream)
    if (scheme_has_zp(scheme)) JF_SCAN_OF(d);
    else if (scheme / 10 == 5) JF_SCAN_OF(e);
    else if (scheme / 10 == 2) JF_SCAN_OF(b);
    else if (scheme == JF_SCHEME_K3V3 || scheme == JF_SCHEME_K4V3) JF_SCAN_OF(c);
    else JF_SCAN_OF(a);
#undef JF_SCAN_OF
  } else if constexpr (MODE == FS_TOPK) {
    JF_FUSED_BY_G(JF_SCHEME_K4V4, 1)
  } else if (scheme == JF_SCHEME_K3V2) {
    if (NGv == 2) JF_FUSED_BY_G(JF_SCHEME_K3V2, 2) else JF_FUSED_BY_G(JF_SCHEME_K3V2, 1)
  } else if (scheme == JF_SCHEME_K4V4) {
    JF_FUSED_BY_G(JF_SCHEME_K4V4, 1)
  } else if constexpr (MODE == FS_STAGE_B) {
    if (scheme == JF_SCHEME_K3V4) {  // INT4 values with either group size (one group: the K4V4 instantiation)
      if (NGv == 2) JF_FUSED_BY_G(JF_SCHEME_K3V4, 2) else JF_FUSED_BY_G(JF_SCHEME_K4V4, 1)
    } else if (NGv == 2) JF_FUSED_BY_G(JF_SCHEME_K3V3, 2) else JF_FUSED_BY_G(JF_SCHEME_K3V3, 1)
  } else if (scheme == JF_SCHEME_K2V2) {  // (Stage A)
    if (NGv == 2) JF_FUSED_BY_G(JF_SCHEME_K2V2, 2) else JF_FUSED_BY_G(JF_SCHEME_K2V2, 1)
  } else if (scheme == JF_SCHEME_B4V2) {
    if (NGv == 2) JF_FUSED_BY_G(JF_SCHEME_B4V2, 2) else JF_FUSED_BY_G(JF_SCHEME_B4V2, 1)
  } else {
    if (NGv == 2) JF_FUSED_BY_G(JF_SCHEME_A2V2, 2) else JF_FUSED_BY_G(JF_SCHEME_A2V2, 1)
  }
#undef JF_FUSED_BY_G
#undef JF_FUSED_CASE
  if (rc != JF_OK || scores_only || p.one_split) return rc;
  const dim3 mgrid(g_act, H_kv, B);
  const bool wide = top_k > FS_LDS_TOPK;  // the winners' arrays do not fit the kernels' static LDS
  if (p.mg_parts > 1) {  // first stage: every part's top_k, as new candidate lists (the same kernel for every form)
    const dim3 pgrid(B, H_q, p.mg_parts);
    const MergeParams mp = merge_params(p, true);
    if (wide) rc = launch_wide_merge<fused_merge_kernel<FS_FULL, 4, 1, 1024, 32, true, true>>(pgrid, mp, st);
    else if ((long long)p.mg_spp * p.Kc > MG_REG_CANDS) hipLaunchKernelGGL((fused_merge_kernel<FS_FULL, 4, 1, 1024, 32, true>), pgrid, dim3(1024), 0, st, mp);
    else hipLaunchKernelGGL((fused_merge_kernel<FS_FULL, 4, 1, 1024, 8, true>), pgrid, dim3(1024), 0, st, mp);
    if (rc != JF_OK) return rc;
    JF_CHECK_LAUNCH();
  }
  const MergeParams mp = merge_params(p, false);
  const bool big = (MODE != FS_STAGE_B) &&
                   (p.mg_parts > 1 ? (long long)p.mg_parts * top_k : (long long)p.n_splits * p.Kc) > MG_REG_CANDS;
  // Many rows with few candidates each (large batches of short or medium sequences): four wavefronts per row and
  // small tables, so that five rows share a CU instead of one (measured from 257 rows up: 42.5 against 47.5 us per
  // layer at 384 rows of 2048 candidates, 38 against 57 at 1024 rows of 512).  Same results (see VGRP in
  // the kernel).
  const bool light = (MODE == FS_FULL) && !big && p.mg_parts == 1 && top_k <= MG_LIGHT_TOPK &&
                     (long long)B * H_q > (long long)device_cus() && (long long)p.n_splits * p.Kc <= MG_LIGHT_THREADS * MG_LIGHT_REGK;
  // More rows than CUs that the light shape does not take: half the wavefronts with twice the candidates each.  What every wavefront
  // does for itself is done half as often, and two rows share a CU (82 vector registers): per layer, 1024 threads / this, 288 rows of 8 lists
  // (9 x 4096 positions, K3V2, top-k 1024) 36.9 / 31.7 us, 384 (12 x 2500) 35.6 / 30.4, 512 (16 x 4096) 42.1 / 37.2, 1024 (32 x
  // 3000) 61.4 / 49.3, K4V4, 2048 84.0 / 73.5.  With a row per CU the sixteen wavefronts are the shorter way: 256 rows 25.2 / 25.8,
  // 128 (4 x 32768, 256) 33.7 / 34.45.
  const bool medium = (MODE == FS_FULL) && !wide && !big && !light && (long long)B * H_q > (long long)device_cus();
  (void)medium;
  // the rows of both of a wavefront's turns at once where there are two and four workgroups per CU hold every row (see PER_CU)
  const bool gather = light && top_k > 256 && (long long)B * H_q <= 4ll * device_cus();
  (void)gather;
#define JF_MERGE(VB, NGG)                                                                                            \
  do {                                                                                                               \
    if (wide) {                                                                                                      \
      if constexpr (MODE == FS_STAGE_B) rc = launch_wide_merge<fused_merge_kernel<MODE, VB, NGG, 1024, 8, false, true>>(mgrid, mp, st); \
      else rc = launch_wide_merge<fused_merge_kernel<MODE, VB, NGG, 1024, 32, false, true>>(mgrid, mp, st);            \
    } else if (big) hipLaunchKernelGGL((fused_merge_kernel<MODE, VB, NGG, 1024, 32, false>), mgrid, dim3(1024), 0, st, mp); \
    else if (light) {                                                                                                \
      if constexpr (MODE == FS_FULL) {                                                                               \
        if (gather) hipLaunchKernelGGL((fused_merge_kernel<FS_FULL, VB, NGG, MG_LIGHT_THREADS, MG_LIGHT_REGK, false, false, 4>), mgrid, dim3(MG_LIGHT_THREADS), 0, st, mp); \
        else hipLaunchKernelGGL((fused_merge_kernel<FS_FULL, VB, NGG, MG_LIGHT_THREADS, MG_LIGHT_REGK, false>), mgrid, dim3(MG_LIGHT_THREADS), 0, st, mp); \
      }                                                                                                              \
    } else if (medium) {                                                                                               \
      if constexpr (MODE == FS_FULL) hipLaunchKernelGGL((fused_merge_kernel<FS_FULL, VB, NGG, MG_MEDIUM_THREADS, MG_MEDIUM_REGK, false>), mgrid, dim3(MG_MEDIUM_THREADS), 0, st, mp); \
    } else hipLaunchKernelGGL((fused_merge_kernel<MODE, VB, NGG, 1024, 8, false>), mgrid, dim3(1024), 0, st, mp);       \
  } while (0)
  if constexpr (MODE == FS_STAGE_A || MODE == FS_TOPK) {  // no value rows are read: one instantiation serves every format
    if (wide) rc = launch_wide_merge<fused_merge_kernel<FS_STAGE_A, 4, 1, 1024, 32, false, true>>(mgrid, mp, st);
    else if (big) hipLaunchKernelGGL((fused_merge_kernel<FS_STAGE_A, 4, 1, 1024, 32, false>), mgrid, dim3(1024), 0, st, mp);
    else hipLaunchKernelGGL((fused_merge_kernel<FS_STAGE_A, 4, 1, 1024, 8, false>), mgrid, dim3(1024), 0, st, mp);
  } else if (scheme % 10 == 2) {  // INT2 values
    if (NGv == 2) JF_MERGE(2, 2);
    else JF_MERGE(2, 1);
  } else if (scheme % 10 == 3) {  // INT3 values
    if (NGv == 2) JF_MERGE(3, 2);
    else JF_MERGE(3, 1);
  } else {
    if (NGv == 2) JF_MERGE(4, 2);
    else JF_MERGE(4, 1);
  }
#undef JF_MERGE
  if (rc != JF_OK) return rc;
  JF_CHECK_LAUNCH();
  return JF_OK;
}

// Stage B merge kernel with the caller's softmax statistics: o_hat is the plain sum of normalised partial rows, and
//   W = sum_j p_j, o_old_unnorm = sum_j p_j * Vhat_j over the given winners, p_j = exp(score_j - m) * inv_z.
template <int VBITS, int NG>
static int launch_precorr_given_stats(const float* scores, const float* softmax_m, const float* softmax_inv_z,
                                      const uint8_t* v_data, const uint16_t* v_scales, const int64_t* block_table,
                                      const int32_t* seq_lens, const int64_t* topk_idx, int B, int H_q, int H_kv,
                                      int max_S, int max_blocks, int64_t num_slots, int top_k, const float* partial,
                                      int n_partial, float* o_hat, float* o_old_unnorm, float* W, hipStream_t st) {
  FusedParams p = {};
  p.v_data = v_data; p.v_scales = v_scales; p.block_table = block_table; p.seq_lens = seq_lens;
  p.B = B; p.H_q = H_q; p.H_kv = H_kv; p.g_act = H_q / H_kv; p.max_S = max_S; p.max_blocks = max_blocks; p.num_slots = num_slots;
  p.top_k = top_k;
  p.n_splits = n_partial; p.part_o = const_cast<float*>(partial); p.o_hat = o_hat; p.mg_parts = 1; p.mg_spp = 0; p.Kc = p.L = 0;
  p.scores_in = scores; p.stats_m = softmax_m; p.stats_iz = softmax_inv_z;
  p.topk_idx = const_cast<int64_t*>(topk_idx);
  p.o_old = o_old_unnorm; p.W = W;
  hipLaunchKernelGGL((fused_merge_kernel<FS_STAGE_B, VBITS, NG, 1024, 8, false>), dim3(p.g_act, H_kv, B), dim3(1024), 0, st, merge_params(p, false));
  JF_CHECK_LAUNCH();
  return JF_OK;
}

}  // namespace
}  // namespace jf
