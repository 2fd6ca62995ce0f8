// Mirror of appended bf16 K/V rows into the host shadow the CPU correction reads.
//
// The shadow lives in pinned host memory that the GPU can address, so one kernel stores every appended row
// straight to shadow[h, slots[t], :] across PCIe: no staging buffer, no host-side scatter, no host callback,
// and the launch can be recorded into a HIP graph like any other kernel.  Rows are 256 bytes and leave as
// 16-byte stores that are contiguous across the sixteen lanes of a row (consecutive slots give longer runs).
// Writes to pinned host memory are visible to the host once the kernel has completed.
//
// append_rows_kernel is the whole append of one layer in one launch: both tensors' rows are quantised into the packed
// cache (quant_rows.h), the slots marked as filled, and, where the mirror belongs to the same stream, the bf16 rows
// stored to the shadow from the registers that were quantised.
#include "quant_rows.h"

namespace jf {
namespace {

struct MirrorSrc {
  const uint16_t* x;
  int64_t stride_t, stride_h;  // elements
};

// LPR lanes own one row: 16 lanes x 16 bytes, or 64 lanes x 4 bytes for rows that are only 4-byte aligned.
// Grid: x = blocks of 256 / LPR tokens, y = kv-head, z = tensor (K, V).
// Mirror launches that have run on this device, replays from a HIP graph included (the reference counts its
// graph-mode append callbacks, jetfire_vllm/csrc/cpu_topk_attn.cpp:1611-1616); device code only.
__device__ unsigned long long shadow_appends;

template <int LPR>
__global__ __launch_bounds__(256) void shadow_write_kernel(MirrorSrc k, MirrorSrc v, uint16_t* __restrict__ k_shadow,
                                                           uint16_t* __restrict__ v_shadow, int64_t stride_h,
                                                           int64_t stride_slot, const int64_t* __restrict__ slots,
                                                           int64_t T, int64_t num_slots) {
  constexpr int RPB = 256 / LPR;
  if ((blockIdx.x | blockIdx.y | blockIdx.z | threadIdx.x) == 0) atomicAdd(&shadow_appends, 1ull);
  const int l = threadIdx.x % LPR;
  const int64_t t = (int64_t)blockIdx.x * RPB + threadIdx.x / LPR;
  if (t >= T) return;
  const int64_t slot = slots[t];
  if (slot < 0 || slot >= num_slots) return;  // padding tokens; a slot outside the shadow is never stored to
  const int h = blockIdx.y;
  const MirrorSrc& s = blockIdx.z ? v : k;
  uint16_t* shadow = blockIdx.z ? v_shadow : k_shadow;
  const uint16_t* src = s.x + t * s.stride_t + (int64_t)h * s.stride_h;
  uint16_t* dst = shadow + (int64_t)h * stride_h + slot * stride_slot;
  if (LPR == 16) {
    const uint4 r = reinterpret_cast<const uint4*>(src)[l];
    uint32_t* d32 = reinterpret_cast<uint32_t*>(dst) + 4 * l;
    __builtin_nontemporal_store(r.x, d32);
    __builtin_nontemporal_store(r.y, d32 + 1);
    __builtin_nontemporal_store(r.z, d32 + 2);
    __builtin_nontemporal_store(r.w, d32 + 3);
  } else {
    __builtin_nontemporal_store(reinterpret_cast<const uint32_t*>(src)[l], reinterpret_cast<uint32_t*>(dst) + l);
  }
}

struct AppendParams {
  RowSrc k, v;
  RowDst kd, vd;
  uint16_t* k_zp;  // asymmetric INT2 keys only
  int64_t zp_stride_h, zp_stride_slot;
  const int64_t* slots;
  int64_t T, num_slots;
  int group_size;
  uint8_t* filled;                   // optional: filled[slot] = 1
  uint16_t *k_shadow, *v_shadow;     // optional: device-visible addresses of the host shadow
  int64_t shadow_stride_h, shadow_stride_slot;
};

// Grid: x = blocks of 16 tokens, y = kv-head, z = tensor (K, V); sixteen lanes per row, as quant_write16_kernel.
// KF: key bits, or 1 for the asymmetric INT2 keys.
// A decode append (a few tokens) is launches: two writers, three small kernels that marked the slots and the mirror took
// 55 us per layer from the host's call on (5 tokens, 8 kv-heads), this one 18 us.  A chunk is HBM traffic, 512 bytes read
// and 76..136 written per token and kv-head; one launch for both tensors has no gap and one tail (16371 tokens, 8
// kv-heads, INT3 / INT2, group 64: 43 us before, 16.6 us = 4.7 TB/s now; a plain device copy reaches 5.1 TB/s).
template <int KF, int VN>
__global__ __launch_bounds__(256) void append_rows_kernel(AppendParams p) {
  const int l16 = threadIdx.x & 15;
  const uint32_t r = threadIdx.x >> 4;
  const int64_t t0 = (int64_t)blockIdx.x * 16;
  const int h = blockIdx.y;
  const bool values = blockIdx.z != 0;
  // rows past the end re-read the block's first row (they take part in the cross-lane steps) and store nothing
  const bool inside = t0 + r < p.T;
  const uint32_t re = inside ? r : 0u;
  const int64_t slot = p.slots[t0 + re];
  const RowSrc& s = values ? p.v : p.k;
  const uint16_t* xrow = s.x + t0 * s.stride_t + (int64_t)h * s.stride_h + (uint64_t)re * (uint32_t)s.stride_t;
  const uint4 raw = reinterpret_cast<const uint4*>(xrow)[l16];
  const bool live = inside && slot >= 0 && slot < p.num_slots;
  if (values) quant16_row<VN>(raw, p.vd, h, (uint32_t)slot, live, l16, p.group_size);
  else if constexpr (KF == 1) quant16_row_int2_asym(raw, p.kd, p.k_zp, p.zp_stride_h, p.zp_stride_slot, h, slot, live, l16, p.group_size);
  else quant16_row<KF>(raw, p.kd, h, (uint32_t)slot, live, l16, p.group_size);
  uint16_t* shadow = values ? p.v_shadow : p.k_shadow;
  if (shadow) {  // (uniform)
    if ((blockIdx.x | blockIdx.y | blockIdx.z | threadIdx.x) == 0) atomicAdd(&shadow_appends, 1ull);
    if (live) {
      typedef uint32_t v4u __attribute__((ext_vector_type(4)));
      v4u* dst = reinterpret_cast<v4u*>(shadow + (int64_t)h * p.shadow_stride_h + slot * p.shadow_stride_slot);
      __builtin_nontemporal_store((v4u){raw.x, raw.y, raw.z, raw.w}, dst + l16);
    }
  }
  if (p.filled && h == 0 && !values && live && l16 == 0) p.filled[slot] = 1;
}

template <int KF>
void launch_append(int v_nbits, dim3 grid, const AppendParams& p, hipStream_t st) {
  if (v_nbits == 2) hipLaunchKernelGGL((append_rows_kernel<KF, 2>), grid, dim3(256), 0, st, p);
  else if (v_nbits == 3) hipLaunchKernelGGL((append_rows_kernel<KF, 3>), grid, dim3(256), 0, st, p);
  else hipLaunchKernelGGL((append_rows_kernel<KF, 4>), grid, dim3(256), 0, st, p);
}

inline bool aligned16(const void* x, int64_t stride_t, int64_t stride_h) {
  return ((uintptr_t)x & 15) == 0 && stride_t % 8 == 0 && stride_h % 8 == 0;
}

}  // namespace
}  // namespace jf

using namespace jf;

extern "C" int jf_host_buffer_device_pointer(const void* host_ptr, void** device_ptr) {
  JF_CHECK_ARG(host_ptr && device_ptr, "host_buffer_device_pointer: null pointer");
  hipPointerAttribute_t attr;
  hipError_t e = hipPointerGetAttributes(&attr, host_ptr);
  if (e != hipSuccess) {
    (void)hipGetLastError();  // an unknown pointer is an answer, not a sticky error
    set_error("host_buffer_device_pointer: %p is not known to the HIP runtime (pageable host memory?): %s", host_ptr,
              hipGetErrorString(e));
    return JF_ERR_ARG;
  }
  JF_CHECK_ARG(attr.type == hipMemoryTypeHost && attr.devicePointer != nullptr,
               "host_buffer_device_pointer: %p is not pinned host memory the GPU can address (memory type %d)",
               host_ptr, (int)attr.type);
  *device_ptr = attr.devicePointer;
  return JF_OK;
}

extern "C" int jf_shadow_write(const uint16_t* key, int64_t k_stride_t, int64_t k_stride_h, const uint16_t* value,
                               int64_t v_stride_t, int64_t v_stride_h, const int64_t* slots, int64_t T, int H_kv,
                               uint16_t* k_shadow, uint16_t* v_shadow, int64_t shadow_stride_h,
                               int64_t shadow_stride_slot, int64_t num_slots, void* stream) {
  JF_CHECK_ARG(T >= 0 && H_kv > 0 && H_kv <= 65535, "shadow_write: bad T=%lld H_kv=%d", (long long)T, H_kv);
  JF_CHECK_ARG(T <= (int64_t)4 * 0x7fffffff, "shadow_write: T=%lld exceeds the launch grid", (long long)T);
  if (T == 0) return JF_OK;
  JF_CHECK_ARG(key && value && slots && k_shadow && v_shadow, "shadow_write: null pointer");
  JF_CHECK_ARG(num_slots > 0 && shadow_stride_slot >= D && shadow_stride_h >= shadow_stride_slot,
               "shadow_write: bad shadow geometry (num_slots=%lld, strides %lld / %lld)", (long long)num_slots,
               (long long)shadow_stride_h, (long long)shadow_stride_slot);
  JF_CHECK_ARG((k_stride_t | k_stride_h | v_stride_t | v_stride_h) % 2 == 0 && (((uintptr_t)key | (uintptr_t)value) & 3) == 0,
               "shadow_write: token rows must be 4-byte aligned");
  JF_CHECK_ARG((((uintptr_t)k_shadow | (uintptr_t)v_shadow) & 15) == 0 && shadow_stride_h % 8 == 0 && shadow_stride_slot % 8 == 0,
               "shadow_write: shadow rows must be 16-byte aligned");
  MirrorSrc k{key, k_stride_t, k_stride_h}, v{value, v_stride_t, v_stride_h};
  hipStream_t st = (hipStream_t)stream;
  if (aligned16(key, k_stride_t, k_stride_h) && aligned16(value, v_stride_t, v_stride_h)) {
    dim3 grid((unsigned)((T + 15) / 16), (unsigned)H_kv, 2);
    hipLaunchKernelGGL(shadow_write_kernel<16>, grid, dim3(256), 0, st, k, v, k_shadow, v_shadow, shadow_stride_h,
                       shadow_stride_slot, slots, T, num_slots);
  } else {
    dim3 grid((unsigned)((T + 3) / 4), (unsigned)H_kv, 2);
    hipLaunchKernelGGL(shadow_write_kernel<64>, grid, dim3(256), 0, st, k, v, k_shadow, v_shadow, shadow_stride_h,
                       shadow_stride_slot, slots, T, num_slots);
  }
  JF_CHECK_LAUNCH();
  return JF_OK;
}

extern "C" int jf_shadow_append_count(int64_t* count, int reset) {
  JF_CHECK_ARG(count, "shadow_append_count: null output");
  unsigned long long v = 0;
  JF_CHECK_HIP(hipMemcpyFromSymbol(&v, HIP_SYMBOL(shadow_appends), sizeof(v)));
  *count = (int64_t)v;
  if (reset) {
    const unsigned long long zero = 0;
    JF_CHECK_HIP(hipMemcpyToSymbol(HIP_SYMBOL(shadow_appends), &zero, sizeof(zero)));
  }
  return JF_OK;
}

extern "C" int jf_append_rows(const uint16_t* key, int64_t k_stride_t, int64_t k_stride_h, const uint16_t* value,
                              int64_t v_stride_t, int64_t v_stride_h, const int64_t* slots, int64_t T, int H_kv,
                              uint8_t* k_data, int64_t k_data_stride_h, int64_t k_data_stride_slot, uint16_t* k_scale,
                              int64_t k_scale_stride_h, int64_t k_scale_stride_slot, uint16_t* k_zp, int64_t zp_stride_h,
                              int64_t zp_stride_slot, uint8_t* v_data, int64_t v_data_stride_h, int64_t v_data_stride_slot,
                              uint16_t* v_scale, int64_t v_scale_stride_h, int64_t v_scale_stride_slot, int64_t num_slots,
                              int group_size, int k_nbits, int v_nbits, uint8_t* slot_filled, uint16_t* k_shadow,
                              uint16_t* v_shadow, int64_t shadow_stride_h, int64_t shadow_stride_slot, void* stream) {
  JF_CHECK_ARG(T >= 0 && T <= (int64_t)16 * 0x7fffffff && H_kv > 0 && H_kv <= 65535, "append_rows: bad T=%lld H_kv=%d",
               (long long)T, H_kv);
  JF_CHECK_ARG(group_size == 32 || group_size == 64 || group_size == 128, "append_rows: group_size must be 32, 64 or 128 (got %d)",
               group_size);
  JF_CHECK_ARG(k_nbits >= 2 && k_nbits <= 4 && v_nbits >= 2 && v_nbits <= 4, "append_rows: bits must be 2, 3 or 4 (got %d / %d)",
               k_nbits, v_nbits);
  JF_CHECK_ARG(!k_zp || k_nbits == 2, "append_rows: zero-points go with INT2 keys");
  JF_CHECK_ARG((k_shadow == nullptr) == (v_shadow == nullptr), "append_rows: the two shadows go together");
  if (T == 0) return JF_OK;
  JF_CHECK_ARG(key && value && slots && k_data && k_scale && v_data && v_scale, "append_rows: null pointer");
  JF_CHECK_ARG(num_slots > 0 && num_slots < ((int64_t)1 << 32), "append_rows: num_slots out of range");
  JF_CHECK_ARG(rows_16b_aligned(key, k_stride_t, k_stride_h) && rows_16b_aligned(value, v_stride_t, v_stride_h),
               "append_rows: token rows must be 16-byte aligned");
  JF_CHECK_ARG(strides_fit_32(k_stride_t, k_data_stride_slot, k_scale_stride_slot) &&
                   strides_fit_32(v_stride_t, v_data_stride_slot, v_scale_stride_slot), "append_rows: strides beyond 32 bits");
  JF_CHECK_ARG((((uintptr_t)k_data | (uintptr_t)v_data) & 3) == 0 && (k_data_stride_slot | k_data_stride_h) % 4 == 0 &&
                   (v_data_stride_slot | v_data_stride_h) % 4 == 0 && k_data_stride_slot >= D * k_nbits / 8 &&
                   v_data_stride_slot >= D * v_nbits / 8, "append_rows: cache rows must be 4-byte aligned and wide enough");
  if (k_shadow)
    JF_CHECK_ARG((((uintptr_t)k_shadow | (uintptr_t)v_shadow) & 15) == 0 && shadow_stride_h % 8 == 0 &&
                     shadow_stride_slot % 8 == 0 && shadow_stride_slot >= D && shadow_stride_h >= shadow_stride_slot,
                 "append_rows: shadow rows must be 16-byte aligned");
  const AppendParams p{{key, k_stride_t, k_stride_h}, {value, v_stride_t, v_stride_h},
                       {k_data, k_data_stride_h, k_data_stride_slot, k_scale, k_scale_stride_h, k_scale_stride_slot},
                       {v_data, v_data_stride_h, v_data_stride_slot, v_scale, v_scale_stride_h, v_scale_stride_slot},
                       k_zp, zp_stride_h, zp_stride_slot, slots, T, num_slots, group_size, slot_filled, k_shadow, v_shadow,
                       shadow_stride_h, shadow_stride_slot};
  const dim3 grid((unsigned)((T + 15) / 16), (unsigned)H_kv, 2);
  hipStream_t st = (hipStream_t)stream;
  if (k_zp) launch_append<1>(v_nbits, grid, p, st);
  else if (k_nbits == 2) launch_append<2>(v_nbits, grid, p, st);
  else if (k_nbits == 3) launch_append<3>(v_nbits, grid, p, st);
  else launch_append<4>(v_nbits, grid, p, st);
  JF_CHECK_LAUNCH();
  return JF_OK;
}
