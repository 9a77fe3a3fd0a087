// Slot-mapped K/V append into the paged cache (gfx950).
//
// Replaces tileInfer's store_kvcache (kernels/kvcache_store.py:43-71). The reference stages a
// block_N x D tile of K and V in shared memory and then scatters it (14-40); here every lane
// moves one 16-byte vector straight from the new-token row to its cache row, so a 2 KiB row
// (4 KV heads x 256 x bf16) is one fully coalesced 128-lane access for K and one for V, with no
// LDS round trip and no per-N specialisation.
#include "ti_common.h"

namespace ti {
namespace {

constexpr int kAppendThreads = 256;

// VecT is the per-lane access: u32x4 (16 B) when rows and strides allow it, else 16-bit. U: items of
// a lane in flight together.
template <typename VecT, int U>
__global__ __launch_bounds__(kAppendThreads) void kv_append_kernel(
    const VecT* __restrict__ key, const VecT* __restrict__ value, int64_t key_stride,
    int64_t value_stride, VecT* __restrict__ k_cache, VecT* __restrict__ v_cache,
    int64_t cache_stride, const int32_t* __restrict__ slot_mapping, uint32_t total,
    uint32_t row_vecs, int64_t num_slots) {
  // Strides are in units of VecT. One item = one vector of one token's K row and the matching
  // vector of its V row; a workgroup takes U blocks of kAppendThreads items at a time, every load
  // issued before the first slot is looked at (a skipped token's rows are read for nothing).
  const uint32_t step = gridDim.x * (U * kAppendThreads);
  for (uint32_t base = blockIdx.x * (U * kAppendThreads) + threadIdx.x; base < total; base += step) {
    VecT kx[U], vx[U];
    int32_t slot[U];
    uint32_t vec[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t i = min(base + u * kAppendThreads, total - 1);
      const uint32_t tok = i / row_vecs;
      vec[u] = i - tok * row_vecs;
      slot[u] = slot_mapping[tok];
      // The new rows are read once: streaming (nt) loads keep them out of the way of the cache rows.
      kx[u] = __builtin_nontemporal_load(key + tok * key_stride + vec[u]);
      vx[u] = __builtin_nontemporal_load(value + tok * value_stride + vec[u]);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // Past the last item, -1 padding, or a slot out of range: skip.
      if (base + u * kAppendThreads >= total || slot[u] < 0 || slot[u] >= num_slots) continue;
      k_cache[slot[u] * cache_stride + vec[u]] = kx[u];
      v_cache[slot[u] * cache_stride + vec[u]] = vx[u];
    }
  }
}

template <typename VecT, int U>
int launch_items(const void* key, const void* value, int64_t key_stride, int64_t value_stride,
                 void* k_cache, void* v_cache, int64_t cache_stride,
                 const int32_t* slot_mapping, int64_t n_tokens, int64_t row_elems,
                 int64_t num_slots, hipStream_t stream) {
  constexpr int64_t per = sizeof(VecT) / 2;  // 16-bit elements per vector
  const int64_t row_vecs = row_elems / per;
  const int64_t total = n_tokens * row_vecs;
  const int64_t blocks_needed = ceil_div(total, kAppendThreads * U);
  const int64_t max_blocks = int64_t(device_cu_count()) * 32;
  const unsigned grid = unsigned(blocks_needed < max_blocks ? blocks_needed : max_blocks);
  hipLaunchKernelGGL((kv_append_kernel<VecT, U>), dim3(grid), dim3(kAppendThreads), 0, stream,
                     static_cast<const VecT*>(key), static_cast<const VecT*>(value),
                     key_stride / per, value_stride / per, static_cast<VecT*>(k_cache),
                     static_cast<VecT*>(v_cache), cache_stride / per, slot_mapping,
                     uint32_t(total), uint32_t(row_vecs), num_slots);
  return check_launch("ti_kv_append");
}

// Items per lane by the call's size. The copy is bound by HBM once enough of it is in flight; a lane
// with one item waits for the memory once per item, one with more has fewer lanes to start. GPU time
// per call in us, rows of 4 x 256 (128 items a token), with 1 / 2 / 4 items per lane: 512 tokens
// 2.7 / 2.8 / 3.2, 2,080 5.2 / 5.1 / 5.4, 5,000 10.0 / 9.0 / 9.6, 16,384 24.7 / 23.8 / 23.8, 65,536
// 84.1 / 82.7 / 79.8, 131,072 219 / 217 / 211; rows of 1 x 256 (32 items): 5,000 3.5 / 3.8 / 3.9,
// 16,384 8.5 / 7.4 / 7.3, 131,072 43.0 / 41.7 / 42.0 (the former kernel, one item a lane and the slot
// looked at first: as 1, within 2 %). The lines are 1,024 and 16,384 items per CU.
template <typename VecT>
int launch_append(const void* key, const void* value, int64_t key_stride, int64_t value_stride,
                  void* k_cache, void* v_cache, int64_t cache_stride,
                  const int32_t* slot_mapping, int64_t n_tokens, int64_t row_elems,
                  int64_t num_slots, hipStream_t stream) {
  const int64_t total = n_tokens * (row_elems / int64_t(sizeof(VecT) / 2));
  if (total >= (int64_t(1) << 31)) {
    return fail(TI_EINVAL, "ti_kv_append: n_tokens*row_elems too large (%lld vectors)",
                (long long)total);
  }
  const int64_t per_cu = total / device_cu_count();
  const auto launch = per_cu < 1024 ? launch_items<VecT, 1>
                      : per_cu <= 16384 ? launch_items<VecT, 2>
                                        : launch_items<VecT, 4>;
  return launch(key, value, key_stride, value_stride, k_cache, v_cache, cache_stride, slot_mapping,
                n_tokens, row_elems, num_slots, stream);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace
}  // namespace ti

extern "C" int ti_kv_append(const void* key, const void* value, int64_t key_row_stride,
                            int64_t value_row_stride, void* k_cache, void* v_cache,
                            int64_t cache_row_stride, const int32_t* slot_mapping,
                            int64_t n_tokens, int64_t row_elems, int64_t num_slots,
                            int32_t dtype, void* stream) {
  using namespace ti;
  if (dtype != TI_DTYPE_BF16 && dtype != TI_DTYPE_F16) {
    return fail(TI_EUNSUPPORTED, "ti_kv_append: dtype code %d is not bf16/fp16", dtype);
  }
  if (n_tokens < 0 || row_elems <= 0 || num_slots < 0) {
    return fail(TI_EINVAL, "ti_kv_append: bad sizes n_tokens=%lld row_elems=%lld num_slots=%lld",
                (long long)n_tokens, (long long)row_elems, (long long)num_slots);
  }
  if (n_tokens == 0) return TI_OK;
  if (!key || !value || !k_cache || !v_cache || !slot_mapping) {
    return fail(TI_EINVAL, "ti_kv_append: null pointer");
  }
  if (key_row_stride < row_elems || value_row_stride < row_elems || cache_row_stride < row_elems) {
    return fail(TI_EINVAL, "ti_kv_append: row strides (%lld, %lld, %lld) < row_elems %lld",
                (long long)key_row_stride, (long long)value_row_stride,
                (long long)cache_row_stride, (long long)row_elems);
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool vec16 = (row_elems % 8 == 0) && (key_row_stride % 8 == 0) &&
                     (value_row_stride % 8 == 0) && (cache_row_stride % 8 == 0) &&
                     aligned16(key) && aligned16(value) && aligned16(k_cache) &&
                     aligned16(v_cache);
  if (vec16) {
    return launch_append<u32x4>(key, value, key_row_stride, value_row_stride, k_cache, v_cache,
                                cache_row_stride, slot_mapping, n_tokens, row_elems, num_slots,
                                s);
  }
  return launch_append<uint16_t>(key, value, key_row_stride, value_row_stride, k_cache, v_cache,
                                 cache_row_stride, slot_mapping, n_tokens, row_elems, num_slots,
                                 s);
}
