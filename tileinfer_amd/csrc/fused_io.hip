// The element-wise work on either side of the paged attention path, fused with it.
//
// Before attention (model/qwen_36.py:977-1018): per-head RMSNorm of q and k with a (1 + w)
// weight, partial rotary embedding on the first rotary_dim dimensions, then the slot-mapped append
// of k and v. The reference runs the first two as one TileLang kernel for a single sequence
// (kernels/qknorm_rope.py:9-56) and as separate torch ops otherwise, then store_kvcache.
//   ti_qknorm_rope         q or k alone (any number of tokens, per-token cos/sin)
//   ti_qknorm_rope_append  q, k and v of one step in one launch: q normalised and rotated to its
//                          output, k normalised and rotated and v as is, written straight into
//                          the cache rows at slot_mapping (no intermediate k)
// After attention (model/qwen_36.py:1083, kernels/act_mul.py:62-79): out = attn * sigmoid(gate).
//   ti_sigmoid_mul         the element-wise product alone (the decode kernel also applies it in
//                          its output epilogue, ti_gqa_decode_paged_gated)
//
// Numerics follow the reference's fused kernel (kernels/qknorm_rope.py:29-49): sum of squares and
// scale in fp32, normalised row rounded to the storage type, rotation in fp32 from those values
// with cos/sin[0 .. rotary_dim/2) for both halves (rotate-half pairing i <-> i + rotary_dim/2),
// rounded once. The fused append writes exactly what ti_qknorm_rope followed by the append would.
#include "decode_common.h"

namespace ti {
namespace {

// x rounded to 32 bits: the compiler may not fold it into what follows, in one kernel and not in
// another; the forms below have to give the same bits.
__device__ __forceinline__ float rounded(float x) {
  asm("" : "+v"(x));
  return x;
}

// A rotated value is own * c + this: the partner's part in the first half of the pair (low) or the
// second.
__device__ __forceinline__ float partner_part(float partner, float s, bool low) {
  const float ps = rounded(partner * s);
  return low ? -ps : ps;
}

struct NormRopeArgs {
  const uint16_t* x;
  int64_t x_st, x_sh;
  uint16_t* out;  // row outputs (q or k) or nullptr
  int64_t o_st, o_sh;
  const uint16_t* w;
  const uint16_t* cos;
  const uint16_t* sin;
  int64_t cs_st;  // cos/sin token stride (0: one vector for every token)
  int32_t n_tokens, n_heads, rotary_dim;
  float eps;
  // Cache-row output (fused append): row slot of token t, head h at cache + slot*row + h*D.
  uint16_t* cache;
  int64_t cache_row;
  const int32_t* slots;
  int64_t num_slots;
};


// Rows of 16-byte aligned vectors (every stride a multiple of 8 elements, rotary_dim of 16): a row is
// D / 8 lanes of 8 elements, so a wave takes 2 (D = 256) or 4 (D = 128) rows at once, and a
// workgroup walks the rows with the next ones' loads in flight. The general form below (one wave per
// row, 4-byte accesses) spends its time on dispatching workgroups and on narrow accesses: 2,080
// tokens of 24 + 2 x 4 heads of 256 took 24.8 us, 17.5 us here (69 MB of unique bytes, 3.9 TB/s).
// What a row needs beside its values: where it goes (nullptr: nowhere) and whether it is a v row
// (copied) or a q or k row (normalised and rotated, with this token's cos / sin).
struct RowJob {
  const uint16_t* src;
  uint16_t* dst;
  int tok;
  int kind;  // 0: q, 1: k, 2: v
};

// Normalises and rotates the row whose elements [8 l, 8 l + 8) lane l of its D / 8 lanes holds in x
// (w: the same elements of the weight).
template <int D, typename Tag>
__device__ __forceinline__ u32x4 norm_rope_vec(const NormRopeArgs& a, u32x4 x, u32x4 w, int t,
                                               int lane) {
  constexpr int LPR = D / 8;
  const int l = lane & (LPR - 1);
  float v[8];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float2 p = unpack2(x[j], Tag{});
    v[2 * j] = p.x;
    v[2 * j + 1] = p.y;
  }
  // The sum of squares in the order of the general form, whose lanes hold EPL elements each: one
  // partial sum per such lane, across the lanes first, then among themselves. Both forms so give
  // the same bits.
  constexpr int EPL = D / 64, PARTS = 8 / EPL;
  float part[PARTS];
#pragma unroll
  for (int i = 0; i < PARTS; ++i) {
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < EPL; ++j) ss += v[EPL * i + j] * v[EPL * i + j];
#pragma unroll
    for (int d = LPR / 2; d > 0; d >>= 1) ss += __shfl_xor(ss, d, 64);
    part[i] = ss;
  }
#pragma unroll
  for (int d = PARTS / 2; d > 0; d >>= 1) {
#pragma unroll
    for (int i = 0; i < d; ++i) part[i] += part[i + d];
  }
  const float ss = part[0];
  const float r = rsqrtf(ss / float(D) + a.eps);
  u32x4 nb;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float2 q = unpack2(w[j], Tag{});
    nb[j] = pack_mul2(rounded(v[2 * j] * r), 1.f + q.x, rounded(v[2 * j + 1] * r), 1.f + q.y, Tag{});
  }
  if (a.rotary_dim == 0) return nb;  // uniform
  const int half = a.rotary_dim / 2;
  const bool low = 8 * l < half;
  // The rotation partners, half elements (half / 8 lanes) away.
  const int from = (lane & ~(LPR - 1)) | ((low ? l + half / 8 : l - half / 8) & (LPR - 1));
  u32x4 pb;
#pragma unroll
  for (int j = 0; j < 4; ++j) pb[j] = uint32_t(__shfl(int(nb[j]), from, 64));
  if (8 * l >= a.rotary_dim) return nb;
  const int64_t cs = int64_t(t) * a.cs_st + (low ? 8 * l : 8 * l - half);
  const u32x4 c = load16(a.cos + cs);
  const u32x4 sn = load16(a.sin + cs);
  u32x4 res;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float2 own = unpack2(nb[j], Tag{});
    const float2 partner = unpack2(pb[j], Tag{});
    const float2 cc = unpack2(c[j], Tag{});
    const float2 s2 = unpack2(sn[j], Tag{});
    res[j] = pack_fma2(own.x, cc.x, partner_part(partner.x, s2.x, low), own.y, cc.y,
                       partner_part(partner.y, s2.y, low), Tag{});
  }
  return res;
}

// Walks rows [0, rows) of job_of(row), the wave's share of them.
template <int D, typename Tag, typename JobOf>
__device__ __forceinline__ void norm_rope_rows(const NormRopeArgs& q, const uint16_t* kw,
                                               int64_t rows, JobOf job_of) {
  constexpr int LPR = D / 8;
  constexpr int RPW = 64 / LPR;  // rows per wave
  const int lane = threadIdx.x & 63;
  const int l8 = 8 * (lane & (LPR - 1));
  const u32x4 w_q = load16(q.w + l8);
  const u32x4 w_k = load16(kw + l8);
  const int64_t step = int64_t(gridDim.x) * 4 * RPW;
  int64_t row = (int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6)) * RPW + lane / LPR;
  // The shuffles inside need whole waves: lanes past the last row repeat it and store nothing.
  RowJob job = job_of(row < rows ? row : rows - 1);
  u32x4 x = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(job.src + l8));
  for (int64_t base = row - lane / LPR; base < rows; base += step) {  // uniform in the wave
    const RowJob now = job;
    const u32x4 xn = x;
    const bool live = row < rows;
    row += step;
    if (base + step < rows) {
      job = job_of(row < rows ? row : rows - 1);
      x = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(job.src + l8));
    }
    const u32x4 y = norm_rope_vec<D, Tag>(q, xn, now.kind == 1 ? w_k : w_q, now.tok, lane);
    if (live && now.dst != nullptr) {
      *reinterpret_cast<u32x4*>(now.dst + l8) = now.kind == 2 ? xn : y;
    }
  }
}

template <int D, typename Tag>
__global__ __launch_bounds__(256) void norm_rope_vec_kernel(NormRopeArgs a) {
  const uint32_t heads = uint32_t(a.n_heads);
  norm_rope_rows<D, Tag>(a, a.w, int64_t(a.n_tokens) * heads, [&](int64_t row) {
    const uint32_t t = uint32_t(row) / heads, h = uint32_t(row) - t * heads;
    return RowJob{a.x + t * a.x_st + h * a.x_sh, a.out + t * a.o_st + h * a.o_sh, int(t), 0};
  });
}

// Normalises and rotates row (t, h) of `a.x` (one wave per row); returns the lane's EPL output
// values, packed. Lane l owns elements [EPL*l, EPL*l + EPL). `sh` is this wave's LDS row of D
// 16-bit values, through which the rotation partners (i <-> i +- rotary_dim/2) are exchanged.
template <int D, typename Tag>
__device__ __forceinline__ void norm_rope_row(const NormRopeArgs& a, int t, int h, uint16_t* sh,
                                              uint32_t (&res)[D / 128]) {
  constexpr int EPL = D / 64;  // 2 or 4 elements per lane
  const int lane = threadIdx.x & 63;
  const uint16_t* xr = a.x + int64_t(t) * a.x_st + int64_t(h) * a.x_sh + EPL * lane;
  float v[EPL], w[EPL];
#pragma unroll
  for (int j = 0; j < EPL; j += 2) {
    const float2 p = unpack2(*reinterpret_cast<const uint32_t*>(xr + j), Tag{});
    const float2 q = unpack2(*reinterpret_cast<const uint32_t*>(a.w + EPL * lane + j), Tag{});
    v[j] = p.x;
    v[j + 1] = p.y;
    w[j] = q.x;
    w[j + 1] = q.y;
  }
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < EPL; ++j) ss += v[j] * v[j];
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) ss += __shfl_xor(ss, d, 64);
  const float r = rsqrtf(ss / float(D) + a.eps);
  uint32_t nb[EPL / 2];
#pragma unroll
  for (int j = 0; j < EPL; j += 2) {
    nb[j / 2] = pack_mul2(rounded(v[j] * r), 1.f + w[j], rounded(v[j + 1] * r), 1.f + w[j + 1], Tag{});
    *reinterpret_cast<uint32_t*>(sh + EPL * lane + j) = nb[j / 2];
  }
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const int half = a.rotary_dim / 2;
  const uint16_t* cr = a.rotary_dim > 0 ? a.cos + int64_t(t) * a.cs_st : nullptr;
  const uint16_t* sr = a.rotary_dim > 0 ? a.sin + int64_t(t) * a.cs_st : nullptr;
#pragma unroll
  for (int j = 0; j < EPL; j += 2) {
    const float2 own = unpack2(nb[j / 2], Tag{});
    float c2[2] = {1.f, 1.f}, p2[2] = {-0.f, -0.f};  // past the rotation: the value itself
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int i = EPL * lane + j + e;
      if (i < a.rotary_dim) {
        const int k = i < half ? i : i - half;          // cos/sin index
        const int pi = i < half ? i + half : i - half;  // rotation partner
        const uint16_t pb = sh[pi];
        const float partner = unpack2(uint32_t(pb), Tag{}).x;
        c2[e] = unpack2(uint32_t(cr[k]), Tag{}).x;
        p2[e] = partner_part(partner, unpack2(uint32_t(sr[k]), Tag{}).x, i < half);
      }
    }
    res[j / 2] = pack_fma2(own.x, c2[0], p2[0], own.y, c2[1], p2[1], Tag{});
  }
}

template <int D, typename Tag>
__global__ __launch_bounds__(256) void norm_rope_kernel(NormRopeArgs a) {
  constexpr int EPL = D / 64;
  __shared__ __align__(16) uint16_t sh[4][D];
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int64_t row = int64_t(blockIdx.x) * 4 + wave;
  if (row >= int64_t(a.n_tokens) * a.n_heads) return;  // uniform per wave
  const int t = int(row / a.n_heads);
  const int h = int(row % a.n_heads);
  uint32_t res[EPL / 2];
  norm_rope_row<D, Tag>(a, t, h, sh[wave], res);
  uint16_t* dst = a.out + int64_t(t) * a.o_st + int64_t(h) * a.o_sh + EPL * lane;
#pragma unroll
  for (int j = 0; j < EPL / 2; ++j) reinterpret_cast<uint32_t*>(dst)[j] = res[j];
}

// One launch for q, k and v of a step: rows [0, T*Hq) are q heads (to q_out), the next T*Hkv
// are k heads (to the k cache at their slots), the last T*Hkv are v heads (copied to the v cache).
struct StepArgs {
  NormRopeArgs q, k;
  const uint16_t* v;
  int64_t v_st, v_sh;
  uint16_t* v_cache;
  int32_t n_kv_heads;
};

template <int D, typename Tag>
__global__ __launch_bounds__(256) void norm_rope_append_vec_kernel(StepArgs a) {
  const uint32_t tokens = uint32_t(a.q.n_tokens), hq = uint32_t(a.q.n_heads),
                 hkv = uint32_t(a.n_kv_heads);
  const uint32_t nq = tokens * hq, nk = tokens * hkv;
  norm_rope_rows<D, Tag>(a.q, a.k.w, int64_t(nq) + 2 * int64_t(nk), [&](int64_t row) {
    uint32_t r = uint32_t(row);
    if (r < nq) {
      const uint32_t t = r / hq, h = r - t * hq;
      return RowJob{a.q.x + t * a.q.x_st + h * a.q.x_sh, a.q.out + t * a.q.o_st + h * a.q.o_sh,
                    int(t), 0};
    }
    r -= nq;
    const bool is_v = r >= nk;
    if (is_v) r -= nk;
    const uint32_t t = r / hkv, h = r - t * hkv;
    const int64_t slot = a.k.slots[t];
    const int64_t at = slot * a.k.cache_row + int64_t(h) * D;
    uint16_t* dst = slot < 0 || slot >= a.k.num_slots ? nullptr : (is_v ? a.v_cache : a.k.cache) + at;
    return RowJob{is_v ? a.v + t * a.v_st + h * a.v_sh : a.k.x + t * a.k.x_st + h * a.k.x_sh, dst,
                  int(t), is_v ? 2 : 1};
  });
}

template <int D, typename Tag>
__global__ __launch_bounds__(256) void norm_rope_append_kernel(StepArgs a) {
  constexpr int EPL = D / 64;
  __shared__ __align__(16) uint16_t sh[4][D];
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  int64_t row = int64_t(blockIdx.x) * 4 + wave;
  const int64_t nq = int64_t(a.q.n_tokens) * a.q.n_heads;
  const int64_t nk = int64_t(a.k.n_tokens) * a.k.n_heads;
  uint32_t res[EPL / 2];
  if (row < nq) {
    const int t = int(row / a.q.n_heads), h = int(row % a.q.n_heads);
    norm_rope_row<D, Tag>(a.q, t, h, sh[wave], res);
    uint16_t* dst = a.q.out + int64_t(t) * a.q.o_st + int64_t(h) * a.q.o_sh + EPL * lane;
#pragma unroll
    for (int j = 0; j < EPL / 2; ++j) reinterpret_cast<uint32_t*>(dst)[j] = res[j];
    return;
  }
  row -= nq;
  if (row < nk) {
    const int t = int(row / a.k.n_heads), h = int(row % a.k.n_heads);
    const int64_t slot = a.k.slots[t];
    norm_rope_row<D, Tag>(a.k, t, h, sh[wave], res);
    if (slot < 0 || slot >= a.k.num_slots) return;
    uint16_t* dst = a.k.cache + slot * a.k.cache_row + int64_t(h) * D + EPL * lane;
#pragma unroll
    for (int j = 0; j < EPL / 2; ++j) reinterpret_cast<uint32_t*>(dst)[j] = res[j];
    return;
  }
  row -= nk;
  if (row < nk) {
    const int t = int(row / a.n_kv_heads), h = int(row % a.n_kv_heads);
    const int64_t slot = a.k.slots[t];
    if (slot < 0 || slot >= a.k.num_slots) return;
    const uint16_t* src = a.v + int64_t(t) * a.v_st + int64_t(h) * a.v_sh + EPL * lane;
    uint16_t* dst = a.v_cache + slot * a.k.cache_row + int64_t(h) * D + EPL * lane;
#pragma unroll
    for (int j = 0; j < EPL / 2; ++j) {
      reinterpret_cast<uint32_t*>(dst)[j] = reinterpret_cast<const uint32_t*>(src)[j];
    }
  }
}

template <typename Tag>
__global__ __launch_bounds__(256) void sigmoid_mul_kernel(const uint32_t* a, const uint32_t* b,
                                                          uint32_t* out, int64_t n_pairs) {
  for (int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < n_pairs;
       i += int64_t(gridDim.x) * 256) {
    out[i] = gate_mul2(a[i], b[i], Tag{});
  }
}

bool rows_aligned(const void* p, int64_t st, int64_t sh) {
  return (reinterpret_cast<uintptr_t>(p) & 3) == 0 && st % 2 == 0 && sh % 2 == 0;
}

int check_common(int32_t n_tokens, int32_t head_dim, int32_t rotary_dim, int32_t dtype,
                 const char* who) {
  if (dtype != TI_DTYPE_BF16 && dtype != TI_DTYPE_F16) {
    return fail(TI_EUNSUPPORTED, "%s: dtype code %d is not bf16/fp16", who, dtype);
  }
  if (head_dim != 128 && head_dim != 256) {
    return fail(TI_EUNSUPPORTED, "%s: head_dim %d not built (128, 256)", who, head_dim);
  }
  if (n_tokens < 0 || rotary_dim < 0 || rotary_dim > head_dim || rotary_dim % 2 != 0) {
    return fail(TI_EINVAL, "%s: bad sizes tokens=%d rotary_dim=%d", who, n_tokens, rotary_dim);
  }
  return TI_OK;
}

unsigned row_blocks(int64_t rows) { return unsigned((rows + 3) / 4); }

// Rows of 16-byte vectors (norm_rope_vec_kernel): pointers and strides of 16 bytes.
bool vec_rows(const void* p, int64_t st, int64_t sh) {
  return (reinterpret_cast<uintptr_t>(p) & 15) == 0 && st % 8 == 0 && sh % 8 == 0;
}
// ... and rotations that pair whole vectors; row numbers are 32-bit there.
bool vec_rope(const void* w, const void* cos, const void* sin, int64_t cs_st, int32_t rotary_dim,
              int64_t rows) {
  return (reinterpret_cast<uintptr_t>(w) & 15) == 0 && rotary_dim % 16 == 0 &&
         (rotary_dim == 0 || (vec_rows(cos, cs_st, 0) && vec_rows(sin, cs_st, 0))) &&
         rows < (int64_t(1) << 31);
}
// Enough workgroups for every wave slot once (8 four-wave workgroups per CU); they walk the rest.
unsigned vec_blocks(int64_t rows, int32_t head_dim) {
  const int64_t want = ceil_div(rows, 4 * (64 / (head_dim / 8)));
  const int64_t cap = int64_t(device_cu_count()) * 8;
  return unsigned(want < cap ? want : cap);
}

}  // namespace
}  // namespace ti

extern "C" int ti_qknorm_rope(const void* x, int64_t x_stride_t, int64_t x_stride_h, void* out,
                              int64_t out_stride_t, int64_t out_stride_h, const void* weight,
                              const void* cos, const void* sin, int64_t cs_stride_t,
                              int32_t n_tokens, int32_t n_heads, int32_t head_dim,
                              int32_t rotary_dim, float eps, int32_t dtype, void* stream) {
  using namespace ti;
  int rc = check_common(n_tokens, head_dim, rotary_dim, dtype, "ti_qknorm_rope");
  if (rc != TI_OK) return rc;
  if (n_heads <= 0) return fail(TI_EINVAL, "ti_qknorm_rope: n_heads %d", n_heads);
  if (n_tokens == 0) return TI_OK;
  if (!x || !out || !weight || (rotary_dim > 0 && (!cos || !sin))) {
    return fail(TI_EINVAL, "ti_qknorm_rope: null pointer");
  }
  if (!rows_aligned(x, x_stride_t, x_stride_h) || !rows_aligned(out, out_stride_t, out_stride_h) ||
      (reinterpret_cast<uintptr_t>(weight) & 3)) {
    return fail(TI_EINVAL, "ti_qknorm_rope: rows must be 4-byte aligned");
  }
  NormRopeArgs a{};
  a.x = static_cast<const uint16_t*>(x);
  a.x_st = x_stride_t;
  a.x_sh = x_stride_h;
  a.out = static_cast<uint16_t*>(out);
  a.o_st = out_stride_t;
  a.o_sh = out_stride_h;
  a.w = static_cast<const uint16_t*>(weight);
  a.cos = static_cast<const uint16_t*>(cos);
  a.sin = static_cast<const uint16_t*>(sin);
  a.cs_st = cs_stride_t;
  a.n_tokens = n_tokens;
  a.n_heads = n_heads;
  a.rotary_dim = rotary_dim;
  a.eps = eps;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool bf16 = dtype == TI_DTYPE_BF16;
  const int64_t rows = int64_t(n_tokens) * n_heads;
  if (vec_rows(x, x_stride_t, x_stride_h) && vec_rows(out, out_stride_t, out_stride_h) &&
      vec_rope(weight, cos, sin, cs_stride_t, rotary_dim, rows)) {
    const dim3 vgrid(vec_blocks(rows, head_dim));
    if (head_dim == 256) {
      if (bf16) hipLaunchKernelGGL((norm_rope_vec_kernel<256, Bf16>), vgrid, dim3(256), 0, s, a);
      else hipLaunchKernelGGL((norm_rope_vec_kernel<256, F16>), vgrid, dim3(256), 0, s, a);
    } else {
      if (bf16) hipLaunchKernelGGL((norm_rope_vec_kernel<128, Bf16>), vgrid, dim3(256), 0, s, a);
      else hipLaunchKernelGGL((norm_rope_vec_kernel<128, F16>), vgrid, dim3(256), 0, s, a);
    }
    return check_launch("ti_qknorm_rope");
  }
  const dim3 grid(row_blocks(rows));
  if (head_dim == 256) {
    if (bf16) hipLaunchKernelGGL((norm_rope_kernel<256, Bf16>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((norm_rope_kernel<256, F16>), grid, dim3(256), 0, s, a);
  } else {
    if (bf16) hipLaunchKernelGGL((norm_rope_kernel<128, Bf16>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((norm_rope_kernel<128, F16>), grid, dim3(256), 0, s, a);
  }
  return check_launch("ti_qknorm_rope");
}

extern "C" int ti_qknorm_rope_append(
    const void* q, int64_t q_stride_t, int64_t q_stride_h, const void* k, int64_t k_stride_t,
    int64_t k_stride_h, const void* v, int64_t v_stride_t, int64_t v_stride_h,
    const void* q_weight, const void* k_weight, const void* cos, const void* sin,
    int64_t cs_stride_t, void* q_out, int64_t q_out_stride_t, int64_t q_out_stride_h,
    void* k_cache, void* v_cache, int64_t cache_row_stride, const int32_t* slot_mapping,
    int64_t num_slots, int32_t n_tokens, int32_t n_q_heads, int32_t n_kv_heads, int32_t head_dim,
    int32_t rotary_dim, float eps, int32_t dtype, void* stream) {
  using namespace ti;
  int rc = check_common(n_tokens, head_dim, rotary_dim, dtype, "ti_qknorm_rope_append");
  if (rc != TI_OK) return rc;
  if (n_q_heads <= 0 || n_kv_heads <= 0 || num_slots < 0 ||
      cache_row_stride < int64_t(n_kv_heads) * head_dim) {
    return fail(TI_EINVAL, "ti_qknorm_rope_append: bad heads/slots/row stride");
  }
  if (n_tokens == 0) return TI_OK;
  if (!q || !k || !v || !q_weight || !k_weight || !q_out || !k_cache || !v_cache ||
      !slot_mapping || (rotary_dim > 0 && (!cos || !sin))) {
    return fail(TI_EINVAL, "ti_qknorm_rope_append: null pointer");
  }
  if (!rows_aligned(q, q_stride_t, q_stride_h) || !rows_aligned(k, k_stride_t, k_stride_h) ||
      !rows_aligned(v, v_stride_t, v_stride_h) ||
      !rows_aligned(q_out, q_out_stride_t, q_out_stride_h) ||
      !rows_aligned(k_cache, cache_row_stride, 2) || !rows_aligned(v_cache, 2, 2)) {
    return fail(TI_EINVAL, "ti_qknorm_rope_append: rows must be 4-byte aligned");
  }
  StepArgs a{};
  a.q.x = static_cast<const uint16_t*>(q);
  a.q.x_st = q_stride_t;
  a.q.x_sh = q_stride_h;
  a.q.out = static_cast<uint16_t*>(q_out);
  a.q.o_st = q_out_stride_t;
  a.q.o_sh = q_out_stride_h;
  a.q.w = static_cast<const uint16_t*>(q_weight);
  a.q.cos = static_cast<const uint16_t*>(cos);
  a.q.sin = static_cast<const uint16_t*>(sin);
  a.q.cs_st = cs_stride_t;
  a.q.n_tokens = n_tokens;
  a.q.n_heads = n_q_heads;
  a.q.rotary_dim = rotary_dim;
  a.q.eps = eps;
  a.k = a.q;
  a.k.x = static_cast<const uint16_t*>(k);
  a.k.x_st = k_stride_t;
  a.k.x_sh = k_stride_h;
  a.k.out = nullptr;
  a.k.w = static_cast<const uint16_t*>(k_weight);
  a.k.n_heads = n_kv_heads;
  a.k.cache = static_cast<uint16_t*>(k_cache);
  a.k.cache_row = cache_row_stride;
  a.k.slots = slot_mapping;
  a.k.num_slots = num_slots;
  a.v = static_cast<const uint16_t*>(v);
  a.v_st = v_stride_t;
  a.v_sh = v_stride_h;
  a.v_cache = static_cast<uint16_t*>(v_cache);
  a.n_kv_heads = n_kv_heads;
  const int64_t rows = int64_t(n_tokens) * (n_q_heads + 2 * n_kv_heads);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool bf16 = dtype == TI_DTYPE_BF16;
  if (vec_rows(q, q_stride_t, q_stride_h) && vec_rows(k, k_stride_t, k_stride_h) &&
      vec_rows(v, v_stride_t, v_stride_h) && vec_rows(q_out, q_out_stride_t, q_out_stride_h) &&
      vec_rows(k_cache, cache_row_stride, 0) && vec_rows(v_cache, cache_row_stride, 0) &&
      vec_rows(k_weight, 0, 0) && vec_rope(q_weight, cos, sin, cs_stride_t, rotary_dim, rows)) {
    const dim3 vgrid(vec_blocks(rows, head_dim));
    if (head_dim == 256) {
      if (bf16) hipLaunchKernelGGL((norm_rope_append_vec_kernel<256, Bf16>), vgrid, dim3(256), 0, s, a);
      else hipLaunchKernelGGL((norm_rope_append_vec_kernel<256, F16>), vgrid, dim3(256), 0, s, a);
    } else {
      if (bf16) hipLaunchKernelGGL((norm_rope_append_vec_kernel<128, Bf16>), vgrid, dim3(256), 0, s, a);
      else hipLaunchKernelGGL((norm_rope_append_vec_kernel<128, F16>), vgrid, dim3(256), 0, s, a);
    }
    return check_launch("ti_qknorm_rope_append");
  }
  const dim3 grid(row_blocks(rows));
  if (head_dim == 256) {
    if (bf16) hipLaunchKernelGGL((norm_rope_append_kernel<256, Bf16>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((norm_rope_append_kernel<256, F16>), grid, dim3(256), 0, s, a);
  } else {
    if (bf16) hipLaunchKernelGGL((norm_rope_append_kernel<128, Bf16>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((norm_rope_append_kernel<128, F16>), grid, dim3(256), 0, s, a);
  }
  return check_launch("ti_qknorm_rope_append");
}

extern "C" int ti_sigmoid_mul(const void* a, const void* b, void* out, int64_t n, int32_t dtype,
                              void* stream) {
  using namespace ti;
  if (dtype != TI_DTYPE_BF16 && dtype != TI_DTYPE_F16) {
    return fail(TI_EUNSUPPORTED, "ti_sigmoid_mul: dtype code %d is not bf16/fp16", dtype);
  }
  if (n < 0 || n % 2 != 0) return fail(TI_EINVAL, "ti_sigmoid_mul: n=%lld must be even", (long long)n);
  if (n == 0) return TI_OK;
  if (!a || !b || !out) return fail(TI_EINVAL, "ti_sigmoid_mul: null pointer");
  if ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b) |
       reinterpret_cast<uintptr_t>(out)) & 3) {
    return fail(TI_EINVAL, "ti_sigmoid_mul: pointers must be 4-byte aligned");
  }
  const int64_t pairs = n / 2;
  const int64_t cap = int64_t(device_cu_count()) * 16;
  const int64_t want = (pairs + 255) / 256;
  const dim3 grid(unsigned(want < cap ? want : cap));
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == TI_DTYPE_BF16) {
    hipLaunchKernelGGL((sigmoid_mul_kernel<Bf16>), grid, dim3(256), 0, s,
                       static_cast<const uint32_t*>(a), static_cast<const uint32_t*>(b),
                       static_cast<uint32_t*>(out), pairs);
  } else {
    hipLaunchKernelGGL((sigmoid_mul_kernel<F16>), grid, dim3(256), 0, s,
                       static_cast<const uint32_t*>(a), static_cast<const uint32_t*>(b),
                       static_cast<uint32_t*>(out), pairs);
  }
  return check_launch("ti_sigmoid_mul");
}
