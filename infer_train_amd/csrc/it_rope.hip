// it_rope.hip -- RoPE then append (src/inference/forward.rs:195-229): the
// rotary embedding of q and k (rope_f32, src/backend/arm/rope.rs:6-44) fused
// into the slot-mapped KV append, so the rotated K goes straight from the
// projection output into its cache page in the cache's format.
//
// The angles' cos/sin come from a table built on the host with the C
// library's float32 powf/cosf/sinf, in rope_f32's operation order, and held
// on the device: the device only multiplies and adds, so its results equal
// the CPU's bit for bit.  One lane rotates one 16-byte vector (two pairs) of
// one (token, head) row; K and V lanes then convert (or quantise: Q8_0,
// Q4_0, Q4_1, Q5_0, Q5_1) and store like the plain append, Q lanes write the
// rotated query.
#include <hip/hip_runtime.h>

#include <cmath>
#include <vector>

#include "it_device.hpp"
#include "it_internal.hpp"
#include "it_quant.hpp"

using namespace itkv;

struct it_rope_table {
  float2* table;  // device [max_pos][n_dims / 2]: (cos, sin)
  int32_t device;
  int32_t n_dims;
  int32_t max_pos;
  float freq_base;
};

namespace {
constexpr int kThreads = 256;
typedef float f32x4 __attribute__((ext_vector_type(4)));

struct RopeAppendArgs {
  const float4* q;
  const float4* k;
  const float4* v;
  void* q_out;
  char* kpool;
  char* vpool;
  const int64_t* slots;
  const int32_t* positions;
  const float2* table;
  int64_t n_tokens;
  int64_t page_bytes;
  int64_t n_slots;
  uint32_t* err;
  int hq, hkv, d, n_dims, max_pos, log2_bs, q_out_dtype;
};


// Four floats to the 16-bit format DT16 (IT_BF16 or IT_F16), packed.
template <int DT16>
__device__ __forceinline__ uint2 pack4(const float4& x) {
  auto cv = [](float f) { return DT16 == IT_BF16 ? f32_to_bf16_bits(f) : f16_bits_rne(f); };
  return make_uint2(cv(x.x) | (cv(x.y) << 16), cv(x.z) | (cv(x.w) << 16));
}


// rope.rs:38-39 on the pairs (x, y) and (z, w) with the table's (cos, sin):
// two products, each rounded, then their difference / sum -- no FMA.
__device__ __forceinline__ float4 rotate(float4 x, float2 cs0, float2 cs1, bool r0, bool r1) {
  float4 o = x;
  if (r0) {
    o.x = mul_rn(x.x, cs0.x) - mul_rn(x.y, cs0.y);
    o.y = mul_rn(x.x, cs0.y) + mul_rn(x.y, cs0.x);
  }
  if (r1) {
    o.z = mul_rn(x.z, cs1.x) - mul_rn(x.w, cs1.y);
    o.w = mul_rn(x.z, cs1.y) + mul_rn(x.w, cs1.x);
  }
  return o;
}

// grid.y: 0 = K, 1 = V, 2 = Q.  DT: the cache dtype.
template <int DT>
__global__ __launch_bounds__(kThreads) void kv_append_rope(RopeAppendArgs a) {
  const int part = blockIdx.y;
  const int H = part == 2 ? a.hq : a.hkv;
  const int vecs = a.d >> 2;
  const int64_t gid = int64_t(blockIdx.x) * kThreads + threadIdx.x;
  const int64_t total = a.n_tokens * H * vecs;
  const bool live = gid < total;
  const int cv = int(gid % vecs);
  const int64_t th = gid / vecs;
  const int h = int(th % H);
  const int64_t t = th / H;
  const float4* src = part == 0 ? a.k : (part == 1 ? a.v : a.q);
  float4 x = live ? src[gid] : make_float4(0.f, 0.f, 0.f, 0.f);
  // A token whose position is outside the table writes nothing (K, V or q).
  bool pos_ok = true;
  if (live) {
    const int pos = a.positions[t];
    pos_ok = pos >= 0 && pos < a.max_pos;
    if (!pos_ok) {
      if (cv == 0 && h == 0 && part == 0) atomicOr(a.err, kErrPos);
    } else if (part != 1) {
      // Elements 4 cv .. 4 cv + 3 are pairs 2 cv and 2 cv + 1.
      const int e0 = 4 * cv;
      const float2* row = a.table + int64_t(pos) * (a.n_dims >> 1) + 2 * cv;
      const bool r0 = e0 < a.n_dims, r1 = e0 + 2 < a.n_dims;
      const float2 cs0 = r0 ? row[0] : make_float2(1.f, 0.f);
      const float2 cs1 = r1 ? row[1] : make_float2(1.f, 0.f);
      x = rotate(x, cs0, cs1, r0, r1);
    }
  }
  if (part == 2) {
    if (!live || !pos_ok) return;
    if (a.q_out_dtype == IT_F32) static_cast<float4*>(a.q_out)[gid] = x;
    else if (a.q_out_dtype == IT_BF16) static_cast<uint2*>(a.q_out)[gid] = pack4<IT_BF16>(x);
    else static_cast<uint2*>(a.q_out)[gid] = pack4<IT_F16>(x);
    return;
  }
  if constexpr (DT == IT_Q8_0 || DT == IT_Q4_0 || DT == IT_Q4_1 || DT == IT_Q5_0 || DT == IT_Q5_1) {
    // Eight lanes own one 32-element group (rows of d/4 vectors, d % 32 ==
    // 0): the group's reductions run before any lane leaves.
    const QuantGroup qg = quant_group<DT>(x, cv & 7);
    if (!live || !pos_ok) return;
    const int64_t slot = a.slots[t];
    if (slot < 0) return;
    if (slot >= a.n_slots) {
      if (cv == 0 && h == 0) atomicOr(a.err, kErrSlot);
      return;
    }
    const int64_t blk = slot >> a.log2_bs;
    const int64_t off = slot & ((int64_t(1) << a.log2_bs) - 1);
    char* page = (part == 1 ? a.vpool : a.kpool) + (blk * a.hkv + h) * a.page_bytes;
    store_group<DT>(page, off, int64_t(1) << a.log2_bs, a.d, cv, qg);
  } else {
    if (!live || !pos_ok) return;
    const int64_t slot = a.slots[t];
    if (slot < 0) return;
    if (slot >= a.n_slots) {
      if (cv == 0 && h == 0) atomicOr(a.err, kErrSlot);
      return;
    }
    const int64_t blk = slot >> a.log2_bs;
    const int64_t off = slot & ((int64_t(1) << a.log2_bs) - 1);
    char* row = (part == 1 ? a.vpool : a.kpool) + (blk * a.hkv + h) * a.page_bytes;
    if constexpr (DT == IT_F32) {
      reinterpret_cast<float4*>(row + off * a.d * 4)[cv] = x;
    } else {
      reinterpret_cast<uint2*>(row + off * a.d * 2)[cv] = pack4<DT>(x);
    }
  }
}

// The same for rows of a power of two of 16-byte vectors, four up to a wave
// (head_dim 16, 32, 64, 128 or 256; other widths take the kernel above).  A wave
// takes one token: its position, slot and angles are read once and serve G
// instructions of RPI = 64 / vecs (token, head) rows each, q's, k's and v's heads
// numbered one after another; all rows are loaded before the first is stored.
// Bound by memory: 4096 tokens of 32 + 2 x 8 heads of 128, bf16 cache (151 MB):
// 28.8 us, 5.2 TB/s, a large copy's rate (one vector per lane, its (token, head)
// found by 64-bit divisions, in a grid of three parts each sized for q: 47.3 us).
// Two rows a lane 30.6, eight 30.9; without the non-temporal hint on the loads
// 30.8.  Small calls are a chain of waits, longer with each row: see launch_rope.
template <int DT, int G>
__global__ __launch_bounds__(kThreads) void kv_append_rope_rows(RopeAppendArgs a, int log2_vecs) {
  const int64_t t = int64_t(blockIdx.x) * (kThreads / 64) + __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  if (t >= a.n_tokens) return;  // uniform
  const int lane = int(threadIdx.x & 63), vecs = 1 << log2_vecs, cv = lane & (vecs - 1);
  const int rpi = 64 >> log2_vecs;
  const int rows = a.hq + 2 * a.hkv;
  const int row0 = int(blockIdx.y) * (rpi * G) + (lane >> log2_vecs);
  const int pos = a.positions[t];
  const int64_t slot = a.slots[t];
  // A token whose position is outside the table writes nothing (K, V or q).
  if (pos < 0 || pos >= a.max_pos) {
    if (blockIdx.y == 0 && lane == 0) atomicOr(a.err, kErrPos);
    return;
  }
  float4 x[G];
#pragma unroll
  for (int j = 0; j < G; ++j) {
    // Past the last row a lane re-reads it; only the stores are predicated.
    const int r = min(row0 + j * rpi, rows - 1);
    const int rk = r - a.hq, rv = rk - a.hkv;
    const float4* const src = rk < 0 ? a.q + ((t * a.hq + r) << log2_vecs)
                              : rv < 0 ? a.k + ((t * a.hkv + rk) << log2_vecs)
                                       : a.v + ((t * a.hkv + rv) << log2_vecs);
    const f32x4 f = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(src + cv));
    x[j] = make_float4(f.x, f.y, f.z, f.w);
  }
  // Elements 4 cv .. 4 cv + 3 are pairs 2 cv and 2 cv + 1.
  const bool r0 = 4 * cv < a.n_dims, r1 = 4 * cv + 2 < a.n_dims;
  const float2* const ang = a.table + int64_t(pos) * (a.n_dims >> 1) + 2 * cv;
  const float2 cs0 = r0 ? ang[0] : make_float2(1.f, 0.f);
  const float2 cs1 = r1 ? ang[1] : make_float2(1.f, 0.f);
  if (slot >= a.n_slots && blockIdx.y == 0 && lane == 0) atomicOr(a.err, kErrSlot);
  const int64_t blk = slot >> a.log2_bs;
  const int64_t off = slot & ((int64_t(1) << a.log2_bs) - 1);
  const bool cached = slot >= 0 && slot < a.n_slots;  // uniform
#pragma unroll
  for (int j = 0; j < G; ++j) {
    const int r = row0 + j * rpi;
    const int rk = r - a.hq, rv = rk - a.hkv;
    if (r >= rows) continue;
    const float4 y = rv < 0 ? rotate(x[j], cs0, cs1, r0, r1) : x[j];
    if (rk < 0) {
      const int64_t at = ((t * a.hq + r) << log2_vecs) + cv;
      if (a.q_out_dtype == IT_F32) static_cast<float4*>(a.q_out)[at] = y;
      else if (a.q_out_dtype == IT_BF16) static_cast<uint2*>(a.q_out)[at] = pack4<IT_BF16>(y);
      else static_cast<uint2*>(a.q_out)[at] = pack4<IT_F16>(y);
    } else if (cached) {
      char* const page = (rv < 0 ? a.kpool : a.vpool) + (blk * a.hkv + (rv < 0 ? rk : rv)) * a.page_bytes;
      if constexpr (DT == IT_Q8_0 || DT == IT_Q4_0 || DT == IT_Q4_1 || DT == IT_Q5_0 || DT == IT_Q5_1) {
        // The eight lanes of a 32-group hold the same row: all of them are here.
        store_group<DT>(page, off, int64_t(1) << a.log2_bs, a.d, cv, quant_group<DT>(y, cv & 7));
      } else if constexpr (DT == IT_F32) {
        reinterpret_cast<float4*>(page + off * a.d * 4)[cv] = y;
      } else {
        reinterpret_cast<uint2*>(page + off * a.d * 2)[cv] = pack4<DT>(y);
      }
    }
  }
}

template <int DT, int G>
void launch_rows(const RopeAppendArgs& a, int vecs, int64_t chunks, hipStream_t s) {
  const dim3 grid(unsigned((a.n_tokens + kThreads / 64 - 1) / (kThreads / 64)), unsigned(chunks));
  hipLaunchKernelGGL((kv_append_rope_rows<DT, G>), grid, dim3(kThreads), 0, s, a, ilog2(vecs));
}

// Rows per lane: one, two or four, the fewest with which all waves are resident
// at once (32 of 256 CUs).  us with one / two / four, bf16: one token of 32 + 2 x
// 8 heads of 128 2.23 / 2.61 / 3.31 (a vector per lane: 2.49), 128 tokens 2.79 /
// 3.11 / 3.98, 256 3.62 / 3.52 / 4.17, 512 5.54 / 4.93 / 5.19, 1024 9.34 / 8.51 /
// 7.97; Q8_0, 128 tokens 3.20 / 3.89 / 4.86, 1024 11.1 / 10.7 / 11.1.
constexpr int64_t kRopeWaves = 256 * 32;

template <int DT>
void launch_rope(const RopeAppendArgs& a, hipStream_t s) {
  const int vecs = a.d / 4;
  if (vecs >= 4 && vecs <= 64 && (vecs & (vecs - 1)) == 0) {
    const int64_t rows = int64_t(a.hq) + 2 * int64_t(a.hkv);
    const auto chunks = [&](int g) { return (rows + 64 / vecs * g - 1) / (64 / vecs * g); };  // waves per token
    if (chunks(1) <= 65535 && a.n_tokens * chunks(1) <= kRopeWaves) return launch_rows<DT, 1>(a, vecs, chunks(1), s);
    if (chunks(2) <= 65535 && a.n_tokens * chunks(2) <= kRopeWaves) return launch_rows<DT, 2>(a, vecs, chunks(2), s);
    if (chunks(4) <= 65535) return launch_rows<DT, 4>(a, vecs, chunks(4), s);
  }
  const int64_t blocks = (a.n_tokens * a.hq * vecs + kThreads - 1) / kThreads;  // Q has the most rows
  hipLaunchKernelGGL(kv_append_rope<DT>, dim3(unsigned(blocks), 3), dim3(kThreads), 0, s, a);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
}  // namespace

extern "C" int32_t it_rope_table_new(int32_t device, int32_t n_dims, float freq_base, int32_t max_pos,
                                     it_rope_table** out) {
  const char* who = "it_rope_table_new";
  if (!out) return fail(IT_INVALID_INPUT, "%s: out is NULL", who);
  *out = nullptr;
  if (n_dims <= 0 || n_dims % 4 || n_dims > 4096)
    return fail(IT_INVALID_INPUT, "%s: n_dims %d must be a positive multiple of 4 (<= 4096)", who, n_dims);
  if (max_pos <= 0) return fail(IT_INVALID_INPUT, "%s: max_pos %d", who, max_pos);
  if (!(freq_base > 0.0f) || !std::isfinite(freq_base))
    return fail(IT_INVALID_INPUT, "%s: freq_base must be positive and finite", who);
  const int pairs = n_dims / 2;
  // rope.rs:30-34, float32: theta = (float)pos * powf(base, -(float)i / (float)n_dims).
  std::vector<float> inv(pairs);
  for (int p = 0; p < pairs; ++p) inv[p] = powf(freq_base, -float(2 * p) / float(n_dims));
  std::vector<float2> host(size_t(max_pos) * pairs);
  for (int64_t pos = 0; pos < max_pos; ++pos)
    for (int p = 0; p < pairs; ++p) {
      const float theta = float(pos) * inv[p];
      host[size_t(pos) * pairs + p] = make_float2(cosf(theta), sinf(theta));
    }
  int prev = -1;
  (void)hipGetDevice(&prev);
  if (hipSetDevice(device) != hipSuccess) return fail(IT_DEVICE_ERROR, "%s: hipSetDevice(%d)", who, device);
  float2* dev = nullptr;
  hipError_t e = hipMalloc(&dev, host.size() * sizeof(float2));
  if (e == hipSuccess) e = hipMemcpy(dev, host.data(), host.size() * sizeof(float2), hipMemcpyHostToDevice);
  if (prev >= 0) (void)hipSetDevice(prev);
  if (e != hipSuccess) {
    if (dev) (void)hipFree(dev);
    return fail(IT_DEVICE_ERROR, "%s: %s", who, hipGetErrorString(e));
  }
  *out = new it_rope_table{dev, device, n_dims, max_pos, freq_base};
  return IT_OK;
}

extern "C" int32_t it_rope_table_destroy(it_rope_table* r) {
  if (!r) return IT_OK;
  int prev = -1;
  (void)hipGetDevice(&prev);
  (void)hipSetDevice(r->device);
  const hipError_t e = hipFree(r->table);
  if (prev >= 0) (void)hipSetDevice(prev);
  delete r;
  return e == hipSuccess ? IT_OK : fail(IT_DEVICE_ERROR, "it_rope_table_destroy: %s", hipGetErrorString(e));
}

extern "C" int32_t it_kv_append_rope(it_kv_cache* c, const it_rope_table* rope, const float* q, int32_t n_heads,
                                     const float* k, const float* v, const int64_t* slot_mapping,
                                     const int32_t* positions, int32_t n_tokens, void* q_out, int32_t q_out_dtype,
                                     void* stream) {
  const char* who = "it_kv_append_rope";
  if (!c || !rope) return fail(IT_INVALID_INPUT, "%s: cache or table is NULL", who);
  if (int32_t rc = one_layer(c, who)) return rc;
  if (n_tokens < 0) return fail(IT_INVALID_INPUT, "%s: n_tokens %d < 0", who, n_tokens);
  if (n_heads <= 0 || n_heads % c->n_kv_heads)
    return fail(IT_INVALID_INPUT, "%s: n_heads %d must be a positive multiple of n_kv_heads %d", who, n_heads,
                c->n_kv_heads);
  if (rope->n_dims > c->head_dim)
    return fail(IT_INVALID_INPUT, "%s: table n_dims %d > head_dim %d", who, rope->n_dims, c->head_dim);
  if (rope->device != c->device) return fail(IT_INVALID_INPUT, "%s: table and cache on different devices", who);
  const bool quant = is_quant(c->dtype);
  if (c->dtype != IT_F32 && c->dtype != IT_BF16 && c->dtype != IT_F16 && !quant)
    return fail(IT_NOT_IMPLEMENTED, "%s: cache dtype %d", who, c->dtype);
  const bool q_ok = q_out_dtype == IT_F32 || ((c->dtype == IT_BF16 || c->dtype == IT_F16) && q_out_dtype == c->dtype);
  if (!q_ok) return fail(IT_NOT_IMPLEMENTED, "%s: q_out dtype %d for cache dtype %d", who, q_out_dtype, c->dtype);
  if (c->head_dim % 4 || (quant && c->head_dim % 32))
    return fail(IT_NOT_IMPLEMENTED, "%s: head_dim %d", who, c->head_dim);
  if (n_tokens == 0) return IT_OK;
  if (!q || !k || !v || !slot_mapping || !positions || !q_out) return fail(IT_INVALID_INPUT, "%s: NULL tensor", who);
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(q_out))
    return fail(IT_INVALID_INPUT, "%s: q/k/v/q_out must be 16-byte aligned", who);
  RopeAppendArgs a{};
  a.q = reinterpret_cast<const float4*>(q);
  a.k = reinterpret_cast<const float4*>(k);
  a.v = reinterpret_cast<const float4*>(v);
  a.q_out = q_out;
  a.kpool = static_cast<char*>(c->k_pool);
  a.vpool = static_cast<char*>(c->v_pool);
  a.slots = slot_mapping;
  a.positions = positions;
  a.table = rope->table;
  a.n_tokens = n_tokens;
  a.page_bytes = c->page_bytes;
  a.n_slots = c->num_blocks * c->block_size;
  a.err = c->err_flag;
  a.hq = n_heads;
  a.hkv = c->n_kv_heads;
  a.d = c->head_dim;
  a.n_dims = rope->n_dims;
  a.max_pos = rope->max_pos;
  a.log2_bs = c->log2_bs;
  a.q_out_dtype = q_out_dtype;
  const int64_t vecs = int64_t(n_tokens) * n_heads * (c->head_dim / 4);  // Q has the most rows
  const int64_t blocks = (vecs + kThreads - 1) / kThreads;
  if (blocks > INT32_MAX) return fail(IT_INVALID_INPUT, "%s: too many tokens", who);
  int dev = -1;
  (void)hipGetDevice(&dev);
  if (dev != c->device) (void)hipSetDevice(c->device);
  hipStream_t s = (hipStream_t)stream;
  switch (c->dtype) {
    case IT_F32: launch_rope<IT_F32>(a, s); break;
    case IT_BF16: launch_rope<IT_BF16>(a, s); break;
    case IT_F16: launch_rope<IT_F16>(a, s); break;
    case IT_Q4_0: launch_rope<IT_Q4_0>(a, s); break;
    case IT_Q4_1: launch_rope<IT_Q4_1>(a, s); break;
    case IT_Q5_0: launch_rope<IT_Q5_0>(a, s); break;
    case IT_Q5_1: launch_rope<IT_Q5_1>(a, s); break;
    default: launch_rope<IT_Q8_0>(a, s); break;
  }
  const hipError_t e = hipGetLastError();
  if (dev >= 0 && dev != c->device) (void)hipSetDevice(dev);
  if (e != hipSuccess) return fail(IT_DEVICE_ERROR, "%s: launch: %s", who, hipGetErrorString(e));
  return IT_OK;
}
