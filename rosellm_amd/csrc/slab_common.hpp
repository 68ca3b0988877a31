// Rows as 16-byte slabs held by a workgroup's lanes: element access, a row's
// split into head, body and tail, and the pieces of the online (max, sum of
// exp) reduction.  Shared by the register-resident kernels
// (logprob_resident.hip) and the streaming forward (logprob_fwd.hip).
#pragma once

#include "policy_math.hpp"
#include "row_common.hpp"
#include "wave_common.hpp"

namespace rrl {
namespace {

// Element access of one 16-byte vector per tag: EPV elements, their float
// values, the packed form written back (round to nearest even for 16-bit),
// the sign bit of every element of a dword, and the single-element loads and
// non-temporal stores of a row's unaligned head and tail.
template <class Tag> struct Pack16;
template <> struct Pack16<TagBF16> {
  static constexpr int EPV = 8, LOG2_EPV = 3;
  static constexpr uint32_t SGN2 = 0x80008000u, SGN1 = 0x8000u;
  static __device__ __forceinline__ void unpack(const u32x4& u, float (&x)[8]) {
    x[0] = __uint_as_float(u.x << 16); x[1] = __uint_as_float(u.x & 0xffff0000u);
    x[2] = __uint_as_float(u.y << 16); x[3] = __uint_as_float(u.y & 0xffff0000u);
    x[4] = __uint_as_float(u.z << 16); x[5] = __uint_as_float(u.z & 0xffff0000u);
    x[6] = __uint_as_float(u.w << 16); x[7] = __uint_as_float(u.w & 0xffff0000u);
  }
  static __device__ __forceinline__ u32x4 pack(const float (&d)[8]) {
    u32x4 o;
    o.x = f32x2_to_bf16x2_bits(d[0], d[1]);
    o.y = f32x2_to_bf16x2_bits(d[2], d[3]);
    o.z = f32x2_to_bf16x2_bits(d[4], d[5]);
    o.w = f32x2_to_bf16x2_bits(d[6], d[7]);
    return o;
  }
  static __device__ __forceinline__ float one(uint32_t b) { return __uint_as_float(b << 16); }
  static __device__ __forceinline__ uint32_t pack_one(float d) { return f32_to_bf16_bits(d); }
  static __device__ __forceinline__ uint32_t load_one(__amdgpu_buffer_rsrc_t r, int off) {
    return __builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0);
  }
  static __device__ __forceinline__ void store_one(uint32_t b, __amdgpu_buffer_rsrc_t r, int off) {
    __builtin_amdgcn_raw_buffer_store_b16((unsigned short)b, r, off, 0, kAuxStoreNT);
  }
};
template <> struct Pack16<TagF16> {
  static constexpr int EPV = 8, LOG2_EPV = 3;
  static constexpr uint32_t SGN2 = 0x80008000u, SGN1 = 0x8000u;
  static __device__ __forceinline__ void unpack(const u32x4& u, float (&x)[8]) {
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[2 * i] = f16_bits_to_f32((uint16_t)(w[i] & 0xffffu));
      x[2 * i + 1] = f16_bits_to_f32((uint16_t)(w[i] >> 16));
    }
  }
  static __device__ __forceinline__ u32x4 pack(const float (&d)[8]) {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      w[i] = (uint32_t)f32_to_f16_bits(d[2 * i]) | ((uint32_t)f32_to_f16_bits(d[2 * i + 1]) << 16);
    u32x4 o;
    o.x = w[0]; o.y = w[1]; o.z = w[2]; o.w = w[3];
    return o;
  }
  static __device__ __forceinline__ float one(uint32_t b) {
    return f16_bits_to_f32((uint16_t)(b & 0xffffu));
  }
  static __device__ __forceinline__ uint32_t pack_one(float d) { return f32_to_f16_bits(d); }
  static __device__ __forceinline__ uint32_t load_one(__amdgpu_buffer_rsrc_t r, int off) {
    return __builtin_amdgcn_raw_buffer_load_b16(r, off, 0, 0);
  }
  static __device__ __forceinline__ void store_one(uint32_t b, __amdgpu_buffer_rsrc_t r, int off) {
    __builtin_amdgcn_raw_buffer_store_b16((unsigned short)b, r, off, 0, kAuxStoreNT);
  }
};
template <> struct Pack16<TagF32> {
  static constexpr int EPV = 4, LOG2_EPV = 2;
  static constexpr uint32_t SGN2 = 0x80000000u, SGN1 = 0x80000000u;
  static __device__ __forceinline__ void unpack(const u32x4& u, float (&x)[4]) {
    x[0] = __uint_as_float(u.x); x[1] = __uint_as_float(u.y);
    x[2] = __uint_as_float(u.z); x[3] = __uint_as_float(u.w);
  }
  static __device__ __forceinline__ u32x4 pack(const float (&d)[4]) {
    u32x4 o;
    o.x = __float_as_uint(d[0]); o.y = __float_as_uint(d[1]);
    o.z = __float_as_uint(d[2]); o.w = __float_as_uint(d[3]);
    return o;
  }
  static __device__ __forceinline__ float one(uint32_t b) { return __uint_as_float(b); }
  static __device__ __forceinline__ uint32_t pack_one(float d) { return __float_as_uint(d); }
  static __device__ __forceinline__ uint32_t load_one(__amdgpu_buffer_rsrc_t r, int off) {
    return __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
  }
  static __device__ __forceinline__ void store_one(uint32_t b, __amdgpu_buffer_rsrc_t r, int off) {
    __builtin_amdgcn_raw_buffer_store_b32(b, r, off, 0, kAuxStoreNT);
  }
};

// A row as the resident kernels hold it: `head` single elements up to the
// first 128-byte boundary, `nbody` 16-byte vectors (the register slabs), then
// `tail` single elements.  The body starts on a 128-byte boundary so that
// each wave's 1 KB run of vector stores covers whole cache lines: runs that
// share a partly written line with the next wave's run cost up to 10% of the
// write rate.  head < 128 / element size (at most 63) and tail <= EPV - 1,
// so lanes 0-63 carry the head and lanes 64-71 the tail in one extra
// register.  Without EXTRAS every row is 16-byte aligned with V % EPV == 0:
// head = tail = 0 and nbody is the same for every row.
constexpr uint32_t kBodyAlign = 128;
constexpr int kHeadLanes = 64;

struct RowGeo {
  uint32_t head, nbody, tail;
};

template <class Tag, bool EXTRAS>
__device__ __forceinline__ RowGeo row_geo(const void* row, uint32_t V, int32_t nvec) {
  constexpr uint32_t EPV = Pack16<Tag>::EPV, ESZ = 16 / EPV;
  RowGeo g;
  if constexpr (EXTRAS) {
    const uint32_t mis = (uint32_t)(reinterpret_cast<uintptr_t>(row) & (kBodyAlign - 1u));
    uint32_t h = mis ? (kBodyAlign - mis) / ESZ : 0u;
    h = h < V ? h : V;
    const uint32_t rem = V - h;
    g.head = h;
    g.nbody = rem / EPV;
    g.tail = rem - g.nbody * EPV;
  } else {
    g.head = 0;
    g.nbody = (uint32_t)nvec;
    g.tail = 0;
  }
  return g;
}

// Vocabulary index of the extra element lane `tid` carries, or -1.
template <class Tag>
__device__ __forceinline__ int32_t extra_index(const RowGeo& g, int tid) {
  constexpr int EPV = Pack16<Tag>::EPV;
  if (tid < kHeadLanes) return tid < (int)g.head ? tid : -1;
  if (tid < kHeadLanes + EPV)
    return tid - kHeadLanes < (int)g.tail ? (int)(g.head + g.nbody * EPV) + tid - kHeadLanes : -1;
  return -1;
}

// s * exp(m - M) for the combine: exact s when m == M (also for M = -inf or
// +inf, where m - M is NaN), 0 for m = -inf below a finite M.
__device__ __forceinline__ float rescale(float s, float m, float M) {
  return m == M ? s : s * exp2_hw((m - M) * kLog2e);
}

// Balanced max / sum of the EPV values of one vector.
template <int N>
__device__ __forceinline__ float vmax(const float (&v)[N]) {
  if constexpr (N == 8)
    return fmaxf(fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])),
                 fmaxf(fmaxf(v[4], v[5]), fmaxf(v[6], v[7])));
  else
    return fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3]));
}
template <int N>
__device__ __forceinline__ float vsum(const float (&e)[N]) {
  if constexpr (N == 8)
    return ((e[0] + e[1]) + (e[2] + e[3])) + ((e[4] + e[5]) + (e[6] + e[7]));
  else
    return (e[0] + e[1]) + (e[2] + e[3]);
}

// Lane-private running (max, sum exp(x - max)) over the non-target columns.
// The running max starts at -inf; the exponent offset is kept finite so that
// -inf entries contribute exp(-inf) = 0 rather than exp(-inf + inf) = NaN,
// while NaN and +inf still poison the row as in log_softmax.
struct LaneLse {
  float m, s;
};

// Folds one vector of a row in.  `is_target`: this lane's vector holds the
// target at element ti, which joins the max, stays out of the sum and goes to
// *xt_slot.
template <class Tag>
__device__ __forceinline__ void fold_vector(LaneLse& q, const u32x4& u, bool is_target, int ti,
                                            float* xt_slot) {
  constexpr int EPV = Pack16<Tag>::EPV;
  float v[EPV];
  Pack16<Tag>::unpack(u, v);
  const float mn = fmaxf(q.m, vmax(v));
  const float mg = fmaxf(mn, -__FLT_MAX__);
  float e[EPV];
#pragma unroll
  for (int i = 0; i < EPV; ++i) e[i] = exp2_hw((v[i] - mg) * kLog2e);
  float se = vsum(e);
  if (is_target) {
    float xv = v[0], so = 0.0f;
#pragma unroll
    for (int i = 0; i < EPV; ++i) {
      xv = (i == ti) ? v[i] : xv;
      so += (i == ti) ? 0.0f : e[i];
    }
    se = so;
    *xt_slot = xv;
  }
  q.s = __builtin_fmaf(q.s, exp2_hw((q.m - mg) * kLog2e), se);
  q.m = mn;
}

// The same for a single head or tail element.
__device__ __forceinline__ void fold_one(LaneLse& q, float v, bool is_target, float* xt_slot) {
  const float mn = fmaxf(q.m, v);
  const float mg = fmaxf(mn, -__FLT_MAX__);
  const float ev = is_target ? 0.0f : exp2_hw((v - mg) * kLog2e);
  if (is_target) *xt_slot = v;
  q.s = __builtin_fmaf(q.s, exp2_hw((q.m - mg) * kLog2e), ev);
  q.m = mn;
}

// The records and row coefficients are read-only for the sweep, so they come through
// the scalar data cache: a uniform load from the constant address space is a
// single s_load_dwordx4, waited on with lgkmcnt and never behind the
// vector-memory queue of slab loads and stores.
struct RowRecord {
  int32_t target;
  float old, adv;
  float weight, coef;
  // Mask weight * row coefficient, formed where it is used: forming it where
  // the record is requested would wait for the loads at the top of every row.
  __device__ __forceinline__ float wcoef() const { return weight_coef(weight, coef); }
};
__device__ __forceinline__ RowRecord load_record(const RowArgs& a, uint32_t r, uint32_t T32) {
  typedef __attribute__((address_space(4))) const u32x4 ConstWords;
  typedef __attribute__((address_space(4))) const float ConstFloat;
  const u32x4 q = reinterpret_cast<ConstWords*>(reinterpret_cast<uintptr_t>(a.records))[r];
  RowRecord rec;
  rec.target = (int32_t)q.x;
  rec.old = __uint_as_float(q.y);
  rec.adv = __uint_as_float(q.z);
  rec.weight = __uint_as_float(q.w);
  rec.coef = reinterpret_cast<ConstFloat*>(reinterpret_cast<uintptr_t>(a.row_coef))[r / T32];
  return rec;
}

}  // namespace
}  // namespace rrl
