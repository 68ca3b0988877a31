// Token log-probs of 16-bit and float32 logits rows (losses.py:14-38), forward
// only: the row is read once and nothing is kept, so this is a pure stream.
//
// HBM reads bound it.  One workgroup owns one row and keeps four 16-byte loads
// per lane in flight: slab k is folded into the lane's running (max, sum of
// exp) and its register takes the load of slab k + 4 at once.  At 53 VGPRs
// eight waves share a SIMD (32 KB in flight per 512 lanes, 128 KB per CU), so
// one row's reduction and the next row's first latency hide behind other
// rows, and the hardware hands out rows as workgroups finish.  The generic
// kernel's plain loop folded each vector before asking for the next.
// Measured, generic kernel -> here: 8188 x 128256 bf16 395 -> 307 us
// (6.84 TB/s; depth 8 306, depth 12 300 but 65.7 against 49.0 at V = 16000),
// 4096 x 50257 f32 149 -> 118 us (7.0 TB/s), 8192 x 4096 bf16 27.5 -> 16.7 us,
// 16 x 128256 bf16 25.8 -> 10.9 us.
#include <hip/hip_runtime.h>

#include "slab_common.hpp"

namespace rrl {

namespace {

constexpr int DEPTH = 4;

template <class Tag, int NT>
__global__ __launch_bounds__(NT) void stream_fwd_kernel(RowArgs a) {
  using P = Pack16<Tag>;
  using S = typename Tag::S;
  constexpr int EPV = P::EPV;
  constexpr int ESZ = (int)sizeof(S);
  constexpr int NW = NT / 64;
  static_assert(NT >= kHeadLanes + EPV, "lanes for the head and the tail");
  __shared__ float sh_m[NW], sh_s[NW], sh_xt;

  const int tid = threadIdx.x;
  const uint32_t r = blockIdx.x;
  const uint32_t T32 = (uint32_t)a.T;
  const uint32_t b = r / T32, t = r - b * T32;
  const int64_t tgt = load_index(a.tgt.ptr, a.tgt.dt, b * a.tgt.sr + t * a.tgt.sc);
  const bool tgt_ok = tgt >= 0 && tgt < a.V;
  // A masked-out row (rrl_logprob_fwd_masked) is never read: 0 and 0.
  if (a.mask.present() && !a.mask.truth(b, t)) {
    if (tid == 0) {
      if (!tgt_ok) raise_flag(a.status, RRL_FLAG_TARGET_RANGE);
      store_as<float>(a.logp, a.logp_dt, r, 0.0f);
      static_cast<float*>(a.lse_out)[r] = 0.0f;
    }
    return;
  }
  const S* row = static_cast<const S*>(a.logits) + (int64_t)b * a.ls_b + (int64_t)t * a.ls_t;
  const uint32_t V32 = (uint32_t)a.V;
  const RowGeo g = row_geo<Tag, true>(row, V32, 0);
  const __amdgpu_buffer_rsrc_t src = row_rsrc(row + g.head, g.nbody * 16);
  const int voff = tid * 16;
  u32x4 x[DEPTH];
#pragma unroll
  for (int k = 0; k < DEPTH; ++k) {
    x[k] = __builtin_amdgcn_raw_buffer_load_b128(src, voff, k * NT * 16, kAuxLoad);
    __builtin_amdgcn_sched_barrier(0);
  }
  // Head and tail elements, one each in lanes 0-71.
  const int32_t ei = extra_index<Tag>(g, tid);
  const __amdgpu_buffer_rsrc_t esrc = row_rsrc(row, V32 * ESZ);
  const uint32_t xe = P::load_one(esrc, ei >= 0 ? ei * ESZ : (int)(V32 * ESZ));
  const int32_t tgt32 = tgt_ok ? (int32_t)tgt : -1;
  const int32_t bt = tgt32 - (int32_t)g.head;
  const bool in_body = tgt_ok && bt >= 0 && bt < (int32_t)(g.nbody * EPV);
  // Slab k of this lane holds the target iff rel == k * NT.
  const int rel = in_body ? (bt >> P::LOG2_EPV) - tid : -1;
  const int ti = bt & (EPV - 1);

  LaneLse acc{-__builtin_huge_valf(), 0.0f};
  const int nbody = (int)g.nbody;
  int base = 0;  // first vector of the slabs held
  for (; base + DEPTH * NT <= nbody; base += DEPTH * NT) {
#pragma unroll
    for (int k = 0; k < DEPTH; ++k) {
      fold_vector<Tag>(acc, x[k], rel == base + k * NT, ti, &sh_xt);
      x[k] = __builtin_amdgcn_raw_buffer_load_b128(src, voff, (base + (DEPTH + k) * NT) * 16,
                                                   kAuxLoad);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int k = 0; k < DEPTH; ++k)
    if (tid < nbody - base - k * NT)
      fold_vector<Tag>(acc, x[k], rel == base + k * NT, ti, &sh_xt);
  if (ei >= 0) fold_one(acc, P::one(xe), ei == tgt32, &sh_xt);
  if (!tgt_ok && tid == 0) sh_xt = -__builtin_huge_valf();
  const float Mw = wave_max_dpp(acc.m);
  const float Sw = wave_sum_dpp(rescale(acc.s, acc.m, Mw));
  if ((tid & 63) == 0) {
    sh_m[tid >> 6] = Mw;
    sh_s[tid >> 6] = Sw;
  }
  __syncthreads();
  if (tid != 0) return;
  float m = sh_m[0];
#pragma unroll
  for (int i = 1; i < NW; ++i) m = fmaxf(m, sh_m[i]);
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < NW; ++i) s += rescale(sh_s[i], sh_m[i], m);
  const RowLogprob<float> fr = finish_row<float>(m, s, sh_xt);
  if (!tgt_ok) raise_flag(a.status, RRL_FLAG_TARGET_RANGE);
  store_as<float>(a.logp, a.logp_dt, r, tgt_ok ? fr.logp : __builtin_nanf(""));
  static_cast<float*>(a.lse_out)[r] = fr.lse;
}

template <class Tag, int NT>
int launch_fwd(const RowArgs& a, hipStream_t stream) {
  hipLaunchKernelGGL((stream_fwd_kernel<Tag, NT>), dim3((unsigned)(a.B * a.T)), dim3(NT), 0, stream,
                     a);
  return check_launch("stream_fwd_kernel");
}

// Lanes per row: enough that a lane's loads fill its depth more than once,
// few enough that a CU holds several rows.  us at 128 / 256 / 512 / 1024
// lanes, 8192 rows bf16: V = 4096 16.7 / 18.0 / 26.7 / 45, V = 16000
// 47.1 / 46.0 / 49.0 / 64, V = 32000 82.9 / 81.4 / 80.0 / 92, 7161 rows of
// V = 50257 113 / 109 / 108 / 110.  Fewer rows than CUs leave nothing to share
// a CU with: 64 rows of V = 32000 take 6.7 / 6.1 / 5.6 us at 256 / 512 / 1024.
template <class Tag>
int dispatch_fwd(const RowArgs& a, hipStream_t stream) {
  const int64_t nvec = a.V / Pack16<Tag>::EPV;
  if (nvec <= 768) return launch_fwd<Tag, 128>(a, stream);
  if (nvec <= 3072) return launch_fwd<Tag, 256>(a, stream);
  if (a.B * a.T >= 256) return launch_fwd<Tag, 512>(a, stream);
  return launch_fwd<Tag, 1024>(a, stream);
}

}  // namespace

// Takes 16-bit and float32 rows of any alignment and stride whose bytes and
// number fit 31 bits; otherwise *launched stays false and the caller runs the
// generic row kernel (float64).
int maybe_launch_fwd(const RowArgs& a, int logits_dtype, hipStream_t stream, bool* launched) {
  *launched = false;
  const int64_t lim = (int64_t)1 << 31;
  if (a.B * a.T == 0 || a.B * a.T >= lim || a.T >= lim) return RRL_OK;
  if (a.V * (logits_dtype == RRL_F32 ? 4 : 2) >= lim - (1 << 20)) return RRL_OK;
  switch (logits_dtype) {
    case RRL_BF16: *launched = true; return dispatch_fwd<TagBF16>(a, stream);
    case RRL_F16: *launched = true; return dispatch_fwd<TagF16>(a, stream);
    case RRL_F32: *launched = true; return dispatch_fwd<TagF32>(a, stream);
    default: return RRL_OK;
  }
}

}  // namespace rrl
