// rrl_fused_logprob_policy for rows past the register-resident kernels' length
// (16-bit V > 163840, float32 V > 81920): log-prob, objective gradient and
// dlogits with one read of the row from HBM.
//
// HBM bounds it, and what to save is the second read: a 151936-entry float32
// row is 608 KB against a CU's 512 KB of registers and 160 KB of LDS, so one
// 512-lane workgroup per CU (two waves per SIMD, 256 VGPRs each) holds kRegs
// slabs of 16 bytes per lane in registers and kLds more in LDS, 508 KB
// together.  Only the slabs past those (97 KB of this row) are read again in
// sweep 2, while the memory-side cache still has them: all CUs' rests are
// 25 MB of its 256 MB.  The generic kernel, which took these rows before,
// reads every row twice.
//
// Per row: the register slabs were requested at the end of the row before;
// the others stream through kDepth more registers, folded as they land and
// kept in LDS where they fit.  After the reduction the register slabs become
// dlogits and are stored, the rest's second read goes into the freed
// registers while the LDS slabs are stored, then the rest, then the next
// row's register slabs are requested.  A lane reads back only LDS that it
// wrote itself, so the one barrier is the reduction's.
#include <hip/hip_runtime.h>

#include "slab_common.hpp"

namespace rrl {

int launch_pack_records(const RowArgs& a, hipStream_t stream);
int cu_count_of_current_device(int* n_out);

namespace {

constexpr int NT = 512;
constexpr int kRegs = 44;   // 176 VGPRs
constexpr int kLds = 18;    // 144 KB
constexpr int kDepth = 6;   // 24 VGPRs, 48 KB in flight per CU
constexpr int kGroup = 8;   // slabs per step of the second read
constexpr int kGroups = kRegs / kGroup;
constexpr int kAuxKeep = 0;  // temporal: the rest is read again

// What sweep 2 needs of a row, besides its data.
struct GradRow {
  float lse, lg;    // log-sum-exp and log2 |g|
  uint32_t sgn;     // sign bits to flip in every packed word
  float tgt_pre;    // the target column's gradient before the flip
  int ti;           // the target's element in its vector
};

// g * (onehot - exp(x - lse)) of one vector, packed.
template <class Tag>
__device__ __forceinline__ u32x4 grad_vector(const u32x4& u, const GradRow& q, bool is_target) {
  using P = Pack16<Tag>;
  constexpr int EPV = P::EPV;
  float v[EPV], d[EPV];
  P::unpack(u, v);
#pragma unroll
  for (int i = 0; i < EPV; ++i) d[i] = exp2_hw(__builtin_fmaf(v[i] - q.lse, kLog2e, q.lg));
  if (is_target) {
#pragma unroll
    for (int i = 0; i < EPV; ++i) d[i] = (i == q.ti) ? q.tgt_pre : d[i];
  }
  u32x4 o = P::pack(d);
  o.x ^= q.sgn; o.y ^= q.sgn; o.z ^= q.sgn; o.w ^= q.sgn;
  return o;
}

template <class Tag>
__global__ __launch_bounds__(NT, 2) void long_fused_kernel(RowArgs a) {
  using P = Pack16<Tag>;
  using S = typename Tag::S;
  constexpr int EPV = P::EPV;
  constexpr int ESZ = (int)sizeof(S);
  constexpr int NW = NT / 64;
  __shared__ u32x4 sh_row[kLds][NT];
  // Double-buffered by row parity: a wave can run at most one reduction ahead.
  __shared__ float sh_m[2][NW], sh_s[2][NW], sh_xt[2];
  int buf = 0;

  const int tid = threadIdx.x;
  const uint32_t rows32 = (uint32_t)(a.B * a.T), T32 = (uint32_t)a.T, V32 = (uint32_t)a.V;
  const int voff = tid * 16;
  const S* logits = static_cast<const S*>(a.logits);
  S* dl = static_cast<S*>(a.dl);
  const PolicyConsts<float> c = PolicyConsts<float>::make(a.pp);
  const bool skip_masked = (a.pp.flags & RRL_POLICY_SKIP_MASKED) != 0;
  uint32_t r = blockIdx.x;
  if (r >= rows32) return;

  auto row_ptr = [&](uint32_t rr) {
    const uint32_t bb = rr / T32, tt = rr - bb * T32;
    return logits + (int64_t)bb * a.ls_b + (int64_t)tt * a.ls_t;
  };
  auto extra_off = [&](const RowGeo& g) {
    const int32_t ei = extra_index<Tag>(g, tid);
    return ei >= 0 ? ei * ESZ : (int)(V32 * ESZ);
  };
  RowRecord rec_next = load_record(a, r, T32);
  u32x4 x[kRegs];
  uint32_t xe;
  {
    const bool skip0 = skip_masked && rec_next.wcoef() == 0.0f;
    const S* p0 = row_ptr(r);
    const RowGeo g0 = row_geo<Tag, true>(p0, V32, 0);
    const __amdgpu_buffer_rsrc_t src =
        skip0 ? row_rsrc(logits, 0u) : row_rsrc(p0 + g0.head, g0.nbody * 16);
#pragma unroll
    for (int k = 0; k < kRegs; ++k) {
      x[k] = __builtin_amdgcn_raw_buffer_load_b128(src, voff, k * NT * 16, kAuxLoad);
      __builtin_amdgcn_sched_barrier(0);
    }
    xe = P::load_one(skip0 ? row_rsrc(logits, 0u) : row_rsrc(p0, V32 * ESZ), extra_off(g0));
  }

  for (; r < rows32; r += gridDim.x) {
    const uint32_t b = r / T32, t = r - b * T32;
    int lane = tid;
    asm volatile("" : "+v"(lane));
    const S* row = row_ptr(r);
    const RowGeo g = row_geo<Tag, true>(row, V32, 0);
    const int32_t ei = extra_index<Tag>(g, tid);
    const RowRecord rec = rec_next;
    const bool skip = skip_masked && rec.wcoef() == 0.0f;
    const uint32_t rn = r + gridDim.x;
    const bool has_next = rn < rows32;
    if (has_next) rec_next = load_record(a, rn, T32);
    const int32_t tgt = rec.target;
    const bool tgt_ok = tgt >= 0;
    const int32_t bt = tgt - (int32_t)g.head;
    const int nbody = (int)g.nbody;
    const int nslab = (nbody + NT - 1) / NT;
    const bool in_body = tgt_ok && bt >= 0 && bt < nbody * EPV;
    const int rel = in_body ? (bt >> P::LOG2_EPV) - lane : -1;
    const int ti = bt & (EPV - 1);
    const bool ex_tgt = tgt_ok && ei == tgt;
    // A skipped row is never read: its descriptor covers 0 bytes.
    const __amdgpu_buffer_rsrc_t cur =
        skip ? row_rsrc(logits, 0u) : row_rsrc(row + g.head, g.nbody * 16);

    float m = -__builtin_huge_valf(), s = 0.0f, xt = 0.0f;
    if (!skip) {
      LaneLse acc{-__builtin_huge_valf(), 0.0f};
      u32x4 w[kDepth];
#pragma unroll
      for (int i = 0; i < kDepth; ++i) {
        w[i] = __builtin_amdgcn_raw_buffer_load_b128(cur, voff, (kRegs + i) * NT * 16, kAuxKeep);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int k = 0; k < kRegs; ++k)
        if (lane < nbody - k * NT)
          fold_vector<Tag>(acc, x[k], rel == k * NT, ti, &sh_xt[buf]);
      // The slabs past the registers: into LDS, then folded only.
#pragma unroll 1
      for (int j = kRegs; j < nslab; j += kDepth) {
        const bool keep = j < kRegs + kLds;
#pragma unroll
        for (int i = 0; i < kDepth; ++i) {
          if (lane < nbody - (j + i) * NT)
            fold_vector<Tag>(acc, w[i], rel == (j + i) * NT, ti, &sh_xt[buf]);
          if (keep) sh_row[j - kRegs + i][tid] = w[i];
          w[i] = __builtin_amdgcn_raw_buffer_load_b128(cur, voff, (j + kDepth + i) * NT * 16,
                                                       kAuxKeep);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if (ei >= 0) fold_one(acc, P::one(xe), ex_tgt, &sh_xt[buf]);
      if (!tgt_ok && tid == 0) sh_xt[buf] = -__builtin_huge_valf();
      const float Mw = wave_max_dpp(acc.m);
      const float Sw = wave_sum_dpp(rescale(acc.s, acc.m, Mw));
      if ((tid & 63) == 0) {
        sh_m[buf][tid >> 6] = Mw;
        sh_s[buf][tid >> 6] = Sw;
      }
      lds_barrier();
      m = sh_m[buf][0];
#pragma unroll
      for (int i = 1; i < NW; ++i) m = fmaxf(m, sh_m[buf][i]);
#pragma unroll
      for (int i = 0; i < NW; ++i) s += rescale(sh_s[buf][i], sh_m[buf][i], m);
      xt = sh_xt[buf];
      buf ^= 1;
    }
    // Opaque: sweep 2 expands the packed slabs again instead of keeping sweep
    // 1's widened copies.
#pragma unroll
    for (int k = 0; k < kRegs; ++k) asm volatile("" : "+v"(x[k]));
    asm volatile("" : "+v"(xe));

    const RowLogprob<float> fr = finish_row<float>(m, s, xt);
    GradRow q;
    q.lse = skip ? 0.0f : fr.lse;
    const float logp = skip ? 0.0f : (tgt_ok ? fr.logp : __builtin_nanf(""));
    const float gr =
        skip ? 0.0f : -(rec.wcoef() * token_local_grad<float>(c, logp, rec.old, rec.adv));
    const float tgt_d = target_grad<float>(gr, logp, true, xt, q.lse);
    if (tid == 0) {
      store_as<float>(a.logp, a.logp_dt, r, logp);
      static_cast<float*>(a.lse_out)[r] = q.lse;
    }
    // The difference x - lse is formed first, so no finite lse overflows and
    // 16-bit rows need no rerun.
    q.lg = __log2f(fabsf(gr));
    const bool flip = gr > 0.0f;
    q.sgn = flip ? P::SGN2 : 0u;
    q.tgt_pre = flip ? -tgt_d : tgt_d;
    q.ti = ti;
    const S* drow = dl + (int64_t)b * a.ds_b + (int64_t)t * a.ds_t;
    const __amdgpu_buffer_rsrc_t dst = row_rsrc(drow + g.head, g.nbody * 16);
    auto put = [&](const u32x4& u, int slab) __attribute__((always_inline)) {
      const u32x4 o = grad_vector<Tag>(u, q, rel == slab * NT);
      store_b128_nt(o, dst, voff, slab * NT * 16);
    };
#pragma unroll
    for (int k = 0; k < kRegs; ++k) put(x[k], k);
    {
      const float dv =
          ex_tgt ? q.tgt_pre : exp2_hw(__builtin_fmaf(P::one(xe) - q.lse, kLog2e, q.lg));
      P::store_one(P::pack_one(dv) ^ (flip ? P::SGN1 : 0u), row_rsrc(drow, V32 * ESZ),
                   extra_off(g));
    }
    auto put_lds = [&]() __attribute__((always_inline)) {
      const int n = nslab - kRegs < kLds ? nslab - kRegs : kLds;
#pragma unroll 2
      for (int l = 0; l < n; ++l) {
        u32x4 u = sh_row[l][tid];
        if (skip) u = u32x4{0u, 0u, 0u, 0u};  // not written for a skipped row
        put(u, kRegs + l);
      }
    };
    if (nslab <= kRegs + kLds) put_lds();
#pragma unroll 1
    for (int s0 = kRegs + kLds; s0 < nslab; s0 += kGroups * kGroup) {
#pragma unroll
      for (int q0 = 0; q0 < kGroups; ++q0) {
        if (s0 + q0 * kGroup < nslab) {
#pragma unroll
          for (int i = 0; i < kGroup; ++i) {
            x[q0 * kGroup + i] = __builtin_amdgcn_raw_buffer_load_b128(
                cur, voff, (s0 + q0 * kGroup + i) * NT * 16, kAuxKeep);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
      if (s0 == kRegs + kLds) put_lds();
#pragma unroll
      for (int q0 = 0; q0 < kGroups; ++q0) {
        if (s0 + q0 * kGroup < nslab) {
#pragma unroll
          for (int i = 0; i < kGroup; ++i) put(x[q0 * kGroup + i], s0 + q0 * kGroup + i);
        }
      }
    }
    const bool load_next = has_next && !(skip_masked && rec_next.wcoef() == 0.0f);
    const S* pn = row_ptr(load_next ? rn : r);
    const RowGeo gn = row_geo<Tag, true>(pn, V32, 0);
    const __amdgpu_buffer_rsrc_t src =
        load_next ? row_rsrc(pn + gn.head, gn.nbody * 16) : row_rsrc(logits, 0u);
#pragma unroll
    for (int k = 0; k < kRegs; ++k) {
      x[k] = __builtin_amdgcn_raw_buffer_load_b128(src, voff, k * NT * 16, kAuxLoad);
      __builtin_amdgcn_sched_barrier(0);
    }
    xe = P::load_one(load_next ? row_rsrc(pn, V32 * ESZ) : row_rsrc(logits, 0u), extra_off(gn));
  }
}

template <class Tag>
int launch_long(const RowArgs& a, hipStream_t stream) {
  int cus = 0;
  if (int rc = cu_count_of_current_device(&cus)) return rc;
  if (int rc = launch_pack_records(a, stream)) return rc;
  const int64_t rows = a.B * a.T;
  const unsigned grid = (unsigned)(rows < cus ? rows : cus);
  hipLaunchKernelGGL((long_fused_kernel<Tag>), dim3(grid), dim3(NT), 0, stream, a);
  return check_launch("long_fused_kernel");
}

}  // namespace

int launch_long_fused(const RowArgs& a, int logits_dtype, hipStream_t stream) {
  switch (logits_dtype) {
    case RRL_BF16: return launch_long<TagBF16>(a, stream);
    case RRL_F16: return launch_long<TagF16>(a, stream);
    default: return launch_long<TagF32>(a, stream);
  }
}

}  // namespace rrl
