// Register-resident 16-bit row kernels: the fast path of
// rrl_fused_logprob_policy (log-prob + token-local objective gradient in one
// read of the logits, losses.py:14-38 composed with :426-486 / :127-203 /
// :355-423), and of rrl_logprob_bwd (resident_bwd_kernel, the backward of
// losses.py:34-38 given the forward's lse and log-probs).
//
// Layout and schedule (gfx950, wave64):
//   * A persistent grid of NT-lane workgroups, as many as fit the CUs, walks
//     rows r = blockIdx.x, blockIdx.x + gridDim.x, ...  NT runs from 64 (short
//     rows, many of them per CU) to 1024 (one row per CU); see launch_variant.
//   * A row of V 16-bit logits is held in VGPRs as SL slabs of one 16-byte
//     vector per lane: slab k, lane j holds vector k*NT + j.  V = 151936
//     (bf16) is 18992 vectors, 19 slabs of 1024 lanes, i.e. 76 VGPRs.
//   * Per-row scalars (target, old log-prob, advantage, mask weight) come from
//     a packed 16-byte record per token (pack_records_kernel, or
//     rrl_policy_prepare), the row coefficient from its array, both read a row
//     ahead through the scalar cache.
//   * Sweep 1 (registers only): online max / sum of exp over the non-target
//     columns per lane, slab by slab as the loads land, then one LDS combine
//     across the workgroup's waves.
//   * Sweep 2: each slab becomes g * (onehot - exp(x - lse)), is packed back to
//     16 bits and stored with a non-temporal buffer store; once the whole row
//     is stored, the same registers are refilled with the workgroup's next
//     row, so the next row's HBM reads overlap the drain of this row's stores.
// Every access is a raw buffer load/store whose descriptor covers exactly one
// row, so a lane past the end of the row reads zeros and its stores are
// dropped by the hardware range check.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "slab_common.hpp"

namespace rrl {

int launch_long_fused(const RowArgs& a, int logits_dtype, hipStream_t stream);

namespace {

constexpr int kMaxSlabs = 20;       // slabs per lane: 80 VGPRs of the 128 at 4 waves per SIMD
constexpr int kWavesPerSimd = 4;
constexpr uint32_t kFmaLse = 0x43000000u;  // 128.0f: up to here the one-FMA exponent keeps 5e-6

// Per-token records for the resident kernel (TokenRecord): the views' dtype
// and stride handling happens here, once per token, so that the row loop reads
// its scalars with one uniform 16-byte load.
__global__ __launch_bounds__(256) void pack_records_kernel(RowArgs a) {
  const PolicyConsts<float> c = PolicyConsts<float>::make(a.pp);
  TokenRecord* rec = static_cast<TokenRecord*>(a.records);
  const int64_t n = a.B * a.T;
  for (int64_t i = blockIdx.x * (int64_t)256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const int64_t b = i / a.T, t = i - (i / a.T) * a.T;
    const int64_t tgt = load_index(a.tgt.ptr, a.tgt.dt, b * a.tgt.sr + t * a.tgt.sc);
    const bool ok = tgt >= 0 && tgt < a.V;
    if (!ok && !target_ignored(c, tgt)) raise_flag(a.status, RRL_FLAG_TARGET_RANGE);
    TokenRecord r;
    r.target = ok ? (int32_t)tgt : -1;
    r.old = a.old.get<float>(b, t);
    r.adv = a.adv.get<float>(b, t);
    r.weight = mask_weight<float>(c, a.mask, b, t);
    rec[i] = r;
  }
}

template <class Tag, int NT, int SL, bool EXTRAS>
__global__ __launch_bounds__(NT, kWavesPerSimd) void resident_fused_kernel(RowArgs a, int32_t nvec) {
  using P = Pack16<Tag>;
  using S = typename Tag::S;
  constexpr int EPV = P::EPV;
  constexpr int ESZ = (int)sizeof(S);
  // Double-buffered by combine parity: a wave can run at most one combine
  // ahead of the slowest (each combine has one barrier), so the buffer it
  // writes is never the one another wave is still reading.
  __shared__ float sh_m[2][NT / 64];
  __shared__ float sh_s[2][NT / 64];
  __shared__ float sh_xt[2];
  int buf = 0;

  const int tid = threadIdx.x;
  const int64_t rows = a.B * a.T;
  const uint32_t V32 = (uint32_t)a.V;
  const int voff = tid * 16;
  const S* logits = static_cast<const S*>(a.logits);
  S* dl = static_cast<S*>(a.dl);
  const PolicyConsts<float> c = PolicyConsts<float>::make(a.pp);
  // Row indices fit in 32 bits (checked on the host); 32-bit division keeps the
  // per-row address arithmetic short.
  const uint32_t T32 = (uint32_t)a.T;
  const uint32_t rows32 = (uint32_t)rows;
  uint32_t r = blockIdx.x;
  if (r >= rows32) return;

  auto row_ptr = [&](uint32_t rr) {
    const uint32_t bb = rr / T32, tt = rr - bb * T32;
    return logits + (int64_t)bb * a.ls_b + (int64_t)tt * a.ls_t;
  };
  // The extra element of this lane (EXTRAS): its byte offset in the row, or
  // the row's end (out of range: loads return 0, stores are dropped).
  auto extra_off = [&](const RowGeo& g) {
    const int32_t ei = extra_index<Tag>(g, tid);
    return ei >= 0 ? ei * ESZ : (int)(V32 * ESZ);
  };
  // RRL_POLICY_SKIP_MASKED: rows whose weight is exactly 0 are never read
  // (their loads use a 0-byte descriptor: no memory traffic) and get zero
  // dlogits and log-prob 0.
  const bool skip_masked = (a.pp.flags & RRL_POLICY_SKIP_MASKED) != 0;
  RowRecord rec_next = load_record(a, r, T32);
  u32x4 x[SL];
  uint32_t xe = 0;  // EXTRAS: the lane's head or tail element, as stored
  {
    const bool skip0 = skip_masked && rec_next.wcoef() == 0.0f;
    const S* p0 = row_ptr(r);
    const RowGeo g0 = row_geo<Tag, EXTRAS>(p0, V32, nvec);
    const __amdgpu_buffer_rsrc_t src = skip0 ? row_rsrc(logits, 0u) : row_rsrc(p0 + g0.head, g0.nbody * 16);
    // Issue in slab order, the order sweep 2 refills them: with one order on
    // both paths into the row loop, sweep 1 waits for slab k only (older
    // loads), not for the whole row.
#pragma unroll
    for (int k = 0; k < SL; ++k) {
      x[k] = __builtin_amdgcn_raw_buffer_load_b128(src, voff, k * NT * 16, kAuxLoad);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (EXTRAS) {
      const __amdgpu_buffer_rsrc_t esrc = skip0 ? row_rsrc(logits, 0u) : row_rsrc(p0, V32 * ESZ);
      xe = P::load_one(esrc, extra_off(g0));
    }
  }

  for (; r < rows32; r += gridDim.x) {
    const uint32_t b = r / T32, t = r - b * T32;
    // An opaque per-row copy of the lane id: the per-slab compares below are
    // then recomputed each row instead of being hoisted (and spilled) as 2*SL
    // loop-invariant masks.
    int lane = tid;
    asm volatile("" : "+v"(lane));
    const RowGeo g = row_geo<Tag, EXTRAS>(row_ptr(r), V32, nvec);
    const int32_t ei = EXTRAS ? extra_index<Tag>(g, tid) : -1;
    // Per-row scalars: one scalar-cache load, issued a row ahead.
    const RowRecord rec = rec_next;
    const bool skip = skip_masked && rec.wcoef() == 0.0f;
    const uint32_t rn = r + gridDim.x;
    const bool has_next = rn < rows32;
    if (has_next) rec_next = load_record(a, rn, T32);
    const int32_t tgt = rec.target;
    const bool tgt_ok = tgt >= 0;
    // Slab k of this lane holds the target iff rel == k * NT; a target in
    // the head or tail is the extra element of lane ei == tgt.
    const int32_t bt = tgt - (int32_t)g.head;
    const bool in_body = tgt_ok && (!EXTRAS || (bt >= 0 && bt < (int32_t)(g.nbody * EPV)));
    const int rel = in_body ? (bt >> P::LOG2_EPV) - lane : -1;
    const int ti = bt & (EPV - 1);
    const bool ex_tgt = EXTRAS && tgt_ok && ei == tgt;

    // Sweep 1: per-lane online (max, sum exp) over the slabs; the target
    // column is left out of the sum in the one lane and slab that hold it.
    LaneLse acc{-__builtin_huge_valf(), 0.0f};
    float m = -__builtin_huge_valf(), s = 0.0f, xt = 0.0f;
    if (!skip) {  // uniform over the workgroup
#pragma unroll
      for (int k = 0; k < SL; ++k)
        if (lane < (int)g.nbody - k * NT)
          fold_vector<Tag>(acc, x[k], rel == k * NT, ti, &sh_xt[buf]);
      if constexpr (EXTRAS) {
        if (ei >= 0) fold_one(acc, P::one(xe), ex_tgt, &sh_xt[buf]);
      }
      // No valid target: xt = -inf keeps the row's log-sum-exp finite (the
      // log-prob is set to NaN below).
      if (!tgt_ok && tid == 0) sh_xt[buf] = -__builtin_huge_valf();
      // Workgroup combine, kept short: the next row's loads are not issued
      // until it ends.  Wave max, then the rescaled sum (one exponential per
      // lane), then the wave pairs through LDS with one barrier.
      const float Mw = wave_max_dpp(acc.m);
      const float Sw = wave_sum_dpp(rescale(acc.s, acc.m, Mw));
      if ((tid & 63) == 0) {
        sh_m[buf][tid >> 6] = Mw;
        sh_s[buf][tid >> 6] = Sw;
      }
      lds_barrier();
      float mw[NT / 64];
#pragma unroll
      for (int i = 0; i < NT / 64; ++i) mw[i] = sh_m[buf][i];
      m = mw[0];
#pragma unroll
      for (int i = 1; i < NT / 64; ++i) m = fmaxf(m, mw[i]);
      float sp[NT / 64];
#pragma unroll
      for (int i = 0; i < NT / 64; ++i) sp[i] = rescale(sh_s[buf][i], mw[i], m);
#pragma unroll
      for (int w = NT / 128; w > 0; w >>= 1)
#pragma unroll
        for (int i = 0; i < w; ++i) sp[i] += sp[i + w];
      s = sp[0];
      xt = sh_xt[buf];
      buf ^= 1;
    }
    // Past the last row (or for a skipped next row) the descriptor covers 0
    // bytes: the refills return zeros without touching memory.
    const bool skip_next = skip_masked && rec_next.wcoef() == 0.0f;
    const bool load_next = has_next && !skip_next;
    const S* pn = row_ptr(load_next ? rn : r);
    const RowGeo gn = row_geo<Tag, EXTRAS>(pn, V32, nvec);
    const __amdgpu_buffer_rsrc_t src =
        load_next ? row_rsrc(pn + gn.head, gn.nbody * 16) : row_rsrc(logits, 0u);

    // Opaque to the optimiser: sweep 2 re-expands the packed slabs instead of
    // keeping sweep 1's widened copies live (twice the registers).
#pragma unroll
    for (int k = 0; k < SL; ++k) asm volatile("" : "+v"(x[k]));
    if constexpr (EXTRAS) asm volatile("" : "+v"(xe));

    const RowLogprob<float> fr = finish_row<float>(m, s, xt);
    const float lse = skip ? 0.0f : fr.lse;
    const float logp = skip ? 0.0f : (tgt_ok ? fr.logp : __builtin_nanf(""));
    const float gr =
        skip ? 0.0f : -(rec.wcoef() * token_local_grad<float>(c, logp, rec.old, rec.adv));
    const float tgt_d = target_grad<float>(gr, logp, true, xt, lse);
    if (tid == 0) {
      store_as<float>(a.logp, a.logp_dt, r, logp);
      static_cast<float*>(a.lse_out)[r] = lse;
    }

    // Sweep 2: dlogits, then refill the register slabs with the next row.
    const S* drow = dl + (int64_t)b * a.ds_b + (int64_t)t * a.ds_t;
    const __amdgpu_buffer_rsrc_t dst = row_rsrc(drow + g.head, g.nbody * 16);
    // -g * exp(x - lse) = -sign(g) * exp2(x * log2e + (log2|g| - lse * log2e)):
    // one FMA per 16-bit element, the difference first for float32, whose 1e-7
    // it keeps.  The FMA leaves the rounding of lse * log2e in the exponent,
    // 5e-6 at |lse| = 128 and doubling with it (at 3e38 nothing else is left),
    // so 16-bit rows past that take the distance from the row's maximum, which
    // is exact at any size, and the sum itself instead of lse, which float32
    // cannot hold beside such a maximum.  The branch is uniform over the
    // workgroup: forming the difference in every row costs 1-2% of the
    // 151936-entry sweep.  The sign is applied to the packed words with one XOR
    // per dword.
    // kFmaLse < |lse| < inf, compared as bits in scalar registers.
    const uint32_t lse_bits =
        (uint32_t)__builtin_amdgcn_readfirstlane((int)(__float_as_uint(lse) & 0x7fffffffu));
    const bool wide = EPV == 8 && lse_bits > kFmaLse && lse_bits < 0x7f800000u;
    const float lg = __log2f(fabsf(gr));
    const bool flip = gr > 0.0f;
    const uint32_t sgn = flip ? P::SGN2 : 0u;
    const float tgt_pre = flip ? -tgt_d : tgt_d;  // the XOR restores tgt_d
    // Every element goes through the same arithmetic, also for a zero-weight
    // row: there log2|g| = -inf and exp2(-inf) = 0 for every finite or -inf
    // logit (a +inf or NaN logit makes lse non-finite and the row NaN, as in
    // log_softmax), so zero-weight rows take no branch.
    auto put_row = [&](auto expo) __attribute__((always_inline)) {
#pragma unroll
      for (int k = 0; k < SL; ++k) {
        float d[EPV];
        float v[EPV];
        P::unpack(x[k], v);
#pragma unroll
        for (int i = 0; i < EPV; ++i) d[i] = exp2_hw(expo(v[i]));
        if (rel == k * NT) {
#pragma unroll
          for (int i = 0; i < EPV; ++i) d[i] = (i == ti) ? tgt_pre : d[i];
        }
        u32x4 o = P::pack(d);
        o.x ^= sgn; o.y ^= sgn; o.z ^= sgn; o.w ^= sgn;
        store_b128_nt(o, dst, voff, k * NT * 16);
      }
      if constexpr (EXTRAS) {
        const float dv = ex_tgt ? tgt_pre : exp2_hw(expo(P::one(xe)));
        P::store_one(P::pack_one(dv) ^ (flip ? P::SGN1 : 0u), row_rsrc(drow, V32 * ESZ),
                     extra_off(g));
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if constexpr (EPV == 8) {
      if (__builtin_expect(wide, 0)) {
        const float cm = lg - __log2f(s + exp2_hw((xt - m) * kLog2e));
        put_row([&](float xv) { return __builtin_fmaf(xv - m, kLog2e, cm); });
      } else {
        const float cg = lg - lse * kLog2e;
        put_row([&](float xv) { return __builtin_fmaf(xv, kLog2e, cg); });
      }
    } else {
      put_row([&](float xv) { return __builtin_fmaf(xv - lse, kLog2e, lg); });
    }
    // Then the next row's loads into the same registers: each CU issues its
    // row's stores as one burst and the next row's loads as another instead
    // of alternating 16-byte stores and loads, which the memory system serves
    // 8-12% faster (5.7 against 5.1-5.3 TB/s for the same 1R + 1W bytes).
#pragma unroll
    for (int k = 0; k < SL; ++k) {
      x[k] = __builtin_amdgcn_raw_buffer_load_b128(src, voff, k * NT * 16, kAuxLoad);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (EXTRAS) {
      const __amdgpu_buffer_rsrc_t esrc = load_next ? row_rsrc(pn, V32 * ESZ) : row_rsrc(logits, 0u);
      xe = P::load_one(esrc, extra_off(gn));
    }
  }
}

// Per-row inputs of the backward (rrl_logprob_bwd): target id, log-sum-exp,
// upstream gradient g = d loss / d logp and the forward's log-prob, each a
// uniform load through the scalar data cache (read-only in this kernel).
struct BwdRow {
  int64_t target;
  float lse, g, logp;
};

__device__ __forceinline__ BwdRow load_bwd_row(const RowArgs& a, uint32_t r, uint32_t T32) {
  typedef __attribute__((address_space(4))) const float CF;
  typedef __attribute__((address_space(4))) const int32_t CI32;
  typedef __attribute__((address_space(4))) const int64_t CI64;
  const uint32_t b = r / T32, t = r - b * T32;
  const int64_t off = (int64_t)b * a.tgt.sr + (int64_t)t * a.tgt.sc;
  const uintptr_t tp = reinterpret_cast<uintptr_t>(a.tgt.ptr);
  BwdRow q;
  q.target = a.tgt.dt == RRL_I32 ? (int64_t)reinterpret_cast<CI32*>(tp)[off]
                                 : reinterpret_cast<CI64*>(tp)[off];
  q.lse = reinterpret_cast<CF*>(reinterpret_cast<uintptr_t>(a.lse))[r];
  q.g = reinterpret_cast<CF*>(reinterpret_cast<uintptr_t>(a.g))[r];
  q.logp = reinterpret_cast<CF*>(reinterpret_cast<uintptr_t>(a.logp_in))[r];
  return q;
}

// A row whose gradient is exactly zero and whose log-sum-exp is finite has
// all-zero dlogits: its logits are never read.
__device__ __forceinline__ bool bwd_zero_row(const BwdRow& q) {
  return q.g == 0.0f && q.lse - q.lse == 0.0f;
}

// rrl_logprob_bwd for 16-bit and float32 rows (losses.py:34-38 backward):
// dlogits = g * (onehot(target) - exp(x - lse)) with lse, g and log-prob given,
// so there is no reduction and no exchange between lanes.  The schedule is the
// fused kernel's sweep 2: the row sits in VGPRs as SL slabs of 16 bytes per
// lane (plus the head and tail elements with EXTRAS), is written back as one
// burst of stores and the registers are refilled with the workgroup's next
// row as one burst of loads.  The waves never synchronise.
//
// PIECES: a row longer than one set of slabs goes through as `pieces` runs of
// SL * NT vectors (there is nothing to reduce, so a piece is a row of its
// own); the head belongs to the first run and the tail to the last.
template <class Tag, int NT, int SL, bool EXTRAS, bool PIECES>
__global__ __launch_bounds__(NT, kWavesPerSimd) void resident_bwd_kernel(RowArgs a, int32_t nvec,
                                                                         uint32_t pieces) {
  using P = Pack16<Tag>;
  using S = typename Tag::S;
  constexpr int EPV = P::EPV;
  constexpr int ESZ = (int)sizeof(S);
  const int tid = threadIdx.x;
  const uint32_t rows32 = (uint32_t)(a.B * a.T) * (PIECES ? pieces : 1u);
  const uint32_t T32 = (uint32_t)a.T;
  const uint32_t V32 = (uint32_t)a.V;
  const int voff = tid * 16;
  const S* logits = static_cast<const S*>(a.logits);
  S* dl = static_cast<S*>(a.dl);
  uint32_t r = blockIdx.x;
  if (r >= rows32) return;

  // Work item rr: row rr, or piece rr % pieces of row rr / pieces.
  auto row_of = [&](uint32_t rr) { return PIECES ? rr / pieces : rr; };
  auto piece_of = [&](uint32_t rr) { return PIECES ? rr - (rr / pieces) * pieces : 0u; };
  auto row_ptr = [&](uint32_t rr) {
    const uint32_t row = row_of(rr);
    const uint32_t bb = row / T32, tt = row - bb * T32;
    return logits + (int64_t)bb * a.ls_b + (int64_t)tt * a.ls_t;
  };
  // The item's first body vector and their number.
  auto body_of = [&](const RowGeo& g, uint32_t rr, uint32_t& count) {
    const uint32_t first = PIECES ? piece_of(rr) * (uint32_t)(SL * NT) : 0u;
    const uint32_t left = g.nbody > first ? g.nbody - first : 0u;
    count = PIECES && left > (uint32_t)(SL * NT) ? (uint32_t)(SL * NT) : left;
    return first;
  };
  auto extra_of = [&](const RowGeo& g, uint32_t rr) {
    if (PIECES && piece_of(rr) != (tid < kHeadLanes ? 0u : pieces - 1)) return -1;
    return extra_index<Tag>(g, tid);
  };
  auto extra_off = [&](const RowGeo& g, uint32_t rr) {
    const int32_t ei = extra_of(g, rr);
    return ei >= 0 ? ei * ESZ : (int)(V32 * ESZ);
  };
  auto body_rsrc = [&](const S* row, const RowGeo& g, uint32_t rr) {
    uint32_t count;
    const uint32_t first = body_of(g, rr, count);
    return row_rsrc(row + g.head + first * EPV, count * 16);
  };
  BwdRow next = load_bwd_row(a, row_of(r), T32);
  u32x4 x[SL];
  uint32_t xe = 0;
  {
    const bool z0 = bwd_zero_row(next);
    const S* p0 = row_ptr(r);
    const RowGeo g0 = row_geo<Tag, EXTRAS>(p0, V32, nvec);
    const __amdgpu_buffer_rsrc_t src = z0 ? row_rsrc(logits, 0u) : body_rsrc(p0, g0, r);
#pragma unroll
    for (int k = 0; k < SL; ++k) {
      x[k] = __builtin_amdgcn_raw_buffer_load_b128(src, voff, k * NT * 16, kAuxLoad);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (EXTRAS)
      xe = P::load_one(z0 ? row_rsrc(logits, 0u) : row_rsrc(p0, V32 * ESZ), extra_off(g0, r));
  }

  // The zero rows' store data: a register quad of its own, opaque so that it
  // is not rematerialised into a slab register whose load is still pending
  // (that would make the zero stores wait on vmcnt, which on gfx9 also waits
  // for every older store to be acknowledged).
  u32x4 zv = {0u, 0u, 0u, 0u};
  asm volatile("" : "+v"(zv));

  for (; r < rows32; r += gridDim.x) {
    const uint32_t row = row_of(r);
    const uint32_t b = row / T32, t = row - b * T32;
    int lane = tid;
    asm volatile("" : "+v"(lane));
    const RowGeo g = row_geo<Tag, EXTRAS>(row_ptr(r), V32, nvec);
    const int32_t ei = EXTRAS ? extra_of(g, r) : -1;
    uint32_t count;
    const uint32_t first = body_of(g, r, count);
    const BwdRow cur = next;
    const uint32_t rn = r + gridDim.x;
    const bool has_next = rn < rows32;
    if (has_next) next = load_bwd_row(a, row_of(rn), T32);
    // A target outside [0, V) has no column: every element takes the
    // exp(x - lse) term, as in the generic kernel.
    const bool tgt_ok = cur.target >= 0 && cur.target < a.V;
    const int32_t tgt = tgt_ok ? (int32_t)cur.target : 0;
    const int32_t bt = tgt - (int32_t)(g.head + first * EPV);
    const bool in_body = tgt_ok && ((!EXTRAS && !PIECES) || (bt >= 0 && bt < (int32_t)(count * EPV)));
    const int rel = in_body ? (bt >> P::LOG2_EPV) - lane : -1;
    const int ti = bt & (EPV - 1);
    const bool ex_tgt = EXTRAS && tgt_ok && ei == tgt;
    const bool zero = bwd_zero_row(cur);
    const float gr = cur.g, lse = cur.lse;
    // -g * exp(x - lse) = -sign(g) * exp2((x - lse) * log2e + log2|g|): the
    // difference is formed first, so no finite lse overflows.
    const float lg = __log2f(fabsf(gr));
    const bool flip = gr > 0.0f;
    const uint32_t sgn = flip ? P::SGN2 : 0u;
    const float tgt_d = zero ? 0.0f : target_grad<float>(gr, cur.logp, true, 0.0f, lse);
    const float tgt_pre = flip ? -tgt_d : tgt_d;  // the XOR restores tgt_d
    const bool load_next = has_next && !bwd_zero_row(next);
    const S* pn = row_ptr(load_next ? rn : r);
    const RowGeo gn = row_geo<Tag, EXTRAS>(pn, V32, nvec);
    const __amdgpu_buffer_rsrc_t src =
        load_next ? body_rsrc(pn, gn, rn) : row_rsrc(logits, 0u);
    const S* drow = dl + (int64_t)b * a.ds_b + (int64_t)t * a.ds_t;
    const __amdgpu_buffer_rsrc_t dst = row_rsrc(drow + g.head + first * EPV, count * 16);
    if (zero) {  // uniform over the workgroup
      // Stores only, with no dependence on the (never read) slabs: a run of
      // zero rows (a clipped GSPO sequence, masked prompt tokens) streams its
      // stores without waiting for earlier ones.  Measured on config 3 (72%
      // zero rows): backward 16.8-18.4 ms against 18.6-20.0 ms when the zero
      // rows went through the arithmetic below.
#pragma unroll
      for (int k = 0; k < SL; ++k) {
        store_b128_nt(zv, dst, voff, k * NT * 16);
      }
      if constexpr (EXTRAS) {
        P::store_one(zv.x, row_rsrc(drow, V32 * ESZ), extra_off(g, r));
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma unroll
      for (int k = 0; k < SL; ++k) {
        float d[EPV];
        float v[EPV];
        P::unpack(x[k], v);
#pragma unroll
        for (int i = 0; i < EPV; ++i) d[i] = exp2_hw(__builtin_fmaf(v[i] - lse, kLog2e, lg));
        if (rel == k * NT) {
#pragma unroll
          for (int i = 0; i < EPV; ++i) d[i] = (i == ti) ? tgt_pre : d[i];
        }
        u32x4 o = P::pack(d);
        o.x ^= sgn; o.y ^= sgn; o.z ^= sgn; o.w ^= sgn;
        store_b128_nt(o, dst, voff, k * NT * 16);
      }
      if constexpr (EXTRAS) {
        const float dv =
            ex_tgt ? tgt_pre : exp2_hw(__builtin_fmaf(P::one(xe) - lse, kLog2e, lg));
        P::store_one(P::pack_one(dv) ^ (flip ? P::SGN1 : 0u), row_rsrc(drow, V32 * ESZ),
                     extra_off(g, r));
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int k = 0; k < SL; ++k) {
      x[k] = __builtin_amdgcn_raw_buffer_load_b128(src, voff, k * NT * 16, kAuxLoad);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (EXTRAS)
      xe = P::load_one(load_next ? row_rsrc(pn, V32 * ESZ) : row_rsrc(logits, 0u), extra_off(gn, rn));
  }
}

}  // namespace

int launch_pack_records(const RowArgs& a, hipStream_t stream) {
  if (a.pp.flags & RRL_POLICY_RECORDS_READY) return RRL_OK;
  const int64_t rows = a.B * a.T;
  const unsigned grid = (unsigned)((rows + 255) / 256 < 65536 ? (rows + 255) / 256 : 65536);
  hipLaunchKernelGGL(pack_records_kernel, dim3(grid), dim3(256), 0, stream, a);
  return check_launch("pack_records_kernel");
}

int cu_count_of_current_device(int* n_out) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return check_launch("hipGetDevice");
  static int cu_count[64] = {0};
  if (dev < 0 || dev >= 64) dev = 0;
  if (cu_count[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    cu_count[dev] = n;
  }
  *n_out = cu_count[dev];
  return RRL_OK;
}

namespace {

// Workgroups per CU by slab count: the waves per SIMD that the kernels'
// registers allow (4 SL of slabs and about 45 more), in NT-lane workgroups.
template <int NT, int SL>
constexpr int wgs_per_cu() {
  constexpr int waves = SL <= 4 ? 7 : SL <= 8 ? 6 : SL <= 12 ? 5 : kWavesPerSimd;
  return waves * 256 / NT > 0 ? waves * 256 / NT : 1;
}

template <class Tag, int NT, int SL, bool EXTRAS>
int launch_resident(int mode, const RowArgs& a, int32_t nvec, int cus, hipStream_t stream) {
  static_assert(!EXTRAS || NT >= kHeadLanes + Pack16<Tag>::EPV, "lanes for the head and the tail");
  const int64_t rows = a.B * a.T;
  const int64_t wgs = (int64_t)cus * wgs_per_cu<NT, SL>();
  const unsigned grid = (unsigned)(rows < wgs ? rows : wgs);
  if (mode == 1) {
    hipLaunchKernelGGL((resident_bwd_kernel<Tag, NT, SL, EXTRAS, false>), dim3(grid), dim3(NT), 0,
                       stream, a, nvec, 1u);
    return check_launch("resident_bwd_kernel");
  }
  hipLaunchKernelGGL((resident_fused_kernel<Tag, NT, SL, EXTRAS>), dim3(grid), dim3(NT), 0, stream,
                     a, nvec);
  return check_launch("resident_fused_kernel");
}

// Lanes per row by its length.  A row's time is its loads' latency, the
// reduction and finish_row's serial chain, then its stores; a CU hides that
// only behind other rows, so a short row takes a small workgroup and the CU
// holds many (24 rows of 4096 bf16 entries with one wave each).  Measured
// with 8192 rows, us at no fewer than 64 / 128 / 256 / 512 / 1024 lanes per
// row, the fused pass and the backward (which has no reduction, and would take
// 256 lanes where the fused pass takes fewer; it shares the fused pass's table):
//   V =  4096 bf16 (  512 vectors)   20 /  29 /  35 /  84 / 198    24 /  24 /  24 /  50 / 123
//   V =  8192 bf16 ( 1024)           47 /  47 /  51 /  88 / 214    45 /  45 /  44 /  53 / 125
//   V = 16000 bf16 ( 2000)            - /  95 /  95 / 107 / 225     - /  92 /  92 /  97 / 129
//   V = 24000 bf16 ( 3000)            - /   - / 146 / 139 / 237     - /   - / 140 / 142 / 153
//   V = 32000 bf16 ( 4000)            - /   - / 185 / 186 / 250     - /   - / 193 / 192 / 195
//   V = 50304 bf16 ( 6288)            - /   - /   - / 294 / 317     - /   - /   - / 306 / 305
//   V = 65536 bf16 ( 8192, 4096 rows) - /   - /   - / 183 / 197     - /   - /   - / 184 / 185
//   V = 20000 f32  ( 5000)            - /   - /   - / 233 / 247     - /   - /   - / 241 / 241
//   V = 32000 f32  ( 8000, 4096 rows) - /   - /   - /   - / 183     - /   - /   - /   - / 186
// A slab past the row's end costs its issue slots though it moves nothing:
// 4000 vectors took 228 us with 13 slabs of 512 lanes against 190 with 8, so
// the slab counts step by one or two from 4 up.  With few rows one- and two-wave
// workgroups leave the chip idle, and 256 lanes finish each row sooner; the fused
// pass's lines cross between 1024 and 2048 rows, the backward's not at all, by
// little (us with one wave, or two at 12000, against 256 lanes):
//   rows            512          1024         1536         2048         4096
//   V =  4096  6.5 /  5.5   7.2 /  7.0   8.6 /  8.9   8.9 / 10.4  11.8 / 18.1  fused
//              4.3 /  4.4   4.9 /  4.3   6.0 /  5.9   7.4 /  6.8  12.5 / 11.7  backward
//   V =  8192  8.5 /  6.5   9.0 /  8.9  11.6 / 10.7  11.9 / 13.8  20.2 / 26.4  fused
//              5.3 /  4.5   7.2 /  6.8  10.0 /  9.7  12.2 / 11.6  23.3 / 22.6  backward
//   V = 12000 10.4 /  8.1  11.3 / 11.1  15.9 / 14.0  16.5 / 16.9  36.8 / 36.3  fused
//              6.4 /  5.3   8.8 /  9.2  13.7 / 12.8  17.4 / 17.1  35.8 / 33.1  backward
template <class Tag, bool EXTRAS>
int launch_variant(int mode, const RowArgs& a, int32_t nvec, hipStream_t stream) {
  int cus = 0;
  if (int rc = cu_count_of_current_device(&cus)) return rc;
  const int64_t rows = a.B * a.T;
  if (mode == 2) {
    if (int rc = launch_pack_records(a, stream)) return rc;
  }
  const bool many = rows >= 2048;
#define RRL_RESIDENT_CASE(NTV, SLV) \
  if (nvec <= NTV * SLV) return launch_resident<Tag, NTV, SLV, EXTRAS>(mode, a, nvec, cus, stream);
  if (many) {
    if constexpr (EXTRAS) {
      RRL_RESIDENT_CASE(128, 4)  // one wave has no lanes for the tail
    } else {
      RRL_RESIDENT_CASE(64, 2)
      RRL_RESIDENT_CASE(64, 4)
      RRL_RESIDENT_CASE(64, 6)
      RRL_RESIDENT_CASE(64, 8)
    }
    RRL_RESIDENT_CASE(128, 5)
    RRL_RESIDENT_CASE(128, 6)
    RRL_RESIDENT_CASE(128, 8)
    RRL_RESIDENT_CASE(128, 10)
    RRL_RESIDENT_CASE(128, 12)
  }
  RRL_RESIDENT_CASE(256, 2)
  RRL_RESIDENT_CASE(256, 4)
  RRL_RESIDENT_CASE(256, 6)
  RRL_RESIDENT_CASE(256, 7)
  RRL_RESIDENT_CASE(256, 8)
  RRL_RESIDENT_CASE(256, 10)
  RRL_RESIDENT_CASE(256, 12)
  RRL_RESIDENT_CASE(512, 7)
  RRL_RESIDENT_CASE(512, 8)
  RRL_RESIDENT_CASE(512, 10)
  RRL_RESIDENT_CASE(512, 12)
  RRL_RESIDENT_CASE(512, 13)
  RRL_RESIDENT_CASE(512, 14)
  if constexpr (Pack16<Tag>::EPV == 8) {
    RRL_RESIDENT_CASE(512, 16)
  } else {
    RRL_RESIDENT_CASE(1024, 8)
  }
  RRL_RESIDENT_CASE(1024, 9)
  RRL_RESIDENT_CASE(1024, 10)
  RRL_RESIDENT_CASE(1024, 12)
  RRL_RESIDENT_CASE(1024, 13)
  RRL_RESIDENT_CASE(1024, 14)
  RRL_RESIDENT_CASE(1024, 16)
  RRL_RESIDENT_CASE(1024, 18)
  RRL_RESIDENT_CASE(1024, 19)
  RRL_RESIDENT_CASE(1024, 20)
#undef RRL_RESIDENT_CASE
  set_error("resident row kernel: row too long");
  return RRL_EINVAL;
}

constexpr int64_t kMaxResidentVec = kMaxSlabs * 1024;  // SL = 20 fits 128 VGPRs without spills

// rrl_logprob_bwd of longer rows, in the fewest pieces and the fewest slabs
// that cover them.
template <class Tag, bool EXTRAS>
int launch_pieces(const RowArgs& a, int32_t nvec, hipStream_t stream) {
  int cus = 0;
  if (int rc = cu_count_of_current_device(&cus)) return rc;
  const int64_t pieces = (nvec + kMaxResidentVec - 1) / kMaxResidentVec;
  const int64_t items = a.B * a.T * pieces;
  const unsigned grid = (unsigned)(items < cus ? items : cus);
#define RRL_PIECES_CASE(SLV)                                                                   \
  if (nvec <= pieces * SLV * 1024) {                                                           \
    hipLaunchKernelGGL((resident_bwd_kernel<Tag, 1024, SLV, EXTRAS, true>), dim3(grid),        \
                       dim3(1024), 0, stream, a, nvec, (uint32_t)pieces);                      \
    return check_launch("resident_bwd_kernel");                                                \
  }
  RRL_PIECES_CASE(12)
  RRL_PIECES_CASE(14)
  RRL_PIECES_CASE(16)
  RRL_PIECES_CASE(18)
  RRL_PIECES_CASE(19)
  RRL_PIECES_CASE(20)
#undef RRL_PIECES_CASE
  set_error("resident_bwd_kernel: row too long");
  return RRL_EINVAL;
}

template <class Tag>
int dispatch_resident(int mode, bool extras, const RowArgs& a, int32_t nvec, hipStream_t st) {
  if (nvec > kMaxResidentVec)
    return extras ? launch_pieces<Tag, true>(a, nvec, st) : launch_pieces<Tag, false>(a, nvec, st);
  return extras ? launch_variant<Tag, true>(mode, a, nvec, st)
                : launch_variant<Tag, false>(mode, a, nvec, st);
}

}  // namespace

// Takes the register-resident kernel (mode 2: the fused single pass; mode 1:
// rrl_logprob_bwd with the forward's log-probs given) for 16-bit and float32
// logits when the row's 16-byte vectors fit the register budget (V <= 163840
// 16-bit or 81920 float32 entries).  Rows that are 128-byte aligned with
// V % (16 / element size) == 0 take the plain variant.  Other rows take the
// variant with head and tail elements, whose body starts on a 128-byte
// boundary, provided every dlogits row sits at its logits row's offset from a
// 128-byte boundary (same strides mod 128 bytes, as for contiguous tensors or
// in place); failing that, 16-byte aligned rows take the plain variant.
// Otherwise *launched stays false and the caller runs the generic row kernel.
int maybe_launch_resident(const RowArgs& a, int mode, int logits_dtype, hipStream_t stream,
                          bool* launched) {
  *launched = false;
  if (mode == 2 && (a.pp.flags & RRL_POLICY_GENERIC)) return RRL_OK;
  if (mode != 1 && mode != 2) return RRL_OK;
  if (logits_dtype != RRL_BF16 && logits_dtype != RRL_F16 && logits_dtype != RRL_F32)
    return RRL_OK;
  if (a.dl_dt != logits_dtype || a.accumulate) return RRL_OK;
  const int64_t esz = logits_dtype == RRL_F32 ? 4 : 2;
  const int64_t epv = 16 / esz;
  const int64_t lim = (int64_t)1 << 31;
  if (a.B * a.T == 0 || a.V * esz >= lim - (1 << 24)) return RRL_OK;
  // Work items (rows, or pieces of long rows) are counted in 32 bits.
  const int64_t pieces = (a.V / epv + kMaxResidentVec - 1) / kMaxResidentVec;
  if (a.B * a.T * std::max<int64_t>(pieces, 1) >= lim || a.T >= lim) return RRL_OK;
  const auto al = [&](int64_t elems, int64_t n) { return ((elems * esz) % n) == 0; };
  const auto rows_aligned = [&](int64_t n) {
    return a.V % epv == 0 && (uintptr_t)a.logits % n == 0 && (uintptr_t)a.dl % n == 0 &&
           al(a.ls_b, n) && al(a.ls_t, n) && al(a.ds_b, n) && al(a.ds_t, n);
  };
  const bool same_offset = ((uintptr_t)a.dl - (uintptr_t)a.logits) % kBodyAlign == 0 &&
                           al(a.ds_b - a.ls_b, kBodyAlign) && al(a.ds_t - a.ls_t, kBodyAlign);
  // Plain: 128-byte aligned rows, or 16-byte aligned ones the head/tail
  // variant cannot take.
  const bool aligned = rows_aligned(kBodyAlign) || (!same_offset && rows_aligned(16));
  if (!aligned && !same_offset) return RRL_OK;
  const int32_t nvec = (int32_t)(a.V / epv);
  if (mode == 1) {
    // Scalar loads need 4-byte aligned operands.
    if (a.logp_in == nullptr || a.tgt.ptr == nullptr) return RRL_OK;
    if (((uintptr_t)a.lse | (uintptr_t)a.g | (uintptr_t)a.logp_in) % 4) return RRL_OK;
    if ((uintptr_t)a.tgt.ptr % (a.tgt.dt == RRL_I32 ? 4 : 8)) return RRL_OK;
  } else {
    if (a.logp_dt != RRL_F32 || a.records == nullptr) return RRL_OK;
    if ((uintptr_t)a.records % 16) return RRL_OK;
  }
  *launched = true;
  // The long kernel's rows may start anywhere on both sides as long as the
  // offsets agree; 16-byte aligned rows at other offsets stay generic.
  if (mode == 2 && nvec > kMaxResidentVec) {
    if (!same_offset) {
      *launched = false;
      return RRL_OK;
    }
    return launch_long_fused(a, logits_dtype, stream);
  }
  switch (logits_dtype) {
    case RRL_BF16: return dispatch_resident<TagBF16>(mode, !aligned, a, nvec, stream);
    case RRL_F16: return dispatch_resident<TagF16>(mode, !aligned, a, nvec, stream);
    default: return dispatch_resident<TagF32>(mode, !aligned, a, nvec, stream);
  }
}

}  // namespace rrl
