// Policy objectives over [B, T] token log-probs (losses.py:104-512): forward
// scalars and diagnostics, closed-form backward to d/d current_logprobs, and
// the mask denominators for the single-pass kernel.
//
// Work split: one workgroup per sequence row accumulates the row's sums
// (policy_rows_kernel), one workgroup combines rows in a fixed order
// (policy_finalize_kernel).  GSPO-token needs the sequence ratio before its
// token surrogate, so it runs a second row pass.  Every reduction is
// deterministic for a given shape.
#include "policy_math.hpp"
#include "row_common.hpp"

namespace rrl {

namespace {

constexpr int RS = 8;  // per-row statistics slots

constexpr int kParts = 8;  // workgroups a sequence's row pass is split over, at most

// Workspace layout (Acc elements): rowstats[B][RS] | seq[B] | globals[8] |
// the row pass's partial sums [B][parts][RS].
template <typename Acc>
struct Workspace {
  Acc* rows;
  Acc* seq;
  Acc* glob;
  Acc* part;
  __host__ __device__ static Workspace at(void* base, int64_t B) {
    Workspace w;
    w.rows = static_cast<Acc*>(base);
    w.seq = w.rows + B * RS;
    w.glob = w.seq + B;
    w.part = w.glob + 8;
    return w;
  }
};

struct PolicyArgs {
  rrl_policy_params pp;
  int64_t B, T;
  View cur, old, adv, mask;
  void* ws;
  void* scalars;
  void* seq_out;
  uint8_t* trusted;
  int32_t* status;
  const void* gscal;
  const void* gseq;
  void* grad;
  void* row_coef;
  rrl_scalars sc;     // rrl_policy_forward's destinations / _backward's upstream gradients
  // rrl_policy_prepare
  int64_t V;
  View tgt;
  TokenRecord* records;
  int parts;  // workgroups per sequence in the row pass
};

// Flags found by a single-workgroup kernel: or-ed into the caller's cleared
// word, or (STORE) stored over whatever it held, through the fabric if it is
// host memory.
template <bool STORE>
__device__ __forceinline__ void report_flags(int32_t* status, int32_t flags) {
  if constexpr (STORE) {
    if (status) {
      *static_cast<volatile int32_t*>(status) = flags;
      __threadfence_system();
    }
  } else {
    if (flags) raise_flag(status, flags);
  }
}

// The objective's scalars: the acc array of rrl_policy_fwd, or one destination
// each with the loss beside them.
template <typename Acc>
__device__ __forceinline__ void put_scalar(const PolicyArgs& a, int k, Acc v) {
  if (a.scalars) static_cast<Acc*>(a.scalars)[k] = v;
  if (k < 4 && a.sc.ptr[k]) store_as<Acc>(a.sc.ptr[k], a.sc.dtype[k], 0, v);
  if (k == 0 && a.sc.ptr[4]) store_as<Acc>(a.sc.ptr[4], a.sc.dtype[4], 0, -v);
}

// What a row pass forms: the objective's sums, the mask's alone (the row
// coefficients), or those with the sweep's records and the target check.
enum RowsMode { ROWS_OBJECTIVE = 0, ROWS_MASK = 1, ROWS_PREPARE = 2 };

// Row pass.  Slots: 0 = #mask-true, 1 = mask weight sum, 2 = sum w*(cur-old),
// 3..6 = objective-specific sums (see policy_finalize_kernel); ROWS_PREPARE
// counts the row's bad target ids in slot 3.
template <typename Acc, int NT, int MODE>
__global__ __launch_bounds__(NT) void policy_rows_kernel(PolicyArgs a) {
  __shared__ Acc sh[(NT / 64) * 7];
  const PolicyConsts<Acc> c = PolicyConsts<Acc>::make(a.pp);
  Workspace<Acc> ws = Workspace<Acc>::at(a.ws, a.B);
  const int64_t chunk = (a.T + a.parts - 1) / a.parts;
  const int64_t t0 = blockIdx.y * chunk, t1 = t0 + chunk < a.T ? t0 + chunk : a.T;
  for (int64_t b = blockIdx.x; b < a.B; b += gridDim.x) {
    Acc v[7] = {Acc(0), Acc(0), Acc(0), Acc(0), Acc(0), Acc(0), Acc(0)};
    for (int64_t t = t0 + threadIdx.x; t < t1; t += NT) {
      const Acc w = mask_weight<Acc>(c, a.mask, b, t);
      const bool mt = c.kind == RRL_OBJ_NLL ? w != Acc(0) : a.mask.truth(b, t);
      v[0] += mt ? Acc(1) : Acc(0);
      v[1] += w;
      if (MODE == ROWS_PREPARE) {
        const int64_t tgt = load_index(a.tgt.ptr, a.tgt.dt, b * a.tgt.sr + t * a.tgt.sc);
        const bool ok = tgt >= 0 && tgt < a.V;
        v[3] += !ok && !target_ignored(c, tgt) ? Acc(1) : Acc(0);
        if (a.records) {
          TokenRecord r;
          r.target = ok ? (int32_t)tgt : -1;
          const bool nll = c.kind == RRL_OBJ_NLL;  // reads neither operand
          r.old = nll ? 0.0f : a.old.get<float>(b, t);
          r.adv = nll ? 0.0f : a.adv.get<float>(b, t);
          r.weight = (float)w;
          a.records[b * a.T + t] = r;
        }
      }
      if (MODE != ROWS_OBJECTIVE) continue;
      const Acc l = a.cur.get<Acc>(b, t);
      const Acc o = a.old.get<Acc>(b, t);
      if (c.kind == RRL_OBJ_NLL) {
        // An ignored token's log-prob may be NaN (no target): select, not multiply.
        v[3] += w != Acc(0) ? l * w : Acc(0);
        continue;
      }
      v[2] += (l - o) * w;
      if (c.kind == RRL_OBJ_PPO) {
        const Acc A = a.adv.get<Acc>(b, t);
        Acc rho, safe, d;
        const Acc surr = ppo_token(c, l, o, A, rho, safe, d);
        v[3] += surr * w;
        v[4] += ((rho - Acc(1)) - safe) * w;
        v[5] += ((rho < c.lo) || (rho > c.hi) ? Acc(1) : Acc(0)) * w;
        v[6] += rho * w;
      } else if (c.kind == RRL_OBJ_SAO) {
        const Acc A = a.adv.get<Acc>(b, t);
        Acc rho, safe, d, drho;
        bool tr;
        const Acc term = sao_token(c, l, o, A, rho, safe, tr, d, drho);
        v[3] += term * w;
        v[4] += ((rho - Acc(1)) - safe) * w;
        v[5] += (tr ? Acc(0) : Acc(1)) * w;
        v[6] += rho * w;
        if (a.trusted) a.trusted[b * a.T + t] = (tr && mt) ? 1 : 0;
      } else if (c.kind == RRL_OBJ_SAPO) {
        const Acc A = a.adv.get<Acc>(b, t);
        Acc rho, safe, p, d, dp;
        const Acc soft = sapo_token(c, l, o, A, rho, safe, p, d, dp);
        v[3] += soft * w;
        v[4] += ((rho - Acc(1)) - safe) * w;
        v[5] += rho * w;
        v[6] += ((Acc(4) * p) * (Acc(1) - p)) * w;
      }
    }
    block_sum<NT, 7, Acc>(v, sh);
    if (threadIdx.x == 0) {
#pragma unroll
      for (int k = 0; k < 7; ++k) ws.part[(b * a.parts + blockIdx.y) * RS + k] = v[k];
    }
  }
}

// A sequence's sums from its parts, in order; kept in ws.rows for the passes
// that follow.
template <typename Acc>
__device__ __forceinline__ void gather_row(const PolicyArgs& a, const Workspace<Acc>& ws, int64_t b,
                                           Acc (&rs)[RS]) {
  const Acc* p = ws.part + b * a.parts * RS;
#pragma unroll
  for (int k = 0; k < 7; ++k) rs[k] = p[k];
  rs[7] = Acc(0);
  for (int c = 1; c < a.parts; ++c)
#pragma unroll
    for (int k = 0; k < 7; ++k) rs[k] += p[c * RS + k];
#pragma unroll
  for (int k = 0; k < 7; ++k) ws.rows[b * RS + k] = rs[k];
}

// GSPO sequence ratio from row sums (losses.py:252-256): returns s, writes the
// clamped log ratio and whether the clamp passed gradient.
template <typename Acc>
__device__ __forceinline__ Acc gspo_seq_ratio(const PolicyConsts<Acc>& c, Acc lr, Acc cnt,
                                              Acc& safe, Acc& pass) {
  const Acc y = lr / cnt;
  safe = clampt(y, -c.K, c.K);
  pass = clamp_pass(y, -c.K, c.K);
  return M<Acc>::exp(safe);
}

// d min(s*A, clamp(s, lo, hi)*A) / d s with torch.minimum's tie split.
template <typename Acc>
__device__ __forceinline__ Acc clipped_surrogate(const PolicyConsts<Acc>& c, Acc s, Acc A,
                                                 Acc& dsurr) {
  const Acc cs = clampt(s, c.lo, c.hi);
  Acc share;
  const Acc surr = min_with_share(s * A, cs * A, share);
  dsurr = share * A + (Acc(1) - share) * A * clamp_pass(s, c.lo, c.hi);
  return surr;
}

template <typename Acc, int NT, bool STORE>
__global__ __launch_bounds__(NT) void policy_finalize_kernel(PolicyArgs a) {
  __shared__ Acc sh[(NT / 64) * 8];
  const PolicyConsts<Acc> c = PolicyConsts<Acc>::make(a.pp);
  Workspace<Acc> ws = Workspace<Acc>::at(a.ws, a.B);
  Acc v[8] = {Acc(0), Acc(0), Acc(0), Acc(0), Acc(0), Acc(0), Acc(0), Acc(0)};
  const bool per_seq = c.kind == RRL_OBJ_GSPO || c.kind == RRL_OBJ_GSPO_TOKEN || c.kind == RRL_OBJ_SAPO;
  for (int64_t b = threadIdx.x; b < a.B; b += NT) {
    Acc rs[RS];
    gather_row<Acc>(a, ws, b, rs);
    const Acc cnt = rs[0];
    if (per_seq) v[7] += (cnt == Acc(0)) ? Acc(1) : Acc(0);
    if (c.kind == RRL_OBJ_PPO || c.kind == RRL_OBJ_SAO || c.kind == RRL_OBJ_NLL) {
      v[0] += rs[1];
      v[3] += rs[3];
      v[4] += rs[4];
      v[5] += rs[5];
      v[6] += rs[6];
    } else if (c.kind == RRL_OBJ_GSPO || c.kind == RRL_OBJ_GSPO_TOKEN) {
      Acc safe, pass, dsurr;
      const Acc s = gspo_seq_ratio(c, rs[2], cnt, safe, pass);
      ws.seq[b] = s;
      if (a.seq_out) store_as<Acc>(a.seq_out, sizeof(Acc) == 8 ? RRL_F64 : RRL_F32, b, s);
      if (c.kind == RRL_OBJ_GSPO) {
        const Acc A = a.adv.get<Acc>(b, 0);
        v[3] += clipped_surrogate(c, s, A, dsurr);
      }
      v[4] += (s - Acc(1)) - safe;
      v[5] += ((s < c.lo) || (s > c.hi)) ? Acc(1) : Acc(0);
      v[6] += s;
    } else {  // SAPO: per-sequence means, then mean over sequences
      v[3] += rs[3] / cnt;
      v[4] += rs[4] / cnt;
      v[5] += rs[5] / cnt;
      v[6] += rs[6] / cnt;
    }
  }
  block_sum<NT, 8, Acc>(v, sh);
  if (threadIdx.x == 0) {
    Acc out[4] = {Acc(0), Acc(0), Acc(0), Acc(0)};
    int32_t flags = 0;
    if (c.kind == RRL_OBJ_NLL) {
      // F.cross_entropy: "mean" divides by the number of non-ignored tokens
      // (NaN when there is none, no error); "sum" does not divide.
      const bool sum = (a.pp.flags & RRL_POLICY_SUM) != 0;
      ws.glob[0] = sum ? Acc(1) : v[0];
      out[0] = sum ? v[3] : v[3] / v[0];
      out[1] = v[0];
    } else if (c.kind == RRL_OBJ_PPO || c.kind == RRL_OBJ_SAO) {
      const Acc Mw = v[0];
      if (Mw == Acc(0)) flags |= RRL_FLAG_EMPTY_MASK;
      ws.glob[0] = Mw;
      out[0] = v[3] / Mw;
      out[1] = v[4] / Mw;
      out[2] = v[5] / Mw;
      out[3] = v[6] / Mw;
    } else {
      if (v[7] != Acc(0)) flags |= RRL_FLAG_EMPTY_ROW;
      const Acc Bf = (Acc)a.B;
      ws.glob[0] = Bf;
      if (c.kind == RRL_OBJ_SAPO) {
        out[0] = v[3] / Bf;
        out[1] = v[4] / Bf;
        out[2] = v[5] / Bf;
        out[3] = v[6] / Bf;
      } else {
        out[0] = v[3] / Bf;  // GSPO-token overwrites after its second pass
        out[1] = v[4] / Bf;
        out[2] = v[5] / Bf;
        out[3] = v[6] / Bf;
      }
    }
    for (int k = 0; k < 4; ++k) put_scalar<Acc>(a, k, out[k]);
    if (a.scalars)
      for (int k = 4; k < RRL_NSCALARS; ++k) static_cast<Acc*>(a.scalars)[k] = Acc(0);
    report_flags<STORE>(a.status, flags);
  }
}

// GSPO-token second pass: per-row sum of mask * min(tau*A, clip(tau)*A) with
// tau = sg(s) * exp(cur - sg(cur)) (losses.py:331-341).
template <typename Acc, int NT>
__global__ __launch_bounds__(NT) void gspo_token_rows_kernel(PolicyArgs a) {
  __shared__ Acc sh[NT / 64];
  const PolicyConsts<Acc> c = PolicyConsts<Acc>::make(a.pp);
  Workspace<Acc> ws = Workspace<Acc>::at(a.ws, a.B);
  for (int64_t b = blockIdx.x; b < a.B; b += gridDim.x) {
    const Acc s = ws.seq[b];
    Acc v[1] = {Acc(0)};
    for (int64_t t = threadIdx.x; t < a.T; t += NT) {
      const Acc w = mask_weight<Acc>(c, a.mask, b, t);
      const Acc l = a.cur.get<Acc>(b, t);
      const Acc tau = s * M<Acc>::exp(l - l);
      Acc d;
      v[0] += clipped_surrogate(c, tau, a.adv.get<Acc>(b, t), d) * w;
    }
    block_sum<NT, 1, Acc>(v, sh);
    if (threadIdx.x == 0) ws.rows[b * RS + 3] = v[0];
  }
}

template <typename Acc, int NT>
__global__ __launch_bounds__(NT) void gspo_token_finalize_kernel(PolicyArgs a) {
  __shared__ Acc sh[NT / 64];
  Workspace<Acc> ws = Workspace<Acc>::at(a.ws, a.B);
  Acc v[1] = {Acc(0)};
  for (int64_t b = threadIdx.x; b < a.B; b += NT) v[0] += ws.rows[b * RS + 3] / ws.rows[b * RS + 0];
  block_sum<NT, 1, Acc>(v, sh);
  if (threadIdx.x == 0) put_scalar<Acc>(a, 0, v[0] / (Acc)a.B);
}

// Backward: grad_cur[b, t] = sum_k G[k] d scalar_k / d cur[b, t].
template <typename Acc, int NT>
__global__ __launch_bounds__(NT) void policy_bwd_kernel(PolicyArgs a) {
  const PolicyConsts<Acc> c = PolicyConsts<Acc>::make(a.pp);
  Workspace<Acc> ws = Workspace<Acc>::at(a.ws, a.B);
  Acc Gk[4];
  if (a.gscal) {
#pragma unroll
    for (int k = 0; k < 4; ++k) Gk[k] = static_cast<const Acc*>(a.gscal)[k];
  } else {
#pragma unroll
    for (int k = 0; k < 4; ++k)
      Gk[k] = a.sc.ptr[k] ? load_as<Acc>(a.sc.ptr[k], a.sc.dtype[k], 0) : Acc(0);
    if (a.sc.ptr[4]) Gk[0] -= load_as<Acc>(a.sc.ptr[4], a.sc.dtype[4], 0);  // loss = -objective
  }
  const Acc G0 = Gk[0], G1 = Gk[1], G2 = Gk[2], G3 = Gk[3];
  Acc* grad = static_cast<Acc*>(a.grad);
  const Acc Bf = (Acc)a.B;
  for (int64_t b = blockIdx.x; b < a.B; b += gridDim.x) {
    const Acc* rs = ws.rows + b * RS;
    const Acc cnt = rs[0];
    // Per-row factor for the GSPO kinds' sequence-ratio terms.
    Acc seq_coef = Acc(0), s = Acc(0);
    if (c.kind == RRL_OBJ_GSPO || c.kind == RRL_OBJ_GSPO_TOKEN) {
      Acc safe, pass, dsurr = Acc(0);
      s = gspo_seq_ratio(c, rs[2], cnt, safe, pass);
      const Acc gs = a.gseq ? static_cast<const Acc*>(a.gseq)[b] : Acc(0);
      Acc dy = (G1 * (s - Acc(1)) + G3 * s) / Bf + gs * s;
      if (c.kind == RRL_OBJ_GSPO) {
        (void)clipped_surrogate(c, s, a.adv.get<Acc>(b, 0), dsurr);
        dy += (G0 * dsurr * s) / Bf;
      }
      seq_coef = dy * pass;
    }
    for (int64_t t = threadIdx.x; t < a.T; t += NT) {
      const Acc w = mask_weight<Acc>(c, a.mask, b, t);
      Acc gr = Acc(0);
      if (c.kind == RRL_OBJ_NLL) {
        gr = w != Acc(0) ? (w / ws.glob[0]) * G0 : Acc(0);
      } else if (c.kind == RRL_OBJ_PPO) {
        const Acc l = a.cur.get<Acc>(b, t), o = a.old.get<Acc>(b, t), A = a.adv.get<Acc>(b, t);
        Acc rho, safe, d;
        (void)ppo_token(c, l, o, A, rho, safe, d);
        const Acc px = clamp_pass(l - o, -c.K, c.K);
        const Acc drho = rho * px;
        gr = (w / ws.glob[0]) * (G0 * d + G1 * (drho - px) + G3 * drho);
      } else if (c.kind == RRL_OBJ_SAO) {
        const Acc l = a.cur.get<Acc>(b, t), o = a.old.get<Acc>(b, t), A = a.adv.get<Acc>(b, t);
        Acc rho, safe, d, drho;
        bool tr;
        (void)sao_token(c, l, o, A, rho, safe, tr, d, drho);
        const Acc px = clamp_pass(l - o, -c.K, c.K);
        gr = (w / ws.glob[0]) * (G0 * d + G1 * (drho - px) + G3 * drho);
      } else if (c.kind == RRL_OBJ_SAPO) {
        const Acc l = a.cur.get<Acc>(b, t), o = a.old.get<Acc>(b, t), A = a.adv.get<Acc>(b, t);
        Acc rho, safe, p, d, dp;
        (void)sapo_token(c, l, o, A, rho, safe, p, d, dp);
        const Acc px = clamp_pass(l - o, -c.K, c.K);
        const Acc drho = rho * px;
        const Acc dgate = (Acc(4) * dp) * (Acc(1) - Acc(2) * p);
        gr = ((w / cnt) / Bf) * (G0 * d + G1 * (drho - px) + G2 * drho + G3 * dgate);
      } else if (c.kind == RRL_OBJ_GSPO) {
        gr = seq_coef * (w / cnt);
      } else {  // GSPO-token
        const Acc l = a.cur.get<Acc>(b, t);
        const Acc tau = s * M<Acc>::exp(l - l);
        Acc d;
        (void)clipped_surrogate(c, tau, a.adv.get<Acc>(b, t), d);
        gr = ((w / cnt) / Bf) * (G0 * d * tau) + seq_coef * (w / cnt);
      }
      grad[b * a.T + t] = gr;
    }
  }
}

// Mask denominators for the single-pass kernel.
template <typename Acc, int NT, bool PREPARE>
__global__ __launch_bounds__(NT) void row_coef_kernel(PolicyArgs a) {
  __shared__ Acc sh[(NT / 64) * 3];
  Workspace<Acc> ws = Workspace<Acc>::at(a.ws, a.B);
  Acc v[3] = {Acc(0), Acc(0), Acc(0)};
  for (int64_t b = threadIdx.x; b < a.B; b += NT) {
    Acc rs[RS];
    gather_row<Acc>(a, ws, b, rs);
    v[0] += rs[1];
    v[1] += rs[0] == Acc(0) ? Acc(1) : Acc(0);
    if (PREPARE) v[2] += rs[3];
  }
  block_sum<NT, 3, Acc>(v, sh);
  const bool per_seq = a.pp.kind != RRL_OBJ_PPO && a.pp.kind != RRL_OBJ_SAO &&
                       a.pp.kind != RRL_OBJ_NLL;
  const bool nll = a.pp.kind == RRL_OBJ_NLL;
  if (threadIdx.x == 0) {
    int32_t flags = 0;
    if (!per_seq && !nll && v[0] == Acc(0)) flags |= RRL_FLAG_EMPTY_MASK;
    if (per_seq && v[1] != Acc(0)) flags |= RRL_FLAG_EMPTY_ROW;
    if (PREPARE && v[2] != Acc(0)) flags |= RRL_FLAG_TARGET_RANGE;
    report_flags<PREPARE>(a.status, flags);
  }
  Acc* coef = static_cast<Acc*>(a.row_coef);
  if (coef == nullptr) return;  // GSPO: the check alone
  const Acc Bf = (Acc)a.B;
  const Acc flat = (nll && (a.pp.flags & RRL_POLICY_SUM)) ? Acc(1) : Acc(1) / v[0];
  for (int64_t b = threadIdx.x; b < a.B; b += NT) {
    coef[b] = per_seq ? (Acc(1) / ws.rows[b * RS + 0]) / Bf : flat;
  }
}

// The row pass takes a sequence in up to kParts pieces of at least 256 tokens:
// its time is the chain of dependent steps of one lane, 51 us for 32 steps (64
// sequences of 8192 tokens, SAPO, one workgroup each) and 7 us for the 4 of
// 8 parts.  1024 lanes per sequence instead spill and took 13-18 us at 1024
// tokens, where one 256-lane workgroup took 7.
template <typename Acc, int MODE>
int launch_policy_rows(const PolicyArgs& a, hipStream_t st) {
  if (a.B == 0) return RRL_OK;
  const unsigned grid = (unsigned)(a.B < 65536 ? a.B : 65536);
  hipLaunchKernelGGL((policy_rows_kernel<Acc, 256, MODE>), dim3(grid, (unsigned)a.parts), dim3(256),
                     0, st, a);
  return check_launch("policy_rows_kernel");
}

void split_rows(PolicyArgs& a) {
  const int64_t want = (a.T + 255) / 256;
  a.parts = (int)(want < 1 ? 1 : want < kParts ? want : kParts);
}

// The single-workgroup kernels over sequences take 256 lanes up to 256 of
// them; a wider workgroup only lengthens the final sum.
#define RRL_ONE_GROUP(KERNEL, ...)                                                            \
  do {                                                                                        \
    if (a.B <= 256)                                                                           \
      hipLaunchKernelGGL((KERNEL<Acc, 256 __VA_ARGS__>), dim3(1), dim3(256), 0, st, a);       \
    else                                                                                      \
      hipLaunchKernelGGL((KERNEL<Acc, 1024 __VA_ARGS__>), dim3(1), dim3(1024), 0, st, a);     \
    if (int rc = check_launch(#KERNEL)) return rc;                                            \
  } while (0)
#define RRL_COMMA ,

template <typename Acc, bool STORE>
int run_policy_fwd(PolicyArgs a, hipStream_t st) {
  constexpr int NT = 256;
  split_rows(a);
  if (int rc = launch_policy_rows<Acc, ROWS_OBJECTIVE>(a, st)) return rc;
  RRL_ONE_GROUP(policy_finalize_kernel, RRL_COMMA STORE);
  if (a.pp.kind == RRL_OBJ_GSPO_TOKEN && a.B > 0) {
    const unsigned grid = (unsigned)(a.B < 65536 ? a.B : 65536);
    hipLaunchKernelGGL((gspo_token_rows_kernel<Acc, NT>), dim3(grid), dim3(NT), 0, st, a);
    if (int rc = check_launch("gspo_token_rows_kernel")) return rc;
    RRL_ONE_GROUP(gspo_token_finalize_kernel, );
  }
  return RRL_OK;
}

template <typename Acc, bool PREPARE>
int run_row_coef(PolicyArgs a, hipStream_t st) {
  split_rows(a);
  if (int rc = launch_policy_rows<Acc, PREPARE ? ROWS_PREPARE : ROWS_MASK>(a, st)) return rc;
  RRL_ONE_GROUP(row_coef_kernel, RRL_COMMA PREPARE);
  return RRL_OK;
}

#undef RRL_COMMA
#undef RRL_ONE_GROUP

// Target ids in [0, V) (NLL's ignore_index exempt), one token per thread,
// ahead of the single-pass sweep that makes the same check.
struct TargetCheckArgs {
  rrl_policy_params pp;
  int64_t B, T, V;
  View tgt;
  int32_t* status;
  int32_t* part;  // one flag per workgroup (rrl_targets_status over many tokens)
};

template <int NT>
__device__ __forceinline__ bool any_bad_target(const TargetCheckArgs& a) {
  const PolicyConsts<float> c = PolicyConsts<float>::make(a.pp);
  const int64_t n = a.B * a.T;
  bool bad = false;
  for (int64_t i = blockIdx.x * (int64_t)NT + threadIdx.x; i < n; i += (int64_t)gridDim.x * NT) {
    const int64_t b = i / a.T, t = i - b * a.T;
    const int64_t tgt = load_index(a.tgt.ptr, a.tgt.dt, b * a.tgt.sr + t * a.tgt.sc);
    bad = bad || ((tgt < 0 || tgt >= a.V) && !target_ignored(c, tgt));
  }
  return bad;
}

__global__ __launch_bounds__(256) void check_targets_kernel(TargetCheckArgs a) {
  const bool bad = any_bad_target<256>(a);
  if (__any(bad) && (threadIdx.x & 63) == 0) raise_flag(a.status, RRL_FLAG_TARGET_RANGE);
}

// The stored form: up to kTargetsOne tokens one workgroup checks them and
// stores the status; beyond, every workgroup stores its own flag and a second
// launch combines them (nothing to clear, no atomics).
constexpr int64_t kTargetsOne = 16384;
constexpr int kTargetsParts = 1024;

template <bool PARTS>
__global__ __launch_bounds__(1024) void targets_status_kernel(TargetCheckArgs a) {
  const int bad = __syncthreads_or(any_bad_target<1024>(a));
  if (threadIdx.x != 0) return;
  if (PARTS) a.part[blockIdx.x] = bad;
  else report_flags<true>(a.status, bad ? RRL_FLAG_TARGET_RANGE : 0);
}

__global__ __launch_bounds__(1024) void targets_combine_kernel(TargetCheckArgs a, int parts) {
  const int bad = __syncthreads_or((int)threadIdx.x < parts && a.part[threadIdx.x] != 0);
  if (threadIdx.x == 0) report_flags<true>(a.status, bad ? RRL_FLAG_TARGET_RANGE : 0);
}

int validate_policy(const rrl_policy_params* p, int64_t B, int64_t T, int acc) {
  RRL_REQUIRE(p != nullptr, RRL_EINVAL, "params is null");
  RRL_REQUIRE(p->kind >= RRL_OBJ_PPO && p->kind <= RRL_OBJ_NLL, RRL_EINVAL, "unknown objective kind");
  RRL_REQUIRE(B >= 0 && T >= 0, RRL_EINVAL, "negative size");
  RRL_REQUIRE(acc == RRL_F32 || acc == RRL_F64, RRL_EDTYPE, "acc dtype must be float32 or float64");
  return RRL_OK;
}

}  // namespace
}  // namespace rrl

using namespace rrl;

extern "C" size_t rrl_policy_workspace_bytes(int64_t B, int32_t acc_dtype) {
  const size_t e = acc_dtype == RRL_F64 ? 8 : 4;
  return (size_t)(B * RS + B + 8 + B * kParts * RS) * e + 256;
}

namespace {

int policy_fwd_args(PolicyArgs& a, const rrl_policy_params* params, int64_t B, int64_t T,
                    const rrl_view& cur, const rrl_view& old, const rrl_view& adv,
                    const rrl_view& mask, int32_t acc_dtype, void* workspace) {
  if (int rc = validate_policy(params, B, T, acc_dtype)) return rc;
  RRL_REQUIRE(workspace, RRL_EINVAL, "workspace and scalars are required");
  RRL_REQUIRE(B * T == 0 || (cur.ptr && old.ptr && adv.ptr && mask.ptr), RRL_EINVAL,
              "null input pointer");
  RRL_REQUIRE(is_float_dtype(cur.dtype) && is_float_dtype(old.dtype) && is_float_dtype(adv.dtype),
              RRL_EDTYPE, "log-probabilities and advantages must be floating point");
  RRL_REQUIRE(is_known_dtype(mask.dtype), RRL_EDTYPE, "unsupported mask dtype");
  RRL_REQUIRE(params->kind != RRL_OBJ_NLL || mask.dtype == RRL_I32 || mask.dtype == RRL_I64,
              RRL_EDTYPE, "NLL: the mask operand holds the target ids (int32 or int64)");
  a.pp = *params; a.B = B; a.T = T;
  a.cur = to_view(cur); a.old = to_view(old); a.adv = to_view(adv); a.mask = to_view(mask);
  a.ws = workspace;
  return RRL_OK;
}

int check_scalars(const rrl_scalars* sc) {
  RRL_REQUIRE(sc, RRL_EINVAL, "workspace and scalars are required");
  for (int k = 0; k < 5; ++k)
    RRL_REQUIRE(!sc->ptr[k] || is_float_dtype(sc->dtype[k]), RRL_EDTYPE,
                "scalars must be floating point");
  return RRL_OK;
}

int run_policy_bwd(const PolicyArgs& a, int32_t acc_dtype, hipStream_t st) {
  const unsigned grid = (unsigned)(a.B < 65536 ? a.B : 65536);
  const bool wide = a.T > 256;  // as launch_policy_rows
  if (acc_dtype == RRL_F64) {
    if (wide) hipLaunchKernelGGL((policy_bwd_kernel<double, 1024>), dim3(grid), dim3(1024), 0, st, a);
    else hipLaunchKernelGGL((policy_bwd_kernel<double, 256>), dim3(grid), dim3(256), 0, st, a);
  } else {
    if (wide) hipLaunchKernelGGL((policy_bwd_kernel<float, 1024>), dim3(grid), dim3(1024), 0, st, a);
    else hipLaunchKernelGGL((policy_bwd_kernel<float, 256>), dim3(grid), dim3(256), 0, st, a);
  }
  return check_launch("policy_bwd_kernel");
}

}  // namespace

extern "C" int rrl_policy_fwd(const rrl_policy_params* params, int64_t B, int64_t T,
                              rrl_view cur, rrl_view old, rrl_view adv, rrl_view mask,
                              int32_t acc_dtype, void* workspace, void* scalars_out,
                              void* seq_out, uint8_t* trusted_out, int32_t* status,
                              void* stream) {
  clear_error();
  PolicyArgs a{};
  if (int rc = policy_fwd_args(a, params, B, T, cur, old, adv, mask, acc_dtype, workspace))
    return rc;
  RRL_REQUIRE(scalars_out, RRL_EINVAL, "workspace and scalars are required");
  a.scalars = scalars_out; a.seq_out = seq_out; a.trusted = trusted_out; a.status = status;
  hipStream_t st = as_stream(stream);
  return acc_dtype == RRL_F64 ? run_policy_fwd<double, false>(a, st)
                              : run_policy_fwd<float, false>(a, st);
}

extern "C" int rrl_policy_forward(const rrl_policy_params* params, int64_t B, int64_t T,
                                  rrl_view cur, rrl_view old, rrl_view adv, rrl_view mask,
                                  int32_t acc_dtype, void* workspace, const rrl_scalars* out,
                                  void* seq_out, uint8_t* trusted_out, int32_t* status,
                                  void* stream) {
  clear_error();
  PolicyArgs a{};
  if (int rc = policy_fwd_args(a, params, B, T, cur, old, adv, mask, acc_dtype, workspace))
    return rc;
  if (int rc = check_scalars(out)) return rc;
  a.sc = *out; a.seq_out = seq_out; a.trusted = trusted_out; a.status = status;
  hipStream_t st = as_stream(stream);
  return acc_dtype == RRL_F64 ? run_policy_fwd<double, true>(a, st)
                              : run_policy_fwd<float, true>(a, st);
}

extern "C" int rrl_policy_bwd(const rrl_policy_params* params, int64_t B, int64_t T,
                              rrl_view cur, rrl_view old, rrl_view adv, rrl_view mask,
                              int32_t acc_dtype, const void* workspace, const void* grad_scalars,
                              const void* grad_seq, void* grad_cur, void* stream) {
  clear_error();
  if (int rc = validate_policy(params, B, T, acc_dtype)) return rc;
  RRL_REQUIRE(workspace && grad_scalars && (B * T == 0 || grad_cur), RRL_EINVAL,
              "workspace, grad_scalars and grad_cur are required");
  if (B * T == 0) return RRL_OK;
  PolicyArgs a{};
  a.pp = *params; a.B = B; a.T = T;
  a.cur = to_view(cur); a.old = to_view(old); a.adv = to_view(adv); a.mask = to_view(mask);
  a.ws = const_cast<void*>(workspace); a.gscal = grad_scalars; a.gseq = grad_seq; a.grad = grad_cur;
  return run_policy_bwd(a, acc_dtype, as_stream(stream));
}

extern "C" int rrl_policy_backward(const rrl_policy_params* params, int64_t B, int64_t T,
                                   rrl_view cur, rrl_view old, rrl_view adv, rrl_view mask,
                                   int32_t acc_dtype, const void* workspace,
                                   const rrl_scalars* grads, const void* grad_seq, void* grad_cur,
                                   void* stream) {
  clear_error();
  if (int rc = validate_policy(params, B, T, acc_dtype)) return rc;
  if (int rc = check_scalars(grads)) return rc;
  RRL_REQUIRE(workspace && (B * T == 0 || grad_cur), RRL_EINVAL,
              "workspace and grad_cur are required");
  if (B * T == 0) return RRL_OK;
  PolicyArgs a{};
  a.pp = *params; a.B = B; a.T = T;
  a.cur = to_view(cur); a.old = to_view(old); a.adv = to_view(adv); a.mask = to_view(mask);
  a.ws = const_cast<void*>(workspace); a.sc = *grads; a.gseq = grad_seq; a.grad = grad_cur;
  return run_policy_bwd(a, acc_dtype, as_stream(stream));
}

namespace {

int row_coef_args(PolicyArgs& a, const rrl_policy_params* params, int64_t B, int64_t T,
                  const rrl_view& mask, int32_t acc_dtype, void* row_coef, void* workspace,
                  int32_t* status) {
  if (int rc = validate_policy(params, B, T, acc_dtype)) return rc;
  const bool gspo = params->kind == RRL_OBJ_GSPO || params->kind == RRL_OBJ_GSPO_TOKEN;
  RRL_REQUIRE(!gspo || !row_coef, RRL_EINVAL,
              "row coefficients exist for the token-local objectives only");
  // An empty mask has no address, and its rows are still counted (as empty).
  RRL_REQUIRE(workspace && (B == 0 || row_coef || gspo) && (B * T == 0 || mask.ptr), RRL_EINVAL,
              "null pointer argument");
  RRL_REQUIRE(is_known_dtype(mask.dtype), RRL_EDTYPE, "unsupported mask dtype");
  RRL_REQUIRE(params->kind != RRL_OBJ_NLL || mask.dtype == RRL_I32 || mask.dtype == RRL_I64,
              RRL_EDTYPE, "NLL: the mask operand holds the target ids (int32 or int64)");
  a.pp = *params; a.B = B; a.T = T; a.mask = to_view(mask);
  a.ws = workspace; a.row_coef = row_coef; a.status = status;
  return RRL_OK;
}

}  // namespace

extern "C" int rrl_policy_row_coef(const rrl_policy_params* params, int64_t B, int64_t T,
                                   rrl_view mask, int32_t acc_dtype, void* row_coef,
                                   void* workspace, int32_t* status, void* stream) {
  clear_error();
  PolicyArgs a{};
  RRL_REQUIRE(B == 0 || (row_coef && mask.ptr), RRL_EINVAL, "null pointer argument");
  RRL_REQUIRE(!params || (params->kind != RRL_OBJ_GSPO && params->kind != RRL_OBJ_GSPO_TOKEN),
              RRL_EINVAL, "row coefficients exist for the token-local objectives only");
  if (int rc = row_coef_args(a, params, B, T, mask, acc_dtype, row_coef, workspace, status))
    return rc;
  hipStream_t st = as_stream(stream);
  return acc_dtype == RRL_F64 ? run_row_coef<double, false>(a, st)
                              : run_row_coef<float, false>(a, st);
}

extern "C" int rrl_policy_prepare(const rrl_policy_params* params, int64_t B, int64_t T, int64_t V,
                                  rrl_view target, rrl_view old, rrl_view adv, rrl_view mask,
                                  int32_t acc_dtype, void* row_coef, void* records,
                                  void* workspace, int32_t* status, void* stream) {
  clear_error();
  PolicyArgs a{};
  if (int rc = row_coef_args(a, params, B, T, mask, acc_dtype, row_coef, workspace, status))
    return rc;
  RRL_REQUIRE(V >= 1, RRL_EINVAL, "vocabulary must be non-empty");
  RRL_REQUIRE(status && (B * T == 0 || target.ptr), RRL_EINVAL, "null pointer argument");
  RRL_REQUIRE(target.dtype == RRL_I32 || target.dtype == RRL_I64, RRL_EDTYPE,
              "target ids must be int32 or int64");
  if (records && params->kind != RRL_OBJ_NLL) {
    RRL_REQUIRE(B * T == 0 || (old.ptr && adv.ptr), RRL_EINVAL, "null pointer argument");
    RRL_REQUIRE(is_float_dtype(old.dtype) && is_float_dtype(adv.dtype), RRL_EDTYPE,
                "old log-probs and advantages must be floating point");
  }
  RRL_REQUIRE((uintptr_t)records % 16 == 0, RRL_EALIGN, "records must be 16-byte aligned");
  a.V = V; a.tgt = to_view(target); a.old = to_view(old); a.adv = to_view(adv);
  a.records = static_cast<TokenRecord*>(records);
  hipStream_t st = as_stream(stream);
  return acc_dtype == RRL_F64 ? run_row_coef<double, true>(a, st)
                              : run_row_coef<float, true>(a, st);
}

extern "C" size_t rrl_targets_workspace_bytes(void) { return kTargetsParts * sizeof(int32_t); }

extern "C" int rrl_targets_status(const rrl_policy_params* params, int64_t B, int64_t T, int64_t V,
                                  rrl_view target, void* workspace, int32_t* status,
                                  void* stream) {
  clear_error();
  if (int rc = validate_policy(params, B, T, RRL_F32)) return rc;
  RRL_REQUIRE(V >= 1, RRL_EINVAL, "vocabulary must be non-empty");
  RRL_REQUIRE(workspace && status && (B * T == 0 || target.ptr), RRL_EINVAL,
              "null pointer argument");
  RRL_REQUIRE(target.dtype == RRL_I32 || target.dtype == RRL_I64, RRL_EDTYPE,
              "target ids must be int32 or int64");
  TargetCheckArgs a{};
  a.pp = *params; a.B = B; a.T = T; a.V = V; a.tgt = to_view(target); a.status = status;
  a.part = static_cast<int32_t*>(workspace);
  const int64_t n = B * T;
  hipStream_t st = as_stream(stream);
  if (n <= kTargetsOne) {
    hipLaunchKernelGGL((targets_status_kernel<false>), dim3(1), dim3(1024), 0, st, a);
    return check_launch("targets_status_kernel");
  }
  const int64_t want = (n + 4095) / 4096;
  const int parts = (int)(want < kTargetsParts ? want : kTargetsParts);
  hipLaunchKernelGGL((targets_status_kernel<true>), dim3(parts), dim3(1024), 0, st, a);
  if (int rc = check_launch("targets_status_kernel")) return rc;
  hipLaunchKernelGGL(targets_combine_kernel, dim3(1), dim3(1024), 0, st, a, parts);
  return check_launch("targets_combine_kernel");
}

extern "C" int rrl_check_targets(const rrl_policy_params* params, int64_t B, int64_t T,
                                 int64_t V, rrl_view target, int32_t* status, void* stream) {
  clear_error();
  if (int rc = validate_policy(params, B, T, RRL_F32)) return rc;
  RRL_REQUIRE(V >= 1, RRL_EINVAL, "vocabulary must be non-empty");
  RRL_REQUIRE(status && (B * T == 0 || target.ptr), RRL_EINVAL, "null pointer argument");
  RRL_REQUIRE(target.dtype == RRL_I32 || target.dtype == RRL_I64, RRL_EDTYPE,
              "target ids must be int32 or int64");
  const int64_t n = B * T;
  if (n == 0) return RRL_OK;
  TargetCheckArgs a{};
  a.pp = *params; a.B = B; a.T = T; a.V = V; a.tgt = to_view(target); a.status = status;
  const int64_t blocks = (n + 255) / 256;
  const unsigned grid = (unsigned)(blocks < 4096 ? blocks : 4096);
  hipLaunchKernelGGL(check_targets_kernel, dim3(grid), dim3(256), 0, as_stream(stream), a);
  return check_launch("check_targets_kernel");
}
