// Return and advantage estimators (advantages.py:25-290), masked reductions
// (losses.py:41-50, :104-124, :489-512) and masked whitening.
//
// The reverse recurrences (discounted returns, GAE, skip-observation GAE) are
// affine maps on a small carried state, with padding acting as the identity.
// One workgroup owns one sequence; each lane owns a few consecutive time steps:
//   1. every lane composes the affine map of its steps (reverse time);
//   2. a suffix scan of the lanes' maps (shuffles in a wave, then the waves'
//      maps through LDS) gives each lane its incoming state;
//   3. every lane replays its steps with the reference's step arithmetic from
//      that state and writes the outputs.
#include "rrl_common.hpp"

#include <type_traits>

namespace rrl {

namespace {

// Sets a bit of the caller's status word: with an atomic, or (RRL_STATUS_HOST in
// its address) with plain stores to a word in host memory, which has no atomics
// from here and belongs to this call alone; every writer in one of these
// launches sets the same single bit.
__device__ __forceinline__ void or_flag(int32_t* status, int32_t bit) {
  const uintptr_t at = reinterpret_cast<uintptr_t>(status);
  if (at & RRL_STATUS_HOST) {
    volatile int32_t* p = reinterpret_cast<volatile int32_t*>(at - RRL_STATUS_HOST);
    *p = *p | bit;
    __threadfence_system();
  } else {
    raise_flag(status, bit);
  }
}

struct ScanArgs {
  int64_t B, T;
  View r, v, nv;      // rewards, values / action_end_values, next_action_values
  View term, valid;   // optional (ptr == nullptr)
  View boot;          // optional [B]
  double gamma, lam;
  void* out0;         // returns / advantages
  void* out1;         // value targets
  int odt;
};

// Per-estimator recurrences.  KIND 0: discounted returns (state: the return).
// KIND 1: GAE (state: next value, next advantage).  KIND 2: skip-observation
// GAE (state: next advantage).
template <int KIND> struct StateDim { static constexpr int D = KIND == 1 ? 2 : 1; };

// A run of steps as a map on the carried state, S' = m S + c.  Padding is the
// identity.  Maps and states between lanes are float64: composed in float32
// they left 64 x 8192 advantages further from 64 bits than the serial walk.
template <typename Acc, int KIND>
struct Run {
  Acc m = Acc(1), c = Acc(0);
  // This run preceded in time by one step with S' = sm S + sc.
  __device__ __forceinline__ void step(Acc sm, Acc sc) {
    c = sc + sm * c;
    m = sm * m;
  }
  // This run applied after `later`.
  __device__ __forceinline__ void after(const Run& later) {
    c = c + m * later.c;
    m = m * later.m;
  }
  __device__ __forceinline__ void apply(Acc (&S)[1]) const { S[0] = c + m * S[0]; }
  template <class F>
  __device__ __forceinline__ Run moved(F f) const {
    Run r;
    r.m = f(m);
    r.c = f(c);
    return r;
  }
};
// GAE: a run with a valid step leaves the value of its first one and an
// advantage affine in the state; the value is carried as such (a product with
// zero would turn an infinite value further on into NaN).
template <typename Acc>
struct Run<Acc, 1> {
  int any = 0;
  Acc v = Acc(0), c = Acc(0), mv = Acc(0), ma = Acc(1);
  // One valid step: delta = rv + gn V', A = delta + gln A', V = sv.
  __device__ __forceinline__ void step(Acc sv, Acc rv, Acc gn, Acc gln) {
    c = any ? (rv + gn * v) + gln * c : rv;
    mv = any ? gln * mv : gn;
    ma = any ? gln * ma : gln;
    v = sv;
    any = 1;
  }
  __device__ __forceinline__ void after(const Run& later) {
    if (!any) {
      *this = later;
    } else if (later.any) {
      c = (c + mv * later.v) + ma * later.c;
      mv = ma * later.mv;
      ma = ma * later.ma;
    }
  }
  __device__ __forceinline__ void apply(Acc (&S)[2]) const {
    if (any) {
      S[1] = (c + mv * S[0]) + ma * S[1];
      S[0] = v;
    }
  }
  template <class F>
  __device__ __forceinline__ Run moved(F f) const {
    Run r;
    r.any = f(any);
    r.v = f(v);
    r.c = f(c);
    r.mv = f(mv);
    r.ma = f(ma);
    return r;
  }
};

// The runs of the wave's later lanes composed (`later`), and the whole wave's.
template <class R>
__device__ __forceinline__ void wave_suffix(const R& f, R& later, R& whole) {
  const int lane = threadIdx.x & 63;
  R p = f;  // this lane's run after those of the lanes behind it
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const R o = p.moved([&](auto x) { return __shfl_down(x, d, 64); });
    if (lane + d < 64) p.after(o);
  }
  later = p.moved([&](auto x) { return __shfl_down(x, 1, 64); });
  whole = p.moved([&](auto x) { return __shfl(x, 0, 64); });
  if (lane == 63) later = R{};
}

// Four consecutive steps of an operand: one 16-byte load of contiguous aligned
// float32 (VEC), or element by element.
template <typename Acc, bool VEC>
__device__ __forceinline__ void load_steps(const View& v, int64_t b, int64_t t, int64_t T,
                                           Acc (&x)[4]) {
  if constexpr (VEC) {
    const float4 u = *reinterpret_cast<const float4*>(static_cast<const float*>(v.ptr) + b * v.sr + t);
    x[0] = u.x; x[1] = u.y; x[2] = u.z; x[3] = u.w;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = t + i < T ? v.get<Acc>(b, t + i) : Acc(0);
  }
}
template <bool VEC>
__device__ __forceinline__ uint32_t load_flags(const View& v, int64_t b, int64_t t, int64_t T,
                                               bool absent) {
  if (!v.present()) return absent ? 0xFu : 0u;
  uint32_t f = 0;
  if constexpr (VEC) {
    const uint32_t u =
        *reinterpret_cast<const uint32_t*>(static_cast<const uint8_t*>(v.ptr) + b * v.sr + t);
#pragma unroll
    for (int i = 0; i < 4; ++i) f |= (u >> (8 * i) & 0xFFu) ? 1u << i : 0u;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) f |= t + i < T && v.truth(b, t + i) ? 1u << i : 0u;
  }
  return f;
}

// One step (the kind's reference: advantages.py:75-79, :129-139, :196-210)
// as an addition to a run and in the
// reference's own arithmetic.
template <typename Acc, int KIND>
struct Step {
  static constexpr int D = StateDim<KIND>::D;
  Acc r, v, nv;
  bool valid, term;
  __device__ __forceinline__ void add_to(Run<double, KIND>& f, Acc g, Acc gl) const {
    if (!valid) return;
    const Acc nt = term ? Acc(0) : Acc(1);
    if constexpr (KIND == 0) f.step(g * nt, r);
    if constexpr (KIND == 1) f.step(v, r - v, g * nt, gl * nt);
    if constexpr (KIND == 2) f.step(gl * nt, (r + (g * nt) * nv) - v);
  }
  __device__ __forceinline__ void replay(Acc g, Acc gl, Acc (&S)[D], Acc& o0, Acc& o1) const {
    const Acc nt = term ? Acc(0) : Acc(1);
    if (KIND == 0) {
      const Acc cand = r + (g * nt) * S[0];
      if (valid) S[0] = cand;
      o0 = valid ? S[0] : Acc(0);
      o1 = Acc(0);
    } else if (KIND == 1) {
      const Acc delta = (r + (g * nt) * S[0]) - v;
      const Acc cand = delta + (gl * nt) * S[1];
      const Acc adv = valid ? cand : Acc(0);
      o0 = adv;
      o1 = valid ? adv + v : Acc(0);
      if (valid) { S[0] = v; S[1] = adv; }
    } else {
      const Acc delta = (r + (g * nt) * nv) - v;
      const Acc cand = delta + (gl * nt) * S[0];
      const Acc adv = valid ? cand : Acc(0);
      o0 = adv;
      o1 = valid ? adv + v : Acc(0);
      if (valid) S[0] = adv;
    }
  }
};

// Latency bounds the scan: 64 sequences of 8192 steps are 9 MB, but a sequence
// is one dependent chain.  A lane holds E = 4 or 8 consecutive steps in
// registers (read once, 16 bytes at a time where the layout allows), a wave
// scans its lanes' runs with shuffles, and each wave carries the incoming
// state through the later waves' runs (up to 15 of them), so a
// tile of NT * E steps costs one barrier; longer sequences go tile by tile
// from the end.  rrl_gae at 64 x 8192: 57.7 us before (32-step chunks read
// twice, 16 barriers), 11.0 us here (9.2 with float32 maps).
template <typename Acc, int KIND, int NT, int E, bool VEC>
__global__ __launch_bounds__(NT) void reverse_scan_kernel(ScanArgs a) {
  constexpr int D = StateDim<KIND>::D;
  constexpr int NW = NT / 64;
  // Raw storage: the runs have initialisers, which LDS cannot.
  __shared__ __align__(16) char sh_raw[2 * NW * sizeof(Run<double, KIND>)];
  auto* sh_wave = reinterpret_cast<Run<double, KIND>*>(sh_raw);
  // gamma and gamma*lambda as the reference forms them: python float products
  // rounded to the tensor dtype.
  const Acc g = (Acc)a.gamma;
  const Acc gl = (Acc)(a.gamma * a.lam);
  const int wave = threadIdx.x >> 6;
  const int64_t tile = (int64_t)NT * E;
  for (int64_t b = blockIdx.x; b < a.B; b += gridDim.x) {
    // The state behind the tile: at first the bootstrap value.
    double C[D];
    C[0] = KIND != 2 && a.boot.present() ? a.boot.get<Acc>(b, 0) : Acc(0);
    if (D == 2) C[D - 1] = 0.0;
    int buf = 0;
    for (int64_t base = (a.T - 1) / tile * tile; base >= 0; base -= tile, buf ^= 1) {
      const int64_t t0 = base + (int64_t)threadIdx.x * E;
      Step<Acc, KIND> st[E];
#pragma unroll
      for (int e = 0; e < E; e += 4) {
        const int64_t t = t0 + e;
        Acc r[4] = {}, v[4] = {}, nv[4] = {};
        uint32_t ok = 0, term = 0;
        if (t < a.T) {
          load_steps<Acc, VEC>(a.r, b, t, a.T, r);
          if (KIND != 0) load_steps<Acc, VEC>(a.v, b, t, a.T, v);
          if (KIND == 2) load_steps<Acc, VEC>(a.nv, b, t, a.T, nv);
          ok = load_flags<VEC>(a.valid, b, t, a.T, true);
          term = load_flags<VEC>(a.term, b, t, a.T, false);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
          st[e + i] = {r[i], v[i], nv[i], (ok >> i & 1u) && t + i < a.T, (term >> i & 1u) != 0};
      }
      Run<double, KIND> f, later, whole;
#pragma unroll
      for (int e = E - 1; e >= 0; --e) st[e].add_to(f, g, gl);
      wave_suffix(f, later, whole);
      if ((threadIdx.x & 63) == 0) sh_wave[buf * NW + wave] = whole;
      __syncthreads();
      // Every wave carries the tile's incoming state down to its own end, and
      // on through the rest for the next tile's.
      double in[D];
#pragma unroll
      for (int i = 0; i < D; ++i) in[i] = C[i];
#pragma unroll
      for (int w = NW - 1; w >= 0; --w) {
        if (w == wave) {
#pragma unroll
          for (int i = 0; i < D; ++i) in[i] = C[i];
        }
        sh_wave[buf * NW + w].apply(C);
      }
      later.apply(in);
      Acc S[D];
#pragma unroll
      for (int i = 0; i < D; ++i) S[i] = (Acc)in[i];
      Acc o0[E], o1[E];
#pragma unroll
      for (int e = E - 1; e >= 0; --e) st[e].replay(g, gl, S, o0[e], o1[e]);
#pragma unroll
      for (int e = 0; e < E; e += 4) {
        const int64_t t = t0 + e;
        if constexpr (VEC) {
          if (t < a.T) {
            float* p = static_cast<float*>(a.out0) + b * a.T + t;
            *reinterpret_cast<float4*>(p) =
                make_float4((float)o0[e], (float)o0[e + 1], (float)o0[e + 2], (float)o0[e + 3]);
            if (KIND != 0) {
              float* q = static_cast<float*>(a.out1) + b * a.T + t;
              *reinterpret_cast<float4*>(q) =
                  make_float4((float)o1[e], (float)o1[e + 1], (float)o1[e + 2], (float)o1[e + 3]);
            }
          }
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            if (t + i >= a.T) continue;
            store_as<Acc>(a.out0, a.odt, b * a.T + t + i, o0[e + i]);
            if (KIND != 0) store_as<Acc>(a.out1, a.odt, b * a.T + t + i, o1[e + i]);
          }
        }
      }
    }
    __syncthreads();  // the next sequence writes sh_wave again
  }
}

// Contiguous float32 steps at 16-byte aligned rows.
bool vec_steps(const View& v, bool used) {
  return !used || (v.dt == RRL_F32 && v.sc == 1 && v.sr % 4 == 0 && (uintptr_t)v.ptr % 16 == 0);
}
// Contiguous one-byte flags at 4-byte aligned rows, or none.
bool vec_flags(const View& v) {
  return !v.present() || ((v.dt == RRL_BOOL || v.dt == RRL_U8 || v.dt == RRL_I8) && v.sc == 1 &&
                          v.sr % 4 == 0 && (uintptr_t)v.ptr % 4 == 0);
}

template <typename Acc, int KIND, bool VEC>
int launch_scan_as(const ScanArgs& a, hipStream_t st) {
  const unsigned grid = (unsigned)(a.B < 65536 ? a.B : 65536);
  // One wave for short sequences: no other wave's map to carry the state through.
  if (a.T <= 256)
    hipLaunchKernelGGL((reverse_scan_kernel<Acc, KIND, 64, 4, VEC>), dim3(grid), dim3(64), 0, st, a);
  else if (a.T <= 1024)
    hipLaunchKernelGGL((reverse_scan_kernel<Acc, KIND, 256, 4, VEC>), dim3(grid), dim3(256), 0, st,
                       a);
  else
    hipLaunchKernelGGL((reverse_scan_kernel<Acc, KIND, 1024, 8, VEC>), dim3(grid), dim3(1024), 0,
                       st, a);
  return check_launch("reverse_scan_kernel");
}

template <int KIND>
int launch_scan(const ScanArgs& a, bool f64, hipStream_t st) {
  if (a.B * a.T == 0) return RRL_OK;
  if (f64) return launch_scan_as<double, KIND, false>(a, st);
  const bool vec = a.T % 4 == 0 && vec_steps(a.r, true) && vec_steps(a.v, KIND != 0) &&
                   vec_steps(a.nv, KIND == 2) && vec_flags(a.term) && vec_flags(a.valid) &&
                   a.odt == RRL_F32 && (uintptr_t)a.out0 % 16 == 0 &&
                   (KIND == 0 || (uintptr_t)a.out1 % 16 == 0);
  return vec ? launch_scan_as<float, KIND, true>(a, st) : launch_scan_as<float, KIND, false>(a, st);
}

// ---------------------------------------------------------------------------
// Group statistics: one lane per group (groups are small: G = 4..64 in GRPO).
// ---------------------------------------------------------------------------
template <typename Acc>
__global__ void group_std_kernel(int64_t n, int64_t G, View r, Acc eps, void* out, int odt) {
  for (int64_t gi = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; gi < n;
       gi += (int64_t)gridDim.x * blockDim.x) {
    Acc sum = Acc(0);
    Acc lo = r.get<Acc>(gi, 0), hi = lo;
    for (int64_t k = 0; k < G; ++k) {
      const Acc x = r.get<Acc>(gi, k);
      sum += x;
      lo = x < lo ? x : lo;
      hi = x > hi ? x : hi;
    }
    const Acc mean = sum / (Acc)G;
    Acc ss = Acc(0);
    for (int64_t k = 0; k < G; ++k) {
      const Acc d = r.get<Acc>(gi, k) - mean;
      ss += d * d;
    }
    // A uniform group has std 0 exactly ("uniform-reward groups return exactly
    // zero", advantages.py:243-244): the float mean of a non-dyadic value is
    // often an ulp off, which would otherwise leave a std above eps.
    const Acc sd = hi == lo ? Acc(0) : M<Acc>::sqrt(ss / (Acc)G);
    const Acc den = sd > eps ? sd : eps;  // clamp_min(eps) (advantages.py:257)
    for (int64_t k = 0; k < G; ++k) {
      const Acc z = (r.get<Acc>(gi, k) - mean) / den;
      store_as<Acc>(out, odt, gi * G + k, sd > eps ? z : Acc(0));
    }
  }
}

template <typename Acc>
__global__ void leave_one_out_kernel(int64_t n, int64_t G, View r, void* out, int odt) {
  for (int64_t gi = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; gi < n;
       gi += (int64_t)gridDim.x * blockDim.x) {
    Acc sum = Acc(0);
    for (int64_t k = 0; k < G; ++k) sum += r.get<Acc>(gi, k);
    for (int64_t k = 0; k < G; ++k) {
      const Acc x = r.get<Acc>(gi, k);
      store_as<Acc>(out, odt, gi * G + k, x - (sum - x) / (Acc)(G - 1));
    }
  }
}

// out[b, t] = mask ? turn_adv[b, id] : 0 (advantages.py:282-290).  The value is
// copied through the accumulation type, which round-trips every float dtype.
template <typename Acc>
__global__ void broadcast_turn_kernel(int64_t B, int64_t K, int64_t T, View adv, View ids,
                                      View mask, void* out, int odt, int32_t* status) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < B * T;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t b = i / T, t = i - (i / T) * T;
    const bool m = mask.truth(b, t);
    const int64_t id = load_as<int64_t>(ids.ptr, ids.dt, b * ids.sr + t * ids.sc);
    Acc v = Acc(0);
    if (m) {
      if (id < 0 || id >= K) {
        or_flag(status, RRL_FLAG_INVALID_TURN);
      } else {
        v = adv.get<Acc>(b, id);
      }
    }
    store_as<Acc>(out, odt, i, v);
  }
}

// ---------------------------------------------------------------------------
// Flat masked reductions over [B, T]: per-block partials, then every consumer
// re-sums the partials in block order (deterministic, no atomics).
// ---------------------------------------------------------------------------
constexpr int RED_NT = 256;
constexpr int RED_MAXB = 1024;

struct RedArgs {
  int64_t B, T;
  View x, mask;
  void* part;      // Acc[RED_MAXB][4]
  double eps;
  int shift;
  void* out;
  int odt;
  int32_t* status;
  const void* grad;
};

inline unsigned red_grid(int64_t n) {
  int64_t g = (n + RED_NT * 8 - 1) / (RED_NT * 8);
  if (g < 1) g = 1;
  if (g > RED_MAXB) g = RED_MAXB;
  return (unsigned)g;
}

// Sum of a partial column over all blocks, in block order.
template <typename Acc>
__device__ void sum_partials(const Acc* part, int nb, int col, Acc& out, Acc* sh) {
  Acc v[1] = {Acc(0)};
  for (int i = threadIdx.x; i < nb; i += RED_NT) v[0] += part[i * 4 + col];
  block_sum<RED_NT, 1, Acc>(v, sh);
  out = v[0];
}

// masked_mean: part = (sum w*x, sum w).
template <typename Acc>
__global__ __launch_bounds__(RED_NT) void masked_partials_kernel(RedArgs a) {
  __shared__ Acc sh[(RED_NT / 64) * 2];
  Acc* part = static_cast<Acc*>(a.part);
  Acc v[2] = {Acc(0), Acc(0)};
  const int64_t n = a.B * a.T;
  for (int64_t i = blockIdx.x * (int64_t)RED_NT + threadIdx.x; i < n; i += (int64_t)gridDim.x * RED_NT) {
    const int64_t b = i / a.T, t = i - (i / a.T) * a.T;
    const Acc w = a.mask.get<Acc>(b, t);
    const Acc x = a.x.get<Acc>(b, t);
    v[0] += x * w;
    v[1] += w;
  }
  block_sum<RED_NT, 2, Acc>(v, sh);
  if (threadIdx.x == 0) {
    part[blockIdx.x * 4 + 0] = v[0];
    part[blockIdx.x * 4 + 1] = v[1];
  }
}

// masked_mean finalize: out = sum(w*x) / sum(w).
template <typename Acc>
__global__ __launch_bounds__(RED_NT) void masked_mean_final_kernel(RedArgs a, int nb) {
  __shared__ Acc sh[RED_NT / 64];
  Acc s0, s1;
  sum_partials<Acc>(static_cast<const Acc*>(a.part), nb, 0, s0, sh);
  sum_partials<Acc>(static_cast<const Acc*>(a.part), nb, 1, s1, sh);
  if (threadIdx.x == 0) {
    if (s1 == Acc(0)) or_flag(a.status, RRL_FLAG_EMPTY_MASK);
    static_cast<Acc*>(a.out)[0] = s0 / s1;
    static_cast<Acc*>(a.part)[RED_MAXB * 4] = s1;  // denominator for the backward
  }
}

template <typename Acc>
__global__ __launch_bounds__(RED_NT) void masked_mean_bwd_kernel(RedArgs a) {
  const Acc G = static_cast<const Acc*>(a.grad)[0];
  const Acc den = static_cast<const Acc*>(a.part)[RED_MAXB * 4];
  const int64_t n = a.B * a.T;
  for (int64_t i = blockIdx.x * (int64_t)RED_NT + threadIdx.x; i < n; i += (int64_t)gridDim.x * RED_NT) {
    const int64_t b = i / a.T, t = i - (i / a.T) * a.T;
    static_cast<Acc*>(a.out)[i] = (G / den) * a.mask.get<Acc>(b, t);
  }
}

// Masked whitening in two launches.  The first forms each tile's count, mean
// and sum of squared deviations from the tile's own mean (the tile sits in
// registers, so that is a two-pass sum without a second read) and merges a
// workgroup's tiles; the second merges the workgroups' and writes.  Bytes are
// few (64 x 8192: 4.7 MB); launches, a lane's serial loads (each waited for
// behind its type's branch) and the 64-bit division per element that strided
// operands need bounded it: three launches took 24 us, two 15.7.  Float32
// values with one-byte flags are read four at a time, and the second launch's
// first tile is requested before the moments are merged: 7.8 us, and GAE +
// whitening of 64 x 8192 50.2 -> 42.3 us per pass.
constexpr int WH_E = 8;  // elements per lane and tile

// (count, mean, M2) <- merged with another group's.  The squared distance of
// the means may pass the type's range where the deviations' squares do not, so
// it is only formed times the weight; means further apart than the range keep a
// finite mean and give an infinite M2, as the sum of squares would be.
template <typename Acc>
struct Moments {
  Acc n, mean, m2;
  __device__ __forceinline__ void merge(Acc n2, Acc mean2, Acc m22) {
    if (n2 == Acc(0)) return;
    if (n == Acc(0)) {
      n = n2, mean = mean2, m2 = m22;
      return;
    }
    const Acc nt = n + n2, d = mean2 - mean, f = n2 / nt;
    const bool apart = d - d != Acc(0) && mean - mean == Acc(0) && mean2 - mean2 == Acc(0);
    mean = apart ? mean * (n / nt) + mean2 * f : mean + d * f;
    m2 += m22 + (d * (n * f)) * d;
    n = nt;
  }
};

// Element offsets of flat index i: FLAT operands are contiguous as a whole.
template <bool FLAT>
__device__ __forceinline__ void split_index(const RedArgs& a, int64_t i, int64_t& b, int64_t& t) {
  if constexpr (FLAT) {
    b = 0;
    t = i;
  } else {
    b = i / a.T;
    t = i - b * a.T;
  }
}

// How a whitening kernel reads its operands: VEC, float32 values (and results)
// and one-byte flags, each contiguous as a whole, four elements per load; FLAT,
// contiguous operands of any type; STRIDED, rows of any strides.
enum WhitenPath { WH_STRIDED, WH_FLAT, WH_VEC };

// A tile's elements of this lane: element e is flat index tile_index(i0, e).
template <int PATH>
__device__ __forceinline__ int64_t tile_index(int64_t i0, int e) {
  if constexpr (PATH == WH_VEC)
    return i0 + (int64_t)(e / 4) * RED_NT * 4 + threadIdx.x * 4 + e % 4;
  else
    return i0 + e * RED_NT + threadIdx.x;
}

// The values and flags of the tile at i0 (0 and unset past the end).
template <typename Acc, int PATH>
__device__ __forceinline__ void load_tile(const RedArgs& a, int64_t i0, int64_t n, Acc (&x)[WH_E],
                                          bool (&m)[WH_E]) {
  if constexpr (PATH == WH_VEC) {
    const float* xp = static_cast<const float*>(a.x.ptr);
    const uint8_t* mp = static_cast<const uint8_t*>(a.mask.ptr);
#pragma unroll
    for (int e = 0; e < WH_E; e += 4) {
      const int64_t i = tile_index<PATH>(i0, e);
      float4 f = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      uint32_t w = 0;
      if (i + 4 <= n) {
        f = *reinterpret_cast<const float4*>(xp + i);
        w = *reinterpret_cast<const uint32_t*>(mp + i);
      } else {  // the last one to three elements
        if (i < n) f.x = xp[i], w = mp[i];
        if (i + 1 < n) f.y = xp[i + 1], w |= (uint32_t)mp[i + 1] << 8;
        if (i + 2 < n) f.z = xp[i + 2], w |= (uint32_t)mp[i + 2] << 16;
      }
      x[e] = f.x, x[e + 1] = f.y, x[e + 2] = f.z, x[e + 3] = f.w;
#pragma unroll
      for (int k = 0; k < 4; ++k) m[e + k] = (w >> (8 * k) & 0xffu) != 0;
    }
  } else {
#pragma unroll
    for (int e = 0; e < WH_E; ++e) {
      const int64_t i = tile_index<PATH>(i0, e);
      m[e] = false;
      x[e] = Acc(0);
      if (i < n) {
        int64_t b, t;
        split_index<PATH == WH_FLAT>(a, i, b, t);
        m[e] = a.mask.truth(b, t);
        x[e] = a.x.get<Acc>(b, t);
      }
    }
  }
}

template <typename Acc, int PATH>
__global__ __launch_bounds__(RED_NT) void whiten_moments_kernel(RedArgs a) {
  __shared__ Acc sh[(RED_NT / 64) * 2];
  Acc* part = static_cast<Acc*>(a.part);
  const int64_t n = a.B * a.T;
  constexpr int64_t kTile = (int64_t)RED_NT * WH_E;
  Moments<Acc> q{Acc(0), Acc(0), Acc(0)};
  for (int64_t i0 = blockIdx.x * kTile; i0 < n; i0 += (int64_t)gridDim.x * kTile) {
    Acc x[WH_E];
    bool m[WH_E];
    Acc v[2] = {Acc(0), Acc(0)};
    load_tile<Acc, PATH>(a, i0, n, x, m);
#pragma unroll
    for (int e = 0; e < WH_E; ++e)
      if (m[e]) {
        v[0] += x[e];
        v[1] += Acc(1);
      }
    block_sum<RED_NT, 2, Acc>(v, sh);
    const Acc mean = v[1] != Acc(0) ? v[0] / v[1] : Acc(0);
    Acc s[1] = {Acc(0)};
#pragma unroll
    for (int e = 0; e < WH_E; ++e) {
      const Acc d = x[e] - mean;
      if (m[e]) s[0] += d * d;
    }
    block_sum<RED_NT, 1, Acc>(s, sh);
    q.merge(v[1], mean, s[0]);
  }
  if (threadIdx.x == 0) {
    part[blockIdx.x * 4 + 0] = q.n * q.mean;
    part[blockIdx.x * 4 + 1] = q.n;
    part[blockIdx.x * 4 + 2] = q.m2;
  }
}

template <typename Acc, int PATH>
__global__ __launch_bounds__(RED_NT) void whiten_write_kernel(RedArgs a, int nb) {
  __shared__ Acc sh[(RED_NT / 64) * 2];
  const Acc* part = static_cast<const Acc*>(a.part);
  const int64_t n = a.B * a.T;
  constexpr int64_t kTile = (int64_t)RED_NT * WH_E;
  // The first tile is on its way while the moments are merged.
  int64_t i0 = blockIdx.x * kTile;
  Acc x[WH_E];
  bool m[WH_E];
  load_tile<Acc, PATH>(a, i0, n, x, m);
  Acc v[2] = {Acc(0), Acc(0)};
  for (int i = threadIdx.x; i < nb; i += RED_NT) {
    v[0] += part[i * 4 + 0];
    v[1] += part[i * 4 + 1];
  }
  block_sum<RED_NT, 2, Acc>(v, sh);
  if (blockIdx.x == 0 && threadIdx.x == 0 && v[1] == Acc(0)) or_flag(a.status, RRL_FLAG_EMPTY_MASK);
  const Acc mean = v[0] / v[1];
  Acc s2[1] = {Acc(0)};
  for (int i = threadIdx.x; i < nb; i += RED_NT) {
    const Acc ni = part[i * 4 + 1];
    const Acc d = ni != Acc(0) ? part[i * 4 + 0] / ni - mean : Acc(0);
    s2[0] += part[i * 4 + 2] + ni * d * d;
  }
  block_sum<RED_NT, 1, Acc>(s2, sh);
  const Acc sd = M<Acc>::sqrt(s2[0] / v[1]);
  const Acc den = sd + (Acc)a.eps;
  while (i0 < n) {
    Acc y[WH_E];
#pragma unroll
    for (int e = 0; e < WH_E; ++e) {
      const Acc z = a.shift ? (x[e] - mean) / den : x[e] / den;
      y[e] = m[e] ? z : Acc(0);
    }
    if constexpr (PATH == WH_VEC) {
      float* out = static_cast<float*>(a.out);
#pragma unroll
      for (int e = 0; e < WH_E; e += 4) {
        const int64_t i = tile_index<PATH>(i0, e);
        if (i + 4 <= n) {
          *reinterpret_cast<float4*>(out + i) = make_float4(y[e], y[e + 1], y[e + 2], y[e + 3]);
        } else {
          if (i < n) out[i] = y[e];
          if (i + 1 < n) out[i + 1] = y[e + 1];
          if (i + 2 < n) out[i + 2] = y[e + 2];
        }
      }
    } else {
#pragma unroll
      for (int e = 0; e < WH_E; ++e) {
        const int64_t i = tile_index<PATH>(i0, e);
        if (i < n) store_as<Acc>(a.out, a.odt, i, y[e]);
      }
    }
    i0 += (int64_t)gridDim.x * kTile;
    if (i0 < n) load_tile<Acc, PATH>(a, i0, n, x, m);
  }
}

template <typename Acc, int PATH>
int launch_whiten_as(const RedArgs& a, unsigned nb, hipStream_t st) {
  hipLaunchKernelGGL((whiten_moments_kernel<Acc, PATH>), dim3(nb), dim3(RED_NT), 0, st, a);
  hipLaunchKernelGGL((whiten_write_kernel<Acc, PATH>), dim3(nb), dim3(RED_NT), 0, st, a, (int)nb);
  return check_launch("masked_whiten");
}

template <typename Acc>
int launch_whiten(const RedArgs& a, unsigned nb, hipStream_t st) {
  const auto flat = [&](const View& v) { return v.sc == 1 && (v.sr == a.T || a.B == 1); };
  if (!flat(a.x) || !flat(a.mask)) return launch_whiten_as<Acc, WH_STRIDED>(a, nb, st);
  if constexpr (std::is_same<Acc, float>::value) {
    const auto aligned = [](const void* p, uintptr_t by) { return (uintptr_t)p % by == 0; };
    const int md = a.mask.dt;
    if (a.x.dt == RRL_F32 && a.odt == RRL_F32 && aligned(a.x.ptr, 16) && aligned(a.out, 16) &&
        (md == RRL_BOOL || md == RRL_U8 || md == RRL_I8) && aligned(a.mask.ptr, 4))
      return launch_whiten_as<Acc, WH_VEC>(a, nb, st);
  }
  return launch_whiten_as<Acc, WH_FLAT>(a, nb, st);
}

// sequence_log_ratio: one workgroup per row.
template <typename Acc>
__global__ __launch_bounds__(RED_NT) void seq_log_ratio_kernel(int64_t B, int64_t T, View cur,
                                                               View old, View mask, int norm,
                                                               Acc* out, Acc* counts,
                                                               int32_t* status) {
  __shared__ Acc sh[(RED_NT / 64) * 2];
  for (int64_t b = blockIdx.x; b < B; b += gridDim.x) {
    Acc v[2] = {Acc(0), Acc(0)};
    for (int64_t t = threadIdx.x; t < T; t += RED_NT) {
      const Acc w = mask.get<Acc>(b, t);
      v[0] += (cur.get<Acc>(b, t) - old.get<Acc>(b, t)) * w;
      v[1] += w;
    }
    block_sum<RED_NT, 2, Acc>(v, sh);
    if (threadIdx.x == 0) {
      if (v[1] == Acc(0)) or_flag(status, RRL_FLAG_EMPTY_ROW);
      out[b] = norm ? v[0] / v[1] : v[0];
      counts[b] = v[1];
    }
  }
}

template <typename Acc>
__global__ void seq_log_ratio_bwd_kernel(int64_t B, int64_t T, View mask, int norm,
                                         const Acc* counts, const Acc* grad, Acc* gcur) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < B * T;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t b = i / T, t = i - (i / T) * T;
    const Acc w = mask.get<Acc>(b, t);
    gcur[i] = norm ? (grad[b] / counts[b]) * w : grad[b] * w;
  }
}

template <typename Acc>
__global__ void double_sided_kernel(int64_t n, const void* r, int dt, Acc lo, Acc hi, uint8_t* out) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const Acc x = load_as<Acc>(r, dt, i);
    out[i] = (x > lo && x < hi) ? 1 : 0;
  }
}

inline unsigned flat_grid(int64_t n, int nt) {
  int64_t g = (n + nt - 1) / nt;
  if (g < 1) g = 1;
  if (g > 65536) g = 65536;
  return (unsigned)g;
}

bool view_ok(const rrl_view& v) { return v.ptr == nullptr || is_known_dtype(v.dtype); }

}  // namespace
}  // namespace rrl

using namespace rrl;

static int scan_common(int kind, int64_t B, int64_t T, rrl_view rewards, rrl_view v1, rrl_view v2,
                       rrl_view terminated, rrl_view valid, rrl_view bootstrap, double gamma,
                       double lam, void* out0, void* out1, int32_t out_dtype, void* stream) {
  clear_error();
  RRL_REQUIRE(B >= 0 && T >= 0, RRL_EINVAL, "negative size");
  RRL_REQUIRE(is_float_dtype(out_dtype), RRL_EDTYPE, "output dtype must be floating point");
  RRL_REQUIRE(B * T == 0 || (rewards.ptr && out0), RRL_EINVAL, "null pointer argument");
  RRL_REQUIRE(view_ok(terminated) && view_ok(valid) && view_ok(bootstrap), RRL_EDTYPE,
              "unsupported dtype");
  ScanArgs a{};
  a.B = B; a.T = T;
  a.r = to_view(rewards); a.v = to_view(v1); a.nv = to_view(v2);
  a.term = to_view(terminated); a.valid = to_view(valid); a.boot = to_view(bootstrap);
  a.gamma = gamma; a.lam = lam; a.out0 = out0; a.out1 = out1; a.odt = out_dtype;
  const bool f64 = out_dtype == RRL_F64;
  hipStream_t st = as_stream(stream);
  if (kind == 0) return launch_scan<0>(a, f64, st);
  if (kind == 1) return launch_scan<1>(a, f64, st);
  return launch_scan<2>(a, f64, st);
}

extern "C" int rrl_discounted_returns(int64_t B, int64_t T, rrl_view rewards, rrl_view terminated,
                                      rrl_view valid, rrl_view bootstrap, double gamma, void* out,
                                      int32_t out_dtype, void* stream) {
  rrl_view none{nullptr, RRL_F32, 0, 0};
  return scan_common(0, B, T, rewards, none, none, terminated, valid, bootstrap, gamma, 1.0, out,
                     nullptr, out_dtype, stream);
}

extern "C" int rrl_gae(int64_t B, int64_t T, rrl_view rewards, rrl_view values,
                       rrl_view terminated, rrl_view valid, rrl_view bootstrap, double gamma,
                       double gae_lambda, void* adv_out, void* targets_out, int32_t out_dtype,
                       void* stream) {
  if (B * T != 0 && (!values.ptr || !targets_out)) {
    set_error("values and targets_out are required");
    return RRL_EINVAL;
  }
  rrl_view none{nullptr, RRL_F32, 0, 0};
  return scan_common(1, B, T, rewards, values, none, terminated, valid, bootstrap, gamma,
                     gae_lambda, adv_out, targets_out, out_dtype, stream);
}

extern "C" int rrl_skip_observation_gae(int64_t B, int64_t T, rrl_view rewards,
                                        rrl_view action_end_values, rrl_view next_action_values,
                                        rrl_view terminated, rrl_view valid, double gamma,
                                        double gae_lambda, void* adv_out, void* targets_out,
                                        int32_t out_dtype, void* stream) {
  if (B * T != 0 && (!action_end_values.ptr || !next_action_values.ptr || !targets_out)) {
    set_error("value inputs and targets_out are required");
    return RRL_EINVAL;
  }
  rrl_view none{nullptr, RRL_F32, 0, 0};
  return scan_common(2, B, T, rewards, action_end_values, next_action_values, terminated, valid,
                     none, gamma, gae_lambda, adv_out, targets_out, out_dtype, stream);
}

extern "C" int rrl_group_standardize(int64_t n_groups, int64_t G, rrl_view rewards, double eps,
                                     void* out, int32_t out_dtype, void* stream) {
  clear_error();
  RRL_REQUIRE(n_groups >= 0 && G >= 1, RRL_EINVAL, "bad group shape");
  RRL_REQUIRE(is_float_dtype(out_dtype) && is_float_dtype(rewards.dtype), RRL_EDTYPE,
              "rewards must be floating point");
  if (n_groups == 0) return RRL_OK;
  RRL_REQUIRE(rewards.ptr && out, RRL_EINVAL, "null pointer argument");
  hipStream_t st = as_stream(stream);
  const unsigned grid = flat_grid(n_groups, 256);
  if (out_dtype == RRL_F64)
    hipLaunchKernelGGL((group_std_kernel<double>), dim3(grid), dim3(256), 0, st, n_groups, G,
                       to_view(rewards), (double)eps, out, (int)out_dtype);
  else
    hipLaunchKernelGGL((group_std_kernel<float>), dim3(grid), dim3(256), 0, st, n_groups, G,
                       to_view(rewards), (float)eps, out, (int)out_dtype);
  return check_launch("group_std_kernel");
}

extern "C" int rrl_leave_one_out(int64_t n_groups, int64_t G, rrl_view rewards, void* out,
                                 int32_t out_dtype, void* stream) {
  clear_error();
  RRL_REQUIRE(n_groups >= 0 && G >= 2, RRL_EINVAL, "leave-one-out needs G >= 2");
  RRL_REQUIRE(is_float_dtype(out_dtype) && is_float_dtype(rewards.dtype), RRL_EDTYPE,
              "rewards must be floating point");
  if (n_groups == 0) return RRL_OK;
  RRL_REQUIRE(rewards.ptr && out, RRL_EINVAL, "null pointer argument");
  hipStream_t st = as_stream(stream);
  const unsigned grid = flat_grid(n_groups, 256);
  if (out_dtype == RRL_F64)
    hipLaunchKernelGGL((leave_one_out_kernel<double>), dim3(grid), dim3(256), 0, st, n_groups, G,
                       to_view(rewards), out, (int)out_dtype);
  else
    hipLaunchKernelGGL((leave_one_out_kernel<float>), dim3(grid), dim3(256), 0, st, n_groups, G,
                       to_view(rewards), out, (int)out_dtype);
  return check_launch("leave_one_out_kernel");
}

extern "C" int rrl_broadcast_turn(int64_t B, int64_t K, int64_t T, rrl_view turn_adv,
                                  rrl_view turn_ids, rrl_view mask, void* out, int32_t out_dtype,
                                  int32_t* status, void* stream) {
  clear_error();
  RRL_REQUIRE(B >= 0 && K >= 0 && T >= 0, RRL_EINVAL, "negative size");
  RRL_REQUIRE(is_float_dtype(out_dtype) && is_known_dtype(turn_ids.dtype) &&
                  is_known_dtype(mask.dtype) && is_known_dtype(turn_adv.dtype),
              RRL_EDTYPE, "unsupported dtype");
  if (B * T == 0) return RRL_OK;
  RRL_REQUIRE(turn_ids.ptr && mask.ptr && out && (K == 0 || turn_adv.ptr), RRL_EINVAL,
              "null pointer argument");
  hipStream_t st = as_stream(stream);
  const unsigned grid = flat_grid(B * T, 256);
  if (out_dtype == RRL_F64)
    hipLaunchKernelGGL((broadcast_turn_kernel<double>), dim3(grid), dim3(256), 0, st, B, K, T,
                       to_view(turn_adv), to_view(turn_ids), to_view(mask), out, (int)out_dtype,
                       status);
  else
    hipLaunchKernelGGL((broadcast_turn_kernel<float>), dim3(grid), dim3(256), 0, st, B, K, T,
                       to_view(turn_adv), to_view(turn_ids), to_view(mask), out, (int)out_dtype,
                       status);
  return check_launch("broadcast_turn_kernel");
}

extern "C" size_t rrl_reduce_workspace_bytes(int64_t n) {
  (void)n;
  return (size_t)(RED_MAXB * 4 + 4) * 8 + 256;
}

extern "C" int rrl_masked_mean_fwd(int64_t B, int64_t T, rrl_view values, rrl_view mask,
                                   int32_t acc_dtype, void* workspace, void* out, int32_t* status,
                                   void* stream) {
  clear_error();
  RRL_REQUIRE(B >= 0 && T >= 0, RRL_EINVAL, "negative size");
  RRL_REQUIRE(workspace && out, RRL_EINVAL, "workspace and out are required");
  RRL_REQUIRE(B * T == 0 || (values.ptr && mask.ptr), RRL_EINVAL, "null pointer argument");
  RRL_REQUIRE(is_float_dtype(values.dtype) && is_known_dtype(mask.dtype), RRL_EDTYPE,
              "unsupported dtype");
  RedArgs a{};
  a.B = B; a.T = T; a.x = to_view(values); a.mask = to_view(mask);
  a.part = workspace; a.out = out; a.status = status;
  const unsigned nb = red_grid(B * T);
  hipStream_t st = as_stream(stream);
  if (acc_dtype == RRL_F64) {
    hipLaunchKernelGGL((masked_partials_kernel<double>), dim3(nb), dim3(RED_NT), 0, st, a);
    if (int rc = check_launch("masked_partials_kernel")) return rc;
    hipLaunchKernelGGL((masked_mean_final_kernel<double>), dim3(1), dim3(RED_NT), 0, st, a, (int)nb);
  } else {
    hipLaunchKernelGGL((masked_partials_kernel<float>), dim3(nb), dim3(RED_NT), 0, st, a);
    if (int rc = check_launch("masked_partials_kernel")) return rc;
    hipLaunchKernelGGL((masked_mean_final_kernel<float>), dim3(1), dim3(RED_NT), 0, st, a, (int)nb);
  }
  return check_launch("masked_mean_final_kernel");
}

extern "C" int rrl_masked_mean_bwd(int64_t B, int64_t T, rrl_view mask, int32_t acc_dtype,
                                   const void* workspace, const void* grad, void* grad_values,
                                   void* stream) {
  clear_error();
  RRL_REQUIRE(workspace && grad && (B * T == 0 || grad_values), RRL_EINVAL, "null pointer argument");
  if (B * T == 0) return RRL_OK;
  RedArgs a{};
  a.B = B; a.T = T; a.mask = to_view(mask);
  a.part = const_cast<void*>(workspace); a.grad = grad; a.out = grad_values;
  hipStream_t st = as_stream(stream);
  const unsigned grid = flat_grid(B * T, RED_NT);
  if (acc_dtype == RRL_F64)
    hipLaunchKernelGGL((masked_mean_bwd_kernel<double>), dim3(grid), dim3(RED_NT), 0, st, a);
  else
    hipLaunchKernelGGL((masked_mean_bwd_kernel<float>), dim3(grid), dim3(RED_NT), 0, st, a);
  return check_launch("masked_mean_bwd_kernel");
}

extern "C" int rrl_masked_whiten(int64_t B, int64_t T, rrl_view x, rrl_view mask, double eps,
                                 int32_t shift_mean, int32_t acc_dtype, void* workspace, void* out,
                                 int32_t out_dtype, int32_t* status, void* stream) {
  clear_error();
  RRL_REQUIRE(B >= 0 && T >= 0, RRL_EINVAL, "negative size");
  RRL_REQUIRE(workspace && (B * T == 0 || (x.ptr && mask.ptr && out)), RRL_EINVAL,
              "null pointer argument");
  RRL_REQUIRE(is_float_dtype(x.dtype) && is_known_dtype(mask.dtype) && is_float_dtype(out_dtype),
              RRL_EDTYPE, "unsupported dtype");
  RedArgs a{};
  a.B = B; a.T = T; a.x = to_view(x); a.mask = to_view(mask);
  a.part = workspace; a.eps = eps; a.shift = shift_mean; a.out = out; a.odt = out_dtype;
  a.status = status;
  const unsigned nb = red_grid(B * T);
  hipStream_t st = as_stream(stream);
  return acc_dtype == RRL_F64 ? launch_whiten<double>(a, nb, st) : launch_whiten<float>(a, nb, st);
}

extern "C" int rrl_sequence_log_ratio_fwd(int64_t B, int64_t T, rrl_view cur, rrl_view old,
                                          rrl_view mask, int32_t length_normalize,
                                          int32_t acc_dtype, void* out, void* counts_out,
                                          int32_t* status, void* stream) {
  clear_error();
  RRL_REQUIRE(B >= 0 && T >= 0, RRL_EINVAL, "negative size");
  RRL_REQUIRE(B == 0 || (cur.ptr && old.ptr && mask.ptr && out && counts_out), RRL_EINVAL,
              "null pointer argument");
  RRL_REQUIRE(is_float_dtype(cur.dtype) && is_float_dtype(old.dtype) && is_known_dtype(mask.dtype),
              RRL_EDTYPE, "unsupported dtype");
  if (B == 0) return RRL_OK;
  hipStream_t st = as_stream(stream);
  const unsigned grid = (unsigned)(B < 65536 ? B : 65536);
  if (acc_dtype == RRL_F64)
    hipLaunchKernelGGL((seq_log_ratio_kernel<double>), dim3(grid), dim3(RED_NT), 0, st, B, T,
                       to_view(cur), to_view(old), to_view(mask), (int)length_normalize,
                       static_cast<double*>(out), static_cast<double*>(counts_out), status);
  else
    hipLaunchKernelGGL((seq_log_ratio_kernel<float>), dim3(grid), dim3(RED_NT), 0, st, B, T,
                       to_view(cur), to_view(old), to_view(mask), (int)length_normalize,
                       static_cast<float*>(out), static_cast<float*>(counts_out), status);
  return check_launch("seq_log_ratio_kernel");
}

extern "C" int rrl_sequence_log_ratio_bwd(int64_t B, int64_t T, rrl_view mask,
                                          int32_t length_normalize, int32_t acc_dtype,
                                          const void* counts, const void* grad, void* grad_cur,
                                          void* stream) {
  clear_error();
  RRL_REQUIRE(B * T == 0 || (mask.ptr && counts && grad && grad_cur), RRL_EINVAL,
              "null pointer argument");
  if (B * T == 0) return RRL_OK;
  hipStream_t st = as_stream(stream);
  const unsigned grid = flat_grid(B * T, 256);
  if (acc_dtype == RRL_F64)
    hipLaunchKernelGGL((seq_log_ratio_bwd_kernel<double>), dim3(grid), dim3(256), 0, st, B, T,
                       to_view(mask), (int)length_normalize, static_cast<const double*>(counts),
                       static_cast<const double*>(grad), static_cast<double*>(grad_cur));
  else
    hipLaunchKernelGGL((seq_log_ratio_bwd_kernel<float>), dim3(grid), dim3(256), 0, st, B, T,
                       to_view(mask), (int)length_normalize, static_cast<const float*>(counts),
                       static_cast<const float*>(grad), static_cast<float*>(grad_cur));
  return check_launch("seq_log_ratio_bwd_kernel");
}

extern "C" int rrl_double_sided_mask(int64_t n, const void* ratios, int32_t dtype, double lo,
                                     double hi, uint8_t* out, void* stream) {
  clear_error();
  RRL_REQUIRE(n >= 0, RRL_EINVAL, "negative size");
  RRL_REQUIRE(is_float_dtype(dtype), RRL_EDTYPE, "ratios must be floating point");
  if (n == 0) return RRL_OK;
  RRL_REQUIRE(ratios && out, RRL_EINVAL, "null pointer argument");
  hipStream_t st = as_stream(stream);
  const unsigned grid = flat_grid(n, 256);
  // Thresholds arrive already rounded to the ratio dtype by the caller.
  if (dtype == RRL_F64)
    hipLaunchKernelGGL((double_sided_kernel<double>), dim3(grid), dim3(256), 0, st, n, ratios,
                       (int)dtype, lo, hi, out);
  else
    hipLaunchKernelGGL((double_sided_kernel<float>), dim3(grid), dim3(256), 0, st, n, ratios,
                       (int)dtype, (float)lo, (float)hi, out);
  return check_launch("double_sided_kernel");
}
