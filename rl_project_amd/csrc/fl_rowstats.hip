// Full-distribution statistics of logits rows in one streaming pass:
//   token log-probability   -cross_entropy(x.float(), label)
//                           (src/forgeline/models/policy.py:47-50)
//   entropy                 -(softmax * log_softmax).sum(-1)
//                           (src/forgeline/training/common/logprobs.py:65-68)
//   KL(new || ref)          (p_new * (log p_new - log p_ref)).sum(-1)
//                           (src/forgeline/training/common/logprobs.py:58-62)
// all in float32 as the reference's .float() computes them.
//
// One work-group per row; the row streams through 16-byte chunks interleaved
// over the threads (coalesced), 2 chunks per thread in flight.  The loads need
// no more than an element's alignment, so rows of an odd vocabulary take them
// too (4096 bf16 rows of V = 50257: element by element 309 us, so 132 us).  Each thread keeps, relative to a reference m
// near its maximum of the row x,
//   s = sum exp(x - m),  u = sum exp(x - m) (x - m),
// and with a reference row y (its m') also
//   s' = sum exp(y - m'),  w = sum exp(x - m) ((x - m) - (y - m')),
// in float64, rescaled when m moves.  The partials are added in a fixed tree
// once all are relative to the row's largest m, so results are deterministic.
// With M that reference and S the row's sum:
//   log p(label) = x_label - M - log S
//   entropy      = log S - u / S
//   KL           = w / S - log S + log S'
// A -inf logit contributes exp(-inf) * (-inf) = NaN to u and w, as 0 * -inf
// does in the reference's expression; a finite one, however low, does not.
#include <type_traits>

#include "fl_device.h"
#include "fl_kernels.h"

namespace fl {

namespace {

constexpr float LOG2E_F = 1.44269504088896340736f;
constexpr double INV_LOG2E_F = 1.0 / static_cast<double>(LOG2E_F);  // (of the float: a base-2 difference over it is exact)
// A thread moves its reference m only once a value passes it by more than
// this: a re-base is a double-precision exponential, and while every new
// maximum took one, some lane of a wave had one in nearly every iteration
// (4096 bf16 rows of V = 128256: 195 us, without it 188 us).  The terms that
// count have exponents up to SLACK log2(e): below 8 they round at 2^-22 like
// those a little under the maximum (a slack of 8 is 1 % faster, but 255 bf16
// rows of V = 50257 are then 6.2e-7 from the KL in 64 bits, with 5.5 3.3e-7).
constexpr float SLACK = 5.5f;

template <class D>
struct RowChunk;
template <>
struct RowChunk<F32> {
  static constexpr int N = 4;
  __device__ static float elem(__amdgpu_buffer_rsrc_t r, int i) {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, 4 * i, 0, 0));
  }
  __device__ static void unpack(const uint4 u, float (&x)[N]) {
    x[0] = __uint_as_float(u.x);
    x[1] = __uint_as_float(u.y);
    x[2] = __uint_as_float(u.z);
    x[3] = __uint_as_float(u.w);
  }
};
template <class H>
struct RowChunk16 {
  static constexpr int N = 8;
  __device__ static float elem(__amdgpu_buffer_rsrc_t r, int i) {
    return H::to_f32(__builtin_amdgcn_raw_buffer_load_b16(r, 2 * i, 0, 0));
  }
  __device__ static void unpack(const uint4 u, float (&x)[N]) {
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      x[2 * k] = H::to_f32(w[k] & 0xFFFFu);
      x[2 * k + 1] = H::to_f32(w[k] >> 16);
    }
  }
};
template <>
struct RowChunk<BF16> : RowChunk16<BF16> {};
template <>
struct RowChunk<F16> : RowChunk16<F16> {};

// Running state of one row for one thread (or a merged set of threads).
struct Acc {
  float m;    // reference of x, its maximum less at most SLACK (-inf: nothing yet)
  double s;   // sum exp(x - m)
  double u;   // sum exp(x - m) (x - m)
  float my;   // reference of y
  double sy;  // sum exp(y - my)
  double w;   // sum exp(x - m) ((x - m) - (y - my))
};

// The reference a partial's terms were taken against.  Exponents are
// fma(x, log2(e), -mb) with mb = RN(m log2(e)), so that is mb / log2(e) and
// not m: half an ulp of mb is up to 3e-7 of every term of the thread.  (255
// f32 rows of V = 50257 with KL, from 64 bits: 3.5e-7 with m, 3.2e-7 with
// mb / log2(e); entropies of scores around 12: 6.4e-8 and 2.6e-8.)  Where mb overflows (a mask of the type's lowest value) the
// exponents are (x - m) log2(e).
__device__ __forceinline__ bool base2_ok(float m) { return __builtin_fabsf(m * LOG2E_F) != __builtin_inff(); }
__device__ __forceinline__ double ref_of(float m) {
  return base2_ok(m) ? static_cast<double>(m * LOG2E_F) * INV_LOG2E_F : static_cast<double>(m);
}

// Re-base a partial on a larger maximum M (m <= M).  A partial with no
// element yet (m == -inf) has zero sums and stays zero.
__device__ __forceinline__ void rebase_x(Acc& a, float M) {
  if (a.m == M || a.m == -__builtin_inff()) {
    a.m = M;
    return;
  }
  const double d = ref_of(a.m) - ref_of(M);
  const double f = exp(d);
  a.u = (a.u + a.s * d) * f;
  a.w = (a.w + a.s * d) * f;
  a.s *= f;
  a.m = M;
}
__device__ __forceinline__ void rebase_y(Acc& a, float M) {
  if (a.my == M || a.my == -__builtin_inff()) {
    a.my = M;
    return;
  }
  const double d = ref_of(a.my) - ref_of(M);
  // (x - m) - (y - M) = (x - m) - (y - my) - d
  a.w -= a.s * d;
  a.sy *= exp(d);
  a.my = M;
}

}  // namespace

template <class D, bool KL, int NT_RS>
__global__ __launch_bounds__(NT_RS) void k_row_stats(const fl_row_stats_args a) {
  using C = RowChunk<D>;
  constexpr int N = C::N;
  constexpr int NW_RS = NT_RS / WAVE;
  // chunks per thread in flight: with 4 the 16-bit instantiations hold too
  // many registers for the waves that keep HBM busy (4096 bf16 rows of V =
  // 128256: 188 us at 4, 174 us at 2, 6.0 TB/s; with KL, 2048 rows: 218 / 214 us)
  constexpr int U_RS = 2;
  __shared__ Acc part[NW_RS];
  __shared__ float ref_m[NW_RS], ref_my[NW_RS];
  const int tid = threadIdx.x;
  const int64_t r = blockIdx.x;
  const int V = static_cast<int>(a.vocab);
  const size_t esz = D::id == FL_DTYPE_F32 ? 4 : 2;
  const char* xp = static_cast<const char*>(a.logits) + r * a.ld * esz;
  const char* yp = KL ? static_cast<const char*>(a.ref_logits) + r * a.ref_ld * esz : xp;
  const __amdgpu_buffer_rsrc_t rx = row_rsrc(xp, static_cast<uint32_t>(V * esz));
  const __amdgpu_buffer_rsrc_t ry = row_rsrc(yp, static_cast<uint32_t>(V * esz));
  const int nch = (V + N - 1) / N;
  const int nfull = V / N;

  Acc acc = {-__builtin_inff(), 0.0, 0.0, -__builtin_inff(), 0.0, 0.0};
  auto load = [&](__amdgpu_buffer_rsrc_t rs, int c, float (&x)[N]) __attribute__((always_inline)) {
    if (c < nfull) {
      C::unpack(buf_load16_once(rs, 16u * c, 0u), x);  // (read once: 207 -> 201 us at 4096 x 128256 bf16)
    } else {
#pragma unroll
      for (int e = 0; e < N; ++e) x[e] = N * c + e < V ? C::elem(rs, N * c + e) : -__builtin_inff();
    }
  };
  for (int c0 = 0; c0 < nch; c0 += U_RS * NT_RS) {
    float xs[U_RS][N], ys[U_RS][N];
#pragma unroll
    for (int k = 0; k < U_RS; ++k) {
      const int c = c0 + k * NT_RS + tid;
      if (c < nch) {
        load(rx, c, xs[k]);
        if (KL) load(ry, c, ys[k]);
      } else {
#pragma unroll
        for (int e = 0; e < N; ++e) xs[k][e] = ys[k][e] = -__builtin_inff();
      }
    }
    // maxima of the iteration's chunks first (padding is -inf)
    float cm = xs[0][0], cmy = ys[0][0];
#pragma unroll
    for (int k = 0; k < U_RS; ++k)
#pragma unroll
      for (int e = 0; e < N; ++e) {
        cm = fmaxf(cm, xs[k][e]);
        if (KL) cmy = fmaxf(cmy, ys[k][e]);
      }
    if (cm > acc.m + SLACK) rebase_x(acc, cm);
    if (KL && cmy > acc.my + SLACK) rebase_y(acc, cmy);
    // exponents in base 2: d2 = (x - m) log2(e) in one rounding; the base-2
    // sums of the iteration (at most U_RS * N terms, each below e^SLACK) are
    // scaled to natural units and added to the float64 partials once
    const float mb = acc.m * LOG2E_F, myb = acc.my * LOG2E_F;
    float fs = 0.0f, fu = 0.0f, fsy = 0.0f, fw = 0.0f;
    double wd = 0.0;
    const bool bx = base2_ok(acc.m), by = !KL || base2_ok(acc.my);
    bool general = !(c0 + (U_RS - 1) * NT_RS + tid < nfull && bx && by);
    if (!general) {
      // whole chunks under a finite maximum: -inf gives d2 = -inf, e = 0 and
      // e * d2 = NaN, the reference's 0 * -inf
#pragma unroll
      for (int k = 0; k < U_RS; ++k)
#pragma unroll
        for (int e = 0; e < N; ++e) {
          const float d2 = fmaf(xs[k][e], LOG2E_F, -mb);
          const float ex = __builtin_amdgcn_exp2f(d2);
          fs += ex;
          fu = fmaf(ex, d2, fu);
          if (KL) {
            const float dy2 = fmaf(ys[k][e], LOG2E_F, -myb);
            fsy += __builtin_amdgcn_exp2f(dy2);
            fw = fmaf(ex, d2 - dy2, fw);
          }
        }
    }
    // A finite value near the type's lowest (a mask) has d2 = -inf too, where
    // the reference's 0 * x is 0 (and p * -y large, but finite): such an
    // iteration is taken again below.  Not once a -inf logit has made the
    // wave's sum NaN, and the row's with it, so that a row with many of them
    // takes one such iteration a wave.
    const bool nan_u = !(__builtin_fabsf(fu) < __builtin_inff());
    const bool nan_w = KL && !(__builtin_fabsf(fw) < __builtin_inff());
    if (__any(nan_u || nan_w)) {
      const bool lost_u = __any(acc.u != acc.u), lost_w = KL && __any(acc.w != acc.w);
      general = general || (nan_u && !lost_u) || (nan_w && !lost_w);
    }
    if (general) {
      // the row's last chunks (partial or past the row), values before any
      // finite one (-inf below a maximum that is still -inf), references whose
      // base-2 form overflows, and values whose exponent does
      auto below = [](float x, float m, float b, bool ok) {
        return x == -__builtin_inff() ? x : ok ? fmaf(x, LOG2E_F, -b) : (x - m) * LOG2E_F;
      };
      // (the difference itself, also where it is past the float range)
      auto wide = [](float d2, float x, float m) -> double {
        return d2 == -__builtin_inff() && x != d2 ? (static_cast<double>(x) - ref_of(m)) * LOG2E_F : d2;
      };
      fs = fu = fsy = 0.0f;
      fw = 0.0f;
#pragma unroll
      for (int k = 0; k < U_RS; ++k) {
        const int c = c0 + k * NT_RS + tid;
#pragma unroll
        for (int e = 0; e < N; ++e) {
          if (N * c + e >= V) continue;
          const float x = xs[k][e], d2 = below(x, acc.m, mb, bx);
          const float ex = __builtin_amdgcn_exp2f(d2);
          fs += ex;
          fu += d2 == -__builtin_inff() && x != d2 ? 0.0f : ex * d2;
          if (KL) {
            const float y = ys[k][e], dy2 = below(y, acc.my, myb, by);
            fsy += __builtin_amdgcn_exp2f(dy2);
            wd += static_cast<double>(ex) * (wide(d2, x, acc.m) - wide(dy2, y, acc.my));
          }
        }
      }
    }
    acc.s += fs;
    acc.u += static_cast<double>(fu) * INV_LOG2E_F;
    if (KL) {
      acc.sy += fsy;
      acc.w += (static_cast<double>(fw) + wd) * INV_LOG2E_F;
    }
  }
  // merge: the row's largest references first, so that each thread re-bases
  // its partial once (two double-precision exponentials), then plain sums in a
  // fixed tree.  (Merging partial by partial re-based twice per step of the
  // tree: 4096 bf16 rows of V = 4099 took 38.0 us, now 28.6.)
  const int wave = tid / WAVE;
  const float wm = wave_reduce(acc.m, OpMax()), wmy = KL ? wave_reduce(acc.my, OpMax()) : 0.0f;
  if ((tid & (WAVE - 1)) == 0) {
    ref_m[wave] = wm;
    ref_my[wave] = wmy;
  }
  __syncthreads();
  float M = ref_m[0], My = ref_my[0];
#pragma unroll
  for (int i = 1; i < NW_RS; ++i) {
    M = fmaxf(M, ref_m[i]);
    My = fmaxf(My, ref_my[i]);
  }
  rebase_x(acc, M);
  if (KL) rebase_y(acc, My);  // (from the thread's own s: before the sums)
  acc.s = wave_reduce(acc.s, OpAdd());
  acc.u = wave_reduce(acc.u, OpAdd());
  if (KL) {
    acc.sy = wave_reduce(acc.sy, OpAdd());
    acc.w = wave_reduce(acc.w, OpAdd());
  }
  // (field by field: a copy of the struct keeps it in memory, which the compiler
  // puts into LDS, indexed through the launch packet in host memory: 255 bf16
  // rows of V = 512 18.2 us, now 4.7)
  if ((tid & (WAVE - 1)) == 0) {
    Acc& p = part[wave];
    p.m = acc.m;
    p.s = acc.s;
    p.u = acc.u;
    if (KL) {
      p.my = acc.my;
      p.sy = acc.sy;
      p.w = acc.w;
    }
  }
  __syncthreads();
  if (tid != 0) return;
  Acc t = {M, 0.0, 0.0, My, 0.0, 0.0};
#pragma unroll
  for (int i = 0; i < NW_RS; ++i) {
    t.s += part[i].s;
    t.u += part[i].u;
    if (KL) {
      t.sy += part[i].sy;
      t.w += part[i].w;
    }
  }
  const double logS = log(t.s);
  if (a.out_entropy) a.out_entropy[r] = static_cast<float>(logS - t.u / t.s);
  if (a.out_lse) a.out_lse[r] = static_cast<float>(ref_of(t.m) + logS);
  if (KL && a.out_kl) a.out_kl[r] = static_cast<float>(t.w / t.s - logS + log(t.sy));
  if (a.labels && a.out_logprob) {
    const int64_t lab = a.labels[r];
    float lp;
    if (lab == a.ignore_index) lp = -0.0f;  // -(cross_entropy = 0) for an ignored target
    else if (lab < 0 || lab >= V) lp = __builtin_nanf("");
    else lp = static_cast<float>(static_cast<double>(C::elem(rx, static_cast<int>(lab))) - ref_of(t.m) - logS);
    a.out_logprob[r] = lp;
  }
}

// Threads per row: 256 where rows are many (their merges overlap other rows'
// reads); 1024 where a CU gets one row at most, so that the row has 16 waves'
// loads in flight instead of 4.  f32 with KL, V = 50257: 255 rows 34.2 us with
// 256 threads, 22.2 us with 1024; 520 rows 41.4 against 47.9 us.
constexpr int64_t RS_FEW_ROWS = 256;

hipError_t launch_row_stats(const fl_row_stats_args& a, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(a.rows));
  const bool few = a.rows <= RS_FEW_ROWS;
  auto run = [&](auto d) {
    using D = decltype(d);
    auto go = [&](auto kl_c) {
      constexpr bool KL = decltype(kl_c)::value;
      if (few) hipLaunchKernelGGL((k_row_stats<D, KL, 1024>), grid, dim3(1024), 0, s, a);
      else hipLaunchKernelGGL((k_row_stats<D, KL, 256>), grid, dim3(256), 0, s, a);
    };
    if (a.ref_logits != nullptr) go(std::true_type{});
    else go(std::false_type{});
  };
  if (a.dtype == FL_DTYPE_F32) run(F32{});
  else if (a.dtype == FL_DTYPE_BF16) run(BF16{});
  else run(F16{});
  return hipGetLastError();
}

}  // namespace fl
