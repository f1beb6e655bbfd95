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
// too (4096 bf16 rows of V = 50257: element by element 309 us, so 86 us).  HBM
// bounds it from some hundred rows on: 4096 bf16 rows of V = 128256 171 us, 6.1
// TB/s.  Each thread keeps, relative to a reference m
// near its maximum of the row x,
//   s = sum exp(x - m),  u = sum exp(x - m) (x - m),
// and with a reference row y (its m') also
//   s' = sum exp(y - m'),  w = sum exp(x - m) ((x - m) - (y - m')),
// in float64, rescaled when m moves.  The partials are added in a fixed tree
// once all are relative to the largest m, the same for every call: a row's
// results are a function of the row alone.
// With M that reference and S the row's sum:
//   log p(label) = x_label - M - log S
//   entropy      = log S - u / S
//   KL           = w / S - log S + log S'
// A -inf logit contributes exp(-inf) * (-inf) = NaN to u and w, as 0 * -inf
// does in the reference's expression; a finite one, however low, does not.
#include <algorithm>
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
// count have exponents up to SLACK log2(e), rounded at that size: of the KL's
// distance from 64 bits, summed over 72 sets of rows each of f32, bf16 and f16,
// 3.5 gives 2.29e-5, 3.14e-5 and 3.28e-5, 5.5 2.38e-5, 3.36e-5 and 3.46e-5 (and
// 162 us in place of 171 for the 4096 rows).  The same for both rows: their differences are
// what counts, and with 1 for the reference row alone the KL is 4.5e-5 off.
constexpr float SLACK = 3.5f;
// Stands for the values past the row's end in its last iteration: nothing to
// any sum, its exponent finite and far below that of any reference in base 2.
constexpr float PAD = -1.0e38f;

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
// mb / log2(e); entropies of scores around 12: 6.4e-8 and 2.6e-8.)  From 2^31 on
// (a mask value as a thread's reference) that half ulp, 2^6 and more, would
// leave the float range as an exponent: the exponents are (x - m) log2(e) there.
__device__ __forceinline__ bool base2_ok(float m) { return __builtin_fabsf(m * LOG2E_F) < 0x1p31f; }
__device__ __forceinline__ double ref_of(float m) {
#pragma clang fp contract(off)
  return base2_ok(m) ? static_cast<double>(m * LOG2E_F) * INV_LOG2E_F : static_cast<double>(m);
}

// (Products and sums are fused where written as fma only, here and in the
// kernel: the same bits from every instantiation.)
// One value below the reference m: its base-2 exponent, and whether that is
// -inf though the value is finite (the difference is past the float range).
struct Below {
  float d2;
  bool under;
  // the base-2 difference itself
  __device__ __forceinline__ double wide(float x, float m) const {
    return under ? (static_cast<double>(x) - ref_of(m)) * static_cast<double>(LOG2E_F) : static_cast<double>(d2);
  }
};
__device__ __forceinline__ Below below(float x, float m) {
  if (x == -__builtin_inff()) return {x, false};
  const float d2 = base2_ok(m) ? fmaf(x, LOG2E_F, -(m * LOG2E_F)) : (x - m) * LOG2E_F;
  return {d2, d2 == -__builtin_inff()};
}

// Re-base a partial on a larger maximum M (m <= M).  A partial with no
// element yet (m == -inf) has zero sums and stays zero.
__device__ __forceinline__ void rebase_x(Acc& a, float M) {
#pragma clang fp contract(off)
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
#pragma clang fp contract(off)
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

// A row's terms are grouped by its length and type alone, so that a row has the
// same bits in any call: 256 lanes take the row's iterations (RS_U chunks per
// lane) in up to RS_SEGS runs, a lane's terms of one run go into one partial,
// and the partials merge wave by wave, then run by run.  How many of the runs
// are taken side by side, by 256 threads each, is the launch's choice.
constexpr int RS_LANES = 256;
constexpr int RS_WAVES = RS_LANES / WAVE;
constexpr int RS_U = 2;     // chunks per lane in flight
constexpr int RS_SEGS = 4;  // most runs of a row

// Runs of a row of `iters` iterations, a power of two, each of four iterations
// or more: of two, the merges cost many rows more than the split gives few (4096
// bf16 rows of V = 32000 with KL: 90 us in two runs, 100 in four; 255 rows 12.4
// and 11.8).
__host__ __device__ __forceinline__ int rs_segs(int iters) { return iters >= 4 * RS_SEGS ? RS_SEGS : iters >= 8 ? 2 : 1; }
template <class D>
__host__ __device__ __forceinline__ int rs_iters(int V) {
  constexpr int E = RS_LANES * RS_U * RowChunk<D>::N;
  return (V + E - 1) / E;
}

// GROUPS: runs taken side by side (a divisor of the row's number of runs)
template <class D, bool KL, int GROUPS>
__global__ __launch_bounds__(RS_LANES * GROUPS) void k_row_stats(const fl_row_stats_args a) {
#pragma clang fp contract(off)
  using C = RowChunk<D>;
  constexpr int N = C::N;
  constexpr int NPART = RS_SEGS * RS_WAVES;
  static_assert(NPART <= WAVE, "one lane per partial");
  __shared__ Acc part[NPART];
  __shared__ float ref_m[RS_WAVES], ref_my[RS_WAVES];
  const int tid = threadIdx.x, lane = tid & (WAVE - 1);
  const int slot = tid % RS_LANES;  // the thread's lane of its run
  const int64_t r = blockIdx.x;
  const int V = static_cast<int>(a.vocab);
  const size_t esz = D::id == FL_DTYPE_F32 ? 4 : 2;
  const char* xp = static_cast<const char*>(a.logits) + r * a.ld * esz;
  const char* yp = KL ? static_cast<const char*>(a.ref_logits) + r * a.ref_ld * esz : xp;
  const __amdgpu_buffer_rsrc_t rx = row_rsrc(xp, static_cast<uint32_t>(V * esz));
  const __amdgpu_buffer_rsrc_t ry = row_rsrc(yp, static_cast<uint32_t>(V * esz));
  const int nfull = V / N;
  const int iters = rs_iters<D>(V), nseg = rs_segs(iters), per = (iters + nseg - 1) / nseg;

  // (the sum is not asked for, or the wave has seen a -inf logit and it is NaN)
  bool lost_u = a.out_entropy == nullptr, lost_w = a.out_kl == nullptr;
  for (int seg = __builtin_amdgcn_readfirstlane(tid / RS_LANES); seg < nseg; seg += GROUPS) {
    Acc acc = {-__builtin_inff(), 0.0, 0.0, -__builtin_inff(), 0.0, 0.0};
    for (int it = seg * per; it < min(iters, (seg + 1) * per); ++it) {
      const int base = it * RS_U * RS_LANES, c0 = base + slot;
      // (chunks past the row, and what lies past it of the last one, load zeros:
      // the range check goes by dwords)
      uint4 qx[RS_U], qy[RS_U];
#pragma unroll
      for (int k = 0; k < RS_U; ++k) {
        // (read once: 207 -> 201 us at 4096 x 128256 bf16)
        qx[k] = buf_load16_once(rx, 16u * static_cast<uint32_t>(c0 + k * RS_LANES), 0u);
        if (KL) qy[k] = buf_load16_once(ry, 16u * static_cast<uint32_t>(c0 + k * RS_LANES), 0u);
      }
      float xs[RS_U][N], ys[RS_U][N];
#pragma unroll
      for (int k = 0; k < RS_U; ++k) {
        C::unpack(qx[k], xs[k]);
        if (KL) C::unpack(qy[k], ys[k]);
      }
      const bool whole = base + RS_U * RS_LANES <= nfull;  // (for all lanes)
      if (!whole) {
        // past the row -inf (for the maximum); the last value of an odd 16-bit
        // row, whose dword reaches past it, by itself
        if (N * c0 >= V) continue;
#pragma unroll
        for (int k = 0; k < RS_U; ++k)
#pragma unroll
          for (int e = 0; e < N; ++e) {
            const int i = N * (c0 + k * RS_LANES) + e;
            if (i >= V) {
              xs[k][e] = -__builtin_inff();
              if (KL) ys[k][e] = -__builtin_inff();
            } else if (D::id != FL_DTYPE_F32 && e % 2 == 0 && i == V - 1) {
              xs[k][e] = C::elem(rx, i);
              if (KL) ys[k][e] = C::elem(ry, i);
            }
          }
      }
      // maxima of the iteration's chunks first (padding is -inf)
      float cm = xs[0][0], cmy = ys[0][0];
#pragma unroll
      for (int k = 0; k < RS_U; ++k)
#pragma unroll
        for (int e = 0; e < N; ++e) {
          cm = fmaxf(cm, xs[k][e]);
          if (KL) cmy = fmaxf(cmy, ys[k][e]);
        }
      if (cm > acc.m + SLACK) rebase_x(acc, cm);
      if (KL && cmy > acc.my + SLACK) rebase_y(acc, cmy);
      // exponents in base 2: d2 = (x - m) log2(e) in one rounding; the base-2
      // sums of the iteration (at most RS_U * N terms, each below e^SLACK) are
      // scaled to natural units and added to the float64 partials once
      // (without a reference, -inf values alone so far, relative to 0: their
      // terms are the same)
      const float mb = acc.m == -__builtin_inff() ? 0.0f : acc.m * LOG2E_F;
      const float myb = acc.my == -__builtin_inff() ? 0.0f : acc.my * LOG2E_F;
      float fs = 0.0f, fu = 0.0f, fsy = 0.0f, fw = 0.0f;
      if (!whole) {
        // (then a finite value whose terms are 0)
#pragma unroll
        for (int k = 0; k < RS_U; ++k)
#pragma unroll
          for (int e = 0; e < N; ++e)
            if (N * (c0 + k * RS_LANES) + e >= V) {
              xs[k][e] = PAD;
              if (KL) ys[k][e] = PAD;
            }
      }
      // -inf gives d2 = -inf, e = 0 and e * d2 = NaN, the reference's 0 * -inf
#pragma unroll
      for (int k = 0; k < RS_U; ++k)
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
      // A finite value near the type's lowest (a mask) has d2 = -inf too, where
      // the reference's 0 * x is 0 (and p * -y large, but finite); and a thread's
      // reference may be such a value.  Such an iteration is taken again, from
      // memory and in float64 where float ends.  Not once a -inf logit has
      // made the wave's sum NaN, and the row's with it, so that a row with many
      // of them takes one such iteration a wave.
      const bool off = !(__builtin_fabsf(mb) < 0x1p31f) || (KL && !(__builtin_fabsf(myb) < 0x1p31f));
      const bool nan_u = !(__builtin_fabsf(fu) < __builtin_inff());
      const bool nan_w = KL && !(__builtin_fabsf(fw) < __builtin_inff());
      double wd = 0.0;
      if (__any(off || nan_u || nan_w)) {
        lost_u = lost_u || __any(acc.u != acc.u);
        lost_w = lost_w || (KL && __any(acc.w != acc.w));
        if (off || (nan_u && !lost_u) || (nan_w && !lost_w)) {
          fs = fu = fsy = fw = 0.0f;
#pragma unroll 1
          for (int k = 0; k < RS_U; ++k) {
            const int c = c0 + k * RS_LANES;
            float x[N], y[N];
            C::unpack(buf_load16(rx, 16u * static_cast<uint32_t>(c), 0u), x);
            if (KL) C::unpack(buf_load16(ry, 16u * static_cast<uint32_t>(c), 0u), y);
#pragma unroll
            for (int e = 0; e < N; ++e) {
              const int i = N * c + e;
              if (i >= V) continue;
              if (D::id != FL_DTYPE_F32 && e % 2 == 0 && i == V - 1) {
                x[e] = C::elem(rx, i);
                if (KL) y[e] = C::elem(ry, i);
              }
              const Below bx = below(x[e], acc.m);
              const float ex = __builtin_amdgcn_exp2f(bx.d2);
              fs += ex;
              fu += bx.under ? 0.0f : ex * bx.d2;
              if (KL) {
                const Below by = below(y[e], acc.my);
                fsy += __builtin_amdgcn_exp2f(by.d2);
                wd += static_cast<double>(ex) * (bx.wide(x[e], acc.m) - by.wide(y[e], acc.my));
              }
            }
          }
        }
      }
      acc.s += fs;
      acc.u = fma(static_cast<double>(fu), INV_LOG2E_F, acc.u);
      if (KL) {
        acc.sy += fsy;
        acc.w = fma(static_cast<double>(fw) + wd, INV_LOG2E_F, acc.w);
      }
    }
    // the wave's partial: its largest references first (of a row of one run, the
    // row's), so that each lane re-bases its own once, then plain sums in a
    // fixed tree.  (Merging partial by partial re-based twice per step of the
    // tree: 4096 bf16 rows of V = 4099 took 38.0 us, now 15.6.)
    const int wave = slot / WAVE;
    float M = wave_reduce(acc.m, OpMax()), My = KL ? wave_reduce(acc.my, OpMax()) : 0.0f;
    if (nseg == 1) {  // (every wave of the group is here)
      if (lane == 0) {
        ref_m[wave] = M;
        ref_my[wave] = My;
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < RS_WAVES; ++i) {
        M = fmaxf(M, ref_m[i]);
        My = fmaxf(My, ref_my[i]);
      }
    }
    rebase_x(acc, M);
    if (KL) rebase_y(acc, My);  // (from the lane's own s: before the sums)
    acc.s = wave_reduce(acc.s, OpAdd());
    acc.u = wave_reduce(acc.u, OpAdd());
    if (KL) {
      acc.sy = wave_reduce(acc.sy, OpAdd());
      acc.w = wave_reduce(acc.w, OpAdd());
    }
    // (field by field: a copy of the struct keeps it in memory, which the
    // compiler puts into LDS, indexed through the launch packet in host memory:
    // 12 us of every launch: 255 bf16 rows of V = 512 18.2 us so, 4.1 without)
    if (lane == 0) {
      Acc& p = part[seg * RS_WAVES + wave];
      p.m = acc.m;
      p.s = acc.s;
      p.u = acc.u;
      if (KL) {
        p.my = acc.my;
        p.sy = acc.sy;
        p.w = acc.w;
      }
    }
  }
  __syncthreads();
  if (tid >= NPART) return;
  Acc t = {-__builtin_inff(), 0.0, 0.0, -__builtin_inff(), 0.0, 0.0};
  if (nseg == 1) {
    // the waves' partials, relative to the row's references, in order
    t.m = part[0].m;
    if (KL) t.my = part[0].my;
#pragma unroll
    for (int i = 0; i < RS_WAVES; ++i) {
      t.s += part[i].s;
      t.u += part[i].u;
      if (KL) {
        t.sy += part[i].sy;
        t.w += part[i].w;
      }
    }
  } else {
    // lane i takes partial i: as above, and again a fixed tree
    if (tid < nseg * RS_WAVES) {
      t.m = part[tid].m;
      t.s = part[tid].s;
      t.u = part[tid].u;
      if (KL) {
        t.my = part[tid].my;
        t.sy = part[tid].sy;
        t.w = part[tid].w;
      }
    }
    rebase_x(t, wave_reduce<float, OpMax, NPART>(t.m, OpMax()));
    if (KL) rebase_y(t, wave_reduce<float, OpMax, NPART>(t.my, OpMax()));
    t.s = wave_reduce<double, OpAdd, NPART>(t.s, OpAdd());
    t.u = wave_reduce<double, OpAdd, NPART>(t.u, OpAdd());
    if (KL) {
      t.sy = wave_reduce<double, OpAdd, NPART>(t.sy, OpAdd());
      t.w = wave_reduce<double, OpAdd, NPART>(t.w, OpAdd());
    }
  }
  if (tid != 0) return;
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

// Runs taken side by side (as far as the row has so many): four, unless the
// launch has rows enough for the CUs and the KL's registers would leave a CU one
// or two work-groups of that size.  Per launch with four / two / one: f32 V =
// 50257 255 rows 12.0 / 16.4 / 25.2 us, 512 20.9 / 20.7 / 28.2, 2048 65.5 / 69.0 /
// 72.2; bf16 4096x128256 175 / 178 / 178; f32 with KL V = 32000 255 rows 18.4 /
// 18.7 / 25.5, 257 23.5 / 22.0 / 27.1, 1024 53.2 / 48.7 / 48.4, 4096 178 / 164 /
// 166; bf16 with KL V = 32000 (two runs) 512 rows - / 19.3 / 21.4, 4096 - / 109 / 99.
constexpr int64_t RS_CU_ROWS = 256, RS_MANY_ROWS = 1024;
int rs_groups(bool kl, bool f32, int64_t rows) {
  if (!kl || rows <= RS_CU_ROWS) return 4;
  return f32 || rows <= RS_MANY_ROWS ? 2 : 1;
}

hipError_t launch_row_stats(const fl_row_stats_args& a, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(a.rows));
  auto run = [&](auto d) {
    using D = decltype(d);
    auto go = [&](auto kl_c, auto groups_c) {
      constexpr int G = decltype(groups_c)::value;
      hipLaunchKernelGGL((k_row_stats<D, decltype(kl_c)::value, G>), grid, dim3(RS_LANES * G), 0, s, a);
    };
    auto go_kl = [&](auto kl_c) {
      const int nseg = rs_segs(rs_iters<D>(static_cast<int>(a.vocab)));
      const int groups = std::min(nseg, rs_groups(a.ref_logits != nullptr, a.dtype == FL_DTYPE_F32, a.rows));
      if (groups == 4) go(kl_c, std::integral_constant<int, 4>{});
      else if (groups == 2) go(kl_c, std::integral_constant<int, 2>{});
      else go(kl_c, std::integral_constant<int, 1>{});
    };
    if (a.ref_logits != nullptr) go_kl(std::true_type{});
    else go_kl(std::false_type{});
  };
  if (a.dtype == FL_DTYPE_F32) run(F32{});
  else if (a.dtype == FL_DTYPE_BF16) run(BF16{});
  else run(F16{});
  return hipGetLastError();
}

}  // namespace fl
