// Inverse-Compton spectrum of a tabulated particle distribution scattering a
// tabulated soft-photon field (ICSpectrum, src/physics/ic.cpp:15-46, with the
// per-triple kernel of src/physics/ic.hpp:28-86).
//
// For every output energy e_ic and every (gamma, e_soft) pair the reference adds
//     f_g (f_s / e_s) e_ic^2 KN(Gamma, q) / g      (/ g^2 for linear gamma bins)
// with Gamma = 4 g e_s, q = (e_ic / g) / (Gamma (1 - e_ic / g)), skipped above
// the kinematic limit e_ic > g Gamma / (1 + Gamma).  The terms of a bin are summed
// in FP64 in a fixed order, so results are reproducible bit for bit.
//
// Layout: one workgroup per (output bin, chunk of gamma bins), enough of them
// to fill the device; its threads take the chunk's (gamma, e_soft) pairs in
// turn, both staged in LDS; a fixed-order tree per block and, with more than one
// chunk, a second pass adding the chunks in order.  No table or plan.
//
// The kernel is bound by its VALU work and its LDS reads, so what depends on one operand only is
// formed once per block.  With x = e_ic / g (from x = 1/2 on the reference's float)
//     q = [x / (4 g (1 - x))] (1 / e_s),   Gamma q = x / (1 - x),
// so a pair's q is one product, KN's quotient (Gamma q)^2 / (1 + Gamma q) is the
// gamma bin's, and the kinematic limit is q = 1: no divide is left in the loop.
// Pairs where rounding could decide differently (q within 2e-6 / (1 - x) of 1:
// the reference's limit is good to 2.4e-7 / (1 - x)) and operands outside the
// ranges below take the reference's own operations (KN's second part is double
// there: its 0.5 literal promotes it).
// q, KN and the quotient by g are FP64, which issues at the rate of FP32 here and
// takes fewer instructions than float factors with their conversions; the
// logarithm is the hardware's float log2.  Error of a term against 64 bits (rms):
// 5.7e-8 at q < 1e-2, 1.2e-7 at 0.5 .. 0.9, 5.2e-7 at 0.9 .. 0.99; of the reference's
// operations 6.7e-8, 2.2e-7 and 1.5e-6.
// Per call, before and after: 200^3 27.6 and 15.5 us (of it the kernel 23.4 and
// 11: the loop's 125000 wave steps take 4.4, loading, staging and the reduction
// the rest), 500^3 235 and 72, 1000^3 1595 and 457 us (72 clocks a step of 64 pairs).
#include <algorithm>
#include <cmath>

#include "rgn_core.hpp"

namespace rgn {
namespace {

constexpr int kIcThreads = 256;
constexpr int kIcGamma = 128;  // gamma bins and
static_assert(kIcGamma <= kIcThreads, "one gamma bin a thread");
constexpr int kIcSoft = 512;   // soft-photon bins staged in LDS at a time

// ic.hpp:20-25.  2 * q * log(q) is float; the 0.5 literal makes the rest double.
__device__ __forceinline__ float kn_func(float Gamma, float q) {
  const float Gq = Gamma * q;
  const float first = 2.0f * q * logf(q);
  const double rest = static_cast<double>(1.0f - q) *
                      (static_cast<double>(1.0f + 2.0f * q) +
                       0.5 * static_cast<double>(Gq) * static_cast<double>(Gq) / static_cast<double>(1.0f + Gq));
  return static_cast<float>(static_cast<double>(first) + rest);
}

// ic.hpp:62-85, float arithmetic in the reference's order.
__device__ __noinline__ float ic_term(float g_prtls, float f_prtls, float e_soft, float fs_es, float e_ic, int g_log) {
  const float Gamma = 4.0f * g_prtls * e_soft;
  if (e_ic > g_prtls * Gamma / (1.0f + Gamma)) return 0.0f;
  const float x = e_ic / g_prtls;
  const float q = x / (Gamma * (1.0f - x));
  const float kn = kn_func(Gamma, q);
  return g_log ? f_prtls * fs_es * e_ic * e_ic * kn / g_prtls
               : f_prtls * fs_es * e_ic * e_ic * kn / (g_prtls * g_prtls);
}

// 1 / x to about one ulp (hardware estimate, two Newton steps).
__device__ __forceinline__ double ic_rcp(double x) {
  double y = __builtin_amdgcn_rcp(x);
  y = fma(fma(-x, y, 1.0), y, y);
  return fma(fma(-x, y, 1.0), y, y);
}

struct __align__(16) IcGamma {
  double c;      // x / (4 g (1 - x)); NaN: outside the ranges, every pair by ic_term
  double h1;     // 1 + (Gamma q)^2 / (1 + Gamma q) / 2
  double ig;     // 1 / g, or 1 / g^2 for linear gamma bins
  float lo, hi;  // below lo (from kIcMinQ): a term; above hi: none; between: ic_term
  float f;
};
constexpr float kIcMinQ = 1e-30f;

__device__ __forceinline__ IcGamma ic_gamma(float g, float f, float e_ic, int g_log) {
  IcGamma o;
  const float x = e_ic / g, one_x = 1.0f - x;
  const bool ok = g >= 1e-6f && g <= 1e12f && x >= 1e-20f && fabsf(one_x) >= 4e-6f && x < INFINITY;
  // x unrounded, but for x near 1, where its rounding decides 1 - x: the reference's
  const double rg = ic_rcp(g);
  const double xd = x < 0.5f ? static_cast<double>(e_ic) * rg : static_cast<double>(x);
  const double gq = xd * ic_rcp(1.0 - xd);
  // past the limit for every e_soft where x > 1
  o.c = !ok ? NAN : one_x > 0.0f ? 0.25 * gq * rg : INFINITY;
  const float margin = 2e-6f * __builtin_amdgcn_rcpf(fabsf(one_x));
  o.lo = 1.0f - margin;
  o.hi = 1.0f + margin;
  o.f = f;
  o.h1 = fma(0.5 * gq * gq, ic_rcp(1.0 + gq), 1.0);
  o.ig = g_log ? rg : rg * rg;
  return o;
}

// One workgroup per (output bin, chunk of gamma bins); its FP64 sum goes to
// partial[chunk][bin], or to the result where there is one chunk.  The pairs of a
// stage go to the threads
//   ROWS   64 soft-photon bins to a wave at a time, every fourth gamma bin: a soft-
//          photon bin's factors stay in registers;
//   else   in turn, soft-photon bins fastest, so that every lane has a pair
//          whatever the counts.
// Summation order: per thread, stage by stage, its pairs in order; then a fixed
// tree over the threads.
template <bool ROWS>
__global__ void __launch_bounds__(kIcThreads) ic_kernel(const float* __restrict__ g, const float* __restrict__ fg,
                                                        int ng, int g_log, const float* __restrict__ es,
                                                        const float* __restrict__ fes, int nes,
                                                        const float* __restrict__ eic, int gper,
                                                        double* __restrict__ partial, float* __restrict__ out) {
  __shared__ double red[kIcThreads];
  __shared__ IcGamma s_g[kIcGamma];
  __shared__ double s_r[kIcSoft];  // 1 / e_soft (NaN: outside the range)
  __shared__ float s_f[kIcSoft];   // f_s / e_soft
  const int e = blockIdx.x, neic = gridDim.x, tid = threadIdx.x;
  const float e_ic = eic[e];
  const int g0 = blockIdx.y * gper, g1 = min(ng, g0 + gper);
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  double acc = 0.0;
  // KN = 2 q ln q + (1 - q) (1 + 2 q + h), of q rounded once to float: of one q in both
  // parts, which cancel near q = 1.  The hardware's log2 rounds down, below q = 1/4 half
  // an ulp on average, 4e-8 of it (0 .. 2e-8 beyond): the constant takes that off (error
  // of 200^3 against 64 bits 5.5e-8 without, 4.0e-8 with it).
  constexpr double kTwoLn2 = 2.0 * 0.69314718055994530942 * (1.0 - 4e-8);
  auto pair = [&](const IcGamma& G, int gi, double r, float fs_es, int si) {
    const float qf = static_cast<float>(G.c * r);
    if (qf > G.hi) return;
    if (qf <= G.lo && qf >= kIcMinQ) {
      const double lg = static_cast<double>(__builtin_amdgcn_logf(qf));
      const double q = static_cast<double>(qf);
      const double rest = (1.0 - q) * fma(q, 2.0, G.h1);
      const double kn = fma(q * kTwoLn2, lg, rest);
      acc = fma(static_cast<double>(G.f * fs_es * e_ic * e_ic), kn * G.ig, acc);
    } else {
      acc += static_cast<double>(ic_term(g[gi], G.f, es[si], fs_es, e_ic, g_log));
    }
  };
  for (int ss = 0; ss < nes; ss += kIcSoft) {
    const int ms = min(kIcSoft, nes - ss);
    const int di = kIcThreads / ms, ds = kIcThreads % ms;  // a step of kIcThreads pairs
    for (int gs = g0; gs < g1; gs += kIcGamma) {
      const int mg = min(kIcGamma, g1 - gs);
      // all loads of a stage at once: in a small call they are most of a block's time
      float soft[kIcSoft / kIcThreads], fsoft[kIcSoft / kIcThreads];
      if (gs == g0) {
#pragma unroll
        for (int j = 0; j < kIcSoft / kIcThreads; ++j) {
          const int i = min(tid + j * kIcThreads, ms - 1);
          soft[j] = es[ss + i];
          fsoft[j] = fes[ss + i];
        }
      }
      const int ig = gs + min(tid, mg - 1);
      const float gv = g[ig], fv = fg[ig];
      __syncthreads();  // the previous stage has been read
      if (tid < mg) s_g[tid] = ic_gamma(gv, fv, e_ic, g_log);
      if (gs == g0) {
#pragma unroll
        for (int j = 0; j < kIcSoft / kIcThreads; ++j) {
          if (tid + j * kIcThreads < ms) {
            s_r[tid + j * kIcThreads] = soft[j] >= 1e-15f && soft[j] <= 1e15f ? ic_rcp(soft[j]) : NAN;
            s_f[tid + j * kIcThreads] = fsoft[j] / soft[j];
          }
        }
      }
      __syncthreads();
      if constexpr (ROWS) {
        for (int si = lane; si < ms; si += 64) {
          const double r = s_r[si];
          const float fs_es = s_f[si];
          for (int i = wave; i < mg; i += kIcThreads / 64) pair(s_g[i], gs + i, r, fs_es, ss + si);
        }
      } else {
        int i = tid / ms, si = tid % ms;
        while (i < mg) {
          pair(s_g[i], gs + i, s_r[si], s_f[si], ss + si);
          i += di;
          si += ds;
          if (si >= ms) {
            si -= ms;
            ++i;
          }
        }
      }
    }
  }
  red[tid] = acc;
  __syncthreads();
  for (int w = kIcThreads / 2; w > 0; w >>= 1) {
    if (tid < w) red[tid] += red[tid + w];
    __syncthreads();
  }
  if (tid == 0) {
    if (gridDim.y == 1) {
      out[e] = static_cast<float>(red[0]);
    } else {
      partial[static_cast<size_t>(blockIdx.y) * neic + e] = red[0];
    }
  }
}

// out[e] = the chunk partials of bin e, summed in chunk order, eight in flight.
constexpr int kIcCombine = 64;

__global__ void __launch_bounds__(kIcCombine) ic_combine(const double* __restrict__ partial, int nchunk, int neic,
                                                         float* __restrict__ out) {
  const int e = blockIdx.x * kIcCombine + threadIdx.x;
  if (e >= neic) return;
  double s = 0.0;
  for (int c = 0; c < nchunk; c += 8) {
    double v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = partial[static_cast<size_t>(min(c + k, nchunk - 1)) * neic + e];
#pragma unroll
    for (int k = 0; k < 8; ++k) s += c + k < nchunk ? v[k] : 0.0;
  }
  out[e] = static_cast<float>(s);
}

}  // namespace
}  // namespace rgn

using namespace rgn;

extern "C" {

int rgn_ic_spectrum(const float* d_g, const float* d_fg, int ng, int g_log, const float* d_es,
                    const float* d_fes, int nes, const float* d_eic, int neic, float* d_out,
                    rgn_stream_t stream) {
  return guarded([&] {
    RGN_REQUIRE(ng >= 0 && nes >= 0 && neic >= 0, RGN_ERR_INVALID, "negative size");
    if (neic == 0) return;
    RGN_REQUIRE(d_eic && d_out, RGN_ERR_INVALID, "null argument");
    RGN_REQUIRE((ng == 0 || (d_g && d_fg)) && (nes == 0 || (d_es && d_fes)), RGN_ERR_INVALID,
                "null argument");
    hipStream_t st = as_stream(stream);
    ScratchUse order(st);
    // Gamma bins in chunks: up to 16 blocks per CU (500^3: 8 blocks 100 us, 16 93),
    // but at least kIcPairs pairs a block, below which its staging and reduction
    // outweigh them (200^3 of 2048, 4096, 8192 pairs: 18.1, 16.2, 18.1 us; 50^3 as
    // 20 chunks and a second pass 15.6, as one 12.6 us)
    constexpr double kIcPairs = 4096.0;
    const double most = std::max(1, (16 * num_cus() + neic - 1) / neic);
    const double pairs = static_cast<double>(ng) * nes;
    const int chunks = std::max(1, static_cast<int>(std::min({most, static_cast<double>(ng), pairs / kIcPairs})));
    const int gper = std::max(1, (ng + chunks - 1) / chunks);
    const int nchunk = std::max(1, (ng + gper - 1) / gper);  // at most 16 CUs + 1
    double* partial = static_cast<double*>(scratch(sizeof(double) * nchunk * static_cast<size_t>(neic), 17));
    // Rows where they fill three quarters of their lanes and a block has 8000
    // pairs: 500^3 92 -> 76 us, 300 x 300 x 400 32.5 -> 30.2; with fewer they are
    // slower (400 x 300 x 60, 4100 pairs a block: 15.6 against 16.5).
    const bool rows = 4 * nes >= 3 * ((nes + 63) / 64 * 64) && pairs >= 8000.0 * nchunk;
    auto kernel = rows ? ic_kernel<true> : ic_kernel<false>;
    kernel<<<dim3(neic, nchunk), kIcThreads, 0, st>>>(d_g, d_fg, ng, g_log ? 1 : 0, d_es, d_fes, nes, d_eic, gper,
                                                      partial, d_out);
    RGN_HIP(hipGetLastError());
    stage_mark(st, "ic_kernel");
    if (nchunk == 1) return;
    ic_combine<<<(neic + kIcCombine - 1) / kIcCombine, kIcCombine, 0, st>>>(partial, nchunk, neic, d_out);
    RGN_HIP(hipGetLastError());
    stage_mark(st, "ic_combine");
  });
}

}  // extern "C"
