// Particles<D>::energyDistribution (particles.cpp:189-260) on gfx950.
//
// Index function.  The reference bins an energy E (double) as
//   E < e_min -> 0,  E >= e_max -> n - 1,
//   else min(n - 1, (size_t)((float)(n - 1) * |log10(E / e_min)| / log10f(e_max / e_min)))
// (particles.cpp:233-245), with e_min / e_max the float MinMax of the bins.
// That function of E is monotone and piecewise constant, so the plan finds its
// n - 1 jump points E_k (the smallest double E with index >= k) on the host by
// bisection over the ordered bit patterns of positive doubles, evaluating the
// reference expression with the host libm.  The energy itself is a monotone
// function of the float |u|^2 (a correctly rounded square root, of |u|^2 or
// of 1 + |u|^2 in double), so each jump is also a float threshold of |u|^2:
// the kernel compares |u|^2 with floats and never forms the
// energy for the index.  It starts from a float log2 estimate of the index, which
// the plan checks to be within one bin everywhere, and corrects it by the
// thresholds on its two sides (plans that fail the check walk, and so do those
// with a threshold among the subnormals, whose log2 the hardware takes to be
// that of zero): the result
// equals the reference expression bit for bit, whatever the device log does.
//
// Accumulation.  Each wave owns private LDS histograms (uint32 counts and FP64
// sums of the per-particle float terms); blocks write per-block partials that a
// second kernel combines in a fixed order.  Counts are exact integers; sums are
// the FP64 sum of the reference's float terms, rounded to float once.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <limits>
#include <mutex>
#include <type_traits>
#include <vector>

#include "rgn_core.hpp"

struct rgn_hist_plan {
  int nb = 0;
  int log_bins = 0;
  float emin = 0.f, emax = 0.f;
  std::vector<double> edges;  // nb + 1 entries: edges[k] = E_k for 1 <= k < nb
  // per energy kind (0: sqrt(1 + u^2), 1: |u|): nb + 1 thresholds of |u|^2,
  // -inf and NaN at the ends; the estimate's coefficients and whether it is
  // within one bin everywhere
  rgn::DeviceBuffer d_thr;  // float[2][nb + 1]
  float est_a[2] = {}, est_b[2] = {};
  bool near[2] = {};
};

namespace rgn {
namespace {

constexpr int kThreads = 256;

// particles.cpp:239-243, evaluated exactly as the reference does on the host.
size_t reference_index(double energy, float emin, float emax, size_t n) {
  if (energy < emin) return 0;
  if (energy >= emax) return n - 1;
  const auto ei = static_cast<std::size_t>(static_cast<float>(n - 1) *
                                           std::fabs(std::log10(energy / emin)) /
                                           std::log10(emax / emin));
  return ei > n - 1 ? n - 1 : ei;
}

uint64_t bits_of(double d) {
  uint64_t b;
  std::memcpy(&b, &d, sizeof b);
  return b;
}

double from_bits(uint64_t b) {
  double d;
  std::memcpy(&d, &b, sizeof d);
  return d;
}

void build_edges(rgn_hist_plan& plan) {
  const size_t n = plan.nb;
  plan.edges.assign(n + 1, std::numeric_limits<double>::infinity());
  plan.edges[0] = -std::numeric_limits<double>::infinity();
  if (n < 2) return;
  // All positive doubles in [emin, emax) are ordered like their bit patterns.
  const uint64_t lo = bits_of(static_cast<double>(plan.emin));
  const uint64_t hi = bits_of(static_cast<double>(plan.emax));  // exclusive
  auto reaches = [&](uint64_t b, size_t k) { return reference_index(from_bits(b), plan.emin, plan.emax, n) >= k; };
  // inverse of the reference expression, good to a few double ulps: brackets
  // the jump, so that the bisection takes ~8 steps instead of ~60
  const double decades = std::log10(plan.emax / plan.emin) / static_cast<double>(static_cast<float>(n - 1));
  for (size_t k = 1; k < n; ++k) {
    // smallest E in [emin, emax) with index >= k, or emax if none
    uint64_t a = lo, b = hi;
    const double guess = plan.emin * std::pow(10.0, k * decades);
    if (guess > plan.emin && guess < plan.emax) {
      const uint64_t g = bits_of(guess);
      if (g - lo > 64 && !reaches(g - 64, k)) a = g - 63;
      if (hi - g > 64 && reaches(g + 64, k)) b = g + 64;
    }
    while (a < b) {
      const uint64_t mid = a + (b - a) / 2;
      if (reaches(mid, k)) {
        b = mid;
      } else {
        a = mid + 1;
      }
    }
    // E >= emax maps to n - 1 regardless; an edge at emax covers that.
    plan.edges[k] = from_bits(a);
  }
}

// The energy of |u|^2 = q, rounded as the reference rounds it.
double energy_of(float q, bool fourvel) {
  return fourvel ? static_cast<double>(std::sqrt(q)) : std::sqrt(1.0 + static_cast<double>(q));
}

// Smallest float q >= 0 with energy_of(q) >= target (NaN for a NaN target).
float first_reaching(double target, bool fourvel) {
  const float inf = std::numeric_limits<float>::infinity();
  if (!(target == target)) return std::numeric_limits<float>::quiet_NaN();
  if (energy_of(0.0f, fourvel) >= target) return 0.0f;
  if (!(energy_of(std::numeric_limits<float>::max(), fourvel) >= target)) return inf;
  // a guess within a few floats, then a step at a time
  float q = static_cast<float>(std::min(target * target - (fourvel ? 0.0 : 1.0), 3e38));
  q = std::max(q, std::numeric_limits<float>::denorm_min());
  for (int step = 0; step < 64; ++step) {
    if (!(energy_of(q, fourvel) >= target)) {
      q = std::nextafter(q, inf);
    } else if (energy_of(std::nextafter(q, 0.0f), fourvel) >= target) {
      q = std::nextafter(q, 0.0f);
    } else {
      return q;
    }
  }
  uint32_t a = 0, b = 0x7f800000u;  // bit patterns of 0 .. inf are ordered like the values
  while (a < b) {
    const uint32_t mid = a + (b - a) / 2;
    std::memcpy(&q, &mid, sizeof q);
    if (energy_of(q, fourvel) >= target) b = mid; else a = mid + 1;
  }
  std::memcpy(&q, &a, sizeof q);
  return q;
}

// Thresholds of |u|^2 and the estimate, for both energy kinds.
void build_thresholds(rgn_hist_plan& plan) {
  const size_t n = plan.nb;
  const float inf = std::numeric_limits<float>::infinity();
  std::vector<float> thr(2 * (n + 1));
  for (int fourvel = 0; fourvel < 2; ++fourvel) {
    float* t = thr.data() + fourvel * (n + 1);
    t[0] = -inf;
    t[n] = std::numeric_limits<float>::quiet_NaN();  // never reached
    for (size_t k = 1; k < n; ++k) {
      // index >= k from edge k on, and from emax on (degenerate bins: edges at infinity)
      t[k] = first_reaching(plan.edges[k] < inf ? plan.edges[k] : static_cast<double>(plan.emax), fourvel);
    }
    // index ~ a log2(|u|^2 or 1 + |u|^2) + b
    plan.near[fourvel] = false;
    if (!(plan.emin > 0.0f && plan.emax > plan.emin && plan.emax < inf)) continue;
    const double lo = std::log2(static_cast<double>(plan.emin)), hi = std::log2(static_cast<double>(plan.emax));
    const double scale = (n - 1) / (hi - lo);
    plan.est_a[fourvel] = static_cast<float>(0.5 * scale);
    plan.est_b[fourvel] = static_cast<float>(-scale * lo);
    // float errors of the estimate: a few ulps of its two terms
    bool near = scale * (std::fabs(lo) + std::fabs(hi) + 2.0) * 1e-6 < 0.1;
    for (size_t k = 1; k < n && near; ++k) {
      const double q = t[k];
      // the kernel's log2 reads a subnormal |u|^2 as zero
      if (!(q < inf) || (fourvel && q > 0.0 && q < std::numeric_limits<float>::min())) {
        near = false;
        break;
      }
      const double est = static_cast<double>(plan.est_a[fourvel]) * std::log2(fourvel ? q : 1.0 + q) + plan.est_b[fourvel];
      // gamma bins from below 1 start at |u| = 0, whose first thresholds are 0
      near = (est > k - 0.85 || (q == 0.0 && est >= k - 0.85)) && (est < k + 0.85 || q == 0.0);
    }
    plan.near[fourvel] = near;
  }
  plan.d_thr.reset(thr.size() * sizeof(float));
  RGN_HIP(hipMemcpy(plan.d_thr.ptr, thr.data(), plan.d_thr.bytes, hipMemcpyHostToDevice));
}

// (float)(1 / E) of particles.cpp:247-252 for log-spaced bins, E = sqrtf(q) or
// sqrt(1 + q), from an FP64 reciprocal square root y (hardware estimate, one
// third-order step).  |u|: E is the root rounded to float, and one Newton step
// from y gives 1 / E to about one double ulp.  The terms are the reference's
// except within a few double ulps of a float rounding boundary (~1e-9 of them).
template <bool FOURVEL>
__device__ __forceinline__ float energy_term(float q) {
  if (!(q >= 0x1p-126f && q < 0x1p127f)) {
    // 0, subnormal, huge, NaN: as 1.0 / e gives them
    const double e = FOURVEL ? static_cast<double>(sqrtf(q)) : sqrt(1.0 + static_cast<double>(q));
    return static_cast<float>(1.0 / e);
  }
  const double d = FOURVEL ? static_cast<double>(q) : 1.0 + static_cast<double>(q);
  const double y0 = __builtin_amdgcn_rsq(d);
  const double r = fma(-d * y0, y0, 1.0);
  const double y = fma(y0 * r, fma(r, 0.375, 0.5), y0);
  if (!FOURVEL) return static_cast<float>(y);
  const double e = static_cast<double>(static_cast<float>(d * y));
  return static_cast<float>(fma(y, fma(-e, y, 1.0), y));
}

struct HistParams {
  const float* thr;  // in LDS
  int nb;
  float a, b;  // the estimate
};

// particles.cpp:228-252 for one particle.  NEAR: the estimate is within one bin.
template <bool FOURVEL, bool LOGB, bool COUNT, bool NEAR>
__device__ __forceinline__ void bin_particle(float x, float y, float z, const HistParams& H,
                                             double* __restrict__ my_sum, unsigned* __restrict__ my_cnt) {
  const float q = x * x + y * y + z * z;  // float, as the reference
  const float est = fmaf(H.a, __builtin_amdgcn_logf(FOURVEL ? q : 1.0f + q), H.b);
  int idx = static_cast<int>(fminf(fmaxf(est, 0.0f), static_cast<float>(H.nb - 1)));
  const float lo = H.thr[idx], hi = H.thr[idx + 1];
  idx += (q >= hi) - (q < lo);
  if (!NEAR) {
    while (idx < H.nb - 1 && q >= H.thr[idx + 1]) ++idx;
    while (idx > 0 && !(q >= H.thr[idx])) --idx;
  }
  if (!(q == q)) idx = H.nb - 1;  // NaN: the x86 reference's size_t conversion lands here
  if (COUNT) atomicAdd(my_cnt + idx, 1u);
  if (LOGB) atomicAdd(my_sum + idx, static_cast<double>(energy_term<FOURVEL>(q)));
}

// Four consecutive floats at any float address (one 16-byte load).
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));

// Each thread keeps two 16-byte loads per component in flight (8 particles); the
// last n % 4 particles go one per thread.  COUNT: integer counts are kept (linear
// bins sum ones, so their sums are the counts).  43 vector instructions a
// particle, 14 of them FP64 (57 when the energy was formed); bound by memory
// latency and LDS atomics (counters: VALU 40%, LDS 45% of the cycles).  2^24 particles with the
// momenta in HBM (201 MB, 39 us at the rate of a copy): 200 log bins 56.6 -> 55.5
// us, 1000 bins 80 -> 64, linear bins 55 -> 49; 2^24 + 3 particles 60 -> 56.
template <bool FOURVEL, bool LOGB, bool COUNT, bool NEAR>
__global__ void __launch_bounds__(kThreads) hist_kernel(const float* __restrict__ ux, const float* __restrict__ uy,
                                                        const float* __restrict__ uz, size_t n,
                                                        const float* __restrict__ g_thr, int nb, float a, float b,
                                                        int qper, unsigned* __restrict__ cpart,
                                                        double* __restrict__ partials) {
  extern __shared__ __align__(16) unsigned char smem[];
  // 4 * qper private sub-histograms per block: one per wave and lane group of
  // 64 / qper lanes (fewer same-address atomics where energies pile up in a
  // few bins); pitch nb + 1 staggers the copies over the LDS banks
  const int copies = 4 * qper, pitch = nb + 1;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  double* lsum = reinterpret_cast<double*>(smem);                                 // LOGB: [copies][pitch]
  unsigned* lcnt = reinterpret_cast<unsigned*>(lsum + (LOGB ? copies * pitch : 0));  // COUNT: [copies][pitch]
  float* lthr = reinterpret_cast<float*>(lcnt + (COUNT ? copies * pitch : 0));    // [nb + 1]
  for (int i = threadIdx.x; i < copies * pitch; i += kThreads) {
    if (LOGB) lsum[i] = 0.0;
    if (COUNT) lcnt[i] = 0u;
  }
  for (int i = threadIdx.x; i <= nb; i += kThreads) lthr[i] = g_thr[i];
  __syncthreads();
  const HistParams H{lthr, nb, a, b};
  const int copy = wave * qper + lane / (64 / qper);
  double* my_sum = lsum + copy * pitch;
  unsigned* my_cnt = lcnt + copy * pitch;
  auto bin = [&](float x, float y, float z) {
    bin_particle<FOURVEL, LOGB, COUNT, NEAR>(x, y, z, H, my_sum, my_cnt);
  };
  const size_t stride = static_cast<size_t>(gridDim.x) * kThreads;
  const size_t tid = blockIdx.x * static_cast<size_t>(kThreads) + threadIdx.x;
  const size_t nq = n / 4;
  const float4u* x4 = reinterpret_cast<const float4u*>(ux);
  const float4u* y4 = reinterpret_cast<const float4u*>(uy);
  const float4u* z4 = reinterpret_cast<const float4u*>(uz);
  for (size_t q = tid; q < nq; q += 2 * stride) {
    const bool two = q + stride < nq;
    const size_t q1 = two ? q + stride : q;
    const float4u a0 = x4[q], b0 = y4[q], c0 = z4[q], a1 = x4[q1], b1 = y4[q1], c1 = z4[q1];
    bin(a0.x, b0.x, c0.x);
    bin(a0.y, b0.y, c0.y);
    bin(a0.z, b0.z, c0.z);
    bin(a0.w, b0.w, c0.w);
    if (two) {
      bin(a1.x, b1.x, c1.x);
      bin(a1.y, b1.y, c1.y);
      bin(a1.z, b1.z, c1.z);
      bin(a1.w, b1.w, c1.w);
    }
  }
  const size_t p = 4 * nq + tid;
  if (p < n) bin(ux[p], uy[p], uz[p]);
  __syncthreads();
  for (int i = threadIdx.x; i < nb; i += kThreads) {
    unsigned c = 0;
    double s = 0.0;
    for (int q = 0; q < copies; ++q) {  // fixed order
      if (COUNT) c += lcnt[q * pitch + i];
      if (LOGB) s += lsum[q * pitch + i];
    }
    if (COUNT) cpart[static_cast<size_t>(blockIdx.x) * nb + i] = c;
    if (LOGB) partials[static_cast<size_t>(blockIdx.x) * nb + i] = s;
  }
}

// Fixed-order sums of the per-block partials.  A block takes BINS bins of the sums
// or of the counts, a part of the rows per thread, kCombineRows of them in flight.
// No global atomics.  The partials are rows of bins: as columns, 8 bytes into
// each of nb cache lines per block, the histogram kernel took 40.3 instead of
// 37.6 us at 2^24 particles and 200 bins, and a call at 1000 bins 54.8 instead of
// 42.1 (4e6 particles 34.1 and 21.5; 200 bins, three stores in turn, 55.1 and
// 49.2).
constexpr int kCombineThreads = 1024;
constexpr int kCombineRows = 16;

// The block's sum of column col; the total of bin threadIdx.x in the first
// BINS threads.
template <int BINS, class Total, class T>
__device__ __forceinline__ Total column_sum(const T* __restrict__ rows, int nblocks, int nb, int col) {
  constexpr int kParts = kCombineThreads / BINS;
  const int bin = threadIdx.x % BINS, part = threadIdx.x / BINS;
  Total s = 0;
  for (int b = part; b < nblocks; b += kCombineRows * kParts) {
    T v[kCombineRows];
#pragma unroll
    for (int k = 0; k < kCombineRows; ++k) {
      v[k] = rows[static_cast<size_t>(b + k * kParts < nblocks ? b + k * kParts : b) * nb + col];
    }
#pragma unroll
    for (int k = 0; k < kCombineRows; ++k) s += b + k * kParts < nblocks ? v[k] : T(0);
  }
  // the wave's parts, then the waves
#pragma unroll
  for (int w = BINS; w < 64; w <<= 1) s += __shfl_xor(s, w);
  __shared__ Total red[kCombineThreads / 64][BINS];
  if ((threadIdx.x & 63) < BINS) red[threadIdx.x / 64][bin] = s;
  __syncthreads();
  s = red[0][bin];
#pragma unroll
  for (int w = 1; w < kCombineThreads / 64; ++w) s += red[w][bin];
  return s;
}

// FP64 sums (LOGB, blocks y = 0; else the counts) to out, uint64 counts (COUNT,
// the last blocks y) to counts where it is not null.
template <int BINS, bool LOGB, bool COUNT>
__global__ void __launch_bounds__(kCombineThreads) hist_combine_kernel(const double* __restrict__ partials,
                                                                       const unsigned* __restrict__ cpart,
                                                                       int nblocks, int nb, float* __restrict__ out,
                                                                       unsigned long long* __restrict__ counts) {
  const int i = blockIdx.x * BINS + threadIdx.x % BINS, col = min(i, nb - 1);
  const bool store = threadIdx.x < BINS && i < nb;
  if (LOGB && blockIdx.y == 0) {
    const double s = column_sum<BINS, double>(partials, nblocks, nb, col);
    if (store) out[i] = static_cast<float>(s);
  } else if (COUNT) {
    const unsigned long long c = column_sum<BINS, unsigned long long>(cpart, nblocks, nb, col);
    if (store && !LOGB) out[i] = static_cast<float>(static_cast<double>(c));
    if (store && counts) counts[i] = c;
  }
}

// Launch shape of one histogram call.
struct HistShape {
  int grid = 1;
  size_t smem = 0;
  int qper = 1;
};

HistShape hist_shape(const rgn_hist_plan& plan, size_t n, bool counts) {
  HistShape sh;
  const int nb = plan.nb;
  const size_t tiles = ceil_div(std::max<size_t>(n, 1), kThreads * 8);
  // lane groups per wave: as many private copies as fit in 24 KB of LDS (at
  // 200 bins two per wave, and seven blocks share a CU: 51 -> 50 us at 2^24
  // against four per wave in 48 KB)
  const size_t per_copy =
    static_cast<size_t>(nb + 1) * ((plan.log_bins ? sizeof(double) : 0) + (counts || !plan.log_bins ? sizeof(unsigned) : 0));
  const size_t thr = (nb + 1) * sizeof(float);
  sh.qper = 4;
  while (sh.qper > 1 && 4 * sh.qper * per_copy + thr > 24 * 1024) sh.qper /= 2;
  sh.smem = 4 * sh.qper * per_copy + thr;
  // one round of blocks: as many per CU as the LDS holds (at most 8), so the
  // per-block clearing and reduction of the private copies is paid once
  const size_t per_cu = std::max<size_t>(1, std::min<size_t>(8, (160 * 1024) / sh.smem));
  sh.grid = static_cast<int>(std::min<size_t>(tiles, static_cast<size_t>(num_cus()) * per_cu));
  return sh;
}

// Bytes of per-block partials a launch of `grid` blocks writes (FP64 sums and
// uint32 counts per bin and block).  Every entry is written before it is read.
size_t hist_partial_bytes(int nb, int grid) {
  return (sizeof(double) + sizeof(unsigned)) * static_cast<size_t>(nb) * grid;
}

void launch_hist(const rgn_hist_plan& plan, const float* const d_u[3], size_t n, int fourvel,
                 float* d_hist, uint64_t* d_counts, const HistShape& sh, double* partials,
                 hipStream_t st) {
  const int nb = plan.nb, kind = fourvel ? 1 : 0;
  const bool count = d_counts || !plan.log_bins;
  unsigned* cpart = reinterpret_cast<unsigned*>(partials + static_cast<size_t>(nb) * sh.grid);
  const float* thr = plan.d_thr.as<float>() + kind * (nb + 1);
  auto launch = [&](auto kernel) {
    kernel<<<sh.grid, kThreads, sh.smem, st>>>(d_u[0], d_u[1], d_u[2], n, thr, nb, plan.est_a[kind], plan.est_b[kind],
                                               sh.qper, cpart, partials);
  };
  const bool near = plan.near[kind];
  switch ((kind ? 8 : 0) + (plan.log_bins ? 4 : 0) + (count ? 2 : 0) + (near ? 1 : 0)) {
#define RGN_HIST_CASES(F_)                                                 \
  case F_ * 8 + 2: launch(hist_kernel<F_, false, true, false>); break;     \
  case F_ * 8 + 3: launch(hist_kernel<F_, false, true, true>); break;      \
  case F_ * 8 + 4: launch(hist_kernel<F_, true, false, false>); break;     \
  case F_ * 8 + 5: launch(hist_kernel<F_, true, false, true>); break;      \
  case F_ * 8 + 6: launch(hist_kernel<F_, true, true, false>); break;      \
  case F_ * 8 + 7: launch(hist_kernel<F_, true, true, true>); break;
    RGN_HIST_CASES(0)
    RGN_HIST_CASES(1)
#undef RGN_HIST_CASES
  }
  RGN_HIP(hipGetLastError());
  stage_mark(st, "hist_kernel");
  auto* out_counts = reinterpret_cast<unsigned long long*>(d_counts);
  auto combine = [&](auto bins) {
    constexpr int BINS = decltype(bins)::value;
    const dim3 blocks(static_cast<unsigned>(ceil_div(nb, BINS)), plan.log_bins && count ? 2 : 1);
    if (!plan.log_bins) {
      hist_combine_kernel<BINS, false, true><<<blocks, kCombineThreads, 0, st>>>(partials, cpart, sh.grid, nb, d_hist,
                                                                                 out_counts);
    } else if (count) {
      hist_combine_kernel<BINS, true, true><<<blocks, kCombineThreads, 0, st>>>(partials, cpart, sh.grid, nb, d_hist,
                                                                                out_counts);
    } else {
      hist_combine_kernel<BINS, true, false><<<blocks, kCombineThreads, 0, st>>>(partials, cpart, sh.grid, nb, d_hist,
                                                                                 nullptr);
    }
  };
  // enough blocks to read the rows, else whole cache lines of them (100 bins 4:
  // 45.0, 8: 44.9, 16: 46.6 us a call; 300 bins 46.1, 44.5, 45.6)
  if (nb <= 128) {
    combine(std::integral_constant<int, 4>{});
  } else if (nb <= 512) {
    combine(std::integral_constant<int, 8>{});
  } else {
    combine(std::integral_constant<int, 16>{});
  }
  RGN_HIP(hipGetLastError());
  stage_mark(st, "hist_combine_kernel");
}

}  // namespace
}  // namespace rgn

// Per-block partials of rgn_energy_hist_noalloc: a fixed device array (each
// device holds its own copy until the process ends), used instead of the
// library's allocated scratch.  Host code reaches it only through the address
// hipGetSymbolAddress returns on each device (noalloc_partials below).
constexpr size_t kHistNoAllocBytes = size_t{8} << 20;
static __device__ __align__(256) unsigned char scratch[kHistNoAllocBytes];

namespace {
std::mutex g_noalloc_mutex;
constexpr int kMaxDevices = 64;
void* g_noalloc_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device, looked up on the first
// call on that device and kept.
void* noalloc_partials() {
  int dev = 0;
  RGN_HIP(hipGetDevice(&dev));
  RGN_REQUIRE(dev >= 0 && dev < kMaxDevices, RGN_ERR_UNSUPPORTED, "device index out of range");
  std::lock_guard<std::mutex> lk(g_noalloc_mutex);
  if (!g_noalloc_ptr[dev]) {
    void* p = nullptr;
    RGN_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(::scratch)));
    RGN_REQUIRE(p != nullptr, RGN_ERR_HIP, "no device address for the histogram's fixed scratch");
    g_noalloc_ptr[dev] = p;
  }
  return g_noalloc_ptr[dev];
}
}  // namespace

using namespace rgn;

extern "C" {

int rgn_hist_plan_create(const float* h_bins, int nb, int log_bins, rgn_hist_plan** out) {
  return guarded([&] {
    RGN_REQUIRE(out != nullptr && h_bins != nullptr, RGN_ERR_INVALID, "null argument");
    RGN_REQUIRE(nb >= 1, RGN_ERR_INVALID, "no energy bins");
    // LDS of the smallest configuration: 4 private copies (pitch nb + 1) and as much again for the thresholds
    RGN_REQUIRE(static_cast<size_t>(nb + 1) * (4 * (sizeof(double) + sizeof(unsigned)) + sizeof(double)) <=
                  150 * 1024,
                RGN_ERR_UNSUPPORTED, "too many energy bins for the LDS histogram (at most 2741)");
    auto* plan = new rgn_hist_plan();
    plan->nb = nb;
    plan->log_bins = log_bins ? 1 : 0;
    // particles.cpp:200-215 ("EnergyBinsMinMax")
    float lo = h_bins[0], hi = h_bins[0];
    for (int i = 0; i < nb; ++i) {
      lo = h_bins[i] < lo ? h_bins[i] : lo;
      hi = h_bins[i] > hi ? h_bins[i] : hi;
    }
    plan->emin = lo;
    plan->emax = hi;
    try {
      if (lo > 0.0f && hi > lo) {
        build_edges(*plan);
      } else {
        // degenerate bins: every finite energy lands in bin 0 or n - 1
        plan->edges.assign(nb + 1, std::numeric_limits<double>::infinity());
        plan->edges[0] = -std::numeric_limits<double>::infinity();
      }
      build_thresholds(*plan);
    } catch (...) {
      delete plan;
      throw;
    }
    *out = plan;
  });
}

int rgn_hist_plan_destroy(rgn_hist_plan* plan) {
  delete plan;
  return RGN_OK;
}

int rgn_energy_hist(const rgn_hist_plan* plan, const float* const d_u[3], size_t n, int fourvel,
                    float* d_hist, uint64_t* d_counts, rgn_stream_t stream) {
  return guarded([&] {
    RGN_REQUIRE(plan != nullptr, RGN_ERR_INVALID, "null plan");
    RGN_REQUIRE(d_u && d_u[0] && d_u[1] && d_u[2] && d_hist, RGN_ERR_INVALID, "null argument");
    hipStream_t st = as_stream(stream);
    ScratchUse order(st);
    const HistShape sh = hist_shape(*plan, n, d_counts != nullptr);
    double* partials = static_cast<double*>(rgn::scratch(hist_partial_bytes(plan->nb, sh.grid), 2));
    launch_hist(*plan, d_u, n, fourvel, d_hist, d_counts, sh, partials, st);
  });
}

int rgn_energy_hist_noalloc(const rgn_hist_plan* plan, const float* const d_u[3], size_t n,
                            int fourvel, float* d_hist, uint64_t* d_counts, rgn_stream_t stream) {
  return guarded([&] {
    RGN_REQUIRE(plan != nullptr, RGN_ERR_INVALID, "null plan");
    RGN_REQUIRE(d_u && d_u[0] && d_u[1] && d_u[2] && d_hist, RGN_ERR_INVALID, "null argument");
    HistShape sh = hist_shape(*plan, n, d_counts != nullptr);
    // the grid is cut to what the fixed array holds: bins x blocks x 12 bytes
    const size_t per_block = hist_partial_bytes(plan->nb, 1);
    RGN_REQUIRE(per_block <= kHistNoAllocBytes, RGN_ERR_UNSUPPORTED,
                "energy bins beyond the fixed scratch of rgn_energy_hist_noalloc");
    sh.grid = static_cast<int>(std::min<size_t>(sh.grid, kHistNoAllocBytes / per_block));
    double* partials = static_cast<double*>(noalloc_partials());
    launch_hist(*plan, d_u, n, fourvel, d_hist, d_counts, sh, partials, as_stream(stream));
  });
}

// Jump points of the index function (nb + 1 doubles), for tests.
int rgn_hist_plan_edges(const rgn_hist_plan* plan, double* h_edges) {
  return guarded([&] {
    RGN_REQUIRE(plan != nullptr && h_edges != nullptr, RGN_ERR_INVALID, "null argument");
    std::copy(plan->edges.begin(), plan->edges.end(), h_edges);
  });
}

}  // extern "C"
