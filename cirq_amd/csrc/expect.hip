// Pauli-string expectations, PauliSum application and norms (FP64 accumulation).
#include <algorithm>
#include <atomic>
#include <numeric>
#include <type_traits>
#include <vector>

#include <string.h>

#include "common.hpp"

namespace cqs {

constexpr int kRedBlocks = 512;  // k_inner: fixed grid => deterministic reduction order

// Pauli terms with any X masks, up to kPauliTerms per launch.
//
// Term t needs sum_i s(i) conj(psi[i ^ x]) psi[i], s(i) = (-1)^popcount(i & z).  The indices i and
// i ^ x give w s and conj(w) s (-1)^popcount(x & z), so the sum is 2 Re w or 2i Im w over half of the
// indices: where x reaches above the chunk, half of the chunks do the work.
// A workgroup owns a slice of the state in chunks of 2^kChunkBits amplitudes and kPauliGroup terms: it holds
// a chunk in registers and reads each term's partner chunk i ^ x (a permutation of one chunk, so reads
// stay coalesced; terms with equal x share it), two amplitudes to a load.  The state is read about
// 1 + kPauliGroup / 2 times per kPauliGroup terms, by workgroups that run side by side (the group is the
// fastest grid index) and find it in cache.  What bounds it is the FP64 arithmetic and, for small
// states, the launch: 200 4-local terms on 20 qubits take 160 us
// (183 X masks; a launch and a final per mask took 2.07 ms), 42 terms on 10 qubits one launch of 10 us (152 us).
// How terms fall into launches and groups does not enter any term's summation order.
constexpr int kPauliTerms = 96;   // arguments stay below 4 KB
constexpr int kPauliGroup = 8;    // terms of one workgroup (FP64 accumulators in registers)
constexpr int kChunkBits = 11;    // 256 threads x 4 pairs of amplitudes
// Slices of a state, fixed by n alone => deterministic reduction order: 512, two workgroups per CU for one group of terms;
// at most 256 below 22 qubits, where a chunk's work does not pay for reducing its sums (200 terms on 20 qubits: 169 us
// against 204).
constexpr int kPauliSlices = 512;
inline int pauli_slices(int n) {
  const int most = n >= 22 ? kPauliSlices : kPauliSlices / 2;
  return n - kChunkBits < 0 ? 1 : (int)std::min<uint64_t>(most, 1ull << (n - kChunkBits));
}
constexpr int kFewPauliTerms = 16;  // launches of so few take 0.6 KB of arguments each (3.4 KB: 3 us more for one term)
template <int kMax>
struct PauliBatch {
  int count;
  int out_idx[kMax];
  uint64_t x[kMax];
  uint64_t z[kMax];
  double cr[kMax], ci[kMax];
};

// Amplitudes i and i + 1 (i even); `pairs`: the state starts on 16 bytes.
__device__ __forceinline__ float4 load_pair(const float2* amps, uint64_t i, int pairs) {
  if (pairs) return *reinterpret_cast<const float4*>(amps + i);
  const float2 u = amps[i], v = amps[i + 1];
  return make_float4(u.x, u.y, v.x, v.y);
}

// Writes out[out_idx] = c * sum when one slice covers the state, else the slice's share of every
// term's sum to partials[(term * slices + slice) * 2 + {0,1}].  pre: as in k_expect_z (1 for density matrices).
template <bool kDm, int kMax>
__global__ __launch_bounds__(256) void k_pauli_terms(const float2* __restrict__ amps, int n, int slices, int pairs,
                                                     float pre, PauliBatch<kMax> tb, double* __restrict__ partials,
                                                     double* __restrict__ out) {
  __shared__ double red[4][kPauliGroup][2];
  const uint64_t N = 1ull << n;
  const int ngroups = (tb.count + kPauliGroup - 1) / kPauliGroup;
  const int slice = blockIdx.x / ngroups, t0 = (blockIdx.x % ngroups) * kPauliGroup;
  const int tid = threadIdx.x;
  const int cnt = tb.count - t0 < kPauliGroup ? tb.count - t0 : kPauliGroup;
  double ar[kPauliGroup], ai[kPauliGroup];
  uint32_t tneg = 0;  // bit t: this thread's part of term t's sign (index bits 1..8)
#pragma unroll
  for (int t = 0; t < kPauliGroup; ++t) {
    ar[t] = ai[t] = 0.0;
    if (t < cnt) tneg |= (uint32_t)(__popcll((uint64_t)(tid << 1) & tb.z[t0 + t]) & 1) << t;
  }
  const uint64_t chunks = N >> kChunkBits ? N >> kChunkBits : 1;
  for (uint64_t c = slice; c < chunks; c += slices) {
    const uint64_t base = c << kChunkBits;
    // element (e, h): index base | e << 9 | tid << 1 | h
    float2 a[8];
    if constexpr (!kDm) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint64_t i = base | ((uint64_t)e << 9) | (tid << 1);
        a[2 * e] = a[2 * e + 1] = make_float2(0.f, 0.f);
        if (i + 1 < N) {
          const float4 v = load_pair(amps, i, pairs);
          a[2 * e] = make_float2(v.x, v.y);
          a[2 * e + 1] = make_float2(v.z, v.w);
        } else if (i < N) {
          a[2 * e] = amps[i];
        }
      }
    }
    float2 b[8];
    uint64_t px = ~0ull;
#pragma unroll
    for (int t = 0; t < kPauliGroup; ++t) {
      if (t >= cnt) break;
      const uint64_t x = tb.x[t0 + t], z = tb.z[t0 + t];
      // Half of the chunks for an x that leaves the chunk (sums are doubled below): of a chunk and its partner the one
      // whose bit at the top of x equals the state's top bit, or, with that in x, the one where it is clear.  The
      // top bit numbers a slice's chunks, so every slice does its share (X on bit 12 of 29: 1.6 ms; taking the lower
      // half of each pair, the chunks of half of the slices, and 256 slices 3.9 ms).
      if (!kDm && (x >> kChunkBits) != 0) {
        const int top = 63 - __builtin_clzll(x);
        if (((base >> top) ^ (top < n - 1 ? base >> (n - 1) : 0)) & 1) continue;
      }
      const bool odd = __popcll(x & z) & 1;
      if (x != px) {
        px = x;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint64_t i = base | ((uint64_t)e << 9) | (tid << 1);
          b[2 * e] = b[2 * e + 1] = make_float2(0.f, 0.f);
          if constexpr (kDm) {
            if (i < N) b[2 * e] = amps[i * N + (i ^ x)];
            if (i + 1 < N) b[2 * e + 1] = amps[(i + 1) * N + ((i + 1) ^ x)];
          } else {
            if (i + 1 < N) {
              const float4 v = load_pair(amps, (i ^ x) & ~1ull, pairs);
              const bool swap = x & 1;
              b[2 * e] = swap ? make_float2(v.z, v.w) : make_float2(v.x, v.y);
              b[2 * e + 1] = swap ? make_float2(v.x, v.y) : make_float2(v.z, v.w);
            } else if (i < N) {
              b[2 * e] = amps[i];
            }
          }
        }
      }
      double sr = 0.0, si = 0.0;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int zk = (int)((z & 1) | ((z >> 8) & 6));  // the z bits of (h, e)
        const double sg = (__popc(k & zk) & 1) ? -1.0 : 1.0;
        if constexpr (kDm) {
          sr = fma(sg, (double)b[k].x, sr);
          si = fma(sg, (double)b[k].y, si);
        } else {  // conj(b) a: its real part, or its imaginary part for an odd number of Y
          const double br = b[k].x * pre, bi = b[k].y * pre, xr = a[k].x * pre, xi = a[k].y * pre;
          const double w = odd ? fma(br, xi, -bi * xr) : fma(br, xr, bi * xi);
          sr = fma(sg, w, sr);
        }
      }
      const bool neg = (((tneg >> t) & 1) ^ (__popcll(base & z) & 1)) != 0;
      ar[t] += neg ? -sr : sr;
      if constexpr (kDm) ai[t] += neg ? -si : si;
    }
  }
  const int lane = tid & 63, w = tid >> 6;
#pragma unroll
  for (int t = 0; t < kPauliGroup; ++t) {
    if (t >= cnt) break;
    const double sr = wave_sum(ar[t]), si = kDm ? wave_sum(ai[t]) : 0.0;
    if (lane == 0) {
      red[w][t][0] = sr;
      red[w][t][1] = si;
    }
  }
  __syncthreads();
  if (tid >= cnt) return;
  const int t = t0 + tid;
  double sr = (red[0][tid][0] + red[1][tid][0]) + (red[2][tid][0] + red[3][tid][0]);
  double si = (red[0][tid][1] + red[1][tid][1]) + (red[2][tid][1] + red[3][tid][1]);
  if constexpr (!kDm) {
    if ((tb.x[t] >> kChunkBits) != 0) sr *= 2.0;
    if (__popcll(tb.x[t] & tb.z[t]) & 1) {
      si = sr;
      sr = 0.0;
    }
  }
  if (slices == 1) {
    out[2 * tb.out_idx[t] + 0] = tb.cr[t] * sr - tb.ci[t] * si;
    out[2 * tb.out_idx[t] + 1] = tb.cr[t] * si + tb.ci[t] * sr;
  } else {
    partials[((size_t)t * slices + slice) * 2 + 0] = sr;
    partials[((size_t)t * slices + slice) * 2 + 1] = si;
  }
}

// One wave per term sums its slices in a fixed order.
template <int kMax>
__global__ __launch_bounds__(64) void k_pauli_final(const double* __restrict__ partials, int slices, PauliBatch<kMax> tb,
                                                    double* __restrict__ out) {
  const int t = blockIdx.x;
  double sr = 0.0, si = 0.0;
  for (int b = threadIdx.x; b < slices; b += 64) {
    sr += partials[((size_t)t * slices + b) * 2 + 0];
    si += partials[((size_t)t * slices + b) * 2 + 1];
  }
  sr = wave_sum(sr);
  si = wave_sum(si);
  if (threadIdx.x == 0) {
    out[2 * tb.out_idx[t] + 0] = tb.cr[t] * sr - tb.ci[t] * si;
    out[2 * tb.out_idx[t] + 1] = tb.cr[t] * si + tb.ci[t] * sr;
  }
}

// partials[2 * blockIdx + {0,1}] = this block's share of sum_i conj(a_i) b_i (FP64, fixed order).
__global__ __launch_bounds__(256) void k_inner(const float2* __restrict__ a, const float2* __restrict__ b,
                                               uint64_t N, double* __restrict__ partials) {
  __shared__ double red[4][2];
  double sr = 0.0, si = 0.0;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += stride) {
    const float2 x = a[i], y = b[i];
    const double xr = x.x, xi = x.y, yr = y.x, yi = y.y;
    sr += xr * yr + xi * yi;
    si += xr * yi - xi * yr;
  }
  sr = wave_sum(sr);
  si = wave_sum(si);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) {
    red[w][0] = sr;
    red[w][1] = si;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    const int c = threadIdx.x;
    partials[2 * blockIdx.x + c] = (red[0][c] + red[1][c]) + (red[2][c] + red[3][c]);
  }
}

__global__ __launch_bounds__(64) void k_inner_final(const double* __restrict__ partials, int nblocks,
                                                    double* __restrict__ out) {
  double sr = 0.0, si = 0.0;
  for (int b = threadIdx.x; b < nblocks; b += 64) {
    sr += partials[2 * b];
    si += partials[2 * b + 1];
  }
  sr = wave_sum(sr);
  si = wave_sum(si);
  if (threadIdx.x == 0) {
    out[0] = sr;
    out[1] = si;
  }
}

// Terms without X or Y (x mask 0): sum_i (-1)^popcount(i & z) |psi_i|^2, up to 64 terms per read
// of the state.  Each thread takes 16 consecutive amplitudes i = 16g + j, so the sign splits into
// (-1)^popcount(g & z>>4), the same for the 16, times (-1)^popcount(j & z&15), the same for every
// thread: one FP64 FMA per amplitude and distinct low mask.  A thread's groups are
// g = lo + k * stride (lo < stride, stride = 2^sbits the grid's threads), so the group sign is
// parity(lo & z>>4), fixed per thread, times parity(k * stride & z>>4), which depends only on the
// z bits at 4 + sbits and above.  Terms that agree in their low 4 bits and in those high bits form
// one class: a thread accumulates one FP64 sum per class (lane j evaluates the iteration sign of
// class j and a ballot shares it) and gives each term its class sum with the term's fixed sign
// (negation is exact, so every term's sum is the same as with the sign applied per group).
// |psi_i|^2 is exact in FP64 up to its final rounding.  Which thread sums which groups does not
// depend on the batch, so every term's reduction order is fixed.
constexpr int kZTerms = 64;       // terms per launch
constexpr int kZBatch = kZTerms;
constexpr int kZClasses = 24;     // classes per launch (FP64 accumulators in registers)
constexpr int kZBlocks = 2048;    // fixed grid => deterministic reduction order
struct ZBatch {
  int count;                      // terms
  int nclass;                     // classes
  uint64_t newrun;                // bit j: class j's low 4 bits differ from class j - 1's (bit 0 set)
  uint64_t z[kZBatch];            // the terms' z masks
  uint64_t zc[kZClasses];         // a z mask of each class (its low 4 bits and high bits)
  uint8_t cls[kZBatch];           // term -> class
};

// pre: every amplitude is multiplied by it (in FP32, as a scaled state would hold it) before its square, so the
// norm of a scaled state is one read of the state (435 us at 28 qubits, where the kernel is bound by that read).
// Copying the state, scaling the copy and reading that were three passes over it: 25.0 -> 23.1 ms for the
// amplitudes of a 28-qubit circuit; the two products per amplitude are hidden behind the loads.
__global__ __launch_bounds__(256) void k_expect_z(const float2* __restrict__ amps, int n, float pre, ZBatch zb,
                                                  double* __restrict__ partials) {
  __shared__ double red[4][kZTerms];
  __shared__ int zls[kZClasses];  // low 4 z bits per class, read inside the loop (not kept in registers)
  const int tid = threadIdx.x;
  const int cnt = zb.count, ncl = zb.nclass;
  if (tid < kZClasses) zls[tid] = tid < ncl ? (int)(zb.zc[tid] & 15) : 0;
  __syncthreads();
  double acc[kZClasses];
#pragma unroll
  for (int j = 0; j < kZClasses; ++j) acc[j] = 0.0;
  const uint64_t G = 1ull << (n - 4);
  const uint64_t stride = (uint64_t)gridDim.x * 256;  // 2^19 whenever G >= 2^19 (full grid)
  const uint64_t lo = (uint64_t)blockIdx.x * 256 + tid;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const uint64_t zh_lane = lane < ncl ? zb.zc[lane] >> 4 : 0;
  const uint64_t iters = G > stride ? G / stride : 1;  // every thread runs them all: the ballot sees all lanes
  for (uint64_t k = 0; k < iters; ++k) {
    const uint64_t kpar = __ballot(__popcll((k * stride) & zh_lane) & 1);
    const uint64_t g = lo + k * stride;
    if (g >= G) continue;
    const float4* src = reinterpret_cast<const float4*>(amps + 16 * g);
    double p[16];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      float4 v = src[q];
      v = make_float4(v.x * pre, v.y * pre, v.z * pre, v.w * pre);
      p[2 * q] = fma((double)v.x, (double)v.x, (double)v.y * (double)v.y);
      p[2 * q + 1] = fma((double)v.z, (double)v.z, (double)v.w * (double)v.w);
    }
    // The host orders classes by their low 4 z bits, so the signed 16-term sum is formed once per
    // run of equal low masks (a uniform branch) and shared by the run's classes.  The run's mask is
    // read from LDS there (a barrier to code motion keeps the masks out of the registers).
    asm volatile("" ::: "memory");
    double w = 0.0;
#pragma unroll
    for (int j = 0; j < kZClasses; ++j) {
      if (j < ncl) {
        if ((zb.newrun >> j) & 1) {
          const int zl = __builtin_amdgcn_readfirstlane(zls[j]);
          w = 0.0;
#pragma unroll
          for (int q = 0; q < 16; ++q) w = fma((__popc(q & zl) & 1) ? -1.0 : 1.0, p[q], w);
        }
        acc[j] += ((kpar >> j) & 1) ? -w : w;
      }
    }
  }
  // each term: its class's sum with the term's fixed sign parity(lo & z>>4)
  for (int t = 0; t < cnt; ++t) {
    const int c = zb.cls[t];
    double v = acc[0];
#pragma unroll
    for (int j = 1; j < kZClasses; ++j) v = c == j ? acc[j] : v;
    const double sv = wave_sum((__popcll(lo & (zb.z[t] >> 4)) & 1) ? -v : v);
    if (lane == 0) red[wv][t] = sv;
  }
  __syncthreads();
  if (tid < cnt) partials[(size_t)blockIdx.x * kZBatch + tid] = (red[0][tid] + red[1][tid]) + (red[2][tid] + red[3][tid]);
}

struct ZFinal {
  int count;
  int nblocks;
  int out_idx[kZBatch];
  double cr[kZBatch], ci[kZBatch];
};

// One wave per term (workgroup k sums term k's block partials in a fixed order).
__global__ __launch_bounds__(64) void k_expect_z_final(const double* __restrict__ partials, ZFinal fb,
                                                       double* __restrict__ out) {
  const int k = blockIdx.x;
  double sv = 0.0;
  for (int b = threadIdx.x; b < fb.nblocks; b += 64) sv += partials[(size_t)b * kZBatch + k];
  sv = wave_sum(sv);
  if (threadIdx.x == 0) {
    out[2 * fb.out_idx[k] + 0] = fb.cr[k] * sv;
    out[2 * fb.out_idx[k] + 1] = fb.ci[k] * sv;
  }
}

constexpr int kApplyTerms = 32;
struct ApplyBatch {
  int count;
  int accumulate;
  uint64_t x[kApplyTerms];
  uint64_t z[kApplyTerms];
  double cr[kApplyTerms], ci[kApplyTerms];
};

// phi[j] (+)= sum_t c_t (-1)^popcount((j ^ x_t) & z_t) psi[j ^ x_t]
__global__ __launch_bounds__(256) void k_apply_paulisum(const float2* __restrict__ psi, float2* __restrict__ phi,
                                                        uint64_t N, ApplyBatch ab) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; j < N; j += stride) {
    double sr = 0.0, si = 0.0;
    if (ab.accumulate) {
      const float2 o = phi[j];
      sr = o.x;
      si = o.y;
    }
    for (int t = 0; t < ab.count; ++t) {
      const uint64_t src = j ^ ab.x[t];
      const float2 v = psi[src];
      const double s = (__popcll(src & ab.z[t]) & 1) ? -1.0 : 1.0;
      const double vr = s * v.x, vi = s * v.y;
      sr += ab.cr[t] * vr - ab.ci[t] * vi;
      si += ab.cr[t] * vi + ab.ci[t] * vr;
    }
    phi[j] = make_float2((float)sr, (float)si);
  }
}

// Term checks shared by the expectation entry points.
static int check_terms(int32_t n_qubits, int32_t is_dm, int32_t n_terms, const uint64_t* xmask, const uint64_t* zmask,
                       const double* coef) {
  CQS_REQUIRE(n_qubits >= 0 && n_qubits <= (is_dm ? 20 : CQS_MAX_BITS), "n_qubits=%d out of range", n_qubits);
  CQS_REQUIRE(n_terms >= 0, "n_terms < 0");
  if (n_terms == 0) return CQS_OK;
  CQS_REQUIRE(xmask && zmask && coef, "NULL term arrays");
  const uint64_t valid = n_qubits >= 64 ? ~0ull : ((1ull << n_qubits) - 1);
  for (int t = 0; t < n_terms; ++t)
    CQS_REQUIRE(!(xmask[t] & ~valid) && !(zmask[t] & ~valid), "term %d has masks beyond %d qubits", t,
                n_qubits);
  return CQS_OK;
}

// Launches over the terms in `order` (identity when NULL): runs of Z-only terms share a k_expect_z
// launch (up to 64), other terms a k_pauli_terms launch (up to 96).  States of one chunk take every
// term through k_pauli_terms, which then needs no second launch (z-only terms included: 7.4 + 3.7 us
// less at 10 qubits).  Every term's sum has a fixed reduction order whatever batch it lands in, so any
// order of the terms gives the same bits.  `partials` holds one launch's per-block partial sums.
static int expect_batches(const void* amps, int32_t n_qubits, int32_t is_dm, int32_t n_terms, const int* order,
                          const uint64_t* xmask, const uint64_t* zmask, const double* coef, double* out,
                          double* partials, hipStream_t s, float pre = 1.f) {
  auto term = [&](int i) { return order ? order[i] : i; };
  const uint64_t N = 1ull << n_qubits;
  const int slices = pauli_slices(n_qubits);
  const int zgrid = n_qubits >= 4 ? (int)std::min<uint64_t>(kZBlocks, ((N >> 4) + 255) / 256) : 0;
  for (int i = 0; i < n_terms;) {
    auto z_only = [&](int k) { return !is_dm && slices > 1 && xmask[term(k)] == 0; };
    if (z_only(i)) {
      ZBatch zb;
      ZFinal zf;
      memset(&zb, 0, sizeof(zb));
      // class key: the low 4 z bits and the z bits that the iteration index reaches (from bit
      // 4 + sbits up; none when the grid covers every group in one iteration)
      const uint64_t G = N >> 4, stride = (uint64_t)zgrid * 256;
      const int sbits = __builtin_ctzll(stride);
      const uint64_t hmask = G > stride ? ~0ull << (4 + sbits) : 0;
      auto key = [&](uint64_t z) { return (z & 15) | (z & hmask); };
      while (i < n_terms && zb.count < kZBatch && xmask[term(i)] == 0) {
        const int t = term(i);
        const uint64_t kz = key(zmask[t]);
        int c = 0;
        while (c < zb.nclass && key(zb.zc[c]) != kz) ++c;
        if (c == zb.nclass) {
          if (zb.nclass == kZClasses) break;  // the next launch takes it
          if (c == 0 || (kz & 15) != (zb.zc[c - 1] & 15)) zb.newrun |= 1ull << c;
          zb.zc[c] = zmask[t];
          ++zb.nclass;
        }
        zb.cls[zb.count] = (uint8_t)c;
        zb.z[zb.count] = zmask[t];
        zf.out_idx[zb.count] = t;
        zf.cr[zb.count] = coef[2 * t];
        zf.ci[zb.count] = coef[2 * t + 1];
        ++zb.count;
        ++i;
      }
      zf.count = zb.count;
      zf.nblocks = zgrid;
      hipLaunchKernelGGL(k_expect_z, dim3(zgrid), dim3(256), 0, s, (const float2*)amps, (int)n_qubits, pre, zb,
                         partials);
      hipLaunchKernelGGL(k_expect_z_final, dim3(zf.count), dim3(64), 0, s, (const double*)partials, zf, out);
      continue;
    }
    const int first = i;
    while (i < n_terms && i - first < kPauliTerms && !z_only(i)) ++i;
    auto launch = [&](auto max) {
      constexpr int kMax = decltype(max)::value;
      PauliBatch<kMax> tb;
      memset(&tb, 0, sizeof(tb));
      for (; tb.count < i - first; ++tb.count) {
        const int t = term(first + tb.count);
        tb.x[tb.count] = xmask[t];
        tb.z[tb.count] = zmask[t];
        tb.out_idx[tb.count] = t;
        tb.cr[tb.count] = coef[2 * t];
        tb.ci[tb.count] = coef[2 * t + 1];
      }
      const int pairs = (reinterpret_cast<uintptr_t>(amps) & 15) == 0;
      const dim3 grid((tb.count + kPauliGroup - 1) / kPauliGroup * slices);
      const auto kernel = is_dm ? &k_pauli_terms<true, kMax> : &k_pauli_terms<false, kMax>;
      hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, (const float2*)amps, (int)n_qubits, slices, pairs, pre, tb,
                         partials, out);
      if (slices > 1)
        hipLaunchKernelGGL(k_pauli_final<kMax>, dim3(tb.count), dim3(64), 0, s, (const double*)partials, slices, tb, out);
    };
    if (i - first <= kFewPauliTerms)
      launch(std::integral_constant<int, kFewPauliTerms>());
    else
      launch(std::integral_constant<int, kPauliTerms>());
  }
  CQS_HIP(hipGetLastError());
  return CQS_OK;
}

// Static scratch for cqs_expect_paulis_noalloc: one launch's partial sums, the largest any batch
// writes (2048 blocks x 64 Z terms, or 512 slices x 96 terms x 2 doubles): 1 MiB per GPU, held
// until the process ends.  In host code `scratch` is only a handle for hipGetSymbolAddress; the
// kernels get the device address that call returns, kept per device.
static __device__ __align__(256) double scratch[kZBatch * kZBlocks];
static_assert(2 * kPauliTerms * kPauliSlices <= kZBatch * kZBlocks && 2 * kRedBlocks <= kZBatch * kZBlocks,
              "the Z batch writes the most partial sums");
constexpr int kMaxDevices = 64;
static std::atomic<double*> g_scratch_ptr[kMaxDevices];

// The current device's address of `scratch`, looked up once per device (hipGetSymbolAddress with
// that device current).
static int scratch_for_current_device(double** out) {
  int dev = 0;
  CQS_HIP(hipGetDevice(&dev));
  CQS_REQUIRE(dev >= 0 && dev < kMaxDevices, "device %d beyond the %d the scratch table covers", dev, kMaxDevices);
  double* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    void* addr = nullptr;
    CQS_HIP(hipGetSymbolAddress(&addr, HIP_SYMBOL(scratch)));
    CQS_REQUIRE(addr != nullptr, "hipGetSymbolAddress returned NULL for the expectation scratch");
    p = (double*)addr;
    g_scratch_ptr[dev].store(p, std::memory_order_release);
  }
  *out = p;
  return CQS_OK;
}

}  // namespace cqs

using namespace cqs;

extern "C" {

size_t cqs_expect_workspace_bytes(int32_t n_terms) {
  (void)n_terms;
  return sizeof(double) * kZBatch * kZBlocks;
}

int cqs_expect_paulis(const void* amps, int32_t n_qubits, int32_t is_dm, int32_t n_terms,
                      const uint64_t* xmask, const uint64_t* zmask, const double* coef, double* out,
                      void* workspace, void* stream) {
  CQS_REQUIRE(amps != nullptr && out != nullptr && workspace != nullptr, "NULL pointer");
  if (int rc = check_terms(n_qubits, is_dm, n_terms, xmask, zmask, coef)) return rc;
  if (n_terms == 0) return CQS_OK;
  std::vector<int> order(n_terms);
  std::iota(order.begin(), order.end(), 0);
  // by X mask (terms with one X mask share reads); Z-only terms also by their low 4 z bits (k_expect_z)
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
    if (xmask[a] != xmask[b]) return xmask[a] < xmask[b];
    return xmask[a] == 0 && (zmask[a] & 15) < (zmask[b] & 15);
  });
  return expect_batches(amps, n_qubits, is_dm, n_terms, order.data(), xmask, zmask, coef, out, (double*)workspace,
                        as_stream(stream));
}

int cqs_expect_paulis_noalloc(const void* amps, int32_t n_qubits, int32_t is_dm, int32_t n_terms,
                              const uint64_t* xmask, const uint64_t* zmask, const double* coef, double* out,
                              void* stream) {
  CQS_REQUIRE(amps != nullptr && out != nullptr, "NULL pointer");
  if (int rc = check_terms(n_qubits, is_dm, n_terms, xmask, zmask, coef)) return rc;
  if (n_terms == 0) return CQS_OK;
  CQS_REQUIRE(cqs_expect_workspace_bytes(n_terms) <= sizeof(scratch),
              "expectation scratch of %zu bytes exceeds the static %zu-byte array", cqs_expect_workspace_bytes(n_terms),
              sizeof(scratch));
  double* partials = nullptr;
  if (int rc = scratch_for_current_device(&partials)) return rc;
  // terms in the caller's order: runs of equal X masks share launches (no host sort, no allocation)
  return expect_batches(amps, n_qubits, is_dm, n_terms, nullptr, xmask, zmask, coef, out, partials,
                        as_stream(stream));
}

int cqs_norm2(const void* amps, int32_t n_bits, double* out, void* workspace, void* stream) {
  return cqs_norm2_scaled(amps, n_bits, 1.f, out, workspace, stream);
}

int cqs_norm2_scaled(const void* amps, int32_t n_bits, float scale, double* out, void* workspace, void* stream) {
  // A 1-term "expectation" of the identity over all 2^n_bits entries, real part in out[0].
  CQS_REQUIRE(amps != nullptr && out != nullptr && workspace != nullptr, "NULL pointer");
  CQS_REQUIRE(n_bits >= 0 && n_bits <= CQS_MAX_BITS, "n_bits=%d out of range", n_bits);
  const uint64_t x = 0, z = 0;
  const double c[2] = {1.0, 0.0};
  return expect_batches(amps, n_bits, 0, 1, nullptr, &x, &z, c, out, (double*)workspace, as_stream(stream), scale);
}

int cqs_inner(const void* a, const void* b, int32_t n_bits, double* out, void* workspace, void* stream) {
  CQS_REQUIRE(a != nullptr && b != nullptr && out != nullptr && workspace != nullptr, "NULL pointer");
  CQS_REQUIRE(n_bits >= 0 && n_bits <= CQS_MAX_BITS, "n_bits=%d out of range", n_bits);
  const uint64_t N = 1ull << n_bits;
  hipStream_t s = as_stream(stream);
  const int grid = (int)std::max<uint64_t>(1, std::min<uint64_t>(kRedBlocks, (N + 255) / 256));
  hipLaunchKernelGGL(k_inner, dim3(grid), dim3(256), 0, s, (const float2*)a, (const float2*)b, N, (double*)workspace);
  hipLaunchKernelGGL(k_inner_final, dim3(1), dim3(64), 0, s, (const double*)workspace, grid, out);
  CQS_HIP(hipGetLastError());
  return CQS_OK;
}

int cqs_apply_paulisum(const void* psi, void* phi, int32_t n_qubits, int32_t n_terms, const uint64_t* xmask,
                       const uint64_t* zmask, const double* coef, void* stream) {
  CQS_REQUIRE(psi != nullptr && phi != nullptr && psi != phi, "psi/phi must be distinct non-NULL");
  CQS_REQUIRE(n_qubits >= 0 && n_qubits <= CQS_MAX_BITS, "n_qubits=%d out of range", n_qubits);
  CQS_REQUIRE(n_terms >= 0, "n_terms < 0");
  CQS_REQUIRE(n_terms == 0 || (xmask && zmask && coef), "NULL term arrays");
  const uint64_t valid = (1ull << n_qubits) - 1;
  for (int t = 0; t < n_terms; ++t)
    CQS_REQUIRE(!(xmask[t] & ~valid) && !(zmask[t] & ~valid), "term %d has masks beyond %d qubits", t, n_qubits);
  const uint64_t N = 1ull << n_qubits;
  hipStream_t s = as_stream(stream);
  int grid = (int)std::min<uint64_t>(65536, (N + 255) / 256);
  if (grid < 1) grid = 1;
  int done = 0;
  do {
    ApplyBatch ab;
    ab.count = std::min(kApplyTerms, n_terms - done);
    ab.accumulate = done > 0;
    for (int k = 0; k < kApplyTerms; ++k) {
      const bool v = k < ab.count;
      ab.x[k] = v ? xmask[done + k] : 0;
      ab.z[k] = v ? zmask[done + k] : 0;
      ab.cr[k] = v ? coef[2 * (done + k)] : 0.0;
      ab.ci[k] = v ? coef[2 * (done + k) + 1] : 0.0;
    }
    hipLaunchKernelGGL(k_apply_paulisum, dim3(grid), dim3(256), 0, s, (const float2*)psi, (float2*)phi, N, ab);
    done += ab.count;
  } while (done < n_terms);
  CQS_HIP(hipGetLastError());
  return CQS_OK;
}

}  // extern "C"
