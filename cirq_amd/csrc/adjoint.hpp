// Device side of adjoint differentiation, shared by the single-state and batched kernels.
//
// The host supplies the reversed program: every gate U_k becomes U_k^dagger on both tiles, preceded,
// where it has a parameter, by GRAD ops that see psi_k and phi_k and accumulate
//   g_k = 2 Re <phi_k | dU_k | psi_{k-1}> = 2 Re <phi_k | G_k | psi_k>,  G_k = dU_k U_k^dagger
// (Jones & Gacon 2020, arXiv:2009.02823) in FP64, one partial per wave of a tile.  The generator G_k is
// the same at every parameter value for gates exp(i t K), and the two states stay consistent between
// any two ops, so a gate is undone by one op instead of one per state.
//
// GRAD sums are sums of the products conj(phi_i) psi_j weighted by G's entries.  The products are formed and
// summed in FP64, only those whose entry of G is not zero (a uniform test): a rotation about X, Y or Z has two
// real numbers in its generator.  Diagonal ops on both states leave conj(phi_j) psi_j as it is, so a run of them
// forms the products once for all its GRAD ops (specialised and decoded passes).  The reverse passes are bound by
// VALU work and latency: a gradient of 24-node QAOA, 8 rounds (36 ZZ and 24 X rotations each), takes 7.1 ms
// against 8.5 with dU, psi-only and phi-only ops; of the 20-qubit ansatz, 400 rotations, compiled, 1.13 against
// 1.34.
#pragma once

#include "tile.hpp"

namespace cqs {

constexpr int kSelBoth = 0, kSelPsi = 1, kSelPhi = 2;

__device__ __forceinline__ int op_kind(sop_t& op) { return op.kind & 0xff; }
__device__ __forceinline__ int op_sel(sop_t& op) { return (op.kind >> 8) & 3; }

// s + conj(f) x, its real or its imaginary part, in FP64: the products of two FP32 values are exact there.
template <bool kImag>
__device__ __forceinline__ double add_overlap(double s, float2 f, float2 x) {
  const double fr = f.x, fi = f.y, xr = x.x, xi = x.y;
  return kImag ? fma(fr, xi, fma(-fi, xr, s)) : fma(fr, xr, fma(fi, xi, s));
}

// 2 Re sum over pairs (m, n) of one bit of conj(f) M x, for a 2x2 M: the products that M's nonzero
// parts need, summed over this thread's pairs, then weighted.  x(i, bit), f(i, bit): pair i's
// amplitudes.
template <class X, class F, class MPtr>
__device__ __forceinline__ double grad_pairs(int pairs, X x, F f, MPtr M) {
  double g = 0.0;
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const float2 m = ldm(M, 2 * r + c);
      if (m.x != 0.f) {
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < pairs; ++i) s = add_overlap<false>(s, f(i, r), x(i, c));
        g = fma((double)m.x, s, g);
      }
      if (m.y != 0.f) {
        double s = 0.0;
#pragma unroll
        for (int i = 0; i < pairs; ++i) s = add_overlap<true>(s, f(i, r), x(i, c));
        g = fma(-(double)m.y, s, g);
      }
    }
  return 2.0 * g;
}

// This thread's share (its groups) of 2 Re sum conj(phi) G psi over the LDS tiles for a dense G on
// one tile bit.
template <int NT, class MPtr>
__device__ __forceinline__ double grad_dense1(const float2* psi, const float2* phi, int L, int t, MPtr M) {
  const int pt = pad(1 << t);
  const int pairs = ((1 << L) >> 1) / NT;
  double g = 0.0;
  if (pairs == 0) {  // fewer pairs than threads
    if ((int)threadIdx.x < ((1 << L) >> 1)) {
      const int j = pad(insert0((int)threadIdx.x, t));
      g = grad_pairs(1, [&](int, int b) { return psi[j + b * pt]; }, [&](int, int b) { return phi[j + b * pt]; }, M);
    }
    return g;
  }
  constexpr int kStep = 4;  // pairs whose amplitudes are held at a time
#pragma unroll 1
  for (int i0 = 0; i0 < pairs; i0 += kStep) {
    float2 x[kStep][2], f[kStep][2];
#pragma unroll
    for (int i = 0; i < kStep; ++i) {
      const bool on = i0 + i < pairs;
      const int j = pad(insert0((int)threadIdx.x + (i0 + (on ? i : 0)) * NT, t));
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        x[i][b] = on ? psi[j + b * pt] : make_float2(0.f, 0.f);
        f[i][b] = phi[j + b * pt];
      }
    }
    g += grad_pairs(kStep, [&](int i, int b) { return x[i][b]; }, [&](int i, int b) { return f[i][b]; }, M);
  }
  return g;
}

// This thread's share (its groups) of 2 Re sum conj(phi) G psi over the LDS tiles for a dense G
// (k <= 3) on tile bits op.t.
template <int K, int NT, class Op>
__device__ __forceinline__ double grad_dense(const float2* psi, const float2* phi, int L, Op& op, smat_t* M) {
  if constexpr (K == 1) return grad_dense1<NT>(psi, phi, L, op.t[0], M);
  constexpr int D = 1 << K;
  int ts[K];
#pragma unroll
  for (int m = 0; m < K; ++m) ts[m] = op.t[m];
#pragma unroll
  for (int a = 1; a < K; ++a)
#pragma unroll
    for (int b = a; b > 0; --b)
      if (ts[b - 1] > ts[b]) {
        int x = ts[b - 1];
        ts[b - 1] = ts[b];
        ts[b] = x;
      }
  int pat[D];
#pragma unroll
  for (int m = 0; m < D; ++m) {
    int p = 0;
#pragma unroll
    for (int b = 0; b < K; ++b) p |= ((m >> b) & 1) << op.t[b];
    pat[m] = p;
  }
  double acc = 0.0;
  const int G = (1 << L) >> K;
  // one group at a time: with the op's bits as constants the trip count is known, and unrolling it
  // would keep several groups' operands live at once (spills at 128 VGPRs)
#pragma unroll 1
  for (int g = threadIdx.x; g < G; g += NT) {
    int j0 = g;
#pragma unroll
    for (int s = 0; s < K; ++s) j0 = insert0(j0, ts[s]);
    float2 x[D];
#pragma unroll
    for (int c = 0; c < D; ++c) x[c] = psi[pad(j0 + pat[c])];
#pragma unroll
    for (int r = 0; r < D; ++r) {
      float2 y = make_float2(0.f, 0.f);  // (dU x)_r in FP32, as the state itself
#pragma unroll
      for (int c = 0; c < D; ++c) y = cfma(ldm(M, r * D + c), x[c], y);
      const float2 f = phi[pad(j0 + pat[r])];
      acc += (double)f.x * y.x + (double)f.y * y.y;  // Re(conj(f) y), summed in FP64
    }
  }
  return 2.0 * acc;
}

// GRAD ops run on register-resident tiles when their targets are register bits; otherwise the
// tile goes through LDS.  A DENSE or GRAD_DENSE op whose targets are register bits (ascending)
// stays in registers.
template <int PER, int NT>
__device__ __forceinline__ bool adj_register_dense(sop_t& op) {
  constexpr int TB = __builtin_ctz(NT);
  constexpr int NR = __builtin_ctz(PER);
  const int kind = op_kind(op);
  if ((kind != CQS_OP_DENSE && kind != CQS_OP_GRAD_DENSE) || op.k < 1 || op.k > 3) return false;
  if (op.t[0] < (op.k == 1 ? kLaneBits : 0)) return true;
  if (op.k > NR || op.t[0] < TB) return false;
#pragma unroll
  for (int m = 1; m < 3; ++m)
    if (m < op.k && op.t[m] <= op.t[m - 1]) return false;
  return true;
}

template <int PER, int NT>
__device__ __forceinline__ bool adj_mixing(sop_t& op) {
  const int kind = op_kind(op);
  if (kind == CQS_OP_BLOCK) return true;
  return (kind == CQS_OP_DENSE || kind == CQS_OP_GRAD_DENSE) && !adj_register_dense<PER, NT>(op);
}

// 2 Re sum conj(f) G x over this thread's groups of a register-bit dense G (targets R0 < R1 < R2,
// matrix index bit m <-> target m): one bit through grad_pairs; more bits with G x in FP32 and the
// products with conj(f) summed in FP64.
template <int PER, int K, int R0, int R1, int R2, class MPtr>
__device__ __forceinline__ double grad_reg_dense_k(const float2 (&x)[PER], const float2 (&f)[PER], MPtr M) {
  if constexpr (K == 1) {
    auto at = [](int i, int b) { return ((i >> R0) << (R0 + 1)) | (i & ((1 << R0) - 1)) | (b << R0); };
    return grad_pairs(PER / 2, [&](int i, int b) { return x[at(i, b)]; }, [&](int i, int b) { return f[at(i, b)]; }, M);
  }
  constexpr int D = 1 << K;
  constexpr int RS[3] = {R0, R1, R2};
  constexpr int TMASK = (1 << R0) | (K > 1 ? 1 << R1 : 0) | (K > 2 ? 1 << R2 : 0);
  double acc = 0.0;
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    if (e & TMASK) continue;
    int idx[D];
#pragma unroll
    for (int m = 0; m < D; ++m) {
      int v = e;
#pragma unroll
      for (int b = 0; b < K; ++b) v |= ((m >> b) & 1) << RS[b];
      idx[m] = v;
    }
#pragma unroll
    for (int r = 0; r < D; ++r) {
      float2 y = make_float2(0.f, 0.f);  // (dU x)_r in FP32, as the state itself
#pragma unroll
      for (int c = 0; c < D; ++c) y = cfma(ldm(M, r * D + c), x[idx[c]], y);
      acc += (double)f[idx[r]].x * y.x + (double)f[idx[r]].y * y.y;  // summed in FP64
    }
  }
  return 2.0 * acc;
}

// 2 Re sum conj(f) G x over this thread's elements for a dense G on lane bit T: every lane weights its
// own products and those with its partner's x by its row of G.
template <int PER, int T, class MPtr>
__device__ __forceinline__ double grad_lane1(const float2 (&x)[PER], const float2 (&f)[PER], MPtr M) {
  const float2 m00 = ldm(M, 0), m01 = ldm(M, 1), m10 = ldm(M, 2), m11 = ldm(M, 3);
  const bool hi = (threadIdx.x >> T) & 1;
  const float2 d = hi ? m11 : m00, o = hi ? m10 : m01;
  double g = 0.0;
  if (m00.x != 0.f || m11.x != 0.f) {
    double s = 0.0;
#pragma unroll
    for (int e = 0; e < PER; ++e) s = add_overlap<false>(s, f[e], x[e]);
    g = fma((double)d.x, s, g);
  }
  if (m00.y != 0.f || m11.y != 0.f) {
    double s = 0.0;
#pragma unroll
    for (int e = 0; e < PER; ++e) s = add_overlap<true>(s, f[e], x[e]);
    g = fma(-(double)d.y, s, g);
  }
  if (m01.x != 0.f || m10.x != 0.f) {
    double s = 0.0;
#pragma unroll
    for (int e = 0; e < PER; ++e)
      s = add_overlap<false>(s, f[e], make_float2(lane_xor<T>(x[e].x), lane_xor<T>(x[e].y)));
    g = fma((double)o.x, s, g);
  }
  if (m01.y != 0.f || m10.y != 0.f) {
    double s = 0.0;
#pragma unroll
    for (int e = 0; e < PER; ++e)
      s = add_overlap<true>(s, f[e], make_float2(lane_xor<T>(x[e].x), lane_xor<T>(x[e].y)));
    g = fma(-(double)o.y, s, g);
  }
  return 2.0 * g;
}

template <int PER, int NT, class Prog>
__device__ __forceinline__ double grad_reg_dense(const float2 (&x)[PER], const float2 (&f)[PER], const Prog& P,
                                                 sop_t& op) {
  constexpr int TB = __builtin_ctz(NT);
  constexpr int NR = __builtin_ctz(PER);
  smat_t* M = scalar_ptr(P.mats) + op.mat;
  if (op.k == 1 && op.t[0] < kLaneBits) {
    switch (op.t[0]) {
      case 0: return grad_lane1<PER, 0>(x, f, M);
      case 1: return grad_lane1<PER, 1>(x, f, M);
      case 2: return grad_lane1<PER, 2>(x, f, M);
      case 3: return grad_lane1<PER, 3>(x, f, M);
      case 4: return grad_lane1<PER, 4>(x, f, M);
      default: return grad_lane1<PER, 5>(x, f, M);
    }
  }
  const int r0 = op.t[0] - TB, r1 = op.t[1] - TB, r2 = op.t[2] - TB;
  const int code = op.k == 1 ? r0 : (op.k == 2 ? 16 + r0 * 4 + r1 : 32 + r0 * 16 + r1 * 4 + r2);
#define CQS_G1(A) \
  case A: if constexpr (NR > A) return grad_reg_dense_k<PER, 1, A, 0, 0>(x, f, M); return 0.0;
#define CQS_G2(A, B) \
  case 16 + A * 4 + B: if constexpr (NR > B) return grad_reg_dense_k<PER, 2, A, B, 0>(x, f, M); return 0.0;
#define CQS_G3(A, B, C) \
  case 32 + A * 16 + B * 4 + C: if constexpr (NR > C) return grad_reg_dense_k<PER, 3, A, B, C>(x, f, M); return 0.0;
  switch (code) {
    CQS_G1(0) CQS_G1(1) CQS_G1(2) CQS_G1(3)
    CQS_G2(0, 1) CQS_G2(0, 2) CQS_G2(0, 3) CQS_G2(1, 2) CQS_G2(1, 3) CQS_G2(2, 3)
    CQS_G3(0, 1, 2) CQS_G3(0, 1, 3) CQS_G3(0, 2, 3) CQS_G3(1, 2, 3)
    default: return 0.0;
  }
#undef CQS_G1
#undef CQS_G2
#undef CQS_G3
}

// Diagonal gradients weight the products w_e = Im conj(f_e) x_e of this thread's elements (x: psi, f: phi).
// Diagonal ops of unit modulus on both states leave the products as they are, so specialised passes form them once for a
// run of such ops.  They are plain arrays of the calling kernel: as members of an object with flags for what was formed
// they went to scratch memory (208 bytes per lane; reverse passes of the 20-qubit ansatz 0.85 ms against 0.52).
template <int PER>
__device__ __forceinline__ void diag_products(double (&w)[PER], const float2 (&x)[PER], const float2 (&f)[PER]) {
#pragma unroll
  for (int e = 0; e < PER; ++e) w[e] = add_overlap<true>(0.0, f[e], x[e]);
}

// 2 Re sum conj(f_e) d(e) x_e for a diagonal d and w(e) the products above.  A generator's entries are imaginary: only
// w is needed; a nonzero real part (a uniform test for tables of up to 4 entries) adds its products.
template <int PER, int NT, class W, class Prog, class Op>
__device__ __forceinline__ double grad_diag(W w, const float2 (&x)[PER], const float2 (&f)[PER], const Prog& P, Op& op,
                                            uint64_t base) {
  const DiagTable<PER, NT, Prog> D(P, op, base);
  double acc = 0.0;
  if (!D.any_reg) {
    const float2 d = D.small ? D.pick(D.fixed) : D.Dg[D.fixed];
#pragma unroll
    for (int e = 0; e < PER; ++e) acc += w(e);
    acc *= -(double)d.y;
  } else if (D.small) {
#pragma unroll
    for (int e = 0; e < PER; ++e) acc = fma(-(double)D.pick(D.index(e)).y, w(e), acc);
  } else {
#pragma unroll
    for (int e = 0; e < PER; ++e) acc = fma(-(double)D.Dg[D.index(e)].y, w(e), acc);
  }
  if (!D.small || D.d0.x != 0.f || D.d1.x != 0.f || D.d2.x != 0.f || D.d3.x != 0.f) {
#pragma unroll
    for (int e = 0; e < PER; ++e) acc = fma((double)D.at(e).x, add_overlap<false>(0.0, f[e], x[e]), acc);
  }
  return 2.0 * acc;
}

// Phases that all of a thread's elements share (no register bit among an op's bits), gathered over a run in FP64 and
// multiplied into both states once; phases that differ between elements are multiplied op by op.
template <int PER, int NT, class Prog, class Op>
__device__ __forceinline__ void gather_diag(double2& ph, const Prog& P, Op& op, uint64_t base) {
  const DiagTable<PER, NT, Prog> D(P, op, base);
  ph = cmul(ph, D.small ? D.pick(D.fixed) : D.Dg[D.fixed]);
}
template <int PER>
__device__ __forceinline__ void apply_phase(float2 (&x)[PER], float2 (&f)[PER], double2 ph) {
  const float2 p = make_float2((float)ph.x, (float)ph.y);
#pragma unroll
  for (int e = 0; e < PER; ++e) {
    x[e] = cmul(x[e], p);
    f[e] = cmul(f[e], p);
  }
}

// Every wave writes its own partial of a GRAD op: partial[slot * stride + tile * NW + wave] (a
// shuffle reduction inside the wave, no workgroup barrier; the host sums the NW entries per tile).
template <int NT>
__device__ __forceinline__ void write_wave_partial(double g, double* __restrict__ partial, int64_t stride,
                                                   int64_t tile, int slot) {
  g = wave_sum(g);
  if ((threadIdx.x & 63) == 0)
    partial[(int64_t)slot * stride + tile * (NT / 64) + (threadIdx.x >> 6)] = g;
}

// Waves per workgroup of the adjoint kernels at tile width L (the factor between tiles and
// per-slot partial entries).
__host__ __device__ constexpr int adjoint_waves(int L) { return (L <= 12 ? 256 : (1 << L) / 16) / 64; }

// One op of a register phase on this thread's elements of both states.
template <int PER, int NT, class Prog>
__device__ __forceinline__ void adjoint_register_op(float2 (&va)[PER], float2 (&vb)[PER], const Prog& P, sop_t& op,
                                                    uint64_t base, bool act, double* __restrict__ partial,
                                                    int64_t stride, int64_t tile) {
  const int kind = op_kind(op), sel = op_sel(op);
  const bool ok = outer_controls_ok(op, base);
  if (kind == CQS_OP_GRAD_DIAG) {
    double g = 0.0;
    if (ok && act)
      g = grad_diag<PER, NT>([&](int e) { return add_overlap<true>(0.0, vb[e], va[e]); }, va, vb, P, op, base);
    write_wave_partial<NT>(g, partial, stride, tile, op.slot);
    return;
  }
  if (kind == CQS_OP_GRAD_DENSE) {
    double g = 0.0;
    if (ok) g = grad_reg_dense<PER, NT>(va, vb, P, op);  // exchanges lanes: every lane takes part
    if (!act) g = 0.0;
    write_wave_partial<NT>(g, partial, stride, tile, op.slot);
    return;
  }
  if (!ok) return;
  if (kind == CQS_OP_DENSE) {
    if (sel != kSelPhi) reg_dense<PER, NT>(va, P, op, base);
    if (sel != kSelPsi) reg_dense<PER, NT>(vb, P, op, base);
  } else if (kind == CQS_OP_DIAG) {
    if (sel != kSelPhi) ew_diag<PER, NT>(va, P, op, base);
    if (sel != kSelPsi) ew_diag<PER, NT>(vb, P, op, base);
  } else if (kind == CQS_OP_PAIRPHASE) {
    if (sel != kSelPhi) ew_pairs<PER, NT>(va, P, op, base);
    if (sel != kSelPsi) ew_pairs<PER, NT>(vb, P, op, base);
  } else if (kind == CQS_OP_SCALE) {
    if (sel != kSelPhi) ew_scale<PER>(va, P, op);
    if (sel != kSelPsi) ew_scale<PER>(vb, P, op);
  }
}

// One op of an LDS phase on both LDS tiles.  The caller fences before.
template <int NT, int L, class Prog>
__device__ __forceinline__ void adjoint_mixing_op(float2* tA, float2* tB, float2* mstage, const Prog& P, sop_t& op,
                                                  uint64_t base, double* __restrict__ partial, int64_t stride,
                                                  int64_t tile) {
  const int kind = op_kind(op), sel = op_sel(op);
  const bool ok = outer_controls_ok(op, base);
  if (kind == CQS_OP_GRAD_DENSE) {
    double g = 0.0;
    if (ok) {
      smat_t* M = scalar_ptr(P.mats) + op.mat;
      if (op.k == 1)
        g = grad_dense<1, NT>(tA, tB, L, op, M);
      else if (op.k == 2)
        g = grad_dense<2, NT>(tA, tB, L, op, M);
      else if (op.k == 3)
        g = grad_dense<3, NT>(tA, tB, L, op, M);
    }
    write_wave_partial<NT>(g, partial, stride, tile, op.slot);
    return;
  }
  if (!ok) return;
  if (sel != kSelPhi) run_mixing_op<NT>(tA, mstage, P, op, base);
  if (sel == kSelBoth) __syncthreads();  // the matrix stage is shared by both tiles
  if (sel != kSelPsi) run_mixing_op<NT>(tB, mstage, P, op, base);
}

struct RunAdjoint {  // the interpreter below
  template <int PER, int NT, int L, class Prog>
  static __device__ __forceinline__ void run(float2 (&va)[PER], float2 (&vb)[PER], float2* tA, float2* tB,
                                             float2* mstage, const Prog& P, uint64_t base, bool act,
                                             double* __restrict__ partial, int64_t stride, int64_t tile);
  template <int NT, class Prog>
  static __device__ __forceinline__ void begin(const Prog& P, uint64_t, float2*) {
    warm_program<NT>(P);
  }
};

// One workgroup's share of a reverse-sweep pass.  psi and phi stay in registers (this thread's
// elements, natural layout) through runs of elementwise ops, register-bit dense ops and GRAD ops on
// register bits; ops that mix elements of different threads (other dense ops, MFMA blocks, GRAD
// ops on thread bits) run on the two LDS tiles between barriers.  GRAD ops write one FP64 partial
// per wave.  `stride` is the per-slot partial stride (tiles x waves).
template <int L, class Run = RunAdjoint, class Prog>
__device__ __forceinline__ void adjoint_tile(float2* __restrict__ psi, float2* __restrict__ phi, const Prog& P,
                                             const int32_t* lpos, uint64_t base, double* __restrict__ partial,
                                             int64_t stride, int64_t tile, float2* lds) {
  constexpr int NT = TileShape<L>::NT, PER = TileShape<L>::PER;
  float2* tA = lds;
  float2* tB = lds + tile_words(L);
  float2* mstage = lds + 2 * tile_words(L);
  const bool act = L >= 8 || (int)threadIdx.x < (1 << L);
  Run::template begin<NT>(P, base, mstage);
  float2 va[PER], vb[PER];
  {  // offsets are recomputed for the store, so they are not live across the program
    uint64_t off_lo, off_hi[PER];
    tile_offsets<L>(lpos, off_lo, off_hi);
    if (act) {
#pragma unroll
      for (int e = 0; e < PER; ++e) {
        va[e] = psi[base + off_lo + off_hi[e]];
        vb[e] = phi[base + off_lo + off_hi[e]];
      }
    } else {
#pragma unroll
      for (int e = 0; e < PER; ++e) va[e] = vb[e] = make_float2(0.f, 0.f);
    }
  }
  Run::template run<PER, NT, L>(va, vb, tA, tB, mstage, P, base, act, partial, stride, tile);
  uint64_t off_lo, off_hi[PER];
  tile_offsets<L>(lpos, off_lo, off_hi);
  if (act) {
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      psi[base + off_lo + off_hi[e]] = va[e];
      phi[base + off_lo + off_hi[e]] = vb[e];
    }
  }
}

template <int PER, int NT, int L, class Prog>
__device__ __forceinline__ void RunAdjoint::run(float2 (&va)[PER], float2 (&vb)[PER], float2* tA, float2* tB,
                                                float2* mstage, const Prog& P, uint64_t base, bool act,
                                                double* __restrict__ partial, int64_t stride, int64_t tile) {
  int i = 0;
  for (;;) {
    // register phase
    for (; i < P.op_count && !adj_mixing<PER, NT>(scalar_ptr(P.ops)[i]); ++i)
      adjoint_register_op<PER, NT>(va, vb, P, scalar_ptr(P.ops)[i], base, act, partial, stride, tile);
    if (i >= P.op_count) break;
    // LDS phase: both tiles out of registers, then every consecutive op that mixes threads
    regs_to_tile<PER, NT>(va, tA, act);
    regs_to_tile<PER, NT>(vb, tB, act);
    for (; i < P.op_count && adj_mixing<PER, NT>(scalar_ptr(P.ops)[i]); ++i) {
      sop_t& op = scalar_ptr(P.ops)[i];
      __syncthreads();
      adjoint_mixing_op<NT, L>(tA, tB, mstage, P, op, base, partial, stride, tile);
    }
    __syncthreads();
    tile_to_regs<PER, NT>(va, tA, act);
    tile_to_regs<PER, NT>(vb, tB, act);  // each thread reads back only its own slots: no barrier until the next mix
  }
}

}  // namespace cqs
