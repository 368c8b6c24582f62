// Programs decoded into LDS: the interpreter of passes with few tiles.
//
// The interpreter of tile.hpp decodes every op on the scalar unit while the wave waits: kind, targets,
// controls, outer bits, matrix variant.  That is 104 vector, 84 scalar and 30 branch instructions and two
// waits for the scalar cache per one-bit gate on 10 qubits (0.75 us), of which 32 are the
// gate; with one wave per SIMD nothing hides them.  Here a pass decodes its program first, one thread
// per op, into 64-byte records in LDS: what depends on the tile's outer bits is resolved (controls, the
// outer bits of diagonals and phases), small matrices lie in the record, and a class number selects
// the code.  Ops without a class of their own run through the functions of tile.hpp and adjoint.hpp.
// A one-bit gate takes 0.32 us instead of 0.74 on 10 qubits, a diagonal 0.37 instead of 0.68; the gradient of
// a 20-qubit ansatz 1.94 ms instead of 2.24, of a 13-qubit one (4 rows) 2.08 instead of 2.50.
#pragma once

#include "adjoint.hpp"

namespace cqs {

constexpr int kRecWords = 16;    // class, word, slot, -, 4 complex entries, 4 pair words
constexpr int kStageOps = 63;    // ops decoded at a time (4 KB of records with the end mark)
constexpr size_t kStagedBytes = (size_t)(kStageOps + 1) * kRecWords * 4;

// Classes.  The last two bits of REG1 and the ELEM_REG classes are a register bit, the last three of the
// LANE1 classes a lane bit.
enum StagedClass : int {
  kNop = 0,
  kGeneric = 1,    // stays in registers, through the scalar path
  kMix = 2,        // on the LDS tile, through the scalar path
  kEnd = 3,
  kMix1 = 4,       // one-bit op on the LDS tile (word: the bit)
  kGradMix1 = 5,
  kGradOff = 6,    // a gradient op that is off here: its partial sums are zero
  kReg1 = 8,
  kLane1 = 16,
  kGradReg1 = 24,
  kGradLane1 = 40,
  kElem = 48,      // elementwise on lane bits (word: two 16-bit lane masks that select the entry)
  kPairs = 49,     // phases of up to 4 bit pairs (word: their number)
  kGradElem = 50,
  kElemReg = 52,   // elementwise, selected by a lane mask and a register bit
  kGradElemReg = 56,
};

// |d| = 1 as far as FP32 holds it.
__device__ __forceinline__ bool unit_modulus(float2 d) { return fabsf(fmaf(d.x, d.x, d.y * d.y) - 1.f) < 1e-6f; }

// Decodes op i of the pass for the tile at `base`.  TB: thread bits.  In reverse passes the elementwise classes are ops of
// unit modulus on both states, which leave conj(phi) psi as it is; others end a run of diagonal ops (kGeneric).
template <int TB, bool kReverse, class Prog>
__device__ __forceinline__ void decode_op(const Prog& P, int i, uint64_t base, int* r) {
  struct Words {
    int w[16];
  };
  static_assert(sizeof(Words) == sizeof(cqs_op), "the descriptor's words");
  const Words o = *reinterpret_cast<const Words*>(P.ops + i);
  const int4 a = make_int4(o.w[0], o.w[1], o.w[2], o.w[3]), b = make_int4(o.w[4], o.w[5], o.w[6], o.w[7]);
  const int4 c = make_int4(o.w[8], o.w[9], o.w[10], o.w[11]), d = make_int4(o.w[12], o.w[13], o.w[14], o.w[15]);
  const int kind = a.x & 0xff, sel = (a.x >> 8) & 3, k = a.y, mat = a.z;
  const int t0 = b.x, t1 = b.y, t2 = b.z, cl_mask = c.z;
  const uint64_t cm = ((uint64_t)(uint32_t)d.y << 32) | (uint32_t)d.x;
  const uint64_t cv = ((uint64_t)(uint32_t)d.w << 32) | (uint32_t)d.z;
  const bool on = (base & cm) == cv;
  const bool grad = kind == CQS_OP_GRAD_DENSE || kind == CQS_OP_GRAD_DIAG;
  float2 e[4];
  int cls = kGeneric, word = 0, pw[4] = {0, 0, 0, 0};
#pragma unroll
  for (int q = 0; q < 4; ++q) e[q] = make_float2(0.f, 0.f);
  if (!on) {
    cls = grad ? kGradOff : kNop;
  } else if (kind == CQS_OP_DENSE || kind == CQS_OP_GRAD_DENSE) {
    bool reg = t0 >= TB && k <= 3;  // ascending register bits
    if (k > 1) reg = reg && t1 > t0;
    if (k > 2) reg = reg && t2 > t1;
    if (k == 1 && cl_mask == 0 && sel == 0) {
      const int code = c.y;  // t[5]: outer bits that select one of several matrices
      int var = 0;
      for (int q = 0; q < ((code >> 24) & 3); ++q) var |= (int)((base >> ((code >> (7 * q)) & 127)) & 1ull) << q;
#pragma unroll
      for (int q = 0; q < 4; ++q) e[q] = P.mats[mat + 4 * var + q];
      word = t0;
      cls = t0 < kLaneBits ? (grad ? kGradLane1 : kLane1) + t0
            : reg          ? (grad ? kGradReg1 : kReg1) + (t0 - TB)
                           : (grad ? kGradMix1 : kMix1);
    } else {
      cls = reg || (k == 1 && t0 < kLaneBits) ? kGeneric : kMix;
    }
  } else if (kind == CQS_OP_BLOCK) {
    cls = kMix;
  } else if (kind == CQS_OP_SCALE && sel == 0) {
#pragma unroll
    for (int q = 0; q < 4; ++q) e[q] = P.mats[mat];
    cls = kReverse && !unit_modulus(e[0]) ? kGeneric : kElem;
  } else if ((kind == CQS_OP_DIAG || kind == CQS_OP_GRAD_DIAG) && k <= 2 && sel == 0) {
    // entry index bit 0 <- s0, bit 1 <- s1: a tile bit, or -1 for none
    int s0 = t0, s1 = k == 2 ? t1 : -1;
    e[0] = P.mats[mat];
    e[1] = P.mats[mat + 1];
    e[2] = k == 2 ? P.mats[mat + 2] : e[0];
    e[3] = k == 2 ? P.mats[mat + 3] : e[1];
    if (s1 >= kOuter) {
      const bool one = (base >> (s1 - kOuter)) & 1ull;
      e[0] = one ? e[2] : e[0];
      e[1] = one ? e[3] : e[1];
      s1 = -1;
    }
    if (s0 >= kOuter) {
      const bool one = (base >> (s0 - kOuter)) & 1ull;
      e[0] = one ? e[1] : e[0];
      e[1] = one ? e[3] : e[2];
      s0 = s1;
      s1 = -1;
    }
    if (s0 >= TB && s1 < TB) {  // the register bit selects last
      const int s = s0;
      s0 = s1;
      s1 = s;
      const float2 x = e[1];
      e[1] = s0 < 0 ? e[0] : e[2];
      e[2] = x;
    }
    if (s1 < 0) e[2] = e[0], e[3] = e[1];
    word = (s0 >= 0 && s0 < TB ? 1 << s0 : 0) | (s1 >= 0 && s1 < TB ? 1 << (s1 + 16) : 0);
    if (s1 >= 0 && s0 < 0) e[3] = e[2];
    const bool real = e[0].x != 0.f || e[1].x != 0.f || e[2].x != 0.f || e[3].x != 0.f;
    const bool unit = unit_modulus(e[0]) && unit_modulus(e[1]) && unit_modulus(e[2]) && unit_modulus(e[3]);
    if (s0 >= TB || (grad && real) || (kReverse && !grad && !unit))
      cls = kGeneric;
    else
      cls = s1 >= TB ? (grad ? kGradElemReg : kElemReg) + (s1 - TB) : grad ? kGradElem : kElem;
  } else if (kind == CQS_OP_PAIRPHASE && k <= 4 && sel == 0) {
    cls = kPairs;
    word = k;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (q >= k) break;
      e[q] = P.mats[mat + q];
      if (kReverse && !unit_modulus(e[q])) cls = kGeneric;
      int lanes = 0, regs = 0;
      bool both = true;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int x = P.aux[t0 + 2 * q + h];
        if (x >= kOuter)
          both = both && ((base >> (x - kOuter)) & 1ull);
        else if (x < TB)
          lanes |= 1 << x;
        else
          regs |= 1 << (x - TB);
      }
      pw[q] = lanes | (regs << 16) | (both ? 1 << 30 : 0);
    }
  }
  reinterpret_cast<int4*>(r)[0] = make_int4(cls, word, a.w, 0);
  reinterpret_cast<float4*>(r)[1] = make_float4(e[0].x, e[0].y, e[1].x, e[1].y);
  reinterpret_cast<float4*>(r)[2] = make_float4(e[2].x, e[2].y, e[3].x, e[3].y);
  reinterpret_cast<int4*>(r)[3] = make_int4(pw[0], pw[1], pw[2], pw[3]);
}

// Records of the pass's ops from `first` on (up to kStageOps), ended by kEnd.  Every thread takes part.
template <int NT, bool kReverse, class Prog>
__device__ __forceinline__ void decode_program(const Prog& P, int first, uint64_t base, int* recs) {
  static_assert(kStageOps < NT, "one thread per op");
  const int left = P.op_count - first, n = left < kStageOps ? left : kStageOps;
  if ((int)threadIdx.x < n) decode_op<__builtin_ctz(NT), kReverse>(P, first + threadIdx.x, base, recs + threadIdx.x * kRecWords);
  if ((int)threadIdx.x == n) recs[n * kRecWords] = kEnd;
  __syncthreads();
}

__device__ __forceinline__ int rec_word(const int* r, int q) { return __builtin_amdgcn_readfirstlane(r[q]); }
__device__ __forceinline__ float2 rec_entry(const int* r, int q) {
  return make_float2(__int_as_float(rec_word(r, 4 + 2 * q)), __int_as_float(rec_word(r, 5 + 2 * q)));
}
__device__ __forceinline__ Mat2 rec_matrix(const int* r) {
  Mat2 m;
#pragma unroll
  for (int q = 0; q < 4; ++q) m.m[q] = rec_entry(r, q);
  return m;
}
// This lane's entries of an elementwise record: lo (the last selector clear) and hi (set).
__device__ __forceinline__ void rec_lane_entries(const int* r, int lanes0, float2& lo, float2& hi) {
  const bool c = (threadIdx.x & lanes0) != 0;
  const float2 e0 = rec_entry(r, 0), e1 = rec_entry(r, 1), e2 = rec_entry(r, 2), e3 = rec_entry(r, 3);
  lo = c ? e1 : e0;
  hi = c ? e3 : e2;
}

template <int PER, int R>
__device__ __forceinline__ void mul_by_reg_bit(float2 (&v)[PER], float2 lo, float2 hi) {
#pragma unroll
  for (int e = 0; e < PER; ++e) v[e] = cmul(v[e], (e >> R) & 1 ? hi : lo);
}

// An elementwise record (kElem, kElemReg, kPairs) on the elements v.
template <int PER>
__device__ __forceinline__ void staged_elementwise(float2 (&v)[PER], const int* r, int cls) {
  constexpr int NR = __builtin_ctz(PER);
  const int word = rec_word(r, 1);
  if (cls == kPairs) {
    float2 cph = make_float2(1.f, 0.f);
    for (int q = 0; q < word; ++q) {
      const int w = rec_word(r, 12 + q), lanes = w & 0xffff, regs = (w >> 16) & 15;
      if (!(w >> 30 & 1)) continue;
      const float2 f = rec_entry(r, q);
      const bool tc = ((int)threadIdx.x & lanes) == lanes;
      if (regs == 0) {
        const float2 g = cmul(cph, f);
        cph = tc ? g : cph;
        continue;
      }
#pragma unroll
      for (int e = 0; e < PER; ++e)
        if ((e & regs) == regs) {
          const float2 g = cmul(v[e], f);
          v[e] = tc ? g : v[e];
        }
    }
#pragma unroll
    for (int e = 0; e < PER; ++e) v[e] = cmul(v[e], cph);
    return;
  }
  float2 lo, hi;
  rec_lane_entries(r, word & 0xffff, lo, hi);
  if (cls == kElem) {
    const float2 d = (threadIdx.x & (word >> 16)) != 0 ? hi : lo;
#pragma unroll
    for (int e = 0; e < PER; ++e) v[e] = cmul(v[e], d);
    return;
  }
  switch (cls & 3) {
    case 0: if constexpr (NR > 0) mul_by_reg_bit<PER, 0>(v, lo, hi); return;
    case 1: if constexpr (NR > 1) mul_by_reg_bit<PER, 1>(v, lo, hi); return;
    case 2: if constexpr (NR > 2) mul_by_reg_bit<PER, 2>(v, lo, hi); return;
    default: if constexpr (NR > 3) mul_by_reg_bit<PER, 3>(v, lo, hi); return;
  }
}

// A one-bit matrix on register bit (kReg1) or lane bit (kLane1) `cls` of the elements v.
template <int PER, int NT>
__device__ __forceinline__ void staged_dense1(float2 (&v)[PER], const Mat2& M, int cls) {
  constexpr int NR = __builtin_ctz(PER);
  switch (cls) {
    case kReg1 + 0: if constexpr (NR > 0) reg_dense_k<PER, NT, 1, 0, 0, 0, false>(v, M, 0, 0); return;
    case kReg1 + 1: if constexpr (NR > 1) reg_dense_k<PER, NT, 1, 1, 0, 0, false>(v, M, 0, 0); return;
    case kReg1 + 2: if constexpr (NR > 2) reg_dense_k<PER, NT, 1, 2, 0, 0, false>(v, M, 0, 0); return;
    case kReg1 + 3: if constexpr (NR > 3) reg_dense_k<PER, NT, 1, 3, 0, 0, false>(v, M, 0, 0); return;
    case kLane1 + 0: lane_reg_dense_k<PER, NT, 0, false>(v, M, 0, 0); return;
    case kLane1 + 1: lane_reg_dense_k<PER, NT, 1, false>(v, M, 0, 0); return;
    case kLane1 + 2: lane_reg_dense_k<PER, NT, 2, false>(v, M, 0, 0); return;
    case kLane1 + 3: lane_reg_dense_k<PER, NT, 3, false>(v, M, 0, 0); return;
    case kLane1 + 4: lane_reg_dense_k<PER, NT, 4, false>(v, M, 0, 0); return;
    default: lane_reg_dense_k<PER, NT, 5, false>(v, M, 0, 0); return;
  }
}

struct OneBit {  // what tile_dense<1> reads of an op
  int t[1], cl_mask, cl_val;
};

// tile.hpp run_program over the records of the ops from `ops` on.
template <int PER, int NT, class Prog>
__device__ __forceinline__ void run_staged(float2 (&v)[PER], float2* tile, float2* mstage, const Prog& P,
                                           const cqs_op* ops, const int* recs, uint64_t base, bool act) {
  for (int i = 0;; ++i) {
    const int* r = recs + i * kRecWords;
    int cls = rec_word(r, 0);
    if (cls >= kElem) {
      staged_elementwise<PER>(v, r, cls);
    } else if (cls >= kReg1) {
      staged_dense1<PER, NT>(v, rec_matrix(r), cls);
    } else if (cls == kMix || cls == kMix1) {
      regs_to_tile<PER, NT>(v, tile, act);
      do {
        if (cls != kNop) __syncthreads();
        if (cls == kMix1) {
          OneBit op{{rec_word(r, 1)}, 0, 0};
          tile_dense<1, NT>(tile, P.L, op, rec_matrix(r));
        } else if (cls == kMix) {
          run_mixing_op<NT>(tile, mstage, P, scalar_ptr(ops)[i], base);
        }
        r = recs + ++i * kRecWords;
        cls = rec_word(r, 0);
      } while (cls == kMix || cls == kMix1 || cls == kNop);
      --i;
      __syncthreads();
      tile_to_regs<PER, NT>(v, tile, act);
    } else if (cls == kGeneric) {
      sop_t& op = scalar_ptr(ops)[i];
      if (op.kind == CQS_OP_PERMUTE) {
        __syncthreads();  // every thread has read its elements before any is overwritten
        regs_to_tile_permuted<PER, NT>(v, tile, P.L, scalar_ptr(P.aux) + op.t[0], act);
        __syncthreads();
        tile_to_regs<PER, NT>(v, tile, act);
      } else if (op.kind == CQS_OP_DENSE) {
        reg_dense<PER, NT>(v, P, op, base);
      } else if (op.kind == CQS_OP_DIAG) {
        ew_diag<PER, NT>(v, P, op, base);
      } else if (op.kind == CQS_OP_PAIRPHASE) {
        ew_pairs<PER, NT>(v, P, op, base);
      }
    } else if (cls == kEnd) {
      return;
    }
  }
}

// adjoint.hpp's reverse pass over the records of the ops from `ops` on.
template <int PER, int NT, int L, class Prog>
__device__ __forceinline__ void adjoint_staged(float2 (&va)[PER], float2 (&vb)[PER], float2* tA, float2* tB,
                                               float2* mstage, const Prog& P, const cqs_op* ops, const int* recs,
                                               uint64_t base, bool act, double* __restrict__ partial, int64_t stride,
                                               int64_t tile) {
  constexpr int NR = __builtin_ctz(PER);
  for (int i = 0;; ++i) {
    const int* r = recs + i * kRecWords;
    int cls = rec_word(r, 0);
    if (cls >= kElem) {
      // a run of diagonal ops on both states, which leave the products conj(f) x as they are: formed once
      // (gathering the run's phases in FP64 as well was slower: 2.48 against 1.85 ms for the 20-qubit ansatz)
      double w[PER];
      double total = 0.0;
      bool have_w = false;
      do {
        if (cls == kGradElem || cls >= kGradElemReg) {
          if (!have_w) {
#pragma unroll
            for (int e = 0; e < PER; ++e) {
              w[e] = add_overlap<true>(0.0, vb[e], va[e]);
              total += w[e];
            }
            have_w = true;
          }
          const int word = rec_word(r, 1);
          float2 lo, hi;
          rec_lane_entries(r, word & 0xffff, lo, hi);
          double g;
          if (cls == kGradElem) {
            const float d = (threadIdx.x & (word >> 16)) != 0 ? hi.y : lo.y;
            g = -2.0 * (double)d * total;
          } else {
            const int bit = 1 << (cls & 3);
            double s = 0.0;  // elements with the register bit set
#pragma unroll
            for (int e = 0; e < PER; ++e)
              if (e & bit) s += w[e];
            g = -2.0 * fma((double)hi.y, s, (double)lo.y * (total - s));
          }
          write_wave_partial<NT>(act ? g : 0.0, partial, stride, tile, rec_word(r, 2));
        } else {
          staged_elementwise<PER>(va, r, cls);
          staged_elementwise<PER>(vb, r, cls);
        }
        r = recs + ++i * kRecWords;
        cls = rec_word(r, 0);
      } while (cls >= kElem);
      --i;
    } else if (cls >= kGradReg1 && (cls < kGradReg1 + 4 || cls >= kGradLane1)) {
      const Mat2 M = rec_matrix(r);
      double g = 0.0;
      switch (cls) {
        case kGradReg1 + 0: if constexpr (NR > 0) g = grad_reg_dense_k<PER, 1, 0, 0, 0>(va, vb, M); break;
        case kGradReg1 + 1: if constexpr (NR > 1) g = grad_reg_dense_k<PER, 1, 1, 0, 0>(va, vb, M); break;
        case kGradReg1 + 2: if constexpr (NR > 2) g = grad_reg_dense_k<PER, 1, 2, 0, 0>(va, vb, M); break;
        case kGradReg1 + 3: if constexpr (NR > 3) g = grad_reg_dense_k<PER, 1, 3, 0, 0>(va, vb, M); break;
        case kGradLane1 + 0: g = grad_lane1<PER, 0>(va, vb, M); break;
        case kGradLane1 + 1: g = grad_lane1<PER, 1>(va, vb, M); break;
        case kGradLane1 + 2: g = grad_lane1<PER, 2>(va, vb, M); break;
        case kGradLane1 + 3: g = grad_lane1<PER, 3>(va, vb, M); break;
        case kGradLane1 + 4: g = grad_lane1<PER, 4>(va, vb, M); break;
        default: g = grad_lane1<PER, 5>(va, vb, M); break;
      }
      write_wave_partial<NT>(act ? g : 0.0, partial, stride, tile, rec_word(r, 2));
    } else if (cls >= kReg1) {
      const Mat2 M = rec_matrix(r);
      staged_dense1<PER, NT>(va, M, cls);
      staged_dense1<PER, NT>(vb, M, cls);
    } else if (cls == kMix || cls == kMix1 || cls == kGradMix1) {
      regs_to_tile<PER, NT>(va, tA, act);
      regs_to_tile<PER, NT>(vb, tB, act);
      do {
        if (cls != kNop) __syncthreads();
        if (cls == kMix1) {
          OneBit op{{rec_word(r, 1)}, 0, 0};
          const Mat2 M = rec_matrix(r);
          tile_dense<1, NT>(tA, L, op, M);
          tile_dense<1, NT>(tB, L, op, M);
        } else if (cls == kGradMix1) {
          const double g = grad_dense1<NT>(tA, tB, L, rec_word(r, 1), rec_matrix(r));
          write_wave_partial<NT>(g, partial, stride, tile, rec_word(r, 2));
        } else if (cls == kMix) {
          adjoint_mixing_op<NT, L>(tA, tB, mstage, P, scalar_ptr(ops)[i], base, partial, stride, tile);
        }
        r = recs + ++i * kRecWords;
        cls = rec_word(r, 0);
      } while (cls == kMix || cls == kMix1 || cls == kGradMix1 || cls == kNop);
      --i;
      __syncthreads();
      tile_to_regs<PER, NT>(va, tA, act);
      tile_to_regs<PER, NT>(vb, tB, act);
    } else if (cls == kGeneric) {
      adjoint_register_op<PER, NT>(va, vb, P, scalar_ptr(ops)[i], base, act, partial, stride, tile);
    } else if (cls == kGradOff) {
      write_wave_partial<NT>(0.0, partial, stride, tile, rec_word(r, 2));
    } else if (cls == kEnd) {
      return;
    }
  }
}

// pass_tile / adjoint_tile with the program decoded behind the tiles and the matrix stage, kStageOps ops
// at a time.
template <bool kReverse>
struct RunDecoded {
  template <class Prog>
  static __device__ __forceinline__ int* records(const Prog& P, float2* mstage) {
    return reinterpret_cast<int*>(mstage + mstage_words(P.max_k));
  }
  template <int NT, class Prog>
  static __device__ __forceinline__ void begin(const Prog& P, uint64_t base, float2* mstage) {
    decode_program<NT, kReverse>(P, 0, base, records(P, mstage));
  }
  template <int PER, int NT, class Prog>
  static __device__ __forceinline__ void run(float2 (&v)[PER], float2* tile, float2* mstage, const Prog& P,
                                             uint64_t base, bool act) {
    int* recs = records(P, mstage);
    for (int first = 0;;) {
      run_staged<PER, NT>(v, tile, mstage, P, P.ops + first, recs, base, act);
      first += kStageOps;
      if (first >= P.op_count) return;
      __syncthreads();
      decode_program<NT, kReverse>(P, first, base, recs);
    }
  }
};
using RunStaged = RunDecoded<false>;
struct RunStagedAdjoint : RunDecoded<true> {
  template <int PER, int NT, int L, class Prog>
  static __device__ __forceinline__ void run(float2 (&va)[PER], float2 (&vb)[PER], float2* tA, float2* tB,
                                             float2* mstage, const Prog& P, uint64_t base, bool act,
                                             double* __restrict__ partial, int64_t stride, int64_t tile) {
    int* recs = records(P, mstage);
    for (int first = 0;;) {
      adjoint_staged<PER, NT, L>(va, vb, tA, tB, mstage, P, P.ops + first, recs, base, act, partial, stride, tile);
      first += kStageOps;
      if (first >= P.op_count) return;
      __syncthreads();
      decode_program<NT, true>(P, first, base, recs);
    }
  }
};

typedef void (*StagedPassKernel)(float2*, TileProg);
typedef void (*StagedAdjKernel)(float2*, float2*, TileProg, double*, int64_t);
extern const StagedPassKernel kPassStaged[15];
extern const StagedAdjKernel kAdjStaged[15];

// Tile widths with a decoding interpreter: the records start on 16 bytes behind the tile from 6 bits on.
constexpr int kStagedMinL = 6, kStagedMaxL = 12;
constexpr int kStagedAdjMaxL = 11;  // two states of 16 elements per thread spill 400 registers here
constexpr bool staged_adjoint_width(int L) { return L >= kStagedMinL && L <= kStagedAdjMaxL; }
constexpr bool staged_width(int L) { return L >= kStagedMinL && L <= kStagedMaxL; }

// Passes that are decoded first: those of many ops.  Decoding costs a start (0.3-1 us on few tiles, a tenth of a
// pass of 2-4 ops) and 0.1-0.2 us more for each op without a class of its own, and saves 0.2-0.4 us for each op
// with one.  The host does not see the kinds (ops lie on the device), but programs of one-bit gates have long
// passes, and those whose gates fuse into two-bit matrices and MFMA blocks short ones: grid circuits and noisy
// density matrices 1-14 ops.  Scalar / decoded in us: 16 one-bit and diagonal ops 14.0 / 10.2 on 10 qubits, 23.0 /
// 18.1 on 20, 31.3 / 31.0 on 22; 8 blocks and phases 10.9 / 11.4, 19.7 / 20.4, 30.2 / 33.2; 16 of them 19.1 /
// 19.0, 34.2 / 34.5, 52.5 / 56.3.  On more tiles the waves hide more of the scalar decoding: 16 gates 56 / 54 on
// 23 qubits, 368 / 357 on 26, 32 gates 100 / 91 and 689 / 627. The same in reverse passes: 8 gates and gradients
// 12.6 / 9.2 on 10 qubits, 18.0 / 15.3 on 20, 130 / 132 on 24, 16 of them 22.1 / 13.8, 29.2 / 22.2, 226 / 201; 4
// blocks 11.7 / 13.0, 17.4 / 19.5, 145 / 187, 16 blocks, gradients and phases 29.5 / 25.8, 38.8 / 38.5, 335 / 392,
// 32 of them 54.4 / 44.9, 68.5 / 66.2, 617 / 702.
constexpr int kStagedOuterBits = 10, kStagedOps = 16, kStagedManyOps = 32;
inline bool staged_ops(const TileProg& P) {
  return P.op_count >= (P.nouter <= kStagedOuterBits ? kStagedOps : kStagedManyOps);
}
inline bool staged_pass(const TileProg& P) { return staged_width(P.L) && staged_ops(P); }
inline bool staged_adjoint_pass(const TileProg& P) { return staged_adjoint_width(P.L) && staged_ops(P); }

}  // namespace cqs
