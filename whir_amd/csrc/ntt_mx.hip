// Reed-Solomon expansion on the matrix cores (CDNA4 int8 MFMA).
//
// The transforms of ntt.hip again (same layout, same values), for cosets of 2^4 .. 2^10
// elements (one pass) and 2^11 .. 2^20 (two passes, 2^12 also one), with the DFTs as integer
// matrix products.  A Goldilocks element is eight signed base-256 digits, x = sum_b s_b 2^(8b),
// -128 <= s_b < 128, and multiplying by a constant w is linear in the digits:
//     w x = sum_b s_b (w 2^(8b) mod p),
// with the constants' own eight digits as the rows of an int8 matrix.  A whole small DFT
// is then one product of a constant digit matrix (8 digits per output by 8 digits per
// input) with the digits of many columns, exact in the int32 accumulators.  Lane l of a
// v_mfma_i32_16x16x64_i8 holds 16 digits, that is two whole elements, of column l % 16 and
// gets four rows of that column back; the matrix's rows are ordered so that two tiles give
// a lane all eight digits of one output, so elements never cross lanes:
//     sum_k c_k 2^(8k) with 0 <= c_k < 2^23 -> two 48-bit halves -> one 64-bit number.
// Digits come out of a number without a carry chain: the bytes of z = x + K0 with
// K0 = 128 (1 + 2^8 + ... + 2^56), each with its top bit flipped, are the digits of x.
// "Biased" below means that K0 has been added; a multiplication by a twiddle factor adds
// it for nothing (it is the addend of the partial products).
//
// What bounds it.  The radix-8 butterflies of ntt.hip spend 219-251 VALU instructions per
// element of a 2^10-point pass, nearly half of them half-rate 64-bit ones.  Here a 16-point
// DFT costs 12 (digits, recombination) and a twiddle 19, and the matrix cores, idle until
// now, take the additions: 71 VALU instructions per element for a 2^8-point pass 2, 98 for
// a 2^10-point one.  Measured on MI355X, 16 messages, two passes, before -> after:
//     Fp  2^20 -> 2^22: 603 + 432 -> 359 + 312 us    Fp  2^18 -> 2^22: 548 + 366 -> 297 + 253 us
//     Fp2 2^16 -> 2^21: 393 + 289 -> 282 + 246 us    Fp3 2^18 -> 2^21: 834 + 619 -> 446 + 418 us (in groups)
//     Fp2 2^12 -> 2^20: 284 -> 210 us                Fp3 2^14 -> 2^17: 79 -> 54 us
//     one pass, Fp2 2^8 -> 2^19: 98 -> 60 us         Fp3 2^10 -> 2^19: 264 -> 104 us
//     small, Fp 2^10 -> 2^11: 15.5 -> 7.2 us         Fp2 2^12 -> 2^13: 21.2 -> 12.9 us
// Pass 2 of 2^8 and 2^9 points moves 1.07 GB in 245-253 us, 4.3 TB/s where a large copy
// reaches 4.7: it is near the memory's rate, and its waves wait 52-64% of their time.  Pass 1
// waits 45-50% and issues 0.87-1.0 VALU instructions per SIMD and four cycles (half of them
// half-rate 64-bit ones, whose mix allows about 1.3) with the matrix cores busy 10-27% of the
// time: VALU issue and the latency of four waves per SIMD together.  128 registers a lane, 64
// of them the matrix, allow no more waves; the 2^10-point pass 2 is between the two (0.68,
// waits 51%).  Measured slower: 12 waves per CU with the next tile's loads in flight in
// registers (pass 2 234 -> 317 us, the late tiles leave waves idle), one block of 16 waves
// per CU, the matrices of a whole 32-point DFT in registers (8 waves per CU, 1.2x slower).
#include "common.h"
#include "gl.h"
#include "ntt_mx.h"

#include <algorithm>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

namespace whir {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr uint32_t K0W = 0x80808080u;  // both halves of K0 = 128 (1 + 2^8 + ... + 2^56)
constexpr int MAT16 = 1026;            // where the 16-point matrix starts, after the eight-point ones
constexpr int TILE = 8192;             // words of one LDS tile (64 KiB)

#define DEV __device__ __forceinline__
// Keeps the scheduler from interleaving the eight-point transforms of a step, which would
// need more registers than four waves per SIMD leave.
#define SCHED_FENCE() __builtin_amdgcn_sched_barrier(0)

DEV uint64_t mk64(uint32_t lo, uint32_t hi) { return ((uint64_t)hi << 32) | lo; }

// Constants the compiler must not see through: a multiply-add by them stays one
// instruction instead of becoming a chain of shifts, adds and carries.
struct Opaque { uint32_t two16; int32_t m1; };
DEV Opaque opaque() {
  Opaque k;
  asm("s_mov_b32 %0, 0x10000" : "=s"(k.two16));
  asm("s_mov_b32 %0, -1" : "=s"(k.m1));
  return k;
}

// [r0, r1] + c (2^32 - 1) for a carry c out of 2^64
DEV uint64_t fix_carry(uint32_t r0, uint32_t r1, uint32_t c) {
  asm("" : "+v"(c));
  uint64_t p = mk64(r0, r1);
  asm("" : "+v"(p));
  return (uint64_t)c * 0xFFFFFFFFu + p;
}
// [r0, r1] + r2 (2^32 - 1) for r2 in -1 .. 1
DEV uint64_t fix_signed(uint32_t r0, uint32_t r1, int32_t r2, const Opaque& k) {
  uint64_t p = mk64(r0, r1 + (uint32_t)r2);
  asm("" : "+v"(p));
  return (uint64_t)((int64_t)r2 * (int64_t)k.m1 + (int64_t)p);
}

// r mod p for r < 2^64
DEV uint64_t canon(uint64_t r) {
  uint32_t c;
  const uint32_t x0 = __builtin_addc((uint32_t)r, 0xFFFFFFFFu, 0u, &c);
  const uint32_t x1 = __builtin_addc((uint32_t)(r >> 32), 0u, c, &c);
  return c ? mk64(x0, x1) : r;
}

// l0 + 2^32 l1 + 2^64 (hl + 2^32 hh) mod p as some 64-bit number:
// 2^64 = 2^32 - 1 and 2^96 = -1, and of a borrow and a carry the difference counts
DEV uint64_t reduce(uint32_t l0, uint32_t l1, uint32_t hl, uint32_t hh, const Opaque& k) {
  uint32_t b, c;
  uint32_t r0 = __builtin_subc(l0, hh, 0u, &b);
  uint32_t r1 = __builtin_subc(l1, 0u, b, &b);
  uint32_t r2 = __builtin_subc(0u, 0u, b, &b);
  const uint64_t q = (uint64_t)hl * 0xFFFFFFFFu;
  r0 = __builtin_addc(r0, (uint32_t)q, 0u, &c);
  r1 = __builtin_addc(r1, (uint32_t)(q >> 32), c, &c);
  r2 = __builtin_addc(r2, 0u, c, &c);
  return fix_signed(r0, r1, (int32_t)r2, k);
}

// a w mod p, below p; BIASED: a w + K0 mod p as some 64-bit number
template <bool BIASED>
DEV uint64_t mulw(uint64_t a, uint64_t w, const Opaque& k) {
  const uint32_t a0 = (uint32_t)a, a1 = (uint32_t)(a >> 32), b0 = (uint32_t)w, b1 = (uint32_t)(w >> 32);
  constexpr uint32_t kb = BIASED ? K0W : 0;
  const uint64_t p00 = (uint64_t)a0 * b0 + kb;
  const uint64_t mid = (uint64_t)a0 * b1 + kb + (p00 >> 32);
  const uint64_t mid2 = (uint64_t)a1 * b0 + (uint32_t)mid;
  const uint64_t hi = (uint64_t)a1 * b1 + (mid >> 32) + (mid2 >> 32);
  const uint64_t r = reduce((uint32_t)p00, (uint32_t)mid2, (uint32_t)hi, (uint32_t)(hi >> 32), k);
  return BIASED ? r : canon(r);
}

// a + b, a - b for any 64-bit a and canonical b
DEV uint64_t addl(uint64_t a, uint64_t b) {
  uint32_t c;
  const uint32_t lo = __builtin_addc((uint32_t)a, (uint32_t)b, 0u, &c);
  const uint32_t hi = __builtin_addc((uint32_t)(a >> 32), (uint32_t)(b >> 32), c, &c);
  return fix_carry(lo, hi, c);
}
DEV uint64_t subl(uint64_t a, uint64_t b) {
  uint32_t c, k;
  uint32_t lo = __builtin_subc((uint32_t)a, (uint32_t)b, 0u, &c);
  uint32_t hi = __builtin_subc((uint32_t)(a >> 32), (uint32_t)(b >> 32), c, &c);
  lo = __builtin_subc(lo, 0u - c, 0u, &k);
  return mk64(lo, hi - k);
}
DEV uint64_t biased(uint64_t x) { return addl(mk64(K0W, K0W), x); }  // x + K0 for canonical x
// x 2^48 for any 64-bit x, below p
DEV uint64_t rot48(uint64_t x, const Opaque& k) {
  const uint32_t x0 = (uint32_t)x, x1 = (uint32_t)(x >> 32);
  return canon(reduce(0, x0 << 16, __builtin_amdgcn_alignbit(x1, x0, 16), x1 >> 16, k));
}

DEV uint64_t recombine(v4i L, v4i H, const Opaque& k) {
  const uint32_t e = (uint32_t)L[0] + ((uint32_t)L[1] << 8), f = (uint32_t)L[2] + ((uint32_t)L[3] << 8);
  const uint32_t g = (uint32_t)H[0] + ((uint32_t)H[1] << 8), h = (uint32_t)H[2] + ((uint32_t)H[3] << 8);
  const uint64_t U = (uint64_t)f * k.two16 + e, V = (uint64_t)h * k.two16 + g;
  const uint64_t T = (uint64_t)(uint32_t)(V >> 32) * 0xFFFFFFFFu + U;
  uint32_t c;
  const uint32_t hi = __builtin_addc((uint32_t)(T >> 32), (uint32_t)V, 0u, &c);
  return fix_carry((uint32_t)T, hi, c);
}

// A radix-R step (R = 8, 16, 32) of 16 columns by one wave.  Lane (n, g), n = lane % 16 and
// g = lane / 16, loads R/4 elements of column n, element i of index g + in_u(i), and ends
// with R/4 outputs, output i of index out_g g + out_u(i).
//   FULL (R = 16): the 16-point transform is one product with the 128 x 128 digit matrix;
//     inputs are biased, any 64-bit numbers.
//   else: radix R/8 butterflies on the lane's own elements, then R/8 eight-point transforms
//     (64 x 64 digit matrices) that have the butterflies' twiddle factors in their entries;
//     inputs are canonical and not biased.
template <int LR, bool FULL>
struct Step {
  static constexpr int N = 1 << (LR - 2);
  static constexpr int out_g = FULL || LR == 3 ? 1 : LR == 4 ? 2 : 4;
  static DEV constexpr int in_u(int i) { return FULL || LR == 3 ? 4 * i : 4 * (i & 1) + (i >> 1) * 8; }
  // which of its elements index j is, for the lane group j % 4 that loads it
  static DEV constexpr int in_i(int j) { return FULL ? j >> 2 : (j >> 2 & 1) + (j >> 3) * 2; }
  static DEV constexpr int out_u(int i) { return FULL || LR == 3 ? 4 * i : LR == 4 ? 8 * (i >> 1) + (i & 1) : 16 * (i >> 2) + (i & 3); }
};

struct Mats {
  v4i a[16];  // FULL: [tile 8][k step 2]; else [residue 4][tile 4]
  v4i bL, bH; // the accumulators' initial values, digits 0-3 and 4-7
  Opaque k;
};
DEV void load_mats(Mats& A, const v4i* mat) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < 16; i++) A.a[i] = mat[i * 64 + lane];
  A.bL = mat[1024];
  A.bH = mat[1025];
  A.k = opaque();
}

DEV v4i digits2(uint64_t z0, uint64_t z1) {
  return v4i{(int)((uint32_t)z0 ^ K0W), (int)((uint32_t)(z0 >> 32) ^ K0W), (int)((uint32_t)z1 ^ K0W),
             (int)((uint32_t)(z1 >> 32) ^ K0W)};
}
#define MX_MFMA(a, b, c) __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0)

template <class F>
DEV void dft8(const Mats& A, int r, uint64_t z0, uint64_t z1, int i0, int i1, F emit) {
  const v4i b = digits2(z0, z1);
  const v4i L0 = MX_MFMA(A.a[4 * r], b, A.bL), H0 = MX_MFMA(A.a[4 * r + 1], b, A.bH);
  const v4i L1 = MX_MFMA(A.a[4 * r + 2], b, A.bL), H1 = MX_MFMA(A.a[4 * r + 3], b, A.bH);
  emit(i0, recombine(L0, H0, A.k));
  emit(i1, recombine(L1, H1, A.k));
}

template <int LR, bool FULL, class F>
DEV void dft(const Mats& A, const uint64_t (&x)[1 << (LR - 2)], F emit) {
  if constexpr (FULL) {
    const v4i b0 = digits2(x[0], x[1]), b1 = digits2(x[2], x[3]);
#pragma unroll
    for (int u = 0; u < 4; u += 2) {
      v4i L0 = MX_MFMA(A.a[4 * u], b0, A.bL), H0 = MX_MFMA(A.a[4 * u + 2], b0, A.bH);
      v4i L1 = MX_MFMA(A.a[4 * u + 4], b0, A.bL), H1 = MX_MFMA(A.a[4 * u + 6], b0, A.bH);
      L0 = MX_MFMA(A.a[4 * u + 1], b1, L0);
      H0 = MX_MFMA(A.a[4 * u + 3], b1, H0);
      L1 = MX_MFMA(A.a[4 * u + 5], b1, L1);
      H1 = MX_MFMA(A.a[4 * u + 7], b1, H1);
      emit(u, recombine(L0, H0, A.k));
      emit(u + 1, recombine(L1, H1, A.k));
    }
  } else if constexpr (LR == 3) {
    dft8(A, 0, biased(x[0]), biased(x[1]), 0, 1, emit);
  } else if constexpr (LR == 4) {
    const uint64_t b0 = biased(x[0]), b1 = biased(x[1]);
    dft8(A, 0, addl(b0, x[2]), addl(b1, x[3]), 0, 2, emit);
    dft8(A, 2, subl(b0, x[2]), subl(b1, x[3]), 1, 3, emit);
  } else {
    uint64_t y[4][2];
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const uint64_t b = biased(x[e]);
      const uint64_t t0 = addl(b, x[4 + e]), t1 = subl(b, x[4 + e]);
      const uint64_t t2 = canon(addl(x[2 + e], x[6 + e])), t3 = rot48(subl(x[2 + e], x[6 + e]), A.k);
      y[0][e] = addl(t0, t2);
      y[2][e] = subl(t0, t2);
      y[1][e] = addl(t1, t3);
      y[3][e] = subl(t1, t3);
    }
#pragma unroll
    for (int b = 0; b < 4; b++) {
      dft8(A, b, y[b][0], y[b][1], b, 4 + b, emit);
      SCHED_FENCE();
    }
  }
}

DEV uint64_t ld(const uint64_t* p, uint32_t voff) { return *(const uint64_t*)((const char*)p + voff); }
DEV void st(uint64_t* p, uint32_t voff, uint64_t v) { *(uint64_t*)((char*)p + voff) = v; }

DEV bool xcd_block(uint32_t nlogical, uint32_t& logical) {
  constexpr uint32_t NX = 8;
  const uint32_t per = (nlogical + NX - 1) / NX;
  logical = (blockIdx.x % NX) * per + blockIdx.x / NX;
  return logical < nlogical;
}

template <int D>
DEV const uint64_t* msg_ptr(const RsArgs& a, size_t j) {
  j += a.j0;
  return a.msg_tab ? a.msg_tab[j / a.mpi] + (j % a.mpi) * a.msg_stride * D : a.msgs + j * a.msg_stride * D;
}
template <int D>
DEV uint64_t* out_ptr(const RsArgs& a, size_t j) {
  j += a.j0;
  return a.out_tab ? a.out_tab[j / a.mpi] + (j % a.mpi) * a.N * D : a.out + j * a.N * D;
}

// Word w of the masked message: message || mask || zeros.
template <int D>
DEV uint64_t word_at(const uint64_t* msg, size_t Lw, const uint64_t* mask, size_t mw, size_t w) {
  if (w < Lw) return msg[w];
  return w - Lw < mw ? mask[w - Lw] : 0;
}

// Threads of a block of pass 2.  Radix 32 over an Fp3 tile of 6144 words is 12 column groups:
// 768 threads take one each (512 would idle half of a second round: pass 2 of 2^20 rows of
// 2^10 points 776 -> 560 us, of 2^9 points 535 -> 508 us).
template <int D, int LA>
constexpr int row_threads() { return D == 3 && LA == 5 ? 768 : 512; }

// Rows of length S that a block of pass 2 transforms.
template <int D>
constexpr int row_block(int S) { return (D == 1 ? 8 : D == 2 ? 4 : 2) * (1024 / S); }

// Most sequences of length S that a block of the single pass transforms.
template <int D>
constexpr int sequences(int S) { return row_block<D>(S); }

// ------------------------------------------------------------------ pass 1: columns
template <int D, int LA, int LB, bool NEXT16>
__global__ __launch_bounds__(512, 4) void k_mx_pass1(RsArgs a, const v4i* mat, const uint64_t* tw, const uint64_t* row,
                                                        const uint64_t* post, uint64_t* Y, int logC1, int logBY, int jn) {
  constexpr int RA = 1 << LA, RB = 1 << LB, S = RA * RB, WB = TILE / S;
  constexpr bool F16 = LA == 4 && LB == 4;
  using SA = Step<LA, F16>;
  using SB = Step<LB, F16>;
  constexpr int NA = RA / 4, NB = RB / 4, KS = RB * WB + 8;
  __shared__ uint64_t s[RA * KS];
  __shared__ uint64_t t1[S];
  __shared__ uint64_t rw[RA];
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t C1w = (uint32_t)D << logC1;  // words of one row of the message matrix
  const size_t C = (size_t)1 << a.logC;
  const uint32_t ntile = C1w / WB;
  const uint32_t njg = (uint32_t)((a.M + jn - 1) / jn);
  uint32_t lb;
  if (!xcd_block(ntile * (uint32_t)a.Q * njg, lb)) return;
  const uint32_t c = lb % (uint32_t)a.Q, rest = lb / (uint32_t)a.Q;
  const uint32_t wc0 = (rest % ntile) * WB;
  const size_t j0 = (size_t)(rest / ntile) * jn, j1 = j0 + jn < a.M ? j0 + jn : a.M;
  Mats A;
  load_mats(A, mat + (F16 ? MAT16 : 0));
  const uint64_t* rowc = row + (size_t)c * S;
  for (int k = threadIdx.x; k < S; k += 512) t1[k] = c ? gl::mul(tw[k], rowc[k / RA]) : tw[k];
  if (threadIdx.x < RA) rw[(threadIdx.x & 3) * NA + SA::in_i(threadIdx.x)] = rowc[threadIdx.x * RB];
  const uint64_t* postc = post + c * C;
  const size_t Lw = a.L * D, mw = a.mask_len * D;
  const bool full = a.L == C;
  const uint32_t nwt = C1w / 8;
  __syncthreads();
  for (size_t j = j0; j < j1; j++) {
    const uint64_t* msg = msg_ptr<D>(a, j) + wc0;
#pragma unroll 1
    for (int t = wave; t < RB * WB / 16; t += 512 / 64) {
      const uint32_t q = t * 16 + n, col = q % WB, lo = q / WB;
      uint64_t x[NA];
      const uint32_t v0 = ((g * RB + lo) * C1w + col) * 8;
      if (full) {
#pragma unroll
        for (int i = 0; i < NA; i++) x[i] = ld(msg + (size_t)SA::in_u(i) * RB * C1w, v0);
      } else {
        const uint64_t* mask = a.masks ? a.masks + (a.j0 + j) * mw : nullptr;
#pragma unroll
        for (int i = 0; i < NA; i++)
          x[i] = word_at<D>(msg - wc0, Lw, mask, mw, (size_t)(SA::in_u(i) * RB) * C1w + (v0 >> 3) + wc0);
      }
      if (c) {
#pragma unroll
        for (int i = 0; i < NA; i++)
          x[i] = mulw<F16>(x[i], rw[g * NA + i], A.k);
      } else if constexpr (F16) {
#pragma unroll
        for (int i = 0; i < NA; i++) x[i] = biased(x[i]);
      }
      SCHED_FENCE();
      const uint64_t* w = t1 + lo * RA + SA::out_g * g;
      uint64_t* d = s + SA::out_g * g * KS + q;
      dft<LA, F16>(A, x, [&](int i, uint64_t o) { d[SA::out_u(i) * KS] = mulw<F16>(o, w[SA::out_u(i)], A.k); });
    }
    __syncthreads();
    uint64_t* yj = Y + (j * a.N + c * C) * D;
#pragma unroll 1
    for (int t = wave; t < RA * WB / 16; t += 512 / 64) {
      const uint32_t q = t * 16 + n, col = q % WB, k1 = q / WB;
      const uint32_t i1 = (wc0 + col) / D, wt = (wc0 + col) >> 3;
      const uint32_t t2 = k1 + RA * SB::out_g * g;
      const uint32_t vp = ((t2 << logC1) + i1) * 8;
      const uint32_t vy = (((((t2 >> logBY) * nwt + wt) << logBY) + (t2 & ((1u << logBY) - 1))) * 8 + (col & 7)) * 8;
      uint64_t x[NB], w[NB];
#pragma unroll
      for (int i = 0; i < NB; i++) w[i] = ld(postc + ((size_t)(RA * SB::out_u(i)) << logC1), vp);
      const uint64_t* src = s + k1 * KS + g * WB + col;
#pragma unroll
      for (int i = 0; i < NB; i++) x[i] = src[SB::in_u(i) * WB];
      dft<LB, F16>(A, x, [&](int i, uint64_t o) { st(yj + (size_t)(RA * SB::out_u(i)) * C1w, vy, mulw<NEXT16>(o, w[i], A.k)); });
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------------ pass 2: rows
template <int D, int LA, int LB, int B>
__global__ __launch_bounds__((row_threads<D, LA>()), 4) void k_mx_pass2(RsArgs a, const v4i* mat, const uint64_t* tw, const uint64_t* Y,
                                                        int logC1) {
  constexpr int TH = row_threads<D, LA>(), RA = 1 << LA, RB = 1 << LB, S = RA * RB;
  constexpr int BY = B < 16 ? B : 16, BD = B * D;
  constexpr bool F16 = LA == 4 && LB == 4;
  using SA = Step<LA, F16>;
  using SB = Step<LB, F16>;
  constexpr int NA = RA / 4, NB = RB / 4, PS = S * D + (D == 1 ? 9 : D == 2 ? 10 : 11);
  __shared__ uint64_t s[B * PS];
  __shared__ uint64_t t1[S];
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int logC2 = a.logC - logC1;
  const uint32_t C2 = 1u << logC2;
  const size_t C = (size_t)1 << a.logC;
  const uint32_t ntile = C2 / B, nl = ntile * (uint32_t)a.Q * (uint32_t)a.M;
  const uint32_t per = (nl + 7) / 8, l1 = min(nl, (blockIdx.x % 8 + 1) * per);
  for (int k = threadIdx.x; k < S; k += TH) t1[k] = tw[k];
  Mats A;
  load_mats(A, mat + (F16 ? MAT16 : 0));
  __syncthreads();
  for (uint32_t lb = (blockIdx.x % 8) * per + blockIdx.x / 8; lb < l1; lb += gridDim.x / 8) {
    const uint32_t t2_0 = (lb % ntile) * B;
    const size_t c = (lb / ntile) % (uint32_t)a.Q, j = (lb / ntile) / (uint32_t)a.Q;
    const uint64_t* yj = Y + (j * a.N + c * C + (size_t)t2_0 * S) * D;
#pragma unroll 1
    for (int t = wave; t < RB * BD / 16; t += TH / 64) {
      const uint32_t q = t * 16 + n, col8 = q & 7, r = (q >> 3) % B, lt = q / (8 * B);
      const uint32_t wl = lt * 8 + col8, lo = wl / D;
      uint64_t x[NA];
      const uint32_t v0 = (((r / BY) * (S * D / 8) + g * (RB * D / 8) + lt) * (BY * 8) + (r % BY) * 8 + col8) * 8;
#pragma unroll
      for (int i = 0; i < NA; i++) x[i] = ld(yj + SA::in_u(i) * (RB * D) * BY, v0);
      const uint64_t* w = t1 + lo * RA + SA::out_g * g;
      uint64_t* d = s + r * PS + SA::out_g * g * (RB * D) + wl;
      dft<LA, F16>(A, x, [&](int i, uint64_t o) { d[SA::out_u(i) * (RB * D)] = mulw<F16>(o, w[SA::out_u(i)], A.k); });
    }
    __syncthreads();
    uint64_t* oj = out_ptr<D>(a, j) + (c * C + t2_0) * D;
#pragma unroll 1
    for (int t = wave; t < RA * BD / 16; t += TH / 64) {
      const uint32_t q = t * 16 + n, line = q % BD, k1 = q / BD;
      uint64_t x[NB];
      const uint64_t* src = s + (line / D) * PS + (k1 * RB + g) * D + line % D;
#pragma unroll
      for (int i = 0; i < NB; i++) x[i] = src[SB::in_u(i) * D];
      const uint32_t vo = (((k1 + RA * SB::out_g * g) << logC2) * D + line) * 8;
      dft<LB, F16>(A, x,
              [&](int i, uint64_t o) { st(oj + ((size_t)(RA * SB::out_u(i)) << logC2) * D, vo, canon(o)); });
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------------ single pass
template <int D, int LA, int LB>
__global__ __launch_bounds__(512, 4) void k_mx_single(RsArgs a, const v4i* mat, const uint64_t* tw, const uint64_t* pre,
                                                    int G) {
  constexpr int TH = 512, RA = 1 << LA, RB = 1 << LB, S = RA * RB;
  constexpr bool F16 = LA == 4 && LB == 4;
  using SA = Step<LA, F16>;
  using SB = Step<LB, F16>;
  constexpr int NA = RA / 4, NB = RB / 4, KS = RB * D + D;
  __shared__ uint64_t s[sequences<D>(S) * RA * KS];
  __shared__ uint64_t t1[S];
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t nseq = (uint32_t)(a.M * a.Q), Q = (uint32_t)a.Q;
  const int logQ = __builtin_ctz(Q);  // a power of two, as the codeword and coset lengths are
  for (int k = threadIdx.x; k < S; k += TH) t1[k] = tw[k];
  Mats A;
  load_mats(A, mat + (F16 ? MAT16 : 0));
  const size_t Lw = a.L * D, mw = a.mask_len * D;
  __syncthreads();
  for (uint32_t seq0 = blockIdx.x * G; seq0 < nseq; seq0 += gridDim.x * G) {
#pragma unroll 1
    for (int t = wave; t < G * RB * D / 16; t += TH / 64) {
      // group: 16 words (lo, d), of one sequence unless a sequence has fewer or 24 of them
      constexpr bool ONE = RB * D % 16 == 0;
      const uint32_t q = t * 16 + n, sq = ONE ? t / (RB * D / 16) : q / (RB * D), wl = q - sq * (RB * D), lo = wl / D;
      if (seq0 + (t * 16) / (RB * D) >= nseq) break;  // uniform: later sequences are past the end too
      const uint32_t seq = min(seq0 + sq, nseq - 1), j = seq >> logQ, c = seq & (Q - 1);
      const uint64_t* msg = msg_ptr<D>(a, j);
      const uint64_t* mask = a.masks ? a.masks + (a.j0 + j) * mw : nullptr;
      uint64_t x[NA], p[NA];
#pragma unroll
      for (int e = 0; e < NA; e++) {
        x[e] = word_at<D>(msg, Lw, mask, mw, (SA::in_u(e) + g) * (RB * D) + wl);
        p[e] = ld(pre + (size_t)c * S + SA::in_u(e) * RB, (g * RB + lo) * 8);
      }
#pragma unroll
      for (int e = 0; e < NA; e++) x[e] = mulw<F16>(x[e], p[e], A.k);
      SCHED_FENCE();
      const uint64_t* w = t1 + lo * RA + SA::out_g * g;
      uint64_t* d = s + (sq * RA + SA::out_g * g) * KS + wl;
      dft<LA, F16>(A, x, [&](int e, uint64_t o) { d[SA::out_u(e) * KS] = mulw<F16>(o, w[SA::out_u(e)], A.k); });
    }
    __syncthreads();
#pragma unroll 1
    for (int t = wave; t < G * RA * D / 16; t += TH / 64) {
      constexpr bool ONE = RA * D % 16 == 0;
      const uint32_t q = t * 16 + n, sq = ONE ? t / (RA * D / 16) : q / (RA * D), kw = q - sq * (RA * D), k1 = kw / D;
      if (seq0 + (t * 16) / (RA * D) >= nseq) break;
      const uint32_t seq = min(seq0 + sq, nseq - 1), j = seq >> logQ, c = seq & (Q - 1);
      uint64_t x[NB];
      const uint64_t* src = s + (sq * RA + k1) * KS + g * D + kw % D;
#pragma unroll
      for (int e = 0; e < NB; e++) x[e] = src[SB::in_u(e) * D];
      uint64_t* out = out_ptr<D>(a, j) + (size_t)c * S * D;
      const uint32_t vo = (RA * D * SB::out_g * g + kw) * 8;
      dft<LB, F16>(A, x, [&](int e, uint64_t o) {
        if (ONE || seq0 + sq < nseq) st(out + RA * D * SB::out_u(e), vo, canon(o));
      });
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------------ pass 1 of one step
// Columns of C2 = 8, 16 or 32 elements: a wave takes 16 word columns of one (message, coset)
// straight from memory to memory, no LDS and no barrier.
template <int D, int LA, bool NEXT16>
__global__ __launch_bounds__(512, 4) void k_mx_column(RsArgs a, const v4i* mat, const uint64_t* row, const uint64_t* post,
                                                     uint64_t* Y, int logC1, int logBY) {
  constexpr int RA = 1 << LA, NA = RA / 4;
  constexpr bool F16 = LA == 4;
  using SA = Step<LA, F16>;
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t C1w = (uint32_t)D << logC1, ntile = C1w / 16, nwt = C1w / 8;
  const size_t C = (size_t)1 << a.logC;
  const size_t Lw = a.L * D, mw = a.mask_len * D;
  const bool full = a.L == C;
  Mats A;
  load_mats(A, mat + (F16 ? MAT16 : 0));
  // column groups: tiles fastest, then cosets (the same message words), then messages
  const uint32_t units = ntile * (uint32_t)a.Q * (uint32_t)a.M;
  const uint32_t per = (units + 7) / 8, u1 = min(units, (blockIdx.x % 8 + 1) * per);
  for (uint32_t u = (blockIdx.x % 8) * per + (blockIdx.x / 8) * 8 + wave; u < u1; u += gridDim.x) {
    const uint32_t wc = (u % ntile) * 16 + n, jc = u / ntile;
    const uint32_t c = jc % (uint32_t)a.Q, j = jc / (uint32_t)a.Q;
    const uint64_t* msg = msg_ptr<D>(a, j);
    const uint64_t* mask = a.masks ? a.masks + (a.j0 + j) * mw : nullptr;
    const uint32_t i1 = wc / D, t2 = SA::out_g * g;
    const uint32_t v0 = (g * C1w + wc) * 8, vp = ((t2 << logC1) + i1) * 8;
    uint64_t x[NA], r[NA], w[NA];
#pragma unroll
    for (int e = 0; e < NA; e++) {
      x[e] = full ? ld(msg + (size_t)SA::in_u(e) * C1w, v0)
                  : word_at<D>(msg, Lw, mask, mw, (size_t)SA::in_u(e) * C1w + (v0 >> 3));
      r[e] = ld(row + (size_t)c * RA + SA::in_u(e), g * 8);
      w[e] = ld(post + c * C + ((size_t)SA::out_u(e) << logC1), vp);
    }
    if (c) {
#pragma unroll
      for (int e = 0; e < NA; e++) x[e] = mulw<F16>(x[e], r[e], A.k);
    } else if constexpr (F16) {
#pragma unroll
      for (int e = 0; e < NA; e++) x[e] = biased(x[e]);
    }
    uint64_t* yj = Y + ((size_t)j * a.N + c * C) * D;
    dft<LA, F16>(A, x, [&](int e, uint64_t o) {
      const uint32_t t = t2 + SA::out_u(e);
      const uint32_t vy = (((((t >> logBY) * nwt + (wc >> 3)) << logBY) + (t & ((1u << logBY) - 1))) * 8 + (wc & 7)) * 8;
      st(yj, vy, mulw<NEXT16>(o, w[e], A.k));
    });
  }
}

// ------------------------------------------------------------------ single pass, three steps
// C = 2^12 = 16 * 16 * 16, each step in place in LDS.  The first step's output factor
// w_N^(lo (c + Q k1)) is the four-step post factor of the split 16 * 256.
template <int D>
__global__ __launch_bounds__(512, 4) void k_mx_cube(RsArgs a, const v4i* mat, const uint64_t* tw256, const uint64_t* row,
                                                   const uint64_t* post) {
  constexpr int S = 4096, G = D == 1 ? 2 : 1, KS = 256 * D + D;
  using SA = Step<4, true>;
  __shared__ uint64_t s[G * 16 * KS];
  __shared__ uint64_t t2[256];
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t nseq = (uint32_t)(a.M * a.Q), Q = (uint32_t)a.Q;
  const int logQ = __builtin_ctz(Q);
  const size_t Lw = a.L * D, mw = a.mask_len * D;
  Mats A;
  load_mats(A, mat + MAT16);
  if (threadIdx.x < 256) t2[threadIdx.x] = tw256[threadIdx.x];
  __syncthreads();
  for (uint32_t seq0 = blockIdx.x * G; seq0 < nseq; seq0 += gridDim.x * G) {
#pragma unroll 1
    for (int t = wave; t < G * 16 * D; t += 8) {
      const uint32_t sq = t / (16 * D), wl = (t % (16 * D)) * 16 + n, lo = wl / D;
      const uint32_t seq = seq0 + sq;
      if (seq >= nseq) break;  // uniform: later sequences are past the end too
      const uint32_t j = seq >> logQ, c = seq & (Q - 1);
      const uint64_t* msg = msg_ptr<D>(a, j);
      const uint64_t* mask = a.masks ? a.masks + (a.j0 + j) * mw : nullptr;
      uint64_t x[4], r[4], w[4];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        x[e] = word_at<D>(msg, Lw, mask, mw, (SA::in_u(e) + g) * (256 * D) + wl);
        r[e] = ld(row + (size_t)c * 16 + SA::in_u(e), g * 8);
      }
#pragma unroll
      for (int e = 0; e < 4; e++) w[e] = ld(post + (size_t)c * S + SA::out_u(e) * 256, (g * 256 + lo) * 8);
#pragma unroll
      for (int e = 0; e < 4; e++) x[e] = mulw<true>(x[e], r[e], A.k);
      SCHED_FENCE();
      uint64_t* d = s + (sq * 16 + g) * KS + wl;
      dft<4, true>(A, x, [&](int e, uint64_t o) { d[SA::out_u(e) * KS] = mulw<true>(o, w[e], A.k); });
    }
    __syncthreads();
#pragma unroll 1
    for (int t = wave; t < G * 16 * D; t += 8) {  // group: 16 words (lo2, d) of one k1
      const uint32_t kq = t / D, wl = (t % D) * 16 + n, lo2 = wl / D;
      uint64_t* p = s + kq * KS + wl + g * (16 * D);
      uint64_t x[4];
#pragma unroll
      for (int e = 0; e < 4; e++) x[e] = p[SA::in_u(e) * 16 * D];
      const uint64_t* w = t2 + lo2 * 16 + g;
      dft<4, true>(A, x, [&](int e, uint64_t o) { p[SA::out_u(e) * 16 * D] = mulw<true>(o, w[SA::out_u(e)], A.k); });
    }
    __syncthreads();
#pragma unroll 1
    for (int t = wave; t < G * 16 * D; t += 8) {  // group: 16 words (k1, d) of one k2
      const uint32_t sq = t / (16 * D), r = t % (16 * D), k2 = r / D, kw = (r % D) * 16 + n, k1 = kw / D, d = kw % D;
      const uint32_t seq = seq0 + sq;
      if (seq >= nseq) break;
      const uint32_t j = seq >> logQ, c = seq & (Q - 1);
      uint64_t x[4];
      const uint64_t* p = s + (sq * 16 + k1) * KS + (k2 * 16 + g) * D + d;
#pragma unroll
      for (int e = 0; e < 4; e++) x[e] = p[SA::in_u(e) * D];
      uint64_t* out = out_ptr<D>(a, j) + ((size_t)c * S + k2 * 16) * D;
      const uint32_t vo = (256 * D * g + kw) * 8;
      dft<4, true>(A, x, [&](int e, uint64_t o) { st(out + 256 * D * SA::out_u(e), vo, canon(o)); });
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------------ single pass, one step
// C = 16 or 32: 16 columns of a wave are 16 (coset, d) words of one message, which all read
// the same coefficients.
template <int D, int LA>
__global__ __launch_bounds__(512, 4) void k_mx_short(RsArgs a, const v4i* mat, const uint64_t* pre) {
  constexpr int RA = 1 << LA, NA = RA / 4;
  constexpr bool F16 = LA == 4;
  using SA = Step<LA, F16>;
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const size_t Lw = a.L * D, mw = a.mask_len * D;
  Mats A;
  load_mats(A, mat + (F16 ? MAT16 : 0));
  const uint64_t words = a.Q * D, groups = (words + 15) / 16, units = groups * a.M;
  for (uint64_t u = (uint64_t)blockIdx.x * 8 + wave; u < units; u += (uint64_t)gridDim.x * 8) {
    const uint64_t j = u / groups, cw = (u % groups) * 16 + n, c = min(cw, words - 1) / D;
    const uint32_t d = (uint32_t)(min(cw, words - 1) % D);
    const uint64_t* msg = msg_ptr<D>(a, j);
    const uint64_t* mask = a.masks ? a.masks + (a.j0 + j) * mw : nullptr;
    uint64_t x[NA], p[NA];
#pragma unroll
    for (int e = 0; e < NA; e++) {
      x[e] = word_at<D>(msg, Lw, mask, mw, (SA::in_u(e) + g) * D + d);
      p[e] = pre[c * RA + SA::in_u(e) + g];
    }
#pragma unroll
    for (int e = 0; e < NA; e++) x[e] = mulw<F16>(x[e], p[e], A.k);
    uint64_t* o = out_ptr<D>(a, j) + (c * RA + SA::out_g * g) * D + d;
    dft<LA, F16>(A, x, [&](int e, uint64_t v) {
      if (cw < words) o[SA::out_u(e) * D] = canon(v);
    });
  }
}

// ------------------------------------------------------------------ host
struct Consts {
  int cus;
  const v4i* mat;
  const uint64_t* tw[11];  // tw[s][lo * RA + k1] = w_S^(lo k1)
};
std::mutex g_mu;
std::map<int, Consts> g_consts;

// log2 of the first radix of a two-step transform of 2^s points: 8*8, 16*8, 16*16, 32*16, 32*32
constexpr int first_step(int s) { return s == 6 ? 3 : s <= 8 ? 4 : 5; }

// Signed digits of v mod p in base 256.
void digits(uint64_t v, int8_t out[8]) {
  if (v > 0x7F7F7F7F7F7F7F7Full) v -= gl::P;
  const uint64_t t = v + 0x8080808080808080ull;
  for (int k = 0; k < 8; k++) out[k] = (int8_t)((uint8_t)(t >> (8 * k)) ^ 0x80);
}

Consts build_consts() {
  // Tables of 16 operand registers (16 bytes a lane) and the two accumulator starts.  Row
  // r of a tile is digit 4 (tile % 2) + r % 4 of output 4 (tile / 2) + r / 4; the 16 bytes
  // of lane group kg are the digits of inputs kg + 8 .. (see the byte index below).
  std::vector<int8_t> m(2 * MAT16 * 16);
  const uint64_t w32 = gl::root_of_unity(32);
  int32_t start[8];
  {
    // accumulators start at 2^21 (above any sum's magnitude) plus the digits of minus that
    uint64_t tot = 0;
    for (int k = 7; k >= 0; k--) {
      for (int x = 0; x < 8; x++) tot = gl::add(tot, tot);
      tot = gl::add(tot, 1ull << 21);
    }
    const uint64_t adj = gl::neg(tot);
    for (int k = 0; k < 8; k++) start[k] = (1 << 21) + (int)((adj >> (8 * k)) & 255);
  }
  for (int full = 0; full < 2; full++) {
    int8_t* base = m.data() + (size_t)full * MAT16 * 16;
    for (int i = 0; i < 16; i++)
      for (int lane = 0; lane < 64; lane++) {
        const int tile = full ? i / 2 : i % 4, r = full ? 0 : i / 4;
        const int k = 4 * (tile / 2) + (lane % 16) / 4, digit = 4 * (tile % 2) + lane % 4;
        for (int b = 0; b < 16; b++) {
          const int j = 4 * ((full ? 2 * (i % 2) : 0) + b / 8) + lane / 16;
          uint64_t v = gl::pow(w32, full ? (uint64_t)(2 * j * k) : (uint64_t)(r * j + 4 * j * k));
          for (int x = 0; x < 8 * (b % 8); x++) v = gl::add(v, v);
          int8_t d[8];
          digits(v, d);
          base[((size_t)i * 64 + lane) * 16 + b] = d[digit];
        }
      }
    memcpy(base + 1024 * 16, start, 32);
  }
  Consts c{};
  int dev = 0;
  WHIR_HIP(hipGetDevice(&dev));
  WHIR_HIP(hipDeviceGetAttribute(&c.cus, hipDeviceAttributeMultiprocessorCount, dev));
  void* p = nullptr;
  WHIR_HIP(hipMalloc(&p, m.size()));
  WHIR_HIP(hipMemcpy(p, m.data(), m.size(), hipMemcpyHostToDevice));
  c.mat = (const v4i*)p;
  for (int s = 6; s <= 10; s++) {
    const int LA = first_step(s), RA = 1 << LA, RB = 1 << (s - LA);
    std::vector<uint64_t> t((size_t)1 << s);
    const uint64_t w = gl::root_of_unity(1ull << s);
    for (int lo = 0; lo < RB; lo++)
      for (int k1 = 0; k1 < RA; k1++) t[lo * RA + k1] = gl::pow(w, (uint64_t)lo * k1);
    void* d = nullptr;
    WHIR_HIP(hipMalloc(&d, t.size() * 8));
    WHIR_HIP(hipMemcpy(d, t.data(), t.size() * 8, hipMemcpyHostToDevice));
    c.tw[s] = (const uint64_t*)d;
  }
  return c;
}

const Consts& consts() {
  int dev = 0;
  WHIR_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> g(g_mu);
  auto it = g_consts.find(dev);
  if (it != g_consts.end()) return it->second;
  WHIR_REQUIRE(!capture_active(), "ntt: tables built during a stream capture");
  return g_consts.emplace(dev, build_consts()).first->second;
}

unsigned xcd_grid(uint64_t nlogical) {
  WHIR_REQUIRE(nlogical < (1ull << 31), "interleaved_encode: too many blocks");
  return (unsigned)((nlogical + 7) / 8 * 8);
}

// Blocks of a kernel whose blocks loop over the work: at most two per CU, a multiple of 8.
unsigned resident(const Consts& k, uint64_t nlogical) {
  WHIR_REQUIRE(nlogical < (1ull << 31), "interleaved_encode: too many blocks");
  return (unsigned)std::min<uint64_t>((nlogical + 7) / 8 * 8, std::max(8, k.cus * 2 / 8 * 8));
}

// log2 of the rows that lie together in pass 1's output, for rows of 2^logC1 in cosets of 2^logC.
template <int D>
int log_by(int logC1, int logC) {
  int by = 0;
  while ((2 << by) <= std::min({16, row_block<D>(1 << logC1), 1 << (logC - logC1)})) by++;
  return by;
}

template <int D, int LA, int LB>
void pass1(const RsArgs& a, const Consts& k, const MxTables& t, uint64_t* scratch, int logC1, hipStream_t st) {
  constexpr int S = 1 << (LA + LB), WB = TILE / S;
  const uint64_t base = ((uint64_t)D << logC1) / WB * a.Q;
  int jn = 1;
  while (jn * 2 <= (int)a.M && base * ((a.M + jn * 2 - 1) / (jn * 2)) >= 512) jn *= 2;
  ProfScope prof(kernel_name("k_mx_pass1", D, LA + LB), st, 8.0 * D * ((double)a.M * a.L + (double)a.M * a.N));
  auto kernel = logC1 == 8 ? k_mx_pass1<D, LA, LB, true> : k_mx_pass1<D, LA, LB, false>;
  kernel<<<xcd_grid(base * ((a.M + jn - 1) / jn)), 512, 0, st>>>(a, k.mat, k.tw[LA + LB], t.row, t.post, scratch, logC1,
                                                                     log_by<D>(logC1, a.logC), jn);
  WHIR_HIP(hipGetLastError());
}
template <int D, int LA, int LB>
void pass2(const RsArgs& a, const Consts& k, const uint64_t* scratch, int logC1, hipStream_t st) {
  constexpr int B = row_block<D>(1 << (LA + LB));
  const uint64_t C2 = 1ull << (a.logC - logC1);
  ProfScope prof(kernel_name("k_mx_pass2", D, LA + LB), st, 16.0 * D * (double)a.M * a.N);
  const auto launch = [&](auto kernel, int rows) {
    kernel<<<resident(k, C2 / rows * a.Q * a.M), row_threads<D, LA>(), 0, st>>>(a, k.mat, k.tw[LA + LB], scratch, logC1);
  };
  // the column steps of 2^11 and 2^12 elements leave 8 and 16 rows
  constexpr int B16 = std::min(B, 16), B8 = std::min(B, 8);
  if (C2 >= B) launch(k_mx_pass2<D, LA, LB, B>, B);
  else if (C2 == 16) launch(k_mx_pass2<D, LA, LB, B16>, B16);
  else launch(k_mx_pass2<D, LA, LB, B8>, B8);
  WHIR_HIP(hipGetLastError());
}
template <int D, int LA, int LB>
void single(const RsArgs& a, const Consts& k, const MxTables& t, hipStream_t st) {
  constexpr int S = 1 << (LA + LB);
  const uint64_t nseq = a.M * a.Q;
  WHIR_REQUIRE(nseq < (1ull << 30), "interleaved_encode: too many cosets");
  // Small encodes spread over the CUs instead of filling their tiles (an even count, so that
  // groups of 16 words end with a sequence's words): 16 messages 2^10 -> 2^11 13.2 -> 7.3 us.
  int G = sequences<D>(S);
  while (G > 2 && nseq <= (uint64_t)k.cus * (G / 2)) G /= 2;
  ProfScope prof(kernel_name("k_mx_single", D, LA + LB), st, 8.0 * D * ((double)a.M * a.L + (double)a.M * a.N));
  k_mx_single<D, LA, LB><<<resident(k, (nseq + G - 1) / G), 512, 0, st>>>(a, k.mat, k.tw[LA + LB], t.pre, G);
  WHIR_HIP(hipGetLastError());
}

template <int D, int LA>
void column(const RsArgs& a, const Consts& k, const MxTables& t, uint64_t* scratch, int logC1, hipStream_t st) {
  const uint64_t units = ((uint64_t)D << logC1) / 16 * a.Q * a.M;
  WHIR_REQUIRE(units < (1ull << 31), "interleaved_encode: too many column groups");
  ProfScope prof(kernel_name("k_mx_column", D, LA), st, 8.0 * D * ((double)a.M * a.L + (double)a.M * a.N));
  auto kernel = logC1 == 8 ? k_mx_column<D, LA, true> : k_mx_column<D, LA, false>;
  kernel<<<resident(k, (units + 7) / 8), 512, 0, st>>>(a, k.mat, t.row, t.post, scratch, logC1, log_by<D>(logC1, a.logC));
  WHIR_HIP(hipGetLastError());
}
template <int D>
void cube(const RsArgs& a, const Consts& k, const MxTables& t, hipStream_t st) {
  WHIR_REQUIRE(a.M * a.Q < (1ull << 30), "interleaved_encode: too many cosets");
  ProfScope prof(kernel_name("k_mx_cube", D), st, 8.0 * D * ((double)a.M * a.L + (double)a.M * a.N));
  k_mx_cube<D><<<resident(k, (a.M * a.Q + (D == 1)) / (D == 1 ? 2 : 1)), 512, 0, st>>>(a, k.mat, k.tw[8], t.row, t.post);
  WHIR_HIP(hipGetLastError());
}
template <int D, int LA>
void shortest(const RsArgs& a, const Consts& k, const MxTables& t, hipStream_t st) {
  const uint64_t units = (a.Q * D + 15) / 16 * a.M;
  ProfScope prof(kernel_name("k_mx_short", D, LA), st, 8.0 * D * ((double)a.M * a.L + (double)a.M * a.N));
  k_mx_short<D, LA><<<resident(k, (units + 7) / 8), 512, 0, st>>>(a, k.mat, t.pre);
  WHIR_HIP(hipGetLastError());
}

template <int D>
void encode(const RsArgs& a, const MxTables& t, uint64_t* scratch, hipStream_t st) {
  const Consts& k = consts();
  int logC1 = 0;
  WHIR_REQUIRE(mx_split(a.logC, &logC1), "interleaved_encode: no matrix-core transform of this size");
  switch (logC1 ? 0 : a.logC) {
    case 0: break;
    case 4: return shortest<D, 4>(a, k, t, st);
    case 5: return shortest<D, 5>(a, k, t, st);
    case 6: return single<D, 3, 3>(a, k, t, st);
    case 7: return single<D, 4, 3>(a, k, t, st);
    case 8: return single<D, 4, 4>(a, k, t, st);
    case 9: return single<D, 5, 4>(a, k, t, st);
    default: return single<D, 5, 5>(a, k, t, st);
  }
  // 2^12: one kernel instead of a column step and rows once the grid is full (Fp 2^22 words
  // 35.2 -> 28.4 us, Fp2 2^25 words 239 -> 204; but Fp 2^19 words 11.6 -> 15.9, Fp2 2^20
  // 16.8 -> 19.9, and Fp2 2^23 words 59.0 and 60.7, the same).
  if constexpr (D < 3) {
    if (a.logC == 12 && a.M * a.N * D >= (D == 1 ? 1ull << 22 : 1ull << 24)) return cube<D>(a, k, t, st);
  }
  // Fp3 messages go through both passes in groups whose intermediate is at most 128 MB:
  // pass 2's reads of it (and its partly written lines) then meet in the 256 MB last-level
  // cache (16 messages 2^18 -> 2^21: pass 1 + 2 471 + 588 -> 535 + 410 us).  Fp and Fp2,
  // whose pass 2 is at the memory's rate already, lose more to the smaller launches than
  // they gain (Fp 2^20 -> 2^22: 670 -> 700 us).
  const size_t per = D < 3 ? (size_t)a.M : std::max<size_t>(1, ((size_t)128 << 20) / (a.N * D * 8));
  for (size_t j0 = 0; j0 < a.M; j0 += per) {
    RsArgs b = a;
    b.j0 = j0;
    b.M = std::min<size_t>(per, a.M - j0);
    switch (a.logC - logC1) {
      case 3: column<D, 3>(b, k, t, scratch, logC1, st); break;
      case 4: column<D, 4>(b, k, t, scratch, logC1, st); break;
      case 5: column<D, 5>(b, k, t, scratch, logC1, st); break;
      case 8: pass1<D, 4, 4>(b, k, t, scratch, logC1, st); break;
      case 9: pass1<D, 5, 4>(b, k, t, scratch, logC1, st); break;
      default: pass1<D, 5, 5>(b, k, t, scratch, logC1, st); break;
    }
    switch (logC1) {
      case 8: pass2<D, 4, 4>(b, k, scratch, logC1, st); break;
      case 9: pass2<D, 5, 4>(b, k, scratch, logC1, st); break;
      default: pass2<D, 5, 5>(b, k, scratch, logC1, st); break;
    }
  }
}

}  // namespace

bool mx_split(int logC, int* logC1) {
  // one pass up to 2^10; 2^11 .. 2^15 a column step of 8, 16 or 32, then rows; from 2^16
  // the balanced split
  *logC1 = logC < 11 ? 0 : logC == 11 ? 8 : logC < 16 ? std::min(logC - 4, 10) : (logC + 1) / 2;
  return logC >= 4 && logC <= 20;
}

void mx_prepare() { (void)consts(); }

void mx_encode(int D, const RsArgs& a, const MxTables& t, uint64_t* scratch, hipStream_t st) {
  switch (D) {
    case 1: return encode<1>(a, t, scratch, st);
    case 2: return encode<2>(a, t, scratch, st);
    case 3: return encode<3>(a, t, scratch, st);
    default: throw Error("rs_encode: extension degree must be 1, 2 or 3");
  }
}

}  // namespace whir
