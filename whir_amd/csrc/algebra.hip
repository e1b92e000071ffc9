// Sumcheck prover round and covector builders on CDNA4.
//
// All of these are streaming passes over HBM with exact Goldilocks arithmetic,
// so their order of summation does not change any result.  Reductions run as
// grid-stride partial sums per block (LDS tree) followed by one small block.
#include "algebra.h"
#include "common.h"
#include "gl.h"
#include "ntt.h"

#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <type_traits>
#include <utility>
#include <vector>

namespace whir {

using gl::Ext;

static constexpr int RT = 256;            // threads per block for streaming kernels
static constexpr unsigned MAX_BLOCKS = 2048;

template <int D>
__device__ __forceinline__ Ext<D> ld(const uint64_t* p, size_t i) {
  Ext<D> r;
#pragma unroll
  for (int d = 0; d < D; d++) r.c[d] = p[i * D + d];
  return r;
}
// f(std::integral_constant<int, 0>{}), ..., f(std::integral_constant<int, N - 1>{}):
// a loop whose index is a compile-time constant in the body, so arrays indexed by it
// stay in registers however large the body is (an unroll pragma gives up on large
// bodies, and the arrays then go to scratch memory).
template <class F, int... J>
__device__ __forceinline__ void static_for_seq(F&& f, std::integer_sequence<int, J...>) {
  (f(std::integral_constant<int, J>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_seq(f, std::make_integer_sequence<int, N>{});
}

template <int D>
__device__ __forceinline__ void st(uint64_t* p, size_t i, const Ext<D>& v) {
#pragma unroll
  for (int d = 0; d < D; d++) p[i * D + d] = v.c[d];
}
template <int D>
__device__ __forceinline__ Ext<D> ld_host(const uint64_t* const* unused, const Ext<D>& v) { return v; }

// Block sums.  The short passes of a proof run these kernels on a wave or a few, where
// straight-line code is fetched once and used once: at about 0.45 us per KB of cold code
// on MI355X the fetch, not the arithmetic, was most of their time.  So the exchanges stay
// a loop over the distance, and the last steps give a word to each thread.

// Sums lane l of every R lanes (R a power of two; lane's role l = lane mod R) over the
// block: tot[(l NV + k) D + d] for the role's value k, in LDS, for all threads.  At most
// 1024 threads.
template <int D, int NV, int R>
__device__ __forceinline__ void block_role_sum(Ext<D> (&v)[NV], uint64_t* tot) {
  constexpr int W = R * NV * D;
  static_assert(W <= 64, "block_role_sum: one wave finishes the words");
  __shared__ uint64_t red[16][W];
#pragma unroll 1
  for (int off = R; off < 64; off <<= 1)
#pragma unroll
    for (int k = 0; k < NV; k++)
#pragma unroll
      for (int d = 0; d < D; d++) v[k].c[d] = gl::add(v[k].c[d], (uint64_t)__shfl_xor(v[k].c[d], off));
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane < R)
#pragma unroll
    for (int k = 0; k < NV; k++)
#pragma unroll
      for (int d = 0; d < D; d++) red[wave][(lane * NV + k) * D + d] = v[k].c[d];
  __syncthreads();
  if (threadIdx.x < W) {
    const int waves = blockDim.x >> 6;
    uint64_t x = red[0][threadIdx.x];
#pragma unroll 1
    for (int w = 1; w < waves; w++) x = gl::add(x, red[w][threadIdx.x]);
    tot[threadIdx.x] = x;
  }
  __syncthreads();
}

// The first W threads (one wave) store a word each; the flag follows when sig asks it to.
template <int W>
__device__ __forceinline__ void store_words(uint64_t word, uint64_t* out, const MailboxSig& sig) {
  if (threadIdx.x < W) out[threadIdx.x] = word;
  if (sig.flag) {
    __syncthreads();  // every word is stored before thread 0 raises the flag
    if (threadIdx.x == 0) mailbox_raise(sig);
  }
}

// Sum NV extension values over the block and write them to out.
template <int D, int NV>
__device__ void block_reduce_store(Ext<D> (&v)[NV], uint64_t* out, MailboxSig sig = {}) {
  __shared__ uint64_t tot[NV * D];
  block_role_sum<D, NV, 1>(v, tot);
  store_words<NV * D>(threadIdx.x < NV * D ? tot[threadIdx.x] : 0, out, sig);
}

// Final reduction of `nparts` block partials of NV*D words each into `out`
// (device memory, or the stream's pinned mailbox).  A second launch rather than a
// last-block-done reduction in the first: on CDNA4 the per-block device-scope
// release that pattern needs writes back the XCD's L2, and the producing kernels
// have just filled it with their outputs (measured 1.5x slower on MI355X).
template <int D, int NV>
__global__ __launch_bounds__(1024) void k_reduce_parts(const uint64_t* parts, size_t nparts, uint64_t* out,
                                                       MailboxSig sig) {
  __shared__ uint64_t tot[NV * D];
  Ext<D> v[1] = {gl::ext_zero<D>()};
  // a value per thread, so that the block reads the partials in order
  for (size_t e = threadIdx.x; e < nparts * NV; e += blockDim.x) v[0] = gl::eadd<D>(v[0], ld<D>(parts, e));
  block_role_sum<D, 1, NV>(v, tot);
  store_words<NV * D>(threadIdx.x < NV * D ? tot[threadIdx.x] : 0, out, sig);
}

// Threads of a one-block reduction of n values: whole waves, at most 1024.
static unsigned reduce_threads(size_t n) { return (unsigned)std::min<size_t>(1024, (n + 63) / 64 * 64); }

// last: this launch ends the work a mailbox wait may be armed for.
template <int D, int NV>
static void finish_reduce(const uint64_t* parts, unsigned nparts, uint64_t* out, hipStream_t s, bool last = true) {
  k_reduce_parts<D, NV><<<1, reduce_threads(nparts * (size_t)NV), 0, s>>>(parts, nparts, out, last ? mailbox_take(out) : MailboxSig{});
  WHIR_HIP(hipGetLastError());
}

static unsigned grid_for(size_t n) { return (unsigned)std::min<size_t>(blocks_for(n, RT), MAX_BLOCKS); }

// Up to this many element pairs a reducing pass runs as one block of up to 1024 threads,
// which stores its sums directly: cheaper than a second launch.
static constexpr size_t SMALL_PAIRS = 1024;

// Pass a small host constant (D words) to kernels by value.
template <int D>
static Ext<D> host_ext(const uint64_t* w) {
  Ext<D> r;
  for (int d = 0; d < D; d++) r.c[d] = w[d];
  return r;
}

static size_t next_pow2(size_t n) {
  size_t p = 1;
  while (p < n) p <<= 1;
  return p;
}

// ------------------------------------------------------------------ sumcheck polynomial
// Element i of a vector of Ds-word elements, embedded in the degree-D extension
// (Ds = 1: a base-field vector, as the initial round sees the committed vector).
template <int Ds, int D>
__device__ __forceinline__ Ext<D> ldx(const uint64_t* p, size_t i) {
  if constexpr (Ds == D) return ld<D>(p, i);
  else return gl::ext_base<D>(p[i]);
}

// a * b with a embedded from Ds words.
template <int Ds, int D>
__device__ __forceinline__ Ext<D> mulx(const uint64_t* a, size_t i, const Ext<D>& b) {
  if constexpr (Ds == D) return gl::emul<D>(ld<D>(a, i), b);
  else return gl::escale<D>(b, a[i]);
}

// w += a b with a embedded from Ds words.
template <int Ds, int D>
__device__ __forceinline__ void mulx_acc(gl::Wide (&w)[D], const Ext<Ds>& a, const Ext<D>& b) {
  if constexpr (Ds == D) {
    gl::emul_acc<D>(w, a, b);
  } else {
#pragma unroll
    for (int d = 0; d < D; d++) gl::wide_mac(w[d], a.c[0], b.c[d]);
  }
}

// The products are summed unreduced (emul_acc) and reduced once per lane.
template <int Ds, int D>
__global__ __launch_bounds__(1024) void k_sc_poly(const uint64_t* __restrict__ a, const uint64_t* __restrict__ b,
                                                size_t half, size_t nhi, uint64_t* parts, MailboxSig sig) {
  gl::Wide w[2][D];
  gl::wide_zero<D>(w[0]);
  gl::wide_zero<D>(w[1]);
#pragma unroll 1
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < half; i += (size_t)gridDim.x * blockDim.x) {
    const Ext<Ds> a0 = ld<Ds>(a, i);
    const Ext<D> b0 = ld<D>(b, i);
    Ext<Ds> a1 = gl::ext_zero<Ds>();  // implicit zero padding past the end
    Ext<D> b1 = gl::ext_zero<D>();
    if (i < nhi) {
      a1 = ld<Ds>(a, half + i);
      b1 = ld<D>(b, half + i);
    }
    mulx_acc<Ds, D>(w[0], a0, b0);
    mulx_acc<Ds, D>(w[1], gl::esub<Ds>(a1, a0), gl::esub<D>(b1, b0));
  }
  Ext<D> acc[2] = {gl::ext_reduce<D>(w[0]), gl::ext_reduce<D>(w[1])};
  block_reduce_store<D, 2>(acc, parts + (size_t)blockIdx.x * 2 * D, sig);
}

template <int Ds, int D>
__global__ void k_sc_single(const uint64_t* a, const uint64_t* b, size_t n, uint64_t* out, MailboxSig sig) {
  if (threadIdx.x != 0) return;
  Ext<D> c0 = n ? mulx<Ds, D>(a, 0, ld<D>(b, 0)) : gl::ext_zero<D>();
  st<D>(out, 0, c0);
  st<D>(out, 1, gl::ext_zero<D>());
  mailbox_raise(sig);
}

template <int Ds, int D>
static void sc_poly(const uint64_t* a, const uint64_t* b, size_t n, uint64_t* out, hipStream_t s) {
  if (n <= 1) {
    k_sc_single<Ds, D><<<1, 64, 0, s>>>(a, b, n, out, mailbox_take(out));
    WHIR_HIP(hipGetLastError());
    return;
  }
  size_t half = next_pow2(n) >> 1, nhi = n - half;
  // Small rounds: one block, which then writes the sums itself (no second launch).
  const unsigned g = half <= SMALL_PAIRS ? 1u : grid_for(half);
  DevBuf parts(g == 1 ? 0 : (size_t)g * 2 * D * 8, s);
  {
    ProfScope prof(kernel_name("k_sc_poly", Ds, D), s, 8.0 * (Ds + D) * (double)n);
    k_sc_poly<Ds, D><<<g, g == 1 ? reduce_threads(half) : RT, 0, s>>>(a, b, half, nhi, g == 1 ? out : parts.as<uint64_t>(),
                                      g == 1 ? mailbox_take(out) : MailboxSig{});
    WHIR_HIP(hipGetLastError());
  }
  if (g > 1) finish_reduce<D, 2>(parts.as<uint64_t>(), g, out, s);
}

void sumcheck_poly_mixed_dev(int Ds, int D, const uint64_t* a, const uint64_t* b, size_t n, uint64_t* out,
                             hipStream_t s) {
  if (Ds == D) {
    switch (D) {
      case 1: sc_poly<1, 1>(a, b, n, out, s); return;
      case 2: sc_poly<2, 2>(a, b, n, out, s); return;
      case 3: sc_poly<3, 3>(a, b, n, out, s); return;
    }
  } else if (Ds == 1) {
    switch (D) {
      case 2: sc_poly<1, 2>(a, b, n, out, s); return;
      case 3: sc_poly<1, 3>(a, b, n, out, s); return;
    }
  }
  throw Error("sumcheck: extension degree must be 1, 2 or 3");
}

void sumcheck_poly_dev(int D, const uint64_t* a, const uint64_t* b, size_t n, uint64_t* out, hipStream_t s) {
  sumcheck_poly_mixed_dev(D, D, a, b, n, out, s);
}

// ------------------------------------------------------------------ fold
// Folded element i of v (pairs (i, half + i), zero padded past n):
//   v[i] + w (v[half + i] - v[i])  or  v[i] (1 - w) when the partner is padding.
template <int Ds, int D>
__device__ __forceinline__ Ext<D> fold_at(const uint64_t* v, size_t i, size_t half, size_t nhi, const Ext<D>& w,
                                          const Ext<D>& om) {
  if constexpr (Ds == D) {
    const Ext<D> lo = ld<D>(v, i);
    if (i < nhi) return gl::eadd<D>(lo, gl::emul<D>(gl::esub<D>(ld<D>(v, half + i), lo), w));
    return gl::emul<D>(lo, om);
  } else {
    const uint64_t lo = v[i];
    if (i < nhi) {
      Ext<D> r = gl::escale<D>(w, gl::sub(v[half + i], lo));
      r.c[0] = gl::add(r.c[0], lo);
      return r;
    }
    return gl::escale<D>(om, lo);
  }
}

// out may alias in when Ds == D: lane i reads positions i and half + i and writes i only.
template <int Ds, int D>
__global__ __launch_bounds__(RT) void k_fold(const uint64_t* in, uint64_t* out, size_t half, size_t nhi, Ext<D> w,
                                             Ext<D> one_minus_w) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < half; i += (size_t)gridDim.x * blockDim.x)
    st<D>(out, i, fold_at<Ds, D>(in, i, half, nhi, w, one_minus_w));
}

template <int Ds, int D>
static size_t fold_t(const uint64_t* in, uint64_t* out, size_t n, const uint64_t* w, hipStream_t s) {
  if (n <= 1) {
    if (n == 1 && Ds != D) lift_dev(D, in, 1, out, s);  // nothing to fold: embed
    if (n == 1 && Ds == D && in != out) WHIR_HIP(hipMemcpyAsync(out, in, D * 8, hipMemcpyDeviceToDevice, s));
    return n;
  }
  size_t half = next_pow2(n) >> 1, nhi = n - half;
  Ext<D> ww = host_ext<D>(w);
  Ext<D> om = gl::esub<D>(gl::ext_base<D>(1), ww);
  ProfScope prof(kernel_name("k_fold", Ds, D), s, 8.0 * ((double)Ds * n + (double)D * half));
  k_fold<Ds, D><<<grid_for(half), RT, 0, s>>>(in, out, half, nhi, ww, om);
  WHIR_HIP(hipGetLastError());
  return half;
}

size_t fold_into_dev(int Ds, int D, const uint64_t* in, uint64_t* out, size_t n, const uint64_t* w, hipStream_t s) {
  if (Ds == D) {
    switch (D) {
      case 1: return fold_t<1, 1>(in, out, n, w, s);
      case 2: return fold_t<2, 2>(in, out, n, w, s);
      case 3: return fold_t<3, 3>(in, out, n, w, s);
    }
  } else if (Ds == 1) {
    switch (D) {
      case 2: return fold_t<1, 2>(in, out, n, w, s);
      case 3: return fold_t<1, 3>(in, out, n, w, s);
    }
  }
  throw Error("fold: extension degree must be 1, 2 or 3");
}

size_t fold_dev(int D, uint64_t* v, size_t n, const uint64_t* w, hipStream_t s) {
  return fold_into_dev(D, D, v, v, n, w, s);
}

// Both sumcheck vectors folded by the same challenge in one launch (a from Ds words
// into a_out, b in place).
template <int Ds, int D>
__global__ __launch_bounds__(RT) void k_fold2(const uint64_t* a_in, uint64_t* a_out, uint64_t* b, size_t half,
                                              size_t nhi, Ext<D> w, Ext<D> one_minus_w) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < half; i += (size_t)gridDim.x * blockDim.x) {
    st<D>(a_out, i, fold_at<Ds, D>(a_in, i, half, nhi, w, one_minus_w));
    st<D>(b, i, fold_at<D, D>(b, i, half, nhi, w, one_minus_w));
  }
}

template <int Ds, int D>
static size_t fold2_t(const uint64_t* a_in, uint64_t* a_out, uint64_t* b, size_t n, const uint64_t* w, hipStream_t s) {
  if (n <= 1) {
    fold_t<Ds, D>(a_in, a_out, n, w, s);
    return n;
  }
  size_t half = next_pow2(n) >> 1, nhi = n - half;
  Ext<D> ww = host_ext<D>(w);
  Ext<D> om = gl::esub<D>(gl::ext_base<D>(1), ww);
  ProfScope prof(kernel_name("k_fold2", Ds, D), s, 8.0 * ((double)(Ds + D) * n + 2.0 * D * half));
  k_fold2<Ds, D><<<grid_for(half), RT, 0, s>>>(a_in, a_out, b, half, nhi, ww, om);
  WHIR_HIP(hipGetLastError());
  return half;
}

size_t fold_both_dev(int Ds, int D, const uint64_t* a_in, uint64_t* a_out, uint64_t* b, size_t n, const uint64_t* w,
                     hipStream_t s) {
  if (Ds == D) {
    switch (D) {
      case 1: return fold2_t<1, 1>(a_in, a_out, b, n, w, s);
      case 2: return fold2_t<2, 2>(a_in, a_out, b, n, w, s);
      case 3: return fold2_t<3, 3>(a_in, a_out, b, n, w, s);
    }
  } else if (Ds == 1) {
    switch (D) {
      case 2: return fold2_t<1, 2>(a_in, a_out, b, n, w, s);
      case 3: return fold2_t<1, 3>(a_in, a_out, b, n, w, s);
    }
  }
  throw Error("fold: extension degree must be 1, 2 or 3");
}

// ------------------------------------------------------------------ fused fold + polynomial
// The value of lane CTRL[l] of each quad of lanes (quad_perm: two bits per lane l).
template <int CTRL>
__device__ __forceinline__ uint64_t quad_get(uint64_t v) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)v, CTRL, 0xf, 0xf, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(v >> 32), CTRL, 0xf, 0xf, true);
  return ((uint64_t)hi << 32) | lo;
}
template <int CTRL, int D>
__device__ __forceinline__ Ext<D> quad_get(const Ext<D>& v) {
  Ext<D> r;
#pragma unroll
  for (int d = 0; d < D; d++) r.c[d] = quad_get<CTRL>(v.c[d]);
  return r;
}
constexpr int quad_ctrl(int a, int b, int c, int d) { return a | b << 2 | c << 4 | d << 6; }

// Lane 0 of a pair of lanes: its own value; lane 1: its value less lane 0's.
template <int D>
__device__ __forceinline__ Ext<D> pair_factor(const Ext<D>& x) {
  const Ext<D> d = gl::esub<D>(x, quad_get<quad_ctrl(0, 0, 2, 2)>(x));
  Ext<D> p;
#pragma unroll
  for (int k = 0; k < D; k++) p.c[k] = (threadIdx.x & 1) ? d.c[k] : x.c[k];
  return p;
}

// Fold a (Ds words, into a_out) and b (in place) by w, then the round polynomial of
// the folded pair.  Folded length h = next_pow2(n)/2 (a power of two >= 2); the new
// pairs are (i, h/2 + i), h/2 = q.  Two lanes share a pair: lane l folds position l q + i of
// both vectors (it writes that position and reads it and h + it, so a_out may alias a_in when
// Ds == D), then lane 0 takes the product of the low halves and lane 1 that of the
// differences: half the code and twice the lanes of a lane per pair.  Fp2 on MI355X: 2^12
// elements 17 -> 12 us, 2^17 9.2 -> 7.5, 2^20 16 -> 17; long vectors move 5 TB/s either way.
template <int Ds, int D>
__global__ __launch_bounds__(1024) void k_fold_poly(const uint64_t* a_in, uint64_t* a_out, uint64_t* b, size_t h,
                                                  size_t nhi, Ext<D> w, Ext<D> om, uint64_t* parts,
                                                  MailboxSig sig) {
  gl::Wide acc[D];
  gl::wide_zero<D>(acc);
  const size_t q = h >> 1, l = threadIdx.x & 1;
#pragma unroll 1
  for (size_t i = (blockIdx.x * (size_t)blockDim.x + threadIdx.x) >> 1; i < q;
       i += ((size_t)gridDim.x * blockDim.x) >> 1) {
    const size_t t = l * q + i;
    const Ext<D> x = fold_at<Ds, D>(a_in, t, h, nhi, w, om), y = fold_at<D, D>(b, t, h, nhi, w, om);
    st<D>(a_out, t, x);
    st<D>(b, t, y);
    gl::emul_acc<D>(acc, pair_factor<D>(x), pair_factor<D>(y));
  }
  // A caller that has seen the flag may read the folded vectors on another stream: every
  // wave's stores are complete before it rises.
  if (sig.flag) __threadfence_system();
  Ext<D> v[1] = {gl::ext_reduce<D>(acc)};
  __shared__ uint64_t tot[2 * D];
  block_role_sum<D, 1, 2>(v, tot);
  store_words<2 * D>(threadIdx.x < 2 * D ? tot[threadIdx.x] : 0, parts + (size_t)blockIdx.x * 2 * D, sig);
}

// Block partials of one fold + polynomial pass: none when one block does it all.
static unsigned fold_poly_grid(size_t n) {
  if (n <= 2) return 1;
  const size_t q = (next_pow2(n) >> 1) >> 1;
  return q <= SMALL_PAIRS ? 1u : grid_for(2 * q);
}

// parts_buf: caller-provided room for the block partials (fold_poly_parts_words), or
// null to take it from the stream's pool.
template <int Ds, int D>
static size_t fold_poly_t(const uint64_t* a_in, uint64_t* a_out, uint64_t* b, size_t n, const uint64_t* w,
                          uint64_t* out, hipStream_t s, uint64_t* parts_buf = nullptr) {
  if (n <= 2) {
    // folded length <= 1: fold then the one-element polynomial
    size_t m = fold_t<Ds, D>(a_in, a_out, n, w, s);
    fold_t<D, D>(b, b, n, w, s);
    sc_poly<D, D>(a_out, b, m, out, s);
    return m;
  }
  size_t h = next_pow2(n) >> 1, nhi = n - h;
  Ext<D> ww = host_ext<D>(w);
  Ext<D> om = gl::esub<D>(gl::ext_base<D>(1), ww);
  const unsigned g = fold_poly_grid(n);
  DevBuf parts(g == 1 || parts_buf ? 0 : (size_t)g * 2 * D * 8, s);
  uint64_t* pp = parts_buf ? parts_buf : parts.as<uint64_t>();
  {
    ProfScope prof(kernel_name("k_fold_poly", Ds, D), s, 8.0 * ((Ds + D) * (double)n + 2.0 * D * h));
    k_fold_poly<Ds, D><<<g, g == 1 ? reduce_threads(h) : RT, 0, s>>>(a_in, a_out, b, h, nhi, ww, om, g == 1 ? out : pp,
                                        g == 1 ? mailbox_take(out) : MailboxSig{});
    WHIR_HIP(hipGetLastError());
  }
  if (g > 1) finish_reduce<D, 2>(pp, g, out, s);
  return h;
}

size_t fold_poly_parts_words(int D, size_t n) {
  const unsigned g = fold_poly_grid(n);
  return g == 1 ? 0 : (size_t)g * 2 * D;
}

size_t fold_and_poly_ws_dev(int D, uint64_t* a, uint64_t* b, size_t n, const uint64_t* w, uint64_t* out,
                            uint64_t* parts, hipStream_t s) {
  WHIR_REQUIRE(fold_poly_parts_words(D, n) == 0 || parts, "fold_and_poly: no room for the block partials");
  switch (D) {
    case 1: return fold_poly_t<1, 1>(a, a, b, n, w, out, s, parts);
    case 2: return fold_poly_t<2, 2>(a, a, b, n, w, out, s, parts);
    case 3: return fold_poly_t<3, 3>(a, a, b, n, w, out, s, parts);
  }
  throw Error("fold: extension degree must be 1, 2 or 3");
}

size_t fold_and_poly_mixed_dev(int Ds, int D, const uint64_t* a_in, uint64_t* a_out, uint64_t* b, size_t n,
                               const uint64_t* w, uint64_t* out, hipStream_t s) {
  if (Ds == D) {
    switch (D) {
      case 1: return fold_poly_t<1, 1>(a_in, a_out, b, n, w, out, s);
      case 2: return fold_poly_t<2, 2>(a_in, a_out, b, n, w, out, s);
      case 3: return fold_poly_t<3, 3>(a_in, a_out, b, n, w, out, s);
    }
  } else if (Ds == 1) {
    switch (D) {
      case 2: return fold_poly_t<1, 2>(a_in, a_out, b, n, w, out, s);
      case 3: return fold_poly_t<1, 3>(a_in, a_out, b, n, w, out, s);
    }
  }
  throw Error("fold: extension degree must be 1, 2 or 3");
}

size_t fold_and_poly_dev(int D, uint64_t* a, uint64_t* b, size_t n, const uint64_t* w, uint64_t* out,
                         hipStream_t s) {
  return fold_and_poly_mixed_dev(D, D, a, a, b, n, w, out, s);
}

// ------------------------------------------------------------------ two sumcheck rounds per pass
// Folding is linear in the challenge, so round k+1's polynomial is a polynomial in
// round k's challenge r whose coefficients the pass over round k's vectors can sum
// too.  For vectors x, y of length L = 4q (a power of two), h = L/2, dx_i = x_(h+i) -
// x_i and, after the fold by r, x'_i = x_i + r dx_i:
//   round k:    c0 = sum_(i<h) x_i y_i,  c2 = sum_(i<h) dx_i dy_i
//   round k+1:  c0' = S0 + r S1 + r^2 S2,  c2' = T0 + r T1 + r^2 T2, with (i < q)
//     S0 = sum x_i y_i,  S1 = sum (x_i dy_i + dx_i y_i),  S2 = sum dx_i dy_i,
//     U = x_(q+i) - x_i,  V = dx_(q+i) - dx_i:  T0 = sum Ux Uy,  T1 = sum (Ux Vy + Vx Uy),
//     T2 = sum Vx Vy
// (the same field values as folding first and summing after, the order of exact
// additions aside).  With FOLD the vectors are first folded by two pending challenges
// (r1, then r2) from length 4L, position t from t, L+t, 2L+t, 3L+t of the source, and
// written (a to a_out, b in place: a lane writes only its own position, the only one
// below L that it reads).  NS: sums per block, 8 (c0, c2, S0, S1, S2, T0, T1, T2) or 2
// (c0, c2).
//
// The position folded by r1 then r2 is bilinear in the challenges:
//   x0 + r1 (x2 - x0) + r2 (x1 - x0) + r1 r2 (x3 - x2 - x1 + x0)
// so its three products are summed unreduced and reduced once per coefficient.
template <int D>
struct Fold4 {
  Ext<D> r1, r2, r12;
};

template <int Ds, int D>
__device__ __forceinline__ Ext<D> fold_twice(const uint64_t* v, size_t t, size_t L, const Fold4<D>& f) {
  gl::Wide w[D];
  gl::wide_zero<D>(w);
  Ext<D> r;
  if constexpr (Ds == 1 && D > 1) {
    const uint64_t x0 = v[t], x1 = v[L + t], x2 = v[2 * L + t], x3 = v[3 * L + t];
    const uint64_t d1 = gl::sub(x2, x0), d2 = gl::sub(x1, x0), d3 = gl::sub(gl::sub(x3, x2), d2);
#pragma unroll
    for (int d = 0; d < D; d++) {
      gl::wide_mac(w[d], d1, f.r1.c[d]);
      gl::wide_mac(w[d], d2, f.r2.c[d]);
      gl::wide_mac(w[d], d3, f.r12.c[d]);
    }
    r = gl::ext_reduce<D>(w);
    r.c[0] = gl::add(r.c[0], x0);
  } else {
    const Ext<D> x0 = ldx<Ds, D>(v, t), x1 = ldx<Ds, D>(v, L + t), x2 = ldx<Ds, D>(v, 2 * L + t),
                 x3 = ldx<Ds, D>(v, 3 * L + t);
    const Ext<D> d2 = gl::esub<D>(x1, x0);
    gl::emul_acc<D>(w, gl::esub<D>(x2, x0), f.r1);
    gl::emul_acc<D>(w, d2, f.r2);
    gl::emul_acc<D>(w, gl::esub<D>(gl::esub<D>(x3, x2), d2), f.r12);
    r = gl::eadd<D>(gl::ext_reduce<D>(w), x0);
  }
  return r;
}

// Element i of a covector view: sum_k hi_k[i >> sh] lo_k[i & (2^sh - 1)].
template <int D>
__device__ __forceinline__ Ext<D> view_at(const CovView& v, size_t i) {
  const size_t h = i >> v.sh, l = i & (((size_t)1 << v.sh) - 1);
  Ext<D> r = gl::emul<D>(ld<D>(v.hi, h), ld<D>(v.lo, l));
  for (uint32_t k = 1; k < v.nt; k++)
    r = gl::eadd<D>(r, gl::emul<D>(ld<D>(v.hi, (size_t)k * v.nhi + h), ld<D>(v.lo, ((size_t)k << v.sh) + l)));
  return r;
}

constexpr int VIEW_MAX_TERMS = 4;

// The double fold alone, one output position per lane.  VIEW: b's folded values come from the
// unfolded view v: the block folds the high-table entries of its 256 positions (at most 128, a
// low table has at least two) into LDS first.
template <int Ds, int D, bool VIEW>
__global__ __launch_bounds__(RT) void k_fold4(const uint64_t* a_in, uint64_t* a_out, uint64_t* b, size_t L,
                                              Fold4<D> f, CovView v) {
  __shared__ uint64_t hi[VIEW ? VIEW_MAX_TERMS * (RT / 2) * D : 1];
  const size_t nhi = v.nhi >> 2;
  const uint32_t cnt = (uint32_t)(v.sh >= 8 ? 1 : nhi < (RT >> v.sh) ? nhi : RT >> v.sh);
  for (size_t t0 = blockIdx.x * (size_t)RT; t0 < L; t0 += (size_t)gridDim.x * RT) {
    const size_t t = t0 + threadIdx.x, h0 = t0 >> v.sh;
    if constexpr (VIEW) {
      for (uint32_t e = threadIdx.x; e < v.nt * cnt; e += RT)
        st<D>(hi, e, fold_twice<D, D>(v.hi + (size_t)(e / cnt) * v.nhi * D, h0 + e % cnt, nhi, f));
      __syncthreads();
    }
    if (t < L) {
      Ext<D> y;
      if constexpr (VIEW) {
        gl::Wide w[D];
        gl::wide_zero<D>(w);
        const size_t l = t & (((size_t)1 << v.sh) - 1);
#pragma unroll 1
        for (uint32_t k = 0; k < v.nt; k++)
          gl::emul_acc<D>(w, ld<D>(hi, k * cnt + (uint32_t)((t >> v.sh) - h0)), ld<D>(v.lo, ((size_t)k << v.sh) + l));
        y = gl::ext_reduce<D>(w);
      } else {
        y = fold_twice<D, D>(b, t, L, f);
      }
      st<D>(a_out, t, fold_twice<Ds, D>(a_in, t, L, f));
      st<D>(b, t, y);
    }
    if constexpr (VIEW) __syncthreads();
  }
}

// The second factor of a quad's lane: the quarter differences 2 - 0, 3 - 1, 3 - 2, 1 - 0,
// and for lane 3 in place of its own quarter (3 - 2) - (1 - 0) as the first factor.
template <int D>
__device__ __forceinline__ void quad_factors(const Ext<D>& x, Ext<D>& p, Ext<D>& q) {
  q = gl::esub<D>(quad_get<quad_ctrl(2, 3, 3, 1)>(x), quad_get<quad_ctrl(0, 1, 2, 0)>(x));
  const Ext<D> w = gl::esub<D>(quad_get<quad_ctrl(2, 2, 2, 2)>(q), q);
  const bool own = (threadIdx.x & 3) != 3;
#pragma unroll
  for (int d = 0; d < D; d++) p.c[d] = own ? x.c[d] : w.c[d];
}
// NS == 2: quarters 0 and 1, then the differences 2 - 0 and 3 - 1.
template <int D>
__device__ __forceinline__ Ext<D> quad_factor2(const Ext<D>& x) {
  const Ext<D> w = gl::esub<D>(x, quad_get<quad_ctrl(0, 1, 0, 1)>(x));
  Ext<D> p;
#pragma unroll
  for (int d = 0; d < D; d++) p.c[d] = (threadIdx.x & 2) ? w.c[d] : x.c[d];
  return p;
}

// Word e of the pass's sums from the quads' products (NS == 8: prod[(2 l + j) D + d], j = 0
// the first factors' product of lane l, j = 1 the second's; slot 8 is zero).  With
// P_l and Q_l for the two: c0 = P0 + P1, c2 = Q0 + Q1, S0 = P0, S1 = P2 - P0 - Q0,
// S2 = Q0, T0 = Q3, T1 = Q2 - Q3 - P3, T2 = P3.  The hex digits are the slots of each
// sum's terms, sum 0 in the lowest.
template <int D>
__device__ __forceinline__ uint64_t pair_sum_word(const uint64_t* prod, unsigned e) {
  const unsigned k = e / D, d = e % D;
  auto at = [&](uint32_t slots) { return prod[((slots >> (4 * k)) & 15) * D + d]; };
  return gl::sub(gl::sub(gl::add(at(0x65714010u), at(0x88888832u)), at(0x87880888u)), at(0x86881888u));
}

// Four lanes share the positions i, q+i, 2q+i, 3q+i: lane l folds and holds quarter l of x
// and y, and the quad forms eight products, two per lane, of which the eight sums are
// differences.  A lane that takes all four positions itself runs 34 extension products and
// the sums of eight values in 42 KB of code, against 8 KB here, and that is what the
// passes of a proof wait for once they are short: Fp2 with the fold on MI355X 20 -> 7.6 us
// from 2^6 to 2^14 elements, without it 12-19 -> 4-6.6.
template <int Ds, int D, bool FOLD, int NS>
__global__ __launch_bounds__(1024) void k_sc_pair(const uint64_t* a_in, uint64_t* a_out, uint64_t* b, size_t L,
                                                  Fold4<D> f, uint64_t* parts, MailboxSig sig) {
  constexpr int Dx = FOLD ? D : Ds, NP = NS == 8 ? 2 : 1;
  gl::Wide w[NP][D];
#pragma unroll
  for (int j = 0; j < NP; j++) gl::wide_zero<D>(w[j]);
  const size_t q = L >> 2, l = threadIdx.x & 3;
  const size_t step = ((size_t)gridDim.x * blockDim.x) >> 2;
#pragma unroll 1
  for (size_t i = (blockIdx.x * (size_t)blockDim.x + threadIdx.x) >> 2; i < q; i += step) {
    const size_t t = l * q + i;
    Ext<Dx> x;
    Ext<D> y;
    if constexpr (FOLD) {
      x = fold_twice<Ds, D>(a_in, t, L, f);
      y = fold_twice<D, D>(b, t, L, f);
      st<D>(a_out, t, x);
      st<D>(b, t, y);
    } else {
      x = ld<Dx>(a_in, t);
      y = ld<D>(b, t);
    }
    if constexpr (NS == 8) {
      Ext<Dx> px, qx;
      Ext<D> py, qy;
      quad_factors<Dx>(x, px, qx);
      quad_factors<D>(y, py, qy);
      mulx_acc<Dx, D>(w[0], px, py);
      mulx_acc<Dx, D>(w[1], qx, qy);
    } else {
      mulx_acc<Dx, D>(w[0], quad_factor2<Dx>(x), quad_factor2<D>(y));
    }
  }
  Ext<D> v[NP];
#pragma unroll
  for (int j = 0; j < NP; j++) v[j] = gl::ext_reduce<D>(w[j]);
  __shared__ uint64_t prod[9 * D];
  if (threadIdx.x < D) prod[8 * D + threadIdx.x] = 0;
  block_role_sum<D, NP, 4>(v, prod);
  const unsigned e = threadIdx.x;
  uint64_t word = 0;
  if (e < NS * D) {
    if constexpr (NS == 8) word = pair_sum_word<D>(prod, e);
    else word = gl::add(prod[e / D * 2 * D + e % D], prod[(e / D * 2 + 1) * D + e % D]);
  }
  store_words<NS * D>(word, parts + (size_t)blockIdx.x * NS * D, sig);
}

template <int D>
static Fold4<D> host_fold4(const uint64_t* r1, const uint64_t* r2) {
  Fold4<D> f{gl::ext_zero<D>(), gl::ext_zero<D>(), gl::ext_zero<D>()};
  if (r1 && r2) {
    f.r1 = host_ext<D>(r1);
    f.r2 = host_ext<D>(r2);
    f.r12 = gl::emul<D>(f.r1, f.r2);
  }
  return f;
}

template <int Ds, int D, bool VIEW>
static void fold4_t(const uint64_t* a_in, uint64_t* a_out, uint64_t* b, size_t L, const uint64_t* r1,
                    const uint64_t* r2, const CovView& v, hipStream_t s) {
  ProfScope prof(kernel_name("k_fold4", Ds, D), s, 8.0 * ((Ds + D) * 4.0 * L + 2.0 * D * L));
  k_fold4<Ds, D, VIEW><<<grid_for(L), RT, 0, s>>>(a_in, a_out, b, L, host_fold4<D>(r1, r2), v);
  WHIR_HIP(hipGetLastError());
}

// Up to this many quads a pass runs as one block of up to 1024 threads, which stores its
// sums itself; above, the second launch (3 us and the gap before it) costs less than the
// further turns on one CU.  Fp2 on MI355X: 256 quads without a fold 6.6 us in one block,
// 1024 13 us against 6.5; with the fold 64 quads 5.8 us, 256 10.6 against 7.4 and the launch.
static constexpr size_t SMALL_PAIRS_SUM = 256, SMALL_PAIRS_FOLD = 64;

template <int Ds, int D, bool FOLD, int NS>
static void sc_pair_t(const uint64_t* a_in, uint64_t* a_out, uint64_t* b, size_t L, const uint64_t* r1,
                      const uint64_t* r2, uint64_t* out, hipStream_t s) {
  const size_t q = L >> 2;
  const bool one = q <= (FOLD ? SMALL_PAIRS_FOLD : SMALL_PAIRS_SUM);
  const unsigned g = one ? 1u : grid_for(4 * q);
  DevBuf parts(one ? 0 : (size_t)g * NS * D * 8, s);
  {
    ProfScope prof(kernel_name(FOLD ? "k_sc_pair_fold" : "k_sc_pair", Ds, D), s,
                   FOLD ? 8.0 * ((Ds + D) * 4.0 * L + 2.0 * D * L) : 8.0 * (Ds + D) * (double)L);
    // one block stores the sums itself
    k_sc_pair<Ds, D, FOLD, NS><<<g, one ? reduce_threads(4 * q) : RT, 0, s>>>(
        a_in, a_out, b, L, host_fold4<D>(r1, r2), one ? out : parts.as<uint64_t>(),
        one ? mailbox_take(out) : MailboxSig{});
    WHIR_HIP(hipGetLastError());
  }
  if (!one) finish_reduce<D, NS>(parts.as<uint64_t>(), g, out, s);
}

template <int Ds, int D, bool VIEW>
static void sc_pair_d(int mode, const uint64_t* a_in, uint64_t* a_out, uint64_t* b, size_t L, const uint64_t* r1,
                      const uint64_t* r2, uint64_t* out, const CovView& v, hipStream_t s) {
  if constexpr (VIEW) {  // the double fold is the only pass that takes a view here
    fold4_t<Ds, D, true>(a_in, a_out, b, L, r1, r2, v, s);
  } else {
    switch (mode) {
      case 0: sc_pair_t<Ds, D, false, 8>(a_in, a_out, b, L, r1, r2, out, s); return;
      case 1: sc_pair_t<Ds, D, true, 8>(a_in, a_out, b, L, r1, r2, out, s); return;
      case 2: sc_pair_t<Ds, D, true, 2>(a_in, a_out, b, L, r1, r2, out, s); return;
      default: fold4_t<Ds, D, false>(a_in, a_out, b, L, r1, r2, v, s); return;
    }
  }
}

template <bool VIEW>
static void sc_pair_any(int mode, int Ds, int D, const uint64_t* a_in, uint64_t* a_out, uint64_t* b, size_t L,
                        const uint64_t* r1, const uint64_t* r2, uint64_t* out, const CovView& v, hipStream_t s) {
  WHIR_REQUIRE(L >= 4 && (L & (L - 1)) == 0, "sumcheck pair: length must be a power of two >= 4");
  if (Ds == D) {
    switch (D) {
      case 1: sc_pair_d<1, 1, VIEW>(mode, a_in, a_out, b, L, r1, r2, out, v, s); return;
      case 2: sc_pair_d<2, 2, VIEW>(mode, a_in, a_out, b, L, r1, r2, out, v, s); return;
      case 3: sc_pair_d<3, 3, VIEW>(mode, a_in, a_out, b, L, r1, r2, out, v, s); return;
    }
  } else if (Ds == 1) {
    switch (D) {
      case 2: sc_pair_d<1, 2, VIEW>(mode, a_in, a_out, b, L, r1, r2, out, v, s); return;
      case 3: sc_pair_d<1, 3, VIEW>(mode, a_in, a_out, b, L, r1, r2, out, v, s); return;
    }
  }
  throw Error("sumcheck pair: extension degree must be 1, 2 or 3");
}

void sumcheck_pair_dev(int mode, int Ds, int D, const uint64_t* a_in, uint64_t* a_out, uint64_t* b, size_t L,
                       const uint64_t* r1, const uint64_t* r2, uint64_t* out, hipStream_t s) {
  sc_pair_any<false>(mode, Ds, D, a_in, a_out, b, L, r1, r2, out, CovView{}, s);
}

// ------------------------------------------------------------------ view passes
// The sums of a pairs pass whose covector y is a view, factored by the view's blocks.
// With quarters x_a(i) = x(a L/4 + i), y_b likewise (i < L/4), every sum of the pass is
// a fixed bilinear combination of the 16 values G[a][b] = sum_i x_a(i) y_b(i), and
//   G[a][b] = sum_t sum_h hi_t[b Qb + h] P_(a,t)(h),  P_(a,t)(h) = sum_l x_a(h 2^sh + l) lo_t[l]
// (Qb = L/4 / 2^sh blocks per quarter): the inner products run against the low tables
// (a base-field x costs D products per term, summed as 128-bit values and reduced once
// per block), and the high tables enter once per block.  One GPU block per (a, h).
template <int Ds, int D, bool FOLD, int NT>
__global__ __launch_bounds__(RT) void k_view_pass(const uint64_t* a_in, uint64_t* a_out, size_t L, Fold4<D> f,
                                                  CovView v, uint64_t* hi_out, uint64_t* parts) {
  const size_t q = L >> 2, B = (size_t)1 << v.sh, Qb = q >> v.sh;
  const size_t a = blockIdx.x / Qb, h = blockIdx.x % Qb;
  const size_t base = a * q + h * B;
  // thread 4 t + b ends with term t of quarter b: its high-table factor is read here
  const unsigned et = threadIdx.x >> 2, eb = threadIdx.x & 3;
  Ext<D> hi = gl::ext_zero<D>();
  if (et < NT) {
    if constexpr (FOLD) {  // v is not folded yet: fold the entry, and keep it for the next pass
      const size_t nhi = v.nhi >> 2, e = eb * Qb + h;
      hi = fold_twice<D, D>(v.hi + et * v.nhi * D, e, nhi, f);
      if (a == 0) st<D>(hi_out, et * nhi + e, hi);
    } else {
      hi = ld<D>(v.hi, (size_t)et * v.nhi + eb * Qb + h);
    }
  }
  Ext<D> P[NT];
  if constexpr (!FOLD && Ds == 1) {
    gl::Wide W[NT][D];
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int d = 0; d < D; d++) W[t][d] = gl::Wide{0, 0, 0};
#pragma unroll 1
    for (size_t l = threadIdx.x; l < B; l += blockDim.x) {
      const uint64_t x = a_in[base + l];
      Ext<D> lo[NT];
#pragma unroll
      for (int t = 0; t < NT; t++) lo[t] = ld<D>(v.lo, ((size_t)t << v.sh) + l);
#pragma unroll
      for (int t = 0; t < NT; t++)
#pragma unroll
        for (int d = 0; d < D; d++) gl::wide_mac(W[t][d], x, lo[t].c[d]);
    }
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int d = 0; d < D; d++) P[t].c[d] = gl::wide_reduce(W[t][d]);
  } else {
    // extension x: the products' coefficients are summed unreduced, one reduction per
    // coefficient per block
    gl::Wide W[NT][D];
#pragma unroll
    for (int t = 0; t < NT; t++) gl::wide_zero<D>(W[t]);
#pragma unroll 1
    for (size_t l = threadIdx.x; l < B; l += blockDim.x) {
      const size_t p = base + l;
      Ext<D> lo[NT];
#pragma unroll
      for (int t = 0; t < NT; t++) lo[t] = ld<D>(v.lo, ((size_t)t << v.sh) + l);
      Ext<D> x;
      if constexpr (FOLD) {
        x = fold_twice<Ds, D>(a_in, p, L, f);
        st<D>(a_out, p, x);
      } else {
        x = ldx<Ds, D>(a_in, p);
      }
#pragma unroll
      for (int t = 0; t < NT; t++) gl::emul_acc<D>(W[t], x, lo[t]);
    }
#pragma unroll
    for (int t = 0; t < NT; t++) P[t] = gl::ext_reduce<D>(W[t]);
  }
  __shared__ uint64_t tot[NT * D];
  block_role_sum<D, NT, 1>(P, tot);
  if (threadIdx.x < 16) {
    Ext<D> g = gl::ext_zero<D>();
    if (et < NT) {
      Ext<D> x;
#pragma unroll
      for (int d = 0; d < D; d++) x.c[d] = tot[et * D + d];
      g = gl::emul<D>(hi, x);
    }
    if constexpr (NT > 1)
#pragma unroll 1
      for (int off = 4; off < 16; off <<= 1)
#pragma unroll
        for (int d = 0; d < D; d++) g.c[d] = gl::add(g.c[d], (uint64_t)__shfl_xor(g.c[d], off));
    if (threadIdx.x < 4) st<D>(parts, (size_t)blockIdx.x * 4 + eb, g);
  }
}

// Sums the blocks' G contributions and writes the pass's NS sums, through the eight
// products of the pairs kernel's quads: each is sum_ab c_a c_b G[a][b] for a vector c of
// 0, 1 and -1 over the quarters.  Thread 16 p + 4 a + b sums G[a][b] over every p-th h.
template <int D, int NS>
__global__ __launch_bounds__(1024) void k_view_reduce(const uint64_t* parts, size_t Qb, uint64_t* out,
                                                      MailboxSig sig) {
  __shared__ uint64_t G[16 * D], prod[9 * D];
  const unsigned a = (threadIdx.x >> 2) & 3, b = threadIdx.x & 3, e = threadIdx.x;
  Ext<D> v[1] = {gl::ext_zero<D>()};
  for (size_t h = threadIdx.x >> 4; h < Qb; h += blockDim.x >> 4)
    v[0] = gl::eadd<D>(v[0], ld<D>(parts, (a * Qb + h) * 4 + b));
  block_role_sum<D, 1, 16>(v, G);
  // c of products P0, Q0, P1, Q1, P2, Q2, P3, Q3 (slot order): the quarters with +1 and
  // those with -1, four bits each
  if (e < 9 * D) {
    const unsigned slot = e / D, d = e % D, sh = 4 * (slot & 7);
    const unsigned pos = slot < 8 ? (0x29848241u >> sh) & 15 : 0, neg = slot < 8 ? (0x16402010u >> sh) & 15 : 0;
    uint64_t r = 0;
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const unsigned pa = pos >> (i >> 2) & 1, na = neg >> (i >> 2) & 1, pb = pos >> (i & 3) & 1, nb = neg >> (i & 3) & 1;
      const uint64_t x = (pa | na) & (pb | nb) ? G[i * D + d] : 0;
      r = (pa ^ pb) & 1 ? gl::sub(r, x) : gl::add(r, x);
    }
    prod[e] = r;
  }
  __syncthreads();
  store_words<NS * D>(e < NS * D ? pair_sum_word<D>(prod, e) : 0, out, sig);
}

template <int Ds, int D>
static void view_pass_t(int mode, const uint64_t* a_in, uint64_t* a_out, size_t L, const uint64_t* r1,
                        const uint64_t* r2, const CovView& v, uint64_t* hi_out, uint64_t* out, hipStream_t s) {
  const size_t Qb = (L >> 2) >> v.sh;
  const unsigned blocks = (unsigned)(4 * Qb);
  DevBuf parts((size_t)blocks * 4 * D * 8, s);
  const Fold4<D> f = host_fold4<D>(r1, r2);
  {
    ProfScope prof(kernel_name(mode ? "k_view_pass_fold" : "k_view_pass", Ds, D), s,
                   mode ? 8.0 * (Ds * 4.0 * L + D * (double)L) : 8.0 * Ds * (double)L);
    uint64_t* pp = parts.as<uint64_t>();
    auto go = [&](auto nt) {
      constexpr int NT = decltype(nt)::value;
      if (mode == 0) k_view_pass<Ds, D, false, NT><<<blocks, RT, 0, s>>>(a_in, a_out, L, f, v, hi_out, pp);
      else k_view_pass<Ds, D, true, NT><<<blocks, RT, 0, s>>>(a_in, a_out, L, f, v, hi_out, pp);
    };
    switch (v.nt) {
      case 1: go(std::integral_constant<int, 1>{}); break;
      case 2: go(std::integral_constant<int, 2>{}); break;
      case 3: go(std::integral_constant<int, 3>{}); break;
      default: go(std::integral_constant<int, 4>{}); break;
    }
    WHIR_HIP(hipGetLastError());
  }
  if (mode == 2) k_view_reduce<D, 2><<<1, reduce_threads(16 * Qb), 0, s>>>(parts.as<uint64_t>(), Qb, out, mailbox_take(out));
  else k_view_reduce<D, 8><<<1, reduce_threads(16 * Qb), 0, s>>>(parts.as<uint64_t>(), Qb, out, mailbox_take(out));
  WHIR_HIP(hipGetLastError());
}

void sumcheck_pair_view_dev(int mode, int Ds, int D, const uint64_t* a_in, uint64_t* a_out, uint64_t* b, size_t L,
                            const uint64_t* r1, const uint64_t* r2, const CovView& v, uint64_t* hi_out, uint64_t* out,
                            hipStream_t s) {
  WHIR_REQUIRE(v.nt > 0 && v.nt <= VIEW_MAX_TERMS && v.hi && v.lo, "sumcheck pair: bad covector view");
  const size_t nhi = mode == 0 ? v.nhi : v.nhi >> 2;
  WHIR_REQUIRE(v.sh >= 1 && nhi > 0 && (nhi << v.sh) == L, "sumcheck pair: covector view length mismatch");
  if (mode == 3) {  // the double fold alone; it writes the view's values into b
    sc_pair_any<true>(mode, Ds, D, a_in, a_out, b, L, r1, r2, out, v, s);
    return;
  }
  WHIR_REQUIRE(nhi >= 4 && mode >= 0 && mode <= 2, "sumcheck pair: covector view too short for a view pass");
  WHIR_REQUIRE(mode == 0 || hi_out, "sumcheck pair: no room for the folded high tables");
  if (Ds == D) {
    switch (D) {
      case 1: return view_pass_t<1, 1>(mode, a_in, a_out, L, r1, r2, v, hi_out, out, s);
      case 2: return view_pass_t<2, 2>(mode, a_in, a_out, L, r1, r2, v, hi_out, out, s);
      case 3: return view_pass_t<3, 3>(mode, a_in, a_out, L, r1, r2, v, hi_out, out, s);
    }
  } else if (Ds == 1) {
    switch (D) {
      case 2: return view_pass_t<1, 2>(mode, a_in, a_out, L, r1, r2, v, hi_out, out, s);
      case 3: return view_pass_t<1, 3>(mode, a_in, a_out, L, r1, r2, v, hi_out, out, s);
    }
  }
  throw Error("sumcheck pair: extension degree must be 1, 2 or 3");
}

// ------------------------------------------------------------------ covector terms
// covector_dev adds (or writes) any mix of
//   eq terms     s_p eq(z_p, i)      eval_eq (src/algebra/multilinear.rs:170-190)
//   power terms  t_j x_j^i           geometric_accumulate (src/algebra/mod.rs:154-177)
// for every i < n in one pass over HBM.  Element layout: block b covers
// [b S, (b+1) S) with S = RT K; lane t owns i = b S + k RT + t (k < K), so loads
// and stores are coalesced.  k_cov_tables builds every table on the device:
//   eq:    hi_p[h] = s_p prod_{v < k1} (h_v ? z_v : 1 - z_v) over the first k1
//          variables (h_0 = MSB), lo_p[l] the same over the last k2; eq = hi lo.
//   power: T0[j nb + b] = t_j x_j^(b S), T1[j RT + t] = x_j^t, X[j] = x_j^RT.
//          Base-field points (upper coefficients zero; the STIR in-domain points)
//          keep T1 and X in the base field, so a step costs D base products
//          instead of an extension product.
struct CovPlan {
  size_t np, nv, k1, k2, nhi, nlo;        // eq terms
  size_t m_e, m_b, nb, S;                 // power terms: extension points, then base points
  size_t in_z, in_s, in_x, in_t;          // uploaded inputs (word offsets)
  size_t hi, lo, T0, T1e, Xe, T1b, Xb;    // tables (word offsets)
  size_t words, entries;
  size_t in_sq;                           // per extension point: x^(S 2^k) for k < kb, then x^(2^k)
  int kb;                                 // for k <= 8 (squares made on the host)
};

// Inputs of the covector tables (eq points and scalars, power points and scalars) up
// to this many words travel with the launch itself, which saves a staged copy and
// its launch; larger inputs are copied into the table buffer first.
static constexpr size_t COV_ARG_WORDS = 320;
// Larger inputs of short tables (few waves) are read in pinned host memory.
static constexpr size_t COV_IN_PLACE = (size_t)1 << 16;
struct CovIn {
  uint64_t w[COV_ARG_WORDS];
};

// Element i (D words) of the input region starting at word `off`: from device memory
// when dev is given, else from the launch's arguments.
template <int D>
__device__ __forceinline__ Ext<D> in_ld(const uint64_t* dev, const CovIn& arg, size_t off, size_t i) {
  Ext<D> r;
#pragma unroll
  for (int d = 0; d < D; d++) r.c[d] = dev ? dev[off + i * D + d] : arg.w[off + i * D + d];
  return r;
}

template <int D>
__global__ void k_cov_tables(uint64_t* buf, CovPlan L, const uint64_t* in_dev, CovIn in_arg) {
  size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (e >= L.entries) return;
  const size_t m = L.m_e + L.m_b;
  const size_t sec[7] = {L.np * L.nhi, L.np * L.nlo, m * L.nb, L.m_e * RT, L.m_e, L.m_b * RT, L.m_b};
  if (e < sec[0]) {
    const size_t p = e / L.nhi, h = e % L.nhi;
    Ext<D> v = in_ld<D>(in_dev, in_arg, L.in_s, p);
    for (size_t q = 0; q < L.k1; q++) {
      Ext<D> zq = in_ld<D>(in_dev, in_arg, L.in_z, p * L.nv + q);
      v = gl::emul<D>(v, ((h >> (L.k1 - 1 - q)) & 1) ? zq : gl::esub<D>(gl::ext_base<D>(1), zq));
    }
    st<D>(buf + L.hi, e, v);
    return;
  }
  e -= sec[0];
  if (e < sec[1]) {
    const size_t p = e / L.nlo, l = e % L.nlo;
    Ext<D> v = gl::ext_base<D>(1);
    for (size_t q = 0; q < L.k2; q++) {
      Ext<D> zq = in_ld<D>(in_dev, in_arg, L.in_z, p * L.nv + L.k1 + q);
      v = gl::emul<D>(v, ((l >> (L.k2 - 1 - q)) & 1) ? zq : gl::esub<D>(gl::ext_base<D>(1), zq));
    }
    st<D>(buf + L.lo, e, v);
    return;
  }
  e -= sec[1];
  // extension points take their powers from squares made on the host (a product per set
  // bit of the exponent instead of a square-and-multiply chain per lane)
  const size_t nsq = (size_t)L.kb + 9;
  if (e < sec[2]) {
    const size_t j = e / L.nb, b = e % L.nb;
    const Ext<D> t = in_ld<D>(in_dev, in_arg, L.in_t, j);
    Ext<D> v;
    if (j < L.m_e) {
      v = t;
      for (int k = 0; k < L.kb; k++)
        if ((b >> k) & 1) v = gl::emul<D>(v, in_ld<D>(in_dev, in_arg, L.in_sq, j * nsq + k));
    } else {
      v = gl::escale<D>(t, gl::pow(in_ld<D>(in_dev, in_arg, L.in_x, j).c[0], (uint64_t)b * L.S));
    }
    st<D>(buf + L.T0, e, v);
    return;
  }
  e -= sec[2];
  if (e < sec[3]) {
    const size_t j = e / RT, r = e % RT;
    Ext<D> v = gl::ext_base<D>(1);
    for (int k = 0; k < 8; k++)
      if ((r >> k) & 1) v = gl::emul<D>(v, in_ld<D>(in_dev, in_arg, L.in_sq, j * nsq + L.kb + k));
    st<D>(buf + L.T1e, e, v);
    return;
  }
  e -= sec[3];
  if (e < sec[4]) {
    static_assert(RT == 256, "x^RT is the square x^(2^8)");
    st<D>(buf + L.Xe, e, in_ld<D>(in_dev, in_arg, L.in_sq, e * nsq + L.kb + 8));
    return;
  }
  e -= sec[4];
  if (e < sec[5]) {
    buf[L.T1b + e] = gl::pow(in_ld<D>(in_dev, in_arg, L.in_x, L.m_e + e / RT).c[0], e % RT);
    return;
  }
  e -= sec[5];
  buf[L.Xb + e] = gl::pow(in_ld<D>(in_dev, in_arg, L.in_x, L.m_e + e).c[0], RT);
}

template <int D, int K>
__global__ __launch_bounds__(RT) void k_cov(uint64_t* acc, size_t n, int accumulate, const uint64_t* buf,
                                            CovPlan L) {
  const size_t b = blockIdx.x;
  const size_t i0 = b * (size_t)RT * K + threadIdx.x;
  Ext<D> sum[K];
#pragma unroll
  for (int k = 0; k < K; k++) sum[k] = gl::ext_zero<D>();
  if (L.np) {
    const size_t mask = L.nlo - 1;
    // term and query loops unrolled so several iterations' loads share one wait
#pragma unroll 2
    for (size_t p = 0; p < L.np; p++) {
      const uint64_t* hi = buf + L.hi + p * L.nhi * D;
      const uint64_t* lo = buf + L.lo + p * L.nlo * D;
#pragma unroll
      for (int k = 0; k < K; k++) {
        const size_t i = i0 + (size_t)k * RT;
        if (i < n) sum[k] = gl::eadd<D>(sum[k], gl::emul<D>(ld<D>(hi, i >> L.k2), ld<D>(lo, i & mask)));
      }
    }
  }
#pragma unroll 2
  for (size_t j = 0; j < L.m_e; j++) {
    Ext<D> p = gl::emul<D>(ld<D>(buf + L.T0, j * L.nb + b), ld<D>(buf + L.T1e, j * RT + threadIdx.x));
    const Ext<D> step = ld<D>(buf + L.Xe, j);
#pragma unroll
    for (int k = 0; k < K; k++) {
      sum[k] = gl::eadd<D>(sum[k], p);
      if (k + 1 < K) p = gl::emul<D>(p, step);
    }
  }
#pragma unroll 4
  for (size_t j = 0; j < L.m_b; j++) {
    Ext<D> p = gl::escale<D>(ld<D>(buf + L.T0, (L.m_e + j) * L.nb + b), buf[L.T1b + j * RT + threadIdx.x]);
    const uint64_t step = buf[L.Xb + j];
#pragma unroll
    for (int k = 0; k < K; k++) {
      sum[k] = gl::eadd<D>(sum[k], p);
      if (k + 1 < K) p = gl::escale<D>(p, step);
    }
  }
#pragma unroll
  for (int k = 0; k < K; k++) {
    const size_t i = i0 + (size_t)k * RT;
    if (i < n) st<D>(acc, i, accumulate ? gl::eadd<D>(ld<D>(acc, i), sum[k]) : sum[k]);
  }
}

// Elements per lane: the largest K (up to a per-degree maximum) that still gives
// >= 1024 blocks.
// The largest K is 16 for Fp, 8 for Fp2 and 4 for Fp3 (fewer accumulators per lane,
// more waves: the d = 24 Fp2 covector 0.198 -> 0.177 ms, the d = 26 Fp3 ones 3.53 ->
// 2.82 ms on MI355X); WHIR_COV_KMAX2 / WHIR_COV_KMAX3 override them.
static int cov_k(size_t n, int D) {
  static const int kmax2 = [] {
    const char* e = getenv("WHIR_COV_KMAX2");
    return e ? atoi(e) : 8;
  }();
  static const int kmax3 = [] {
    const char* e = getenv("WHIR_COV_KMAX3");
    return e ? atoi(e) : 4;
  }();
  int K = D == 3 ? kmax3 : (D == 2 ? kmax2 : 16);
  while (K > 1 && (n + (size_t)RT * K - 1) / ((size_t)RT * K) < 1024) K >>= 1;
  return K;
}

// ------------------------------------------------------------------ many power terms
// sum_j t_j x_j^i for many points (the STIR terms of a round: the OOD samples and the
// in-domain queries), factored by i = 256 h + l:
//   t_j x_j^i = HI_j[h] * LO_j[l],  HI_j[h] = t_j x_j^(256 h),  LO_j[l] = x_j^l.
// Lane l of a block holds LO_j[l] for one point at a time and adds it times the block's
// K high values (the same for every lane: scalar loads) into 128-bit sums, reduced once
// per element at the end; in-domain points lie in the base field, so their terms cost D
// 64x64 products per element instead of an extension scale and an addition.  In-domain
// points come as exponents of the domain's root of unity (x = w_N^e), so each of their
// table entries is one twiddle-table product (exponents multiply mod N); the few OOD
// points' tables are powers computed in short runs.
constexpr int GEO_RUN = 8;      // consecutive OOD-point table entries per thread
struct GeoPlan {
  size_t m_e, m_b, H;           // OOD points first, then in-domain points; H = n / 256
  size_t in_x, in_t, in_e;      // inputs: OOD points (m_e D words), scalars (all points),
                                // in-domain exponents (m_b words)
  size_t hi, lo_e, lo_b;        // tables: HI (m H elements), LO of OOD points (m_e 256
                                // elements), LO of in-domain points (m_b 256 words)
  uint64_t N;                   // domain size of the in-domain points (a power of two)
  size_t in_sq;                 // inputs: per OOD point, x^(256 2^k) for k < kh, then x^(2^k)
  int kh;                       // for k < 8 (squares made on the host)
};

template <int D>
__global__ void k_geo_tables(uint64_t* buf, GeoPlan L, const uint64_t* in_dev, CovIn in_arg, TwTable tw) {
  const size_t runs_hi = (L.H + GEO_RUN - 1) / GEO_RUN;
  const size_t sec[4] = {L.m_b * L.H, L.m_b * 256, L.m_e * runs_hi, L.m_e * (256 / GEO_RUN)};
  size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (e < sec[0]) {  // in-domain HI: t_j w^(256 h e_j)
    const size_t j = e / L.H, h = e % L.H;
    const uint64_t ej = in_dev ? in_dev[L.in_e + j] : in_arg.w[L.in_e + j];
    const uint64_t x = tw_at(tw, ((uint64_t)h * 256 * ej) & (L.N - 1));
    st<D>(buf + L.hi, (L.m_e + j) * L.H + h, gl::escale<D>(in_ld<D>(in_dev, in_arg, L.in_t, L.m_e + j), x));
    return;
  }
  e -= sec[0];
  if (e < sec[1]) {  // in-domain LO: w^(l e_j)
    const size_t j = e / 256, l = e % 256;
    const uint64_t ej = in_dev ? in_dev[L.in_e + j] : in_arg.w[L.in_e + j];
    buf[L.lo_b + e] = tw_at(tw, ((uint64_t)l * ej) & (L.N - 1));
    return;
  }
  e -= sec[1];
  const size_t nsq = (size_t)L.kh + 8;  // squares per OOD point
  if (e < sec[2]) {  // OOD HI in runs: t_j x_j^(256 h), x^(256 h0) from the squares of x^256
    const size_t j = e / runs_hi, h0 = (e % runs_hi) * GEO_RUN;
    const Ext<D> step = in_ld<D>(in_dev, in_arg, L.in_sq, j * nsq);
    Ext<D> v = in_ld<D>(in_dev, in_arg, L.in_t, j);
    for (int k = 0; k < L.kh; k++)
      if ((h0 >> k) & 1) v = gl::emul<D>(v, in_ld<D>(in_dev, in_arg, L.in_sq, j * nsq + k));
    for (size_t h = h0; h < h0 + GEO_RUN && h < L.H; h++) {
      st<D>(buf + L.hi, j * L.H + h, v);
      v = gl::emul<D>(v, step);
    }
    return;
  }
  e -= sec[2];
  if (e >= sec[3]) return;
  const size_t j = e / (256 / GEO_RUN), l0 = (e % (256 / GEO_RUN)) * GEO_RUN;  // OOD LO in runs: x_j^l
  const Ext<D> x = in_ld<D>(in_dev, in_arg, L.in_x, j);
  Ext<D> v = gl::ext_base<D>(1);
  for (int k = 0; k < 8; k++)
    if ((l0 >> k) & 1) v = gl::emul<D>(v, in_ld<D>(in_dev, in_arg, L.in_sq, j * nsq + L.kh + k));
  for (size_t l = l0; l < l0 + GEO_RUN; l++) {
    st<D>(buf + L.lo_e, j * 256 + l, v);
    v = gl::emul<D>(v, x);
  }
}

// K rows h per block, the points dealt out to QG groups of 256 lanes (each group sums every
// QG-th point, then group 0 adds the groups' reduced sums from LDS).  A lane's work is a
// serial sum over the points, so a short vector needs the groups to fill the chip; the rows
// a lane shares its LO loads among matter only once it is full.
template <int D, int K, int QG>
__global__ __launch_bounds__(256 * QG) void k_geo(uint64_t* acc, size_t n, int accumulate, const uint64_t* buf, GeoPlan L) {
  __shared__ uint64_t part[QG > 1 ? (QG - 1) * 256 * K * D : 1];
  const size_t l = threadIdx.x & 255, h0 = (size_t)blockIdx.x * K;
  const size_t q = QG > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
  gl::Wide W[K][D];
#pragma unroll
  for (int k = 0; k < K; k++)
#pragma unroll
    for (int d = 0; d < D; d++) W[k][d] = gl::Wide{0, 0, 0};
  const uint64_t* hi = buf + L.hi;
  // in-domain points: HI (extension) x LO (base), D products per row.  The query loops
  // are unrolled so that the loads of several queries share one wait (short vectors run
  // a few waves per SIMD, with little else to hide the latency).
#pragma unroll 4
  for (size_t j = q; j < L.m_b; j += QG) {
    const uint64_t lo = buf[L.lo_b + j * 256 + l];
    const uint64_t* hj = hi + ((L.m_e + j) * L.H + h0) * D;
#pragma unroll
    for (int k = 0; k < K; k++)
#pragma unroll
      for (int d = 0; d < D; d++) gl::wide_mac(W[k][d], hj[k * D + d], lo);
  }
  Ext<D> sum[K];
#pragma unroll
  for (int k = 0; k < K; k++)
#pragma unroll
    for (int d = 0; d < D; d++) sum[k].c[d] = gl::wide_reduce(W[k][d]);
  // OOD points: full extension products
#pragma unroll 2
  for (size_t j = q; j < L.m_e; j += QG) {
    const Ext<D> lo = ld<D>(buf + L.lo_e, j * 256 + l);
#pragma unroll
    for (int k = 0; k < K; k++) sum[k] = gl::eadd<D>(sum[k], gl::emul<D>(ld<D>(hi, j * L.H + h0 + k), lo));
  }
  if constexpr (QG > 1) {
    if (q) {
#pragma unroll
      for (int k = 0; k < K; k++)
#pragma unroll
        for (int d = 0; d < D; d++) part[(((q - 1) * K + k) * D + d) * 256 + l] = sum[k].c[d];
    }
    __syncthreads();
    if (q) return;
#pragma unroll
    for (int g = 0; g < QG - 1; g++)
#pragma unroll
      for (int k = 0; k < K; k++)
#pragma unroll
        for (int d = 0; d < D; d++) sum[k].c[d] = gl::add(sum[k].c[d], part[((g * K + k) * D + d) * 256 + l]);
  }
#pragma unroll
  for (int k = 0; k < K; k++) {
    const size_t i = (h0 + k) * 256 + l;
    if (i < n) st<D>(acc, i, accumulate ? gl::eadd<D>(ld<D>(acc, i), sum[k]) : sum[k]);
  }
}

template <int D>
static void geo_terms_t(uint64_t* acc, size_t n, bool accumulate, const uint64_t* scalars, const uint64_t* ext_points,
                        size_t m_e, const uint64_t* exps, size_t m_b, int logN, hipStream_t s) {
  GeoPlan L{};
  L.H = n / 256;
  L.m_e = m_e;
  L.m_b = m_b;
  L.N = (uint64_t)1 << logN;
  const size_t m = m_e + m_b;
  std::vector<uint64_t> in;
  L.in_x = 0;
  in.insert(in.end(), ext_points, ext_points + m_e * D);
  L.in_t = in.size();
  in.insert(in.end(), scalars, scalars + m * D);
  L.in_e = in.size();
  in.insert(in.end(), exps, exps + m_b);
  // Squares for the OOD tables: x^(256 2^k) for k < kh (2^kh >= H) and x^(2^k) for k < 8,
  // so a lane forms its run's first power from the bits of its index.
  L.kh = 0;
  while (((size_t)1 << L.kh) < L.H) L.kh++;
  L.in_sq = in.size();
  for (size_t j = 0; j < m_e; j++) {
    Ext<D> x;
    for (int d = 0; d < D; d++) x.c[d] = ext_points[j * D + d];
    Ext<D> lo[8];
    for (int k = 0; k < 8; k++) {
      lo[k] = x;
      x = gl::emul<D>(x, x);
    }
    for (int k = 0; k < L.kh; k++) {  // x is x_j^256 here
      in.insert(in.end(), x.c, x.c + D);
      x = gl::emul<D>(x, x);
    }
    for (int k = 0; k < 8; k++) in.insert(in.end(), lo[k].c, lo[k].c + D);
  }
  const bool by_arg = in.size() <= COV_ARG_WORDS;
  const size_t entries = m_b * L.H + m_b * 256 + m_e * ((L.H + GEO_RUN - 1) / GEO_RUN) + m_e * (256 / GEO_RUN);
  const uint64_t* in_place = nullptr;
  if (!by_arg && entries <= COV_IN_PLACE) in_place = (const uint64_t*)stage_async(in.data(), in.size() * 8, s);
  size_t w = by_arg || in_place ? 0 : in.size();
  L.hi = w;   w += m * L.H * D;
  L.lo_e = w; w += m_e * 256 * D;
  L.lo_b = w; w += m_b * 256;
  DevBuf buf(w * 8, s);
  CovIn args{};
  if (by_arg) std::copy(in.begin(), in.end(), args.w);
  else if (!in_place) upload_async(buf.ptr, in.data(), in.size() * 8, s);
  const TwTable tw = m_b ? twiddles(logN) : TwTable{};
  k_geo_tables<D><<<blocks_for(entries, RT), RT, 0, s>>>(
      buf.as<uint64_t>(), L, by_arg ? nullptr : in_place ? in_place : buf.as<uint64_t>(), args, tw);
  WHIR_HIP(hipGetLastError());
  ProfScope prof(kernel_name("k_geo", D), s, 8.0 * D * (accumulate ? 2.0 : 1.0) * (double)n);
  const int ac = accumulate ? 1 : 0;
  const uint64_t* tb = buf.as<uint64_t>();
  // The shapes measured at n = 2^10, 2^16, 2^18, 2^20 (Fp2, all STIR launches of a proof):
  // four rows and one group 74 (k_cov), 70, 96, 173 us; four rows and two groups -, -, 71, 167;
  // one row and four groups 15, 18, 61, 309.
  if (L.H >= 2048 && L.H % 4 == 0) k_geo<D, 4, 2><<<(unsigned)(L.H / 4), 512, 0, s>>>(acc, n, ac, tb, L);
  else k_geo<D, 1, 4><<<(unsigned)L.H, 1024, 0, s>>>(acc, n, ac, tb, L);
  WHIR_HIP(hipGetLastError());
}

// The same terms over a short vector in one launch: a block makes its own factors in LDS
// (HI of its row h, one twiddle product per in-domain point; for an OOD point x^l as the
// product of x^(16 a) and x^b, l = 16 a + b), deals the points to the groups of LW lanes that
// its 1024 threads form, takes LO of an in-domain point straight from the twiddle tables, and
// adds the groups in LDS.
// Its rule: up to 64 blocks of 16 to 256 lanes (every block reads all the inputs, from host
// memory), 256 lanes above; points times lanes at most 2^14, since a lane's turns over the
// points gather from the twiddle tables.  Fp2 on MI355X against the table launch, k_geo and the
// 3 us between them: 2^10 elements, 180 points 9 us against 25; 2^12, 85 points 8 against 20;
// 2^13, 85 points 20 against 29; 2^16, 45 points 12 against 20; but 2^14, 85 points 32 against 30.
constexpr size_t GEO_SHORT_N = (size_t)1 << 16, GEO_SHORT_WORK = (size_t)1 << 14;
constexpr size_t GEO_SHORT_M = 256, GEO_SHORT_ME = 4, GEO_SHORT_IN = 1536;
struct GeoShort {
  uint64_t N;
  uint32_t m_e, m_b, lw;          // points; LW = 2^lw
  uint32_t in_t, in_sq, nsq, words;  // inputs: exponents, then scalars, then per OOD point x^(2^k), k < nsq
};

template <int D>
__global__ __launch_bounds__(1024) void k_geo_short(uint64_t* acc, size_t n, int accumulate, GeoShort L,
                                                    const uint64_t* in_dev, CovIn in_arg, TwTable tw) {
  __shared__ uint64_t in[GEO_SHORT_IN], hi[GEO_SHORT_M * D], ab[GEO_SHORT_ME * 32 * D], part[D][1024];
  const uint32_t tid = threadIdx.x;
  const uint64_t h = blockIdx.x;
  for (uint32_t i = tid; i < L.words; i += 1024) in[i] = in_dev ? in_dev[i] : in_arg.w[i];
  __syncthreads();
  for (uint32_t e = tid; e < L.m_b + L.m_e * 33; e += 1024) {
    if (e < L.m_b) {
      const uint64_t x = tw_at(tw, ((h << L.lw) * in[e]) & (L.N - 1));
      st<D>(hi, L.m_e + e, gl::escale<D>(ld<D>(in + L.in_t, L.m_e + e), x));
    } else {
      const uint32_t j = (e - L.m_b) / 33, i = (e - L.m_b) % 33;
      Ext<D> v = i == 32 ? ld<D>(in + L.in_t, j) : gl::ext_base<D>(1);
      const uint64_t* sq = in + L.in_sq + j * L.nsq * D;
#pragma unroll 1
      for (uint64_t x = i == 32 ? h << L.lw : i < 16 ? i << 4 : i - 16; x; x &= x - 1)
        v = gl::emul<D>(v, ld<D>(sq, __builtin_ctzll(x)));
      if (i == 32) st<D>(hi, j, v);
      else st<D>(ab, j * 32 + i, v);
    }
  }
  __syncthreads();
  const uint32_t LW = 1u << L.lw, l = tid & (LW - 1), G = 1024u >> L.lw;
  gl::Wide W[D];
  gl::wide_zero<D>(W);
#pragma unroll 4
  for (uint32_t j = tid >> L.lw; j < L.m_b; j += G) {
    const uint64_t lo = tw_at(tw, (l * in[j]) & (L.N - 1));
#pragma unroll
    for (int d = 0; d < D; d++) gl::wide_mac(W[d], hi[(L.m_e + j) * D + d], lo);
  }
  // (from the last group on: the first ones have the odd in-domain points)
#pragma unroll 1
  for (uint32_t j = G - 1 - (tid >> L.lw); j < L.m_e; j += G)
    gl::emul_acc<D>(W, ld<D>(hi, j), gl::emul<D>(ld<D>(ab, j * 32 + (l >> 4)), ld<D>(ab, j * 32 + 16 + (l & 15))));
  const Ext<D> sum = gl::ext_reduce<D>(W);
#pragma unroll
  for (int d = 0; d < D; d++) part[d][tid] = sum.c[d];
#pragma unroll 1
  for (uint32_t s = 512; s >= LW; s >>= 1) {
    __syncthreads();
    if (tid < s)
#pragma unroll
      for (int d = 0; d < D; d++) part[d][tid] = gl::add(part[d][tid], part[d][tid + s]);
  }
  const size_t i = (h << L.lw) + l;
  if (tid < LW && i < n) {
    Ext<D> v;
#pragma unroll
    for (int d = 0; d < D; d++) v.c[d] = part[d][tid];
    st<D>(acc, i, accumulate ? gl::eadd<D>(ld<D>(acc, i), v) : v);
  }
}

template <int D>
static bool geo_short_t(uint64_t* acc, size_t n, bool accumulate, const uint64_t* scalars, const uint64_t* ext_points,
                        size_t m_e, const uint64_t* exps, size_t m_b, int logN, hipStream_t s) {
  const size_t m = m_e + m_b;
  GeoShort L{};
  for (L.nsq = 8; ((size_t)1 << L.nsq) < n;) L.nsq++;
  L.words = (uint32_t)std::min<size_t>(m_b + m * D + m_e * L.nsq * D, ~0u);
  if (n > GEO_SHORT_N || m > GEO_SHORT_M || m_e > GEO_SHORT_ME || L.words > GEO_SHORT_IN) return false;
  L.N = (uint64_t)1 << logN;
  L.m_e = (uint32_t)m_e;
  L.m_b = (uint32_t)m_b;
  L.in_t = (uint32_t)m_b;
  L.in_sq = (uint32_t)(m_b + m * D);
  for (L.lw = 4; L.lw < 8 && ((size_t)64 << L.lw) < n;) L.lw++;
  if ((m << L.lw) > GEO_SHORT_WORK) return false;
  const size_t H = (n + ((size_t)1 << L.lw) - 1) >> L.lw;
  std::vector<uint64_t> in(exps, exps + m_b);
  in.insert(in.end(), scalars, scalars + m * D);
  for (size_t j = 0; j < m_e; j++) {
    Ext<D> x;
    for (int d = 0; d < D; d++) x.c[d] = ext_points[j * D + d];
    for (uint32_t k = 0; k < L.nsq; k++) {
      in.insert(in.end(), x.c, x.c + D);
      x = gl::emul<D>(x, x);
    }
  }
  CovIn args{};
  const uint64_t* in_dev = nullptr;
  DevBuf buf;
  if (in.size() <= COV_ARG_WORDS) {
    std::copy(in.begin(), in.end(), args.w);
  } else if (!(in_dev = (const uint64_t*)stage_async(in.data(), in.size() * 8, s))) {
    buf = DevBuf(in.size() * 8, s);
    upload_async(buf.ptr, in.data(), in.size() * 8, s);
    in_dev = buf.as<uint64_t>();
  }
  const TwTable tw = m_b ? twiddles(logN) : TwTable{};
  ProfScope prof(kernel_name("k_geo_short", D), s, 8.0 * D * (accumulate ? 2.0 : 1.0) * (double)n);
  k_geo_short<D><<<(unsigned)H, 1024, 0, s>>>(acc, n, accumulate ? 1 : 0, L, in_dev, args, tw);
  WHIR_HIP(hipGetLastError());
  return true;
}

// WHIR_COV_GEO=0 keeps power terms on the one-pass kernel (for comparison).
static bool geo_path_enabled() {
  static const bool on = [] {
    const char* e = getenv("WHIR_COV_GEO");
    return !e || atoi(e) != 0;
  }();
  return on;
}

template <int D>
static void covector_t(uint64_t* acc, size_t n, bool accumulate, const uint64_t* eq_points,
                       const uint64_t* eq_scalars, size_t np, size_t nv, const uint64_t* scalars,
                       const uint64_t* points, size_t m, hipStream_t s) {
  if (!n) return;
  WHIR_REQUIRE(!np || n == ((size_t)1 << nv), "eval_eq: the covector length must be 2^(number of variables)");
  if (!np && !m) {
    if (!accumulate) fill_zero(acc, n * D * 8, s);
    return;
  }
  const int K = cov_k(n, D);
  CovPlan L{};
  L.np = np;
  L.nv = np ? nv : 0;
  L.k1 = L.nv / 2;
  L.k2 = L.nv - L.k1;
  L.nhi = (size_t)1 << L.k1;
  L.nlo = (size_t)1 << L.k2;
  L.S = (size_t)RT * K;
  L.nb = (n + L.S - 1) / L.S;
  // Extension points first, then points that lie in the base field.
  std::vector<size_t> order_e, order_b;
  for (size_t j = 0; j < m; j++) {
    bool base = D > 1;
    for (int d = 1; d < D; d++) base = base && points[j * D + d] == 0;
    (base ? order_b : order_e).push_back(j);
  }
  L.m_e = order_e.size();
  L.m_b = order_b.size();
  std::vector<uint64_t> in;
  L.in_z = 0;
  if (np) in.insert(in.end(), eq_points, eq_points + np * L.nv * D);
  L.in_s = in.size();
  if (np) in.insert(in.end(), eq_scalars, eq_scalars + np * D);
  L.in_x = in.size();
  for (size_t j : order_e) in.insert(in.end(), points + j * D, points + (j + 1) * D);
  for (size_t j : order_b) in.insert(in.end(), points + j * D, points + (j + 1) * D);
  L.in_t = in.size();
  for (size_t j : order_e) in.insert(in.end(), scalars + j * D, scalars + (j + 1) * D);
  for (size_t j : order_b) in.insert(in.end(), scalars + j * D, scalars + (j + 1) * D);
  // Squares of the extension points: x^(S 2^k) for k < kb (2^kb >= nb), then x^(2^k)
  // for k <= 8.
  L.kb = 0;
  while (((size_t)1 << L.kb) < L.nb) L.kb++;
  L.in_sq = in.size();
  for (size_t j : order_e) {
    Ext<D> x;
    for (int d = 0; d < D; d++) x.c[d] = points[j * D + d];
    Ext<D> xs = gl::epow<D>(x, L.S);
    for (int k = 0; k < L.kb; k++) {
      in.insert(in.end(), xs.c, xs.c + D);
      xs = gl::emul<D>(xs, xs);
    }
    for (int k = 0; k <= 8; k++) {
      in.insert(in.end(), x.c, x.c + D);
      x = gl::emul<D>(x, x);
    }
  }
  // Small inputs go with the launch; larger ones are copied to the front of the buffer.
  const bool by_arg = in.size() <= COV_ARG_WORDS;
  L.entries = np * (L.nhi + L.nlo) + m * L.nb + L.m_e * (RT + 1) + L.m_b * (RT + 1);
  const uint64_t* in_place = nullptr;
  if (!by_arg && L.entries <= COV_IN_PLACE) in_place = (const uint64_t*)stage_async(in.data(), in.size() * 8, s);
  size_t w = by_arg || in_place ? 0 : in.size();
  L.hi = w;  w += np * L.nhi * D;
  L.lo = w;  w += np * L.nlo * D;
  L.T0 = w;  w += m * L.nb * D;
  L.T1e = w; w += L.m_e * RT * D;
  L.Xe = w;  w += L.m_e * D;
  L.T1b = w; w += L.m_b * RT;
  L.Xb = w;  w += L.m_b;
  L.words = w;
  DevBuf buf(L.words * 8, s);
  CovIn args{};
  if (by_arg) std::copy(in.begin(), in.end(), args.w);
  else if (!in_place) upload_async(buf.ptr, in.data(), in.size() * 8, s);
  k_cov_tables<D><<<blocks_for(L.entries, RT), RT, 0, s>>>(
      buf.as<uint64_t>(), L, by_arg ? nullptr : in_place ? in_place : buf.as<uint64_t>(), args);
  WHIR_HIP(hipGetLastError());
  ProfScope prof(kernel_name("k_cov", D, K), s, 8.0 * D * (accumulate ? 2.0 : 1.0) * (double)n);
  const unsigned g = (unsigned)L.nb;
  const int ac = accumulate ? 1 : 0;
  uint64_t* tb = buf.as<uint64_t>();
  switch (K) {
    case 16: k_cov<D, 16><<<g, RT, 0, s>>>(acc, n, ac, tb, L); break;
    case 8: k_cov<D, 8><<<g, RT, 0, s>>>(acc, n, ac, tb, L); break;
    case 4: k_cov<D, 4><<<g, RT, 0, s>>>(acc, n, ac, tb, L); break;
    case 2: k_cov<D, 2><<<g, RT, 0, s>>>(acc, n, ac, tb, L); break;
    default: k_cov<D, 1><<<g, RT, 0, s>>>(acc, n, ac, tb, L); break;
  }
  WHIR_HIP(hipGetLastError());
}

void covector_dev(int D, uint64_t* acc, size_t n, bool accumulate, const uint64_t* eq_points,
                  const uint64_t* eq_scalars, size_t np, size_t nv, const uint64_t* scalars, const uint64_t* points,
                  size_t m, hipStream_t s) {
  switch (D) {
    case 1: covector_t<1>(acc, n, accumulate, eq_points, eq_scalars, np, nv, scalars, points, m, s); break;
    case 2: covector_t<2>(acc, n, accumulate, eq_points, eq_scalars, np, nv, scalars, points, m, s); break;
    case 3: covector_t<3>(acc, n, accumulate, eq_points, eq_scalars, np, nv, scalars, points, m, s); break;
    default: throw Error("covector: extension degree must be 1, 2 or 3");
  }
}

// ------------------------------------------------------------------ covector views
// Table layout in the buffer: the uploaded inputs (when they do not travel with the
// launch), then the nt hi tables, then the nt lo tables.  Terms: np eq terms (points
// z_p of nv elements, scalars s_p), then m geometric terms (points x_j, scalars t_j):
//   eq:  hi[h] = s_p prod_{q < nv-sh} (h_q ? z_q : 1 - z_q)   (h_0 = MSB of h)
//        lo[l] = prod_{q < sh} (l_q ? z_(nv-sh+q) : 1 - z_(nv-sh+q))
//   geo: hi[h] = t_j x_j^(h 2^sh), lo[l] = x_j^l.
struct CovViewPlan {
  size_t np, m, nv, sh, nhi, nlo;
  size_t in_z, in_s, in_t, in_sq;  // input offsets (words); in_sq: per point x^(2^b), b < nv
  size_t hi, lo;                   // table offsets (words)
};

// A block makes 256 consecutive entries of one table.  An entry is a product over the bits of
// its index, (bit ? f1 : f0) per bit, the scalar in front for a hi table: the block has the
// pairs (f0, f1) in LDS, forms the 16 products of each half of the low byte and the product of
// the bits above it, and an entry is two products (the tables of 2^14 coefficients on MI355X
// 4.1 us; 9.0 when every entry was a chain of its own products or a power by squaring).
template <int D>
__global__ __launch_bounds__(256) void k_covview_tables(uint64_t* buf, CovViewPlan L, const uint64_t* in_dev,
                                                        CovIn in_arg) {
  __shared__ uint64_t f[64 * 2 * D], half[32 * D], top[D];
  const uint32_t tid = threadIdx.x;
  const size_t bh = (L.nhi + 255) >> 8, bl = (L.nlo + 255) >> 8;
  const size_t k = blockIdx.x / (bh + bl), c = blockIdx.x % (bh + bl);
  const bool hi = c < bh;
  const size_t chunk = hi ? c : c - bh, size = hi ? L.nhi : L.nlo;
  const int bits = (int)(hi ? L.nv - L.sh : L.sh);
  if (tid < (uint32_t)bits) {  // bit tid of the index
    Ext<D> f0 = gl::ext_base<D>(1), f1;
    if (k < L.np) {
      f1 = in_ld<D>(in_dev, in_arg, L.in_z, k * L.nv + (hi ? L.nv - L.sh : L.nv) - 1 - tid);
      f0 = gl::esub<D>(f0, f1);
    } else {
      f1 = in_ld<D>(in_dev, in_arg, L.in_sq, (k - L.np) * L.nv + (hi ? L.sh : 0) + tid);
    }
    st<D>(f, 2 * tid, f0);
    st<D>(f, 2 * tid + 1, f1);
  }
  Ext<D> v = gl::ext_base<D>(1);
  if (tid == 64 && hi) v = k < L.np ? in_ld<D>(in_dev, in_arg, L.in_s, k) : in_ld<D>(in_dev, in_arg, L.in_t, k - L.np);
  __syncthreads();
  if (tid < 32 || tid == 64) {  // bits 0..3, bits 4..7, and from 8 on
    const size_t e = tid < 32 ? tid & 15 : chunk;
    const int b0 = tid < 16 ? 0 : tid < 32 ? 4 : 8, b1 = tid < 32 ? b0 + 4 : bits;
#pragma unroll 1
    for (int b = b0; b < b1 && b < bits; b++) v = gl::emul<D>(v, ld<D>(f, 2 * b + ((e >> (b - b0)) & 1)));
    st<D>(tid < 32 ? half : top, tid < 32 ? tid : 0, v);
  }
  __syncthreads();
  const size_t e = (chunk << 8) + tid;
  if (e < size)
    st<D>(buf + (hi ? L.hi : L.lo), k * size + e,
          gl::emul<D>(gl::emul<D>(ld<D>(half, tid & 15), ld<D>(half, 16 + (tid >> 4))), ld<D>(top, 0)));
}

size_t covview_words(int D, size_t np, size_t m, size_t nv) {
  const size_t sh = nv - nv / 2, nt = np + m;
  return (np * nv + np + m + m * nv) * D + nt * (((size_t)1 << (nv - sh)) + ((size_t)1 << sh)) * D;
}

template <int D>
static CovView covview_build_t(uint64_t* buf, size_t nv, const uint64_t* eq_points, const uint64_t* eq_scalars,
                               size_t np, const uint64_t* scalars, const uint64_t* points, size_t m, hipStream_t s) {
  CovViewPlan L{};
  L.np = np;
  L.m = m;
  L.nv = nv;
  L.sh = nv - nv / 2;
  L.nhi = (size_t)1 << (nv - L.sh);
  L.nlo = (size_t)1 << L.sh;
  std::vector<uint64_t> in;
  L.in_z = 0;
  in.insert(in.end(), eq_points, eq_points + np * nv * D);
  L.in_s = in.size();
  in.insert(in.end(), eq_scalars, eq_scalars + np * D);
  L.in_t = in.size();
  in.insert(in.end(), scalars, scalars + m * D);
  L.in_sq = in.size();
  for (size_t j = 0; j < m; j++) {
    Ext<D> x;
    for (int d = 0; d < D; d++) x.c[d] = points[j * D + d];
    for (size_t b = 0; b < nv; b++) {
      in.insert(in.end(), x.c, x.c + D);
      x = gl::emul<D>(x, x);
    }
  }
  const bool by_arg = in.size() <= COV_ARG_WORDS;
  const size_t nt = np + m;
  L.hi = in.size();  // the input region stays reserved either way (covview_words)
  L.lo = L.hi + nt * L.nhi * D;
  CovIn args{};
  if (by_arg) std::copy(in.begin(), in.end(), args.w);
  else upload_async(buf, in.data(), in.size() * 8, s);
  const size_t blocks = nt * (((L.nhi + 255) >> 8) + ((L.nlo + 255) >> 8));
  k_covview_tables<D><<<(unsigned)blocks, 256, 0, s>>>(buf, L, by_arg ? nullptr : buf, args);
  WHIR_HIP(hipGetLastError());
  CovView v;
  v.hi = buf + L.hi;
  v.lo = buf + L.lo;
  v.nt = (uint32_t)nt;
  v.sh = (uint32_t)L.sh;
  v.nhi = L.nhi;
  return v;
}

CovView covview_build_dev(int D, uint64_t* buf, size_t nv, const uint64_t* eq_points, const uint64_t* eq_scalars,
                          size_t np, const uint64_t* scalars, const uint64_t* points, size_t m, hipStream_t s) {
  WHIR_REQUIRE(np + m > 0 && nv >= 2 && nv < 63, "covector view: needs terms and 2 <= nv < 63");
  switch (D) {
    case 1: return covview_build_t<1>(buf, nv, eq_points, eq_scalars, np, scalars, points, m, s);
    case 2: return covview_build_t<2>(buf, nv, eq_points, eq_scalars, np, scalars, points, m, s);
    case 3: return covview_build_t<3>(buf, nv, eq_points, eq_scalars, np, scalars, points, m, s);
    default: throw Error("covector view: extension degree must be 1, 2 or 3");
  }
}

template <int D>
__global__ void k_covview_write(CovView v, uint64_t* out, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    st<D>(out, i, view_at<D>(v, i));
}

void covview_write_dev(int D, const CovView& v, uint64_t* out, size_t n, hipStream_t s) {
  WHIR_REQUIRE(n <= ((size_t)v.nhi << v.sh), "covector view: output longer than the view");
  if (!n) return;
  const unsigned g = grid_for(n);
  switch (D) {
    case 1: k_covview_write<1><<<g, RT, 0, s>>>(v, out, n); break;
    case 2: k_covview_write<2><<<g, RT, 0, s>>>(v, out, n); break;
    case 3: k_covview_write<3><<<g, RT, 0, s>>>(v, out, n); break;
    default: throw Error("covector view: extension degree must be 1, 2 or 3");
  }
  WHIR_HIP(hipGetLastError());
}

void covector_stir_dev(int D, uint64_t* acc, size_t n, bool accumulate, const uint64_t* scalars,
                       const uint64_t* ext_points, size_t m_e, const uint64_t* exps, const uint64_t* points, size_t m_b,
                       int logN, hipStream_t s) {
  const size_t m = m_e + m_b;
  if (geo_path_enabled() && m && n && logN <= 62) {
    bool done = false;
    switch (D) {
      case 1: done = geo_short_t<1>(acc, n, accumulate, scalars, ext_points, m_e, exps, m_b, logN, s); break;
      case 2: done = geo_short_t<2>(acc, n, accumulate, scalars, ext_points, m_e, exps, m_b, logN, s); break;
      case 3: done = geo_short_t<3>(acc, n, accumulate, scalars, ext_points, m_e, exps, m_b, logN, s); break;
    }
    if (done) return;
  }
  if (!geo_path_enabled() || m < 8 || !n || n % 256 || logN > 62) {
    // the one-pass kernel, with every point as a field element (in-domain points lifted)
    std::vector<uint64_t> pts(ext_points, ext_points + m_e * D);
    for (size_t j = 0; j < m_b; j++) {
      pts.push_back(points[j]);
      for (int d = 1; d < D; d++) pts.push_back(0);
    }
    covector_dev(D, acc, n, accumulate, nullptr, nullptr, 0, 0, scalars, pts.data(), m, s);
    return;
  }
  switch (D) {
    case 1: geo_terms_t<1>(acc, n, accumulate, scalars, ext_points, m_e, exps, m_b, logN, s); break;
    case 2: geo_terms_t<2>(acc, n, accumulate, scalars, ext_points, m_e, exps, m_b, logN, s); break;
    case 3: geo_terms_t<3>(acc, n, accumulate, scalars, ext_points, m_e, exps, m_b, logN, s); break;
    default: throw Error("covector: extension degree must be 1, 2 or 3");
  }
}

void eval_eq_dev(int D, uint64_t* acc, const uint64_t* point, size_t k, const uint64_t* scalar, hipStream_t s) {
  covector_dev(D, acc, (size_t)1 << k, true, point, scalar, 1, k, nullptr, nullptr, 0, s);
}

void geometric_accumulate_dev(int D, uint64_t* acc, size_t n, const uint64_t* scalars, const uint64_t* points,
                              size_t m, hipStream_t s) {
  covector_dev(D, acc, n, true, nullptr, nullptr, 0, 0, scalars, points, m, s);
}

// ------------------------------------------------------------------ univariate evaluation
// mixed_univariate_evaluate (src/algebra/mod.rs:105-129) of several vectors at several
// points.  A block of T <= 256 threads takes G segments of T K elements; thread t holds
//   a_t = sum_k c_(k T + t) x^(k T)   over all its k, by Horner's rule in x^(T K) over the
// segments, and within a segment against the powers x^(k T), k < K, which are the same for
// every thread and come with the launch (through LDS: the arguments are read in one go
// while the elements are on their way).  A segment's products and the Horner step are
// summed unreduced and reduced once.  Then one wave forms sum_t a_t x^t: Horner's rule in
// x^64 over the waves, and a tree of lo + x^(2^i) hi over its lanes, so no thread makes a
// power of its own; the block's sum times x^(first element) is its part.  A short vector
// waits for the code as much as for the arithmetic, so the loops stay loops: 4 KB against
// 27 KB of a lane that steps its own power through sixteen unrolled elements.
static constexpr int UNI_MP = 4;   // points per launch
static constexpr int UNI_MV = 16;  // vectors per launch, times points (both rounded up to a power of two)
static constexpr int UNI_PW = 32;  // squares x^(2^b): vectors of up to 2^32 elements
static constexpr int UNI_K = 16;   // elements per thread of a segment of k_uni_many

// Per point: the squares x^(2^b), then the powers x^(k T).  MP points (at most 3.6 KB, 0.7 to
// 1.1 KB for the usual single point: the launch copies them).
template <int D, int K, int MP>
struct UniArgs {
  static constexpr int POINT = (UNI_PW + K) * D;
  const uint64_t* c[UNI_MV];
  uint64_t w[MP * POINT];
};
struct UniGrid {
  size_t n, G;
  int lt;      // T = 2^lt threads, 64 <= T <= 256
  int nv, m;   // slots per vector (points rounded up to a power of two), points
  int rows;    // slots per block of parts (vectors rounded up, times nv)
};

template <int D>
__device__ __forceinline__ Ext<D> uni_arg(const uint64_t* w, int i) {
  Ext<D> r;
#pragma unroll
  for (int d = 0; d < D; d++) r.c[d] = w[i * D + d];
  return r;
}

// Blocks z take a vector, blocks y a slot.  rows == 0: the block is the only one and stores
// its points' values to parts in order (sig).
template <int Ds, int D, int K, int MP>
__global__ __launch_bounds__(RT) void k_uni(UniArgs<D, K, MP> A, UniGrid U, uint64_t* parts, MailboxSig sig) {
  constexpr int POINT = (UNI_PW + K) * D;
  static_assert(K == 4 || K == 8, "k_uni: the step x^(T K) is one of the squares");
  __shared__ uint64_t arg[POINT], sum[RT * D], first[D];
  const uint64_t* c = A.c[blockIdx.z];
  const unsigned T = blockDim.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = T >> 6;
  const size_t S = (size_t)T * K, base = blockIdx.x * U.G * S;
  const int step_bit = U.lt + (K == 4 ? 2 : 3);
#pragma unroll 1
  for (int j = blockIdx.y; j < U.nv; j += gridDim.y) {
    Ext<Ds> cv[K];
    auto load = [&](size_t g) {
      const size_t i0 = base + g * S + threadIdx.x;
#pragma unroll
      for (int k = 0; k < K; k++) {
        const size_t i = i0 + (size_t)k * T;
        cv[k] = i < U.n ? ld<Ds>(c, i) : gl::ext_zero<Ds>();
      }
    };
    load(U.G - 1);
#pragma unroll 1
    for (int i = threadIdx.x; i < POINT; i += T) arg[i] = A.w[j * POINT + i];
    __syncthreads();
    Ext<D> acc = gl::ext_zero<D>();
    // many segments: scalar registers hold the factors best (the loop's factors in vector
    // registers halve the waves per SIMD)
    const uint64_t* aj = K == 4 ? arg : A.w + j * POINT;
#pragma unroll 1
    for (size_t g = U.G;;) {
      gl::Wide w[D];
      gl::wide_zero<D>(w);
#pragma unroll
      for (int d = 0; d < Ds; d++) w[d].lo = cv[0].c[d];
      if (g != U.G) gl::emul_acc<D>(w, acc, uni_arg<D>(aj, step_bit));
#pragma unroll
      for (int k = 1; k < K; k++) {
        const Ext<D> p = uni_arg<D>(aj, UNI_PW + k);
        if constexpr (Ds == D) {
          gl::emul_acc<D>(w, cv[k], p);
        } else {
#pragma unroll
          for (int d = 0; d < D; d++) gl::wide_mac(w[d], cv[k].c[0], p.c[d]);
        }
      }
      acc = gl::ext_reduce<D>(w);
      if (--g == 0) break;
      load(g - 1);
    }
    st<D>(sum, threadIdx.x, acc);
    __syncthreads();
    // wave 0 sums the threads' values while wave 1 forms x^base (several blocks: T = 256)
    if (base && wave == 1) {
      Ext<D> f = gl::ext_base<D>(1);
#pragma unroll 1
      for (size_t e = base; e; e &= e - 1) f = gl::emul<D>(f, uni_arg<D>(arg, __builtin_ctzll(e)));
      if (lane == 0) st<D>(first, 0, f);
    }
    Ext<D> v = gl::ext_zero<D>();
    if (wave == 0) {
#pragma unroll 1
      for (int w = waves - 1; w >= 0; w--)
        v = gl::eadd<D>(ld<D>(sum, w * 64 + lane), gl::emul<D>(v, uni_arg<D>(arg, 6)));
#pragma unroll 1
      for (int bit = 5; bit >= 0; bit--) {
        Ext<D> hi;
#pragma unroll
        for (int d = 0; d < D; d++) hi.c[d] = __shfl_xor(v.c[d], 1 << bit);
        v = gl::eadd<D>(v, gl::emul<D>(hi, uni_arg<D>(arg, bit)));  // right in lanes below 2^bit
      }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      if (base) v = gl::emul<D>(v, ld<D>(first, 0));
      if (j >= U.m) v = gl::ext_zero<D>();
      if (U.rows > 0) st<D>(parts, blockIdx.x * (size_t)U.rows + (size_t)blockIdx.z * U.nv + j, v);
      else if (j < U.m) st<D>(parts, j, v);
    }
  }
  if (sig.flag && threadIdx.x == 0) mailbox_raise(sig);  // the thread that stored the values
}

// The vectors' values from the blocks' parts (R slots per block, nv per vector): value j of
// vector z goes to out[z ms + j].
template <int D, int R>
__global__ __launch_bounds__(1024) void k_uni_reduce(const uint64_t* parts, size_t nparts, int nv, int m, int ms,
                                                     int count, uint64_t* out, MailboxSig sig) {
  __shared__ uint64_t tot[R * D];
  Ext<D> v[1] = {gl::ext_zero<D>()};
  for (size_t e = threadIdx.x; e < nparts * R; e += blockDim.x)
    if ((int)(e % R) < nv * count) v[0] = gl::eadd<D>(v[0], ld<D>(parts, e));
  block_role_sum<D, 1, R>(v, tot);
  const int r = threadIdx.x / D, z = r / nv, j = r % nv;
  if (threadIdx.x < R * D && z < count && j < m) out[(z * ms + j) * D + threadIdx.x % D] = tot[threadIdx.x];
  if (sig.flag) {
    __syncthreads();  // every word is stored before thread 0 raises the flag
    if (threadIdx.x == 0) mailbox_raise(sig);
  }
}

static int next_pow2_int(int n) {
  int p = 1;
  while (p < n) p <<= 1;
  return p;
}

// One launch (and its reduction): count vectors at m points, values to out[z ms + j].
template <int Ds, int D, int K, int MP>
static void uni_launch(const uint64_t* const* c, int count, size_t n, const uint64_t* xs, int m, uint64_t* out,
                       int ms, bool last, hipStream_t s) {
  UniArgs<D, K, MP> A{};
  UniGrid U{};
  std::copy(c, c + count, A.c);
  U.n = n;
  U.m = m;
  U.nv = next_pow2_int(m);
  U.lt = 8;
  if (K == 4)
    while (U.lt > 6 && n <= ((size_t)K << (U.lt - 1))) U.lt--;
  const size_t S = (size_t)K << U.lt, segs = (n + S - 1) / S;
  U.G = (segs + MAX_BLOCKS - 1) / MAX_BLOCKS;
  const size_t nb = (segs + U.G - 1) / U.G;
  WHIR_REQUIRE(n <= ((size_t)1 << UNI_PW), "univariate: vector too long");
  for (int j = 0; j < m; j++) {
    Ext<D> p, k = gl::ext_base<D>(1);
    for (int d = 0; d < D; d++) p.c[d] = xs[j * D + d];
    Ext<D> xt = k;
    for (int b = 0; b < UNI_PW; b++) {
      std::copy(p.c, p.c + D, &A.w[j * A.POINT + b * D]);
      if (b == U.lt) xt = p;
      p = gl::emul<D>(p, p);
    }
    for (int i = 0; i < K; i++, k = gl::emul<D>(k, xt)) std::copy(k.c, k.c + D, &A.w[j * A.POINT + (UNI_PW + i) * D]);
  }
  const bool one = nb == 1 && count == 1;
  U.rows = one ? 0 : next_pow2_int(count) * U.nv;
  DevBuf parts(one ? 0 : nb * U.rows * D * 8, s);
  {
    ProfScope prof(kernel_name("k_uni", Ds, D), s, 8.0 * Ds * (double)n * count);
    const dim3 grid((unsigned)nb, one ? 1u : (unsigned)U.nv, (unsigned)count);
    k_uni<Ds, D, K, MP><<<grid, 1u << U.lt, 0, s>>>(A, U, one ? out : parts.as<uint64_t>(),
                                                   one && last ? mailbox_take(out) : MailboxSig{});
    WHIR_HIP(hipGetLastError());
  }
  if (one) return;
  const MailboxSig sig = last ? mailbox_take(out) : MailboxSig{};
  const unsigned th = reduce_threads(nb * U.rows);
  const uint64_t* pp = parts.as<uint64_t>();
  switch (U.rows) {
    case 1: k_uni_reduce<D, 1><<<1, th, 0, s>>>(pp, nb, U.nv, m, ms, count, out, sig); break;
    case 2: k_uni_reduce<D, 2><<<1, th, 0, s>>>(pp, nb, U.nv, m, ms, count, out, sig); break;
    case 4: k_uni_reduce<D, 4><<<1, th, 0, s>>>(pp, nb, U.nv, m, ms, count, out, sig); break;
    case 8: k_uni_reduce<D, 8><<<1, th, 0, s>>>(pp, nb, U.nv, m, ms, count, out, sig); break;
    default: k_uni_reduce<D, 16><<<1, th, 0, s>>>(pp, nb, U.nv, m, ms, count, out, sig); break;
  }
  WHIR_HIP(hipGetLastError());
}

// Up to this many elements a segment is 4 per thread, which spreads a short vector over the
// most CUs; above, 8 per thread halve the Horner steps (2^20 base elements at an Fp2 point on
// MI355X 13.2 us against 14.1).  2^24 take 42 us (3.2 TB/s; 54 with a table of powers read
// beside the elements), 2^12 Fp2 7 us (15 with a power chain per lane).
static constexpr size_t UNI_SHORT = (size_t)1 << 18;

template <int Ds, int D>
static void uni_t(const uint64_t* const* vecs, size_t count, size_t n, const uint64_t* xs, size_t m, uint64_t* out,
                  hipStream_t s) {
  if (!n) {
    fill_zero(out, count * m * D * 8, s);
    return;
  }
  // Fp3 with K = 8: two points fill the launch's arguments
  const size_t gm = std::min<size_t>(m, D == 3 && n > UNI_SHORT ? 2 : UNI_MP);
  const size_t gv = UNI_MV / next_pow2_int((int)gm);
  for (size_t v = 0; v < count; v += gv)
    for (size_t j = 0; j < m; j += gm) {
      const size_t kv = std::min(gv, count - v), kj = std::min(gm, m - j);
      const bool last = v + kv == count && j + kj == m;
      uint64_t* o = out + (v * m + j) * D;
      auto go = [&](auto k, auto mp) {
        uni_launch<Ds, D, decltype(k)::value, decltype(mp)::value>(vecs + v, (int)kv, n, xs + j * D, (int)kj, o, (int)m,
                                                                   last, s);
      };
      using One = std::integral_constant<int, 1>;
      using K4 = std::integral_constant<int, 4>;
      using K8 = std::integral_constant<int, 8>;
      if (n <= UNI_SHORT) kj == 1 ? go(K4{}, One{}) : go(K4{}, std::integral_constant<int, UNI_MP>{});
      else kj == 1 ? go(K8{}, One{}) : go(K8{}, std::integral_constant<int, D == 3 ? 2 : UNI_MP>{});
    }
}

void univariate_eval_many_dev(int Ds, int D, const uint64_t* const* vecs, size_t count, size_t n, const uint64_t* xs,
                              size_t m, uint64_t* out, hipStream_t s) {
  if (!m || !count) return;
  if (Ds == 1) {
    switch (D) {
      case 1: uni_t<1, 1>(vecs, count, n, xs, m, out, s); return;
      case 2: uni_t<1, 2>(vecs, count, n, xs, m, out, s); return;
      case 3: uni_t<1, 3>(vecs, count, n, xs, m, out, s); return;
    }
  } else if (Ds == D) {
    switch (D) {
      case 2: uni_t<2, 2>(vecs, count, n, xs, m, out, s); return;
      case 3: uni_t<3, 3>(vecs, count, n, xs, m, out, s); return;
    }
  }
  throw Error("univariate_evaluate: unsupported degrees");
}

// ------------------------------------------------------------------ batched univariate evaluation
// Evaluations f_e(x_e) = sum_i c_e[i] x_e^i of many base-field vectors (e < count),
// each at its own point, in three launches for the whole batch: tables (x_e^q for
// q < S and x_e^(b S) per segment, from host-computed squarings), segment sums (one
// block per segment of S = RT * UNI_K coefficients, found by a binary search over the
// jobs' first segments), and one reducing block per job.
struct UniJobDev {
  const uint64_t* c;
  uint64_t n, nb, blk0, P, B;
};

template <int D>
__global__ void k_uni_many_tables(uint64_t* buf, const UniJobDev* jobs, const uint64_t* pw, size_t count,
                                  size_t entries_per_job_p) {
  const size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  const size_t S = (size_t)RT * UNI_K;
  // entries: count * S powers x^q, then every job's segment offsets x^(b S)
  size_t j, i;
  uint64_t ex;
  uint64_t* dst;
  if (e < count * S) {
    j = e / S;
    i = e % S;
    ex = i;
    dst = buf + jobs[j].P + i * D;
  } else {
    size_t r = e - count * S;
    // job of segment entry r: jobs are laid out with their segment counts in order
    size_t lo = 0, hi = count;
    while (hi - lo > 1) {
      const size_t mid = (lo + hi) / 2;
      if (jobs[mid].blk0 <= r) lo = mid; else hi = mid;
    }
    j = lo;
    if (r >= jobs[j].blk0 + jobs[j].nb) return;
    i = r - jobs[j].blk0;
    ex = (uint64_t)i * S;
    dst = buf + jobs[j].B + i * D;
  }
  (void)entries_per_job_p;
  Ext<D> acc = gl::ext_base<D>(1);
  for (int b = 0; ex; b++, ex >>= 1)
    if (ex & 1) acc = gl::emul<D>(acc, ld<D>(pw, (j * UNI_PW + b)));
  st<D>(dst, 0, acc);
}

template <int D>
__global__ __launch_bounds__(RT) void k_uni_many(const UniJobDev* jobs, size_t count, const uint64_t* buf,
                                                 uint64_t* parts) {
  const size_t b = blockIdx.x;
  size_t lo = 0, hi = count;
  while (hi - lo > 1) {
    const size_t mid = (lo + hi) / 2;
    if (jobs[mid].blk0 <= b) lo = mid; else hi = mid;
  }
  const UniJobDev J = jobs[lo];
  const size_t seg = b - J.blk0;
  const size_t S = (size_t)RT * UNI_K;
  const size_t i0 = seg * S + threadIdx.x;
  Ext<D> acc[1] = {gl::ext_zero<D>()};
#pragma unroll
  for (int k = 0; k < UNI_K; k++) {
    const size_t i = i0 + (size_t)k * RT;
    if (i >= J.n) break;
    const size_t q = (size_t)k * RT + threadIdx.x;
    acc[0] = gl::eadd<D>(acc[0], gl::escale<D>(ld<D>(buf + J.P, q), J.c[i]));
  }
  acc[0] = gl::emul<D>(acc[0], ld<D>(buf + J.B, seg));
  block_reduce_store<D, 1>(acc, parts + b * D);
}

template <int D>
__global__ __launch_bounds__(RT) void k_uni_many_reduce(const UniJobDev* jobs, const uint64_t* parts,
                                                        uint64_t* out) {
  const UniJobDev J = jobs[blockIdx.x];
  Ext<D> v[1] = {gl::ext_zero<D>()};
  for (size_t p = threadIdx.x; p < J.nb; p += blockDim.x) v[0] = gl::eadd<D>(v[0], ld<D>(parts, J.blk0 + p));
  block_reduce_store<D, 1>(v, out + blockIdx.x * D);
}

template <int D>
static void uni_batch_t(const UniJob* jobs, size_t count, uint64_t* out, hipStream_t s) {
  const size_t S = (size_t)RT * UNI_K;
  std::vector<UniJobDev> dj(count);
  size_t blk = 0, words = 0;
  for (size_t j = 0; j < count; j++) {
    WHIR_REQUIRE(jobs[j].n > 0, "univariate batch: empty vector");
    dj[j].c = jobs[j].coeffs;
    dj[j].n = jobs[j].n;
    dj[j].nb = (jobs[j].n + S - 1) / S;
    WHIR_REQUIRE((uint64_t)(dj[j].nb - 1) * S < ((uint64_t)1 << UNI_PW), "univariate batch: vector too long");
    dj[j].blk0 = blk;
    blk += dj[j].nb;
  }
  for (size_t j = 0; j < count; j++) {
    dj[j].P = words;
    words += S * D;
  }
  for (size_t j = 0; j < count; j++) {
    dj[j].B = words;
    words += dj[j].nb * D;
  }
  // squarings x^(2^b), b < UNI_PW, per job
  std::vector<uint64_t> pw(count * UNI_PW * D);
  for (size_t j = 0; j < count; j++) {
    Ext<D> p;
    for (int d = 0; d < D; d++) p.c[d] = jobs[j].x[d];
    for (int b = 0; b < UNI_PW; b++) {
      for (int d = 0; d < D; d++) pw[(j * UNI_PW + b) * D + d] = p.c[d];
      p = gl::emul<D>(p, p);
    }
  }
  const size_t job_words = (count * sizeof(UniJobDev) + 7) / 8;
  DevBuf in(job_words * 8 + pw.size() * 8, s), buf(words * 8, s), parts(blk * D * 8, s);
  {
    std::vector<uint64_t> host(job_words + pw.size());
    memcpy(host.data(), dj.data(), count * sizeof(UniJobDev));
    std::copy(pw.begin(), pw.end(), host.begin() + job_words);
    upload_async(in.ptr, host.data(), host.size() * 8, s);
  }
  const UniJobDev* djobs = (const UniJobDev*)in.ptr;
  const uint64_t* dpw = in.as<uint64_t>() + job_words;
  const size_t entries = count * S + blk;
  k_uni_many_tables<D><<<blocks_for(entries, RT), RT, 0, s>>>(buf.as<uint64_t>(), djobs, dpw, count, S);
  WHIR_HIP(hipGetLastError());
  {
    ProfScope prof(kernel_name("k_uni_many", 1, D), s, 8.0 * (double)blk * S);
    k_uni_many<D><<<(unsigned)blk, RT, 0, s>>>(djobs, count, buf.as<uint64_t>(), parts.as<uint64_t>());
    WHIR_HIP(hipGetLastError());
  }
  k_uni_many_reduce<D><<<(unsigned)count, RT, 0, s>>>(djobs, parts.as<uint64_t>(), out);
  WHIR_HIP(hipGetLastError());
}

void univariate_eval_batch_dev(int D, const UniJob* jobs, size_t count, uint64_t* out, hipStream_t s) {
  if (!count) return;
  switch (D) {
    case 1: uni_batch_t<1>(jobs, count, out, s); return;
    case 2: uni_batch_t<2>(jobs, count, out, s); return;
    case 3: uni_batch_t<3>(jobs, count, out, s); return;
  }
  throw Error("univariate batch: extension degree must be 1, 2 or 3");
}

void univariate_eval_dev(int Ds, int D, const uint64_t* c, size_t n, const uint64_t* x, uint64_t* out,
                         hipStream_t s) {
  univariate_eval_many_dev(Ds, D, &c, 1, n, x, 1, out, s);
}

// ------------------------------------------------------------------ lift, axpy, dot, gather
template <int D>
__global__ void k_lift(const uint64_t* src, size_t n, uint64_t* dst) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    st<D>(dst, i, gl::ext_base<D>(src[i]));
}

void lift_dev(int D, const uint64_t* src, size_t n, uint64_t* dst, hipStream_t s) {
  if (!n) return;
  ProfScope prof(kernel_name("k_lift", D), s, 8.0 * (1.0 + D) * (double)n);
  switch (D) {
    case 1: k_lift<1><<<grid_for(n), RT, 0, s>>>(src, n, dst); break;
    case 2: k_lift<2><<<grid_for(n), RT, 0, s>>>(src, n, dst); break;
    case 3: k_lift<3><<<grid_for(n), RT, 0, s>>>(src, n, dst); break;
    default: throw Error("lift: extension degree must be 1, 2 or 3");
  }
  WHIR_HIP(hipGetLastError());
}

template <int D>
__global__ void k_axpy(uint64_t* acc, Ext<D> w, const uint64_t* v, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    st<D>(acc, i, gl::eadd<D>(ld<D>(acc, i), gl::escale<D>(w, v[i])));
}

void mixed_scalar_mul_add_dev(int D, uint64_t* acc, const uint64_t* w, const uint64_t* v, size_t n, hipStream_t s) {
  if (!n) return;
  switch (D) {
    case 1: k_axpy<1><<<grid_for(n), RT, 0, s>>>(acc, host_ext<1>(w), v, n); break;
    case 2: k_axpy<2><<<grid_for(n), RT, 0, s>>>(acc, host_ext<2>(w), v, n); break;
    case 3: k_axpy<3><<<grid_for(n), RT, 0, s>>>(acc, host_ext<3>(w), v, n); break;
    default: throw Error("mixed_scalar_mul_add: extension degree must be 1, 2 or 3");
  }
  WHIR_HIP(hipGetLastError());
}

template <int D>
__global__ void k_axpy_ext(uint64_t* acc, Ext<D> w, const uint64_t* v, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    st<D>(acc, i, gl::eadd<D>(ld<D>(acc, i), gl::emul<D>(w, ld<D>(v, i))));
}

void scalar_mul_add_dev(int D, uint64_t* acc, const uint64_t* w, const uint64_t* v, size_t n, hipStream_t s) {
  if (!n) return;
  switch (D) {
    case 1: k_axpy_ext<1><<<grid_for(n), RT, 0, s>>>(acc, host_ext<1>(w), v, n); break;
    case 2: k_axpy_ext<2><<<grid_for(n), RT, 0, s>>>(acc, host_ext<2>(w), v, n); break;
    case 3: k_axpy_ext<3><<<grid_for(n), RT, 0, s>>>(acc, host_ext<3>(w), v, n); break;
    default: throw Error("scalar_mul_add: extension degree must be 1, 2 or 3");
  }
  WHIR_HIP(hipGetLastError());
}

template <int D>
__global__ __launch_bounds__(RT) void k_dot(const uint64_t* a, const uint64_t* b, size_t n, uint64_t* parts) {
  Ext<D> acc[1] = {gl::ext_zero<D>()};
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    acc[0] = gl::eadd<D>(acc[0], gl::emul<D>(ld<D>(a, i), ld<D>(b, i)));
  block_reduce_store<D, 1>(acc, parts + (size_t)blockIdx.x * D);
}

template <int D>
static void dot_t(const uint64_t* a, const uint64_t* b, size_t n, uint64_t* out, hipStream_t s) {
  unsigned g = grid_for(n ? n : 1);
  DevBuf parts((size_t)g * D * 8, s);
  k_dot<D><<<g, RT, 0, s>>>(a, b, n, parts.as<uint64_t>());
  WHIR_HIP(hipGetLastError());
  finish_reduce<D, 1>(parts.as<uint64_t>(), g, out, s);
}

void dot_dev(int D, const uint64_t* a, const uint64_t* b, size_t n, uint64_t* out, hipStream_t s) {
  switch (D) {
    case 1: dot_t<1>(a, b, n, out, s); break;
    case 2: dot_t<2>(a, b, n, out, s); break;
    case 3: dot_t<3>(a, b, n, out, s); break;
    default: throw Error("dot: extension degree must be 1, 2 or 3");
  }
}

template <int D>
__global__ void k_gather(const uint64_t* cw, size_t N, size_t M, const uint64_t* idx, size_t k, uint64_t* out) {
  size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (e >= k * M) return;
  size_t q = e / M, j = e % M;
  size_t r = idx[q];
  if (r >= N) return;
  st<D>(out, q * M + j, ld<D>(cw, j * N + r));
}

// Opening gather in one launch: rows (out_rows[q*M + j] = cw[j*N + idx[q]], Ds words
// each) and Merkle sibling hashes (out_hashes[i] = nodes[sib[i]]); idx_sib holds the
// k row indices followed by the ns node indices.  With D > 0 it also sums each opened
// row against per-column weights of degree D (wts[j], D words):
// out_vals[q] = sum_j wts[j] cw[j*N + idx[q]].  When M is a power of two up to 64 the
// M lanes that gather a row each weight their element and sum across the row with
// XOR shuffles (the row's lanes are aligned within one wave), so no lane waits on M
// loads in turn; other widths sum each row on one lane.
template <int Ds, int D>
__global__ void k_gather_open(const uint64_t* __restrict__ cw, size_t N, size_t M, const uint64_t* __restrict__ idx_sib,
                              size_t k, const uint4* __restrict__ nodes, size_t ns, uint64_t* out_rows,
                              uint4* out_hashes, const uint64_t* __restrict__ wts, uint64_t* out_vals,
                              bool lane_sums) {
  size_t e = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
  if (e < k * M) {
    const size_t q = e / M, j = e % M, r = idx_sib[q];
    const Ext<Ds> x = r < N ? ld<Ds>(cw, j * N + r) : gl::ext_zero<Ds>();
    if (r < N) st<Ds>(out_rows, e, x);
    if constexpr (D > 0) {
      if (lane_sums) {
        Ext<D> p;
        if constexpr (Ds == 1) p = gl::escale<D>(ld<D>(wts, j), x.c[0]);
        else p = gl::emul<D>(ld<D>(wts, j), x);
        for (unsigned o = 1; o < (unsigned)M; o <<= 1) {
          Ext<D> t;
#pragma unroll
          for (int d = 0; d < D; d++) t.c[d] = __shfl_xor(p.c[d], (int)o);
          p = gl::eadd<D>(p, t);
        }
        if (j == 0) st<D>(out_vals, q, p);  // zero for an index past the codeword
      }
    }
    return;
  }
  e -= k * M;
  if (e < 2 * ns) {
    out_hashes[e] = nodes[2 * idx_sib[k + (e >> 1)] + (e & 1)];
    return;
  }
  if constexpr (D > 0) {
    e -= 2 * ns;
    if (!lane_sums && e < k) {
      const size_t r = idx_sib[e];
      Ext<D> acc = gl::ext_zero<D>();
      if (r < N) {
#pragma unroll 8
        for (size_t j = 0; j < M; j++) {
          if constexpr (Ds == 1) acc = gl::eadd<D>(acc, gl::escale<D>(ld<D>(wts, j), cw[j * N + r]));
          else acc = gl::eadd<D>(acc, gl::emul<D>(ld<D>(wts, j), ld<D>(cw, j * N + r)));
        }
      }
      st<D>(out_vals, e, acc);
    }
  }
}

template <int Ds, int D>
static void gather_open_t(const uint64_t* cw, size_t N, size_t M, const uint64_t* idx_sib, size_t k,
                          const uint8_t* nodes, size_t ns, uint64_t* out_rows, uint8_t* out_hashes,
                          const uint64_t* wts, uint64_t* out_vals, hipStream_t s) {
  const bool lane_sums = D > 0 && M >= 1 && M <= 64 && (M & (M - 1)) == 0;
  const size_t total = k * M + 2 * ns + (D > 0 && !lane_sums ? k : 0);
  if (!total) return;
  // Rows start at multiples of M within each block (RT % M == 0), so a row's lanes
  // are aligned within one wave.
  static_assert(RT % 64 == 0, "block size must be a multiple of the wave size");
  k_gather_open<Ds, D><<<blocks_for(total, RT), RT, 0, s>>>(cw, N, M, idx_sib, k, (const uint4*)nodes, ns, out_rows,
                                                              (uint4*)out_hashes, wts, out_vals, lane_sums);
  WHIR_HIP(hipGetLastError());
}

void gather_open_dev(int Ds, const uint64_t* cw, size_t N, size_t M, const uint64_t* idx_sib, size_t k,
                     const uint8_t* nodes, size_t ns, uint64_t* out_rows, uint8_t* out_hashes, hipStream_t s, int D,
                     const uint64_t* wts, uint64_t* out_vals) {
  WHIR_REQUIRE(ns == 0 || ((uintptr_t)out_hashes & 15) == 0, "gather_open: hash output must be 16-byte aligned");
  WHIR_REQUIRE(D == 0 || (wts && out_vals), "gather_open: row sums need weights and an output");
  const int key = Ds * 10 + D;
  switch (key) {
    case 10: gather_open_t<1, 0>(cw, N, M, idx_sib, k, nodes, ns, out_rows, out_hashes, wts, out_vals, s); return;
    case 20: gather_open_t<2, 0>(cw, N, M, idx_sib, k, nodes, ns, out_rows, out_hashes, wts, out_vals, s); return;
    case 30: gather_open_t<3, 0>(cw, N, M, idx_sib, k, nodes, ns, out_rows, out_hashes, wts, out_vals, s); return;
    case 11: gather_open_t<1, 1>(cw, N, M, idx_sib, k, nodes, ns, out_rows, out_hashes, wts, out_vals, s); return;
    case 12: gather_open_t<1, 2>(cw, N, M, idx_sib, k, nodes, ns, out_rows, out_hashes, wts, out_vals, s); return;
    case 13: gather_open_t<1, 3>(cw, N, M, idx_sib, k, nodes, ns, out_rows, out_hashes, wts, out_vals, s); return;
    case 22: gather_open_t<2, 2>(cw, N, M, idx_sib, k, nodes, ns, out_rows, out_hashes, wts, out_vals, s); return;
    case 33: gather_open_t<3, 3>(cw, N, M, idx_sib, k, nodes, ns, out_rows, out_hashes, wts, out_vals, s); return;
    default: throw Error("gather: unsupported row / weight degrees");
  }
}

void gather_rows_dev(int D, const uint64_t* cw, size_t N, size_t M, const uint64_t* idx, size_t k, uint64_t* out,
                     hipStream_t s) {
  if (!k || !M) return;
  unsigned g = blocks_for(k * M, RT);
  switch (D) {
    case 1: k_gather<1><<<g, RT, 0, s>>>(cw, N, M, idx, k, out); break;
    case 2: k_gather<2><<<g, RT, 0, s>>>(cw, N, M, idx, k, out); break;
    case 3: k_gather<3><<<g, RT, 0, s>>>(cw, N, M, idx, k, out); break;
    default: throw Error("gather: extension degree must be 1, 2 or 3");
  }
  WHIR_HIP(hipGetLastError());
}

}  // namespace whir
