// Restarted, right-preconditioned GMRES(m) on the device.
//
// Reference: krylov::gmres_preconditioned[_with_workspace]
// (crates/cfd-math/src/linear_solver/krylov.rs:150-251) delegating to the
// un-vendored athena Gmres<B, M>; the restart width is rounded up the ladder
// 8/16/32/64/128/256 (krylov.rs:84-114) when restart_ladder is set.
//
// Arnoldi uses classical Gram-Schmidt applied twice (CGS2): a multi-dot over
// all basis vectors, and a multi-axpy, per pass, instead of the j+1 dependent
// dots of modified Gram-Schmidt.  The first pass's multi-axpy and the second
// pass's multi-dot read the same basis entries and run as one kernel.  The
// Hessenberg column, Givens rotations and residual estimate are updated on
// the device by the kernel that scales the new basis vector, so a whole
// restart cycle is enqueued without a host round trip.
// The preconditioner is linear, so the cycle's update is
// x += M^-1 (V_k y) with a single preconditioner application.
#include <algorithm>
#include <cmath>

#include "reduce.hpp"
#include "solver.hpp"

namespace cfdla {
namespace {

constexpr int kGramBlocks = 512;  // partials per vector of k_gram
constexpr int kMdotBlocks = 256;  // and of k_mdot

struct GmLayout {
  int m;
  double *H, *cs, *sn, *g, *y, *hc, *hp, *part;
  static size_t doubles(int m) { return (size_t)(m + 1) * m + 2 * m + (m + 1) + m + 2 * (m + 1) + (size_t)(m + 1) * kGramBlocks; }
  GmLayout(double *base, int m_) : m(m_) {
    H = base;
    cs = H + (size_t)(m + 1) * m;
    sn = cs + m;
    g = sn + m;
    y = g + (m + 1);
    hc = y + m;
    hp = hc + (m + 1);
    part = hp + (m + 1);
  }
};

// part[k * NB + bx] = sum over the block's slice of V_k . w, k = blockIdx.y
template <typename T>
__global__ __launch_bounds__(kBlock) void k_mdot(int n, const T *__restrict__ V, size_t ld, const T *__restrict__ w,
                                                 double *__restrict__ part, Scal *s) {
  if (s->done) return;
  const int k = blockIdx.y;
  const T *v = V + (size_t)k * ld;
  double acc = 0.0;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) acc += (double)v[i] * (double)w[i];
  __shared__ double sh[kBlock / 64];
  acc = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int q = 0; q < kBlock / 64; ++q) t += sh[q];
    part[(size_t)k * gridDim.x + blockIdx.x] = t;
  }
}

// hp[k] = sum_b part[k * nb + b]; hc[k] (+)= hp[k]
__global__ __launch_bounds__(kBlock) void k_mdot_fin(int nb, const double *__restrict__ part, double *__restrict__ hp,
                                                     double *__restrict__ hc, int first, Scal *s) {
  if (s->done) return;
  const int k = blockIdx.x;
  double acc = 0.0;
  for (int b = threadIdx.x; b < nb; b += kBlock) acc += part[(size_t)k * nb + b];
  __shared__ double sh[kBlock / 64];
  acc = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int q = 0; q < kBlock / 64; ++q) t += sh[q];
    hp[k] = t;
    hc[k] = first ? t : hc[k] + t;
  }
}

// w -= sum_{k<=j} hp[k] V_k; with NORM, also the block partials of ||w||^2
// of the updated w (the last Gram-Schmidt pass: the norm needs no pass of
// its own).  (Summing the multi-dot partials here instead of in k_mdot_fin,
// with 64 partials per vector, was slower: 22.1 -> 23.2 ms for the 512^2
// momentum GMRES.)
template <typename T, bool NORM>
__global__ __launch_bounds__(kBlock) void k_maxpy(int n, int jp1, const T *__restrict__ V, size_t ld,
                                                  const double *__restrict__ hp, T *__restrict__ w, Scal *s,
                                                  double *partials) {
  if (s->done) return;
  __shared__ double h[257];
  for (int k = threadIdx.x; k < jp1; k += kBlock) h[k] = hp[k];
  __syncthreads();
  double v[1] = {0.0};
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    double acc = (double)w[i];
    for (int k = 0; k < jp1; ++k) acc -= h[k] * (double)V[(size_t)k * ld + i];
    const T wi = (T)acc;
    w[i] = wi;
    if (NORM) v[0] += (double)wi * (double)wi;
  }
  if (NORM) block_partials<1>(v, partials);
}

// ---- Gram-Schmidt passes over at most JB basis vectors, held in registers ------
// Bound: the basis bytes (L2 and Infinity Cache).  A lane owns whole elements
// of w and reads the JB entries of its element together, so w is read once
// per pass and a pass that updates and then dots reads the basis once.
//
// The block's sums of JB accumulators per lane: each lane swap halves the
// accumulators instead of the lanes that hold a sum (lane ^ 32, then lane ^
// 16: the lower half keeps the first accumulator of a pair, the upper half
// the second), then rotations add the 16 lanes of a row.  About 5
// instructions per accumulator against 24 for a wavefront sum each.
template <int SWAP>
__device__ __forceinline__ double swap_add(double a, double b) {
  const unsigned long long x = __builtin_bit_cast(unsigned long long, a), y = __builtin_bit_cast(unsigned long long, b);
  unsigned l0, l1, h0, h1;
  if constexpr (SWAP == 32) {
    const auto l = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    l0 = l[0]; l1 = l[1]; h0 = h[0]; h1 = h[1];
  } else {
    const auto l = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
    l0 = l[0]; l1 = l[1]; h0 = h[0]; h1 = h[1];
  }
  return __builtin_bit_cast(double, (unsigned long long)h0 << 32 | l0) +
         __builtin_bit_cast(double, (unsigned long long)h1 << 32 | l1);
}

// part[k * nb + blockIdx.x] = the block's sum of accumulator k, k < jp1
template <int JB, int THREADS>
__device__ __forceinline__ void block_sums(double (&acc)[JB], int jp1, double *__restrict__ part) {
  static_assert(JB % 4 == 0, "four rows of 16 lanes hold a quarter of the sums each");
  __shared__ double sh[THREADS / 64][JB];
  constexpr int Q = JB / 4;
  double half[2 * Q], quarter[Q];
#pragma unroll
  for (int k = 0; k < 2 * Q; ++k) half[k] = swap_add<32>(acc[k], acc[k + 2 * Q]);
#pragma unroll
  for (int k = 0; k < Q; ++k) quarter[k] = swap_add<16>(half[k], half[k + Q]);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < Q; ++k) {
    double v = quarter[k];
    v += dpp_move<0x128>(v);
    v += dpp_move<0x124>(v);
    v += dpp_move<0x122>(v);
    v += dpp_move<0x121>(v);
    if ((lane & 15) == 0) sh[wave][(lane >> 4) * Q + k] = v;  // row r of lanes: sums r Q .. r Q + Q - 1
  }
  __syncthreads();
  for (int k = threadIdx.x; k < jp1; k += THREADS) {
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < THREADS / 64; ++w) t += sh[w][k];
    part[(size_t)k * gridDim.x + blockIdx.x] = t;
  }
}

// One element: its basis entries, and with UPDATE w_i -= sum_k h[k] V_k,i in
// ascending k.
template <typename T, int JB, bool UPDATE, bool DOTS, bool NORM>
__global__ __launch_bounds__(kBlock) void k_gram(int n, int jp1, const T *__restrict__ V, size_t ld,
                                                 const double *__restrict__ hp, T *__restrict__ w, Scal *s,
                                                 double *__restrict__ part) {
  if (s->done) return;
  __shared__ double h[JB];
  if constexpr (UPDATE) {
    if (threadIdx.x < JB) h[threadIdx.x] = (int)threadIdx.x < jp1 ? hp[threadIdx.x] : 0.0;
    __syncthreads();
  }
  double acc[JB], nv[1] = {0.0};
#pragma unroll
  for (int k = 0; k < JB; ++k) acc[k] = 0.0;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    T v[JB];
    const T wi = w[i];
    // jp1 is the same for the grid: vectors past it repeat the last one
    // (a cached line) and are not used
#pragma unroll
    for (int k = 0; k < JB; ++k) v[k] = V[(size_t)min(k, jp1 - 1) * ld + i];
    T wn = wi;
    if constexpr (UPDATE) {
      double t = (double)wi;
#pragma unroll
      for (int k = 0; k < JB; ++k)
        if (k < jp1) t -= h[k] * (double)v[k];
      wn = (T)t;
      w[i] = wn;
    }
    if constexpr (DOTS) {
#pragma unroll
      for (int k = 0; k < JB; ++k) acc[k] += (double)v[k] * (double)wn;
    }
    if constexpr (NORM) nv[0] += (double)wn * (double)wn;
  }
  if constexpr (DOTS) block_sums<JB, kBlock>(acc, jp1, part);
  if constexpr (NORM) block_partials<1>(nv, part);
}

// ---- the same passes with one element per thread -------------------------------
// Up to kRowBlocks blocks of 1024 rows: so few partials that the next pass's
// blocks sum them themselves, each wavefront a vector's, while their own
// entries are in flight, instead of a launch between (k_mdot_fin, 2.7 us); and
// the first pass forms its element of w itself where A is diagonal storage,
// which saves the product's launch (3.6 us).  Bound: the basis bytes out of the
// Infinity Cache for long bases, two round trips of latency for short ones.  384
// x 384 momentum matrix, 8 / 16 / 24 / 32 vectors: dots with the product 6.1 /
// 7.4 / 9.2 / 10.7 us, update and dots 5.1 / 6.8 / 8.2 / 10.3, update and norm 4.6 /
// 5.7 / 6.4 / 8.2; a step 36 -> 27 us with the start of the sweep in the scaling
// (k_gm_arnoldi_sor), GMRES(30) with SOR there 8.9 -> 6.7 ms.  (Smaller blocks,
// one on every CU, cost more in the partials: 6.9 ms; visiting the vectors
// backwards in every other pass gained nothing.)
// PASS_DOTS: dots of w; PASS_PRODUCT: w = A z and its dots; PASS_BOTH: w -=
// sum_k h_k V_k, then dots; PASS_LAST: w -= sum_k h_k V_k and its norm.  h from
// in (nb partials per vector); hc collects them over the two passes.
constexpr int kRowThreads = 1024;
constexpr int kRowBlocks = 256;
enum { PASS_DOTS, PASS_PRODUCT, PASS_BOTH, PASS_LAST };
template <typename T, int JB, int PASS, int NS>
__global__ __launch_bounds__(kRowThreads) void k_gram_row(int n, int jp1, const T *__restrict__ V, size_t ld,
                                                          DiaRows A, const T *__restrict__ av,
                                                          const T *__restrict__ z, const double *__restrict__ in,
                                                          double *__restrict__ hc, T *__restrict__ w, const Scal *s,
                                                          double *__restrict__ out) {
  if (s->done) return;
  constexpr int W = kRowThreads / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nb = gridDim.x;
  const int mine = blockIdx.x * kRowThreads + tid;
  const bool live = mine < n;
  const int i = live ? mine : n - 1;
  constexpr bool UPDATE = PASS == PASS_BOTH || PASS == PASS_LAST;
  constexpr int R = (JB + W - 1) / W, Q = kRowBlocks / 64;
  // the partials first: loads return in order, and h is summed while the
  // entries are on their way
  double hv[R][Q];
  if constexpr (UPDATE) {
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int k = min(wave + r * W, jp1 - 1), b = lane + 64 * q;
        const double t = in[(size_t)k * nb + min(b, nb - 1)];
        hv[r][q] = b < nb ? t : 0.0;
      }
    __builtin_amdgcn_sched_barrier(0);
  }
  T v[JB];
#pragma unroll
  for (int k = 0; k < JB; ++k) v[k] = V[(size_t)min(k, jp1 - 1) * ld + i];
  double wn;
  if constexpr (PASS == PASS_PRODUCT) {
    T a[NS], g[NS];
#pragma unroll
    for (int q = 0; q < NS; ++q) {
      const int c = i + A.off[q];
      const bool ok = q < A.count && c >= 0 && c < n;
      const T e = av[(size_t)A.k[q] * n + (ok && A.lower[q] ? c : i)];
      a[q] = ok ? e : T(0);
      g[q] = z[ok ? c : i];
    }
    T sum = T(0);
#pragma unroll
    for (int q = 0; q < NS; ++q) sum += a[q] != T(0) ? a[q] * g[q] : T(0);
    wn = (double)sum;
    if (live) w[i] = sum;
  } else {
    wn = (double)w[i];
  }
  if constexpr (UPDATE) {
    __shared__ double h[R * W];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      double t = hv[r][0];
#pragma unroll
      for (int q = 1; q < Q; ++q) t += hv[r][q];
      t = wave_sum(t);
      if (lane == 0) h[wave + r * W] = t;
    }
    __syncthreads();
    if (blockIdx.x == 0 && tid < jp1) hc[tid] = PASS == PASS_BOTH ? h[tid] : hc[tid] + h[tid];
#pragma unroll
    for (int k = 0; k < JB; ++k)
      if (k < jp1) wn -= h[k] * (double)v[k];
    const T t = (T)wn;
    wn = (double)t;
    if (live) w[i] = t;
  }
  if constexpr (PASS == PASS_LAST) {
    __shared__ double sh[W];
    const double t = wave_sum(live ? wn * wn : 0.0);
    if (lane == 0) sh[wave] = t;
    __syncthreads();
    if (wave == 0) {
      const double sum = wave_sum(lane < W ? sh[lane] : 0.0);
      if (lane == 0) out[blockIdx.x] = sum;
    }
  } else {
    double acc[JB];
#pragma unroll
    for (int k = 0; k < JB; ++k) acc[k] = live ? (double)v[k] * wn : 0.0;
    block_sums<JB, kRowThreads>(acc, jp1, out);
  }
}

// ||w|| from its partials, v_{j+1} = w / ||w|| in place, and (block 0) the
// Hessenberg column j, Givens rotation and residual estimate.  Every block
// sums the partials itself; the scalars go from in to out, so no block reads
// what block 0 has already advanced.  Block 0 stages the column and the
// earlier rotations in LDS, so thread 0's rotation chain waits on arithmetic,
// not on global memory, beside the other blocks' scaling (4.8 us; 3.7 + 2.9 us
// with the scaling as a launch of its own, 147,456 rows).
struct Column {
  double h[258], cs[256], sn[256];
  Scal sc;
};
// block 0, before the norm is summed
__device__ __forceinline__ void load_column(Column &c, int j, const Scal *in, const GmLayout &L) {
  const int tid = threadIdx.x;
  if (tid < (int)(sizeof(Scal) / sizeof(int))) reinterpret_cast<int *>(&c.sc)[tid] = reinterpret_cast<const int *>(in)[tid];
  for (int k = tid; k <= j; k += kBlock) c.h[k] = L.hc[k];
  for (int k = tid; k < j; k += kBlock) {
    c.cs[k] = L.cs[k];
    c.sn[k] = L.sn[k];
  }
}
// block 0, with the norm hn and its reciprocal a
__device__ __forceinline__ void finish_column(Column &c, int j, double hn, double a, Scal *out, const GmLayout &L) {
  const int tid = threadIdx.x, m = L.m;
  if (tid == 0) {
    Scal &sc = c.sc;
    double *col = c.h;
    sc.hn = hn;
    col[j + 1] = hn;
    for (int k = 0; k < j; ++k) {
      const double t0 = col[k], t1 = col[k + 1];
      col[k] = c.cs[k] * t0 + c.sn[k] * t1;
      col[k + 1] = -c.sn[k] * t0 + c.cs[k] * t1;
    }
    const double h0 = col[j], h1 = col[j + 1];
    const double den = hypot(h0, h1);
    if (den == 0.0 || !isfinite(den)) {
      sc.done = 4;  // breakdown: the cycle ends with kstep = j
    } else {
      const double cj = h0 / den, sj = h1 / den;
      L.cs[j] = cj;
      L.sn[j] = sj;
      col[j] = den;
      col[j + 1] = 0.0;
      const double gj = L.g[j];
      L.g[j + 1] = -sj * gj;
      L.g[j] = cj * gj;
      sc.kstep = j + 1;
      sc.iters += 1;
      sc.alpha = a;
      if (fabs(L.g[j + 1]) <= sqrt(sc.thr2) || hn == 0.0) sc.done = 1;
    }
  }
  __syncthreads();
  if (tid < (int)(sizeof(Scal) / sizeof(int))) reinterpret_cast<int *>(out)[tid] = reinterpret_cast<const int *>(&c.sc)[tid];
  // the column as the host-visible Hessenberg H(0:j+1, j); on breakdown the
  // rotated entries up to j + 1, as before the rotation that failed
  for (int k = tid; k <= j + 1; k += kBlock) L.H[(size_t)k * m + j] = c.h[k];
}
__device__ __forceinline__ void keep_scal(const Scal *in, Scal *out) {
  const int tid = threadIdx.x;
  if (blockIdx.x == 0 && tid < (int)(sizeof(Scal) / sizeof(int)))
    reinterpret_cast<int *>(out)[tid] = reinterpret_cast<const int *>(in)[tid];
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_gm_arnoldi(int j, int n, T *__restrict__ w, int nblocks,
                                                       const double *partials, const Scal *in, Scal *out, GmLayout L) {
  __shared__ Column c;
  const int tid = threadIdx.x;
  const bool first = blockIdx.x == 0;
  if (in->done) {
    keep_scal(in, out);
    return;
  }
  const int i0 = blockIdx.x * kBlock + tid, step = gridDim.x * kBlock;
  T w0 = T(0);
  if (i0 < n) w0 = w[i0];
  if (first) load_column(c, j, in, L);
  double tot[1];
  sum_partials<1>(nblocks, partials, tot);  // synchronizes the block
  const double hn = sqrt(tot[0]);
  const double a = hn > 0.0 ? 1.0 / hn : 0.0;
  // (a breakdown or a non-finite norm ends the cycle: the vector is not used)
  for (int i = i0; i < n; i += step) w[i] = (T)((double)(i == i0 ? w0 : w[i]) * a);
  if (first) finish_column(c, j, hn, a, out, L);
}

// The same with v_{j+1} = w / ||w|| going to its own place and, in the same
// launch, the start of the multicolour sweep on it (k_sor_start in
// kernels.hip: the first colour z_i = piv_i v_i, the second from the first's
// values formed at the gathers; the other colours 0).  The neighbours' entries
// of v are formed from w as the own one is, so z has the bits of the sweep on
// the stored v.
template <typename T, int W>
__global__ __launch_bounds__(kBlock) void k_gm_arnoldi_sor(int j, int n, const T *__restrict__ w, T *__restrict__ v,
                                                           T *__restrict__ z, const uint8_t *__restrict__ cls,
                                                           const int *__restrict__ ci, const T *__restrict__ sv,
                                                           const T *__restrict__ piv, int nblocks,
                                                           const double *partials, const Scal *in, Scal *out,
                                                           GmLayout L) {
  __shared__ Column c;
  const bool first = blockIdx.x == 0;
  if (in->done) {
    keep_scal(in, out);
    return;
  }
  if (first) load_column(c, j, in, L);
  double hn = 0.0, a = 0.0;
  bool summed = false;
  for (int base = blockIdx.x * kBlock; base < n; base += gridDim.x * kBlock) {
    const bool live = base + (int)threadIdx.x < n;
    const int i = live ? base + (int)threadIdx.x : n - 1;
    const int k = cls[i];
    const T pi = piv[i], wi = w[i];
    int col[W];
    T e[W], pj[W], wj[W];
#pragma unroll
    for (int q = 0; q < W; ++q) {
      col[q] = ci[(size_t)q * n + i];
      e[q] = sv[(size_t)q * n + i];
    }
#pragma unroll
    for (int q = 0; q < W; ++q) {
      pj[q] = piv[col[q]];
      wj[q] = w[col[q]];
    }
    if (!summed) {
      double tot[1];
      sum_partials<1>(nblocks, partials, tot);  // synchronizes the block
      hn = sqrt(tot[0]);
      a = hn > 0.0 ? 1.0 / hn : 0.0;
      summed = true;
    }
    const T ri = (T)((double)wi * a);
    T acc = ri;
#pragma unroll
    for (int q = 0; q < W; ++q)
      if (col[q] != i) {
        const T zj = pj[q] * (T)((double)wj[q] * a);
        acc -= e[q] * zj;
      }
    if (live) {
      v[i] = ri;
      z[i] = k > 1 ? T(0) : pi * acc;
    }
  }
  if (first) finish_column(c, j, hn, a, out, L);
}

// Back substitution H(0:k,0:k) y = g(0:k), k = kstep, by one wavefront: the
// triangle is staged in LDS and each lane keeps the right-hand sides of its
// rows, from which every solved unknown is taken at once (a single thread
// walking the triangle in global memory took 46 us at k = 32, this 10 us).
constexpr int kSolveLds = 64;  // largest restart width staged in LDS
__global__ __launch_bounds__(64) void k_gm_solve(const Scal *s, GmLayout L) {
  const int k = s->kstep, m = L.m, lane = threadIdx.x;
  __shared__ double h[kSolveLds * kSolveLds];
  if (m > kSolveLds) {
    if (lane != 0) return;
    for (int i = k - 1; i >= 0; --i) {
      double t = L.g[i];
      for (int q = i + 1; q < k; ++q) t -= L.H[(size_t)i * m + q] * L.y[q];
      L.y[i] = t / L.H[(size_t)i * m + i];
    }
    return;
  }
  for (int e = lane; e < k * m; e += 64) h[e] = L.H[e];
  double t = lane < k ? L.g[lane] : 0.0;
  __syncthreads();
  for (int i = k - 1; i >= 0; --i) {
    const double yi = __shfl(t, i, 64) / h[i * m + i];
    if (lane == i) L.y[i] = yi;
    if (lane < i) t -= h[lane * m + i] * yi;
  }
}

// u = sum_{k < kstep} y_k V_k
template <typename T>
__global__ __launch_bounds__(kBlock) void k_gm_combine(int n, const T *__restrict__ V, size_t ld, Scal *s, GmLayout L,
                                                       T *__restrict__ u) {
  const int k = s->kstep;
  __shared__ double y[256];
  for (int q = threadIdx.x; q < k; q += kBlock) y[q] = L.y[q];
  __syncthreads();
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
    double acc = 0.0;
    for (int q = 0; q < k; ++q) acc += y[q] * (double)V[(size_t)q * ld + i];
    u[i] = (T)acc;
  }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void k_axpy1(int n, const T *__restrict__ z, T *__restrict__ x) {
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) x[i] += z[i];
}

// v_0 = r / beta, g = beta e_1, new cycle.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_gm_restart(int n, const T *__restrict__ r, double beta,
                                                       T *__restrict__ v0, Scal *s, GmLayout L) {
  const double a = 1.0 / beta;
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) v0[i] = (T)((double)r[i] * a);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    for (int q = 0; q <= L.m; ++q) L.g[q] = 0.0;
    L.g[0] = beta;
    s->kstep = 0;
    s->done = 0;
  }
}

template <typename T> T *vec(int slot, size_t n);
template <> double *vec<double>(int slot, size_t n) { return ctx().dv_at(slot, n); }
template <> float *vec<float>(int slot, size_t n) { return ctx().fv_at(slot, n); }

struct GmWork {
  DevBuf<double> V64, st;
  DevBuf<float> V32;
};
GmWork &gmwork() {
  static GmWork w;
  return w;
}

template <typename T> T *basis(size_t count);
template <> double *basis<double>(size_t count) { gmwork().V64.ensure(count); return gmwork().V64.p; }
template <> float *basis<float>(size_t count) { gmwork().V32.ensure(count); return gmwork().V32.p; }

template <typename T>
double residual_norm(const DevCsr &A, const T *b, const T *x, T *r, Scal *s) {
  csr_apply<T>(A, EPI_RESID, x, b, nullptr, 0.0, r, s, false, OP_INIT_RR, r, ctx().ws);
  return std::sqrt(ctx().read(s).rr);
}

template <typename T>
SolveOut gmres(const DevCsr &A, Precond *M, const T *b, T *x, double thr, int64_t max_it, int m, bool confirm) {
  Context &c = ctx();
  RedWs &ws = c.ws;
  const int n = A.n;
  const size_t ld = (size_t)n;
  T *V = basis<T>((size_t)(m + 1) * ld);
  gmwork().st.ensure(GmLayout::doubles(m));
  GmLayout L(gmwork().st.p, m);
  T *r = vec<T>(0, n), *z = vec<T>(1, n), *u = vec<T>(2, n);
  Scal *s = c.s(0);
  SolveOut o;
  o.thr = thr;
  scal_reset(s, thr * thr);
  double beta = residual_norm<T>(A, b, x, r, s);
  o.rn0 = o.rn = beta;
  if (beta <= thr) {
    o.term = CFDLA_TERM_INITIAL_RESIDUAL;
    return o;
  }
  const int eb = blocks_for(n, kBlock * 4);
  const int gb = std::min(kGramBlocks, blocks_for(n, kBlock));
  // k_mdot runs this many blocks for every vector, so each takes several rows
  // per lane: with gb of them a cycle of 256 vectors on 147,456 rows, of which
  // 87 steps run and the others find the solve done, takes 15.3 ms, with these
  // 10.5 (262,144 rows: 21.1 and 17.9; FP32 33.0 and 26.3)
  const int mb = std::min(kMdotBlocks, blocks_for(n, kBlock * 4));
  // Gram-Schmidt over basis vectors 0..j of w.  Up to 32 vectors fit the
  // registers of k_gram (384 x 384 momentum matrix, m = 32: 16.7 us per step on
  // average against 21.6 us in the separate multi-dots and multi-axpys); a
  // longer basis takes those.
  auto gram = [&](int j, T *w, Scal *sc) {
    const int jp1 = j + 1;
    auto fin = [&](int pass, int nb) {
      hipLaunchKernelGGL(k_mdot_fin, dim3(jp1), dim3(kBlock), 0, stream(), nb, L.part, L.hp, L.hc, pass == 0 ? 1 : 0,
                         sc);
    };
#define CFDLA_GRAM(JB)                                                                                                \
  do {                                                                                                                \
    hipLaunchKernelGGL((k_gram<T, JB, false, true, false>), dim3(gb), dim3(kBlock), 0, stream(), n, jp1, V, ld, L.hp, \
                       w, sc, L.part);                                                                                \
    fin(0, gb);                                                                                                       \
    hipLaunchKernelGGL((k_gram<T, JB, true, true, false>), dim3(gb), dim3(kBlock), 0, stream(), n, jp1, V, ld, L.hp,  \
                       w, sc, L.part);                                                                                \
    fin(1, gb);                                                                                                       \
    hipLaunchKernelGGL((k_gram<T, JB, true, false, true>), dim3(gb), dim3(kBlock), 0, stream(), n, jp1, V, ld, L.hp,  \
                       w, sc, ws.current());                                                                          \
    return gb;                                                                                                        \
  } while (0)
    if (jp1 <= 4) CFDLA_GRAM(4);
    if (jp1 <= 8) CFDLA_GRAM(8);
    if (jp1 <= 16) CFDLA_GRAM(16);
    if (jp1 <= 24) CFDLA_GRAM(24);
    if (jp1 <= 32) CFDLA_GRAM(32);
#undef CFDLA_GRAM
    for (int pass = 0; pass < 2; ++pass) {
      hipLaunchKernelGGL((k_mdot<T>), dim3(mb, jp1), dim3(kBlock), 0, stream(), n, V, ld, w, L.part, sc);
      fin(pass, mb);
      if (pass == 0)
        hipLaunchKernelGGL((k_maxpy<T, false>), dim3(eb), dim3(kBlock), 0, stream(), n, jp1, V, ld, L.hp, w, sc,
                           nullptr);
      else
        hipLaunchKernelGGL((k_maxpy<T, true>), dim3(eb), dim3(kBlock), 0, stream(), n, jp1, V, ld, L.hp, w, sc,
                           ws.current());
    }
    return eb;
  };
  // One row per thread, as long as the blocks' partials are few (above, and
  // for a basis of more than 32 vectors: gram).
  const DiaRows rows = dia_rows<T>(A);
  const int rb = (n + kRowThreads - 1) / kRowThreads;
  const bool by_row = rb <= kRowBlocks && m <= 32;
  auto gram_row = [&](int j, const T *zj, T *w, Scal *sc) {
    const int jp1 = j + 1;
    double *part[2] = {L.part, L.part + (size_t)(m + 1) * kRowBlocks};
    const T *av = rows.count > 0 ? A.dia_vals<T>() : nullptr;
    if (rows.count == 0) csr_apply<T>(A, EPI_Y, zj, nullptr, nullptr, 0.0, w, sc, true, OP_NONE, nullptr, ws);
    const auto go = [&](auto *kernel, const double *in, double *out) {
      hipLaunchKernelGGL(kernel, dim3(rb), dim3(kRowThreads), 0, stream(), n, jp1, V, ld, rows, av, zj, in, L.hc, w,
                         sc, out);
    };
#define CFDLA_GRAM_ROW(JB)                                                                  \
  do {                                                                                      \
    if (rows.count == 0) go(k_gram_row<T, JB, PASS_DOTS, 1>, nullptr, part[0]);              \
    else if (rows.count <= 5) go(k_gram_row<T, JB, PASS_PRODUCT, 5>, nullptr, part[0]);      \
    else go(k_gram_row<T, JB, PASS_PRODUCT, kDiaRowMax>, nullptr, part[0]);                  \
    go(k_gram_row<T, JB, PASS_BOTH, 1>, part[0], part[1]);                                   \
    go(k_gram_row<T, JB, PASS_LAST, 1>, part[1], ws.current());                              \
  } while (0)
    if (jp1 <= 8) CFDLA_GRAM_ROW(8);
    else if (jp1 <= 16) CFDLA_GRAM_ROW(16);
    else if (jp1 <= 24) CFDLA_GRAM_ROW(24);
    else CFDLA_GRAM_ROW(32);
#undef CFDLA_GRAM_ROW
    return rb;
  };
  // a multicolour sweep whose start takes the scaling of its argument along
  auto *sor = by_row ? dynamic_cast<ColoredSorPrecond *>(M) : nullptr;
  if (sor && sor->start_w == 0) sor = nullptr;
  T *wt = sor ? vec<T>(3, n) : nullptr;
  auto arnoldi_sor = [&](const ColoredSorPrecond &p, int j, const T *w, T *v, int parts, const Scal *in, Scal *out) {
    const auto go = [&](auto *kernel) {
      hipLaunchKernelGGL(kernel, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, stream(), j, n, w, v, z, p.cls.p,
                         p.start_ci.p, p.start_v<T>(), p.piv<T>(), parts, ws.current(), in, out, L);
    };
    if (p.start_w == 4) go(k_gm_arnoldi_sor<T, 4>);
    else if (p.start_w == 6) go(k_gm_arnoldi_sor<T, 6>);
    else go(k_gm_arnoldi_sor<T, 8>);
  };
  int64_t enq = 0;
  while (true) {
    // the residual's read left no reduction pending, and the cycle's kernels
    // start none: the scalars stay where they are until its end
    s = settled_scal(s);
    hipLaunchKernelGGL((k_gm_restart<T>), dim3(eb), dim3(kBlock), 0, stream(), n, r, beta, V, s, L);
    int steps = (int)std::min<int64_t>(m, max_it - enq);
    for (int j = 0; j < steps; ++j) {
      T *vj = V + (size_t)j * ld, *w = sor ? wt : V + (size_t)(j + 1) * ld;
      if (!sor || j == 0) M->apply(vj, z, s, true);
      int parts;
      if (by_row) {
        parts = gram_row(j, z, w, s);
      } else {
        csr_apply<T>(A, EPI_Y, z, nullptr, nullptr, 0.0, w, s, true, OP_NONE, nullptr, ws);
        parts = gram(j, w, s);
      }
      Scal *next = twin_scal(s);
      if (sor && j + 1 < steps) {
        arnoldi_sor(*sor, j, w, vj + ld, parts, s, next);
        s = next;
        sor->rest(vj + ld, z, s, true);
        continue;
      }
      hipLaunchKernelGGL((k_gm_arnoldi<T>), dim3(eb), dim3(kBlock), 0, stream(), j, n, w, parts, ws.current(), s, next,
                         L);
      s = next;
    }
    enq += steps;
    CFDLA_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_gm_solve, dim3(1), dim3(64), 0, stream(), s, L);
    hipLaunchKernelGGL((k_gm_combine<T>), dim3(eb), dim3(kBlock), 0, stream(), n, V, ld, s, L, u);
    M->apply(u, z, s, false);
    hipLaunchKernelGGL((k_axpy1<T>), dim3(eb), dim3(kBlock), 0, stream(), n, z, x);
    CFDLA_HIP(hipGetLastError());
    Scal h = c.read(s);
    o.iters = h.iters;
    beta = residual_norm<T>(A, b, x, r, s);
    o.rn = beta;
    if (beta <= thr || (!confirm && h.done == 1)) {
      o.term = CFDLA_TERM_CONVERGED;
      return o;
    }
    if (h.done == 4 && h.kstep == 0) {
      o.term = CFDLA_TERM_BREAKDOWN;
      return o;
    }
    if (enq >= max_it) {
      o.term = CFDLA_TERM_MAX_ITERATIONS;
      return o;
    }
    if (!std::isfinite(beta)) {
      o.term = CFDLA_TERM_BREAKDOWN;
      return o;
    }
  }
}

}  // namespace

int restart_width(const cfdla_solver_config &cfg) {
  int req = cfg.restart > 0 ? cfg.restart : 30;
  if (cfg.restart_ladder) {
    if (req <= 8) return 8;
    if (req <= 16) return 16;
    if (req <= 32) return 32;
    if (req <= 64) return 64;
    if (req <= 128) return 128;
    return 256;
  }
  return std::min(req, 256);
}

SolveOut gmres_fp64(const DevCsr &A, Precond *M, const double *b, double *x, double thr,
                    const cfdla_solver_config &cfg) {
  return gmres<double>(A, M, b, x, thr, cfg.max_iter, restart_width(cfg), true);
}

SolveOut gmres_fp32_inner(const DevCsr &A, Precond *M, const float *b, float *x, double thr, int64_t max_it,
                          const cfdla_solver_config &cfg) {
  return gmres<float>(A, M, b, x, thr, max_it, restart_width(cfg), false);
}

}  // namespace cfdla
