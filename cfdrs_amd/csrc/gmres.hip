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

constexpr int kMdotBlocks = 512;

struct GmLayout {
  int m;
  double *H, *cs, *sn, *g, *y, *hc, *hp, *part;
  static size_t doubles(int m) { return (size_t)(m + 1) * m + 2 * m + (m + 1) + m + 2 * (m + 1) + (size_t)(m + 1) * kMdotBlocks; }
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
template <int JB>
__device__ __forceinline__ void block_sums(double (&acc)[JB], int jp1, double *__restrict__ part) {
  static_assert(JB % 4 == 0, "four rows of 16 lanes hold a quarter of the sums each");
  __shared__ double sh[kBlock / 64][JB];
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
  for (int k = threadIdx.x; k < jp1; k += kBlock) {
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) t += sh[w][k];
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
  if constexpr (DOTS) block_sums<JB>(acc, jp1, part);
  if constexpr (NORM) block_partials<1>(nv, part);
}

// ||w|| from its partials, v_{j+1} = w / ||w|| in place, and (block 0) the
// Hessenberg column j, Givens rotation and residual estimate.  Every block
// sums the partials itself; the scalars go from in to out, so no block reads
// what block 0 has already advanced.  Block 0 stages the column and the
// earlier rotations in LDS, so thread 0's rotation chain waits on arithmetic,
// not on global memory, beside the other blocks' scaling (4.8 us; 3.7 + 2.9 us
// with the scaling as a launch of its own, 147,456 rows).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_gm_arnoldi(int j, int n, T *__restrict__ w, int nblocks,
                                                       const double *partials, const Scal *in, Scal *out, GmLayout L) {
  __shared__ double col[258], cs[256], sn[256];
  const int tid = threadIdx.x;
  constexpr int kWords = sizeof(Scal) / sizeof(int);
  const bool first = blockIdx.x == 0;
  if (in->done) {
    if (first && tid < kWords) reinterpret_cast<int *>(out)[tid] = reinterpret_cast<const int *>(in)[tid];
    return;
  }
  const int i0 = blockIdx.x * kBlock + tid, step = gridDim.x * kBlock;
  T w0 = T(0);
  if (i0 < n) w0 = w[i0];
  __shared__ Scal sc;
  if (first) {
    if (tid < kWords) reinterpret_cast<int *>(&sc)[tid] = reinterpret_cast<const int *>(in)[tid];
    for (int k = tid; k <= j; k += kBlock) col[k] = L.hc[k];
    for (int k = tid; k < j; k += kBlock) {
      cs[k] = L.cs[k];
      sn[k] = L.sn[k];
    }
  }
  double tot[1];
  sum_partials<1>(nblocks, partials, tot);  // synchronizes the block
  const double hn = sqrt(tot[0]);
  const double a = hn > 0.0 ? 1.0 / hn : 0.0;
  // (a breakdown or a non-finite norm ends the cycle: the vector is not used)
  for (int i = i0; i < n; i += step) w[i] = (T)((double)(i == i0 ? w0 : w[i]) * a);
  if (!first) return;
  const int m = L.m;
  if (tid == 0) {
    sc.hn = hn;
    col[j + 1] = hn;
    for (int k = 0; k < j; ++k) {
      const double t0 = col[k], t1 = col[k + 1];
      col[k] = cs[k] * t0 + sn[k] * t1;
      col[k + 1] = -sn[k] * t0 + cs[k] * t1;
    }
    const double h0 = col[j], h1 = col[j + 1];
    const double den = hypot(h0, h1);
    if (den == 0.0 || !isfinite(den)) {
      sc.done = 4;  // breakdown: the cycle ends with kstep = j
    } else {
      const double c = h0 / den, sj = h1 / den;
      L.cs[j] = c;
      L.sn[j] = sj;
      col[j] = den;
      col[j + 1] = 0.0;
      const double gj = L.g[j];
      L.g[j + 1] = -sj * gj;
      L.g[j] = c * gj;
      sc.kstep = j + 1;
      sc.iters += 1;
      sc.alpha = a;
      if (fabs(L.g[j + 1]) <= sqrt(sc.thr2) || hn == 0.0) sc.done = 1;
    }
  }
  __syncthreads();
  if (tid < kWords) reinterpret_cast<int *>(out)[tid] = reinterpret_cast<const int *>(&sc)[tid];
  // the column as the host-visible Hessenberg H(0:j+1, j); on breakdown the
  // rotated entries up to j + 1, as before the rotation that failed
  for (int k = tid; k <= j + 1; k += kBlock) L.H[(size_t)k * m + j] = col[k];
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
  const int nb = std::min(kMdotBlocks, blocks_for(n, kBlock));
  // Gram-Schmidt over basis vectors 0..j of w.  Up to 32 vectors fit the
  // registers of k_gram (384 x 384 momentum matrix, m = 32: 16.7 us per step on
  // average against 21.6 us in the separate multi-dots and multi-axpys); a
  // longer basis takes those.
  auto gram = [&](int j, T *w, Scal *sc) {
    const int jp1 = j + 1;
    auto fin = [&](int pass) {
      hipLaunchKernelGGL(k_mdot_fin, dim3(jp1), dim3(kBlock), 0, stream(), nb, L.part, L.hp, L.hc, pass == 0 ? 1 : 0,
                         sc);
    };
#define CFDLA_GRAM(JB)                                                                                                \
  do {                                                                                                                \
    hipLaunchKernelGGL((k_gram<T, JB, false, true, false>), dim3(nb), dim3(kBlock), 0, stream(), n, jp1, V, ld, L.hp, \
                       w, sc, L.part);                                                                                \
    fin(0);                                                                                                           \
    hipLaunchKernelGGL((k_gram<T, JB, true, true, false>), dim3(nb), dim3(kBlock), 0, stream(), n, jp1, V, ld, L.hp,  \
                       w, sc, L.part);                                                                                \
    fin(1);                                                                                                           \
    hipLaunchKernelGGL((k_gram<T, JB, true, false, true>), dim3(nb), dim3(kBlock), 0, stream(), n, jp1, V, ld, L.hp,  \
                       w, sc, ws.current());                                                                          \
    return nb;                                                                                                        \
  } while (0)
    if (jp1 <= 4) CFDLA_GRAM(4);
    if (jp1 <= 8) CFDLA_GRAM(8);
    if (jp1 <= 16) CFDLA_GRAM(16);
    if (jp1 <= 24) CFDLA_GRAM(24);
    if (jp1 <= 32) CFDLA_GRAM(32);
#undef CFDLA_GRAM
    for (int pass = 0; pass < 2; ++pass) {
      hipLaunchKernelGGL((k_mdot<T>), dim3(nb, jp1), dim3(kBlock), 0, stream(), n, V, ld, w, L.part, sc);
      fin(pass);
      if (pass == 0)
        hipLaunchKernelGGL((k_maxpy<T, false>), dim3(eb), dim3(kBlock), 0, stream(), n, jp1, V, ld, L.hp, w, sc,
                           nullptr);
      else
        hipLaunchKernelGGL((k_maxpy<T, true>), dim3(eb), dim3(kBlock), 0, stream(), n, jp1, V, ld, L.hp, w, sc,
                           ws.current());
    }
    return eb;
  };
  int64_t enq = 0;
  while (true) {
    // the residual's read left no reduction pending, and the cycle's kernels
    // start none: the scalars stay where they are until its end
    s = settled_scal(s);
    hipLaunchKernelGGL((k_gm_restart<T>), dim3(eb), dim3(kBlock), 0, stream(), n, r, beta, V, s, L);
    int steps = (int)std::min<int64_t>(m, max_it - enq);
    for (int j = 0; j < steps; ++j) {
      T *vj = V + (size_t)j * ld, *w = V + (size_t)(j + 1) * ld;
      M->apply(vj, z, s, true);
      csr_apply<T>(A, EPI_Y, z, nullptr, nullptr, 0.0, w, s, true, OP_NONE, nullptr, ws);
      const int parts = gram(j, w, s);
      Scal *next = twin_scal(s);
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
