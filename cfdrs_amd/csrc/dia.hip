// Diagonal-format (DIA) products of libcfdla for stencil matrices.
//
// One lane per row, rows dealt in 256-row tiles: on every stored diagonal a
// wavefront reads 64 consecutive values (512 B FP64 / 256 B FP32), and no
// column index is stored, so a symmetric 7-point operator moves 4 values per
// row (main diagonal + 3 upper ones) where CSR moves 7 values and 7 indices.
// The lower entries of a symmetric matrix are the upper ones of the rows
// above (a(i, i - d) = a(i - d, i)): the same diagonal array read d rows
// back, which the L2 of the XCD still holds (the tiles of an XCD are
// contiguous, and d rows are at most one grid plane).
//
// Entries are summed in ascending column order, as a sequential CSR row sum.
// Structurally absent entries (zero on the diagonal arrays) are skipped, so
// a non-finite x at an absent column does not leak into the row.
//
// Tiles are split into 8 contiguous ranges, one per XCD (block b runs on XCD
// b % 8), so the x gathers of neighbouring rows hit the L2 of the XCD that
// owns them.
#include "epilogue.hpp"
#include "finalize.hpp"
#include "internal.hpp"
#include "reduce.hpp"

namespace cfdla {
namespace {

// EPI_DIR on a stopped solve: the product is skipped, but the new-direction
// buffer still receives the current direction, so the caller's buffer swap
// keeps pointing at the latest one when the iteration resumes (after a
// residual replacement).  Every block copies its strips, also one that has no
// tile of the product.
template <typename T>
__device__ __forceinline__ void keep_direction(int n, const T *__restrict__ p, T *__restrict__ pn) {
  for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) pn[i] = p[i];
}

// A block of a consuming product (CONS below) that the dealing of the tiles
// left without one: the tile loop, where the others learn that the solve has
// stopped, does not run there.
template <typename T>
__device__ __forceinline__ void idle_direction(int n, const T *__restrict__ p, T *__restrict__ pn, const Pend &pd,
                                               int check_done) {
  __shared__ Scal sc;
  consume(pd, sc);
  if (check_done && sc.done) keep_direction(n, p, pn);
}

// CONS: the reduction before this product is still pending (finalize.hpp).
// Every load of the block's tile is issued, then the block sums the partials
// and advances the scalars while they are in flight; one tile per block.
template <typename T, int EPI, bool DOT, bool SYM, int ND, bool CONS>
__global__ __launch_bounds__(kBlock) void k_dia(int n, DiaDesc dd, const T *__restrict__ dv,
                                                const T *__restrict__ x, const T *__restrict__ b,
                                                const T *__restrict__ dinv, T omega, T *y, const T *dotw, Scal *s,
                                                int check_done, double *partials, T *y2, Pend pd) {
  if constexpr (!CONS) {
    if (check_done && s->done) {
      if constexpr (EPI == EPI_DIR) keep_direction(n, x, y2);
      return;
    }
    if constexpr (EPI == EPI_DIR) omega = (T)s->beta;
  }
  // entries per row in column order: SYM lower k = ND-1..1, main, upper k = 1..ND-1
  constexpr int NS = SYM ? 2 * ND - 1 : ND;
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3, per = gridDim.x >> 3;
  const int tiles = (n + kBlock - 1) / kBlock;
  const int chunk = (tiles + 7) >> 3;
  const int t1 = min(tiles, xcd * chunk + chunk);
  double dacc[EPI == EPI_DOT2 ? 2 : 1] = {};
  if constexpr (CONS && EPI == EPI_DIR) {
    if (xcd * chunk + local >= t1) idle_direction(n, x, y2, pd, check_done);
  }
  for (int t = xcd * chunk + local; t < t1; t += per) {
    const int mine = t * kBlock + (int)threadIdx.x;
    const bool live = mine < n;
    if constexpr (!CONS) {
      if (!live) continue;
    }
    const int row = CONS && !live ? n - 1 : mine;
    EpiIn<T> e = epi_load<T, EPI, DOT>(row, x, b, dinv, omega, y, dotw);
    T ou = T(0), ow = T(0);  // the row's own direction operands
    if constexpr (CONS && EPI == EPI_DIR) gather_raw<T, EPI>(row, x, b, dinv, ou, ow);
    // Branch-free: every value and gather load is issued before the sums;
    // an out-of-range column re-reads row's own slot and is masked.
    int c[NS];
    bool ok[NS];
    T v[NS], gu[NS], gw[NS];
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      const bool lower = SYM && j < ND - 1;
      const int k = lower ? ND - 1 - j : (SYM ? j - (ND - 1) : j);
      const int col = lower ? row - dd.off[k] : row + dd.off[k];
      ok[j] = col >= 0 && col < n;
      c[j] = ok[j] ? col : row;
      v[j] = dv[k * n + (lower && ok[j] ? col : row)];
    }
#pragma unroll
    for (int j = 0; j < NS; ++j) gather_raw<T, EPI>(c[j], x, b, dinv, gu[j], gw[j]);
    if constexpr (CONS) {
      __shared__ Scal sc;
      consume(pd, sc);
      if (check_done && sc.done) {
        if constexpr (EPI == EPI_DIR) keep_direction(n, x, y2);
        return;
      }
      if constexpr (EPI == EPI_DIR) {
        omega = (T)sc.beta;
        e.x = gather_combine<T, EPI>(ou, ow, omega);
      }
    }
    T sum = T(0);
#pragma unroll
    for (int j = 0; j < NS; ++j)
      sum += (ok[j] && v[j] != T(0)) ? v[j] * gather_combine<T, EPI>(gu[j], gw[j], omega) : T(0);
    if (live) {
      epi_store<T, EPI, DOT>(e, row, sum, omega, y, dotw, dacc[0], y2);
      if constexpr (EPI == EPI_DOT2) dacc[1] += (double)sum * (double)sum;
    }
    if constexpr (CONS) break;
  }
  if constexpr (DOT) block_partials<EPI == EPI_DOT2 ? 2 : 1>(dacc, partials);
}

// ---- R rows per lane, 16-byte loads ------------------------------------------
// The same product with R consecutive rows per lane (R = 2 in FP64), so
// every diagonal, x, epilogue and y access is one 16-byte load or store per
// lane.  It applies to symmetric storage when n is a multiple of R, the first
// off-diagonal offset is 1 and the others are multiples of R (the 2D 5-point
// and 3D 7-point operators with nx % R == 0): a multiple-of-R offset keeps a
// lane's R columns one aligned vector, and the unit offset takes its R - 1
// inner neighbours from the lane's own main-diagonal vectors plus one scalar
// load at each end.
// Each row sums the same terms in the same column order as k_dia.
template <typename T, int R>
using vec_t = T __attribute__((ext_vector_type(R)));

template <typename T, int R>
__device__ __forceinline__ void ldv(const T *p, T (&o)[R]) {
  const vec_t<T, R> v = *reinterpret_cast<const vec_t<T, R> *>(p);
#pragma unroll
  for (int r = 0; r < R; ++r) o[r] = v[r];
}

// loaded operands of the gathers at the R aligned columns c..c+R-1 (gather_raw)
template <typename T, int EPI, int R>
__device__ __forceinline__ void gatherv(int c, const T *__restrict__ x, const T *__restrict__ b,
                                        const T *__restrict__ dinv, T (&u)[R], T (&w)[R]) {
  if constexpr (EPI == EPI_JACOBI0) {
    ldv<T, R>(dinv + c, u);
    ldv<T, R>(b + c, w);
  } else {
    ldv<T, R>(x + c, u);
    if constexpr (EPI == EPI_DIR) ldv<T, R>(b + c, w);
  }
}

template <typename T, int EPI, bool DOT, int ND, int R, bool CONS>
__global__ __launch_bounds__(kBlock) void k_dia_vec(int n, DiaDesc dd, const T *__restrict__ dv,
                                                    const T *__restrict__ x, const T *__restrict__ b,
                                                    const T *__restrict__ dinv, T omega, T *y, const T *dotw,
                                                    Scal *s, int check_done, double *partials, T *y2, Pend pd) {
  if constexpr (!CONS) {
    if (check_done && s->done) {
      if constexpr (EPI == EPI_DIR) keep_direction(n, x, y2);
      return;
    }
    if constexpr (EPI == EPI_DIR) omega = (T)s->beta;
  }
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3, per = gridDim.x >> 3;
  const int groups = n / R;
  const int tiles = (groups + kBlock - 1) / kBlock;
  const int chunk = (tiles + 7) >> 3;
  const int t1 = min(tiles, xcd * chunk + chunk);
  double dacc[EPI == EPI_DOT2 ? 2 : 1] = {};
  if constexpr (CONS && EPI == EPI_DIR) {
    if (xcd * chunk + local >= t1) idle_direction(n, x, y2, pd, check_done);
  }
  for (int t = xcd * chunk + local; t < t1; t += per) {
    const int g = t * kBlock + (int)threadIdx.x;
    const bool live = g < groups;
    if constexpr (!CONS) {
      if (!live) continue;
    }
    const int row = (CONS && !live ? groups - 1 : g) * R;
    // epilogue operands, then every entry and gather load before the sums
    EpiIn<T> e[R];
    {
      T tb[R], td[R], tx[R], ty[R], tw[R];
      if constexpr (EPI == EPI_RESID || EPI == EPI_JACOBI || EPI == EPI_JACOBI0) ldv<T, R>(b + row, tb);
      if constexpr (EPI == EPI_JACOBI || EPI == EPI_JACOBI0) ldv<T, R>(dinv + row, td);
      if constexpr (EPI == EPI_JACOBI) ldv<T, R>(x + row, tx);
      if constexpr (EPI == EPI_ADD) ldv<T, R>(y + row, ty);
      if constexpr (DOT && EPI != EPI_DIR) {
        if (dotw != y) ldv<T, R>(dotw + row, tw);
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        e[r] = EpiIn<T>{T(0), T(0), T(0), T(0), T(0)};
        if constexpr (EPI == EPI_RESID || EPI == EPI_JACOBI || EPI == EPI_JACOBI0) e[r].b = tb[r];
        if constexpr (EPI == EPI_JACOBI) {
          e[r].d = td[r];
          e[r].x = tx[r];
        }
        if constexpr (EPI == EPI_JACOBI0) {
          e[r].d = td[r];
          e[r].x = omega * td[r] * tb[r];
        }
        if constexpr (EPI == EPI_ADD) e[r].y = ty[r];
        if constexpr (DOT && EPI != EPI_DIR) {
          if (dotw != y) e[r].w = tw[r];
        }
      }
    }
    // main diagonal and the operand at the lane's own columns
    // (loads only; the gathered operands are combined below, once omega is known)
    T vm[R], mu[R], mw[R];
    ldv<T, R>(dv + row, vm);
    gatherv<T, EPI, R>(row, x, b, dinv, mu, mw);
    // off-diagonals: lower (column row + r - off) and upper (row + r + off)
    T vl[ND][R], lu[ND][R], lw[ND][R], vu[ND][R], uu[ND][R], uw[ND][R];
    bool okl[ND][R], oku[ND][R];
#pragma unroll
    for (int k = 1; k < ND; ++k) {
      const int off = dd.off[k];
      const T *dk = dv + (size_t)k * n;
      ldv<T, R>(dk + row, vu[k]);
      if (k == 1) {  // off == 1
        // inner neighbours come from the lane's own vectors
        const bool okf = row > 0, okb = row + R < n;
        const T vfirst = dk[okf ? row - 1 : row];
        gather_raw<T, EPI>(okf ? row - 1 : row, x, b, dinv, lu[k][0], lw[k][0]);
        gather_raw<T, EPI>(okb ? row + R : row, x, b, dinv, uu[k][R - 1], uw[k][R - 1]);
#pragma unroll
        for (int r = 0; r < R; ++r) {
          vl[k][r] = r == 0 ? vfirst : vu[k][r - 1];
          okl[k][r] = r > 0 || okf;
          oku[k][r] = r < R - 1 || okb;
        }
      } else {
        // whole vectors are in or out of range (row, off and n are multiples of R)
        const bool okL = row - off >= 0, okU = row + off < n;
        ldv<T, R>(dk + (okL ? row - off : row), vl[k]);
        gatherv<T, EPI, R>(okL ? row - off : row, x, b, dinv, lu[k], lw[k]);
        gatherv<T, EPI, R>(okU ? row + off : row, x, b, dinv, uu[k], uw[k]);
#pragma unroll
        for (int r = 0; r < R; ++r) {
          okl[k][r] = okL;
          oku[k][r] = okU;
        }
      }
    }
    if constexpr (CONS) {
      __shared__ Scal sc;
      consume(pd, sc);
      if (check_done && sc.done) {
        if constexpr (EPI == EPI_DIR) keep_direction(n, x, y2);
        return;
      }
      if constexpr (EPI == EPI_DIR) omega = (T)sc.beta;
    }
    T xm[R], xl[ND][R], xu[ND][R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      xm[r] = gather_combine<T, EPI>(mu[r], mw[r], omega);
      if constexpr (EPI == EPI_DIR) e[r].x = xm[r];  // the direction at the lane's own rows
    }
#pragma unroll
    for (int k = 1; k < ND; ++k)
#pragma unroll
      for (int r = 0; r < R; ++r) {
        xl[k][r] = k == 1 && r > 0 ? xm[r - 1] : gather_combine<T, EPI>(lu[k][r], lw[k][r], omega);
        xu[k][r] = k == 1 && r < R - 1 ? xm[r + 1] : gather_combine<T, EPI>(uu[k][r], uw[k][r], omega);
      }
    T out[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      // column order: lower k = ND-1..1, main, upper k = 1..ND-1
      T sum = T(0);
#pragma unroll
      for (int k = ND - 1; k >= 1; --k)
        sum += (okl[k][r] && vl[k][r] != T(0)) ? vl[k][r] * xl[k][r] : T(0);
      sum += vm[r] != T(0) ? vm[r] * xm[r] : T(0);
#pragma unroll
      for (int k = 1; k < ND; ++k)
        sum += (oku[k][r] && vu[k][r] != T(0)) ? vu[k][r] * xu[k][r] : T(0);
      out[r] = epi_out<T, EPI>(e[r], sum, omega);
      if constexpr (DOT) {
        if (live) {
          dacc[0] += (double)(EPI == EPI_DIR ? e[r].x : (dotw == y ? out[r] : e[r].w)) * (double)out[r];
          if constexpr (EPI == EPI_DOT2) dacc[1] += (double)out[r] * (double)out[r];
        }
      }
    }
    if (CONS && !live) break;
    vec_t<T, R> ov;
#pragma unroll
    for (int r = 0; r < R; ++r) ov[r] = out[r];
    *reinterpret_cast<vec_t<T, R> *>(y + row) = ov;
    if constexpr (EPI == EPI_DIR) {
      vec_t<T, R> pv;
#pragma unroll
      for (int r = 0; r < R; ++r) pv[r] = e[r].x;
      *reinterpret_cast<vec_t<T, R> *>(y2 + row) = pv;
    }
    if constexpr (CONS) break;
  }
  if constexpr (DOT) block_partials<EPI == EPI_DOT2 ? 2 : 1>(dacc, partials);
}

// Products that follow a reduction within an iteration take it along while it
// is pending: the CG direction, the first product of a V-cycle (the residual
// where the update has made the first sweeps), BiCGSTAB's second product.
template <int EPI, bool DOT>
constexpr bool consumes() {
  return EPI == EPI_DIR || EPI == EPI_JACOBI0 || EPI == EPI_DOT2 || (EPI == EPI_RESID && !DOT);
}

template <typename T, int EPI, bool DOT, bool SYM, int ND>
void launch_shape(const DevCsr &A, int blocks, const T *x, const T *b, const T *dinv, double omega, T *y,
                  const T *dotw, Scal *s, bool check_done, RedWs &ws, T *y2) {
  double *part = DOT ? nullptr : ws.partials.p;
  if constexpr (consumes<EPI, DOT>()) {
    if (pending_on(s) && blocks <= kConsumeBlocks) {
      const Pend pd = take_pending(s);
      if (DOT) part = ws.next();
      hipLaunchKernelGGL((k_dia<T, EPI, DOT, SYM, ND, true>), dim3(blocks), dim3(kBlock), 0, stream(), A.n, A.dia_desc,
                         A.dia_vals<T>(), x, b, dinv, (T)omega, y, dotw, pd.out, check_done ? 1 : 0, part, y2, pd);
      return;
    }
  }
  s = settled_scal(s);
  if (DOT) part = ws.next();
  hipLaunchKernelGGL((k_dia<T, EPI, DOT, SYM, ND, false>), dim3(blocks), dim3(kBlock), 0, stream(), A.n, A.dia_desc,
                     A.dia_vals<T>(), x, b, dinv, (T)omega, y, dotw, s, check_done ? 1 : 0, part, y2, Pend{});
}

template <typename T, int EPI, bool DOT, int ND, int R>
void launch_vec(const DevCsr &A, const T *x, const T *b, const T *dinv, double omega, T *y, const T *dotw,
                Scal *s, bool check_done, RedWs &ws, int blocks, T *y2) {
  double *part = DOT ? nullptr : ws.partials.p;
  if constexpr (consumes<EPI, DOT>()) {
    if (pending_on(s) && blocks <= kConsumeBlocks) {
      const Pend pd = take_pending(s);
      if (DOT) part = ws.next();
      hipLaunchKernelGGL((k_dia_vec<T, EPI, DOT, ND, R, true>), dim3(blocks), dim3(kBlock), 0, stream(), A.n,
                         A.dia_desc, A.dia_vals<T>(), x, b, dinv, (T)omega, y, dotw, pd.out, check_done ? 1 : 0, part,
                         y2, pd);
      return;
    }
  }
  s = settled_scal(s);
  if (DOT) part = ws.next();
  hipLaunchKernelGGL((k_dia_vec<T, EPI, DOT, ND, R, false>), dim3(blocks), dim3(kBlock), 0, stream(), A.n, A.dia_desc,
                     A.dia_vals<T>(), x, b, dinv, (T)omega, y, dotw, s, check_done ? 1 : 0, part, y2, Pend{});
}

// The PCG update and the first two Jacobi sweeps of the V-cycle that follows it
// on symmetric diagonal storage, in one pass: x += alpha p, rn = r - alpha q
// with its norm, and the sweeps of rn from zero (EPI_JACOBI0), whose neighbours'
// entries of rn are formed at the gathers as the own one is.  rn is not r:
// other blocks still read that.  Bound by latency: a launch saved per iteration
// is the gain, three gathers per entry instead of two the cost.  On 97,665 rows
// 5.5 us, and 4.2 for the residual product that now finishes the norm, against
// 4.5, 4.3 and 3.2; FP64 AMG-PCG solves of five-point systems, 64x64 / 100x90 /
// 200x151 / 383x255 / 512x512: 0.53 / 0.605 / 0.78 / 0.945 / 1.38 ms with two
// launches, 0.50 / 0.57 / 0.735 / 0.905 / 1.33 ms.
template <typename T, int ND>
__global__ __launch_bounds__(kBlock) void k_cg_start(int n, DiaDesc dd, const T *__restrict__ dv,
                                                     const T *__restrict__ r, const T *__restrict__ q,
                                                     const T *__restrict__ dinv, T omega, const T *__restrict__ p,
                                                     T *__restrict__ x, T *__restrict__ rn, T *__restrict__ y,
                                                     double *partials, Pend pd) {
  constexpr int NS = 2 * ND - 1;
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int chunk = ((n + kBlock - 1) / kBlock + 7) >> 3;
  const int mine = (xcd * chunk + local) * kBlock + (int)threadIdx.x;
  const bool live = local < chunk && mine < n;
  const int row = live ? mine : n - 1;
  int c[NS];
  bool ok[NS];
  T v[NS], rv[NS], qv[NS], jv[NS];
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    const bool lower = j < ND - 1;
    const int k = lower ? ND - 1 - j : j - (ND - 1);
    const int col = lower ? row - dd.off[k] : row + dd.off[k];
    ok[j] = col >= 0 && col < n;
    c[j] = ok[j] ? col : row;
    v[j] = dv[k * n + (lower && ok[j] ? col : row)];
  }
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    rv[j] = r[c[j]];
    qv[j] = q[c[j]];
    jv[j] = dinv[c[j]];
  }
  const T r0 = r[row], q0 = q[row], d0 = dinv[row], p0 = p[row], x0 = x[row];
  __shared__ Scal sc;
  consume(pd, sc);
  if (sc.done) return;
  const T alpha = (T)sc.alpha;
  const T ri = r0 - alpha * q0;
  T sum = T(0);
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    const T rj = rv[j] - alpha * qv[j];
    sum += (ok[j] && v[j] != T(0)) ? v[j] * (omega * jv[j] * rj) : T(0);
  }
  double acc[1] = {0.0};
  if (live) {
    x[row] = x0 + alpha * p0;
    rn[row] = ri;
    y[row] = omega * d0 * ri + omega * d0 * (ri - sum);
    acc[0] = (double)ri * (double)ri;
  }
  block_partials<1>(acc, partials);
}

bool aligned(const void *p, size_t bytes) { return (reinterpret_cast<uintptr_t>(p) & (bytes - 1)) == 0; }

// Rows per lane of the 16-byte-load product for this operator and these
// vectors, or 1 when its conditions do not hold.
// FP64 only: in FP32 the 4-row form measured no faster in the 128^3 solve
// (Jacobi sweep 11.4 against 10.8 us, y = A x 9.7 against 9.6 us; 2 rows per
// lane slower still), since at 50 MB per pass launch and ramp-up dominate.
template <typename T>
constexpr int dia_r() { return sizeof(T) == 8 ? 2 : 1; }

template <typename T>
int dia_rows_per_lane(const DevCsr &A, const void *x, const void *b, const void *dinv, const void *y,
                      const void *dotw, const void *y2) {
  constexpr int R = dia_r<T>();
  if (R == 1) return 1;
  const DiaDesc &d = A.dia_desc;
  if (!d.sym || d.nd < 2 || d.nd > 4 || A.n % R != 0) return 1;
  if (d.off[1] != 1) return 1;
  for (int k = 2; k < d.nd; ++k)
    if (d.off[k] % R != 0) return 1;
  for (const void *p : {x, b, dinv, y, dotw, y2, static_cast<const void *>(A.dia_vals<T>())})
    if (p != nullptr && !aligned(p, R * sizeof(T))) return 1;
  return R;
}

}  // namespace

// Instantiated shapes: symmetric with 2..5 stored diagonals (1D 3-point,
// 2D 5-point, 3D 7-point, 2D 9-point), general with 3, 5, 7 or 9.
bool dia_supported(const DiaDesc &d) {
  if (d.sym) return d.nd >= 2 && d.nd <= 5 && d.off[0] == 0;
  return d.nd == 3 || d.nd == 5 || d.nd == 7 || d.nd == 9;
}

template <typename T, int EPI, bool DOT>
void launch_dia(const DevCsr &A, const T *x, const T *b, const T *dinv, double omega, T *y, const T *dotw,
                Scal *s, bool check_done, int op, RedWs &ws, T *y2) {
  // one 256-row tile per block up to the partials capacity: blocks that
  // finish hand their CU to the next tile without a loop-carried wait
  // (26.2 us against 29.1 us with 4 tiles per block, FP64 y = A x, 128^3)
  const DiaDesc &d = A.dia_desc;
  constexpr int R = dia_r<T>();
  if constexpr (R > 1) {
    if (dia_rows_per_lane<T>(A, x, b, dinv, y, dotw, y2) == R) {
      const int vblocks = xcd_grid((A.n / R + kBlock - 1) / kBlock, 1, kMaxBlocks);
      switch (d.nd) {
        case 2: launch_vec<T, EPI, DOT, 2, R>(A, x, b, dinv, omega, y, dotw, s, check_done, ws, vblocks, y2); break;
        case 3: launch_vec<T, EPI, DOT, 3, R>(A, x, b, dinv, omega, y, dotw, s, check_done, ws, vblocks, y2); break;
        default: launch_vec<T, EPI, DOT, 4, R>(A, x, b, dinv, omega, y, dotw, s, check_done, ws, vblocks, y2); break;
      }
      if (DOT) finish(EPI == EPI_DOT2 ? 2 : 1, s, op, vblocks, ws, check_done);
      return;
    }
  }
  const int blocks = xcd_grid((A.n + kBlock - 1) / kBlock, 1, kMaxBlocks);
#define CFDLA_DIA(SYM, ND) launch_shape<T, EPI, DOT, SYM, ND>(A, blocks, x, b, dinv, omega, y, dotw, s, check_done, ws, y2)
  if (d.sym) {
    switch (d.nd) {
      case 2: CFDLA_DIA(true, 2); break;
      case 3: CFDLA_DIA(true, 3); break;
      case 4: CFDLA_DIA(true, 4); break;
      case 5: CFDLA_DIA(true, 5); break;
      default: throw Error(CFDLA_ERR_INVALID_ARG, "unsupported symmetric diagonal count");
    }
  } else {
    switch (d.nd) {
      case 3: CFDLA_DIA(false, 3); break;
      case 5: CFDLA_DIA(false, 5); break;
      case 7: CFDLA_DIA(false, 7); break;
      case 9: CFDLA_DIA(false, 9); break;
      default: throw Error(CFDLA_ERR_INVALID_ARG, "unsupported diagonal count");
    }
  }
#undef CFDLA_DIA
  if (DOT) finish(EPI == EPI_DOT2 ? 2 : 1, s, op, blocks, ws, check_done);
}

// At most five entries per row: with seven the gathers eat the launch saved
// (32^3 and 64^3 rows 0.80 and 1.565 ms, fused 0.81 and 1.58).  Its norm stays
// pending for the residual product, hence the limit of kConsumeBlocks.
template <typename T>
bool cg_start_takes(const DevCsr &A) {
  return A.dia && A.dia_vals<T>() != nullptr && dia_supported(A.dia_desc) && A.dia_desc.sym && A.dia_desc.nd <= 3 &&
         xcd_grid((A.n + kBlock - 1) / kBlock, 1, kMaxBlocks) <= kConsumeBlocks;
}

template <typename T>
void cg_start(const DevCsr &A, const T *r, const T *q, const T *dinv, double omega, const T *p, T *x, T *rn, T *y,
              Scal *s, RedWs &ws) {
  const int blocks = xcd_grid((A.n + kBlock - 1) / kBlock, 1, kMaxBlocks);
  const Pend pd = take_pending(s);
  double *part = ws.next();
#define CFDLA_START(ND)                                                                                        \
  hipLaunchKernelGGL((k_cg_start<T, ND>), dim3(blocks), dim3(kBlock), 0, stream(), A.n, A.dia_desc,             \
                     A.dia_vals<T>(), r, q, dinv, (T)omega, p, x, rn, y, part, pd)
  if (A.dia_desc.nd == 2) CFDLA_START(2);
  else CFDLA_START(3);
#undef CFDLA_START
  CFDLA_HIP(hipGetLastError());
  finish(1, s, OP_CG_RR, blocks, ws, true);
}
template bool cg_start_takes<double>(const DevCsr &);
template bool cg_start_takes<float>(const DevCsr &);
template void cg_start<double>(const DevCsr &, const double *, const double *, const double *, double, const double *,
                               double *, double *, double *, Scal *, RedWs &);
template void cg_start<float>(const DevCsr &, const float *, const float *, const float *, double, const float *,
                              float *, float *, float *, Scal *, RedWs &);

#define CFDLA_DIA_INST(T, E)                                                                                   \
  template void launch_dia<T, E, false>(const DevCsr &, const T *, const T *, const T *, double, T *, const T *, \
                                        Scal *, bool, int, RedWs &, T *);                                      \
  template void launch_dia<T, E, true>(const DevCsr &, const T *, const T *, const T *, double, T *, const T *,  \
                                       Scal *, bool, int, RedWs &, T *);
#define CFDLA_DIA_ALL(T)         \
  CFDLA_DIA_INST(T, EPI_Y)       \
  CFDLA_DIA_INST(T, EPI_RESID)   \
  CFDLA_DIA_INST(T, EPI_JACOBI)  \
  CFDLA_DIA_INST(T, EPI_ADD)     \
  CFDLA_DIA_INST(T, EPI_JACOBI0) \
  template void launch_dia<T, EPI_DIR, true>(const DevCsr &, const T *, const T *, const T *, double, T *, const T *, \
                                             Scal *, bool, int, RedWs &, T *);                                   \
  template void launch_dia<T, EPI_DOT2, true>(const DevCsr &, const T *, const T *, const T *, double, T *, const T *, \
                                              Scal *, bool, int, RedWs &, T *);
CFDLA_DIA_ALL(double)
CFDLA_DIA_ALL(float)

}  // namespace cfdla
