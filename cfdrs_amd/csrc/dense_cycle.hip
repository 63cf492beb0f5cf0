// The V-cycle from a small level on as one dense operator.
//
// From the zero guess a V-cycle is linear in its right-hand side.  Below about
// 2,000 rows it is a dozen launches or colour steps of pure latency per level,
// while its matrix, formed once per set of level values, is at most 33 MB that
// the eight L2s and the memory-side cache hold between applications: x = C b is
// one launch.  C is formed on the device by running the cycle itself on the
// columns of the identity, all at once (Jacobi: sparse times dense products over
// the columns; Gauss-Seidel: the one-workgroup tail, one workgroup per column).
//
// One application, alone / with 12 MB of other data between two: 889 rows 2.7 /
// 2.9 us, 1,186 rows 3.9 / 4.0, 1,564 rows 4.2 / 6.2, 1,858 rows 4.5 / 8.5, 2,048
// rows 5.3 / 10.5, against 14.5 us in the five launches of two Jacobi levels and
// some 65 us in the Gauss-Seidel tail.  Forming it takes 0.13 ms for 1,564 rows
// (Jacobi) and some 0.3 ms for 889 rows (Gauss-Seidel).  AMG-PCG on 383x255 1.00 ->
// 0.92 ms, BiCGSTAB with the default AMG on 96x80 2.30 -> 1.39 ms, a SIMPLE step
// on 320x256 cells 3.49 -> 3.24 ms, the adjoint of a 256x256 solve 3.09 -> 2.73 ms.
// Above kDenseCycleRows the matrix no longer comes out of the caches.
#include "solver.hpp"
#include "reduce.hpp"

#include <algorithm>

namespace cfdla {
namespace {

// x = C b: one wavefront per row, the whole row in flight (16 bytes per load),
// b in LDS meanwhile.
template <typename T, int U>
__global__ __launch_bounds__(kBlock) void k_cycle_gemv(int n, int ld, const double *__restrict__ c,
                                                       const T *__restrict__ b, T *__restrict__ x,
                                                       const int *__restrict__ done) {
  const int stop = *done;  // (tested at the store, so that no load waits for it)
  __shared__ __align__(16) double bs[128 * U];
  const int lane = threadIdx.x & 63;
  const int row = (int)((blockIdx.x * (unsigned)kBlock + threadIdx.x) >> 6);
  const double *cr = c + (size_t)(row < n ? row : n - 1) * ld;
  double2 v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int j = 2 * (lane + 64 * u);
    v[u] = *reinterpret_cast<const double2 *>(cr + (j < ld ? j : 0));
  }
  for (int j = threadIdx.x; j < 128 * U; j += kBlock) bs[j] = j < n ? (double)b[j] : 0.0;
  __syncthreads();
  double acc = 0.0;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int j = 2 * (lane + 64 * u);
    const double2 w = *reinterpret_cast<const double2 *>(bs + j);
    if (j < n) acc += v[u].x * w.x;
    if (j + 1 < n) acc += v[u].y * w.y;
  }
  acc = wave_sum(acc);
  if (lane == 0 && row < n && !stop) x[row] = (T)acc;
}

// Row i of Y (columns c of ld): PLAIN: sum_j a_ij X_j; ADD: Y + that; RESID:
// E - that; JACOBI: X_i + w d_i (E_i - that).  e null: E is the identity.
// A wavefront takes a row and 128 columns, 16 bytes per lane, a block four
// consecutive rows of the same columns, and all blocks of a column tile run on
// one XCD, whose L2 holds the tiles' part of X.  Bound by the gathered rows of
// X: a sweep over 1,564 rows of 13 entries 19 us (16 rows per block 25; tiles
// over all XCDs and 8 bytes per lane 30).
enum { MM_PLAIN, MM_ADD, MM_RESID, MM_JACOBI };
constexpr int kMmBlock = kBlock / 64;
template <int MODE>
__global__ __launch_bounds__(kBlock) void k_cycle_mm(int ld, const int32_t *__restrict__ rp,
                                                     const int32_t *__restrict__ ci, const double *__restrict__ av,
                                                     const double *__restrict__ x, const double *__restrict__ e,
                                                     const double *__restrict__ dinv, double w, int n, double *y) {
  const int tiles = (ld + 127) / 128, per = (tiles + 7) / 8, local = blockIdx.x >> 3;
  const int c = ((int)(blockIdx.x & 7) + 8 * (local % per)) * 128 + 2 * (int)(threadIdx.x & 63);
  if (c >= ld) return;
  const int i = __builtin_amdgcn_readfirstlane(local / per * kMmBlock + (int)(threadIdx.x >> 6));
  if (i >= n) return;
  const int k1 = rp[i + 1];
  double s0 = 0.0, s1 = 0.0;
  int k = rp[i];
  for (; k + 8 <= k1; k += 8) {
    double2 t[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) t[q] = *reinterpret_cast<const double2 *>(x + (size_t)ci[k + q] * ld + c);
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      s0 += av[k + q] * t[q].x;
      s1 += av[k + q] * t[q].y;
    }
  }
  for (; k < k1; ++k) {
    const double2 t = *reinterpret_cast<const double2 *>(x + (size_t)ci[k] * ld + c);
    s0 += av[k] * t.x;
    s1 += av[k] * t.y;
  }
  const size_t at = (size_t)i * ld + c;
  double2 *out = reinterpret_cast<double2 *>(y + at);
  if constexpr (MODE == MM_PLAIN) *out = make_double2(s0, s1);
  if constexpr (MODE == MM_ADD) *out = make_double2(out->x + s0, out->y + s1);
  if constexpr (MODE == MM_RESID || MODE == MM_JACOBI) {
    const double2 b =
        e ? *reinterpret_cast<const double2 *>(e + at) : make_double2(c == i ? 1.0 : 0.0, c + 1 == i ? 1.0 : 0.0);
    const double r0 = b.x - s0, r1 = b.y - s1;
    if constexpr (MODE == MM_RESID) {
      *out = make_double2(r0, r1);
    } else {
      const double2 own = *reinterpret_cast<const double2 *>(x + at);
      const double wd = w * dinv[i];
      *out = make_double2(own.x + wd * r0, own.y + wd * r1);
    }
  }
}

// y = w D E (a sweep from zero), or zero without dinv
__global__ __launch_bounds__(kBlock) void k_cycle_first(int ld, const double *__restrict__ e,
                                                        const double *__restrict__ dinv, double w, double *y) {
  const int i = blockIdx.x, c = blockIdx.y * kBlock + (int)threadIdx.x;
  if (c >= ld) return;
  const size_t at = (size_t)i * ld + c;
  y[at] = dinv ? (w * dinv[i]) * (e ? e[at] : (c == i ? 1.0 : 0.0)) : 0.0;
}

// Y = Inv X, n x n times n x ld, kMmRows rows of 64 columns per wavefront
constexpr int kMmRows = 4;
__global__ __launch_bounds__(kBlock) void k_cycle_dense(int n, int ld, const double *__restrict__ inv,
                                                        const double *__restrict__ x, double *__restrict__ y) {
  const int i0 = __builtin_amdgcn_readfirstlane((blockIdx.x * (kBlock / 64) + (int)(threadIdx.x >> 6)) * kMmRows);
  const int c = blockIdx.y * 64 + (int)(threadIdx.x & 63);
  if (c >= ld) return;
  double acc[kMmRows] = {};
  const double *row[kMmRows];
#pragma unroll
  for (int q = 0; q < kMmRows; ++q) row[q] = inv + (size_t)min(i0 + q, n - 1) * n;
  int j = 0;
  for (; j + 8 <= n; j += 8) {
    double t[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) t[u] = x[(size_t)(j + u) * ld + c];
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int q = 0; q < kMmRows; ++q) acc[q] += row[q][j + u] * t[u];
  }
  for (; j < n; ++j)
#pragma unroll
    for (int q = 0; q < kMmRows; ++q) acc[q] += row[q][j] * x[(size_t)j * ld + c];
#pragma unroll
  for (int q = 0; q < kMmRows; ++q)
    if (i0 + q < n) y[(size_t)(i0 + q) * ld + c] = acc[q];
}

// c[i ld + j] = t[j n + i], 32 x 32 tiles through LDS
__global__ __launch_bounds__(kBlock) void k_cycle_transpose(int n, int ld, const double *__restrict__ t,
                                                            double *__restrict__ c) {
  __shared__ double tile[32][33];
  const int lx = threadIdx.x & 31, ly = threadIdx.x >> 5, i0 = blockIdx.x * 32, j0 = blockIdx.y * 32;
  for (int q = ly; q < 32; q += kBlock / 32)
    if (j0 + q < n && i0 + lx < n) tile[q][lx] = t[(size_t)(j0 + q) * n + i0 + lx];
  __syncthreads();
  for (int q = ly; q < 32; q += kBlock / 32)
    if (i0 + q < n && j0 + lx < n) c[(size_t)(i0 + q) * ld + j0 + lx] = tile[lx][q];
}

struct Cycle {
  std::vector<DevLevel> &lv;
  const cfdla_amg_config &cfg;
  const double *inv;
  int ld;
  std::vector<DevBuf<double>> &ws;  // per level from the first: X, T, E

  dim3 grid(int rows, int per_block, int cols) const {
    return dim3((unsigned)((rows + per_block - 1) / per_block), (unsigned)((ld + cols - 1) / cols));
  }
  double *buf(size_t q, int k, int rows) {
    DevBuf<double> &b = ws[3 * q + (size_t)k];
    b.ensure((size_t)rows * (size_t)ld);
    return b.p;
  }
  template <int MODE>
  void mm(const DevCsr &A, const double *x, const double *e, double w, double *y) const {
    hipLaunchKernelGGL((k_cycle_mm<MODE>), dim3((unsigned)(8 * (((ld + 127) / 128 + 7) / 8) * ((A.n + kMmBlock - 1) / kMmBlock))),
                       dim3(kBlock), 0, stream(), ld, A.rp.p, A.ci.p,
                       A.v64.p, x, e, MODE == MM_JACOBI ? A.sdinv64.p : nullptr, w, A.n, y);
  }
  // X of the cycle from level l (the q-th here) for the right-hand sides e;
  // the first level's goes to out.
  double *run(size_t l, size_t q, const double *e, double *out) {
    DevLevel &L = lv[l];
    const int n = L.A.n;
    const bool last = l + 1 == lv.size();
    const double w = cfg.relaxation_factor;
    double *cur = out ? out : buf(q, 0, n), *nxt = buf(q, 1, n);
    if (last && cfg.coarse_solver == 1) {
      hipLaunchKernelGGL(k_cycle_dense, grid(n, kMmRows * kBlock / 64, 64), dim3(kBlock), 0, stream(), n, ld, inv, e,
                         cur);
      return cur;
    }
    const int down = last ? cfg.pre_smooth_iterations + 10 : cfg.pre_smooth_iterations;
    const int up = last ? 0 : cfg.post_smooth_iterations;
    // the iterate has to end in `cur` of the end: start in the other one if
    // the number of flips is odd
    if (((std::max(down, 1) - 1 + up) & 1) != 0) std::swap(cur, nxt);
    hipLaunchKernelGGL(k_cycle_first, grid(n, 1, kBlock), dim3(kBlock), 0, stream(), ld, e,
                       down > 0 ? L.A.sdinv64.p : nullptr, w, cur);
    for (int k = 1; k < down; ++k) {
      mm<MM_JACOBI>(L.A, cur, e, w, nxt);
      std::swap(cur, nxt);
    }
    if (!last) {
      mm<MM_RESID>(L.A, cur, e, 0.0, nxt);
      double *ec = buf(q + 1, 2, lv[l + 1].A.n);
      mm<MM_PLAIN>(L.R, nxt, nullptr, 0.0, ec);
      const double *xc = run(l + 1, q + 1, ec, nullptr);
      mm<MM_ADD>(L.P, xc, nullptr, 0.0, cur);
      for (int k = 0; k < up; ++k) {
        mm<MM_JACOBI>(L.A, cur, e, w, nxt);
        std::swap(cur, nxt);
      }
    }
    return cur;
  }
};
}  // namespace

template <typename T>
void DenseCycle::apply(const T *b, T *x, Scal *s, bool check_done) const {
  s = settled_scal(s);
  const dim3 blocks((unsigned)((n + kBlock / 64 - 1) / (kBlock / 64)));
#define CFDLA_GEMV(U)                                                                                             \
  hipLaunchKernelGGL((k_cycle_gemv<T, U>), blocks, dim3(kBlock), 0, stream(), n, ld, c.p, b, x, done_flag(s, check_done))
  if (ld <= 512) CFDLA_GEMV(4);
  else if (ld <= 1024) CFDLA_GEMV(8);
  else if (ld <= 1536) CFDLA_GEMV(12);
  else CFDLA_GEMV(16);
#undef CFDLA_GEMV
  CFDLA_HIP(hipGetLastError());
}
template void DenseCycle::apply<double>(const double *, double *, Scal *, bool) const;
template void DenseCycle::apply<float>(const float *, float *, Scal *, bool) const;

void DenseCycle::form_jacobi(std::vector<DevLevel> &lv, const cfdla_amg_config &cfg, const double *inv) {
  n = lv[(size_t)level].A.n;
  ld = (n + 15) / 16 * 16;
  c.ensure((size_t)n * (size_t)ld);
  ws.resize(3 * (lv.size() - (size_t)level));
  Cycle{lv, cfg, inv, ld, ws}.run((size_t)level, 0, nullptr, c.p);
  CFDLA_HIP(hipGetLastError());
}

void DenseCycle::from_columns(const double *columns) {
  hipLaunchKernelGGL(k_cycle_transpose, dim3((unsigned)((n + 31) / 32), (unsigned)((n + 31) / 32)), dim3(kBlock), 0,
                     stream(), n, ld, columns, c.p);
  CFDLA_HIP(hipGetLastError());
}

}  // namespace cfdla
