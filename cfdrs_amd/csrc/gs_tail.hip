// The small levels of a Gauss-Seidel V-cycle in one launch.
//
// The reference's default AMG (crates/cfd-math/src/linear_solver/
// preconditioners/multigrid/amg.rs:423-503 with the Gauss-Seidel smoothers of
// smoothers.rs:42-137) sweeps a handful of levels of a few thousand rows or
// fewer.  Colour by colour, one launch each, a 7,680-row hierarchy took about
// 160 launches of 4.7 us per V-cycle, nearly all of it launch latency and the
// chain perm -> row pointer -> column -> x of one row.
//
// Bound: the latency of one compute unit's L2 stream.  One workgroup of 16
// wavefronts runs every level from the first small one down and back up.  A
// barrier of the workgroup separates the colours, so a colour costs a round
// trip to its entries instead of a launch.  The iterate of the current level
// and the residual (or the coarser iterate, on the way up) live in LDS, where
// the gathers go.  The rows of a colour lie one after the other, each padded
// to the colour's longest row in groups of 4 entries, so a lane reads its row
// with 16-byte loads that depend on nothing but its position: a colour of a
// small level runs on one or two wavefronts, and their instruction count is
// its time (entries slot-major, with a mask per entry, took 1.0 us per colour
// of an 18-row level).  The last levels, which take most of the colour steps,
// are copied to LDS whole (inner levels); the larger ones are streamed from
// the L2.  A padding entry is 0 times the zero kept behind the gathered
// vector, so it adds nothing whatever the vector holds.
//
// V-cycle of the 7,680 -> 3,840 -> 977 -> 250 -> 65 -> 18 row hierarchy: about
// 760 us in launches, 154 us in one (the two largest levels 70, the coarsest
// one's 60 colour steps 28); BiCGSTAB to 1e-12 with it 11.25 -> 2.24 ms.  With
// the levels from 977 rows on as one dense operator (dense_cycle.hip) between a
// launch down and one up, 35 us each, 1.39 ms.
//
// Rows of a colour are not coupled, so the update order within a colour does
// not matter and the iterates are those of k_gs_colour bit for bit; the
// residual, restriction and prolongation sum in their own order.
#include "solver.hpp"
#include "reduce.hpp"

#include <algorithm>

namespace cfdla {

namespace {

constexpr int kTailThreads = 1024;
// The level arrays' addresses are read from memory, so their address space
// has to be named: loads through them would be flat ones otherwise.
#define CFDLA_GLOBAL __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ CFDLA_GLOBAL T *global_ptr(T *p) {
  return (CFDLA_GLOBAL T *)p;
}

template <typename T> struct TailVals;
template <> struct TailVals<double> {
  __device__ static auto v(const TailLevelDev &d) { return global_ptr(d.v64); }
  __device__ static auto d(const TailLevelDev &d) { return global_ptr(d.d64); }
  __device__ static auto p(const TailLevelDev &d) { return global_ptr(d.p64); }
  __device__ static auto r(const TailLevelDev &d) { return global_ptr(d.r64); }
  __device__ static auto b(const TailLevelDev &d) { return global_ptr(d.b64); }
  __device__ static auto x(const TailLevelDev &d) { return global_ptr(d.x64); }
};
template <> struct TailVals<float> {
  __device__ static auto v(const TailLevelDev &d) { return global_ptr(d.v32); }
  __device__ static auto d(const TailLevelDev &d) { return global_ptr(d.d32); }
  __device__ static auto p(const TailLevelDev &d) { return global_ptr(d.p32); }
  __device__ static auto r(const TailLevelDev &d) { return global_ptr(d.r32); }
  __device__ static auto b(const TailLevelDev &d) { return global_ptr(d.b32); }
  __device__ static auto x(const TailLevelDev &d) { return global_ptr(d.x32); }
};

// A level's entries as the sweeps read them: in LDS for the levels that fit
// there together, in memory (the L2) for the larger ones.  b is in position
// order.
template <typename T>
struct LdsRows {
  const T *v, *d, *b;
  const uint16_t *col, *row;
};
template <typename T>
struct MemRows {
  const CFDLA_GLOBAL T *v, *d, *b;
  const CFDLA_GLOBAL uint16_t *col, *row;
};
// (of workgroup k: the k-th right-hand side and iterate)
template <typename T>
__device__ __forceinline__ auto rhs_of(const TailLevelDev &D) {
  return TailVals<T>::b(D) + (size_t)blockIdx.x * D.n;
}
template <typename T>
__device__ __forceinline__ auto iterate_of(const TailLevelDev &D) {
  return TailVals<T>::x(D) + (size_t)blockIdx.x * D.n;
}
template <typename T>
__device__ __forceinline__ MemRows<T> mem_rows(const TailLevelDev &D) {
  return {TailVals<T>::v(D), TailVals<T>::d(D), rhs_of<T>(D), global_ptr(D.col), global_ptr(D.row)};
}

typedef unsigned short v4u16 __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));

// Four consecutive entries (4-entry aligned), in LDS or global memory.
__device__ __forceinline__ void quad(const double *p, double (&v)[4]) {
  const v2d a = reinterpret_cast<const v2d *>(p)[0], b = reinterpret_cast<const v2d *>(p)[1];
  v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
}
__device__ __forceinline__ void quad(const float *p, float (&v)[4]) {
  const v4f a = *reinterpret_cast<const v4f *>(p);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}
__device__ __forceinline__ void quad(const uint16_t *p, int (&v)[4]) {
  const v4u16 a = *reinterpret_cast<const v4u16 *>(p);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}
__device__ __forceinline__ void quad(const CFDLA_GLOBAL double *p, double (&v)[4]) {
  const v2d a = reinterpret_cast<const CFDLA_GLOBAL v2d *>(p)[0], b = reinterpret_cast<const CFDLA_GLOBAL v2d *>(p)[1];
  v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
}
__device__ __forceinline__ void quad(const CFDLA_GLOBAL float *p, float (&v)[4]) {
  const v4f a = *reinterpret_cast<const CFDLA_GLOBAL v4f *>(p);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}
__device__ __forceinline__ void quad(const CFDLA_GLOBAL uint16_t *p, int (&v)[4]) {
  const v4u16 a = *reinterpret_cast<const CFDLA_GLOBAL v4u16 *>(p);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}

// sum[r] += sum over Q groups of 4 entries of row r (rows rstep entries
// apart) of value * u[column], in entry order: all entries read before any
// gather, all gathers before any sum.
template <typename T, int NR, int Q, typename CP, typename VP>
__device__ __forceinline__ void tail_groups(CP c, VP v, int rstep, const T *u, T (&sum)[NR]) {
  int cc[NR][Q][4];
  T vv[NR][Q][4], xx[NR][Q][4];
#pragma unroll
  for (int r = 0; r < NR; ++r)
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      quad(c + r * rstep + 4 * q, cc[r][q]);
      quad(v + r * rstep + 4 * q, vv[r][q]);
    }
#pragma unroll
  for (int r = 0; r < NR; ++r)
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int j = 0; j < 4; ++j) xx[r][q][j] = u[cc[r][q][j]];
#pragma unroll
  for (int r = 0; r < NR; ++r)
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int j = 0; j < 4; ++j) sum[r] += vv[r][q][j] * xx[r][q][j];
}

// sums of NR rows of w entries (a multiple of 4, the same for the workgroup)
template <typename T, int NR, typename CP, typename VP>
__device__ __forceinline__ void tail_rows(CP c, VP v, int w, int rstep, const T *u, T (&sum)[NR]) {
#pragma unroll
  for (int r = 0; r < NR; ++r) sum[r] = T(0);
  if (w == 8) {
    tail_groups<T, NR, 2>(c, v, rstep, u, sum);
    return;
  }
  if constexpr (NR == 1) {
    if (w == 12) {
      tail_groups<T, NR, 3>(c, v, rstep, u, sum);
      return;
    }
  }
  for (int k = 0; k < w; k += 4) tail_groups<T, NR, 1>(c + k, v + k, rstep, u, sum);
}

// NR rows of colour m = (first position, rows, first entry, entries per row)
// from its t-th on, one every kTailThreads: x_i += omega ((b_i - sum) / d_i - x_i)
// unless |d_i| <= 1e-15, or (RESID) res_i = b_i - (d_i x_i + sum).
template <typename T, int NR, bool RESID, typename Rows>
__device__ __forceinline__ void tail_update(const Rows &A, int4 m, int t, T omega, T *u, T *res) {
  int i[NR];
  T diag[NR], bi[NR], sum[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    i[r] = A.row[m.x + t + r * kTailThreads];
    diag[r] = A.d[m.x + t + r * kTailThreads];
    bi[r] = A.b[m.x + t + r * kTailThreads];
  }
  tail_rows<T, NR>(A.col + m.z + t * m.w, A.v + m.z + t * m.w, m.w, m.w * kTailThreads, u, sum);
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    if constexpr (RESID) {
      res[i[r]] = bi[r] - (diag[r] * u[i[r]] + sum[r]);
    } else if (fabs((double)diag[r]) > 1e-15) {
      const T nv = (bi[r] - sum[r]) / diag[r];
      u[i[r]] = u[i[r]] + omega * (nv - u[i[r]]);
    }
  }
}

template <typename T, bool RESID, typename Rows>
__device__ __forceinline__ void tail_colour(const Rows &A, int4 m, T omega, T *u, T *res) {
  int t = threadIdx.x;
  for (; t + kTailThreads < m.y; t += 2 * kTailThreads) tail_update<T, 2, RESID>(A, m, t, omega, u, res);
  if (t < m.y) tail_update<T, 1, RESID>(A, m, t, omega, u, res);
}

// the colour's meta data in scalar registers
__device__ __forceinline__ int4 uniform(int4 m) {
  return make_int4(__builtin_amdgcn_readfirstlane(m.x), __builtin_amdgcn_readfirstlane(m.y),
                   __builtin_amdgcn_readfirstlane(m.z), __builtin_amdgcn_readfirstlane(m.w));
}

template <typename T, typename Rows>
__device__ __forceinline__ void tail_sweeps(const Rows &A, const int4 *meta, int nc, T omega, int sweeps,
                                            int symmetric, T *u) {
  for (int dir = 0; dir <= symmetric; ++dir)
    for (int k = 0; k < sweeps; ++k)
      for (int c = 0; c < nc; ++c) {
        tail_colour<T, false>(A, uniform(meta[dir ? nc - 1 - c : c]), omega, u, nullptr);
        __syncthreads();
      }
}

// lv[0 .. L): the tail's levels, finest first, the last L - inner of them with
// their entries in LDS; b, x: the finest level's vectors; LDS: the colours'
// meta data, two vectors u and w of the most rows of a level, and for the
// inner levels two vectors of icap rows and their entries.
//
// part: TAIL_WHOLE; TAIL_DOWN to the right-hand side of level L - 1; TAIL_UP
// from its iterate; TAIL_COLUMN the whole, workgroup k on the k-th unit vector
// in position order, into column k of x.
enum { TAIL_WHOLE, TAIL_DOWN, TAIL_UP, TAIL_COLUMN };
template <typename T>
__global__ __launch_bounds__(kTailThreads) void k_gs_tail(int part, const TailLevelDev *__restrict__ lv, int L, int inner,
                                                          int cap, int icap, int itotal,
                                                          const int4 *__restrict__ gmeta, int ncol, const T *b, T *x,
                                                          T omega, int pre, int post, int symmetric,
                                                          const double *__restrict__ inv, Scal *s, int check_done) {
  if (check_done && s->done) return;
  extern __shared__ double tail_lds[];
  __shared__ int4 meta[kTailColours];
  T *const base = reinterpret_cast<T *>(tail_lds);
  T *const store = base + 2 * (icap + 1);  // entries, diagonals, right-hand sides and iterates of the inner levels
  uint16_t *const istore = reinterpret_cast<uint16_t *>(store + itotal);
  const int tid = threadIdx.x;
  for (int c = tid; c < ncol; c += kTailThreads) meta[c] = gmeta[c];
  T *u = base, *w = base + cap + 1;
  // right-hand side of the finest level in position order
  auto rhs = [&](int p) {
    return part == TAIL_COLUMN ? T(p == (int)blockIdx.x ? 1 : 0) : b[global_ptr(lv[0].row)[p]];
  };
  if (inner > 0 && part != TAIL_UP) {
    auto bp = rhs_of<T>(lv[0]);
    for (int p = tid; p < lv[0].n; p += kTailThreads) bp[p] = rhs(p);
  }
  auto lds_rows = [&](const TailLevelDev &D) {
    return LdsRows<T>{store + D.iv, store + D.id, store + D.ib, istore + D.icol, istore + D.irow};
  };
  for (int l = part == TAIL_UP ? L : 0; l < L; ++l) {
    const TailLevelDev &D = lv[l];
    if (part == TAIL_DOWN && l + 1 == L) return;  // its right-hand side is in memory
    if (l == inner) {
      // The larger levels' iterates are in memory now: the inner levels take
      // the LDS over.  Their first right-hand side came through memory.
      u = base;
      w = base + icap + 1;
      for (int q = l; q < L; ++q) {
        const TailLevelDev &I = lv[q];
        for (int k = tid; k < I.slots; k += kTailThreads) {
          store[I.iv + k] = TailVals<T>::v(I)[k];
          istore[I.icol + k] = global_ptr(I.col)[k];
        }
        for (int k = tid; k < I.n; k += kTailThreads) {
          store[I.id + k] = TailVals<T>::d(I)[k];
          istore[I.irow + k] = global_ptr(I.row)[k];
        }
      }
      for (int k = tid; k < D.n; k += kTailThreads) store[D.ib + k] = l == 0 ? rhs(k) : rhs_of<T>(D)[k];
      __syncthreads();
    }
    const bool in = l >= inner;
    if (l + 1 == L && inv) {
      // dense coarsest level: the right-hand side in row order, one
      // wavefront per row
      for (int p = tid; p < D.n; p += kTailThreads) w[global_ptr(D.row)[p]] = in ? store[D.ib + p] : rhs_of<T>(D)[p];
      __syncthreads();
      for (int i = tid >> 6; i < D.n; i += kTailThreads / 64) {
        double acc = 0.0;
        for (int j = tid & 63; j < D.n; j += 64) acc += inv[(size_t)i * D.n + j] * (double)w[j];
        acc = wave_sum(acc);
        if ((tid & 63) == 0) u[i] = (T)acc;
      }
      if (tid == 0) u[D.n] = T(0);
      __syncthreads();
      break;
    }
    for (int i = tid; i <= D.n; i += kTailThreads) u[i] = T(0);
    if (tid == 0) w[D.n] = T(0);
    __syncthreads();
    const int4 *mt = meta + D.meta;
    const bool last = l + 1 == L;
    // the coarsest level is the pre-smoothing and 10 more sweeps (amg.rs:501)
    for (int more = 0; more < (last ? 2 : 1); ++more) {
      const int k = more == 0 ? pre : 10;
      if (in) {
        const LdsRows<T> A = lds_rows(D);
        tail_sweeps<T>(A, mt, D.nc, omega, k, symmetric, u);
      } else {
        const MemRows<T> A = mem_rows<T>(D);
        tail_sweeps<T>(A, mt, D.nc, omega, k, symmetric, u);
      }
    }
    if (last) break;
    if (in) {
      const LdsRows<T> A = lds_rows(D);
      for (int c = 0; c < D.nc; ++c) tail_colour<T, true>(A, uniform(mt[c]), omega, u, w);
      for (int i = tid; i < D.n; i += kTailThreads) store[D.ix + i] = u[i];
    } else {
      const MemRows<T> A = mem_rows<T>(D);
      for (int c = 0; c < D.nc; ++c) tail_colour<T, true>(A, uniform(mt[c]), omega, u, w);
      auto xl = iterate_of<T>(D);
      for (int i = tid; i < D.n; i += kTailThreads) xl[i] = u[i];
    }
    __syncthreads();
    // restriction, rows in the coarse level's position order
    const TailLevelDev &C = lv[l + 1];
    for (int p = tid; p < C.n; p += kTailThreads) {
      T sum[1];
      tail_rows<T, 1>(global_ptr(D.rcol) + p * D.rw, TailVals<T>::r(D) + p * D.rw, D.rw, 0, w, sum);
      if (in) store[C.ib + p] = sum[0];
      else rhs_of<T>(C)[p] = sum[0];
    }
    __syncthreads();
  }
  if (part == TAIL_UP) {
    auto xc = iterate_of<T>(lv[L - 1]);
    for (int i = tid; i < lv[L - 1].n; i += kTailThreads) u[i] = xc[i];
    if (tid == 0) u[lv[L - 1].n] = T(0);
    __syncthreads();
  }
  for (int l = L - 2; l >= 0; --l) {
    const TailLevelDev &D = lv[l];
    const bool in = l >= inner;
    if (l + 1 == inner && part != TAIL_UP) {
      // back to the larger levels: the coarse iterate moves behind the room
      // of the level's own, through memory
      auto xc = iterate_of<T>(lv[inner]);
      const int nc = lv[inner].n;
      for (int i = tid; i < nc; i += kTailThreads) xc[i] = u[i];
      __syncthreads();
      u = base;
      w = base + cap + 1;
      for (int i = tid; i < nc; i += kTailThreads) u[i] = xc[i];
      if (tid == 0) u[nc] = T(0);
      __syncthreads();
    }
    if (in) {
      for (int i = tid; i < D.n; i += kTailThreads) {
        T sum[1];
        tail_rows<T, 1>(global_ptr(D.pcol) + i * D.pw, TailVals<T>::p(D) + i * D.pw, D.pw, 0, u, sum);
        w[i] = store[D.ix + i] + sum[0];
      }
    } else {
      auto xl = iterate_of<T>(D);
      for (int i = tid; i < D.n; i += kTailThreads) {
        T sum[1];
        tail_rows<T, 1>(global_ptr(D.pcol) + i * D.pw, TailVals<T>::p(D) + i * D.pw, D.pw, 0, u, sum);
        w[i] = xl[i] + sum[0];
      }
    }
    if (tid == 0) w[D.n] = T(0);
    __syncthreads();
    T *sw = u;
    u = w;
    w = sw;
    const int4 *mt = meta + D.meta;
    if (in) {
      const LdsRows<T> A = lds_rows(D);
      tail_sweeps<T>(A, mt, D.nc, omega, post, symmetric, u);
    } else {
      const MemRows<T> A = mem_rows<T>(D);
      tail_sweeps<T>(A, mt, D.nc, omega, post, symmetric, u);
    }
  }
  const int n0 = lv[0].n;
  for (int i = tid; i < n0; i += kTailThreads) x[(size_t)blockIdx.x * n0 + i] = u[i];
}

// Slot values from the level's CSR values (src: CSR slot or -1), after a device refresh.
__global__ __launch_bounds__(kBlock) void k_tail_values(int n, const int *__restrict__ src,
                                                        const double *__restrict__ v64, double *o64, float *o32) {
  for (int k = blockIdx.x * kBlock + threadIdx.x; k < n; k += gridDim.x * kBlock) {
    const double a = src[k] >= 0 ? v64[src[k]] : 0.0;
    o64[k] = a;
    o32[k] = (float)a;
  }
}

int64_t widest(const HostCsr &h) {
  int64_t w = 0;
  for (int64_t i = 0; i < h.n; ++i) w = std::max<int64_t>(w, h.rp[i + 1] - h.rp[i]);
  return w;
}

int64_t group4(int64_t w) { return (w + 3) & ~int64_t(3); }

// Copy of a CSR matrix with every row padded to the longest, in groups of 4
// (padding: 0 at column m); position p holds row order[p] (order null: row p).
int padded_rows(const HostCsr &h, const std::vector<int32_t> *order, std::vector<uint16_t> &col,
                std::vector<double> &val) {
  const int64_t w = group4(widest(h));
  col.assign((size_t)(w * h.n), (uint16_t)h.m);
  val.assign((size_t)(w * h.n), 0.0);
  for (int64_t p = 0; p < h.n; ++p) {
    const int64_t i = order ? (*order)[(size_t)p] : p;
    for (int64_t k = h.rp[i]; k < h.rp[i + 1]; ++k) {
      const size_t o = (size_t)(p * w + k - h.rp[i]);
      col[o] = (uint16_t)h.ci[k];
      val[o] = h.v[k];
    }
  }
  return (int)w;
}

void put_pair(DevBuf<double> &d, DevBuf<float> &f, const std::vector<double> &v) {
  std::vector<float> t(v.begin(), v.end());
  d.upload(v.data(), v.size());
  f.upload(t.data(), t.size());
  sync_stream();
}

// Entries of colour c's padded rows of A without the diagonal.
int64_t colour_width(const HostCsr &a, const std::vector<int32_t> &order, const std::vector<int32_t> &off, size_t c) {
  int64_t w = 0;
  for (int32_t q = off[c]; q < off[c + 1]; ++q) {
    const int32_t i = order[(size_t)q];
    int64_t m = 0;
    for (int64_t e = a.rp[i]; e < a.rp[i + 1]; ++e) m += a.ci[e] != i;
    w = std::max(w, m);
  }
  return group4(w);
}

}  // namespace

// The first level from which the rest of the hierarchy runs in one
// workgroup, or -1.
int gs_tail_first(const HostHierarchy &h, const std::vector<std::vector<int32_t>> &order,
                  const std::vector<std::vector<int32_t>> &off, bool direct) {
  const int L = (int)h.levels.size();
  if (direct && h.levels.back().A.n > kTailDenseRows) return -1;
  int first = -1;
  int64_t colours = 0;
  for (int l = L - 1; l >= 0; --l) {
    const HostLevel &lv = h.levels[(size_t)l];
    const int64_t n = lv.A.n, nc = (int64_t)off[(size_t)l].size() - 1;
    colours += nc;
    if (colours > kTailColours) break;
    bool ok = n >= 1 && n <= kTailRows && lv.A.nnz() <= kTailNnzPerColour * nc;
    if (ok) {
      // padding may at most double an operator
      int64_t total = 0;
      for (size_t c = 0; c < (size_t)nc; ++c)
        total += colour_width(lv.A, order[(size_t)l], off[(size_t)l], c) * (off[(size_t)l][c + 1] - off[(size_t)l][c]);
      ok = total <= 2 * lv.A.nnz() + 4096;
    }
    if (ok && l + 1 < L)
      ok = group4(widest(lv.P)) * lv.P.n <= 2 * lv.P.nnz() + 4096 &&
           group4(widest(lv.R)) * lv.R.n <= 3 * lv.R.nnz() + 4096 && lv.R.n >= 1;
    if (!ok) break;
    first = l;
  }
  return first;
}

void GsTail::build(const HostHierarchy &h, int first, const std::vector<std::vector<int32_t>> &order,
                   const std::vector<std::vector<int32_t>> &off) {
  level = first;
  const size_t L = h.levels.size();
  lv.clear();
  lv.resize(L - (size_t)first);
  std::vector<TailLevelDev> desc(lv.size());
  std::vector<int32_t> meta;
  for (size_t q = 0; q < lv.size(); ++q) {
    const size_t l = (size_t)first + q;
    const HostLevel &H = h.levels[l];
    const HostCsr &a = H.A;
    TailLevel &t = lv[q];
    const std::vector<int32_t> &ord = order[l], &of = off[l];
    const int nc = (int)of.size() - 1;
    std::vector<int32_t> eoff((size_t)nc + 1, 0), dsrc((size_t)a.n, -1), src;
    std::vector<uint16_t> row((size_t)a.n), col;
    for (int c = 0; c < nc; ++c) {
      const int cnt = of[(size_t)c + 1] - of[(size_t)c];
      const int w = (int)colour_width(a, ord, of, (size_t)c);
      eoff[(size_t)c + 1] = eoff[(size_t)c] + w * cnt;
      col.resize((size_t)eoff[(size_t)c + 1], (uint16_t)a.n);  // padding
      src.resize((size_t)eoff[(size_t)c + 1], -1);
      for (int k = 0; k < cnt; ++k) {
        const int p = of[(size_t)c] + k;
        const int32_t i = ord[(size_t)p];
        row[(size_t)p] = (uint16_t)i;
        int m = 0;
        for (int64_t e = a.rp[i]; e < a.rp[i + 1]; ++e) {
          if (a.ci[e] == i) {
            dsrc[(size_t)p] = (int32_t)e;
            continue;
          }
          const size_t o = (size_t)(eoff[(size_t)c] + k * w + m++);
          col[o] = (uint16_t)a.ci[e];
          src[o] = (int32_t)e;
        }
      }
    }
    std::vector<double> v(src.size()), d((size_t)a.n);
    for (size_t k = 0; k < src.size(); ++k) v[k] = src[k] >= 0 ? a.v[(size_t)src[k]] : 0.0;
    for (size_t k = 0; k < d.size(); ++k) d[k] = dsrc[k] >= 0 ? a.v[(size_t)dsrc[k]] : 0.0;
    t.row.upload(row.data(), row.size());
    t.col.upload(col.data(), col.size());
    t.src.upload(src.data(), src.size());
    t.dsrc.upload(dsrc.data(), dsrc.size());
    t.slots = (int)src.size();
    put_pair(t.v64, t.v32, v);
    put_pair(t.d64, t.d32, d);
    TailLevelDev &D = desc[q];
    D = TailLevelDev{};
    D.meta = (int)meta.size() / 4;
    for (int c = 0; c < nc; ++c) {
      const int cnt = of[(size_t)c + 1] - of[(size_t)c];
      meta.insert(meta.end(), {of[(size_t)c], cnt, eoff[(size_t)c],
                               cnt > 0 ? (eoff[(size_t)c + 1] - eoff[(size_t)c]) / cnt : 0});
    }
    t.b64.alloc((size_t)a.n);
    t.x64.alloc((size_t)a.n);
    t.b32.alloc((size_t)a.n);
    t.x32.alloc((size_t)a.n);
    if (l + 1 < L) {
      std::vector<uint16_t> c;
      D.pw = padded_rows(H.P, nullptr, c, v);
      t.pcol.upload(c.data(), c.size());
      put_pair(t.p64, t.p32, v);
      D.rw = padded_rows(H.R, &order[l + 1], c, v);
      t.rcol.upload(c.data(), c.size());
      put_pair(t.r64, t.r32, v);
    }
    D.n = (int)a.n;
    D.nc = nc;
    D.slots = t.slots;
    D.row = t.row.p;
    D.col = t.col.p;
    D.pcol = t.pcol.p;
    D.rcol = t.rcol.p;
    D.v64 = t.v64.p; D.d64 = t.d64.p; D.p64 = t.p64.p; D.r64 = t.r64.p;
    D.v32 = t.v32.p; D.d32 = t.d32.p; D.p32 = t.p32.p; D.r32 = t.r32.p;
    D.b64 = t.b64.p; D.x64 = t.x64.p;
    D.b32 = t.b32.p; D.x32 = t.x32.p;
  }
  cap = 0;
  for (const TailLevelDev &D : desc) cap = std::max(cap, D.n);
  // The inner levels: as many of the last ones as fit in LDS with their
  // entries (value, column), diagonal, right-hand side, iterate and row.
  inner = (int)desc.size();
  icap = itotal = 0;
  int iwords = 0;
  for (int q = (int)desc.size() - 1; q >= 0; --q) {
    TailLevelDev &D = desc[(size_t)q];
    // every part starts at a multiple of 4 elements (16-byte groups)
    const int n4 = (int)group4(D.n);
    const int64_t vals = (int64_t)itotal + D.slots + 3 * n4, words = (int64_t)iwords + D.slots + n4;
    const int64_t most = std::max<int64_t>(icap, group4(D.n + 1) + 1);  // 2 (most + 1) is a multiple of 4
    if ((2 * (most + 1) + vals) * (int64_t)sizeof(double) + words * (int64_t)sizeof(uint16_t) > kTailLds) break;
    D.iv = itotal;
    D.id = D.iv + D.slots;
    D.ib = D.id + n4;
    D.ix = D.ib + n4;
    D.icol = iwords;
    D.irow = iwords + D.slots;
    itotal = (int)vals;
    iwords = (int)words;
    icap = (int)most;
    inner = q;
  }
  lds_vals = inner > 0 ? 2 * (cap + 1) : 0;
  lds_words = iwords;
  ncolours = (int)meta.size() / 4;
  // The dense operator: from the first small level behind the first one.  A
  // hierarchy that fits in LDS whole (inner = 0) runs there faster than in
  // three launches.
  dense.level = -1;
  for (int q = inner; q >= 1 && desc[(size_t)std::min<int>(q, (int)desc.size() - 1)].n <= kDenseCycleRows; --q)
    if (q < (int)desc.size()) dense.level = q;
  if (dense.level >= 0) {
    dense.n = desc[(size_t)dense.level].n;
    dense.ld = (dense.n + 15) / 16 * 16;
    dense.c.ensure((size_t)dense.n * (size_t)dense.ld);
  }
  d_meta.upload(meta.data(), meta.size());
  d_desc.upload(desc.data(), desc.size());
  sync_stream();
  const int bytes = kTailLds;
  CFDLA_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(k_gs_tail<double>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
  CFDLA_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(k_gs_tail<float>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
}

void GsTail::refresh(const std::vector<DevLevel> &dev) {
  for (size_t q = 0; q < lv.size(); ++q) {
    const double *v = dev[(size_t)level + q].A.v64.p;
    TailLevel &t = lv[q];
    const int n = dev[(size_t)level + q].A.n;
    if (t.slots > 0)
      hipLaunchKernelGGL(k_tail_values, dim3(blocks_for(t.slots, kBlock)), dim3(kBlock), 0, stream(), t.slots, t.src.p,
                         v, t.v64.p, t.v32.p);
    hipLaunchKernelGGL(k_tail_values, dim3(blocks_for(n, kBlock)), dim3(kBlock), 0, stream(), n, t.dsrc.p, v, t.d64.p,
                       t.d32.p);
  }
  CFDLA_HIP(hipGetLastError());
}

namespace {
template <typename T> T *tail_rhs(const TailLevel &t);
template <> double *tail_rhs<double>(const TailLevel &t) { return t.b64.p; }
template <> float *tail_rhs<float>(const TailLevel &t) { return t.b32.p; }
template <typename T> T *tail_iterate(const TailLevel &t);
template <> double *tail_iterate<double>(const TailLevel &t) { return t.x64.p; }
template <> float *tail_iterate<float>(const TailLevel &t) { return t.x32.p; }

// The LDS of k_gs_tail: the 16-bit words follow the inner levels' values,
// inside or past the larger levels' two vectors.
size_t tail_bytes(const GsTail &t, size_t elem) {
  return std::max((size_t)t.lds_vals * elem,
                  (2 * ((size_t)t.icap + 1) + t.itotal) * elem + (size_t)t.lds_words * sizeof(uint16_t));
}
}  // namespace

// The columns of the dense operator, one workgroup each, with the larger of
// its levels' vectors in memory once per column.
void GsTail::form_dense(double omega, int pre, int post, bool symmetric, const double *inv) {
  const size_t L = lv.size(), q0 = (size_t)dense.level;
  std::vector<TailLevelDev> desc(L);
  if (dense.ws.empty()) {
    dense.ws.resize(1 + 2 * (L - q0));
    dense.ws[0].ensure((size_t)dense.n * (size_t)dense.n);
    d_desc.download(desc.data(), L);
    sync_stream();
    for (size_t q = q0; q < L && q <= (size_t)inner; ++q) {
      const size_t count = (size_t)dense.n * (size_t)desc[q].n;
      DevBuf<double> &b = dense.ws[1 + 2 * (q - q0)], &x = dense.ws[2 + 2 * (q - q0)];
      b.ensure(count);
      x.ensure(count);
      desc[q].b64 = b.p;
      desc[q].x64 = x.p;
    }
    d_column.upload(desc.data(), L);
    sync_stream();
  }
  hipLaunchKernelGGL((k_gs_tail<double>), dim3((unsigned)dense.n), dim3(kTailThreads), tail_bytes(*this, sizeof(double)),
                     stream(), (int)TAIL_COLUMN, d_column.p + q0, (int)(L - q0), inner - (int)q0, dense.n, icap, itotal,
                     reinterpret_cast<const int4 *>(d_meta.p), ncolours, (const double *)nullptr, dense.ws[0].p, omega,
                     pre, post, symmetric ? 1 : 0, inv, (Scal *)nullptr, 0);
  CFDLA_HIP(hipGetLastError());
  dense.from_columns(dense.ws[0].p);
}

template <typename T>
void gs_tail(const GsTail &t, const T *b, T *x, double omega, int pre, int post, bool symmetric, const double *inv,
             Scal *s, bool check_done) {
  s = settled_scal(s);
  const auto run = [&](int part, int L, int inner) {
    hipLaunchKernelGGL((k_gs_tail<T>), dim3(1), dim3(kTailThreads), tail_bytes(t, sizeof(T)), stream(), part,
                       t.d_desc.p, L, inner, t.cap, t.icap, t.itotal, reinterpret_cast<const int4 *>(t.d_meta.p),
                       t.ncolours, b, x, (T)omega, pre, post, symmetric ? 1 : 0, inv, s, check_done ? 1 : 0);
  };
  const int q = t.dense.level;
  if (q >= 0) {
    const TailLevel &D = t.lv[(size_t)q];
    run(TAIL_DOWN, q + 1, t.inner);
    t.dense.apply<T>(tail_rhs<T>(D), tail_iterate<T>(D), s, check_done);
    run(TAIL_UP, q + 1, t.inner);
  } else {
    run(TAIL_WHOLE, (int)t.lv.size(), t.inner);
  }
  CFDLA_HIP(hipGetLastError());
}
template void gs_tail<double>(const GsTail &, const double *, double *, double, int, int, bool, const double *, Scal *,
                              bool);
template void gs_tail<float>(const GsTail &, const float *, float *, double, int, int, bool, const double *, Scal *,
                             bool);

}  // namespace cfdla
