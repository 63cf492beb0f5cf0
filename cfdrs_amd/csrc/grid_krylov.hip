// CG and BiCGSTAB with a Jacobi (or no) preconditioner on diagonal storage,
// many iterations per launch.  On grids of 10^4 - 10^5 rows an iteration is a
// chain of short dependent phases, and a launch per phase costs 4.3-5.5 us
// each.  Here the vectors and the matrix rows stay in the registers of up to
// kGridBlocks resident blocks, and a phase ends with an exchange of one or a few
// sums between all blocks (exchange below).  The rows a block's product needs
// from its neighbours are published before the exchange that follows the
// product, and each block carries r and p of those rows along itself, so a
// product needs no exchange of its own.
//
// us per iteration, a launch per phase and here: CG on 4,096 / 16,384 / 65,536 /
// 262,144 / 524,176 rows 8.6 / 8.8 / 9.5 / 12.5 / 17.3 -> 3.4 / 4.1 / 4.8 / 7.1 /
// 8.1; BiCGSTAB up to 262,144 rows 18.7 / 19.2 / 20.2 / 27.6 -> 6.5 / 7.3 / 9.5 /
// 12.1.  Bound by the two (CG) or three exchanges of an iteration.  Larger
// systems would need every CU or rows that no longer fit the registers: the
// 128 of 1,024 threads hold all of a thread's rows but in FP64 CG with 4 rows
// (10 spilled with 5 entries per row, 34 with 7) and FP64 BiCGSTAB with 2 rows of
// 7 entries (8 spilled).
//
// Every wait is bounded: a block that does not see the others' sums within
// DevCsr::resident_polls polls reports it in Scal::pad.  The new iterate and
// scalars replace the old ones in a launch of their own (k_grid_commit), if no
// block did: a solve whose blocks did not meet goes on with a launch per phase
// from where it was.
#include "finalize.hpp"
#include "internal.hpp"
#include "solver.hpp"

namespace cfdla {
namespace {

constexpr int kGridThreads = 1024;
constexpr int kGridWaves = kGridThreads / 64;
constexpr int kGridBlocks = 128;
constexpr int kGridHalo = 1024;   // largest |offset|: 2 halo entries per thread
constexpr int kGridSums = 3;      // sums per exchange
constexpr int kGridSet = kGridSums * kGridBlocks;
constexpr unsigned long long kEmpty = 0x7ff8dead0000beefull;  // a NaN that no sum is stored as
constexpr int kScalWords = (int)(sizeof(Scal) / sizeof(int));

struct GridShared {
  Scal sc;
  double red[kGridSums][kGridWaves];
  int failed;
};

template <typename T>
__device__ __forceinline__ void publish(T *p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ T fetch(const T *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Sums v over all blocks and runs fin(scalars, sums) on this block's copy of
// the scalars; false when a block's sum did not come in time.  Each block
// stores its sums into its places of set `phase` mod 4 and waits until no
// place of the set is empty; all blocks add them in the same order, so all
// have the same bits.  A block passing exchange k knows that every block has
// left exchange k - 1, so at k its places of set k - 2 = k + 2 can be
// emptied again, and that is in memory before its sum of k + 1 is.
// EDGES: the caller published values (publish) that the other blocks fetch
// after this exchange.
// 16 / 32 / 64 / 128 blocks: 1.2 / 1.8 / 2.2 / 3.0 us, two trips to the memory
// side of the eight L2s and the polls that queue there.
template <int NV, bool EDGES, typename Fin>
__device__ __forceinline__ bool exchange(GridShared &sh, unsigned long long *slots, int &phase, int polls,
                                         const double (&v)[NV], Fin &&fin) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nb = gridDim.x;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const double w = wave_sum(v[i]);
    if (lane == 0) sh.red[i][wave] = w;
  }
  if constexpr (EDGES) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (wave == 0) {
    double tot[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) tot[i] = wave_sum(lane < kGridWaves ? sh.red[i][lane] : 0.0);
    bool ok = true;
    if (nb > 1) {
      unsigned long long *set = slots + (phase & 3) * kGridSet, *old = slots + ((phase + 2) & 3) * kGridSet;
      if (lane == 0) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          const double t = tot[i] == tot[i] ? tot[i] : __builtin_nan("");
          publish(set + i * kGridBlocks + blockIdx.x, __builtin_bit_cast(unsigned long long, t));
        }
#pragma unroll
        for (int i = 0; i < kGridSums; ++i) publish(old + i * kGridBlocks + blockIdx.x, kEmpty);
      }
      unsigned long long got[NV][2];
      int left = polls;
      do {
        ok = true;
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            got[i][h] = 0;  // +0.0
            if (lane + 64 * h < nb) got[i][h] = fetch(set + i * kGridBlocks + lane + 64 * h);
            ok = ok && got[i][h] != kEmpty;
          }
        ok = __all(ok);
      } while (!ok && --left > 0);
#pragma unroll
      for (int i = 0; i < NV; ++i)
        tot[i] = wave_sum(__builtin_bit_cast(double, got[i][0]) + __builtin_bit_cast(double, got[i][1]));
    }
    if (lane == 0) {
      sh.failed = !ok;
      if (ok) fin(sh.sc, tot);
    }
  }
  __syncthreads();
  ++phase;
  return !sh.failed;
}

// The product's operand in LDS: rows r0 - halo .. r0 + rows + halo - 1.  Halo
// entry e < halo is row r0 - halo + e, the others follow the block's rows.
template <typename T, int NS, int RPT>
struct GridRows {
  static constexpr int rows = kGridThreads * RPT;
  T a[RPT][NS];
  const DiaRows &g;
  const int r0;

  __device__ GridRows(const DiaRows &g_, const T *__restrict__ dv) : g(g_), r0(blockIdx.x * rows) {
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
      const int row = r0 + u * kGridThreads + (int)threadIdx.x;
#pragma unroll
      for (int j = 0; j < NS; ++j) {
        const int col = row + g.off[j];
        const bool ok = row < g.n && col >= 0 && col < g.n;
        const T v = dv[(size_t)g.k[j] * g.n + (ok ? (g.lower[j] ? col : row) : 0)];
        a[u][j] = ok ? v : T(0);
      }
    }
  }
  __device__ int row(int u) const { return r0 + u * kGridThreads + (int)threadIdx.x; }
  __device__ int slot(int u) const { return g.halo + u * kGridThreads + (int)threadIdx.x; }
  __device__ T load(const T *__restrict__ x, int u) const { return row(u) < g.n ? x[row(u)] : T(0); }
  __device__ void store(T *x, int u, T v) const {
    if (row(u) < g.n) x[row(u)] = v;
  }
  __device__ T product(const T *op, int u) const {
    T s = T(0);
#pragma unroll
    for (int j = 0; j < NS; ++j) s += a[u][j] * op[slot(u) + g.off[j]];
    return s;
  }
  // rows that a neighbour's product reads
  __device__ void publish_edge(T *edge, int u, T v) const {
    const int li = u * kGridThreads + (int)threadIdx.x;
    if ((li < g.halo || li >= rows - g.halo) && row(u) < g.n) publish(edge + row(u), v);
  }
  // this thread's halo entries h = 0, 1
  __device__ bool halo(int h, int &e, int &at, int &grow) const {
    e = (int)threadIdx.x + h * kGridThreads;
    at = e < g.halo ? e : rows + e;
    grow = e < g.halo ? r0 - g.halo + e : r0 + rows + e - g.halo;
    return e < 2 * g.halo && grow >= 0 && grow < g.n;
  }
};

__global__ __launch_bounds__(256) void k_grid_reset(unsigned long long *slots, Scal *s) {
  for (int i = threadIdx.x; i < 4 * kGridSet; i += 256) slots[i] = kEmpty;
  if (threadIdx.x == 0) s->pad = 0;
}

template <typename T>
__device__ __forceinline__ void load_scal(GridShared &sh, const Scal *s) {
  if (threadIdx.x < kScalWords) reinterpret_cast<int *>(&sh.sc)[threadIdx.x] = reinterpret_cast<const int *>(s)[threadIdx.x];
  if (threadIdx.x == 0) sh.failed = 0;
}
__device__ __forceinline__ void store_scal(const GridShared &sh, Scal *s) {
  const int i = threadIdx.x;
  if (blockIdx.x == 0 && i < kScalWords) reinterpret_cast<int *>(s)[i] = reinterpret_cast<const int *>(&sh.sc)[i];
}

template <typename T>
__global__ __launch_bounds__(256) void k_grid_commit(int n, const T *__restrict__ xn, T *__restrict__ x,
                                                     const Scal *__restrict__ sn, Scal *s) {
  if (s->pad) return;  // (never written here: the new scalars' pad is 0 too)
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) x[i] = xn[i];
  if (i < kScalWords && i != (int)(offsetof(Scal, pad) / sizeof(int)))
    reinterpret_cast<int *>(s)[i] = reinterpret_cast<const int *>(sn)[i];
}

// Up to `steps` iterations of Jacobi-preconditioned CG (jd null: none) from
// x, r, p and the scalars, with p the next direction; the new x and scalars go
// to xn and sn.  edge: 2 n values.
template <typename T, int NS, int RPT>
__global__ __launch_bounds__(kGridThreads) void k_grid_cg(DiaRows g, const T *__restrict__ dv,
                                                          const T *__restrict__ jd, const T *__restrict__ x,
                                                          T *xn, T *r, T *p, T *edge, Scal *s, Scal *sn,
                                                          unsigned long long *slots, int steps, int polls) {
  extern __shared__ char grid_lds[];
  __shared__ GridShared sh;
  GridRows<T, NS, RPT> A(g, dv);
  T *pl = reinterpret_cast<T *>(grid_lds);
  load_scal<T>(sh, s);
  T xv[RPT], rv[RPT], jv[RPT], q[RPT];
#pragma unroll
  for (int u = 0; u < RPT; ++u) {
    xv[u] = A.load(x, u);
    rv[u] = A.load(r, u);
    jv[u] = jd ? A.load(jd, u) : T(1);
    pl[A.slot(u)] = A.load(p, u);
  }
  T rh[2], jh[2];
  int e, at, grow;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const bool live = A.halo(h, e, at, grow);
    rh[h] = live ? r[grow] : T(0);
    jh[h] = live ? (jd ? jd[grow] : T(1)) : T(0);
    if (e < 2 * g.halo) pl[at] = live ? p[grow] : T(0);
  }
  __syncthreads();
  if (sh.sc.done) steps = 0;
  int phase = 0;
  for (int it = 0; it < steps; ++it) {
    T *out = edge + (size_t)(it & 1) * g.n;
    double pq[1] = {0.0};
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
      q[u] = A.product(pl, u);
      A.publish_edge(out, u, q[u]);
      pq[0] += (double)pl[A.slot(u)] * (double)q[u];
    }
    if (!exchange<1, true>(sh, slots, phase, polls, pq, [](Scal &sc, const double(&t)[1]) {
          sc.red[0] = t[0];
          finalize(&sc, OP_CG_ALPHA);
        })) {
      if (threadIdx.x == 0) s->pad = 1;
      return;
    }
    if (sh.sc.done) break;
    const T alpha = (T)sh.sc.alpha;
    T qh[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) qh[h] = A.halo(h, e, at, grow) ? fetch(out + grow) : T(0);
    double rr[2] = {0.0, 0.0};
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
      xv[u] = fma(alpha, pl[A.slot(u)], xv[u]);
      rv[u] = fma(-alpha, q[u], rv[u]);
      rr[0] += (double)rv[u] * (double)rv[u];
      rr[1] += (double)rv[u] * (double)(jv[u] * rv[u]);
    }
    if (!exchange<2, false>(sh, slots, phase, polls, rr, [](Scal &sc, const double(&t)[2]) {
          sc.red[0] = t[0];
          sc.red[1] = t[1];
          finalize(&sc, OP_CG_RR_RZ);
        })) {
      if (threadIdx.x == 0) s->pad = 1;
      return;
    }
    if (sh.sc.done) break;
    const T beta = (T)sh.sc.beta;
#pragma unroll
    for (int u = 0; u < RPT; ++u) pl[A.slot(u)] = fma(beta, pl[A.slot(u)], jv[u] * rv[u]);
#pragma unroll
    for (int h = 0; h < 2; ++h)
      if (A.halo(h, e, at, grow)) {
        rh[h] = fma(-alpha, qh[h], rh[h]);
        pl[at] = fma(beta, pl[at], jh[h] * rh[h]);
      }
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < RPT; ++u) {
    A.store(xn, u, xv[u]);
    A.store(r, u, rv[u]);
    A.store(p, u, pl[A.slot(u)]);
  }
  store_scal(sh, sn);
}

// Up to `steps` iterations of BiCGSTAB from x, r, rhat, p, v and the scalars
// (beta of the first iteration formed), the new x and scalars into xn and sn;
// leaves jd .* p in ph.  edge: 3 n values.
template <typename T, int NS, int RPT>
__global__ __launch_bounds__(kGridThreads) void k_grid_bicg(DiaRows g, const T *__restrict__ dv,
                                                            const T *__restrict__ jd, const T *__restrict__ x,
                                                            T *xn, T *r, const T *__restrict__ rhat, T *p, T *v,
                                                            T *ph, T *edge, Scal *s, Scal *sn,
                                                            unsigned long long *slots, int steps, int polls) {
  extern __shared__ char grid_lds[];
  __shared__ GridShared sh;
  GridRows<T, NS, RPT> A(g, dv);
  T *op = reinterpret_cast<T *>(grid_lds);
  load_scal<T>(sh, s);
  T xv[RPT], rv[RPT], hv[RPT], pv[RPT], vv[RPT], jv[RPT];
#pragma unroll
  for (int u = 0; u < RPT; ++u) {
    xv[u] = A.load(x, u);
    rv[u] = A.load(r, u);
    hv[u] = A.load(rhat, u);
    pv[u] = A.load(p, u);
    vv[u] = A.load(v, u);
    jv[u] = jd ? A.load(jd, u) : T(1);
  }
  T rh[2], jh[2], pe[2], ve[2];
  int e, at, grow;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const bool live = A.halo(h, e, at, grow);
    rh[h] = live ? r[grow] : T(0);
    pe[h] = live ? p[grow] : T(0);
    ve[h] = live ? v[grow] : T(0);
    jh[h] = live ? (jd ? jd[grow] : T(1)) : T(0);
    if (e < 2 * g.halo) op[at] = T(0);
  }
  __syncthreads();
  if (sh.sc.done) steps = 0;
  int phase = 0;
  bool failed = false;
  for (int it = 0; it < steps; ++it) {
    T *vout = edge, *tout = edge + (size_t)(1 + (it & 1)) * g.n;
    {
      const T beta = (T)sh.sc.beta, omega = (T)sh.sc.omega;
#pragma unroll
      for (int u = 0; u < RPT; ++u) {
        pv[u] = fma(beta, fma(-omega, vv[u], pv[u]), rv[u]);
        op[A.slot(u)] = jv[u] * pv[u];
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
        if (A.halo(h, e, at, grow)) {
          pe[h] = fma(beta, fma(-omega, ve[h], pe[h]), rh[h]);
          op[at] = jh[h] * pe[h];
        }
    }
    __syncthreads();
    double rhv[1] = {0.0};
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
      vv[u] = A.product(op, u);
      A.publish_edge(vout, u, vv[u]);
      rhv[0] += (double)hv[u] * (double)vv[u];
    }
    failed = !exchange<1, true>(sh, slots, phase, polls, rhv, [](Scal &sc, const double(&t)[1]) {
      sc.red[0] = t[0];
      finalize(&sc, OP_BI_ALPHA);
    });
    if (failed || sh.sc.done) break;
    const T alpha = (T)sh.sc.alpha;
    // rv holds s from here to the update of r
    double sums[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int h = 0; h < 2; ++h) ve[h] = A.halo(h, e, at, grow) ? fetch(vout + grow) : T(0);
    T sv[RPT], t[RPT];
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
      sv[u] = fma(-alpha, vv[u], rv[u]);
      sums[0] += (double)sv[u] * (double)sv[u];
      op[A.slot(u)] = jv[u] * sv[u];
    }
    T se[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      se[h] = fma(-alpha, ve[h], rh[h]);
      if (A.halo(h, e, at, grow)) op[at] = jh[h] * se[h];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
      t[u] = A.product(op, u);
      A.publish_edge(tout, u, t[u]);
      sums[1] += (double)t[u] * (double)sv[u];
      sums[2] += (double)t[u] * (double)t[u];
    }
    failed = !exchange<3, true>(sh, slots, phase, polls, sums, [](Scal &sc, const double(&w)[3]) {
      sc.red[0] = w[0];
      finalize(&sc, OP_BI_SNORM);
      if (!sc.done) {
        sc.red[0] = w[1];
        sc.red[1] = w[2];
        finalize(&sc, OP_BI_OMEGA);
      }
    });
    if (failed || sh.sc.done) break;
    const T omega = (T)sh.sc.omega;
    T te[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) te[h] = A.halo(h, e, at, grow) ? fetch(tout + grow) : T(0);
    double rr[2] = {0.0, 0.0};
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
      xv[u] += alpha * (jv[u] * pv[u]) + omega * (jv[u] * sv[u]);
      rv[u] = fma(-omega, t[u], sv[u]);
      rr[0] += (double)rv[u] * (double)rv[u];
      rr[1] += (double)hv[u] * (double)rv[u];
    }
    failed = !exchange<2, false>(sh, slots, phase, polls, rr, [](Scal &sc, const double(&w)[2]) {
      sc.red[0] = w[0];
      sc.red[1] = w[1];
      finalize(&sc, OP_BI_RR_RHO);
    });
    if (failed || sh.sc.done) break;
#pragma unroll
    for (int h = 0; h < 2; ++h) rh[h] = fma(-omega, te[h], se[h]);
  }
  if (failed) {
    if (threadIdx.x == 0) s->pad = 1;
    return;
  }
#pragma unroll
  for (int u = 0; u < RPT; ++u) {
    A.store(xn, u, xv[u]);
    A.store(r, u, rv[u]);
    A.store(p, u, pv[u]);
    A.store(v, u, vv[u]);
    A.store(ph, u, jv[u] * pv[u]);
  }
  store_scal(sh, sn);
}

// Rows per thread: an exchange costs more with every block that takes part,
// the phases between cost more with every row.  CG on 16,384 / 36,864 / 65,536
// / 131,044 rows, us per iteration with 1, 2 and 4 rows: 4.1, 4.3, 4.3 / 5.4,
// 4.6, 4.7 / 6.0, 5.7, 4.8 / 6.8, 6.5, 6.1; BiCGSTAB with 1 and 2: 7.3, 7.5 / 9.3,
// 7.9 / 10.1, 9.5 / 11.7, 11.0.  7 entries in 4 rows no longer fit the registers
// in FP64 (32,768 rows: 5.5, 4.6, 7.5), nor do BiCGSTAB's vectors, so CG takes 2
// such rows as long as 128 blocks hold them.  Above, 4 rows still beat a launch
// per phase: 263,168 / 409,600 / 524,288 rows 10.6 / 10.9 / 11.2 us against 14.2 /
// 16.0 / 18.4, FP32, where they fit, 7.5 / 7.9 / 8.1 against 15.9 / 18.1 / 17.9.
int rows_per_thread(int n, int ns, bool bicg) {
  const int most = bicg || (ns > 5 && n <= 2 * kGridThreads * kGridBlocks) ? 2 : 4;
  int rpt = 1;
  while (rpt < most && (n + kGridThreads * rpt - 1) / (kGridThreads * rpt) > 18) rpt *= 2;
  return rpt;
}

template <typename T>
void commit(int n, const T *xn, T *x, const Scal *sn, Scal *s) {
  const int words = std::max(n, kScalWords);
  hipLaunchKernelGGL((k_grid_commit<T>), dim3((words + 255) / 256), dim3(256), 0, stream(), n, xn, x, sn, s);
  CFDLA_HIP(hipGetLastError());
}
}  // namespace

template <typename T>
DiaRows dia_rows(const DevCsr &A) {
  DiaRows g;
  const DiaDesc &d = A.dia_desc;
  if (!A.dia || A.dia_vals<T>() == nullptr || A.n != A.m || (d.sym ? 2 * d.nd - 1 : d.nd) > kDiaRowMax) return g;
  g.n = A.n;
  int m = 0;
  if (d.sym)
    for (int k = d.nd - 1; k > 0; --k, ++m) {
      g.off[m] = -d.off[k];
      g.k[m] = k;
      g.lower[m] = 1;
    }
  for (int k = 0; k < d.nd; ++k, ++m) {
    g.off[m] = d.off[k];
    g.k[m] = k;
  }
  g.count = m;
  for (int j = 0; j < m; ++j) g.halo = std::max(g.halo, std::abs(g.off[j]));
  return g;
}
template DiaRows dia_rows<double>(const DevCsr &);
template DiaRows dia_rows<float>(const DevCsr &);

template <typename T>
bool grid_krylov_takes(const DevCsr &A, bool bicg) {
  const DiaRows g = dia_rows<T>(A);
  const int ns = g.count;
  if (A.resident_polls < 1 || ns < 1 || A.n < 1 || g.halo > kGridHalo) return false;
  // one block per CU, and no more than half of the CUs
  const int rows = kGridThreads * rows_per_thread(A.n, ns, bicg);
  return (A.n + rows - 1) / rows <= std::min(kGridBlocks, num_cus() / 2);
}

template <typename T>
void grid_cg(const DevCsr &A, const T *jd, T *x, T *r, T *p, T *edge, Scal *s, int steps) {
  Context &c = ctx();
  s = settled_scal(s);
  c.grid_slots.ensure(4 * kGridSet + (sizeof(Scal) + 7) / 8);
  Scal *sn = reinterpret_cast<Scal *>(c.grid_slots.p + 4 * kGridSet);
  hipLaunchKernelGGL(k_grid_reset, dim3(1), dim3(256), 0, stream(), c.grid_slots.p, s);
  const DiaRows g = dia_rows<T>(A);
  const int ns = g.count, rpt = rows_per_thread(A.n, ns, false), rows = kGridThreads * rpt;
  const auto go = [&](auto *kernel) {
    const int lds = (rows + 2 * g.halo) * (int)sizeof(T);
    hipLaunchKernelGGL(kernel, dim3((A.n + rows - 1) / rows), dim3(kGridThreads), lds, stream(), g,
                       A.dia_vals<T>(), jd, x, edge + 2 * (size_t)A.n, r, p, edge, s, sn, c.grid_slots.p, steps,
                       A.resident_polls);
  };
#define CFDLA_GRID(RPT)                     \
  if (ns <= 3) go(k_grid_cg<T, 3, RPT>);    \
  else if (ns <= 5) go(k_grid_cg<T, 5, RPT>); \
  else go(k_grid_cg<T, 7, RPT>);
  if (rpt == 1) { CFDLA_GRID(1) } else if (rpt == 2) { CFDLA_GRID(2) } else { CFDLA_GRID(4) }
#undef CFDLA_GRID
  commit<T>(A.n, edge + 2 * (size_t)A.n, x, sn, s);
}

template <typename T>
void grid_bicgstab(const DevCsr &A, const T *jd, T *x, T *r, const T *rhat, T *p, T *v, T *ph, T *edge, Scal *s,
                   int steps) {
  Context &c = ctx();
  s = settled_scal(s);
  c.grid_slots.ensure(4 * kGridSet + (sizeof(Scal) + 7) / 8);
  Scal *sn = reinterpret_cast<Scal *>(c.grid_slots.p + 4 * kGridSet);
  hipLaunchKernelGGL(k_grid_reset, dim3(1), dim3(256), 0, stream(), c.grid_slots.p, s);
  const DiaRows g = dia_rows<T>(A);
  const int ns = g.count, rpt = rows_per_thread(A.n, ns, true), rows = kGridThreads * rpt;
  const auto go = [&](auto *kernel) {
    const int lds = (rows + 2 * g.halo) * (int)sizeof(T);
    hipLaunchKernelGGL(kernel, dim3((A.n + rows - 1) / rows), dim3(kGridThreads), lds, stream(), g,
                       A.dia_vals<T>(), jd, x, edge + 3 * (size_t)A.n, r, rhat, p, v, ph, edge, s, sn, c.grid_slots.p, steps,
                       A.resident_polls);
  };
#define CFDLA_GRID(RPT)                       \
  if (ns <= 3) go(k_grid_bicg<T, 3, RPT>);    \
  else if (ns <= 5) go(k_grid_bicg<T, 5, RPT>); \
  else go(k_grid_bicg<T, 7, RPT>);
  if (rpt == 1) { CFDLA_GRID(1) } else { CFDLA_GRID(2) }
#undef CFDLA_GRID
  commit<T>(A.n, edge + 3 * (size_t)A.n, x, sn, s);
}

#define CFDLA_INST(T)                                                                                          \
  template bool grid_krylov_takes<T>(const DevCsr &, bool);                                                    \
  template void grid_cg<T>(const DevCsr &, const T *, T *, T *, T *, T *, Scal *, int);                        \
  template void grid_bicgstab<T>(const DevCsr &, const T *, T *, T *, const T *, T *, T *, T *, T *, Scal *, int);
CFDLA_INST(double)
CFDLA_INST(float)
#undef CFDLA_INST

}  // namespace cfdla
