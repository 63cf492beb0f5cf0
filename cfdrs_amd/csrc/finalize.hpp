// The finalize ops that advance the Krylov scalars once a reduction's block
// partials are summed, and their evaluation inside the next kernel.
//
// A reduction over few blocks is not finalized by a launch of its own (2.6-3 us
// of latency for a sum of at most kConsumeBlocks values): it stays pending
// (take_pending in kernels.hip) and every block of the next kernel that
// depends on it sums the partials itself, in k_finalize's order, and runs the
// op on a copy of the scalars in LDS; block 0 writes that copy to the other
// slot of the pair, so no block reads a value that another one has already
// advanced.  The result is k_finalize's bit for bit.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

#include "internal.hpp"
#include "reduce.hpp"

namespace cfdla {

__device__ inline void finalize(Scal *s, int op) {
  switch (op) {
    case OP_INIT_RR:
      s->rr = s->red[0];
      break;
    case OP_SET_RZ:
      s->rz = s->red[0];
      break;
    case OP_CG_ALPHA: {
      double pq = s->red[0];
      s->pq = pq;
      if (!(pq > 0.0) || !isfinite(pq)) {
        s->term = CFDLA_TERM_NONPOSITIVE_CURVATURE;
        s->done = 2;
      } else {
        s->alpha = s->rz / pq;
      }
    } break;
    case OP_CG_RR: {
      double rr = s->red[0];
      s->rr = rr;
      s->iters += 1;
      if (!isfinite(rr)) {
        s->term = CFDLA_TERM_BREAKDOWN;
        s->done = 2;
      } else if (rr <= s->thr2) {
        s->done = 1;
      }
    } break;
    case OP_CG_BETA: {
      double rzn = s->red[0];
      if (rzn == 0.0 || !isfinite(rzn)) {
        s->term = CFDLA_TERM_BREAKDOWN;
        s->done = 2;
      } else {
        s->beta = s->restart_dir ? 0.0 : rzn / s->rz;
        s->restart_dir = 0;
        s->rz = rzn;
      }
    } break;
    case OP_CG_RR_RZ: {
      double rr = s->red[0], rzn = s->red[1];
      s->rr = rr;
      s->iters += 1;
      if (!isfinite(rr)) {
        s->term = CFDLA_TERM_BREAKDOWN;
        s->done = 2;
      } else if (rr <= s->thr2) {
        s->done = 1;
      } else if (rzn == 0.0 || !isfinite(rzn)) {
        s->term = CFDLA_TERM_BREAKDOWN;
        s->done = 2;
      } else {
        s->beta = rzn / s->rz;
        s->rz = rzn;
      }
    } break;
    case OP_BI_RHO: {
      double rho_new = s->red[0];
      if (rho_new == 0.0 || !isfinite(rho_new)) {
        s->term = CFDLA_TERM_BREAKDOWN;
        s->done = 2;
      } else {
        // a residual replacement far from the recurrence restarts p = r
        s->beta = s->restart_dir ? 0.0 : (rho_new / s->rho) * (s->alpha / s->omega);
        s->restart_dir = 0;
        s->rho = rho_new;
      }
    } break;
    case OP_BI_ALPHA: {
      double rv = s->red[0];
      if (rv == 0.0 || !isfinite(rv)) {
        s->term = CFDLA_TERM_BREAKDOWN;
        s->done = 2;
      } else {
        s->alpha = s->rho / rv;
      }
    } break;
    case OP_BI_SNORM: {
      double ss = s->red[0];
      s->iters += 1;
      if (!isfinite(ss)) {
        s->term = CFDLA_TERM_BREAKDOWN;
        s->done = 2;
      } else if (ss <= s->thr2) {
        s->done = 3;  // x += alpha * phat, then confirm on the host
      }
    } break;
    case OP_BI_OMEGA: {
      double ts = s->red[0], tt = s->red[1];
      s->omega = tt > 0.0 ? ts / tt : 0.0;
    } break;
    case OP_RELIABLE: {
      // FP64 residual of the accumulated FP64 solution (reliable-update CG)
      // A replaced residual far above the recursive one it replaces (the
      // FP32 operator's rounding caps what one cycle can gain) would make
      // beta = r.z / rz blow up and wreck the direction: restart it.
      double rr = s->red[0];
      const double rec = s->rr;
      s->rr = rr;
      s->rr_true = rr;
      s->nupd += 1;
      if (!isfinite(rr)) {
        s->term = CFDLA_TERM_BREAKDOWN;
        s->done = 2;
      } else {
        s->done = rr <= s->thr_final2 ? 4 : 0;
        s->restart_dir = rr > 4.0 * rec ? 1 : 0;
        s->nrestart += s->restart_dir;
      }
    } break;
    case OP_BI_RR:
    case OP_BI_RR_RHO: {
      double rr = s->red[0];
      s->rr = rr;
      if (!isfinite(rr)) {
        s->term = CFDLA_TERM_BREAKDOWN;
        s->done = 2;
      } else if (rr <= s->thr2) {
        s->done = 1;
      } else if (s->omega == 0.0 || !isfinite(s->omega)) {
        s->term = CFDLA_TERM_BREAKDOWN;
        s->done = 2;
      } else if (op == OP_BI_RR_RHO) {
        // the next iteration's OP_BI_RHO, with rho_new = rhat . r
        double rho_new = s->red[1];
        if (rho_new == 0.0 || !isfinite(rho_new)) {
          s->term = CFDLA_TERM_BREAKDOWN;
          s->done = 2;
        } else {
          s->beta = s->restart_dir ? 0.0 : (rho_new / s->rho) * (s->alpha / s->omega);
          s->restart_dir = 0;
          s->rho = rho_new;
        }
      }
    } break;
    default:
      break;
  }
}


// Sums the pending partials and leaves the advanced scalars in sc (LDS, valid
// after the call).  Every thread of the block calls it.
__device__ __forceinline__ void consume(const Pend &pd, Scal &sc) {
  constexpr int kWords = sizeof(Scal) / sizeof(int);
  static_assert(kWords <= kBlock, "one word of the scalars per thread");
  const int tid = threadIdx.x;
  if (tid < kWords) reinterpret_cast<int *>(&sc)[tid] = reinterpret_cast<const int *>(pd.in)[tid];
  if (pd.nblocks > 0) {
    double tot[2] = {0.0, 0.0};
    if (pd.nv == 1) {
      double t[1];
      sum_partials<1>(pd.nblocks, pd.partials, t);
      tot[0] = t[0];
    } else {
      sum_partials<2>(pd.nblocks, pd.partials, tot);
    }
    if (tid == 0 && !(pd.check_done && sc.done)) {
      sc.red[0] = tot[0];
      if (pd.nv > 1) sc.red[1] = tot[1];
      finalize(&sc, pd.op);
    }
  }
  __syncthreads();
  if (blockIdx.x == 0 && pd.out != pd.in && tid < kWords)
    reinterpret_cast<int *>(pd.out)[tid] = reinterpret_cast<const int *>(&sc)[tid];
}

}  // namespace cfdla
