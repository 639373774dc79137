// Device-side FP64 bookkeeping of the SP2 loop: the branch decision for the
// next step and the absorption of a step's partial sums.  The mixed-precision
// loops, and the FP64 loop above 1280 tiles (leading dimension 2432 on), run
// them in a one-block kernel after each step.  The FP64 loop of smaller
// matrices runs them at the start of the next step's launch, in every
// workgroup, on an LDS copy of the state header: the launch and its gap (4.5 +
// 1 us per step) give way to about 2 us of reads that a workgroup needs anyway.  (A last-workgroup
// absorb at the end of the step was slower than a launch of its own: the
// device-scope fences it needs write back and invalidate the per-XCD L2s.)
#pragma once

#include "prg_internal.h"
#include "prg_tile.h"

#include <cmath>
#include <cstddef>

namespace prg {

// Decide the next SP2 step from the current X's traces (runs in thread 0).
// The branch rules restate src/prg_sp2_mod.F90: alg2 :319-363, genseq
// :469-513, alg1 :801-849, alg1_genseq :941-982, basic :89-119, replay
// variants :581-600 / :1060-1072 / :1288-1300, and the response loop of
// src/prg_response_mod.F90:730-770.
// pp: the branch log (pp[] of the state, or of the state the header was
// copied from).
__device__ inline void sp2_plan(Sp2State* s, const int* pp) {
  s->planned = 0;
  s->apply = 0;
  s->last = 0;
  if (s->done) return;
  const double occ = s->occ, tol = s->idemtol;
  const int v = s->variant;
  const int k = s->iter + 1;
  if (!isfinite(s->fro2) || !isfinite(s->trx) || !isfinite(s->trx_fresh)) {
    s->status = ERR_NUMERIC;
    s->done = 1;
    return;
  }
  switch (v) {
    case V_ALG2:
    case V_ALG2_GENSEQ:
    case V_RESPONSE: {
      if (s->iter >= s->maxit) { s->done = 1; return; }
      const double trx = (v == V_ALG2_GENSEQ) ? s->trx_fresh : s->trx;
      const double trx2 = s->fro2;
      if (s->refine_phase && s->refine_steps >= s->refine_max) { s->done = 1; return; }
      if (s->noise_stop && !s->refine_phase) {
        // low-precision products: stop where the idempotency error stops
        // falling quadratically (numerical noise floor)
        const double e = trx - trx2;
        const int it0 = s->iter;  // 0-based index of the step being planned
        const bool alt = it0 > 2 && pp[it0 - 1] != pp[it0 - 2];
        s->ie2 = s->ie1;
        s->ie1 = s->ie0;
        s->ie0 = e;
        if (e <= 0.0 || (alt && e >= 4.5 * s->ie2 * s->ie2)) {
          s->done = 1;
          return;
        }
      }
      const double tr2xx2 = 2.0 * trx - trx2;
      const double limdiff = fabs(trx2 - occ) - fabs(tr2xx2 - occ);
      s->trx2 = trx2;
      s->limdiff = limdiff;
      int stop = 0;
      if (limdiff >= tol) {
        s->sigma = 0;
        s->trx_next = tr2xx2;
      } else if (limdiff < -tol) {
        s->sigma = 1;
        s->trx_next = trx2;
      } else {
        stop = 1;
        s->trx_next = trx;
      }
      const double e_new = fabs(s->trx_next - trx);
      const int keff = (stop && v != V_RESPONSE) ? k - 1 : k;
      int last = stop;
      if (s->rel && keff >= s->minit && (e_new >= s->e1 || e_new < tol)) last = 1;
      if (!stop && k == s->maxit) {
        s->status = ERR_NOT_CONVERGED;
        last = 1;
      }
      if (s->refine_phase && s->refine_steps + 1 >= s->refine_max) last = 1;
      s->last = last;
      s->apply = !stop;
      s->planned = !stop || (v == V_ALG2_GENSEQ);
      if (!s->planned) {
        s->trx = s->trx_next;
        s->done = 1;
      }
      break;
    }
    case V_ALG1:
    case V_ALG1_GENSEQ: {
      if (s->iter >= s->maxit) { s->done = 1; return; }
      const double trx = s->trx;
      const double trx2 = s->trx_fresh - s->fro2;  // Tr(X - X^2)
      const double limdiff = fabs(trx - trx2 - occ) - fabs(trx + trx2 - occ);
      s->trx2 = trx2;
      s->limdiff = limdiff;
      int stop = 0;
      if (limdiff >= tol) {
        s->sigma = 0;
        s->trx_next = trx + trx2;
      } else if (limdiff < -tol) {
        s->sigma = 1;
        s->trx_next = trx - trx2;
      } else if (v == V_ALG1 && limdiff == 0.0 && k == 1) {
        s->sigma = 1;
        s->trx_next = trx - trx2;
      } else {
        stop = 1;
        s->trx_next = trx;
      }
      const double e_new = fabs(trx2);
      const int keff = stop ? k - 1 : k;
      int last = stop;
      if (s->rel && keff >= s->minit && (s->e1 <= e_new || e_new < tol)) last = 1;
      if (v == V_ALG1_GENSEQ && s->absconv && fabs(limdiff) < tol) last = 1;
      if (!stop && k == s->maxit) {
        s->status = ERR_NOT_CONVERGED;
        last = 1;
      }
      s->last = last;
      s->apply = !stop;
      s->planned = !stop || (v == V_ALG1_GENSEQ);
      if (!s->planned) s->done = 1;
      break;
    }
    case V_BASIC:
    case V_BASIC_FIXED: {
      // V_BASIC_FIXED (src/prg_sp2_mod.F90:138-246): the same branch rule run
      // for iterations 0..maxit with the convergence exit commented out
      // (:214) and only a message at maxit (:216-219)
      const int it = s->iter;  // reference loop index, starting at 0
      if (it > s->maxit) { s->done = 1; return; }
      const double trx = s->trx_fresh;
      s->trx2 = s->fro2;
      if (trx - occ <= 0.0) {
        s->sigma = 0;
        s->trx_next = 2.0 * trx - s->fro2;
      } else {
        s->sigma = 1;
        s->trx_next = s->fro2;
      }
      int last = (v == V_BASIC_FIXED) ? (it == s->maxit)
                                      : (fabs(occ - s->trx_next) < tol && it > s->minit);
      if (!last && it == s->maxit) {
        s->status = ERR_NOT_CONVERGED;
        last = 1;
      }
      s->last = last;
      s->apply = 1;
      s->planned = 1;
      break;
    }
    case V_SEQ_ALG2:
    case V_SEQ_ALG1:
    case V_SUBMATRIX: {
      if (s->iter >= s->icount) { s->done = 1; return; }
      s->sigma = pp[s->iter] != 0;
      s->trx_next = s->sigma ? s->fro2 : 2.0 * s->trx_fresh - s->fro2;
      s->apply = 1;
      s->planned = 1;
      s->last = (k == s->icount);
      break;
    }
    default:
      s->status = ERR_ARG;
      s->done = 1;
  }
}

// Fixed-order block sum of nb records of 4 partials (32 bytes each): one
// pass over the records, wave shuffles, then the BT / 64 wave totals (BT threads).
template <int BT>
__device__ inline void block_sum4(const double* part, int nb, double* out /*shared*/) {
  __shared__ double red[BT / 64][4];
  double a[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
  for (int b = threadIdx.x; b < nb; b += BT) {
    const double2 lo = *(const double2*)(part + 4 * (size_t)b);
    const double2 hi = *(const double2*)(part + 4 * (size_t)b + 2);
    a[0] += lo.x;
    a[1] += lo.y;
    a[2] += hi.x;
    a[3] += hi.y;
  }
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) a[q] += __shfl_xor(a[q], off);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) {
#pragma unroll
    for (int q = 0; q < 4; ++q) red[w][q] = a[q];
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    double t = 0.0;
#pragma unroll
    for (int ww = 0; ww < BT / 64; ++ww) t += red[ww][threadIdx.x];
    out[threadIdx.x] = t;
  }
  __syncthreads();
}

// Absorb the sums of the product just computed, then plan the next step (one
// thread).  pp, vv: the logs; written only if `log` (one workgroup of a
// launch that plans in all of them).
__device__ inline void sp2_absorb_sums(Sp2State* s, const double* sums, int* pp, double* vv,
                                       bool log) {
  const double fro2 = sums[0], trf = sums[1], idem = sums[2];
  s->x2_trace = sums[3];
  const int v = s->variant;
  const int k = s->iter + 1;
  const int idx = k - 1;
  if (log && idx < kMaxIter) {
    if (v == V_ALG2_GENSEQ || v == V_ALG1_GENSEQ || v == V_SEQ_ALG2 || v == V_SEQ_ALG1)
      vv[idx] = sqrt(idem);
    else if (v == V_SUBMATRIX)
      vv[idx] += idem;
  }
  double trx_old = (v == V_ALG2_GENSEQ) ? s->trx_fresh : s->trx;
  if (v == V_BASIC || v == V_BASIC_FIXED) trx_old = s->trx_fresh;
  if (s->apply) {
    if (log && v != V_SEQ_ALG2 && v != V_SEQ_ALG1 && v != V_SUBMATRIX && idx < kMaxIter)
      pp[idx] = s->sigma;
    s->iter = k;
    s->cur ^= 1;
    s->fro2 = fro2;
    s->trx_fresh = trf;
    s->trx = s->trx_next;
  } else {
    s->trx = s->trx_next;
  }
  // idempotency-error history (src/prg_sp2_mod.F90:352-354, :830-832)
  double e_new;
  if (v == V_ALG1 || v == V_ALG1_GENSEQ) e_new = fabs(s->trx2);
  else e_new = fabs(s->trx - trx_old);
  s->e2 = s->e1;
  s->e1 = s->e0;
  s->e0 = e_new;
  if (s->refine_phase && s->apply) s->refine_steps += 1;
  if (s->last) s->done = 1;
  sp2_plan(s, pp);
}

// The same from ntiles records of 4 partials.  Called by every thread of one
// BT-thread block of a launch whose step was planned.
template <int BT>
__device__ inline void sp2_absorb_plan_block(Sp2State* s, const double* part, int ntiles) {
  __shared__ double sums[4];
  block_sum4<BT>(part, ntiles, sums);
  if (threadIdx.x == 0) sp2_absorb_sums(s, sums, s->pp, s->vv, true);
}

// What an FP64 step launch reads first: the state header as the previous
// launch left it and the partial sums of the step that launch ran.  Every
// workgroup absorbs them into its own copy (the same operations in the same
// order everywhere) and workgroup 0 stores that copy as the next header, in
// the other slot, so that no workgroup reads what another writes.
struct Sp2Link {
  const Sp2State* in;
  Sp2State* out;       // null: the header is already planned and stays as it is
  int* pp;             // logs, in the first slot
  double* vv;
  const double* part;  // null: nothing to absorb (first step)
  int nparts;
};

constexpr int kSp2HeadBytes = (int)offsetof(Sp2State, pp);

// The reads of a link, issued before anything waits for them (wave 0 of the
// workgroup; every thread learns `planned`, the header's flag before the
// absorption: 0 when the loop had ended).
struct Sp2LinkReads {
  static constexpr int kRecords = 4;  // per lane: 256 workgroups' sums
  uint32_t word;
  double2 lo[kRecords], hi[kRecords];
  int planned;
};

__device__ __forceinline__ void sp2_link_read(const Sp2Link& l, Sp2LinkReads& r) {
  static_assert(kSp2HeadBytes % 4 == 0 && kSp2HeadBytes / 4 <= 64, "one header word per lane");
  r.planned = l.in->planned;
  if (threadIdx.x >= 64) return;
  if (threadIdx.x < kSp2HeadBytes / 4) r.word = ((const uint32_t*)l.in)[threadIdx.x];
#pragma unroll
  for (int i = 0; i < Sp2LinkReads::kRecords; ++i) {
    const int b = threadIdx.x + 64 * i;
    r.lo[i] = r.hi[i] = double2{0.0, 0.0};
    if (l.part && b < l.nparts) {
      r.lo[i] = *(const double2*)(l.part + 4 * (size_t)b);
      r.hi[i] = *(const double2*)(l.part + 4 * (size_t)b + 2);
    }
  }
}

// Wave 0 leaves the planned header in `head` (LDS, kSp2HeadBytes; the other
// waves see it after the next barrier), workgroup 0's also in the other slot.
__device__ __forceinline__ void sp2_link(const Sp2Link& l, Sp2LinkReads& r, char* head) {
  if (threadIdx.x >= 64) return;
  constexpr int words = kSp2HeadBytes / 4;
  if (threadIdx.x < words) ((uint32_t*)head)[threadIdx.x] = r.word;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  if (l.part && r.planned) {
    double a[4] = {0.0, 0.0, 0.0, 0.0};
    auto add = [&](double2 lo, double2 hi) {
      a[0] += lo.x;
      a[1] += lo.y;
      a[2] += hi.x;
      a[3] += hi.y;
    };
#pragma unroll
    for (int i = 0; i < Sp2LinkReads::kRecords; ++i) add(r.lo[i], r.hi[i]);
#pragma unroll 4
    for (int b = threadIdx.x + 64 * Sp2LinkReads::kRecords; b < l.nparts; b += 64)
      add(*(const double2*)(l.part + 4 * (size_t)b), *(const double2*)(l.part + 4 * (size_t)b + 2));
    tile::wave_sum4(a);
    if (threadIdx.x == 0) sp2_absorb_sums((Sp2State*)head, a, l.pp, l.vv, blockIdx.x == 0);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  if (l.out && blockIdx.x == 0 && threadIdx.x < words)
    ((uint32_t*)l.out)[threadIdx.x] = ((const volatile uint32_t*)head)[threadIdx.x];
}

}  // namespace prg
