// Scalars of the CG iterations (Jacobi-PCG and AMG-CG) and the reductions that a consuming
// kernel does itself (pcg.hip, amg.hip, patch.hip).
#pragma once
#include "fem_common.hpp"

namespace fem {

struct PcgScalars {
  double rz;             // <r, z> of the current iteration
  double alpha, beta;
  double rr;             // <r, r> of the current iteration
  double rr_true;        // |b - A x|^2 of the last true-residual evaluation
  double pad0[3];
  int32_t done, iter, nan;
  int32_t ready;         // 1: rz, rr and beta are those of the partials last written; 0: to be summed
  int32_t pad2[4];
};
static_assert(sizeof(PcgScalars) <= 128, "host status buffer");

// Sum of `n` partials starting at p, identical in every block (blockDim == 256).
__device__ inline double block_reduce_partials(const double* __restrict__ p, int n, double* smem) {
  double acc = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) acc += p[i];
  return block_sum_256(acc, smem);
}

// End of an iteration, done by every block of the kernel that begins the next one: <r, z> and
// <r, r> from the update kernel's partials, the stop test and beta.  The state is read from
// `cur` and block 0 writes it to `next` (two slots, so no block reads what another writes).
// A reduction of at most 1024 partials by every block costs about 1 us of latency where a
// kernel of its own cost 3 us and its launch 1.6 us.
struct PcgHead {
  const PcgScalars* cur;
  PcgScalars* next;
  const double* part;    // (2 * parts): <r, z>, then <r, r>
  int parts;
  double tol2;
  int maxiter;
};

// The state after the partials; smem holds 2 * NT / 64 doubles.  The partials are loaded with
// the state, not after it.
struct PcgState {
  double rz, rr, beta;
  int32_t done, iter, nan;
};

// What a kernel loads for its head.  A kernel takes this first, issues its own loads and only then
// finishes the head: the reduction's latency (two barriers and the loads, 1.5 us) runs beside them
// (per iteration: 2,184-node J2 system 12.1 -> 10.3 us, 65,536-cell elastic system 26 -> 22.5).
constexpr int kHeadParts = 1024;  // partials held in registers; more are summed when the head ends
template <int NT>
struct PcgRaw {
  static constexpr int PER = kHeadParts / NT;
  double a0[PER], a1[PER];
  PcgState s;
  int32_t ready;
};
template <int NT>
__device__ inline PcgRaw<NT> pcg_raw(const PcgHead& h) {
  PcgRaw<NT> r;
#pragma unroll
  for (int k = 0; k < PcgRaw<NT>::PER; ++k) {
    const int i = threadIdx.x + k * NT;
    const bool in = i < h.parts;
    r.a0[k] = in ? h.part[i] : 0.0;
    r.a1[k] = in ? h.part[h.parts + i] : 0.0;
  }
  r.s = PcgState{h.cur->rz, h.cur->rr, h.cur->beta, h.cur->done, h.cur->iter, h.cur->nan};
  r.ready = h.cur->ready;
  return r;
}

template <int NT>
__device__ inline PcgState pcg_state(const PcgHead& h, const PcgRaw<NT>& raw, double* smem) {
  PcgState s = raw.s;
  if (s.done || raw.ready) return s;
  double a0 = 0.0, a1 = 0.0;
#pragma unroll
  for (int k = 0; k < PcgRaw<NT>::PER; ++k) {
    a0 += raw.a0[k];
    a1 += raw.a1[k];
  }
  for (int i = threadIdx.x + PcgRaw<NT>::PER * NT; i < h.parts; i += NT) {
    a0 += h.part[i];
    a1 += h.part[h.parts + i];
  }
  block_sum2<NT>(a0, a1, smem);
  const bool bad = !isfinite(a1) || !isfinite(a0);
  s.beta = a0 / s.rz;
  s.rz = a0;
  s.rr = a1;
  s.iter += 1;
  if (bad) s.nan = 1;
  if (bad || a1 <= h.tol2 || s.iter >= h.maxiter) s.done = 1;
  return s;
}

__device__ inline void pcg_store(PcgScalars* out, const PcgState& s, int ready) {
  out->rz = s.rz;
  out->rr = s.rr;
  out->beta = s.beta;
  out->done = s.done;
  out->iter = s.iter;
  out->nan = s.nan;
  out->ready = ready;
}

// beta of the iteration that begins, or done = true.
template <int NT>
__device__ inline double pcg_head(const PcgHead& h, const PcgRaw<NT>& raw, double* smem, bool* done) {
  const PcgState s = pcg_state<NT>(h, raw, smem);
  if (blockIdx.x == 0 && threadIdx.x == 0) pcg_store(h.next, s, 0);
  *done = s.done != 0;
  return s.beta;
}

constexpr int kSumParts = 2048;  // most partials that every block of a consuming kernel sums itself

// AMG-CG.  rz: <r, z> of the last two iterations (slot = iteration & 1), so that the kernel that
// forms a new one reads what none of its blocks writes.
struct AmgScalars {
  double rz[2], alpha, beta, rr, stop2, bb;
  int32_t done, iter, nan, pad;
};
static_assert(sizeof(AmgScalars) <= 128, "host status buffer");

// beta of iteration `it` (0: the first), summed by every block of the product that needs it from
// the <r, z> partials of the V-cycle's last kernel.
struct CgHead {
  AmgScalars* sc;
  const double* part;
  int parts, it;
};

template <int NT>
struct CgRaw {
  static constexpr int PER = kHeadParts / NT;
  double a[PER], old;
  int32_t done;
};
template <int NT>
__device__ inline CgRaw<NT> cg_raw(const CgHead& h) {
  CgRaw<NT> r;
#pragma unroll
  for (int k = 0; k < CgRaw<NT>::PER; ++k) {
    const int i = threadIdx.x + k * NT;
    r.a[k] = i < h.parts ? h.part[i] : 0.0;
  }
  r.old = h.sc->rz[(h.it + 1) & 1];
  r.done = h.sc->done;
  return r;
}

template <int NT>
__device__ inline double cg_head(const CgHead& h, const CgRaw<NT>& raw, double* smem, bool* done) {
  const double old = raw.old;
  if (raw.done) {
    *done = true;
    return 0.0;
  }
  double a = 0.0;
#pragma unroll
  for (int k = 0; k < CgRaw<NT>::PER; ++k) a += raw.a[k];
  for (int i = threadIdx.x + CgRaw<NT>::PER * NT; i < h.parts; i += NT) a += h.part[i];
  a = block_sum<NT>(a, smem);
  *done = !isfinite(a);
  const double beta = h.it == 0 ? 0.0 : a / old;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    if (*done) {
      h.sc->nan = 1;
      h.sc->done = 1;
    } else {
      h.sc->rz[h.it & 1] = a;
      h.sc->beta = beta;
    }
  }
  return beta;
}

}  // namespace fem
