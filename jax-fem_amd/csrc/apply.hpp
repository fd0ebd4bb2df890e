// Epilogues of the operator products: what a kernel does with (A x)_i once it
// has the sum.  Shared by the AMG operators and the matrix-free products.
#pragma once
#include "fem_common.hpp"

namespace fem {

// AP_CHEBZ: AP_CHEB and the partials of <rhs, y> (matrix-free products only); AP_FIRST: the
// product as right-hand side of the next level, and that level's first Chebyshev step.
enum { AP_STORE = 0, AP_ADD = 1, AP_RESID = 2, AP_CHEB = 3, AP_DSTORE = 4, AP_PQ = 5, AP_CHEBZ = 6, AP_FIRST = 7 };

// TX: storage of the input vector and of the Chebyshev direction, TY: of the
// output.  Arithmetic is FP64 whatever the storage; the V-cycle's vectors are
// FP64, the level-0 power iteration on the FP32 copy keeps FP32 iterates.
template <typename TX = double, typename TY = double>
struct ApplyArgsT {
  const TX* x;         // gathered input
  TY* y;               // output (CHEB: the new iterate)
  const double* rhs;   // RESID, CHEB
  const double* dinv;  // CHEB, DSTORE, FIRST
  TX* d;               // CHEB: search direction (in/out)
  double c1, c2;       // CHEB: d = c1 d + c2 D^-1 (rhs - A x), y = x + d
  double* part;        // PQ: per-block partials of <x, A x>; CHEBZ: of <rhs, y>
  const int32_t* done; // NULL, or a flag: the kernel returns at once when it is set
                       // (V-cycles queued after the outer CG converged)
  TY* first = nullptr; // FIRST: d = first = c2 D^-1 A x, the iterate after a step from zero
};
using ApplyArgs = ApplyArgsT<double, double>;

// The epilogue's own-entry operands (loaded ahead of the product where a kernel can
// overlap their latency with it) and the epilogue itself.
struct EpiOperands {
  double y, rhs, dinv, d, x;
};

template <int MODE, typename TX, typename TY>
__device__ inline EpiOperands epilogue_load(const ApplyArgsT<TX, TY>& a, int64_t idx) {
  EpiOperands e{0.0, 0.0, 0.0, 0.0, 0.0};
  if (MODE == AP_ADD) e.y = double(a.y[idx]);
  if (MODE == AP_RESID || MODE == AP_CHEB) e.rhs = a.rhs[idx];
  if (MODE == AP_CHEB || MODE == AP_DSTORE || MODE == AP_FIRST) e.dinv = a.dinv[idx];
  if (MODE == AP_CHEB && a.c1 != 0.0) e.d = double(a.d[idx]);
  if (MODE == AP_CHEB) e.x = double(a.x[idx]);
  return e;
}

// (returns what y received)
template <int MODE, typename TX, typename TY>
__device__ inline double epilogue_store(const ApplyArgsT<TX, TY>& a, int64_t idx, double ax, const EpiOperands& e) {
  double y = ax;
  if (MODE == AP_ADD) {
    y = e.y + ax;
  } else if (MODE == AP_RESID) {
    y = e.rhs - ax;
  } else if (MODE == AP_DSTORE) {
    y = e.dinv * ax;
  } else if (MODE == AP_FIRST) {
    const TX v = TX(a.c2 * e.dinv * ax);
    a.d[idx] = v;
    a.first[idx] = TY(v);
  } else if (MODE == AP_CHEB) {
    const double r = e.dinv * (e.rhs - ax);
    const double dn = a.c1 != 0.0 ? fma(a.c1, e.d, a.c2 * r) : a.c2 * r;
    a.d[idx] = TX(dn);
    y = e.x + dn;
  }
  a.y[idx] = TY(y);
  return double(TY(y));
}

template <int MODE, typename TX, typename TY>
__device__ inline void apply_epilogue(const ApplyArgsT<TX, TY>& a, int64_t idx, double ax) {
  epilogue_store<MODE>(a, idx, ax, epilogue_load<MODE>(a, idx));
}

}  // namespace fem
