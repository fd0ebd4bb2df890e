// Jacobi-preconditioned conjugate gradients on the SELL-64 block matrix.
//
// Replaces the default linear solve of jax-fem (solver.py:63-92, jax_solve:
// host CSR -> scipy -> BCOO conversion on every call, then BiCGSTAB with
// M = x / diag(A), tol = atol = 1e-10, maxiter 10000).  The Dirichlet rows of
// A are identity rows (solver.py:527-528) and the initial guess carries the
// exact boundary increment (solver.py:402-409), so the residual and search
// direction vanish on those rows and CG runs on the SPD free block.
//
// Launches per iteration k:
//   P_k : ends iteration k-1 (rz, rr, stop test, beta from B's partials, summed by
//         every block); p = z + beta p (row-local, in place)
//   A_k : q = A p, per-block <p, q> (one 64-row slice per block, W waves
//         splitting its slots; the product gathers p only), or the two kernels
//         of a matrix-free product (patch.hip)
//   B_k : alpha = rz / pq from A's partials, summed by every block;
//         x += alpha p, r -= alpha q, z = D^-1 r, per-block <r,z>, <r,r>
// Where the matrix stays in the caches, and in the matrix-free products, P's
// work is done by the product's kernel, which gathers z and the old direction.
// (On matrices read from HBM that gather costs ~20% of the product's bandwidth;
// there P streams 3 vectors once, and a one-block kernel RA sums more than 2048
// partials.)  The five kernels of separate reductions took 26 us per iteration
// on small systems, of which 6 in the reductions and 8 in gaps; two take 13.
// The reductions sum per-block partials in a fixed order (bit-reproducible);
// no grid-wide fence or atomic is used.  Scalars live in device memory and
// are written by one kernel and read by the next.
//
// Precision FEM_F64: everything FP64, standard matrix form.
// FEM_F32: FP32 matrix in difference form, FP32 r, z, p, q (FP32 storage,
// FP64 arithmetic inside the product); x accumulated in FP64; the recursive
// residual is replaced by the FP64 true residual b - A x
// (A applied matrix-free in FP64) each time it has dropped by reliable_delta
// and at convergence; beta keeps the value of the recursion across a
// replacement.
#include "patch.hpp"
#include "pcg_scalars.hpp"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <vector>

int fem_operator_apply_impl(const fem_operator_t* op, const double* x, double* y, hipStream_t s);

namespace fem {

// Kernel P: begins the iteration; p = z + beta p in place (beta = 0 at a start).
template <typename T>
__global__ __launch_bounds__(256) void k_pcg_p(int64_t n, const T* __restrict__ z, T* __restrict__ p, PcgHead head) {
  __shared__ double smem[8];
  bool done;
  const T beta = T(pcg_head<256>(head, pcg_raw<256>(head), smem, &done));
  if (done) return;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = fma(beta, p[i], z[i]);
}

// Kernel A: one 64-row slice per block; the W waves split the slots
// (sell_slice_partial) and wave 0 combines them through LDS, stores
// q = A p and the block's <p, q>.
// FUSED: the kernel begins the iteration (pcg_head) and multiplies p = z + beta p_old, formed
// where it is gathered; each row's own entries go to pn.
template <int V, bool DIFF, typename T, bool FUSED, int W = SliceCfg<T>::W>
__global__ __launch_bounds__(64 * W) void k_pcg_a(fem_pattern_t pat, const T* __restrict__ vals,
                                                           const T* __restrict__ p, const T* __restrict__ z,
                                                           T* __restrict__ pn, T* __restrict__ q,
                                                           const PcgScalars* sc, PcgHead head,
                                                           double* __restrict__ partA, int remap) {
  constexpr int U = SliceCfg<T>::U, NT = 64 * W;
  // small matrices (W >= 8): a wave's first slots (all of them for rows of up to 32 blocks at W = 16
  // or scalar blocks) are loaded, and their vector entries gathered, before the head's reduction is
  // waited for; as many as leave two workgroups on a CU
  constexpr int NS = FUSED && W >= 8 && V <= 3 ? (W == 8 && V == 1 ? 4 : 2) : 0, VV = V * V;
  __shared__ double smem[2 * (NT / 64)];
  __shared__ double red[W][kSlice][V];
  PcgRaw<NT> raw;
  if constexpr (FUSED)
    raw = pcg_raw<NT>(head);
  else if (sc->done)
    return;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t s = remap ? xcd_logical_block(blockIdx.x, gridDim.x) : blockIdx.x;
  const int64_t row = pat.sell_row[s * kSlice + lane];
  const bool real = row >= 0;
  const int base = NS ? pat.slice_ptr[s] : 0, L = NS ? (pat.slice_ptr[s + 1] - base) >> 6 : 0;
  int32_t sc_[NS ? NS : 1];
  T sv[NS ? NS : 1][VV], sp[NS ? NS : 1][V], sz[NS ? NS : 1][V], rp[V], rz[V];
  if constexpr (NS > 0) {
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      const int k = w + W * i;
      sc_[i] = k < L ? pat.sell_col[base + lane + k * kSlice] : 0;
#pragma unroll
      for (int v = 0; v < VV; ++v)
        sv[i][v] = k < L ? vals[((size_t)base + (size_t)k * kSlice) * VV + (size_t)v * kSlice + lane] : T(0);
    }
#pragma unroll
    for (int i = 0; i < NS; ++i)
#pragma unroll
      for (int j = 0; j < V; ++j) {
        sp[i][j] = p[(int64_t)sc_[i] * V + j];
        sz[i][j] = z[(int64_t)sc_[i] * V + j];
      }
#pragma unroll
    for (int j = 0; j < V; ++j) {
      rp[j] = p[(real ? row : 0) * V + j];
      rz[j] = z[(real ? row : 0) * V + j];
    }
  }
  T beta = T(0);
  if constexpr (FUSED) {
    bool done;
    beta = T(pcg_head<NT>(head, raw, smem, &done));
    if (done) return;
  }
  auto xat = [&](int64_t c, T (&xc)[V]) {
#pragma unroll
    for (int j = 0; j < V; ++j) xc[j] = FUSED ? fma(beta, p[c * V + j], z[c * V + j]) : p[c * V + j];
  };
  T pr[V];
  if constexpr (NS > 0) {
#pragma unroll
    for (int j = 0; j < V; ++j) pr[j] = fma(beta, rp[j], rz[j]);
  } else {
    xat(real ? row : 0, pr);
  }
  double xr[V], acc[V];
#pragma unroll
  for (int j = 0; j < V; ++j) xr[j] = double(pr[j]);
  if constexpr (NS > 0) {
#pragma unroll
    for (int i = 0; i < V; ++i) acc[i] = 0.0;
    auto add = [&](int64_t c, const T (&xt)[V], const T (&a)[VV]) {
      double xc[V];
#pragma unroll
      for (int j = 0; j < V; ++j) xc[j] = (DIFF && c != row) ? double(xt[j]) - xr[j] : double(xt[j]);
#pragma unroll
      for (int i = 0; i < V; ++i)
#pragma unroll
        for (int j = 0; j < V; ++j) acc[i] = fma(double(a[i * V + j]), xc[j], acc[i]);
    };
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      if (w + W * i >= L) continue;
      T xt[V];
#pragma unroll
      for (int j = 0; j < V; ++j) xt[j] = fma(beta, sp[i][j], sz[i][j]);
      add(sc_[i], xt, sv[i]);
    }
    for (int k = w + W * NS; k < L; k += W) {
      const int64_t c = pat.sell_col[base + lane + k * kSlice];
      T xt[V], a[VV];
      xat(c, xt);
#pragma unroll
      for (int v = 0; v < VV; ++v) a[v] = vals[((size_t)base + (size_t)k * kSlice) * VV + (size_t)v * kSlice + lane];
      add(c, xt, a);
    }
  } else {
    sell_slice_partial<V, DIFF, W, U, T>(pat, vals, s, w, lane, row, xat, xr, acc);
  }
  if (FUSED && w == 0 && real) {
#pragma unroll
    for (int j = 0; j < V; ++j) pn[row * V + j] = pr[j];
  }
  if (w > 0) {
#pragma unroll
    for (int i = 0; i < V; ++i) red[w][lane][i] = acc[i];
  }
  __syncthreads();
  double dot = 0.0;
  if (w == 0 && real) {
#pragma unroll
    for (int i = 0; i < V; ++i) {
      double t = acc[i];
#pragma unroll
      for (int o = 1; o < W; ++o) t += red[o][lane][i];
      const T qi = T(t);
      q[row * V + i] = qi;
      dot += xr[i] * double(qi);
    }
  }
  const double d = block_sum<NT>(dot, smem);
  if (threadIdx.x == 0) partA[blockIdx.x] = d;
}

// A batch of iterations of a small scalar system in one workgroup: nothing is launched and no
// vector or partial passes through memory between iterations.  Wave w takes the slices w and 8 + w
// with their matrix in registers and, of systems of more than 16 slices, slice 16 + w with its matrix
// in LDS (the first kOneSlots entries of each row; longer rows read the rest where it is); x, r, z, p
// and D^-1 stay in registers and the direction is exchanged through LDS.  The limit is what registers
// (256 per lane of eight waves) and LDS hold.  Two launches per iteration take 9 us, most of it launch and load latency;
// this 4.7 (1,331 rows; Poisson solve of 1,000 cells 2.50 -> 2.13 ms).
constexpr int kOneWaves = 8, kOneExtra = 6, kOneSlots = 32;
constexpr int kOneSlices = 2 * kOneWaves + kOneExtra, kOneGroup = 8;
template <typename T>
struct OneLds {
  T p[kOneSlices * kSlice];
  T a[kOneExtra][kOneSlots][kSlice];
  uint16_t col[kOneExtra][kOneSlots][kSlice];
  double smem[2 * kOneWaves];
};
template <bool DIFF, typename T>
__global__ __launch_bounds__(64 * kOneWaves) void k_pcg_one(fem_pattern_t pat, const T* __restrict__ vals,
                                                            double* __restrict__ x, T* __restrict__ r,
                                                            T* __restrict__ z, T* __restrict__ p,
                                                            const T* __restrict__ dinv, PcgHead head, int batch) {
  constexpr int NT = 64 * kOneWaves;
  __shared__ OneLds<T> S;
  const PcgRaw<NT> raw = pcg_raw<NT>(head);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  constexpr int H = 3;  // slices of a wave: two in registers, one in LDS
  int row[H], base[H], L[H];
  double xi[H];
  T ri[H], zi[H], pi[H], di[H];
#pragma unroll
  for (int h = 0; h < H; ++h) {
    const int sl = w + h * kOneWaves;
    const bool in = sl < pat.num_slices;
    row[h] = in ? pat.sell_row[sl * kSlice + lane] : -1;
    base[h] = in ? pat.slice_ptr[sl] : 0;
    L[h] = in ? (pat.slice_ptr[sl + 1] - base[h]) >> 6 : 0;
    xi[h] = 0.0;
    ri[h] = zi[h] = pi[h] = di[h] = T(0);
    if (row[h] >= 0) {
      xi[h] = x[row[h]];
      ri[h] = r[row[h]];
      zi[h] = z[row[h]];
      pi[h] = p[row[h]];
      di[h] = dinv[row[h]];
    }
  }
  T a[2][kOneSlots];
  uint32_t col[2][kOneSlots / 2];  // two 16-bit columns each
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int k = 0; k < kOneSlots; ++k) {
      a[h][k] = k < L[h] ? vals[base[h] + k * kSlice + lane] : T(0);
      const uint32_t c = k < L[h] ? (uint32_t)pat.sell_col[base[h] + k * kSlice + lane] : 0u;
      col[h][k / 2] = k & 1 ? col[h][k / 2] | c << 16 : c;
    }
  // padded with zeros to whole groups of slots
  const int l2 = (min(L[2], kOneSlots) + kOneGroup - 1) / kOneGroup * kOneGroup;
  for (int k = 0; k < l2; ++k) {
    S.a[w][k][lane] = k < L[2] ? vals[base[2] + k * kSlice + lane] : T(0);
    S.col[w][k][lane] = k < L[2] ? (uint16_t)pat.sell_col[base[2] + k * kSlice + lane] : (uint16_t)0;
  }
  PcgState st = pcg_state<NT>(head, raw, S.smem);
  for (int m = 0; m < batch && !st.done; ++m) {
    __syncthreads();  // the last iteration's directions are no longer read
#pragma unroll
    for (int h = 0; h < H; ++h) {
      pi[h] = fma(T(st.beta), pi[h], zi[h]);
      if (row[h] >= 0) S.p[row[h]] = pi[h];
    }
    __syncthreads();
    double acc[H] = {0.0, 0.0, 0.0};
    auto add = [&](int h, T v, int c) {
      const double xc = double(S.p[c]);
      acc[h] = fma(double(v), DIFF && c != row[h] ? xc - double(pi[h]) : xc, acc[h]);
    };
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int k0 = 0; k0 < kOneSlots; k0 += kOneGroup)
        if (k0 < L[h])  // (a branch for every slot would wait for each gather in turn)
#pragma unroll
          for (int k = k0; k < k0 + kOneGroup; ++k)
            add(h, a[h][k], (int)((col[h][k / 2] >> (k & 1 ? 16 : 0)) & 0xffffu));
    for (int k0 = 0; k0 < l2; k0 += kOneGroup)
#pragma unroll
      for (int k = 0; k < kOneGroup; ++k) add(2, S.a[w][k0 + k][lane], S.col[w][k0 + k][lane]);
#pragma unroll
    for (int h = 0; h < H; ++h)
      for (int k = kOneSlots; k < L[h]; ++k)
        add(h, vals[base[h] + k * kSlice + lane], pat.sell_col[base[h] + k * kSlice + lane]);
    T qi[H];
    double dot = 0.0;
#pragma unroll
    for (int h = 0; h < H; ++h) {
      qi[h] = row[h] >= 0 ? T(acc[h]) : T(0);
      dot = fma(double(pi[h]), double(qi[h]), dot);
    }
    const double alpha = st.rz / block_sum<NT>(dot, S.smem);
    double a0 = 0.0, a1 = 0.0;
#pragma unroll
    for (int h = 0; h < H; ++h)
      if (row[h] >= 0) {
        xi[h] += alpha * double(pi[h]);
        ri[h] = ri[h] - T(alpha) * qi[h];
        zi[h] = di[h] * ri[h];
        a0 += double(ri[h] * zi[h]);
        a1 += double(ri[h] * ri[h]);
      }
    block_sum2<NT>(a0, a1, S.smem);
    const bool bad = !isfinite(a1) || !isfinite(a0);
    st.beta = a0 / st.rz;
    st.rz = a0;
    st.rr = a1;
    st.iter += 1;
    if (bad) st.nan = 1;
    if (bad || a1 <= head.tol2 || st.iter >= head.maxiter) st.done = 1;
  }
#pragma unroll
  for (int h = 0; h < H; ++h)
    if (row[h] >= 0) {
      x[row[h]] = xi[h];
      r[row[h]] = ri[h];
      z[row[h]] = zi[h];
      p[row[h]] = pi[h];
    }
  if (threadIdx.x == 0) pcg_store(head.next, st, 1);
}

// RA: alpha = rz / sum(partA).  Eight independent loads per thread are in
// flight at once (the sum is latency-bound); the order of the sum is fixed.
__global__ __launch_bounds__(1024) void k_pcg_ra(const double* __restrict__ partA, int nA, PcgScalars* sc) {
  __shared__ double smem[16];
  double a[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) a[u] = 0.0;
  for (int base = 0; base < nA; base += 8 * 1024) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = base + u * 1024 + (int)threadIdx.x;
      if (i < nA) a[u] += partA[i];
    }
  }
  const double t = ((a[0] + a[1]) + (a[2] + a[3])) + ((a[4] + a[5]) + (a[6] + a[7]));
  const double pq = block_sum<1024>(t, smem);
  if (sc->done) return;
  if (threadIdx.x == 0) sc->alpha = sc->rz / pq;
}

// RB: rz, rr and beta of the iteration that ended, its stop test (head.next may be head.cur).
__global__ __launch_bounds__(1024) void k_pcg_rb(PcgHead head) {
  __shared__ double smem[32];
  const PcgState s = pcg_state<1024>(head, pcg_raw<1024>(head), smem);
  __syncthreads();
  if (threadIdx.x == 0) pcg_store(head.next, s, 1);
}

template <typename T, typename TX>
__global__ __launch_bounds__(256) void k_pcg_b(int64_t n, TX* __restrict__ x, T* __restrict__ r,
                                               T* __restrict__ z, const T* __restrict__ p,
                                               const T* __restrict__ q, const T* __restrict__ dinv,
                                               const PcgScalars* sc, const double* __restrict__ partA, int nA,
                                               double* __restrict__ partB) {
  __shared__ double smem[8];
  // the first entry's loads and the partials' are in flight together, and with the state's
  int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  TX xi = TX(0);
  T pi = T(0), ri = T(0), qi = T(0), di = T(0);
  auto load = [&]() {
    if (i < n) {
      xi = x[i];
      pi = p[i];
      ri = r[i];
      qi = q[i];
      di = dinv[i];
    }
  };
  double pa[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int k = 0; k < 4; ++k)
    if ((int)threadIdx.x + 256 * k < nA) pa[k] = partA[threadIdx.x + 256 * k];
  load();
  if (sc->done) return;
  // nA > 0: every block sums the <p, q> partials itself
  double alpha_d = sc->alpha;
  if (nA > 0) {
    double s = (pa[0] + pa[1]) + (pa[2] + pa[3]);
    for (int k = threadIdx.x + 1024; k < nA; k += 256) s += partA[k];
    alpha_d = sc->rz / block_sum_256(s, smem);
  }
  const T alpha = T(alpha_d);
  T rz = T(0), rr = T(0);
  while (i < n) {
    x[i] = xi + TX(alpha_d) * TX(pi);
    const T rn = ri - alpha * qi;
    const T zi = di * rn;
    r[i] = rn;
    z[i] = zi;
    rz += rn * zi;
    rr += rn * rn;
    i += (int64_t)gridDim.x * blockDim.x;
    load();
  }
  const double s1 = block_sum_256(double(rz), smem);
  const double s2 = block_sum_256(double(rr), smem + 4);
  if (threadIdx.x == 0) {
    partB[blockIdx.x] = s1;
    partB[gridDim.x + blockIdx.x] = s2;
  }
}

// r = (T)(b - y) (y = NULL: r = b); per-block partials of |b - y|^2.
template <typename T>
__global__ __launch_bounds__(256) void k_pcg_resid(int64_t n, const double* __restrict__ b, const double* __restrict__ y,
                                                   T* __restrict__ r, double* __restrict__ part) {
  __shared__ double smem[8];
  double rr = 0;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const double ri = b[i] - (y ? y[i] : 0.0);
    r[i] = T(ri);
    rr += ri * ri;
  }
  const double s = block_sum_256(rr, smem);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

__global__ __launch_bounds__(256) void k_pcg_finish_rr(const double* __restrict__ part, int n, PcgScalars* sc) {
  __shared__ double smem[8];
  const double s = block_reduce_partials(part, n, smem);
  if (threadIdx.x == 0) sc->rr_true = s;
}

// z = D^-1 r and the partials of <r,z>, <r,r> (start or residual replacement).
template <typename T>
__global__ __launch_bounds__(256) void k_pcg_restart(int64_t n, const T* __restrict__ r, T* __restrict__ z,
                                                     const T* __restrict__ dinv, double* __restrict__ partR) {
  __shared__ double smem[8];
  T rz = T(0), rr = T(0);
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const T zi = dinv[i] * r[i];
    z[i] = zi;
    rz += r[i] * zi;
    rr += r[i] * r[i];
  }
  const double s1 = block_sum_256(double(rz), smem);
  const double s2 = block_sum_256(double(rr), smem + 4);
  if (threadIdx.x == 0) {
    partR[blockIdx.x] = s1;
    partR[gridDim.x + blockIdx.x] = s2;
  }
}

// Start (init = 1: beta = 0, counters reset) or residual replacement at
// iteration k (beta keeps the recursion's value; only rz and rr change).
__global__ __launch_bounds__(1024) void k_pcg_rr(const double* __restrict__ partR, int n, PcgScalars* sc, int init,
                                                 int k) {
  __shared__ double smem[16];
  double a0 = 0.0, a1 = 0.0;
  for (int i = threadIdx.x; i < n; i += 1024) {
    a0 += partR[i];
    a1 += partR[n + i];
  }
  const double rz = block_sum<1024>(a0, smem);
  const double rr = block_sum<1024>(a1, smem);
  if (threadIdx.x == 0) {
    sc->rz = rz;
    sc->rr = rr;
    sc->done = 0;
    sc->iter = k;
    sc->ready = 1;
    if (init) {
      sc->beta = 0.0;
      sc->nan = 0;
    }
  }
}

template <typename T>
__global__ void k_fill(int64_t n, T* __restrict__ v, T val) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    v[i] = val;
}

template <typename T>
__global__ void k_pcg_copy(int64_t n, const T* __restrict__ a, T* __restrict__ b) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    b[i] = a[i];
}

constexpr int kVecGrid = 1024;  // blocks of the vector kernels (partials per reduction)
// Largest matrix whose product forms its direction itself (us per iteration, with and without).
// Scalar rows: FP64 37 MB 19.7 / 19.9, 59 MB 28 / 25.6; FP32 39 MB 25.0 / 26.1, 58 MB 33.0 / 32.7.  Blocks in
// FP64: 72 MB 22.5 / 24.2, 139 MB 33.8 / 37.2, 237 MB 52.7 / 55.2 (HEX27 52 / 71), 325 MB 96 / 83; in FP32:
// 45 MB 17.0 / 19.2, 73 MB 23.2 / 24.9, 125 MB 34.4 / 34.2, of long rows 125 MB 39 / 46, 171 MB 50 / 53.
// (3 x 3 blocks.)  2 x 2 blocks, to the largest measured: FP64 28 MB 13.2 / 17.0, 87 MB 24.9 / 27.3, FP32
// 16 MB 12.7 / 16.1, 48 MB 20.2 / 22.6.  4 x 4 blocks: FP64 52 MB 18.8 / 19.2, 104 MB 27.5 / 27.8, 177 MB
// 45.6 / 43.7; FP32 27 MB 14.6 / 14.8, 53 MB 19.0 / 20.8, 90 MB 28.5 / 30.3.
template <int V, typename T>
inline double fuse_bytes(bool longs) {
  if (V == 1 || V > 3) return 45e6;
  return sizeof(T) == 8 ? 240e6 : longs ? 180e6 : 100e6;
}

struct EventPool {
  std::vector<hipEvent_t> e;
  bool ok = true;
  explicit EventPool(int n) : e(n, nullptr) {
    for (auto& x : e)
      if (hipEventCreate(&x) != hipSuccess) ok = false;
  }
  ~EventPool() {
    for (auto& x : e)
      if (x) (void)hipEventDestroy(x);
  }
};

struct Ws {
  void* r;
  void* z;
  void* p;
  void* q;
  void* ones;
  double* y;
  double* partA;
  double* partB;
  double* partR;
  double* partT;
  PcgScalars* sc;
};

static int64_t align256(int64_t b) { return (b + 255) / 256 * 256; }

static int64_t grid_a(const fem_pattern_t* pat) { return pat->num_slices; }

static int64_t ws_layout(const fem_pattern_t* pat, int precision, void* base, Ws* w) {
  const int64_t n = pat->num_rows * pat->vec;
  const int64_t es = precision == FEM_F32 ? 4 : 8;
  int64_t off = 0;
  auto take = [&](int64_t bytes) {
    char* p = base ? reinterpret_cast<char*>(base) + off : nullptr;
    off += align256(bytes);
    return p;
  };
  Ws tmp;
  Ws* o = w ? w : &tmp;
  o->r = take(n * es);
  o->z = take(n * es);
  o->p = take(n * es);
  o->q = take(n * es);
  o->ones = take(n * es);
  o->y = reinterpret_cast<double*>(take(n * 8));
  o->partA = reinterpret_cast<double*>(take(std::max<int64_t>(grid_a(pat), kPatchDotBlocks) * 8));
  o->partB = reinterpret_cast<double*>(take(2 * kVecGrid * 8));
  o->partR = reinterpret_cast<double*>(take(2 * kVecGrid * 8));
  o->partT = reinterpret_cast<double*>(take(kVecGrid * 8));
  o->sc = reinterpret_cast<PcgScalars*>(take(2 * sizeof(PcgScalars)));
  return off;
}

// pop != NULL: the products run matrix-free on it (vals and op are not read).
template <int V, typename T>
static int pcg_run(const fem_pattern_t* pat, const T* vals, const T* dinv_in, const fem_operator_t* op,
                   const fem_patch_operator_t* pop, const double* b, double* x, const fem_pcg_options_t* opt, void* ws_base,
                   PcgScalars* host_sc, fem_pcg_result_t* res, hipStream_t s) {
  constexpr bool kMixed = std::is_same<T, float>::value;
  constexpr bool kDiff = kMixed;  // the FP32 matrix is stored in difference form
  const int64_t n = pat->num_rows * V;
  Ws w;
  ws_layout(pat, kMixed ? FEM_F32 : FEM_F64, ws_base, &w);
  T* r = (T*)w.r;
  T* z = (T*)w.z;
  T* p = (T*)w.p;
  T* q = (T*)w.q;
  const T* dinv = dinv_in;
  if (!opt->precond || !dinv) {
    hipLaunchKernelGGL(k_fill<T>, dim3(256), dim3(256), 0, s, n, (T*)w.ones, T(1));
    FEM_LAUNCHED();
    dinv = (T*)w.ones;
  }
  int gA = (int)grid_a(pat);  // partials of <p, q>
  const int gV = (int)std::min<int64_t>(ceil_div(n, 256), kVecGrid);
  FEM_HIP(hipMemsetAsync(w.sc, 0, 2 * sizeof(PcgScalars), s));
  hipLaunchKernelGGL(k_fill<T>, dim3(256), dim3(256), 0, s, n, p, T(0));
  FEM_LAUNCHED();

  auto read_status = [&]() -> int {
    FEM_HIP(hipMemcpyAsync(host_sc, w.sc, sizeof(PcgScalars), hipMemcpyDeviceToHost, s));
    FEM_HIP(hipStreamSynchronize(s));
    return FEM_OK;
  };
  // r = b - y (y = NULL: r = b), |r|^2 -> rr_true
  auto residual_from = [&](const double* y) -> int {
    hipLaunchKernelGGL(k_pcg_resid<T>, dim3(gV), dim3(256), 0, s, n, b, y, r, w.partT);
    hipLaunchKernelGGL(k_pcg_finish_rr, dim3(1), dim3(256), 0, s, (const double*)w.partT, gV, w.sc);
    FEM_LAUNCHED();
    return read_status();
  };
  auto true_residual = [&]() -> int {
    if (pop) {
      ApplyArgs a{x, w.y, nullptr, nullptr, nullptr, 0.0, 0.0, nullptr, nullptr};
      if (int rc = patch_apply<AP_STORE, double, double>(*pop, a, s)) return rc;
    } else if (kMixed) {
      if (int rc = fem_operator_apply_impl(op, x, w.y, s)) return rc;
    } else {
      if (int rc = fem_spmv(pat, FEM_F64, FEM_FORM_STANDARD, vals, x, w.y, s)) return rc;
    }
    return residual_from(w.y);
  };

  if (int rc = residual_from(nullptr)) return rc;  // |b|^2
  const double bb = host_sc->rr_true;
  const double tol2 = std::max(opt->rtol * opt->rtol * bb, opt->atol * opt->atol);
  res->b_norm = std::sqrt(bb);
  res->iterations = 0;
  res->replacements = 0;
  res->status = FEM_OK;
  res->timed_launches = 0;
  res->spmv_ms = res->update_ms = 0.0;

  if (int rc = true_residual()) return rc;
  double rr_true = host_sc->rr_true;
  if (!std::isfinite(rr_true)) {
    res->status = FEM_ERR_NAN;
    res->res_norm = rr_true;
    return FEM_OK;
  }
  if (rr_true <= tol2) {
    res->res_norm = std::sqrt(rr_true);
    return FEM_OK;
  }
  hipLaunchKernelGGL(k_pcg_restart<T>, dim3(gV), dim3(256), 0, s, n, (const T*)r, z, dinv, w.partR);
  hipLaunchKernelGGL(k_pcg_rr, dim3(1), dim3(1024), 0, s, (const double*)w.partR, gV, w.sc, 1, 0);
  FEM_LAUNCHED();
  double rr_ref = rr_true;
  const int check = std::max(1, opt->check_every);
  // Small matrices leave most of the chip idle at one workgroup of W waves per slice: up to 256
  // slices (one per CU) 16 waves share a slice's slots, up to 768 eight (FP64 Poisson of 13,824
  // cells 15.3 -> 12.0 us per iteration, of 32,768 cells 16.0 -> 14.9).  FP32 blocks leave room for two
  // workgroups of eight waves on a CU: eight waves only up to 512 slices (562 slices: 25 us, with four
  // 16.3) unless the direction has its own kernel.  FP64 blocks keep eight at any size (139 MB: 33.8 us,
  // with two 37.7).
  // The direction update runs inside the product (which then gathers z and the old direction) where
  // the matrix stays in the caches or is not read; the new direction goes to a second buffer.  That is
  // y's, free between the true residuals: so a batch of status-free iterations has to be even.
  T* p2 = (T*)w.y;
  const double sell_bytes = double(pat->sell_blocks) * (V * V * sizeof(T) + 4);
  const bool fused = check % 2 == 0 && (pop ? true : sell_bytes <= fuse_bytes<V, T>(long_rows(*pat)));
  const bool eight = long_rows(*pat) || (V == 1 ? fused && gA <= 768 : !fused || gA <= 512 || sizeof(T) == 8);
  // one workgroup for the whole batch: few scalar rows of, on average, at most kOneSlots slots (a timed
  // solve takes the launches that its events can stand between)
  const bool one = V == 1 && !pop && !opt->timing && pat->num_slices <= kOneSlices &&
                   pat->sell_blocks <= pat->num_slices * kSlice * kOneSlots;
  const double delta2 = kMixed ? opt->reliable_delta * opt->reliable_delta : 0.0;
  EventPool ev(opt->timing ? 4 * check : 0);
  if (!ev.ok) {
    set_error("fem_pcg_solve: hipEventCreate failed");
    return FEM_ERR_HIP;
  }
  double spmv_ms = 0.0, upd_ms = 0.0;
  int timed = 0;
  int iter = 0;
  for (;;) {
    const int iter0 = iter;
    T* pc = p;  // the current direction
    if constexpr (V == 1)
      if (one) {
        hipLaunchKernelGGL((k_pcg_one<kDiff, T>), dim3(1), dim3(64 * kOneWaves), 0, s, *pat, vals, x, r, z, p, dinv,
                           PcgHead{w.sc, w.sc, w.partB, 0, tol2, opt->maxiter}, check);
        FEM_LAUNCHED();
      }
    for (int m = 0; m < (one ? 0 : check); ++m) {
      PcgScalars* sc = w.sc + 1 - (m & 1);  // the state of this iteration
      const PcgHead head{w.sc + (m & 1), sc, w.partB, gV, tol2, opt->maxiter};
      T* pn = fused ? (pc == p ? p2 : p) : p;
      if (opt->timing) FEM_HIP(hipEventRecord(ev.e[4 * m], s));
      if (!fused) hipLaunchKernelGGL(k_pcg_p<T>, dim3(gV), dim3(256), 0, s, n, (const T*)z, p, head);
      if (opt->timing) FEM_HIP(hipEventRecord(ev.e[4 * m + 1], s));
      if (pop && fused) {
        if (int rc = patch_pcg_product<PcgHead, T>(*pop, head, z, pc, pn, q, w.partA, s, &gA)) return rc;
      } else if (pop) {
        ApplyArgsT<T, T> a{p, q, nullptr, nullptr, nullptr, 0.0, 0.0, w.partA, &sc->done};
        if (int rc = patch_apply<AP_PQ, T, T>(*pop, a, s, &gA)) return rc;
      } else {
        auto product = [&](auto fuse, auto waves) {
          constexpr int W = decltype(waves)::value;
          hipLaunchKernelGGL((k_pcg_a<V, kDiff, T, decltype(fuse)::value, W>), dim3(gA), dim3(64 * W), 0, s, *pat, vals,
                             (const T*)pc, (const T*)z, pn, q, (const PcgScalars*)sc, head, w.partA, opt->xcd_remap);
        };
        using Few = std::integral_constant<int, 16>;
        using Some = std::integral_constant<int, 8>;
        using Many = std::integral_constant<int, SliceCfg<T>::W>;
        // (blocks always take eight waves in FP64 and where the direction has its own kernel)
        constexpr bool kManyFused = V == 1 || sizeof(T) == 4, kMany = V == 1;
        if (fused && gA <= 256)
          product(std::true_type{}, Few{});
        else if (fused && (eight || !kManyFused))
          product(std::true_type{}, Some{});
        else if (!fused && (eight || !kMany))
          product(std::false_type{}, Some{});
        else if (fused) {
          if constexpr (kManyFused) product(std::true_type{}, Many{});
        } else {
          if constexpr (kMany) product(std::false_type{}, Many{});
        }
      }
      if (opt->timing) FEM_HIP(hipEventRecord(ev.e[4 * m + 2], s));
      const int sumA = gA <= kSumParts ? gA : 0;
      if (!sumA) hipLaunchKernelGGL(k_pcg_ra, dim3(1), dim3(1024), 0, s, (const double*)w.partA, gA, sc);
      hipLaunchKernelGGL((k_pcg_b<T, double>), dim3(gV), dim3(256), 0, s, n, x, r, z, (const T*)pn, (const T*)q, dinv,
                         (const PcgScalars*)sc, (const double*)w.partA, sumA, w.partB);
      if (opt->timing) FEM_HIP(hipEventRecord(ev.e[4 * m + 3], s));
      pc = pn;
    }
    if (!one) {
      hipLaunchKernelGGL(k_pcg_rb, dim3(1), dim3(1024), 0, s,
                         PcgHead{w.sc + (check & 1), w.sc, w.partB, gV, tol2, opt->maxiter});
      FEM_LAUNCHED();
    }
    if (int rc = read_status()) return rc;
    iter = host_sc->iter;
    // the last direction of a batch that ended inside: back from the shared buffer
    if (fused && !one && ((iter - iter0) & 1)) {
      hipLaunchKernelGGL(k_pcg_copy<T>, dim3(gV), dim3(256), 0, s, n, (const T*)p2, p);
      FEM_LAUNCHED();
    }
    if (opt->timing) {
      // only the launches that ran an iteration (the rest returned on `done`)
      for (int m = 0; m < std::min(check, iter - iter0); ++m) {
        float t0 = 0.f, t1 = 0.f, t2 = 0.f;
        FEM_HIP(hipEventElapsedTime(&t0, ev.e[4 * m], ev.e[4 * m + 1]));
        FEM_HIP(hipEventElapsedTime(&t1, ev.e[4 * m + 1], ev.e[4 * m + 2]));
        FEM_HIP(hipEventElapsedTime(&t2, ev.e[4 * m + 2], ev.e[4 * m + 3]));
        spmv_ms += t1;
        upd_ms += t0 + t2;
        ++timed;
      }
    }
    if (host_sc->nan) {
      res->status = FEM_ERR_NAN;
      break;
    }
    const bool conv_rec = host_sc->done && host_sc->rr <= tol2;
    const bool trigger = kMixed && !host_sc->done && host_sc->rr < delta2 * rr_ref;
    if (conv_rec || trigger) {
      if (int rc = true_residual()) return rc;
      rr_true = host_sc->rr_true;
      if (rr_true <= tol2) break;
      if (!std::isfinite(rr_true)) {
        res->status = FEM_ERR_NAN;
        break;
      }
      if (iter >= opt->maxiter) {
        res->status = FEM_ERR_NOT_CONVERGED;
        break;
      }
      // residual replacement at iteration `iter`: keep the search direction
      hipLaunchKernelGGL(k_pcg_restart<T>, dim3(gV), dim3(256), 0, s, n, (const T*)r, z, dinv, w.partR);
      hipLaunchKernelGGL(k_pcg_rr, dim3(1), dim3(1024), 0, s, (const double*)w.partR, gV, w.sc, 0, iter);
      FEM_LAUNCHED();
      rr_ref = rr_true;
      res->replacements += 1;
      continue;
    }
    if (host_sc->done || iter >= opt->maxiter) {  // maxiter reached
      res->status = FEM_ERR_NOT_CONVERGED;
      break;
    }
  }
  if (!(rr_true <= tol2) || res->status != FEM_OK) {
    if (int rc = true_residual()) return rc;
    rr_true = host_sc->rr_true;
  }
  res->iterations = iter;
  res->res_norm = std::sqrt(rr_true);
  res->timed_launches = timed;
  res->spmv_ms = timed ? spmv_ms / timed : 0.0;
  res->update_ms = timed ? upd_ms / timed : 0.0;
  return FEM_OK;
}

// ------------------------------------------------- no-allocation variant
// The workspace of fem_pcg_solve_noalloc: a library-held device array, one
// copy per GPU (each device that loads this code object holds it until the
// process ends).  Host code never passes `scratch` itself to a kernel: its
// device address comes from hipGetSymbolAddress, looked up once per device.
static __device__ __align__(256) unsigned char scratch[FEM_PCG_NOALLOC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static void* g_scratch_ptr[kMaxDevices] = {};

// Device address of the current device's scratch array.
static int scratch_address(void** out) {
  int dev = -1;
  FEM_HIP(hipGetDevice(&dev));
  FEM_CHECK_ARG(dev >= 0 && dev < kMaxDevices, "fem_pcg_solve_noalloc: device %d out of range", dev);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    FEM_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    FEM_CHECK_ARG(p != nullptr, "fem_pcg_solve_noalloc: no device address for the scratch array");
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return FEM_OK;
}

}  // namespace fem

using namespace fem;

extern "C" {

int64_t fem_pcg_ws_bytes(const fem_pattern_t* pat, int32_t precision) {
  if (!pat || pat->num_rows <= 0) return -1;
  return ws_layout(pat, precision, nullptr, nullptr) + 256;
}

static int pcg_dispatch(const fem_pattern_t* pat, const void* vals, const void* dinv, const fem_operator_t* op,
                        const fem_patch_operator_t* pop, const double* b, double* x, const fem_pcg_options_t* opt,
                        void* ws, void* host_status, fem_pcg_result_t* result, void* stream) {
  hipStream_t s = as_stream(stream);
  PcgScalars* hsc = reinterpret_cast<PcgScalars*>(host_status);
  auto run = [&](auto vc) -> int {
    constexpr int V = decltype(vc)::value;
    if (opt->precision == FEM_F32)
      return pcg_run<V, float>(pat, (const float*)vals, (const float*)dinv, op, pop, b, x, opt, ws, hsc, result, s);
    return pcg_run<V, double>(pat, (const double*)vals, (const double*)dinv, op, pop, b, x, opt, ws, hsc, result, s);
  };
  switch (pat->vec) {
    case 1: return run(std::integral_constant<int, 1>{});
    case 2: return run(std::integral_constant<int, 2>{});
    case 3: return run(std::integral_constant<int, 3>{});
    case 4: return run(std::integral_constant<int, 4>{});
    default: break;
  }
  set_error("fem_pcg_solve: unsupported vec %d", pat->vec);
  return FEM_ERR_BAD_ARG;
}

int fem_pcg_solve(const fem_pattern_t* pat, const void* vals, const void* dinv, const fem_operator_t* op,
                  const double* b, double* x, const fem_pcg_options_t* opt, void* ws, void* host_status,
                  fem_pcg_result_t* result, void* stream) {
  FEM_CHECK_ARG(pat && pat->slice_ptr && pat->sell_col && pat->sell_row && pat->sell_pos && pat->num_rows > 0,
                "fem_pcg_solve: bad pattern");
  FEM_CHECK_ARG(vals && b && x && opt && ws && host_status && result, "fem_pcg_solve: NULL argument");
  FEM_CHECK_ARG(opt->precision == FEM_F32 || opt->precision == FEM_F64, "fem_pcg_solve: bad precision");
  FEM_CHECK_ARG(opt->precision == FEM_F64 || op, "fem_pcg_solve: FP32 mode needs the FP64 operator");
  FEM_CHECK_ARG(opt->maxiter > 0 && opt->rtol >= 0 && opt->atol >= 0, "fem_pcg_solve: bad tolerances");
  FEM_CHECK_ARG(!opt->precond || dinv, "fem_pcg_solve: Jacobi requested without dinv");
  return pcg_dispatch(pat, vals, dinv, op, nullptr, b, x, opt, ws, host_status, result, stream);
}

int fem_pcg_solve_patch(const fem_pattern_t* pat, const fem_patch_operator_t* op, const void* dinv, const double* b,
                        double* x, const fem_pcg_options_t* opt, void* ws, void* host_status,
                        fem_pcg_result_t* result, void* stream) {
  FEM_CHECK_ARG(pat && pat->num_rows > 0 && b && x && opt && ws && host_status && result,
                "fem_pcg_solve_patch: NULL argument");
  FEM_CHECK_ARG(patch_operator_ok(op), "fem_pcg_solve_patch: the operator is incomplete or not covered");
  FEM_CHECK_ARG(op->mesh->num_nodes == pat->num_rows && op->mesh->vec == pat->vec,
                "fem_pcg_solve_patch: operator and pattern disagree");
  FEM_CHECK_ARG(opt->precision == FEM_F32 || opt->precision == FEM_F64, "fem_pcg_solve_patch: bad precision");
  FEM_CHECK_ARG(opt->maxiter > 0 && opt->rtol >= 0 && opt->atol >= 0, "fem_pcg_solve_patch: bad tolerances");
  FEM_CHECK_ARG(!opt->precond || dinv, "fem_pcg_solve_patch: Jacobi requested without dinv");
  return pcg_dispatch(pat, nullptr, dinv, nullptr, op, b, x, opt, ws, host_status, result, stream);
}

int fem_pcg_solve_noalloc(const fem_pattern_t* pat, const void* vals, const void* dinv, const fem_operator_t* op,
                          const double* b, double* x, const fem_pcg_options_t* opt, void* host_status,
                          fem_pcg_result_t* result, void* stream) {
  FEM_CHECK_ARG(pat && opt, "fem_pcg_solve_noalloc: NULL argument");
  FEM_CHECK_ARG(opt->timing == 0, "fem_pcg_solve_noalloc: timing=1 creates HIP events; use fem_pcg_solve");
  const int64_t need = fem_pcg_ws_bytes(pat, opt->precision);
  FEM_CHECK_ARG(need > 0, "fem_pcg_solve_noalloc: bad pattern");
  if (need > (int64_t)FEM_PCG_NOALLOC_SCRATCH_BYTES) {
    set_error("fem_pcg_solve_noalloc: the system needs %lld workspace bytes, more than the %lld-byte scratch "
              "(%lld rows of %d); use fem_pcg_solve with a caller workspace",
              (long long)need, (long long)FEM_PCG_NOALLOC_SCRATCH_BYTES, (long long)pat->num_rows, pat->vec);
    return FEM_ERR_CAPACITY;
  }
  void* ws = nullptr;
  if (int rc = scratch_address(&ws)) return rc;
  // every workspace entry the solve reads is written by it first (scalars and p are
  // cleared at its start), so the previous call's contents do not matter
  return fem_pcg_solve(pat, vals, dinv, op, b, x, opt, ws, host_status, result, stream);
}

}  // extern "C"
