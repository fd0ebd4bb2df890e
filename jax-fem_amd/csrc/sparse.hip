// Global matrix and vector kernels over the SELL-64 block layout.
//
// Replaces jax-fem's host-side global assembly and BC handling:
//   problem.py:426-437  scatter-add of cell residuals into nodal residuals
//   solver.py:522-529   PETSc setValuesCOO (sum duplicates) + zeroRows(diag=1)
//   solver.py:290-304   apply_bc_vec (residual rows of Dirichlet dofs)
//   solver.py:65-68     CSR export / Jacobi diagonal of jax_solve
// All sums run in a fixed order (cells ascending), so results are
// bit-reproducible run to run.
#include "fem_common.hpp"

#include <algorithm>
#include <type_traits>

namespace fem {

// ------------------------------------------------------- nodal gather
// V is a template parameter so the per-node sums stay in registers; the
// incident entries are visited two at a time to keep two gathers in flight.
template <int V>
__global__ __launch_bounds__(256) void k_gather_nodal(int64_t num_nodes, const int32_t* __restrict__ inc_ptr,
                                                      const int32_t* __restrict__ inc_idx,
                                                      const double* __restrict__ ent, const double* base,
                                                      double* out) {
  for (int64_t n = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; n < num_nodes;
       n += (int64_t)gridDim.x * blockDim.x) {
    const int b = inc_ptr[n], e = inc_ptr[n + 1];
    double acc[V], acc2[V];
#pragma unroll
    for (int i = 0; i < V; ++i) acc[i] = acc2[i] = 0.0;
    int t = b;
    for (; t + 1 < e; t += 2) {
      const double* p0 = ent + (int64_t)inc_idx[t] * V;
      const double* p1 = ent + (int64_t)inc_idx[t + 1] * V;
#pragma unroll
      for (int i = 0; i < V; ++i) {
        acc[i] += p0[i];
        acc2[i] += p1[i];
      }
    }
    if (t < e) {
      const double* p0 = ent + (int64_t)inc_idx[t] * V;
#pragma unroll
      for (int i = 0; i < V; ++i) acc[i] += p0[i];
    }
#pragma unroll
    for (int i = 0; i < V; ++i) out[n * V + i] = (base ? base[n * V + i] : 0.0) + (acc[i] + acc2[i]);
  }
}

// ------------------------------------------------------- matrix values
// One workgroup per slice, lane = row: for every SELL slot k, sum the cell blocks that land in
// block (row, col_k) and store them (zeros in padding slots).  Wave w takes the slots
// [w K, (w + 1) K), K = slots / waves rounded up, so the lists a lane reads stay contiguous (they
// are read through windows).  DIFF stores the row-sum block R_row = sum_k A(row, k) (accumulated
// in TS, the waves' sums added in their order) in the diagonal slot instead of the diagonal block
// (difference form of the SpMV).  dinv (may be NULL) receives 1 / A(row*V+c, row*V+c).
// Bound by the blocks' addresses (every lane reads 72 bytes of its own: five wide loads where
// element loads are nine); one thread per row walked a dependent chain of up to 125 slots on 1840
// waves in all: 24^3 HEX27 cells 800 -> 630 us (4 and 16 waves per slice: 650 and 690).
constexpr int kGatherWaves = 8;

template <int VV, typename TS>
__device__ inline void add_block(const TS* __restrict__ src, TS (&acc)[VV]) {
  // two values a load; a block is aligned to one value
  typedef TS Pair __attribute__((ext_vector_type(2), aligned(alignof(TS))));
#pragma unroll
  for (int v = 0; v + 1 < VV; v += 2) {
    const Pair p = *reinterpret_cast<const Pair*>(src + v);
    acc[v] += p.x;
    acc[v + 1] += p.y;
  }
  if (VV & 1) acc[VV - 1] += src[VV - 1];
}

template <int V, bool DIFF, typename TS, typename T>
__global__ __launch_bounds__(64 * kGatherWaves) void k_gather_matrix(fem_pattern_t pat, const TS* __restrict__ Ke,
                                                                     T* __restrict__ vals, T* __restrict__ dinv) {
  constexpr int VV = V * V;
  __shared__ double s_sum[DIFF ? kGatherWaves : 1][DIFF ? VV : 1][DIFF ? kSlice : 1];
  const int64_t s = blockIdx.x;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int base = pat.slice_ptr[s];
  const int L = (pat.slice_ptr[s + 1] - base) >> 6;
  const int row = pat.sell_row[s * kSlice + lane];
  const bool real = row >= 0;
  const int rb = real ? pat.row_ptr[row] : 0;
  const int len = real ? pat.row_ptr[row + 1] - rb : 0;
  const int ds = real ? pat.diag_slot[row] : -1;
  T* vp = vals + (size_t)base * VV + lane;
  // (FP64 whatever the tangents' type: rounded row sums let CG stagnate, 64x32x32 cantilever)
  double rsum[VV];
#pragma unroll
  for (int v = 0; v < VV; ++v) rsum[v] = 0.;
  ListWindow<4> cptr(pat.contrib_ptr, pat.nnzb + 1);
  ListWindow<8> cidx(pat.contrib_idx, (int64_t)pat.num_cells * pat.nodes_per_cell * pat.nodes_per_cell);
  const int K = (L + kGatherWaves - 1) / kGatherWaves, k0 = w * K, k1 = min(L, k0 + K);
  int c1 = k0 < len ? cptr[rb + k0] : 0;
  for (int k = k0; k < k1; ++k) {
    TS acc[VV];
#pragma unroll
    for (int v = 0; v < VV; ++v) acc[v] = TS(0);
    if (k < len) {
      const int c0 = c1;
      c1 = cptr[rb + k + 1];
      for (int ci = c0; ci < c1; ++ci) add_block<VV>(Ke + (size_t)cidx[ci] * VV, acc);
    }
    if (DIFF)
#pragma unroll
      for (int v = 0; v < VV; ++v) rsum[v] += acc[v];
    if (k == ds && dinv) {
#pragma unroll
      for (int c = 0; c < V; ++c) {
        const TS d = acc[c * V + c];
        dinv[(int64_t)row * V + c] = d != TS(0) ? T(TS(1) / d) : T(0);
      }
    }
    if (!(DIFF && k == ds)) {
#pragma unroll
      for (int v = 0; v < VV; ++v) __builtin_nontemporal_store(T(acc[v]), &vp[((size_t)k * VV + v) * kSlice]);
    }
  }
  if (w == 0 && real && ds < 0 && dinv) {  // a node of no cell
#pragma unroll
    for (int c = 0; c < V; ++c) dinv[(int64_t)row * V + c] = T(0);
  }
  if (DIFF) {
#pragma unroll
    for (int v = 0; v < VV; ++v) s_sum[w][v][lane] = rsum[v];
    __syncthreads();
    if (ds >= 0)
      for (int v = w; v < VV; v += kGatherWaves) {
        double t = s_sum[0][v][lane];
#pragma unroll
        for (int o = 1; o < kGatherWaves; ++o) t += s_sum[o][v][lane];
        vp[((size_t)ds * VV + v) * kSlice] = T(t);
      }
  }
}

// The same sums for cells of 27 nodes: the 27 blocks of a (cell, row node) pair are one run of 1944
// bytes (FP64), which the slot-by-slot gather above reads 72 bytes at a time at moments far apart.
// A wave takes a row: it lists the row's pairs (the diagonal slot's contributions) and the slot of
// each of their blocks, then adds run after run, lane-contiguous, to the row's slots in LDS; the
// workgroup's eight rows are stored together (64-byte segments).  Sums run over the cells in
// ascending order, as above.  Rows of more than kRowSlots slots are done in windows; rows of more
// than kRowPairs pairs, and rows of a cell that names a node twice (two lanes of one run on one
// slot: their order would be the hardware's), slot by slot, into the same LDS.
// The adds are LDS atomics in FP64 (one instruction; loads, adds and stores 416 us instead of 405 in
// the same run) and plain ones in FP32, whose atomics are the slower ones (777 us; plain 400).
// 24^3 cells: 610 -> 365 us (1.29 GB, 250 us at the copy rate), from FP32 tangents 553 -> 400; with two
// rows to a wave 525: what is left is the chain row -> lists -> runs, which 16 waves on a CU (the LDS's
// limit) do not cover.
constexpr int kRowSlots = 128, kRowPairs = 16, kRowWaves = 8, kRowsPerGroup = 8;

template <int V, int N, bool DIFF, typename TS, typename T>
__global__ __launch_bounds__(64 * kRowWaves) void k_gather_rows(fem_pattern_t pat, const TS* __restrict__ Ke,
                                                                T* __restrict__ vals, T* __restrict__ dinv) {
  constexpr int VV = V * V, RUN = N * VV, PER = (RUN + 63) / 64, STRIDE = kRowSlots * VV + 1;
  constexpr bool kPlainAdds = sizeof(TS) == 4;
  __shared__ TS s_acc[kRowsPerGroup][STRIDE];
  __shared__ uint8_t s_slot[kRowWaves][kRowPairs][N + 1];
  __shared__ uint8_t s_first[kRowWaves][kRowPairs * N + 64];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t s = blockIdx.x / (kSlice / kRowsPerGroup);
  const int l0 = (blockIdx.x % (kSlice / kRowsPerGroup)) * kRowsPerGroup;
  const int base = pat.slice_ptr[s], L = (pat.slice_ptr[s + 1] - base) >> 6;
  T* vp = vals + (size_t)base * VV + l0;
  constexpr int RPW = kRowsPerGroup / kRowWaves;
  double rsum[RPW][VV];
#pragma unroll
  for (int r = 0; r < RPW; ++r)
#pragma unroll
    for (int v = 0; v < VV; ++v) rsum[r][v] = 0.;
  for (int k0 = 0; k0 < L; k0 += kRowSlots) {
    const int kn = min(kRowSlots, L - k0);
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
      const int rl = w + r * kRowWaves;
      TS* acc = s_acc[rl];
      for (int i = lane; i < kn * VV; i += 64) acc[i] = TS(0);
      const int row = pat.sell_row[s * kSlice + l0 + rl];
      if (row < 0) continue;
      const int rb = pat.row_ptr[row], len = pat.row_ptr[row + 1] - rb, ds = pat.diag_slot[row];
      if (k0 > 0 && len <= k0) continue;  // only padding in this window
      const int d0 = ds >= 0 ? pat.contrib_ptr[rb + ds] : 0;
      const int n = ds >= 0 ? pat.contrib_ptr[rb + ds + 1] - d0 : 0;
      const int t0 = pat.contrib_ptr[rb], t1 = pat.contrib_ptr[rb + len];
      bool listed = len <= kRowSlots && n <= kRowPairs && t1 - t0 == n * N;
      int first = 0;
      if (listed) {
        // first block of each pair (the diagonal's contribution is its block a)
        if (lane < n) {
          const int32_t e = pat.contrib_idx[d0 + lane];
          first = e - e % N;
        }
        for (int i = lane; i < n * N; i += 64) s_first[w][i] = 0;
        wave_fence();
        for (int k = lane; k < len; k += 64) s_first[w][pat.contrib_ptr[rb + k] - t0] = 1;
        wave_fence();
        bool twice = false;
        int slots = 0;  // slots that begin before the 64 contributions at hand
        int last = -1;  // pair of the contribution before them
        for (int i = lane; i - lane < n * N; i += 64) {
          const bool in = i < n * N;
          const unsigned long long begins = __ballot(in && s_first[w][i]);
          const int slot = slots + __popcll(begins & (~0ull >> (63 - lane))) - 1;
          slots += __popcll(begins);
          const int e = in ? pat.contrib_idx[t0 + i] : -1;
          int pair = -1;
          for (int p = 0; p < n; ++p) {
            const int b = e - __shfl(first, p, 64);
            if (in && b >= 0 && b < N) {
              s_slot[w][p][b] = (uint8_t)slot;
              pair = p;
            }
          }
          // (a slot's contributions are in ascending order: a pair's two blocks of it are neighbours)
          const int up = __shfl_up(pair, 1, 64);
          twice |= in && !(begins >> lane & 1) && pair == (lane ? up : last);
          last = __shfl(pair, 63, 64);
        }
        wave_fence();
        listed = !__any(twice);
      }
      if (listed) {
        for (int p = 0; p < n; p += 4) {
          TS x[4][PER];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const TS* src = Ke + (size_t)__shfl(first, min(p + j, n - 1), 64) * VV;
#pragma unroll
            for (int i = 0; i < PER; ++i) x[j][i] = p + j < n && lane + 64 * i < RUN ? src[lane + 64 * i] : TS(0);
          }
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            if (p + j >= n) break;
            if constexpr (kPlainAdds) {
              int at[PER];
              TS y[PER];
#pragma unroll
              for (int i = 0; i < PER; ++i) {
                const int o = min(lane + 64 * i, RUN - 1);
                at[i] = s_slot[w][p + j][o / VV] * VV + o % VV;
                y[i] = acc[at[i]];
              }
#pragma unroll
              for (int i = 0; i < PER; ++i)
                if (lane + 64 * i < RUN) acc[at[i]] = y[i] + x[j][i];
              wave_fence();
            } else {
#pragma unroll
              for (int i = 0; i < PER; ++i) {
                const int o = lane + 64 * i;
                if (o < RUN) atomicAdd(&acc[s_slot[w][p + j][o / VV] * VV + o % VV], x[j][i]);
              }
            }
          }
        }
      } else {
        for (int k = lane; k < kn; k += 64) {
          TS a[VV];
#pragma unroll
          for (int v = 0; v < VV; ++v) a[v] = TS(0);
          if (k0 + k < len)
            for (int ci = pat.contrib_ptr[rb + k0 + k]; ci < pat.contrib_ptr[rb + k0 + k + 1]; ++ci)
              add_block<VV>(Ke + (size_t)pat.contrib_idx[ci] * VV, a);
#pragma unroll
          for (int v = 0; v < VV; ++v) acc[k * VV + v] = a[v];
        }
      }
      wave_fence();
      if (DIFF)
        for (int k = lane; k < kn; k += 64)
#pragma unroll
          for (int v = 0; v < VV; ++v) rsum[r][v] += acc[k * VV + v];
      if (dinv && lane < V && k0 == (ds >= 0 ? ds / kRowSlots * kRowSlots : 0)) {
        const TS d = ds >= 0 ? acc[(ds - k0) * VV + lane * (V + 1)] : TS(0);  // 0: a node of no cell
        dinv[(int64_t)row * V + lane] = d != TS(0) ? T(TS(1) / d) : T(0);
      }
    }
    __syncthreads();
    const int rl = threadIdx.x % kRowsPerGroup;
    const int row = pat.sell_row[s * kSlice + l0 + rl];
    const int ds = DIFF && row >= 0 ? pat.diag_slot[row] : -1;
    for (int k = threadIdx.x / kRowsPerGroup; k < kn; k += 64 * kRowWaves / kRowsPerGroup)
      if (!DIFF || k0 + k != ds)
#pragma unroll
        for (int v = 0; v < VV; ++v)
          __builtin_nontemporal_store(T(s_acc[rl][k * VV + v]), &vp[((size_t)(k0 + k) * VV + v) * kSlice + rl]);
    __syncthreads();
  }
  if (DIFF)
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
      const int rl = w + r * kRowWaves;
      const int row = pat.sell_row[s * kSlice + l0 + rl];
      const int ds = row >= 0 ? pat.diag_slot[row] : -1;
#pragma unroll
      for (int v = 0; v < VV; ++v) {
        const double t = wave_sum(rsum[r][v]);
        if (ds >= 0 && lane == 0) vp[((size_t)ds * VV + v) * kSlice + rl] = T(t);
      }
    }
}

// Zero row d of the matrix and put 1 on its diagonal (PETSc zeroRows, diag = 1).
// The row of an identity row sums to e_d, so the same values serve both
// forms; dinv[d] = 1.
template <int V, typename T>
__global__ void k_bc_rows(fem_pattern_t pat, T* __restrict__ vals, int64_t n_bc, const int32_t* __restrict__ dofs,
                          T* __restrict__ dinv) {
  constexpr int VV = V * V;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n_bc; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t d = dofs[i];
    const int64_t row = d / V;
    const int ci = (int)(d % V);
    const int64_t pos = pat.sell_pos[row];
    const int64_t s = pos >> 6;
    const int lane = (int)(pos & 63);
    const int base = pat.slice_ptr[s];
    const int L = (pat.slice_ptr[s + 1] - base) >> 6;
    T* vp = vals + (size_t)base * VV + lane;
    for (int k = 0; k < L; ++k)
#pragma unroll
      for (int cj = 0; cj < V; ++cj) vp[((size_t)k * VV + ci * V + cj) * kSlice] = T(0);
    const int ds = pat.diag_slot[row];
    if (ds >= 0) vp[((size_t)ds * VV + ci * V + ci) * kSlice] = T(1);
    if (dinv) dinv[d] = T(1);
  }
}

template <int V, typename T>
__global__ void k_jacobi(fem_pattern_t pat, const T* __restrict__ vals, T* __restrict__ dinv) {
  constexpr int VV = V * V;
  for (int64_t row = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; row < pat.num_rows;
       row += (int64_t)gridDim.x * blockDim.x) {
    const int64_t pos = pat.sell_pos[row];
    const int64_t s = pos >> 6;
    const int lane = (int)(pos & 63);
    const int base = pat.slice_ptr[s];
    const T* vp = vals + (size_t)base * VV + lane;
    const int ds = pat.diag_slot[row];
#pragma unroll
    for (int c = 0; c < V; ++c) {
      const T d = ds >= 0 ? vp[((size_t)ds * VV + c * V + c) * kSlice] : T(0);
      dinv[row * V + c] = d != T(0) ? T(1) / d : T(0);
    }
  }
}

__global__ void k_residual_bc(int64_t n_bc, const int32_t* __restrict__ dofs, const double* __restrict__ g,
                              const double* __restrict__ u, double* __restrict__ res, double scale) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n_bc; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t d = dofs[i];
    res[d] = u[d] - g[i] * scale;
  }
}

// ------------------------------------------------------------ SpMV
// One block per slice; the W waves split the slots and wave 0 combines them.
template <int V, bool DIFF, typename T, int W>
__global__ __launch_bounds__(64 * W) void k_spmv(fem_pattern_t pat, const T* __restrict__ vals,
                                                 const T* __restrict__ x, T* __restrict__ y) {
  constexpr int U = SliceCfg<T>::U;
  __shared__ double red[W][kSlice][V];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t s = blockIdx.x;
  const int64_t row = pat.sell_row[s * kSlice + lane];
  const bool real = row >= 0;
  auto xat = [&](int64_t c, T (&xc)[V]) {
#pragma unroll
    for (int j = 0; j < V; ++j) xc[j] = x[c * V + j];
  };
  T xt[V];
  xat(real ? row : 0, xt);
  double xr[V], acc[V];
#pragma unroll
  for (int j = 0; j < V; ++j) xr[j] = double(xt[j]);
  sell_slice_partial<V, DIFF, W, U, T>(pat, vals, s, w, lane, row, xat, xr, acc);
  if (w > 0) {
#pragma unroll
    for (int i = 0; i < V; ++i) red[w][lane][i] = acc[i];
  }
  __syncthreads();
  if (w == 0 && real) {
#pragma unroll
    for (int i = 0; i < V; ++i) {
      double t = acc[i];
#pragma unroll
      for (int o = 1; o < W; ++o) t += red[o][lane][i];
      y[row * V + i] = T(t);
    }
  }
}

// Scalar CSR of the block matrix: row r = V*node + ci holds the blocks of node
// row `node` in column order, each contributing V consecutive columns.  In
// difference form the diagonal block is recovered as R - sum of the others
// (in FP64).
template <int V, typename T>
__global__ void k_export_csr(fem_pattern_t pat, const T* __restrict__ vals, int form, int32_t* __restrict__ indptr,
                             int32_t* __restrict__ indices, double* __restrict__ data) {
  constexpr int VV = V * V;
  for (int64_t row = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; row < pat.num_rows;
       row += (int64_t)gridDim.x * blockDim.x) {
    const int rb = pat.row_ptr[row];
    const int len = pat.row_ptr[row + 1] - rb;
    const int ds = pat.diag_slot[row];
    const int64_t pos = pat.sell_pos[row];
    const int64_t s = pos >> 6;
    const int lane = (int)(pos & 63);
    const T* vp = vals + (size_t)pat.slice_ptr[s] * VV + lane;
    for (int ci = 0; ci < V; ++ci) {
      const int64_t start = (int64_t)VV * rb + (int64_t)ci * V * len;
      if (indptr) indptr[row * V + ci] = (int32_t)start;
      for (int k = 0; k < len; ++k)
        for (int cj = 0; cj < V; ++cj) {
          const int64_t pos = start + (int64_t)k * V + cj;
          if (indices) indices[pos] = pat.col_idx[rb + k] * V + cj;
          if (data && vals) {
            double v = double(vp[((size_t)k * VV + ci * V + cj) * kSlice]);
            if (form == FEM_FORM_DIFFERENCE && k == ds)
              for (int kk = 0; kk < len; ++kk)
                if (kk != ds) v -= double(vp[((size_t)kk * VV + ci * V + cj) * kSlice]);
            data[pos] = v;
          }
        }
    }
    if (indptr && row == pat.num_rows - 1) indptr[pat.num_rows * V] = (int32_t)((int64_t)VV * pat.row_ptr[pat.num_rows]);
  }
}

// ------------------------------------------------------- small vector ops
__global__ void k_copy_bc(int64_t n_bc, const int32_t* __restrict__ dofs, const double* __restrict__ x,
                          double* __restrict__ y) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n_bc; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t d = dofs[i];
    y[d] = x[d];
  }
}

__global__ __launch_bounds__(256) void k_dot(int64_t n, const double* __restrict__ x, const double* __restrict__ y,
                                             double* __restrict__ partials) {
  __shared__ double smem[8];
  double s = 0;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    s += x[i] * y[i];
  s = block_sum_256(s, smem);
  if (threadIdx.x == 0) partials[blockIdx.x] = s;
}

__global__ __launch_bounds__(256) void k_dot_finish(const double* __restrict__ partials, int n, double* __restrict__ out) {
  __shared__ double smem[8];
  double s = 0;
  for (int i = threadIdx.x; i < n; i += 256) s += partials[i];
  s = block_sum_256(s, smem);
  if (threadIdx.x == 0) *out = s;
}

static int grid_for(int64_t n, int threads, int cap = 65536) {
  int64_t g = ceil_div(n, threads);
  if (g < 1) g = 1;
  return (int)(g > cap ? cap : g);
}

template <class F>
static int with_vt(int vec, int precision, F&& f) {
  if (vec == 1 && precision == FEM_F32) return f(std::integral_constant<int, 1>{}, float{});
  if (vec == 1 && precision == FEM_F64) return f(std::integral_constant<int, 1>{}, double{});
  if (vec == 3 && precision == FEM_F32) return f(std::integral_constant<int, 3>{}, float{});
  if (vec == 3 && precision == FEM_F64) return f(std::integral_constant<int, 3>{}, double{});
  // block sizes of several variables on one mesh (sum of their vec)
  if (vec == 2 && precision == FEM_F32) return f(std::integral_constant<int, 2>{}, float{});
  if (vec == 2 && precision == FEM_F64) return f(std::integral_constant<int, 2>{}, double{});
  if (vec == 4 && precision == FEM_F32) return f(std::integral_constant<int, 4>{}, float{});
  if (vec == 4 && precision == FEM_F64) return f(std::integral_constant<int, 4>{}, double{});
  set_error("unsupported vec=%d / precision=%d", vec, precision);
  return FEM_ERR_BAD_ARG;
}

static int check_pat(const fem_pattern_t* p) {
  FEM_CHECK_ARG(p && p->row_ptr && p->slice_ptr && p->sell_row && p->sell_pos && p->num_rows > 0,
                "pattern descriptor invalid");
  FEM_CHECK_ARG(p->num_slices == ceil_div(p->num_rows, kSlice), "pattern num_slices mismatch");
  return FEM_OK;
}

}  // namespace fem

using namespace fem;

// Implemented here, used by the PCG driver.
int fem_operator_apply_impl(const fem_operator_t* op, const double* x, double* y, hipStream_t s);

int fem_operator_apply_impl(const fem_operator_t* op, const double* x, double* y, hipStream_t s) {
  FEM_CHECK_ARG(op && op->mesh && op->mat && op->u && op->inc_ptr && op->inc_idx && op->cell_scratch && x && y,
                "fem_operator_apply: NULL argument");
  int rc = fem_cell_jvp(op->mesh, op->mat, op->u, x, op->cell_scratch, s);
  if (rc) return rc;
  if (op->mass_M && (rc = fem_cell_mass_jvp(op->mesh, op->mass_M, x, op->cell_scratch, s))) return rc;
  if (op->cell_K && (rc = fem_cell_matvec(op->mesh, op->cell_K, x, op->cell_scratch, s))) return rc;
  rc = fem_gather_nodal(op->mesh->num_nodes, op->mesh->vec, op->inc_ptr, op->inc_idx, op->cell_scratch, nullptr, y, s);
  if (rc) return rc;
  if (op->n_bc > 0) {
    hipLaunchKernelGGL(k_copy_bc, dim3(grid_for(op->n_bc, 256)), dim3(256), 0, s, op->n_bc, op->bc_dofs, x, y);
    FEM_LAUNCHED();
  }
  return FEM_OK;
}

extern "C" {

int fem_gather_nodal(int64_t num_nodes, int32_t vec, const int32_t* inc_ptr, const int32_t* inc_idx,
                     const double* ent, const double* base, double* out, void* stream) {
  FEM_CHECK_ARG(num_nodes > 0 && vec >= 1 && vec <= 4 && inc_ptr && inc_idx && ent && out,
                "fem_gather_nodal: bad arguments");
  const dim3 grid(grid_for(num_nodes, 256));
  hipStream_t s = as_stream(stream);
  if (vec == 3)
    hipLaunchKernelGGL(k_gather_nodal<3>, grid, dim3(256), 0, s, num_nodes, inc_ptr, inc_idx, ent, base, out);
  else if (vec == 1)
    hipLaunchKernelGGL(k_gather_nodal<1>, grid, dim3(256), 0, s, num_nodes, inc_ptr, inc_idx, ent, base, out);
  else if (vec == 2)
    hipLaunchKernelGGL(k_gather_nodal<2>, grid, dim3(256), 0, s, num_nodes, inc_ptr, inc_idx, ent, base, out);
  else
    hipLaunchKernelGGL(k_gather_nodal<4>, grid, dim3(256), 0, s, num_nodes, inc_ptr, inc_idx, ent, base, out);
  FEM_LAUNCHED();
  return FEM_OK;
}

int fem_gather_matrix(const fem_pattern_t* pat, int32_t ke_precision, const void* Ke, int32_t precision, int32_t form,
                      void* vals, void* dinv, void* stream) {
  if (int rc = check_pat(pat)) return rc;
  FEM_CHECK_ARG(Ke && vals && pat->contrib_ptr && pat->contrib_idx && pat->diag_slot,
                "fem_gather_matrix: NULL argument");
  FEM_CHECK_ARG(pat->nnzb > 0 && pat->num_cells > 0 && pat->nodes_per_cell > 0,
                "fem_gather_matrix: pattern nnzb, num_cells and nodes_per_cell must be set");
  FEM_CHECK_ARG(ke_precision == precision || (ke_precision == FEM_F64 && precision == FEM_F32),
                "fem_gather_matrix: Ke precision must equal the matrix precision or be FP64");
  FEM_CHECK_ARG(form == FEM_FORM_STANDARD || form == FEM_FORM_DIFFERENCE, "fem_gather_matrix: bad form");
  if (pat->num_slices == 0) return FEM_OK;
  const dim3 grid((unsigned)pat->num_slices), block(64 * kGatherWaves);
  return with_vt(pat->vec, precision, [&](auto vc, auto tv) -> int {
    constexpr int V = decltype(vc)::value;
    using T = decltype(tv);
    hipStream_t s = as_stream(stream);
    if constexpr (V == 3) {
      if (pat->nodes_per_cell == 27) {
        const dim3 rows((unsigned)(pat->num_slices * (kSlice / kRowsPerGroup))), nt(64 * kRowWaves);
        auto go = [&](auto ts, auto diff) {
          using TS = decltype(ts);
          hipLaunchKernelGGL((k_gather_rows<3, 27, decltype(diff)::value, TS, T>), rows, nt, 0, s, *pat,
                             (const TS*)Ke, (T*)vals, (T*)dinv);
        };
        const bool d = form == FEM_FORM_DIFFERENCE;
        if (ke_precision == FEM_F64)
          d ? go(double{}, std::true_type{}) : go(double{}, std::false_type{});
        else
          d ? go(T{}, std::true_type{}) : go(T{}, std::false_type{});
        FEM_LAUNCHED();
        return FEM_OK;
      }
    }
    if (ke_precision == FEM_F64) {
      if (form == FEM_FORM_DIFFERENCE)
        hipLaunchKernelGGL((k_gather_matrix<V, true, double, T>), grid, block, 0, s, *pat, (const double*)Ke,
                           (T*)vals, (T*)dinv);
      else
        hipLaunchKernelGGL((k_gather_matrix<V, false, double, T>), grid, block, 0, s, *pat, (const double*)Ke,
                           (T*)vals, (T*)dinv);
    } else {
      if (form == FEM_FORM_DIFFERENCE)
        hipLaunchKernelGGL((k_gather_matrix<V, true, T, T>), grid, block, 0, s, *pat, (const T*)Ke, (T*)vals,
                           (T*)dinv);
      else
        hipLaunchKernelGGL((k_gather_matrix<V, false, T, T>), grid, block, 0, s, *pat, (const T*)Ke, (T*)vals,
                           (T*)dinv);
    }
    FEM_LAUNCHED();
    return FEM_OK;
  });
}

int fem_matrix_bc_rows(const fem_pattern_t* pat, int32_t precision, void* vals, int64_t n_bc, const int32_t* bc_dofs,
                       void* dinv, void* stream) {
  if (int rc = check_pat(pat)) return rc;
  FEM_CHECK_ARG(vals && (n_bc == 0 || bc_dofs) && pat->diag_slot, "fem_matrix_bc_rows: NULL argument");
  if (n_bc == 0) return FEM_OK;
  return with_vt(pat->vec, precision, [&](auto vc, auto tv) -> int {
    constexpr int V = decltype(vc)::value;
    using T = decltype(tv);
    hipLaunchKernelGGL((k_bc_rows<V, T>), dim3(grid_for(n_bc, 256)), dim3(256), 0, as_stream(stream), *pat, (T*)vals,
                       n_bc, bc_dofs, (T*)dinv);
    FEM_LAUNCHED();
    return FEM_OK;
  });
}

int fem_jacobi(const fem_pattern_t* pat, int32_t precision, const void* vals, void* dinv, void* stream) {
  if (int rc = check_pat(pat)) return rc;
  FEM_CHECK_ARG(vals && dinv && pat->diag_slot, "fem_jacobi: NULL argument");
  return with_vt(pat->vec, precision, [&](auto vc, auto tv) -> int {
    constexpr int V = decltype(vc)::value;
    using T = decltype(tv);
    hipLaunchKernelGGL((k_jacobi<V, T>), dim3(grid_for(pat->num_rows, 256)), dim3(256), 0, as_stream(stream), *pat,
                       (const T*)vals, (T*)dinv);
    FEM_LAUNCHED();
    return FEM_OK;
  });
}

int fem_residual_bc(int64_t n_bc, const int32_t* bc_dofs, const double* bc_vals, const double* u, double* res,
                    double scale, void* stream) {
  FEM_CHECK_ARG(n_bc >= 0 && (n_bc == 0 || (bc_dofs && bc_vals && u && res)), "fem_residual_bc: bad arguments");
  if (n_bc == 0) return FEM_OK;
  hipLaunchKernelGGL(k_residual_bc, dim3(grid_for(n_bc, 256)), dim3(256), 0, as_stream(stream), n_bc, bc_dofs,
                     bc_vals, u, res, scale);
  FEM_LAUNCHED();
  return FEM_OK;
}

int fem_spmv(const fem_pattern_t* pat, int32_t precision, int32_t form, const void* vals, const void* x, void* y,
             void* stream) {
  if (int rc = check_pat(pat)) return rc;
  FEM_CHECK_ARG(vals && x && y && pat->sell_col, "fem_spmv: NULL argument");
  FEM_CHECK_ARG(form == FEM_FORM_STANDARD || form == FEM_FORM_DIFFERENCE, "fem_spmv: bad form");
  return with_vt(pat->vec, precision, [&](auto vc, auto tv) -> int {
    constexpr int V = decltype(vc)::value;
    using T = decltype(tv);
    const dim3 grid((unsigned)pat->num_slices);
    auto product = [&](auto diff, auto waves) {
      constexpr int W = decltype(waves)::value;
      hipLaunchKernelGGL((k_spmv<V, decltype(diff)::value, T, W>), grid, dim3(64 * W), 0, as_stream(stream), *pat,
                         (const T*)vals, (const T*)x, (T*)y);
    };
    // Eight waves per slice for blocks and long rows, SliceCfg's for short scalar rows.  us with SliceCfg's
    // and with eight: HEX8 elastic 64^3 FP64 97 / 92, FP32 49.6 / 48.2, HEX27 12^3 32 / 20 and 17 / 11.5, 32^3
    // 343 / 319 and 165 / 161, HEX27 scalar 32^3 72 / 57 and 45 / 45; HEX8 scalar 64^3 19.6 / 18.5 and 16 / 18.2,
    // 100^3 66 / 68 and 54 / 64.
    using Some = std::integral_constant<int, 8>;
    using Many = std::integral_constant<int, SliceCfg<T>::W>;
    auto go = [&](auto diff) {
      if constexpr (V == 1) {
        if (!long_rows(*pat)) return product(diff, Many{});
      }
      product(diff, Some{});
    };
    if (form == FEM_FORM_DIFFERENCE)
      go(std::true_type{});
    else
      go(std::false_type{});
    FEM_LAUNCHED();
    return FEM_OK;
  });
}

int fem_export_csr(const fem_pattern_t* pat, int32_t precision, int32_t form, const void* vals, int32_t* indptr,
                   int32_t* indices, double* data, void* stream) {
  if (int rc = check_pat(pat)) return rc;
  FEM_CHECK_ARG(pat->col_idx && pat->diag_slot, "fem_export_csr: pattern without col_idx");
  FEM_CHECK_ARG((int64_t)pat->vec * pat->vec * pat->nnzb < (int64_t)INT32_MAX, "fem_export_csr: nnz exceeds int32");
  return with_vt(pat->vec, precision, [&](auto vc, auto tv) -> int {
    constexpr int V = decltype(vc)::value;
    using T = decltype(tv);
    hipLaunchKernelGGL((k_export_csr<V, T>), dim3(grid_for(pat->num_rows, 256)), dim3(256), 0, as_stream(stream),
                       *pat, (const T*)vals, form, indptr, indices, data);
    FEM_LAUNCHED();
    return FEM_OK;
  });
}

int fem_operator_apply(const fem_operator_t* op, const double* x, double* y, void* stream) {
  return fem_operator_apply_impl(op, x, y, as_stream(stream));
}

int fem_dot(int64_t n, const double* x, const double* y, double* out, void* ws, void* stream) {
  FEM_CHECK_ARG(n >= 0 && x && y && out && ws, "fem_dot: bad arguments");
  const int grid = grid_for(n, 256, 512);
  double* partials = reinterpret_cast<double*>(ws);
  hipStream_t s = as_stream(stream);
  hipLaunchKernelGGL(k_dot, dim3(grid), dim3(256), 0, s, n, x, y, partials);
  hipLaunchKernelGGL(k_dot_finish, dim3(1), dim3(256), 0, s, (const double*)partials, grid, out);
  FEM_LAUNCHED();
  return FEM_OK;
}

}  // extern "C"
