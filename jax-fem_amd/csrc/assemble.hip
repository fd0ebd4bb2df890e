// Single-pass HEX8 assembly: per-cell tangents (and optionally the residual)
// computed and summed straight into the SELL-64 matrix, with no per-cell
// tangent buffer in between.
//
// Replaces, in one kernel, what jax-fem does in two host-visible stages:
//   problem.py:447-460  compute_newton_vars: vmapped jacfwd per cell -> problem.V
//   solver.py:522-526   PETSc setValuesCOO: sum the COO duplicates into AIJ
//   problem.py:426-437  scatter of the cell residuals (optional, same pass)
//
// Work split.  A wave owns eight block rows (a group: eight consecutive lanes
// of one SELL slice) and shares nothing with other waves but the table of
// reference gradients: no barrier after the start, no atomics.  The plan lists
// the group's incident cells by ascending id and, for each row, its pairs
// (cell, local node a) in the same order, with the slots of the row that the
// pair's eight blocks go to.
//
// A cell's geometry and point records are recomputed once per group that
// touches it (about 4.5 times per 8 rows for a structured HEX8 box, against 4.1
// with 64-row groups); each tangent block is computed exactly once.
//
// What bounds it: LDS (60 to 70 % of its cycles: gradients read per block, blocks
// handed over) and the latencies that two waves per SIMD leave open; the matrix
// itself is written at 6 TB/s, past the caches.  64^3 Neo-Hookean cells with FP64
// values 2630 -> 925 us, 128 x 64 x 64 elastic cells 2000 -> 850 us (the stores alone
// take 220 us of these, a wave's first loads 130 us), 80 x 31 x 31 SIMP cells 342 ->
// 160 us, against one workgroup per slice that met at four barriers per chunk (80 to
// 110 KB of LDS, one or two workgroups per CU, most threads idle in most phases).
#include "element.hpp"

#include <algorithm>
#include <type_traits>

namespace fem {

constexpr int kGroupRows = 8;                // rows (and cells per chunk) of a wave
constexpr int kGroups = kSlice / kGroupRows; // groups per slice: the header of its cell list
constexpr int kSliceIncCap = 4096;           // incident (cell, node) entries of one slice's rows
constexpr int kSlicePairCap = 1024;          // pairs of a slice the assembly takes (the rank has 12 bits)
constexpr int kAsmMaxK = 4;                  // slots per lane: rows of at most 8 * 4 = 32 blocks

// A pair's word for slot class j (slots j, j + 8, j + 16, j + 24 of its row):
//   bits 0-15   four nibbles: the column node b whose block goes to slot j + 8 m, 8 = none
//   bits 16-18  a     bit 19  the cell names a node twice     bits 20-31  rank of the cell
constexpr uint32_t kNoSlots = 0x8888u, kTwice = 1u << 19;
constexpr int kRankShift = 20;

// An LDS pointer whose value the compiler does not know: constant offsets from it go into the
// instructions (from a known address it adds each of them up anew).
using LdsD = __attribute__((address_space(3))) double;
__device__ inline LdsD* lds_base(double* p) {
  LdsD* q = (LdsD*)p;
  asm volatile("" : "+v"(q));
  return q;
}

// ------------------------------------------------------------------ plan
// Cell lists of each slice: kGroups end offsets, then the groups' unique incident
// cells, ascending.  FILL = false writes the slice's entry and pair counts;
// FILL = true writes the entries at out_ptr[s].  One wave per group.
template <bool FILL>
__global__ __launch_bounds__(64 * kGroups) void k_slice_cells(int64_t num_slices,
                                                              const int32_t* __restrict__ sell_row,
                                                              const int32_t* __restrict__ inc_ptr,
                                                              const int32_t* __restrict__ inc_idx,
                                                              const int32_t* __restrict__ out_ptr,
                                                              int32_t* __restrict__ out,
                                                              int32_t* __restrict__ pair_out,
                                                              int32_t* __restrict__ err) {
  __shared__ int32_t s_buf[2 * kSliceIncCap];  // the groups' entries, each padded to a power of two
  __shared__ int32_t s_off[kSlice + 1];        // first entry of each row
  __shared__ int32_t s_n[kGroups];             // unique cells of each group
  const int64_t s = blockIdx.x;
  const int t = threadIdx.x, w = t >> 6, lane = t & 63;
  if (s >= num_slices) return;
  int row = -1, b = 0, e = 0;
  if (t < kSlice) {
    row = sell_row[s * kSlice + t];
    if (row >= 0) {
      b = inc_ptr[row];
      e = inc_ptr[row + 1];
    }
    s_off[t + 1] = e - b;
  }
  if (t == 0) s_off[0] = 0;
  __syncthreads();
  if (t == 0)
    for (int i = 1; i <= kSlice; ++i) s_off[i] += s_off[i - 1];
  __syncthreads();
  const int total = s_off[kSlice];
  if (!FILL && t == 0) pair_out[s] = total <= kSliceIncCap ? total : 0;
  if (total > kSliceIncCap) {
    if (t == 0) {
      atomicMax(err, total);
      if (!FILL) out[s] = 0;
    }
    return;
  }
  // the group's entries at s_buf[beg, beg + n), padded to P <= max(1, 2 n): the segments of the
  // groups start at twice their entry offset and do not overlap (P <= 2 n for n >= 1)
  const int g0 = s_off[w * kGroupRows], n = s_off[(w + 1) * kGroupRows] - g0;
  int32_t* buf = s_buf + 2 * g0;
  if (t < kSlice) {
    const int q0 = s_off[(t / kGroupRows) * kGroupRows];
    for (int j = b; j < e; ++j) s_buf[2 * q0 + (s_off[t] - q0) + (j - b)] = inc_idx[j] >> 3;
  }
  int P = n > 0 ? 1 : 0;
  while (P < n) P <<= 1;
  for (int i = n + lane; i < P; i += 64) buf[i] = INT32_MAX;
  __syncthreads();
  for (int k = 2; k <= P; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = lane; i < P; i += 64) {
        const int l = i ^ j;
        if (l > i) {
          const int32_t x = buf[i], y = buf[l];
          if ((x > y) == ((i & k) == 0)) {
            buf[i] = y;
            buf[l] = x;
          }
        }
      }
      wave_fence();
    }
  // unique entries: each lane takes a contiguous run of the sorted list
  const int per = (n + 63) / 64, i0 = min(n, lane * per), i1 = min(n, i0 + per);
  int cnt = 0;
  for (int i = i0; i < i1; ++i) cnt += (i == 0 || buf[i] != buf[i - 1]) ? 1 : 0;
  int scan = cnt;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int v = __shfl_up(scan, off, 64);
    if (lane >= off) scan += v;
  }
  if (lane == 63) s_n[w] = scan;
  __syncthreads();
  int before = 0, all = 0;
  for (int i = 0; i < kGroups; ++i) {
    if (i < w) before += s_n[i];
    all += s_n[i];
  }
  if (!FILL) {
    if (t == 0) out[s] = kGroups + all;
    return;
  }
  int32_t* o = out + out_ptr[s];
  if (lane == 63) o[w] = before + scan;
  o += kGroups + before + scan - cnt;
  for (int i = i0; i < i1; ++i)
    if (i == 0 || buf[i] != buf[i - 1]) *o++ = buf[i];
}

// The words of every pair: loc[8 p + j] for slot class j of the row's pair p, rows' pairs by
// ascending cell (a row with n pairs has 8 n contributions, so its words start where its
// contributions do).  One thread per (row, j).
__global__ __launch_bounds__(kSlice* kGroupRows) void k_pair_words(fem_pattern_t pat,
                                                                   const int32_t* __restrict__ inc_ptr,
                                                                   const int32_t* __restrict__ inc_idx,
                                                                   const int32_t* __restrict__ sc_ptr,
                                                                   const int32_t* __restrict__ sc,
                                                                   uint32_t* __restrict__ loc,
                                                                   int32_t* __restrict__ err) {
  if (*err) return;  // the plan is refused
  const int64_t s = blockIdx.x;
  const int l = threadIdx.x >> 3, j = threadIdx.x & 7, g = l / kGroupRows;
  const int row = pat.sell_row[s * kSlice + l];
  if (row < 0) return;
  const int32_t* hd = sc + sc_ptr[s];
  const int first = g ? hd[g - 1] : 0, nc = hd[g] - first;
  const int32_t* list = hd + kGroups + first;
  const int32_t* inc = inc_idx + inc_ptr[row];
  const int np = inc_ptr[row + 1] - inc_ptr[row];
  const int rb = pat.row_ptr[row], len = pat.row_ptr[row + 1] - rb, t0 = pat.contrib_ptr[rb];
  if (pat.contrib_ptr[rb + len] - t0 != 8 * np) {
    atomicMax(err, 1);
    return;
  }
  auto order = [&](int32_t e) {  // position of incidence e among the row's
    int p = 0;
    for (int i = 0; i < np; ++i) p += inc[i] < e ? 1 : 0;
    return p;
  };
  for (int i = 0; i < np; ++i) {
    const int32_t e = inc[i], c = e >> 3;
    int lo = 0, hi = nc;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (list[mid] < c) lo = mid + 1; else hi = mid;
    }
    if (lo >= nc || list[lo] != c || lo >= kSlicePairCap) {
      atomicMax(err, 1);
      return;
    }
    loc[t0 + 8 * order(e) + j] = ((uint32_t)lo << kRankShift) | ((uint32_t)(e & 7) << 16) | kNoSlots;
  }
  // every slot of the row: its own class' nibbles, and whether a pair has two blocks for it
  for (int k = 0; k < len; ++k) {
    const int c0 = pat.contrib_ptr[rb + k], c1 = pat.contrib_ptr[rb + k + 1];
    int32_t prev = -1;
    for (int t = c0; t < c1; ++t) {
      const int32_t v = pat.contrib_idx[t], e = v >> 3;
      if ((k & 7) != j && e != prev) {
        prev = e;
        continue;
      }
      uint32_t& word = loc[t0 + 8 * order(e) + j];
      if (e == prev) word |= kTwice;
      if ((k & 7) == j && k < 8 * kAsmMaxK) {
        const int sh = 4 * (k >> 3);
        const uint32_t b = v & 7, old = (word >> sh) & 15u;
        word = (word & ~(15u << sh)) | (min(b, old) << sh);  // 8 = none yet; the lowest of two
      }
      prev = e;
    }
  }
}

// The pairs of each slice for callers that ask for them (the assembly reads their words above):
// keys (rank * 8 + a) * 64 + lane, rank = place of the cell among the slice's lists, ascending.
__global__ __launch_bounds__(256) void k_slice_pairs(fem_pattern_t pat, const int32_t* __restrict__ inc_ptr,
                                                     const int32_t* __restrict__ inc_idx,
                                                     const int32_t* __restrict__ sc_ptr,
                                                     const int32_t* __restrict__ sc,
                                                     const int32_t* __restrict__ pair_ptr,
                                                     int32_t* __restrict__ pairs, const int32_t* __restrict__ err) {
  __shared__ int32_t s_key[kSliceIncCap];
  __shared__ int32_t s_off[kSlice + 1];
  if (*err) return;  // the plan is refused
  const int64_t s = blockIdx.x;
  const int t = threadIdx.x;
  const int row = t < kSlice ? pat.sell_row[s * kSlice + t] : -1;
  const int b = row >= 0 ? inc_ptr[row] : 0, e = row >= 0 ? inc_ptr[row + 1] : 0;
  if (t < kSlice) s_off[t + 1] = e - b;
  if (t == 0) s_off[0] = 0;
  __syncthreads();
  if (t == 0)
    for (int i = 1; i <= kSlice; ++i) s_off[i] += s_off[i - 1];
  __syncthreads();
  const int n = s_off[kSlice];
  if (n > kSliceIncCap || pair_ptr[s + 1] - pair_ptr[s] != n) return;
  if (t < kSlice) {
    const int32_t* hd = sc + sc_ptr[s];
    const int g = t / kGroupRows, first = g ? hd[g - 1] : 0, end = hd[g];
    const int32_t* list = hd + kGroups;
    for (int j = b; j < e; ++j) {
      int lo = first, hi = end;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (list[mid] < inc_idx[j] >> 3) lo = mid + 1; else hi = mid;
      }
      s_key[s_off[t] + j - b] = (lo * 8 + (inc_idx[j] & 7)) * kSlice + t;
    }
  }
  int P = 1;
  while (P < n) P <<= 1;
  for (int i = n + t; i < P; i += 256) s_key[i] = INT32_MAX;
  __syncthreads();
  for (int k = 2; k <= P; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = t; i < P; i += 256) {
        const int l = i ^ j;
        if (l > i) {
          const int32_t x = s_key[i], y = s_key[l];
          if ((x > y) == ((i & k) == 0)) {
            s_key[i] = y;
            s_key[l] = x;
          }
        }
      }
      __syncthreads();
    }
  for (int i = t; i < n; i += 256) pairs[pair_ptr[s] + i] = s_key[i];
}

// ------------------------------------------------------- point records
// What a block K_ab needs of a quadrature point besides the gradients h_a, h_b of its
// shape functions: NR doubles, weighted with JxW (point()), and the block itself (add(),
// summed over the points, then finish()).  kSpatial: the gradients are taken in the
// current configuration.  kRow: the law has a vector per (a, q) that all b share.
template <class MAT>
struct TanPoint;

// K = w k g_a . g_b
template <>
struct TanPoint<MatPoisson> {
  static constexpr int NR = 1;
  static constexpr bool kSpatial = false, kRow = false, kIso = false;
  __device__ static void point(const MatPoisson::St<double>& s, double w, double (&r)[NR]) { r[0] = w * s.k; }
  __device__ static void add(const LdsD* r, const double (&)[3], const double (&a)[3], const double (&b)[3], double&,
                             double (&K)[1][1]) {
    K[0][0] += r[0] * (a[0] * b[0] + a[1] * b[1] + a[2] * b[2]);
  }
};

// Isotropic linear laws: lambda = c0 E and mu = c1 E at every point, so with
// M = sum_q JxW E g_a (x) g_b,  K_ab = c0 M + c1 M^T + c1 tr(M) I.  The slots sum M.
template <bool S>
struct TanPoint<MatElastic<S>> {
  static constexpr int NR = 1;
  static constexpr bool kSpatial = false, kRow = false, kIso = true;
  __device__ static void add(const LdsD* r, const double (&)[3], const double (&a)[3], const double (&b)[3], double&,
                             double (&K)[3][3]) {
    const double w = r[0];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const double wa = w * a[i];
#pragma unroll
      for (int k = 0; k < 3; ++k) K[i][k] += wa * b[k];
    }
  }
};

// Neo-Hookean in the current configuration: with h = F^-T grad N, b = F F^T,
//   K_ab = c_fh (b h_a (x) h_b + h_a (x) b h_b) + c_hh h_a (x) h_b + c_tr h_b (x) h_a
//          + ma (h_a . b h_b) I,   c_fh = -2/3 ma
// (MatNeoHookean::tangent with F g = b h).  Record: c_fh b (6), c_hh, c_tr.  The
// row vector is t_a = c_fh b h_a + c_hh h_a: 42 operations per point instead of 106.
template <>
struct TanPoint<MatNeoHookean> {
  static constexpr int NR = 8;
  static constexpr bool kSpatial = true, kRow = true, kIso = false;
  __device__ static void bh(const LdsD* r, const double (&h)[3], double (&f)[3]) {
    f[0] = r[0] * h[0] + r[3 * 64] * h[1] + r[4 * 64] * h[2];
    f[1] = r[3 * 64] * h[0] + r[1 * 64] * h[1] + r[5 * 64] * h[2];
    f[2] = r[4 * 64] * h[0] + r[5 * 64] * h[1] + r[2 * 64] * h[2];
  }
  __device__ static void row(const LdsD* r, const double (&a)[3], double (&t)[3]) {
    bh(r, a, t);
#pragma unroll
    for (int i = 0; i < 3; ++i) t[i] += r[6 * 64] * a[i];
  }
  __device__ static void add(const LdsD* r, const double (&t)[3], const double (&a)[3], const double (&b)[3],
                             double& d, double (&K)[3][3]) {
    double f[3];
    bh(r, b, f);
    d += a[0] * f[0] + a[1] * f[1] + a[2] * f[2];
    const double ct = r[7 * 64];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const double cb = ct * b[i];
#pragma unroll
      for (int k = 0; k < 3; ++k) K[i][k] += t[i] * b[k] + a[i] * f[k] + cb * a[k];
    }
  }
};

// J2: MatJ2::tangent with the symmetric deviator.  Record: s (6), w lam_t, w mu_t, w gam.
template <>
struct TanPoint<MatJ2> {
  static constexpr int NR = 9;
  static constexpr bool kSpatial = false, kRow = true, kIso = false;
  __device__ static void point(const MatJ2::St<double>& s, double w, double (&r)[NR]) {
    r[0] = s.s[0], r[1] = s.s[4], r[2] = s.s[8], r[3] = s.s[1], r[4] = s.s[2], r[5] = s.s[5];
    r[6] = w * s.lam_t, r[7] = w * s.mu_t, r[8] = w * s.gam;
  }
  __device__ static void row(const LdsD* r, const double (&a)[3], double (&t)[3]) {
    TanPoint<MatNeoHookean>::bh(r, a, t);
#pragma unroll
    for (int i = 0; i < 3; ++i) t[i] *= r[8 * 64];
  }
  __device__ static void add(const LdsD* r, const double (&t)[3], const double (&a)[3], const double (&b)[3],
                             double& d, double (&K)[3][3]) {
    double sb[3];
    TanPoint<MatNeoHookean>::bh(r, b, sb);
    const double l = r[6 * 64], m = r[7 * 64];
    d += m * (a[0] * b[0] + a[1] * b[1] + a[2] * b[2]);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const double la = l * a[i], mb = m * b[i];
#pragma unroll
      for (int k = 0; k < 3; ++k) K[i][k] += la * b[k] + mb * a[k] - t[i] * sb[k];
    }
  }
};

// ------------------------------------------------------------- assembly
constexpr int kAsmThreads = 128;             // 2 waves: 16 rows, whole 128-byte lines of FP64 values
constexpr int kGQ = 25, kGC = 8 * kGQ;       // strides of the staged gradients: [cell][q][node][3]
constexpr int kXC = 49;                      // stride of a cell's staged coordinates and u

// LDS of one wave: the chunk's gradients (its coordinates and u before them), point
// records, weighted stresses and the blocks in exchange.
template <class MAT, bool RES>
struct AsmWave {
  static constexpr int NP = RES ? (MAT::V == 1 ? 3 : 6) : 0, NR = TanPoint<MAT>::NR;
  // values of a block exchanged at a time: as many as leave eight waves' LDS on a CU (20,480 bytes
  // each with the table), at least a row vector's three
  static constexpr int NX = MAT::V == 1 ? 1 : NR == 1 ? 9 : NR <= 8 ? 5 : 3;
  double g[8 * kGC];
  double rec[NR + NP][64];
  double ex[65 * NX];  // the last entry stays zero: the block of a slot that receives none
};

// One wave per group.  The group's cells are walked in chunks of eight; per chunk
//   1  lane (cell, node): coordinates (and u) to LDS, loaded one chunk ahead;
//   2  lane (cell, q): Jacobian, inverse, the eight gradients, the point record (and the
//      weighted stress);
//   3  while a row has pairs in the chunk: lane (row, b) forms block K_ab of the row's next
//      pair (the eight lanes share h_a and the records) and hands it to the lane that owns
//      its slot (lane j of a row owns the slots j, j + 8, ...), which adds it in registers.
// Every sum runs in the plan's order, so the result does not depend on scheduling.
// With the residual, lane (row, q) sums its point's part over the row's pairs and the
// eight lanes are added at the end.
template <class MAT, typename TO, bool DIFF, bool RES>
__global__ __launch_bounds__(kAsmThreads, 2) void k_assemble_hex8(
    fem_mesh_t mesh, fem_material_t mat, fem_pattern_t pat, const int32_t* __restrict__ sc_ptr,
    const int32_t* __restrict__ sc, const uint32_t* __restrict__ loc, const double* __restrict__ u,
    TO* __restrict__ vals, TO* __restrict__ dinv, const double* __restrict__ base, double* __restrict__ res) {
  using TP = TanPoint<MAT>;
  constexpr int V = MAT::V, VV = V * V, M = kAsmMaxK, NR = TP::NR;
  constexpr bool kU = MAT::kNeedsU || RES;
  constexpr bool kParam = !std::is_same<MAT, MatJ2>::value;
  __shared__ double s_dN[8 * kGQ], s_w[8];
  __shared__ AsmWave<MAT, RES> s_wave[kAsmThreads / 64];
  AsmWave<MAT, RES>& L = s_wave[threadIdx.x >> 6];
  const int lane = threadIdx.x & 63, hi8 = lane >> 3, j = lane & 7;
  // (uniform in the wave, and known to be: what follows from it stays in scalar registers)
  const int gid = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (kAsmThreads / 64) + (threadIdx.x >> 6)));
  const int s = gid / kGroups;
  const int gr = gid % kGroups, rl = gr * kGroupRows + hi8;  // the lane's row in the slice

  // The wave's two chains of lists, row -> pairs and group -> cells -> nodes -> coordinates, are
  // begun side by side and before the tables' barrier (one after the other: 128 x 64 x 64 elastic
  // cells 867 us instead of 849, 64^3 Neo-Hookean with the residual 1070 instead of 1045).
  const int sbase = pat.slice_ptr[s], nslots = (pat.slice_ptr[s + 1] - sbase) >> 6;
  const int row = pat.sell_row[s * kSlice + rl];
  const int32_t* cl = sc + sc_ptr[s];
  const int first = gr ? cl[gr - 1] : 0, nc = cl[gr] - first;
  cl += kGroups + first;
  auto cell_at = [&](int k) { return cl[min(k * 8 + hi8, nc - 1)]; };
  // loaded ahead: cell, node, coordinates and parameter of the coming chunk (1), cell and node of
  // the one after it (2), cells of the third
  int32_t c1 = 0, n1 = 0, c2 = 0, n2 = 0, c3 = 0;
  if (nc > 0) c1 = cell_at(0), c2 = cell_at(1), c3 = cell_at(2);
  for (int i = threadIdx.x; i < 8 * 24; i += kAsmThreads) s_dN[(i / 24) * kGQ + i % 24] = mesh.shape_grads_ref[i];
  if (threadIdx.x < 8) s_w[threadIdx.x] = mesh.quad_weights[threadIdx.x];
  const int rr = max(row, 0), rb = pat.row_ptr[rr], re = pat.row_ptr[rr + 1];
  int ds = pat.diag_slot[rr];
  if (nc > 0) n1 = mesh.cells[(int64_t)c1 * 8 + j], n2 = mesh.cells[(int64_t)c2 * 8 + j];
  const int t0 = pat.contrib_ptr[rb];
  int np = (pat.contrib_ptr[re] - t0) >> 3;  // pairs of the row
  __syncthreads();
  double xr[3] = {0, 0, 0}, ur[V], par = 1.0;
#pragma unroll
  for (int i = 0; i < V; ++i) ur[i] = 0.0;
  // without parameters the load reads a weight and is not used (a branch would split the geometry)
  const bool has_par = kParam && mat.has_param;
  const double* par_base = has_par ? mat.param : mesh.quad_weights;
  auto load_chunk = [&]() {
#pragma unroll
    for (int i = 0; i < 3; ++i) xr[i] = mesh.points[(int64_t)n1 * 3 + i];
    if constexpr (kU)
#pragma unroll
      for (int i = 0; i < V; ++i) ur[i] = u[(int64_t)n1 * V + i];
    if constexpr (kParam) par = par_base[has_par ? (int64_t)c1 * 8 + j : 0];
  };
  if (nc > 0) load_chunk();
  np = row >= 0 ? np : 0;
  ds = row >= 0 ? ds : -1;
  const uint32_t* pw = loc + (np > 0 ? t0 : 0) + j;
  // word: the row's next pair; ahead: what was loaded for pair ip, the one after it (beyond the
  // row's last pair the load repeats that one and is not used)
  int ip = 1;
  uint32_t word = pw[0], ahead = pw[8 * min(1, max(np - 1, 0))];
  if (np == 0) word = ~0u;
  constexpr int NX = AsmWave<MAT, RES>::NX;
  LdsD *const lg = lds_base(L.g), *const lr = lds_base(&L.rec[0][0]), *const lx = lds_base(L.ex);
  if (lane < NX) lx[64 * NX + lane] = 0.0;

  // the point's reference gradients: kept where the registers suffice, else read from LDS each time
  constexpr bool kKeep = TP::kIso && !RES;
  double kept[kKeep ? 24 : 1];
  if constexpr (kKeep)
#pragma unroll
    for (int i = 0; i < 24; ++i) kept[i] = s_dN[j * kGQ + i];
  double acc[M][VV];
#pragma unroll
  for (int m = 0; m < M; ++m)
#pragma unroll
    for (int v = 0; v < VV; ++v) acc[m][v] = 0.0;
  double rs[V];
#pragma unroll
  for (int i = 0; i < V; ++i) rs[i] = 0.0;

  for (int k = 0; k * 8 < nc; ++k) {
    // ---- 1: the chunk's coordinates to LDS; fetch the next chunk's
    wave_fence();
    const int32_t c0 = c1;
    const double p0 = has_par ? par : 1.0;
    {
      LdsD* x = lg + hi8 * kXC + j * 6;
#pragma unroll
      for (int i = 0; i < 3; ++i) x[i] = xr[i];
      if constexpr (kU)
#pragma unroll
        for (int i = 0; i < V; ++i) x[3 + i] = ur[i];
    }
    c1 = c2, n1 = n2;
    c2 = c3;
    load_chunk();
    n2 = mesh.cells[(int64_t)c2 * 8 + j];
    c3 = cell_at(k + 3);
    wave_fence();
    __builtin_amdgcn_sched_barrier(0);
    double E = 1.0;
    if constexpr (std::is_same<MAT, MatElastic<true>>::value) {
      E = MAT::modulus(mat, p0);
      __builtin_amdgcn_sched_barrier(0);  // the power's temporaries end before the Jacobian's begin
    }
    // ---- 2: geometry, gradients and records of (cell hi8, point j)
    {
      double J[9], U[V][3];
#pragma unroll
      for (int i = 0; i < 9; ++i) J[i] = 0.0;
#pragma unroll
      for (int i = 0; i < V; ++i) U[i][0] = U[i][1] = U[i][2] = 0.0;
      const LdsD* x = lg + hi8 * kXC;
      const LdsD* tab = lds_base(&s_dN[j * kGQ]);
      auto dn = [&](int i) { return kKeep ? kept[kKeep ? i : 0] : tab[i]; };
#pragma unroll
      for (int a = 1; a < 8; ++a) {
        const double e0 = dn(a * 3), e1 = dn(a * 3 + 1), e2 = dn(a * 3 + 2);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const double d = x[a * 6 + i] - x[i];
          J[i * 3 + 0] += d * e0;
          J[i * 3 + 1] += d * e1;
          J[i * 3 + 2] += d * e2;
        }
        if constexpr (kU)
#pragma unroll
          for (int i = 0; i < V; ++i) {
            const double d = x[a * 6 + 3 + i] - x[3 + i];
            U[i][0] += d * e0;
            U[i][1] += d * e1;
            U[i][2] += d * e2;
          }
        if (a == 3 || a == 5) __builtin_amdgcn_sched_barrier(0);
      }
      const double det = det3(J), w = det * s_w[j];
      double iJ[9], r[NR];
      inv3(J, det, iJ);
      [[maybe_unused]] double P[6];
      if constexpr (TP::kSpatial) {
        // F = I + grad_ref u J^-1; h = j^-T dN with j = J + grad_ref u.  (F, and its determinant, from
        // the displacement's gradient: from j they carry j's rounding, which the stress of a small
        // strain, a difference of terms of order 1, shows undiminished.)
        double jc[9], F[9];
#pragma unroll
        for (int i = 0; i < 9; ++i) jc[i] = J[i] + U[i / 3][i % 3];
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int l = 0; l < 3; ++l)
            F[i * 3 + l] = (U[i][0] * iJ[l] + U[i][1] * iJ[3 + l] + U[i][2] * iJ[6 + l]) + (i == l ? 1.0 : 0.0);
        const double b[6] = {F[0] * F[0] + F[1] * F[1] + F[2] * F[2], F[3] * F[3] + F[4] * F[4] + F[5] * F[5],
                             F[6] * F[6] + F[7] * F[7] + F[8] * F[8], F[0] * F[3] + F[1] * F[4] + F[2] * F[5],
                             F[0] * F[6] + F[1] * F[7] + F[2] * F[8], F[3] * F[6] + F[4] * F[7] + F[5] * F[8]};
        const double Jd = det3(F);
        inv3(jc, det3(jc), iJ);
        const double wp = w * p0, I1 = b[0] + b[1] + b[2];
        const double ma = mat.c[0] * wp * pow_m23(Jd), kp = mat.c[1] * wp;
#pragma unroll
        for (int i = 0; i < 6; ++i) r[i] = (-2.0 / 3.0) * ma * b[i];
        const double kj = kp * Jd * (Jd - 1.0), mi = ma * I1 * (1.0 / 3.0);
        r[6] = (2.0 / 3.0) * mi + kj + kp * (Jd * Jd);
        r[7] = mi - kj;
        if constexpr (RES)
#pragma unroll
          for (int i = 0; i < 6; ++i) P[i] = ma * b[i] + (i < 3 ? kj - mi : 0.0);  // Kirchhoff stress
      } else {
        double G[V][3];
        if constexpr (kU)
#pragma unroll
          for (int i = 0; i < V; ++i)
#pragma unroll
            for (int l = 0; l < 3; ++l) G[i][l] = U[i][0] * iJ[l] + U[i][1] * iJ[3 + l] + U[i][2] * iJ[6 + l];
        typename MAT::template St<double> st;
        if constexpr (TP::kIso) {
          r[0] = w * E;
          st.lam = mat.c[0] * E;
          st.mu = mat.c[1] * E;
        } else {
          if constexpr (std::is_same<MAT, MatPoisson>::value)
            st.k = mat.c[0] * p0;
          else
            st = MAT::template prep<double>(mat, (int64_t)c0 * 8 + j, G);
          TP::point(st, w, r);
        }
        if constexpr (RES) {
          double S[V][3];
          MAT::stress(st, G, S);
          if constexpr (V == 1) {
#pragma unroll
            for (int i = 0; i < 3; ++i) P[i] = w * S[0][i];
          } else {  // symmetric
            P[0] = w * S[0][0], P[1] = w * S[1][1], P[2] = w * S[2][2];
            P[3] = w * S[0][1], P[4] = w * S[0][2], P[5] = w * S[1][2];
          }
        }
      }
      wave_fence();  // the gradients overwrite the coordinates
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < NR; ++i) lr[i * 64 + lane] = r[i];
      if constexpr (RES)
#pragma unroll
        for (int i = 0; i < AsmWave<MAT, RES>::NP; ++i) lr[(NR + i) * 64 + lane] = P[i];
      tab = lds_base(&s_dN[j * kGQ]);
      LdsD* g = lg + hi8 * kGC + j * kGQ;
#pragma unroll
      for (int a = 0; a < 8; ++a) {
        const double e0 = dn(a * 3), e1 = dn(a * 3 + 1), e2 = dn(a * 3 + 2);
#pragma unroll
        for (int l = 0; l < 3; ++l) g[a * 3 + l] = e0 * iJ[l] + e1 * iJ[3 + l] + e2 * iJ[6 + l];
      }
    }
    // ---- 3: the rows' pairs of this chunk
    const uint32_t lim = (uint32_t)(k + 1) * 8u;
    do {  // every chunk has a pair
      const bool active = (word >> kRankShift) < lim;
      const uint32_t cur = active ? word : kNoSlots | ((uint32_t)k * 8u << kRankShift);
      // no branch around the fetch: one would make the compiler copy every accumulator
      word = active ? (ip < np ? ahead : ~0u) : word;
      ip += active ? 1 : 0;
      ahead = pw[8 * max(min(ip, np - 1), 0)];
      const int cc = (int)(cur >> kRankShift) - k * 8, a = (cur >> 16) & 7;
      const LdsD* ga = lg + cc * kGC + a * 3;
      const LdsD* gb = lg + cc * kGC + j * 3;
      const LdsD* rec = lr + cc * 8;
      wave_fence();
      if constexpr (TP::kRow || RES) {  // lane (row, q = j)
        const double ha[3] = {ga[j * kGQ], ga[j * kGQ + 1], ga[j * kGQ + 2]};
        if constexpr (TP::kRow) {
          double t[3];
          TP::row(rec + j, ha, t);
#pragma unroll
          for (int i = 0; i < 3; ++i) lx[lane * 3 + i] = t[i];
        }
        if constexpr (RES) {
          const LdsD* p = rec + j + NR * 64;
          double f[3];
          if constexpr (V == 1)
            f[0] = p[0] * ha[0] + p[64] * ha[1] + p[128] * ha[2];
          else
            TanPoint<MatNeoHookean>::bh(p, ha, f);
#pragma unroll
          for (int i = 0; i < V; ++i) rs[i] += active ? f[i] : 0.0;
        }
        wave_fence();
      }
      double K[V][V], d = 0.0;
#pragma unroll
      for (int i = 0; i < V; ++i)
#pragma unroll
        for (int l = 0; l < V; ++l) K[i][l] = 0.0;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const double ha[3] = {ga[q * kGQ], ga[q * kGQ + 1], ga[q * kGQ + 2]};
        const double hb[3] = {gb[q * kGQ], gb[q * kGQ + 1], gb[q * kGQ + 2]};
        double t[3] = {0, 0, 0};
        if constexpr (TP::kRow)
#pragma unroll
          for (int i = 0; i < 3; ++i) t[i] = lx[(hi8 * 8 + q) * 3 + i];
        TP::add(rec + q, t, ha, hb, d, K);
      }
      if constexpr (TP::kRow) {
        const double dd = TP::kSpatial ? -1.5 * d : d;  // Neo-Hookean: the records hold c_fh = -2/3 ma
#pragma unroll
        for (int i = 0; i < V; ++i) K[i][i] += dd;
      }
      if (__any((cur & kTwice) != 0)) {
        // a cell naming a node twice: the lowest lane of equal columns takes their sum
        const int32_t node = mesh.cells[(int64_t)cl[min((int)(cur >> kRankShift), nc - 1)] * 8 + j];
        double S[V][V];
#pragma unroll
        for (int i = 0; i < V; ++i)
#pragma unroll
          for (int l = 0; l < V; ++l) S[i][l] = 0.0;
        for (int b = 0; b < 8; ++b) {
          const bool same = __shfl(node, (lane & 56) + b, 64) == node;
#pragma unroll
          for (int i = 0; i < V; ++i)
#pragma unroll
            for (int l = 0; l < V; ++l) {
              const double v = __shfl(K[i][l], (lane & 56) + b, 64);
              if (same) S[i][l] += v;
            }
        }
#pragma unroll
        for (int i = 0; i < V; ++i)
#pragma unroll
          for (int l = 0; l < V; ++l) K[i][l] = S[i][l];
      }
      // hand the blocks to their slots, NX values at a time
#pragma unroll
      for (int r0 = 0; r0 < (VV + NX - 1) / NX; ++r0) {
        wave_fence();
#pragma unroll
        for (int v = 0; v < NX; ++v)
          if (r0 * NX + v < VV) lx[lane * NX + v] = K[(r0 * NX + v) / V][(r0 * NX + v) % V];
        wave_fence();
#pragma unroll
        for (int m = 0; m < M; ++m) {
          const int b = (cur >> (4 * m)) & 15;
          if (!__any(b < 8)) continue;  // a HEX8 box: two or three of the four
          const LdsD* e = lx + (b < 8 ? (lane & 56) + b : 64) * NX;
#pragma unroll
          for (int v = 0; v < NX; ++v)
            if (r0 * NX + v < VV) acc[m][r0 * NX + v] += e[v];
        }
      }
    } while (__any((word >> kRankShift) < lim));
  }

  if constexpr (TP::kIso) {
    const double l = mat.c[0], mu = mat.c[1];
#pragma unroll
    for (int m = 0; m < M; ++m) {
      double A[9];
#pragma unroll
      for (int v = 0; v < 9; ++v) A[v] = acc[m][v];
      const double tr = mu * (A[0] + A[4] + A[8]);
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int k = 0; k < 3; ++k) acc[m][i * 3 + k] = l * A[i * 3 + k] + mu * A[k * 3 + i] + (i == k ? tr : 0.0);
    }
  }
  // sums over the eight lanes of a row, the same in every lane
  auto row_sum = [](double v) {
    v += dpp_move<kDppXor1>(v);
    v += dpp_move<kDppXor2>(v);
    return v + dpp_move<kDppHalfMirror>(v);
  };
  double rsum[DIFF ? VV : 1];  // difference form: the diagonal block holds the row sum
  if constexpr (DIFF)
#pragma unroll
    for (int v = 0; v < VV; ++v) {
      double p = 0.0;
#pragma unroll
      for (int m = 0; m < M; ++m) p += acc[m][v];
      rsum[v] = row_sum(p);
    }
  if (dinv && row >= 0 && ds < 0 && j < V) dinv[(int64_t)row * V + j] = TO(0);  // a node of no cell
  // the diagonal block: its inverse diagonal, then the difference form's row sum in its place
#pragma unroll
  for (int c = 0; c < V; ++c) {
    double d = 0.0;
#pragma unroll
    for (int m = 0; m < M; ++m) d = ds == j + 8 * m ? acc[m][c * V + c] : d;
    if (dinv && ds >= 0 && (ds & 7) == j) dinv[(int64_t)row * V + c] = d != 0.0 ? TO(1.0 / d) : TO(0);
  }
  TO* vp = vals + (size_t)sbase * VV + rl;
#pragma unroll
  for (int m = 0; m < M; ++m) {
    const int k = j + 8 * m;
    if (k < nslots)
#pragma unroll
      for (int v = 0; v < VV; ++v)
        __builtin_nontemporal_store(TO((DIFF && k == ds) ? rsum[v] : acc[m][v]), &vp[((size_t)k * VV + v) * kSlice]);
  }
  if constexpr (RES) {
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const double r = row_sum(rs[i]);
      if (j == i && row >= 0) {
        const int64_t idx = (int64_t)row * V + i;
        res[idx] = (base ? base[idx] : 0.0) + r;
      }
    }
  }
}

// ------------------------------------------------------------- dispatch
template <class F>
static int with_mat8(const fem_material_t& mat, int vec, F&& f) {
  switch (mat.kind) {
    case FEM_MAT_POISSON:
      if (vec == 1) return f(MatPoisson{});
      break;
    case FEM_MAT_LINEAR_ELASTIC:
      if (vec == 3) return f(MatElastic<false>{});
      break;
    case FEM_MAT_SIMP:
      if (vec == 3 && mat.has_param) return f(MatElastic<true>{});
      break;
    case FEM_MAT_NEO_HOOKEAN:
      if (vec == 3) return f(MatNeoHookean{});
      break;
    case FEM_MAT_J2_PLASTIC:
      if (vec == 3 && mat.state) return f(MatJ2{});
      break;
    default:
      break;
  }
  set_error("fem_assemble: material kind %d (vec=%d) is assembled by the two-pass path "
            "(fem_cell_tangent + fem_gather_matrix)", mat.kind, vec);
  return FEM_ERR_BAD_ARG;
}

}  // namespace fem

using namespace fem;

extern "C" {

int fem_assembly_plan_counts(const fem_pattern_t* pat, const int32_t* inc_ptr, const int32_t* inc_idx,
                             int32_t* slice_cell_counts, int32_t* slice_pair_counts, int32_t* err_flag,
                             void* stream) {
  FEM_CHECK_ARG(pat && inc_ptr && inc_idx && slice_cell_counts && slice_pair_counts && err_flag,
                "fem_assembly_plan_counts: NULL argument");
  FEM_CHECK_ARG(pat->nodes_per_cell == 8, "fem_assembly_plan_counts: HEX8 patterns only");
  if (pat->num_slices == 0) return FEM_OK;
  hipStream_t st = as_stream(stream);
  FEM_HIP(hipMemsetAsync(err_flag, 0, sizeof(int32_t), st));
  hipLaunchKernelGGL(k_slice_cells<false>, dim3((unsigned)pat->num_slices), dim3(64 * kGroups), 0, st,
                     pat->num_slices, pat->sell_row, inc_ptr, inc_idx, (const int32_t*)nullptr,
                     slice_cell_counts, slice_pair_counts, err_flag);
  FEM_LAUNCHED();
  return FEM_OK;
}

int fem_assembly_plan_fill(const fem_pattern_t* pat, const int32_t* inc_ptr, const int32_t* inc_idx,
                           const int32_t* slice_cell_ptr, const int32_t* slice_pair_ptr, int32_t* slice_cells,
                           int32_t* slice_pairs, int32_t* contrib_loc, int32_t* err_flag, void* stream) {
  FEM_CHECK_ARG(pat && inc_ptr && inc_idx && slice_cell_ptr && slice_cells && contrib_loc && err_flag,
                "fem_assembly_plan_fill: NULL argument");
  FEM_CHECK_ARG(!slice_pairs || slice_pair_ptr, "fem_assembly_plan_fill: slice_pairs without slice_pair_ptr");
  FEM_CHECK_ARG(pat->nodes_per_cell == 8, "fem_assembly_plan_fill: HEX8 patterns only");
  if (pat->num_slices == 0) return FEM_OK;
  hipStream_t st = as_stream(stream);
  hipLaunchKernelGGL(k_slice_cells<true>, dim3((unsigned)pat->num_slices), dim3(64 * kGroups), 0, st,
                     pat->num_slices, pat->sell_row, inc_ptr, inc_idx, slice_cell_ptr, slice_cells,
                     (int32_t*)nullptr, err_flag);
  FEM_LAUNCHED();
  hipLaunchKernelGGL(k_pair_words, dim3((unsigned)pat->num_slices), dim3(kSlice * kGroupRows), 0, st, *pat, inc_ptr,
                     inc_idx, slice_cell_ptr, slice_cells, (uint32_t*)contrib_loc, err_flag);
  FEM_LAUNCHED();
  if (slice_pairs) {
    hipLaunchKernelGGL(k_slice_pairs, dim3((unsigned)pat->num_slices), dim3(256), 0, st, *pat, inc_ptr, inc_idx,
                       slice_cell_ptr, slice_cells, slice_pair_ptr, slice_pairs, err_flag);
    FEM_LAUNCHED();
  }
  return FEM_OK;
}

int fem_assemble(const fem_mesh_t* mesh, const fem_material_t* mat, const fem_pattern_t* pat,
                 const fem_assembly_plan_t* plan, const double* u, int32_t precision, int32_t form, void* vals,
                 void* dinv, const double* base, double* res, void* stream) {
  FEM_CHECK_ARG(mesh && mat && pat && plan && u && vals, "fem_assemble: NULL argument");
  FEM_CHECK_ARG(mesh->nodes_per_cell == 8 && mesh->num_quads == 8,
                "fem_assemble: single-pass assembly covers HEX8 cells with 8 quadrature points");
  FEM_CHECK_ARG(pat->nodes_per_cell == 8 && pat->vec == mesh->vec && pat->num_cells == mesh->num_cells,
                "fem_assemble: pattern and mesh disagree");
  FEM_CHECK_ARG(plan->slice_cell_ptr && plan->slice_cells && plan->contrib_loc, "fem_assemble: plan not built");
  FEM_CHECK_ARG(plan->max_slots >= 0 && plan->max_slots <= 8 * kAsmMaxK,
                "fem_assemble: a slice has %d blocks per row (at most %d)", plan->max_slots, 8 * kAsmMaxK);
  FEM_CHECK_ARG(plan->max_pairs >= 0 && plan->max_pairs <= kSlicePairCap,
                "fem_assemble: a slice has %d (cell, row node) pairs (at most %d)", plan->max_pairs, kSlicePairCap);
  FEM_CHECK_ARG((precision == FEM_F64 && form == FEM_FORM_STANDARD) ||
                    (precision == FEM_F32 && form == FEM_FORM_DIFFERENCE),
                "fem_assemble: FP64 standard-form or FP32 difference-form storage");
  FEM_CHECK_ARG(!mat->has_param || mat->param, "fem_assemble: material param missing");
  if (pat->num_slices == 0) return FEM_OK;
  hipStream_t st = as_stream(stream);
  const dim3 grid((unsigned)(pat->num_slices * kGroups * 64 / kAsmThreads)), block(kAsmThreads);
  return with_mat8(*mat, mesh->vec, [&](auto m) -> int {
    using MAT = decltype(m);
    auto go = [&](auto res_c) {
      constexpr bool R = decltype(res_c)::value;
      if (precision == FEM_F64)
        hipLaunchKernelGGL((k_assemble_hex8<MAT, double, false, R>), grid, block, 0, st, *mesh, *mat, *pat,
                           plan->slice_cell_ptr, plan->slice_cells, (const uint32_t*)plan->contrib_loc, u, (double*)vals, (double*)dinv, base, res);
      else
        hipLaunchKernelGGL((k_assemble_hex8<MAT, float, true, R>), grid, block, 0, st, *mesh, *mat, *pat,
                           plan->slice_cell_ptr, plan->slice_cells, (const uint32_t*)plan->contrib_loc, u, (float*)vals, (float*)dinv, base, res);
    };
    if (res)
      go(std::true_type{});
    else
      go(std::false_type{});
    FEM_LAUNCHED();
    return FEM_OK;
  });
}

}  // extern "C"
