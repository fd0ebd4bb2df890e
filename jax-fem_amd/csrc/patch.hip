// Matrix-free residuals and tangent products over patches of consecutive cells.
//
// Replaces, for the element integrals the solvers repeat, the reference's
// vmapped cell kernels and scatter (problem.py:261-296, 426-445) and the
// products with the assembled matrix (solver.py:63-92): the cells' integrals
// are recomputed from the nodal coordinates instead of read from HBM.
//
// Two kernels per product.
//   k_patch_hex8, k_patch_hex27
//                   one workgroup per patch of consecutive cells (128 or 28).
//                   Every cell's nodal vector is formed in registers, staged in
//                   LDS and summed per distinct node of the patch (a fixed
//                   order): one partial per (patch, node) goes to memory
//                   instead of one per (cell, node).
//   k_patch_gather  one thread per dof sums the partials of its node (one to
//                   four for a structured mesh, a fixed order) and applies the
//                   product's epilogue (Dirichlet identity rows, residual,
//                   Chebyshev step, <x, A x> partials).
// Nothing depends on scheduling: the products are bit-reproducible.
//
// On the 1.6M-dof HEX8 cantilever (524,288 cells, a modulus per point) a product
// takes 55 us (40 + 15) where the FP64 SELL matrix takes 190 and its FP32
// difference form 103 (1116 and 587 MB against 180), a residual 56 us where the
// cell vectors and their nodal gather took 193.  The cells' pass issues 890
// vector instructions per thread (720 FP64), about 26 us of the chip's issue
// rate at three waves per SIMD; the gather moves 64 MB at about 5 TB/s.  Patches
// of 64 / 128 / 256 cells: 63, 61, 71 us before the plan's entries were fetched
// ahead (61 -> 55).
#include "patch.hpp"

#include "element.hpp"

#include <algorithm>
#include <type_traits>

namespace fem {

constexpr int kPatchCells = 128;  // HEX8 cells per patch
constexpr int kPatchCells27 = 28;  // HEX27 cells per patch: 7 per wave, 9 lanes each
constexpr int kPatchCap = 2048;   // most (cell, node) entries of a patch

// ------------------------------------------------------------------ plan
// Per patch, the (cell in patch, local node) entries sorted by node: bitonic
// sort of (node << 11 | entry) in LDS.  FILL = false writes the number of
// distinct nodes; FILL = true writes the sorted entries, each distinct node
// and the end of its entries.
template <bool FILL>
__global__ __launch_bounds__(256) void k_patch_nodes(int64_t num_cells, int N, int cpp,
                                                     const int32_t* __restrict__ cells, int32_t* __restrict__ counts,
                                                     const int32_t* __restrict__ slot_ptr,
                                                     int32_t* __restrict__ slot_node, uint16_t* __restrict__ slot_end,
                                                     uint16_t* __restrict__ contrib) {
  __shared__ unsigned long long key[kPatchCap];
  __shared__ int32_t s_scan[256];
  const int t = threadIdx.x;
  const int64_t c0 = (int64_t)blockIdx.x * cpp;
  const int total = (int)min((int64_t)cpp, num_cells - c0) * N;
  int P = 1;
  while (P < total) P <<= 1;
  for (int i = t; i < P; i += 256)
    key[i] = i < total ? ((unsigned long long)(uint32_t)cells[c0 * N + i] << 11) | (unsigned)i : ~0ull;
  __syncthreads();
  for (int k = 2; k <= P; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int i = t; i < P; i += 256) {
        const int l = i ^ j;
        if (l > i) {
          const unsigned long long a = key[i], b = key[l];
          if ((a > b) == ((i & k) == 0)) {
            key[i] = b;
            key[l] = a;
          }
        }
      }
      __syncthreads();
    }
  // each thread owns a contiguous run; a run counts the last entries of its nodes
  const int per = (total + 255) / 256;
  const int i0 = min(total, t * per), i1 = min(total, i0 + per);
  int cnt = 0;
  for (int i = i0; i < i1; ++i) cnt += (i + 1 == total || (key[i + 1] >> 11) != (key[i] >> 11)) ? 1 : 0;
  s_scan[t] = cnt;
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {
    const int a = t >= off ? s_scan[t - off] : 0;
    __syncthreads();
    s_scan[t] += a;
    __syncthreads();
  }
  if (!FILL) {
    if (t == 255) counts[blockIdx.x] = s_scan[255];
    return;
  }
  int pos = slot_ptr[blockIdx.x] + s_scan[t] - cnt;
  for (int i = i0; i < i1; ++i) {
    contrib[c0 * N + i] = (uint16_t)(key[i] & 2047u);
    if (i + 1 == total || (key[i + 1] >> 11) != (key[i] >> 11)) {
      slot_node[pos] = (int32_t)(key[i] >> 11);
      slot_end[pos++] = (uint16_t)(i + 1);
    }
  }
}

// ------------------------------------------------------------ element layer
// value of the neighbouring lane (lane ^ 1)
__device__ inline double swap_lane1(double x) { return dpp_move<kDppXor1>(x); }

// Reference gradients of NC nodal fields on one layer of quadrature points of a
// trilinear cell, sum-factorised.  Two neighbouring lanes share a cell: lane h = 0
// holds the nodes 0-3 of the face z = 0 and integrates the points nearest to it,
// h = 1 the nodes 4-7 and the points nearest z = 1.  With the third reference
// coordinate counted from the lane's own face (z' = z or 1 - z) both lanes run the
// same code; J and the fields use the same coordinate, so physical gradients agree
// and only det J changes sign on h = 1.
//   d/dx at point (i, j):  e[j];   d/dy:  f[i];   d/dz':  a[i] and b[i], the values on
//   the edges y = 0 and y = 1, interpolated to j.
template <int NC>
struct Layer {
  double e[2][NC], f[2][NC], a[2][NC], b[2][NC];
};

template <int NC>
__device__ inline void layer_grad(const double (&n)[4][NC], double g, Layer<NC>& L) {
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    double dl[4], p[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      dl[k] = swap_lane1(n[k][c]) - n[k][c];
      p[k] = fma(g, dl[k], n[k][c]);
    }
    const double e0 = p[1] - p[0], e1 = p[2] - p[3], de = e1 - e0;
    L.e[0][c] = fma(g, de, e0);
    L.e[1][c] = fma(-g, de, e1);
    const double f0 = p[3] - p[0], f1 = p[2] - p[1], df = f1 - f0;
    L.f[0][c] = fma(g, df, f0);
    L.f[1][c] = fma(-g, df, f1);
    const double da = dl[1] - dl[0], db = dl[2] - dl[3];
    L.a[0][c] = fma(g, da, dl[0]);
    L.a[1][c] = fma(-g, da, dl[1]);
    L.b[0][c] = fma(g, db, dl[3]);
    L.b[1][c] = fma(-g, db, dl[2]);
  }
}

// d/dz' at point (i, j)
template <int NC>
__device__ inline double layer_dz(const Layer<NC>& L, int i, int j, int c, double g) {
  const double d = L.b[i][c] - L.a[i][c];
  return j == 0 ? fma(g, d, L.a[i][c]) : fma(-g, d, L.b[i][c]);
}

// Transpose of layer_grad: S holds the sums of the weighted stresses against e, f, a, b;
// r[k] receives the vector of the lane's node k (both layers' points summed).
template <int NC>
__device__ inline void layer_div(const Layer<NC>& S, double g, double (&r)[4][NC]) {
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const double de = S.e[1][c] - S.e[0][c], e0 = fma(g, de, S.e[0][c]), e1 = fma(-g, de, S.e[1][c]);
    const double df = S.f[1][c] - S.f[0][c], f0 = fma(g, df, S.f[0][c]), f1 = fma(-g, df, S.f[1][c]);
    const double da = S.a[1][c] - S.a[0][c], db = S.b[1][c] - S.b[0][c];
    const double p[4] = {-e0 - f0, e0 - f1, e1 + f1, f0 - e1};
    const double d[4] = {fma(g, da, S.a[0][c]), fma(-g, da, S.a[1][c]), fma(-g, db, S.b[1][c]), fma(g, db, S.b[0][c])};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const double other = fma(g, p[k], d[k]);
      r[k][c] = (p[k] - other) + swap_lane1(other);
    }
  }
}

// adjugate of the row-major 3x3 A (A^-1 = adj / det)
__device__ inline void adj3(const double (&A)[9], double (&B)[9]) {
  B[0] = A[4] * A[8] - A[5] * A[7];
  B[1] = A[2] * A[7] - A[1] * A[8];
  B[2] = A[1] * A[5] - A[2] * A[4];
  B[3] = A[5] * A[6] - A[3] * A[8];
  B[4] = A[0] * A[8] - A[2] * A[6];
  B[5] = A[2] * A[3] - A[0] * A[5];
  B[6] = A[3] * A[7] - A[4] * A[6];
  B[7] = A[1] * A[6] - A[0] * A[7];
  B[8] = A[0] * A[4] - A[1] * A[3];
}

// 1 / x by the hardware estimate (2^-24) and two Newton steps: rounds as the division does (0.5 ulp at
// most over 0.5 .. 1.5 and e^-50 .. e^50); 0, inf and NaN give a non-finite result
__device__ inline double rcp_newton(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  return fma(fma(-x, r, 1.0), r, r);
}

// Laws whose stress is linear in grad u take the weight and the Jacobian's scaling into
// their constants instead of the nine stresses.
__device__ inline void scale_state(MatPoisson::St<double>& st, double s) { st.k *= s; }
template <class St>
__device__ inline void scale_state(St& st, double s) {
  st.lam *= s;
  st.mu *= s;
}

// The isotropic elastic law with a given modulus factor per point (the SIMP law with its
// power already taken): lambda = c0 E, mu = c1 E.
struct MatModulus : MatElastic<false> {
  template <typename T>
  __device__ static St<T> prep(const fem_material_t& m, int64_t cq, const T (&)[3][3]) {
    St<T> s;
    const double E = m.param[cq];
    s.lam = T(m.c[0] * E);
    s.mu = T(m.c[1] * E);
    return s;
  }
};

// Sum of the patch's staged cell vectors per distinct node, to its partials.  The plan's
// entries are fetched when the kernel starts (load) and put beside the staged vectors before
// the barrier (stage), so that no wave waits for them after it: the cells' pass is bound by
// such waits (its arithmetic alone takes half its time).
template <int N, int V, int STRIDE, int CELLS, int NT>
struct PatchSums {
  static constexpr int kEntries = CELLS * N;         // entries and, at most, slots of a patch
  static constexpr int EPT = (kEntries + NT - 1) / NT;
  int64_t n0;
  int cnt;
  uint16_t ent[EPT], end[EPT];

  struct Lds {
    uint16_t ent[kEntries], end[kEntries + 1];
  };

  __device__ void load(const fem_patch_plan_t& plan, int64_t patch, int64_t num_cells) {
    n0 = plan.slot_ptr[patch];
    cnt = (int)(plan.slot_ptr[patch + 1] - n0);
    const int total = (int)min((int64_t)CELLS, num_cells - patch * CELLS) * N;
    const uint16_t* lst = plan.contrib + patch * kEntries;
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
      const int i = threadIdx.x + k * NT;
      ent[k] = i < total ? lst[i] : 0;
      end[k] = i < cnt ? plan.slot_end[n0 + i] : 0;
    }
  }
  __device__ void stage(Lds& L) const {
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
      const int i = threadIdx.x + k * NT;
      if (i < kEntries) {
        L.ent[i] = ent[k];
        L.end[i + 1] = end[k];
      }
    }
    if (threadIdx.x == 0) L.end[0] = 0;
  }
  __device__ void store(const Lds& L, const double* s_r, double* __restrict__ part) const {
    for (int i = threadIdx.x; i < cnt; i += NT) {
      const int stop = L.end[i + 1];
      double t[V];
#pragma unroll
      for (int v = 0; v < V; ++v) t[v] = 0.0;
      for (int k = L.end[i]; k < stop; ++k) {
        const int e = L.ent[k];
        const double* r = s_r + (e / N) * STRIDE + (e % N) * V;
#pragma unroll
        for (int v = 0; v < V; ++v) t[v] += r[v];
      }
#pragma unroll
      for (int v = 0; v < V; ++v) part[(n0 + i) * V + v] = t[v];
    }
  }
};

// Kirchhoff form of the Neo-Hookean tangent (MatNeoHookean::jvp pushed to the current
// configuration): with L = grad v in current coordinates, b = F F^T and the weighted
// constants m = mu J^-2/3 and k = kappa,
//   dtau = m (L b - 2/3 tr(L) b - 2/3 (b : L) I + 2/9 I1 tr(L) I) + k (2 J^2 - J) tr(L) I
//          + (m I1 / 3 - k (J^2 - J)) L^T,
// integrated against current gradients.  Fewer products than the material form and, with b
// (6 values) in place of F and its inverse, fewer live registers.
// jr, jc: reference and current Jacobians; Lr: reference gradient of v; w: quadrature
// weight with the sign of the lane's det jr; T: weighted stress against reference gradients.
__device__ inline void neo_hookean_tangent(const fem_material_t& m, int64_t cq, const double (&jr)[9],
                                           const double (&jc)[9], const double (&Lr)[3][3], double w,
                                           double (&T)[3][3]) {
  double b[6], J, W;
  {
    double A[9], F[3][3];
    adj3(jr, A);
    const double det = jr[0] * A[0] + jr[1] * A[3] + jr[2] * A[6], id = rcp_newton(det);
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int l = 0; l < 3; ++l) F[i][l] = jc[3 * i] * A[l] + jc[3 * i + 1] * A[3 + l] + jc[3 * i + 2] * A[6 + l];
    const double s = id * id;
    b[0] = s * (F[0][0] * F[0][0] + F[0][1] * F[0][1] + F[0][2] * F[0][2]);
    b[1] = s * (F[1][0] * F[1][0] + F[1][1] * F[1][1] + F[1][2] * F[1][2]);
    b[2] = s * (F[2][0] * F[2][0] + F[2][1] * F[2][1] + F[2][2] * F[2][2]);
    b[3] = s * (F[0][0] * F[1][0] + F[0][1] * F[1][1] + F[0][2] * F[1][2]);
    b[4] = s * (F[0][0] * F[2][0] + F[0][1] * F[2][1] + F[0][2] * F[2][2]);
    b[5] = s * (F[1][0] * F[2][0] + F[1][1] * F[2][1] + F[1][2] * F[2][2]);
    J = id;
    W = w * det;
  }
  double A[9], L[3][3];
  adj3(jc, A);
  const double det = jc[0] * A[0] + jc[1] * A[3] + jc[2] * A[6], id = rcp_newton(det);
  J *= det;
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int l = 0; l < 3; ++l) L[i][l] = Lr[i][0] * A[l] + Lr[i][1] * A[3 + l] + Lr[i][2] * A[6 + l];
  const double s = W * id * id * param_at(m, cq);
  const double ma = m.c[0] * s * pow_m23(J), k = m.c[1] * s, I1 = b[0] + b[1] + b[2];
  const double tr = L[0][0] + L[1][1] + L[2][2];
  const double bL = b[0] * L[0][0] + b[1] * L[1][1] + b[2] * L[2][2] + b[3] * (L[0][1] + L[1][0]) +
                    b[4] * (L[0][2] + L[2][0]) + b[5] * (L[1][2] + L[2][1]);
  const double cb = ma * (-2.0 / 3.0) * tr;
  const double ci = (ma * (2.0 / 9.0) * I1 + k * (2.0 * J * J - J)) * tr - ma * (2.0 / 3.0) * bL;
  const double ct = ma * I1 * (1.0 / 3.0) - k * (J * J - J);
  const double B[3][3] = {{b[0], b[3], b[4]}, {b[3], b[1], b[5]}, {b[4], b[5], b[2]}};
  double D[3][3];
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const double Lb = L[i][0] * B[0][j] + L[i][1] * B[1][j] + L[i][2] * B[2][j];
      D[i][j] = ma * Lb + cb * B[i][j] + ct * L[j][i] + (i == j ? ci : 0.0);
    }
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int d = 0; d < 3; ++d) T[i][d] = D[i][0] * A[3 * d] + D[i][1] * A[3 * d + 1] + D[i][2] * A[3 * d + 2];
}

// The field a cells' pass gathers: x, or z + beta x (the direction of a CG iteration that the
// pass begins, in the vectors' precision as the gather kernel stores it).
struct NoHead {
  const int32_t* done;
};
template <typename TX, typename HEAD>
struct PatchField {
  const TX* x;
  const TX* z;
  HEAD head;
};

// A cells' pass takes raw() first, loads its cells' data and then finishes the head (begin()).
struct NoRaw {
  int32_t done;
};
template <int NT>
__device__ inline NoRaw raw(const NoHead& h) {
  return NoRaw{h.done ? *h.done : 0};
}
template <int NT>
__device__ inline PcgRaw<NT> raw(const PcgHead& h) {
  return pcg_raw<NT>(h);
}
template <int NT>
__device__ inline CgRaw<NT> raw(const CgHead& h) {
  return cg_raw<NT>(h);
}
template <int NT>
__device__ inline double begin(const NoHead&, const NoRaw& r, double*, bool* done) {
  *done = r.done != 0;
  return 0.0;
}
template <int NT>
__device__ inline double begin(const PcgHead& h, const PcgRaw<NT>& r, double* smem, bool* done) {
  return pcg_head<NT>(h, r, smem, done);
}
template <int NT>
__device__ inline double begin(const CgHead& h, const CgRaw<NT>& r, double* smem, bool* done) {
  return cg_head<NT>(h, r, smem, done);
}
template <int NT, typename TX, typename HEAD, typename RAW>
__device__ inline TX patch_begin(const PatchField<TX, HEAD>& f, const RAW& r, bool* done) {
  if constexpr (std::is_same<HEAD, NoHead>::value) {
    return TX(begin<NT>(f.head, r, nullptr, done));
  } else {
    __shared__ double smem[2 * (NT / 64)];
    return TX(begin<NT>(f.head, r, smem, done));
  }
}

// MODE 0: internal force at x (u unused); MODE 1: tangent at u times x.
template <class MAT, int MODE, typename TX, typename HEAD>
__global__ __launch_bounds__(2 * kPatchCells) void k_patch_hex8(fem_mesh_t mesh, fem_material_t mat,
                                                                fem_patch_plan_t plan, const double* __restrict__ u,
                                                                PatchField<TX, HEAD> field, double* __restrict__ part) {
  constexpr int N = 8, V = MAT::V, NT = 2 * kPatchCells, STRIDE = N * V + 1;  // odd: no bank conflicts between cells
  constexpr bool kNeo = MODE == 1 && MAT::kNeedsU;     // the tangent of the hyperelastic law
  constexpr bool kLinear = !MAT::kNeedsU;
  static_assert(!MAT::kNeedsU || std::is_same<MAT, MatNeoHookean>::value, "one nonlinear law");
  constexpr bool CG = !std::is_same<HEAD, NoHead>::value;
  using Sums = PatchSums<N, V, STRIDE, kPatchCells, NT>;
  __shared__ double s_r[kPatchCells * STRIDE];
  __shared__ typename Sums::Lds s_plan;
  const auto head = raw<NT>(field.head);
  const int64_t patch = xcd_logical_block(blockIdx.x, gridDim.x);
  Sums sums;
  const int h = threadIdx.x & 1, cl = threadIdx.x >> 1;
  // lanes past the last cell repeat it; the plan does not list their results
  const int64_t c = min(patch * kPatchCells + cl, mesh.num_cells - 1);
  const double g = plan.val[1];
  Layer<3> X;       // coordinates
  Layer<V> F;       // the field
  Layer<3> C;       // kNeo: current coordinates
  {
    const int4 node = *reinterpret_cast<const int4*>(mesh.cells + c * N + 4 * h);
    const int id[4] = {node.x, node.y, node.z, node.w};
    double nx[4][3], nf[4][V];
    TX fx[4][V], fz[CG ? 4 : 1][V];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
#pragma unroll
      for (int j = 0; j < 3; ++j) nx[k][j] = mesh.points[(int64_t)id[k] * 3 + j];
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const int64_t at = (int64_t)id[k] * V + v;
        fx[k][v] = field.x[at];
        if (CG) fz[k][v] = field.z[at];
      }
    }
    sums.load(plan, patch, mesh.num_cells);
    bool done;
    const TX beta = patch_begin<NT>(field, head, &done);
    if (done) return;
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int v = 0; v < V; ++v) nf[k][v] = double(CG ? fma(beta, fx[k][v], fz[k][v]) : fx[k][v]);
    // coordinates, and the residual's field, from the cell's first node, so that their differences
    // round like the cell's size and the field's change over it
    auto from_first = [&](auto& n) {
      constexpr int NC = sizeof(n[0]) / sizeof(double);
#pragma unroll
      for (int j = 0; j < NC; ++j) {
        const double o = swap_lane1(n[0][j]), n0 = h ? o : n[0][j];
#pragma unroll
        for (int k = 0; k < 4; ++k) n[k][j] -= n0;
      }
    };
    from_first(nx);
    if constexpr (MODE == 0) from_first(nf);
    layer_grad<3>(nx, g, X);
    layer_grad<V>(nf, g, F);
    if constexpr (kNeo) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int j = 0; j < 3; ++j) nx[k][j] += u[(int64_t)id[k] * 3 + j];
      layer_grad<3>(nx, g, C);
    }
  }
  Layer<V> S;
#pragma unroll
  for (int v = 0; v < V; ++v) S.e[0][v] = S.e[1][v] = 0.0;
  auto columns = [&](auto& L, int i, int j, auto& M) {  // M[k][dir]: reference gradients at point (i, j)
    constexpr int NC = sizeof(M) / sizeof(M[0]);
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      M[k][0] = L.e[j][k];
      M[k][1] = L.f[i][k];
      M[k][2] = layer_dz(L, i, j, k, g);
    }
  };
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    double sf[V], sz[2][V];
#pragma unroll
    for (int v = 0; v < V; ++v) sf[v] = 0.0;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int64_t cq = c * 8 + (4 * i + 2 * j + h);
      const double w0 = mesh.quad_weights[4 * i + 2 * j], w1 = mesh.quad_weights[4 * i + 2 * j + 1];
      const double w = h ? -w1 : w0;
      double J3[3][3], R[V][3], T[V][3];
      columns(X, i, j, J3);
      columns(F, i, j, R);
      double J[9];
#pragma unroll
      for (int k = 0; k < 9; ++k) J[k] = J3[k / 3][k % 3];
      if constexpr (kNeo) {
        double C3[3][3], Jc[9];
        columns(C, i, j, C3);
#pragma unroll
        for (int k = 0; k < 9; ++k) Jc[k] = C3[k / 3][k % 3];
        neo_hookean_tangent(mat, cq, J, Jc, R, w, T);
      } else {
        double A[9], G[V][3], P[V][3];
        adj3(J, A);
        const double det = J[0] * A[0] + J[1] * A[3] + J[2] * A[6];
        // linear laws: grad u = G / det and the second 1 / det and JxW go into the constants
        const double id = rcp_newton(det);
        if constexpr (!kLinear)
#pragma unroll
          for (int k = 0; k < 9; ++k) A[k] *= id;
#pragma unroll
        for (int v = 0; v < V; ++v)
#pragma unroll
          for (int k = 0; k < 3; ++k) G[v][k] = R[v][0] * A[k] + R[v][1] * A[3 + k] + R[v][2] * A[6 + k];
        auto st = MAT::template prep<double>(mat, cq, G);
        if constexpr (kLinear) {
          scale_state(st, w * id);
          MAT::stress(st, G, P);
        } else {
          MAT::stress(st, G, P);
          const double jxw = w * det;
#pragma unroll
          for (int v = 0; v < V; ++v)
#pragma unroll
            for (int k = 0; k < 3; ++k) P[v][k] *= jxw;
        }
#pragma unroll
        for (int v = 0; v < V; ++v)
#pragma unroll
          for (int d = 0; d < 3; ++d) T[v][d] = P[v][0] * A[3 * d] + P[v][1] * A[3 * d + 1] + P[v][2] * A[3 * d + 2];
      }
#pragma unroll
      for (int v = 0; v < V; ++v) {
        S.e[j][v] += T[v][0];
        sf[v] += T[v][1];
        sz[j][v] = T[v][2];
      }
    }
#pragma unroll
    for (int v = 0; v < V; ++v) {
      S.f[i][v] = sf[v];
      const double d = sz[1][v] - sz[0][v];
      S.a[i][v] = fma(g, d, sz[0][v]);
      S.b[i][v] = fma(-g, d, sz[1][v]);
    }
  }
  double r[4][V];
  layer_div<V>(S, g, r);
#pragma unroll
  for (int k = 0; k < 4; ++k)
#pragma unroll
    for (int v = 0; v < V; ++v) s_r[cl * STRIDE + (4 * h + k) * V + v] = r[k][v];
  sums.stage(s_plan);
  __syncthreads();
  sums.store(s_plan, s_r, part);
}

// ------------------------------------------------------------ HEX27 cells
// LDS written by a wave and read by the same wave: its DS instructions execute in order, the
// fence keeps the compiler from reordering them.
__device__ inline void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// VTK number of lattice node (i, j, k) of the triquadratic cell, at 9 i + 3 j + k
__device__ const int8_t kVtk27[27] = {0, 16, 4, 11, 20, 15, 3,  19, 7,  8, 22, 12, 24, 26,
                                      25, 10, 23, 14, 1, 17, 5, 9, 21, 13, 2, 18, 6};

// Triquadratic cells with the 3x3x3 Gauss rule, sum-factorised: nine lanes per cell, each
// holding a line of three values, contract one axis at a time with the 1-D tables and hand
// the results on through LDS (seven cells per wave, so no barrier is needed).  MODE as in
// k_patch_hex8; the tangent covers the laws that are linear in grad u.
template <class MAT, int MODE, typename TX, typename HEAD>
__global__ __launch_bounds__(256) void k_patch_hex27(fem_mesh_t mesh, fem_material_t mat, fem_patch_plan_t plan,
                                                     PatchField<TX, HEAD> field, double* __restrict__ part) {
  constexpr int N = 27, V = MAT::V, NT = 256, STRIDE = 243;  // doubles of LDS per cell: 3 fields, 3 kinds, 27 points
  constexpr bool kLinear = !MAT::kNeedsU;
  static_assert(MODE == 0 || kLinear, "the hyperelastic tangent runs on HEX8 patches only");
  constexpr bool CG = !std::is_same<HEAD, NoHead>::value;
  using Sums = PatchSums<N, V, STRIDE, kPatchCells27, NT>;
  __shared__ double s_r[kPatchCells27 * STRIDE];
  __shared__ typename Sums::Lds s_plan;
  const auto head = raw<NT>(field.head);
  const int64_t patch = xcd_logical_block(blockIdx.x, gridDim.x);
  const int lane = min((int)(threadIdx.x & 63), 62);  // lane 63 repeats lane 62
  const int cl = (threadIdx.x >> 6) * 7 + lane / 9, t = lane % 9, ta = t / 3, tb = t % 3;
  const int64_t c = min(patch * kPatchCells27 + cl, mesh.num_cells - 1);
  double* L = s_r + cl * STRIDE;
  Sums sums;
  auto val = [&](int q, int n) { return plan.val[3 * q + n]; };
  auto der = [&](int q, int n) { return plan.der[3 * q + n]; };
  // nodal lines n[i][field] of lane (j, k) -> h[field][kind][k] of lane (qx, qy): kind 0 the value
  // along both axes, 1 the y derivative, 2 the x derivative
  auto contract = [&](auto& n, auto& h) {
    constexpr int NC = sizeof(n[0]) / sizeof(double);
#pragma unroll
    for (int f = 0; f < NC; ++f)
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        L[(2 * f) * 27 + q * 9 + t] = val(q, 0) * n[0][f] + val(q, 1) * n[1][f] + val(q, 2) * n[2][f];
        L[(2 * f + 1) * 27 + q * 9 + t] = der(q, 0) * n[0][f] + der(q, 1) * n[1][f] + der(q, 2) * n[2][f];
      }
    wave_lds_fence();
    double a[NC][3], b[NC][3];
#pragma unroll
    for (int f = 0; f < NC; ++f)
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        a[f][j] = L[(2 * f) * 27 + ta * 9 + j * 3 + tb];
        b[f][j] = L[(2 * f + 1) * 27 + ta * 9 + j * 3 + tb];
      }
    wave_lds_fence();
#pragma unroll
    for (int f = 0; f < NC; ++f)
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        double* o = L + (3 * f) * 27 + ta * 9 + q * 3 + tb;
        o[0] = val(q, 0) * a[f][0] + val(q, 1) * a[f][1] + val(q, 2) * a[f][2];
        o[27] = der(q, 0) * a[f][0] + der(q, 1) * a[f][1] + der(q, 2) * a[f][2];
        o[54] = val(q, 0) * b[f][0] + val(q, 1) * b[f][1] + val(q, 2) * b[f][2];
      }
    wave_lds_fence();
#pragma unroll
    for (int f = 0; f < NC; ++f)
#pragma unroll
      for (int kind = 0; kind < 3; ++kind)
#pragma unroll
        for (int k = 0; k < 3; ++k) h[f][kind][k] = L[(3 * f + kind) * 27 + t * 3 + k];
    wave_lds_fence();
  };
  double hx[3][3][3], hf[V][3][3];
  int vtk[3];
  {
    double nx[3][3], nf[3][V];
    TX fx[3][V], fz[CG ? 3 : 1][V];
    const int32_t* cn = mesh.cells + c * N;
    const double* p0 = mesh.points + (int64_t)cn[0] * 3;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      vtk[i] = kVtk27[9 * i + t];
      const int64_t id = cn[vtk[i]];
#pragma unroll
      for (int j = 0; j < 3; ++j) nx[i][j] = mesh.points[id * 3 + j] - p0[j];
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const int64_t at = id * V + v;
        fx[i][v] = field.x[at];
        if (CG) fz[i][v] = field.z[at];
      }
    }
    sums.load(plan, patch, mesh.num_cells);
    bool done;
    const TX beta = patch_begin<NT>(field, head, &done);
    if (done) return;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int v = 0; v < V; ++v) nf[i][v] = double(CG ? fma(beta, fx[i][v], fz[i][v]) : fx[i][v]);
    if constexpr (MODE == 0)  // from the cell's first node (held by its first lane), as the coordinates
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const double f0 = __shfl(nf[0][v], lane - t, 64);
#pragma unroll
        for (int i = 0; i < 3; ++i) nf[i][v] -= f0;
      }
    contract(nx, hx);
    contract(nf, hf);
  }
  double s[V][3][3];
#pragma unroll
  for (int v = 0; v < V; ++v)
#pragma unroll
    for (int kind = 0; kind < 3; ++kind)
#pragma unroll
      for (int k = 0; k < 3; ++k) s[v][kind][k] = 0.0;
  // reference gradients at point q of the lane's line: M[f][dir]
  auto columns = [&](auto& h, int q, auto& M) {
    constexpr int NC = sizeof(M) / sizeof(M[0]);
#pragma unroll
    for (int f = 0; f < NC; ++f) {
      M[f][0] = val(q, 0) * h[f][2][0] + val(q, 1) * h[f][2][1] + val(q, 2) * h[f][2][2];
      M[f][1] = val(q, 0) * h[f][1][0] + val(q, 1) * h[f][1][1] + val(q, 2) * h[f][1][2];
      M[f][2] = der(q, 0) * h[f][0][0] + der(q, 1) * h[f][0][1] + der(q, 2) * h[f][0][2];
    }
  };
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    double J3[3][3], R[V][3], J[9], A[9], G[V][3], P[V][3];
    columns(hx, q, J3);
    columns(hf, q, R);
#pragma unroll
    for (int k = 0; k < 9; ++k) J[k] = J3[k / 3][k % 3];
    adj3(J, A);
    const double det = J[0] * A[0] + J[1] * A[3] + J[2] * A[6], id = rcp_newton(det);
    const double w = mesh.quad_weights[t * 3 + q];
    if constexpr (!kLinear)
#pragma unroll
      for (int k = 0; k < 9; ++k) A[k] *= id;
#pragma unroll
    for (int v = 0; v < V; ++v)
#pragma unroll
      for (int k = 0; k < 3; ++k) G[v][k] = R[v][0] * A[k] + R[v][1] * A[3 + k] + R[v][2] * A[6 + k];
    auto st = MAT::template prep<double>(mat, c * 27 + t * 3 + q, G);
    if constexpr (kLinear) scale_state(st, w * id);
    MAT::stress(st, G, P);
    if constexpr (!kLinear) {
      const double jxw = w * det;
#pragma unroll
      for (int v = 0; v < V; ++v)
#pragma unroll
        for (int k = 0; k < 3; ++k) P[v][k] *= jxw;
    }
#pragma unroll
    for (int v = 0; v < V; ++v) {
      double T[3];
#pragma unroll
      for (int d = 0; d < 3; ++d) T[d] = P[v][0] * A[3 * d] + P[v][1] * A[3 * d + 1] + P[v][2] * A[3 * d + 2];
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        s[v][2][k] = fma(val(q, k), T[0], s[v][2][k]);
        s[v][1][k] = fma(val(q, k), T[1], s[v][1][k]);
        s[v][0][k] = fma(der(q, k), T[2], s[v][0][k]);
      }
    }
  }
  // the transposed contractions, back to the lane's nodes
#pragma unroll
  for (int v = 0; v < V; ++v)
#pragma unroll
    for (int kind = 0; kind < 3; ++kind)
#pragma unroll
      for (int k = 0; k < 3; ++k) L[(3 * v + kind) * 27 + t * 3 + k] = s[v][kind][k];
  wave_lds_fence();
  double a[V][3], b[V][3];
#pragma unroll
  for (int v = 0; v < V; ++v) {
#pragma unroll
    for (int j = 0; j < 3; ++j) a[v][j] = b[v][j] = 0.0;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const double* o = L + (3 * v) * 27 + ta * 9 + q * 3 + tb;
      const double vv = o[0], vd = o[27], dv = o[54];
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        a[v][j] = fma(val(q, j), vv, fma(der(q, j), vd, a[v][j]));
        b[v][j] = fma(val(q, j), dv, b[v][j]);
      }
    }
  }
  wave_lds_fence();
#pragma unroll
  for (int v = 0; v < V; ++v)
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      L[(2 * v) * 27 + ta * 9 + j * 3 + tb] = a[v][j];
      L[(2 * v + 1) * 27 + ta * 9 + j * 3 + tb] = b[v][j];
    }
  wave_lds_fence();
  double r[3][V];
#pragma unroll
  for (int v = 0; v < V; ++v) {
#pragma unroll
    for (int i = 0; i < 3; ++i) r[i][v] = 0.0;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const double va = L[(2 * v) * 27 + q * 9 + t], de = L[(2 * v + 1) * 27 + q * 9 + t];
#pragma unroll
      for (int i = 0; i < 3; ++i) r[i][v] = fma(val(q, i), va, fma(der(q, i), de, r[i][v]));
    }
  }
  wave_lds_fence();
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int v = 0; v < V; ++v) L[vtk[i] * V + v] = r[i][v];
  sums.stage(s_plan);
  __syncthreads();
  sums.store(s_plan, s_r, part);
}

// ------------------------------------------------------------------ gather
// AP_STORE adds a.rhs where it is given (the residual's constant loads).
// AP_PQ and AP_CHEBZ run at most kPatchDotBlocks blocks (one partial each) of kDotThreads threads, which
// still fill the chip; the others one thread per dof.
constexpr int kDotThreads = 512;

// sum of the partials of dof idx
template <int V>
__device__ inline double patch_sum(int64_t idx, int2 inc, const int32_t* __restrict__ inc_idx,
                                   const double* __restrict__ part) {
  const int v = (int)(idx % V);
  double t = 0.0;
  for (int k = inc.x; k < inc.y; ++k) t += part[(int64_t)inc_idx[k] * V + v];
  return t;
}
template <int V>
__device__ inline int2 patch_inc(int64_t idx, const int32_t* __restrict__ inc_ptr) {
  return make_int2(inc_ptr[idx / V], inc_ptr[idx / V + 1]);
}

// the dofs of a block: one contiguous range, in the order of the patches
__device__ inline void patch_range(int64_t n, int64_t* begin, int64_t* end) {
  const int lb = xcd_logical_block(blockIdx.x, gridDim.x);
  const int64_t per = ((n + gridDim.x - 1) / gridDim.x + blockDim.x - 1) / blockDim.x * blockDim.x;
  *begin = (int64_t)lb * per;
  *end = min(n, *begin + per);
}

constexpr bool has_dot(int mode) { return mode == AP_PQ || mode == AP_CHEBZ; }

template <int V, int MODE0, typename TX, typename TY>
__global__ __launch_bounds__(has_dot(MODE0) ? kDotThreads : 256) void k_patch_gather(int64_t n, const int32_t* __restrict__ inc_ptr,
                                                      const int32_t* __restrict__ inc_idx,
                                                      const double* __restrict__ part,
                                                      const uint8_t* __restrict__ mask, ApplyArgsT<TX, TY> a) {
  constexpr int MODE = MODE0 == AP_CHEBZ ? AP_CHEB : MODE0, NT = has_dot(MODE0) ? kDotThreads : 256;
  __shared__ double red[NT / 64];
  const int32_t done = a.done ? *a.done : 0;  // looked at once the first loads are on their way
  double pq = 0.0;
  int64_t begin, end;
  patch_range(n, &begin, &end);
  for (int64_t idx = begin + threadIdx.x; idx < end; idx += NT) {
    EpiOperands e = epilogue_load<MODE>(a, idx);
    if (MODE == AP_PQ) e.x = double(a.x[idx]);
    if (MODE == AP_STORE && a.rhs) e.rhs = a.rhs[idx];
    const bool fixed = mask && mask[idx];
    const int2 inc = patch_inc<V>(idx, inc_ptr);
    if (done) break;
    double t = patch_sum<V>(idx, inc, inc_idx, part);
    if (fixed) t = double(a.x[idx]);
    if (MODE == AP_STORE) t += e.rhs;
    const double y = epilogue_store<MODE>(a, idx, t, e);
    if (has_dot(MODE0)) pq = fma(MODE == AP_PQ ? e.x : e.rhs, y, pq);
  }
  if (has_dot(MODE0) && !done) {
    pq = block_sum<NT>(pq, red);
    if (threadIdx.x == 0) a.part[blockIdx.x] = pq;
  }
}

// The gather of a CG product: p_new = z + beta p_old (as the cells' pass formed it), q, <p, q>.
// (p_old and p_new may be one vector: an entry is read and written by one thread)
template <int V, typename T, typename SC>
__global__ __launch_bounds__(kDotThreads) void k_patch_gather_cg(
    int64_t n, const int32_t* __restrict__ inc_ptr, const int32_t* __restrict__ inc_idx,
    const double* __restrict__ part, const uint8_t* __restrict__ mask, const SC* __restrict__ sc,
    const T* __restrict__ z, const T* p_old, T* p_new, T* __restrict__ q,
    double* __restrict__ pq_part) {
  __shared__ double red[kDotThreads / 64];
  const int32_t done = sc->done;  // (as above)
  const T beta = T(sc->beta);
  double pq = 0.0;
  int64_t begin, end;
  patch_range(n, &begin, &end);
  for (int64_t idx = begin + threadIdx.x; idx < end; idx += kDotThreads) {
    const T po = p_old[idx], zi = z[idx];
    const bool fixed = mask && mask[idx];
    const int2 inc = patch_inc<V>(idx, inc_ptr);
    if (done) return;
    const T p = fma(beta, po, zi);
    const double t = patch_sum<V>(idx, inc, inc_idx, part);
    const T qi = fixed ? p : T(t);
    p_new[idx] = p;
    q[idx] = qi;
    pq = fma(double(p), double(qi), pq);
  }
  if (done) return;
  pq = block_sum<kDotThreads>(pq, red);
  if (threadIdx.x == 0) pq_part[blockIdx.x] = pq;
}

// ---------------------------------------------------------------- dispatch
template <class F>
static int with_patch_law(const fem_patch_operator_t& op, fem_material_t* mat, F&& f) {
  *mat = *op.mat;
  const int vec = op.mesh->vec;
  switch (mat->kind) {
    case FEM_MAT_POISSON:
      if (vec == 1) return f(MatPoisson{});
      break;
    case FEM_MAT_LINEAR_ELASTIC:
      if (vec == 3) return f(MatElastic<false>{});
      break;
    case FEM_MAT_SIMP:
      if (vec != 3) break;
      if (op.modulus) {
        mat->param = op.modulus;
        return f(MatModulus{});
      }
      return f(MatElastic<true>{});
    case FEM_MAT_NEO_HOOKEAN:
      if (vec == 3) return f(MatNeoHookean{});
      break;
    default:
      break;
  }
  set_error("patch product: material kind %d (vec=%d) is not covered", mat->kind, vec);
  return FEM_ERR_BAD_ARG;
}

bool patch_operator_ok(const fem_patch_operator_t* op, bool residual) {
  if (!op || !op->mesh || !op->mat || !op->plan || !op->partials) return false;
  const fem_mesh_t& m = *op->mesh;
  const fem_patch_plan_t& p = *op->plan;
  const int cpp = fem_patch_cells(&m);
  if (cpp <= 0 || m.num_cells <= 0 || m.num_nodes <= 0) return false;
  if (p.cells_per_patch != cpp || p.num_patches != ceil_div(m.num_cells, cpp)) return false;
  if (!m.cells || ((uintptr_t)m.cells & 15) || !m.points || !m.quad_weights) return false;  // 16-byte node id loads
  if (!p.slot_ptr || !p.slot_end || !p.contrib || !p.inc_ptr || !p.inc_idx) return false;
  const fem_material_t& t = *op->mat;
  if (t.has_param && !t.param) return false;
  switch (t.kind) {
    case FEM_MAT_POISSON: return m.vec == 1;
    case FEM_MAT_LINEAR_ELASTIC: return m.vec == 3;
    case FEM_MAT_SIMP: return m.vec == 3 && t.has_param;
    case FEM_MAT_NEO_HOOKEAN: return m.vec == 3 && op->u && (residual || m.nodes_per_cell == 8);
    default: return false;
  }
}

// the cells' pass: partials of the internal force (MODE 0) or of the tangent product (MODE 1)
template <int MODE, typename TX, typename HEAD>
static int patch_cells(const fem_patch_operator_t& op, const PatchField<TX, HEAD>& field, hipStream_t s) {
  fem_material_t mat;
  const fem_mesh_t& m = *op.mesh;
  return with_patch_law(op, &mat, [&](auto tag) -> int {
    using MAT = decltype(tag);
    if (m.nodes_per_cell == 27) {
      if constexpr (MODE == 0 || !MAT::kNeedsU) {
        hipLaunchKernelGGL((k_patch_hex27<MAT, MODE, TX, HEAD>), dim3((unsigned)op.plan->num_patches), dim3(256), 0, s,
                           m, mat, *op.plan, field, op.partials);
        FEM_LAUNCHED();
      }
      return FEM_OK;
    }
    hipLaunchKernelGGL((k_patch_hex8<MAT, MODE, TX, HEAD>), dim3((unsigned)op.plan->num_patches), dim3(2 * kPatchCells),
                       0, s, m, mat, *op.plan, op.u, field, op.partials);
    FEM_LAUNCHED();
    return FEM_OK;
  });
}

template <int MODE, typename TX, typename TY>
static int patch_gather(const fem_patch_operator_t& op, const uint8_t* mask, const ApplyArgsT<TX, TY>& a, hipStream_t s,
                        int* parts) {
  const int64_t n = op.mesh->num_nodes * op.mesh->vec;
  constexpr int NT = has_dot(MODE) ? kDotThreads : 256;
  const int64_t want = ceil_div(n, NT);
  const unsigned grid = (unsigned)(has_dot(MODE) ? std::min<int64_t>(want, kPatchDotBlocks) : want);
  if (parts) *parts = (int)grid;
  if (op.mesh->vec == 3)
    hipLaunchKernelGGL((k_patch_gather<3, MODE, TX, TY>), dim3(grid), dim3(NT), 0, s, n, op.plan->inc_ptr,
                       op.plan->inc_idx, op.partials, mask, a);
  else
    hipLaunchKernelGGL((k_patch_gather<1, MODE, TX, TY>), dim3(grid), dim3(NT), 0, s, n, op.plan->inc_ptr,
                       op.plan->inc_idx, op.partials, mask, a);
  FEM_LAUNCHED();
  return FEM_OK;
}

template <int MODE, typename TX, typename TY>
int patch_apply(const fem_patch_operator_t& op, const ApplyArgsT<TX, TY>& a, hipStream_t s, int* parts) {
  if (int rc = patch_cells<1>(op, PatchField<TX, NoHead>{a.x, nullptr, NoHead{a.done}}, s)) return rc;
  return patch_gather<MODE, TX, TY>(op, op.bc_mask, a, s, parts);
}

inline const PcgScalars* head_scalars(const PcgHead& h) { return h.next; }
inline const AmgScalars* head_scalars(const CgHead& h) { return h.sc; }

template <typename HEAD, typename T>
int patch_pcg_product(const fem_patch_operator_t& op, const HEAD& head, const T* z, const T* p_old, T* p_new, T* q,
                      double* part, hipStream_t s, int* parts) {
  if (int rc = patch_cells<1>(op, PatchField<T, HEAD>{p_old, z, head}, s)) return rc;
  const int64_t n = op.mesh->num_nodes * op.mesh->vec;
  *parts = (int)std::min<int64_t>(ceil_div(n, kDotThreads), kPatchDotBlocks);
  auto go = [&](auto vc) {
    constexpr int V = decltype(vc)::value;
    using S = typename std::remove_pointer<decltype(head_scalars(head))>::type;
    hipLaunchKernelGGL((k_patch_gather_cg<V, T, S>), dim3((unsigned)*parts), dim3(kDotThreads), 0, s, n,
                       op.plan->inc_ptr, op.plan->inc_idx, op.partials, op.bc_mask, head_scalars(head), z,
                       p_old, p_new, q, part);
  };
  if (op.mesh->vec == 3)
    go(std::integral_constant<int, 3>{});
  else
    go(std::integral_constant<int, 1>{});
  FEM_LAUNCHED();
  return FEM_OK;
}

template int patch_pcg_product(const fem_patch_operator_t&, const PcgHead&, const double*, const double*, double*,
                               double*, double*, hipStream_t, int*);
template int patch_pcg_product(const fem_patch_operator_t&, const PcgHead&, const float*, const float*, float*, float*,
                               double*, hipStream_t, int*);
template int patch_pcg_product(const fem_patch_operator_t&, const CgHead&, const double*, const double*, double*,
                               double*, double*, hipStream_t, int*);

template int patch_apply<AP_STORE, double, double>(const fem_patch_operator_t&, const ApplyArgsT<double, double>&,
                                                   hipStream_t, int*);
template int patch_apply<AP_RESID, double, double>(const fem_patch_operator_t&, const ApplyArgsT<double, double>&,
                                                   hipStream_t, int*);
template int patch_apply<AP_CHEB, double, double>(const fem_patch_operator_t&, const ApplyArgsT<double, double>&,
                                                  hipStream_t, int*);
template int patch_apply<AP_CHEBZ, double, double>(const fem_patch_operator_t&, const ApplyArgsT<double, double>&,
                                                   hipStream_t, int*);
template int patch_apply<AP_DSTORE, double, double>(const fem_patch_operator_t&, const ApplyArgsT<double, double>&,
                                                    hipStream_t, int*);
template int patch_apply<AP_PQ, double, double>(const fem_patch_operator_t&, const ApplyArgsT<double, double>&,
                                                hipStream_t, int*);
template int patch_apply<AP_PQ, float, float>(const fem_patch_operator_t&, const ApplyArgsT<float, float>&,
                                              hipStream_t, int*);

// E of every point of a SIMP law: the power is taken once per tangent, not once per product
__global__ __launch_bounds__(256) void k_modulus(int64_t n, fem_material_t mat, double* __restrict__ out) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) out[i] = MatElastic<true>::modulus(mat, mat.param[i]);
}

static int check_patch_mesh(const fem_mesh_t* m) {
  FEM_CHECK_ARG(m && m->cells && m->num_cells > 0 && m->num_nodes > 0, "patch plan: mesh descriptor incomplete");
  FEM_CHECK_ARG(fem_patch_cells(m) > 0,
                "patch plan: covers HEX8 cells with the 2x2x2 and HEX27 cells with the 3x3x3 Gauss rule (got %d nodes, "
                "%d points)", m->nodes_per_cell, m->num_quads);
  return FEM_OK;
}

}  // namespace fem

using namespace fem;

extern "C" {

int fem_patch_cells(const fem_mesh_t* mesh) {
  if (!mesh) return 0;
  if (mesh->nodes_per_cell == 8 && mesh->num_quads == 8) return kPatchCells;
  return mesh->nodes_per_cell == 27 && mesh->num_quads == 27 ? kPatchCells27 : 0;
}

int fem_patch_counts(const fem_mesh_t* mesh, int32_t* counts, void* stream) {
  if (int rc = check_patch_mesh(mesh)) return rc;
  FEM_CHECK_ARG(counts, "fem_patch_counts: NULL argument");
  const int cpp = fem_patch_cells(mesh);
  hipLaunchKernelGGL(k_patch_nodes<false>, dim3((unsigned)ceil_div(mesh->num_cells, cpp)), dim3(256), 0,
                     as_stream(stream), mesh->num_cells, mesh->nodes_per_cell, cpp, mesh->cells, counts,
                     (const int32_t*)nullptr, (int32_t*)nullptr, (uint16_t*)nullptr, (uint16_t*)nullptr);
  FEM_LAUNCHED();
  return FEM_OK;
}

int fem_patch_fill(const fem_mesh_t* mesh, const int32_t* slot_ptr, int32_t* slot_node, uint16_t* slot_end,
                   uint16_t* contrib, void* stream) {
  if (int rc = check_patch_mesh(mesh)) return rc;
  FEM_CHECK_ARG(slot_ptr && slot_node && slot_end && contrib, "fem_patch_fill: NULL argument");
  const int cpp = fem_patch_cells(mesh);
  hipLaunchKernelGGL(k_patch_nodes<true>, dim3((unsigned)ceil_div(mesh->num_cells, cpp)), dim3(256), 0,
                     as_stream(stream), mesh->num_cells, mesh->nodes_per_cell, cpp, mesh->cells, (int32_t*)nullptr,
                     slot_ptr, slot_node, slot_end, contrib);
  FEM_LAUNCHED();
  return FEM_OK;
}

int fem_patch_modulus(const fem_mesh_t* mesh, const fem_material_t* mat, double* modulus, void* stream) {
  FEM_CHECK_ARG(mesh && mat && modulus && mat->kind == FEM_MAT_SIMP && mat->has_param && mat->param,
                "fem_patch_modulus: needs a SIMP law with its parameter");
  const int64_t n = mesh->num_cells * mesh->num_quads;
  if (n == 0) return FEM_OK;
  hipLaunchKernelGGL(k_modulus, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, as_stream(stream), n, *mat, modulus);
  FEM_LAUNCHED();
  return FEM_OK;
}

int fem_patch_apply(const fem_patch_operator_t* op, const double* x, double* y, void* stream) {
  FEM_CHECK_ARG(patch_operator_ok(op) && x && y, "fem_patch_apply: the operator is incomplete or not covered");
  ApplyArgs a{x, y, nullptr, nullptr, nullptr, 0.0, 0.0, nullptr, nullptr};
  return patch_apply<AP_STORE, double, double>(*op, a, as_stream(stream));
}

int fem_patch_residual(const fem_patch_operator_t* op, const double* u, const double* base, double* res,
                       void* stream) {
  FEM_CHECK_ARG(op && u && res, "fem_patch_residual: NULL argument");
  fem_patch_operator_t o = *op;
  o.u = u;
  FEM_CHECK_ARG(patch_operator_ok(&o, true), "fem_patch_residual: the operator is incomplete or not covered");
  hipStream_t s = as_stream(stream);
  if (int rc = patch_cells<0>(o, PatchField<double, NoHead>{u, nullptr, NoHead{nullptr}}, s)) return rc;
  ApplyArgs a{u, res, base, nullptr, nullptr, 0.0, 0.0, nullptr, nullptr};
  return patch_gather<AP_STORE, double, double>(o, nullptr, a, s, nullptr);
}

}  // extern "C"
