// Per-cell staging shared by the element kernels: configuration, LDS cell
// state, geometry staging (Jacobian, inverse, physical gradients, JxW) and
// the reference tables.
#pragma once
#include "materials.hpp"

namespace fem {

// Q is the number of quadrature points staged at a time: kernels walk the
// mesh's num_quads points in chunks of Q (one chunk when they are equal), so
// any quadrature order runs with the LDS footprint of Q points.
template <int N_, int Q_>
struct ElemCfg {
  static constexpr int N = N_;
  static constexpr int Q = Q_;
  static constexpr int TPC = (N_ * N_ <= 64) ? 64 : 256;  // threads per cell
  static constexpr int CPW = 256 / TPC;                   // cells per workgroup
};

// LDS state of one cell: coordinates, (inverse) Jacobians and JxW; with the physical gradients.
template <int N, int Q, typename T>
struct JacLds {
  double xd[N][3];
  T invJ[Q][9];
  T jxw[Q];
};
template <int N, int Q, typename T>
struct CellLds : JacLds<N, Q, T> {
  T g[Q][N][3];
};

// Reference gradients r[q][i][j] = sum_a f[a][i] dN_a/dxi_j of a nodal field in LDS, one lane per
// entry (q, i, j): a serial sum of N products, where a lane per point had 3 V of them one after
// the other and left nine lanes of ten idle.
template <int N, int Q, int TPC, int V, typename T, typename TF>
__device__ inline void ref_grads(const T (&dN)[Q][N][3], const TF (*f)[V], int qn, int t, T* r) {
  for (int it = t; it < qn * V * 3; it += TPC) {
    const int q = it / (V * 3), i = (it / 3) % V, j = it % 3;
    T s = T(0);
#pragma unroll
    for (int a = 0; a < N; ++a) s += f[a][i] * dN[q][a][j];
    r[it] = s;
  }
}

// Stage the node numbers and coordinates of cell c and the inverse Jacobians and JxW of the
// first qn (default Q) staged quadrature points.
// Must be called by all threads of the workgroup (contains barriers).
template <int N, int Q, int TPC, typename T>
__device__ inline void stage_jacobian(const fem_mesh_t& mesh, int64_t c, bool active, int t,
                                      const T (&dN)[Q][N][3], const double (&w)[Q], JacLds<N, Q, T>& L,
                                      int32_t (&node)[N], int qn = Q) {
  if (active && t < N) {
    const int32_t n = mesh.cells[c * N + t];
    node[t] = n;
    L.xd[t][0] = mesh.points[(int64_t)n * 3 + 0];
    L.xd[t][1] = mesh.points[(int64_t)n * 3 + 1];
    L.xd[t][2] = mesh.points[(int64_t)n * 3 + 2];
  }
  __syncthreads();
  if (active)
    for (int it = t; it < qn * 9; it += TPC) {
      const int q = it / 9, i = (it / 3) % 3, j = it % 3;
      const double x0 = L.xd[0][i];
      T s = T(0);
#pragma unroll
      for (int a = 1; a < N; ++a) s += T(L.xd[a][i] - x0) * dN[q][a][j];
      L.invJ[q][i * 3 + j] = s;
    }
  __syncthreads();
  if (active)
    for (int q = t; q < qn; q += TPC) {
      T J[9], iJ[9];
#pragma unroll
      for (int k = 0; k < 9; ++k) J[k] = L.invJ[q][k];
      const T det = det3(J);
      inv3(J, det, iJ);
#pragma unroll
      for (int k = 0; k < 9; ++k) L.invJ[q][k] = iJ[k];
      L.jxw[q] = det * T(w[q]);
    }
  __syncthreads();
}

// stage_jacobian and the physical gradients.
template <int N, int Q, int TPC, typename T>
__device__ inline void stage_geometry(const fem_mesh_t& mesh, int64_t c, bool active, int t,
                                      const T (&dN)[Q][N][3], const double (&w)[Q], CellLds<N, Q, T>& L,
                                      int32_t (&node)[N], int qn = Q) {
  stage_jacobian<N, Q, TPC, T>(mesh, c, active, t, dN, w, L, node, qn);
  if (active) {
    for (int it = t; it < qn * N; it += TPC) {
      const int q = it / N, a = it % N;
      const T* iJ = L.invJ[q];
      const T d0 = dN[q][a][0], d1 = dN[q][a][1], d2 = dN[q][a][2];
#pragma unroll
      for (int j = 0; j < 3; ++j) L.g[q][a][j] = d0 * iJ[0 * 3 + j] + d1 * iJ[1 * 3 + j] + d2 * iJ[2 * 3 + j];
    }
  }
  __syncthreads();
}

template <int N, int Q, typename T>
__device__ inline void load_tables(const fem_mesh_t& mesh, T (&dN)[Q][N][3], double (&w)[Q]) {
  T* flat = &dN[0][0][0];
  for (int i = threadIdx.x; i < Q * N * 3; i += blockDim.x) flat[i] = T(mesh.shape_grads_ref[i]);
  for (int i = threadIdx.x; i < Q; i += blockDim.x) w[i] = mesh.quad_weights[i];
}

// Reference gradients and weights of quadrature points q0 .. q0 + qn - 1 (qn <= Q).
template <int N, int Q, typename T>
__device__ inline void load_tables_chunk(const fem_mesh_t& mesh, int q0, int qn, T (&dN)[Q][N][3], double (&w)[Q]) {
  T* flat = &dN[0][0][0];
  const double* src = mesh.shape_grads_ref + (size_t)q0 * N * 3;
  for (int i = threadIdx.x; i < qn * N * 3; i += blockDim.x) flat[i] = T(src[i]);
  for (int i = threadIdx.x; i < qn; i += blockDim.x) w[i] = mesh.quad_weights[q0 + i];
}

// grad f at quad q from nodal values f[N][V] (LDS)
template <int N, int Q, int V, typename T>
__device__ inline void quad_grad(const CellLds<N, Q, T>& L, const T (&f)[N][V], int q, T (&G)[V][3]) {
#pragma unroll
  for (int i = 0; i < V; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) G[i][j] = T(0);
  for (int a = 0; a < N; ++a) {
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const T fa = f[a][i];
#pragma unroll
      for (int j = 0; j < 3; ++j) G[i][j] += fa * L.g[q][a][j];
    }
  }
}

}  // namespace fem
