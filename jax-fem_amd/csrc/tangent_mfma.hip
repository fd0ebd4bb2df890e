// HEX27 tangents of the isotropic elastic laws on the matrix cores.
//
// Replaces the per-cell jacfwd of jax-fem (problem.py:262-266) for
// LINEAR_ELASTIC and SIMP materials on 27-node cells with 27 quadrature
// points.  With X[q][(a,i)] = dN_a/dx_i at quad q (27 x 81) and
// W_q = JxW_q E_q, all of the 81 x 81 cell tangent follows from one GEMM
//   Z = X^T diag(W) X                                  (81 x 81, inner dim 27)
// because lambda = c0 E and mu = c1 E share the modulus E:
//   K[(a,i),(b,k)] = c0 Z[(a,i),(b,k)] + c1 Z[(a,k),(b,i)]
//                  + delta_ik c1 (Z[(a,0),(b,0)] + Z[(a,1),(b,1)] + Z[(a,2),(b,2)]).
// Z is formed on MFMA in tiles of 15 x 15 (five nodes by five: whole 3 x 3 blocks in a 16 x 16
// result) and is symmetric, so the 21 tile pairs of the upper triangle are shared out over the
// four waves; a wave stages its tile in LDS of its own and writes the blocks of Ke[c][a][b][i][k]
// and, off the diagonal, their transposes, 45 consecutive values at a time.  Operand layouts:
// A[i][k] in lane i + 16 k (f64; for bf16 the four
// k of one lane are k = 4 (lane / 16) + e), B[k][j] in lane j + 16 k; the two
// instructions place the 16 x 16 result differently (see the stores).  Two arithmetic modes:
//   FP64 : v_mfma_f64_16x16x4f64, exact FP64 products and sums.
//   BF16x3: each operand split x = hi + lo (hi = bf16(x), lo = bf16(x - hi));
//          hi*hi + hi*lo + lo*hi on v_mfma_f32_16x16x16bf16_1k with FP32
//          accumulation (about 16 significant bits per product); Ke in FP32.
// One workgroup of 4 waves per cell, persistent over cells.  46 KB of LDS, so three of them share
// a CU and one's Jacobians run beside another's products and stores; with all of Z in LDS (91 KB)
// there was one, which waited for each phase in turn: 24^3 cells 940 -> 350 us (726 MB written, 115 us).
#include "element.hpp"
#include "tangent_mfma.hpp"

#include <algorithm>
#include <type_traits>

namespace fem {

namespace {

constexpr int kN = 27, kQ = 27, kM = 81;
constexpr int kTN = 5, kTiles = 6;  // nodes per tile; 27 nodes padded to 6 tiles
constexpr int kZS = 3 * kTN + 2;    // row stride of a staged tile (its entries number below 256)
constexpr int kEntries = (kTN * kTN * 9 + 63) / 64;
constexpr uint32_t kDiag = 1u << 24;
constexpr int kGrid = 768;          // persistent workgroups: three per CU

typedef double double4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef short short4_t __attribute__((ext_vector_type(4)));

// round-to-nearest-even FP32 -> BF16 (finite inputs)
__device__ inline unsigned short bf16_bits(float x) {
  unsigned int b = __float_as_uint(x);
  b += 0x7FFFu + ((b >> 16) & 1u);
  return (unsigned short)(b >> 16);
}
__device__ inline float bf16_value(unsigned short h) { return __uint_as_float((unsigned int)h << 16); }

struct Hex27Lds {
  double dN[kQ][kN][3];
  double w[kQ];
  double W[kQ];
  CellLds<kN, kQ, double> cell;
  int32_t node[kN];
};

}  // namespace

template <bool kSimp, bool kBf16, typename TO>
__global__ __launch_bounds__(256) void k_tangent_hex27_mfma(fem_mesh_t mesh, fem_material_t mat,
                                                            TO* __restrict__ Ke) {
  using TZ = typename std::conditional<kBf16, float, double>::type;
  __shared__ Hex27Lds S;
  __shared__ TZ s_z[4][3 * kTN][kZS];
  const int t = threadIdx.x;
  const int wave = t >> 6, lane = t & 63;
  load_tables(mesh, S.dN, S.w);
  const double c0 = mat.c[0], c1 = mat.c[1];
  TZ(*z)[kZS] = s_z[wave];
  // The lane's values of a tile, the same in every tile: where Z[(a,i),(b,k)], Z[(a,k),(b,i)] and the
  // block's trace stand, whether i = k, and (a, b) against the last tile's edge; off: the value's
  // place in Ke.  ent of the tile's blocks, entT of their transposes (45 values of a block row are
  // consecutive in either).  Taken apart again in every tile, the indices cost more than the MFMA.
  uint32_t ent[kEntries], entT[kEntries];
  int off[kEntries];
#pragma unroll
  for (int t = 0; t < kEntries; ++t) {
    const int e = lane + 64 * t, hi = e / (9 * kTN), lo = (e / 9) % kTN, i = (e % 9) / 3, k = e % 3;
    auto pack = [&](int a, int b, int i, int k) {
      return (uint32_t)((3 * a + i) * kZS + 3 * b + k) | (uint32_t)((3 * a + k) * kZS + 3 * b + i) << 8 |
             (uint32_t)(3 * a * kZS + 3 * b) << 16 | (i == k ? kDiag : 0u) | (uint32_t)a << 25 | (uint32_t)b << 28;
    };
    const bool in = e < kTN * kTN * 9;
    ent[t] = in ? pack(hi, lo, i, k) : 7u << 25;    // a = 7: outside every tile
    entT[t] = in ? pack(lo, hi, k, i) : 7u << 25;
    off[t] = (hi * kN + lo) * 9 + e % 9;
  }
  const int l = lane & 15;  // row of A, column of B and of the result; 15 is padding
  for (int64_t c = blockIdx.x; c < mesh.num_cells; c += gridDim.x) {
    __syncthreads();  // the previous cell's gradients are no longer read
    stage_geometry<kN, kQ, 256, double>(mesh, c, true, t, S.dN, S.w, S.cell, S.node);
    if (t < kQ) {
      const double E = kSimp ? MatElastic<true>::modulus(mat, mat.param[c * kQ + t]) : 1.0;
      S.W[t] = S.cell.jxw[t] * E;
    }
    __syncthreads();
    const double(*g)[kN][3] = S.cell.g;
    TO* out = Ke + (size_t)c * kM * kM;
    // pair p of the upper triangle (row by row): (tm, tn), tm <= tn
    for (int p = wave; p < kTiles * (kTiles + 1) / 2; p += 4) {
      int tm = 0, first = 0;
      while (p >= first + kTiles - tm) first += kTiles - tm++;
      const int tn = tm + (p - first);
      const int m = tm * 3 * kTN + l, n = tn * 3 * kTN + l;
      const bool om = l < 3 * kTN && m < kM, on = l < 3 * kTN && n < kM;
      if (!kBf16) {
        double4_t acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int kk = 0; kk < 7; ++kk) {          // inner dim 27 padded to 28
          const int q = kk * 4 + (lane >> 4);
          const double a = (q < kQ && om) ? S.W[q] * g[q][m / 3][m % 3] : 0.0;
          const double b = (q < kQ && on) ? g[q][n / 3][n % 3] : 0.0;
          acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
        }
        // f64 16x16x4 result: D[i][j] in lane j + 16 (i % 4), register i / 4
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = (lane >> 4) + 4 * r;
          if (row < 3 * kTN && l < 3 * kTN) z[row][l] = TZ(acc[r]);
        }
      } else {
        float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {          // inner dim 27 padded to 32
          short4_t ahi, alo, bhi, blo;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int q = kk * 16 + 4 * (lane >> 4) + e;
            const float a = (q < kQ && om) ? float(S.W[q] * g[q][m / 3][m % 3]) : 0.f;
            const float b = (q < kQ && on) ? float(g[q][n / 3][n % 3]) : 0.f;
            const unsigned short ah = bf16_bits(a), bh = bf16_bits(b);
            ahi[e] = (short)ah;
            alo[e] = (short)bf16_bits(a - bf16_value(ah));
            bhi[e] = (short)bh;
            blo[e] = (short)bf16_bits(b - bf16_value(bh));
          }
          acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ahi, bhi, acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ahi, blo, acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(alo, bhi, acc, 0, 0, 0);
        }
        // bf16 16x16x16 result: D[i][j] in lane j + 16 (i / 4), register i % 4
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = 4 * (lane >> 4) + r;
          if (row < 3 * kTN && l < 3 * kTN) z[row][l] = TZ(acc[r]);
        }
      }
      // (the hardware executes a wave's LDS accesses in order; the fences keep the compiler's)
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      const int a0 = tm * kTN, b0 = tn * kTN;
      const int na = min(kTN, kN - a0), nb = min(kTN, kN - b0);
      const TZ* zf = &z[0][0];
      auto emit = [&](uint32_t e, TO* o) {
        double v = c0 * double(zf[e & 255u]) + c1 * double(zf[(e >> 8) & 255u]);
        const TZ* d = zf + ((e >> 16) & 255u);
        const double tr = double(d[0]) + double(d[kZS + 1]) + double(d[2 * kZS + 2]);
        if (e & kDiag) v += c1 * tr;
        *o = TO(v);
      };
#pragma unroll
      for (int t = 0; t < kEntries; ++t) {
        const int a = (ent[t] >> 25) & 7, b = (int)(ent[t] >> 28) & 7;
        if (a < na && b < nb) emit(ent[t], out + (a0 * kN + b0) * 9 + off[t]);
      }
      if (tm != tn)
#pragma unroll
        for (int t = 0; t < kEntries; ++t) {
          const int a = (entT[t] >> 25) & 7, b = (int)(entT[t] >> 28) & 7;
          if (a < na && b < nb) emit(entT[t], out + (b0 * kN + a0) * 9 + off[t]);
        }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }
}

bool hex27_tangent_mfma_applies(const fem_mesh_t& mesh, const fem_material_t& mat) {
  return mesh.nodes_per_cell == kN && mesh.num_quads == kQ && mesh.vec == 3 &&
         (mat.kind == FEM_MAT_LINEAR_ELASTIC || (mat.kind == FEM_MAT_SIMP && mat.has_param));
}

int hex27_tangent_mfma(const fem_mesh_t& mesh, const fem_material_t& mat, int precision, void* Ke, hipStream_t s) {
  const unsigned grid = (unsigned)std::min<int64_t>(mesh.num_cells, kGrid);
  const bool simp = mat.kind == FEM_MAT_SIMP;
  if (precision == FEM_F64) {
    if (simp)
      hipLaunchKernelGGL((k_tangent_hex27_mfma<true, false, double>), dim3(grid), dim3(256), 0, s, mesh, mat,
                         (double*)Ke);
    else
      hipLaunchKernelGGL((k_tangent_hex27_mfma<false, false, double>), dim3(grid), dim3(256), 0, s, mesh, mat,
                         (double*)Ke);
  } else {
    if (simp)
      hipLaunchKernelGGL((k_tangent_hex27_mfma<true, true, float>), dim3(grid), dim3(256), 0, s, mesh, mat,
                         (float*)Ke);
    else
      hipLaunchKernelGGL((k_tangent_hex27_mfma<false, true, float>), dim3(grid), dim3(256), 0, s, mesh, mat,
                         (float*)Ke);
  }
  FEM_LAUNCHED();
  return FEM_OK;
}

}  // namespace fem
