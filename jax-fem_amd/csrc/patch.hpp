// Matrix-free element products over patches of consecutive cells (patch.hip):
// the entry points the solvers call.
#pragma once
#include "apply.hpp"
#include "pcg_scalars.hpp"

namespace fem {

constexpr int kPatchDotBlocks = 1024;  // most <x, A x> partials of an AP_PQ product

// True when `op` describes an element, rule and law whose tangent (or residual) the patch kernels run.
bool patch_operator_ok(const fem_patch_operator_t* op, bool residual = false);

// y = epilogue(A x), A the tangent at op->u with identity rows on op->bc_mask; *parts
// receives the number of partials an AP_PQ or AP_CHEBZ product writes to a.part.  TX / TY: FP64, or
// FP32 vectors (the arithmetic is FP64).
template <int MODE, typename TX, typename TY>
int patch_apply(const fem_patch_operator_t& op, const ApplyArgsT<TX, TY>& a, hipStream_t s, int* parts = nullptr);

// One CG product: begins the iteration (HEAD: PcgHead or CgHead), p_new = z + beta p_old (p_new may
// be p_old), q = A p_new and the *parts partials of <p_new, q> in part.
template <typename HEAD, typename T>
int patch_pcg_product(const fem_patch_operator_t& op, const HEAD& head, const T* z, const T* p_old, T* p_new, T* q,
                      double* part, hipStream_t s, int* parts);

}  // namespace fem
