// Plan-free SDDMM over a device CSR that allocates no memory and keeps none: the row-gather kernel in one
// launch, or one per slice of K (gather_slice), finding the rows of its nonzeros from the row pointers.
#include <hip/hip_runtime.h>
#include "internal.hpp"
#include "kernels.hpp"
#include "launch.hpp"

using namespace sddmm;

extern "C" int sddmm_csr_noalloc(int64_t n_rows, int64_t n_cols, int64_t nnz, const int32_t *d_row_ptr,
                                 const int32_t *d_col_ind, const float *d_val, int32_t K, const float *d_W,
                                 const float *d_H, float *d_out, void *stream)
{
    if (n_rows < 0 || n_cols < 0 || nnz < 0 || K < 1) return fail(SDDMM_ERR_ARG, "sddmm_csr_noalloc: negative size or K < 1");
    if (nnz > (int64_t)SDDMM_NOALLOC_MAX_NNZ)
        return fail(SDDMM_ERR_RANGE, "sddmm_csr_noalloc: nnz = %lld exceeds the limit of %lld nonzeros",
                    (long long)nnz, (long long)(int64_t)SDDMM_NOALLOC_MAX_NNZ);
    if (n_rows >= INT32_MAX || n_cols >= INT32_MAX) return fail(SDDMM_ERR_RANGE, "sddmm_csr_noalloc: sizes beyond int32 offsets");
    if (nnz == 0) return SDDMM_OK;
    if (n_rows == 0 || n_cols == 0) return fail(SDDMM_ERR_ARG, "sddmm_csr_noalloc: %lld nonzeros in an empty matrix", (long long)nnz);
    if (!d_row_ptr || !d_col_ind || !d_W || !d_H || !d_out) return fail(SDDMM_ERR_ARG, "sddmm_csr_noalloc: NULL device pointer");
    if ((((uintptr_t)d_W | (uintptr_t)d_H) & 15u) && K % 4 == 0)
        return fail(SDDMM_ERR_ARG, "sddmm_csr_noalloc: W and H must be 16-byte aligned");

    KArgs a{};
    a.col_ind = d_col_ind; a.val = d_val; a.W = d_W; a.H = d_H; a.out = d_out;
    a.row_ptr = d_row_ptr; a.n_rows = (int32_t)n_rows;
    a.nnz = (int32_t)nnz; a.K = K; a.n_cols = (int32_t)n_cols; a.tile_x = (int32_t)n_cols;
    const bool wide = gather_wide(n_rows, n_cols, K);
    const int slice = gather_slice(nnz, n_cols, K);
    hipError_t e;
    if (slice < K) {
        e = launch_gather_slices(a, n_rows, n_rows, wide, slice, stream);
    } else {
        const GatherShape shape = gather_shape(nnz, n_rows, n_rows, K);
        const KernelFn fn = shape.v.G ? gather_kernel(shape.v, shape.once, wide) : generic_kernel();
        a.chunk = shape.chunk;
        const int grid = (int)((nnz + a.chunk - 1) / a.chunk);
        e = launch(fn, dim3((unsigned)grid), dim3(kRowGatherBlock), 0, (hipStream_t)stream, a);
    }
    if (e != hipSuccess) return fail(SDDMM_ERR_HIP, "sddmm_csr_noalloc: launch failed: %s", hipGetErrorString(e));
    return SDDMM_OK;
}
