"""The padded gather on groups of 4 positions (eight lanes, two rows of W at a time): streams that end inside a batch, with one
group or two in the last eight positions, padding flagged or repeated, one K slice or several (in one launch and one by one),
against 64-bit sums."""
import pytest
import torch

from sddmm_gpu_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,fuse", [(32, -1), (64, -1), (128, -1), (384, -1), (384, 0)])
@pytest.mark.parametrize("n_rows,n_cols,nnz", [(1, 5, 1), (2, 9, 7), (3, 40, 64), (17, 50, 130), (301, 97, 5003), (40, 3000, 9001)])
@pytest.mark.parametrize("sink,slab", [(1, 16), (0, 16), (1, 1 << 20)])
def test_against_64_bits(n_rows, n_cols, nnz, K, fuse, sink, slab):
    g = torch.Generator().manual_seed(nnz + K)
    keys = torch.randperm(n_rows * n_cols, generator=g)[:nnz].sort().values
    rows, cols = keys // n_cols, keys % n_cols
    nnz = keys.numel()
    row_ptr = torch.zeros(n_rows + 1, dtype=torch.int64)
    row_ptr[1:] = torch.cumsum(torch.bincount(rows, minlength=n_rows), 0)
    W, H, val = torch.randn(n_rows, K, generator=g), torch.randn(n_cols, K, generator=g), torch.rand(nnz, generator=g)
    p = W.double()[rows] * H.double()[cols]
    dot, size, v = p.sum(1), p.abs().sum(1), val.double()
    rp, ci, dW, dH, dv = (t.cuda() for t in (row_ptr.int(), cols.int(), W, H, val))
    plan = capi.Plan.from_device_csr(n_rows, n_cols, nnz, rp.data_ptr(), ci.data_ptr(), K,
                                     options=capi.PlanOptions.defaults(kernel=capi.KERNEL_ROW_GATHER, row_padded=1, gather_lanes=4, gather_sink=sink,
                                                                       k_slice=128 if K > 128 else 0, fuse_slices=fuse, gather_slab_cols=slab, ignore_env=1))
    assert plan.info()["padded_positions"] % 4 == 0 and plan.info()["padded_positions"] >= nnz
    assert plan.info()["n_launches"] == (3 if fuse == 0 else 1)
    stream = torch.cuda.current_stream().cuda_stream
    out = torch.full((nnz + 1,), 7.0, device="cuda")

    def check(run, ref, scale):
        out.fill_(7.0)
        run()
        torch.cuda.synchronize()
        # a rounding per product and sum, per K slice one more, and of the scaling
        assert bool(((out[:nnz].cpu().double() - ref).abs() <= (K + 8) * 2.0 ** -24 * scale + 1e-30).all()) and float(out[nnz]) == 7.0

    a = (dW.data_ptr(), dH.data_ptr(), out.data_ptr())
    check(lambda: plan.execute(0, *a, stream), dot, size)
    check(lambda: plan.execute(dv.data_ptr(), *a, stream), v * dot, v * size)
    check(lambda: plan.execute_epilogue(dv.data_ptr(), *a, capi.EPILOGUE_RESIDUAL, stream), v - dot, v + size)
    plan.set_values(dv.data_ptr(), stream)
    check(lambda: plan.execute(0, *a, stream), v * dot, v * size)
    check(lambda: plan.execute_epilogue(0, *a, capi.EPILOGUE_RESIDUAL, stream), v - dot, v + size)


# the K slices of a gathered class keep partial results in the plan like those of tiles: k_slice < K says so to its callers
@pytest.mark.parametrize("opts,kernel,launches", [(dict(fuse_slices=0), capi.KERNEL_AUTO, 3), (dict(fuse_slices=1), capi.KERNEL_AUTO, 1),
                                                  (dict(fuse_slices=0, row_padded=1), capi.KERNEL_ROW_GATHER, 3)])
def test_slices_are_reported(opts, kernel, launches):
    n, K = 200000, 384  # (factors of 307 MB: slabs)
    g = torch.Generator().manual_seed(5)
    cols = torch.randint(0, n // 2, (n, 2), generator=g)
    cols[:, 1] += n // 2
    rp, ci = torch.arange(0, 2 * n + 1, 2).int().cuda(), cols.reshape(-1).int().cuda()
    plan = capi.Plan.from_device_csr(n, n, 2 * n, rp.data_ptr(), ci.data_ptr(), K,
                                     options=capi.PlanOptions.defaults(kernel=kernel, short_row_max=1 << 20, ignore_env=1, **opts))
    info = plan.info()
    assert info["kernel"] == capi.KERNEL_ROW_GATHER and info["n_launches"] == launches and info["k_slice"] == 128, info
    assert plan.workspace_bytes() >= 4 * info["padded_positions"] >= 8 * n
