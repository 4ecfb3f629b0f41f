"""Wide banded matrices on column tiles, walked by groups of workgroups whose waves take batches in turn: items of less batches
than a workgroup has waves, of whole batches and of a last one cut short, in every width, K slices in one launch and one by one,
with every source of the values, against 64 bits."""
import pytest
import torch

from sddmm_gpu_amd import capi, synth

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("K,fuse", [(32, -1), (50, -1), (64, -1), (128, -1), (150, 0), (150, 1), (200, 0), (200, 1), (256, 0), (256, 1)])
@pytest.mark.parametrize("n_rows,per_row,half_band,tile_x", [(60000, 2, 150, 32), (350000, 3, 500, 0), (370001, 9, 1500, 0)])
def test_bands(n_rows, per_row, half_band, tile_x, K, fuse):
    d = synth.banded(n_rows, per_row, half_band, K=K, seed=K + per_row, device=DEV)
    nnz = d["nnz"]
    plan = capi.Plan.from_device_csr(n_rows, n_rows, nnz, d["row_ptr"].data_ptr(), d["col_ind"].data_ptr(), K,
                                     options=capi.PlanOptions.defaults(kernel=capi.KERNEL_LDS_TILE, tile_runs=2, tile_size_x=tile_x, fuse_slices=fuse, ignore_env=1))
    info = plan.info()
    assert info["n_row_panels"] > 1 and info["n_launches"] == (-(-K // 128) if fuse == 0 else 1), info  # (dealt out to groups of workgroups)
    if tile_x:  # most items are smaller than the 12 or 16 batches of 64 that would give every wave one
        assert info["padded_positions"] < 12 * 64 * info["n_col_tiles"], info
    rows, cols = d["row_ind"].long(), d["col_ind"].long()
    W, H, val = d["W"], d["H"], d["val"]
    dot, size = torch.empty(nnz, dtype=torch.float64, device=DEV), torch.empty(nnz, dtype=torch.float64, device=DEV)
    for b in range(0, nnz, 1 << 19):
        p = W[rows[b:b + (1 << 19)]].double() * H[cols[b:b + (1 << 19)]].double()
        dot[b:b + (1 << 19)] = p.sum(1)
        size[b:b + (1 << 19)] = p.abs().sum(1)
    out = torch.empty(nnz + 1, device=DEV)
    stream = torch.cuda.current_stream().cuda_stream

    def check(run, ref, scale):
        out.fill_(7.0)
        run()
        torch.cuda.synchronize()
        # a rounding per product and sum, a few per K slice, and the scaling
        assert float(out[nnz]) == 7.0 and bool(((out[:nnz].double() - ref).abs() <= (K + 16) * 2.0 ** -24 * scale).all())

    a, v = (W.data_ptr(), H.data_ptr(), out.data_ptr()), val.double()
    check(lambda: plan.execute(0, *a, stream), dot, size)
    check(lambda: plan.execute(val.data_ptr(), *a, stream), v * dot, v * size)
    check(lambda: plan.execute_epilogue(val.data_ptr(), *a, capi.EPILOGUE_RESIDUAL, stream), v - dot, v + size)
    plan.set_values(val.data_ptr(), stream)
    check(lambda: plan.execute(0, *a, stream), v * dot, v * size)
    check(lambda: plan.execute_epilogue(0, *a, capi.EPILOGUE_RESIDUAL, stream), v - dot, v + size)
