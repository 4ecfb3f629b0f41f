"""Wide banded matrices on column tiles, walked by groups of workgroups whose waves take batches in turn: items of less batches
than a workgroup has waves, of whole batches and of a last one cut short, in every width and number of K slices, against 64 bits."""
import pytest
import torch

from sddmm_gpu_amd import capi, synth

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("K", [32, 50, 64, 128, 256])
@pytest.mark.parametrize("n_rows,per_row,half_band", [(400000, 1, 900), (350000, 3, 500), (370001, 9, 1500)])
def test_bands(n_rows, per_row, half_band, K):
    d = synth.banded(n_rows, per_row, half_band, K=K, seed=K + per_row, device=DEV)
    nnz = d["nnz"]
    plan = capi.Plan.from_device_csr(n_rows, n_rows, nnz, d["row_ptr"].data_ptr(), d["col_ind"].data_ptr(), K,
                                     options=capi.PlanOptions.defaults(kernel=capi.KERNEL_LDS_TILE, tile_runs=2, ignore_env=1))
    rows, cols = d["row_ind"].long(), d["col_ind"].long()
    W, H, val = d["W"], d["H"], d["val"]
    out = torch.full((nnz + 1,), 7.0, device=DEV)
    stream = torch.cuda.current_stream().cuda_stream
    for given in (False, True):
        if given:
            plan.set_values(val.data_ptr(), stream)
        out.fill_(7.0)
        plan.execute(0 if given else val.data_ptr(), W.data_ptr(), H.data_ptr(), out.data_ptr(), stream)
        torch.cuda.synchronize()
        assert float(out[nnz]) == 7.0
        for b in range(0, nnz, 1 << 19):
            s = slice(b, min(nnz, b + (1 << 19)))
            p = W[rows[s]].double() * H[cols[s]].double() * val[s].double()[:, None]
            # a rounding per product and sum, a few per K slice, and the scaling
            assert bool(((out[s].double() - p.sum(1)).abs() <= (K + 16) * 2.0 ** -24 * p.abs().sum(1)).all())
