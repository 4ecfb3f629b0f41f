"""Plans whose H does not fit a die's L2 walk S in column slabs of a width that the planner chooses: against 64-bit sums,
with every source of the values, on both kinds of column popularity and with a last slab cut short."""
import pytest
import torch

from sddmm_gpu_amd import capi, synth

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("kind,K", [("uniform", 64), ("uniform", 128), ("uniform", 320), ("graph", 128), ("graph", 512)])
def test_slabs_chosen_by_the_planner(kind, K):
    if kind == "uniform":
        d = synth.uniform_random(3001, 100003, 0.002, K=K, seed=2, device=DEV)
    else:
        d = synth.rmat(17, 1500000, K=K, seed=2, device=DEV)
    nnz = d["nnz"]
    plan = capi.Plan.from_device_csr(d["n_rows"], d["n_cols"], nnz, d["row_ptr"].data_ptr(), d["col_ind"].data_ptr(), K,
                                     options=capi.PlanOptions.defaults(ignore_env=1))
    info = plan.info()
    assert info["kernel"] == capi.KERNEL_ROW_GATHER and info["padded_positions"] >= nnz, info
    rows, cols, val = d["row_ind"].long(), d["col_ind"].long(), d["val"].double()
    dot = torch.empty(nnz, dtype=torch.float64, device=DEV)
    mag = torch.empty_like(dot)
    for b in range(0, nnz, 1 << 18):
        p = d["W"][rows[b:b + (1 << 18)]].double() * d["H"][cols[b:b + (1 << 18)]].double()
        dot[b:b + (1 << 18)] = p.sum(1)
        mag[b:b + (1 << 18)] = p.abs().sum(1)
    W, H, out = d["W"].data_ptr(), d["H"].data_ptr(), torch.empty(nnz, device=DEV)

    def close(ref, scale):  # a rounding per product, sum and scaling
        torch.cuda.synchronize()
        assert bool((torch.abs(out.double() - ref) <= (K + 4) * 2.0 ** -24 * scale).all())
        out.fill_(float("nan"))

    out.fill_(float("nan"))
    plan.execute(0, W, H, out.data_ptr())
    close(dot, mag)
    plan.execute(d["val"].data_ptr(), W, H, out.data_ptr())
    close(val * dot, val.abs() * mag)
    plan.set_values(d["val"].data_ptr())
    plan.execute(0, W, H, out.data_ptr())
    close(val * dot, val.abs() * mag)
    plan.execute_epilogue(0, W, H, out.data_ptr(), capi.EPILOGUE_RESIDUAL)
    close(val - dot, val.abs() + mag)
