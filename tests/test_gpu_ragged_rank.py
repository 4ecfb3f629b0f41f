"""The padded tile kernel at ranks it has no exact width for (32, 64 and 128 elements, slices of 128): all value
modes and the residual, one launch and several slices in one launch or in one each, rows of W and H at any 4-byte
address; NaN and infinity outside a row must not reach its results."""
import numpy as np
import pytest
import torch

from conftest import parity_report
from sddmm_gpu_amd import capi
from test_gpu_parity import _dict_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [8, 9, 15, 16, 31, 33, 50, 63, 66, 96, 100, 127, 129, 130, 131, 160, 205, 255, 300])
@pytest.mark.parametrize("fuse", [0, 1])
def test_ragged_ranks_on_the_tile_kernel(oracle, K, fuse):
    if K <= 128 and not fuse:
        pytest.skip("one launch either way")
    rng = np.random.default_rng(K)
    n, m = 700, 900
    key = np.unique(np.concatenate([rng.integers(0, n * m, 30000), np.arange(40) * m + 7, np.arange(899) + 5 * m]))
    d = _dict_of(n, m, key // m, key % m, K, rng)
    dev = torch.device("cuda:0")
    # W and H inside larger arrays of NaN, at an address that is no multiple of 16 where the rank allows it
    shift = 0 if K % 4 == 0 else 3

    def surrounded(x):
        big = torch.full((x.numel() + 64,), float("nan"), device=dev)
        big[32 + shift:32 + shift + x.numel()] = x.reshape(-1).to(dev)
        return big, big.data_ptr() + 4 * (32 + shift)

    (_, W), (_, H) = keep = surrounded(d["W"]), surrounded(d["H"])
    t = {k: d[k].to(dev) for k in ("row_ptr", "col_ind", "val")}
    nnz = d["nnz"]
    plan = capi.Plan.from_device_csr(n, m, nnz, t["row_ptr"].data_ptr(), t["col_ind"].data_ptr(), K, options=capi.PlanOptions.defaults(
        kernel=capi.KERNEL_HYBRID, split_min_nnz=0, stage_factor=0, short_row_max=42, tile_size_x=200, fuse_slices=fuse, ignore_env=1))
    info = plan.info()
    assert info["class_nnz"][0] > 0 and info["class_nnz"][2] > 0 and info["k_slice"] == min(K, 128)

    def run(f):
        out = torch.full((nnz,), float("nan"), device=dev)
        f(out.data_ptr())
        torch.cuda.synchronize()
        return out.cpu().numpy()

    def check(vals, out):
        args = d["row_ind"].numpy(), d["col_ind"].numpy(), vals, d["W"].numpy(), d["H"].numpy()
        assert np.all(np.isfinite(out))
        assert parity_report(out, oracle.sddmm_coo(*args), K, oracle.sddmm_f64(*args)[1])["violations"] == 0

    check(np.ones(nnz, np.float32), run(lambda o: plan.execute(0, W, H, o)))
    by_call = run(lambda o: plan.execute(t["val"].data_ptr(), W, H, o))
    check(d["val"].numpy(), by_call)
    res_call = run(lambda o: plan.execute_epilogue(t["val"].data_ptr(), W, H, o, capi.EPILOGUE_RESIDUAL))
    plan.set_values(t["val"].data_ptr())
    assert np.array_equal(by_call, run(lambda o: plan.execute(0, W, H, o)))
    res_plan = run(lambda o: plan.execute_epilogue(0, W, H, o, capi.EPILOGUE_RESIDUAL))
    assert np.array_equal(res_call, res_plan)
    cpu = oracle.sddmm_residual_csr(d["row_ptr"].numpy(), d["col_ind"].numpy(), d["val"].numpy(), d["W"].numpy(), d["H"].numpy())
    _, absp = oracle.sddmm_f64(d["row_ind"].numpy(), d["col_ind"].numpy(), np.ones(nnz, np.float32), d["W"].numpy(), d["H"].numpy())
    assert np.all(np.abs(res_call.astype(np.float64) - cpu) <= 1e-5 * np.sqrt(K) * absp + 2.0 ** -22 * np.abs(cpu))
    plan.close()
    del keep
