"""Tile launches whose (row block, tile) items are uneven, so that they are cut into pieces and dealt out anew:
windows around the diagonal with a few full rows and columns, a few crowded columns, everything in one tile."""
import numpy as np
import pytest
import torch

from sddmm_gpu_amd import capi
from test_gpu_parity import _dict_of, check

pytestmark = pytest.mark.gpu


def pattern(kind, rng):
    if kind == "window":
        n = m = 2500
        r = np.repeat(np.arange(n), 81); c = r + np.tile(np.arange(-40, 41), n)
        keep = (c >= 0) & (c < m); r, c = r[keep], c[keep]
        g = np.arange(0, n, 311)
        r = np.concatenate([r, np.repeat(g, m), np.tile(np.arange(n), len(g))]); c = np.concatenate([c, np.tile(np.arange(m), len(g)), np.repeat(g, n)])
    elif kind == "crowded":
        n, m = 3000, 6000
        r = np.concatenate([np.repeat(np.arange(n), 60), rng.integers(0, n, 40000)])
        c = np.concatenate([rng.integers(2000, 2130, n * 60), rng.integers(0, m, 40000)])
    else:
        n, m = 1200, 9000
        r = np.repeat(np.arange(n), 90); c = np.tile(np.arange(90), n) + 4321
    key = np.unique(r.astype(np.int64) * m + c)
    return n, m, key // m, key % m


@pytest.mark.parametrize("K", [32, 64, 128, 256])
@pytest.mark.parametrize("kind", ["window", "crowded", "one tile"])
@pytest.mark.parametrize("few", [-1, 0])
def test_uneven_items(oracle, kind, K, few):
    rng = np.random.default_rng(5)
    n, m, r, c = pattern(kind, rng)
    d = _dict_of(n, m, r, c, K, rng)
    dev = torch.device("cuda:0")
    t = {k: d[k].to(dev) for k in ("row_ptr", "col_ind", "val", "W", "H")}
    plan = capi.Plan.from_device_csr(n, m, d["nnz"], t["row_ptr"].data_ptr(), t["col_ind"].data_ptr(), K, options=capi.PlanOptions.defaults(
        kernel=capi.KERNEL_HYBRID, split_min_nnz=0, stage_factor=0, short_row_max=0, tile_few_blocks=few, spmm_stream=1, ignore_env=1))
    out = torch.full((d["nnz"],), float("nan"), device=dev)
    plan.execute(t["val"].data_ptr(), t["W"].data_ptr(), t["H"].data_ptr(), out.data_ptr())
    torch.cuda.synchronize()
    check(d, out.cpu().numpy(), oracle, K=K)
    # (cut and dealt out anew or not: the product of these goes over the pattern, as the runs are short or the matrix is small)
    assert plan.spmm_form() == capi.SPMM_WALK
    Y = torch.full((n, K), float("nan"), device=dev)
    plan.spmm(t["val"].data_ptr(), t["H"].data_ptr(), Y.data_ptr())
    torch.cuda.synchronize()
    ref, mag = oracle.spmm_csr(d["row_ptr"].numpy(), d["col_ind"].numpy(), d["val"].numpy(), d["H"].numpy(), with_abs=True)
    deg = np.diff(d["row_ptr"].numpy())
    assert np.all(np.abs(Y.cpu().numpy().astype(np.float64) - ref) <= 1e-5 * np.sqrt(np.maximum(deg, 1))[:, None] * mag)
