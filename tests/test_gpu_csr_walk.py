"""The kernels that walk a plain CSR pattern by nonzeros (sddmm_csr_noalloc, ROW_GATHER plans,
sddmm_spmm_csr) at ranks that are no multiple of their 16-byte pieces and on patterns whose rows
begin and end at the edges of a group's, a wave's and a workgroup's share."""
import numpy as np
import pytest
import torch

from conftest import parity_report
from sddmm_gpu_amd import capi

pytestmark = pytest.mark.gpu


def pattern(kind, n_cols, rng):
    if kind == "edges of shares":  # rows that end on, before and after multiples of 4 to 512, empty rows between
        counts = [0, 64, 63, 1, 0, 0, 65, 31, 32, 33, 4, 3, 1, 512, 511, 1, 0, 128, 100, 27, 1] + [0] * 150 + [5, 0]
    elif kind == "one long row":   # a row over many workgroups among short ones; nothing behind it
        counts = [3, 0, 40000, 2]
    elif kind == "single":
        counts = [0, 0, 1, 0]
    else:                          # many short rows, more than 64 row starts in one batch
        counts = list(rng.integers(0, 3, 3000))
    counts = np.minimum(np.asarray(counts), n_cols)
    rp = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    ci = np.concatenate([np.sort(rng.choice(n_cols, c, replace=False)) for c in counts] or [[]]).astype(np.int32)
    return rp, ci


@pytest.mark.parametrize("K", [4, 5, 15, 17, 33, 50, 66, 97, 130, 193, 255, 257, 300, 515, 1030])
@pytest.mark.parametrize("kind", ["edges of shares", "one long row", "single", "short rows"])
def test_any_rank_on_awkward_patterns(oracle, kind, K):
    if kind == "one long row" and K > 300:
        pytest.skip("covered by the smaller ranks")
    rng = np.random.default_rng(K)
    n_cols = 50000 if kind == "one long row" else 700
    rp, ci = pattern(kind, n_cols, rng)
    n, nnz = len(rp) - 1, len(ci)
    W = rng.standard_normal((n, K)).astype(np.float32); H = rng.standard_normal((n_cols, K)).astype(np.float32)
    val = rng.standard_normal(nnz).astype(np.float32)
    dev = torch.device("cuda:0")
    d = [torch.from_numpy(x).to(dev) for x in (rp, ci, val, W, H)]
    p = [x.data_ptr() for x in d]
    cpu = oracle.sddmm_csr(rp, ci, val, W, H)
    rows = np.repeat(np.arange(n), np.diff(rp)).astype(np.int32)
    _, absp = oracle.sddmm_f64(rows, ci, val, W, H)
    out = torch.full((nnz,), float("nan"), device=dev)
    capi.csr_noalloc(n, n_cols, nnz, p[0], p[1], p[2], K, p[3], p[4], out.data_ptr())
    torch.cuda.synchronize()
    assert parity_report(out.cpu().numpy(), cpu, K, absp)["violations"] == 0
    plan = capi.Plan.from_device_csr(n, n_cols, nnz, p[0], p[1], K, kernel=capi.KERNEL_ROW_GATHER)
    out2 = torch.full((nnz,), float("nan"), device=dev)
    plan.execute(p[2], p[3], p[4], out2.data_ptr())
    torch.cuda.synchronize()
    plan.close()
    assert torch.equal(out, out2)
    Y = torch.full((n, K), float("nan"), device=dev)
    capi.spmm_csr(n, n_cols, nnz, p[0], p[1], p[2], K, p[4], Y.data_ptr())
    torch.cuda.synchronize()
    ref, mag = oracle.spmm_csr(rp, ci, val, H, with_abs=True)
    bound = 1e-5 * np.sqrt(np.maximum(np.diff(rp), 1))[:, None] * mag
    assert np.all(np.abs(Y.cpu().numpy().astype(np.float64) - ref) <= bound)
