"""Long runs of empty rows in a plain CSR pattern: behind the last nonzero (padded batches), in the
middle, in front, and between all nonzeros (more empty rows among a wave's nonzeros than it walks over)."""
import numpy as np
import pytest
import torch

from conftest import parity_report
from sddmm_gpu_amd import capi

pytestmark = pytest.mark.gpu
RUN = 1 << 20  # empty rows in a run


def pattern(kind, nnz, rng):
    """(row_ptr, rows) of nnz nonzeros over 1024 rows and RUN empty ones, or spread over RUN rows."""
    if kind == "spread":
        rows = np.sort(rng.integers(0, RUN, nnz))
        n = RUN
    else:
        rows = np.sort(rng.integers(0, 1024, nnz))
        n = 1024 + RUN
        rows += {"behind": 0, "in front": RUN, "in the middle": 0}[kind]
        if kind == "in the middle":
            rows[rows >= 512] += RUN
    rp = np.zeros(n + 1, np.int32)
    rp[1:] = np.cumsum(np.bincount(rows, minlength=n))
    return rp, rows.astype(np.int32)


# (one nonzero, less than a share, many shares of 64 or fewer with a partial last one)
@pytest.mark.parametrize("nnz", [1, 50, 5000, 70001])
@pytest.mark.parametrize("kind", ["behind", "in front", "in the middle", "spread"])
def test_runs_of_empty_rows(oracle, kind, nnz):
    K, n_cols = 8, 300
    rng = np.random.default_rng(nnz)
    rp, rows = pattern(kind, nnz, rng)
    n = len(rp) - 1
    ci = rng.integers(0, n_cols, nnz).astype(np.int32)
    ci = ci[np.lexsort((ci, rows))]
    W = rng.standard_normal((n, K)).astype(np.float32); H = rng.standard_normal((n_cols, K)).astype(np.float32)
    val = rng.standard_normal(nnz).astype(np.float32)
    dev = torch.device("cuda:0")
    d = [torch.from_numpy(x).to(dev) for x in (rp, ci, val, W, H)]
    p = [x.data_ptr() for x in d]
    _, absp = oracle.sddmm_f64(rows, ci, val, W, H)
    out = torch.full((nnz,), float("nan"), device=dev)
    Y = torch.full((n, K), float("nan"), device=dev)
    stream = torch.cuda.current_stream().cuda_stream
    sddmm = lambda: capi.csr_noalloc(n, n_cols, nnz, p[0], p[1], p[2], K, p[3], p[4], out.data_ptr(), stream)
    spmm = lambda: capi.spmm_csr(n, n_cols, nnz, p[0], p[1], p[2], K, p[4], Y.data_ptr(), stream)
    for call in (sddmm, spmm):
        # one wave that steps over the run 64 rows at a time takes 5 ms for it; the whole call takes
        # 60 us where nothing walks it (most of that zeroing 32 MB of Y)
        call()
        best = 1e30
        for _ in range(5):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record(); call(); e1.record(); e1.synchronize()
            best = min(best, e0.elapsed_time(e1))
        assert best < 1.0, f"{best} ms"
    assert parity_report(out.cpu().numpy(), oracle.sddmm_csr(rp, ci, val, W, H), K, absp)["violations"] == 0
    ref, mag = oracle.spmm_csr(rp, ci, val, H, with_abs=True)
    # sums of c products in any order: c 2^-24 of their magnitude (and never less than a rounding)
    bound = (np.diff(rp)[:, None] + 1) * 2.0 ** -24 * mag
    assert np.all(np.abs(Y.cpu().numpy().astype(np.float64) - ref) <= bound)


def test_share_of_512_nonzeros_among_empty_rows(oracle):
    """The largest share of a wave (five million nonzeros at K = 8), eight rows to a nonzero: searched, not walked."""
    K, n_cols, nnz = 8, 64, 5_000_000
    rng = np.random.default_rng(7)
    rows = np.sort(rng.integers(0, 8 * nnz, nnz))
    n = 8 * nnz
    dev = torch.device("cuda:0")
    rows_d = torch.from_numpy(rows).to(dev)
    rp = torch.zeros(n + 1, dtype=torch.int64, device=dev)
    rp[1:] = torch.cumsum(torch.bincount(rows_d, minlength=n), 0)
    rp = rp.int()
    ci = torch.from_numpy(rng.integers(0, n_cols, nnz).astype(np.int32)).to(dev)
    g = torch.Generator(device=dev); g.manual_seed(3)
    W = torch.randn(n, K, device=dev, generator=g); H = torch.randn(n_cols, K, device=dev, generator=g)
    val = torch.randn(nnz, device=dev, generator=g)
    out = torch.full((nnz,), float("nan"), device=dev)
    Y = torch.full((n, K), float("nan"), device=dev)
    capi.csr_noalloc(n, n_cols, nnz, rp.data_ptr(), ci.data_ptr(), val.data_ptr(), K, W.data_ptr(), H.data_ptr(), out.data_ptr())
    capi.spmm_csr(n, n_cols, nnz, rp.data_ptr(), ci.data_ptr(), val.data_ptr(), K, H.data_ptr(), Y.data_ptr())
    torch.cuda.synchronize()
    w, h = W[rows_d].double(), H[ci.long()].double()
    ref = val.double() * (w * h).sum(1)
    mag = val.double().abs() * (w * h).abs().sum(1)
    assert bool(((out.double() - ref).abs() <= (K + 2) * 2.0 ** -24 * mag).all())
    yref = torch.zeros(n, K, dtype=torch.float64, device=dev).index_add_(0, rows_d, val.double()[:, None] * h)
    ymag = torch.zeros(n, K, dtype=torch.float64, device=dev).index_add_(0, rows_d, (val.double()[:, None] * h).abs())
    count = (rp[1:] - rp[:-1]).double()[:, None]
    assert bool(((Y.double() - yref).abs() <= (count + 1) * 2.0 ** -24 * ymag).all())
