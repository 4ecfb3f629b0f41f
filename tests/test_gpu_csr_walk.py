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


# The slices of H's rows that the product takes in turn (slice_pieces_most in kernels_spmm_csr.hip): 8 pieces from 1.5 million nonzeros
# on, two slices at K = 64 from 4 million and 20 MB of H on, 16 pieces at ranks beyond 256 across lines and where columns are used
# less than four times, whole rows on the other side of those lines and where rows have next to no nonzeros.  Rows: lengths that differ,
# every seventh empty.
@pytest.mark.parametrize("n_rows,n_cols,nnz,K", [
    (30000, 40000, 1500000, 192), (30000, 40000, 1499999, 192), (30000, 40000, 2000001, 96), (60000, 100000, 4000000, 64), (60000, 100000, 3999999, 64),
    (20000, 20000, 1500001, 300), (20000, 20000, 1499999, 300), (20000, 400000, 1599999, 192), (20000, 400000, 1600000, 192), (20000, 400000, 1599999, 301),
    (20000, 100000, 399999, 256), (20000, 100000, 400001, 256), (40000, 3000, 65536, 192), (40001, 3000, 65536, 192), (43690, 3000, 65536, 200),
    (43692, 3000, 65536, 200), (3000, 3000, 65537, 192)])
def test_product_in_slices_against_64_bits(n_rows, n_cols, nnz, K):
    g = torch.Generator(device="cuda")
    g.manual_seed(nnz + K)
    lens = torch.rand(n_rows, generator=g, device="cuda") ** 2
    lens[torch.arange(n_rows, device="cuda") % 7 == 3] = 0
    rows = torch.searchsorted(torch.cumsum(lens, 0) / lens.sum(), torch.rand(nnz, generator=g, device="cuda")).clamp_(max=n_rows - 1).sort().values
    rp = torch.zeros(n_rows + 1, dtype=torch.int64, device="cuda")
    rp[1:] = torch.cumsum(torch.bincount(rows, minlength=n_rows), 0)
    ci = torch.randint(0, n_cols, (nnz,), generator=g, device="cuda")  # (any order, pairs may repeat: the product allows it)
    x, H = torch.randn(nnz, generator=g, device="cuda"), torch.randn(n_cols, K, generator=g, device="cuda")
    rp32, ci32 = rp.int(), ci.int()
    Y = torch.full((n_rows, K), float("nan"), device="cuda")
    capi.spmm_csr(n_rows, n_cols, nnz, rp32.data_ptr(), ci32.data_ptr(), x.data_ptr(), K, H.data_ptr(), Y.data_ptr(), torch.cuda.current_stream().cuda_stream)
    for k in range(0, K, 64):
        want = torch.zeros(n_rows, min(64, K - k), dtype=torch.float64, device="cuda")
        mag = torch.zeros_like(want)
        for i in range(0, nnz, 1 << 19):
            part = x[i:i + (1 << 19), None].double() * H[ci[i:i + (1 << 19)], k:k + 64].double()
            want.index_add_(0, rows[i:i + (1 << 19)], part)
            mag.index_add_(0, rows[i:i + (1 << 19)], part.abs())
        bound = 1e-5 * torch.diff(rp).clamp(min=1).double().sqrt()[:, None] * mag
        assert bool(((Y[:, k:k + 64].double() - want).abs() <= bound).all())


def test_product_of_more_slices_than_a_grid_has():
    """Rows of 16 MB: in slices of 16 pieces more than a grid's second dimension holds."""
    K = 4 * 16 * 65535 + 4
    rp = torch.tensor([0, 2, 3], dtype=torch.int32, device="cuda")
    ci = torch.tensor([0, 1, 1], dtype=torch.int32, device="cuda")
    x, H = torch.randn(3, device="cuda"), torch.randn(2, K, device="cuda")
    Y = torch.full((2, K), float("nan"), device="cuda")
    capi.spmm_csr(2, 2, 3, rp.data_ptr(), ci.data_ptr(), x.data_ptr(), K, H.data_ptr(), Y.data_ptr(), torch.cuda.current_stream().cuda_stream)
    want = torch.stack([x[0].double() * H[0].double() + x[1].double() * H[1].double(), x[2].double() * H[1].double()])
    mag = torch.stack([(x[0] * H[0]).abs() + (x[1] * H[1]).abs(), (x[2] * H[1]).abs()])
    assert bool(((Y.double() - want).abs() <= 1e-6 * mag.double() + 1e-30).all())
