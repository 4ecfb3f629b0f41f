"""Row gather in slices of K (gather_slice in kernels_gather.hip): without and with a plan, from where the rule takes over,
against 64 bits; every value mode; values that lie where the results go (all slices in one launch then), bit for bit the same."""
import pytest
import torch

from sddmm_gpu_amd import capi

pytestmark = pytest.mark.gpu


def make(n_rows, n_cols, nnz, K, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    keys = torch.randint(0, n_rows * n_cols, (int(1.2 * nnz),), generator=g, device="cuda")
    keys = torch.unique(keys[keys // n_cols % 7 != 3])  # (every seventh row is empty)
    keys = keys[torch.randperm(keys.numel(), generator=g, device="cuda")[:nnz].sort().values]
    assert keys.numel() == nnz
    rows = keys // n_cols
    rp = torch.zeros(n_rows + 1, dtype=torch.int64, device="cuda")
    rp[1:] = torch.cumsum(torch.bincount(rows, minlength=n_rows), 0)
    W, H, val = (torch.randn(*s, generator=g, device="cuda") for s in ((n_rows, K), (n_cols, K), (nnz,)))
    cols = keys - rows * n_cols
    dot = torch.cat([(W[rows[i:i + (1 << 18)]].double() * H[cols[i:i + (1 << 18)]].double()).sum(1) for i in range(0, nnz, 1 << 18)])
    return rp.int(), cols.int(), val, W, H, dot


# On both sides of each line: nonzeros, columns, rank.  Slices: launches of a plan that gathers all rows.  40,000 and 300,000
# rows: kernels with several batches a wave and with one; W or H beyond 4 GB: rows found
# with 64-bit offsets.
@pytest.mark.parametrize("n_rows,n_cols,nnz,K,slices", [
    (40000, 24000, 2500000, 256, 4), (300000, 25001, 2500003, 256, 4), (40000, 23999, 2500000, 256, 1), (40000, 24000, 2499999, 256, 1),
    (40000, 11000, 3000000, 448, 7), (40000, 11000, 2999999, 448, 1), (150000, 11000, 1400001, 512, 8), (40000, 11000, 1399999, 512, 1),
    (9000, 350001, 1400003, 512, 1), (9000, 350000, 1400001, 512, 8), (40000, 24000, 3000000, 384, 1),
    (2101248, 11000, 1500001, 512, 8), (100000, 2101248, 8405000, 512, 8)])
def test_slices_against_64_bits(n_rows, n_cols, nnz, K, slices):
    rp, ci, val, W, H, dot = make(n_rows, n_cols, nnz, K, K + slices)
    st = torch.cuda.current_stream().cuda_stream
    plan = capi.Plan.from_device_csr(n_rows, n_cols, nnz, rp.data_ptr(), ci.data_ptr(), K, options=capi.PlanOptions.defaults(kernel=capi.KERNEL_ROW_GATHER))
    assert plan.info()["n_launches"] == slices
    p = lambda t: t.data_ptr()

    def noalloc(v, out):
        capi.csr_noalloc(n_rows, n_cols, nnz, p(rp), p(ci), v, K, p(W), p(H), p(out), st)

    def close(out, want):  # (fp32 chains of 16 and sums of those: 1e-7, measured)
        assert float((out.double() - want).norm() / want.norm()) < 2e-7

    out, out2 = torch.full_like(val, 7.0), torch.full_like(val, -7.0)
    noalloc(p(val), out)
    close(out, val.double() * dot)
    plan.execute(p(val), p(W), p(H), p(out2), st)
    assert torch.equal(out, out2)
    scaled = out.clone()
    noalloc(0, out)
    close(out, dot)
    plan.execute_epilogue(p(val), p(W), p(H), p(out2), capi.EPILOGUE_RESIDUAL, st)
    close(out2, val.double() - dot)
    for run in (lambda v: noalloc(p(v), v), lambda v: plan.execute(p(v), p(W), p(H), p(v), st)):
        v = val.clone()
        run(v)
        assert torch.equal(v, scaled)
    v = val.clone()
    plan.execute_epilogue(p(v), p(W), p(H), p(v), capi.EPILOGUE_RESIDUAL, st)
    assert torch.equal(v, out2)
    for v, d_out, launches in ((val, out, slices), (v, v, 1)):
        prof = plan.execute_profiled(p(v), p(W), p(H), p(d_out), st)
        lanes = 8 if nnz > 32 * n_rows else 16  # (those of the kernel on slices)
        assert [q["n_kernel_launches"] for q in prof] == [launches] and (slices == 1 or prof[0]["lanes_per_nnz"] == plan.info()["lanes_per_nnz"] == lanes)
    plan.close()


def test_slices_replayed_from_a_graph():
    n_rows, n_cols, nnz, K = 60000, 11001, 1500001, 512
    rp, ci, val, W, H, dot = make(n_rows, n_cols, nnz, K, 5)
    out = torch.zeros_like(val)
    run = lambda: capi.csr_noalloc(n_rows, n_cols, nnz, rp.data_ptr(), ci.data_ptr(), val.data_ptr(), K, W.data_ptr(), H.data_ptr(),
                                   out.data_ptr(), torch.cuda.current_stream().cuda_stream)
    run()
    torch.cuda.synchronize()
    want = out.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run()
    for _ in range(3):
        out.fill_(3.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
