"""The row gather with one batch a wave: the edges of its batches, rounds of steps and rule, against 64 bits."""
import pytest
import torch

from sddmm_gpu_amd import capi

pytestmark = pytest.mark.gpu


def _case(n_rows, n_cols, nnz, K, seed):
    g = torch.Generator().manual_seed(seed)
    keys = torch.randperm(n_rows * n_cols, generator=g)[:nnz].sort().values
    rows, cols = keys // n_cols, keys % n_cols
    row_ptr = torch.zeros(n_rows + 1, dtype=torch.int64)
    row_ptr[1:] = torch.cumsum(torch.bincount(rows, minlength=n_rows), 0)
    W, H = torch.randn(n_rows, K, generator=g), torch.randn(n_cols, K, generator=g)
    val = torch.rand(nnz, generator=g)
    dot, size = torch.empty(nnz, dtype=torch.float64), torch.empty(nnz, dtype=torch.float64)
    for b in range(0, nnz, 1 << 14):
        w, h = W[rows[b:b + (1 << 14)]].double(), H[cols[b:b + (1 << 14)]].double()
        dot[b:b + (1 << 14)] = (w * h).sum(1)
        size[b:b + (1 << 14)] = (w * h).abs().sum(1)
    dev = [t.cuda() for t in (row_ptr.int(), cols.int(), val, W, H)]
    # a sum of K rounded products in any order, then one product with the value
    return dev, dot * val.double(), (K + 1) * 2.0 ** -24 * size * val.double() + 1e-30


@pytest.mark.parametrize("K", [4, 7, 16, 32, 33, 64, 72, 96, 100, 128, 180, 256, 300, 512, 700, 1024, 2048])
@pytest.mark.parametrize("n_rows,n_cols,nnz", [(1, 1, 1), (40, 90, 63), (3, 400, 64), (700, 30, 65), (64, 64, 257), (5000, 40, 3000)])
def test_sizes_and_ranks(n_rows, n_cols, nnz, K):
    (rp, ci, val, W, H), ref, bound = _case(n_rows, n_cols, nnz, K, 100 * K + nnz)
    stream = torch.cuda.current_stream().cuda_stream
    out = torch.full((nnz + 1,), 7.0, device="cuda")
    capi.csr_noalloc(n_rows, n_cols, nnz, rp.data_ptr(), ci.data_ptr(), val.data_ptr(), K, W.data_ptr(), H.data_ptr(), out.data_ptr(), stream)
    planned = torch.full((nnz + 1,), 7.0, device="cuda")
    plan = capi.Plan.from_device_csr(n_rows, n_cols, nnz, rp.data_ptr(), ci.data_ptr(), K,
                                     options=capi.PlanOptions.defaults(kernel=capi.KERNEL_ROW_GATHER))
    plan.execute(val.data_ptr(), W.data_ptr(), H.data_ptr(), planned.data_ptr(), stream)
    torch.cuda.synchronize()
    assert ((out[:nnz].cpu().double() - ref).abs() <= bound).all()
    assert torch.equal(out, planned) and float(out[nnz]) == 7.0


# either side of each line of the rule: 2^16 nonzeros, 32 a row, and 2^18 nonzeros at up to 32 floats a row
@pytest.mark.parametrize("K", [32, 64, 128])
@pytest.mark.parametrize("n_rows,nnz", [(1024, 65536), (1024, 65537), (3000, 96000), (3000, 96001), (2000, 262144), (2000, 262145)])
def test_rule(n_rows, nnz, K):
    (rp, ci, val, W, H), ref, bound = _case(n_rows, 500, nnz, K, nnz + K)
    out = torch.full((nnz + 1,), 7.0, device="cuda")
    capi.csr_noalloc(n_rows, 500, nnz, rp.data_ptr(), ci.data_ptr(), val.data_ptr(), K, W.data_ptr(), H.data_ptr(), out.data_ptr(),
                     torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert ((out[:nnz].cpu().double() - ref).abs() <= bound).all() and float(out[nnz]) == 7.0


@pytest.mark.parametrize("repeat", [40, 12000])  # one batch a wave, several
def test_h_beyond_32_bit_offsets(repeat):
    n_rows, n_cols, K = 3, (1 << 22) + 3, 256  # 4.3 GB
    cols = torch.tensor([n_cols - 1, 0, n_cols - 2, 1 << 21, 5, (1 << 22) - 1, 1 << 22], dtype=torch.int32, device="cuda").repeat(repeat)
    nnz = cols.numel()
    rp = torch.tensor([0, 5, 5, nnz], dtype=torch.int32, device="cuda")
    g = torch.Generator(device="cuda").manual_seed(repeat)
    W = torch.randn(n_rows, K, generator=g, device="cuda")
    H = torch.empty(n_cols, K, device="cuda").normal_(generator=g)
    out = torch.full((nnz + 1,), 7.0, device="cuda")
    capi.csr_noalloc(n_rows, n_cols, nnz, rp.data_ptr(), cols.data_ptr(), 0, K, W.data_ptr(), H.data_ptr(), out.data_ptr(),
                     torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    rows = torch.repeat_interleave(torch.arange(n_rows, device="cuda"), (rp[1:] - rp[:-1]).long())
    terms = W[rows].double() * H[cols.long()].double()
    assert bool(((out[:nnz].double() - terms.sum(1)).abs() <= K * 2.0 ** -24 * terms.abs().sum(1)).all()) and float(out[nnz]) == 7.0


# half a million nonzeros at K = 64 (exact; 60: masked), and rows of 16 and 32: 32 from 8 million pieces on (a third of a million
# nonzeros at K = 96, a million at K = 32)
@pytest.mark.parametrize("K", [16, 32, 60, 64, 96])
@pytest.mark.parametrize("n_rows,nnz", [(33000, 2 ** 19 - 1), (33000, 2 ** 19), (16000, 2 ** 19), (16384, 2 ** 19), (12000, 333333), (12000, 333334), (10416, 333334), (34000, 1000000)])
def test_rule_for_larger_matrices(n_rows, nnz, K):
    (rp, ci, val, W, H), ref, bound = _case(n_rows, 200, nnz, K, nnz + K)
    out = torch.full((nnz + 1,), 7.0, device="cuda")
    capi.csr_noalloc(n_rows, 200, nnz, rp.data_ptr(), ci.data_ptr(), val.data_ptr(), K, W.data_ptr(), H.data_ptr(), out.data_ptr(),
                     torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert ((out[:nnz].cpu().double() - ref).abs() <= bound).all() and float(out[nnz]) == 7.0


# the ranks read line by line from 2^18 nonzeros on (K = 33 to 36 up to 2^20)
@pytest.mark.parametrize("K", [33, 36, 37, 40, 60, 64, 97, 125, 128])
@pytest.mark.parametrize("n_rows,nnz", [(17000, 2 ** 18 - 1), (17000, 2 ** 18), (66000, 2 ** 20 - 1), (66000, 2 ** 20)])
def test_ranks_read_line_by_line(n_rows, nnz, K):
    (rp, ci, val, W, H), ref, bound = _case(n_rows, 200, nnz, K, nnz + K)
    out = torch.full((nnz + 1,), 7.0, device="cuda")
    capi.csr_noalloc(n_rows, 200, nnz, rp.data_ptr(), ci.data_ptr(), val.data_ptr(), K, W.data_ptr(), H.data_ptr(), out.data_ptr(),
                     torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert ((out[:nnz].cpu().double() - ref).abs() <= bound).all() and float(out[nnz]) == 7.0


# many empty rows: the plan lists the others, the call without a plan knows only how many there are of both
@pytest.mark.parametrize("K", [33, 50, 64, 100])
def test_same_bits_with_and_without_a_plan_beside_empty_rows(K):
    used, n_rows, n_cols, nnz = 5000, 40000, 200, 2 ** 18
    (rp, ci, val, W, H), ref, bound = _case(used, n_cols, nnz, K, K)
    rp = torch.cat([rp, rp[-1:].repeat(n_rows - used)])
    W = torch.cat([W, W.new_zeros(n_rows - used, K)])
    outs = [torch.full((nnz + 1,), 7.0, device="cuda") for _ in range(2)]
    stream = torch.cuda.current_stream().cuda_stream
    capi.csr_noalloc(n_rows, n_cols, nnz, rp.data_ptr(), ci.data_ptr(), val.data_ptr(), K, W.data_ptr(), H.data_ptr(), outs[0].data_ptr(), stream)
    plan = capi.Plan.from_device_csr(n_rows, n_cols, nnz, rp.data_ptr(), ci.data_ptr(), K,
                                     options=capi.PlanOptions.defaults(kernel=capi.KERNEL_ROW_GATHER))
    plan.execute(val.data_ptr(), W.data_ptr(), H.data_ptr(), outs[1].data_ptr(), stream)
    torch.cuda.synchronize()
    assert ((outs[0][:nnz].cpu().double() - ref).abs() <= bound).all()
    assert torch.equal(outs[0], outs[1]) and float(outs[0][nnz]) == 7.0
