"""The product over a CSR pattern where its groups of lanes meet the rows (a mark beside each entry says that a row begins):
rows that begin and end at, before and behind a group's share and the steps of four in it; an H beyond 32-bit byte offsets."""
import pytest
import torch

from sddmm_gpu_amd import capi

pytestmark = pytest.mark.gpu


def check(lens, n_cols, K, cols=None, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    lens = torch.tensor(lens, device="cuda")
    nnz, n_rows = int(lens.sum()), lens.numel()
    row_ptr = torch.zeros(n_rows + 1, dtype=torch.int32, device="cuda")
    row_ptr[1:] = torch.cumsum(lens, 0)
    if cols is None:
        cols = torch.randint(0, n_cols, (nnz,), generator=g, device="cuda")
    cols = cols.int()
    x = torch.randn(nnz, generator=g, device="cuda")
    H = torch.empty(n_cols, K, device="cuda").normal_(generator=g)
    Y = torch.full((n_rows, K), float("nan"), device="cuda")
    capi.spmm_csr(n_rows, n_cols, nnz, row_ptr.data_ptr(), cols.data_ptr(), x.data_ptr(), K, H.data_ptr(), Y.data_ptr(),
                  torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    rows = torch.repeat_interleave(torch.arange(n_rows, device="cuda"), lens)
    terms = x[:, None].double() * H[cols.long()].double()
    want = torch.zeros(n_rows, K, dtype=torch.float64, device="cuda").index_add_(0, rows, terms)
    size = torch.zeros(n_rows, K, dtype=torch.float64, device="cuda").index_add_(0, rows, terms.abs())
    # a rounding per term and a few for the parts of cut rows
    bound = (lens[:, None].double() + 16) * 2.0 ** -24 * size
    assert bool(((Y.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("K", [4, 16, 30, 50, 64, 100, 128, 256, 300])
@pytest.mark.parametrize("lens", [[1] * 300, [3, 5] * 200, [4] * 130, [63, 1, 64, 65, 0, 0, 128, 2] * 5, [1000, 7, 0, 1], [0] * 9 + [1], [2, 6] * 3000 + [5000]])
def test_rows_at_the_edges_of_shares(lens, K):
    check(lens, 77, K, seed=K)


def test_h_beyond_32_bit_offsets():
    n_cols, K = (1 << 22) + 3, 256  # 4.3 GB
    cols = torch.tensor([n_cols - 1, 0, n_cols - 2, 1 << 21, 5, (1 << 22) - 1, 1 << 22], device="cuda").repeat(40)
    check([3, 50, 1, 0, 100, 126], n_cols, K, cols=cols)
