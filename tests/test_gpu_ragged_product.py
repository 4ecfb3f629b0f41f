"""The product with the dense factor on column tiles at ranks that are no multiple of the tiles' width: one piece more or less than
a whole one, several slices with a short last one, factors at any 4-byte address, short and empty rows, against 64 bits."""
import pytest
import torch

from sddmm_gpu_amd import capi, synth

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module", params=["ratings", "dense"])
def matrix(request):
    if request.param == "ratings":
        d = synth.recommender(44000, 5600, K=4, seed=5, device=DEV, max_deg=5000)
    else:
        d = synth.uniform_random(8000, 2000, 0.33, K=4, seed=5, device=DEV)
    assert d["nnz"] >= 4000000
    n_rows = d["n_rows"] + 7  # empty ones at the end
    rp = torch.cat([d["row_ptr"], d["row_ptr"][-1:].repeat(7)]).int()
    return n_rows, d["n_cols"], d["nnz"], rp, d["col_ind"].int(), d["row_ind"].long()


@pytest.mark.parametrize("K", [28, 31, 33, 50, 61, 63, 65, 99, 100, 127, 187, 253, 382])
def test_against_64_bits(matrix, K):
    n_rows, n_cols, nnz, rp, ci, rows = matrix
    g = torch.Generator(device=DEV).manual_seed(K)
    x = torch.randn(nnz, generator=g, device=DEV)
    shift = 0 if K % 4 == 0 else 1  # (multiples of 4 need 16-byte alignment)
    H = torch.randn(n_cols * K + shift, generator=g, device=DEV)[shift:].view(n_cols, K)
    Yb = torch.full((n_rows * K + shift + 1,), 7.0, device=DEV)
    Y = Yb[shift:-1].view(n_rows, K)
    plan = capi.Plan.from_device_csr(n_rows, n_cols, nnz, rp.data_ptr(), ci.data_ptr(), K,
                                     options=capi.PlanOptions.defaults(spmm_stream=1, ignore_env=1))
    if n_cols == 2000:  # (long runs)
        assert plan.spmm_form() == (capi.SPMM_TILES if K > 32 else capi.SPMM_WALK)
    stream = torch.cuda.current_stream().cuda_stream
    plan.spmm(x.data_ptr(), H.data_ptr(), Y.data_ptr(), stream=stream)
    first = Y.clone()
    ws = torch.empty(plan.workspace_bytes() + 256, dtype=torch.uint8, device=DEV)
    at = (ws.data_ptr() + 255) // 256 * 256
    Yb.fill_(7.0)
    plan.spmm(x.data_ptr(), H.data_ptr(), Y.data_ptr(), at, plan.workspace_bytes(), stream=stream)
    torch.cuda.synchronize()
    assert torch.equal(first, Y) and float(Yb[-1]) == 7.0 and (not shift or float(Yb[0]) == 7.0)
    ref = torch.zeros(n_rows, K, dtype=torch.float64, device=DEV)
    size = torch.zeros(n_rows, K, dtype=torch.float64, device=DEV)
    for b in range(0, nnz, 1 << 19):
        t = x[b:b + (1 << 19), None].double() * H[ci[b:b + (1 << 19)].long()].double()
        ref.index_add_(0, rows[b:b + (1 << 19)], t)
        size.index_add_(0, rows[b:b + (1 << 19)], t.abs())
    n = (rp[1:] - rp[:-1]).double()[:, None]  # a rounding per term of a row, however they are added up
    assert bool(((Y.double() - ref).abs() <= (n + 16) * 2.0 ** -24 * size).all())
    assert float(Y[-7:].abs().max()) == 0.0


# all rows tiled for the SDDMM, the long ones alone for the product (K slices of up to 64), or the long ones alone for both
@pytest.mark.parametrize("K", [32, 50, 64, 96, 128])
def test_sddmm_and_product_of_one_plan(matrix, K):
    n_rows, n_cols, nnz, rp, ci, rows = matrix
    g = torch.Generator(device=DEV).manual_seed(K)
    W, H = torch.randn(n_rows, K, generator=g, device=DEV), torch.randn(n_cols, K, generator=g, device=DEV)
    out, Y = torch.full((nnz + 1,), 7.0, device=DEV), torch.full((n_rows * K + 1,), 7.0, device=DEV)
    plan = capi.Plan.from_device_csr(n_rows, n_cols, nnz, rp.data_ptr(), ci.data_ptr(), K,
                                     options=capi.PlanOptions.defaults(spmm_stream=1, ignore_env=1))
    stream = torch.cuda.current_stream().cuda_stream
    plan.execute(0, W.data_ptr(), H.data_ptr(), out.data_ptr(), stream)
    plan.spmm(out.data_ptr(), H.data_ptr(), Y.data_ptr(), stream=stream)
    torch.cuda.synchronize()
    assert float(out[-1]) == 7.0 and float(Y[-1]) == 7.0
    ref, size = torch.zeros(n_rows, K, dtype=torch.float64, device=DEV), torch.zeros(n_rows, K, dtype=torch.float64, device=DEV)
    for b in range(0, nnz, 1 << 19):
        r, h, o = rows[b:b + (1 << 19)], H[ci[b:b + (1 << 19)].long()].double(), out[b:min(nnz, b + (1 << 19))].double()
        p = W[r].double() * h
        assert bool(((o - p.sum(1)).abs() <= (K + 4) * 2.0 ** -24 * p.abs().sum(1)).all())
        t = o[:, None] * h
        ref.index_add_(0, r, t)
        size.index_add_(0, r, t.abs())
    n = (rp[1:] - rp[:-1]).double()[:, None]
    assert bool(((Y[:-1].view(n_rows, K).double() - ref).abs() <= (n + 16) * 2.0 ** -24 * size).all())
