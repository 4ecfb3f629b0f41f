"""The row softmax where its units meet the rows: every share size, rows at the limits of each kind of work, huge rows
that begin, cross and end units, runs of empty rows, in place; against the oracle (relative 1e-5 per entry)."""
import numpy as np
import pytest
import torch

from sddmm_gpu_amd import capi
from test_gpu_fused import softmax_ok

pytestmark = pytest.mark.gpu

LIMITS = [8, 9, 96, 97, 512, 513, 1024, 1025, 4088, 4089, 17400, 17401, 20000, 1, 70000, 3]


# (entries of filler rows, their length): totals from a few thousand to 20 million on the kernel's scale, so shares of 64 to 4096
@pytest.mark.parametrize("filler,length", [(0, 1), (40000, 7), (300000, 50), (700000, 300), (2000000, 40), (4000000, 700), (16000000, 100)])
def test_limits_among_fillers(oracle, filler, length):
    rng = np.random.default_rng(filler + length)
    n = filler // length
    lens = np.concatenate([np.full(n // 2, length), np.repeat(LIMITS, 2), np.zeros(3000), np.full(n - n // 2, length), rng.permutation(LIMITS),
                           np.zeros(500), [1025] * 9, [17401]]).astype(np.int64)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    x = rng.normal(0, 4, rp[-1]).astype(np.float32)
    x[rp[np.flatnonzero(lens == 70000)] + 69999] = 60.0
    want = oracle.row_softmax(rp, x)
    xd, rpd = torch.from_numpy(x).cuda(), torch.from_numpy(rp).cuda()
    out = torch.full((len(x) + 1,), float("nan"), device="cuda")
    capi.row_softmax(len(lens), rpd.data_ptr(), xd.data_ptr(), out.data_ptr())
    capi.row_softmax(len(lens), rpd.data_ptr(), xd.data_ptr(), xd.data_ptr())
    torch.cuda.synchronize()
    softmax_ok(out[:-1].cpu().numpy(), want)
    assert torch.equal(out[:-1], xd) and bool(torch.isnan(out[-1]))


@pytest.mark.parametrize("at", [0, 5, 2000, 19999])
@pytest.mark.parametrize("value", ["nan", "inf", "-inf"])
def test_special_values_stay_in_their_row(oracle, at, value):
    lens = np.array([30, 20000, 700, 0, 5, 3000], dtype=np.int64)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    x = np.random.default_rng(3).normal(0, 2, rp[-1]).astype(np.float32)
    want = oracle.row_softmax(rp, x)
    x[rp[1] + at] = float(value)
    out = torch.empty(len(x), device="cuda")
    xd, rpd = torch.from_numpy(x).cuda(), torch.from_numpy(rp).cuda()
    capi.row_softmax(len(lens), rpd.data_ptr(), xd.data_ptr(), out.data_ptr())
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    touched = slice(rp[1], rp[2])
    softmax_ok(np.delete(got, np.r_[touched]), np.delete(want, np.r_[touched]))
    if value == "-inf":
        softmax_ok(got[touched], oracle.row_softmax(rp, x)[touched])
    else:
        assert np.isnan(got[touched]).sum() >= 1


# Short rows alone and among longer ones in shares of 64, both sides of the scale's lines between shares (entries + 4 rows = 2^18,
# 2^19, 2^20, 2^22), and the smallest matrices.
@pytest.mark.parametrize("lens", [[0], [1], [1, 0, 0, 2], [1] * 3000, [8] * 3000, [8, 8, 8, 8, 8, 20, 20, 20] * 200, [8, 8, 8, 8, 8, 8, 20, 20, 20] * 200,
                                  [1, 9, 1, 1, 1, 1, 1, 1, 1, 1, 1] * 200, [3, 0, 96, 0, 1, 97, 7, 513, 8, 9] * 40, [5] * 29126 + [6], [5] * 29126 + [7],
                                  [28] * 16384, [28] * 16384 + [0], [28] * 32768, [28] * 32768 + [1], [60] * 65535 + [59], [60] * 65536])
def test_short_rows_and_lines_between_shares(oracle, lens):
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    x = np.random.default_rng(len(lens)).normal(0, 4, rp[-1]).astype(np.float32)
    xd, rpd = torch.from_numpy(x).cuda(), torch.from_numpy(rp).cuda()
    out = torch.full((len(x) + 1,), float("nan"), device="cuda")
    capi.row_softmax(len(lens), rpd.data_ptr(), xd.data_ptr() if len(x) else out.data_ptr(), out.data_ptr())
    torch.cuda.synchronize()
    softmax_ok(out[:-1].cpu().numpy(), oracle.row_softmax(rp, x))
    assert bool(torch.isnan(out[-1]))


# Pieces are 256 entries without filler rows and 2048 with them; a lane merges every 64th piece of a row.
@pytest.mark.parametrize("filler,masked", [(0, [(0, 700)]), (0, [(16384, 18000)]), (0, [(0, 19999)]), (0, [(500, 20000)]),
                                           (1200000, [(0, 5000)]), (1200000, [(0, 9000), (12000, 20000)])])
def test_huge_row_with_pieces_all_masked(oracle, filler, masked):
    """Pieces of a huge row in which every entry is minus infinity have weight 0 and leave the others theirs."""
    lens = np.array([30, 20000, 700] + [300] * (filler // 300), dtype=np.int64)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    x = np.random.default_rng(3).normal(0, 2, rp[-1]).astype(np.float32)
    for b, e in masked:
        x[rp[1] + b:rp[1] + e] = -np.inf
    out = torch.empty(len(x), device="cuda")
    xd, rpd = torch.from_numpy(x).cuda(), torch.from_numpy(rp).cuda()
    capi.row_softmax(len(lens), rpd.data_ptr(), xd.data_ptr(), out.data_ptr())
    torch.cuda.synchronize()
    softmax_ok(out.cpu().numpy(), oracle.row_softmax(rp, x))


@pytest.mark.parametrize("value", [float("nan"), -float("inf")])
def test_huge_row_without_weights(oracle, value):
    """A huge row of nothing but minus infinity, and one with a piece of nothing but NaN, are NaN throughout."""
    lens = np.array([30, 20000, 700], dtype=np.int64)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    x = np.random.default_rng(3).normal(0, 2, rp[-1]).astype(np.float32)
    want = oracle.row_softmax(rp, x)
    b, e = (0, 20000) if np.isinf(value) else (20 * 256 - 34, 22 * 256 - 34)  # (the row starts at 30 + 4 on the kernel's scale)
    x[rp[1] + b:rp[1] + e] = value
    out = torch.empty(len(x), device="cuda")
    xd, rpd = torch.from_numpy(x).cuda(), torch.from_numpy(rp).cuda()
    capi.row_softmax(len(lens), rpd.data_ptr(), xd.data_ptr(), out.data_ptr())
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert np.isnan(got[rp[1]:rp[2]]).all()
    softmax_ok(np.delete(got, np.r_[rp[1]:rp[2]]), np.delete(want, np.r_[rp[1]:rp[2]]))


# (the grids grow at 2^18 and at 2^20 rows; a row of 600,000 entries alone is more pieces than the smaller merge grid has workgroups)
@pytest.mark.parametrize("rows", [2 ** 18 - 40, 2 ** 18, 2 ** 20 - 40, 2 ** 20])
def test_many_rows(oracle, rows):
    rng = np.random.default_rng(rows)
    lens = rng.integers(0, 4, rows)
    lens[[5, rows // 2, rows // 2 + 1, rows - 2]] = 600000, 17401, 3000, 40000
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    x = rng.normal(0, 4, rp[-1]).astype(np.float32)
    xd, rpd = torch.from_numpy(x).cuda(), torch.from_numpy(rp).cuda()
    out = torch.full((len(x) + 1,), float("nan"), device="cuda")
    capi.row_softmax(rows, rpd.data_ptr(), xd.data_ptr(), out.data_ptr())
    torch.cuda.synchronize()
    softmax_ok(out[:-1].cpu().numpy(), oracle.row_softmax(rp, x))
    assert bool(torch.isnan(out[-1]))


# A plan knows its longest row and leaves the kernel that joins the pieces of huge rows out where there are none: the longest row that
# is none, the shortest that is one, one of several pieces.
@pytest.mark.parametrize("longest", [17400, 17401, 40000])
@pytest.mark.parametrize("kernel", [capi.KERNEL_ROW_GATHER, capi.KERNEL_LDS_TILE, capi.KERNEL_HYBRID])
def test_longest_row_of_a_plan(oracle, tmp_path, kernel, longest):
    rng = np.random.default_rng(longest)
    n_cols, K = 40000, 32
    lens = np.concatenate([rng.integers(0, 200, 150), [longest, 0, 1100], rng.integers(0, 200, 150)])
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    ci = np.concatenate([np.sort(rng.choice(n_cols, c, replace=False)) for c in lens]).astype(np.int32)
    n, nnz = len(lens), len(ci)
    rpd, cid = torch.from_numpy(rp).cuda(), torch.from_numpy(ci).cuda()
    g = torch.Generator(device="cuda")
    g.manual_seed(longest)
    W, H, val = (torch.randn(*s, generator=g, device="cuda") for s in ((n, K), (n_cols, K), (nnz,)))
    plan = capi.Plan.from_device_csr(n, n_cols, nnz, rpd.data_ptr(), cid.data_ptr(), K, options=capi.PlanOptions.defaults(kernel=kernel, dense_blocks=0, ignore_env=1))
    plan.set_values(val.data_ptr())
    scores = torch.empty(nnz, device="cuda")
    plan.execute(0, W.data_ptr(), H.data_ptr(), scores.data_ptr())
    path = tmp_path / "softmax.plan"
    plan.save(path)
    loaded = capi.Plan.load_device(path, n, n_cols, nnz, rpd.data_ptr(), cid.data_ptr(), K, keep=(rpd, cid))
    want = oracle.row_softmax(rp, scores.cpu().numpy())
    for p in (plan, loaded):
        nbytes = p.workspace_bytes()
        ws = torch.full((nbytes // 4 + 1,), float("nan"), device="cuda")
        for run in (lambda o: p.execute_softmax(0, W.data_ptr(), H.data_ptr(), o),
                    lambda o: p.execute_ws(0, W.data_ptr(), H.data_ptr(), o, ws.data_ptr(), nbytes, capi.FORM_SOFTMAX)):
            out = torch.full((nnz,), float("nan"), device="cuda")
            run(out.data_ptr())
            torch.cuda.synchronize()
            softmax_ok(out.cpu().numpy(), want)
