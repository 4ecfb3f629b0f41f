"""Row blocks: locally dense patterns whose SDDMM, row softmax and product run as whole 32 x 32 tiles on the matrix cores,
against the oracle and against the general path (dense_blocks = 0) of the same plan."""
import numpy as np
import pytest
import torch

from sddmm_gpu_amd import capi, synth
from test_gpu_parity import _dict_of, check

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def window(n, m, half, every, K, seed=3, empty=0, drop=0.0):
    """Columns within `half` of the diagonal, every `every`-th row and column full; rows from the `empty` last on left out,
    a share of the entries left out at random."""
    rng = np.random.default_rng(seed)
    r = np.repeat(np.arange(n), 2 * half + 1)
    c = r * m // n + np.tile(np.arange(-half, half + 1), n)
    g, h = np.arange(0, n, every), np.arange(0, m, every)
    r = np.concatenate([r, np.repeat(g, m), np.tile(np.arange(n), len(h))])
    c = np.concatenate([c, np.tile(np.arange(m), len(g)), np.repeat(h, n)])
    keep = (c >= 0) & (c < m) & (r < n - empty) & (rng.random(len(r)) >= drop)
    key = np.unique(r[keep].astype(np.int64) * m + c[keep])
    return _dict_of(n, m, key // m, key % m, K, rng)


def plans(d, K, values=True, product=1, **kw):
    dev = torch.device(DEV)
    t = {k: d[k].to(dev) for k in ("row_ptr", "col_ind", "val", "W", "H")}
    out = []
    for dense in (2, 0):  # (2: also where few blocks make the general path the faster one)
        plan = capi.Plan.from_device_csr(d["n_rows"], d["n_cols"], d["nnz"], t["row_ptr"].data_ptr(), t["col_ind"].data_ptr(), K,
                                         options=capi.PlanOptions.defaults(spmm_stream=product, ignore_env=1, dense_blocks=dense, **kw))
        if values:
            plan.set_values(t["val"].data_ptr())
        out.append(plan)
    return t, out


def is_blocks(plan, d):
    return plan.info()["dense_nnz"] == d["nnz"] and plan.spmm_form() == capi.SPMM_BLOCKS


# n = 1500: the full rows' blocks are several units (47 tiles); 700: they are whole (22); 33 and 65: one row behind a whole
# block; wide and narrow matrices; K at every number of steps
CASES = [(1500, 1500, 24, 97, 64), (1500, 1500, 150, 211, 128), (700, 700, 40, 50, 32), (700, 900, 60, 60, 48), (1300, 1100, 33, 400, 80),
         (33, 64, 31, 6, 96), (65, 65, 64, 16, 112), (2100, 2100, 300, 1000, 64), (32, 200, 10, 1, 64)]


@pytest.mark.parametrize("n,m,half,every,K", CASES)
def test_row_blocks(oracle, n, m, half, every, K):
    d = window(n, m, half, every, K, empty=5 if n > 1000 else 0, drop=0.1 if K == 80 else 0.0)
    t, (plan, general) = plans(d, K)
    assert is_blocks(plan, d) and general.info()["dense_nnz"] == 0, plan.info()
    dev = torch.device(DEV)
    W, H = t["W"].data_ptr(), t["H"].data_ptr()
    deg = np.diff(d["row_ptr"].numpy())

    def run(f):
        out = torch.full((d["nnz"],), float("nan"), device=dev)
        f(out.data_ptr())
        torch.cuda.synchronize()
        return out
    # out = val * dot, with the plan's values, with the call's, without; the residual
    out = run(lambda o: plan.execute(0, W, H, o))
    check(d, out.cpu().numpy(), oracle, K=K)
    assert torch.equal(out, run(lambda o: plan.execute(t["val"].data_ptr(), W, H, o)))
    _, (bare, bare_general) = plans(d, K, values=False)
    dots = run(lambda o: bare.execute(0, W, H, o))
    res = run(lambda o: plan.execute_epilogue(0, W, H, o, capi.EPILOGUE_RESIDUAL))
    assert torch.equal(dots * t["val"], out) and torch.equal(t["val"] - dots, res)
    # the softmax: within what the scores' difference moves it (1e-5 sqrt(K) of the sum of magnitudes, absolute)
    soft, want = run(lambda o: plan.execute_softmax(0, W, H, o)), run(lambda o: general.execute_softmax(0, W, H, o))
    scores = out.cpu().numpy()
    row = np.repeat(np.arange(n), deg)
    mag = (np.abs(d["W"].numpy()[row]) * np.abs(d["H"].numpy()[d["col_ind"].numpy()])).sum(1) * np.abs(d["val"].numpy())
    bound = 1e-5 + 4e-6 * np.sqrt(K) * (mag + np.maximum.reduceat(mag, d["row_ptr"].numpy()[:-1][deg > 0]).repeat(deg[deg > 0]))
    assert np.all(np.abs(soft.cpu().numpy() - want.cpu().numpy()) <= bound * want.cpu().numpy() + 1e-30)
    assert np.allclose(soft.cpu().numpy(), oracle.row_softmax(d["row_ptr"].numpy(), scores), rtol=1e-5, atol=1e-30)
    assert torch.equal(soft, run(lambda o: plan.execute_softmax(0, W, H, o)))
    # the product
    x = torch.randn(d["nnz"], generator=torch.Generator().manual_seed(K))
    xd = x.to(dev)
    Y = torch.full((n, K), float("nan"), device=dev)
    plan.spmm(xd.data_ptr(), H, Y.data_ptr())
    Y2 = torch.full((n, K), float("nan"), device=dev)
    nbytes = plan.workspace_bytes()
    ws = torch.full((nbytes // 4,), float("nan"), device=dev)
    plan.spmm(xd.data_ptr(), H, Y2.data_ptr(), ws.data_ptr(), nbytes)
    torch.cuda.synchronize()
    assert torch.equal(Y, Y2)
    ref, absum = oracle.spmm_csr(d["row_ptr"].numpy(), d["col_ind"].numpy(), x.numpy(), d["H"].numpy(), with_abs=True)
    assert np.all(np.abs(Y.cpu().numpy().astype(np.float64) - ref) <= 1e-5 * np.sqrt(np.maximum(deg, 1))[:, None] * absum)
    assert np.all(Y.cpu().numpy()[deg == 0] == 0)


@pytest.mark.parametrize("K", [64, 80])
@pytest.mark.parametrize("what", ["infinity", "nan", "overflow", "tiny"])
def test_row_blocks_values_that_parts_do_not_hold(oracle, what, K):
    """Operands with infinities, NaNs, products beyond the range, bits under bf16's smallest subnormal: those results are
    what fp32 gives, the others unchanged."""
    d = window(1500, 1500, 30, 400, K)
    W, H = d["W"].clone(), d["H"].clone()
    x = torch.randn(d["nnz"], generator=torch.Generator().manual_seed(1))
    if what == "infinity":
        W[100, 3] = float("inf"); H[640, 5] = -float("inf"); x[5000] = float("inf")
    elif what == "nan":
        W[100, 3] = float("nan"); H[640, 5] = float("nan"); x[5000] = float("nan")
    elif what == "overflow":
        W[100] *= 1e30; H[110] *= 1e30; H[640] *= 3e38; x[20000] = 3e38
    else:
        W[100:140] *= 1e-37; H[640:700] *= 1e-37; x[20000:30000] *= 1e-38
    d = dict(d, W=W, H=H)
    t, (plan, general) = plans(d, K, values=False)
    assert is_blocks(plan, d)
    dev = torch.device(DEV)
    xd = x.to(dev)
    got, want = [], []
    for p, into in ((plan, got), (general, want)):
        out = torch.full((d["nnz"],), 7.0, device=dev); Y = torch.full((1500, K), 7.0, device=dev)
        p.execute(0, t["W"].data_ptr(), t["H"].data_ptr(), out.data_ptr())
        p.spmm(xd.data_ptr(), t["H"].data_ptr(), Y.data_ptr())
        torch.cuda.synchronize()
        into += [out.double().cpu(), Y.double().cpu()]
    row, col = d["row_ind"].long(), d["col_ind"].long()
    size = (W.double().abs()[row] * H.double().abs()[col]).sum(1)
    ysize = torch.zeros(1500, K, dtype=torch.float64).index_add_(0, row, x.double().abs()[:, None] * H.double().abs()[col])
    for g, w, s in zip(got, want, (size, ysize)):
        finite = torch.isfinite(w) & (s < 1e38)  # (beyond, an order of summation may overflow where another does not)
        assert bool((torch.isfinite(g) | ~finite).all()) and bool((torch.isnan(g) == torch.isnan(w))[~torch.isfinite(s)].all())
        assert bool(((g - w).abs() <= 1e-5 * s + 1e-44)[finite].all())
        assert bool((g == w)[torch.isinf(w) & ~torch.isfinite(s)].all())


def test_row_blocks_masked_scores():
    """A score of minus infinity (a masked entry) has weight 0; a row of nothing else is NaN."""
    d = window(700, 700, 40, 50, 64)
    t, (plan, _) = plans(d, 64, values=False)
    bias = torch.zeros(d["nnz"]); rp = d["row_ptr"].numpy()
    bias[rp[10]:rp[11]:2] = -float("inf"); bias[rp[33]:rp[34]] = -float("inf"); bias[rp[50]:rp[51]:3] = -float("inf")
    dev = torch.device(DEV)
    out = torch.empty(d["nnz"], device=dev)
    nbytes = plan.workspace_bytes()
    ws = torch.empty(nbytes // 4, device=dev)
    plan.execute_ws(bias.to(dev).data_ptr(), t["W"].data_ptr(), t["H"].data_ptr(), out.data_ptr(),
                    ws.data_ptr(), nbytes, form=capi.EPILOGUE_RESIDUAL | capi.FORM_SOFTMAX)
    torch.cuda.synchronize()
    s = (bias.double() - (d["W"].double()[d["row_ind"].long()] * d["H"].double()[d["col_ind"].long()]).sum(1))
    for r in (10, 33, 50, 51):
        got, want = out[rp[r]:rp[r + 1]].double().cpu(), torch.softmax(s[rp[r]:rp[r + 1]], 0)
        assert torch.allclose(got, want, rtol=1e-4, atol=1e-12, equal_nan=True)


def test_row_blocks_are_left_to_patterns_that_are_dense():
    """Not: a band filled by a third, a pattern with an entry twice, ranks without such a kernel, layouts a caller chose, small
    matrices where the product does not use them."""
    rng = np.random.default_rng(2)
    d = window(700, 700, 40, 50, 64, drop=0.7)
    assert plans(d, 64)[1][0].info()["dense_nnz"] == 0
    d = window(700, 700, 40, 50, 64)
    for K in (16, 50, 144):
        e = dict(d, W=torch.rand(700, K), H=torch.rand(700, K))
        assert plans(e, K)[1][0].info()["dense_nnz"] == 0
    assert plans(d, 64, tile_size_x=100)[1][0].info()["dense_nnz"] == 0
    key = np.sort(np.concatenate([d["row_ind"].numpy().astype(np.int64) * 700 + d["col_ind"].numpy(), [5 * 700 + 7]]))
    twice = _dict_of(700, 700, key // 700, key % 700, 64, rng)
    assert plans(twice, 64)[1][0].info()["dense_nnz"] == 0
    assert plans(d, 64, product=0)[1][0].info()["dense_nnz"] == 0
    large = window(2100, 2100, 300, 1000, 64)
    assert plans(large, 64, product=0)[1][0].info()["dense_nnz"] == large["nnz"]


@pytest.mark.parametrize("n", [700, 1500])
def test_row_blocks_saved_and_loaded(tmp_path, n):
    d = window(n, n, 40, 100, 64)
    t, (plan, _) = plans(d, 64)
    path = str(tmp_path / "p.bin")
    plan.save(path)
    loaded = capi.Plan.load_device(path, n, n, d["nnz"], t["row_ptr"].data_ptr(), t["col_ind"].data_ptr(), 64)
    assert is_blocks(loaded, d)
    dev = torch.device(DEV)
    for f in (lambda p, o, Y: p.execute(0, t["W"].data_ptr(), t["H"].data_ptr(), o.data_ptr()),
              lambda p, o, Y: p.execute_softmax(0, t["W"].data_ptr(), t["H"].data_ptr(), o.data_ptr()),
              lambda p, o, Y: p.spmm(t["val"].data_ptr(), t["H"].data_ptr(), Y.data_ptr())):
        got = []
        for p in (plan, loaded):
            o = torch.zeros(d["nnz"], device=dev); Y = torch.zeros(n, 64, device=dev)
            f(p, o, Y)
            torch.cuda.synchronize()
            got.append((o, Y))
        assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("n,half,every,K,blocks", [(559, 83, 24, 80, False), (1000, 40, 60, 32, False), (2000, 100, 100, 128, True), (334, 167, 38, 32, True)])
def test_few_row_blocks_only_where_they_are_faster(n, half, every, K, blocks):
    """Left to itself the planner takes the general path where one workgroup's tiles would be all that runs."""
    d = window(n, n, half, every, K)
    t = {k: d[k].to(torch.device(DEV)) for k in ("row_ptr", "col_ind")}
    plan = capi.Plan.from_device_csr(n, n, d["nnz"], t["row_ptr"].data_ptr(), t["col_ind"].data_ptr(), K,
                                     options=capi.PlanOptions.defaults(spmm_stream=1, ignore_env=1))
    assert is_blocks(plan, d) == blocks


@pytest.mark.parametrize("dense", [-1, 0, 1, 2, 3])
def test_what_dense_blocks_asks_for(dense):
    """Every value but 0 leaves the dense core on (-1: from K = 384 on), and row blocks; 2 takes row blocks where they are few, too."""
    def plan(d, K, **kw):
        t = {k: d[k].to(torch.device(DEV)) for k in ("row_ptr", "col_ind")}
        return capi.Plan.from_device_csr(d["n_rows"], d["n_cols"], d["nnz"], t["row_ptr"].data_ptr(), t["col_ind"].data_ptr(), K,
                                         options=capi.PlanOptions.defaults(ignore_env=1, dense_blocks=dense, **kw))
    ratings = synth.make(3, 0.03, K=4, device=DEV)
    for K in (128, 512):
        core = plan(ratings, K, dense_min_nnz=1000, split_min_nnz=0).info()["dense_nnz"]
        assert (core > ratings["nnz"] // 10) == (dense > 0 or (dense < 0 and K == 512)) and core < ratings["nnz"]
    many, few = window(2100, 2100, 300, 1000, 32), window(1000, 1000, 40, 60, 32)
    assert is_blocks(plan(many, 32, spmm_stream=1), many) == (dense != 0)
    assert is_blocks(plan(few, 32, spmm_stream=1), few) == (dense == 2)


@pytest.mark.parametrize("n,half,every,K", [(700, 40, 50, 64), (1500, 30, 400, 80)])
def test_product_with_small_and_large_weights(oracle, n, half, every, K):
    """X times a power of two gives Y times it, bit for bit, where nothing is subnormal: one path for weights of any size.
    At the ends of the range the product is right."""
    d = window(n, n, half, every, K)
    t, (plan, _) = plans(d, K, values=False)
    assert is_blocks(plan, d)
    row, col, H = d["row_ind"].long(), d["col_ind"].long(), d["H"].double()

    def product(x):
        xd, Y = x.to(DEV), torch.full((n, K), float("nan"), device=DEV)
        plan.spmm(xd.data_ptr(), t["H"].data_ptr(), Y.data_ptr())
        torch.cuda.synchronize()
        return Y.cpu()
    g = torch.Generator().manual_seed(5)
    x = (0.5 + 0.5 * torch.rand(d["nnz"], generator=g)) * (2 * torch.randint(0, 2, (d["nnz"],), generator=g) - 1)
    Y = product(x)
    for e in (-112, -60, 40, 70):
        assert torch.equal(product(torch.ldexp(x, torch.tensor(e))), torch.ldexp(Y, torch.tensor(e))), e
    # a few that vanish beside the others
    mixed = torch.where(torch.rand(d["nnz"], generator=g) < 0.01, torch.ldexp(x, torch.tensor(-112)), x)
    assert torch.equal(product(torch.ldexp(mixed, torch.tensor(30))), torch.ldexp(product(mixed), torch.tensor(30)))
    deg = np.diff(d["row_ptr"].numpy())
    for e in (-147, -125, 78, 83, 85, 88, 110, 118):
        xe = torch.ldexp(x, torch.tensor(e))
        mag = torch.zeros(n, K, dtype=torch.float64).index_add_(0, row, xe.double().abs()[:, None] * H.abs()[col])
        ref = torch.zeros(n, K, dtype=torch.float64).index_add_(0, row, xe.double()[:, None] * H[col])
        bound = 1e-5 * torch.from_numpy(np.sqrt(np.maximum(deg, 1)))[:, None] * mag + 2.0 ** -149 * torch.from_numpy(deg)[:, None]
        assert bool(((product(xe).double() - ref).abs() <= bound).all()), e


@pytest.mark.parametrize("n,half,every,K", [(700, 40, 50, 64), (1500, 30, 400, 80), (700, 60, 60, 128)])
def test_small_values_in_dense_factors(n, half, every, K):
    """W, H times a power of two: the results times it, bit for bit, where nothing is subnormal; one small value among large
    ones changes what it should."""
    d = window(n, n, half, every, K)
    t, (plan, _) = plans(d, K, values=False)
    assert is_blocks(plan, d)
    row, col = d["row_ind"].long(), d["col_ind"].long()
    g = torch.Generator().manual_seed(6)
    x = 0.5 + torch.rand(d["nnz"], generator=g)
    W, H = (0.5 + torch.rand(n, K, generator=g) for _ in range(2))

    def both(W, H, x):
        out, Y = torch.full((d["nnz"],), float("nan"), device=DEV), torch.full((n, K), float("nan"), device=DEV)
        W, H, x = W.to(DEV), H.to(DEV), x.to(DEV)
        plan.execute(0, W.data_ptr(), H.data_ptr(), out.data_ptr())
        plan.spmm(x.data_ptr(), H.data_ptr(), Y.data_ptr())
        torch.cuda.synchronize()
        return out.cpu(), Y.cpu()
    s = lambda v, e: torch.ldexp(v, torch.tensor(e))
    out, Y = both(W, H, x)
    for ew, eh, ex in ((0, -112, 0), (-112, 0, 0), (-112, 80, 0), (30, -115, 20)):
        o, y = both(s(W, ew), s(H, eh), s(x, ex))
        assert torch.equal(o, s(out, ew + eh)) and (eh > 60 or torch.equal(y, s(Y, eh + ex))), (ew, eh)
    # small values among others, and others so large that they leave the range once scaled
    for what, e in (("H", 0), ("W", 0), ("H", 46), ("H", 100), ("W", 100)):
        W2, H2 = s(W, e), H.clone()
        (H2 if what == "H" else W2)[n // 2, 3:20] = s(H[n // 2, 3:20], -115)
        if what == "H":
            H2[:, K - 1] = s(H[:, K - 1], -140)
        o, y = both(W2, H2, s(x, e))
        size = (W2.double()[row] * H2.double()[col]).sum(1)
        ysize = torch.zeros(n, K, dtype=torch.float64).index_add_(0, row, s(x, e).double()[:, None] * H2.double()[col])
        # (one rounding per product and sum, in any order)
        bound = (torch.from_numpy(np.diff(d["row_ptr"].numpy())) + 4)[:, None] * 2.0 ** -24 * ysize + 1e-42
        assert bool(((o.double() - size).abs() <= (K + 4) * 2.0 ** -24 * size).all()) and bool(((y.double() - ysize).abs() <= bound).all()), (what, e)


# Full rows of one piece of 16,384 entries, of two with one entry in the last, of three: their softmax joins the pieces' records.
@pytest.mark.parametrize("m", [16384, 16385, 32769, 40000])
def test_full_rows_in_pieces(oracle, tmp_path, m):
    n, K = 608, 64
    rng = np.random.default_rng(m)
    full = np.arange(0, n, 19)  # (32 rows: a block)
    r, c = np.repeat(np.arange(n), 49), (np.arange(n)[:, None] + np.arange(49)).reshape(-1)
    keep = ~np.isin(r, full)
    key = np.unique(np.concatenate([r[keep].astype(np.int64) * m + c[keep], (full[:, None].astype(np.int64) * m + np.arange(m)).reshape(-1)]))
    d = _dict_of(n, m, key // m, key % m, K, rng)
    t, (plan, general) = plans(d, K)
    assert is_blocks(plan, d), plan.info()
    W, H = t["W"].data_ptr(), t["H"].data_ptr()
    scores = torch.empty(d["nnz"], device=DEV)
    plan.execute(0, W, H, scores.data_ptr())
    want = oracle.row_softmax(d["row_ptr"].numpy(), scores.cpu().numpy())
    path = tmp_path / "blocks.plan"
    plan.save(path)
    loaded = capi.Plan.load_device(path, n, m, d["nnz"], t["row_ptr"].data_ptr(), t["col_ind"].data_ptr(), K, keep=t)
    first = None
    for p in (plan, loaded):
        nbytes = p.workspace_bytes()
        ws = torch.full((nbytes // 4 + 1,), float("nan"), device=DEV)
        for run in (lambda o: p.execute_softmax(0, W, H, o), lambda o: p.execute_ws(0, W, H, o, ws.data_ptr(), nbytes, capi.FORM_SOFTMAX)):
            out = torch.full((d["nnz"],), float("nan"), device=DEV)
            run(out.data_ptr())
            torch.cuda.synchronize()
            first = out if first is None else first
            assert torch.equal(out, first)
    assert np.allclose(first.cpu().numpy(), want, rtol=1e-5, atol=1e-30)
