"""Plans that also serve the product with the dense factor, where their column tiles would hold little or nothing of it: the form
that is chosen, SDDMM and product against 64-bit sums, the same bits on every call, and the plan saved and loaded."""
import pytest
import torch

from sddmm_gpu_amd import capi, synth

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def even_rows(n_rows, n_cols, per_row, n_long=0, long_row=0):
    """per_row nonzeros a row, one in each of as many stretches of the columns; the first n_long rows have long_row."""
    g = torch.Generator(device=DEV).manual_seed(per_row)

    def rows(n, per):
        step = n_cols // per
        return (torch.arange(per, device=DEV) * step + torch.randint(0, step, (n, per), generator=g, device=DEV)).reshape(-1)
    cols = torch.cat([rows(n_long, long_row)] * (n_long > 0) + [rows(n_rows - n_long, per_row)]).int()
    deg = torch.full((n_rows,), per_row, device=DEV)
    deg[:n_long] = long_row
    return dict(n_rows=n_rows, n_cols=n_cols, nnz=int(cols.numel()), row_ptr=torch.cat([deg.new_zeros(1), deg.cumsum(0)]).int(), col_ind=cols)


def plan_of(d, K, **opts):
    return capi.Plan.from_device_csr(d["n_rows"], d["n_cols"], d["nnz"], d["row_ptr"].data_ptr(), d["col_ind"].data_ptr(), K,
                                     options=capi.PlanOptions.defaults(spmm_stream=1, ignore_env=1, **opts))


def check(d, K, plan, path):
    n_rows, nnz, ci, stream = d["n_rows"], d["nnz"], d["col_ind"].long(), torch.cuda.current_stream().cuda_stream
    rows = torch.repeat_interleave(torch.arange(n_rows, device=DEV), (d["row_ptr"][1:] - d["row_ptr"][:-1]).long())
    g = torch.Generator(device=DEV).manual_seed(K)
    W, H = torch.randn(n_rows, K, generator=g, device=DEV), torch.randn(d["n_cols"], K, generator=g, device=DEV)

    def run(p):
        out, Y = torch.full((nnz + 1,), 7.0, device=DEV), torch.full((n_rows * K + 1,), 7.0, device=DEV)
        p.execute(0, W.data_ptr(), H.data_ptr(), out.data_ptr(), stream)
        p.spmm(out.data_ptr(), H.data_ptr(), Y.data_ptr(), stream=stream)
        torch.cuda.synchronize()
        return out, Y
    out, Y = run(plan)
    assert float(out[-1]) == 7.0 and float(Y[-1]) == 7.0
    ref, size = torch.zeros(n_rows, K, dtype=torch.float64, device=DEV), torch.zeros(n_rows, K, dtype=torch.float64, device=DEV)
    for b in range(0, nnz, 1 << 19):
        r, h, o = rows[b:b + (1 << 19)], H[ci[b:b + (1 << 19)]].double(), out[b:min(nnz, b + (1 << 19))].double()
        p = W[r].double() * h
        assert bool(((o - p.sum(1)).abs() <= (K + 16) * 2.0 ** -24 * p.abs().sum(1)).all())
        ref.index_add_(0, r, o[:, None] * h)
        size.index_add_(0, r, (o[:, None] * h).abs())
    n = (d["row_ptr"][1:] - d["row_ptr"][:-1]).double()[:, None]  # a rounding per term of a row, however they are added up
    assert bool(((Y[:-1].view(n_rows, K).double() - ref).abs() <= (n + 16) * 2.0 ** -24 * size).all())
    plan.save(path)
    loaded = capi.Plan.load_device(path, n_rows, d["n_cols"], nnz, d["row_ptr"].data_ptr(), d["col_ind"].data_ptr(), K)
    assert loaded.spmm_form() == plan.spmm_form()
    for a, b in zip(run(loaded), (out, Y)):
        assert torch.equal(a, b)


# no row is long enough for the tiles, or a few are
@pytest.mark.parametrize("n_long", [0, 10])
@pytest.mark.parametrize("n_rows,n_cols,per_row,K", [(100000, 17770, 50, 32), (100000, 17770, 50, 64), (30000, 40000, 156, 50), (30000, 40000, 156, 64)])
def test_rows_too_short_for_the_tiles(tmp_path, n_rows, n_cols, per_row, K, n_long):
    d = even_rows(n_rows, n_cols, per_row, n_long, 5000)
    plan = plan_of(d, K)
    assert plan.spmm_form() == capi.SPMM_WALK and plan.info()["class_nnz"] == [d["nnz"], 0, 0]
    check(d, K, plan, tmp_path / "p.plan")


# ranks without a tile width of their own: the SDDMM is planned as in a plan without the product, whose rows are too short for tiles
@pytest.mark.parametrize("K", [96, 100])
def test_sddmm_as_without_the_product(tmp_path, K):
    d = synth.uniform_random(30000, 40000, 0.0039, K=4, device=DEV)
    plan = plan_of(d, K)
    alone = capi.Plan.from_device_csr(d["n_rows"], d["n_cols"], d["nnz"], d["row_ptr"].data_ptr(), d["col_ind"].data_ptr(), K,
                                      options=capi.PlanOptions.defaults(ignore_env=1))
    assert plan.spmm_form() == capi.SPMM_WALK and plan.info()["class_nnz"] == alone.info()["class_nnz"] == [d["nnz"], 0, 0]
    check(d, K, plan, tmp_path / "p.plan")


# ranks without a tile width of their own: tiles where the runs, times the share of the width that is used, are long enough
@pytest.mark.parametrize("kind,sizes,K,form", [
    ("bag_of_words", (20000, 17000, 480), 28, capi.SPMM_WALK),
    ("bag_of_words", (20000, 17000, 480), 36, capi.SPMM_WALK),
    ("bag_of_words", (20000, 17000, 480), 60, capi.SPMM_TILES),
    ("bag_of_words", (20000, 17000, 480), 100, capi.SPMM_WALK),
    ("bag_of_words", (20000, 17000, 480), 300, capi.SPMM_WALK),
    ("bag_of_words", (8000, 17000, 1500), 100, capi.SPMM_TILES),
    ("uniform_random", (20000, 12000, 0.05), 300, capi.SPMM_TILES),
    # (and where SDDMM + product, one after the other, gain by the tiles)
    ("bag_of_words", (3545, 33207, 1354), 59, capi.SPMM_WALK),  # few runs in an item
    ("bag_of_words", (6074, 42148, 2706), 55, capi.SPMM_TILES),
    ("recommender", (54211, 5638), 117, capi.SPMM_TILES),
    ("recommender", (96122, 7724), 75, capi.SPMM_WALK),
    ("recommender", (46295, 5912), 187, capi.SPMM_WALK),
    ("uniform_random", (35484, 2456, 0.0524), 189, capi.SPMM_WALK),
    ("recommender", (38596, 4965), 437, capi.SPMM_WALK),
    ("uniform_random", (8615, 6969, 0.0569), 450, capi.SPMM_TILES),
])
def test_form_by_the_length_of_runs(tmp_path, kind, sizes, K, form):
    d = getattr(synth, kind)(*sizes, K=4, device=DEV, **(dict(max_deg=int(0.9 * sizes[1])) if kind == "recommender" else {}))
    plan = plan_of(d, K)
    assert plan.spmm_form() == form
    check(d, K, plan, tmp_path / "p.plan")


# ranks without a tile width of their own, rows dealt out to groups of workgroups or a stream of several panels: no runs for the
# product, which walks the pattern and gives the same bits on every call
@pytest.mark.parametrize("sizes,K,opts", [((100000, 64, 512), 100, {}), ((100000, 64, 512), 300, {}), ((20000, 300, 1000), 100, dict(tile_size_x=250, tile_size_y=5000))])
def test_launches_without_runs(tmp_path, sizes, K, opts):
    d = synth.banded(*sizes, K=4, device=DEV)
    plan = plan_of(d, K, **opts)
    assert plan.spmm_form() == capi.SPMM_WALK and plan.info()["n_row_panels"] > 1
    check(d, K, plan, tmp_path / "p.plan")


# small matrices whose SDDMM alone would be gathered: beside a product it stays on tiles, for the product walks with its cut rows kept
@pytest.mark.parametrize("kind,sizes,K", [("banded", (4000, 60, 400), 96), ("banded", (10000, 40, 300), 64), ("rmat", (15, 800000), 100)])
def test_small_matrices_keep_the_walk(tmp_path, kind, sizes, K):
    d = getattr(synth, kind)(*sizes, K=4, device=DEV)
    alone = capi.Plan.from_device_csr(d["n_rows"], d["n_cols"], d["nnz"], d["row_ptr"].data_ptr(), d["col_ind"].data_ptr(), K,
                                      options=capi.PlanOptions.defaults(ignore_env=1))
    plan = plan_of(d, K)
    assert alone.info()["kernel"] == capi.KERNEL_ROW_GATHER and plan.spmm_form() == capi.SPMM_WALK
    check(d, K, plan, tmp_path / "p.plan")


# where rows are long the product takes the column tiles, without a dense core, unless the caller has said how that is to be found
@pytest.mark.parametrize("opts,core", [({}, False), (dict(dense_permille=250), True), (dict(dense_min_nnz=0), True), (dict(dense_blocks=1), True), (dict(dense_blocks=0), False)])
def test_dense_core_that_was_asked_for(opts, core):
    d = synth.recommender(44000, 5600, K=4, seed=5, device=DEV, max_deg=5000)
    plan = plan_of(d, 512, **opts)
    assert (plan.info()["dense_blocks"] > 0) == core and plan.spmm_form() == (capi.SPMM_CSR if core else capi.SPMM_TILES)


# columns that are used unevenly: the short rows, most of the nonzeros, are gathered beside the tiled ones, and the product keeps the walk
@pytest.mark.parametrize("scale,edges,K", [(17, 9369749, 32), (18, 14678406, 192)])
def test_rows_stay_split(tmp_path, scale, edges, K):
    d = synth.rmat(scale, edges, K=4, device=DEV)
    plan = plan_of(d, K)
    long_rows, _, short_rows = plan.info()["class_nnz"]
    assert long_rows > 0 and short_rows > 0 and plan.spmm_form() == capi.SPMM_WALK
    check(d, K, plan, tmp_path / "p.plan")
