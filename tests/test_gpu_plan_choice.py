"""Plans whose kernels the planner chooses by the busiest workgroup, by the lines a row of H lies in, or in thinner K slices than
the widest: what is chosen, the results with every source of the values against 64-bit sums, and calls that overlap in time."""
import pytest
import torch

from sddmm_gpu_amd import capi, synth

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("kind,sizes,K,kernel,k_slice", [
    ("banded", (4000, 60, 400), 96, capi.KERNEL_ROW_GATHER, 96),         # a few tiles hold most
    ("banded", (4000, 60, 400), 100, capi.KERNEL_ROW_GATHER, 100),
    ("banded", (4000, 60, 400), 1024, capi.KERNEL_LDS_TILE, 128),        # beyond the ranks that was measured at
    ("bag_of_words", (3000, 20000, 900), 11, capi.KERNEL_LDS_TILE, 11),  # 44-byte rows of H
    ("uniform_random", (16598, 15299, 0.0091), 96, capi.KERNEL_LDS_TILE, 96),  # runs of one and two: no slices of the planner's own up to K = 128
    ("uniform_random", (30281, 34347, 0.0063), 128, capi.KERNEL_LDS_TILE, 128),
    ("uniform_random", (30281, 34347, 0.0063), 256, capi.KERNEL_LDS_TILE, 32),
])
def test_choice(kind, sizes, K, kernel, k_slice):
    d = getattr(synth, kind)(*sizes, K=K, seed=3, device=DEV)
    nnz = d["nnz"]
    plan = capi.Plan.from_device_csr(d["n_rows"], d["n_cols"], nnz, d["row_ptr"].data_ptr(), d["col_ind"].data_ptr(), K,
                                     options=capi.PlanOptions.defaults(ignore_env=1))
    info = plan.info()
    assert info["kernel"] == kernel and info["k_slice"] == k_slice, info
    rows, cols, val = d["row_ind"].long(), d["col_ind"].long(), d["val"].double()
    dot = torch.empty(nnz, dtype=torch.float64, device=DEV)
    size = torch.empty_like(dot)
    for b in range(0, nnz, 1 << 18):
        p = d["W"][rows[b:b + (1 << 18)]].double() * d["H"][cols[b:b + (1 << 18)]].double()
        dot[b:b + (1 << 18)] = p.sum(1)
        size[b:b + (1 << 18)] = p.abs().sum(1)
    W, H, out = d["W"].data_ptr(), d["H"].data_ptr(), torch.empty(nnz + 1, device=DEV)
    stream = torch.cuda.current_stream().cuda_stream

    def check(run, ref, scale):
        out.fill_(7.0)
        run()
        torch.cuda.synchronize()
        # a rounding per product and sum, a few per K slice, and the scaling
        assert bool(((out[:nnz].double() - ref).abs() <= (K + 16) * 2.0 ** -24 * scale).all()) and float(out[nnz]) == 7.0

    check(lambda: plan.execute(0, W, H, out.data_ptr(), stream), dot, size)
    check(lambda: plan.execute(d["val"].data_ptr(), W, H, out.data_ptr(), stream), val * dot, val.abs() * size)
    plan.set_values(d["val"].data_ptr(), stream)
    check(lambda: plan.execute(0, W, H, out.data_ptr(), stream), val * dot, val.abs() * size)
    check(lambda: plan.execute_epilogue(0, W, H, out.data_ptr(), capi.EPILOGUE_RESIDUAL, stream), val - dot, val.abs() + size)


# runs of one to four: a plan of one launch keeps no scratch memory, so its calls may overlap in time
@pytest.mark.parametrize("kind,sizes,K", [
    ("uniform_random", (16598, 15299, 0.0091), 96),
    ("uniform_random", (30281, 34347, 0.0063), 128),
    ("uniform_random", (30000, 40000, 0.0039), 128),
    ("even", (120000, 5600, 34), 256),
    ("even", (100000, 17770, 50), 64),
])
def test_overlapping_calls(kind, sizes, K):
    if kind == "even":  # every row has one nonzero in each of as many stretches of the columns
        n_rows, n_cols, per_row = sizes
        g = torch.Generator(device=DEV).manual_seed(3)
        step = n_cols // per_row
        cols = (torch.arange(per_row, device=DEV) * step + torch.randint(0, step, (n_rows, per_row), generator=g, device=DEV)).reshape(-1).int()
        rp, W, H = (torch.arange(n_rows + 1, device=DEV) * per_row).int(), torch.randn(n_rows, K, generator=g, device=DEV), torch.randn(n_cols, K, generator=g, device=DEV)
    else:
        d = synth.uniform_random(*sizes, K=K, seed=3, device=DEV)
        n_rows, n_cols, rp, cols, W, H = (d[k] for k in ("n_rows", "n_cols", "row_ptr", "col_ind", "W", "H"))
    nnz = cols.numel()
    plan = capi.Plan.from_device_csr(n_rows, n_cols, nnz, rp.data_ptr(), cols.data_ptr(), K, options=capi.PlanOptions.defaults(ignore_env=1))
    assert plan.info()["n_launches"] == 1 and plan.info()["k_slice"] == K and plan.workspace_bytes() < 4 * nnz, plan.info()
    factors = [(W, H), (H.new_tensor(2.0) * W, H)]
    want = [torch.empty(nnz, device=DEV) for _ in factors]
    for (w, h), o in zip(factors, want):
        plan.execute(0, w.data_ptr(), h.data_ptr(), o.data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    streams, outs = [torch.cuda.Stream() for _ in range(4)], [torch.empty(nnz, device=DEV) for _ in range(4)]
    torch.cuda.synchronize()
    for _ in range(8):
        for i, (st, o) in enumerate(zip(streams, outs)):
            w, h = factors[i % 2]
            plan.execute(0, w.data_ptr(), h.data_ptr(), o.data_ptr(), st.cuda_stream)
    torch.cuda.synchronize()
    for i, o in enumerate(outs):
        assert torch.equal(o, want[i % 2])


def test_one_launch_that_was_asked_for():
    d = synth.uniform_random(30281, 34347, 0.0063, K=4, seed=3, device=DEV)
    plan = capi.Plan.from_device_csr(d["n_rows"], d["n_cols"], d["nnz"], d["row_ptr"].data_ptr(), d["col_ind"].data_ptr(), 256,
                                     options=capi.PlanOptions.defaults(fuse_slices=1, ignore_env=1))
    assert plan.info()["n_launches"] == 1 and plan.info()["k_slice"] == 128
