"""The dense-block launch multiplies operands cut into three bf16 parts.  Values that three parts hold exactly give an
error of fp32 size; infinities, NaNs, sums beyond the range and values with bits below bf16's smallest subnormal give
what fp32 arithmetic gives."""
import numpy as np
import pytest
import torch

from sddmm_gpu_amd import capi, synth

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def dense_plan(K, scale=0.03):
    d = synth.make(3, scale, K=K, device=DEV)
    opts = capi.PlanOptions.defaults(kernel=capi.KERNEL_HYBRID, dense_blocks=1, dense_min_nnz=1000, split_min_nnz=0, ignore_env=1)
    plan = capi.Plan.from_device_csr(d["n_rows"], d["n_cols"], d["nnz"], d["row_ptr"].data_ptr(), d["col_ind"].data_ptr(), K, options=opts)
    assert plan.info()["dense_nnz"] > d["nnz"] // 10
    return d, plan


def product(d, plan, W, H):
    out = torch.full((d["nnz"],), 7.0, device=DEV)
    plan.execute(0, W.data_ptr(), H.data_ptr(), out.data_ptr())
    torch.cuda.synchronize()
    rows = torch.repeat_interleave(torch.arange(d["n_rows"], device=DEV), torch.diff(d["row_ptr"].long()))
    cols = d["col_ind"].long()
    ref = torch.empty(d["nnz"], dtype=torch.float64, device=DEV)
    mag = torch.empty_like(ref)  # sum of the products' magnitudes
    for b in range(0, d["nnz"], 1 << 18):
        p = W[rows[b:b + (1 << 18)]].double() * H[cols[b:b + (1 << 18)]].double()
        ref[b:b + (1 << 18)] = p.sum(1)
        mag[b:b + (1 << 18)] = p.abs().sum(1)
    return out, ref, mag, rows, cols


# Full 24-bit significands; 2^-105 .. 2^-125 puts the third, then the second part below bf16's smallest subnormal
# (2^-133), 2^-140 is subnormal itself; H brings the products back into the range.
@pytest.mark.parametrize("K", [96, 512])
@pytest.mark.parametrize("we,he", [(0, 0), (60, -70), (-100, 90), (-108, 100), (-125, 110), (-140, 120)])
def test_magnitudes(K, we, he):
    d, plan = dense_plan(K)
    g = torch.Generator(device=DEV); g.manual_seed(3)
    W = torch.ldexp(torch.randn(d["n_rows"], K, generator=g, device=DEV), torch.tensor(we, device=DEV))
    H = torch.ldexp(torch.randn(d["n_cols"], K, generator=g, device=DEV), torch.tensor(he, device=DEV))
    out, ref, mag, _, _ = product(d, plan, W, H)
    assert bool((torch.abs(out.double() - ref) <= (K + 4) * 2.0 ** -24 * mag).all())  # one rounding per product and sum


def test_infinities_nans_and_sums_beyond_the_range():
    K = 128
    d, plan = dense_plan(K)
    g = torch.Generator(device=DEV); g.manual_seed(4)
    W = torch.randn(d["n_rows"], K, generator=g, device=DEV).abs() + 0.1
    H = torch.randn(d["n_cols"], K, generator=g, device=DEV).abs() + 0.1
    low_nan = torch.tensor([0x7f800001], dtype=torch.int32, device=DEV).view(torch.float32)  # payload in the last bit
    W[0::7, 5] = float("inf")
    W[1::7, 9] = float("-inf")
    W[2::7, 100] = low_nan
    H[0::5, 77] = float("inf")
    H[1::5, 3] = 1.0e20  # 10^40 where it meets the next line, small elsewhere, so no second infinity meets -inf
    W[3::7, 3] = 1.0e20
    out, ref, mag, rows, cols = product(d, plan, W, H)
    ref32 = ref.float()  # beyond the range: infinity
    assert torch.equal(torch.isnan(out), torch.isnan(ref32))
    inf = torch.isinf(ref32)
    assert torch.equal(out[inf], ref32[inf]) and bool(inf.any())
    fin = torch.isfinite(ref32)
    assert bool((torch.abs(out.double() - ref)[fin] <= (K + 4) * 2.0 ** -24 * mag[fin]).all())


@pytest.mark.parametrize("K", [96, 512])
@pytest.mark.parametrize("kind", ["dense", "positive", "four a row", "one a row", "small"])
def test_no_less_precise_than_fp32_sums(K, kind):
    """The error against 64 bits beside that of fp32 sums which round once for every two products (what an fp32 matrix
    instruction of two elements does at best), also where a row of W has one or a few elements, so that each product's
    own rounding shows."""
    d, plan = dense_plan(K)
    g = torch.Generator(device=DEV); g.manual_seed(5)
    W = torch.randn(d["n_rows"], K, generator=g, device=DEV)
    H = torch.randn(d["n_cols"], K, generator=g, device=DEV)
    if kind == "positive":
        W, H = W.abs(), H.abs()
    elif kind in ("four a row", "one a row"):
        n = 4 if kind == "four a row" else 1
        W *= torch.zeros_like(W).scatter_(1, torch.randint(0, K, (W.shape[0], n), generator=g, device=DEV), 1.0)
    elif kind == "small":  # products of 2^-122, parts of them subnormal
        W, H = torch.ldexp(W, torch.tensor(-60, device=DEV)), torch.ldexp(H, torch.tensor(-62, device=DEV))
    out, ref, _, rows, cols = product(d, plan, W, H)
    sums = torch.zeros(d["nnz"], device=DEV)
    for k in range(0, K, 2):
        sums = (sums.double() + (W[rows, k:k + 2].double() * H[cols, k:k + 2].double()).sum(1)).float()
    scale = 2.0 ** 122 if kind == "small" else 1.0
    err, err32 = (out.double() - ref) * scale, (sums.double() - ref) * scale
    # A product alone is rounded once, to half a unit in the last place (2^-24 of it); next to others the sum of its 16
    # is rounded, and then the running sum: at most a quarter more in the 2-norm than the sums of two, and less the
    # denser the rows are.
    if kind == "one a row":
        assert bool((err.abs() <= 2.0 ** -24 * (1 + 2.0 ** -6) * ref.abs() * scale).all())
    assert float(err.norm()) <= 1.25 * float(err32.norm()), (float(err.norm()), float(err32.norm()))
