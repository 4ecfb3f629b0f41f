"""The tile kernel's K slices: dot products kept between the slices, positions and values in the last one only."""
import numpy as np
import pytest
import torch

from sddmm_gpu_amd import capi
from test_gpu_parity import _dict_of, plan_options

pytestmark = pytest.mark.gpu


def pattern(K, seed=5):
    """Runs of every length from 1 to 21 in column tiles of 64, and rows without entries."""
    rng = np.random.default_rng(seed)
    r, c = [], []
    for row in range(0, 200, 3):
        for tile in range(4):
            n = (row + 5 * tile) % 21 + 1
            r += [row] * n
            c += sorted(64 * tile + rng.choice(64, n, replace=False))
    return _dict_of(201, 256, r, c, K, rng)


def results(d, fuse, **kw):
    dev = torch.device("cuda:0")
    t = {k: d[k].to(dev) for k in ("row_ptr", "col_ind", "val", "W", "H")}
    make = lambda: capi.Plan.from_device_csr(d["n_rows"], d["n_cols"], d["nnz"], t["row_ptr"].data_ptr(), t["col_ind"].data_ptr(), d["K"],
                                             options=plan_options(capi.KERNEL_LDS_TILE, tile_x=64, fuse_slices=fuse, **kw))
    plan, bare = make(), make()
    plan.set_values(t["val"].data_ptr())
    out = []
    for p, val, form in ((plan, 0, 0), (plan, t["val"].data_ptr(), 0), (plan, 0, capi.EPILOGUE_RESIDUAL),
                         (bare, t["val"].data_ptr(), capi.EPILOGUE_RESIDUAL), (bare, 0, 0)):
        o = torch.full((d["nnz"],), float("nan"), device=dev)
        p.execute_epilogue(val, t["W"].data_ptr(), t["H"].data_ptr(), o.data_ptr(), form)
        torch.cuda.synchronize()
        out.append(o.cpu())
    assert plan.info()["k_slice"] < d["K"]
    return out


# two slices, several, the last one cut short; slices of 64 (the compact stream); groups of 16 lanes
@pytest.mark.parametrize("K,kw", [(256, {}), (384, {}), (512, {}), (300, {}), (515, {}), (192, {}), (320, {}), (512, dict(k_slice=256))])
@pytest.mark.parametrize("fuse", [0, 1])
def test_slices(K, kw, fuse):
    d = pattern(K)
    scaled, scaled_call, residual, residual_call, dots = results(d, fuse, **kw)
    assert torch.equal(scaled, scaled_call) and torch.equal(residual, residual_call)
    w, h, v = d["W"].double()[d["row_ind"].long()], d["H"].double()[d["col_ind"].long()], d["val"].double()
    dot, size = (w * h).sum(1), (w * h).abs().sum(1)
    u = 2.0 ** -24  # K + 2 roundings at most, whatever the order
    for got, want, scale in ((scaled, v * dot, v.abs() * size), (residual, v - dot, v.abs() + size), (dots, dot, size)):
        assert bool(((got.double() - want).abs() <= 1.01 * (K + 2) * u * scale).all())


@pytest.mark.parametrize("fuse", [0, 1])
def test_slices_infinities_and_nan(fuse):
    """In any slice, and sums that leave the range, come out as the formula has them."""
    K = 512
    d = pattern(K)
    inf = float("inf")
    d["W"][3, 5] = inf; d["W"][6, 200] = -inf; d["W"][9, 511] = inf; d["W"][12, 300] = float("nan")
    d["W"][15, :128] = 3e38; d["H"][:, 0] = 1.0; d["W"][18, 130:256] = 3e38
    d["val"][7] = inf
    scaled, _, residual, _, dots = results(d, fuse)
    w, h, v = d["W"].double()[d["row_ind"].long()], d["H"].double()[d["col_ind"].long()], d["val"].double()
    dot, size = (w * h).sum(1), (w * h).abs().sum(1)
    # (sums beyond fp32's range: left out where the order of the terms decides)
    clear = ~torch.isfinite(size) | (size < 1e38)
    for got, want in ((scaled, v * dot), (residual, v - dot), (dots, dot)):
        want32 = want.float()
        special = clear & ~torch.isfinite(want32)
        assert bool((torch.isnan(got) == torch.isnan(want32))[clear].all())
        assert torch.equal(got[special & ~torch.isnan(want32)], want32[special & ~torch.isnan(want32)])
        assert bool(torch.isfinite(got)[clear & torch.isfinite(want32)].all())
