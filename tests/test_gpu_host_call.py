"""sddmm_gpu (host arrays in and out): transfers from one value to several pieces, with tails that are no multiple
of 16 bytes and host arrays at any 4-byte address, against the device form of the same plan; calls from two threads."""
import threading

import numpy as np
import pytest
import torch

from sddmm_gpu_amd import capi

pytestmark = pytest.mark.gpu


def make(n_rows, n_cols, nnz, K, seed):
    rng = np.random.default_rng(seed)
    keys = np.sort(rng.choice(n_rows * n_cols, nnz, replace=False))
    S = capi.Coo.from_arrays(n_rows, n_cols, keys // n_cols, keys % n_cols, rng.standard_normal(nnz).astype(np.float32))
    W = rng.standard_normal(n_rows * K + 1).astype(np.float32)[1:].reshape(n_rows, K)  # (not 16-byte aligned)
    H = rng.standard_normal((n_cols, K)).astype(np.float32)
    return S.plan(K), W, H


def expected(plan, W, H, nnz):
    dev = torch.device("cuda:0")
    Wd, Hd, out = torch.from_numpy(W.copy()).to(dev), torch.from_numpy(H).to(dev), torch.empty(nnz, device=dev)
    plan.execute(0, Wd.data_ptr(), Hd.data_ptr(), out.data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("n_rows,n_cols,nnz,K", [(1, 1, 1, 1), (3, 5, 7, 5), (257, 256, 65536, 32), (4001, 1999, 300_001, 64), (5000, 3001, 1_500_001, 64),
                                                 (40001, 999, 3_000_003, 50)])
def test_transfers_of_all_sizes(n_rows, n_cols, nnz, K):
    plan, W, H = make(n_rows, n_cols, nnz, K, nnz)
    want = expected(plan, W, H, nnz)
    for _ in range(2):
        out, ms = plan.gpu(W, H)
        assert np.array_equal(out, want) and ms > 0
    plan.close()


def test_two_threads_with_a_plan_each_and_one_plan():
    plans = [make(3000 + i, 2000, 700_000, 64, i) for i in range(2)]
    want = [expected(p, W, H, 700_000) for p, W, H in plans]
    bad = []

    def work(i):
        p, W, H = plans[i % 2]
        for _ in range(5):
            if not np.array_equal(p.gpu(W, H)[0], want[i % 2]):
                bad.append(i)

    th = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad


def test_what_a_call_keeps_is_counted_and_given_back():
    plan, W, H = make(60000, 30000, 400_000, 128, 9)
    want = expected(plan, W, H, 400_000)
    kept = 4 * (W.size + H.size + 400_000)  # 47 MB
    before = plan.info()["device_bytes"]
    for _ in range(2):
        assert np.array_equal(plan.gpu(W, H)[0], want)
        assert plan.info()["device_bytes"] == before + kept
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        plan.release_host()
        assert plan.info()["device_bytes"] == before
        assert torch.cuda.mem_get_info()[0] >= free + kept // 2
    plan.release_host()  # nothing to give back
    plan.close()
