"""Workloads that performance is measured on: what a user of this framework has it do, over the sizes they do it at.

A case is a dict of plain values.  "op" says which calls one pass makes:
  product    out = val * (W H^T) on the pattern of S, through a plan that the program keeps (the framework's main call);
             "values": "plan" (S.val handed over with the plan), "call" (passed with each call) or "none" (out = dot)
  factorise  matrix factorisation: the residual val - W H^T at the nonzeros, and its product with H, which is the
             gradient step of the row factor (the backward direction of the same pattern)
  attention  sparse attention: row softmax of the sampled scores Q K^T, then the weighted sum of the V rows
  edges      a graph layer whose pattern is new in every batch, so no plan: edge scores, softmax over each vertex's
             edges, aggregation -- the three calls that work on a plain CSR pattern
  host       host arrays in, host array out through a kept plan: the calling convention of the command line tool
"pattern" says how the nonzeros lie, with the sizes beside it; "K" is the rank (row length of the dense factors).
The patterns and the distributions of the values are those of sddmm_gpu_amd.synth, the five benchmark shapes among
them, and a local attention window.
"""
import math

import torch

from sddmm_gpu_amd import capi, synth


def listed():
    return [
        # The smallest graph layer in earnest: a few thousand vertices with a handful of edges each.  Launches count.
        dict(name="edges_small_k16", op="edges", pattern="graph", log2_n=12, edges=20000, K=16),
        # Benchmark shape 1, one small SDDMM per step: the work fits the caches, the latency of the call counts.
        dict(name="uniform_k32", op="product", pattern="uniform", n_rows=4096, n_cols=4096, density=0.01, K=32, values="plan"),
        # Benchmark shape 2, bag of words at a high rank: small, skewed columns, cache-resident.
        dict(name="words_k256", op="product", pattern="words", n_rows=1500, n_cols=12419, mean_row=497.5, K=256, values="plan"),
        # A sampled batch of a larger graph at a feature length that is no power of two, edge weights with the call.
        dict(name="edges_k100", op="edges", pattern="graph", log2_n=17, edges=2000000, K=100),
        # Attention over 16k tokens: a local window and a few tokens that all others look at, one head of 64.
        dict(name="attention_k64", op="attention", pattern="window", n=16384, half_band=128, every=512, K=64),
        # A factorisation step on a medium ratings matrix at the customary rank of 50 (rows are not 16-byte multiples).
        dict(name="factorise_k50", op="factorise", pattern="ratings", n_rows=48000, n_cols=5600, max_deg=5000, K=50),
        # The same from host memory and back, as the command line tool runs it.
        dict(name="host_k128", op="host", pattern="ratings", n_rows=48000, n_cols=5600, max_deg=5000, K=128),
        # Benchmark shape 3 (recommender ratings, 100 M nonzeros) at three ranks of the headline sweep.
        dict(name="ratings_k32", op="product", pattern="ratings", n_rows=480189, n_cols=17770, max_deg=17000, K=32, values="plan"),
        dict(name="ratings_k128", op="product", pattern="ratings", n_rows=480189, n_cols=17770, max_deg=17000, K=128, values="plan"),
        dict(name="ratings_k512", op="product", pattern="ratings", n_rows=480189, n_cols=17770, max_deg=17000, K=512, values="plan"),
        # Benchmark shape 4 (power-law graph, 4 M vertices, 190 M edges): dense factors of 1 GB each, irregular gathers.
        dict(name="graph_k64", op="product", pattern="graph", log2_n=22, edges=200000000, K=64, values="plan"),
        # Benchmark shape 5 (band of 64 nonzeros a row in +-2048, high rank): the largest number of operations.
        dict(name="banded_k512", op="product", pattern="band", n_rows=1 << 20, per_row=64, half_band=2048, K=512, values="plan"),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _draw_pattern(rng, kind, nnz):
    """Sizes of a pattern of about nnz nonzeros."""
    if kind == "uniform":
        density = _log_uniform(rng, 0.002, 0.05)
        side = math.sqrt(nnz / density)
        skew = _log_uniform(rng, 0.5, 2.0)
        return dict(n_rows=max(64, int(side * skew)), n_cols=max(64, int(side / skew)), density=density)
    if kind == "words":
        n_rows = int(math.sqrt(nnz / 500.0 / 1500.0) * 1500 * _log_uniform(rng, 0.7, 1.4)) + 64
        mean_row = nnz / n_rows
        return dict(n_rows=n_rows, n_cols=int(mean_row * rng.uniform(15, 35)), mean_row=mean_row)
    if kind == "ratings":
        s = nnz / 1.0e8
        n_cols = int(17770 * min(1.0, s ** 0.33) * rng.uniform(0.8, 1.0)) + 64
        max_deg = int(0.9 * n_cols)
        return dict(n_rows=max(64, int(nnz / _ratings_mean(max_deg))), n_cols=n_cols, max_deg=max_deg)
    if kind == "graph":
        edges = int(nnz)
        return dict(log2_n=max(8, min(22, round(math.log2(edges / _log_uniform(rng, 8, 60))))), edges=edges)
    if kind == "band":
        per_row = rng.randint(16, 96)
        n_rows = max(4 * per_row, int(nnz / per_row))
        return dict(n_rows=n_rows, per_row=per_row, half_band=int(min(n_rows / 2, per_row * _log_uniform(rng, 4, 32))))
    half_band, seen_by_all = rng.randint(24, 300), rng.randint(4, 32)
    n = max(2 * half_band, int(nnz / (2 * half_band + 2 * seen_by_all)))
    return dict(n=n, half_band=half_band, every=-(-n // seen_by_all))


def draw(rng):
    """One more case of the ranges above: any operation, 20,000 to 10^8 nonzeros, ranks from 8 to 512 (odd ones too),
    at most the operations of the largest listed case."""
    op = rng.choice(["product", "product", "product", "factorise", "attention", "edges", "host"])
    if op == "attention":
        K = rng.choice([32, 64, 64, 80, 128])
    elif rng.random() < 0.6:
        K = rng.choice([16, 32, 64, 96, 128, 192, 256, 384, 512])
    else:
        K = int(_log_uniform(rng, 8, 300))
    most = {"product": 1.0e8, "factorise": 2.0e7, "attention": 2.0e7, "edges": 1.0e7, "host": 2.0e7}[op]
    if K % 4:
        most = min(most, 4.0e6)
    least = 2.0e4 if op == "edges" else 1.0e5
    nnz = _log_uniform(rng, least, min(most, 2.5e10 / K))
    kind = {"product": rng.choice(["uniform", "words", "ratings", "graph", "band"]), "factorise": "ratings",
            "attention": "window", "edges": "graph", "host": rng.choice(["words", "ratings"])}[op]
    case = dict(op=op, pattern=kind, K=K, **_draw_pattern(rng, kind, nnz))
    if op == "product":
        case["values"] = rng.choice(["plan", "plan", "call", "none"])
    return case


def _window(n, half_band, every, K, seed, device):
    """Local attention: every token looks at the half_band tokens on either side of it and at each token whose number
    is a multiple of `every`; those tokens look at all.  Q, K, V from N(0, 1), Q scaled by K^-1/2."""
    g = torch.Generator(device=device)
    g.manual_seed(int(seed))
    rows = torch.arange(n, device=device)
    cols = rows[:, None] + torch.arange(-half_band, half_band + 1, device=device)[None, :]
    keys = (rows[:, None] * n + cols)[(cols >= 0) & (cols < n)]
    seen = torch.arange(0, n, every, device=device)
    keys = torch.unique(torch.cat([keys, (rows[:, None] * n + seen[None, :]).reshape(-1),
                                   (seen[:, None] * n + rows[None, :]).reshape(-1)]))
    dense = [torch.randn(n, K, generator=g, device=device) for _ in range(3)]
    return dict(n_rows=n, n_cols=n, **_csr(keys, n, n), val=None, W=dense[0] * K ** -0.5, H=dense[1], V=dense[2])


def _csr(keys, n_rows, n_cols):
    """Sorted keys row * n_cols + column as a CSR pattern."""
    rows = torch.div(keys, n_cols, rounding_mode="floor")
    row_ptr = torch.zeros(n_rows + 1, dtype=torch.int64, device=keys.device)
    row_ptr[1:] = torch.cumsum(torch.bincount(rows, minlength=n_rows), 0)
    return dict(nnz=int(keys.numel()), row_ptr=row_ptr.to(torch.int32), col_ind=(keys - rows * n_cols).to(torch.int32))


def _of_size(d, nnz, seed):
    """The pattern brought to exactly nnz nonzeros, so that every seed gives outputs of one size: evenly spaced ones
    left out, or further ones added that pair the row and the column of two nonzeros drawn at random (rows and columns
    stay as popular as they are)."""
    n_rows, n_cols, dev = d["n_rows"], d["n_cols"], d["col_ind"].device
    keys = d.pop("row_ind").long() * n_cols + d["col_ind"]
    g = torch.Generator(device=dev)
    g.manual_seed(int(seed) + 2)
    while keys.numel() < nnz:
        more = int(1.3 * (nnz - keys.numel())) + 64
        at = torch.randint(0, keys.numel(), (2, more), generator=g, device=dev)
        keys = torch.unique(torch.cat([keys, torch.div(keys[at[0]], n_cols, rounding_mode="floor") * n_cols + keys[at[1]] % n_cols]))
    left_out = keys.numel() - nnz
    if left_out:
        keep = torch.ones(keys.numel(), dtype=torch.bool, device=dev)
        keep[torch.div(torch.arange(left_out, device=dev) * keys.numel(), left_out, rounding_mode="floor")] = False
        keys = keys[keep]
    d.update(_csr(keys, n_rows, n_cols))
    val = d["val"]
    d["val"] = val[:nnz].clone() if val.numel() >= nnz else val.repeat(-(-nnz // val.numel()))[:nnz]
    return d


def _matrix(case, seed, device):
    kind, K = case["pattern"], case["K"]
    kw = dict(K=K, seed=seed, device=device)
    if kind == "window":
        return _window(case["n"], case["half_band"], case["every"], K, seed, device)
    if kind == "uniform":
        d = synth.uniform_random(case["n_rows"], case["n_cols"], case["density"], **kw)
    elif kind == "words":
        d = synth.bag_of_words(case["n_rows"], case["n_cols"], case["mean_row"], **kw)
    elif kind == "ratings":
        d = synth.recommender(case["n_rows"], case["n_cols"], max_deg=case["max_deg"], **kw)
    elif kind == "graph":
        d = synth.rmat(case["log2_n"], case["edges"], **kw)
    else:
        d = synth.banded(case["n_rows"], case["per_row"], case["half_band"], **kw)
    d = _of_size(d, _nonzeros(case), seed)
    if case["op"] == "edges":  # edge weights, and features of a size that keeps the scores moderate
        g = torch.Generator(device=device)
        g.manual_seed(int(seed) + 1)
        d["val"] = 0.5 + torch.rand(d["nnz"], generator=g, device=device)
        d["W"] *= K ** -0.25
        d["H"] *= K ** -0.25
    return d


def prepare(case, seed):
    dev = torch.device("cuda")
    d = _matrix(case, seed, dev)
    op, K, n_rows, n_cols, nnz = case["op"], case["K"], d["n_rows"], d["n_cols"], d["nnz"]
    d["op"], d["K"] = op, K
    if op == "edges":
        d["score"] = torch.empty(nnz, device=dev)
        d["weight"] = torch.empty(nnz, device=dev)
        d["Y"] = torch.empty(n_rows, K, device=dev)
        torch.cuda.synchronize()
        return d
    torch.cuda.synchronize()
    both = op in ("factorise", "attention")  # plans that also serve the product with the dense factor
    plan = capi.Plan.from_device_csr(n_rows, n_cols, nnz, d["row_ptr"].data_ptr(), d["col_ind"].data_ptr(), K,
                                     options=capi.PlanOptions.defaults(spmm_stream=1) if both else None)
    d["plan"] = plan
    d["values"] = 0
    if op == "product" and case["values"] == "call":
        d["values"] = d["val"].data_ptr()
    elif d["val"] is not None and case.get("values") != "none":
        plan.set_values(d["val"].data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    if op == "host":
        d["W"], d["H"] = d["W"].cpu().numpy(), d["H"].cpu().numpy()
        return d
    d["out"] = torch.empty(nnz, device=dev)
    if both:
        d["Y"] = torch.empty(n_rows, K, device=dev)
    return d


def run(s):
    op = s["op"]
    if op == "host":
        return s["plan"].gpu(s["W"], s["H"])[0]
    stream = torch.cuda.current_stream().cuda_stream
    W, H = s["W"].data_ptr(), s["H"].data_ptr()
    if op == "product":
        s["plan"].execute(s["values"], W, H, s["out"].data_ptr(), stream)
        return s["out"]
    if op == "factorise":
        s["plan"].execute_epilogue(0, W, H, s["out"].data_ptr(), capi.EPILOGUE_RESIDUAL, stream)
        s["plan"].spmm(s["out"].data_ptr(), H, s["Y"].data_ptr(), stream=stream)
        return s["out"], s["Y"]
    if op == "attention":
        s["plan"].execute_softmax(0, W, H, s["out"].data_ptr(), stream)
        s["plan"].spmm(s["out"].data_ptr(), s["V"].data_ptr(), s["Y"].data_ptr(), stream=stream)
        return s["out"], s["Y"]
    rp, ci = s["row_ptr"].data_ptr(), s["col_ind"].data_ptr()
    capi.csr_noalloc(s["n_rows"], s["n_cols"], s["nnz"], rp, ci, s["val"].data_ptr(), s["K"], W, H, s["score"].data_ptr(), stream)
    capi.row_softmax(s["n_rows"], rp, s["score"].data_ptr(), s["weight"].data_ptr(), stream)
    capi.spmm_csr(s["n_rows"], s["n_cols"], s["nnz"], rp, ci, s["weight"].data_ptr(), s["K"], H, s["Y"].data_ptr(), stream)
    return s["score"], s["weight"], s["Y"]


def _ratings_mean(max_deg, beta=1.42):
    """Mean of the power law x^-beta on [1, max_deg] that the row lengths follow."""
    return (max_deg ** (2 - beta) - 1) / (2 - beta) * (1 - beta) / (max_deg ** (1 - beta) - 1)


def _nonzeros(case):
    """Nonzeros of a generated pattern: a little less than the generator gives on average."""
    kind = case["pattern"]
    if kind == "uniform":
        nnz = case["n_rows"] * case["n_cols"] * -math.expm1(-case["density"])
    elif kind == "words":
        nnz = case["n_rows"] * case["mean_row"]
    elif kind == "ratings":
        nnz = case["n_rows"] * _ratings_mean(min(case["max_deg"], 0.95 * case["n_cols"]))
    elif kind == "graph":
        # every level of an edge falls into quadrant a, into b or c, or into d: cells with i, j and k such levels are
        # equally likely, and the distinct edges are a sum over those kinds of cells
        s, e, nnz = case["log2_n"], case["edges"], 0.0
        for i in range(s + 1):
            for j in range(s - i + 1):
                cells = math.comb(s, i) * math.comb(s - i, j) * 2.0 ** j
                nnz += cells * -math.expm1(-e * 0.57 ** i * 0.19 ** j * 0.05 ** (s - i - j))
    else:
        width = 2 * case["half_band"] + 1
        nnz = case["n_rows"] * width * -math.expm1(-case["per_row"] / width)
    return int(0.98 * nnz)


def _extent(case):
    """(rows, columns, nonzeros, rows with a nonzero, columns with a nonzero), the last two as expected."""
    if case["pattern"] == "window":
        n, hb = case["n"], case["half_band"]
        seen = -(-n // case["every"])
        nnz = n * (2 * hb + 1) - hb * (hb + 1) + 2 * seen * n - seen * (4 * hb + 2)
        return n, n, nnz, n, n
    nnz = _nonzeros(case)
    if case["pattern"] == "graph":  # vertices whose number has k one bits are drawn with probability 0.24^k 0.76^(s - k)
        s, e = case["log2_n"], case["edges"]
        touched = sum(math.comb(s, k) * -math.expm1(-e * 0.24 ** k * 0.76 ** (s - k)) for k in range(s + 1))
        return 1 << s, 1 << s, nnz, touched, touched
    n, m = case["n_rows"], case.get("n_cols", case["n_rows"])
    return n, m, nnz, n, m


def work(case):
    n, m, nnz, rows, cols = _extent(case)
    K, op = case["K"], case["op"]
    pattern = 4.0 * nnz + 4.0 * (n + 1)
    product = 4.0 * K * (rows + cols) + 4.0 * nnz  # W, H and the results
    flops = 2.0 * nnz * K
    if op == "product":
        return dict(bytes=pattern + product + (0.0 if case["values"] == "none" else 4.0 * nnz), flops=flops)
    if op == "host":  # W and H from host memory, the results into it
        return dict(bytes=pattern + 4.0 * K * (n + m) + 8.0 * nnz, flops=flops)
    if op == "factorise":
        return dict(bytes=pattern + product + 4.0 * nnz + 4.0 * K * n, flops=2 * flops)
    if op == "attention":
        return dict(bytes=pattern + product + 4.0 * K * (cols + n), flops=2 * flops + 4.0 * nnz)
    return dict(bytes=pattern + product + 8.0 * nnz + 4.0 * K * n, flops=2 * flops + 4.0 * nnz)


def tolerance(case):
    """Sums of 32-bit products in another order."""
    return {"rel": 1e-5}
