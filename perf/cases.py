"""The calls whose speed this repository answers for: the decode linears of a Llama-2-7B-shaped
model and the generic shapes around them, through the package's public entry points.

A case is one pass of a user's decode loop over one kind of linear: the same call on each of
`layers` weights, so that a pass finds its weights in HBM as a model of many layers does, either
captured as a HIP graph (as the drivers of the per-step benchmark do) or called eagerly.

op        what is called
decode    bsa_mi355x.decode.DecodeStep: every linear of `layers` layers with the exact-L1
          selection in front of each, one graph
list      the drop-in `_prepacked_block_sparse_gemm_from_active_blocks` on an unsorted block list
bitmap    `..._bitmap_preload` on a prebuilt bitmap
dense     dense_gemm: every block active
select    select_sparse_gemm with the exact-L1 rule
rule      select_sparse_gemm with a rule of the reference (l2_mean, energy) and, with `budget`,
          an energy budget that decides the number of kept blocks on the device
cols      the 2-D entry: only `ncols` of the 64-column output blocks are computed
pack      pack_weight of an nn.Linear weight, what loading a model does once per linear
"""
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "towards-batched-activation-sparsity_amd"))

import bsa_mi355x as bsa  # noqa: E402
from bsa_mi355x.decode import DecodeStep  # noqa: E402

DEV = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def _c(name, op, bt, k, n, density, layers, dtype="fp16", graph=True, seqlen=1, score="", budget=0.0, ncols=0):
    return {"name": name, "op": op, "bt": bt, "seqlen": seqlen, "K": k, "N": n, "density": density, "layers": layers,
            "dtype": dtype, "graph": graph, "score": score, "budget": budget, "ncols": ncols}


def listed():
    return [
        # the decode step of linears at the largest batch, 0.52 sparsity: what a server replays per token
        _c("decode_b64", "decode", 64, 4096, 4096, 0.48, 8),
        # the same step for a handful of sequences, where masks are sparser and launches count
        _c("decode_b4", "decode", 4, 4096, 4096, 0.25, 8),
        # attention projections for two sequences with a given mask: the per-step replay's smallest GEMMs
        _c("list_b2_qkvo", "list", 2, 4096, 4096, 0.197, 32),
        # MLP down projection, 16 sequences, half the blocks, called eagerly with an unsorted list
        _c("list_b16_down", "list", 16, 11008, 4096, 0.5, 8, graph=False),
        # one eager selection + GEMM for a single sequence: latency
        _c("select_b1_qkvo", "select", 1, 4096, 4096, 0.5, 1, graph=False),
        # the decode linear of the reference's own selection rule at 64 sequences, a bf16 model
        _c("rule_b64_gate_bf16", "rule", 64, 4096, 11008, 0.48, 8, dtype="bf16", score="l2_mean"),
        # selection with an energy budget: the kept count is found on the device
        _c("budget_b16_gate", "rule", 16, 4096, 11008, 0.2, 8, score="energy", budget=0.6),
        # a bitmap-driven linear of another model: odd width, ragged last block, an odd batch
        _c("bitmap_b37_odd", "bitmap", 37, 5000, 13827, 0.4, 8),
        # the dense baseline of the same kernels, fused q/k/v at 32 sequences
        _c("dense_b32_qkv", "dense", 32, 4096, 12288, 1.0, 4),
        # output sparsity too: half of down's output blocks at 16 sequences
        _c("cols_b16_down", "cols", 16, 11008, 4096, 0.5, 8, ncols=32),
        # the most rows one call meets: 64 sequences checking 4 drafted tokens each
        _c("list_b256_gate", "list", 64, 4096, 11008, 0.48, 4, seqlen=4),
        # loading: one MLP weight packed
        _c("pack_gate", "pack", 0, 4096, 11008, 1.0, 1, graph=False),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    op = rng.choice(["decode", "list", "list", "list", "bitmap", "dense", "select", "rule", "rule", "cols", "pack"])
    dtype = "fp16" if op in ("decode", "select") else rng.choice(["fp16", "fp16", "bf16"])
    bt = _log(rng, 1, 64)
    # the model's own linears as often as those of other models (K a multiple of 8, N any)
    k, n = rng.choice([(4096, 4096), (4096, 11008), (11008, 4096), (4096, 12288), (4096, 22016)])
    if rng.random() < 0.5:
        k, n = 8 * _log(rng, 128, 1536), _log(rng, 1000, 16384)
        if rng.random() < 0.5:
            k, n = k - k % 64, n - n % 64
    density = round(rng.uniform(0.15, 0.9), 3)
    if op == "decode":
        return _c("", "decode", bt, 4096, 4096, round(rng.uniform(0.15, 0.5), 3), rng.randint(2, 6))
    if op == "pack":
        return _c("", "pack", 0, k, n, 1.0, 1, dtype=dtype, graph=False)
    graph = rng.random() < 0.75
    seqlen = rng.choice([2, 3, 4]) if op in ("list", "dense") and rng.random() < 0.3 else 1
    layers = max(1, min(16, int(4e8 / (2.0 * k * n * density))))
    score, budget, ncols = "", 0.0, 0
    if op == "rule":
        score = rng.choice(["l2_mean", "energy"])
        budget = round(rng.uniform(0.5, 0.9), 3) if rng.random() < 0.3 else 0.0
    if op == "cols":
        nnb = -(-n // 64)
        ncols = max(1, int(rng.uniform(0.2, 0.9) * nnb))
    return _c("", op, bt, k, n, 1.0 if op == "dense" else density, layers, dtype=dtype, graph=graph, seqlen=seqlen,
              score=score, budget=budget, ncols=ncols)


def _nblk(k):
    return -(-k // 64)


def _keep(c):
    # the reference's rules score whole blocks only
    nb = c["K"] // 64 if c["op"] == "rule" else _nblk(c["K"])
    return max(1, min(nb, int(round(c["density"] * nb))))


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _inputs(c, seed):
    """The tensors of a case, the same for prepare() and exact(): weights [N, K] ~ N(0, 0.02); x ~ N(0, 1) with
    channels of unequal strength (what makes a selection worth while), Laplace(0, 0.05) into the wide-K linears;
    unsorted lists of distinct blocks."""
    g = _gen(seed)
    dt = DTYPES[c["dtype"]]
    k, n, rows = c["K"], c["N"], c["bt"] * c["seqlen"]
    for _ in range(c["layers"]):
        w = torch.randn(n, k, generator=g, device=DEV, dtype=torch.float32).mul_(0.02).to(dt)
        if c["op"] == "pack":
            yield {"w": w}
            continue
        if k > n:
            u = torch.rand(rows, k, generator=g, device=DEV) - 0.5
            x = -0.05 * torch.sign(u) * torch.log1p(-2 * u.abs())
        else:
            x = torch.randn(rows, k, generator=g, device=DEV)
        x = (x * torch.exp(0.5 * torch.randn(k, generator=g, device=DEV))).to(dt).view(c["bt"], c["seqlen"], k)
        blocks = torch.randperm(_nblk(k), generator=g, device=DEV)[: _keep(c)].to(torch.int32)
        cols = torch.randperm(_nblk(n), generator=g, device=DEV)[: max(1, c["ncols"])].sort()[0].to(torch.int32)
        yield {"w": w, "x": x, "blocks": blocks, "cols": cols}


def prepare(case, seed):
    c = dict(case)
    if c["op"] == "decode":
        step = DecodeStep(batch=c["bt"], density=c["density"], n_layers=c["layers"], seed=seed)
        step.capture()
        return {"case": c, "step": step}
    state = {"case": c, "items": [], "graph": None}
    for t in _inputs(c, seed):
        if c["op"] != "pack":
            dt = DTYPES[c["dtype"]]
            t["y"] = torch.zeros(c["bt"], c["seqlen"], c["N"], device=DEV, dtype=dt)
            cap = c["K"] // 64 if c["budget"] > 0 else _keep(c)
            t["idx"] = torch.zeros(cap, device=DEV, dtype=torch.int32)
            t["cnt"] = torch.zeros(1, device=DEV, dtype=torch.int32)
            t["ratio"] = torch.zeros(1, device=DEV, dtype=torch.float32)
            if c["op"] == "bitmap":
                t["bitmap"] = bsa._build_active_k_bitmap(t["blocks"], _nblk(c["K"]), DEV)
        state["items"].append(t)
    if c["op"] != "pack":
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            _calls(state)  # packs the weights, settles plans and workspaces
        torch.cuda.current_stream().wait_stream(s)
        torch.cuda.synchronize()
    if c["graph"]:
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            state["out"] = _calls(state)
        torch.cuda.synchronize()
        state["graph"] = g
    return state


def _calls(state):
    c = state["case"]
    op, out = c["op"], []
    for t in state["items"]:
        if op == "pack":
            out.append(bsa.pack_weight(t["w"], layout="nk"))
            continue
        x, w, y = t["x"], t["w"], t["y"]
        if op == "list":
            bsa._prepacked_block_sparse_gemm_from_active_blocks(x, w, t["blocks"], y, cache_prefix="perf_list")
        elif op == "bitmap":
            bsa._prepacked_block_sparse_gemm_from_active_blocks_bitmap_preload(
                x, w, t["blocks"], y, cache_prefix="perf_bitmap", prebuilt_bitmap=t["bitmap"])
        elif op == "dense":
            bsa.dense_gemm(x, w, y, cache_prefix="perf_dense")
        elif op == "cols":
            bsa._prepacked_block_sparse_gemm_2d_from_active_blocks(x, w, t["blocks"], t["cols"], y,
                                                                   cache_prefix="perf_cols")
        elif op == "select":
            bsa.select_sparse_gemm(x, w, y, _keep(c), cache_prefix="perf_sel", idx_out=t["idx"], count_out=t["cnt"])
            out.append(t["idx"])
        else:
            rule = {"energy_keep": c["budget"], "ratio_out": t["ratio"]} if c["budget"] > 0 else {}
            bsa.select_sparse_gemm(x, w, y, _keep(c), cache_prefix="perf_rule", idx_out=t["idx"], count_out=t["cnt"],
                                   score=c["score"], **rule)
            out += [t["idx"], t["cnt"]]
            if rule:
                out.append(t["ratio"])
        out.append(y)
    return out


def run(state):
    if "step" in state:
        state["step"].replay()
        return [v for _, p in state["step"].projections() for v in (p.idx, p.y)]
    if state["graph"] is not None:
        state["graph"].replay()
        return state["out"]
    return _calls(state)


def _kept_by_budget(c):
    """About how many blocks an energy budget keeps of channels of the inputs' spread (for work())."""
    nb = c["K"] // 64
    return max(_keep(c), int(0.92 * c["budget"] * nb))


def _gemm_work(bt, k, n, na, x_cols):
    return 2.0 * na * 64 * n + 2.0 * bt * x_cols + 2.0 * bt * n, 2.0 * bt * na * 64 * n


def work(case):
    c = case
    if c["op"] == "pack":
        return {"bytes": 2.0 * c["K"] * c["N"] + 2.0 * _nblk(c["K"]) * 64 * (-(-c["N"] // 16) * 16), "flops": 0.0}
    b = f = 0.0
    if c["op"] == "decode":
        for k, n in ((4096, 12288), (4096, 4096), (4096, 22016), (11008, 4096)):
            na = max(1, min(k // 64, int(round(c["density"] * (k // 64)))))
            wb, wf = _gemm_work(c["bt"], k, n, na, k)
            b, f = b + wb, f + wf
    else:
        rows = c["bt"] * c["seqlen"]
        na = _kept_by_budget(c) if c["budget"] > 0 else _nblk(c["K"]) if c["op"] == "dense" else _keep(c)
        n = min(c["N"], 64 * c["ncols"]) if c["op"] == "cols" else c["N"]
        # a selection reads the whole of x, a given list only its blocks
        b, f = _gemm_work(rows, c["K"], n, na, c["K"] if c["op"] in ("select", "rule") else min(c["K"], 64 * na))
    return {"bytes": b * c["layers"], "flops": f * c["layers"]}


def tolerance(case):
    if case["op"] == "pack":
        return "exact"
    # 16-bit outputs of 32-bit sums: the rounding of the output itself is 2.1e-4 (fp16), 1.7e-3 (bf16); four times that
    return {"rel": 8e-4 if case["dtype"] == "fp16" else 6.6e-3}


def _decode_exact(c, seed):
    """The tensors that DecodeStep draws from this seed, and what its linears give."""
    g = _gen(seed)
    out = []
    for _ in range(c["layers"]):
        for k, n in ((4096, 12288), (4096, 4096), (4096, 22016), (11008, 4096)):
            w = (torch.randn(k, n, generator=g, device=DEV, dtype=torch.float32) * 0.02).to(torch.float16)
            if k > 4096:
                u = torch.rand(c["bt"], k, generator=g, device=DEV) - 0.5
                x = (-0.05 * torch.sign(u) * torch.log1p(-2 * u.abs())).to(torch.float16)
            else:
                x = torch.randn(c["bt"], k, generator=g, device=DEV).to(torch.float16)
            nb = k // 64
            idx = _top(x.double().abs().view(c["bt"], nb, 64).sum((0, 2)), max(1, min(nb, int(round(c["density"] * nb)))))
            out += [idx, _product(x, w.t(), idx)]
    return out


def _top(score, k):
    return score.sort(descending=True, stable=True)[1][:k].sort()[0]


def _product(x2d, w, blocks):
    ch = (blocks.long()[:, None] * 64 + torch.arange(64, device=DEV)).reshape(-1)
    ch = ch[ch < x2d.shape[1]]
    return x2d[:, ch].double() @ w[:, ch].double().t()


def _packed_exact(w):
    n, k = w.shape
    full = torch.zeros(-(-n // 16) * 16, _nblk(k) * 64, device=DEV, dtype=torch.float64)
    full[:n, :k] = w.double()
    # [tile, column, block, half, group, element] -> [block, tile, half, group, column, element]
    p = full.view(full.shape[0] // 16, 16, _nblk(k), 2, 4, 8).permute(2, 0, 3, 4, 1, 5)
    return p.reshape(_nblk(k), full.shape[0] // 16, 1024)


def exact(case, seed):
    c = dict(case)
    if c["op"] == "decode":
        return _decode_exact(c, seed)
    out = []
    for t in _inputs(c, seed):
        w = t["w"]
        if c["op"] == "pack":
            out.append(_packed_exact(w))
            continue
        x = t["x"].view(-1, c["K"])
        shape = (c["bt"], c["seqlen"], c["N"])
        blocks = t["blocks"]
        if c["op"] == "dense":
            blocks = torch.arange(_nblk(c["K"]), device=DEV)
        elif c["op"] == "select":
            pad = torch.nn.functional.pad(x.double().abs(), (0, _nblk(c["K"]) * 64 - c["K"]))
            blocks = _top(pad.view(x.shape[0], -1, 64).sum((0, 2)), _keep(c))
            out.append(blocks)
        elif c["op"] == "rule":
            nb = c["K"] // 64
            sq = x.double()[:, : nb * 64].reshape(-1, nb, 64).square().sum(2)
            energy = sq.mean(0)
            order = (sq.sqrt().mean(0) if c["score"] == "l2_mean" else energy).sort(descending=True, stable=True)[1]
            keep = _keep(c)
            cum = energy[order].cumsum(0)
            if c["budget"] > 0:
                # the budget is a 32-bit number to the framework
                b = float(torch.tensor(c["budget"], dtype=torch.float32))
                keep = max(keep, min(nb, int((cum < b * cum[-1]).sum()) + 1))
            blocks = order[:keep].sort()[0]
            idx = torch.zeros(nb if c["budget"] > 0 else keep, device=DEV, dtype=torch.int64)
            idx[:keep] = blocks
            out += [idx, torch.tensor([keep], device=DEV)]
            if c["budget"] > 0:
                out.append(cum[keep - 1:keep] / cum[-1])
        y = _product(x, w, blocks).view(shape)
        if c["op"] == "cols":
            on = torch.zeros(_nblk(c["N"]), dtype=torch.bool, device=DEV)
            on[t["cols"].long()] = True
            y = y * on.repeat_interleave(64)[: c["N"]]
        out.append(y)
    return out
