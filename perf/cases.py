"""The calls whose speed is measured: what a program that trains or evaluates
Graph Clifford networks has this package do, over the range of graphs, widths,
types and options such programs use.

Kinds of case:
  multihop  the three-hop (or other hop set) propagation of a fixed operator,
            forward and backward (multihop_csr_pipeline, graph)
  gat       collapsed GAT message passing, forward and backward; with dropout
            through the extension object, whose seed is an argument
  conv      the context GAT module (projection, logits, message passing),
            forward and backward
  pack      the Clifford interaction pack, forward and backward
  block     a GraphCliffordBlock, forward and backward
  train     a GraphCliffordNet training step up to the gradients
  eval      a GraphCliffordNet full-graph evaluation (logits)

A graph belongs to its case (a program works on one graph for a whole run);
features, gradients and weights come from the seed. Dropout inside the modules
is 0, since their seeds count the calls of the process.
"""
from __future__ import annotations

import functools

import numpy as np
import torch
import torch.nn.functional as F

from cign_amd import graph, graphgen, train_cign
from cign_amd.collapsed_gat import collapsed_gat_mean_bias_silu, ensure_collapsed_gat_loaded
from cign_amd.fused_clifford_cign_pack import fused_clifford_switch_pack
from cign_amd.model_cign import CompatibleCollapsedFusedGATConv, GraphCliffordBlock, GraphCliffordNet
from cign_amd.multihop_csr_pipeline import MultiHopCSR3GraphOperator, prepare_multihop_csr_operator

DEV = "cuda"
SLOPE = 0.2
CLASSES = 5


def listed():
    return [
        # A small citation-sized graph at the width of a small model: a call
        # is a few launches, so latency is what the user sees.
        dict(name="multihop_small_f32", kind="multihop", n=2000, degree=16, cols=64, dtype="f32", powers="1,2,3"),
        # The propagation of a hidden-256 block ([H | C] is 512 wide) on the
        # 24,492-node benchmark graph.
        dict(name="multihop_d512_f32", kind="multihop", n=24492, degree=8, cols=512, dtype="f32", powers="1,2,3"),
        # The scale configuration's shape at a tenth of its size: denser graph,
        # bf16 storage, tensors beyond the caches' comfort.
        dict(name="multihop_large_bf16", kind="multihop", n=240000, degree=25, cols=256, dtype="bf16",
             powers="1,2,3"),
        # Attention message passing of the benchmark layer, with the dropout
        # training uses.
        dict(name="gat_4x16_f32_drop", kind="gat", n=24492, degree=8, heads=4, channels=16, dtype="f32", drop=0.32),
        # The scale configuration's attention at a tenth of its size.
        dict(name="gat_large_4x32_bf16", kind="gat", n=240000, degree=25, heads=4, channels=32, dtype="bf16",
             drop=0.0),
        # Attention at head counts and widths that are no powers of two, on a
        # graph of odd size.
        dict(name="gat_5x48_f32", kind="gat", n=10007, degree=7, heads=5, channels=48, dtype="f32", drop=0.0),
        # The context GAT of the production block under selective bf16.
        dict(name="conv_6x256_bf16", kind="conv", n=24492, degree=8, in_dim=256, heads=6, channels=256, amp=True),
        # The interaction pack alone at the production width.
        dict(name="pack_d256_f32", kind="pack", n=24492, hidden=256),
        # One production block, forward and backward, selective bf16.
        dict(name="block_256_bf16", kind="block", n=24492, degree=8, hidden=256, heads=6, powers="1,2,3", amp=True),
        # A block away from the tuned widths, in float32, on an odd size.
        dict(name="block_96_f32", kind="block", n=11003, degree=9, hidden=96, heads=5, powers="1,2,3", amp=False),
        # Training step of a two-layer model on a small graph: many launches
        # of little work each.
        dict(name="train_small_f32", kind="train", n=2000, degree=16, in_dim=64, hidden=64, heads=4, layers=2,
             powers="1,2", amp=False),
        # Evaluation of the four-layer production model.
        dict(name="eval_256_bf16", kind="eval", n=24492, degree=8, in_dim=300, hidden=256, heads=6, layers=4,
             powers="1,2,3", amp=True),
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm, odd half of the time."""
    v = int(round(lo * (hi / lo) ** rng.random()))
    return min(hi, max(lo, v | 1 if rng.random() < 0.5 else v))


def draw(rng):
    kind = rng.choice(["multihop", "multihop", "gat", "gat", "conv", "pack", "block", "block", "train", "eval"])
    degree = rng.randint(4, 26)
    dtype = rng.choice(["f32", "bf16"])
    amp = rng.random() < 0.5
    hidden = rng.choice([32, 48, 64, 64, 96, 100, 128, 128, 192, 256, 256, rng.randint(17, 255)])
    powers = rng.choice(["1,2,3", "1,2,3", "1,2", "0,1,3", "1,2,3,4"])
    heads = rng.choice([1, 2, 3, 4, 4, 5, 6, 6, 8])
    n = _log_int(rng, 1200, 24492)
    if kind == "multihop":
        cols = rng.choice([32, 64, 128, 200, 256, 384, 512, rng.randint(33, 511)])
        n = _log_int(rng, 1200, min(240000, 240000 * 25 * 256 // ((degree + 1) * cols * (2 if dtype == "f32" else 1))))
        return dict(kind=kind, n=n, degree=degree, cols=cols, dtype=dtype, powers=rng.choice(["1,2,3", powers]))
    if kind == "gat":
        channels = rng.choice([16, 16, 32, 32, 64, 128, 256, hidden])
        top = 240000 * 25 * 128 // ((degree + 1) * heads * channels * (2 if dtype == "f32" else 1))
        return dict(kind=kind, n=_log_int(rng, 1200, min(240000, max(2400, top))), degree=degree, heads=heads,
                    channels=channels, dtype=dtype, drop=rng.choice([0.0, 0.32]))
    if kind == "conv":
        return dict(kind=kind, n=n, degree=degree, in_dim=rng.choice([64, 128, 256, 300, rng.randint(33, 300)]),
                    heads=heads, channels=rng.choice([16, 32, hidden]), amp=amp)
    if kind == "pack":
        return dict(kind=kind, n=n, hidden=hidden)
    degree = min(degree, 12)
    if kind == "block":
        return dict(kind=kind, n=n, degree=degree, hidden=hidden, heads=heads, powers=powers, amp=amp)
    top = 24492 if kind == "eval" else 8000
    return dict(kind=kind, n=_log_int(rng, 1200, top), degree=degree, in_dim=rng.choice([64, 128, 300]),
                hidden=hidden, heads=min(heads, 6), layers=rng.randint(1, 3), powers=powers, amp=amp)


# ---------------------------------------------------------------------------
# Graphs and inputs
# ---------------------------------------------------------------------------


@functools.lru_cache(maxsize=32)
def _host_graph(n, degree):
    """(edge_index [2, E] as a loader returns it, P on the host, GAT graph on
    the host) of a power-law graph whose hubs grow with it."""
    ei = torch.from_numpy(graphgen.chung_lu_directed(n, n * degree // 2 * 2, gamma=2.5, max_degree=max(32.0, n / 22.0),
                                                     seed=n + degree))
    used, P = graph.build_sparse_normalized_adjacency(ei, n)
    return ei, graph.prepare_fixed_csr_operator(P), graph.prepare_fused_gat_graph(
        graph.prepare_gat_edge_index(used, n), n)


def _operator(case):
    host = _host_graph(case["n"], case["degree"])[1]
    up = lambda c: torch.sparse_csr_tensor(c.crow_indices().to(DEV), c.col_indices().to(DEV), c.values().to(DEV),
                                           size=c.shape)
    return graph.FixedCSRGraphOperator(up(host.csr), up(host.csr_t))


def _gat_graph(case):
    (rowptr, col), (row, colptr), perm = _host_graph(case["n"], case["degree"])[2]
    rowptr, col, row, colptr, perm = (t.to(DEV) for t in (rowptr, col, row, colptr, perm))
    return (rowptr, col), (row, colptr), perm


def _powers(case):
    return tuple(int(p) for p in case["powers"].split(","))


def _dtype(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float32


class _Inputs:
    """Random values in the order of the calls, from one seed."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEV).manual_seed(int(seed))

    def normal(self, *shape, scale=1.0, dtype=torch.float32, grad=False):
        t = torch.randn(*shape, generator=self.gen, device=DEV).mul_(scale).to(dtype)
        return t.requires_grad_(grad)

    def uniform(self, *shape):
        return torch.rand(*shape, generator=self.gen, device=DEV)


def _module(case, seed):
    """The case's module with the weights of the seed, in its training state."""
    with torch.random.fork_rng(devices=[]):
        torch.manual_seed(int(seed))
        if case["kind"] == "conv":
            m = CompatibleCollapsedFusedGATConv(case["in_dim"], case["channels"], heads=case["heads"], dropout=0.0)
            m._selective_amp_enabled = case["amp"]
        elif case["kind"] == "block":
            m = GraphCliffordBlock(hidden_dim=case["hidden"], order_set=_powers(case), dropout=0.0,
                                   gat_heads=case["heads"], gat_dropout=0.0, use_selective_amp=case["amp"])
        else:
            m = GraphCliffordNet(in_dim=case["in_dim"], hidden_dim=case["hidden"], out_dim=CLASSES,
                                 num_layers=case["layers"], order_set=_powers(case), dropout=0.0,
                                 gat_heads=case["heads"], gat_dropout=0.0, use_selective_amp=case["amp"])
    return m.to(DEV).train()


def prepare(case, seed):
    """Inputs, weights and graph operators as a program holds them."""
    kind, n = case["kind"], case["n"]
    inp = _Inputs(seed)
    s = {"case": case}
    if kind == "multihop":
        base = _operator(case)
        powers, dt = _powers(case), _dtype(case)
        if dt is torch.bfloat16:
            powers = (1, 2, 3)  # the operator that has the bf16 option
            s["op"] = MultiHopCSR3GraphOperator(base, dense_cols=case["cols"], dense_dtype=dt)
        else:
            s["op"] = prepare_multihop_csr_operator(base, dense_cols=case["cols"], powers=powers)
        s["powers"] = powers
        s["x"] = inp.normal(n, case["cols"], dtype=dt, grad=True)
        s["gy"] = [inp.normal(n, case["cols"], dtype=dt) for _ in powers]
    elif kind == "gat":
        H, C, dt = case["heads"], case["channels"], _dtype(case)
        s["graph"] = _gat_graph(case)
        s["x"] = inp.normal(n, H, C, dtype=dt, grad=True)
        s["a_dst"], s["a_src"] = inp.normal(n, H, grad=True), inp.normal(n, H, grad=True)
        s["bias"] = inp.normal(C, scale=0.1, grad=True)
        s["gy"] = inp.normal(n, C, dtype=dt)
        s["seed"] = (int(seed) * 7919 + 12345) % (1 << 62)
    elif kind == "conv":
        s["graph"] = _gat_graph(case)
        s["module"] = _module(case, seed)
        s["x"] = inp.normal(n, case["in_dim"], grad=True)
        s["gy"] = inp.normal(n, case["channels"])
    elif kind == "pack":
        D = case["hidden"]
        s["H"], s["C"] = inp.normal(n, D, grad=True), inp.normal(n, D, grad=True)
        s["props"] = [inp.normal(n, 2 * D, scale=0.5, grad=True) for _ in range(3)]
        s["alpha"] = torch.softmax(inp.normal(n, 3), -1).requires_grad_(True)
        s["gy"] = inp.normal(n, 6 * D)
    elif kind == "block":
        s["graph"] = _gat_graph(case)
        s["op"] = prepare_multihop_csr_operator(_operator(case), dense_cols=2 * case["hidden"], powers=_powers(case))
        s["module"] = _module(case, seed)
        s["x"] = inp.normal(n, case["hidden"], grad=True)
        s["gy"] = inp.normal(n, case["hidden"])
    else:
        m = s["module"] = _module(case, seed)
        x = inp.normal(n, case["in_dim"])
        y = (inp.uniform(n) * CLASSES).long().clamp_(max=CLASSES - 1)
        mask = inp.uniform(n) < 0.5
        host = train_cign.GraphData(x=x, y=y, edge_index=_host_graph(n, case["degree"])[0], train_mask=mask)
        ready = train_cign.prepare_graph(m, host, torch.device(DEV), hop_scales=_powers(case))
        s["op"] = ready.graph_operator
        s["data"] = train_cign.GraphData(x=x, y=y, edge_index=ready.edge_index, train_mask=mask)
    if "module" in s:
        s["params"] = [p for p in s["module"].parameters() if p.requires_grad]
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "multihop":
        out = graph.selected_sparse_powers(s["op"], s["x"], s["powers"])
        ys = [out[p] for p in s["powers"]]
        return [y.detach() for y in ys], torch.autograd.grad(ys, s["x"], s["gy"])
    if kind == "gat":
        (rowptr, col), (row, colptr), perm = s["graph"]
        if case["drop"] > 0.0:
            ext = ensure_collapsed_gat_loaded()
            x, a_dst, a_src, bias = (s[k].detach() for k in ("x", "a_dst", "a_src", "bias"))
            (y, pre, mx, sm, mask), agg = ext.forward_agg(a_dst, a_src, rowptr, col, SLOPE, x, bias, case["drop"],
                                                          s["seed"], True)
            gx, g_dst, g_src, g_bias = ext.backward(SLOPE, case["drop"], rowptr, col, colptr, row, perm, mx, sm, mask,
                                                    x, a_dst, a_src, pre, s["gy"], agg)
            return y, gx, g_dst, g_src, g_bias
        y = collapsed_gat_mean_bias_silu(s["a_dst"], s["a_src"], (rowptr, col), (row, colptr), perm, SLOPE, s["x"],
                                         s["bias"], 0.0)
        grads = torch.autograd.grad(y, [s["x"], s["a_dst"], s["a_src"], s["bias"]], s["gy"])
        return (y.detach(), *grads)
    if kind == "conv":
        csr, csc, perm = s["graph"]
        y = s["module"](s["x"], csr, csc, perm)
        return (y.detach(), *torch.autograd.grad(y, [s["x"], *s["params"]], s["gy"]))
    if kind == "pack":
        leaves = [s["H"], s["C"], *s["props"], s["alpha"]]
        y = fused_clifford_switch_pack(s["H"], s["C"], s["props"], s["alpha"], "new", "old")
        return (y.detach(), *torch.autograd.grad(y, leaves, s["gy"]))
    if kind == "block":
        y = s["module"](s["x"], None, s["op"], fused_gat_graph=s["graph"])
        return (y.detach(), *torch.autograd.grad(y, [s["x"], *s["params"]], s["gy"]))
    if kind == "train":
        data = s["data"]
        logits = train_cign.forward_model(s["module"], data, s["op"])
        loss = F.cross_entropy(logits[data.train_mask], data.y[data.train_mask])
        return (logits.detach(), *torch.autograd.grad(loss, s["params"]))
    return train_cign.evaluate_logits(s["module"], s["data"], s["op"])


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how exact its results are
# ---------------------------------------------------------------------------


def _conv_work(n, E, in_dim, H, C, train):
    """The projection's operands and results and the graph; x_proj itself is
    an intermediate."""
    w = in_dim * H * C
    flops = 2 * n * w + 4 * n * H * C + 2 * E * H * C + 8 * E * H
    nbytes = 4 * (n * in_dim + w + n * C + E + n)
    if train:
        flops += 4 * n * w + 4 * E * H * C + 12 * n * H * C
        nbytes += 4 * (n * C + n * in_dim + w + 2 * E + n)
    return nbytes, flops


def _block_work(n, E, hidden, heads, powers, train):
    """A block's input, output and weights and the graph's arrays (each read
    once in each direction)."""
    D, K, top = hidden, len(powers), max(powers)
    nbytes, flops = _conv_work(n, E, D, heads, D, train)
    nbytes = 4 * (2 * n * D + heads * D * D + 2 * K * D * D + 3 * E + 2 * n)
    fwd = 4 * E * D * top + 2 * n * 2 * K * D * D + 30 * n * D * K
    flops += fwd
    if train:
        nbytes += 4 * (2 * n * D + heads * D * D + 2 * K * D * D + 4 * E + 2 * n)
        flops += 2 * fwd
    return nbytes, flops


def work(case):
    kind, n = case["kind"], case["n"]
    E = n * case.get("degree", 0) // 2 * 2 + n  # one self-loop a node
    if kind == "multihop":
        s = 2 if case["dtype"] == "bf16" else 4
        powers = _powers(case) if s == 4 else (1, 2, 3)
        D, K = case["cols"], len([p for p in powers if p])
        return dict(bytes=s * n * D * (2 * K + 2) + 2 * (8 * E + 4 * n), flops=4 * E * D * max(powers))
    if kind == "gat":
        s = 2 if case["dtype"] == "bf16" else 4
        H, C = case["heads"], case["channels"]
        return dict(bytes=2 * s * n * H * C + 2 * s * n * C + 16 * n * H + 4 * (3 * E + 2 * n) + 8 * C,
                    flops=6 * E * H * C + 30 * E * H)
    if kind == "conv":
        b, f = _conv_work(n, E, case["in_dim"], case["heads"], case["channels"], True)
        return dict(bytes=b, flops=f)
    if kind == "pack":
        D = case["hidden"]
        return dict(bytes=4 * n * (2 * (2 + 6) * D + 2 * 6 * D + 6), flops=90 * n * D)
    if kind == "block":
        b, f = _block_work(n, E, case["hidden"], case["heads"], _powers(case), True)
        return dict(bytes=b, flops=f)
    train = kind == "train"
    b, f = _block_work(n, E, case["hidden"], case["heads"], _powers(case), train)
    final = case["hidden"] * (case["layers"] + 1)
    ends = 2 * n * (2 * case["in_dim"] * case["hidden"] + final * CLASSES)
    # a layer's states are intermediates of the model: its weights are not
    weights = case["layers"] * (case["heads"] + 2 * len(_powers(case))) * case["hidden"] ** 2
    return dict(bytes=4 * (n * case["in_dim"] + n * CLASSES + (2 if train else 1) * (weights + 3 * E)),
                flops=case["layers"] * f + (3 if train else 1) * ends)


def tolerance(case):
    """About four times what the same path shows against 64 bits or against
    its unfused composition. Where logits are computed, not given, a sum near
    0 may fall on the other side of LeakyReLU's kink in another order of the
    same float32 arithmetic; one such edge moves an attention gradient by up
    to 4e-4 of its norm. Under autocast the roundings to bf16 follow each
    other through the gradients (7e-3 between two orders of the same model,
    6e-2 against 64 bits for the attention vectors)."""
    kind = case["kind"]
    if kind == "multihop":
        return {"rel": 1e-2 if case["dtype"] == "bf16" else 2e-6}
    if kind == "gat":
        return {"rel": 1e-2 if case["dtype"] == "bf16" else 1e-5}
    if kind == "pack":
        return {"rel": 2e-6}
    if kind == "eval":
        return {"rel": 1.5e-2 if case["amp"] else 5e-6}
    return {"rel": 3e-2 if case["amp"] else 2e-3}


# ---------------------------------------------------------------------------
# The same results in 64 bits, in plain torch
# ---------------------------------------------------------------------------


class _SpMM64(torch.autograd.Function):
    """y[r] += w x[c] over a list of entries, and its transpose."""

    @staticmethod
    def forward(ctx, x, r, c, w):
        ctx.save_for_backward(r, c, w)
        return _entries(x, r, c, w)

    @staticmethod
    def backward(ctx, g):
        r, c, w = ctx.saved_tensors
        return _entries(g, c, r, w), None, None, None


def _entries(x, r, c, w, chunk=1 << 20):
    y = torch.zeros_like(x)
    for at in range(0, r.numel(), chunk):
        sl = slice(at, at + chunk)
        y.index_add_(0, r[sl], w[sl, None] * x[c[sl]])
    return y


def _adjacency64(case):
    csr = _host_graph(case["n"], case["degree"])[1].csr
    crow = csr.crow_indices()
    r = torch.repeat_interleave(torch.arange(case["n"]), crow.diff()).to(DEV)
    return r, csr.col_indices().to(DEV), csr.values().to(DEV).double()


def _edges64(case):
    (rowptr, col), _, _ = _host_graph(case["n"], case["degree"])[2]
    r = torch.repeat_interleave(torch.arange(case["n"]), rowptr.long().diff()).to(DEV)
    return r, col.long().to(DEV)


def _powers64(x, adj, powers):
    out, cur = {0: x}, x
    for p in range(1, max(powers) + 1):
        cur = _SpMM64.apply(cur, *adj)
        out[p] = cur
    return [out[p] for p in powers]


def _keep64(seed, total, p):
    """The dropout mask of the package's documented bit stream: splitmix64 of
    seed ^ (index * constant), its upper half as a float32 uniform > p."""
    with np.errstate(over="ignore"):
        z = np.uint64(seed) ^ (np.arange(total, dtype=np.uint64) * np.uint64(0xD2B74407B1CE6E93))
        z = z + np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z = z ^ (z >> np.uint64(31))
    u = ((z >> np.uint64(32)).astype(np.float32) + np.float32(0.5)) * np.float32(2.0 ** -32)
    return torch.from_numpy(u > np.float32(p)).to(DEV)


def _gat64(x, a_dst, a_src, bias, edges, drop=0.0, seed=0):
    r, c = edges
    n, H, _ = x.shape
    e = F.leaky_relu(a_dst[r] + a_src[c], SLOPE)
    top = torch.full((n, H), -torch.inf, dtype=e.dtype, device=DEV).scatter_reduce(
        0, r[:, None].expand_as(e), e.detach(), "amax")
    ex = torch.exp(e - top[r])
    w = ex / torch.zeros(n, H, dtype=e.dtype, device=DEV).index_add(0, r, ex)[r]
    if drop > 0.0:
        # the mask compares with p, and the scale is that of p, in float32
        keep = _keep64(seed, w.numel(), drop).view_as(w)
        w = w * keep / (1.0 - float(np.float32(drop)))
    mean = sum(torch.zeros(n, x.size(2), dtype=x.dtype, device=DEV).index_add(0, r, w[:, h, None] * x[c, h])
               for h in range(H)) / H
    return F.silu(mean + bias)


def _conv64(x, g, pre, heads, edges):
    xp = F.linear(x, g[pre + "lin.weight"]).view(x.size(0), heads, -1)
    return _gat64(xp, (xp * g[pre + "att_dst"]).sum(-1), (xp * g[pre + "att_src"]).sum(-1), g[pre + "bias"], edges)


def _pack64(H, C, props, alpha):
    D = H.size(1)
    parts = []
    for k, P in enumerate(props):
        hc, ch = H * P[:, D:], C * P[:, :D]
        parts.append(alpha[:, k, None] * torch.cat([0.5 * (hc - ch), F.silu(0.5 * (hc + ch))], -1))
    return torch.cat(parts, -1)


def _block64(H, g, pre, case, edges, adj):
    D = H.size(1)
    Hn = F.layer_norm(H, (D,), g[pre + "h_norm.weight"], g[pre + "h_norm.bias"])
    Cg = _conv64(Hn, g, pre + "context_gat.", case["heads"], edges)
    Cn = F.layer_norm(Cg + Hn, (D,), g[pre + "c_norm.weight"], g[pre + "c_norm.bias"])
    props = _powers64(torch.cat([Hn, Cn], -1), adj, _powers(case))
    score = torch.cat([Hn + Cn, (Hn - Cn).abs()], -1)
    alpha = torch.softmax(F.linear(score, g[pre + "hop_gate_mlp.weight"], g[pre + "hop_gate_mlp.bias"]), -1)
    G = F.linear(_pack64(Hn, Cn, props, alpha), g[pre + "proj.weight"], g[pre + "proj.bias"])
    return H + g[pre + "gamma"] * G


def _net64(x, g, case, edges, adj):
    H = F.silu(F.linear(x, g["input_proj_0.weight"], g["input_proj_0.bias"]))
    H = H + g["input_eta"] * F.silu(F.linear(x, g["input_proj_1.weight"], g["input_proj_1.bias"]))
    states = [H]
    for i in range(case["layers"]):
        states.append(_block64(states[-1], g, f"blocks.{i}.", case, edges, adj))
    out = torch.cat(states, -1)
    out = F.layer_norm(out, (out.size(1),), g["output_norm.weight"], g["output_norm.bias"])
    return F.linear(out, g["classifier.weight"], g["classifier.bias"])


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    up = lambda t: t.detach().double().requires_grad_(t.requires_grad)
    if kind == "multihop":
        x = up(s["x"])
        ys = _powers64(x, _adjacency64(case), s["powers"])
        return [y.detach() for y in ys], torch.autograd.grad(ys, x, [t.double() for t in s["gy"]])
    if kind == "gat":
        leaves = [up(s[k]) for k in ("x", "a_dst", "a_src", "bias")]
        y = _gat64(*leaves, _edges64(case), case["drop"], s["seed"])
        return (y.detach(), *torch.autograd.grad(y, leaves, s["gy"].double()))
    if kind == "pack":
        leaves = [up(t) for t in (s["H"], s["C"], *s["props"], s["alpha"])]
        y = _pack64(leaves[0], leaves[1], leaves[2:5], leaves[5])
        return (y.detach(), *torch.autograd.grad(y, leaves, s["gy"].double()))
    g = {k: up(p) for k, p in s["module"].named_parameters()}
    edges = _edges64(case)
    if kind == "conv":
        x = up(s["x"])
        y = _conv64(x, g, "", case["heads"], edges)
        return (y.detach(), *torch.autograd.grad(y, [x, *g.values()], s["gy"].double()))
    adj = _adjacency64(case)
    if kind == "block":
        x = up(s["x"])
        y = _block64(x, g, "", case, edges, adj)
        return (y.detach(), *torch.autograd.grad(y, [x, *g.values()], s["gy"].double()))
    data = s["data"]
    if kind == "eval":
        with torch.no_grad():
            return _net64(data.x.double(), g, case, edges, adj)
    logits = _net64(data.x.double(), g, case, edges, adj)
    loss = F.cross_entropy(logits[data.train_mask], data.y[data.train_mask])
    return (logits.detach(), *torch.autograd.grad(loss, list(g.values())))
