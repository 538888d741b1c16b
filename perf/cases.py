"""The work this library is measured on: calls of its public entry points over the sizes they serve.

Sizes are the benchmark configurations' (hidden 4096, inter 2048, 256 experts, top-6; bench.py) and
those of the tests (smaller hidden and inter, other counts of experts and routes). Weights are
experts in the container layout with uniform codes and the block scales that quantised normal
weights have, permuted to the device layout by the library, as a loader does.

Kinds:
  decode    M <= 8 tokens through a stack of MoE layers (one fused launch a layer). Weights come
            from HBM: a pass reads more than the 256 MB cache holds, as a real stack does.
  sublayer  one token through whole MoE sublayers: router, routed experts, shared expert,
            hyper-connection post; each a call of its own.
  prefill   a batch or chunk of tokens through one layer's experts, grouped by expert.
  hook      the engine's batch hook: routes in host memory, f32 dim-major activations.
  shared    a chunk through the FP8 shared expert.
  steps     the separable pipeline: W8A8 GEMM, SwiGLU + requantise, W8A8 GEMM, scatter.
  quantize  the producer: one f32 matrix to codes, fields and row scales.
"""
import ctypes as C
import math

import numpy as np
import torch

import affinity_amd.experts as ax
from affinity_amd import _lib

LIMIT = 10.0
DENSE = {"hidden": 4096, "inter": 2048, "experts": 256, "top_k": 6}


def listed():
    return [
        # a chat turn's token: batch 1, the step a serving loop keeps in a HIP graph
        {"name": "decode-1", "kind": "decode", "tokens": 1, "layers": 8, "graph": True, "arena": False, **DENSE},
        # three speculative tokens, called layer by layer
        {"name": "decode-3", "kind": "decode", "tokens": 3, "layers": 4, "graph": False, "arena": False, **DENSE},
        # a six-token verify step in the engine's dim-major arena, added into its block
        {"name": "decode-6-arena", "kind": "decode", "tokens": 6, "layers": 4, "graph": False, "arena": True, **DENSE},
        # the widest decode: eight tokens, most experts serve one or two of them
        {"name": "decode-8", "kind": "decode", "tokens": 8, "layers": 4, "graph": False, "arena": False, **DENSE},
        # every call that a layer's token makes, one after the other: latency and launches
        {"name": "sublayer-1", "kind": "sublayer", "tokens": 1, "layers": 8, **DENSE},
        # a small batch of sequences decoding together, just above the decode entry's range
        {"name": "prefill-24", "kind": "prefill", "tokens": 24, "lo": False, "zipf": False, **DENSE},
        # a short ragged prompt with f32 activations as a bf16 pair
        {"name": "prefill-333-lo", "kind": "prefill", "tokens": 333, "lo": True, "zipf": False, **DENSE},
        # the benchmark's chunk: 4096 tokens, Zipf routes (a few heavy experts, many light ones)
        {"name": "prefill-4096", "kind": "prefill", "tokens": 4096, "lo": False, "zipf": True, **DENSE},
        # the engine's prefill chunk through its hook: host routes, arenas, a wait at the end
        {"name": "hook-512", "kind": "hook", "tokens": 512, "zipf": True, **DENSE},
        # a ragged chunk through the shared expert
        {"name": "shared-1500", "kind": "shared", "tokens": 1500, "lo": False, "hidden": 4096, "inter": 2048},
        # an engine that drives the separable steps itself, over a 256-token batch
        {"name": "steps-256", "kind": "steps", "tokens": 256, "zipf": True, **DENSE},
        # quantising one gate matrix of a checkpoint
        {"name": "quantize-gate", "kind": "quantize", "rows": 2048, "cols": 4096},
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "sublayer", "prefill", "prefill", "prefill", "hook", "hook",
                       "shared", "steps", "quantize"])
    dims = {"hidden": rng.choice([2048, 4096, 4096]), "inter": rng.choice([1024, 2048, 2048])}
    moe = {**dims, "experts": rng.choice([64, 128, 200, 256, 256]), "top_k": rng.choice([4, 6, 6, 8])}
    if kind == "decode":
        return {"kind": kind, "tokens": rng.randint(1, 8), "layers": rng.randint(4, 8), "graph": rng.random() < 0.5,
                "arena": rng.random() < 0.4, **moe}
    if kind == "sublayer":
        return {"kind": kind, "tokens": rng.randint(1, 4), "layers": rng.randint(6, 10), **moe}
    if kind == "prefill":
        return {"kind": kind, "tokens": _spread(rng, 9, 3000), "lo": rng.random() < 0.4, "zipf": rng.random() < 0.5, **moe}
    if kind == "hook":
        return {"kind": kind, "tokens": _spread(rng, 1, 2048), "zipf": rng.random() < 0.5, **moe}
    if kind == "shared":
        return {"kind": kind, "tokens": _spread(rng, 9, 4096), "lo": rng.random() < 0.4, **dims}
    if kind == "steps":
        return {"kind": kind, "tokens": _spread(rng, 24, 700), "zipf": rng.random() < 0.5, **moe}
    return {"kind": "quantize", "rows": _spread(rng, 64, 2048), "cols": 64 * rng.randint(8, 64)}


# ---- inputs, from the seed alone ------------------------------------------------------------------

def _gen(seed, part):
    return torch.Generator(device="cuda").manual_seed((seed * 1009 + part) & 0x7FFFFFFF)


def _bytes(g, n):
    r = torch.empty((n + 7) // 8, dtype=torch.int64, device="cuda").random_(-2 ** 63, None, generator=g)
    return r.view(torch.uint8)[:n]


def _layout(hidden, inter):
    """A container expert: its stride and the (offset, bytes) of its nine planes (gate, up, down:
    codes, fields, row scales). In memory the code planes come first, then the fields, then the
    scales, each on 256 bytes, the expert on 4096."""
    size = [n for r, k in ((inter, hidden), (inter, hidden), (hidden, inter))
            for n in (r * k * 10 // 32, r * k * 6 // 128, 2 * r)]
    off, at = [0] * 9, 0
    for p in (0, 3, 6, 1, 4, 7, 2, 5, 8):
        off[p] = at
        at = (at + size[p] + 255) // 256 * 256
    return (at + 4095) // 4096 * 4096, list(zip(off, size))


def _codebook():
    """The benchmark's fitted codebook: uint32 [2048], four E4M3 bytes each."""
    return np.fromfile("tests/golden/c1_codebook.bin", dtype="<u4")


def _container(c, seed, part):
    """One layer's experts, uint8 [experts][stride], in the container layout: uniform 10-bit codes,
    uniform sign, rotation and variant, and a block scale of 2^6 (82 %), 2^5 (13 %) or 2^7 (5 %)
    with row scales near 6e-4: what normal weights of deviation 0.02 quantise to."""
    n, h, i = c["experts"], c["hidden"], c["inter"]
    stride, planes = _layout(h, i)
    g = _gen(seed, 16 * part + 1)
    out = torch.zeros((n, stride), dtype=torch.uint8, device="cuda")
    for e0 in range(0, n, 64):
        m = min(64, n - e0)
        for k in range(3):
            (oc, sc), (of, sf), (orr, sr) = planes[3 * k:3 * k + 3]
            out[e0:e0 + m, oc:oc + sc] = _bytes(g, m * sc).view(m, sc)
            blocks = sf // 3 * 4
            r = _bytes(g, m * blocks)
            s = torch.full_like(r, 6)
            s[r < 33] = 5
            s[r > 242] = 7
            f = (s | ((_bytes(g, m * blocks) & 7) << 3)).view(m, blocks // 4, 4)
            packed = torch.stack([f[..., 0] | (f[..., 1] << 6), (f[..., 1] >> 2) | (f[..., 2] << 4),
                                  (f[..., 2] >> 4) | (f[..., 3] << 2)], dim=-1)
            out[e0:e0 + m, of:of + sf] = packed.view(m, sf)
            rs = 6e-4 * (1 + 0.08 * torch.randn(m, sr // 2, generator=g, device="cuda"))
            out[e0:e0 + m, orr:orr + sr] = rs.clamp(4e-4, 9e-4).to(torch.bfloat16).view(torch.uint8).view(m, sr)
    return out


def _routes(c, T, seed, part):
    """sel int32 [T][k], w f32 [T][k]: distinct experts, by N(0,1) router logits or with Zipf(1.1)
    popularity over a permutation of the experts; the weights a softmax."""
    g, n, k = _gen(seed, 16 * part + 2), c["experts"], c["top_k"]
    if c.get("zipf"):
        p = -1.1 * torch.log(torch.arange(1, n + 1, device="cuda", dtype=torch.float32))
        p = p[torch.randperm(n, generator=g, device="cuda")]
        u = torch.rand(T, n, generator=g, device="cuda").clamp_min(1e-20)
        sel = torch.topk(p - torch.log(-torch.log(u)), k, dim=1).indices
        w = torch.softmax(torch.randn(T, k, generator=g, device="cuda"), dim=1)
    else:
        top = torch.topk(torch.randn(T, n, generator=g, device="cuda"), k, dim=1)
        sel, w = top.indices, torch.softmax(top.values, dim=1)
    return sel.to(torch.int32).contiguous(), w.float().contiguous()


def _x(c, T, seed, part):
    return torch.randn(T, c["hidden"], generator=_gen(seed, 16 * part + 3), device="cuda")


def _pool(c, seed, part):
    return ax.ExpertPool.from_container(_container(c, seed, part).view(-1), _codebook(), c["hidden"],
                                        c["inter"], swiglu_limit=LIMIT)


def _fp8(rows, cols, g):
    """Dense FP8 weights as a checkpoint holds them: E4M3 bytes, UE8M0 scales per 128 x 128 tile."""
    w = (48 * torch.randn(rows, cols, generator=g, device="cuda")).clamp(-448, 448).to(torch.float8_e4m3fn)
    s = torch.randint(115, 118, (rows // 128, cols // 128), generator=g, device="cuda", dtype=torch.uint8)
    return w.view(torch.uint8), s


def _shared_weights(c, seed, part):
    g, h, i = _gen(seed, 16 * part + 4), c["hidden"], c["inter"]
    return [t for rows, cols in ((i, h), (i, h), (h, i)) for t in _fp8(rows, cols, g)]


def _hc_inputs(c, T, seed, part):
    """The hyper-connection state and control of one sublayer: hc [4][hidden], post [4], comb [16]."""
    g = _gen(seed, 16 * part + 5)
    return (torch.randn(T, 4, c["hidden"], generator=g, device="cuda"), torch.rand(T, 4, generator=g, device="cuda"),
            torch.softmax(torch.randn(T, 16, generator=g, device="cuda"), dim=1))


def _logits(c, T, seed, part):
    g = _gen(seed, 16 * part + 6)
    return (torch.randn(T, c["experts"], generator=g, device="cuda"),
            0.05 * torch.randn(c["experts"], generator=g, device="cuda"))


def _a8(T, cols, seed):
    """E4M3 activations with one scale per (token, 128 columns): what the batch quantiser makes."""
    x = torch.randn(T, cols, generator=_gen(seed, 7), device="cuda").view(T, cols // 128, 128)
    s = x.abs().amax(-1, keepdim=True) / 448
    return (x / s).to(torch.float8_e4m3fn).view(T, cols).view(torch.uint8), s.view(T, cols // 128).contiguous()


def _slots(sel, n):
    """The slot list of a batch's routes (host): slots sorted by expert, then token; each token's
    slots in route order."""
    T, k = sel.shape
    order = np.argsort(sel.reshape(-1), kind="stable")
    count = np.bincount(sel.reshape(-1), minlength=n)
    ordv = np.empty(T * k, np.int32)
    ordv[order] = np.arange(T * k, dtype=np.int32)
    return (order // k).astype(np.int32), order, count, ordv, (np.arange(T + 1) * k).astype(np.int32)


# ---- prepare: what a program has in hand before the call ------------------------------------------

def prepare(case, seed):
    return {"decode": _prepare_decode, "sublayer": _prepare_sublayer, "prefill": _prepare_prefill,
            "hook": _prepare_hook, "shared": _prepare_shared, "steps": _prepare_steps,
            "quantize": _prepare_quantize}[case["kind"]](case, seed)


def _prepare_decode(c, seed):
    ax.init()
    M, n = c["tokens"], c["layers"]
    s = {"run": _run_decode, "arena": c["arena"], "pools": [_pool(c, seed, l) for l in range(n)],
         "routes": [_routes(c, M, seed, l) for l in range(n)],
         "ws": ax.DecodeWorkspace(M, c["top_k"], c["hidden"], c["inter"])}
    x = [_x(c, M, seed, l) for l in range(n)]
    if c["arena"]:  # the engine's dim-major arenas, 16 tokens wide
        s["xa"] = torch.zeros((n, c["hidden"], 16), device="cuda")
        s["ya"] = torch.zeros((n, c["hidden"], 16), device="cuda")
        for l in range(n):
            s["xa"][l, :, :M] = x[l].t()
        s["x"], s["y"] = [a[:, :M] for a in s["xa"]], [a[:, :M] for a in s["ya"]]
    else:
        s["x"], s["y"] = x, [torch.zeros_like(a) for a in x]
    if c["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _decode_stack(s)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            _decode_stack(s)
        s["run"] = _replay
    return s


def _decode_stack(s):
    if s["arena"]:
        s["ya"].zero_()
    for pool, x, (sel, w), y in zip(s["pools"], s["x"], s["routes"], s["y"]):
        ax.expert_ffn_decode(pool, x, sel, w, y=y, accumulate=s["arena"], workspace=s["ws"], dim_major=s["arena"])


def _run_decode(s):
    _decode_stack(s)
    return s["y"]


def _replay(s):
    s["graph"].replay()
    return s["y"]


def _prepare_sublayer(c, seed):
    ax.init()
    M, k, layers = c["tokens"], c["top_k"], []
    for l in range(c["layers"]):
        logits, bias = _logits(c, M, seed, l)
        hc, post, comb = _hc_inputs(c, M, seed, l)
        layers.append({"pool": _pool(c, seed, l), "shared": ax.SharedExpert(*_shared_weights(c, seed, l), LIMIT),
                       "x": _x(c, M, seed, l), "logits": logits, "bias": bias, "hc": hc, "post": post, "comb": comb,
                       "sel": torch.zeros((M, k), dtype=torch.int32, device="cuda"),
                       "w": torch.zeros((M, k), device="cuda"), "block": torch.zeros((M, c["hidden"]), device="cuda"),
                       "out": torch.zeros_like(hc)})
    return {"run": _run_sublayer, "layers": layers, "case": c,
            "ws": ax.DecodeWorkspace(M, k, c["hidden"], c["inter"])}


def _run_sublayer(s):
    c = s["case"]
    M, n, k = c["tokens"], c["experts"], c["top_k"]
    for a in s["layers"]:
        _lib.check(_lib.lib().affx_route_topk(a["logits"].data_ptr(), n, 1, a["bias"].data_ptr(), M, n, k,
                                              _lib.AFFX_ROUTE_ENGINE, 1, 1.5, a["sel"].data_ptr(), a["w"].data_ptr(),
                                              torch.cuda.current_stream().cuda_stream), "route_topk")
        ax.expert_ffn_decode(a["pool"], a["x"], a["sel"], a["w"], y=a["block"], workspace=s["ws"])
        a["shared"].decode(a["x"], a["block"], accumulate=True)
        for t in range(M):
            ax.hc_post(a["block"][t], a["hc"][t], a["post"][t], a["comb"][t], out_hc=a["out"][t], zero_block=True)
    return {"hc": [a["out"] for a in s["layers"]], "sel": [a["sel"] for a in s["layers"]],
            "w": [a["w"] for a in s["layers"]]}


def _split(x):
    hi = x.to(torch.bfloat16)
    return hi, (x - hi.float()).to(torch.bfloat16)


def _prepare_prefill(c, seed):
    ax.init()
    T = c["tokens"]
    hi, lo = _split(_x(c, T, seed, 0))
    sel, w = _routes(c, T, seed, 0)
    return {"run": _run_prefill, "pool": _pool(c, seed, 0), "x": hi, "lo": lo if c["lo"] else None, "sel": sel, "w": w,
            "y": torch.zeros((T, c["hidden"]), device="cuda"),
            "ws": ax.GroupedWorkspace(T, c["top_k"], c["experts"], c["hidden"], c["inter"])}


def _run_prefill(s):
    return ax.expert_ffn_grouped(s["pool"], s["x"], s["sel"], s["w"], y=s["y"], x_lo=s["lo"], workspace=s["ws"])


def _prepare_hook(c, seed):
    ax.init()
    T = c["tokens"]
    sel, w = _routes(c, T, seed, 0)
    pool = _pool(c, seed, 0)
    x = _x(c, T, seed, 0).t().contiguous()
    block = torch.zeros((c["hidden"], T), device="cuda")
    n = int(_lib.lib().affx_batch_workspace_size(T, c["top_k"], c["experts"], c["hidden"], c["inter"]))
    ws = torch.zeros(n, dtype=torch.uint8, device="cuda")
    layers = (_lib.AffxLayer * 1)(pool.layer())
    ctx = _lib.AffxEngineCtx(layers, 1, x.data_ptr(), block.data_ptr(), T, ws.data_ptr(), n,
                             torch.cuda.current_stream().cuda_stream)
    return {"run": _run_hook, "ctx": ctx, "keep": (pool, layers, ws, x), "block": block, "T": T, "k": c["top_k"],
            "sel": sel.cpu().numpy().astype(np.uint32), "w": w.cpu().numpy(),
            "handled": np.zeros((T, c["top_k"]), np.uint8)}


def _run_hook(s):
    s["block"].zero_()
    taken = _lib.lib().affx_expert_ffn_batch(C.addressof(s["ctx"]), 0, s["sel"].ctypes.data, s["w"].ctypes.data, s["T"],
                                             s["k"], s["handled"].ctypes.data)
    return {"block": s["block"], "taken": taken, "handled": s["handled"]}


def _prepare_shared(c, seed):
    ax.init()
    hi, lo = _split(_x(c, c["tokens"], seed, 0))
    return {"run": _run_shared, "shared": ax.SharedExpert(*_shared_weights(c, seed, 0), LIMIT), "x": hi,
            "lo": lo if c["lo"] else None, "y": torch.zeros((c["tokens"], c["hidden"]), device="cuda")}


def _run_shared(s):
    return s["shared"].batch(s["x"], s["y"], x_lo=s["lo"], accumulate=False)


def _prepare_steps(c, seed):
    ax.init()
    T, h, i, n, k = c["tokens"], c["hidden"], c["inter"], c["experts"], c["top_k"]
    pool = _pool(c, seed, 0)
    x8, xs = _a8(T, h, seed)
    sel, w = _routes(c, T, seed, 0)
    tok, order, count, ordv, run = _slots(sel.cpu().numpy(), n)
    S = T * k
    dev = {"tok": torch.from_numpy(tok).cuda(), "slot": torch.arange(S, dtype=torch.int32, device="cuda"),
           "wt": torch.from_numpy(w.cpu().numpy().reshape(-1)[order].copy()).cuda(),
           "ord": torch.from_numpy(ordv).cuda(), "runs": torch.from_numpy(run).cuda(),
           "g": torch.zeros((i, S), dtype=torch.bfloat16, device="cuda"),
           "u": torch.zeros((i, S), dtype=torch.bfloat16, device="cuda"),
           "a8": torch.zeros((S, i), dtype=torch.uint8, device="cuda"), "as": torch.zeros((S, i // 128), device="cuda"),
           "z": torch.zeros((h, S), dtype=torch.bfloat16, device="cuda"), "block": torch.zeros((h, T), device="cuda")}
    # one descriptor for every 64 slots of an expert, for gate, up and down
    spans, at = [], 0
    for e in range(n):
        for b in range(0, int(count[e]), 64):
            spans.append((e, at + b, min(64, int(count[e]) - b)))
        at += int(count[e])
    tiles = []
    for m, (ids, out) in enumerate((("tok", "g"), ("tok", "u"), ("slot", "z"))):
        d = (_lib.AffxExpertTile * len(spans))()
        for q, (e, s0, nt) in enumerate(spans):
            a = pool.matrix(e, m)
            d[q] = _lib.AffxExpertTile(a.codes, a.fields, a.rscales, dev[ids].data_ptr() + 4 * s0,
                                       dev[out].data_ptr() + 2 * s0, nt, S)
        tiles.append(torch.from_numpy(np.frombuffer(bytes(d), np.uint8).copy()).cuda())
    return {"run": _run_steps, "case": c, "pool": pool, "x8": x8, "xs": xs, "tiles": tiles, "n_tiles": len(spans),
            "max_nt": max(t[2] for t in spans), "S": S, **dev}


def _run_steps(s):
    c, L, stream = s["case"], _lib.lib(), torch.cuda.current_stream().cuda_stream
    T, h, i, S, cb = c["tokens"], c["hidden"], c["inter"], s["S"], s["pool"].codebook.data_ptr()

    def gemm(m, x8, xs, rows, cols):
        _lib.check(L.affx_expert_gemm_w8a8(s["tiles"][m].data_ptr(), s["n_tiles"], s["max_nt"], x8.data_ptr(),
                                           xs.data_ptr(), cb, rows, cols, 1.0, 1, stream), "gemm_w8a8")

    gemm(0, s["x8"], s["xs"], i, h)
    gemm(1, s["x8"], s["xs"], i, h)
    _lib.check(L.affx_expert_swiglu_quant(s["g"].data_ptr(), s["u"].data_ptr(), s["wt"].data_ptr(), s["a8"].data_ptr(),
                                          s["as"].data_ptr(), i, S, LIMIT, stream), "swiglu_quant")
    gemm(2, s["a8"], s["as"], h, i)
    s["block"].zero_()
    _lib.check(L.affx_expert_scatter_slots(s["z"].data_ptr(), s["block"].data_ptr(), s["ord"].data_ptr(),
                                           s["runs"].data_ptr(), h, T, T, S, stream), "scatter_slots")
    return {"g": s["g"], "u": s["u"], "block": s["block"]}


def _prepare_quantize(c, seed):
    ax.init()
    g = _gen(seed, 8)
    w = (0.02 * torch.randn(c["rows"], c["cols"], generator=g, device="cuda")).to(torch.bfloat16).float()
    cb = torch.from_numpy(ax.codebook_floats(_codebook())).cuda()
    return {"run": _run_quantize, "w": w, "cb": cb}


def _run_quantize(s):
    return ax.quantize_matrix(s["w"], s["cb"])


def run(state):
    return state["run"](state)


# ---- what a pass cannot do without ----------------------------------------------------------------

def _distinct(c, T):
    """Expected number of experts that T tokens' routes name."""
    n, k = c["experts"], c["top_k"]
    p = np.ones(n) / n
    if c.get("zipf"):
        p = 1.0 / np.arange(1, n + 1) ** 1.1
        p /= p.sum()
    # chance that one token's k draws without replacement name the expert: scaled to sum to k
    q, a = None, 0.0
    for a in np.linspace(1.0, 8.0 * k, 2000):
        q = 1 - np.exp(-a * p)
        if q.sum() >= min(k, n - 0.5):
            break
    return float(np.sum(1 - (1 - q) ** T))


def _expert_bytes(h, i):
    return 3 * h * i * (10 / 32 + 6 / 128) + 2 * (2 * i + h)


def work(case):
    c, kind = case, case["kind"]
    if kind == "quantize":
        n = c["rows"] * c["cols"]
        # one search of the 1024 entries for every quad (difference, square, sum in four dimensions);
        # how many settings of a block have to be searched in full is the algorithm's own business
        return {"bytes": n * 4 + n * (10 / 32 + 6 / 128), "flops": n / 4 * 1024 * 12}
    h, i, T = c["hidden"], c["inter"], c["tokens"]
    if kind == "shared":
        io = T * h * (2 * (2 if c["lo"] else 1) + 4)
        return {"bytes": 3 * h * i + io, "flops": 6 * h * i * T}
    k, per_slot = c["top_k"], 6 * h * i
    w = _distinct(c, T) * _expert_bytes(h, i)
    if kind == "decode":
        return {"bytes": c["layers"] * (w + 8 * T * h), "flops": c["layers"] * T * k * per_slot}
    if kind == "sublayer":
        return {"bytes": c["layers"] * (w + 3 * h * i + T * h * 4 * 10), "flops": c["layers"] * T * (k + 1) * per_slot}
    if kind == "prefill":
        return {"bytes": w + T * h * (2 * (2 if c["lo"] else 1) + 4), "flops": T * k * per_slot}
    if kind == "hook":
        return {"bytes": w + T * h * 12, "flops": T * k * per_slot}
    # steps: the arenas between the calls are results of the calls
    return {"bytes": w + T * h * (1 + 8) + T * k * (2 * 2 * 2 * i + 2 * i + 2 * 2 * h), "flops": T * k * per_slot}


def tolerance(case):
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    if kind == "shared":
        # bf16 products with f32 sums, the SwiGLU output as two bf16 terms: 2.5e-6 against 64 bits
        return {"rel": 1e-5, "max": 1e-4}
    if kind == "sublayer":
        # the shared expert's three E4M3 terms: about 3e-4 of its output
        return {"rel": 4e-4, "max": 4e-3, "differ": 0.0}
    if kind == "steps":
        # bf16 arenas, and an E4M3 requantisation that turns a flipped bf16 bit into a flipped code
        return {"rel": 1e-2, "max": 5e-2}
    # three E4M3 terms an activation (about 12 bits) and the MFMA's own accumulation: 4.5e-5
    return {"rel": 2e-4, "max": 2e-3, "differ": 0.0}


# ---- the same in 64 bits, by plain torch ----------------------------------------------------------

def _codebook64():
    by = torch.from_numpy(_codebook().view(np.uint8).astype(np.int64)).cuda()
    e, m = by >> 3 & 15, by & 7
    return ((1 - 2 * (by >> 7)) * (1 + m.double() / 8) * torch.pow(2.0, (e - 7).double())).view(2, 1024, 4)


def _dequant(expert, planes, m, rows, cols, cb):
    """One matrix of a container expert in float64 [rows][cols]."""
    (oc, sc), (of, sf), (orr, sr) = planes[3 * m:3 * m + 3]
    b = expert[oc:oc + sc].view(-1, 5).to(torch.int32)
    q = torch.stack([b[:, 0] | (b[:, 1] & 3) << 8, b[:, 1] >> 2 | (b[:, 2] & 15) << 6,
                     b[:, 2] >> 4 | (b[:, 3] & 63) << 4, b[:, 3] >> 6 | b[:, 4] << 2], dim=1).view(-1, 4)
    f = expert[of:of + sf].view(-1, 3).to(torch.int32)
    f = torch.stack([f[:, 0] & 63, f[:, 0] >> 6 | (f[:, 1] & 15) << 2, f[:, 1] >> 4 | (f[:, 2] & 3) << 4,
                     f[:, 2] >> 2], dim=1).view(-1)
    v = cb[(f >> 5).long()[:, None], q.long()]                               # [blocks][4 quads][4]
    v = torch.where((f >> 4 & 1).bool()[:, None, None], v.roll(2, dims=2), v)
    v = v * (torch.pow(2.0, (f & 7).double()) * (1 - 2 * (f >> 3 & 1)))[:, None, None]
    rs = expert[orr:orr + sr].view(torch.bfloat16).double()
    return v.view(rows, cols) * rs[:, None]


def _swiglu(g, u):
    g, u = g.clamp(max=LIMIT), u.clamp(-LIMIT, LIMIT)
    return g * torch.sigmoid(g) * u


def _ffn64(c, container, x, sel, w):
    """y[t] = sum_j w[t][j] FFN_sel[t][j](x[t]) in float64, expert by expert."""
    h, i = c["hidden"], c["inter"]
    planes, cb = _layout(h, i)[1], _codebook64()
    y = torch.zeros((x.shape[0], h), dtype=torch.float64, device="cuda")
    for e in torch.unique(sel).tolist():
        t, j = torch.nonzero(sel == e, as_tuple=True)
        a = x[t]
        a = _swiglu(a @ _dequant(container[e], planes, 0, i, h, cb).t(), a @ _dequant(container[e], planes, 1, i, h, cb).t())
        y.index_add_(0, t, (a @ _dequant(container[e], planes, 2, h, i, cb).t()) * w[t, j].double()[:, None])
    return y


def _shared64(weights, x):
    m = [w.view(torch.float8_e4m3fn).double() * torch.pow(2.0, s.double() - 127).repeat_interleave(128, 0)
         .repeat_interleave(128, 1) for w, s in zip(weights[::2], weights[1::2])]
    return _swiglu(x @ m[0].t(), x @ m[1].t()) @ m[2].t()


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "quantize":  # bytes: compared as they are
        return None
    if kind == "decode":
        ys = [_ffn64(c, _container(c, seed, l), _x(c, c["tokens"], seed, l).double(), *_routes(c, c["tokens"], seed, l))
              for l in range(c["layers"])]
        return [y.t() for y in ys] if c["arena"] else ys
    if kind == "sublayer":
        return _exact_sublayer(c, seed)
    T = c["tokens"]
    x = _x(c, T, seed, 0)
    if kind == "hook":
        y = _ffn64(c, _container(c, seed, 0), x.double(), *_routes(c, T, seed, 0))
        return {"block": y.t(), "taken": None, "handled": None}
    if kind == "steps":
        return _exact_steps(c, seed)
    hi, lo = _split(x)
    x = hi.double() + (lo.double() if c["lo"] else 0)
    if kind == "shared":
        return _shared64(_shared_weights(c, seed, 0), x)
    return _ffn64(c, _container(c, seed, 0), x, *_routes(c, T, seed, 0))


def _exact_sublayer(c, seed):
    M, k, hcs, ws = c["tokens"], c["top_k"], [], []
    for l in range(c["layers"]):
        logits, bias = _logits(c, M, seed, l)
        score = torch.sqrt(torch.nn.functional.softplus(logits.double()))
        sel = torch.topk(score + bias.double(), k, dim=1).indices
        w = torch.gather(score, 1, sel)
        w = w / w.sum(1, keepdim=True) * 1.5
        x = _x(c, M, seed, l).double()
        block = _ffn64(c, _container(c, seed, l), x, sel, w) + _shared64(_shared_weights(c, seed, l), x)
        hc, post, comb = (t.double() for t in _hc_inputs(c, M, seed, l))
        mix = comb.view(M, 4, 4)  # [src][dst]
        hcs.append(block[:, None, :] * post[:, :, None] + torch.einsum("tsd,tsh->tdh", mix, hc))
        ws.append(w)
    return {"hc": hcs, "sel": [None] * c["layers"], "w": ws}


def _exact_steps(c, seed):
    """Without the roundings between the steps (bf16 and E4M3 arenas)."""
    T, h, i, n = c["tokens"], c["hidden"], c["inter"], c["experts"]
    cont = _container(c, seed, 0)
    planes, cb = _layout(h, i)[1], _codebook64()
    x8, xs = _a8(T, h, seed)
    x = x8.view(torch.float8_e4m3fn).double() * xs.double().repeat_interleave(128, 1)
    sel, w = _routes(c, T, seed, 0)
    tok, order, count, _, _ = _slots(sel.cpu().numpy(), n)
    tok, wt = torch.from_numpy(tok).long().cuda(), w.reshape(-1)[torch.from_numpy(order).cuda()].double()
    g = torch.empty((i, tok.numel()), dtype=torch.float64, device="cuda")
    u, block, at = torch.empty_like(g), torch.zeros((h, T), dtype=torch.float64, device="cuda"), 0
    for e in range(n):
        m = int(count[e])
        if m == 0:
            continue
        s = slice(at, at + m)
        g[:, s] = _dequant(cont[e], planes, 0, i, h, cb) @ x[tok[s]].t()
        u[:, s] = _dequant(cont[e], planes, 1, i, h, cb) @ x[tok[s]].t()
        z = _dequant(cont[e], planes, 2, h, i, cb) @ (_swiglu(g[:, s], u[:, s]) * wt[s])
        block.index_add_(1, tok[s], z)
        at += m
    return {"g": g, "u": u, "block": block}
