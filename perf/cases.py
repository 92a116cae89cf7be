"""The work whose speed is measured: what a program that serves weight-only quantized models has
this package do, through its public entry points.

A case is one of five kinds:

``stack``    decoder layers of ``QuantLinear4`` modules (bound by ``prepare_fused``) over a decode
             step's rows; one HIP graph replay per pass, as a decode loop runs them.
``layer``    the same modules called one after the other without a graph.
``linear``   fused linears through the operators a module binds: the line-tiled layout where the
             weight fits it (``ops.line_tile``), the row layout otherwise.
``moe``      one MoE layer's routed experts (``ops.moe_experts_w4``).
``convert``  load-time quantization of a weight and its dequantization back (the packers that
             ``_quantize_int4_`` and its siblings run, the dequant behind ``_dequant``).

Weights are N(0, 0.02) quantized round-to-nearest (int4 asymmetric groups of 128, int8 symmetric per
row) or, for int2, uniform codes with fp16 scale ~U(0.005, 0.05) and zero ~U(0, 3) in groups of 64;
activations are bf16 N(0, 1). Shapes are ``K``x``N`` (in features x out features).
"""
from __future__ import annotations

import torch

LLAMA8B = "4096x6144,4096x4096,4096x28672,14336x4096"      # qkv, o, gate_up, down
BF16, FP16, F64 = torch.bfloat16, torch.float16, torch.float64
ALPHA, LIMIT = 1.702, 7.0                                  # gpt-oss's clamped GLU


def listed():
    return [
        # one decode row through one attention projection: the smallest call a program makes
        dict(name="w4 o_proj M=1", kind="linear", bits=4, M=1, shapes="4096x4096"),
        # single-stream decode of a Llama-3-8B-shaped model: eight layers' linears, one graph replay
        dict(name="w4 decode stack M=1", kind="stack", M=1, layers=8, shapes=LLAMA8B),
        # one layer of the same model over 32 rows: batched decode, a draft's verification
        dict(name="w4 layer M=32", kind="layer", M=32, layers=1, shapes=LLAMA8B),
        # a short prompt or a ragged chunk through the MLP
        dict(name="w4 mlp M=200", kind="linear", bits=4, M=200, shapes="4096x28672,14336x4096"),
        # the production prefill chunk, int4
        dict(name="w4 prefill M=2048", kind="linear", bits=4, M=2048, shapes="4096x14336,14336x4096"),
        # prefill chunk, int8 per-row weights
        dict(name="w8 prefill M=512", kind="linear", bits=8, M=512, shapes="4096x14336,14336x4096"),
        # an int8 lm_head (head_quant=int8 at Qwen2.5-7B) over a small decode batch
        dict(name="w8 lm_head M=4", kind="linear", bits=8, M=4, shapes="3584x152064"),
        # int2 at 70B shapes, a small decode batch
        dict(name="w2 decode M=8", kind="linear", bits=2, M=8, shapes="8192x28672,28672x8192"),
        # int2 prefill of a ragged prompt at 70B shapes
        dict(name="w2 prefill M=777", kind="linear", bits=2, M=777, shapes="8192x28672"),
        # gpt-oss-20b experts over a small decode batch (2880 columns: not whole groups)
        dict(name="moe gpt-oss T=4", kind="moe", act="gptoss", T=4, E=32, top=4, H=2880, I=2880),
        # OLMoE experts over a prompt
        dict(name="moe olmoe T=600", kind="moe", act="silu_glu", T=600, E=64, top=8, H=2048, I=1024),
        # quantize a gate_up weight at load and dequantize it (the naive path, the bind-time check)
        dict(name="convert w4 gate_up", kind="convert", bits=4, shapes="4096x28672"),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """One more case: the same kinds over rows 1 .. 2048 and weights 0.25 .. 117 M codes, odd row
    counts and ragged widths among them; no more work than the largest listed case."""
    kind = rng.choice(["linear", "linear", "linear", "linear", "linear", "moe", "moe", "convert", "layer", "stack"])
    if kind in ("stack", "layer"):
        layers = rng.randint(2, 8)
        return dict(kind=kind, M=_log_int(rng, 1, 16 if kind == "stack" else 64),
                    layers=layers if kind == "stack" else 1, shapes=LLAMA8B)
    if kind == "moe":
        act = rng.choice(["silu_glu", "silu_glu", "gptoss"])
        E = rng.choice([16, 32, 64, 128])
        H, I = 64 * _log_int(rng, 12, 48), 64 * _log_int(rng, 8, 46)
        while E * H * I > 300e6:
            E //= 2
        return dict(kind=kind, act=act, T=_log_int(rng, 1, 2048), E=E, top=rng.choice([2, 4, 8]), H=H, I=I)
    if rng.random() < 0.5:      # widths of the models this package is tested at
        K, N = rng.choice([(4096, 4096), (4096, 6144), (4096, 14336), (4096, 28672), (14336, 4096), (3584, 4608),
                           (3584, 18944), (2880, 5120), (4096, 2880), (2048, 2048), (8192, 8192)])
    else:
        K, N = 64 * _log_int(rng, 12, 224), _log_int(rng, 384, 16384)
        if rng.random() < 0.75:
            N = max(1, N // 64) * 64
    bits = rng.choice([4, 4, 4, 8, 2])
    if kind == "convert":
        return dict(kind=kind, bits=bits, shapes=f"{K}x{N}")
    M = min(_log_int(rng, 1, 2048), max(1, int(240e9 / (2 * K * N))))
    return dict(kind=kind, bits=bits, M=M, shapes=f"{K}x{N}")


# ---- inputs ---------------------------------------------------------------------------------------
def _shapes(case):
    return [tuple(int(v) for v in s.split("x")) for s in case["shapes"].split(",")]


def _gen(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 13)
    return g


def _normal(g, *shape, std=1.0, dtype=BF16):
    return (torch.randn(*shape, generator=g, device="cuda") * std).to(dtype)


def _nibbles(codes):
    return (codes[..., 0::2] | (codes[..., 1::2] << 4)).contiguous()


def _rtn4(g, N, K, G=128, W=None):
    """Row-layout int4: (qweight u8 [N, Kpad/2], scale, zero bf16 [N, ng])."""
    W = _normal(g, N, K, std=0.02) if W is None else W
    ng = -(-K // G)
    Wg = torch.nn.functional.pad(W, (0, ng * G - K)).float().reshape(N, ng, G)
    lo, hi = Wg.amin(2), Wg.amax(2)
    s = ((hi - lo) / 15.0).clamp(min=1e-8)
    z = torch.round(-lo / s).clamp(0, 15)
    q = torch.round(Wg / s.unsqueeze(2) + z.unsqueeze(2)).clamp(0, 15).to(torch.uint8)
    return _nibbles(q.reshape(N, ng * G)), s.to(BF16), z.to(BF16)


def _uniform2(g, N, K, G=64):
    """Row-layout int2: (qweight u8 [N, Kpad/4], scale, zero fp16 [N, ng]), zero codes past K."""
    ng = -(-K // G)
    q = torch.randint(0, 256, (N, ng * G // 4), generator=g, device="cuda", dtype=torch.uint8)
    s = (torch.rand(N, ng, generator=g, device="cuda") * 0.045 + 0.005).to(FP16)
    z = (torch.rand(N, ng, generator=g, device="cuda") * 3.0).to(FP16)
    return q, s, z


def _rows8(g, N, K):
    W = _normal(g, N, K, std=0.02, dtype=FP16)
    s = (W.abs().amax(1, keepdim=True) / 127.0).clamp(min=1e-8)
    return (W / s).round().clamp(-127, 127).to(torch.int8), s


def _weight(g, bits, N, K):
    return _rtn4(g, N, K) if bits == 4 else _uniform2(g, N, K) if bits == 2 else _rows8(g, N, K)


def _experts(g, case):
    """(gate_up, down) stacks [E, N, Kpad/2] with scale and zero, the routing and the biases."""
    E, H, I, T = case["E"], case["H"], case["I"], case["T"]
    gu = [torch.stack(p) for p in zip(*[_rtn4(g, 2 * I, H) for _ in range(E)])]
    dn = [torch.stack(p) for p in zip(*[_rtn4(g, H, I) for _ in range(E)])]
    x = _normal(g, T, H)
    p = torch.softmax(torch.randn(T, E, generator=g, device="cuda"), dim=-1)
    top, idx = torch.topk(p, case["top"], dim=-1)
    w = (top / top.sum(-1, keepdim=True)).to(BF16)
    bias = (_normal(g, E, 2 * I, std=0.02), _normal(g, E, H, std=0.02)) if case["act"] == "gptoss" else (None, None)
    return gu, dn, x, idx, w, bias


def _module_set(g, case):
    """Row-layout weights and activations of ``layers`` layers' linears, in call order."""
    return [(*_rtn4(g, N, K), _normal(g, case["M"], K)) for _ in range(case["layers"]) for K, N in _shapes(case)]


def _tiles(bits, N, K):
    """Whether a module would bind the weight line-tiled: whole 16-row tiles and 128-byte line-steps."""
    return N % 16 == 0 and K % {4: 256, 2: 512, 8: 128}[bits] == 0


# ---- the measured path ----------------------------------------------------------------------------
def prepare(case, seed):
    from infinitemodel_amd import ops, worker_quant as wq
    g, kind = _gen(case, seed), case["kind"]
    if kind in ("stack", "layer"):
        calls = []
        for (K, N), (q, s, z, x) in zip(_shapes(case) * case["layers"], _module_set(g, case)):
            mod = wq._quant4_linear_cls()(q, s, z, None, K, 128)
            mod.prepare_fused()
            calls.append((mod, x))
        if kind == "layer":
            return dict(kind=kind, calls=calls)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _call_all(calls)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            ys = _call_all(calls)
        return dict(kind=kind, graph=graph, ys=ys, calls=calls)
    if kind == "linear":
        bits, calls = case["bits"], []
        for K, N in _shapes(case):
            w = _weight(g, bits, N, K)
            x = _normal(g, case["M"], K)
            tiled = _tiles(bits, N, K)
            q = ops.line_tile(w[0]) if tiled else w[0]
            if bits == 8:
                calls.append((ops.linear_w8_tiled if tiled else ops.linear_w8, (x, q, w[1])))
            else:
                op = {4: (ops.linear_w4, ops.linear_w4_tiled), 2: (ops.linear_w2, ops.linear_w2_tiled)}[bits][tiled]
                calls.append((op, (x, q, 128 if bits == 4 else 64, (w[1], w[2]))))
        return dict(kind=kind, calls=calls)
    if kind == "moe":
        gu, dn, x, idx, w, bias = _experts(g, case)
        holder = wq._packed4_3d_cls()
        gu = (*holder(*gu, case["H"], 128)._kernel_tensors(), case["H"])
        dn = (*holder(*dn, case["I"], 128)._kernel_tensors(), case["I"])
        return dict(kind=kind, args=(x, idx, w, gu, dn, 128), act=case["act"], bias=bias)
    (K, N), = _shapes(case)
    return dict(kind=kind, bits=case["bits"], W=_normal(g, N, K, std=0.02))


def _call_all(calls):
    with torch.no_grad():
        return [mod(x) for mod, x in calls]


def run(state):
    from infinitemodel_amd import ops, shard_compile
    kind = state["kind"]
    if kind == "stack":
        state["graph"].replay()
        return state["ys"]
    if kind == "layer":
        return _call_all(state["calls"])
    if kind == "linear":
        return [op(*args) for op, args in state["calls"]]
    if kind == "moe":
        return ops.moe_experts_w4(*state["args"], act=state["act"], gu_bias=state["bias"][0],
                                  dn_bias=state["bias"][1], alpha=ALPHA, limit=LIMIT, check_ids=False)
    W, bits = state["W"], state["bits"]
    if bits == 8:
        q, s = shard_compile.pack_linear_int8(W)
        return dict(q=q, s=s, w=ops.dequant_w8(q, s, W.dtype))
    if bits == 4:
        q, s, z, in_f = shard_compile.pack_linear_int4(W)
        return dict(q=q, s=s, z=z, w=ops.dequant_w4(q, s, z, in_f, 128, W.dtype))
    q, s, z, in_f = shard_compile.pack_linear_int2(W)
    return dict(q=q, s=s, z=z, w=ops.dequant_w2(q, s, z, in_f, 64, W.dtype))


# ---- what a pass cannot do without ----------------------------------------------------------------
def _weight_bytes(bits, N, K):
    if bits == 8:
        return N * K + 2 * N
    G = 128 if bits == 4 else 64
    ng = -(-K // G)
    return N * ng * (G * bits // 8 + 4)


def work(case):
    kind = case["kind"]
    if kind in ("stack", "layer", "linear"):
        M, L, bits = case["M"], case.get("layers", 1), case.get("bits", 4)
        return dict(bytes=L * sum(_weight_bytes(bits, N, K) + 2 * M * (K + N) for K, N in _shapes(case)),
                    flops=L * sum(2 * M * N * K for K, N in _shapes(case)))
    if kind == "moe":
        E, H, I, T = case["E"], case["H"], case["I"], case["T"]
        rows = T * case["top"]
        hit = E * (1 - (1 - case["top"] / E) ** T)       # experts that some row is expected to reach
        per = _weight_bytes(4, 2 * I, H) + _weight_bytes(4, H, I)
        if case["act"] == "gptoss":
            per += 2 * (2 * I + H)
        return dict(bytes=int(hit * per) + 4 * T * H + 10 * rows, flops=rows * 6 * H * I)
    (K, N), = _shapes(case)
    return dict(bytes=4 * N * K + 2 * _weight_bytes(case["bits"], N, K), flops=4 * N * K)


def tolerance(case):
    """Linears: bf16 results with fp32 sums measured 1.6e-3 (unrounded weights) to 2.2e-3 (weights
    rounded to bf16 once) from the 64-bit product, 3.6e-3 for int2's non-integer zeros; the experts,
    which round their intermediate rows too, 2.9e-3. Packers and dequant round as the reference does,
    bit for bit."""
    return "exact" if case["kind"] == "convert" else {"rel": 1e-2}


# ---- the same in 64 bits, in plain torch ----------------------------------------------------------
def _codes(q, bits):
    return torch.stack([(q >> (bits * i)) & ((1 << bits) - 1) for i in range(8 // bits)], dim=-1).flatten(-2)


def _dense(w, bits, K):
    if bits == 8:
        return w[0].to(F64) * w[1].to(F64)
    q, s, z = w
    c = _codes(q, bits).to(F64)
    c = c.reshape(*s.shape, -1)
    return ((c - z.to(F64).unsqueeze(-1)) * s.to(F64).unsqueeze(-1)).flatten(-2)[..., :K]


def exact(case, seed):
    g, kind = _gen(case, seed), case["kind"]
    if kind in ("stack", "layer"):
        return [x.to(F64) @ _dense((q, s, z), 4, x.shape[1]).t() for q, s, z, x in _module_set(g, case)]
    if kind == "linear":
        ys = []
        for K, N in _shapes(case):
            w = _weight(g, case["bits"], N, K)
            x = _normal(g, case["M"], K)
            ys.append(x.to(F64) @ _dense(w, case["bits"], K).t())
        return ys
    if kind == "moe":
        gu, dn, x, idx, w, (gb, db) = _experts(g, case)
        H, I = case["H"], case["I"]
        out = torch.zeros(case["T"], H, dtype=F64, device="cuda")
        for e in range(case["E"]):
            t, j = torch.nonzero(idx == e, as_tuple=True)
            if t.numel() == 0:
                continue
            u = x[t].to(F64) @ _dense([p[e] for p in gu], 4, H).t()
            if case["act"] == "gptoss":
                u = u + gb[e].to(F64)
                gate, up = u[:, 0::2].clamp(max=LIMIT), u[:, 1::2].clamp(-LIMIT, LIMIT)
                h = (up + 1) * gate * torch.sigmoid(ALPHA * gate)
            else:
                h = torch.nn.functional.silu(u[:, :I]) * u[:, I:]
            y = h @ _dense([p[e] for p in dn], 4, I).t()
            if db is not None:
                y = y + db[e].to(F64)
            out.index_add_(0, t, y * w[t, j].to(F64).unsqueeze(1))
        return out
    (K, N), = _shapes(case)
    W = _normal(g, N, K, std=0.02).to(F64)
    if case["bits"] == 8:
        return dict(q=None, s=(W.abs().amax(1, keepdim=True) / 127).clamp(min=1e-8), w=None)
    G, top = (128, 15) if case["bits"] == 4 else (64, 3)
    ng = -(-K // G)
    Wg = torch.nn.functional.pad(W, (0, ng * G - K)).reshape(N, ng, G)
    lo, hi = Wg.amin(2), Wg.amax(2)
    s = ((hi - lo) / top).clamp(min=1e-8)
    z = torch.round(-lo / s).clamp(0, top)
    return dict(q=None, s=s, z=z, w=None)
