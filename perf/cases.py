"""Performance cases of the quantized matmul path: what a program built on this package has it do.

A case is one pass over the projections of a number of decoder layers through the package's
public calls: ``q_gemm_dequant_grouped`` for q/k/v, ``Linear`` for the output projection and
the vocabulary head, ``MLP`` for gate/up/down.  Decode steps (few rows, many launches) are
captured once per model in a graph and replayed, as a decode loop does; prompts and single
calls run eagerly.  Weights are GGUF blocks made on the device from the seed, packed before
the pass as a program packs them at load time; every layer has its own, so a decode pass
streams them from memory.  Model sizes are those of the tests and the benchmark (TinyLlama,
Llama-3-8B, Llama-3-70B) or generic.

``exact`` recomputes a pass in float64 from the same GGUF bytes with plain torch.
"""
import math

import torch

import mlxr_amd as mx

# (elements, bytes) of a GGUF block
BLOCK = {"Q4_0": (32, 18), "Q4_1": (32, 20), "Q8_0": (32, 34), "Q4_K": (256, 144), "Q5_K": (256, 176),
         "Q6_K": (256, 210)}
DTYPE = {"bf16": torch.bfloat16, "f16": torch.float16}
# standard deviation the generated weights are centred on
SIGMA = 0.02


def _case(name, op, qt, qt2, rows, hidden, inter, kv, layers, dtype="bf16", bias=False, graph=False):
    """op: "layer" (q/k/v, o and the MLP), "mlp", "linear" (hidden -> inter).  qt2: the type of
    v and down, as the mixed K-quant files have it.  rows: M, tokens of the pass."""
    return {"name": name, "op": op, "qt": qt, "qt2": qt2, "rows": rows, "hidden": hidden, "inter": inter, "kv": kv,
            "layers": layers, "dtype": dtype, "bias": bias, "graph": graph}


def listed():
    return [
        # the smallest call: one TinyLlama projection for one token, called by itself
        _case("tinyllama_q_m1", "linear", "Q8_0", "Q8_0", 1, 2048, 2048, 0, 1, dtype="f16"),
        # one sequence being generated: a token through eight Llama-3-8B layers
        _case("8b_decode_m1", "layer", "Q4_K", "Q4_K", 1, 4096, 14336, 1024, 8, graph=True),
        # a small server's decode batch
        _case("8b_decode_m8", "layer", "Q4_K", "Q4_K", 8, 4096, 14336, 1024, 8, graph=True),
        # a ragged decode batch on a large model in the usual mixed file (Q6_K v and down)
        _case("70b_decode_m13", "layer", "Q4_K", "Q6_K", 13, 8192, 28672, 1024, 2, graph=True),
        # the MLPs of a model whose file is plain 4-bit, a decode batch of 24
        _case("mlp_q4_0_m24", "mlp", "Q4_0", "Q4_0", 24, 4096, 11008, 0, 8, graph=True),
        # a full decode batch (or the drafts of a speculative step)
        _case("8b_decode_m64", "layer", "Q4_K", "Q4_K", 64, 4096, 14336, 1024, 8, graph=True),
        # the vocabulary head over a decode batch (Q6_K in the usual files)
        _case("lm_head_q6k_m6", "linear", "Q6_K", "Q6_K", 6, 4096, 128256, 0, 1),
        # a short prompt of odd length, a mixed five-bit file
        _case("8b_prompt_m100_q5k", "layer", "Q5_K", "Q6_K", 100, 4096, 14336, 1024, 1),
        # a prompt on a small eight-bit model with q/k/v biases, fp16 activations
        _case("small_prompt_m333_q8", "layer", "Q8_0", "Q8_0", 333, 2048, 5632, 256, 2, dtype="f16", bias=True),
        # a prompt chunk on the large model
        _case("70b_prompt_m256", "layer", "Q4_K", "Q6_K", 256, 8192, 28672, 1024, 1),
        # prompts on the 8B model: a chunk of 512 and the longest pass
        _case("8b_prompt_m512", "layer", "Q4_K", "Q4_K", 512, 4096, 14336, 1024, 1),
        _case("8b_prompt_m2048", "layer", "Q4_K", "Q4_K", 2048, 4096, 14336, 1024, 1),
    ]


def draw(rng):
    largest = max(work(c)["flops"] for c in listed())
    while True:
        op = rng.choice(["layer", "layer", "mlp", "linear"])
        qt = rng.choice(["Q4_K", "Q4_K", "Q4_K", "Q5_K", "Q6_K", "Q8_0", "Q4_0", "Q4_1"])
        qt2 = rng.choice([qt, "Q6_K"]) if qt in ("Q4_K", "Q5_K") else qt
        unit = BLOCK[qt][0]
        rows = int(round(math.exp(rng.uniform(0.0, math.log(2048)))))
        hidden = unit * max(1, int(round(math.exp(rng.uniform(math.log(1024), math.log(8192))) / unit)))
        if op == "linear" and rng.random() < 0.3:
            inter = rng.randrange(32000, 128257)  # a vocabulary
        elif op == "linear":
            inter = int(round(math.exp(rng.uniform(math.log(1000), math.log(16384)))))
        else:
            inter = unit * int(round(hidden * rng.uniform(2.6, 3.6) / unit))
        kv = 64 * max(1, hidden // 64 // rng.choice([1, 4, 8]))
        dtype = "bf16" if rng.random() < 0.75 else "f16"
        graph = rows <= 64 and rng.random() < 0.8
        c = _case("", op, qt, qt2, rows, hidden, inter, kv if op == "layer" else 0, 1, dtype=dtype,
                  bias=op != "mlp" and rng.random() < 0.25, graph=graph)
        del c["name"]
        if graph:  # as many layers as leave the caches behind, at most twelve
            c["layers"] = max(1, min(12, int(1 + 4e8 // sum(_nbytes(q, n, k) for q, n, k in _shapes(c)))))
        w = work(c)
        if w["flops"] <= largest and w["bytes"] <= 1.3e9:
            return c


# ------------------------------------------------------------------------- the weights

def _nbytes(qt, n, k):
    e, b = BLOCK[qt]
    return n * (k // e) * b


def _shapes(c):
    """(type, N, K) of the weights of one layer, in the order of their use."""
    h, i, kv = c["hidden"], c["inter"], c["kv"]
    if c["op"] == "linear":
        return [(c["qt"], i, h)]
    mlp = [(c["qt"], i, h), (c["qt"], i, h), (c["qt2"], h, i)]
    if c["op"] == "mlp":
        return mlp
    return [(c["qt"], h, h), (c["qt"], kv, h), (c["qt2"], kv, h), (c["qt"], h, h)] + mlp


def _gen(seed, *ids):
    s = int(seed)
    for i in ids:
        s = (s * 1000003 + int(i) + 12345) % (1 << 62)
    return torch.Generator(device="cuda").manual_seed(s)


def _f16_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(v.shape[0], 2)


def _blocks(qt, n, k, g):
    """GGUF blocks [n * k / elements, bytes] of weights centred on zero with deviation SIGMA."""
    e, nb = BLOCK[qt]
    rows = n * (k // e)
    w = torch.randint(0, 256, (rows, nb), dtype=torch.uint8, device="cuda", generator=g)
    spread = 0.6 + 0.8 * torch.rand(rows, device="cuda", generator=g)  # block scales differ within a tensor
    if qt == "Q8_0":
        w[:, 0:2] = _f16_bytes(spread * (SIGMA / 73.9))
    elif qt in ("Q4_0", "Q4_1"):
        d = spread * (SIGMA / 4.61)
        w[:, 0:2] = _f16_bytes(d)
        if qt == "Q4_1":
            w[:, 2:4] = _f16_bytes(-7.5 * d)
    elif qt in ("Q4_K", "Q5_K"):
        top = 7.5 if qt == "Q4_K" else 15.5
        d = spread * (SIGMA / (47.5 * (4.61 if qt == "Q4_K" else 9.23)))
        w[:, 0:2] = _f16_bytes(d)
        w[:, 2:4] = _f16_bytes(top * d)
        # sub-block scales 32..63, mins equal to them: each sub-block is centred on zero
        sc = 32 + (w[:, 4:12] & 31)
        lo, hi = sc[:, :4], sc[:, 4:]
        w[:, 4:8] = lo | ((hi >> 4) << 6)
        w[:, 8:12] = lo | ((hi >> 4) << 6)
        w[:, 12:16] = (hi & 15) | ((hi & 15) << 4)
    else:  # Q6_K: int8 scales over their range, either sign
        w[:, 208:210] = _f16_bytes(spread * (SIGMA / (18.5 * 37.0)))
        w[:, 192:208] = ((w[:, 192:208] & 63).to(torch.int16) - 32).to(torch.int8).view(torch.uint8)
    return w


def _half(w, at):
    return w[:, at:at + 2].contiguous().view(torch.float16).to(torch.float64)


def _dense(qt, w, n, k):
    """The float64 weights [n, k] of GGUF blocks (the formats' definitions)."""
    d = _half(w, 208 if qt == "Q6_K" else 0)
    if qt == "Q8_0":
        return (d * w[:, 2:].contiguous().view(torch.int8)).reshape(n, k)
    if qt in ("Q4_0", "Q4_1"):
        q = w[:, 2 if qt == "Q4_0" else 4:]
        q = torch.cat([q & 15, q >> 4], dim=1).to(torch.float64)
        return (d * (q - 8) if qt == "Q4_0" else d * q + _half(w, 2)).reshape(n, k)
    r = w.shape[0]
    if qt in ("Q4_K", "Q5_K"):
        b = w[:, 4:16]
        sc = torch.cat([b[:, 0:4] & 63, (b[:, 8:12] & 15) | ((b[:, 0:4] >> 6) << 4)], dim=1).to(torch.float64)
        mn = torch.cat([b[:, 4:8] & 63, (b[:, 8:12] >> 4) | ((b[:, 4:8] >> 6) << 4)], dim=1).to(torch.float64)
        qs = w[:, 16 if qt == "Q4_K" else 48:].reshape(r, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], dim=2).reshape(r, 8, 32)
        if qt == "Q5_K":
            at = torch.arange(8, device=w.device, dtype=torch.uint8).reshape(1, 8, 1)
            q = q | (((w[:, 16:48].reshape(r, 1, 32) >> at) & 1) << 4)
        q = q.to(torch.float64)
        return ((d * sc).unsqueeze(2) * q - (_half(w, 2) * mn).unsqueeze(2)).reshape(n, k)
    ql, qh = w[:, 0:128].reshape(r, 2, 2, 32), w[:, 128:192].reshape(r, 2, 1, 32)
    lo = torch.cat([ql & 15, ql >> 4], dim=2)
    hi = torch.cat([(qh >> s) & 3 for s in (0, 2, 4, 6)], dim=2) << 4
    q = (lo | hi).to(torch.float64).reshape(r, 16, 16) - 32
    sc = w[:, 192:208].contiguous().view(torch.int8).to(torch.float64)
    return ((d * sc).unsqueeze(2) * q).reshape(n, k)


# -------------------------------------------------------------------------- the inputs

def _act(c, seed, layer, which, width):
    """Activations after a norm (or a gated product): N(0, 1) in the compute type."""
    g = _gen(seed, 1, layer, which)
    return torch.randn(c["rows"], width, device="cuda", generator=g).to(DTYPE[c["dtype"]])


def _bias(c, seed, layer, which, n):
    if not c["bias"]:
        return None
    return (0.5 * torch.randn(n, device="cuda", generator=_gen(seed, 2, layer, which))).to(DTYPE[c["dtype"]])


def _weights(c, seed, layer):
    return [(qt, n, k, _blocks(qt, n, k, _gen(seed, 3, layer, j))) for j, (qt, n, k) in enumerate(_shapes(c))]


def _linear(qt, n, k, blocks, bias=None):
    lin = mx.Linear(k, n, bias=bias is not None)
    lin.load_weight(mx.pack_weights(blocks.reshape(-1), n, k, mx.QuantType[qt]))
    if bias is not None:
        lin.set_bias(bias)
    return lin


def _mlp(c, ws):
    m = mx.MLP(c["hidden"], c["inter"])
    for lin, (qt, n, k, b) in zip((m.gate_proj, m.up_proj, m.down_proj), ws):
        lin.load_weight(mx.pack_weights(b.reshape(-1), n, k, mx.QuantType[qt]))
    return m


def prepare(case, seed):
    c, layers = case, []
    for i in range(c["layers"]):
        ws = _weights(c, seed, i)
        s = {"x": _act(c, seed, i, 0, c["hidden"])}
        if c["op"] == "linear":
            qt, n, k, b = ws[0]
            s["linear"] = _linear(qt, n, k, b, _bias(c, seed, i, 0, n))
        else:
            s["mlp"] = _mlp(c, ws[-3:])
        if c["op"] == "layer":
            s["qkv"] = [mx.pack_weights(b.reshape(-1), n, k, mx.QuantType[qt]) for qt, n, k, b in ws[:3]]
            s["biases"] = [_bias(c, seed, i, j, ws[j][1]) for j in range(3)]
            qt, n, k, b = ws[3]
            s["o"] = _linear(qt, n, k, b)
            s["a"] = _act(c, seed, i, 1, c["hidden"])  # what attention hands to o
            s["m"] = _act(c, seed, i, 2, c["hidden"])  # what the second norm hands to the MLP
        layers.append(s)
    state = {"layers": layers}
    if c["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):  # once before the capture: the layers' workspaces
            _pass(layers)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            state["outputs"] = _pass(layers)
        state["graph"] = graph
    return state


def _pass(layers):
    out = []
    for s in layers:
        if "linear" in s:
            out.append([s["linear"](s["x"])])
            continue
        if "qkv" not in s:
            out.append([s["mlp"](s["x"])])
            continue
        q, k, v = mx.q_gemm_dequant_grouped(s["x"], s["qkv"], biases=s["biases"])
        out.append([q, k, v, s["o"](s["a"]), s["mlp"](s["m"])])
    return out


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["outputs"]
    return _pass(state["layers"])


# ---------------------------------------------------------------------- what is expected

def work(case):
    c = case
    nbytes = flops = 0
    for qt, n, k in _shapes(c):
        nbytes += _nbytes(qt, n, k)
        flops += 2 * c["rows"] * n * k
    h, i, kv, m = c["hidden"], c["inter"], c["kv"], c["rows"]
    elems = m * (h + i) if c["op"] == "linear" else m * 2 * h  # the MLP's input and output
    if c["op"] == "layer":
        elems += m * (h + h + 2 * kv) + m * 2 * h
    return {"bytes": c["layers"] * (nbytes + 2 * elems), "flops": c["layers"] * flops}


def tolerance(case):
    # Outputs are bf16 or fp16 (half a unit: 2^-9, 2^-12 of the value) of products over weights
    # that the matrix instructions take in the same type; the MLP's intermediate is rounded too.
    # Measured against exact(): bf16 2.4e-3 for one product and 3.8e-3 for an MLP, fp16 2.9e-4
    # and 4.7e-4.
    return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 1.6e-3}


def exact(case, seed):
    c, out = case, []
    for i in range(c["layers"]):
        ws = _weights(c, seed, i)

        def mul(x, j):
            qt, n, k, b = ws[j]
            return x.to(torch.float64) @ _dense(qt, b, n, k).T

        def mlp(x, j):
            g, u = mul(x, j), mul(x, j + 1)
            return mul(g * torch.sigmoid(g) * u, j + 2)

        def with_bias(y, j):
            b = _bias(c, seed, i, j, y.shape[1])
            return y if b is None else y + b.to(torch.float64)

        x = _act(c, seed, i, 0, c["hidden"])
        if c["op"] == "linear":
            out.append([with_bias(mul(x, 0), 0)])
        elif c["op"] == "mlp":
            out.append([mlp(x, 0)])
        else:
            a, m = _act(c, seed, i, 1, c["hidden"]), _act(c, seed, i, 2, c["hidden"])
            out.append([with_bias(mul(x, j), j) for j in range(3)] + [mul(a, 3), mlp(m, 4)])
    return out
