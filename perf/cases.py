"""The calls that a program running quantized models makes through libhipq, as measurable cases.

A case is one of four kinds of call, each through the Python binding of the C ABI:

* ``matmul``: ``hipq.matmul_q`` of F32 activations (M, K) and a GGUF weight (N, K);
* ``mlp``: ``hipq.mlp_q``, the gated MLP block (H -> I -> H) of a decoder layer;
* ``int4``: ``hipq.int4_matmul`` of F32 / BF16 / F16 activations and a GPTQ / AWQ style weight;
* ``moe``: ``hipq.moe_block_q``, routing and experts of a sparse decoder layer.

``layers`` is how many layers, each with weights and activations of its own, one pass goes
through.  ``graph`` says that the program replays the pass from a captured graph, as decode loops
do; the others are plain calls.  Workspaces are sized once, outputs are allocated once.

Weights look like a checkpoint's: about 0.02 standard deviation, roughly centred, scales spread
over a factor of a few.  Activations are N(0, 1), as behind a norm.
"""
import math

import torch

from light_amd import hipq

DTYPES = {"Q4_0": hipq.Q4_0, "Q5_0": hipq.Q5_0, "Q8_0": hipq.Q8_0, "Q4_K": hipq.Q4_K, "Q5_K": hipq.Q5_K,
          "Q6_K": hipq.Q6_K}
XTYPES = {"F32": torch.float32, "BF16": torch.bfloat16, "F16": torch.float16}


def listed():
    return [
        # One token through the square attention projections of eight layers: the smallest calls,
        # where launch and start-up latency count as much as bytes.
        dict(name="decode_attn_q8_0", kind="matmul", dt="Q8_0", M=1, N=4096, K=4096, layers=8, graph=True),
        # One token through a dense layer's MLP, called directly.
        dict(name="decode_mlp_q4_k", kind="mlp", dt="Q4_K", M=1, H=4096, I=14336, layers=1, graph=False),
        # A small batch of decoding sequences, not a power of two, through the same MLP.
        dict(name="decode_mlp_q4_k_b6", kind="mlp", dt="Q4_K", M=6, H=4096, I=14336, layers=1, graph=False),
        # One token's logits: the largest weight a decode step reads, in its GGUF bytes.
        dict(name="decode_head_q6_k", kind="matmul", dt="Q6_K", M=1, N=128256, K=4096, layers=1, graph=False),
        # Three sequences decoding on a GPTQ / AWQ checkpoint: the long rows of a down projection.
        dict(name="decode_int4_b3", kind="int4", x="BF16", M=3, N=3584, K=18944, G=128, layers=4, graph=True),
        # A serving batch of forty sequences, or a speculative step: between decode and prefill.
        dict(name="batch_q4_k_m40", kind="matmul", dt="Q4_K", M=40, N=14336, K=4096, layers=1, graph=False),
        # The same on 4-bit groups with half-precision activations.
        dict(name="batch_int4_m64", kind="int4", x="F16", M=64, N=18944, K=3584, G=128, layers=1, graph=False),
        # A 512-token prompt (or chunk of one) through a dense layer's MLP.
        dict(name="prefill_mlp_q4_k", kind="mlp", dt="Q4_K", M=512, H=4096, I=14336, layers=1, graph=False),
        # A prompt of no round length on another GGUF format, long rows.
        dict(name="prefill_q6_k_m777", kind="matmul", dt="Q6_K", M=777, N=4096, K=14336, layers=1, graph=False),
        # A long prompt on 4-bit groups: the largest call.
        dict(name="prefill_int4_m2048", kind="int4", x="BF16", M=2048, N=18944, K=3584, G=128, layers=1, graph=False),
        # Five sequences decoding through the sparse layers of a mixture-of-experts model.
        dict(name="decode_moe_t5", kind="moe", dt="Q4_K", T=5, E=128, topk=8, H=2048, I=768, layers=4, graph=True),
        # A prompt of 500 tokens through one sparse layer.
        dict(name="prefill_moe_t500", kind="moe", dt="Q4_K", T=500, E=128, topk=8, H=2048, I=768, layers=1,
             graph=False),
    ]


# A drawn call stays below these: the largest listed one's operations, and weights of a head.
MAX_FLOPS = 2.0 * 2048 * 18944 * 3584
MAX_WEIGHTS = 128256 * 4096


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _rows(rng):
    """Rows of x: a token, a decode batch, a serving batch, a prompt."""
    return rng.choice([1, _log_int(rng, 2, 8), _log_int(rng, 9, 64), _log_int(rng, 65, 2048)])


def _layers(rng, rows):
    """Decode loops replay several layers, larger passes are called one by one."""
    graph = rows <= 8 and rng.random() < 0.7
    return dict(layers=rng.randint(4, 8) if graph else 1, graph=graph)


def draw(rng):
    while True:
        kind = rng.choice(["matmul", "matmul", "mlp", "int4", "int4", "moe"])
        if kind == "matmul":
            M = _rows(rng)
            N = _log_int(rng, 1024, 32768)
            N = N if rng.random() < 0.25 else (N + 127) // 128 * 128
            K = 256 * _log_int(rng, 4, 64)
            c = dict(kind=kind, dt=rng.choice(["Q4_K", "Q4_K", "Q5_K", "Q6_K", "Q8_0", "Q4_0", "Q5_0"]), M=M, N=N, K=K)
            flops, weights = 2.0 * M * N * K, N * K
        elif kind == "mlp":
            M = _rows(rng)
            H, I = 256 * _log_int(rng, 6, 32), 256 * _log_int(rng, 16, 112)
            c = dict(kind=kind, dt=rng.choice(["Q4_K", "Q4_K", "Q5_K"]), M=M, H=H, I=I)
            flops, weights = 6.0 * M * H * I, 3 * H * I
        elif kind == "int4":
            M = _rows(rng)
            N = 8 * _log_int(rng, 128, 4096)
            G = rng.choice([64, 128, 128])
            K = 128 * _log_int(rng, 8, 160)
            c = dict(kind=kind, x=rng.choice(["F32", "BF16", "F16"]), M=M, N=N, K=K, G=G)
            flops, weights = 2.0 * M * N * K, N * K
        else:
            M = rng.choice([1, _log_int(rng, 2, 8), _log_int(rng, 9, 64), _log_int(rng, 65, 1024)])
            E, topk = rng.choice([(8, 2), (64, 6), (64, 8), (128, 8)])
            H, I = 256 * _log_int(rng, 4, 16), 256 * _log_int(rng, 2, 14 if E > 8 else 40)
            c = dict(kind=kind, dt=rng.choice(["Q4_K", "Q4_K", "Q5_K"]), T=M, E=E, topk=topk, H=H, I=I)
            flops, weights = 6.0 * M * topk * H * I, 3 * E * H * I
        if kind == "moe" and c["dt"] == "Q5_K" and M > 64:
            continue  # prompts through experts: Q4_K
        c.update(_layers(rng, M))
        if flops * c["layers"] <= MAX_FLOPS and weights * c["layers"] <= 2 * MAX_WEIGHTS:
            return c


# ---- inputs ------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _f16_bytes(v):
    return v.to(torch.float16).view(torch.uint8).view(*v.shape, 2)


def _scales(n, g, per):
    """Positive scales (n,): `per` times a spread of about a factor of three."""
    return per * (0.4 + 1.2 * torch.rand(n, device="cuda", generator=g))


def _bytes(nb, size, g):
    return torch.randint(0, 256, (nb, size), dtype=torch.uint8, device="cuda", generator=g)


def _gguf(dt, n, g):
    """The bytes of n weights in format dt: random quants under scales that give about 0.02 rms."""
    if dt in ("Q8_0", "Q4_0", "Q5_0"):
        size, rms = {"Q8_0": (34, 73.9), "Q4_0": (18, 4.6), "Q5_0": (22, 9.2)}[dt]
        b = _bytes(n // 32, size, g)
        b[:, 0:2] = _f16_bytes(_scales(n // 32, g, 0.02 / rms))
        if dt == "Q8_0":  # quants of a block lie in [-127, 127]
            q = b[:, 2:].view(torch.int8)
            q.copy_(torch.where(q == -128, torch.full_like(q, -127), q))
        return b.reshape(-1)
    nb = n // 256
    if dt == "Q6_K":
        b = _bytes(nb, 210, g)
        sc = torch.randint(16, 65, (nb, 16), dtype=torch.int32, device="cuda", generator=g)
        sign = 2 * torch.randint(0, 2, (nb, 16), dtype=torch.int32, device="cuda", generator=g) - 1
        b[:, 192:208] = (sc * sign).to(torch.int8).view(torch.uint8)
        b[:, 208:210] = _f16_bytes(_scales(nb, g, 0.02 / (40 * 18.5)))
        return b
    q_max = 15 if dt == "Q4_K" else 31
    b = _bytes(nb, 144 if dt == "Q4_K" else 176, g)
    d = _scales(nb, g, 0.02 / (43 * 0.3 * q_max))
    b[:, 0:2] = _f16_bytes(d)
    b[:, 2:4] = _f16_bytes(d * (q_max / 2))
    # 6-bit scales and mins of eight sub-blocks; a min near its scale centres the sub-block.
    sc = torch.randint(24, 64, (nb, 8), dtype=torch.int32, device="cuda", generator=g)
    mn = (sc + torch.randint(-4, 5, (nb, 8), dtype=torch.int32, device="cuda", generator=g)).clamp(0, 63)
    b[:, 4:8] = (sc[:, :4] | ((sc[:, 4:] >> 4) << 6)).to(torch.uint8)
    b[:, 8:12] = (mn[:, :4] | ((mn[:, 4:] >> 4) << 6)).to(torch.uint8)
    b[:, 12:16] = ((sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)).to(torch.uint8)
    return b


def _int4(N, K, G, g):
    codes = torch.randint(-2 ** 31, 2 ** 31, (N, K // 8), dtype=torch.int64, device="cuda", generator=g).to(torch.int32)
    scales = _scales(N * (K // G), g, 0.02 / 4.8).to(torch.float16).float().reshape(N, K // G)
    zeros = torch.randint(6, 11, (N, K // G), device="cuda", generator=g).float()
    return codes, scales, zeros


def _x(M, K, g, dtype=torch.float32):
    return torch.randn((M, K), device="cuda", generator=g).to(dtype)


def _inputs(case, seed):
    """Per layer: the activations and weights of the call."""
    g, kind, out = _gen(seed), case["kind"], []
    for _ in range(case["layers"]):
        if kind == "matmul":
            out.append(dict(x=_x(case["M"], case["K"], g), w=_gguf(case["dt"], case["N"] * case["K"], g)))
        elif kind == "mlp":
            n = case["H"] * case["I"]
            out.append(dict(x=_x(case["M"], case["H"], g), wg=_gguf(case["dt"], n, g), wu=_gguf(case["dt"], n, g),
                            wd=_gguf(case["dt"], n, g)))
        elif kind == "int4":
            codes, s, z = _int4(case["N"], case["K"], case["G"], g)
            out.append(dict(x=_x(case["M"], case["K"], g, XTYPES[case["x"]]), codes=codes, s=s, z=z))
        else:
            n = case["E"] * case["I"] * case["H"]
            logits = torch.randn((case["T"], case["E"]), device="cuda", generator=g)
            out.append(dict(probs=torch.softmax(logits, dim=1), x=_x(case["T"], case["H"], g),
                            wgu=_gguf(case["dt"], 2 * n, g), wd=_gguf(case["dt"], n, g)))
    return out


def _workspace_bytes(case):
    L, kind = hipq.lib(), case["kind"]
    if kind == "matmul":
        return L.hq_matmul_q_ws_bytes(case["M"], case["N"], case["K"], DTYPES[case["dt"]])
    if kind == "mlp":
        return L.hq_mlp_q_ws_bytes(case["M"], case["H"], case["I"], DTYPES[case["dt"]])
    if kind == "int4":
        code = {"F32": hipq.F32, "BF16": hipq.BF16, "F16": hipq.F16}[case["x"]]
        return L.hq_int4_matmul_ws_bytes(case["M"], case["N"], case["K"], case["G"], code)
    return L.hq_moe_block_q_ws_bytes(case["T"], case["topk"], case["E"], case["H"], case["I"], DTYPES[case["dt"]])


def _call(case, layer, ws):
    kind = case["kind"]
    if kind == "matmul":
        return hipq.matmul_q(layer["x"], layer["w"], case["N"], case["K"], DTYPES[case["dt"]], out=layer["out"], ws=ws)
    if kind == "mlp":
        return hipq.mlp_q(layer["x"], layer["wg"], layer["wu"], layer["wd"], case["H"], case["I"], DTYPES[case["dt"]],
                          out=layer["out"], ws=ws)
    if kind == "int4":
        return hipq.int4_matmul(layer["x"], layer["codes"], layer["s"], layer["z"], case["G"], out=layer["out"], ws=ws)
    # (y, topk_ids, weights, sorted_pairs, sorted_expts, h)
    return hipq.moe_block_q(layer["probs"], layer["x"], layer["wgu"], layer["wd"], case["E"], case["H"], case["I"],
                            DTYPES[case["dt"]], case["topk"], out=layer["out"], h=layer["h"], ws=ws)


def prepare(case, seed):
    layers, kind = _inputs(case, seed), case["kind"]
    for layer in layers:
        rows, dtype = layer["x"].shape[0], layer["x"].dtype
        layer["out"] = torch.empty((rows, case["N"] if kind in ("matmul", "int4") else case["H"]), dtype=dtype,
                                   device="cuda")
        if kind == "moe":
            layer["h"] = torch.empty((rows * case["topk"], case["I"]), dtype=torch.float32, device="cuda")
    # Never empty: without a workspace a call would use the library's own.
    state = dict(case=case, layers=layers, ws=torch.empty(max(256, _workspace_bytes(case)), dtype=torch.uint8,
                                                          device="cuda"))
    if case["graph"]:
        _call(case, layers[0], state["ws"])  # a program's first step runs before it captures one
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            state["outs"] = [_call(case, layer, state["ws"]) for layer in layers]
    return state


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["outs"]
    return [_call(state["case"], layer, state["ws"]) for layer in state["layers"]]


# ---- what a pass cannot do without ---------------------------------------------------------

def _weight_bytes(dt, n):
    per, size = hipq.BLOCK[DTYPES[dt]]
    return n // per * size


def work(case):
    kind, L = case["kind"], case["layers"]
    if kind == "matmul":
        M, N, K = case["M"], case["N"], case["K"]
        return dict(bytes=L * (_weight_bytes(case["dt"], N * K) + 4 * M * (N + K)), flops=L * 2 * M * N * K)
    if kind == "mlp":
        M, H, I = case["M"], case["H"], case["I"]
        return dict(bytes=L * (3 * _weight_bytes(case["dt"], H * I) + 8 * M * H), flops=L * 6 * M * H * I)
    if kind == "int4":
        M, N, K = case["M"], case["N"], case["K"]
        size = 4 if case["x"] == "F32" else 2
        return dict(bytes=L * (N * K // 2 + 8 * N * (K // case["G"]) + size * M * (N + K)), flops=L * 2 * M * N * K)
    T, E, k, H, I = (case[n] for n in ("T", "E", "topk", "H", "I"))
    used = E * (1 - (1 - k / E) ** T)  # experts that a random routing meets
    weights = _weight_bytes(case["dt"], 3 * H * I) * used
    return dict(bytes=L * (weights + 4 * T * E + 8 * T * H + 4 * T * k * I), flops=L * 6 * T * k * H * I)


def tolerance(case):
    """8-bit activations in the decode calls (each block of 32 at 1/127 of its largest value) and
    bf16 operands elsewhere; an MLP's error is that of three products and of the quantized h.
    Four times what the calls differ by from 64 bits (0.5% to 2% for the first, 0.23% for the
    second), and no more than 3%."""
    if case["kind"] in ("matmul", "int4") and case["M"] > 8:
        return {"rel": 0.01, "max": 0.1}
    return {"rel": 0.03, "max": 0.4}


# ---- the same in 64 bits -------------------------------------------------------------------

def _f16_values(b):
    return b.contiguous().view(torch.float16).double()


def _dequant(dt, b, N, K):
    """(N, K) float64 of GGUF bytes, by the formats' definitions."""
    if dt in ("Q8_0", "Q4_0", "Q5_0"):
        b = b.view(-1, {"Q8_0": 34, "Q4_0": 18, "Q5_0": 22}[dt])
        d = _f16_values(b[:, 0:2])
        if dt == "Q8_0":
            return (b[:, 2:].contiguous().view(torch.int8).double() * d).view(N, K)
        qs = b[:, 2:] if dt == "Q4_0" else b[:, 6:]
        q = torch.cat([qs & 15, qs >> 4], dim=1).int()
        if dt == "Q5_0":
            bits = torch.arange(32, device=b.device)
            q = q + (((b[:, 2:6].int()[:, bits // 8] >> (bits % 8)) & 1) << 4)
        return ((q - (8 if dt == "Q4_0" else 16)).double() * d).view(N, K)
    if dt == "Q6_K":
        b = b.view(-1, 210)
        ql, qh = b[:, :128].view(-1, 2, 2, 32).int(), b[:, 128:192].view(-1, 2, 1, 32).int()
        shift = torch.tensor([0, 2, 4, 6], device=b.device).view(1, 1, 4, 1)
        low = torch.cat([ql & 15, ql >> 4], dim=2)  # (block, half, group of 32, element)
        q = (low | (((qh >> shift) & 3) << 4)) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        return (q.reshape(-1, 16, 16).double() * (sc * _f16_values(b[:, 208:210]))[:, :, None]).view(N, K)
    b = b.view(-1, 144 if dt == "Q4_K" else 176)
    s = b[:, 4:16].int()
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], dim=1)
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], dim=1)
    qs = (b[:, 16:] if dt == "Q4_K" else b[:, 48:]).reshape(-1, 4, 1, 32).int()
    q = torch.cat([qs & 15, qs >> 4], dim=2).view(-1, 8, 32)
    if dt == "Q5_K":
        bit = torch.arange(8, device=b.device).view(1, 8, 1)
        q = q + (((b[:, None, 16:48].int() >> bit) & 1) << 4)
    d, m = sc.double() * _f16_values(b[:, 0:2]), mn.double() * _f16_values(b[:, 2:4])
    return (q.double() * d[:, :, None] - m[:, :, None]).view(N, K)


def _product(x, dt, w, N, K):
    """x (M, K) float64 times the transposed weight, a slice of its rows at a time."""
    out, rows = torch.empty((x.shape[0], N), dtype=torch.float64, device=x.device), max(1, (1 << 28) // K)
    wb = w.reshape(N, -1)
    for n in range(0, N, rows):
        part = wb[n:n + rows]
        out[:, n:n + rows] = x @ _dequant(dt, part.reshape(-1), part.shape[0], K).t()
    return out


def _exact_layer(case, layer):
    kind, x = case["kind"], layer["x"].double()
    if kind == "matmul":
        return _product(x, case["dt"], layer["w"], case["N"], case["K"])
    if kind == "mlp":
        H, I, dt = case["H"], case["I"], case["dt"]
        h = torch.nn.functional.silu(_product(x, dt, layer["wg"], I, H)) * _product(x, dt, layer["wu"], I, H)
        return _product(h, dt, layer["wd"], H, I)
    if kind == "int4":
        N, K, G = case["N"], case["K"], case["G"]
        out = torch.empty((x.shape[0], N), dtype=torch.float64, device=x.device)
        nibble = 4 * torch.arange(8, device=x.device, dtype=torch.int32)
        for n in range(0, N, 4096):
            q = ((layer["codes"][n:n + 4096, :, None] >> nibble) & 15).reshape(-1, K // G, G).double()
            w = (q - layer["z"][n:n + 4096].double()[:, :, None]) * layer["s"][n:n + 4096].double()[:, :, None]
            out[:, n:n + 4096] = x @ w.view(-1, K).t()
        return out
    T, E, k, H, I, dt = (case[n] for n in ("T", "E", "topk", "H", "I", "dt"))
    ids = torch.topk(layer["probs"], k, dim=1).indices
    weights = torch.gather(layer["probs"].double(), 1, ids)
    weights = weights / weights.sum(dim=1, keepdim=True)
    h = torch.empty((T, k, I), dtype=torch.float64, device=x.device)
    y = torch.zeros((T, H), dtype=torch.float64, device=x.device)
    wgu, wd = layer["wgu"].reshape(E, -1), layer["wd"].reshape(E, -1)
    for e in range(E):
        t, slot = torch.nonzero(ids == e, as_tuple=True)
        if t.numel():
            gu = _product(x[t], dt, wgu[e], 2 * I, H)
            he = torch.nn.functional.silu(gu[:, :I]) * gu[:, I:]
            h[t, slot] = he
            y[t] += weights[t, slot][:, None] * _product(he, dt, wd[e], H, I)
    return y, ids, weights.reshape(-1), None, None, h.view(T * k, I)


def exact(case, seed):
    return [_exact_layer(case, layer) for layer in _inputs(case, seed)]
