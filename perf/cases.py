"""The work this library is used for, as cases that can be timed and checked.

Every case is one pass through public entry points on the sizes of decoder
models: single projections and whole decode steps (batch 1), batched decode,
SwiGLU blocks over prompts of 17 to 4096 tokens, routed experts, GGUF tensors
executed from their blocks, and the load-time converters and quantizer.
``listed()`` names representative points, ``draw()`` picks others from the
same ranges.  ``exact()`` restates each path in 64-bit torch, with decoders
for the packed formats written here, so that a result can be held against
something that shares no code with the library.
"""
import math

import torch

from eredu_amd import QuantizedLinear, dequantize, gather_qmm, quantize, quantized_matmul, quantized_matmul_batched
from eredu_amd import decode as D
from eredu_amd import gguf as G

DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
ROPE = dict(base=500000.0, factor=8.0, low=1.0, high=4.0, original=8192)
EPS = 1e-5
HEAD_DIM = 128
KV_HEADS = 8


def listed():
    return [
        # One projection for one token: the smallest call, host latency and one launch.
        dict(name="linear-m1", kind="linear", M=1, N=4096, K=4096, bits=4, gs=64, dtype="bf16"),
        # A decode batch of 16 sequences in an f16 model kept at 8 bits: the down projection.
        dict(name="linear-m16-8bit-f16", kind="linear", M=16, N=4096, K=14336, bits=8, gs=64, dtype="f16"),
        # Greedy decode of one token after 1024: embedding, layers, LM head, argmax, in one graph.
        dict(name="decode-step", kind="decode", layers=8, hidden=4096, ffn=14336, vocab=128256, pos=1024, bits=4),
        # The feed-forward block over a short, a usual and a long prompt.
        dict(name="mlp-prompt-77", kind="mlp", M=77, hidden=4096, ffn=14336, bits=4, gs=64, dtype="bf16"),
        dict(name="mlp-prompt-512", kind="mlp", M=512, hidden=4096, ffn=14336, bits=4, gs=64, dtype="bf16"),
        dict(name="mlp-prompt-4096", kind="mlp", M=4096, hidden=4096, ffn=14336, bits=4, gs=64, dtype="bf16"),
        # GGUF files keep the output head in Q6_K blocks: one token's logits.
        dict(name="gguf-head-q6k-m1", kind="gguf", type="Q6K", M=1, N=128256, K=4096),
        # A projection kept in Q4_K blocks over a usual prompt.
        dict(name="gguf-q4k-prompt-512", kind="gguf", type="Q4K", M=512, N=4096, K=14336),
        # Routed experts: one token through 2 of 8 large experts, and a prompt
        # of 512 tokens through 8 of 128 small ones.
        dict(name="moe-token", kind="moe", tokens=1, experts=8, top=2, hidden=4096, ffn=14336, bits=4, gs=64),
        dict(name="moe-prompt-512", kind="moe", tokens=512, experts=128, top=8, hidden=2048, ffn=768, bits=4, gs=64),
        # Loading: a Q4_0 tensor re-packed to the affine triple.
        dict(name="gguf-load-q4_0", kind="load", type="Q4_0", rows=14336, cols=4096),
        # Quantize on load, and the way back to dense weights.
        dict(name="quantize-4bit", kind="quantize", rows=4096, cols=14336, bits=4, gs=64, dtype="bf16"),
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step` in [lo, hi], spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(hi, max(lo, round(v / step) * step)))


def draw(rng):
    kind = rng.choice(("linear", "linear", "decode", "mlp", "mlp", "mlp", "gguf", "gguf", "moe", "moe", "load", "quantize"))
    if kind == "linear":
        return dict(kind=kind, M=_log(rng, 1, 16), N=_log(rng, 512, 16384, 128), K=_log(rng, 1024, 14336, 128),
                    bits=rng.choice((4, 4, 8)), gs=rng.choice((32, 64, 64, 128)), dtype=rng.choice(("bf16", "bf16", "f16")))
    if kind == "decode":
        return dict(kind=kind, layers=rng.randint(2, 6), hidden=rng.choice((2048, 3072, 4096)),
                    ffn=_log(rng, 4096, 14336, 512), vocab=rng.choice((32000, 49152, 128256)), pos=_log(rng, 16, 4000),
                    bits=rng.choice((4, 4, 8)))
    if kind == "mlp":
        M, hidden = _log(rng, 17, 4096), _log(rng, 1024, 5120, 128)
        ffn = _log(rng, 2048, 14336, 128)
        while M * hidden * ffn > 4096 * 4096 * 14336 // 2:
            M = M * 2 // 3
        return dict(kind=kind, M=M, hidden=hidden, ffn=ffn, bits=rng.choice((4, 4, 4, 8, 6)),
                    gs=rng.choice((32, 64, 64, 128)), dtype=rng.choice(("bf16", "bf16", "f16")))
    if kind == "gguf":
        M = rng.choice((1, _log(rng, 2, 16), _log(rng, 17, 2048)))
        return dict(kind=kind, type=rng.choice(("Q4K", "Q5K", "Q6K", "Q8_0")), M=M,
                    N=_log(rng, 1024, 32768 if M <= 16 else 14336, 128), K=_log(rng, 1024, 14336, 256))
    if kind == "moe":
        experts = rng.choice((8, 16, 64, 128))
        large = experts <= 16
        return dict(kind=kind, tokens=rng.choice((1, _log(rng, 1, 8), _log(rng, 32, 1024))), experts=experts,
                    top=2 if large else rng.choice((4, 8)), hidden=_log(rng, 1024, 4096, 512),
                    ffn=_log(rng, 1024, 8192, 512) if large else _log(rng, 512, 1536, 256),
                    bits=rng.choice((4, 4, 8)), gs=rng.choice((32, 64, 64, 128)))
    if kind == "load":
        return dict(kind=kind, type=rng.choice(("Q4_0", "Q4_1", "Q5_0")), rows=_log(rng, 512, 14336),
                    cols=_log(rng, 1024, 14336, 256))
    return dict(kind=kind, rows=_log(rng, 512, 14336), cols=_log(rng, 1024, 14336, 256), bits=rng.choice((4, 4, 8)),
                gs=rng.choice((32, 64, 128)), dtype=rng.choice(("bf16", "f16", "f32")))


# ------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEVICE, dtype=torch.float32)


def _pack(codes, bits):
    """Codes [..., 32 n] -> int32 words [..., bits n], an LSB-first bit stream."""
    c = codes.reshape(*codes.shape[:-1], -1, 32)
    out = torch.zeros((*c.shape[:-1], bits), dtype=torch.int64, device=c.device)
    for i in range(32):
        at, sh = i * bits // 32, i * bits % 32
        v = c[..., i].to(torch.int64) << sh
        out[..., at] |= v & 0xFFFFFFFF
        if sh + bits > 32:
            out[..., at + 1] |= v >> 32
    out = torch.where(out >= 2 ** 31, out - 2 ** 32, out).to(torch.int32)
    return out.reshape(*codes.shape[:-1], -1)


def _unpack(words, bits):
    w = (words.to(torch.int64) & 0xFFFFFFFF).reshape(*words.shape[:-1], -1, bits)
    out = torch.empty((*w.shape[:-1], 32), dtype=torch.int16, device=w.device)
    for i in range(32):
        at, sh = i * bits // 32, i * bits % 32
        v = w[..., at] >> sh
        if sh + bits > 32:
            v = v | (w[..., at + 1] << (32 - sh))
        out[..., i] = (v & ((1 << bits) - 1)).to(torch.int16)
    return out.reshape(*words.shape[:-1], -1)


def _affine(g, rows, cols, bits, gs, dtype, std=0.02):
    """A packed projection: N(0, std) weights, per-group minimum and step."""
    words = torch.empty((rows, cols * bits // 32), dtype=torch.int32, device=DEVICE)
    scales = torch.empty((rows, cols // gs), dtype=dtype, device=DEVICE)
    biases = torch.empty_like(scales)
    step = max(1, (1 << 25) // cols)
    for r in range(0, rows, step):
        w = _randn(g, min(step, rows - r), cols // gs, gs) * std
        lo, hi = w.amin(-1, keepdim=True), w.amax(-1, keepdim=True)
        s, b = ((hi - lo) / (2 ** bits - 1)).to(dtype), lo.to(dtype)
        q = ((w - b.float()) / s.float()).round_().clamp_(0, 2 ** bits - 1).to(torch.uint8)
        words[r:r + step] = _pack(q.reshape(w.shape[0], cols), bits)
        scales[r:r + step], biases[r:r + step] = s[..., 0], b[..., 0]
    return words, scales, biases


def _affine64(triple, bits):
    words, scales, biases = triple
    q = _unpack(words, bits).reshape(*scales.shape, -1)
    return (q.double() * scales.double()[..., None] + biases.double()[..., None]).reshape(words.shape[0], -1)


def _matmul64(x, triple, bits):
    """x . W^T in 64 bits, a slice of W's rows at a time."""
    step = max(1, (1 << 27) // x.shape[-1])
    return torch.cat([x @ _affine64([t[r:r + step] for t in triple], bits).t()
                      for r in range(0, triple[0].shape[0], step)], dim=-1)


def _half_bytes(v):
    return v.to(torch.float16).view(torch.uint8).reshape(*v.shape, 2)


def _bytes(g, *shape):
    return torch.randint(0, 256, shape, generator=g, device=DEVICE, dtype=torch.uint8)


def _spread(g, n, value):
    return value * (0.8 + 0.4 * torch.rand((n,), generator=g, device=DEVICE))


def _blocks(g, name, rows, cols):
    """GGML blocks whose decoded weights have a standard deviation near 0.02."""
    n = rows * cols // (256 if name.endswith("K") else 32)
    if name == "Q8_0":
        q = (_randn(g, n, 32) * 42).round_().clamp_(-127, 127).to(torch.int8).view(torch.uint8)
        parts = [_half_bytes(_spread(g, n, 0.02 / 42)), q]
    elif name in ("Q4_0", "Q4_1", "Q5_0"):
        d = _half_bytes(_spread(g, n, 0.0045 if name != "Q5_0" else 0.00225))
        m = _half_bytes(-_spread(g, n, 0.034))
        parts = {"Q4_0": [d], "Q4_1": [d, m], "Q5_0": [d, _bytes(g, n, 4)]}[name] + [_bytes(g, n, 16)]
    elif name in ("Q4K", "Q5K"):
        top = 15 if name == "Q4K" else 31
        six = torch.randint(32, 64, (2, n, 8), generator=g, device=DEVICE, dtype=torch.int32)
        sc, mn = six[0], six[1]
        scales = torch.cat([sc[:, :4] | (sc[:, 4:] >> 4 << 6), mn[:, :4] | (mn[:, 4:] >> 4 << 6),
                            (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], dim=1).to(torch.uint8)
        d = _spread(g, n, 0.07 / (top * 47.5))
        parts = [_half_bytes(d), _half_bytes(d * top / 2), scales]
        parts += [_bytes(g, n, 32)] * (name == "Q5K") + [_bytes(g, n, 128)]
    else:
        sc = torch.randint(32, 96, (n, 16), generator=g, device=DEVICE, dtype=torch.int32)
        sign = torch.randint(0, 2, (n, 16), generator=g, device=DEVICE, dtype=torch.int32) * 2 - 1
        sc = (sc * sign).to(torch.int8).view(torch.uint8)
        parts = [_bytes(g, n, 128), _bytes(g, n, 64), sc, _half_bytes(_spread(g, n, 0.035 / (32 * 64)))]
    return torch.cat(parts, dim=1).reshape(-1)


def _half64(b):
    return b.contiguous().view(torch.float16).double()


def _blocks64(name, raw, cols):
    """The weights of GGML blocks, [rows, cols] in 64 bits (ggml's block layouts)."""
    b = raw.reshape(-1, {"Q8_0": 34, "Q4K": 144, "Q5K": 176, "Q6K": 210}[name])
    n = b.shape[0]
    if name == "Q8_0":
        return (_half64(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).double()).reshape(-1, cols)
    if name == "Q6K":
        ql, qh = b[:, :128].int().reshape(n, 2, 2, 32), b[:, 128:192].int().reshape(n, 2, 1, 32)
        sc = b[:, 192:208].contiguous().view(torch.int8).double().reshape(n, 2, 4, 2, 1)
        low = torch.cat([ql & 15, ql >> 4], dim=2)  # [n, half, quarter, 32]
        high = torch.cat([qh >> s & 3 for s in (0, 2, 4, 6)], dim=2)
        q = ((low | high << 4) - 32).double().reshape(n, 2, 4, 2, 16)
        return (_half64(b[:, 208:210]).reshape(n, 1, 1, 1, 1) * sc * q).reshape(-1, cols)
    s = b[:, 4:16].int()
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | (s[:, :4] >> 6 << 4)], dim=1).double()
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | (s[:, 4:8] >> 6 << 4)], dim=1).double()
    qs = b[:, -128:].int().reshape(n, 4, 1, 32)
    q = torch.cat([qs & 15, qs >> 4], dim=2).reshape(n, 8, 32)
    if name == "Q5K":
        q = q | (b[:, 16:48].int()[:, None, :] >> torch.arange(8, device=b.device)[None, :, None] & 1) << 4
    d, dmin = _half64(b[:, :2]), _half64(b[:, 2:4])
    return ((d * sc)[..., None] * q.double() - (dmin * mn)[..., None]).reshape(-1, cols)


def _descriptor(name, rows, cols, raw):
    return G.TensorDescriptor("blk.weight", [cols, rows], G.GgmlType[name], raw.numel())


def _rope_freqs64():
    f = float(ROPE["base"]) ** (torch.arange(HEAD_DIM // 2, device=DEVICE, dtype=torch.float64) * 2 / HEAD_DIM)
    wave, old = f * 2 * math.pi, ROPE["original"]
    lo, hi = old / ROPE["low"], old / ROPE["high"]
    smooth = ((old / wave - ROPE["low"]) / (ROPE["high"] - ROPE["low"])).clamp(0, 1)
    mid = f / ((1 - smooth) / ROPE["factor"] + smooth)
    return torch.where(wave > lo, f * ROPE["factor"], torch.where(wave > hi, mid, f))


def _inputs(case, seed):
    """The tensors of a case, made from the seed alone."""
    g, kind = _gen(seed), case["kind"]
    if kind == "linear":
        dt = DTYPES[case["dtype"]]
        return dict(w=_affine(g, case["N"], case["K"], case["bits"], case["gs"], dt),
                    x=_randn(g, case["M"], case["K"]).to(dt))
    if kind == "mlp":
        dt, h, f = DTYPES[case["dtype"]], case["hidden"], case["ffn"]
        w = {n: _affine(g, o, i, case["bits"], case["gs"], dt) for n, o, i in (("gate", f, h), ("up", f, h), ("down", h, f))}
        return dict(w, x=_randn(g, case["M"], h).to(dt))
    if kind == "decode":
        h, f, bf = case["hidden"], case["ffn"], torch.bfloat16
        kv = KV_HEADS * HEAD_DIM
        shapes = dict(q=(h, h), k=(kv, h), v=(kv, h), o=(h, h), gate=(f, h), up=(f, h), down=(h, f))
        norm = lambda: (1.0 + 0.1 * _randn(g, h)).to(bf)  # noqa: E731
        layers = [dict({n: _affine(g, *s, case["bits"], 64, bf) for n, s in shapes.items()}, in_norm=norm(),
                       post_norm=norm()) for _ in range(case["layers"])]
        rows = (case["pos"] + 64) // 32 * 32
        cache = lambda: [_randn(g, KV_HEADS, rows, HEAD_DIM).to(bf) for _ in range(case["layers"])]  # noqa: E731
        embed = torch.empty((case["vocab"], h), dtype=bf, device=DEVICE).normal_(generator=g)
        return dict(layers=layers, head=_affine(g, case["vocab"], h, case["bits"], 64, bf), norm=norm(), embed=embed,
                    k=cache(), v=cache(), rows=rows,
                    token=torch.randint(0, case["vocab"], (1,), generator=g, device=DEVICE, dtype=torch.int32))
    if kind == "gguf":
        return dict(raw=_blocks(g, case["type"], case["N"], case["K"]),
                    x=_randn(g, case["M"], case["K"]).to(torch.bfloat16))
    if kind == "moe":
        bf, h, f, E = torch.bfloat16, case["hidden"], case["ffn"], case["experts"]
        w = {}
        for n, o, i in (("gate", f, h), ("up", f, h), ("down", h, f)):
            t = _affine(g, E * o, i, case["bits"], case["gs"], bf)
            w[n] = tuple(a.reshape(E, o, -1) for a in t)
        # a router's choice of `top` different experts per token, the popular ones more often
        logits = _randn(g, case["tokens"], E) + 0.5 * _randn(g, 1, E)
        picks = logits.topk(case["top"], dim=-1).indices.reshape(-1)
        if picks.numel() > 16:  # a prompt's routes are sorted by expert
            picks, order = torch.sort(picks, stable=True)
        else:
            order = torch.arange(picks.numel(), device=DEVICE)
        return dict(w, x=_randn(g, case["tokens"], 1, h).to(bf), token=(order // case["top"]).to(torch.int32),
                    expert=picks.to(torch.int32), by_expert=bool(picks.numel() > 16))
    if kind == "load":
        return dict(raw=_blocks(g, case["type"], case["rows"], case["cols"]))
    return dict(w=(_randn(g, case["rows"], case["cols"]) * 0.02).to(DTYPES[case["dtype"]]))


# ------------------------------------------------------------ the library's side

def prepare(case, seed):
    kind, s = case["kind"], _inputs(case, seed)
    s["case"] = case
    if kind == "linear":
        s["layer"] = QuantizedLinear(*s["w"], case["gs"], case["bits"])
    elif kind == "gguf":
        native = G.NativeTensor("blk.weight", [case["N"], case["K"]], G.GgmlType[case["type"]], G.Endian.Little, s["raw"])
        s["layer"] = QuantizedLinear.from_native(native)
    elif kind == "load":
        s["desc"] = _descriptor(case["type"], case["rows"], case["cols"], s["raw"])
    elif kind == "decode":
        lin = lambda t: D.QLinear(*t, case["bits"], 64)  # noqa: E731
        names = ("q", "k", "v", "o", "gate", "up", "down")
        layers = [D.DecoderLayer(L["in_norm"], L["post_norm"], *(lin(L[n]) for n in names)) for L in s["layers"]]
        freqs = D.llama3_rope_freqs(HEAD_DIM, ROPE["base"], ROPE["factor"], ROPE["low"], ROPE["high"], ROPE["original"])
        dec = D.LlamaDecoder(layers, s["embed"], s["norm"], lin(s["head"]), n_heads=case["hidden"] // HEAD_DIM,
                             n_kv_heads=KV_HEADS, eps=EPS, freqs=freqs, max_seq=s["rows"], k_caches=s["k"], v_caches=s["v"])
        start = torch.full((1,), case["pos"], dtype=torch.int32, device=DEVICE)
        stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        stream.wait_stream(torch.cuda.current_stream())

        def step():  # the request's token and position, then one token of the decode loop
            torch.add(s["token"], 0, out=dec.token)
            torch.add(start, 0, out=dec.position)
            dec.step_device()

        with torch.cuda.stream(stream):
            step()
        torch.cuda.current_stream().wait_stream(stream)
        with torch.cuda.graph(graph, stream=stream):
            step()
        s.update(decoder=dec, graph=graph, start=start)
    return s


def run(state):
    s, case = state, state["case"]
    kind = case["kind"]
    if kind == "linear" or kind == "gguf":
        return s["layer"](s["x"])
    if kind == "mlp":
        gate, up = quantized_matmul_batched([(s["x"], *s["gate"]), (s["x"], *s["up"])], True, case["gs"], case["bits"])
        act = D.silu_mul(gate, up) if case["dtype"] == "bf16" else torch.nn.functional.silu(gate) * up
        return quantized_matmul(act, *s["down"], True, case["gs"], case["bits"])
    if kind == "decode":
        s["graph"].replay()
        return dict(logits=s["decoder"].logits, k=s["k"], v=s["v"])
    if kind == "moe":
        routed = dict(transpose=True, group_size=case["gs"], bits=case["bits"], sorted_indices=s["by_expert"])
        gate = gather_qmm(s["x"], *s["gate"], s["token"], s["expert"], **routed)
        up = gather_qmm(s["x"], *s["up"], s["token"], s["expert"], **routed)
        return gather_qmm(D.silu_mul(gate, up), *s["down"], None, s["expert"], **routed)
    if kind == "load":
        t = G.convert(s["desc"], s["raw"])
        return dict(weights=t.weights, scales=t.scales, biases=t.biases)
    w, scales, biases = quantize(s["w"], case["gs"], case["bits"])
    return dict(weights=w, scales=scales, biases=biases, dense=dequantize(w, scales, biases, case["gs"], case["bits"]))


# ------------------------------------------------------------ what it is held against

def _packed_bytes(rows, cols, bits, gs):
    return rows * cols * bits // 8 + 4 * rows * (cols // gs)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return dict(bytes=_packed_bytes(N, K, case["bits"], case["gs"]) + 2 * M * (N + K), flops=2 * M * N * K)
    if kind == "mlp":
        M, h, f = case["M"], case["hidden"], case["ffn"]
        return dict(bytes=3 * _packed_bytes(f, h, case["bits"], case["gs"]) + 4 * M * h, flops=6 * M * h * f)
    if kind == "decode":
        h, f, kv, L = case["hidden"], case["ffn"], KV_HEADS * HEAD_DIM, case["layers"]
        weights = L * (2 * h * h + 2 * kv * h + 3 * f * h) + case["vocab"] * h
        rows = 2 * L * kv * (case["pos"] + 2) * 2  # K and V rows read, one of each written
        return dict(bytes=_packed_bytes(weights // 64, 64, case["bits"], 64) + rows + 2 * case["vocab"] + 4 * h * (L + 1),
                    flops=2 * weights + 4 * L * h * (case["pos"] + 1))
    if kind == "gguf":
        M, N, K = case["M"], case["N"], case["K"]
        values, nbytes = G.GgmlType[case["type"]].block_and_bytes()
        return dict(bytes=N * K // values * nbytes + 2 * M * (N + K), flops=2 * M * N * K)
    if kind == "moe":
        R, h, f = case["tokens"] * case["top"], case["hidden"], case["ffn"]
        hit = case["experts"] * (1 - (1 - case["top"] / case["experts"]) ** case["tokens"])  # experts reached
        return dict(bytes=int(3 * hit * _packed_bytes(f, h, case["bits"], case["gs"])) + 2 * h * (case["tokens"] + R),
                    flops=6 * R * h * f)
    n = case["rows"] * case["cols"]
    if kind == "load":
        values, nbytes = G.GgmlType[case["type"]].block_and_bytes()
        bits, gs = G.affine_config(G.GgmlType[case["type"]])
        return dict(bytes=n // values * nbytes + _packed_bytes(case["rows"], case["cols"], bits, gs), flops=0)
    width = 4 if case["dtype"] == "f32" else 2
    return dict(bytes=2 * n * width + n * case["bits"] // 8 + 2 * width * n // case["gs"], flops=0)


def tolerance(case):
    """About four times the error that the data types give against 64 bits."""
    kind = case["kind"]
    if kind in ("load", "quantize"):
        return "exact"
    if kind == "decode":  # bf16 states rounded through every layer
        return {"rel": 0.03, "max": 0.3}
    if case.get("dtype") == "f16":
        return {"rel": 2e-3, "max": 2e-2}
    return {"rel": 1e-2, "max": 1e-1}


def exact(case, seed):
    kind, s = case["kind"], _inputs(case, seed)
    silu = lambda g: g * torch.sigmoid(g)  # noqa: E731
    if kind == "linear":
        return _matmul64(s["x"].double(), s["w"], case["bits"])
    if kind == "mlp":
        x = s["x"].double()
        act = silu(_matmul64(x, s["gate"], case["bits"])) * _matmul64(x, s["up"], case["bits"])
        return _matmul64(act, s["down"], case["bits"])
    if kind == "decode":
        return _decode64(case, s, silu)
    if kind == "gguf":
        values, nbytes = G.GgmlType[case["type"]].block_and_bytes()
        row, step, x = case["K"] // values * nbytes, max(1, (1 << 26) // case["K"]), s["x"].double()
        return torch.cat([x @ _blocks64(case["type"], s["raw"][r * row:(r + step) * row], case["K"]).t()
                          for r in range(0, case["N"], step)], dim=-1)
    if kind == "moe":
        out = torch.empty((s["expert"].numel(), 1, case["hidden"]), dtype=torch.float64, device=DEVICE)
        for e in s["expert"].unique().tolist():
            at = (s["expert"] == e).nonzero()[:, 0]
            x = s["x"][s["token"][at].long(), 0].double()
            one = lambda n, v: _matmul64(v, [t[e] for t in s[n]], case["bits"])  # noqa: E731
            out[at, 0] = one("down", silu(one("gate", x)) * one("up", x))
        return out
    if kind == "load":
        b = s["raw"].reshape(-1, {"Q4_0": 18, "Q4_1": 20, "Q5_0": 22}[case["type"]])
        d = _half64(b[:, :2])
        bias = {"Q4_0": lambda: -8 * d, "Q4_1": lambda: _half64(b[:, 2:4]), "Q5_0": lambda: -16 * d}[case["type"]]()
        shape = (case["rows"], case["cols"] // 32)
        return dict(weights=None, scales=d.reshape(shape), biases=bias.reshape(shape))
    # the affine rule: the larger end of a group is kept exactly, codes count from it
    w = s["w"].double().reshape(case["rows"], -1, case["gs"])
    lo, hi = w.amin(-1), w.amax(-1)
    low = lo.abs() > hi.abs()
    step = (hi - lo) / (2 ** case["bits"] - 1)
    edge, step = torch.where(low, lo, hi), torch.where(low, step, -step)
    zero = torch.round(edge / step)
    return dict(weights=None, scales=torch.where(zero != 0, edge / zero, step), biases=edge, dense=None)


def _decode64(case, s, silu):
    h, pos, bits = case["hidden"], case["pos"], case["bits"]
    angle = pos / _rope_freqs64()
    cos, sin = torch.cos(angle), torch.sin(angle)

    def rope(v):
        a, b = v[:, :HEAD_DIM // 2], v[:, HEAD_DIM // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=1)

    def norm(v, weight):
        return v * torch.rsqrt((v * v).mean() + EPS) * weight.double()

    x = s["embed"][s["token"].long()].double()
    ks, vs = [], []
    for i, L in enumerate(s["layers"]):
        one = lambda n, v: _matmul64(v, L[n], bits)  # noqa: E731
        a = norm(x, L["in_norm"])
        q = rope(one("q", a).reshape(-1, HEAD_DIM))
        k, v = s["k"][i].double(), s["v"][i].double()
        k[:, pos], v[:, pos] = rope(one("k", a).reshape(KV_HEADS, HEAD_DIM)), one("v", a).reshape(KV_HEADS, HEAD_DIM)
        q = q.reshape(KV_HEADS, -1, HEAD_DIM)
        p = torch.softmax(q @ k[:, :pos + 1].transpose(1, 2).contiguous() / math.sqrt(HEAD_DIM), dim=-1)
        x = x + one("o", (p @ v[:, :pos + 1].contiguous()).reshape(1, h))
        b = norm(x, L["post_norm"])
        x = x + one("down", silu(one("gate", b)) * one("up", b))
        ks.append(k)
        vs.append(v)
    return dict(logits=_matmul64(norm(x, s["norm"]), s["head"], bits)[0], k=ks, v=vs)
