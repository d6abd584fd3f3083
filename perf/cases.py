"""The calls whose speed this framework is measured by, over the range that a decoder built on it meets.

Four kinds of use, each through the public entry points of comp_amd.host:

  call     one eager GEMV from f32 activations, as a caller that drives the decoder from Python makes it: quantize()
           and gemv() (the reference's two launches), or gemv_f32() (one).
  step     a decode step's linear layers captured once into a HIP graph and replayed: f32 activations of m sequences
           in, f32 outputs out.  1 to 3 columns run gemv_f32_into, larger batches quantize_into and gemv_into.
  prefill  a prompt's m tokens through one linear layer: quantize() and gemm(), eager.
  ingest   ggml block bytes already on the device into the split planes (split_device), once per weight at load time.

Every layer gets an input of its own (attention, norms and activation functions between the layers are the caller's).
Weights are seeded ggml-like planes: the formats' quant codes of bell-shaped values, f16 scales that vary from block
to block.  Activations are normal with a few large channels, as transformer activations have them.
"""

import math

import torch

from comp_amd import host

# block values, quant bytes, ggml block bytes, offset of the quants, scale-plane bytes, activation block
_FORMATS = {
    "q4_0": (32, 16, 18, 2, 2, 32),
    "iq4_nl": (32, 16, 18, 2, 2, 32),
    "q8_0": (32, 32, 34, 2, 2, 32),
    "tq2_0": (256, 64, 66, 0, 2, 256),
    "q4_k": (256, 128, 144, 16, 16, 256),
}
_IQ4_NL = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)
_LLAMA = "6144x4096,4096x4096,28672x4096,4096x14336"  # Llama-3-8B: Q+K+V, output, gate+up, down
_BITNET = "6912x2560,2560x6912"                       # BitNet-2B: the FFN's two matrices


def listed():
    return [
        # a Python-driven decoder's smallest call: one BitNet-2B matrix, one token
        {"name": "call_tq2_0_one_token", "kind": "call", "entry": "fused", "fmt": "tq2_0", "m": 1, "n": 6912, "k": 2560,
         "mode": 2},
        # a caller that switched over from the reference: its two launches, its default knobs, dp4a mode
        {"name": "call_q4_0_two_launches", "kind": "call", "entry": "knobs", "fmt": "q4_0", "m": 1, "n": 4096,
         "k": 4096, "mode": 2},
        # one token through BitNet-2B's FFN matrices, eight layers
        {"name": "step_tq2_0_bitnet_m1", "kind": "step", "fmt": "tq2_0", "m": 1, "shapes": _BITNET, "layers": 8},
        # one token through a Llama-3-8B layer and the LM head
        {"name": "step_q4_0_llama_head_m1", "kind": "step", "fmt": "q4_0", "m": 1, "shapes": _LLAMA + ",128256x4096",
         "layers": 1},
        # three tokens (two drafted ones to verify) through two Llama-3-8B layers in Q4_K
        {"name": "step_q4_k_llama_m3", "kind": "step", "fmt": "q4_k", "m": 3, "shapes": _LLAMA, "layers": 2},
        # a small batch of sequences on BitNet-2B
        {"name": "step_tq2_0_bitnet_m8", "kind": "step", "fmt": "tq2_0", "m": 8, "shapes": _BITNET, "layers": 8},
        # a serving batch of 16 on Llama-3-8B
        {"name": "step_q4_0_llama_m16", "kind": "step", "fmt": "q4_0", "m": 16, "shapes": _LLAMA, "layers": 2},
        # a larger batch over ragged matrices: odd row counts, K not a power of two
        {"name": "step_q8_0_ragged_m50", "kind": "step", "fmt": "q8_0", "m": 50,
         "shapes": "4097x4192,6913x4192,127x4192", "layers": 2},
        # a prompt of 512 tokens through Llama-3-8B's gate projection
        {"name": "prefill_q4_0_m512", "kind": "prefill", "fmt": "q4_0", "m": 512, "n": 14336, "k": 4096},
        # a prompt of 2048 tokens through BitNet-2B's gate projection
        {"name": "prefill_tq2_0_m2048", "kind": "prefill", "fmt": "tq2_0", "m": 2048, "n": 6912, "k": 2560},
        # a prompt of an odd length through Llama-3-8B's down projection in Q4_K
        {"name": "prefill_q4_k_m1001", "kind": "prefill", "fmt": "q4_k", "m": 1001, "n": 4096, "k": 14336},
        # a GGUF file's LM head on its way into the split planes
        {"name": "ingest_q4_0_head", "kind": "ingest", "fmt": "q4_0", "n": 128256, "k": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, fmt, lo=256, hi=14336):
    """A K of the format's blocks."""
    blk = _FORMATS[fmt][0]
    return max(1, _log(rng, lo, hi) // blk) * blk


def draw(rng):
    kind = rng.choice(["call", "step", "step", "prefill", "prefill", "ingest"])
    fmt = rng.choice(sorted(_FORMATS))
    if kind == "call":
        entry = rng.choice(["fused", "plan", "knobs"])
        return {"kind": kind, "entry": entry, "fmt": fmt, "m": rng.randint(1, 3), "n": _log(rng, 100, 16384),
                "k": _size(rng, fmt, 512), "mode": rng.choice([2, 2, 0])}
    if kind == "step":
        shapes = ",".join("%dx%d" % (_log(rng, 100, 30000), _size(rng, fmt)) for _ in range(rng.randint(2, 4)))
        return {"kind": kind, "fmt": fmt, "m": rng.choice([1, 2, 3, _log(rng, 4, 64)]), "shapes": shapes, "layers": 2}
    if kind == "prefill":
        k = _size(rng, fmt)
        n = _log(rng, 100, 14336)
        return {"kind": kind, "fmt": fmt, "m": min(_log(rng, 65, 2048), max(65, 3 * 10**10 // (n * k))), "n": n, "k": k}
    return {"kind": kind, "fmt": fmt, "n": _log(rng, 1000, 60000), "k": _size(rng, fmt, 1024, 8192)}


# ---- inputs -----------------------------------------------------------------------------------------------------------


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _f16_scales(g, shape, level):
    """Positive f16 scales around `level`, spread by about a factor of two, a sign now and then."""
    s = level * torch.exp2(torch.randn(shape, generator=g, device="cuda") * 0.5)
    s = torch.where(torch.rand(shape, generator=g, device="cuda") < 0.5, -s, s)
    return s.to(torch.float16).view(torch.int16)


def _planes(fmt, n, k, g):
    """Split planes (WQ uint8 [n][quant bytes], WS int16 [n][scale words]) of seeded weights."""
    blk, qb = _FORMATS[fmt][:2]
    nb = k // blk
    if fmt == "tq2_0":  # crumbs 0, 1, 2
        c = torch.randint(0, 3, (4, n, nb * qb), generator=g, device="cuda", dtype=torch.uint8)
        wq = c[0] | (c[1] << 2) | (c[2] << 4) | (c[3] << 6)
    elif fmt == "q8_0":
        wq = (torch.randn((n, nb * qb), generator=g, device="cuda") * 40).round_().clamp_(-127, 127)
        wq = wq.to(torch.int8).view(torch.uint8)
    else:  # two nibbles a byte
        lo, hi = (
            (torch.randn((n, nb * qb), generator=g, device="cuda") * 2.7 + 8).round_().clamp_(0, 15).to(torch.uint8)
            for _ in range(2)
        )
        wq = lo | (hi << 4)
    level = {"q4_0": 0.01, "iq4_nl": 6e-4, "q8_0": 6e-4, "tq2_0": 0.03, "q4_k": 2e-4}[fmt]
    if fmt == "q4_k":
        ws = torch.randint(0, 256, (n, nb, 16), generator=g, device="cuda", dtype=torch.uint8).view(torch.int16)
        ws[:, :, 0] = _f16_scales(g, (n, nb), level)
        ws[:, :, 1] = _f16_scales(g, (n, nb), 8 * level) & 0x7FFF
        return wq, ws.reshape(n, nb * 8)
    return wq, _f16_scales(g, (n, nb), level)


def _activations(m, k, g):
    x = torch.randn((m, k), generator=g, device="cuda")
    return x * torch.where(torch.rand((k,), generator=g, device="cuda") < 0.01, 12.0, 1.0)


def _matrices(case):
    """(n, k) of every linear layer of a step, in order."""
    one = [tuple(int(v) for v in s.split("x")) for s in case["shapes"].split(",")]
    return one * case["layers"]


def _inputs(case, seed):
    """What both prepare() and exact() start from."""
    g = _generator(seed)
    fmt = case["fmt"]
    if case["kind"] == "ingest":
        return torch.randint(0, 256, (case["n"] * (case["k"] // _FORMATS[fmt][0]) * _FORMATS[fmt][2],), generator=g,
                             device="cuda", dtype=torch.uint8)  # fmt: skip
    shapes = _matrices(case) if case["kind"] == "step" else [(case["n"], case["k"])]
    return [(n, k, *_planes(fmt, n, k, g), _activations(case["m"], k, g)) for n, k in shapes]


def _step(state):
    """One decode step's launches into the state's buffers."""
    fmt = state["fmt"]
    for n, k, wq, ws, x, xq, xd, y in state["layers"]:
        if xq is None:
            host.gemv_f32_into(fmt, wq, ws, x, y, n, k)
        else:
            host.quantize_into(fmt, x, xq, xd)
            host.gemv_into(fmt, wq, ws, xq, xd, y, n, k)


def prepare(case, seed):
    fmt = case["fmt"]
    if case["kind"] == "ingest":
        return {"case": case, "W": _inputs(case, seed)}
    if case["kind"] != "step":
        n, k, wq, ws, x = _inputs(case, seed)[0]
        return {"case": case, "wq": wq, "ws": ws, "x": x}
    m, ablk = case["m"], _FORMATS[fmt][5]
    layers = []
    for n, k, wq, ws, x in _inputs(case, seed):
        xq = xd = None
        if m > 3:
            xq = torch.empty((m, k), dtype=torch.int8, device="cuda")
            xd = torch.empty((m, k // ablk), dtype=torch.float32, device="cuda")
        layers.append((n, k, wq, ws, x, xq, xd, torch.empty((m, n), dtype=torch.float32, device="cuda")))
    state = {"case": case, "fmt": fmt, "layers": layers}
    _step(state)  # every kernel is loaded before the capture
    torch.cuda.synchronize()
    state["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(state["graph"]):
        _step(state)
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "step":
        state["graph"].replay()
        return [layer[-1] for layer in state["layers"]]
    fmt, n, k = case["fmt"], case["n"], case["k"]
    if case["kind"] == "ingest":
        return list(host.split_device(fmt, state["W"], n, k))
    wq, ws, x = state["wq"], state["ws"], state["x"]
    if case["kind"] == "call" and case["entry"] == "fused":
        return [host.gemv_f32(fmt, wq, ws, x, n, k, mode=case["mode"])[0]]
    xq, xd = host.quantize(fmt, x)
    if case["kind"] == "prefill":
        return [host.gemm(fmt, wq, ws, xq, xd, n, k)[0]]
    if case["entry"] == "knobs":
        return [host.gemv(fmt, wq, ws, xq, xd, n, k, mode=case["mode"])[0]]
    return [host.gemv(fmt, wq, ws, xq, xd, n, k, block_n=None, mode=case["mode"])[0]]


# ---- what a pass cannot do without, and what its outputs are ----------------------------------------------------------


def work(case):
    blk, qb, nbytes, _, sb, _ = _FORMATS[case["fmt"]]
    if case["kind"] == "ingest":
        return {"bytes": 2 * case["n"] * (case["k"] // blk) * nbytes, "flops": 0}
    shapes = _matrices(case) if case["kind"] == "step" else [(case["n"], case["k"])]
    m = case["m"]
    return {
        "bytes": sum(n * (k // blk) * (qb + sb) + 4 * m * k + 4 * m * n for n, k in shapes),
        "flops": sum(2 * m * n * k for n, k in shapes),
    }


def tolerance(case):
    """Bytes are the same bytes.  The outputs are f32 sums of exact integer dots times f32 scales: against the 64-bit
    sums the furthest case is 2.1e-7 off (relative 2-norm), whichever order the blocks are summed in."""
    return "exact" if case["kind"] == "ingest" else {"rel": 1e-6, "max": 2e-5}


def _quantized(fmt, x):
    """The quantizers' definition in plain torch: x (f32) -> the f64 values the q8 codes and scales stand for.  Their
    f32 steps (the scale, its reciprocal, the product) are part of the definition; a quotient rounded to f64 and then to
    f32 is the correctly rounded f32 quotient."""
    m, k = x.shape
    if _FORMATS[fmt][5] == 32:  # q8_0: d = amax / 127, codes rounded half away from zero, the scale stored as f16
        b = x.view(m, k // 32, 32)
        d = (b.abs().amax(2, keepdim=True).double() / 127.0).float()
        v = b * torch.where(d != 0, 1.0 / d.double(), torch.zeros_like(d)).float()
        q = torch.copysign((v.abs().double() + 0.5).floor(), v.double())
        return (q * d.to(torch.float16).double()).view(m, k)
    b = x.view(m, k // 256, 256)  # q8_K: -127 / (the value of largest magnitude), codes rounded half to even
    at = b.abs().argmax(2, keepdim=True)
    mx = torch.gather(b, 2, at)
    scale = torch.where(mx != 0, -127.0 / mx.double(), torch.zeros_like(mx)).float()
    q = (b * scale).round().clamp_(max=127).double()
    d = torch.where(mx != 0, 1.0 / scale.double(), torch.zeros_like(scale)).float()
    return (q * d.double()).view(m, k)


def _half(bits):
    return bits.contiguous().view(torch.float16).double()


def _dequantized(fmt, wq, ws, n, k):
    """f64 [n][k] weights of the split planes."""
    blk, qb = _FORMATS[fmt][:2]
    nb = k // blk
    b = wq.view(n, nb, qb)
    if fmt == "q8_0":
        v = b.view(torch.int8).double() * _half(ws).view(n, nb, 1)
    elif fmt == "tq2_0":  # byte 32 h + i, bits 2 j: value 128 h + 32 j + i
        c = torch.stack([(b.view(n, nb, 2, 32) >> (2 * j)) & 3 for j in range(4)], 3)
        v = (c.double() - 1).view(n, nb, 256) * _half(ws).view(n, nb, 1)
    elif fmt == "q4_k":  # byte 32 j + i: value 64 j + i (low nibble), 64 j + 32 + i (high)
        q = torch.stack([b.view(n, nb, 4, 32) & 15, b.view(n, nb, 4, 32) >> 4], 3).view(n, nb, 8, 32).double()
        w = ws.view(n, nb, 8)
        p = w[:, :, 2:].contiguous().view(torch.uint8).view(n, nb, 12)
        sc = torch.cat([p[:, :, :4] & 63, (p[:, :, 8:] & 15) | ((p[:, :, :4] >> 6) << 4)], 2)
        mn = torch.cat([p[:, :, 4:8] & 63, (p[:, :, 8:] >> 4) | ((p[:, :, 4:8] >> 6) << 4)], 2)
        v = q * (_half(w[:, :, :1]) * sc.double()).unsqueeze(3) - (_half(w[:, :, 1:2]) * mn.double()).unsqueeze(3)
    else:
        q = torch.cat([b & 15, b >> 4], 2)
        if fmt == "iq4_nl":
            v = torch.tensor(_IQ4_NL, dtype=torch.float64, device=q.device)[q.long()]
        else:
            v = q.double() - 8
        v = v * _half(ws).view(n, nb, 1)
    return v.reshape(n, k)


def exact(case, seed):
    if case["kind"] == "ingest":
        return None  # bytes
    fmt = case["fmt"]
    outs = []
    for n, k, wq, ws, x in _inputs(case, seed):
        xv = _quantized(fmt, x)
        y = torch.empty((case["m"], n), dtype=torch.float64, device=x.device)
        for r in range(0, n, 16384):  # a slice of rows at a time
            e = min(n, r + 16384)
            y[:, r:e] = xv @ _dequantized(fmt, wq[r:e], ws[r:e], e - r, k).T.contiguous()
        outs.append(y)
    return outs
