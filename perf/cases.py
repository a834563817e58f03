"""The work that performance is judged by: what a program built on `dtas_amd.ops` runs, over the range it runs it.

Four kinds of pass, each a chain of destination-passing calls whose buffers the program allocated once:

  layer   one transformer layer of the dolly-v2-3b graph (hidden 2560, 32 heads of 80, 20 of them rotated), call by call
          as its `prefill` and `decode` issue them: n new positions against m = past + n keys.  n = 1 is the decode step,
          past = 0 a prompt, both above zero a prompt that continues a conversation.  `q8` takes the 8-bit weights.
  ends    what a step runs outside its layers: the embedding lookup of n tokens and the causal mask before them, the last
          layer norm, the vocabulary projection of the last position and the sampling softmax behind them.
  block   the projections at hidden 4096 / 11008 with RMSNorm and residual adds: output projection, up, down.
  rows    the memory-bound calls over [n, H] activations: both casts, add, RMSNorm, layer norm, copy, fp16 softmax.

Every call reads its operands and writes a buffer of the caller's, so `work` counts each call's operands once each.
"""
import math

import torch

from dtas_amd import _lib, ops

HIDDEN, HEADS, DIM, ROT, FF, VOCAB, MAX_POS = 2560, 32, 80, 20, 10240, 50280, 4096
SCALE = 0.11179039301310044
WIDE, WIDE_FF = 4096, 11008


def listed():
    return [
        # a handful of rows: nothing but launches
        {"name": "rows_3", "kind": "rows", "n": 3, "H": 4096},
        # the far end of the elementwise and norm sweeps
        {"name": "rows_4096", "kind": "rows", "n": 4096, "H": 4096},
        # the decode step early in a conversation, and late in a long one (any key count occurs: every step adds one)
        {"name": "decode_127", "kind": "layer", "n": 1, "past": 126, "q8": False},
        {"name": "decode_3001", "kind": "layer", "n": 1, "past": 3000, "q8": False},
        # the same with 8-bit weights, which is what they are for
        {"name": "decode_q8_1024", "kind": "layer", "n": 1, "past": 1023, "q8": True},
        # a one-line prompt
        {"name": "prompt_17", "kind": "layer", "n": 17, "past": 0, "q8": False},
        # the next message of a conversation, 8-bit weights
        {"name": "continue_q8_203", "kind": "layer", "n": 203, "past": 500, "q8": True},
        # prompts as they come (off every vector width), and the largest
        {"name": "prompt_1025", "kind": "layer", "n": 1025, "past": 0, "q8": False},
        {"name": "prompt_2048", "kind": "layer", "n": 2048, "past": 0, "q8": False},
        # the two ends of a decode step
        {"name": "ends_1", "kind": "ends", "n": 1, "past": 600, "q8": False},
        # 48 sequences decoded together, and the largest batch of rows
        {"name": "block_48", "kind": "block", "n": 48},
        {"name": "block_8192", "kind": "block", "n": 8192},
    ]


def _log_int(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(("layer", "layer", "layer", "ends", "block", "rows"))
    if kind == "rows":
        H = rng.choice((2560, 4096, 5120, 8192))
        return {"kind": kind, "n": _log_int(rng, 1, (4096 * 4096) // H), "H": H}
    if kind == "block":
        return {"kind": kind, "n": _log_int(rng, 1, 8192)}
    q8 = rng.random() < 0.4
    if kind == "ends":
        n = _log_int(rng, 1, 2048)
        return {"kind": kind, "n": n, "past": rng.choice((0, _log_int(rng, 1, MAX_POS - n))), "q8": q8}
    form = rng.choice(("decode", "prompt", "continue"))
    if form == "decode":
        return {"kind": kind, "n": 1, "past": _log_int(rng, 15, MAX_POS - 1), "q8": q8}
    if form == "prompt":
        return {"kind": kind, "n": _log_int(rng, 2, 2048), "past": 0, "q8": q8}
    return {"kind": kind, "n": _log_int(rng, 2, 768), "past": _log_int(rng, 16, 3072), "q8": q8}


# --------------------------------------------------------------------------------------------- inputs
class _Make:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=torch.float16):
        return (torch.randn(shape, device="cuda", generator=self.g) * std).to(dtype)

    def uniform(self, *shape, lo, hi, dtype=torch.float32):
        return (torch.rand(shape, device="cuda", generator=self.g) * (hi - lo) + lo).to(dtype)

    def ids(self, n, V):
        return torch.randint(0, V, (n,), device="cuda", generator=self.g, dtype=torch.int32)

    def q8(self, N, K, scale_dtype=torch.float16):
        """Normally distributed weights of standard deviation 0.02 as bytes around 127, four to a word, and a scale per 32."""
        b = (torch.randn((N, K), device="cuda", generator=self.g) * 40 + 127).round_().clamp_(0, 254).to(torch.uint8)
        scale = self.uniform(N, K // 32, lo=0.0004, hi=0.0006, dtype=scale_dtype)
        return b.view(torch.int32), scale


def _empty(*shape, dtype=torch.float16):
    return torch.empty(shape, dtype=dtype, device="cuda")


def _prepare_layer(case, mk):
    n, past, q8 = case["n"], case["past"], case["q8"]
    m = n + past
    weight = mk.q8 if q8 else (lambda N, K: (mk.normal(N, K, std=0.02),))
    pos = torch.arange(MAX_POS, device="cuda", dtype=torch.float32)[:, None]
    angle = pos / 10000.0 ** (torch.arange(ROT, device="cuda") % (ROT // 2) * 2.0 / ROT)[None, :]
    cache = lambda: torch.cat([mk.normal(past, HEADS, DIM), torch.zeros(n, HEADS, DIM, dtype=torch.float16, device="cuda")])
    mask = _empty(1, 1, n, m)
    ops.attn_mask(mask)
    heads = lambda rows: _empty(HEADS, rows, DIM)
    rows = lambda: _empty(n, HEADS, DIM)
    s = {
        "q8": q8, "n": n, "m": m, "past": past, "x": mk.normal(n, HIDDEN), "mask": mask,
        "keys": cache(), "values": cache(), "cos": angle.cos().half(), "sin": angle.sin().half(),
        "ln1": (mk.uniform(HIDDEN, lo=0.5, hi=1.5), mk.uniform(HIDDEN, lo=-0.2, hi=0.2)),
        "ln2": (mk.uniform(HIDDEN, lo=0.5, hi=1.5), mk.uniform(HIDDEN, lo=-0.2, hi=0.2)),
        "qkv_w": weight(3 * HIDDEN, HIDDEN), "o_w": weight(HIDDEN, HIDDEN), "up_w": weight(FF, HIDDEN), "down_w": weight(HIDDEN, FF),
        "qkv_b": mk.normal(3 * HIDDEN, std=0.02), "o_b": mk.normal(HIDDEN, std=0.02), "up_b": mk.normal(FF, std=0.02),
        "down_b": mk.normal(HIDDEN, std=0.02),
        "x32": _empty(n, HIDDEN, dtype=torch.float32), "h1": _empty(n, HIDDEN), "qkv": _empty(n, 3 * HIDDEN),
        "q": rows(), "k": rows(), "v": rows(), "qr": rows(), "kr": rows(), "qh": heads(n), "kh": heads(m), "vh": heads(m),
        "scores": _empty(HEADS, n, m, dtype=torch.float32), "probs": _empty(HEADS, n, m), "ctx": heads(n), "merged": rows(),
        "h2": _empty(n, HIDDEN), "up": _empty(n, FF), "down": _empty(n, HIDDEN), "y": _empty(n, HIDDEN),
    }
    if q8:
        s["o_f16"] = _empty(HIDDEN, HIDDEN)
    return s


def _prepare_ends(case, mk):
    n, m, q8 = case["n"], case["n"] + case["past"], case["q8"]
    table = mk.q8(VOCAB, HIDDEN) if q8 else (mk.normal(VOCAB, HIDDEN),)
    head = mk.q8(VOCAB, HIDDEN, torch.float32) if q8 else (mk.normal(VOCAB, HIDDEN, std=0.02, dtype=torch.float32),)
    return {
        "q8": q8, "n": n, "table": table, "head": head, "ids": mk.ids(n, VOCAB), "hidden": mk.normal(n, HIDDEN, dtype=torch.float32),
        "ln": (mk.uniform(HIDDEN, lo=0.5, hi=1.5), mk.uniform(HIDDEN, lo=-0.2, hi=0.2)),
        "temperature": torch.tensor(0.7, dtype=torch.float32, device="cuda"),
        "embedded": _empty(n, HIDDEN), "mask": _empty(1, 1, n, m), "normed": _empty(n, HIDDEN, dtype=torch.float32),
        "last": _empty(1, HIDDEN, dtype=torch.float32), "logits": _empty(1, VOCAB, dtype=torch.float32),
        "probs": _empty(1, VOCAB, dtype=torch.float32),
    }


def _prepare_block(case, mk):
    n = case["n"]
    rows = lambda: _empty(n, WIDE)
    return {
        "n": n, "x": mk.normal(n, WIDE), "ctx": mk.normal(n, WIDE), "norm": mk.uniform(WIDE, lo=0.5, hi=1.5, dtype=torch.float16),
        "o_w": mk.normal(WIDE, WIDE, std=0.02), "up_w": mk.normal(WIDE_FF, WIDE, std=0.02), "down_w": mk.normal(WIDE, WIDE_FF, std=0.02),
        "o": rows(), "mid": rows(), "h": rows(), "up": _empty(n, WIDE_FF), "down": rows(), "y": rows(),
    }


def _prepare_rows(case, mk):
    n, H = case["n"], case["H"]
    rows = lambda dtype=torch.float16: _empty(n, H, dtype=dtype)
    return {
        "x32": mk.normal(n, H, dtype=torch.float32), "res": mk.normal(n, H), "w": mk.uniform(H, lo=0.5, hi=1.5, dtype=torch.float16),
        "ln": (mk.uniform(H, lo=0.5, hi=1.5), mk.uniform(H, lo=-0.2, hi=0.2)),
        "x": rows(), "sum": rows(), "h": rows(), "h32": rows(torch.float32), "normed": rows(), "kept": rows(), "probs": rows(),
    }


def prepare(case, seed):
    mk = _Make(seed)
    make = {"layer": _prepare_layer, "ends": _prepare_ends, "block": _prepare_block, "rows": _prepare_rows}[case["kind"]]
    return case["kind"], make(case, mk)


# --------------------------------------------------------------------------------------------- one pass
def _run_layer(s):
    n, past, q8 = s["n"], s["past"], s["q8"]
    if n == 1:
        mm, mm8 = ops.gemv, ops.gemv_q8
    else:
        mm, mm8 = ops.gemm, ops.gemm_q8
    project = mm8 if q8 else mm
    ops.cast(s["x"], s["x32"])
    ops.layer_norm(s["x32"], *s["ln1"], s["h1"])
    project(s["h1"], *s["qkv_w"], s["qkv_b"], s["qkv"])
    ops.split3(s["qkv"].view(n, HEADS, 3 * DIM), s["q"], s["k"], s["v"])
    ops.rotary(s["q"], s["cos"], s["sin"], s["qr"], s["m"])
    ops.rotary(s["k"], s["cos"], s["sin"], s["kr"], s["m"])
    ops.copy(s["kr"], s["keys"][past:])
    ops.copy(s["v"], s["values"][past:])
    ops.swap_axes(s["qr"], s["qh"])
    ops.swap_axes(s["keys"], s["kh"])
    ops.swap_axes(s["values"], s["vh"])
    ops.attn_scores(s["qh"], s["kh"], s["mask"], s["scores"], SCALE)
    ops.softmax(s["scores"], s["probs"])
    ops.attn_pv(s["probs"], s["vh"], s["ctx"])
    ops.swap_axes(s["ctx"], s["merged"])
    ops.layer_norm(s["x32"], *s["ln2"], s["h2"])
    project(s["h2"], *s["up_w"], s["up_b"], s["up"], epilogue=_lib.EPI_BIAS_GELU)
    project(s["up"], *s["down_w"], s["down_b"], s["down"])
    if q8:      # the 8-bit graph dequantises this one weight and runs the fp16 product with the residuals
        ops.decode_q8(*s["o_w"], s["o_f16"])
        o_w = s["o_f16"]
    else:
        o_w = s["o_w"][0]
    mm(s["merged"].view(n, HIDDEN), o_w, s["o_b"], s["y"], epilogue=_lib.EPI_BIAS_ADD2, res1=s["down"], res2=s["x"])
    return s["y"], s["keys"], s["values"], s["probs"], s["ctx"]


def _run_ends(s):
    if s["q8"]:
        ops.take_q8(*s["table"], s["ids"], s["embedded"])
    else:
        ops.take(*s["table"], s["ids"], s["embedded"])
    ops.attn_mask(s["mask"])
    ops.layer_norm_f32(s["hidden"], *s["ln"], s["normed"])
    ops.copy(s["normed"][s["n"] - 1:], s["last"])
    (ops.gemv_q8_f32 if s["q8"] else ops.gemv_f32)(s["last"], *s["head"], s["logits"])
    ops.softmax_temperature(s["logits"], s["temperature"], s["probs"])
    return s["embedded"], s["mask"], s["normed"], s["logits"], s["probs"]


def _run_block(s):
    mm = ops.gemv if s["n"] == 1 else ops.gemm
    mm(s["ctx"], s["o_w"], None, s["o"])
    ops.add(s["x"], s["o"], s["mid"])
    ops.rms_norm(s["mid"], s["norm"], s["h"])
    mm(s["h"], s["up_w"], None, s["up"])
    mm(s["up"], s["down_w"], None, s["down"])
    ops.add(s["mid"], s["down"], s["y"])
    return s["up"], s["y"]


def _run_rows(s):
    ops.cast(s["x32"], s["x"])
    ops.add(s["x"], s["res"], s["sum"])
    ops.rms_norm(s["sum"], s["w"], s["h"])
    ops.cast(s["h"], s["h32"])
    ops.layer_norm(s["h32"], *s["ln"], s["normed"])
    ops.copy(s["normed"], s["kept"])
    ops.softmax(s["kept"], s["probs"])
    return s["x"], s["sum"], s["h"], s["h32"], s["normed"], s["kept"], s["probs"]


def run(state):
    kind, s = state
    return {"layer": _run_layer, "ends": _run_ends, "block": _run_block, "rows": _run_rows}[kind](s)


# --------------------------------------------------------------------------------------------- what a pass amounts to
def _matmul(n, N, K, q8=False, streams=0):
    """Bytes and flops of one projection; `streams`: further [n, N] operands (residuals)."""
    w = N * K + 2 * N * (K // 32) if q8 else 2 * N * K
    return 2 * n * K + w + 2 * N + (1 + streams) * 2 * n * N, 2 * n * N * K


def work(case):
    kind, n = case["kind"], case["n"]
    if kind == "rows":
        H = case["H"]
        return {"bytes": n * H * (6 + 6 + 4 + 6 + 6 + 4 + 4) + 10 * H, "flops": 0}
    if kind == "block":
        parts = [_matmul(n, WIDE, WIDE), _matmul(n, WIDE_FF, WIDE), _matmul(n, WIDE, WIDE_FF)]
        return {"bytes": sum(p[0] for p in parts) + n * WIDE * (6 + 4 + 6) + 2 * WIDE, "flops": sum(p[1] for p in parts)}
    m, q8 = n + case["past"], case["q8"]
    if kind == "ends":
        row = HIDDEN + HIDDEN // 16 if q8 else 2 * HIDDEN
        head = VOCAB * (HIDDEN + HIDDEN // 8) if q8 else 4 * VOCAB * HIDDEN
        return {"bytes": n * (row + 2 * HIDDEN + 4) + 2 * n * m + 8 * n * HIDDEN + 8 * HIDDEN + 8 * HIDDEN + head + 12 * VOCAB,
                "flops": 2 * VOCAB * HIDDEN}
    act = n * HIDDEN
    parts = [_matmul(n, 3 * HIDDEN, HIDDEN, q8), _matmul(n, FF, HIDDEN, q8), _matmul(n, HIDDEN, FF, q8),
             _matmul(n, HIDDEN, HIDDEN, False, streams=2)]
    by = sum(p[0] for p in parts)
    by += 6 * act + 2 * (6 * act + 8 * HIDDEN)                         # cast, two layer norms
    by += 12 * act + 2 * 4 * act + 2 * 4 * act                         # split, rotary of q and k, the two appends
    by += 4 * act + 2 * 4 * m * HIDDEN + 4 * act                       # axis swaps of q, keys, values and the output
    by += 2 * act + 2 * m * HIDDEN + 2 * n * m + 4 * HEADS * n * m     # scores
    by += 6 * HEADS * n * m                                            # softmax
    by += 2 * HEADS * n * m + 2 * m * HIDDEN + 2 * act                 # P.V
    if q8:
        by += HIDDEN * HIDDEN + HIDDEN * HIDDEN // 16 + 2 * HIDDEN * HIDDEN
    return {"bytes": by, "flops": sum(p[1] for p in parts) + 4 * n * m * HIDDEN}


def tolerance(case):
    """Four times what the chains differ from the same chains with every sum in float64 (fp16 roundings at the same places)."""
    return {"layer": {"rel": 2e-3, "max": 4e-2}, "ends": {"rel": 4e-6, "max": 1e-5}, "block": {"rel": 8e-4, "max": 1e-2},
            "rows": {"rel": 1e-4, "max": 2e-2}}[case["kind"]]
