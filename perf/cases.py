"""Performance cases of the decode path: the work that a program on this framework has it do.

Single layers and blocks of the Qwen2.5-1.5B decode step and prompt prefill (quantised mat-vecs, batched
projections, split-KV attention), each through its public entry point, and whole engine calls (a batch-1 step, a
ragged-size batch of 16, a 2048-token prompt).  Sizes are those of the repository's benchmark, tests and model
configurations; ``draw`` spreads them over the ranges around these.
"""
from __future__ import annotations

import math
import os

import numpy as np
import torch

import vte_amd.core.hip_graph_executor as hge
from vte_amd.bridge import HIPRuntime
from vte_amd.core.hip_graph_executor import HIPGraphExecutor
from vte_amd.core.model_config import QWEN25_1P5B
from vte_amd.core.prefill import PrefillRunner
from vte_amd.core.rope_cache import build_rope_cache
from vte_amd.core.split_kv_attention import SplitKVAttentionDispatcher
from vte_amd.core.weights import PROJ, SyntheticQwen2, proj_shape
from vte_amd.kernels import kernels

HD = 128
EPS = 1e-6
BYTES = {"q4_k": (144, 256), "q6_k": (210, 256), "q8_0": (34, 32)}
MAX_SEQ = 2304  # cache rows of the step and prompt cases: a 2048-token prefix and room to decode


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest call: a square Q8_0 mat-vec of one token, fp32 in and out; launch and latency
        {"name": "gemv_q8_0_2048", "kind": "gemv", "fmt": "q8_0", "rows": 2048, "cols": 2048, "batch": 1, "io": "f32"},
        # the FFN gate (or up) projection of one decoded token, the mat-vec that a decode step runs most
        {"name": "gemv_q4_k_8960x1536", "kind": "gemv", "fmt": "q4_k", "rows": 8960, "cols": 1536, "batch": 1,
         "io": "f32"},
        # the LM head of one token: the largest matrix of the model, fp16 hidden state to fp32 logits
        {"name": "lm_head_q6_k", "kind": "gemv", "fmt": "q6_k", "rows": 151936, "cols": 1536, "batch": 1,
         "io": "f16f32"},
        # one projection of 16 decoded sequences, fp32 in and out
        {"name": "gemm_q4_k_16", "kind": "gemm", "fmt": "q4_k", "rows": 8960, "cols": 1536, "batch": 16, "io": "f32"},
        # one layer's decode attention of 16 sequences of very different lengths (128 to 8192 cached rows)
        {"name": "attn_ragged_16", "kind": "attn", "batch": 16, "low": 128, "high": 8192, "n_q": 12, "n_kv": 2},
        # one layer's attention of a 512-token prompt chunk that follows 1536 cached tokens
        {"name": "attn_prompt_512", "kind": "attn_prompt", "cols": 512, "start": 1536, "n_q": 12, "n_kv": 2},
        # the three blocks of a layer that read a prompt chunk's activations: q/k/v with RoPE and the K/V append,
        # gate/up with SwiGLU, and down with the residual add and the next layer's norm
        {"name": "qkv_prompt_512", "kind": "qkv", "cols": 512, "hidden": 1536, "n_q": 12, "n_kv": 2, "start": 1536},
        {"name": "ffn_prompt_512", "kind": "ffn", "cols": 512, "hidden": 1536, "ffn": 8960},
        {"name": "down_prompt_512", "kind": "proj", "cols": 512, "hidden": 1536, "in": 8960, "fmt": "q6_k"},
        # whole steps at a 2048-token prefix, as a serving loop calls them: tokens in, top-k candidates out
        {"name": "step_1", "kind": "step", "batch": 1, "prefix": 2048, "layers": 28},
        {"name": "step_16", "kind": "step", "batch": 16, "prefix": 2048, "layers": 28},
        # a whole prompt through the engine's prefill: the wait for the first token
        {"name": "prompt_2048", "kind": "prompt", "tokens": 2048, "start": 0, "layers": 28},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "gemm", "gemm", "attn", "attn", "attn_prompt", "attn_prompt", "qkv", "qkv",
                       "ffn", "ffn", "proj", "proj", "step", "prompt"])
    hidden = rng.choice([1536, 1536, 1536, 256 * _log(rng, 2, 14)])
    n_kv = rng.choice([1, 2, 2, 4])
    n_q = rng.choice([12, 12, 4 * n_kv, 7 * n_kv]) if n_kv != 1 else rng.choice([4, 6, 8])
    if kind == "gemv":
        fmt = rng.choice(["q4_k", "q6_k", "q8_0"])
        cols = (32 if fmt == "q8_0" else 256) * _log(rng, 2, 35) * (8 if fmt == "q8_0" and rng.random() < 0.7 else 1)
        return {"kind": kind, "fmt": fmt, "rows": _log(rng, 256, 151936), "cols": cols,
                "batch": rng.choice([1, 1, 2, 3, 4]), "io": rng.choice(["f32", "f16", "f16f32"])}
    if kind == "gemm":
        return {"kind": kind, "fmt": rng.choice(["q4_k", "q6_k"]), "rows": _log(rng, 256, 17920),
                "cols": rng.choice([1536, 256 * _log(rng, 2, 35)]), "batch": _log(rng, 3, 512),
                "io": rng.choice(["f32", "f16", "f16f32"])}
    if kind == "attn":
        high = _log(rng, 64, 32768)
        return {"kind": kind, "batch": rng.randint(1, 16), "low": max(1, high // rng.randint(1, 40)), "high": high,
                "n_q": n_q, "n_kv": n_kv}
    if kind == "attn_prompt":
        return {"kind": kind, "cols": _log(rng, 3, 512), "start": rng.choice([0, _log(rng, 1, 3500)]), "n_q": n_q,
                "n_kv": n_kv}
    if kind == "qkv":
        return {"kind": kind, "cols": _log(rng, 3, 512), "hidden": hidden, "n_q": n_q, "n_kv": n_kv,
                "start": rng.randint(0, 1700)}
    if kind == "ffn":
        return {"kind": kind, "cols": _log(rng, 3, 512), "hidden": hidden, "ffn": _log(rng, 500, 9500)}
    if kind == "proj":
        return {"kind": kind, "cols": _log(rng, 3, 512), "hidden": hidden, "in": 256 * _log(rng, 2, 37),
                "fmt": rng.choice(["q4_k", "q6_k"])}
    if kind == "step":
        return {"kind": kind, "batch": rng.randint(1, 16), "prefix": _log(rng, 1, MAX_SEQ - 1), "layers": 28}
    return {"kind": kind, "tokens": _log(rng, 4, 2048), "start": rng.randint(0, MAX_SEQ - 2048), "layers": 28}


# ------------------------------------------------------------------------------------------------ inputs
_HIP = None


def _hip():
    """The program's one runtime, on the HIP library that torch has loaded."""
    global _HIP
    if _HIP is None:
        lib = os.path.join(os.path.dirname(torch.__file__), "lib", "libamdhip64.so")
        _HIP = HIPRuntime(lib if os.path.exists(lib) else None)
        if not _HIP.initialize():
            raise RuntimeError("no GPU visible")
    return _HIP


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _blocks(fmt, rows, cols, g):
    """A random rows x cols matrix as raw GGUF blocks: zero-mean weights of standard deviation about 1/sqrt(cols)."""
    size, per = BYTES[fmt]
    nb = rows * cols // per
    b = torch.randint(0, 256, (nb, size), dtype=torch.uint8, device="cuda", generator=g)
    r = 0.5 + torch.rand(nb, 1, device="cuda", generator=g)
    root = math.sqrt(cols)
    if fmt == "q4_k":
        d = r / (200.0 * root)
        b[:, 0:2] = d.half().view(torch.uint8)
        b[:, 2:4] = (7.5 * d).half().view(torch.uint8)
    elif fmt == "q6_k":
        sc = torch.randint(-32, 32, (nb, 16), dtype=torch.int8, device="cuda", generator=g)
        b[:, 192:208] = sc.view(torch.uint8)
        b[:, 208:210] = (r / (340.0 * root)).half().view(torch.uint8)
    else:
        b[:, 0:2] = (r / (73.0 * root)).half().view(torch.uint8)
    return b.reshape(-1)


def _normal(g, shape, scale=1.0, dtype=torch.float16):
    return (scale * torch.randn(shape, device="cuda", generator=g)).to(dtype)


def _with_slack(t):
    """A copy of t followed by 256 readable bytes, as the framework's own device arrays have."""
    b = torch.zeros(t.numel() * t.element_size() + 256, dtype=torch.uint8, device="cuda")
    b = b[:-256].view(t.dtype).reshape(t.shape)
    return b.copy_(t)


def _splits_of(case):
    return hge.splitk_splits(case["in"])


def _lengths(case):
    """Cached rows of each sequence of an attention case: evenly spread from low to high."""
    B = case["batch"]
    return [case["high"] if B == 1 else case["low"] + (case["high"] - case["low"]) * b // (B - 1) for b in range(B)]


def _inputs(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        it = torch.float32 if case["io"] == "f32" else torch.float16
        return {"x": _normal(g, (case["batch"], case["cols"]), dtype=it),
                "w": _blocks(case["fmt"], case["rows"], case["cols"], g)}
    if kind == "attn":
        B, nkv = case["batch"], case["n_kv"]
        lens = torch.tensor(_lengths(case), dtype=torch.int32, device="cuda")
        lens = lens[torch.randperm(B, device="cuda", generator=g)]
        return {"q": _normal(g, (B, case["n_q"], HD)), "k": _normal(g, (B, case["high"], nkv, HD), 0.5),
                "v": _normal(g, (B, case["high"], nkv, HD), 0.5), "off": (lens - 1).contiguous()}
    if kind == "attn_prompt":
        rows = case["start"] + case["cols"]
        off = torch.arange(case["start"], rows, dtype=torch.int32, device="cuda")
        return {"q": _normal(g, (case["cols"], case["n_q"], HD)), "k": _normal(g, (rows, case["n_kv"], HD), 0.5),
                "v": _normal(g, (rows, case["n_kv"], HD), 0.5), "off": off}
    if kind == "qkv":
        H, qd, kd = case["hidden"], case["n_q"] * HD, case["n_kv"] * HD
        off = torch.arange(case["start"], case["start"] + case["cols"], dtype=torch.int32, device="cuda")
        cos, sin = build_rope_cache(case["start"] + case["cols"], HD, QWEN25_1P5B.rope_theta)
        return {"x": _normal(g, (case["cols"], H)), "wq": _blocks("q4_k", qd, H, g), "wk": _blocks("q4_k", kd, H, g),
                "wv": _blocks("q6_k", kd, H, g), "bq": _normal(g, qd, 0.1), "bk": _normal(g, kd, 0.1),
                "bv": _normal(g, kd, 0.1), "off": off, "cos": torch.from_numpy(np.ascontiguousarray(cos)).cuda(),
                "sin": torch.from_numpy(np.ascontiguousarray(sin)).cuda()}
    if kind == "ffn":
        H, F = case["hidden"], case["ffn"]
        return {"x": _normal(g, (case["cols"], H)), "wg": _blocks("q4_k", F, H, g), "wu": _blocks("q4_k", F, H, g)}
    H, C = case["hidden"], case["cols"]  # proj
    return {"x": _normal(g, (C, case["in"])), "w": _blocks(case["fmt"], H, case["in"], g), "h": _normal(g, (C, H)),
            "norm": (1 + 0.1 * torch.randn(H, device="cuda", generator=g)).half()}


def _model(case, seed):
    return SyntheticQwen2(QWEN25_1P5B.with_(n_layers=case["layers"], max_seq=MAX_SEQ), seed=int(seed) % (1 << 31))


def _engine_inputs(case, seed):
    """Tokens, and the K/V rows of every layer that are in the cache before the call ([B][rows][n_kv][hd])."""
    cfg, g = QWEN25_1P5B, _gen(seed)
    if case["kind"] == "step":
        B, rows = case["batch"], case["prefix"]
        toks = torch.randint(0, cfg.vocab, (B,), device="cuda", generator=g).tolist()
    else:
        B, rows = 1, case["start"]
        toks = torch.randint(0, cfg.vocab, (case["tokens"],), device="cuda", generator=g).tolist()
    kv = [(_normal(g, (B, rows, cfg.n_kv, HD), 0.5), _normal(g, (B, rows, cfg.n_kv, HD), 0.5))
          for _ in range(case["layers"])]
    return toks, kv


class _Owner:
    """Closes an executor (or frees a dispatcher's scratch) once no state or output refers to it."""

    def __init__(self, thing):
        self.thing = thing

    def __del__(self):
        try:
            _hip().synchronize()
            if isinstance(self.thing, HIPGraphExecutor):
                self.thing.close()
            else:
                for a in (self.thing.part_m, self.thing.part_l, self.thing.part_o, self.thing.counters):
                    a.free()
        except Exception:  # the process is ending
            pass


class _Memory:
    """Device memory of an executor, for torch.as_tensor."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (int(ptr), False), "shape": tuple(shape), "typestr": typestr,
                                         "version": 2}


def _view(owner, ptr, shape, typestr):
    return torch.as_tensor(_Memory(owner, ptr, shape, typestr), device="cuda")


def prepare(case, seed):
    hip, K, kind = _hip(), kernels(), case["kind"]
    if kind in ("step", "prompt"):
        return _prepare_engine(case, seed)
    s = {n: _with_slack(t) for n, t in _inputs(case, seed).items()}
    p = {n: t.data_ptr() for n, t in s.items()}
    if kind in ("gemv", "gemm"):
        out_f32 = case["io"] != "f16"
        s["y"] = torch.zeros(case["batch"], case["rows"], device="cuda",
                             dtype=torch.float32 if out_f32 else torch.float16)
        call = K.gemv if kind == "gemv" else K.gemm_mfma
        args = (case["fmt"], p["x"], p["w"], s["y"].data_ptr(), case["batch"], case["cols"], case["rows"])
        kw = {"in_dtype": "f32" if case["io"] == "f32" else "f16", "out_dtype": "f32" if out_f32 else "f16"}
        s["run"], s["out"] = (lambda: call(*args, stream=hip.stream, **kw)), s["y"]
    elif kind in ("attn", "attn_prompt"):
        B = case["batch"] if kind == "attn" else case["cols"]
        rows = case["high"] if kind == "attn" else case["start"] + case["cols"]
        stride = rows * case["n_kv"] * HD if kind == "attn" else 0
        s["o"] = torch.zeros(B, case["n_q"], HD, dtype=torch.float16, device="cuda")
        d = SplitKVAttentionDispatcher(hip, case["n_q"], case["n_kv"], HD, rows, B)
        s["owner"], po = _Owner(d), s["o"].data_ptr()
        s["run"] = lambda: d.launch(p["q"], p["k"], p["v"], po, p["off"], stride, dtype="f16", batch=B)
        s["out"] = s["o"]
    elif kind == "qkv":
        C, rows, nkv = case["cols"], case["start"] + case["cols"], case["n_kv"]
        s["q"] = torch.zeros(C, case["n_q"] * HD, dtype=torch.float16, device="cuda")
        s["kc"] = torch.zeros(rows, nkv, HD, dtype=torch.float16, device="cuda")
        s["vc"] = torch.zeros(rows, nkv, HD, dtype=torch.float16, device="cuda")
        o = [s[n].data_ptr() for n in ("q", "kc", "vc")]
        s["run"] = lambda: K.attn_in(p["x"], None, EPS, p["wq"], p["bq"], "q4_k", p["wk"], p["bk"], "q4_k", p["wv"],
                                     p["bv"], "q6_k", o[0], o[1], o[2], p["off"], 0, p["cos"], p["sin"], C,
                                     case["hidden"], case["n_q"], nkv, HD, stream=hip.stream)
        s["out"] = [s["q"], s["kc"], s["vc"]]
    elif kind == "ffn":
        s["a"] = torch.zeros(case["cols"], case["ffn"], dtype=torch.float16, device="cuda")
        po = s["a"].data_ptr()
        s["run"] = lambda: K.ffn_in(p["x"], None, EPS, p["wg"], p["wu"], "q4_k", po, case["cols"], case["hidden"],
                                    case["ffn"], stream=hip.stream)
        s["out"] = s["a"]
    else:
        C, H, n = case["cols"], case["hidden"], _splits_of(case)
        s["part"] = torch.zeros(n, C, H, dtype=torch.float32, device="cuda")
        s["ho"], s["xn"] = torch.zeros_like(s["h"]), torch.zeros_like(s["h"])
        o = [s[k].data_ptr() for k in ("part", "ho", "xn")]

        def both():
            K.gemm_mfma_splitk(case["fmt"], p["x"], p["w"], o[0], C, case["in"], H, n, stream=hip.stream)
            K.add_rmsnorm(p["h"], o[0], n, p["norm"], o[1], o[2], C, H, EPS, stream=hip.stream)

        s["run"], s["out"] = both, [s["ho"], s["xn"]]
    torch.cuda.synchronize()
    return s


def _prepare_engine(case, seed):
    hip, model = _hip(), _model(case, seed)
    cfg = model.cfg
    toks, kv = _engine_inputs(case, seed)
    B, step = (case["batch"], True) if case["kind"] == "step" else (1, False)
    ex = HIPGraphExecutor(hip, model, batch_size=B, max_seq=MAX_SEQ, top_k=40)
    owner = _Owner(ex)
    at, n = (case["prefix"], 1) if step else (case["start"], case["tokens"])
    full = [np.zeros((B, MAX_SEQ, cfg.n_kv, HD), np.float16) for _ in range(2)]
    rows = []
    for L, pair in enumerate(kv):
        for f, t in zip(full, pair):
            f[:, :at] = t.cpu().numpy()
        ex.upload_kv(L, *full)
        rows += [_view(owner, c.ptr, (B, MAX_SEQ, cfg.n_kv, HD), "<f2")[:, at:at + n] for c in (ex.k_cache[L],
                                                                                              ex.v_cache[L])]
    s = {"owner": owner, "rows": rows}
    if step:
        off = [at] * B
        logits = _view(owner, ex.logits.ptr, (B, cfg.vocab), "<f4")

        def run():
            ex.execute_decode_batch(toks, off)
            val, _ = ex.read_topk()
            return {"logits": logits, "top": val, "rows": rows}
    else:
        runner = PrefillRunner(ex)

        def run():
            sub = runner.prefill(toks, seq=0, start=at)
            return {"logits": _view(owner, sub.logits.ptr, (1, cfg.vocab), "<f4"), "rows": rows}
    s["run"], s["out"] = run, None
    torch.cuda.synchronize()
    return s


def run(state):
    r = state["run"]()
    return r if state["out"] is None else state["out"]


# ------------------------------------------------------------------------------------------------ what it takes
def _matrix(fmt, rows, cols):
    size, per = BYTES[fmt]
    return rows * (cols // per) * size


def _layer_work(case):
    """(weight bytes, weights) of the layers and the LM head of an engine case."""
    cfg = QWEN25_1P5B
    b = n = 0
    for L in range(case["layers"]):
        for p in PROJ:
            o, i = proj_shape(cfg, p)
            b += _matrix("q6_k" if p == "v" or (p == "down" and L % 2 == 0) else "q4_k", o, i)
            n += o * i
    return b, n


def work(case):
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        M, N, K = case["batch"], case["rows"], case["cols"]
        return {"bytes": _matrix(case["fmt"], N, K) + M * K * (4 if case["io"] == "f32" else 2)
                + M * N * (2 if case["io"] == "f16" else 4), "flops": 2 * M * N * K}
    if kind == "attn":
        tot = sum(_lengths(case))
        return {"bytes": tot * case["n_kv"] * HD * 4 + 4 * case["batch"] * case["n_q"] * HD,
                "flops": 4 * tot * case["n_q"] * HD}
    if kind == "attn_prompt":
        C, s = case["cols"], case["start"]
        return {"bytes": (s + C) * case["n_kv"] * HD * 4 + 4 * C * case["n_q"] * HD,
                "flops": 4 * HD * case["n_q"] * (C * s + C * (C + 1) // 2)}
    if kind == "qkv":
        C, H, qd, kd = case["cols"], case["hidden"], case["n_q"] * HD, case["n_kv"] * HD
        return {"bytes": _matrix("q4_k", qd + kd, H) + _matrix("q6_k", kd, H) + 2 * C * (H + qd + 2 * kd + 2 * HD),
                "flops": 2 * C * H * (qd + 2 * kd)}
    if kind == "ffn":
        C, H, F = case["cols"], case["hidden"], case["ffn"]
        return {"bytes": 2 * _matrix("q4_k", F, H) + 2 * C * (H + F), "flops": 4 * C * H * F}
    if kind == "proj":
        C, H, I = case["cols"], case["hidden"], case["in"]
        return {"bytes": _matrix(case["fmt"], H, I) + 2 * C * (I + 3 * H), "flops": 2 * C * H * I}
    cfg = QWEN25_1P5B
    wb, wn = _layer_work(case)
    head = _matrix("q6_k", cfg.vocab, cfg.hidden)
    if kind == "step":
        B, kv = case["batch"], case["batch"] * (case["prefix"] + 1)
        out = 1
        cols = B
    else:
        n, s = case["tokens"], case["start"]
        B, cols, out, kv = n, n, 0, s + n
    rows = B if out else 1  # logits rows
    pairs = kv if kind == "step" else cols * case["start"] + cols * (cols + 1) // 2
    return {"bytes": wb + head + case["layers"] * (kv + cols) * cfg.kv_dim * 4 + rows * cfg.vocab * 4,
            "flops": 2 * cols * wn + 2 * rows * cfg.vocab * cfg.hidden + 4 * pairs * cfg.q_dim * case["layers"]}


def tolerance(case):
    kind = case["kind"]
    if kind in ("gemv", "gemm"):
        if case["io"] == "f16f32":
            return {"rel": 1e-5}  # fp32 sums of exact products
        return {"rel": 1e-3}  # fp32 activations enter the products as fp16, or the results are fp16
    if kind in ("attn", "attn_prompt"):
        return {"rel": 1.2e-3}  # fp16 probabilities into P.V, fp16 results
    if kind in ("qkv", "ffn", "proj"):
        return {"rel": 1.5e-3}  # fp16 results
    # 28 layers of fp16 rounding points: two correct summation orders drift apart by about 4e-3 to 9e-3
    return {"rel": 0.02, "max": 0.5, "differ": 0.01}


# ------------------------------------------------------------------------------------------------ in 64 bits
def _dequant(fmt, raw, rows, cols):
    """[rows][cols] float64 values of raw GGUF blocks."""
    size, per = BYTES[fmt]
    b = raw.reshape(-1, size)
    half = lambda lo: b[:, lo:lo + 2].contiguous().view(torch.float16).double()
    if fmt == "q8_0":
        w = half(0) * b[:, 2:].contiguous().view(torch.int8).double()
    elif fmt == "q4_k":
        s = b[:, 4:16].to(torch.int32)
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).double()
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).double()
        q = b[:, 16:].reshape(-1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
        w = half(0)[:, :, None] * sc[:, :, None] * q - half(2)[:, :, None] * mn[:, :, None]
    else:
        ql = b[:, :128].reshape(-1, 2, 2, 32).to(torch.int32)
        qh = b[:, 128:192].reshape(-1, 2, 1, 32).to(torch.int32)
        lo = torch.cat([ql & 15, ql >> 4], 2)  # quarters 0, 1 (low nibbles) and 2, 3 (high nibbles)
        hi = torch.cat([(qh >> (2 * i)) & 3 for i in range(4)], 2)
        q = ((lo | (hi << 4)) - 32).double().reshape(-1, 16, 16)
        w = half(208)[:, :, None] * b[:, 192:208].contiguous().view(torch.int8).double()[:, :, None] * q
    return w.reshape(rows, cols)


def _linear(x, fmt, raw, rows):
    """x [M][cols] float64 times the transposed matrix, row blocks at a time."""
    cols = x.shape[1]
    raw = raw.reshape(rows, -1)
    return torch.cat([x @ _dequant(fmt, r, r.shape[0], cols).T for r in raw.split(16384)], 1)


def _norm(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, cos, sin):
    """x [M][heads][128] rotated by the fp16 table rows cos/sin [M][128] (pairs d, d + 64)."""
    c, s = cos.double()[:, None, :64], sin.double()[:, None, :64]
    a, b = x[..., :64], x[..., 64:]
    return torch.cat([a * c - b * s, a * s + b * c], -1)


def _attend(q, k, v, lens):
    """q [M][n_q][128] against one cache k/v [rows][n_kv][128], column m over its first lens[m] rows."""
    M, nq, _ = q.shape
    nkv = k.shape[1]
    out = torch.empty_like(q)
    seen = torch.arange(k.shape[0], device="cuda")[None, :]
    for h in range(nq):
        kh = h // (nq // nkv)
        s = q[:, h] @ k[:, kh].T / math.sqrt(HD)
        s = s.masked_fill(seen >= lens[:, None], -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, kh]
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("step", "prompt"):
        return _exact_engine(case, seed)
    s = _inputs(case, seed)
    if kind in ("gemv", "gemm"):
        return _linear(s["x"].double(), case["fmt"], s["w"], case["rows"])
    if kind == "attn":
        lens = s["off"].long() + 1
        return torch.cat([_attend(s["q"][b:b + 1].double(), s["k"][b].double(), s["v"][b].double(), lens[b:b + 1])
                          for b in range(case["batch"])])
    if kind == "attn_prompt":
        return _attend(s["q"].double(), s["k"].double(), s["v"].double(), s["off"].long() + 1)
    if kind == "qkv":
        x, C, nq, nkv, at = s["x"].double(), case["cols"], case["n_q"], case["n_kv"], s["off"].long()
        q = (_linear(x, "q4_k", s["wq"], nq * HD) + s["bq"].double()).reshape(C, nq, HD)
        k = (_linear(x, "q4_k", s["wk"], nkv * HD) + s["bk"].double()).reshape(C, nkv, HD)
        v = (_linear(x, "q6_k", s["wv"], nkv * HD) + s["bv"].double()).reshape(C, nkv, HD)
        kc = torch.zeros(case["start"] + C, nkv, HD, dtype=torch.float64, device="cuda")
        vc = torch.zeros_like(kc)
        kc[at], vc[at] = _rope(k, s["cos"][at], s["sin"][at]), v
        return [_rope(q, s["cos"][at], s["sin"][at]).reshape(C, nq * HD), kc, vc]
    if kind == "ffn":
        g, u = (_linear(s["x"].double(), "q4_k", s[n], case["ffn"]) for n in ("wg", "wu"))
        return torch.nn.functional.silu(g) * u
    h = s["h"].double() + _linear(s["x"].double(), case["fmt"], s["w"], case["hidden"])
    return [h, _norm(h, s["norm"])]


def _exact_engine(case, seed):
    model = _model(case, seed)
    cfg = model.cfg
    toks, kv = _engine_inputs(case, seed)
    step = case["kind"] == "step"
    at, M = (case["prefix"], case["batch"]) if step else (case["start"], case["tokens"])
    dev = lambda a: torch.from_numpy(a).cuda()
    size, per = BYTES["q6_k"]
    rows = dev(model.token_embd).reshape(cfg.vocab, -1)[torch.tensor(toks, device="cuda")]
    h = _dequant("q6_k", rows.contiguous(), M, cfg.hidden)
    pos = torch.full((M,), at, device="cuda") if step else torch.arange(at, at + M, device="cuda")
    inv = torch.tensor(cfg.rope_theta, dtype=torch.float64, device="cuda") ** (
        -torch.arange(0, HD, 2, device="cuda", dtype=torch.float64) / HD)
    ang = (pos[:, None].double() * inv).repeat(1, 2)
    cos, sin = ang.cos().half(), ang.sin().half()
    new = []
    for lw, (kp, vp) in zip(model.layers, kv):
        lin = lambda x, p: _linear(x, lw[p + "_fmt"], dev(lw[p]), proj_shape(cfg, p)[0])
        x = _norm(h, dev(lw["attn_norm"]))
        q = _rope((lin(x, "q") + dev(lw["q_bias"]).double()).reshape(M, cfg.n_q, HD), cos, sin)
        k = _rope((lin(x, "k") + dev(lw["k_bias"]).double()).reshape(M, cfg.n_kv, HD), cos, sin)
        v = (lin(x, "v") + dev(lw["v_bias"]).double()).reshape(M, cfg.n_kv, HD)
        new += [k[:, None], v[:, None]] if step else [k[None], v[None]]
        if step:
            one = torch.full((1,), at + 1, device="cuda")
            a = torch.cat([_attend(q[b:b + 1], torch.cat([kp[b].double(), k[b:b + 1]]),
                                   torch.cat([vp[b].double(), v[b:b + 1]]), one) for b in range(M)])
        else:
            a = _attend(q, torch.cat([kp[0].double(), k]), torch.cat([vp[0].double(), v]), pos + 1)
        h = h + lin(a.reshape(M, -1), "o")
        x = _norm(h, dev(lw["ffn_norm"]))
        h = h + lin(torch.nn.functional.silu(lin(x, "gate")) * lin(x, "up"), "down")
    out = h if step else h[-1:]
    logits = _linear(_norm(out, dev(model.output_norm)), model.lm_head_fmt, dev(model.lm_head), cfg.vocab)
    if step:
        return {"logits": logits, "top": None, "rows": new}
    return {"logits": logits, "rows": new}
