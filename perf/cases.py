"""Timed cases of the decode backend: the calls a serving program makes.

Every case goes through the package's public entry points (Matrix, the C ABI
bound in pagoda_amd._lib, Model / Session). Weights, activations and KV are
random, in the formats and distributions of the real path: N(0, 0.02) weights
quantized to MLX affine-8 (group 64), Q4_K or Q6_K; unit-variance activation
rows as an RMSNorm leaves them. Kinds of case (`kind`):

  mlp    the hybrid model's feed-forward block over A8 weights: activations
         prepared once, fused gate/up SwiGLU, down projection plus residual.
         1 row is a single user's decode step, 32 a served batch, hundreds to
         thousands a prompt.
  kq     one projection of a GGUF model with dequantized weights (the GPU-side
         arithmetic): f16 or f32 rows against a Q4_K / Q6_K matrix.
  q8     the same projection in the GGUF path's default arithmetic (activation
         rows quantized to Q8_K, integer block dots): a decode row, or the
         rows of a prompt.
  gdn    the Gated-DeltaNet recurrence of one layer: a decode batch (one or a
         few tokens per sequence) or a prefill (ragged prompts).
  attn   paged GQA attention of one layer: a decode batch over ragged
         contexts, or the rows of prompt chunks.
  qwen2  a whole request on the 0.5B Qwen2 architecture (Q4_K / Q6_K): begin a
         session, prefill the prompt, decode fed tokens; logits of the prompt
         and of the last step.
  hybrid a whole batch on the 27B-class hybrid's layer widths at reduced
         depth: ragged prompts in one step, then batched decode steps; logits
         of the prompt step and of the last step.
"""
from __future__ import annotations

import ctypes as C
import math
from dataclasses import replace

import numpy as np
import torch

from pagoda_amd import Device, Matrix
from pagoda_amd._lib import call
from pagoda_amd.engine import QWEN2_05B, QWEN35_27B, Model
from pagoda_amd.matrix import FMT_Q4K, FMT_Q6K, act_bytes, act_prep_dev

BLOCK = 16       # positions per KV page
GDN_DIM = 128    # key and value width of a Gated-DeltaNet head


def listed() -> list[dict]:
    return [
        # the smallest call: the 0.5B model's key / value projection of one decode row, f16 activations
        {"name": "kq_q4k_kv_1", "kind": "kq", "fmt": "q4k", "n": 256, "k": 896, "rows": 1, "f16": True},
        # its tied embedding as lm_head for a decode batch
        {"name": "kq_q6k_head_32", "kind": "kq", "fmt": "q6k", "n": 151936, "k": 896, "rows": 32, "f16": True},
        # a feed-forward matrix of the same model in the default arithmetic: one decode row with the residual
        {"name": "q8_q6k_down_1", "kind": "q8", "fmt": "q6k", "n": 896, "k": 4864, "rows": 1, "res": True},
        # and over a prompt of a few hundred tokens
        {"name": "q8_q4k_up_333", "kind": "q8", "fmt": "q4k", "n": 4864, "k": 896, "rows": 333, "res": False},
        # the 27B-class feed-forward block: one user, a served batch, a long prompt
        {"name": "mlp_1", "kind": "mlp", "hidden": 5120, "inter": 17408, "rows": 1},
        {"name": "mlp_32", "kind": "mlp", "hidden": 5120, "inter": 17408, "rows": 32},
        {"name": "mlp_2048", "kind": "mlp", "hidden": 5120, "inter": 17408, "rows": 2048},
        # a decode batch's recurrence, and the ragged prompts of a few requests
        {"name": "gdn_step_32", "kind": "gdn", "k_heads": 16, "v_heads": 32, "nseq": 32, "shortest": 1, "longest": 1},
        {"name": "gdn_prefill_3", "kind": "gdn", "k_heads": 16, "v_heads": 32, "nseq": 3, "shortest": 211,
         "longest": 1500},
        # decode attention of a batch whose contexts range over two decades, and a prompt chunk on a cached prefix
        {"name": "attn_decode_32", "kind": "attn", "heads": 24, "kv_heads": 4, "head_dim": 256, "nseq": 32,
         "tokens": 1, "shortest": 40, "longest": 4000, "gate": True},
        # whole calls: an 81-token prompt and 32 decoded tokens on the 0.5B model
        {"name": "qwen2_request", "kind": "qwen2", "prompt": 81, "gen": 32},
        # sixteen chat-sized prompts and eight decode steps on 8 layers of the hybrid (6 recurrent, 2 attention)
        {"name": "hybrid_batch", "kind": "hybrid", "layers": 8, "nseq": 16, "shortest": 19, "longest": 200, "gen": 8},
    ]


def _log(rng, lo: int, hi: int, step: int = 1) -> int:
    """A multiple of step, spread over the logarithm of [lo, hi]."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng) -> dict:
    kind = rng.choice(["mlp", "kq", "q8", "gdn", "gdn", "attn", "attn", "qwen2", "hybrid"])
    if kind == "mlp":
        return {"kind": kind, "hidden": _log(rng, 1024, 5120, 64), "inter": _log(rng, 2048, 17408, 64),
                "rows": _log(rng, 1, 2048)}
    if kind in ("kq", "q8"):
        fmt = rng.choice(["q4k", "q6k"])
        n = _log(rng, 256, 151936) if rng.random() < 0.2 else _log(rng, 256, 18944)
        k = _log(rng, 896, 8960, 128 if fmt == "q6k" else 64)
        if n > 18944:
            k = 896
        if kind == "kq":
            return {"kind": kind, "fmt": fmt, "n": n, "k": k, "rows": _log(rng, 1, 64), "f16": rng.random() < 0.5}
        return {"kind": kind, "fmt": fmt, "n": n, "k": k, "rows": _log(rng, 1, 32 if n > 18944 else 1024),
                "res": rng.random() < 0.5}
    if kind == "gdn":
        heads = rng.choice([(16, 32), (16, 16), (8, 32), (16, 48)])
        if rng.random() < 0.5:  # decode and verify batches
            lo = rng.randint(1, 4)
            return {"kind": kind, "k_heads": heads[0], "v_heads": heads[1], "nseq": _log(rng, 1, 64),
                    "shortest": lo, "longest": rng.randint(lo, 4)}
        lo = _log(rng, 5, 600)
        return {"kind": kind, "k_heads": heads[0], "v_heads": heads[1], "nseq": _log(rng, 1, 8), "shortest": lo,
                "longest": _log(rng, lo, 2000)}
    if kind == "attn":
        heads, kv, hd = rng.choice([(24, 4, 256), (14, 2, 64), (16, 2, 256), (28, 4, 128)])
        if rng.random() < 0.6:
            return {"kind": kind, "heads": heads, "kv_heads": kv, "head_dim": hd, "nseq": _log(rng, 1, 64),
                    "tokens": rng.choice([1, 1, 4]), "shortest": _log(rng, 16, 400), "longest": _log(rng, 400, 4000),
                    "gate": hd == 256}
        tokens = _log(rng, 16, 400)
        return {"kind": kind, "heads": heads, "kv_heads": kv, "head_dim": hd, "nseq": rng.randint(1, 2),
                "tokens": tokens, "shortest": tokens, "longest": _log(rng, tokens, 2000), "gate": hd == 256}
    if kind == "qwen2":
        return {"kind": kind, "prompt": _log(rng, 1, 400), "gen": _log(rng, 1, 32)}
    lo = _log(rng, 4, 100)
    return {"kind": kind, "layers": rng.choice([4, 8]), "nseq": _log(rng, 1, 16), "shortest": lo,
            "longest": _log(rng, lo, 200), "gen": rng.randint(1, 8)}


# ---- inputs -------------------------------------------------------------------

_dev: Device | None = None


def _device() -> Device:
    """The program's one device handle."""
    global _dev
    if _dev is None:
        _dev = Device("hip")
    return _dev


def _gen(seed: int, stream: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1_000_003 + stream) & 0x7FFFFFFFFFFFFFFF)
    return g


def _normal(shape, seed: int, stream: int, scale: float = 1.0) -> torch.Tensor:
    return torch.randn(shape, generator=_gen(seed, stream), device="cuda") * scale


def _spread(lo: int, hi: int, n: int, seed: int) -> list[int]:
    """n whole numbers over the logarithm of [lo, hi], both ends among them, in a seeded order."""
    v = [int(round(math.exp(math.log(lo) + (math.log(hi) - math.log(lo)) * (i / max(1, n - 1))))) for i in range(n)]
    if n == 1:
        v = [hi]
    return [v[i] for i in np.random.default_rng(seed).permutation(n)]


def _a8_weights(n: int, k: int, seed: int, stream: int):
    """MLX affine-8 of N(0, 0.02) weights: u8 codes [n, k], bf16 scales and biases [n, k / 64]."""
    w = _normal((n, k // 64, 64), seed, stream, 0.02)
    lo, hi = w.amin(-1, keepdim=True), w.amax(-1, keepdim=True)
    scale = ((hi - lo) / 255).bfloat16()
    bias = lo.bfloat16()
    codes = ((w - bias.float()) / scale.float()).round().clamp(0, 255).to(torch.uint8)
    return codes.reshape(n, k), scale.reshape(n, -1), bias.reshape(n, -1)


def _a8_matrix(dev: Device, parts) -> Matrix:
    codes, scale, bias = parts
    n, k = codes.shape

    def u16(t):
        return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)

    return Matrix.upload_a8(dev, codes.cpu().numpy().view(np.uint32), u16(scale), u16(bias), n, k)


def _a8_dequant(parts) -> torch.Tensor:
    codes, scale, bias = parts
    n, k = codes.shape
    w = codes.reshape(n, -1, 64).double() * scale.double()[..., None] + bias.double()[..., None]
    return w.reshape(n, k)


def _f16_bytes(t: torch.Tensor) -> torch.Tensor:
    return t.half().contiguous().view(torch.uint8).reshape(*t.shape, 2)


def _padded_weights(n: int, k: int, seed: int) -> torch.Tensor:
    """N(0, 0.02) rows of k weights, padded with zeros to whole 256-weight blocks: [n, blocks, 256]."""
    nsb = (k + 255) // 256
    w = torch.zeros((n, nsb * 256), device="cuda")
    w[:, :k] = _normal((n, k), seed, 1, 0.02)
    return w.reshape(n, nsb, 256)


def _q4k(n: int, k: int, seed: int):
    """GGML block_q4_K bytes [n, blocks, 144], and a function giving the float64 weights [n, k]."""
    w = _padded_weights(n, k, seed).reshape(n, -1, 8, 32)
    low = (-w.amin(-1)).clamp_min(0)
    step = (w.amax(-1) + low) / 15
    d = (step.amax(-1) / 63).half()
    dmin = (low.amax(-1) / 63).half()
    sc = (step / d.float()[..., None]).nan_to_num(0.0, 0.0, 0.0).round().clamp(0, 63)
    mn = (low / dmin.float()[..., None]).nan_to_num(0.0, 0.0, 0.0).round().clamp(0, 63)
    scale, off = d.float()[..., None] * sc, dmin.float()[..., None] * mn
    q = ((w + off[..., None]) / scale[..., None]).nan_to_num(0.0, 0.0, 0.0).round().clamp(0, 15)
    s, m, qi = sc.to(torch.uint8), mn.to(torch.uint8), q.to(torch.uint8)
    packed = torch.cat([s[..., :4] | ((s[..., 4:] >> 4) << 6), m[..., :4] | ((m[..., 4:] >> 4) << 6),
                        (s[..., 4:] & 15) | ((m[..., 4:] & 15) << 4)], -1)
    nib = (qi[..., 0::2, :] | (qi[..., 1::2, :] << 4)).reshape(*d.shape, 128)
    blocks = torch.cat([_f16_bytes(d), _f16_bytes(dmin), packed, nib], -1)

    def weights() -> torch.Tensor:
        v = (d.double()[..., None] * sc.double())[..., None] * q.double()
        return (v - (dmin.double()[..., None] * mn.double())[..., None]).reshape(n, -1)[:, :k]

    return blocks, weights


def _q6k(n: int, k: int, seed: int):
    """GGML block_q6_K bytes [n, blocks, 210], and a function giving the float64 weights [n, k]."""
    w = _padded_weights(n, k, seed).reshape(n, -1, 16, 16)
    step = w.abs().amax(-1) / 31
    d = (step.amax(-1) / 127).half()
    sc = (step / d.float()[..., None]).nan_to_num(0.0, 0.0, 0.0).round().clamp(-128, 127)
    scale = d.float()[..., None] * sc
    q = (w / scale[..., None]).nan_to_num(0.0, 0.0, 0.0).round().clamp(-32, 31)
    u = (q + 32).to(torch.uint8).reshape(n, -1, 2, 4, 32)  # [half][quarter][element]
    ql = torch.stack([(u[..., 0, :] & 15) | ((u[..., 2, :] & 15) << 4),
                      (u[..., 1, :] & 15) | ((u[..., 3, :] & 15) << 4)], -2).reshape(*d.shape, 128)
    hi = u >> 4
    qh = (hi[..., 0, :] | (hi[..., 1, :] << 2) | (hi[..., 2, :] << 4) | (hi[..., 3, :] << 6)).reshape(*d.shape, 64)
    blocks = torch.cat([ql, qh, sc.to(torch.int8).view(torch.uint8), _f16_bytes(d)], -1)

    def weights() -> torch.Tensor:
        return ((d.double()[..., None] * sc.double())[..., None] * q.double()).reshape(n, -1)[:, :k]

    return blocks, weights


def _kq(case: dict, seed: int):
    return (_q4k if case["fmt"] == "q4k" else _q6k)(case["n"], case["k"], seed)


def _rows_in(case: dict, seed: int) -> torch.Tensor:
    """Activation rows of a kq / q8 case, padded to a row stride that is a multiple of 8."""
    x = _normal((case["rows"], case["k"]), seed, 2)
    return x.half() if case.get("f16") else x


def _mlp_inputs(case: dict, seed: int):
    h, i, r = case["hidden"], case["inter"], case["rows"]
    w = [_a8_weights(i, h, seed, 1), _a8_weights(i, h, seed, 2), _a8_weights(h, i, seed, 3)]
    return w, _normal((r, h), seed, 4), _normal((r, h), seed, 5)


def _gdn_inputs(case: dict, seed: int) -> dict:
    kh, vh, d = case["k_heads"], case["v_heads"], GDN_DIM
    lens = _spread(case["shortest"], case["longest"], case["nseq"], seed)
    rows = sum(lens)
    return {
        "lens": lens,
        "conv": torch.nn.functional.silu(_normal((rows, (2 * kh + vh) * d), seed, 1)),
        "a": _normal((rows, vh), seed, 2),
        "b": _normal((rows, vh), seed, 3),
        "z": _normal((rows, vh * d), seed, 4),
        "a_log": (1 + 15 * torch.rand(vh, generator=_gen(seed, 5), device="cuda")).log(),
        "dt_bias": _normal((vh,), seed, 6, 0.1),
        "norm": 1 + _normal((d,), seed, 7, 0.1),
        "states": _normal((len(lens), vh, d, d), seed, 8, 0.1),
    }


def _attn_inputs(case: dict, seed: int) -> dict:
    h, kv, hd, nseq, t = case["heads"], case["kv_heads"], case["head_dim"], case["nseq"], case["tokens"]
    ctx = [max(c, t) for c in _spread(case["shortest"], max(case["shortest"], case["longest"]), nseq, seed)]
    rows = nseq * t
    need = [(c + BLOCK - 1) // BLOCK for c in ctx]
    pages = np.random.default_rng(seed + 1).permutation(sum(need)).astype(np.int32)
    tables = np.zeros((nseq, max(need)), np.int32)
    at = 0
    for s, m in enumerate(need):
        tables[s, :m] = pages[at:at + m]
        at += m
    out = {
        "ctx": ctx,
        "q": _normal((rows, h, hd), seed, 1),
        "gate": _normal((rows, h, hd), seed, 2) if case["gate"] else None,
        "k": _normal((sum(need), kv, BLOCK, hd), seed, 3),
        "v": _normal((sum(need), kv, BLOCK, hd), seed, 4),
        "seq": np.repeat(np.arange(nseq, dtype=np.int32), t),
        "pos": np.concatenate([np.arange(c - t, c, dtype=np.int32) for c in ctx]),
        "tables": tables,
    }
    return out


def _cuda(a: np.ndarray) -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _p(t: torch.Tensor | None):
    return C.c_void_p(t.data_ptr() if t is not None else None)


# ---- states ---------------------------------------------------------------------


class _Mlp:
    def __init__(self, case: dict, seed: int):
        dev = _device()
        w, self.x, self.res = _mlp_inputs(case, seed)
        self.gate, self.up, self.down = (_a8_matrix(dev, p) for p in w)
        self.dev, self.rows, self.h, self.i = dev, case["rows"], case["hidden"], case["inter"]
        self.act = torch.empty(act_bytes(self.rows, self.h), dtype=torch.uint8, device="cuda")
        self.mid = torch.empty((self.rows, self.i), device="cuda")
        self.mid_act = torch.empty(act_bytes(self.rows, self.i), dtype=torch.uint8, device="cuda")
        self.y = torch.empty((self.rows, self.h), device="cuda")

    def run(self):
        act_prep_dev(self.dev, self.x.data_ptr(), self.h, self.rows, self.h, self.act.data_ptr())
        Matrix.gemv_swiglu_act_dev(self.gate, self.up, self.act.data_ptr(), self.rows, self.mid.data_ptr(), self.i)
        act_prep_dev(self.dev, self.mid.data_ptr(), self.i, self.rows, self.i, self.mid_act.data_ptr())
        self.down.gemv_act_dev(self.mid_act.data_ptr(), self.rows, self.y.data_ptr(), self.h, self.res.data_ptr(),
                               self.h)
        return [self.mid, self.y]


class _Linear:
    """One GGUF projection, in either arithmetic."""

    def __init__(self, case: dict, seed: int):
        blocks, _ = _kq(case, seed)
        self.w = Matrix.upload_kq(_device(), FMT_Q4K if case["fmt"] == "q4k" else FMT_Q6K, blocks.cpu().numpy(),
                                  case["n"], case["k"])
        self.x = _rows_in(case, seed)
        self.rows, self.n, self.k = case["rows"], case["n"], case["k"]
        self.q8, self.f16 = case["kind"] == "q8", bool(case.get("f16"))
        self.res = _normal((self.rows, self.n), seed, 3) if case.get("res") else None
        self.y = torch.empty((self.rows, self.n), device="cuda")

    def run(self):
        if self.q8:
            self.w.gemv_q8act_dev(self.x.data_ptr(), self.k, self.rows, self.y.data_ptr(), self.n,
                                  self.res.data_ptr() if self.res is not None else 0, self.n)
        else:
            self.w.gemv_dev(self.x.data_ptr(), self.k, self.rows, self.y.data_ptr(), self.n, x_f16=self.f16)
        return self.y


class _Gdn:
    def __init__(self, case: dict, seed: int):
        self.case, self.dev = case, _device()
        self.t = t = _gdn_inputs(case, seed)
        start = np.concatenate([[0], np.cumsum(t["lens"])[:-1]]).astype(np.int32)
        self.start, self.count = _cuda(start), _cuda(np.asarray(t["lens"], np.int32))
        self.ptrs = torch.tensor([s.data_ptr() for s in t["states"]], dtype=torch.int64, device="cuda")
        self.rows, self.longest = sum(t["lens"]), max(t["lens"])
        self.out = torch.empty((self.rows, case["v_heads"] * GDN_DIM), device="cuda")

    def run(self):
        c, t = self.case, self.t
        args = [self.dev.handle, c["k_heads"], c["v_heads"], _p(t["conv"]), _p(t["a"]), _p(t["b"]), _p(t["z"]),
                _p(t["a_log"]), _p(t["dt_bias"]), _p(t["norm"]), _p(self.ptrs), _p(self.start), _p(self.count),
                len(t["lens"])]
        if self.longest > 4:
            call("pgd_gdn_prefill_dev", *args, self.rows, self.longest, _p(self.out))
        else:
            call("pgd_gdn_step_dev", *args, _p(self.out))
        return [self.out, t["states"]]


class _Attn:
    def __init__(self, case: dict, seed: int):
        self.case, self.dev = case, _device()
        self.t = t = _attn_inputs(case, seed)
        self.seq, self.pos, self.tables = _cuda(t["seq"]), _cuda(t["pos"]), _cuda(t["tables"])
        self.out = torch.empty_like(t["q"])

    def run(self):
        c, t = self.case, self.t
        call("pgd_attn_decode_dev", self.dev.handle, c["heads"], c["kv_heads"], c["head_dim"], BLOCK, _p(t["q"]),
             _p(t["gate"]), _p(t["k"]), _p(t["v"]), _p(self.seq), _p(self.pos), _p(self.tables),
             int(t["tables"].shape[1]), int(t["q"].shape[0]), _p(self.out))
        return self.out


class _Whole:
    """A model and the token ids of a batch of requests."""

    def __init__(self, case: dict, seed: int):
        rng = np.random.default_rng(seed)
        if case["kind"] == "qwen2":
            cfg = replace(QWEN2_05B, max_pos=1024, kv_blocks=64)
            lens = [case["prompt"]]
        else:
            lens = _spread(case["shortest"], case["longest"], case["nseq"], seed)
            pages = sum((n + case["gen"] + BLOCK - 1) // BLOCK for n in lens)
            cfg = replace(QWEN35_27B, n_layers=case["layers"], max_pos=1024, kv_blocks=pages + 8)
        self.model = Model.synth(_device(), cfg, int(seed) & 0xFFFFFFFF)
        self.prompts = [rng.integers(0, cfg.vocab, n) for n in lens]
        self.feeds = rng.integers(0, cfg.vocab, (case["gen"], len(lens)))

    def run(self):
        sessions = [self.model.new_session() for _ in self.prompts]
        _, first = self.model.step_ragged(sessions, self.prompts, want_logits=True)
        for toks in self.feeds[:-1]:
            self.model.step_ragged(sessions, [[t] for t in toks])
        _, last = self.model.step_ragged(sessions, [[t] for t in self.feeds[-1]], want_logits=True)
        for s in sessions:
            s.free()
        return [first, last]

    def __del__(self):
        try:
            self.model.free()
        except Exception:
            pass


_STATES = {"mlp": _Mlp, "kq": _Linear, "q8": _Linear, "gdn": _Gdn, "attn": _Attn, "qwen2": _Whole, "hybrid": _Whole}


def prepare(case: dict, seed: int):
    state = _STATES[case["kind"]](case, seed)
    torch.cuda.synchronize()  # inputs come from torch's stream, the calls run on the device handle's
    return state


def run(state):
    return state.run()


# ---- what a pass cannot do without ------------------------------------------------

_BPW = {"q4k": 4.5, "q6k": 6.5625}


def _model_step(cfg, rows: int, seqs: int, weight_bytes: float, weights: float) -> tuple[float, float]:
    return weight_bytes + seqs * cfg.vocab * 4, 2.0 * weights * rows + 2.0 * cfg.hidden * cfg.vocab * seqs


def work(case: dict) -> dict:
    k = case["kind"]
    if k == "mlp":
        h, i, r = case["hidden"], case["inter"], case["rows"]
        return {"bytes": 3 * h * i * 8.5 / 8 + 3 * r * h * 4 + r * i * 4, "flops": 6.0 * r * h * i}
    if k in ("kq", "q8"):
        n, kk, r = case["n"], case["k"], case["rows"]
        x = 2 if case.get("f16") else 4
        return {"bytes": n * kk * _BPW[case["fmt"]] / 8 + r * kk * x + r * n * 4 * (2 if case.get("res") else 1),
                "flops": 2.0 * r * n * kk}
    if k == "gdn":
        kh, vh, d = case["k_heads"], case["v_heads"], GDN_DIM
        lens = _spread(case["shortest"], case["longest"], case["nseq"], 0)
        rows = sum(lens)
        return {"bytes": len(lens) * vh * d * d * 8 + rows * 4.0 * ((2 * kh + vh) * d + 2 * vh + 2 * vh * d),
                "flops": rows * vh * d * d * 7.0}
    if k == "attn":
        h, kv, hd, t, n = case["heads"], case["kv_heads"], case["head_dim"], case["tokens"], case["nseq"]
        ctx = [max(c, t) for c in _spread(case["shortest"], max(case["shortest"], case["longest"]), n, 0)]
        pairs = sum(t * (c - t) + t * (t + 1) / 2 for c in ctx)
        return {"bytes": sum(ctx) * kv * hd * 8 + n * t * h * hd * 4.0 * (3 if case["gate"] else 2),
                "flops": 4.0 * pairs * h * hd}
    gen = case["gen"]
    if k == "qwen2":
        cfg, lens = QWEN2_05B, [case["prompt"]]
        weights = cfg.n_layers * cfg.hidden * (cfg.hidden * 2 + 2 * cfg.kv_heads * cfg.head_dim + 3 * cfg.intermediate)
        step_bytes = weights * 5.0 / 8 + cfg.hidden * cfg.vocab * 6.5625 / 8
    else:
        cfg = QWEN35_27B
        lens = _spread(case["shortest"], case["longest"], case["nseq"], 0)
        conv = (2 * cfg.k_heads + cfg.v_heads) * GDN_DIM
        lin = cfg.hidden * (conv + 2 * cfg.v_heads * GDN_DIM + 2 * cfg.v_heads)
        full = cfg.hidden * cfg.head_dim * (3 * cfg.heads + 2 * cfg.kv_heads)
        mlp = 3 * cfg.hidden * cfg.intermediate
        weights = case["layers"] * (0.75 * lin + 0.25 * full + mlp)
        step_bytes = (weights + cfg.hidden * cfg.vocab) * 8.5 / 8
    seqs = len(lens)
    b0, f0 = _model_step(cfg, sum(lens), seqs, step_bytes, weights)
    b1, f1 = _model_step(cfg, seqs, seqs, step_bytes, weights)
    if k == "hybrid":  # recurrent state in and out on every step
        b = seqs * 0.75 * case["layers"] * cfg.v_heads * GDN_DIM * GDN_DIM * 8
        b0, b1 = b0 + b, b1 + b
    return {"bytes": b0 + gen * b1, "flops": f0 + gen * f1}


def tolerance(case: dict):
    """About four times the error against exact() (mlp 4e-6, kq 2.5e-5, gdn
    1.1e-6, attn 3e-7) or, for hybrid, the difference between the batch and the
    same requests one by one (1.5e-5). The q8 arithmetic fixes the order of
    every sum, so q8 and qwen2 have one right answer."""
    return {
        "mlp": {"rel": 2e-5},
        "kq": {"rel": 1e-4},
        "q8": "exact",
        "gdn": {"rel": 5e-6},
        "attn": {"rel": 2e-6},
        "qwen2": "exact",
        "hybrid": {"rel": 1e-4},
    }[case["kind"]]


# ---- the same values in 64 bits -----------------------------------------------------


def _q8k_rows(x: torch.Tensor) -> torch.Tensor:
    """Rows as Q8_K holds them (256-element blocks, the first element of
    largest magnitude mapped to -128, round half away from zero), dequantized
    to float64. The rounding to 8 bits is part of the arithmetic."""
    rows, k = x.shape
    nsb = (k + 255) // 256
    v = torch.zeros((rows, nsb * 256), device=x.device)
    v[:, :k] = x
    v = v.reshape(rows, nsb, 256)
    top = v.gather(-1, v.abs().argmax(-1, keepdim=True))
    inv = torch.where(top == 0, torch.zeros_like(top), -128.0 / top)
    t = inv * v
    q = torch.where(t < 0, (t.double() - 0.5).ceil(), (t.double() + 0.5).floor()).clamp_max(127)
    d = torch.where(top == 0, torch.zeros_like(top), 1.0 / inv)
    return (q * d.double()).reshape(rows, -1)[:, :k]


def _gdn_exact(case: dict, seed: int):
    t = _gdn_inputs(case, seed)
    kh, vh, d = case["k_heads"], case["v_heads"], GDN_DIM
    conv = t["conv"].double()
    rows = conv.shape[0]

    def heads(cols, scale):
        v = cols.reshape(rows, kh, d)
        v = v / (v.square().sum(-1, keepdim=True) + 1e-6).sqrt() * scale
        return v.repeat_interleave(vh // kh, 1)

    q = heads(conv[:, :kh * d], d ** -0.5)
    k = heads(conv[:, kh * d:2 * kh * d], 1.0)
    v = conv[:, 2 * kh * d:].reshape(rows, vh, d)
    decay = torch.exp(-t["a_log"].double().exp() * torch.nn.functional.softplus(t["a"].double() + t["dt_bias"].double()))
    beta = torch.sigmoid(t["b"].double())
    state = t["states"].double().clone()
    o = torch.empty((rows, vh, d), dtype=torch.float64, device="cuda")
    start = np.concatenate([[0], np.cumsum(t["lens"])[:-1]])
    for step in range(max(t["lens"])):
        live = [s for s, n in enumerate(t["lens"]) if step < n]
        r = torch.tensor([int(start[s]) + step for s in live], device="cuda")
        li = torch.tensor(live, device="cuda")
        st = state[li] * decay[r][..., None, None]
        delta = beta[r][..., None] * (v[r] - (st * k[r][..., None]).sum(-2))
        st = st + k[r][..., None] * delta[..., None, :]
        state[li] = st
        o[r] = (st * q[r][..., None]).sum(-2)
    o = o / (o.square().mean(-1, keepdim=True) + 1e-6).sqrt() * t["norm"].double()
    z = t["z"].double().reshape(rows, vh, d)
    return [(o * z * torch.sigmoid(z)).reshape(rows, vh * d), state]


def _attn_exact(case: dict, seed: int):
    t = _attn_inputs(case, seed)
    h, kv, hd, n = case["heads"], case["kv_heads"], case["head_dim"], case["tokens"]
    out = torch.empty(t["q"].shape, dtype=torch.float64, device="cuda")
    for s, c in enumerate(t["ctx"]):
        pages = torch.from_numpy(t["tables"][s, :(c + BLOCK - 1) // BLOCK].astype(np.int64)).cuda()
        k, v = (t[x][pages].double().transpose(0, 1).reshape(kv, -1, hd)[:, :c] for x in ("k", "v"))
        mask = torch.arange(c, device="cuda")[None, :] > torch.arange(c - n, c, device="cuda")[:, None]
        for g in range(kv):
            per = h // kv
            q = t["q"][s * n:(s + 1) * n, g * per:(g + 1) * per].double().transpose(0, 1).reshape(per * n, hd)
            scores = (q @ k[g].t().contiguous() / math.sqrt(hd)).reshape(per, n, c).masked_fill(mask, -math.inf)
            o = torch.softmax(scores, -1).reshape(per * n, c) @ v[g]
            out[s * n:(s + 1) * n, g * per:(g + 1) * per] = o.reshape(per, n, hd).transpose(0, 1)
    return out if t["gate"] is None else out * torch.sigmoid(t["gate"].double())


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "mlp":
        w, x, res = _mlp_inputs(case, seed)
        gate = x.double() @ _a8_dequant(w[0]).t()
        mid = gate * torch.sigmoid(gate) * (x.double() @ _a8_dequant(w[1]).t())
        return [mid, res.double() + mid @ _a8_dequant(w[2]).t()]
    if kind in ("kq", "q8"):
        w = _kq(case, seed)[1]()
        x = _rows_in(case, seed)
        y = (x.double() if kind == "kq" else _q8k_rows(x)) @ w.t()
        return y + _normal(y.shape, seed, 3).double() if case.get("res") else y
    if kind == "gdn":
        return _gdn_exact(case, seed)
    if kind == "attn":
        return _attn_exact(case, seed)
    return None  # whole models: weights the library generates, and no 64-bit value of their quantized activations
