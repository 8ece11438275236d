"""What the executor's speed is measured on.

Each case is one thing a user's program has the framework do, through its
public entry points (``see-ai_amd/hip.py``, the plan writer's plans): the
W8A8 products of a quantized model from a decode step to a prefill, the three
attention families forward and backward, the loss turn over a vocabulary, an
optimizer step, and whole plan-engine calls -- the LoRA MLP step, the
decoder's train and eval steps, the int8-base decoder's train step.

``listed()`` are the fixed cases, ``draw(rng)`` more of the same ranges,
``prepare`` / ``run`` what a program holds and calls, ``work`` what a pass
cannot do without, ``exact`` the same results in float64 from plain torch.
"""
from __future__ import annotations

import ctypes
import functools
import importlib
import math

import numpy as np
import torch
import torch.utils.checkpoint

hip = importlib.import_module("see-ai_amd.hip")
pw = importlib.import_module("see-ai_amd.planwriter")

F64 = torch.float64


# --- the cases ------------------------------------------------------------------------------------

def listed():
    return [
        # Decode: 32 sequences, one token each, through one 4096 x 4096 layer.
        {"name": "w8a8_decode", "kind": "w8a8", "M": 32, "N": 4096, "K": 4096},
        # One prompt's prefill chunk into a gated FFN (2048 -> 5632), a row
        # count off every tile.
        {"name": "w8a8_chunk", "kind": "w8a8", "M": 500, "N": 5632, "K": 2048},
        # The benchmark's product: a full prefill batch, 4096 cubed.
        {"name": "w8a8_prefill", "kind": "w8a8", "M": 4096, "N": 4096, "K": 4096},
        # The benchmark's attention: training in bf16 activations.
        {"name": "attn_bf16", "kind": "attn", "held": "bf16", "B": 16, "S": 2048, "H": 16,
         "d": 64, "doc": 0},
        # The decoder's attention in the exact (f32) family: every eval, and
        # every plan whose attention is not let run on bf16.
        {"name": "attn_f32", "kind": "attn", "held": "f32", "B": 8, "S": 1024, "H": 12, "d": 64,
         "doc": 0},
        # Relaxed attention on f32 operands at the wider head, packed
        # documents, a sequence length off every block.
        {"name": "attn_relaxed", "kind": "attn", "held": "relaxed", "B": 4, "S": 1500, "H": 8,
         "d": 128, "doc": 400},
        # The loss turn of both decoders: 8192 tokens over 32000 classes.
        {"name": "xent", "kind": "xent", "N": 8192, "C": 32000, "masked": False},
        # AdamW over the larger decoder's 4,194,304 adapter parameters.
        {"name": "adamw", "kind": "adamw", "n": 4194304, "clip": 0.0},
        # The smallest whole call: one optimizer step of the LoRA MLP on a
        # batch of 32 rows.
        {"name": "mlp_step", "kind": "mlp", "batch": 32, "din": 256, "hidden": 512, "dout": 256},
        # One optimizer step of the 12-layer decoder, 8 x 1024 tokens, bf16
        # activations.
        {"name": "decoder_step", "kind": "decoder", "vocab": 32000, "dim": 768, "ffn": 3072,
         "layers": 12, "seq": 1024, "batch": 8, "rank": 8, "bf16": True},
        # Scoring what ships: the exact eval of four decoder layers on two
        # sequences.
        {"name": "decoder_eval", "kind": "eval", "vocab": 32000, "dim": 768, "ffn": 3072,
         "layers": 4, "seq": 1024, "batch": 2, "rank": 8, "bf16": False},
        # One optimizer step of the larger decoder's blocks (four of its
        # sixteen) on the frozen int8 base, 4 x 2048 tokens, bf16 activations.
        {"name": "q8_step", "kind": "q8", "vocab": 32000, "dim": 2048, "ffn": 5632, "layers": 4,
         "seq": 2048, "batch": 4, "rank": 16, "bf16": True},
    ]


def _spread(rng, lo, hi):
    """A whole number from lo to hi, even over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["w8a8", "w8a8", "attn", "attn", "attn", "xent", "adamw", "mlp", "decoder",
                       "eval", "q8"])
    if kind == "w8a8":
        while True:
            c = {"kind": kind, "M": _spread(rng, 1, 4096), "N": _spread(rng, 256, 5632),
                 "K": _spread(rng, 256, 5632)}
            if rng.random() < 0.5:  # model widths are multiples of 64 as often as not
                c["N"], c["K"] = c["N"] // 64 * 64, c["K"] // 64 * 64
            if c["M"] * c["N"] * c["K"] <= 4096 ** 3:
                return c
    if kind == "attn":
        held = rng.choice(["bf16", "f32", "relaxed"])
        while True:
            c = {"kind": kind, "held": held, "B": _spread(rng, 1, 16), "S": _spread(rng, 64, 2048),
                 "H": _spread(rng, 2, 32), "d": 64 if held == "bf16" else rng.choice([64, 128]),
                 "doc": rng.choice([0, 0, _spread(rng, 32, 1024)])}
            pairs = c["B"] * c["H"] * c["S"] * c["S"] * c["d"]
            if pairs <= (16 * 16 * 2048 * 2048 * 64 if held == "bf16" else 4 << 30):
                return c
    if kind == "xent":
        return {"kind": kind, "N": _spread(rng, 32, 8192), "C": _spread(rng, 256, 32000),
                "masked": rng.random() < 0.5}
    if kind == "adamw":
        return {"kind": kind, "n": _spread(rng, 2048, 4194304), "clip": rng.choice([0.0, 1.0])}
    if kind == "mlp":
        return {"kind": kind, "batch": _spread(rng, 4, 256), "din": 4 * _spread(rng, 16, 256),
                "hidden": 4 * _spread(rng, 16, 512), "dout": 4 * _spread(rng, 8, 256)}
    dim = 64 * (rng.randint(2, 12) if kind != "q8" else rng.randint(2, 32))
    c = {"kind": kind, "vocab": 4 * _spread(rng, 24, 8000), "dim": dim,
         "ffn": 32 * max(4, dim // 32 * rng.randint(2, 4) + rng.randint(-2, 2)),
         "layers": rng.randint(1, 4), "seq": 8 * _spread(rng, 8, 128), "batch": _spread(rng, 1, 8),
         "rank": rng.choice([8, 16]), "bf16": kind != "eval" and rng.random() < 0.7}
    if kind == "eval":
        c["batch"] = min(c["batch"], 4)
    return c


# --- what a program holds -------------------------------------------------------------------------

@functools.lru_cache(maxsize=1)
def _context():
    """One backend context for the whole program, on torch's stream."""
    ctx = hip.Context(0)
    ctx.use_torch_stream()
    return ctx


@functools.lru_cache(maxsize=2)
def _plan(kind, **cfg):
    if kind == "mlp":
        return pw.mlp_lora(hip.plan_self_hash, **cfg)
    make = pw.decoder_q8_lora if kind == "q8" else pw.decoder_lora
    return make(hip.plan_self_hash, relaxed=True, heads=cfg["dim"] // 64, alpha=2.0 * cfg["rank"],
                **cfg)


def _plan_of(case):
    keys = (("batch", "din", "hidden", "dout") if case["kind"] == "mlp" else
            ("vocab", "dim", "ffn", "layers", "seq", "batch", "rank"))
    return _plan("decoder" if case["kind"] == "eval" else case["kind"],
                 **{k: case[k] for k in keys})


class _Extent:
    """`count` floats of an engine's arena, for torch to look at in place; it
    holds the engine for as long as torch looks."""

    def __init__(self, eng, base, offset, count):
        self.eng = eng
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": "<f4", "version": 2,
                                         "data": (base + offset, False)}


def _view(eng, offset, nbytes):
    base = hip.lib().seeai_arena(hip.lib().seeai_engine_context(eng.h))
    return torch.as_tensor(_Extent(eng, base, offset, nbytes // 4), device="cuda")


def _run_of(img, names):
    """(offset, bytes) of the arena extent the named tensors fill, in order."""
    spans = [img.arena[n] for n in names]
    lo = min(o for o, _ in spans)
    return lo, max(o + b for o, b in spans) - lo


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _starts(case, seed):
    """First key of each token's document, documents of about `doc` tokens
    packed one after another."""
    if not case["doc"]:
        return None
    r = np.random.default_rng(seed)
    out = np.zeros((case["B"], case["S"]), np.int32)
    for b in range(case["B"]):
        at = 0
        while at < case["S"]:
            n = int(r.integers(max(1, case["doc"] // 2), 2 * case["doc"]))
            out[b, at:at + n] = at
            at += n
    return torch.from_numpy(out.reshape(-1)).cuda()


def _inputs(case, seed):
    """The call's inputs, from the seed alone."""
    kind, g = case["kind"], _gen(seed)
    rnd = lambda *s: torch.randn(s, device="cuda", generator=g)  # noqa: E731
    if kind == "w8a8":
        return {"X": rnd(case["M"], case["K"]), "W": rnd(case["K"], case["N"]) * 0.02}
    if kind == "attn":
        T, W = case["B"] * case["S"], case["H"] * case["d"]
        x = {n: rnd(T, W) for n in ("q", "k", "v", "do")}
        if case["held"] == "bf16":
            x = {n: t.to(torch.bfloat16) for n, t in x.items()}
        x["starts"] = _starts(case, seed)
        return x
    if kind == "xent":
        N, C = case["N"], case["C"]
        lab = torch.randint(0, C, (N,), dtype=torch.int32, device="cuda", generator=g)
        if case["masked"]:
            lab[torch.rand(N, device="cuda", generator=g) < 0.2] = -1
        return {"logits": rnd(N, C) * 3, "labels": lab, "seed": torch.ones(1, device="cuda")}
    if kind == "adamw":
        n = case["n"]
        return {"p": rnd(n) * 0.02, "g": rnd(n) * 1e-3, "m": rnd(n) * 1e-4,
                "v": (rnd(n) * 1e-3) ** 2}
    if kind == "mlp":
        return {"x": pw.normal(2 * seed + 1, (case["batch"], case["din"])),
                "y": pw.uniform_ints(2 * seed + 2, case["batch"], case["dout"])}
    T = case["seq"] * case["batch"]
    tok = pw.uniform_ints(seed, T + 1, case["vocab"])
    return {"x": tok[:T].copy().view(np.float32), "y": tok[1:].copy()}


def _planted(case, img, seed):
    """The adapters' B matrices as a run under way holds them (a fresh plan's
    are zero, and their A gradients with them)."""
    names = [n for n in img.arrays if n.split(".")[-1][0] == "B"]
    return {n: pw.normal(7919 * (seed + 1) + i, img.arrays[n].shape, 0.02)
            for i, n in enumerate(names)}


ADAMW = dict(lr=1e-3, beta1=0.9, beta2=0.999, eps=1e-8, weight_decay=0.01, step=3)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, **_inputs(case, seed)}
    new = lambda *shape, dtype=torch.float32: torch.empty(shape, dtype=dtype, device="cuda")  # noqa: E731
    if kind in ("w8a8", "attn", "xent", "adamw"):
        s["ctx"] = ctx = _context()
    if kind == "w8a8":
        M, N, K = case["M"], case["N"], case["K"]
        s.update(QA=new(M, K, dtype=torch.int8), sa=new(M), QWt=new(N, K, dtype=torch.int8),
                 sw=new(N), C=new(M, N))
        ctx.call("seeai_w8a8_pack_weights", s["W"].data_ptr(), s["QWt"].data_ptr(),
                 s["sw"].data_ptr(), K, N)
        torch.cuda.synchronize()
        del s["W"]  # the weights are packed once and kept packed
    elif kind == "attn":
        T, W = s["q"].shape
        s.update(o=new(T, W), stats=new(case["B"] * case["H"] * case["S"], 4), dq=new(T, W),
                 dk=new(T, W), dv=new(T, W))
    elif kind == "xent":
        s.update(loss=new(1), probs=new(case["N"], case["C"]), dlogits=new(case["N"], case["C"]))
    elif kind == "adamw":
        s["params"] = hip.StepParams(ADAMW["lr"], ADAMW["beta1"], ADAMW["beta2"], ADAMW["eps"],
                                     ADAMW["weight_decay"], 0, ADAMW["step"])
    else:
        img = _plan_of(case)
        s["eng"] = eng = hip.Engine(img.blob)
        eng.use_torch_stream()
        if kind != "mlp":
            eng.set_attention_bf16(case["bf16"])
        for n, b in _planted(case, img, seed).items():
            eng.write(img.arena[n][0], b.tobytes())
        params = [n for n in img.arrays if "m_" + n in img.arena]
        if kind == "eval":
            s["logits"] = _view(eng, *img.arena["logits"])
        else:
            s["adapters"] = _view(eng, *_run_of(img, params))
            s["grads"] = [_view(eng, *img.arena[n]) for n in _grad_names(params)] if kind == "mlp" \
                else [_view(eng, *_run_of(img, _grad_names(params)))]
    return s


def _grad_names(params):
    """An adapter's gradient buffer: A1 -> dA1, l0.Aq -> l0.dAq."""
    return [".".join(n.split(".")[:-1] + ["d" + n.split(".")[-1]]) for n in params]


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    P = lambda n: s[n].data_ptr()  # noqa: E731
    if kind == "w8a8":
        M, N, K = case["M"], case["N"], case["K"]
        call = s["ctx"].call
        call("seeai_w8a8_quantize_rows", P("X"), P("QA"), P("sa"), M, K)
        call("seeai_w8a8_gemm", P("QA"), P("sa"), P("QWt"), P("sw"), P("C"), None, M, N, K)
        return {"C": s["C"], "QA": s["QA"], "sa": s["sa"]}
    if kind == "attn":
        call, geo = s["ctx"].call, (case["B"], case["S"], case["H"], case["d"])
        starts = s["starts"].data_ptr() if s["starts"] is not None else None
        if case["held"] == "bf16":
            call("seeai_attn_fwd_bf16", P("q"), P("k"), P("v"), P("o"), P("stats"), *geo, starts)
            call("seeai_attn_dq_bf16", P("q"), P("k"), P("v"), P("do"), P("stats"), P("dq"), *geo)
            call("seeai_attn_dkdv_bf16", P("q"), P("k"), P("v"), P("do"), P("stats"), P("dk"),
                 P("dv"), *geo)
        else:
            dt = int(case["held"] == "relaxed")
            call("seeai_attn_fwd", dt, P("q"), P("k"), P("v"), P("o"), P("stats"), *geo, starts)
            call("seeai_attn_dq", dt, P("q"), P("k"), P("v"), P("do"), P("stats"), P("dq"), *geo)
            if dt == 0:
                call("seeai_attn_dkdv_f32", P("q"), P("k"), P("v"), P("do"), P("stats"), P("dk"),
                     P("dv"), *geo)
            elif case["d"] == 64:
                call("seeai_attn_dkdv", P("q"), P("k"), P("v"), P("do"), P("stats"), P("dk"),
                     P("dv"), *geo)
            else:  # the fused relaxed pass is for head width 64
                call("seeai_attn_dk", dt, P("q"), P("k"), P("v"), P("do"), P("stats"), P("dk"), *geo)
                call("seeai_attn_dv", dt, P("q"), P("k"), P("do"), P("stats"), P("dv"), *geo)
        return {n: s[n] for n in ("o", "stats", "dq", "dk", "dv")}
    if kind == "xent":
        N, C, masked = case["N"], case["C"], int(case["masked"])
        call = s["ctx"].call
        call("seeai_xent_fwd", P("logits"), P("labels"), P("loss"), P("probs"), N, C, masked)
        call("seeai_xent_bwd", P("probs"), P("labels"), P("seed"), P("dlogits"), N, C, masked)
        return {n: s[n] for n in ("loss", "probs", "dlogits")}
    if kind == "adamw":
        s["ctx"].call("seeai_adamw_step", P("p"), P("g"), P("m"), P("v"), case["n"],
                      ctypes.byref(s["params"]), ctypes.c_float(case["clip"]))
        return {n: s[n] for n in ("p", "m", "v")}
    if kind == "eval":
        return {"loss": s["eng"].evaluate(s["x"], s["y"]), "logits": s["logits"]}
    return {"loss": s["eng"].train_step(s["x"], s["y"]), "grads": s["grads"],
            "adapters": s["adapters"]}


# --- what a pass cannot do without ----------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "w8a8":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 4 * M * K + M * K + N * K + 4 * M * N + 4 * (M + N),
                "flops": 2 * M * N * K}
    if kind == "attn":
        units, S, d = case["B"] * case["H"], case["S"], case["d"]
        e = units * S * d
        per = S * (S + 1) // 2
        if case["doc"]:  # about 5/4 doc tokens a document, by the lengths' mean and spread
            n = min(S, int(1.4 * case["doc"]))
            per = S * (n + 1) // 2
        return {"bytes": e * (4 * (2 if case["held"] == "bf16" else 4) + 4 * 4) + units * S * 16,
                "flops": 12 * d * per * units}
    if kind == "xent":  # the logits in, probabilities and gradient out
        return {"bytes": 12 * case["N"] * case["C"], "flops": 8 * case["N"] * case["C"]}
    if kind == "adamw":
        return {"bytes": 28 * case["n"], "flops": 15 * case["n"]}
    if kind == "mlp":
        n, w = case["batch"], case["din"] * case["hidden"] + case["hidden"] * case["dout"]
        r = 8 * (case["din"] + 2 * case["hidden"] + case["dout"])
        return {"bytes": 4 * w + 28 * r + 4 * n * (case["din"] + 1),
                "flops": 2 * n * (w + case["hidden"] * case["dout"] + 3 * r)}
    T, D, F, L, r = case["seq"] * case["batch"], case["dim"], case["ffn"], case["layers"], case["rank"]
    frozen = L * (4 * D * D + (3 if kind == "q8" else 2) * D * F)
    sites = 4 if kind == "q8" else 2
    attn = L * case["batch"] * case["seq"] * (case["seq"] + 1) // 2 * D * 4
    passes = 1 if kind == "eval" else 2
    adapters = L * sites * 2 * D * r
    weights = frozen * (1 if kind == "q8" else 4) + 4 * D * case["vocab"]
    return {"bytes": passes * weights + 4 * D * min(T, case["vocab"]) +
            (0 if kind == "eval" else 28 * adapters) + (4 * T * case["vocab"] if kind == "eval" else 0),
            "flops": 2 * T * passes * (frozen + D * case["vocab"]) +
            2 * T * adapters * (1 if kind == "eval" else 3) +
            attn * (1 if kind == "eval" else 3)}


def tolerance(case):
    kind = case["kind"]
    if kind == "w8a8":  # whole-number sums; the dequantization is one expression
        return "exact"
    if kind == "attn":
        return {"rel": 1e-2, "max": 0.2} if case["held"] != "f32" else {"rel": 1e-5, "max": 1e-3}
    if kind == "xent":
        return {"rel": 1e-5, "max": 1e-3}
    if kind == "adamw":
        return {"rel": 1e-6, "max": 1e-4}
    if kind == "mlp":
        return {"rel": 1e-4, "max": 5e-2}
    if kind == "eval":
        return {"rel": 1e-5, "max": 1e-3}
    # A gradient that changes sign moves its weight by two learning rates at
    # AdamW's first steps: the largest difference is that, over the adapters'
    # spread.
    return {"rel": 2e-2, "max": 0.5}


# --- the same in float64 --------------------------------------------------------------------------

def _attention64(q, k, v, starts, B, S, H, d):
    """Causal attention of [B*S, H*d] rows: (o, m, 1/l), per-unit tensors."""
    split = lambda t: t.view(B, S, H, d).transpose(1, 2).contiguous()  # noqa: E731
    q, k, v = split(q), split(k), split(v)
    i = torch.arange(S, device=q.device)
    ok = (i[None, :] <= i[:, None])[None, None]
    if starts is not None:
        ok = ok & (i[None, None, None, :] >= starts.view(B, 1, S, 1))
    sc = (torch.matmul(q, k.transpose(2, 3).contiguous()) / math.sqrt(d)).masked_fill(~ok, -math.inf)
    m = sc.amax(dim=3, keepdim=True)
    e = torch.exp(sc - m)
    l = e.sum(dim=3, keepdim=True)
    p = e / l
    o = torch.matmul(p, v)
    return o.transpose(1, 2).reshape(B * S, H * d), p, m, l


def _exact_attn(case, x):
    B, S, H, d = case["B"], case["S"], case["H"], case["d"]
    T, W = B * S, H * d
    out = {n: torch.empty((T, W), dtype=F64, device="cuda") for n in ("o", "dq", "dk", "dv")}
    stats = torch.empty((B, H, S, 4), dtype=F64, device="cuda")
    for b in range(B):
        rows = slice(b * S, (b + 1) * S)
        st = x["starts"][rows] if x["starts"] is not None else None
        for h0 in range(0, H, 8):
            h1 = min(H, h0 + 8)
            cols, n = slice(h0 * d, h1 * d), h1 - h0
            q, k, v, do = (x[t][rows, cols].to(F64).contiguous() for t in ("q", "k", "v", "do"))
            o, p, m, l = _attention64(q, k, v, st, 1, S, n, d)
            split = lambda t: t.view(1, S, n, d).transpose(1, 2).contiguous()  # noqa: E731
            join = lambda t: t.transpose(1, 2).reshape(S, n * d)  # noqa: E731
            dp = torch.matmul(split(do), split(v).transpose(2, 3).contiguous())
            delta = (p * dp).sum(dim=3, keepdim=True)
            ds = p * (dp - delta) / math.sqrt(d)
            out["o"][rows, cols] = o
            out["dq"][rows, cols] = join(torch.matmul(ds, split(k)))
            out["dk"][rows, cols] = join(torch.matmul(ds.transpose(2, 3).contiguous(), split(q)))
            out["dv"][rows, cols] = join(torch.matmul(p.transpose(2, 3).contiguous(), split(do)))
            stats[b, h0:h1, :, 0] = m[0, :, :, 0]
            stats[b, h0:h1, :, 1] = 1 / l[0, :, :, 0]
            stats[b, h0:h1, :, 2] = delta[0, :, :, 0]
            stats[b, h0:h1, :, 3] = 0 if st is None else st.to(F64)[None]
    return {**out, "stats": stats.view(B * H * S, 4)}


def _quantized64(x, dim):
    """Symmetric int8 levels and scales along `dim` (max|x| / 127, halves away
    from zero), the scale rounded to f32 as it is stored."""
    s = x.abs().amax(dim=dim, keepdim=True) / 127.0
    s = torch.where(s == 0, torch.ones_like(s), s.clamp_min(torch.finfo(torch.float32).tiny))
    r = x / s
    lv = torch.sign(r) * torch.floor(r.abs() + 0.5)
    return lv.clamp(-127, 127).to(F64), s.to(F64)


def _xent64(logits, labels, masked):
    keep = labels >= 0 if masked else torch.ones_like(labels, dtype=torch.bool)
    m = logits.amax(dim=1, keepdim=True)
    e = torch.exp(logits - m)
    p = e / e.sum(dim=1, keepdim=True)
    at = labels.clamp_min(0).long()[:, None]
    count = keep.sum().to(F64)
    term = -torch.log(p.gather(1, at)[:, 0])
    loss = (term * keep).sum() / count if int(count) else torch.zeros((), dtype=F64, device="cuda")
    g = p.clone()
    g.scatter_add_(1, at, torch.full_like(at, -1, dtype=F64))
    g = g * keep[:, None] / count if int(count) else torch.zeros_like(p)
    return loss.view(1), p, g


def _adamw64(p, g, m, v, clip, step, lr):
    if clip > 0:
        norm = g.square().sum().sqrt()
        g = g * torch.clamp(clip / norm, max=1.0)
    b1, b2 = ADAMW["beta1"], ADAMW["beta2"]
    m = b1 * m + (1 - b1) * g
    v = b2 * v + (1 - b2) * g * g
    mh, vh = m / (1 - b1 ** step), v / (1 - b2 ** step)
    return p - lr * (mh / (vh.sqrt() + ADAMW["eps"]) + ADAMW["weight_decay"] * p), m, v


def _rope64(x, B, S, H, d, base=10000.0):
    pos = torch.arange(S, device=x.device, dtype=F64)[:, None]
    ang = pos * base ** (-2.0 * torch.arange(d // 2, device=x.device, dtype=F64) / d)[None]
    c, s = torch.cos(ang)[None, :, None], torch.sin(ang)[None, :, None]
    y = x.view(B, S, H, d // 2, 2)
    a, b = y[..., 0], y[..., 1]
    return torch.stack((a * c - b * s, a * s + b * c), dim=-1).view(B * S, H * d)


def _model64(case, img, planted, x, y, backward):
    """(loss, logits, gradients by adapter) of the plan's model."""
    P = {}
    for n, a in img.arrays.items():
        if n.endswith(".s"):
            continue
        t = torch.from_numpy(np.ascontiguousarray(planted.get(n, a))).cuda().to(F64)
        if a.dtype == np.int8:
            t = t * torch.from_numpy(img.arrays[n + ".s"]).cuda().to(F64)[None]
        P[n] = t
    params = [n for n in img.arrays if "m_" + n in img.arena]
    for n in params:
        P[n].requires_grad_(backward)
    site = lambda t, w, A, Bm: t @ P[w] + 2.0 * ((t @ P[A]) @ P[Bm])  # noqa: E731
    labels = torch.from_numpy(np.asarray(y)).cuda().long()
    if case["kind"] == "mlp":
        t = torch.from_numpy(x).cuda().to(F64)
        h = torch.relu(site(t, "W1", "A1", "B1") + P["b1"])
        logits = site(h, "W2", "A2", "B2") + P["b2"]
    else:
        q8, B, S, D = case["kind"] == "q8", case["batch"], case["seq"], case["dim"]
        H = D // 64

        def norm(t, g, b):
            if q8:
                return t / torch.sqrt((t * t).mean(dim=1, keepdim=True) + 1e-5) * P[g]
            c = t - t.mean(dim=1, keepdim=True)
            return c / torch.sqrt((c * c).mean(dim=1, keepdim=True) + 1e-5) * P[g] + P[b]

        def block(t, l):
            p = f"l{l}."
            n1 = norm(t, p + "g1", p + "b1")
            qkv = []
            for w in "qkv":
                on = q8 or w != "k"
                qkv.append(site(n1, p + "w" + w, p + "A" + w, p + "B" + w) if on else n1 @ P[p + "wk"])
            qkv[:2] = [_rope64(u, B, S, H, 64) for u in qkv[:2]]
            a = torch.cat([_attention64(*(u[i * S:(i + 1) * S] for u in qkv), None, 1, S, H, 64)[0]
                           for i in range(B)])
            t = t + (site(a, p + "wo", p + "Ao", p + "Bo") if q8 else a @ P[p + "wo"])
            n2 = norm(t, p + "g2", p + "b2")
            if q8:
                return t + (torch.nn.functional.silu(n2 @ P[p + "wg"]) * (n2 @ P[p + "wu"])) @ P[p + "wd"]
            return t + torch.nn.functional.gelu(n2 @ P[p + "wu"], approximate="tanh") @ P[p + "wd"]

        t = P["emb"][torch.from_numpy(x.view(np.int32)).cuda().long()]
        for l in range(case["layers"]):
            t = torch.utils.checkpoint.checkpoint(block, t, l, use_reentrant=False) if backward \
                else block(t, l)
        logits = norm(t, "gf", "bf") @ P["wh"]
    loss = torch.nn.functional.cross_entropy(logits, labels)
    if not backward:
        return loss.detach(), logits.detach(), None
    return loss.detach(), logits.detach(), dict(zip(params, torch.autograd.grad(
        loss, [P[n] for n in params])))


def exact(case, seed):
    kind, x = case["kind"], _inputs(case, seed)
    if kind == "w8a8":
        qa, sa = _quantized64(x["X"], 1)
        qw, sw = _quantized64(x["W"], 0)
        return {"C": (qa @ qw) * sa * sw, "QA": None, "sa": sa[:, 0]}
    if kind == "attn":
        return _exact_attn(case, x)
    if kind == "xent":
        loss, p, g = _xent64(x["logits"].to(F64), x["labels"], case["masked"])
        return {"loss": loss, "probs": p, "dlogits": g}
    if kind == "adamw":
        p, m, v = _adamw64(*(x[n].to(F64) for n in ("p", "g", "m", "v")), case["clip"],
                           ADAMW["step"], ADAMW["lr"])
        return {"p": p, "m": m, "v": v}
    img = _plan_of(case)
    planted = _planted(case, img, seed)
    loss, logits, grads = _model64(case, img, planted, x["x"], x["y"], kind != "eval")
    if kind == "eval":
        return {"loss": float(loss), "logits": logits.reshape(-1)}
    flat, order = [grads[n].reshape(-1) for n in grads], list(grads)
    new = []
    for n, g in zip(order, flat):
        p = torch.from_numpy(np.ascontiguousarray(planted.get(n, img.arrays[n]))).cuda().to(F64).view(-1)
        z = torch.zeros_like(p)
        new.append(_adamw64(p, g, z, z, 0.0, 1, 1e-3)[0])
    return {"loss": float(loss), "grads": flat if kind == "mlp" else [torch.cat(flat)],
            "adapters": torch.cat(new)}
