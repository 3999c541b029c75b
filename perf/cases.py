"""Performance cases of the BF16X engine: what a program that serves a model
with compressed weights has it do, each through a public entry point.

A case names a `kind` and its sizes:

  gemv      one token through a BF16X linear (generation, batch 1)
  linear    many tokens through a BF16X linear (batched generation, prefill)
  saturated the reference's plan-less product (bf16x_fused_gemm without the
            overflow table), any activation type
  decode    a compressed weight expanded to bf16
  encode    a bf16 weight on the GPU packed into the dict format
  plan      the overflow plan of a packed weight (part of loading a layer)
  gguf      tokens through a GGUF half-block weight, with the lossless table
  llama     a prompt through a small Llama-style stack, then decode steps

Weights follow the distributions the repository's benchmark uses: N(0, 0.02)
with 1 % of entries x 30 for the dict format, Student-t(3) x 0.015 for GGUF.
"""
import math

import torch

import bfloat16x_amd as bx
from bfloat16x_amd import gguf, llama

DEV = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# The linears of an 8B Llama-style layer (configuration 4) and of a 70B-class
# layer in GGUF blocks (configuration 5), as (out_f, in_f).
LISTED = [
    # k or v projection, one token: a launch of a few microseconds, so the
    # host call and the launch count most
    dict(name="gemv 1024x4096", kind="gemv", out_f=1024, in_f=4096, x="bf16"),
    # gate or up projection, one token: the headline of batch-1 generation
    dict(name="gemv 14336x4096", kind="gemv", out_f=14336, in_f=4096, x="bf16"),
    # down projection, 16 sequences decoded together
    dict(name="linear 4096x14336 M=16", kind="linear", out_f=4096, in_f=14336, rows=16, x="bf16"),
    # a short prompt (or a large decode batch) of odd length
    dict(name="linear 14336x4096 M=101", kind="linear", out_f=14336, in_f=4096, rows=101, x="bf16"),
    # a 512-token prompt
    dict(name="linear 14336x4096 M=512", kind="linear", out_f=14336, in_f=4096, rows=512, x="bf16"),
    # fused gate + up projection of a 2048-token prompt: the largest product
    dict(name="linear 28672x4096 M=2048", kind="linear", out_f=28672, in_f=4096, rows=2048, x="bf16"),
    # fp16 model: the reference's own product (saturated weight), 64 tokens
    dict(name="saturated 4096x4096 fp16", kind="saturated", out_f=4096, in_f=4096, rows=64, x="fp16"),
    # a weight expanded for a program that wants it in bf16
    dict(name="decode 14336x4096", kind="decode", out_f=14336, in_f=4096),
    # packing a layer of a bf16 model when it is deployed
    dict(name="encode 4096x14336", kind="encode", out_f=4096, in_f=14336),
    # the other half of deploying a layer: its overflow plan
    dict(name="plan 14336x4096", kind="plan", out_f=14336, in_f=4096),
    # GGUF o projection, lossless, a decode batch of 24
    dict(name="gguf 8192x8192 M=24", kind="gguf", out_f=8192, in_f=8192, rows=24),
    # a 512-token prompt and eight decode steps of a stack; three layers with
    # configuration 4's sizes and the vocabulary cut in proportion (3 / 32),
    # so the head keeps its share of a step
    dict(name="llama 512+8", kind="llama", layers=3, vocab=12032, prompt=512, steps=8),
]


def listed():
    return [dict(c) for c in LISTED]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "linear", "linear", "linear", "saturated", "decode", "encode", "plan", "gguf",
                       "gguf", "llama"])
    if kind == "llama":
        return dict(kind=kind, layers=rng.choice([2, 3]), vocab=8 * rng.randrange(500, 1505),
                    prompt=_log(rng, 17, 512), steps=rng.randrange(1, 9))
    # out_f: any number (a tensor-parallel shard, an odd head); in_f: the 64-
    # and 32-multiples that hidden and FFN sizes come in
    out_f = _log(rng, 256, 16384)
    if rng.random() < 0.6:
        out_f = -(-out_f // 128) * 128
    in_f = _log(rng, 512, 16384) // 256 * 256
    if rng.random() < 0.3:
        in_f += rng.choice([32, 64, 128])
    while out_f * in_f > 14336 * 4096:                 # no larger than a listed weight
        out_f = -(-out_f // 2)
    x = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
    if kind == "gemv":
        return dict(kind=kind, out_f=out_f, in_f=in_f, x=x)
    if kind == "linear":
        return dict(kind=kind, out_f=out_f, in_f=in_f, rows=_log(rng, 2, 1024), x=x)
    if kind == "saturated":
        return dict(kind=kind, out_f=out_f, in_f=in_f, rows=_log(rng, 2, 512), x=x)
    if kind == "gguf":
        return dict(kind=kind, out_f=min(out_f, 8192), in_f=min(in_f, 8192), rows=_log(rng, 1, 512))
    if kind == "decode" and rng.random() < 0.25:
        in_f -= 8 * rng.randrange(1, 4)                # rows that do not end on a block
    return dict(kind=kind, out_f=out_f, in_f=in_f)


def _gen(seed, k):
    return torch.Generator(device=DEV).manual_seed(1_000_003 * (seed + 1) + k)


def _weight(case, seed):
    g = _gen(seed, 1)
    w = torch.randn(case["out_f"], case["in_f"], generator=g, device=DEV) * 0.02
    big = torch.rand(w.shape, generator=g, device=DEV) < 0.01
    return torch.where(big, w * 30.0, w).to(torch.bfloat16)


def _weight_t(case, seed):
    """Student-t(3) x 0.015, in bf16."""
    g = _gen(seed, 2)
    shape = (case["out_f"], case["in_f"])
    z = torch.randn(shape, generator=g, device=DEV)
    c = torch.zeros(shape, device=DEV)
    for _ in range(3):
        c += torch.randn(shape, generator=g, device=DEV).square_()
    return (z * torch.rsqrt(c / 3.0) * 0.015).to(torch.bfloat16)


def _x(case, seed):
    g = _gen(seed, 3)
    x = torch.randn(case.get("rows", 1), case["in_f"], generator=g, device=DEV)
    return x.to(DTYPES[case.get("x", "bf16")])


def _tokens(case, seed):
    g = _gen(seed, 4)
    return (torch.randint(0, case["vocab"], (case["prompt"],), generator=g, device=DEV),
            torch.randint(0, case["vocab"], (case["steps"],), generator=g, device=DEV))


def _stack(case, seed):
    cfg = llama.LlamaConfig(n_layers=case["layers"], vocab=case["vocab"])
    return llama.LlamaStack(cfg, device=DEV, seed=seed)


def _weight_rows(case, seed):
    """_weight's rows in an order, with signs, of the seed's own: the table
    that packing writes has the same length for every seed."""
    g = _gen(seed, 5)
    w = _weight(case, 0)[torch.randperm(case["out_f"], generator=g, device=DEV)]
    flip = torch.rand(w.shape, generator=g, device=DEV) < 0.5
    return torch.where(flip, -w, w)


@torch.no_grad()
def prepare(case, seed):
    kind = case["kind"]
    if kind in ("gemv", "linear"):
        mod = bx.Bf16xFused(bx.bf16x_quantize(_weight(case, seed)), keep_cpu=False)
        return dict(kind=kind, mod=mod, x=_x(case, seed))
    if kind == "saturated":
        return dict(kind=kind, d=bx.bf16x_quantize(_weight(case, seed)), x=_x(case, seed))
    if kind == "decode":
        d = bx.bf16x_quantize(_weight(case, seed))
        return dict(kind=kind, d=d, plan=bx.build_plan_host(d, device=DEV))
    if kind == "encode":
        return dict(kind=kind, w=_weight_rows(case, seed))
    if kind == "plan":
        return dict(kind=kind, d=bx.bf16x_quantize(_weight_rows(case, seed)))
    if kind == "gguf":
        w = _weight_t(case, seed)
        blocks = gguf.quantize_blocks(w)
        return dict(kind=kind, blocks=gguf.device_blocks(blocks, DEV), x=_x(case, seed),
                    ovf=gguf.device_ovf(gguf.pack_ovf(w), blocks, DEV), out_f=case["out_f"], in_f=case["in_f"])
    model = _stack(case, seed)
    bx.deploy_bf16x_fused(model, verbose=False)
    ids, forced = _tokens(case, seed)
    runner = llama.LlamaRunner(model, max_len=case["prompt"] + case["steps"] + 120, max_new=case["steps"] + 1,
                               max_prompt=case["prompt"])
    runner.prefill(ids)
    runner.capture()
    return dict(kind=kind, runner=runner, ids=ids, forced=forced)


@torch.no_grad()
def run(state):
    kind = state["kind"]
    if kind in ("gemv", "linear"):
        return state["mod"](state["x"])
    if kind == "saturated":
        d = state["d"]
        return bx.bf16x_fused_gemm(state["x"], d["sign_packed"], d["mant_packed"], d["delta_packed"], d["emax"],
                                   d["out_f"], d["in_f"])
    if kind == "decode":
        d = state["d"]
        return bx.bf16x_decode(d["sign_packed"], d["mant_packed"], d["delta_packed"], d["emax"], d["out_f"],
                               d["in_f"], plan=state["plan"])
    if kind == "encode":
        d = bx.bf16x_quantize(state["w"])
        return {k: d[k] for k in ("emax", "sign_packed", "mant_packed", "delta_packed", "delta_ovf_idx",
                                  "delta_ovf_val")}
    if kind == "plan":
        p = bx.build_plan_host(state["d"], device=DEV)
        return {"tile_off": p.tile_off, "tile_ent": p.tile_ent, "tile_sat": p.tile_sat, "n_fix": p.n_fix}
    if kind == "gguf":
        return gguf.gguf_gemm(state["x"], state["blocks"], state["out_f"], state["in_f"], ovf=state["ovf"])
    r, forced = state["runner"], state["forced"]
    r.prefill(state["ids"])
    first = r.logits
    for i in range(forced.numel()):                    # scoring a given continuation
        r.token.copy_(forced[i:i + 1])
        r.decode(1, check=False)
    return {"prompt": first, "last": r.logits}


def _dict_bytes(out_f, in_f):
    """Streams and emax of a packed weight (11 bits and 1/16 byte per element)."""
    n = out_f * in_f
    return n * 11 / 8 + n / 16


OVF = 0.0264     # delta >= 7 entries per element at this distribution
FIX = 0.0231     # of them, delta > 7


def work(case):
    kind = case["kind"]
    if kind == "llama":
        cfg = llama.LlamaConfig(n_layers=case["layers"], vocab=case["vocab"])
        lin = cfg.linear_params()
        passes, tok = 1 + case["steps"], case["prompt"] + case["steps"]
        kv = 2 * 2 * cfg.n_layers * cfg.n_kv_heads * 128 * (case["prompt"] * (1 + case["steps"]))
        attn = 4 * cfg.n_layers * cfg.hidden * (case["prompt"] ** 2 / 2 + case["steps"] * case["prompt"])
        head = cfg.vocab * cfg.hidden
        return {"bytes": passes * (lin * (11 / 8 + 1 / 16) + 2 * head) + kv,
                "flops": 2 * lin * tok + 2 * head * passes + attn}
    out_f, in_f = case["out_f"], case["in_f"]
    n = out_f * in_f
    if kind == "decode":
        return {"bytes": _dict_bytes(out_f, in_f) + 5 * FIX * n + 2 * n, "flops": 0}
    if kind == "encode":
        return {"bytes": 2 * n + _dict_bytes(out_f, in_f) + 5 * OVF * n, "flops": 0}
    if kind == "plan":
        return {"bytes": (5 * OVF + 5 * FIX) * n + 4 * out_f, "flops": 0}
    rows = case.get("rows", 1)
    xb = 2 if case.get("x", "bf16") != "fp32" else 4
    yb = 2 if kind == "gemv" else xb
    if kind == "gguf":
        wb = n * 46 / 32 + 4 * 0.033 * n
    else:
        wb = _dict_bytes(out_f, in_f) + (0 if kind == "saturated" else 5 * FIX * n)
    return {"bytes": wb + rows * (xb * in_f + yb * out_f), "flops": 2 * rows * n}


def tolerance(case):
    """Products are held in fp32 and rounded once to the output type.  Measured
    against float64 (2-norm / largest): bf16 outputs 1.7e-3 / 3.9e-3, fp16
    2.1e-4 / 4.9e-4, fp32 2.5e-6 / 1.6e-5 (activations split into two bf16
    terms, 16 significant bits); allowed is four times that.  The stack's
    logits move by 1.0e-2 / 4.3e-2 when its products run through the decode
    and a library GEMM instead.  Integers and decoded weights are bit for
    bit."""
    kind = case["kind"]
    if kind in ("decode", "encode", "plan"):
        return "exact"
    if kind == "llama":
        return {"rel": 3e-2, "max": 1.6e-1}
    if kind != "gemv" and case.get("x") == "fp32":
        return {"rel": 1e-5, "max": 7e-5}
    if kind != "gemv" and case.get("x") == "fp16":
        return {"rel": 8e-4, "max": 2e-3}
    return {"rel": 6e-3, "max": 1.6e-2}


def _saturated(w):
    """The weight with every overflowing exponent raised to its block's
    maximum minus 7 (at least 0), as the plan-less product uses it."""
    bits = w.view(torch.int16).to(torch.int32) & 0xFFFF
    e = (bits >> 7) & 0xFF
    pad = (-bits.numel()) % 16
    em = torch.nn.functional.pad(e.reshape(-1), (0, pad)).view(-1, 16).amax(1).repeat_interleave(16)[:e.numel()]
    e = torch.maximum(e, (em.view_as(e) - 7).clamp_min(0))
    return ((bits & 0x807F) | (e << 7)).to(torch.int16).view(torch.bfloat16)


def _rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w


def _forward64(model, ids):
    """Logits of every position, the stack's bf16 weights in float64."""
    cfg = model.cfg
    H, KV, D, T = cfg.n_heads, cfg.n_kv_heads, 128, ids.numel()
    inv = 1.0 / (cfg.rope_theta ** (torch.arange(0, D, 2, dtype=torch.int64).float() / D))
    ang = torch.outer(torch.arange(T, dtype=torch.float32), inv).to(DEV)
    c, s = ang.cos().double()[:, None], ang.sin().double()[:, None]

    def rope(t):
        a, b = t[..., :64], t[..., 64:]
        return torch.cat([a * c - b * s, b * c + a * s], dim=-1)

    def lin(t, mod):
        return t @ mod.weight.double().t().contiguous()

    b4 = torch.arange(cfg.ffn // 4, device=DEV)[:, None] * 8 + torch.arange(4, device=DEV)
    gate, up = b4.reshape(-1), (b4 + 4).reshape(-1)      # gate_up rows come in groups of 4 gate, 4 up
    mask = torch.full((T, T), float("-inf"), device=DEV, dtype=torch.float64).triu(1)
    x = model.embed[ids].double()
    for lay in model.layers:
        qkv = lin(_rms(x, lay.attn_norm.double(), cfg.eps), lay.qkv).view(T, H + 2 * KV, D)
        q, k = rope(qkv[:, :H]), rope(qkv[:, H:H + KV]).repeat_interleave(H // KV, 1)
        v = qkv[:, H + KV:].repeat_interleave(H // KV, 1)
        heads = []
        for h in range(H):
            p = torch.softmax(q[:, h] @ k[:, h].t().contiguous() / math.sqrt(D) + mask, dim=-1)
            heads.append(p @ v[:, h].contiguous())
        x = x + lin(torch.cat(heads, dim=-1), lay.o)
        gu = lin(_rms(x, lay.mlp_norm.double(), cfg.eps), lay.gate_up)
        x = x + lin(torch.nn.functional.silu(gu[:, gate]) * gu[:, up], lay.down)
    return lin(_rms(x, model.norm.double(), cfg.eps), model.lm_head)


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind in ("encode", "plan"):
        return None
    if kind == "decode":
        return _weight(case, seed)
    if kind == "llama":
        ids, forced = _tokens(case, seed)
        y = _forward64(_stack(case, seed), torch.cat([ids, forced]))
        return {"prompt": y[ids.numel() - 1], "last": y[-1]}
    w = _weight_t(case, seed) if kind == "gguf" else _weight(case, seed)
    if kind == "saturated":
        w = _saturated(w)
    return _x(case, seed).double() @ w.double().t().contiguous()
