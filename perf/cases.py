"""The work that a user of this package has it do, as cases that can be timed and compared.

Every case goes through the package's public entry points on inputs made from
a seed.  The kinds, and what each stands for in use:

* ``linear``: one W4A16 g128 linear, fp16 or bf16, any row count from the
  single camera token of one frame to the tokens of eight frames: ``WQLinear``
  for a plain or biased layer, ``w4a16_linear`` for a biased layer with GELU,
  ``gemm_forward_cuda_new`` for the extension's own op (no bias).
* ``w8a8_linear``: the extension's W8A8 pair, per-token quantisation of the
  activations and the int8 GEMM with bias on the stored weight.
* ``attention``: the flash attention op on a packed qkv buffer; ``batch``
  sequences of ``seq`` tokens, 16 heads of 64 (frame attention: one sequence
  of 1374 tokens a frame; global attention: one sequence of all frames).
* ``block``: one alternating-attention block (frame or global attention, W4A16
  or W8A8 linears), what a program with its own model graph calls per layer.
* ``dino``: one fp16 block of the DINOv2 patch embed.
* ``camera``: the whole camera head (4 iterations), eager or as the recorded
  HIP graph, one pose token a frame.
* ``aggregator``: the whole VGGT-1B aggregator, images to the layer outputs
  that the model's heads read.
"""
from __future__ import annotations

import math

import torch

from qvggt_amd import awq_inference_engine as engine
from qvggt_amd import camera_head as ch
from qvggt_amd.aggregator import AABlock, Aggregator, AggregatorConfig, DinoBlock, W8A8Linear
from qvggt_amd.awq import WQLinear, pack_intweight

TOKENS = 1374                 # tokens of one frame: 1 camera + 4 registers + 37 x 37 patches
DIM, HEADS, HD, MLP = 1024, 16, 64, 4096
DEPTH = 24                    # frame, global and patch-embed blocks of the aggregator
HEAD_LAYERS = (4, 11, 17, 23)
BLOCK_EPS = 1e-6
ROPE_ROWS = 38                # positions 0..37 of the 37 x 37 patch grid
# (in, out) of the quantised linears: the aggregator's blocks, the camera head's trunk
SHAPES = ((1024, 3072), (1024, 1024), (1024, 4096), (4096, 1024),
          (2048, 6144), (2048, 2048), (2048, 8192), (8192, 2048))


def _dev():
    return torch.device("cuda", torch.cuda.current_device())


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # a camera-head trunk layer for one frame: launch latency and the weight stream
        dict(name="linear_1_token", kind="linear", m=1, k=2048, n=8192, dtype="float16", epilogue="bias"),
        # the qkv projection of one frame: the smallest call of an aggregator block
        dict(name="linear_qkv_1_frame", kind="linear", m=1374, k=1024, n=3072, dtype="float16", epilogue="bias"),
        # the extension's GEMM in bf16 on a ragged number of tokens (crops, merged tokens), long K
        dict(name="linear_bf16_ragged", kind="linear", m=3001, k=4096, n=1024, dtype="bfloat16", epilogue="none"),
        # fc1 with its GELU for eight frames: the benchmark's layer
        dict(name="linear_fc1_8_frames", kind="linear", m=10992, k=1024, n=4096, dtype="float16", epilogue="gelu"),
        # the drop-in W8A8 ops on the weight as stored, four frames, fc2's shape
        dict(name="w8a8_linear_4_frames", kind="w8a8_linear", m=5496, k=4096, n=1024),
        # attention inside one frame: the smallest attention call
        dict(name="attention_1_frame", kind="attention", batch=1, seq=1374),
        # global attention over 32 frames: the largest single call of the model
        dict(name="attention_global_32", kind="attention", batch=1, seq=43968),
        # a frame block with W4A16 linears at eight frames
        dict(name="block_w4_frame_8", kind="block", quant="w4", frames=8, rows=37, attend="frame"),
        # a global block with W8A8 linears at three frames
        dict(name="block_w8_global_3", kind="block", quant="w8", frames=3, rows=37, attend="global"),
        # a patch-embed block at six frames
        dict(name="dino_block_6", kind="dino", frames=6),
        # the camera head as a program calls it, eight frames
        dict(name="camera_head_8", kind="camera", frames=8, graph=False),
        # the whole aggregator on four frames
        dict(name="aggregator_w4_4", kind="aggregator", quant="w4", frames=4),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("linear",) * 6 + ("w8a8_linear",) * 2 + ("attention",) * 4 + ("block",) * 4 + ("dino",) + ("camera",) * 2
                      + ("aggregator",))
    if kind == "linear":
        m = _log(rng, 1, 12288)
        k, n = rng.choice(SHAPES) if rng.random() < 0.75 else (128 * rng.randint(1, 48), 16 * rng.randint(8, 320))
        return dict(kind=kind, m=m, k=k, n=n, dtype=rng.choice(("float16", "float16", "bfloat16")),
                    epilogue=rng.choice(("none", "bias", "gelu")))
    if kind == "w8a8_linear":
        k, n = rng.choice(SHAPES[:4])
        return dict(kind=kind, m=_log(rng, 1, 12288), k=k, n=n)
    if kind == "attention":
        if rng.random() < 0.5:
            return dict(kind=kind, batch=rng.randint(1, 32), seq=_log(rng, 70, 1500))
        return dict(kind=kind, batch=1, seq=_log(rng, 1000, 40000))
    if kind == "block":
        # 518 pixels wide, 294 to 518 high: 21 to 37 rows of 37 patches
        return dict(kind=kind, quant=rng.choice(("w4", "w4", "w8")), frames=_log(rng, 1, 16), rows=rng.randint(21, 37),
                    attend=rng.choice(("frame", "global")))
    if kind == "dino":
        return dict(kind=kind, frames=rng.choice((1, 2, 3, 4, 5, 7, 9, 11, 13, 16)))
    if kind == "camera":
        return dict(kind=kind, frames=_log(rng, 1, 80), graph=rng.random() < 0.5)
    quant, frames = rng.choice((("w4", 1), ("w4", 2), ("w4", 3), ("w8", 1), ("w8", 2), ("w8", 3), ("w8", 4)))
    return dict(kind=kind, quant=quant, frames=frames)


# ------------------------------------------------- inputs and weights from a seed
def _gen(seed, part):
    return torch.Generator(device=_dev()).manual_seed((int(seed) * 1000003 + part * 7919) % (1 << 62))


def _randn(g, *shape, std=1.0, mean=0.0, dtype=torch.float16):
    return (torch.randn(*shape, generator=g, device=g.device) * std + mean).to(dtype)


def _w4_layer(g, k, n, dtype=torch.float16):
    """int4 codes, group scales and integer zeros of an (n, k) layer whose
    weights spread about like N(0, 0.03), and its bias."""
    return {
        "q": torch.randint(0, 16, (n, k), generator=g, device=g.device, dtype=torch.uint8),
        "s": (torch.rand(k // 128, n, generator=g, device=g.device) * 0.004 + 0.004).to(dtype),
        "z": torch.randint(6, 11, (k // 128, n), generator=g, device=g.device).float(),
        "b": _randn(g, n, std=0.02, dtype=dtype),
    }


def _w4_module(p, bias=True):
    n, k = p["q"].shape
    m = WQLinear(4, 128, k, n, bias, p["q"].device, dtype=p["s"].dtype)
    m.qweight.copy_(pack_intweight(p["q"], 4, 64))
    m.scales[:k // 128] = p["s"]
    m.scaled_zeros[:k // 128] = -(p["s"].float() * p["z"]).to(p["s"].dtype)
    if bias:
        m.bias.copy_(p["b"])
    return m


def _w4_weight(p):
    """The (n, k) weights that the codes stand for, as the format defines them
    (one rounding to the tables' type), in 64 bits."""
    dt = p["s"].dtype
    s = p["s"].double().t().repeat_interleave(128, 1)
    sz = (p["s"].float() * p["z"]).to(dt).double().t().repeat_interleave(128, 1)
    return (p["q"].double() * s - sz).to(dt).double()


def _w8_layer(g, k, n):
    return {
        "w": torch.randint(-127, 128, (n, k), generator=g, device=g.device, dtype=torch.int16).to(torch.int8),
        "ws": (torch.rand(n, generator=g, device=g.device) * 2e-4 + 2e-4).half(),
        "b": _randn(g, n, std=0.02),
    }


def _w8_module(p):
    n, k = p["w"].shape
    m = W8A8Linear(k, n, True, p["w"].device)
    m.weight.copy_(p["w"])
    m.wscales.copy_(p["ws"])
    m.bias.copy_(p["b"])
    return m


def _fp16_layer(g, k, n):
    return {"w": _randn(g, n, k, std=0.02), "b": _randn(g, n, std=0.02)}


def _ln_params(g, d):
    return _randn(g, d, std=0.1, mean=1.0), _randn(g, d, std=0.1)


def _gamma(g, d):
    return ((torch.rand(d, generator=g, device=g.device) + 0.5) * 0.1).half()


def _block_params(g, quant):
    layer = {"w4": _w4_layer, "w8": _w8_layer, "fp16": _fp16_layer}[quant]
    p = {"qkv": layer(g, DIM, 3 * DIM), "proj": layer(g, DIM, DIM), "fc1": layer(g, DIM, MLP), "fc2": layer(g, MLP, DIM),
         "norm1": _ln_params(g, DIM), "norm2": _ln_params(g, DIM), "ls1": _gamma(g, DIM), "ls2": _gamma(g, DIM)}
    if quant != "fp16":
        p["q_norm"], p["k_norm"] = _ln_params(g, HD), _ln_params(g, HD)
    return p


def _set_norm(ln, p):
    ln.weight.data.copy_(p[0])
    ln.bias.data.copy_(p[1])


def _set_linear(l, p):
    l.weight.data.copy_(p["w"])
    l.bias.data.copy_(p["b"])


def _block_module(p, quant):
    make = _w4_module if quant == "w4" else _w8_module
    b = AABlock(make(p["qkv"]), make(p["proj"]), make(p["fc1"]), make(p["fc2"]), quant == "w8", _dev(), BLOCK_EPS)
    for ln, name in ((b.norm1, "norm1"), (b.norm2, "norm2"), (b.attn.q_norm, "q_norm"), (b.attn.k_norm, "k_norm")):
        _set_norm(ln, p[name])
    b.ls1.gamma.data.copy_(p["ls1"])
    b.ls2.gamma.data.copy_(p["ls2"])
    return b


def _fill_dino(blk, p):
    _set_norm(blk.norm1, p["norm1"])
    _set_norm(blk.norm2, p["norm2"])
    for l, name in ((blk.attn.qkv, "qkv"), (blk.attn.proj, "proj"), (blk.mlp.fc1, "fc1"), (blk.mlp.fc2, "fc2")):
        _set_linear(l, p[name])
    blk.ls1.gamma.data.copy_(p["ls1"])
    blk.ls2.gamma.data.copy_(p["ls2"])
    return blk


def _scratch(m, w8):
    """The scratch buffers that a block works in, kept by its caller."""
    f16 = dict(dtype=torch.float16, device=_dev())
    ws = {"h": torch.empty(m, DIM, **f16), "qkv": torch.empty(m, 3 * DIM, **f16), "att": torch.empty(m, DIM, **f16),
          "o": torch.empty(m, DIM, **f16), "f": torch.empty(m, MLP, **f16)}
    if w8:
        ws.update(q8=torch.empty(m, DIM, dtype=torch.int8, device=_dev()),
                  q8f=torch.empty(m, MLP, dtype=torch.int8, device=_dev()), s8=torch.empty(m, **f16))
    return ws


def _camera_params(seed):
    g = _gen(seed, 1)
    d = ch.DIM
    p = {"trunk": []}
    for _ in range(ch.TRUNK_DEPTH):
        p["trunk"].append({
            "qkv": _w4_layer(g, d, 3 * d), "proj": _w4_layer(g, d, d), "fc1": _w4_layer(g, d, 4 * d),
            "fc2": _w4_layer(g, 4 * d, d), "norm1": _ln_params(g, d), "norm2": _ln_params(g, d),
            "ls1": _gamma(g, d), "ls2": _gamma(g, d)})
    p["token_norm"], p["trunk_norm"] = _ln_params(g, d), _ln_params(g, d)
    p["embed"], p["mod"] = _fp16_layer(g, ch.POSE_DIM, d), _fp16_layer(g, d, 3 * d)
    p["fc1"], p["fc2"] = _fp16_layer(g, d, d // 2), _fp16_layer(g, d // 2, ch.POSE_DIM)
    p["empty"] = _randn(g, 1, 1, ch.POSE_DIM, std=0.02)
    return p


def _camera_module(p):
    head = ch.CameraHead([tuple(_w4_module(t[n]) for n in ("qkv", "proj", "fc1", "fc2")) for t in p["trunk"]], _dev())
    for blk, t in zip(head.trunk, p["trunk"]):
        _set_norm(blk.norm1, t["norm1"])
        _set_norm(blk.norm2, t["norm2"])
        blk.ls1.gamma.data.copy_(t["ls1"])
        blk.ls2.gamma.data.copy_(t["ls2"])
    _set_norm(head.token_norm, p["token_norm"])
    _set_norm(head.trunk_norm, p["trunk_norm"])
    _set_linear(head.embed_pose, p["embed"])
    _set_linear(head.poseLN_modulation[1], p["mod"])
    _set_linear(head.pose_branch.fc1, p["fc1"])
    _set_linear(head.pose_branch.fc2, p["fc2"])
    head.empty_pose_tokens.data.copy_(p["empty"])
    return head


# part numbers of the aggregator's generators: one a block, so that a block's
# weights can be made again without those before it
_FRAME, _GLOBAL, _DINO, _REST = 100, 200, 300, 400


def _embed_params(seed):
    g = _gen(seed, _REST)
    return {"proj_w": _randn(g, DIM, 3, 14, 14, std=0.02), "proj_b": _randn(g, DIM, std=0.02),
            "cls": _randn(g, 1, 1, DIM, std=0.02), "reg": _randn(g, 1, 4, DIM, std=0.02),
            "pos": _randn(g, 1, 1 + 37 * 37, DIM, std=0.02), "norm": _ln_params(g, DIM),
            "camera": _randn(g, 1, 2, 1, DIM, std=0.02), "register": _randn(g, 1, 2, 4, DIM, std=0.02)}


def _images(case, seed):
    g = _gen(seed, 2)
    return torch.rand(case["frames"], 3, 518, 518, generator=g, device=g.device).half()


def _frame_tokens(case):
    return 5 + 37 * case.get("rows", 37)


def _tokens(case, seed):
    """Residual-stream tokens of a block's input."""
    return _randn(_gen(seed, 2), case["frames"] * _frame_tokens(case), DIM)


def _positions(case):
    """(y, x) of every token: 0 for the 5 special tokens of a frame, patch (i, j) at (i + 1, j + 1)."""
    i = torch.arange(_frame_tokens(case) - 5, device=_dev())
    patch = torch.stack([i // 37 + 1, i % 37 + 1], 1)
    frame = torch.cat([torch.zeros(5, 2, dtype=torch.long, device=_dev()), patch])
    return frame.repeat(case["frames"], 1).to(torch.int32)


# ------------------------------------------------------------ prepare and run
@torch.no_grad()
def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        dt = getattr(torch, case["dtype"])
        p = _w4_layer(_gen(seed, 1), case["k"], case["n"], dt)
        return {"case": case, "x": _randn(_gen(seed, 2), case["m"], case["k"], dtype=dt),
                "layer": _w4_module(p, case["epilogue"] != "none")}
    if kind == "w8a8_linear":
        p = _w8_layer(_gen(seed, 1), case["k"], case["n"])
        return dict(p, case=case, x=_randn(_gen(seed, 2), case["m"], case["k"]))
    if kind == "attention":
        return {"case": case, "qkv": _randn(_gen(seed, 2), case["batch"] * case["seq"], 3, HEADS, HD)}
    if kind == "block":
        m = case["frames"] * _frame_tokens(case)
        return {"case": case, "block": _block_module(_block_params(_gen(seed, 1), case["quant"]), case["quant"]),
                "x": _tokens(case, seed), "pos": _positions(case),
                "tables": engine.rope2d_tables(ROPE_ROWS, 100.0, device=_dev()),
                "ws": _scratch(m, case["quant"] == "w8")}
    if kind == "dino":
        return {"case": case, "block": _fill_dino(DinoBlock(_dev()), _block_params(_gen(seed, 1), "fp16")),
                "x": _tokens(case, seed), "ws": _scratch(case["frames"] * TOKENS, False)}
    if kind == "camera":
        head = _camera_module(_camera_params(seed))
        call = ch.GraphedCameraHead(head, case["frames"]) if case["graph"] else head
        return {"case": case, "head": call, "tokens": _randn(_gen(seed, 2), case["frames"], ch.DIM)}
    quant = case["quant"]
    blocks = [[_block_module(_block_params(_gen(seed, part + i), quant), quant) for i in range(DEPTH)]
              for part in (_FRAME, _GLOBAL)]
    agg = Aggregator(blocks[0], blocks[1], quant == "w8", _dev(), AggregatorConfig())
    for i, blk in enumerate(agg.patch_embed.blocks):
        _fill_dino(blk, _block_params(_gen(seed, _DINO + i), "fp16"))
    e, pe = _embed_params(seed), agg.patch_embed
    pe.patch_embed.proj.weight.data.copy_(e["proj_w"])
    pe.patch_embed.proj.bias.data.copy_(e["proj_b"])
    pe.cls_token.data.copy_(e["cls"])
    pe.register_tokens.data.copy_(e["reg"])
    pe.pos_embed.data.copy_(e["pos"])
    _set_norm(pe.norm, e["norm"])
    agg.camera_token.data.copy_(e["camera"])
    agg.register_token.data.copy_(e["register"])
    return {"case": case, "model": agg, "images": _images(case, seed)}


@torch.no_grad()
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        x, l = state["x"], state["layer"]
        if case["epilogue"] == "none":
            return engine.gemm_forward_cuda_new(x, l.qweight, l.scales, l.scaled_zeros)
        if case["epilogue"] == "gelu":
            return engine.w4a16_linear(x, l.qweight, l.scales, l.scaled_zeros, bias=l.bias, epilogue=2)
        return l(x)
    if kind == "w8a8_linear":
        x = state["x"]
        q = torch.empty(x.shape, dtype=torch.int8, device=x.device)
        s = torch.empty(x.shape[0], dtype=torch.float16, device=x.device)
        out = torch.empty(x.shape[0], case["n"], dtype=torch.float16, device=x.device)
        engine.invoke_quant(q, x, s)
        engine.w8a8_gemm_fuse_bias_forward_cuda(q, state["w"], state["ws"], s, out, state["b"])
        return q, s, out
    if kind == "attention":
        qkv = state["qkv"]
        return engine.attention(qkv[:, 0], qkv[:, 1], qkv[:, 2], case["seq"])
    if kind == "block":
        x = state["x"].clone()          # the block works in place on its caller's residual stream
        seq = _frame_tokens(case) if case["attend"] == "frame" else x.shape[0]
        return state["block"](x, seq, state["pos"], state["tables"], state["ws"])
    if kind == "dino":
        return state["block"](state["x"].clone(), state["ws"])
    if kind == "camera":
        return state["head"](state["tokens"])
    return state["model"](state["images"])


# ------------------------------------------------------------- work, tolerance
def _block_flops(m, seq):
    return 2.0 * m * DIM * (3 * DIM + DIM + 2 * MLP) + 4.0 * m * seq * DIM


def _weight_bytes(k, n, quant):
    return {"w4": n * k / 2 + 4 * (k / 128) * n, "w8": n * k + 2 * n, "fp16": 2 * n * k}[quant] + 2 * n


def _block_bytes(m, quant):
    return 4.0 * m * DIM + sum(_weight_bytes(k, n, quant) for k, n in SHAPES[:4])


def work(case):
    kind = case["kind"]
    if kind in ("linear", "w8a8_linear"):
        m, k, n = case["m"], case["k"], case["n"]
        extra = m * k + 2 * m if kind == "w8a8_linear" else 0   # the int8 codes and scales are results too
        return {"bytes": 2 * m * k + 2 * m * n + extra + _weight_bytes(k, n, "w4" if kind == "linear" else "w8"),
                "flops": 2.0 * m * k * n}
    if kind == "attention":
        t = case["batch"] * case["seq"]
        return {"bytes": 8.0 * t * DIM, "flops": 4.0 * t * case["seq"] * DIM}
    if kind == "camera":
        s, d = case["frames"], ch.DIM
        w4 = sum(_weight_bytes(k, n, "w4") for k, n in SHAPES[4:]) * ch.TRUNK_DEPTH
        flops = 4 * (ch.TRUNK_DEPTH * (2.0 * s * d * 12 * d + 4.0 * s * s * d) + 2.0 * s * d * (3 * d + d // 2))
        return {"bytes": w4 + 2 * (3 * d * d + d * d // 2) + 2 * s * d + 4 * 36 * s, "flops": flops}
    seq = _frame_tokens(case)
    m = case["frames"] * seq
    if kind == "block":
        return {"bytes": _block_bytes(m, case["quant"]),
                "flops": _block_flops(m, seq if case["attend"] == "frame" else m)}
    if kind == "dino":
        return {"bytes": _block_bytes(m, "fp16"), "flops": _block_flops(m, TOKENS)}
    weights = DEPTH * (2 * (_block_bytes(0, case["quant"])) + _block_bytes(0, "fp16"))
    return {"bytes": weights + 2.0 * case["frames"] * 3 * 518 * 518 + 2.0 * m * DIM * (1 + 2 * len(HEAD_LAYERS)),
            "flops": DEPTH * (2 * _block_flops(m, TOKENS) + _block_flops(m, m)) + 2.0 * m * 588 * DIM}


# About four times the largest error against 64 bits that a correct path at
# these types shows (measured): one rounding of a 16-bit output for a linear
# (2.1e-4 in fp16, 1.7e-3 in bf16); attention rounds its probabilities to fp16
# too (3.7e-4); the blocks add the roundings of their intermediate tensors
# (3.0e-4, W8A8 7e-4 from activation codes next to a rounding boundary); the
# camera head feeds its fp16 residual stream through 16 blocks (1.7e-3) and
# the aggregator through 72 (1.2e-3, W8A8 8.8e-3).
def tolerance(case):
    kind = case["kind"]
    if kind == "linear":
        return {"rel": 7e-3} if case["dtype"] == "bfloat16" else {"rel": 1e-3}
    if kind == "w8a8_linear":
        # the int8 codes are whole numbers and fixed by the op's definition
        return {"rel": 1e-3, "differ": 0.0}
    if kind == "attention":
        return {"rel": 1.5e-3}
    if kind == "block":
        return {"rel": 1.2e-3} if case["quant"] == "w4" else {"rel": 3e-3}
    if kind == "dino":
        return {"rel": 1.2e-3}
    if kind == "camera":
        return {"rel": 7e-3}
    return {"rel": 5e-3} if case["quant"] == "w4" else {"rel": 3.5e-2}


# ------------------------------------------------------ the same in 64 bits
def _ln64(x, p, eps):
    return torch.nn.functional.layer_norm(x, (x.shape[-1],), p[0].double(), p[1].double(), eps)


def _gelu64(x):
    return 0.5 * x * (1.0 + torch.erf(x * math.sqrt(0.5)))


def _gelu_tanh64(x):
    return 0.5 * x * (1.0 + torch.tanh(0.7978845608028654 * (x + 0.044715 * x ** 3)))


def _quant64(y):
    """Per-token int8 codes (as 64-bit values) and fp16 scales."""
    amax = y.abs().amax(-1, keepdim=True)
    return torch.round(y * (127.0 / amax)).clamp(-128, 127), (amax / 127.0).half().double()


def _linear64(x, p, quant):
    if quant == "w8":
        q, s = _quant64(x)
        return (q @ p["w"].double().t()) * p["ws"].double() * s + p["b"].double()
    w = _w4_weight(p) if quant == "w4" else p["w"].double()
    return x @ w.t() + p["b"].double()


def _attend64(q, k, v, seq, scale):
    """(T, H, d) each; sequences of ``seq`` tokens; one head and up to 4096 queries at a time."""
    out = torch.empty_like(q)
    for t0 in range(0, q.shape[0], seq):
        for h in range(q.shape[1]):
            kt, vh = k[t0:t0 + seq, h].t().contiguous(), v[t0:t0 + seq, h].contiguous()
            for r in range(t0, t0 + seq, 4096):
                e = min(r + 4096, t0 + seq)
                out[r:e, h] = torch.softmax((q[r:e, h] @ kt) * scale, -1) @ vh
    return out


def _rope64(x, pos, heads):
    """2-D RoPE (base 100) of x (T, heads, 64): columns [0, 32) by y, [32, 64) by x."""
    inv = 100.0 ** (-torch.arange(16, dtype=torch.float64, device=x.device) / 16.0)
    out = torch.empty_like(x)
    for half in range(2):
        ang = pos[:, half].double()[:, None] * inv
        c, s = ang.cos()[:, None], ang.sin()[:, None]
        a, b = x[..., 32 * half:32 * half + 16], x[..., 32 * half + 16:32 * half + 32]
        out[..., 32 * half:32 * half + 16] = a * c - b * s
        out[..., 32 * half + 16:32 * half + 32] = b * c + a * s
    return out


def _block64(x, p, quant, seq, pos, eps=BLOCK_EPS):
    m = x.shape[0]
    qkv = _linear64(_ln64(x, p["norm1"], eps), p["qkv"], quant).view(m, 3, HEADS, HD)
    q, k, v = qkv[:, 0], qkv[:, 1], qkv[:, 2]
    if quant != "fp16":
        q = _rope64(_ln64(q, p["q_norm"], eps), pos, HEADS)
        k = _rope64(_ln64(k, p["k_norm"], eps), pos, HEADS)
    att = _attend64(q.contiguous(), k.contiguous(), v.contiguous(), seq, 0.125).view(m, DIM)
    x = x + p["ls1"].double() * _linear64(att, p["proj"], quant)
    f = _linear64(_ln64(x, p["norm2"], eps), p["fc1"], quant)
    f = _gelu_tanh64(f) if quant == "w8" else _gelu64(f)
    return x + p["ls2"].double() * _linear64(f, p["fc2"], quant)


def _camera64(case, seed):
    p, s = _camera_params(seed), case["frames"]
    d, heads = ch.DIM, ch.HEADS
    ones, zeros = torch.ones(d, device=_dev()), torch.zeros(d, device=_dev())
    weights = [{n: _w4_weight(t[n]) for n in ("qkv", "proj", "fc1", "fc2")} for t in p["trunk"]]
    pose = _ln64(_randn(_gen(seed, 2), s, d).double(), p["token_norm"], 1e-5)
    adaln = _ln64(pose, (ones, zeros), 1e-6)
    pred, outs = None, []
    for _ in range(4):
        src = p["empty"].double().view(1, -1).expand(s, -1) if pred is None else pred
        e = _linear64(src, p["embed"], "fp16")
        shift, scale, gate = _linear64(e * torch.sigmoid(e), p["mod"], "fp16").chunk(3, -1)
        x = gate * (adaln * (1.0 + scale) + shift) + pose
        for t, w in zip(p["trunk"], weights):
            qkv = (_ln64(x, t["norm1"], 1e-5) @ w["qkv"].t() + t["qkv"]["b"].double()).view(s, 3, heads, d // heads)
            att = _attend64(*(qkv[:, i].contiguous() for i in range(3)), s, (d // heads) ** -0.5).reshape(s, d)
            x = x + t["ls1"].double() * (att @ w["proj"].t() + t["proj"]["b"].double())
            f = _gelu64(_ln64(x, t["norm2"], 1e-5) @ w["fc1"].t() + t["fc1"]["b"].double())
            x = x + t["ls2"].double() * (f @ w["fc2"].t() + t["fc2"]["b"].double())
        h = _gelu64(_linear64(_ln64(x, p["trunk_norm"], 1e-5), p["fc1"], "fp16"))
        delta = _linear64(h, p["fc2"], "fp16")
        pred = delta if pred is None else pred + delta
        outs.append(torch.cat([pred[:, :7], pred[:, 7:].clamp(min=0)], -1))
    return outs


def _aggregator64(case, seed):
    s, quant = case["frames"], case["quant"]
    m, e, pos = s * TOKENS, _embed_params(seed), _positions(case)
    mean = torch.tensor((0.485, 0.456, 0.406), device=_dev()).half().double().view(1, 3, 1, 1)
    std = torch.tensor((0.229, 0.224, 0.225), device=_dev()).half().double().view(1, 3, 1, 1)
    img = (_images(case, seed).double() - mean) / std
    patches = img.view(s, 3, 37, 14, 37, 14).permute(0, 2, 4, 1, 3, 5).reshape(s * 37 * 37, 3 * 14 * 14)
    pt = (patches @ e["proj_w"].double().view(DIM, -1).t() + e["proj_b"].double()).view(s, 37 * 37, DIM)
    x = torch.cat([(e["cls"].double() + e["pos"].double()[:, :1]).expand(s, 1, DIM), e["reg"].double().expand(s, 4, DIM),
                   pt + e["pos"].double()[:, 1:]], 1).reshape(m, DIM)
    for i in range(DEPTH):
        x = _block64(x, _block_params(_gen(seed, _DINO + i), "fp16"), "fp16", TOKENS, pos, 1e-6)
    x = _ln64(x, e["norm"], 1e-6).view(s, TOKENS, DIM)
    first = torch.arange(s, device=_dev()).clamp(max=1)      # token set 0 for the first frame, 1 for the others
    x[:, :1] = e["camera"].double()[0, first]
    x[:, 1:5] = e["register"].double()[0, first]
    x = x.reshape(m, DIM)
    outs = {}
    for i in range(DEPTH):
        x = _block64(x, _block_params(_gen(seed, _FRAME + i), quant), quant, TOKENS, pos)
        frame = x
        x = _block64(x, _block_params(_gen(seed, _GLOBAL + i), quant), quant, m, pos)
        if i in HEAD_LAYERS:
            outs[i] = torch.cat([frame, x], -1).view(s, TOKENS, 2 * DIM)
    return x, outs


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        dt = getattr(torch, case["dtype"])
        p = _w4_layer(_gen(seed, 1), case["k"], case["n"], dt)
        y = _randn(_gen(seed, 2), case["m"], case["k"], dtype=dt).double() @ _w4_weight(p).t()
        if case["epilogue"] == "none":
            return y
        y = y + p["b"].double()
        return _gelu64(y) if case["epilogue"] == "gelu" else y
    if kind == "w8a8_linear":
        p = _w8_layer(_gen(seed, 1), case["k"], case["n"])
        return None, None, _linear64(_randn(_gen(seed, 2), case["m"], case["k"]).double(), p, "w8")
    if kind == "attention":
        qkv = _randn(_gen(seed, 2), case["batch"] * case["seq"], 3, HEADS, HD).double()
        return _attend64(*(qkv[:, i].contiguous() for i in range(3)), case["seq"], 0.125)
    if kind in ("block", "dino"):
        quant = "fp16" if kind == "dino" else case["quant"]
        x = _tokens(case, seed).double()
        seq = x.shape[0] if case.get("attend") == "global" else _frame_tokens(case)
        return _block64(x, _block_params(_gen(seed, 1), quant), quant, seq, _positions(case))
    if kind == "camera":
        return _camera64(case, seed)
    return _aggregator64(case, seed)
