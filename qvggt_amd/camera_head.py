"""VGGT camera head with a W4A16 trunk: the small-M consumer of the GEMV path.

QVGGT quantises the camera head's trunk linears (``camera_head.trunk.*``,
loader.py:204-206, 338-344) and keeps the rest in floating point; the head
itself lives in the external vggt-hf, so this restates the public VGGT camera
head under the same module names:

* pose tokens = the camera token of every frame from the last aggregator
  output ([frame | global], 2048 wide), LayerNorm'd (``token_norm``);
* 4 refinement iterations: the current pose encoding (9 values: translation 3,
  quaternion 4, field of view 2; ``empty_pose_tokens`` on the first pass) is
  embedded (``embed_pose``), turned into adaLN shift / scale / gate
  (``poseLN_modulation`` = SiLU + Linear) that modulate the normalised pose
  tokens (``adaln_norm``, no affine), a residual is added, the 4-block trunk
  runs (dim 2048, 16 heads of 128, MLP 8192, LayerScale, no qk-norm / RoPE),
  then ``trunk_norm`` and ``pose_branch`` (2048 -> 1024 -> GELU -> 9) predict a
  delta that is accumulated; translation and quaternion are passed through,
  the field of view through ReLU.

LayerNorm eps: 1e-5 (torch's default) for ``token_norm``, ``trunk_norm`` and
the trunk blocks, 1e-6 for ``adaln_norm``.

Per frame there is one pose token, so the trunk linears run at M = S: every
S <= 64 runs on the skinny-M MFMA kernel (through the GEMV entry for
S <= 16 and the GEMM entry above).  Attention over the S tokens (head_dim
128, fp32; up to 256 frames) is one kernel; up to 64 frames the head's own fp16
linears run with what surrounds them (SiLU, the adaLN modulation, GELU, the
pose update) in four.
``GraphedCameraHead`` records the whole forward as one HIP graph.  The CICT token
QVGGT's loader can attach (loader.py:224-246) has no public definition and is
not modelled.
"""
from __future__ import annotations

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import awq_inference_engine as E
from ._lib import QV_EPI_BIAS, QV_EPI_BIAS_GELU
from .aggregator import LayerScale, Mlp, _affine, _aligned, _linear, _linear_residual, quantize_w4
from .awq.qmodule import WQLinear, w4_buffers

DIM = 2048
HEADS = 16
HEAD_DIM = DIM // HEADS      # 128
MLP_DIM = 4 * DIM
TRUNK_DEPTH = 4
POSE_DIM = 9                 # absT (3) + quaternion (4) + FoV (2)
POSE_LINEAR = 7              # leading columns without an activation (translation, quaternion)
LN_EPS = 1e-5               # token_norm, trunk_norm, trunk blocks (torch's default)
ADALN_EPS = 1e-6
# Frames up to which the pose attention runs in its one fp32 kernel; above, the
# fp32 batched products of torch are as fast or faster (256 frames: 24 us
# against 96; 512: 74 / 63; 1024: 262 / 150).
POSE_ATTENTION_MAX = 256


# Frames up to which the head's own fp16 linears run on the few-token kernels,
# which read the weights once per 16 tokens (beyond, the library's products).
POSE_LINEAR_MAX = 64


def _unhooked(*modules) -> bool:
    """Whether calling the modules does nothing but their own forward."""
    g = nn.modules.module
    if g._global_forward_hooks or g._global_forward_pre_hooks or g._global_backward_hooks or g._global_backward_pre_hooks:
        return False
    return not any(m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks
                   or "forward" in m.__dict__ for m in modules)


def _plain_linear(m, k: int, n: int | None = None) -> int:
    """The output channels of m if it is a plain fp16 linear from k (to n)
    channels with a bias and weights that 16-byte loads can read, else 0."""
    if type(m) is not nn.Linear:
        return 0
    w, b = m._parameters.get("weight"), m._parameters.get("bias")
    if type(w) is not nn.Parameter or type(b) is not nn.Parameter:
        return 0
    shape = w.shape
    ok = (w.dtype == b.dtype == torch.float16 and len(shape) == 2 and shape[1] == k and n in (None, shape[0])
          and b.shape == shape[:1] and w.data_ptr() % 16 == 0)
    return shape[0] if ok else 0


def _fusable(embed, modulation, fc1, fc2) -> bool:
    """Whether the head's own modules are what the few-token kernels compute:
    embed, (SiLU, linear), fc1 and fc2 as built here, or of other inner widths
    that the kernels' K steps of 32 divide."""
    if type(modulation) is not nn.Sequential or len(modulation) != 2:
        return False
    silu, lin = modulation
    e, m = _plain_linear(embed, POSE_DIM), _plain_linear(fc1, DIM)
    return (type(silu) is nn.SiLU and e > 0 and e % 32 == 0 and m > 0 and m % 32 == 0
            and _plain_linear(lin, e, 3 * DIM) > 0 and _plain_linear(fc2, m, POSE_DIM) > 0
            and _unhooked(embed, modulation, silu, lin, fc1, fc2))


def _modulate(mod: torch.Tensor, adaln: torch.Tensor, pose: torch.Tensor) -> torch.Tensor:
    """gate * (adaln * (1 + scale) + shift) + pose for mod = (shift | scale | gate):
    one kernel for the modulation that the head's own modules make, torch for
    what else a replaced one returns (another type, one row for all frames)."""
    S, D = pose.shape
    if mod.dtype == pose.dtype == torch.float16 and mod.shape == (S, 3 * D) and _aligned(mod):
        return E.adaln_modulate(mod, adaln, pose)
    shift, scale, gate = mod.chunk(3, dim=-1)
    return (gate * (adaln * (1 + scale) + shift) + pose).contiguous()


def _norm_linear(norm, layer, x: torch.Tensor, epilogue: int, n: int) -> torch.Tensor:
    """layer(norm(x)) with its bias (+ GELU): one kernel for a ``WQLinear`` on up
    to 16 tokens (one MFMA tile; 6.3-9.0 us against 7.5-9.5 for the two, and
    one call less), else the norm, then the linear."""
    if 0 < x.shape[0] <= 16 and isinstance(layer, WQLinear) and x.dtype == torch.float16:
        qweight, scales, scaled_zeros, bias = w4_buffers(layer)
        weight, shift = _affine(norm)
        if bias is not None and qweight.shape[0] * 4 == n and _aligned(x, weight, shift):
            return E.w4a16_ln_linear(x, weight, shift, LN_EPS, qweight, scales, scaled_zeros, bias, epilogue)
    h = E.layer_norm(x, *_affine(norm), LN_EPS)
    return _linear(layer, h, epilogue, x.new_empty((x.shape[0], n)))


def activate_pose(enc: torch.Tensor) -> torch.Tensor:
    """absT_quaR_FoV with linear translation / quaternion and ReLU field of view."""
    return torch.cat([enc[..., :POSE_LINEAR], F.relu(enc[..., POSE_LINEAR:])], dim=-1)


class TrunkBlock(nn.Module):
    """Camera-head trunk block: LN -> qkv -> attention over the frames -> proj ->
    LayerScale residual; LN -> fc1 -> GELU -> fc2 -> LayerScale residual."""

    def __init__(self, qkv, proj, fc1, fc2, dev=None):
        super().__init__()
        kw = dict(device=dev, dtype=torch.float16)
        self.norm1 = nn.LayerNorm(DIM, eps=LN_EPS, **kw)
        self.attn = nn.Module()
        self.attn.qkv, self.attn.proj = qkv, proj
        self.ls1 = LayerScale(DIM, 0.01, dev)
        self.norm2 = nn.LayerNorm(DIM, eps=LN_EPS, **kw)
        self.mlp = Mlp(fc1, fc2)
        self.ls2 = LayerScale(DIM, 0.01, dev)

    @torch.no_grad()
    def forward(self, x: torch.Tensor) -> torch.Tensor:
        S = x.shape[0]
        attn, mlp = self.attn, self.mlp
        qkv = _norm_linear(self.norm1, attn.qkv, x, QV_EPI_BIAS, 3 * DIM)
        if S <= POSE_ATTENTION_MAX:
            att = E.pose_attention(qkv, HEADS, HEAD_DIM ** -0.5)
        else:
            q, k, v = qkv.float().view(S, 3, HEADS, HEAD_DIM).permute(1, 2, 0, 3)   # (H, S, 128) each
            a = torch.softmax(torch.bmm(q, k.transpose(1, 2).contiguous()) * HEAD_DIM ** -0.5, dim=-1) @ v
            att = a.permute(1, 0, 2).reshape(S, DIM).half()
        o = x.new_empty((S, DIM))   # for a linear that is not fused with its residual update
        _linear_residual(attn.proj, att, self.ls1.gamma, x, o)
        f = _norm_linear(self.norm2, mlp.fc1, x, QV_EPI_BIAS_GELU, MLP_DIM)
        _linear_residual(mlp.fc2, f, self.ls2.gamma, x, o)
        return x


class CameraHead(nn.Module):
    """Iterative camera-pose head (module names as in the checkpoint, under
    ``camera_head.``).  ``forward(tokens)``: tokens (S, 2048) fp16 camera tokens;
    returns the activated pose encodings (S, 9) fp32 of every iteration."""

    def __init__(self, trunk_layers, dev=None):
        super().__init__()
        kw = dict(device=dev, dtype=torch.float16)
        self.trunk = nn.Sequential(*[TrunkBlock(*layers, dev=dev) for layers in trunk_layers])
        self.token_norm = nn.LayerNorm(DIM, eps=LN_EPS, **kw)
        self.trunk_norm = nn.LayerNorm(DIM, eps=LN_EPS, **kw)
        self.empty_pose_tokens = nn.Parameter(torch.zeros(1, 1, POSE_DIM, **kw), requires_grad=False)
        self.embed_pose = nn.Linear(POSE_DIM, DIM, **kw)
        self.poseLN_modulation = nn.Sequential(nn.SiLU(), nn.Linear(DIM, 3 * DIM, **kw))
        self.pose_branch = Mlp(nn.Linear(DIM, DIM // 2, **kw), nn.Linear(DIM // 2, POSE_DIM, **kw))
        self.register_buffer("_ones", torch.ones(DIM, **kw), persistent=False)
        self.register_buffer("_zeros", torch.zeros(DIM, **kw), persistent=False)

    @classmethod
    def empty(cls, device="cuda"):
        """fp16 ``nn.Linear`` trunk (the loader swaps the quantised ones)."""
        dev = torch.device(device)

        def lin(k, n):
            return nn.Linear(k, n, device=dev, dtype=torch.float16)

        return cls([(lin(DIM, 3 * DIM), lin(DIM, DIM), lin(DIM, MLP_DIM), lin(MLP_DIM, DIM))
                    for _ in range(TRUNK_DEPTH)], dev)

    @classmethod
    @torch.no_grad()
    def random(cls, seed: int = 0, device="cuda", w4: bool = True):
        """Seeded random weights (N(0, 0.02) linears); trunk linears W4 g128."""
        dev = torch.device(device)
        g = torch.Generator(device=dev).manual_seed(seed)

        def lin(k, n):
            l = nn.Linear(k, n, device=dev, dtype=torch.float16)
            l.weight.copy_((torch.randn(n, k, generator=g, device=dev) * 0.02).half())
            l.bias.copy_((torch.randn(n, generator=g, device=dev) * 0.02).half())
            return quantize_w4(l) if w4 else l

        layers = [(lin(DIM, 3 * DIM), lin(DIM, DIM), lin(DIM, MLP_DIM), lin(MLP_DIM, DIM)) for _ in range(TRUNK_DEPTH)]
        head = cls(layers, dev)
        for blk in head.trunk:
            for ln in (blk.norm1, blk.norm2):
                ln.weight.copy_((1 + 0.1 * torch.randn(DIM, generator=g, device=dev)).half())
                ln.bias.copy_((0.1 * torch.randn(DIM, generator=g, device=dev)).half())
            blk.ls1.gamma.copy_((0.5 + torch.rand(DIM, generator=g, device=dev)).half())
            blk.ls2.gamma.copy_((0.5 + torch.rand(DIM, generator=g, device=dev)).half())
        for ln in (head.token_norm, head.trunk_norm):
            ln.weight.copy_((1 + 0.1 * torch.randn(DIM, generator=g, device=dev)).half())
            ln.bias.copy_((0.1 * torch.randn(DIM, generator=g, device=dev)).half())
        for l in (head.embed_pose, head.poseLN_modulation[1], head.pose_branch.fc1, head.pose_branch.fc2):
            l.weight.copy_((torch.randn(l.weight.shape, generator=g, device=dev) * 0.02).half())
            l.bias.copy_((torch.randn(l.bias.shape, generator=g, device=dev) * 0.02).half())
        head.empty_pose_tokens.copy_((torch.randn(1, 1, POSE_DIM, generator=g, device=dev) * 0.02).half())
        return head

    @staticmethod
    def pose_tokens(layer_out: torch.Tensor) -> torch.Tensor:
        """Camera token (token 0) of every frame of a (S, tokens, 2048)
        [frame | global] aggregator output: the head's input."""
        return layer_out[:, 0].contiguous()

    # the pose update's kernels hold this one; another (a subclass's, an
    # instance's) is called on the prediction
    activate = staticmethod(activate_pose)

    @torch.no_grad()
    def forward(self, tokens: torch.Tensor, num_iterations: int = 4):
        S = tokens.shape[0]
        pose = E.layer_norm(tokens.contiguous(), self.token_norm.weight, self.token_norm.bias, LN_EPS)
        adaln = E.layer_norm(pose, self._ones, self._zeros, ADALN_EPS)
        # the first iteration embeds empty_pose_tokens, the later ones the prediction
        src = self.empty_pose_tokens.view(1, POSE_DIM).expand(S, POSE_DIM)
        pred = torch.empty(S, POSE_DIM, dtype=torch.float32, device=tokens.device)
        outs = []
        embed, modulation, fc1, fc2 = self.embed_pose, self.poseLN_modulation, self.pose_branch.fc1, self.pose_branch.fc2
        kernel_act = self.activate is activate_pose
        fused = (kernel_act and S <= POSE_LINEAR_MAX and _fusable(embed, modulation, fc1, fc2)
                 and not torch.is_autocast_enabled())
        for i in range(num_iterations):
            if fused:
                x = E.pose_modulate(E.pose_embed(src, *_affine(embed)), *_affine(modulation[1]), adaln, pose)
            else:
                x = _modulate(modulation(embed(src)), adaln, pose)
            for blk in self.trunk:
                blk(x)
            h = E.layer_norm(x, *_affine(self.trunk_norm), LN_EPS)
            if fused:
                act, src = E.pose_delta(E.pose_linear_gelu(h, *_affine(fc1)), *_affine(fc2), pred, i == 0, POSE_LINEAR)
            else:
                delta = fc2(F.gelu(fc1(h)))
                if kernel_act and delta.dtype == torch.float16 and delta.shape == pred.shape:
                    act, src = E.pose_update(delta, pred, i == 0, POSE_LINEAR)
                else:
                    pred = delta.float() if i == 0 else pred + delta.float()
                    act, src = self.activate(pred), pred.half()
            outs.append(act)
        return outs


class GraphedCameraHead:
    """``CameraHead.forward`` for a fixed frame count S, recorded once as a HIP
    graph and replayed: the head is 102 small launches per call up to 16
    frames (4 iterations x 4 trunk blocks of two norm + linear, attention and
    two linear + residual launches, and what surrounds the trunk), 134 with the
    norms apart, so replay removes the host launch cost that otherwise dominates
    at small S (8 frames 1.13 -> 0.60 ms, 32 frames 1.37 -> 0.85).
    ``__call__(tokens)`` copies ``tokens`` (S, 2048) into the graph's input
    buffer, replays, and returns the graph's output tensors (overwritten by the
    next call; clone to keep them)."""

    def __init__(self, head: CameraHead, S: int, num_iterations: int = 4):
        dev = head.token_norm.weight.device
        self.head, self.S = head, S
        self.tokens = torch.zeros(S, DIM, dtype=torch.float16, device=dev)
        side = torch.cuda.Stream(device=dev)
        side.wait_stream(torch.cuda.current_stream(dev))
        with torch.cuda.stream(side):
            for _ in range(2):
                head(self.tokens, num_iterations)
        torch.cuda.current_stream(dev).wait_stream(side)
        self.graph = torch.cuda.CUDAGraph()
        # The eager calls above made every shape's tile plan; the W4 ops'
        # split-K launches in the graph use the device's scratch array (never
        # an eager stream's workspace), so replays may run on any stream, but
        # two graphs with split launches must not replay concurrently.
        with torch.cuda.graph(self.graph, stream=side):
            self.outs = head(self.tokens, num_iterations)

    @torch.no_grad()
    def __call__(self, tokens: torch.Tensor):
        if tokens.shape != self.tokens.shape:
            raise ValueError(f"GraphedCameraHead: recorded for {tuple(self.tokens.shape)} tokens, got {tuple(tokens.shape)}")
        self.tokens.copy_(tokens)
        self.graph.replay()
        return self.outs
