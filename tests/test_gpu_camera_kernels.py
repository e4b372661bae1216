"""The camera head's small kernels against torch in float64.

Bounds: the kernels compute in fp32 and round once to fp16, so an output is
within half an fp16 step (2^-11 relative, 2^-25 absolute below the normal
range) of the exact value plus the fp32 error of the sums, which 1e-5 of the
largest term covers (under 300 terms at 6e-8 each).
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _close(got, ref, scale):
    got, ref = got.double(), ref.double()
    assert torch.isfinite(got).all()
    assert ((got - ref).abs() <= ref.abs() * 2.0 ** -11 + 2.0 ** -25 + 1e-5 * scale).all()


@pytest.mark.parametrize("S", [1, 3, 4, 5, 16, 17, 63, 64, 65, 127, 129, 200])
@pytest.mark.parametrize("H,sigma", [(16, 1.0), (3, 6.0)])
def test_pose_attention(gpu, S, H, sigma):
    """Around the query blocks (4), the 64-key tiles and their
    remainders; sigma = 6 spreads the scores over hundreds, so the running
    maximum moves between tiles."""
    from qvggt_amd import awq_inference_engine as E
    g = torch.Generator(device=gpu).manual_seed(S)
    qkv = (torch.randn(S, 3, H, 128, generator=g, device=gpu) * sigma).half()
    out = E.pose_attention(qkv.view(S, -1), H, 128 ** -0.5)
    q, k, v = (qkv[:, i].double().transpose(0, 1).contiguous() for i in range(3))
    s = q @ k.transpose(1, 2).contiguous() * 128 ** -0.5
    ref = (torch.softmax(s, -1) @ v).transpose(0, 1).reshape(S, H * 128)
    # an fp32 score is off by up to ~1e-6 of the largest, and p by that factor
    _close(out, ref, v.abs().max().item() * max(1.0, s.abs().max().item() / 5))


@pytest.mark.parametrize("S,D", [(1, 8), (3, 2048), (80, 2048), (5, 264)])
def test_adaln_modulate(gpu, S, D):
    from qvggt_amd import awq_inference_engine as E
    g = torch.Generator(device=gpu).manual_seed(S + D)
    mod, a, p = (torch.randn(S, n, generator=g, device=gpu).half() for n in (3 * D, D, D))
    x = E.adaln_modulate(mod, a, p)
    sh, sc, ga = mod.double().chunk(3, -1)
    _close(x, ga * (a.double() * (1 + sc) + sh) + p.double(), 1.0)
    wide = torch.randn(S, 3 * D + 8, generator=g, device=gpu).half()
    wide[:, :3 * D] = mod
    assert torch.equal(E.adaln_modulate(wide[:, :3 * D], a, p), x)      # a strided input


@pytest.mark.parametrize("S", [1, 28, 29, 300])
def test_pose_update(gpu, S):
    """Exact: the fp32 add, ReLU (NaN stays) and the rounding to fp16."""
    from qvggt_amd import awq_inference_engine as E
    g = torch.Generator(device=gpu).manual_seed(S)
    pred = torch.full((S, 9), float("nan"), device=gpu)
    want = None
    for i in range(3):
        d = torch.randn(S, 9, generator=g, device=gpu).half()
        if i == 2:
            d[0, 8], d[0, 0] = float("nan"), float("inf")
        want = d.float() if want is None else want + d.float()
        act, half = E.pose_update(d, pred, i == 0, 7)
        ref = torch.cat([want[:, :7], torch.relu(want[:, 7:])], -1)
        assert torch.equal(act.nan_to_num(123.0), ref.nan_to_num(123.0))
        assert torch.equal(half.nan_to_num(123.0), want.half().nan_to_num(123.0))
        assert torch.equal(pred.nan_to_num(123.0), want.nan_to_num(123.0))


def test_empty(gpu):
    from qvggt_amd import awq_inference_engine as E
    assert E.pose_attention(torch.empty(0, 6144, device=gpu, dtype=torch.float16), 16, 0.1).shape == (0, 2048)


@pytest.mark.parametrize("S,N,K", [(1, 1024, 2048), (8, 40, 32), (16, 1024, 2048), (17, 33, 96), (64, 1024, 288)])
def test_pose_linears(gpu, S, N, K):
    """The few-token fp16 linears with their tails, at token and channel
    remainders and K below, at and above one pass of the eight waves."""
    from qvggt_amd import awq_inference_engine as E
    g = torch.Generator(device=gpu).manual_seed(S + N + K)
    x = torch.randn(S, K, generator=g, device=gpu).half()
    w = (torch.randn(3 * N, K, generator=g, device=gpu) * K ** -0.5).half()
    b, (a, p) = torch.randn(3 * N, generator=g, device=gpu).half(), torch.randn(2, S, N, generator=g, device=gpu).half()
    lin = x.double() @ w.double().t().contiguous() + b.double()
    _close(E.pose_modulate(x, w, b, a, p), lin[:, 2 * N:] * (a.double() * (1 + lin[:, N:2 * N]) + lin[:, :N]) + p.double(), 20.0)
    # gelu: its fitted tail adds 3e-6 of the result
    got, ref = E.pose_linear_gelu(x, w[:N], b[:N]).double(), torch.nn.functional.gelu(lin[:, :N])
    assert ((got - ref).abs() <= ref.abs() * (2.0 ** -11 + 4e-6) + 1e-4).all()
    pred = torch.randn(S, 9, generator=g, device=gpu)
    want = pred.double() + lin[:, :9]
    act, half = E.pose_delta(x, w[:9], b[:9], pred, False, 7)
    assert ((pred.double() - want).abs() <= 1e-5 * 20).all()
    assert torch.equal(act, torch.cat([pred[:, :7], torch.relu(pred[:, 7:])], -1)) and torch.equal(half, pred.half())
    E.pose_delta(x, w[:9], b[:9], pred, True, 7)
    assert ((pred.double() - lin[:, :9]).abs() <= 1e-5 * 20).all()


def test_pose_embed(gpu):
    from qvggt_amd import awq_inference_engine as E
    g = torch.Generator(device=gpu).manual_seed(3)
    w, b = torch.randn(2048, 9, generator=g, device=gpu).half(), torch.randn(2048, generator=g, device=gpu).half()
    for src in (torch.randn(5, 9, generator=g, device=gpu).half(), torch.randn(1, 9, generator=g, device=gpu).half().expand(3, 9)):
        e = src.double() @ w.double().t().contiguous() + b.double()
        _close(E.pose_embed(src, w, b), torch.nn.functional.silu(e), 10.0)


def test_camera_head_hooks_still_run(gpu):
    """A hook on one of the head's own linears sends the forward through the
    module calls (so the hook sees its output), with the fused path's result."""
    from qvggt_amd.camera_head import CameraHead
    head = CameraHead.random(seed=2, device=gpu)
    t = torch.randn(3, 2048, generator=torch.Generator(device=gpu).manual_seed(1), device=gpu).half()
    plain, seen = head(t), []
    handle = head.pose_branch.fc1.register_forward_hook(lambda m, i, o: seen.append(o.shape))
    hooked = head(t)
    handle.remove()
    assert seen == [(3, 1024)] * 4
    for a, b in zip(plain, hooked):
        assert (a - b).abs().max().item() <= 1e-2 * b.abs().max().item()


@pytest.mark.parametrize("M,N,K", [(1, 32, 128), (5, 6144, 2048), (8, 8192, 2048), (16, 64, 1920), (13, 4096, 640), (7, 96, 384)])
@pytest.mark.parametrize("gelu", [False, True])
def test_w4a16_ln_linear(gpu, M, N, K, gelu):
    """LayerNorm + W4A16 linear in one kernel against the two ops: the norm's
    fp16 output differs by at most one step in a few places (its fp32 sums run
    in another order, moving a value by 1e-6 of its size), so the sums differ by
    that share of a step, 2^-11 * sqrt(K) of the typical term, and the output by
    one more rounding."""
    from qvggt_amd import awq_inference_engine as E
    g = torch.Generator(device=gpu).manual_seed(M + N + K)
    x = (torch.randn(M, K, generator=g, device=gpu) * 3 + 1).half()
    w, b = (1 + 0.1 * torch.randn(K, generator=g, device=gpu)).half(), (0.1 * torch.randn(K, generator=g, device=gpu)).half()
    qw = torch.randint(-32768, 32768, (N // 4, K), generator=g, device=gpu, dtype=torch.int32).to(torch.int16)
    rows = (K // 128 + 7) // 8 * 8
    s = (torch.rand(rows, N, generator=g, device=gpu) * 0.01 + 0.005).half()
    z = -(s.float() * 7).half()
    bias = torch.randn(N, generator=g, device=gpu).half()
    got = E.w4a16_ln_linear(x, w, b, 1e-5, qw, s, z, bias, 2 if gelu else 1).double()
    h = E.layer_norm(x, w, b, 1e-5)
    lin = h.double() @ E.w4a16_dequantize(qw, s, z, K).double().t().contiguous() + bias.double()
    ref = torch.nn.functional.gelu(lin) if gelu else lin
    term = (h.double().abs().mean() * 0.05)
    assert ((got - ref).abs() <= ref.abs() * 2.0 ** -10 + term * 2.0 ** -11 * K ** 0.5 + 1e-4).all()


class _Call(torch.nn.Module):
    """A module that calls another: no longer one that the head can look into."""

    def __init__(self, inner, post=lambda y: y):
        super().__init__()
        self.inner, self.post = inner, post

    def forward(self, x):
        return self.post(self.inner(x))


def _head_and_tokens(gpu, S=3):
    from qvggt_amd.camera_head import CameraHead
    return CameraHead.random(seed=2, device=gpu), torch.randn(
        S, 2048, generator=torch.Generator(device=gpu).manual_seed(1), device=gpu).half()


def _linear(gpu, k, n, seed):
    l = torch.nn.Linear(k, n, device=gpu, dtype=torch.float16)
    g = torch.Generator(device=gpu).manual_seed(seed)
    l.weight.data.copy_(torch.randn(n, k, generator=g, device=gpu) * 0.02)
    l.bias.data.copy_(torch.randn(n, generator=g, device=gpu) * 0.02)
    return l


def _rel(a, b):
    return max(((x - y).abs().max() / y.abs().max()).item() for x, y in zip(a, b))


def test_camera_head_activation_can_be_replaced(gpu):
    """``activate`` of a subclass or of an instance makes the outputs, and one
    that returns its argument is not overwritten by the next iteration."""
    from qvggt_amd.camera_head import CameraHead

    class Plain(CameraHead):
        @staticmethod
        def activate(enc):
            return enc

    head, t = _head_and_tokens(gpu)
    want = head(t)
    head.__class__ = Plain
    got = head(t)
    assert any((o[:, 7:] < 0).any() for o in got) and _rel([CameraHead.activate(o) for o in got], want) <= 1e-2
    head.__class__ = CameraHead
    head.activate = lambda enc: 2 * CameraHead.activate(enc)
    assert _rel([o / 2 for o in head(t)], want) <= 1e-2
    del head.activate
    assert all(torch.equal(a, b) for a, b in zip(head(t), want))


@pytest.mark.parametrize("kind", ["low_rank", "appended", "order", "narrow", "call"])
def test_camera_head_modulation_can_be_replaced(gpu, kind):
    """A ``poseLN_modulation`` of another build runs as built: equal, bit for
    bit, to the same modules behind a module that the head cannot look into."""
    from qvggt_amd.camera_head import _fusable
    head, t = _head_and_tokens(gpu)
    assert _fusable(head.embed_pose, head.poseLN_modulation, head.pose_branch.fc1, head.pose_branch.fc2)
    silu, lin = head.poseLN_modulation
    seq = {"low_rank": lambda: torch.nn.Sequential(silu, _linear(gpu, 2048, 64, 5), _linear(gpu, 64, 6144, 6)),
           "appended": lambda: torch.nn.Sequential(silu, lin, torch.nn.SiLU()),
           "order": lambda: torch.nn.Sequential(lin, torch.nn.SiLU()),
           "narrow": lambda: torch.nn.Sequential(silu, _linear(gpu, 100, 6144, 7)),
           "call": lambda: _Call(head.poseLN_modulation)}[kind]()
    if kind == "narrow":
        head.embed_pose = _linear(gpu, 9, 100, 8)
    own = (head.embed_pose, head.pose_branch.fc1, head.pose_branch.fc2)
    assert _fusable(own[0], seq, *own[1:]) is False
    head.poseLN_modulation = seq
    got = head(t)
    head.poseLN_modulation = _Call(seq)
    assert all(torch.equal(a, b) for a, b in zip(got, head(t)))


def test_camera_head_pose_branch_can_be_replaced(gpu):
    """Pose branches of other widths, and one that ends in fp32."""
    head, t = _head_and_tokens(gpu)
    want = head(t)
    fc1, fc2 = head.pose_branch.fc1, head.pose_branch.fc2
    head.pose_branch.fc2 = _Call(fc2, lambda y: y.float())
    assert _rel(head(t), want) <= 1e-2
    head.pose_branch.fc1, head.pose_branch.fc2 = _linear(gpu, 2048, 100, 3), _linear(gpu, 100, 9, 4)
    got = head(t)
    head.pose_branch.fc2 = _Call(head.pose_branch.fc2)
    assert _rel(got, head(t)) <= 1e-2


@pytest.mark.parametrize("post", ["one_row", "unaligned"])
def test_camera_head_takes_modulations_of_other_forms(gpu, post):
    """One modulation row for all frames, and one off 16-byte addresses."""
    head, t = _head_and_tokens(gpu)
    mod = head.poseLN_modulation

    def unaligned(y):
        return torch.empty(y.numel() + 1, device=gpu, dtype=y.dtype)[1:].view_as(y).copy_(y)

    head.poseLN_modulation = _Call(mod, (lambda y: y[:1]) if post == "one_row" else unaligned)
    got = head(t)
    head.poseLN_modulation = _Call(mod, (lambda y: y[:1].expand(3, -1)) if post == "one_row" else lambda y: y)
    assert _rel(got, head(t)) <= 1e-2
