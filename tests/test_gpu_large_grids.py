"""Edge values on grids that fill the GPU: the scales, NaN rows, later keys and strided views that
the small-batch tests check, at the batches where the kernels run with one wave per
row group and the bf16 backward in two launches. Sampled slices are compared with float64."""
import math

import pytest
import torch

from dadgpt_amd import attention as A

pytestmark = pytest.mark.gpu

# On 256 CUs: bf16 forward and backward with one wave per row group, dQ and dK/dV apart; the fp32
# kernels with one wave per row group, delta summed by the backward (300) or by its own pass (600).
BH = 200
F32_S = [300, 600]
BF16_S = 600


def _inputs(S, D, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn((BH, S, D), generator=g, device="cuda").to(dtype) for _ in range(4)]


def _reference(q, k, v, dout, scale, heads):
    """out, lse, dq, dk, dv of the given slices in float64."""
    q, k, v, dout = (x[heads].double() for x in (q, k, v, dout))
    S = q.shape[1]
    future = torch.ones((S, S), dtype=torch.bool, device="cuda").triu(1)
    s = torch.bmm(q, k.transpose(1, 2).contiguous()) * scale
    s.masked_fill_(future, float("-inf"))
    lse = torch.logsumexp(s, -1)
    P = torch.exp(s - lse.unsqueeze(-1))
    o = torch.bmm(P, v)
    dP = torch.bmm(dout, v.transpose(1, 2).contiguous())
    dS = P * (dP - (dout * o).sum(-1, keepdim=True)) * scale
    return (o, lse, torch.bmm(dS, k), torch.bmm(dS.transpose(1, 2).contiguous(), q),
            torch.bmm(P.transpose(1, 2).contiguous(), dout))


HEADS = [0, BH // 2, BH - 1]


@pytest.mark.parametrize("scale", [0.0, -0.125, 1.0])
@pytest.mark.parametrize("D", [64, 32])
def test_bf16_scales(gpu, scale, D):
    """Zero, negative and large scales at the bf16 bounds; the gradients' grows with the scale, as
    dQ and dK carry it and a large one sharpens P."""
    print(f"[case] bf16 scale={scale} BH={BH} S={BF16_S} D={D}", flush=True)
    q, k, v, dout = _inputs(BF16_S, D, torch.bfloat16, 17 + D)
    out, lse = A.attention_forward(q, k, v, scale)
    grads = A.attention_backward(dout, out, lse, q, k, v, scale)[:3]
    want = _reference(q, k, v, dout, scale, HEADS)
    grad = 5e-2 * max(1.0, abs(scale) * math.sqrt(D))
    for name, x, y, tol in zip(("out", "lse", "dq", "dk", "dv"), (out, lse, *grads), want,
                               (2e-2, 1e-3, grad, grad, grad)):
        assert torch.isfinite(x).all().item(), name
        assert (x[HEADS].double() - y).abs().max().item() <= tol, name


@pytest.mark.parametrize("scale", [0.0, -0.125, 1.0, 4.0])
@pytest.mark.parametrize("S", F32_S)
@pytest.mark.parametrize("D", [64, 32])
def test_f32_scales(gpu, scale, S, D):
    """The same in fp32: 1e-5 of the largest value, growing with the scale above the default one
    (a rounding of a score moves its weight that much more)."""
    print(f"[case] fp32 scale={scale} BH={BH} S={S} D={D}", flush=True)
    q, k, v, dout = _inputs(S, D, torch.float32, 27 + D)
    out, lse = A.attention_forward(q, k, v, scale)
    grads = A.attention_backward(dout, out, lse, q, k, v, scale)[:3]
    want = _reference(q, k, v, dout, scale, HEADS)
    tol = 1e-5 * max(1.0, abs(scale) * math.sqrt(D))
    for name, x, y in zip(("out", "lse", "dq", "dk", "dv"), (out, lse, *grads), want):
        assert torch.isfinite(x).all().item(), name
        bound = tol * max(1.0, y.abs().max().item())
        assert (x[HEADS].double() - y).abs().max().item() <= bound, name


@pytest.mark.parametrize("bad", [[599], [150], list(range(40, 50)), list(range(576, 600))])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_forward_rows_with_nan_rows_beside_them(gpu, bad, dtype):
    """NaN query rows leave every other row's output and logsumexp bit-identical."""
    S, D = 600, 64
    print(f"[case] NaN query rows {bad[0]}..{bad[-1]} {dtype}", flush=True)
    q, k, v, _ = _inputs(S, D, dtype, 37)
    o1, l1 = A.attention_forward(q, k, v, 0.125)
    q2 = q.clone()
    q2[BH // 2, bad] = float("nan")
    o2, l2 = A.attention_forward(q2, k, v, 0.125)
    same = torch.ones((BH, S), dtype=torch.bool, device="cuda")
    same[BH // 2, bad] = False
    assert torch.equal(o1[same], o2[same]) and torch.equal(l1[same], l2[same])
    assert torch.isnan(o2[BH // 2, bad]).all().item()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_later_keys(gpu, dtype):
    """K and V rows after a cut leave the earlier rows' outputs bit-identical."""
    S, D, cut = 600, 64, 150
    q, k, v, _ = _inputs(S, D, dtype, 47)
    k2, v2 = k.clone(), v.clone()
    k2[:, cut + 1:] = k[:, cut + 1:].flip(1) * 2
    v2[:, cut + 1:] = v[:, cut + 1:].flip(1) * 2
    o1, l1 = A.attention_forward(q, k, v, 0.125)
    o2, l2 = A.attention_forward(q, k2, v2, 0.125)
    assert torch.equal(o1[:, :cut + 1], o2[:, :cut + 1])
    assert torch.equal(l1[:, :cut + 1], l2[:, :cut + 1])
    assert not torch.equal(o1[:, cut + 1:], o2[:, cut + 1:])


@pytest.mark.parametrize("S,D", [(600, 64), (577, 32), (130, 64)])
def test_token_major_equals_contiguous(gpu, S, D):
    """The token-major calls (fused QKV, padded output rows) give the contiguous ones' bits; padding
    stays untouched."""
    B, H, pad = 20, 10, 8
    HD = H * D
    print(f"[case] token-major B={B} H={H} S={S} D={D}", flush=True)
    q, k, v, dout = _inputs(S, D, torch.bfloat16, 57 + S)
    scale = A.default_scale(D)
    out, lse = A.attention_forward(q, k, v, scale)
    want = (out, *A.attention_backward(dout, out, lse, q, k, v, scale)[:3])

    def tokens(x):
        return x.view(B, H, S, D).transpose(1, 2).reshape(B * S, HD)

    def heads(x):
        return x.reshape(B, S, H, D).transpose(1, 2).reshape(BH, S, D)

    qkv = torch.cat([tokens(x) for x in (q, k, v)], 1)
    o = torch.full((B * S, HD + pad), -77.0, dtype=torch.bfloat16, device="cuda")
    g = torch.zeros_like(o)
    g[:, :HD] = tokens(dout)
    dqkv = torch.empty_like(qkv)
    l2, delta = torch.empty_like(lse), torch.empty_like(lse)
    views = qkv, qkv[:, HD:], qkv[:, 2 * HD:]
    A.flash_attention_forward_bf16_tokens(o, HD + pad, l2, *views, 3 * HD, B, H, S, D, scale)
    A.flash_attention_backward_bf16_tokens(dqkv, dqkv[:, HD:], dqkv[:, 2 * HD:], 3 * HD, delta, g,
                                           o, HD + pad, l2, *views, 3 * HD, B, H, S, D, scale)
    assert torch.equal(o[:, HD:], torch.full_like(o[:, HD:], -77.0))
    got = [heads(o[:, :HD]), *(heads(dqkv[:, i * HD:(i + 1) * HD]) for i in range(3))]
    for name, x, y in zip(("out", "dq", "dk", "dv"), got, want):
        assert torch.equal(x, y), name
    assert torch.equal(l2, lse)
