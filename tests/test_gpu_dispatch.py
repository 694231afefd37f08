"""Attention at the sizes where the kernels' shape rules change course (waves per row group,
workgroups per grid, chunks per sequence), against float64 on the GPU."""
import pytest
import torch

from dadgpt_amd import attention as A

pytestmark = pytest.mark.gpu


def _inputs(BH, S, D, dtype, seed):
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


def _check(BH, S, D, dtype, tols):
    print(f"[case] BH={BH} S={S} D={D} {dtype}", flush=True)
    q, k, v, dout = _inputs(BH, S, D, dtype, 7 * S + BH)
    scale = A.default_scale(D)
    out, lse = A.attention_forward(q, k, v, scale)
    dq, dk, dv, _ = A.attention_backward(dout, out, lse, q, k, v, scale)
    heads = sorted({0, BH // 2, BH - 1})
    want = _reference(q, k, v, dout, scale, heads)
    for name, x, y, tol in zip(("out", "lse", "dq", "dk", "dv"), (out, lse, dq, dk, dv), want,
                               tols):
        err = (x[heads].double() - y).abs().max().item()
        assert err <= tol, (name, err, tol)
    # every other slice against the checked kind of result: finite, and repeatable bit for bit
    again, lse2 = A.attention_forward(q, k, v, scale)
    dq2, dk2, dv2, _ = A.attention_backward(dout, out, lse, q, k, v, scale)
    for x, y in ((out, again), (lse, lse2), (dq, dq2), (dk, dk2), (dv, dv2)):
        assert torch.isfinite(x).all().item() and torch.equal(x, y)


# One or two waves per row group: S on both sides of three chunks (96), and grids of 512 and
# more 128-row workgroups (two per CU of 256) around the line.
F32_SHAPES = [(3, 96, 64), (3, 97, 64), (2, 129, 64), (5, 160, 32), (1, 500, 64), (64, 1000, 64),
              (65, 1000, 64), (128, 385, 32), (129, 390, 32), (512, 100, 64), (513, 100, 32)]


@pytest.mark.parametrize("BH,S,D", F32_SHAPES)
def test_f32_shapes(gpu, BH, S, D):
    """The fp32 kernels' bounds (1e-5) hold against float64 whatever the split."""
    _check(BH, S, D, torch.float32, (1e-5,) * 5)
