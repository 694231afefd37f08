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


# One or two waves per row group: S on both sides of three chunks (96), grids of 256, 384 and 512
# 128-row workgroups (the forward's lines on 256 CUs by length), 256 (the backward's) and 64 (its
# line for short sequences), and delta held for up to 512 rows or in its own pass.
F32_SHAPES = [(3, 96, 64), (3, 97, 64), (2, 129, 64), (5, 160, 32), (1, 500, 64), (64, 1000, 64),
              (65, 1000, 64), (128, 385, 32), (129, 390, 32), (512, 100, 64), (513, 100, 32),
              (64, 40, 64), (65, 33, 64), (32, 1000, 64), (33, 1000, 32), (3, 512, 64),
              (3, 513, 64), (86, 300, 64), (85, 300, 64), (76, 600, 32), (77, 600, 64),
              (24, 600, 32), (160, 1000, 64)]


@pytest.mark.parametrize("BH,S,D", F32_SHAPES)
def test_f32_shapes(gpu, BH, S, D):
    """The fp32 kernels' bounds (1e-5) hold against float64 whatever the split."""
    _check(BH, S, D, torch.float32, (1e-5,) * 5)


# One or two waves per row group in the bf16 kernels: one tile and two (S 64, 65), the short rule
# (S 128, 256) and the long one (S 257, 800, 1000) on both sides of their lines at 256 CUs, tiles
# that end inside a chunk, and more heads than a round of workgroups.
BF16_SHAPES = [(1, 64, 64), (1, 65, 64), (3, 95, 64), (2, 97, 32), (128, 128, 64), (129, 128, 64),
               (64, 256, 64), (65, 250, 64), (128, 257, 64), (129, 330, 64), (64, 800, 64),
               (74, 790, 64), (24, 2047, 64), (384, 100, 32), (385, 70, 32), (96, 800, 32),
               (110, 800, 32),
               # the backward in one launch or two: delta held for up to 1,024 rows, its own pass
               # past them, the lines in heads x length (one and two row blocks, longer rows, rows
               # with the pass), a full round of heads, and the line for two waves
               (3, 1024, 64), (3, 1025, 64), (2, 1030, 32), (128, 1000, 64), (129, 1000, 64),
               (192, 500, 64), (300, 270, 64), (48, 511, 64), (49, 511, 64), (600, 200, 32),
               (3328, 40, 64), (3329, 40, 64), (640, 140, 64), (641, 140, 64), (1024, 140, 32),
               (1025, 140, 32), (115, 1100, 64), (116, 1100, 64), (223, 300, 64), (224, 300, 64)]
BF16_TOLS = (2e-2, 1e-3, 5e-2, 5e-2, 5e-2)


@pytest.mark.parametrize("BH,S,D", BF16_SHAPES)
def test_bf16_shapes(gpu, BH, S, D):
    """The bf16 kernels' bounds against float64 (of the same bf16 inputs) whatever the split."""
    _check(BH, S, D, torch.bfloat16, BF16_TOLS)


@pytest.mark.parametrize("BH,S,D", [(2, 70, 64), (5, 300, 64), (99, 520, 64), (150, 520, 64),
                                    (3, 1030, 64), (30, 600, 64), (100, 257, 64), (60, 700, 64),
                                    (60, 1100, 64), (60, 1100, 32), (3, 1030, 32), (300, 150, 32),
                                    (200, 600, 32)])
def test_bf16_strided_shapes(gpu, BH, S, D):
    """The strided instantiations give the contiguous ones' bits on both sides of the lines, and a
    dropout rate of zero, which runs the plain kernels, too."""
    print(f"[case] strided BH={BH} S={S} D={D}", flush=True)
    q, k, v, dout = _inputs(BH, S, D, torch.bfloat16, S)
    scale = A.default_scale(D)
    out, lse = A.attention_forward(q, k, v, scale)
    want = (out, lse) + A.attention_backward(dout, out, lse, q, k, v, scale)[:3]
    o2, l2, delta = torch.empty_like(out), torch.empty_like(lse), torch.empty_like(lse)
    A.flash_attention_forward_bf16_dropout(o2, l2, q, k, v, BH, S, D, scale, 0.0, 5)
    grads = [torch.empty_like(q) for _ in range(3)]
    A.flash_attention_backward_bf16_dropout(*grads, delta, dout, o2, l2, q, k, v, BH, S, D, scale,
                                            0.0, 5)
    tokens = [x.view(1, BH, S, D).transpose(1, 2).contiguous().transpose(1, 2)
              for x in (q, k, v, dout)]
    o3 = torch.empty_like(tokens[0])
    l3 = torch.empty_like(lse)
    A.flash_attention_forward_bf16_strided(o3, l3, *tokens[:3], scale)
    g3 = [torch.empty_like(tokens[0]) for _ in range(3)]
    A.flash_attention_backward_bf16_strided(*g3, delta, tokens[3], o3, l3, *tokens[:3], scale)
    for got in ((o2, l2, *grads),
                (o3.reshape(BH, S, D), l3, *[x.reshape(BH, S, D) for x in g3])):
        for x, y in zip(got, want):
            assert torch.equal(x, y)


# (3 slices: two waves per group; 400 slices: one wave per group, at S = 160 in D = 64 and 32)
@pytest.mark.parametrize("BH,S,D", [(3, 160, 64), (3, 700, 64), (3, 160, 32), (400, 160, 64),
                                    (400, 160, 32)])
@pytest.mark.parametrize("first", [0, 32, 64])
def test_bf16_chunk_of_minus_infinity(gpu, BH, S, D, first):
    """Scores that overflow to -inf weigh nothing, in the bf16 forward, also where they fill a
    whole 32-key chunk: the first of the row, the first that a group's second wave sees, or a
    later one. Rows that see no other key (those up to first + 31, for the first chunk) are left
    out: they have no defined softmax."""
    print(f"[case] -inf scores of keys {first}..{first + 31} BH={BH} S={S} D={D}", flush=True)
    q, k, v, _ = _inputs(BH, S, D, torch.bfloat16, 3 * S + first)
    # one column decides: 2^60 x -2^90 is far below fp32's range, 2^60 x 0 adds nothing
    q[..., 0], k[..., 0] = 2.0 ** 60, 0.0
    k[:, first:first + 32, 0] = -(2.0 ** 90)
    scale = A.default_scale(D)
    runs = [A.attention_forward(q, k, v, scale)]
    out, lse = torch.empty_like(q), torch.empty((BH, S), device="cuda")
    A.flash_attention_forward_bf16_dropout(out, lse, q, k, v, BH, S, D, scale, 0.1, 5)
    x = [t.view(1, BH, S, D).transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v)]
    o3, l3 = torch.empty_like(x[0]), torch.empty_like(lse)
    A.flash_attention_forward_bf16_strided(o3, l3, *x, scale)
    runs.append((o3.reshape(BH, S, D), l3))
    rows = slice(first + 32 if first == 0 else 0, S)
    hidden = torch.ones((S, S), dtype=torch.bool, device="cuda").triu(1)
    hidden[:, first:first + 32] = True
    heads = [0, BH // 2, BH - 1]
    q6, k6, v6 = (t[heads].double() for t in (q, k, v))
    s = torch.bmm(q6, k6.transpose(1, 2).contiguous()) * scale
    s = s.masked_fill(hidden, float("-inf"))[:, rows]
    want_lse, want = torch.logsumexp(s, -1), torch.bmm(torch.softmax(s, -1), v6)
    for o, l in runs:
        assert torch.isfinite(o[:, rows]).all().item() and torch.isfinite(l[:, rows]).all().item()
        assert (o[heads][:, rows].double() - want).abs().max().item() <= BF16_TOLS[0]
        assert (l[heads][:, rows].double() - want_lse).abs().max().item() <= BF16_TOLS[1]
    assert torch.isfinite(out[:, rows]).all().item()
    assert (lse[heads][:, rows].double() - want_lse).abs().max().item() <= BF16_TOLS[1]


@pytest.mark.parametrize("BH,S,D", [(4, 70, 64), (24, 300, 32), (24, 1024, 64), (3, 1030, 64),
                                    (160, 520, 64)])
def test_bf16_backward_in_place(gpu, BH, S, D):
    """Gradients that take the place of an input which only their own workgroup reads (dk = k,
    dv = v, dq = out, and dk or dv = out): dQ and dK/dV then run one after the other, as the phase
    calls do, bit for bit; contiguous and token-major."""
    print(f"[case] bf16 backward in place BH={BH} S={S} D={D}", flush=True)
    q, k, v, dout = _inputs(BH, S, D, torch.bfloat16, S)
    scale = A.default_scale(D)
    out, lse = A.attention_forward(q, k, v, scale)
    delta = torch.empty_like(lse)
    want = [torch.empty_like(q) for _ in range(3)]
    for phase in (1, 2):
        A.flash_attention_backward_bf16_phase(phase, *want, delta, dout, out, lse, q, k, v, BH, S,
                                              D, scale)
    for places in (("out", "k", "v"), ("q2", "out", "v"), ("q2", "k", "out"), ("q2", "k2", "v")):
        t = {"q": q.clone(), "k": k.clone(), "v": v.clone(), "out": out.clone(),
             "q2": torch.empty_like(q), "k2": torch.empty_like(q)}
        A.flash_attention_backward_bf16(t[places[0]], t[places[1]], t[places[2]], delta, dout,
                                        t["out"], lse, t["q"], t["k"], t["v"], BH, S, D, scale)
        for x, y in zip(places, want):
            assert torch.equal(t[x], y), places
    tok = {n: x.view(1, BH, S, D).transpose(1, 2).contiguous().transpose(1, 2)
           for n, x in (("q", q), ("k", k), ("v", v), ("out", out), ("dout", dout))}
    A.flash_attention_backward_bf16_strided(tok["out"], tok["k"], tok["v"], delta, tok["dout"],
                                            tok["out"], lse, tok["q"], tok["k"], tok["v"], scale)
    for x, y in zip(("out", "k", "v"), want):
        assert torch.equal(tok[x].reshape(BH, S, D), y), x
    # with dropout (p = 0.1) against the call with buffers of its own, to the rounding of another
    # summation order: 2^-8 of values below 8
    shape = (BH, S, D, scale, 0.1, 5)
    A.flash_attention_forward_bf16_dropout(out, lse, q, k, v, *shape)
    A.flash_attention_backward_bf16_dropout(*want, delta, dout, out, lse, q, k, v, *shape)
    A.flash_attention_backward_bf16_dropout(out, k, v, delta, dout, out, lse, q, k, v, *shape)
    for x, y in zip((out, k, v), want):
        assert (x.float() - y.float()).abs().max().item() <= 8 * 2.0 ** -8


@pytest.mark.parametrize("BH,S,D", [(4, 70, 64), (24, 300, 32), (24, 600, 64), (160, 300, 64)])
@pytest.mark.parametrize("p", [0.0, 0.2])
def test_f32_backward_in_place(gpu, BH, S, D, p):
    """As above in fp32, where the delta pass, dK/dV and dQ run in this order: dq = q, dq = dout,
    and any gradient = out. Up to 512 rows delta is otherwise summed in another order, so the
    gradients agree to the fp32 bound."""
    print(f"[case] fp32 backward in place BH={BH} S={S} D={D} p={p}", flush=True)
    q, k, v, dout = _inputs(BH, S, D, torch.float32, S)
    shape = (BH, S, D, A.default_scale(D)) + ((p, 11) if p else ())
    out, lse = torch.empty_like(q), torch.empty((BH, S), device="cuda")
    forward, backward = ((A.flash_attention_forward_dropout, A.flash_attention_backward_dropout)
                         if p else (A.flash_attention_forward, A.flash_attention_backward))
    forward(out, lse, q, k, v, *shape)
    delta = torch.empty_like(lse)
    want = [torch.empty_like(q) for _ in range(3)]
    backward(*want, delta, dout, out, lse, q, k, v, *shape)
    for places in (("q", "out", "v2"), ("dout", "k2", "out"), ("out", "k2", "v2")):
        t = {"q": q.clone(), "dout": dout.clone(), "out": out.clone(),
             "k2": torch.empty_like(q), "v2": torch.empty_like(q)}
        backward(t[places[0]], t[places[1]], t[places[2]], delta, t["dout"], t["out"], lse, t["q"],
                 k, v, *shape)
        for x, y in zip(places, want):
            assert (t[x] - y).abs().max().item() <= 1e-5, places
