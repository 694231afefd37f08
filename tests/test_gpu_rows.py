"""The row kernels of the materialized path at the edges of their shapes: rows of one column a lane
(up to 64) and of 16-byte pieces, rows that end inside a piece, one row and several per wave,
register rows (up to 1,024 columns) and looped ones, against float64."""
import numpy as np
import pytest
import torch

from dadgpt_amd import attention as A

pytestmark = pytest.mark.gpu

# (columns, rows): 16-byte remainders 0-3, both sides of 64, 256, 512 and 1,024 columns, and row
# counts that give one, two and four rows per wave with a last wave that is not full.
SHAPES = [(1, 5), (3, 4099), (4, 9), (5, 16387), (66, 8193), (255, 16389), (256, 16384),
          (257, 8195), (511, 8193), (512, 4097), (513, 33), (1021, 7), (1024, 5), (1025, 6),
          (2047, 3), (2048, 3), (2, 8193), (31, 4097), (63, 16387), (64, 33), (65, 16385),
          (100, 9), (100, 8193), (511, 33), (512, 8193)]


def _normal(shape, seed, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(shape, generator=g, device="cuda") * scale


@pytest.mark.parametrize("cols,rows", SHAPES)
def test_plain_rows(gpu, cols, rows):
    """softmax and the accumulating softmax_backward. A probability p = e^(x - max) / sum is off
    by at most p (|x - max| + 4) 2^-23 <= 6e-7, each product of the backward by 2^-23 of its
    terms (|g| < 6, and a row sum below 6 in magnitude): 2e-6."""
    print(f"[case] rows={rows} cols={cols}", flush=True)
    x, g, d = (_normal((rows, cols), 10 + i, s) for i, s in enumerate((3.0, 1.0, 1.0)))
    out = torch.full_like(x, float("nan"))
    A.softmax(out, x, rows, cols)
    same = x.clone()
    A.softmax(same, same, rows, cols)
    assert torch.equal(out, same)
    p = torch.softmax(x.double(), -1)
    assert (out.double() - p).abs().max().item() <= 1e-6
    din = d.clone()
    A.softmax_backward(din, g, out, rows, cols)
    o, g6 = out.double(), g.double()
    want = d.double() + o * (g6 - (g6 * o).sum(-1, keepdim=True))
    assert (din.double() - want).abs().max().item() <= 2e-6


@pytest.mark.parametrize("S,BH", [(1, 3), (3, 5), (4, 2), (63, 70), (64, 260), (130, 127),
                                  (256, 65), (257, 32), (509, 17), (512, 9), (515, 2), (1023, 1),
                                  (1030, 1), (31, 260), (65, 127), (1032, 1), (50, 170), (128, 70),
                                  (130, 20), (257, 10), (512, 17), (1024, 1)])
def test_causal_rows(gpu, S, BH):
    """attention_probs and attention_probs_backward, without and with dropout (p = 0, whose
    factors are exactly 1, must give the plain result's values). What lies past the diagonal of
    the scores does not matter; past that of the probabilities it counts in the row sum."""
    print(f"[case] BH={BH} S={S}", flush=True)
    scale = 0.25
    s, g = _normal((BH, S, S), 20, 6.0), _normal((BH, S, S), 21)
    upper = torch.ones((S, S), dtype=torch.bool, device="cuda").triu(1)
    probs = s.masked_fill(upper, float("nan"))
    A.attention_probs(probs, BH, S, scale)
    p = torch.softmax((s.double() * scale).masked_fill(upper, float("-inf")), -1)
    assert (probs.double() - p).abs().max().item() <= 1e-6
    assert torch.count_nonzero(probs[:, upper]).item() == 0
    full = probs + 0.01 * upper  # not a causal matrix
    for pr in (probs, full):
        ds = torch.full_like(g, float("nan"))
        A.attention_probs_backward(ds, g, pr, BH, S, scale)
        p6, g6 = pr.double(), g.double()
        want = p6 * (g6 - (g6 * p6).sum(-1, keepdim=True)) * scale
        want.masked_fill_(upper, 0.0)
        # products and the sum of up to S terms of at most 0.06 past the diagonal
        tol = 2e-6 * (1 if pr is probs else 1 + 0.06 * S ** 0.5)
        assert (ds.double() - want).abs().max().item() <= tol
        drop = torch.full_like(g, float("nan"))
        A.attention_probs_backward_dropout(drop, g, pr, BH, S, scale, 0.0, 9)
        assert (drop.double() - want).abs().max().item() <= tol
        inplace = g.clone()
        A.attention_probs_backward(inplace, inplace, pr, BH, S, scale)
        assert torch.equal(inplace, ds)
    dropped = torch.full_like(g, float("nan"))
    A.attention_dropout(dropped, probs, BH, S, 0.0, 9)
    assert torch.equal(dropped, probs)


@pytest.mark.parametrize("S", [50, 70, 72, 1100, 1101])
def test_rows_at_the_mask_value(gpu, S):
    """Visible scores at and below the mask's -1e9: the masked columns then carry weight, as in
    the reference's fill-then-softmax."""
    s = torch.full((1, S, S), -1e9, device="cuda")
    s[0, 5] = -2e9
    s[0, 6] = float("-inf")
    A.attention_probs(s, 1, S, 1.0)
    assert torch.equal(s[0, 0], torch.full((S,), np.float32(1.0) / np.float32(S), device="cuda"))
    want = torch.zeros(S, device="cuda")
    want[6:] = 1.0 / (S - 6)
    assert torch.allclose(s[0, 5], want, rtol=1e-6, atol=0)
    want = torch.zeros(S, device="cuda")
    want[7:] = 1.0 / (S - 7)
    assert torch.allclose(s[0, 6], want, rtol=1e-6, atol=0)


@pytest.mark.parametrize("cols", [33, 64, 255, 256, 1025, 1028])
def test_rows_of_special_values(gpu, cols):
    """A NaN, an infinity or nothing but -inf makes its own row NaN and no other (rows share a
    wave); a -inf among finite scores weighs nothing. Tolerance as for the plain rows."""
    rows = 16387
    x = _normal((rows, cols), 40, 3.0)
    for r, value in ((1, float("nan")), (6, float("inf")), (16384, float("-inf"))):
        x[r, cols // 2] = value
    x[10] = float("-inf")
    out = torch.empty_like(x)
    A.softmax(out, x, rows, cols)
    p = torch.softmax(x.double(), -1)
    assert torch.equal(out.isnan(), p.isnan())
    assert (out.double() - p).nan_to_num().abs().max().item() <= 1e-6
    assert out[16384, cols // 2].item() == 0.0


@pytest.mark.parametrize("L,H", [(1022, 700), (3, 700), (33, 700), (64, 1400), (65, 700),
                                 (1300, 700), (1301, 700), (64, 2800), (100, 700), (100, 1400),
                                 (101, 1400), (100, 2800), (101, 2800), (300, 700), (301, 700),
                                 (300, 1400), (301, 1400), (1000, 700)])
def test_length_rows(gpu, L, H):
    """decode_probs over rows of `L` columns: only the first lens keys, zero past them, a zero
    row for an empty cache."""
    n = 6
    s = _normal((n * H, L), 30, 4.0)
    lens = torch.tensor([1, 0, L // 2 + 1, L, min(4, L), L // 4 + 1], dtype=torch.int32,
                        device="cuda")
    keep = torch.arange(L, device="cuda") < lens.repeat_interleave(H).unsqueeze(1)
    probs = s.masked_fill(~keep, float("nan"))
    A.decode_probs(probs, lens, n, H, L, 0.5)
    p = torch.softmax((s.double() * 0.5).masked_fill(~keep, float("-inf")), -1)
    p[lens.repeat_interleave(H) == 0] = 0.0
    assert (probs.double() - p).abs().max().item() <= 1e-6
    assert torch.count_nonzero(probs[~keep]).item() == 0
