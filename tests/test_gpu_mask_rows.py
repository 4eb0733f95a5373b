"""Additive masks as the kernels read them from the caller's tensor: rows at any element alignment and stride, broadcast
axes, a partial last key tile, the causal diagonal, and rows further apart than a 32-bit offset reaches.  However a mask
is laid out, the output must be that of its contiguous copy bit for bit; the copy's is checked against float64."""
import pytest
import torch

import cdna4_sage

pytestmark = pytest.mark.gpu
BF16, F16 = torch.bfloat16, torch.float16


def _qkv(dev, B, H, Sq, Skv, D, dt, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    r = lambda s: torch.randn((B, H, s, D), generator=g, device=dev, dtype=torch.float32).to(dt)  # noqa: E731
    return (r(Sq), r(Skv), r(Skv)), g


def _values(g, shape, dev, dt):
    """Biases with every class of tile: general values, all-zero and all -inf blocks, 0 / -inf blocks."""
    m = torch.randn(shape, generator=g, device=dev, dtype=torch.float32) * 2
    m[..., :64] = torch.where(m[..., :64] > 1.5, float("-inf"), 0.0)
    if shape[-1] > 192:
        m[..., 64:128] = 0.0
        m[..., 128:192] = float("-inf")
    return m.to(dt)


@pytest.mark.parametrize("B,H,Sq,Skv,D,dt,causal,rows", [
    (1, 2, 200, 448, 64, BF16, False, "b1h"), (2, 2, 129, 333, 64, F16, False, "bh"), (1, 3, 70, 65, 128, BF16, False, "1h"),
    (2, 2, 257, 511, 128, F16, True, "b1"), (1, 2, 96, 700, 96, BF16, True, "h"), (1, 2, 130, 321, 256, BF16, True, "1h"),
    (1, 2, 300, 1088, 256, F16, False, "keys"), (1, 2, 40, 127, 64, BF16, False, "keys"),
    (1, 4, 300, 1500, 128, BF16, True, "keys"),
])
def test_mask_layouts_give_the_same_bits(dev, B, H, Sq, Skv, D, dt, causal, rows):
    (q, k, v), g = _qkv(dev, B, H, Sq, Skv, D, dt, Sq + Skv)
    shape = {"b1h": (B, 1, Sq), "bh": (B, H, Sq), "1h": (1, H, Sq), "b1": (B, 1, Sq), "h": (1, H, Sq),
             "keys": (1, 1, 1)}[rows] + (Skv,)
    mask = _values(g, shape, dev, dt)
    out = cdna4_sage.attention(q, k, v, "HND", is_causal=causal, attn_mask=mask)
    s = q.double() @ k.double().transpose(-1, -2).contiguous() * D ** -0.5 + mask.double()
    if causal:
        s.masked_fill_(torch.ones(Sq, Skv, dtype=torch.bool, device=dev).triu(Skv - Sq + 1), float("-inf"))
    ref = torch.nan_to_num(torch.softmax(s, -1)) @ v.double()
    assert torch.isfinite(out).all()
    # E4M3 probabilities and V: 4e-2 of the outputs' 2-norm on random values, as on every dense shape
    assert (out.double() - ref).norm() <= 0.06 * ref.norm()
    # the same values at other alignments and strides, NaN around every row: nothing outside the rows may be read into
    # the scores
    for before, after in ((1, 0), (8, 3), (5, 61), (64, 64)):
        wide = torch.full(shape[:-1] + (before + Skv + after,), float("nan"), device=dev, dtype=dt)
        wide[..., before:before + Skv] = mask
        view = wide[..., before:before + Skv]
        assert torch.equal(cdna4_sage.attention(q, k, v, "HND", is_causal=causal, attn_mask=view), out), (before, after)
    full = mask.expand(B, H, Sq, Skv)
    assert torch.equal(cdna4_sage.attention(q, k, v, "HND", is_causal=causal, attn_mask=full), out)
    assert torch.equal(cdna4_sage.attention(q, k, v, "HND", is_causal=causal, attn_mask=full.contiguous()), out)


@pytest.mark.parametrize("D", [64, 256])
def test_mask_rows_further_apart_than_32_bits(dev, D):
    B, H, Sq, Skv = 1, 2, 40, 200
    (q, k, v), g = _qkv(dev, B, H, Sq, Skv, D, BF16, 3)
    mask = _values(g, (Sq, Skv), dev, BF16)
    out = cdna4_sage.attention(q, k, v, "HND", attn_mask=mask)
    stride = (1 << 26) + 24                                     # 40 rows: 5 GiB, the lanes of a wave past 4 GiB
    view = torch.empty(Sq * stride, device=dev, dtype=BF16).as_strided((Sq, Skv), (stride, 1))
    view.copy_(mask)
    assert torch.equal(cdna4_sage.attention(q, k, v, "HND", attn_mask=view), out)
