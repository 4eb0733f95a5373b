"""Masked calls whose plan splits tiles with fp32 partials (the mask kernels choose the format at run time, and the host the
merge kernel).  The inputs of the last head, whose tiles are split, are those of the first, whose tiles are whole.  Where
every range starts from the walk's max (a mask of keys) the two outputs differ by the order of fp32 sums alone; where some
row's does not (its first visible tile comes later, or a bias raises its max) other E4M3 roundings are as close to float64.
Masks that hide nothing give the unmasked call bit for bit, and masks of 0 and -inf the bool mask's."""
import pytest
import torch

import cdna4_sage
from cdna4_sage import _capi

pytestmark = pytest.mark.gpu
BF16, F16 = torch.bfloat16, torch.float16
SHAPES = [  # B, H, Sq, Skv, D, dtype, whole tiles, ranges (256 CUs)
    (1, 33, 2040, 2047, 128, BF16, 512, 8), (2, 10, 4096, 4096, 64, F16, 512, 2),
    (1, 30, 4480, 2111, 96, BF16, 1024, 8), (1, 32, 1100, 3073, 256, BF16, 256, 8)]


def _case(dev, B, H, Sq, Skv, D, dt, n_full, chunks):
    full, ch, ws = _capi.attn_plan(dev.index or 0, B, H, Sq, Skv, D, False)
    units = (B * H * ((Sq + 127) // 128) - full) * ch
    assert (full, ch) == (n_full, chunks) and ws == units * 128 * (4 * _capi.layout_dim(D) + 8)
    g = torch.Generator(device=dev).manual_seed(Sq + D)
    q, k, v = (torch.randn((B, H, s, D), generator=g, device=dev).to(dt) for s in (Sq, Skv, Skv))
    for t in (q, k, v):
        t[-1, -1] = t[0, 0]
    return q, k, v, g


def _masks(dev, g, Sq, Skv, dt):
    """name -> (mask, causal): every walk the plan tells apart, with class 0 to 3 tiles and a hidden first tile."""
    keys = torch.rand(Skv, generator=g, device=dev) < 0.8
    keys[:70] = False
    row, key = torch.arange(Sq, device=dev)[:, None], torch.arange(Skv, device=dev)[None]
    band = (key * Sq // Skv - row).abs() < Sq // 2
    bias = torch.randn(Sq, Skv, generator=g, device=dev) * 2
    bias[:, 128:192] = float("-inf")
    bias[:, 256:320] = 0.0
    bias[:, 320:384] = torch.where(bias[:, 320:384] > 0, 0.0, float("-inf"))

    def inf(m):
        return torch.where(m, 0.0, float("-inf")).to(dt)

    out = {"keys": (keys[None, None, None], False), "keys inf": (inf(keys), False), "band": (band, False),
           "band inf": (inf(band), False), "bias": (bias.to(dt), False), "key bias": (bias[7].to(dt), False)}
    if Sq <= Skv:
        out["bias causal"] = (bias.to(dt), True)
    return out


@pytest.mark.parametrize("shape", SHAPES)
def test_split_head_is_the_whole_one(dev, shape):
    B, H, Sq, Skv, D, dt = shape[:6]
    q, k, v, g = _case(dev, *shape)
    outs = {}
    for name, (mask, causal) in _masks(dev, g, Sq, Skv, dt).items():
        out = outs[name] = cdna4_sage.attention(q, k, v, "HND", is_causal=causal, attn_mask=mask)
        assert torch.isfinite(out).all(), name
        whole, split = out[0, 0].double(), out[-1, -1].double()
        if name.startswith("keys"):
            # fp32 sums in another order move a few outputs to the neighbouring bf16 / fp16 value
            step = 2.0 ** (-8 if dt == BF16 else -11)
            assert ((split - whole).abs() <= 1.01 * step * whole.abs().clamp_min(1e-3)).double().mean() >= 0.999, name
        m = mask.reshape(-1, Skv)
        s = q[0, 0].double() @ k[0, 0].double().t().contiguous() * D ** -0.5
        s = s.masked_fill(~m, float("-inf")) if mask.dtype == torch.bool else s + m.double()
        if causal:
            s.masked_fill_(torch.ones(Sq, Skv, dtype=torch.bool, device=dev).triu(Skv - Sq + 1), float("-inf"))
        ref = torch.nan_to_num(torch.softmax(s, -1)) @ v[0, 0].double()
        # E4M3 probabilities and V, as on every dense shape; the two heads' errors are two draws of the same roundings,
        # each the norm over at least 261120 values (1 / sqrt(n) = 2e-3 of it)
        own = (whole - ref).norm()
        assert own <= 0.06 * ref.norm() and (split - ref).norm() <= 1.02 * own, name
    assert torch.equal(outs["keys"], outs["keys inf"])
    assert torch.equal(outs["band"][0, 0], outs["band inf"][0, 0])  # whole tiles (the bool mask's are whole in every head)
    assert torch.equal(outs["band"][-1, -1], outs["band"][0, 0])


@pytest.mark.parametrize("shape", SHAPES)
def test_masks_that_hide_nothing(dev, shape):
    B, H, Sq, Skv, D, dt = shape[:6]
    q, k, v, _ = _case(dev, *shape)
    want = cdna4_sage.attention(q, k, v, "HND")
    for mask in (torch.ones(Skv, dtype=torch.bool, device=dev), torch.zeros(Skv, dtype=dt, device=dev),
                 torch.zeros(Sq, Skv, dtype=dt, device=dev)):
        assert torch.equal(cdna4_sage.attention(q, k, v, "HND", attn_mask=mask), want)
