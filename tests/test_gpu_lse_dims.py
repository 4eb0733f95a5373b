"""The logsumexp kernel at the head dims that return_lse took the fp32 torch formula for, 96 (128-channel LDS rows) and
256, against float64: at most 2^-23 of the value (its own rounding is 2^-24) plus the scores' fp32 accumulation, on lengths
around a tile, both layouts, strided heads, grouped heads and the causal diagonal."""
import pytest
import torch

import cdna4_sage
import sageattention
from sageattention import core
from cdna4_sage._attention import row_lse

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [96, 256])
@pytest.mark.parametrize("B,H,Hkv,Sq,Skv,dt,layout,causal,sm", [
    (1, 2, 2, 1, 1, "bf16", "HND", False, None), (2, 4, 2, 33, 63, "f16", "NHD", False, 0.05),
    (1, 4, 1, 128, 64, "bf16", "NHD", False, None), (1, 2, 2, 129, 65, "f16", "HND", False, None),
    (1, 3, 3, 257, 1031, "bf16", "NHD", True, None), (2, 4, 2, 500, 500, "f16", "HND", True, 0.2),
    (1, 8, 8, 1000, 1000, "bf16", "HND", True, None)])
def test_lse_of_head_dims_96_and_256(dev, D, B, H, Hkv, Sq, Skv, dt, layout, causal, sm):
    dtype = torch.bfloat16 if dt == "bf16" else torch.float16
    g = torch.Generator(device=dev).manual_seed(D + Skv)

    def draw(h, s):  # a slice of wider rows: neither contiguous nor without a gap between heads
        t = torch.randn((B, s, h, D + 32) if layout == "NHD" else (B, h, s, D + 32), generator=g, device=dev)
        return (t * 2).to(dtype)[..., 8:8 + D]

    q, k = draw(H, Sq), draw(Hkv, Skv)
    got = row_lse(q, k, layout, sm, causal)
    qh, kh = (t if layout == "HND" else t.transpose(1, 2) for t in (q, k))
    kt = kh.double().repeat_interleave(H // Hkv, 1).transpose(-1, -2).contiguous()
    scale = D ** -0.5 if sm is None else sm
    s = (qh.double() @ kt) * scale
    # fp32 accumulation of D products, each below |q||k|: D 2^-24 of the sum of their magnitudes, and the fp32 scale
    # of an exponent
    bound = (qh.double().abs() @ kt.abs()).amax(-1) * scale * (D * 2.0 ** -24)
    if causal:
        s.masked_fill_(torch.ones(Sq, Skv, dtype=torch.bool, device=dev).triu(Skv - Sq + 1), float("-inf"))
    ref = torch.logsumexp(s, -1)
    assert ((got.double() - ref).abs() <= ref.abs() * 2.0 ** -23 + bound + 1e-6).all()
    with pytest.raises(cdna4_sage.Unsupported):
        cdna4_sage.lse(q, k, layout, sm, causal)


def test_return_lse_uses_the_kernel(dev):
    g = torch.Generator(device=dev).manual_seed(2)
    q, k, v = (torch.randn(1, 16, 3000, 256, generator=g, device=dev).to(torch.bfloat16) for _ in range(3))
    out, lse = sageattention.sageattn(q, k, v, is_causal=True, return_lse=True)
    assert torch.equal(lse, row_lse(q, k, "HND", None, True))
    assert torch.equal(out, sageattention.sageattn(q, k, v, is_causal=True))


@pytest.mark.parametrize("D", [96, 256])
def test_return_lse_with_gradients_keeps_the_torch_formula(dev, D):
    g = torch.Generator(device=dev).manual_seed(D)
    q, k = (torch.randn(1, 2, 70, D, generator=g, device=dev).to(torch.bfloat16).requires_grad_() for _ in range(2))
    lse = core._lse(q, k, "HND", True, None)
    lse.sum().backward()
    with torch.no_grad():
        # both are within 1e-6 of float64 in the 2-norm
        assert (core._lse(q, k, "HND", True, None) - lse).norm() <= 2e-6 * lse.norm()
    qd, kd = (t.detach().double().requires_grad_() for t in (q, k))
    s = (qd @ kd.transpose(-1, -2).contiguous()) * D ** -0.5
    s = s.masked_fill(torch.ones(70, 70, dtype=torch.bool, device=dev).triu(1), float("-inf"))
    torch.logsumexp(s, -1).sum().backward()
    for got, want in ((q.grad, qd.grad), (k.grad, kd.grad)):
        # the gradient's own bf16 rounding, 2^-9 an element
        assert (got.double() - want).norm() <= 2.0 ** -8 * want.norm()


@pytest.mark.parametrize("D", [64, 96, 128, 256])
@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("causal", [False, True])
def test_lse_of_infinite_scores_is_the_formula_s(dev, D, dt, causal):
    """Rows with infinite or very large scores (from infinite inputs, from products past fp32, of one sign or both, in the first key tile or
    a later one) and with NaN: infinite or NaN exactly where torch.logsumexp of the scores is, the other rows as always."""
    dtype = torch.bfloat16 if dt == "bf16" else torch.float16
    g = torch.Generator(device=dev).manual_seed(D)
    S, inf = 200, float("inf")
    q, k = (torch.randn(1, 3, S, D, generator=g, device=dev) for _ in range(2))
    q[..., 0] = 0.0                     # channel 0 meets the keys below in the rows that set it
    k[..., 0] = 1.0
    q[0, :, 3, 0] = q[0, :, 150, 0] = inf
    q[0, :, 40, 0] = q[0, :, 199, 0] = -inf
    k[0, 1, 70, 0] = -1.0               # head 1: one score of the other sign
    k[0, 2, 71, 0] = 0.0                # head 2: one NaN
    q[0, 0, 100, 5] = float("nan")
    # scores so large that the rounding of one in fp32 is far above the terms' exponents (f16: 65000 x 65000)
    q[0, :, 20:24, 0] = torch.tensor([1.0, -1.0, 1.0, -1.0], device=dev) * (1e9 if dt == "bf16" else 65000.0)
    k[0, 0, 10:13, 0] = 3e9 if dt == "bf16" else 65000.0
    if dt == "bf16":                    # products past the largest fp32
        q[0, 0, 60:64, 0] = torch.tensor([1e30, -1e30, 1e30, -1e30], device=dev)
        k[0, 0, 90:94, 0] = 1e30
    q, k = q.to(dtype), k.to(dtype)
    got = row_lse(q, k, "HND", None, causal)
    s = (q.float() @ k.float().transpose(-1, -2).contiguous()) * D ** -0.5
    if causal:
        s.masked_fill_(torch.ones(S, S, dtype=torch.bool, device=dev).triu(1), -inf)
    want = torch.logsumexp(s, -1)
    assert int((want == inf).sum()) >= 2 and int((want == -inf).sum()) >= 2 and int(want.isnan().sum()) >= 2
    assert torch.equal(got.isnan(), want.isnan())
    odd = want.isinf()
    assert torch.equal(got[odd], want[odd])
    rest = want.isfinite()
    torch.testing.assert_close(got[rest], want[rest], atol=1e-5, rtol=1e-6)
