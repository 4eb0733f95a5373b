"""sage_forward's one-launch quantization of short key ranges (every workgroup of V owns 16 channels of a head over all its
keys) against the stage path (V maxima, Q, K and V in launches of their own): the same bytes at the edges of its passes,
of the padding and of its range, for every head dim, both dtypes and token-major strides."""
import pytest
import torch

from cdna4_sage import _capi

pytestmark = pytest.mark.gpu
CASES = [(1, 2, 2, 70, n, D, dt, layout) for n, D, dt, layout in (
    (1, 64, "bf16", "HND"), (63, 128, "f16", "NHD"), (64, 96, "bf16", "HND"), (77, 64, "f16", "NHD"),
    (128, 256, "bf16", "NHD"), (129, 96, "f16", "NHD"), (511, 128, "bf16", "HND"), (512, 256, "f16", "HND"),
    (513, 64, "bf16", "NHD"), (897, 256, "bf16", "NHD"), (1000, 96, "bf16", "NHD"), (1024, 128, "f16", "HND"),
    (1024, 64, "bf16", "NHD"), (1025, 64, "bf16", "HND"))]
CASES += [(2, 6, 3, 300, 333, 128, "bf16", "NHD"),
          (2, 16, 16, 64, 1024, 128, "bf16", "HND"),    # 8 MiB of V: the last one-launch size
          (1, 33, 33, 64, 1024, 128, "bf16", "HND"),    # past it
          (2, 24, 24, 64, 77, 256, "f16", "HND"), (1, 49, 49, 64, 77, 256, "f16", "NHD"),   # 768 slices, and past it
          (3, 64, 32, 64, 77, 96, "bf16", "NHD"), (3, 65, 65, 64, 77, 64, "bf16", "HND")]


@pytest.mark.parametrize("B,H,Hkv,Sq,Skv,D,dt,layout", CASES)
def test_one_launch_quantization_is_the_stages(dev, B, H, Hkv, Sq, Skv, D, dt, layout):
    dtype, code = (torch.bfloat16, _capi.DTYPE_BF16) if dt == "bf16" else (torch.float16, _capi.DTYPE_F16)
    g = torch.Generator(device=dev).manual_seed(Skv + D)

    def draw(h, s):
        t = torch.randn((B, s, h, D) if layout == "NHD" else (B, h, s, D), generator=g, device=dev)
        t[..., 3] = 0.0                     # a channel without a maximum
        t[..., 5] *= 100.0
        t = t.to(dtype)
        return t if layout == "NHD" else t.transpose(1, 2)

    q, k, v = draw(H, Sq), draw(Hkv, Skv), draw(Hkv, Skv)      # [B, S, heads, D], either stride order
    dl, skp = _capi.layout_dim(D), _capi.kv_pad(Skv)
    ws = _capi.forward_workspace(dev.index or 0, B, H, Hkv, Sq, Skv, D, False)
    got = []
    for size in (ws, 0):
        t = [torch.full((n,), 0xA5, device=dev, dtype=torch.uint8) for n in (
            B * H * Sq * dl, B * H * Sq * 4, B * Hkv * skp * dl, B * Hkv * skp // 8, B * Hkv * dl * skp, B * Hkv * dl * 4)]
        buf = torch.full((max(size, 1),), 0xFF, device=dev, dtype=torch.uint8)
        out = torch.empty(B, Sq, H, D, device=dev, dtype=dtype)
        _capi.call("sage_forward", q.data_ptr(), *q.stride()[:3], k.data_ptr(), *k.stride()[:3], v.data_ptr(),
                   *v.stride()[:3], out.data_ptr(), *out.stride()[:3], B, H, Hkv, Sq, Skv, D, code, 0, 1.0,
                   *(x.data_ptr() for x in t), buf.data_ptr() if size else None, size,
                   torch.cuda.current_stream(dev).cuda_stream)
        torch.cuda.synchronize(dev)
        assert torch.isfinite(out).all()
        got.append(t)
    for name, one, stages in zip(("q8", "qs", "k8", "ks", "v8t", "vs"), *got):
        assert torch.equal(one, stages), name
