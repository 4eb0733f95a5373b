"""The attention's split plans that keep fp32 partials: dense launches that split the tiles past a multiple of the CUs,
causal launches of few tiles, and their boundaries.  A split call (its workspace filled with NaN first) is compared with
the same call without a workspace, which runs every tile whole: the ranges start from the whole walk's running max, so
they form its own probabilities and only the fp32 sums differ in order."""
import ctypes

import pytest
import torch

from cdna4_sage import _capi

pytestmark = pytest.mark.gpu
BF16, F16 = torch.bfloat16, torch.float16
CASES = [  # B, H, Hkv, Sq, Skv, D, dtype, causal, whole tiles, ranges (256 CUs)
    (1, 20, 20, 3333, 2050, 64, F16, False, 512, 8),      # 28 tiles past 2 x 256, 33 key tiles
    (2, 10, 10, 4096, 4096, 64, F16, False, 512, 2),      # 128 tiles past 2 x 256
    (1, 33, 33, 2040, 2047, 128, BF16, False, 512, 8),    # 16 tiles past, 32 key tiles (the last partial): the line
    (1, 33, 33, 2040, 1984, 128, BF16, False, 528, 1),    # 31 key tiles: below it
    (1, 27, 27, 4000, 1281, 128, BF16, False, 768, 2),    # past the first round, 21 key tiles
    (1, 32, 32, 1100, 3073, 256, F16, False, 256, 8),     # one tile per CU and 32 more, head dim 256
    (1, 30, 30, 4480, 2111, 96, BF16, False, 1024, 8),
    (1, 4, 2, 300, 1500, 128, BF16, True, 0, 6),          # causal chunk, the last range short
    (1, 6, 6, 1, 700, 64, F16, True, 0, 2),               # one query row
    (2, 3, 1, 257, 513, 256, F16, True, 0, 2),
    (1, 8, 8, 2048, 2048, 96, BF16, True, 0, 6),          # square: the first tiles' later ranges are empty
    (1, 3, 3, 130, 8191, 128, BF16, True, 0, 16),
    (1, 16, 16, 2048, 2048, 128, BF16, True, 256, 1),     # square, as many tiles as CUs and a short walk: whole
    (1, 12, 12, 4096, 6300, 64, BF16, True, 384, 1),      # more tiles than CUs, fewer than half the keys before them
]


def _quantized(dev, B, H, Hkv, Sq, Skv, D, dt, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    q, k, v = (torch.randn((B, h, s, D), generator=g, device=dev, dtype=torch.float32).to(dt)
               for h, s in ((H, Sq), (Hkv, Skv), (Hkv, Skv)))
    dl, skp, code = _capi.layout_dim(D), _capi.kv_pad(Skv), _capi.DTYPE_BF16 if dt == BF16 else _capi.DTYPE_F16
    q8 = torch.empty(B, H, Sq, dl, dtype=torch.int8, device=dev)
    qs = torch.empty(B, H, Sq, device=dev)
    k8 = torch.empty(B, Hkv, skp, dl, dtype=torch.int8, device=dev)
    ks = torch.empty(B, Hkv, skp // 32, device=dev)
    v8t = torch.empty(B, Hkv, dl, skp, dtype=torch.uint8, device=dev)
    vs = torch.empty(B, Hkv, dl, device=dev)
    st = torch.cuda.current_stream(dev).cuda_stream
    p = [t.data_ptr() for t in (q8, qs, k8, ks, v8t, vs)]
    qst, kst = (H * Sq * D, D, Sq * D), (Hkv * Skv * D, D, Skv * D)
    _capi.call("sage_quant_q", q.data_ptr(), *qst, B, H, Sq, D, code, 1.0, p[0], p[1], st)
    _capi.call("sage_v_amax", v.data_ptr(), *kst, B, Hkv, Skv, D, code, p[5], st)
    _capi.call("sage_quant_kv", k.data_ptr(), *kst, v.data_ptr(), *kst, B, Hkv, Skv, D, code, p[5], p[2], p[3], p[4], st)
    torch.cuda.synchronize(dev)
    return (q8, qs, k8, ks, v8t, vs), code


@pytest.mark.parametrize("B,H,Hkv,Sq,Skv,D,dt,causal,n_full,chunks", CASES)
def test_split_plan_against_whole_tiles(dev, B, H, Hkv, Sq, Skv, D, dt, causal, n_full, chunks):
    full, ch, ws = _capi.attn_plan(dev.index or 0, B, H, Sq, Skv, D, causal)
    assert (full, ch) == (n_full, chunks)
    n = B * H * ((Sq + 127) // 128)
    dl = _capi.layout_dim(D)
    wide = causal or n > 256
    assert ws == (n - full) * (ch if ch > 1 else 0) * 128 * ((4 if wide else 2) * dl + 8)
    t, code = _quantized(dev, B, H, Hkv, Sq, Skv, D, dt, seed=Sq + D)
    outs, lses = [], []
    for size in (0, ws):
        out = torch.full((B, Sq, H, D), float("nan"), device=dev, dtype=dt)
        lse = torch.full((B, H, Sq), float("nan"), device=dev)
        buf = torch.full((max(size, 4) // 4,), float("nan"), device=dev)
        _capi.call("sage_attn_fwd", *(x.data_ptr() for x in t), out.data_ptr(), *out.stride()[:3], B, H, Hkv, Sq, Skv, D,
                   int(causal), code, lse.data_ptr(), buf.data_ptr() if size else None, size,
                   torch.cuda.current_stream(dev).cuda_stream)
        torch.cuda.synchronize(dev)
        outs.append(out.float())
        lses.append(lse)
    whole, split = outs
    assert torch.isfinite(split).all() and torch.isfinite(lses[1]).all()
    if ch == 1:
        assert torch.equal(split, whole)
        return
    # Rows whose ranges all start from the walk's max form its probabilities; their fp32 sums in another order move a
    # few outputs to the neighbouring bf16 / fp16 value (2^-8 / 2^-11 relative).
    # The first 32-row group of a causal tile that does not see all of key tile 0 takes its ranges from -inf, with other
    # E4M3 roundings (a relative 2^-4 of single probabilities): within 2e-2, like every output against the emulation.
    step = 2.0 ** (-8 if dt == BF16 else -11)
    near = (split - whole).abs() <= 1.01 * step * whole.abs().clamp_min(1e-3)
    seeded = torch.ones(Sq, dtype=torch.bool, device=dev)
    if causal:
        first = torch.arange(Sq, device=dev) // 32 * 32
        seeded = first + (Skv - Sq) >= 63
    assert near[:, seeded].float().mean() >= 0.999
    assert (split - whole).abs().max() <= 2e-2
    torch.testing.assert_close(lses[1], lses[0], atol=1e-5 if bool(seeded.all()) else 2e-3, rtol=1e-6)


def test_noalloc_runs_whole_where_only_the_partials_do_not_fit(dev):
    """A shape whose intermediates fill the library's scratch array up to less than its split tiles' partials: the call
    is accepted as before and gives the whole-tile output."""
    B, H, Sq, Skv, D = 1, 32, 1024, 12000, 128
    dl, skp, n = D, _capi.kv_pad(Skv), 32
    inter = n * (Sq * (dl + 4) + skp * (2 * dl) + skp // 8 + dl * 4)
    full, ch, ws = _capi.attn_plan(dev.index or 0, B, H, Sq, Skv, D, True)
    assert ch > 1 and inter < 128 << 20 < inter + ws
    g = torch.Generator(device=dev).manual_seed(5)
    q, k, v = (torch.randn((B, H, s, D), generator=g, device=dev, dtype=torch.float32).to(BF16) for s in (Sq, Skv, Skv))
    lib = _capi.lib()
    out = torch.empty(B, Sq, H, D, device=dev, dtype=BF16)
    qst, kst = (H * Sq * D, D, Sq * D), (H * Skv * D, D, Skv * D)
    rc = lib.sage_forward_noalloc(q.data_ptr(), *qst, k.data_ptr(), *kst, v.data_ptr(), *kst, out.data_ptr(),
                                  *out.stride()[:3], B, H, H, Sq, Skv, D, _capi.DTYPE_BF16, 1, 1.0,
                                  ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream))
    assert rc == _capi.SAGE_OK, _capi.lib().sage_last_error()
    t, code = _quantized(dev, B, H, H, Sq, Skv, D, BF16, seed=5)
    whole = torch.empty_like(out)
    _capi.call("sage_attn_fwd", *(x.data_ptr() for x in t), whole.data_ptr(), *whole.stride()[:3], B, H, H, Sq, Skv, D, 1,
               code, None, None, 0, torch.cuda.current_stream(dev).cuda_stream)
    torch.cuda.synchronize(dev)
    assert torch.equal(out, whole)


@pytest.mark.parametrize("B,H,Sq,L,D,n_full,chunks", [
    (1, 22, 3840, 47, 256, 660, 1), (1, 22, 3840, 48, 256, 512, 3),        # 148 tiles in the last round: three ranges
    (1, 32, 4096, 111, 128, 1024, 1), (1, 32, 4096, 112, 128, 768, 3),     # a tile for every CU in it
    (1, 21, 8192, 111, 64, 1280, 4), (1, 21, 8192, 112, 64, 1024, 3),      # fp32 past the CUs before, 320 tiles after
    (1, 12, 8192, 127, 256, 768, 1), (1, 12, 8192, 128, 256, 512, 2),      # two ranges
    (1, 14, 4096, 127, 64, 448, 1), (1, 14, 4096, 128, 64, 0, 2),
    (1, 24, 8192, 512, 64, 1536, 1),                                        # two full tiles per CU: whole
    (1, 40, 32760, 512, 128, 9984, 3),
])
def test_plan_of_long_walks(dev, B, H, Sq, L, D, n_full, chunks):
    full, ch, ws = _capi.attn_plan(dev.index or 0, B, H, Sq, L * 64, D, 0)
    assert (full, ch) == (n_full, chunks)
    rem = B * H * ((Sq + 127) // 128) - full
    assert ws == (rem * ch * 128 * ((4 if ch == 4 else 2) * D + 8) if ch > 1 else 0)


def test_three_ranges_of_head_dim_256_against_whole_tiles(dev):
    B, H, Sq, Skv, D, dt = 1, 22, 3801, 3067, 256, BF16
    full, ch, ws = _capi.attn_plan(dev.index or 0, B, H, Sq, Skv, D, 0)
    assert (full, ch) == (512, 3)
    t, code = _quantized(dev, B, H, H, Sq, Skv, D, dt, seed=11)
    outs = []
    for size in (0, ws):
        out = torch.full((B, Sq, H, D), float("nan"), device=dev, dtype=dt)
        buf = torch.full((max(size, 4) // 4,), float("nan"), device=dev)
        _capi.call("sage_attn_fwd", *(x.data_ptr() for x in t), out.data_ptr(), *out.stride()[:3], B, H, H, Sq, Skv, D, 0,
                   code, None, buf.data_ptr() if size else None, size, torch.cuda.current_stream(dev).cuda_stream)
        torch.cuda.synchronize(dev)
        outs.append(out.double())
    whole, split = outs
    # the same probabilities: the fp16 partials' rounding (2^-11) and the output's own (2^-9, twice)
    assert (split - whole).norm() <= 2.0 ** -8 * whole.norm()


@pytest.mark.parametrize("B,H,Sq,L,D,n_full,chunks,fp32", [
    (1, 16, 2304, 31, 64, 288, 1, False), (1, 16, 2304, 32, 64, 0, 3, False),     # up to half a tile per CU past the first
    (1, 16, 2944, 47, 64, 368, 1, False), (1, 16, 2944, 48, 64, 0, 2, False),
    (1, 16, 6400, 7, 128, 800, 1, False), (1, 16, 6400, 8, 128, 768, 2, False),   # 32 tiles past a full round
    (1, 16, 6656, 11, 128, 832, 1, False), (1, 16, 6656, 12, 128, 768, 3, False),  # 64: from three ranges, one unit a CU
    (1, 16, 6656, 19, 96, 768, 4, False), (1, 16, 6656, 20, 96, 768, 4, True),     # five would not fit: past the CUs, fp32
    (1, 16, 7296, 39, 128, 912, 1, False), (1, 16, 7296, 40, 128, 768, 5, False),  # more than half a tile per CU
    (1, 16, 4352, 16, 256, 512, 4, False), (1, 16, 4352, 20, 256, 512, 5, False),
    (1, 16, 7168, 31, 256, 896, 1, False), (1, 16, 7168, 32, 256, 768, 2, True),   # two workgroups per CU
    (1, 16, 6272, 20, 256, 768, 5, True),
    (1, 12, 7680, 95, 256, 720, 1, False), (1, 12, 7680, 96, 256, 512, 2, False),  # 208 tiles: CUs without one
])
def test_plan_of_short_walks(dev, B, H, Sq, L, D, n_full, chunks, fp32):
    full, ch, ws = _capi.attn_plan(dev.index or 0, B, H, Sq, L * 64, D, 0)
    assert (full, ch) == (n_full, chunks)
    rem, dl = B * H * ((Sq + 127) // 128) - full, _capi.layout_dim(D)
    assert ws == (rem * ch * 128 * ((4 if fp32 else 2) * dl + 8) if ch > 1 else 0)


@pytest.mark.parametrize("H,Sq,L,D,chunks", [
    (8, 250, 7, 64, 1), (8, 250, 8, 64, 2), (8, 500, 9, 128, 1), (8, 500, 10, 128, 2),           # 16 and 32 tiles
    (32, 250, 15, 256, 1), (32, 250, 16, 256, 4), (8, 1250, 47, 128, 3), (8, 1250, 48, 128, 9),  # 64 and 80
    (32, 350, 23, 128, 1), (32, 350, 24, 128, 6), (32, 500, 31, 256, 1), (32, 500, 32, 256, 2),  # 96 and 128
    (32, 500, 39, 256, 2), (32, 500, 40, 256, 4), (32, 1000, 63, 128, 1), (32, 1000, 64, 128, 3),
    (32, 1000, 79, 256, 1), (32, 1000, 80, 256, 2), (32, 850, 55, 256, 1), (32, 850, 56, 256, 2),  # 256 and 224
    (8, 4096, 64, 256, 2),
])
def test_causal_plan_of_short_walks(dev, H, Sq, L, D, chunks):
    n = H * ((Sq + 127) // 128)
    full, ch, ws = _capi.attn_plan(dev.index or 0, 1, H, Sq, L * 64, D, True)
    assert (full, ch) == (n if chunks == 1 else 0, chunks)
    assert ws == (n * ch * 128 * (4 * _capi.layout_dim(D) + 8) if ch > 1 else 0)
