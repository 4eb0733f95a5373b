"""The tables of a packed batch, made in one launch for at most 64 sequences and in two past that: the padded key offsets,
the owner of every padded 128-key block, and every (sequence, head, query tile) once, sequences with more keys first."""
import random

import pytest
import torch

from cdna4_sage import _capi

pytestmark = pytest.mark.gpu


def _align(n):
    return (n + 255) // 256 * 256


@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("batch,H,broken", [(1, 8, None), (2, 3, None), (63, 2, None), (64, 8, None), (65, 8, None),
                                            (64, 2, "past"), (3, 2, "down"), (65, 2, "past")])
def test_tables(dev, batch, H, broken, causal):
    rng = random.Random(batch * 8 + H)
    lens_q = [rng.choice([0, 1, 127, 128, 129, 300]) for _ in range(batch)]
    lens_k = [rng.choice([0, 1, 64, 65, 128, 400]) for _ in range(batch)]
    lens_q[-1], lens_k[0] = 200, 250
    cu_q, cu_k = ([sum(n[:i]) for i in range(batch + 1)] for n in (lens_q, lens_k))
    TQ, TK, D = cu_q[-1], cu_k[-1], 64
    if broken == "past":
        cu_k[-1] += 1
    elif broken == "down":
        cu_q[1] = cu_q[2] + 1
    tkp, wsb = _capi.varlen_layout(batch, H, H, TQ, TK)
    g = torch.Generator(device=dev).manual_seed(batch)
    q, k, v = (torch.randn(n, H, D, generator=g, device=dev).to(torch.bfloat16) for n in (TQ, TK, TK))
    out = torch.full((TQ, H, D), 7.0, device=dev, dtype=torch.bfloat16)
    sizes = (H * TQ * D, H * TQ * 4, H * tkp * D, H * tkp // 32 * 4, H * D * tkp, batch * H * D * 4, wsb)
    bufs = [torch.full((_align(n),), 0x5A, dtype=torch.uint8, device=dev) for n in sizes]
    cq, ck = (torch.tensor(c, dtype=torch.int32, device=dev) for c in (cu_q, cu_k))
    _capi.call("sage_forward_varlen", q.data_ptr(), H * D, D, k.data_ptr(), H * D, D, v.data_ptr(), H * D, D, out.data_ptr(),
               H * D, D, cq.data_ptr(), ck.data_ptr(), batch, H, H, TQ, TK, D, _capi.DTYPE_BF16, causal, 1.0,
               *(b.data_ptr() for b in bufs), wsb, torch.cuda.current_stream(dev).cuda_stream)
    torch.cuda.synchronize(dev)
    words = bufs[-1].view(torch.int32).cpu().tolist()
    o_kp = 256
    o_ktab = _align(_align(_align(o_kp + (batch + 1) * 4) + batch * 4) + (batch + 1) * 4)
    o_tiles = _align(o_ktab + tkp // 128 * 4)
    n_blocks = H * ((TQ + 127 * batch) // 128)
    ktab = words[o_ktab // 4:o_ktab // 4 + tkp // 128]
    tiles = [tuple(words[o_tiles // 4 + 4 * i:o_tiles // 4 + 4 * i + 3]) for i in range(n_blocks)]
    if broken:
        assert words[0] == 1 and set(ktab) == {-1} and all(t[0] == -1 for t in tiles) and bool((out == 7.0).all())
        return
    pads = [(n + 127) // 128 * 128 for n in lens_k]
    kp = [sum(pads[:i]) for i in range(batch + 1)]
    assert words[0] == 0 and words[o_kp // 4:o_kp // 4 + batch + 1] == kp
    owners = [b for b in range(batch) for _ in range(pads[b] // 128)]
    assert ktab == owners + [-1] * (tkp // 128 - len(owners))
    want = [(b, h, t) for b in range(batch) for h in range(H) for t in range((lens_q[b] + 127) // 128)]
    n = len(want)
    assert sorted(tiles[:n]) == want and all(t[0] == -1 for t in tiles[n:])
    walks = [(lens_k[b] + 63) // 64 for b, _, _ in tiles[:n]]
    assert walks == sorted(walks, reverse=True)
    seqs = [b for i, (b, _, _) in enumerate(tiles[:n]) if i == 0 or tiles[i - 1][0] != b]
    assert len(seqs) == len(set(seqs))  # a sequence's tiles follow one another
    assert torch.isfinite(out).all()
