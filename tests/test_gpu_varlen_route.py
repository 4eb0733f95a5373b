"""The packed pass of the sequences that the router sends to the kernel (sage_forward_varlen_routed): the others have no query
tile and no key block, their output rows stay as they are, and a batch without a sequence for the kernel is not even
quantized.  What it takes is the unrouted pass, bit for bit."""
import random

import pytest
import torch

import cdna4_sage
import sageattention
from cdna4_sage import _capi
from sageattention import core

pytestmark = pytest.mark.gpu


def _align(n):
    return (n + 255) // 256 * 256


def _run(dev, lens_q, lens_k, H, Hkv, D, causal, route, seed):
    cu_q, cu_k = ([sum(n[:i]) for i in range(len(n) + 1)] for n in (lens_q, lens_k))
    TQ, TK, batch = cu_q[-1], cu_k[-1], len(lens_q)
    g = torch.Generator(device=dev).manual_seed(seed)
    q, k, v = (torch.randn(n, h, D, generator=g, device=dev).to(torch.bfloat16) for n, h in ((TQ, H), (TK, Hkv), (TK, Hkv)))
    out = torch.full((TQ, H, D), 7.0, device=dev, dtype=torch.bfloat16)
    tkp, wsb = _capi.varlen_layout(batch, H, Hkv, TQ, TK)
    sizes = (H * TQ * D, H * TQ * 4, Hkv * tkp * D, Hkv * tkp // 32 * 4, Hkv * D * tkp, batch * Hkv * D * 4, wsb)
    bufs = [torch.full((_align(n),), 0x5A, dtype=torch.uint8, device=dev) for n in sizes]
    cq, ck = (torch.tensor(c, dtype=torch.int32, device=dev) for c in (cu_q, cu_k))
    entry = "sage_forward_varlen" + ("" if route is None else "_routed")
    _capi.call(entry, q.data_ptr(), H * D, D, k.data_ptr(), Hkv * D, D, v.data_ptr(), Hkv * D, D, out.data_ptr(), H * D, D,
               cq.data_ptr(), ck.data_ptr(), batch, H, Hkv, TQ, TK, D, _capi.DTYPE_BF16, causal, 1.0, *(route or ()),
               *(b.data_ptr() for b in bufs), wsb, torch.cuda.current_stream(dev).cuda_stream)
    torch.cuda.synchronize(dev)
    return out, bufs, cu_q


@pytest.mark.parametrize("causal", [0, 1])
@pytest.mark.parametrize("batch,H,Hkv", [(1, 8, 8), (2, 3, 1), (7, 4, 2), (64, 2, 2), (65, 8, 4), (130, 2, 1)])
def test_routed_pass(dev, batch, H, Hkv, causal):
    rng = random.Random(batch + H)
    lens_q = [rng.choice([0, 1, 127, 128, 200, 300]) for _ in range(batch)]
    lens_k = [rng.choice([1, 64, 65, 128, 250, 400]) for _ in range(batch)]
    lens_q[-1], lens_k[-1] = 128, 250                      # exactly the least work below
    work = H * 128 * 250 // (2 if causal else 1)

    def taken(sq, sk, min_kv, min_work):
        return sk >= min_kv and H * sq * sk // (2 if causal else 1) >= min_work and not (causal and sq > sk)

    whole, _, cu = _run(dev, lens_q, lens_k, H, Hkv, 64, causal, None, batch)
    for route in ((250, work), (65, work + 1), (-2**63, -2**63), (2**63 - 1, 0), (0, 2**63 - 1)):
        out, bufs, _ = _run(dev, lens_q, lens_k, H, Hkv, 64, causal, route, batch)
        words = bufs[-1].view(torch.int32).cpu().tolist()
        takes = [taken(a, b, *route) for a, b in zip(lens_q, lens_k)]
        assert words[0] == 0 and words[1] == H * sum((a + 127) // 128 for a, t in zip(lens_q, takes) if t)
        assert words[2] == sum((b + 127) // 128 * 128 for b, t in zip(lens_k, takes) if t)
        for b, t in enumerate(takes):
            rows = slice(cu[b], cu[b + 1])
            assert torch.equal(out[rows], whole[rows]) if t else bool((out[rows] == 7.0).all()), (route, b, t)
        if words[1] == 0:                                  # nothing quantized, V's maxima only cleared
            assert all(bool((x == 0x5A).all()) for x in bufs[:5])


def test_maximum_lengths_that_are_upper_bounds(dev, monkeypatch):
    """A model's maximum lengths over short sequences: the result is the per-sequence route's, and the offsets are read
    once."""
    g = torch.Generator(device=dev).manual_seed(1)
    ends = torch.tensor([0, 1100, 2000, 3200], dtype=torch.int32, device=dev)
    q, k, v = (torch.randn(3200, 8, 64, generator=g, device=dev).to(torch.bfloat16) for _ in range(3))
    want = torch.cat([cdna4_sage.sageattn(*(t[a:b].unsqueeze(0) for t in (q, k, v)), tensor_layout="NHD")[0]
                      for a, b in ((0, 1100), (1100, 2000), (2000, 3200))])
    reads, sequences = [], core._sequences
    monkeypatch.setattr(core, "_sequences", lambda *a: reads.append(1) or sequences(*a))
    for bound in (40960, 3000):                            # past the totals, and one that a sequence might have
        assert cdna4_sage.MIN_WORK <= 8 * 3000 * 3000
        assert torch.equal(sageattention.sageattn_varlen(q, k, v, ends, ends, bound, bound), want)
        assert len(reads) == 1
        reads.clear()
