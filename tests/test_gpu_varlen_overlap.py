"""sageattn_varlen with the offsets on the GPU queues the packed pass before it reads them and runs the torch SDPA sequences
on a side stream.  Offsets on the CPU take the plain order (read, pass, sequences one by one): the results must be the same
bits, with offsets and inputs still being produced on the caller's stream, from any stream, and when the caller's maximum
lengths promise a kernel sequence that the offsets do not hold."""
import pytest
import torch

import cdna4_sage
import sageattention

pytestmark = pytest.mark.gpu


def _batch(dev, lens, H, D, dt, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    q, k, v = (torch.randn(sum(lens), H, D, generator=g, device=dev).to(dt) for _ in range(3))
    ends = [0]
    for n in lens:
        ends.append(ends[-1] + n)
    return q, k, v, torch.tensor(ends, dtype=torch.int32)


@pytest.mark.parametrize("lens,H,D,causal,claim", [
    ([3000, 500, 2900, 64, 1], 8, 128, False, None),      # both routes
    ([3000, 500, 4200], 8, 64, True, None),               # the first is too small for the kernel when causal
    ([3000, 2900], 8, 128, False, None),                  # the kernel alone
    ([1100, 900, 1200], 8, 64, False, (5000, 5000)),      # no kernel sequence, maximum lengths that promise one
    ([1100, 900, 1200], 8, 64, False, None),              # no kernel sequence, by the maximum lengths
])
def test_offsets_on_the_gpu_give_the_same_bits(dev, lens, H, D, causal, claim):
    mq, mk = claim or (max(lens), max(lens))
    stream = torch.cuda.Stream(device=dev)
    for seed in range(3):
        q, k, v, ends = _batch(dev, lens, H, D, torch.bfloat16, seed)
        want = sageattention.sageattn_varlen(q, k, v, ends, ends, mq, mk, is_causal=causal)
        torch.cuda.synchronize(dev)
        for s in (torch.cuda.current_stream(dev), stream):
            with torch.cuda.stream(s):
                # inputs and offsets written late on the caller's stream, from memory the allocator hands out again
                cu = torch.zeros(len(ends), dtype=torch.int32, device=dev)
                late = [torch.full_like(t, float("nan")) for t in (q, k, v)]
                torch.cuda._sleep(20_000_000)
                for a, b in zip(late, (q, k, v)):
                    a.copy_(b)
                cu.copy_(ends.to(dev))
                got = sageattention.sageattn_varlen(*late, cu, cu, mq, mk, is_causal=causal)
                del late, cu
                churn = [torch.full_like(q, float("nan")) for _ in range(4)]
                same = torch.equal(got, want)
                del churn
            assert same, (seed, s)


def test_lengths_that_are_not_plain_numbers(dev):
    """Maximum query lengths on the GPU, or none: never read back, so the call can be captured, and the results are those
    of plain numbers."""
    q, k, v, ends = _batch(dev, [3000, 500, 2900], 8, 128, torch.bfloat16, 7)
    cu = ends.to(dev)
    on_gpu = torch.tensor(3000, device=dev)
    want = sageattention.sageattn_varlen(q, k, v, ends, ends, 3000, 3000)
    for mq in (on_gpu, None, 1):
        assert torch.equal(sageattention.sageattn_varlen(q, k, v, cu, cu, mq, 3000), want)
    packed = cdna4_sage.attention_varlen(q, k, v, cu, cu)
    torch.cuda.synchronize(dev)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = sageattention.sageattn_varlen(q, k, v, cu, cu, on_gpu, 3000)
    for _ in range(3):
        noise = torch.randn(1 << 20, device=dev)
        out.zero_()
        graph.replay()
        torch.cuda.synchronize(dev)
        assert torch.equal(out, packed) and torch.isfinite(noise).all()
