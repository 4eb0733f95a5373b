"""return_lse of head dims 96 and 256 where somebody else has to see it: the logsumexp kernel is launched outside torch, so
a traced, transformed or differentiated call must take the torch formula.  The kernel is stood in for by a function that
fills its result outside torch, as the launch does."""
import pytest
import torch
from torch.autograd import forward_ad
from torch.fx.experimental.proxy_tensor import make_fx

from sageattention import core


@pytest.fixture
def kernel(monkeypatch):
    calls = []

    def row_lse(q, k, layout="HND", sm_scale=None, is_causal=False):
        calls.append(q.shape)
        out = torch.empty(q.shape[:3])
        out.detach().numpy()[...] = 7.0
        return out

    monkeypatch.setattr(core, "row_lse", row_lse)
    return calls


def _qk(D, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(1, 2, 7, D, generator=g), torch.randn(1, 2, 9, D, generator=g)


def _want(q, k):
    return torch.logsumexp(q @ k.transpose(-1, -2) * q.shape[-1] ** -0.5, -1)


def _lse(q, k):
    return core._lse(q, k, "HND", False, None)


@pytest.mark.parametrize("D", [96, 256])
def test_plain_calls_take_the_kernel(kernel, D):
    q, k = _qk(D, 1)
    assert bool((_lse(q, k) == 7.0).all())
    with torch.no_grad():
        assert bool((_lse(torch.nn.Parameter(q), k) == 7.0).all())
    assert len(kernel) == 2


@pytest.mark.parametrize("D", [96, 256])
@pytest.mark.parametrize("trace", ["jit", "real", "fake", "symbolic"])
def test_traces_hold_the_formula(kernel, D, trace):
    q, k = _qk(D, 2)
    graph = torch.jit.trace(_lse, (q, k), check_trace=False) if trace == "jit" else make_fx(_lse, tracing_mode=trace)(q, k)
    q2, k2 = _qk(D, 3)
    torch.testing.assert_close(graph(q2, k2), _want(q2, k2))
    assert not kernel


@pytest.mark.parametrize("D", [96, 256])
def test_forward_mode_keeps_the_tangent(kernel, D):
    (q, k), (tq, tk) = _qk(D, 4), _qk(D, 5)
    want, wt = torch.func.jvp(_want, (q, k), (tq, tk))
    for i in range(2):  # a tangent on either input
        with forward_ad.dual_level():
            a, b = (forward_ad.make_dual(q, tq), k) if i == 0 else (q, forward_ad.make_dual(k, tk))
            got = forward_ad.unpack_dual(_lse(a, b))
        ti = torch.func.jvp(_want, (q, k), (tq, torch.zeros_like(k)) if i == 0 else (torch.zeros_like(q), tk))[1]
        torch.testing.assert_close(got.primal, want)
        torch.testing.assert_close(got.tangent, ti)
    assert not kernel


@pytest.mark.parametrize("D", [96, 256])
def test_transforms_do_not_reach_the_kernel(kernel, D):
    """Under vmap the formula raises (it writes rows of a result of its own), as it did before the kernel took these head
    dims; what matters is that no pointer of a wrapped tensor is taken."""
    q, k = _qk(D, 6)
    with pytest.raises(RuntimeError):
        torch.vmap(_lse, in_dims=(0, None))(torch.stack([q, q]), k)
    assert not kernel
