"""torch.jit.trace of the operators: a trace computes what the eager call computes, on inputs other than the
traced ones, with its gradients. (A trace that looked into a native call would hold the allocation of its
outputs and nothing that fills them.)"""

import warnings

import pytest
import torch

import atlas_rnn_amd as am
from atlas_rnn_amd import _lib
from atlas_rnn_amd import functional as F
from atlas_rnn_amd.omega import omega_store_chain

BF16 = torch.bfloat16


def _check(f, x):
    """f traced on x without and with a gradient, run on another input of that shape."""
    other = x * 0.5 + 0.1
    for grad in (False, True):
        with warnings.catch_warnings():
            warnings.simplefilter("ignore")   # sizes of the traced inputs become constants
            traced = torch.jit.trace(f, (x.clone().requires_grad_(grad),))
        a, b = (other.clone().requires_grad_(grad) for _ in range(2))
        got, want = traced(a), f(b)
        assert torch.equal(got, want)
        if grad:
            g = torch.ones_like(want)
            assert torch.equal(torch.autograd.grad(got, [a], g)[0], torch.autograd.grad(want, [b], g)[0])


def test_trace_on_the_cpu():
    w = torch.randn(4, 6)
    _check(lambda x: F.linear(x, w), torch.randn(5, 6))


def test_native_entries_refuse_to_be_traced():
    x, w = torch.randn(5, 6), torch.randn(4, 6)
    host = _lib.native()
    with pytest.raises(RuntimeError, match="not traced"):
        torch.jit.trace(lambda x: host.linear(x, w), (x,))


def _recurrence(t, d):
    g = torch.Generator(device="cuda").manual_seed(t + d)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)
    u = lambda: torch.rand(2, t, device="cuda", generator=g).to(BF16)
    kw = dict(q=r(2, t, d).to(BF16), v=r(2, t, d).to(BF16), lr=0.1 * u(), decay=u(), beta=u())
    return lambda k: torch.cat([x.flatten().float() for x in am.memory_recurrence(k, **kw, window=3) if x is not None]), \
        (r(2, t, d) * d ** -0.5).to(BF16)


def _operator(name):
    g = torch.Generator(device="cuda").manual_seed(7)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)
    if name.startswith("recurrence"):
        return _recurrence(*map(int, name.split("_")[1:]))
    if name == "linear":
        w = r(16, 64).to(BF16)
        return lambda x: F.linear(x, w), r(9, 64).to(BF16)
    if name == "map":
        proj = (r(64 + 64 * 64, 64) / 64).to(BF16)
        return lambda x: F.tensor_feature_map(x, proj), r(9, 64).to(BF16)
    if name == "chain":
        kw = dict(adaptive_momentum=r(1, 2, 5).sigmoid(), last_momentum=r(1, 2, 8), omega_gate=r(2, 5).sigmoid(),
                  omega_buf=r(2, 2, 8))
        decay, last = r(2, 5).sigmoid(), r(2, 8)
        return lambda s: torch.cat([o.flatten() for o in omega_store_chain(s, decay, last, omega_window=3, **kw)]), r(2, 5, 8)
    assert name == "prologue"
    p = dict(norm=r(64), convs=[r(64, 1, 4) for _ in range(3)], projs=[r(64, 64) / 8 for _ in range(3)],
             gw=[r(2, 64) for _ in range(3)], gb=[r(2) for _ in range(3)])

    def f(x):
        xn, q, k, v, gates = F.cell_prologue(x, p["norm"], 1e-6, p["convs"], p["projs"], p["gw"], p["gb"], None, None, 2, 32)
        return torch.cat([t.flatten() for t in (xn, q, k, v, *gates)])

    return f, r(2, 10, 64)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["recurrence_8_64", "recurrence_1_64", "recurrence_8_128", "recurrence_8_24", "linear",
                                  "map", "chain", "prologue"])
def test_trace(name):
    print("trace", name, flush=True)
    _check(*_operator(name))
