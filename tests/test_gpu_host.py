"""The native host path (csrc/host.cpp): operands in other strides, types and alignments give what their
canonical copies give, and the autograd nodes keep what a Python autograd function keeps - saved-tensor
hooks, in-place version checks, gradients only where asked - and refuse functorch transforms and
forward-mode differentiation."""

import pytest
import torch
import torch.autograd.forward_ad as fwd_ad

import atlas_rnn_amd as am
from atlas_rnn_amd import functional as F

pytestmark = pytest.mark.gpu
BH, T, D, E = 3, 70, 64, 4
BF16 = torch.bfloat16


def _ops(dt=BF16, t=T, seed=0):
    g = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g)
    k = r(BH, t, D)
    x = dict(k=k / k.norm(dim=-1, keepdim=True), q=r(BH, t, D), v=r(BH, t, D), lr=0.1 * torch.sigmoid(r(BH, t)),
             decay=torch.sigmoid(r(BH, t) + 2), beta=torch.sigmoid(r(BH, t)), gate=torch.softmax(r(BH, t, E), -1))
    x = {n: v.to("cuda", dt) for n, v in x.items()}
    for n in ("S_ref", "S0", "Z0"):
        x[n] = (0.1 * r(BH, D, D)).cuda()
    x["buffer"] = (0.1 * r(BH, E - 1, D, D)).cuda()
    return x


def _misaligned(x):
    flat = torch.empty(x.numel() + 1, device=x.device, dtype=x.dtype)
    flat[1:] = x.reshape(-1)
    return flat[1:].view(x.shape)


@pytest.mark.parametrize("t", [T, 1])
def test_forms_of_the_operands(t):
    print("forms", t, flush=True)
    x = _ops(t=t)
    want = am.memory_recurrence(**x, window=E)
    forms = dict(
        strides={n: v.transpose(0, 1).contiguous().transpose(0, 1) for n, v in x.items()},
        misaligned={n: _misaligned(v) for n, v in x.items()},
        wider={n: (v.float() if n not in ("k",) else v) for n, v in x.items()},
        states={n: (v.double() if n in ("S_ref", "S0", "Z0", "buffer") else v) for n, v in x.items()})
    for name, f in forms.items():
        got = am.memory_recurrence(**f, window=E)
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want)), name


def test_refusals_stay():
    x = _ops(t=8)
    call = lambda k, **kw: am.memory_recurrence(**{**x, "k": k, **kw}, window=E)[0]
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda k: call(k).float().sum())(x["k"])
    with pytest.raises(RuntimeError):
        torch.vmap(call)(torch.stack([x["k"], x["k"]]))
    with fwd_ad.dual_level(), pytest.raises(RuntimeError):
        call(fwd_ad.make_dual(x["k"], torch.ones_like(x["k"])))
    for bad, kw in ((ValueError, dict(lr=x["lr"][:, :4])), (ValueError, dict(gate=x["gate"][..., :2])),
                    (RuntimeError, dict(S0=x["S0"].cpu())), (RuntimeError, dict(q=x["q"].cpu()))):
        with pytest.raises(bad):
            call(x["k"], **kw)
    with pytest.raises(RuntimeError, match="status"):
        am.memory_recurrence(x["k"], x["q"], x["v"], x["lr"], x["decay"], window=34)


@pytest.mark.parametrize("name", ["k", "beta", "S0", "buffer"])
def test_one_token_refuses_transforms_too(name):
    x = _ops(t=1)
    call = lambda t: am.memory_recurrence(**{**x, name: t}, window=E)[0]
    with fwd_ad.dual_level(), pytest.raises(RuntimeError):
        call(fwd_ad.make_dual(x[name], torch.ones_like(x[name])))
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda t: call(t).float().sum())(x[name])
    with pytest.raises(RuntimeError):
        torch.vmap(call)(torch.stack([x[name], x[name]]))


def test_hooks_versions_and_partial_gradients():
    x = _ops(seed=1)
    packed = []
    k = x["k"].clone().requires_grad_()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t) or t.cpu(), lambda t: t.cuda()):
        y, S, _, _ = am.memory_recurrence(**{**x, "k": k}, window=E)
    g = torch.randn_like(y)
    (a,) = torch.autograd.grad(y, [k], g, retain_graph=True)
    assert packed
    y2, S2, _, _ = am.memory_recurrence(**{**x, "k": k}, window=E)
    (b,) = torch.autograd.grad(y2, [k], g, retain_graph=True)
    assert torch.equal(a, b)
    # only the final state's gradient, and only for one of the inputs
    lr = x["lr"].clone().requires_grad_()
    S3 = am.memory_recurrence(**{**x, "lr": lr}, window=E)[1]
    (c,) = torch.autograd.grad(S3.sum(), [lr])
    assert c.shape == lr.shape and torch.isfinite(c).all()
    with torch.no_grad():
        k.mul_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace"):
        torch.autograd.grad(y2, [k], g)
    w = torch.randn(16, D, device="cuda").to(BF16).requires_grad_()
    z = F.linear(x["q"], w)
    (dw,) = torch.autograd.grad(z.float().sum(), [w])
    torch.cuda.synchronize()
    assert dw.shape == w.shape


def test_side_stream_uses_its_own_stream():
    x = _ops(seed=2)
    want = am.memory_recurrence(**x, window=E)[0]
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        big = torch.zeros(1 << 26, device="cuda")
        for _ in range(20):
            big.add_(1.0)          # the stream is busy when the operands are made on it
        k = x["k"] + (big[:1] - 20.0).to(BF16)
        got = am.memory_recurrence(**{**x, "k": k}, window=E)[0]
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    assert torch.equal(got, want)


@pytest.mark.parametrize("clamp", [None, 16])
def test_recurrence_function_on_canonical_operands(clamp):
    x = _ops(seed=3)
    cfg = F.RecurrenceConfig(window=E, clamp_every=clamp, clamp_final=False)
    names = ("k", "q", "v", "lr", "decay", "beta", "gate", "S_ref", "S0", "Z0", "buffer")
    grads, outs = [], []
    for call in (lambda o: F.MemoryRecurrenceFn.apply(*o, cfg),
                 lambda o: am.memory_recurrence(*o, window=E, clamp_every=clamp, clamp_final=False)):
        o = [x[n].clone().requires_grad_() for n in names]
        out = call(o)
        outs.append(out)
        grads.append(torch.autograd.grad(sum(t.float().square().sum() for t in out), o))
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(*outs))
    for a, b in zip(*grads):   # (the clamped plan's scalar gradients add in any order: a bf16 rounding apart)
        a, b = a.float(), b.float()
        assert torch.equal(a, b) if clamp is None else (a - b).abs().max() <= 2 ** -7 * b.abs().max()
    y, S, Z, B = F.MemoryRecurrenceFn.apply(*[x[n] for n in names[:5]], None, None, x["S_ref"], x["S0"], None, None,
                                            F.RecurrenceConfig(window=1))
    assert y.shape == x["v"].shape and S.shape == x["S0"].shape and Z.numel() == 0 and B.numel() == 0
    with pytest.raises(RuntimeError, match="status"):   # a buffer without a window
        F.MemoryRecurrenceFn.apply(*[x[n] for n in names[:5]], None, None, x["S_ref"], x["S0"], None, x["buffer"],
                                   F.RecurrenceConfig(window=1))


def test_the_cell_runs_its_merge_heads_module():
    cell = am.OmegaRNNMemoryCell(dim=32, dim_head=32, heads=2, omega_window=2).cuda()
    seen = []
    cell.merge_heads.register_forward_hook(lambda m, args, out: seen.append((args[0].shape, out.shape)) or 2 * out)
    x = torch.randn(3, 5, 32, device="cuda")
    doubled = cell(x)[0]
    assert seen == [((3, 2, 5, 32), (3, 5, 64))]
    cell.merge_heads._forward_hooks.clear()
    assert torch.allclose(doubled, 2 * cell(x)[0])


def test_clamp_final_is_a_truth_value():
    x = _ops(t=8)
    for bad, error in ((None, TypeError), ("yes", ValueError), (2, RuntimeError)):
        with pytest.raises(error):
            am.memory_recurrence(**x, window=E, clamp_final=bad)
    assert torch.equal(am.memory_recurrence(**x, window=E, clamp_final=1)[1], am.memory_recurrence(**x, window=E)[1])
