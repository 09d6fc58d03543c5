"""The native host path of the operators around the recurrence (linear layers, cell prologue, state blocks,
replicas, tensor map, weight-update chain): operands in other strides and alignments give what their canonical
copies give, saved-tensor hooks see what the nodes keep, and functorch transforms and forward mode are refused."""

import pytest
import torch
import torch.autograd.forward_ad as fwd_ad

import atlas_rnn_amd as am
from atlas_rnn_amd import functional as F
from atlas_rnn_amd.omega import omega_store_chain

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _strided(x):
    """x's values in another memory order (the last two axes swapped)."""
    return x.transpose(-1, -2).contiguous().transpose(-1, -2) if x.dim() > 1 else torch.stack([x, x], dim=1)[:, 0]


def _misaligned(x):
    flat = torch.empty(x.numel() + 1, device=x.device, dtype=x.dtype)
    flat[1:] = x.reshape(-1)
    return flat[1:].view(x.shape)


def _operator(name):
    """(f, its tensors): f takes them in that order and returns a list of tensors."""
    g = torch.Generator(device="cuda").manual_seed(len(name))
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)
    if name in ("linear", "linear_f32"):
        dt = BF16 if name == "linear" else torch.float32
        return lambda x, w: [F.linear(x, w)], [r(3, 20, 24).to(dt), r(16, 24).to(dt)]
    if name == "prologue":
        p = [r(2, 20, 32), 1 + 0.1 * r(32), *[r(32, 1, 4) for _ in range(3)], *[r(32, 32) / 6 for _ in range(3)],
             *[r(2, 32) / 6 for _ in range(3)], *[r(2) for _ in range(3)], 1 + 0.1 * r(2, 1, 16), 1 + 0.1 * r(2, 1, 16)]

        def f(x, norm, c0, c1, c2, p0, p1, p2, g0, g1, g2, b0, b1, b2, qg, kg):
            xn, q, k, v, gates = F.cell_prologue(x, norm, 1e-6, [c0, c1, c2], [p0, p1, p2], [g0, g1, g2], [b0, b1, b2], qg,
                                                 kg, 2, 16)
            return [xn, q, k, v, *gates]

        return f, [t.to(BF16) for t in p]
    if name == "blocks":
        u = lambda: torch.rand(2, 19, device="cuda", generator=g).to(BF16)

        def f(k, q, v, lr, decay, beta, gate, S_ref, S0, Z0, buffer):
            return list(am.memory_recurrence(k, q, v, lr, decay, beta, gate, S_ref, S0, Z0, buffer, window=3))

        k, q = ((r(2, 19, 128) / 12).to(BF16) for _ in range(2))
        return f, [k, q, r(2, 19, 64).to(BF16), u(), u(), u(), u(), *[0.1 * r(2, 64, 128) for _ in range(3)],
                   0.1 * r(2, 2, 64, 128)]
    if name == "replicas":
        return lambda a, b: [*F._ReplicateFn.apply(3, a, b), *F._ReplicaSumFn.apply(2, a, b)], [r(4, 5), r(2, 3, 7).to(BF16)]
    if name == "map":
        proj = (r(32 + 32 * 32, 48) / 32).to(BF16)
        return lambda x: [F.tensor_feature_map(x, proj, 3)], [(r(50, 32) / 6).to(BF16)]
    assert name == "chain"

    def f(s, decay, last, am_, lm, gate, buf):
        return list(omega_store_chain(s, decay, last, adaptive_momentum=am_, last_momentum=lm, omega_gate=gate,
                                      omega_window=3, omega_buf=buf))

    u = lambda *s: torch.rand(*s, device="cuda", generator=g)
    return f, [r(3, 9, 6, 4), u(3, 9), r(3, 6, 4), u(2, 3, 9), r(2, 3, 6, 4), u(3, 9), r(3, 2, 6, 4)]


OPERATORS = ["linear", "linear_f32", "prologue", "blocks", "replicas", "map", "chain"]


def _grads(outs, leaves):
    loss = sum((o.float() * torch.linspace(-1, 1, o.numel(), device="cuda").view(o.shape)).sum() for o in outs)
    return torch.autograd.grad(loss, leaves)


@pytest.mark.parametrize("name", OPERATORS)
def test_forms_of_the_operands(name):
    print("forms", name, flush=True)
    f, x = _operator(name)

    def run(form):
        leaves = [t.clone().requires_grad_() for t in x]
        # (the prologue's norm weight is the one operand that has to be aligned)
        outs = f(*[form(t) if (name, i, form) != ("prologue", 1, _misaligned) else t for i, t in enumerate(leaves)])
        return [o.detach() for o in outs], _grads(outs, leaves)

    want = run(lambda t: t)
    # torch's fp32 products may take another order of their sums for other strides
    same = torch.equal if name != "linear_f32" else lambda a, b: torch.allclose(a, b, rtol=1e-5, atol=1e-4)
    for form in (_strided, _misaligned):
        got = run(form)
        torch.cuda.synchronize()
        for a, b in zip((*want[0], *want[1]), (*got[0], *got[1])):
            assert a.shape == b.shape and same(a, b), form.__name__


@pytest.mark.parametrize("name", OPERATORS)
def test_saved_tensor_hooks(name):
    f, x = _operator(name)
    leaves = [t.clone().requires_grad_() for t in x]
    want = _grads(f(*leaves), leaves)
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.cpu(), lambda t: t.cuda()):
        outs = f(*leaves)
    got = _grads(outs, leaves)
    torch.cuda.synchronize()
    assert bool(packed) == (name != "replicas")   # (the replicas' node keeps a number)
    assert all(torch.equal(a, b) for a, b in zip(want, got))


@pytest.mark.parametrize("name", OPERATORS)
def test_transforms_are_refused(name):
    f, x = _operator(name)
    first = lambda t: f(t, *x[1:])[0]
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda t: first(t).float().sum())(x[0])
    with pytest.raises(RuntimeError):
        torch.vmap(first)(torch.stack([x[0], x[0]]))
    with fwd_ad.dual_level(), pytest.raises(RuntimeError):
        first(fwd_ad.make_dual(x[0], torch.ones_like(x[0])))


def test_a_misaligned_norm_weight_is_refused():
    f, x = _operator("prologue")
    with pytest.raises(RuntimeError, match="aligned"):
        f(x[0], _misaligned(x[1]), *x[2:])
