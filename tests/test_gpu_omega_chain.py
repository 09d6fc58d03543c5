"""The fused Omega weight-update chain (csrc/chain.hip) at the sizes where its waves, load groups and
window registers end, against oracle/omega.py in float64: outputs and the gradient of every input.

Bounds: fp32 sums of at most a few hundred terms, 1e-5; bf16 2e-2 (inputs, updates and momenta are
stored in bf16, relative rounding 2^-9 each)."""

import pytest
import torch

from _cases import compare
from atlas_rnn_amd.omega import _fused_chain, omega_store_chain
from oracle.omega import omega_store_chain as oracle_chain
from test_gpu_omega import _inputs

pytestmark = pytest.mark.gpu
F64 = torch.float64
BF16 = torch.bfloat16

CASES = [
    # BH, n, param shape, momentum order, gate, window, carried buffer, dtype
    (1, 1, (1,), 0, False, 1, False, torch.float32),      # one step, one column
    (3, 7, (63,), 1, True, 2, True, torch.float32),       # a short load group, one column per lane, a part wave
    (2, 8, (65,), 2, True, 4, True, torch.float32),       # a whole group, a second wave with one column
    (2, 9, (128,), 1, False, 5, False, torch.float32),    # a group and one step, two columns per lane, no buffer
    (3, 17, (2, 65), 0, True, 16, True, torch.float32),   # the widest window, two waves per row
    (2, 3, (6,), 2, True, 16, True, torch.float32),       # fewer tokens than buffer slots
    (4, 40, (20, 16), 1, True, 3, True, BF16),
    (2, 11, (7, 9), 2, False, 8, True, BF16),
]


def _run(chain, x, e, weights, dev):
    out = chain(**x, omega_window=e)
    loss = sum((o.to(w.dtype) * w).sum() for o, w in zip(out, weights) if o is not None and w is not None)
    names = [k for k in sorted(x) if x[k].requires_grad]
    return out, dict(zip(names, torch.autograd.grad(loss, [x[k] for k in names], allow_unused=True)))


def _check(x, e, dt, name, drop=()):
    ref_in = {k: v.to(F64).requires_grad_() for k, v in x.items()}
    shapes = oracle_chain(**ref_in, omega_window=e)
    g = torch.Generator().manual_seed(11)
    w = [None if r is None or i in drop else torch.randn(r.shape, generator=g, dtype=F64) for i, r in enumerate(shapes)]
    ref, gr = _run(oracle_chain, ref_in, e, w, "cpu")
    got_in = {k: v.to("cuda", dt).requires_grad_() for k, v in x.items()}
    got, gd = _run(omega_store_chain, got_in, e, [None if v is None else v.to("cuda", torch.float32) for v in w], "cuda")
    torch.cuda.synchronize()
    tol = 1e-5 if dt == torch.float32 else 2e-2
    for i, (o, r) in enumerate(zip(got, ref)):
        assert (o is None) == (r is None)
        if r is not None:
            assert o.shape == r.shape
            compare(f"{name}.out{i}", o.detach().float().cpu(), r.detach(), tol)
    for k, r in gr.items():
        r = torch.zeros_like(ref_in[k]) if r is None else r
        a = torch.zeros_like(got_in[k]) if gd[k] is None else gd[k]
        compare(f"{name}.d{k}", a.float().cpu(), r, tol)


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"bh{c[0]}_n{c[1]}_p{'x'.join(map(str, c[2]))}_o{c[3]}_e{c[5]}")
def test_chain_edges(case):
    BH, n, p, O, gate, e, buf, dt = case
    print("chain", case, flush=True)
    x = _inputs(BH, n, p, O, False, gate, e, buf, seed=BH * 100 + n, dt=dt)
    _check(x, e, dt, f"chain_{BH}_{n}_{e}")


def test_chain_partial_gradients_and_strides():
    """Outputs that get no gradient, and inputs in other orders and strides than row-major."""
    x = _inputs(3, 12, (10, 6), 2, False, True, 4, True, seed=5, dt=torch.float32)
    _check(x, 4, torch.float32, "chain_no_dupdate", drop=(0, 1))
    _check(x, 4, torch.float32, "chain_only_dupdate", drop=(1, 2, 3))
    y = dict(x)
    y["surprise"] = x["surprise"].transpose(2, 3).contiguous().transpose(2, 3)
    y["adaptive_momentum"] = x["adaptive_momentum"].transpose(1, 2).contiguous().transpose(1, 2)
    a = omega_store_chain(**{k: v.cuda() for k, v in x.items()}, omega_window=4)
    b = omega_store_chain(**{k: v.cuda() for k, v in y.items()}, omega_window=4)
    torch.cuda.synchronize()
    assert all(torch.equal(p, q) for p, q in zip(a, b))


def test_chain_switched_off_keeps_momentum_and_buffer():
    """Every gate below 1e-3: no update and no gradient through it; the momentum and the buffer carry on."""
    x = _inputs(2, 9, (33,), 1, False, True, 3, True, seed=6, dt=torch.float32)
    x["omega_gate"] = torch.full_like(x["omega_gate"], 5e-4)
    ref_in = {k: v.to(F64).requires_grad_() for k, v in x.items()}
    got_in = {k: v.cuda().requires_grad_() for k, v in x.items()}
    ref, got = oracle_chain(**ref_in, omega_window=3), omega_store_chain(**got_in, omega_window=3)
    assert torch.count_nonzero(got[0]).item() == 0
    for o, r in zip(got[2:], ref[2:]):
        compare("chain_off.carried", o.detach().cpu(), r.detach(), 1e-5)
    g = torch.Generator().manual_seed(12)
    w = [torch.randn(r.shape, generator=g, dtype=F64) for r in ref]
    names = sorted(x)
    gr = torch.autograd.grad(sum((o * v).sum() for o, v in zip(ref[2:], w[2:])), [ref_in[k] for k in names], allow_unused=True)
    gd = torch.autograd.grad(sum((o * v.cuda().float()).sum() for o, v in zip(got, w)), [got_in[k] for k in names])
    torch.cuda.synchronize()
    for k, a, b in zip(names, gd, gr):
        compare(f"chain_off.d{k}", a.cpu(), torch.zeros_like(ref_in[k]) if b is None else b, 1e-5)


def test_chain_route():
    """What the fused kernels take and what stays on the separate ones."""
    x = {k: v.cuda() for k, v in _inputs(2, 5, (8,), 1, False, True, 3, True, seed=7, dt=torch.float32).items()}
    call = lambda **kw: _fused_chain(*[{**x, "window": 3, **kw}[k] for k in (
        "surprise", "decay_factor", "last_update", "adaptive_momentum", "last_momentum", "omega_gate", "window", "omega_buf")])
    assert call() is not None
    assert call(window=17, omega_buf=None) is None
    assert call(omega_gate=x["omega_gate"].double()) is None
    assert call(adaptive_momentum=x["adaptive_momentum"].expand(3, -1, -1)) is None
    assert call(surprise=x["surprise"][..., :0]) is None


@pytest.mark.parametrize("order,gate", [(0, False), (0, True), (1, True), (2, False)])
def test_chain_edits_in_place_before_the_backward(order, gate):
    """The returned tensors may be edited in place before the backward, and so may the surprises and decays (the
    surprises not where the gradient of a gate on them reads them: a version error)."""
    x = {k: v.cuda() for k, v in _inputs(2, 11, (70,), order, False, gate, 3, True, seed=8, dt=torch.float32).items()}

    def run(edit):
        leaves = {k: v.clone().requires_grad_() for k, v in x.items()}
        ins = {k: v * 1 for k, v in leaves.items()}
        out = omega_store_chain(**ins, omega_window=3)
        loss = sum((o * torch.linspace(-1, 1, o.numel(), device="cuda").view(o.shape)).sum() for o in out if o is not None)
        with torch.no_grad():
            for t in edit(ins, out):
                t.mul_(0.5)
        names = sorted(leaves)
        return torch.autograd.grad(loss, [leaves[k] for k in names])

    want = run(lambda ins, out: ())
    for edit in (lambda ins, out: (o for o in out if o is not None), lambda ins, out: (ins["decay_factor"],)):
        assert all(torch.equal(a, b) for a, b in zip(run(edit), want))
    edit = lambda ins, out: (ins["surprise"],)
    if order == 0 and gate:
        with pytest.raises(RuntimeError, match="modified by an inplace"):
            run(edit)
    else:
        assert all(torch.equal(a, b) for a, b in zip(run(edit), want))


def test_chain_without_a_gradient_of_the_gate():
    """A gate that asks for no gradient: the other gradients are those of one that does."""
    for order in (0, 1):
        x = {k: v.cuda() for k, v in _inputs(3, 9, (70,), order, False, True, 4, True, seed=9, dt=torch.float32).items()}
        grads = []
        for ask in (True, False):
            leaves = {k: v.clone().requires_grad_(ask or k != "omega_gate") for k, v in x.items()}
            out = omega_store_chain(**leaves, omega_window=4)
            names = sorted(k for k in leaves if k != "omega_gate")
            grads.append(torch.autograd.grad(sum((o * o).sum() for o in out if o is not None), [leaves[k] for k in names]))
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(*grads))


@pytest.mark.parametrize("BH,n,p,O,gate,e,dt", [
    (2, 16, (64,), 0, False, 1, torch.float32),    # whole groups of steps alone; half a wave of columns
    (1, 24, (130,), 2, True, 1, torch.float32),    # a second wave of one lane
    (3, 25, (129,), 1, False, 2, torch.float32),   # a step past the groups; one column a lane
    (2, 33, (256,), 0, True, 1, BF16),
])
def test_chain_groups_of_steps(BH, n, p, O, gate, e, dt):
    print("chain groups", BH, n, p, O, gate, e, dt, flush=True)
    _check(_inputs(BH, n, p, O, False, gate, e, e > 1, seed=n, dt=dt), e, dt, f"chain_groups_{n}")
