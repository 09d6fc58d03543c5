"""functional.cell_prologue's operand lists: a list that is too short or does not fit the sizes is refused
with a ValueError before anything is read past its end (no GPU needed: the checks come before the device's),
and biases in another split than the gate weights are taken."""

import pytest
import torch

from atlas_rnn_amd import _lib
from atlas_rnn_amd.functional import cell_prologue

DIM, H, D, NG = 32, 2, 16, 4


def _lists(device="cpu", dt=torch.float32):
    g = torch.Generator().manual_seed(3)
    r = lambda *s: torch.randn(*s, generator=g).to(device, dt)
    return dict(x=r(2, 9, DIM), norm=1 + 0.1 * r(DIM), convs=[r(DIM, 1, 4) for _ in range(3)],
                projs=[r(H * D, DIM) / 6 for _ in range(3)], gw=[r(H, DIM) / 6 for _ in range(NG)], gb=[r(H) for _ in range(NG)])


def _host(p):
    return _lib.native().cell_prologue(p["x"], p["norm"], 1e-6, p["convs"], p["projs"], p["gw"], p["gb"], None, None, H, D)


@pytest.mark.parametrize("name,edit", [
    ("two projections", lambda p: p.update(projs=p["projs"][:2])),
    ("no projections", lambda p: p.update(projs=[])),
    ("one convolution", lambda p: p.update(convs=p["convs"][:1])),
    ("no biases", lambda p: p.update(gb=[])),
    ("three biases", lambda p: p.update(gb=p["gb"][:3])),
    ("biases without weights", lambda p: p.update(gw=[])),
    ("half a gate", lambda p: p.update(gw=p["gw"] + [p["gw"][0][:1]], gb=p["gb"] + [p["gb"][0][:1]])),
    ("a short bias", lambda p: p["gb"].__setitem__(1, p["gb"][1][:1])),
    ("a projection of other rows", lambda p: p["projs"].__setitem__(2, p["projs"][2][:H * D - 8])),
    ("a projection of other columns", lambda p: p["projs"].__setitem__(0, p["projs"][0][:, :8])),
    ("a gate of other columns", lambda p: p["gw"].__setitem__(0, p["gw"][0][:, :8])),
    ("a short norm", lambda p: p.update(norm=p["norm"][:8])),
], ids=lambda v: v if isinstance(v, str) else "")
def test_lists_that_do_not_fit_are_refused(name, edit):
    p = _lists()
    edit(p)
    with pytest.raises(ValueError):
        _host(p)


def test_cpu_tensors_are_refused():
    with pytest.raises(RuntimeError, match="GPU"):
        _host(_lists())


@pytest.mark.gpu
def test_other_devices_are_refused():
    p = _lists("cuda")
    p["gb"][2] = p["gb"][2].cpu()
    with pytest.raises(RuntimeError, match="one device"):
        _host(p)


@pytest.mark.gpu
@pytest.mark.parametrize("split", [lambda b: [torch.cat(b)], lambda b: [torch.cat(b[:3]), b[3]],
                                   lambda b: [t.reshape(-1)[i:i + 1] for t in b for i in range(H)]],
                         ids=["one", "two", "eight"])
def test_biases_in_another_split(split):
    outs = []
    for cut in (lambda b: b, split):
        p = _lists("cuda", torch.bfloat16)
        leaves = [t.requires_grad_() for t in (p["x"], *p["gw"], *p["gb"])]
        xn, q, k, v, gates = cell_prologue(p["x"], p["norm"], 1e-6, p["convs"], p["projs"], p["gw"], cut(p["gb"]), None, None,
                                           H, D)
        assert len(gates) == NG
        loss = sum((t.float() * t.float()).sum() for t in (xn, q, k, v, *gates))
        outs.append([xn, q, k, v, *gates, *torch.autograd.grad(loss, leaves)])
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(*outs))
