"""A forward that no backward follows leaves out what only the backward reads; its results are the training
forward's bit for bit, on every plan: the walks, a carried buffer, clamps (also where they act, the exact
sequence), fp32, heads of 32, windows past the short halo, ragged ends."""

import pytest
import torch

import atlas_rnn_amd as am

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16

CASES = [
    ("walk", dict(BH=5, T=130, d=64, e=4, dtype=BF16)),
    ("walk_gate", dict(BH=3, T=333, d=64, e=9, gate=True, dtype=BF16)),
    ("walk_buffer", dict(BH=4, T=200, d=64, e=4, buffer=True, dtype=BF16)),
    ("clamp", dict(BH=4, T=257, d=64, e=4, buffer=True, clamp=64, dtype=BF16)),
    ("clamp_acts", dict(BH=2, T=256, d=64, e=2, clamp=64, scale=2e4, dtype=BF16)),
    ("clamp_off_chunk", dict(BH=2, T=150, d=64, e=2, clamp=48, dtype=BF16)),
    ("window_33", dict(BH=3, T=120, d=64, e=33, buffer=True, dtype=BF16)),
    ("d32", dict(BH=7, T=99, d=32, e=4, gate=True, dtype=BF16)),
    ("f32", dict(BH=3, T=140, d=64, e=4, buffer=True, dtype=torch.float32)),
    ("f32_clamp", dict(BH=3, T=96, d=64, e=2, clamp=16, dtype=torch.float32)),
    ("f32_d32", dict(BH=3, T=41, d=32, e=1, dtype=torch.float32)),
]


@pytest.mark.parametrize("name,c", CASES, ids=[n for n, _ in CASES])
def test_same_results_without_a_backward(name, c):
    print("infer:", name, flush=True)
    g = torch.Generator(device="cuda").manual_seed(77)
    BH, T, d, e, dt = c["BH"], c["T"], c["d"], c["e"], c["dtype"]

    def rnd(*s, scale=1.0):
        return scale * torch.randn(*s, device="cuda", generator=g)

    k, q, v = (rnd(BH, T, d, scale=d ** -0.5).to(dt) for _ in range(3))
    v = v * c.get("scale", 1.0)
    sc = [torch.rand(BH, T, device="cuda", generator=g) for _ in range(4)]
    lr, decay, beta = (0.1 * sc[0]).to(dt), (0.05 * sc[1]).to(dt), (0.9 * sc[2]).to(dt)
    gate = sc[3].to(dt) if c.get("gate") else None
    S_ref, S0, Z0 = (rnd(BH, d, d, scale=0.1) for _ in range(3))
    buf = rnd(BH, e - 1, d, d, scale=0.1) if c.get("buffer") else None
    kw = dict(beta=beta, gate=gate, S_ref=S_ref, S0=S0, Z0=Z0, buffer=buf, window=e, clamp_every=c.get("clamp"))
    with torch.no_grad():
        a = am.memory_recurrence(k, q, v, lr, decay, **kw)
    b = am.memory_recurrence(k.clone().requires_grad_(), q, v, lr, decay, **kw)
    for n, x, y in zip(("y", "S_T", "Z_T", "buffer_out"), a, b):
        if x is None:
            assert y is None
            continue
        assert torch.equal(x, y.detach()), n
        assert not x.requires_grad
    if name == "clamp_acts":
        assert b[1].abs().max() == 100


@pytest.mark.parametrize("name,c", [
    ("walk", dict(BH=300, T=333, e=4)),                              # one segment of six chunks a row
    ("walk_buffer", dict(BH=260, T=200, e=4, buffer=True)),          # two saved states a chunk
    ("clamp", dict(BH=257, T=321, e=2, clamp=64)),                   # the same, checked at every chunk's end
    ("walk_segments", dict(BH=40, T=1500, e=9, gate=True)),          # several segments of several chunks
    ("d32", dict(BH=600, T=200, d=32, e=4)),
], ids=lambda v: v if isinstance(v, str) else "")
def test_same_results_over_several_chunks_a_segment(name, c):
    test_same_results_without_a_backward(name, {"d": 64, "dtype": BF16, **c})
