"""A loss on the final state alone gives y no gradient: atlas_mem_bwd gets dy = NULL and reads it as zeros,
on the walks (with and without a carried buffer, clamped) and on the general kernels. Gradients against
the fp64 oracle with the suite's tolerances."""

import pytest
import torch

from _cases import F64, TENSOR_INPUTS, Case, compare, make_inputs, tol_for
from oracle import memory_recurrence_vectorised

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16

CASES = [
    Case("walk", BH=3, T=200, d=64, e=4, gate='lag', states=0.1, dtype=BF16, seed=301),
    Case("walk_nomom", BH=2, T=70, d=64, e=1, momentum=False, states=0.1, dtype=BF16, seed=302),
    Case("walk_buffer", BH=3, T=200, d=64, e=4, gate='token', buffer=True, states=0.1, dtype=BF16, seed=303),
    Case("walk_clamp", BH=2, T=200, d=64, e=2, gate='token', states=0.1, clamp_every=64, dtype=BF16, seed=304),
    Case("general_d32", BH=2, T=90, d=32, e=3, gate='token', buffer=True, states=0.1, dtype=BF16, seed=305),
    Case("general_fp32", BH=2, T=90, d=64, e=3, gate='lag', states=0.1, seed=306),
]


@pytest.mark.parametrize("case", CASES, ids=[c.name for c in CASES])
def test_final_state_loss(case):
    from atlas_rnn_amd.functional import memory_recurrence
    print("no dy:", case.name, flush=True)
    p = make_inputs(case)
    leaves = [n for n in TENSOR_INPUTS if p[n] is not None]

    def grads(fn, conv, **kw):
        x = {n: (conv(n, p[n]).requires_grad_() if p[n] is not None else None) for n in TENSOR_INPUTS}
        S = fn(*(x[n] for n in TENSOR_INPUTS), window=case.e, clamp_every=case.clamp_every, **kw)[1]
        gs = torch.autograd.grad((S * p["gS"].to(S.device, S.dtype)).sum(), [x[n] for n in leaves], allow_unused=True)
        return [torch.zeros_like(x[n]) if g is None else g for n, g in zip(leaves, gs)]

    ref = grads(memory_recurrence_vectorised, lambda n, t: t.to(F64).clone(), clamp_final=True)
    small = ("S_ref", "S0", "Z0", "buffer")
    got = grads(memory_recurrence, lambda n, t: t.to("cuda", torch.float32 if n in small else case.dtype).clone())
    torch.cuda.synchronize()
    for n, a, b in zip(leaves, got, ref):
        compare(f"{case.name}.d{n}", a.float().cpu(), b, tol_for(case))
