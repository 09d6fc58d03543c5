"""The general segment kernels (fp32, and bf16 with heads of 32 or windows past 17) at the edges of their
source tiles: windows on both sides of the 16-slot halo, one token, chunk remainders, clamp chunks that
are not whole tiles. Outputs and gradients against the fp64 oracle with the suite's tolerances."""

import pytest
import torch

from _cases import Case, compare, make_inputs, run_gpu, run_oracle, tol_for

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16

CASES = [
    Case("f32_e17", BH=2, T=95, d=64, e=17, gate='lag', buffer=True, states=0.1, seed=401),
    Case("f32_e16_T17", BH=3, T=17, d=64, e=16, gate='token', buffer=True, states=0.1, seed=402),
    Case("f32_e1_T33", BH=2, T=33, d=64, e=1, states=0.1, seed=403),
    Case("f32_d32_e17_nomom", BH=2, T=65, d=32, e=17, gate='token', momentum=False, buffer=True, states=0.1, seed=404),
    Case("f32_clamp16", BH=2, T=100, d=64, e=4, gate='token', clamp_every=16, states=0.1, seed=405),
    Case("bf16_d32_e17", BH=3, T=130, d=32, e=17, gate='lag', buffer=True, states=0.1, dtype=BF16, seed=406),
    Case("bf16_d32_e18", BH=3, T=130, d=32, e=18, gate='lag', buffer=True, states=0.1, dtype=BF16, seed=407),
    Case("bf16_d32_T1", BH=2, T=1, d=32, e=4, gate='token', buffer=True, states=0.1, dtype=BF16, seed=408),
    Case("bf16_d64_e18_multiseg", BH=40, T=300, d=64, e=18, gate='token', states=0.1, dtype=BF16, seed=409),
    Case("bf16_d32_clamp24", BH=2, T=100, d=32, e=4, gate='token', clamp_every=24, states=0.1, dtype=BF16, seed=410),
]


@pytest.mark.parametrize("case", CASES, ids=[c.name for c in CASES])
def test_halo_edges(case):
    print("general halo:", case.name, flush=True)
    p = make_inputs(case)
    ref_out, ref_grads = run_oracle(case, p)
    got_out, got_grads = run_gpu(case, p)
    tol = tol_for(case)
    for n, g, r in zip(("y", "S_T", "Z_T", "buffer_out"), got_out, ref_out):
        if r is not None:
            compare(f"{case.name}.{n}", g, r, tol)
    for n, r in ref_grads.items():
        compare(f"{case.name}.d{n}", got_grads[n], r, tol)
