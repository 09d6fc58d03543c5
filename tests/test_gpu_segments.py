"""Row counts that do not divide the CU count: the segment split of the rows (fewer, longer segments or a
pair of workgroups per CU) against the fp64 oracle on a few rows, which are independent of the others."""

import pytest
import torch

from _cases import Case, compare, make_inputs, run_gpu, run_oracle_rows, tol_for

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16

CASES = [
    Case("bf16_96", BH=96, T=330, d=64, e=4, gate='token', states=0.1, dtype=BF16, seed=501),
    Case("bf16_160_buffer", BH=160, T=200, d=64, e=3, gate='lag', buffer=True, states=0.1, dtype=BF16, seed=502),
    Case("bf16_12_clamp", BH=12, T=1500, d=64, e=2, gate='token', clamp_every=64, states=0.1, dtype=BF16, seed=503),
    Case("bf16_d32_24", BH=24, T=900, d=32, e=4, gate='token', buffer=True, states=0.1, dtype=BF16, seed=504),
    Case("f32_24", BH=24, T=700, d=64, e=4, gate='lag', buffer=True, states=0.1, seed=505),
    Case("f32_d32_200", BH=200, T=90, d=32, e=2, states=0.1, seed=506),
]


@pytest.mark.parametrize("case", CASES, ids=[c.name for c in CASES])
def test_rows_that_do_not_divide_the_card(case):
    print("segments:", case.name, flush=True)
    p = make_inputs(case)
    rows = [0, case.BH // 2, case.BH - 1]
    block = 256 if case.clamp_every is None else 256 // case.clamp_every * case.clamp_every
    ref_out, ref_grads = run_oracle_rows(case, p, rows, block=block)
    got_out, got_grads = run_gpu(case, p)
    tol = tol_for(case)
    for n, g, r in zip(("y", "S_T", "Z_T", "buffer_out"), got_out, ref_out):
        if r is not None:
            compare(f"{case.name}.{n}", g[rows], r, tol)
    for n, r in ref_grads.items():
        compare(f"{case.name}.d{n}", got_grads[n][rows], r, tol)
