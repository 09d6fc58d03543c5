"""scan_chunk_len values whose chunks cannot be halved on a group of eight tokens (100 in bf16 gives chunks of 25):
outputs and gradients against the fp64 oracle with the suite's tolerances, and the same results without a
backward."""

import pytest
import torch

from _cases import TENSOR_INPUTS, Case, compare, make_inputs, run_gpu, run_oracle, tol_for

import atlas_rnn_amd as am

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16

CASES = [
    Case("bf16_clamp100", BH=2, T=307, d=64, e=4, gate='lag', buffer=True, clamp_every=100, states=0.1, dtype=BF16, seed=601),
    Case("bf16_clamp40", BH=3, T=163, d=64, e=2, gate='token', clamp_every=40, states=0.1, dtype=BF16, seed=602),
    Case("bf16_clamp50_fires", BH=2, T=151, d=64, e=4, gate='token', clamp_every=50, states=150.0, dtype=BF16, seed=603),
    Case("bf16_d32_clamp300", BH=2, T=301, d=32, e=16, gate='token', buffer=True, clamp_every=300, states=0.1, dtype=BF16,
         seed=604),
    Case("f32_clamp48", BH=2, T=100, d=64, e=4, gate='lag', buffer=True, clamp_every=48, states=0.1, seed=605),
    Case("f32_clamp20_fires", BH=2, T=61, d=64, e=2, gate='token', clamp_every=20, states=150.0, seed=606),
    Case("f32_d32_clamp120_nomom", BH=2, T=245, d=32, e=8, momentum=False, gate='token', clamp_every=120, states=0.1, seed=607),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: c.name)
def test_clamp_chunks(case):
    print("clamp chunks", case.name, flush=True)
    p = make_inputs(case)
    ref, gref = run_oracle(case, p)
    out, g = run_gpu(case, p)
    tol = tol_for(case)
    for nm, a, b in zip(("y", "S_T", "Z_T", "buffer"), out, ref):
        if b is not None:
            compare(f"{case.name}.{nm}", a, b, tol)
    for kk, b in gref.items():
        compare(f"{case.name}.d{kk}", g[kk], b, tol)
    x = {n: None if p[n] is None else p[n].to("cuda", case.dtype if n not in ("S_ref", "S0", "Z0", "buffer") else torch.float32)
         for n in TENSOR_INPUTS}
    with torch.no_grad():
        same = am.memory_recurrence(**x, window=case.e, clamp_every=case.clamp_every, clamp_final=case.clamp_final)
    for a, b in zip(same, out):
        if b is not None:
            assert torch.equal(a.float().cpu(), b.float().cpu())
