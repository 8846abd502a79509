"""The kernels of chunk 16 at head dim 128 (one wave per workgroup, D x D states staged in halves), forward and
backward, on whole and partly filled chunks with segment cuts, against the oracle's fp64 chunked rule:
relative L2 1e-5 at "highest" (fp32 sums), 1e-4 at "high" (three bf16 passes: terms of 2^-16 dropped from each
product) and 2e-2 at "mixed" and "bf16" (one bf16 pass on the state path: operands rounded by 2^-9)."""

from __future__ import annotations

import pytest
import torch

from gdn_cases import case_inputs, hip_outputs, oracle_outputs, rel_l2

pytestmark = pytest.mark.gpu

SHAPE = dict(key_heads=1, key_dim=128, value_heads=2, value_dim=128)
TOL = {"highest": 1e-5, "high": 1e-4, "mixed": 2e-2, "bf16": 2e-2}


@pytest.mark.parametrize("residuals", ["states", "tinv"])
@pytest.mark.parametrize("precision", list(TOL))
@pytest.mark.parametrize("length,cuts", [(16, [5]), (17, [16]), (83, [15, 40])])
def test_matches_the_oracle(length, cuts, precision, residuals):
    inputs, cot = case_inputs(1, length, 1, 2, 128, cuts=cuts, trailing_pad=2)
    print(f"chunk 16 T={length} {precision} {residuals}", flush=True)
    got = hip_outputs(inputs, cot, chunk=16, precision=precision, residuals=residuals, **SHAPE)
    want = oracle_outputs(inputs, cot, dtype=torch.float64, **SHAPE)
    errs = {n: rel_l2(got[n], want[n]) for n in got}
    print({n: f"{e:.1e}" for n, e in errs.items()}, flush=True)
    # the gate parameters' gradients are sums over all tokens whose terms cancel: 5 times the bar
    assert all(e <= TOL[precision] * (5 if n in ("A_log", "dt_bias") else 1) for n, e in errs.items()), errs
