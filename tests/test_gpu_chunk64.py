"""The kernels of chunk 64 at head dim 128 (two workgroups per CU, D x D states staged in halves),
forward and backward with the norm, on unit counts at and around the two workgroups per CU of the
grid (32 units a row: 1, 16 and 17 rows), ragged lengths and segment cuts.

- Rows are independent: each row of a batch equals the row run alone, outputs and per-token
  gradients bit for bit.
- One row against the oracle's fp64 chunked rule: relative L2 1e-4 at "high" (three bf16 passes: terms of
  2^-16 dropped from each product), 1e-5 at "highest" (whose kernels keep one workgroup per CU)."""

from __future__ import annotations

import pytest
import torch

from gdn_cases import hip_outputs, oracle_outputs, rel_l2

pytestmark = pytest.mark.gpu

SHAPE = dict(key_heads=1, key_dim=128, value_heads=2, value_dim=128)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,length,precision", [(1, 1024, "high"), (16, 1024, "high"), (17, 1021, "high"), (17, 1024, "mixed"),
                                                   (3, 961, "bf16")])
def test_rows_of_a_batch_equal_the_rows_alone(rows, length, precision, dtype):
    from tjev_amd import gdn_megakernel_normed
    from tjev_amd.testing import gdn_inputs

    qkv, a, b, a_log, dt_bias, w, seg = (x.cuda() for x in gdn_inputs(
        batch=rows, length=length, key_heads=1, value_heads=2, dim=128, dtype=dtype, seed=length, segments="random4"))
    gen = torch.Generator(device="cuda").manual_seed(1)
    z, dy = (torch.randn(rows, length, 2, 128, generator=gen, device="cuda").to(dtype) for _ in range(2))
    print(f"chunk 64 rows={rows} T={length} {precision} {dtype}", flush=True)

    def run(i):
        lv = [x[i].clone().requires_grad_(True) for x in (qkv, a, b, z)]
        y = gdn_megakernel_normed(lv[0], lv[1], lv[2], a_log, dt_bias, w, seg[i], lv[3], torch.ones(128, device="cuda"),
                                  chunk=64, precision=precision, **SHAPE)
        return [y.detach(), *torch.autograd.grad(y, lv, dy[i])]

    whole = run(slice(None))
    assert all(bool(torch.isfinite(x.float()).all()) for x in whole)
    for i in sorted({0, rows // 2, rows - 1}):
        for x, y in zip(whole, run(slice(i, i + 1))):
            assert torch.equal(x[i:i + 1], y)


@pytest.mark.parametrize("precision,tol", [("highest", 1e-5), ("high", 1e-4)])
@pytest.mark.parametrize("length,cuts", [(64, [20]), (65, [64]), (200, [63, 130])])
def test_matches_the_oracle(precision, tol, length, cuts):
    from gdn_cases import case_inputs

    inputs, cot = case_inputs(1, length, 1, 2, 128, cuts=cuts, trailing_pad=3)
    got = hip_outputs(inputs, cot, chunk=64, precision=precision, **SHAPE)
    want = oracle_outputs(inputs, cot, dtype=torch.float64, **SHAPE)
    errs = {n: rel_l2(got[n], want[n]) for n in got}
    print(f"chunk 64 T={length} {precision}: {({n: f'{e:.1e}' for n, e in errs.items()})}", flush=True)
    # the gate parameters' gradients are sums over all tokens whose terms cancel: 5 times the bar
    assert all(e <= tol * (5 if n in ("A_log", "dt_bias") else 1) for n, e in errs.items()), errs
