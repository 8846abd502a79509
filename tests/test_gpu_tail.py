"""The decode state a prefill leaves (k_tail), at the edges of its tiles: lengths at, before and
after a chunk's end and shorter than the conv's history, every head dim's tile split, a segment
that starts inside the last chunk or one token before the end, and a continued row. The state
against the oracle's fp64 token recurrence at the fp32 bar (max relative error 1e-5), the history
bit for bit."""

from __future__ import annotations

import pytest
import torch

from gdn_cases import rel

pytestmark = pytest.mark.gpu


def _want_history(qkv, seg, hist, k1):
    rows = torch.zeros(qkv.shape[0], k1, qkv.shape[2], dtype=qkv.dtype)
    last = qkv.shape[1] - 1
    for b in range(qkv.shape[0]):
        for r in range(k1):
            t = last - k1 + 1 + r
            if int(seg[b, max(t, 0)]) != int(seg[b, last]):
                continue
            if t >= 0:
                rows[b, r] = qkv[b, t]
            elif hist is not None:
                rows[b, r] = hist[b, k1 + t]
    return rows


@pytest.mark.parametrize("dim,chunk", [(16, 16), (32, 128), (64, 64), (128, 128), (128, 64)])
@pytest.mark.parametrize("length,cut,fresh", [(1, None, True), (2, None, False), (3, 2, True), (127, None, False),
                                              (128, 127, True), (129, 100, True), (200, 150, False)])
def test_prefill_state_at_tile_edges(dim, chunk, length, cut, fresh):
    from oracle.gdn_oracle import core_inputs, recurrent_gated_delta_rule
    from tjev_amd.serve import gdn_prefill
    from tjev_amd.testing import gdn_inputs

    shape = dict(key_heads=1, key_dim=dim, value_heads=2, value_dim=dim)
    taps = 5 if chunk == 64 else 4
    pre = 0 if fresh else 40  # a continued row: its first piece is part of the oracle's row
    inputs = gdn_inputs(batch=2, length=pre + length, key_heads=1, value_heads=2, dim=dim, taps=taps, seed=5,
                        style="reference", segments="cuts" if cut else "one", cuts=[pre + cut] if cut else None)
    qkv, a, b, a_log, dt_bias, w, seg = inputs
    dev = [x.cuda() for x in inputs]
    kw = dict(chunk=chunk, precision="highest", **shape)
    state = hist = None
    if pre:
        _, state, hist = gdn_prefill(*(x[:, :pre] for x in dev[:3]), *dev[3:6], dev[6][:, :pre], **kw)
    print(f"tail D={dim} C={chunk} T={length} cut={cut} fresh={fresh}", flush=True)
    _, got, got_hist = gdn_prefill(*(x[:, pre:] for x in dev[:3]), *dev[3:6], dev[6][:, pre:], initial_state=state,
                                   initial_conv=hist, **kw)
    torch.cuda.synchronize()
    f64 = [x.double() if x.is_floating_point() else x for x in inputs]
    want = recurrent_gated_delta_rule(*core_inputs(*f64, dtype=torch.float64, **shape))[1]
    assert rel(got.cpu(), want) <= 1e-5, rel(got.cpu(), want)
    assert torch.equal(got_hist.cpu(), _want_history(qkv[:, pre:], seg[:, pre:], None if hist is None else hist.cpu(),
                                                     taps - 1))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_unaligned_history_output(dtype):
    """The C ABI takes the conv history's output at any address of its element type."""
    import ctypes

    from tjev_amd import _lib
    from tjev_amd.gdn import GdnPlan
    from tjev_amd.testing import gdn_inputs

    dev = [x.cuda() for x in gdn_inputs(batch=1, length=20, key_heads=1, value_heads=1, dim=16, dtype=dtype, seed=2)]
    qkv = dev[0]
    plan = GdnPlan(batch=1, length=20, key_heads=1, key_dim=16, value_heads=1, value_dim=16, taps=4, chunk=16,
                   io_dtype=dtype, gate_dtype=dtype)
    out = torch.empty((1, 20, 1, 16), dtype=dtype, device="cuda")
    res, ws = plan.residuals(qkv.device), plan.workspace(False, qkv.device)
    buf = torch.full((3 * 48 + 2,), 7.0, dtype=dtype, device="cuda")
    ptr = [x.data_ptr() for x in dev]
    _lib.check_status(plan.lib.tjev_gdn_mega2_fwd_cont(
        ctypes.byref(plan.params), plan._stream(qkv.device), *ptr, None, None, out.data_ptr(), res.data_ptr(), None,
        buf[1:].data_ptr(), ws.data_ptr(), ws.numel()))
    torch.cuda.synchronize()
    assert torch.equal(buf[1:-1].view(1, 3, 48), qkv[:, -3:])
    assert float(buf[0]) == 7.0 and float(buf[-1]) == 7.0
