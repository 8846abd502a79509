"""The merged projections' kernel (tjev_gdn_lora_merge) at the edges of its tiles (rows and columns
below, at and past a 16-row strip, a 128-row and a 128-column tile), every rank, several projections in one
launch: round(w + s a b) with a and b rounded to bf16, against fp64 on the same rounded values.
The kernel's fp32 sum is within 2^-24 (rank + 2) of sum |a b| s + |w| of the exact one, so a result
is the bf16 rounding of a value that far off: half a bf16 spacing past it (bf16 keeps 8 bits: the
spacing at |v| in [2^e, 2^(e+1)) is 2^(e-7), half of it at most 2^-8 |v|)."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

GUARD = 64  # elements before and after an output


@pytest.mark.parametrize("rank", [32, 64, 96, 128])
@pytest.mark.parametrize("shapes", [[(1, 8)], [(15, 136), (17, 128), (16, 120)],
                                    [(127, 136), (128, 8), (129, 128)], [(257, 256), (255, 32), (256, 264), (2560, 64)]])
def test_merge_matches_fp64(rank, shapes):
    from tjev_amd import _lib

    gen = torch.Generator().manual_seed(rank)
    rn = lambda *s: torch.randn(s, generator=gen)  # noqa: E731
    ws = [rn(i, o).to(torch.bfloat16) for i, o in shapes]
    a_s, b_s = [rn(i, rank) * rank ** -0.5 for i, o in shapes], [rn(rank, o) * 0.3 for i, o in shapes]
    scales = [0.5 + n for n in range(len(shapes))]
    print(f"merge rank={rank} {shapes}", flush=True)
    # the library's entry point itself; each output lies between guard words that must stay
    dev = [[t.cuda() for t in ts] for ts in (ws, a_s, b_s)]
    bufs = [torch.full((w.numel() + 2 * GUARD,), 7.0, dtype=torch.bfloat16, device="cuda") for w in ws]
    got = [x[GUARD:-GUARD].view(w.shape) for x, w in zip(bufs, ws)]
    args = (_lib.Merge * len(ws))(*(_lib.Merge(w.data_ptr(), a.data_ptr(), b.data_ptr(), y.data_ptr(), *w.shape, rank, s)
                                    for w, a, b, y, s in zip(*dev, got, scales)))
    _lib.check_status(_lib.load().tjev_gdn_lora_merge(args, len(ws), torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    for x in bufs:
        assert bool((x[:GUARD] == 7.0).all()) and bool((x[-GUARD:] == 7.0).all())
    for w, a, b, s, y in zip(ws, a_s, b_s, scales, got):
        a, b, w = a.bfloat16().double(), b.bfloat16().double(), w.double()
        want = w + s * (a @ b)
        room = 2.0 ** -24 * (rank + 2) * (w.abs() + s * (a.abs() @ b.abs()))
        err = (y.double().cpu() - want).abs()
        assert bool((err <= 2.0 ** -8 * (want.abs() + room) + room).all()), float((err / want.abs()).max())


def test_block_projections_take_the_kernel(monkeypatch):
    """The shapes of a block's projections (bf16 weights, fp32 adapters) go to the kernel, not to the GEMM it
    replaces (which would pass the numeric bar too)."""
    from tjev_amd import block

    gen = torch.Generator().manual_seed(5)
    shapes, rank = [(256, 512), (256, 256), (256, 16), (256, 16)], 64
    ws = [torch.randn(s, generator=gen).to(torch.bfloat16).cuda() for s in shapes]
    a_s = [torch.nn.Parameter(torch.randn(i, rank, generator=gen).cuda()) for i, _ in shapes]
    b_s = [torch.nn.Parameter(torch.randn(rank, o, generator=gen).cuda()) for _, o in shapes]
    want = [block._merge(w, a, b, 0.5, torch.bfloat16) for w, a, b in zip(ws, a_s, b_s)]

    def refuse(*args):
        raise AssertionError("the GEMM ran")

    monkeypatch.setattr(block, "_merge", refuse)
    print("merge of a block's projections", flush=True)
    with torch.no_grad():
        got = block._merge_all(ws, a_s, b_s, [0.5] * len(ws), torch.bfloat16)
    for w, a, b, y, z in zip(ws, a_s, b_s, got, want):
        # two roundings of fp32 sums of the same products: one bf16 spacing and twice the sums' error apart
        room = 2.0 ** -24 * (rank + 2) * (w.float().abs() + 0.5 * (a.detach().abs() @ b.detach().abs()) * 1.01)
        assert bool(((y.float() - z.float()).abs() <= 2.0 ** -7 * (z.float().abs() + room) + 2 * room).all())


def test_merge_refuses_what_it_does_not_hold():
    from tjev_amd import _lib

    lib = _lib.load()
    t = torch.zeros(64, 64, device="cuda")
    p = t.data_ptr()
    ok = dict(w=p, a=p, b=p, merged=p, inputs=16, outputs=16, rank=32, scale=1.0)
    for bad, status in ((dict(outputs=12), 2), (dict(rank=48), 2), (dict(rank=160), 2), (dict(inputs=0), 1), (dict(w=None), 1),
                        (dict(b=p + 4), 1)):
        assert lib.tjev_gdn_lora_merge((_lib.Merge * 1)(_lib.Merge(**{**ok, **bad})), 1, None) == status, bad
    assert lib.tjev_gdn_lora_merge((_lib.Merge * 9)(*[_lib.Merge(**ok)] * 9), 9, None) == 1
    assert lib.tjev_gdn_lora_merge(None, 1, None) == 1


@pytest.mark.parametrize("inputs,outputs", [(0, 64), (64, 0), (64, 12)])
def test_merge_of_other_forms_takes_the_gemm(inputs, outputs):
    """What the kernel does not hold (no rows, no columns, columns not in multiples of 8) merges as before."""
    from tjev_amd.block import _merge, _merge_all

    gen = torch.Generator().manual_seed(3)
    w = torch.randn(inputs, outputs, generator=gen).to(torch.bfloat16).cuda()
    a, b = torch.randn(inputs, 64, generator=gen).cuda(), torch.randn(64, outputs, generator=gen).cuda()
    print(f"merge {inputs} x {outputs}", flush=True)
    (got,) = _merge_all([w], [a], [b], [0.5], torch.bfloat16)
    assert got.shape == w.shape and torch.equal(got, _merge(w, a, b, 0.5, torch.bfloat16))


@pytest.mark.parametrize("pre_dispatch", [False, True])
def test_recorded_merge_stays_in_the_graph(pre_dispatch):
    """A graph of the projections recorded by make_fx holds the merge as an operator (the kernel's launch is
    none: its output would be recorded as uninitialised memory) and replays to the same values."""
    from torch.fx.experimental.proxy_tensor import make_fx

    from tjev_amd.block import LoRALinear, grouped

    gen = torch.Generator().manual_seed(4)
    w = torch.randn(256, 128, generator=gen).to(torch.bfloat16).cuda()
    a, b = torch.randn(256, 32, generator=gen).cuda(), torch.randn(32, 128, generator=gen).cuda()
    x = torch.randn(64, 256, generator=gen).to(torch.bfloat16).cuda()
    linear = LoRALinear(w, a, b, 0.5)
    print(f"recorded merge, pre_dispatch={pre_dispatch}", flush=True)
    want = grouped(x, linear)[0]
    graph = make_fx(lambda t: grouped(t, linear)[0], pre_dispatch=pre_dispatch)(x)
    names = [str(n.target) for n in graph.graph.nodes if n.op == "call_function"]
    assert any("addmm" in n for n in names) and not any("empty" in n for n in names), names
    assert torch.equal(graph(x), want)
