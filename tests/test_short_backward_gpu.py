"""Many short documents take one kernel for the whole backward (bwd_short_kernel; above head_dim 64 those of up to 64 tokens, and long ones among many short): lengths on either side of its blocks of 32
and of its teams (64, 128, 256 tokens), classes that do not fill a workgroup, in every form, against the oracle and the general two passes."""
import ctypes
import random

import pytest
import torch

from oracle import sb_oracle as orc
from stickbreaking_attention import sb_attn, sb_attn_fused, sb_attn_varlen, sb_attn_varlen_fused
from tests.helpers import assert_close, cu_from_lengths, oracle_varlen
from tests.test_chained_backward_gpu import form  # noqa: F401
from tests.test_fused_gpu import check, fused_reference
from tests.test_head_dim_256_gpu import DEV, _need_gpu, _run  # noqa: F401

pytestmark = pytest.mark.gpu
EDGES = [256, 1, 255, 225, 64, 129, 128, 0, 127, 97, 96, 65, 63, 224, 33, 32, 31, 2, 160, 161]
_ROUND = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 2.0 ** -7}   # one step of the output (float32 inputs round to bfloat16)


@pytest.mark.parametrize("d,lengths", [(64, EDGES), (32, EDGES), (40, [64] * 21), (8, [128, 1] * 11), (64, [128, 65, 64] * 5 + [33]), (64, [17] * 99),
                                       (128, [64, 1, 63, 33, 32, 31, 0, 2] * 3 + [17]), (72, [64] * 9), (96, [33, 7] * 10)])
@pytest.mark.parametrize("ac,fused", [(False, False), (True, False), (False, True), (True, True)])
def test_against_the_oracle(d, lengths, ac, fused):
    T, H = sum(lengths), 40000 // sum(lengths) + 1
    q, k, v, do = orc.make_inputs((H, T, d), d + T)
    if fused:
        check(_run(q, k, v, do, lengths, ac, fused=True), fused_reference(q, k, v, do, lengths, ac))
        return
    drem = torch.randn((H, T), generator=torch.Generator().manual_seed(d)).to(torch.bfloat16)
    ref = oracle_varlen(q, k, v, do, lengths, ac, drem=drem)
    for name, g, r in zip(("o", "rem", "dq", "dk", "dv"), _run(q, k, v, do, lengths, ac, drem=drem), ref):
        assert_close(name, g, r)


@pytest.mark.parametrize("d,lengths,taken", [(128, EDGES, True), (96, EDGES, True), (72, [128, 1, 31, 97] * 7, True), (128, [200] * 3 + [17] * 40, True),
                                             (128, [128] * 16, True), (96, [200, 100] * 5, False), (128, [65, 66] * 5, False)])
@pytest.mark.parametrize("ac,fused", [(False, False), (True, False), (False, True)])
def test_longer_documents_above_head_dim_64(d, lengths, taken, ac, fused):
    from stickbreaking_attention import _native as nat
    T, H = sum(lengths), 40000 // sum(lengths) + 1
    p = nat.SbaProblem(nat.SBA_BF16, d, H, 1, T, len(lengths), max(lengths), nat.FLAG_PRODUCT_SPACE, 1.0, 16)
    g = nat.SbaGeometry()
    nat.check(nat.load().sba_launch_geometry(ctypes.byref(p), ctypes.byref(g)), "sba_launch_geometry")
    assert (g.bwd_short_workgroups > 0) == taken
    test_against_the_oracle(d, lengths, ac, fused)


@pytest.mark.parametrize("dtype", list(_ROUND))
@pytest.mark.parametrize("d,shape,layout", [(64, None, "heads"), (48, None, "tokens"), (64, (5, 250), "tokens"), (32, (70, 70), "heads"), (24, (9, 128), "heads"),
                                            (128, (33, 50), "heads"), (80, (20, 64), "tokens")])
@pytest.mark.parametrize("ac,fused,zero_start", [(False, False, False), (True, False, True), (False, True, True)])
def test_like_the_two_passes(d, shape, layout, dtype, ac, fused, zero_start, form):  # noqa: F811
    """Weights and logit gradients are rounded to 16 bits before the same products, from float32 values that differ in the last bits: now and then a
    term lands on the neighbour (one step, independently of the others), and so may the output."""
    lengths = [random.Random(4).randint(1, 200) for _ in range(20)] + EDGES if shape is None else None
    B, T = (1, sum(lengths)) if shape is None else shape
    H = 40000 // (B * T) + 1
    gen = torch.Generator(device=DEV).manual_seed(d)

    def tensor(*tail):
        t = torch.randn((B, T, H) + tail if layout == "tokens" else (B, H, T) + tail, generator=gen, device=DEV).to(dtype)
        t = t.transpose(1, 2) if layout == "tokens" else t
        return t[0] if shape is None else t

    q, k, v = (tensor(d).requires_grad_() for _ in range(3))
    do, drem = tensor(d), tensor()
    results = []
    for which in (0, 1):
        form(which)
        if shape is None:
            cu = cu_from_lengths(lengths, leading_zero=zero_start, dtype=torch.int64, device=DEV)
            out = (sb_attn_varlen_fused if fused else sb_attn_varlen)(q, k, v, cu, max(lengths), zero_start=zero_start, attend_current=ac)
        else:
            out = (sb_attn_fused if fused else sb_attn)(q, k, v, attend_current=ac)
        results.append(torch.autograd.grad(out, (q, k, v), do if fused else (do, drem)))
    for g, r in zip(*results):
        torch.testing.assert_close(g, r, rtol=_ROUND[dtype], atol=_ROUND[dtype] / 4 * float(r.float().abs().max()))
        assert float((g.float() - r.float()).norm()) <= _ROUND[dtype] / 4 * float(r.float().norm())


def test_rows_of_no_document_are_cleared_and_refused_input_is_not_computed(monkeypatch):
    from stickbreaking_attention import _ops
    monkeypatch.setattr(_ops, "SYNC_FREE", True)
    lengths = [100, 30, 64, 200]
    q, k, v, do = (t.to(DEV) for t in orc.make_inputs((70, 700, 64), 5))
    q, k, v = (t.requires_grad_() for t in (q, k, v))
    cu = cu_from_lengths(lengths, device=DEV)
    for longest in (200, 150):
        _ops.release_workspaces()
        junk = [torch.full_like(q, 3.0) for _ in range(3)]
        del junk                                  # what the gradients' memory holds before
        o, _ = sb_attn_varlen(q, k, v, cu, longest, zero_start=False)
        grads = torch.autograd.grad(o, (q, k, v), do)
        for g in grads:
            if longest == 200:
                assert not g[:, sum(lengths):].any() and bool(g[:, :sum(lengths)].isfinite().all())
            else:
                assert bool(g.isnan().all())


def test_rows_that_are_not_finite_stay_in_their_documents():
    lengths = [40, 200, 64, 90, 30]
    T = sum(lengths)
    tensors = orc.make_inputs((100, T, 64), 9)
    clean = _run(*tensors, lengths)[2:]
    for which in range(4):
        x = [t.clone() for t in tensors]
        x[which][:, 240 + 20] = float("inf")      # in the third
        for got, want in zip(_run(*x, lengths)[2:], clean):
            assert torch.equal(got[:, :240], want[:, :240]) and torch.equal(got[:, 304:], want[:, 304:]), which


def test_replays_from_a_hip_graph():
    from stickbreaking_attention import _ops
    lengths, H, d = [256, 40, 128, 90, 64, 33, 200], 64, 64
    T = sum(lengths) + 7
    cu = cu_from_lengths(lengths, device=DEV)

    def launch(q, k, v, do):
        o, rem, state = _ops.run_forward(q, k, v, False, cu, max(lengths), d ** -0.5, False, need_table=True)
        return (o, rem) + tuple(_ops.run_backward(q, k, v, do, None, False, state, d ** -0.5, False))

    def inputs(seed):
        return [t.to(DEV) for t in orc.make_inputs((H, T, d), seed)]

    static = inputs(100)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        launch(*static)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = launch(*static)
    for seed in (101, 102, 103):
        fresh = inputs(seed)
        for dst, src in zip(static, fresh):
            dst.copy_(src)
        graph.replay()
        torch.cuda.synchronize()
        eager = launch(*fresh)
        torch.cuda.synchronize()
        for name, a, b in zip(("o", "rem", "dq", "dk", "dv"), captured, eager):
            assert torch.equal(a, b), (seed, name)
