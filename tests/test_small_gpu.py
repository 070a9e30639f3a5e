"""Problems of few tiles take kernels of their own (sba_small.hip): on either side of their blocks of 32 and rounds of 128, in every form
that the rule lets in, against the oracle and against the general kernels."""
import pytest
import torch

from oracle import sb_oracle as orc
from stickbreaking_attention import sb_attn, sb_attn_fused
from stickbreaking_attention import _native as nat
from stickbreaking_attention import _ops
from tests.helpers import assert_close, cu_from_lengths, kernels_of, oracle_varlen
from tests.test_fused_gpu import check, fused_reference
from tests.test_head_dim_256_gpu import DEV, _need_gpu, _run  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,lengths", [(64, [193, 128, 1]), (64, [129, 31, 32, 33]), (64, [161, 129, 33, 32, 31]), (64, [255, 257, 300]), (64, [1, 1025]), (32, [500, 129]),
                                       (8, [385, 384]), (40, [640]), (72, [161, 260]), (96, [513]), (104, [290, 100]), (128, [401, 2]),
                                       (128, [256, 255, 257]), (136, [300, 31]), (192, [255, 257]), (200, [513]), (256, [129, 385, 33])])
@pytest.mark.parametrize("ac,fused", [(False, False), (True, False), (False, True), (True, True)])
def test_packed_edges(d, lengths, ac, fused, monkeypatch):
    monkeypatch.setattr(_ops, "FORWARD_FLAGS", nat.FLAG_FEW_TILES_FORWARD)
    T = sum(lengths)
    q, k, v, do = orc.make_inputs((3, T, d), d + T)
    ran = kernels_of(q, lengths)
    assert ran.fwd_small_workgroups > 0 and (ran.bwd_small_workgroups > 0) == (d <= 128 and lengths != [129, 31, 32, 33])
    if fused:
        check(_run(q, k, v, do, lengths, ac, fused=True), fused_reference(q, k, v, do, lengths, ac))
        return
    drem = torch.randn((3, T), generator=torch.Generator().manual_seed(d)).to(torch.bfloat16)
    ref = oracle_varlen(q, k, v, do, lengths, ac, drem=drem)
    for name, g, r in zip(("o", "rem", "dq", "dk", "dv"), _run(q, k, v, do, lengths, ac, drem=drem), ref):
        assert_close(name, g, r)


_ROUND = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 2.0 ** -7}   # one step of the output (float32 inputs round to bfloat16)


def _both(shape, dtype, times, layout, ac, fused, with_rem):
    """Outputs and gradients of a small call, and those of the same heads `times` over."""
    gen = torch.Generator(device=DEV).manual_seed(shape[-2])
    B, H, T, d = shape
    t = [torch.randn((B, T, H, d) if layout == "tokens" else shape, generator=gen, device=DEV).to(dtype) for _ in range(4)]
    if layout == "tokens":
        t = [x.transpose(1, 2) for x in t]
    drem = torch.randn((B, H, T), generator=gen, device=DEV).to(dtype)
    results = []
    for n in (1, times):
        q, k, v, do = (x.repeat(1, n, 1, 1) if n > 1 else x for x in t)
        q, k, v = (x.detach().requires_grad_() for x in (q, k, v))
        if fused:
            out = (sb_attn_fused(q, k, v, attend_current=ac),)
            grads = torch.autograd.grad(out, (q, k, v), do)
        else:
            out = sb_attn(q, k, v, attend_current=ac)
            grads = torch.autograd.grad(out if with_rem else out[:1], (q, k, v), (do, drem.repeat(1, n, 1)) if with_rem else (do,))
        results.append([x.detach()[:, :H] for x in out + tuple(grads)])
    return results


@pytest.mark.parametrize("dtype", list(_ROUND))
@pytest.mark.parametrize("d,batch,T,layout", [(64, 1, 600, "heads"), (64, 2, 257, "tokens"), (32, 3, 130, "heads"), (96, 1, 400, "tokens"), (128, 2, 321, "heads")])
@pytest.mark.parametrize("ac,fused,with_rem", [(False, False, True), (True, False, False), (False, True, False), (True, True, False)])
def test_gradients_like_the_general_kernels(d, batch, T, layout, dtype, ac, fused, with_rem):
    """Both round weights and logit gradients to 16 bits before the same products, from float32 values that differ in the last bits: of the at most T terms
    of an element some land on the neighbour (one step, independently), and the output may."""
    small, many = _both((batch, 2, T, d), dtype, 64 * 1024 // T, layout, ac, fused, with_rem)
    for g, r in zip(small, many):
        scale = float(r.float().abs().max())
        torch.testing.assert_close(g, r, rtol=_ROUND[dtype], atol=_ROUND[dtype] / 4 * scale)
        assert float((g.float() - r.float()).norm()) <= _ROUND[dtype] / 4 * float(r.float().norm())


@pytest.mark.parametrize("dtype", list(_ROUND))
@pytest.mark.parametrize("d,batch,T,layout", [(64, 1, 600, "heads"), (64, 2, 257, "tokens"), (32, 3, 130, "heads"), (96, 1, 400, "tokens"), (128, 2, 321, "heads"),
                                              (256, 1, 260, "tokens"), (160, 2, 383, "heads")])
@pytest.mark.parametrize("ac", [False, True])
def test_the_same_as_the_general_kernels(d, batch, T, layout, dtype, ac):
    """Remainders to the bit (the table goes to the backward of either form), outputs up to the order of a float32 sum."""
    gen = torch.Generator(device=DEV).manual_seed(T)
    shape = (batch, 2, T, d) if layout == "heads" else (batch, T, 2, d)
    q, k, v = (torch.randn(shape, generator=gen, device=DEV).to(dtype) for _ in range(3))
    if layout == "tokens":
        q, k, v = (t.transpose(1, 2) for t in (q, k, v))
    times = 64 * 1024 // T                    # (fills the chip several times over)
    o, rem = sb_attn(q, k, v, attend_current=ac)
    o_many, rem_many = sb_attn(*(t.repeat(1, times, 1, 1) for t in (q, k, v)), attend_current=ac)
    assert torch.equal(rem, rem_many[:, :2])
    # a float32 sum of T weighted values below 6 in another order, which may round to the neighbour
    torch.testing.assert_close(o, o_many[:, :2], rtol=_ROUND[dtype], atol=T * 6 * 2.0 ** -24)


@pytest.mark.parametrize("d,H,lengths", [(64, 2, [700, 40, 129]), (32, 1, [513]), (96, 3, [400, 33]), (128, 2, [321, 1]), (256, 2, [300, 65])])
def test_a_sequence_in_any_company(d, H, lengths, monkeypatch):
    """On the general kernels a sequence's outputs and gradients are the same bits alone, beside more heads, beside other documents and
    where the weights are returned too; by size, its remainders are."""
    from stickbreaking_attention import sb_attn_varlen
    from stickbreaking_attention.sb_varlen import varlen_fwd
    lib = nat.load()
    gen = torch.Generator(device=DEV).manual_seed(d)
    T, others = sum(lengths), [900, 31, 128] * 6
    mine = [torch.randn((H, T, d), generator=gen, device=DEV).to(torch.bfloat16) for _ in range(4)]
    theirs = [torch.randn((H, sum(others), d), generator=gen, device=DEV).to(torch.bfloat16) for _ in range(4)]

    def run(tensors, lens):
        q, k, v = (t.requires_grad_() for t in tensors[:3])
        o, rem = sb_attn_varlen(q, k, v, cu_from_lengths(lens, device=DEV), max(lens), zero_start=False)
        return [t.detach()[:H, :T] for t in (o, rem) + torch.autograd.grad(o, (q, k, v), tensors[3])]

    def calls():
        yield run([t.clone() for t in mine], lengths)
        yield run([t.repeat(200, 1, 1) for t in mine], lengths)
        yield run([torch.cat([a, b], 1).repeat(12, 1, 1) for a, b in zip(mine, theirs)], lengths + others)

    assert kernels_of(mine[0], lengths).fwd_small_workgroups > 0 and kernels_of(mine[0].repeat(200, 1, 1), lengths).fwd_small_workgroups == 0
    alone, *company = calls()
    for other in company:
        assert torch.equal(alone[1], other[1])
    monkeypatch.setattr(_ops, "FORWARD_FLAGS", nat.FLAG_GENERAL_FORWARD)
    lib.sba_set_backward_form(1)
    try:
        alone, *company = calls()
    finally:
        lib.sba_set_backward_form(0)
    for other in company:
        for name, a, b in zip(("o", "rem", "dq", "dk", "dv"), alone, other):
            assert torch.equal(a, b), name
    with torch.no_grad():
        o, rem = varlen_fwd(*(t.detach() for t in mine[:3]), cu_from_lengths(lengths, device=DEV), max(lengths), logit_scale=d ** -0.5,
                            no_grad=True, return_attention=True)[:2]
    assert torch.equal(o, alone[0]) and torch.equal(rem, alone[1])
