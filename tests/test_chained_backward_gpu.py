"""The one-pass backward (csrc/sba_chain.hip), forced wherever it is possible: documents at the edges of its steps of 32 and
64 queries and 128-key tiles and of the three steps a tile lags behind its predecessor, both kernel widths and heads
narrower than them, against the oracle; and queues of many items per workgroup and many groups, against the two-pass form."""
import ctypes

import pytest
import torch

from oracle import sb_oracle as orc
from tests.helpers import assert_close, cu_from_lengths, oracle_varlen

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture
def form():
    from stickbreaking_attention import _native
    lib = _native.load()
    yield lib.sba_set_backward_form
    lib.sba_set_backward_form(0)


def gradients(op, tensors, cu, longest, ac, grads):
    x = [t.to(DEV).requires_grad_() for t in tensors]
    out = op(*x, cu, longest, zero_start=False, attend_current=ac)
    out = out if isinstance(out, tuple) else (out,)
    return torch.autograd.grad(out, x, [g.to(DEV) for g in grads[:len(out)]])


@pytest.mark.parametrize("ac", [False, True])
@pytest.mark.parametrize("steps,d,dtype", [(2, 128, torch.bfloat16), (2, 96, torch.float16), (2, 104, torch.bfloat16),
                                           (2, 64, torch.bfloat16), (2, 32, torch.float16), (3, 64, torch.bfloat16),
                                           (3, 40, torch.float16), (3, 24, torch.bfloat16),
                                           # the two passes, which problems of these sizes no longer take by themselves
                                           (1, 128, torch.bfloat16), (1, 96, torch.float16), (1, 64, torch.bfloat16), (1, 40, torch.float16), (1, 32, torch.bfloat16)])
def test_tile_edges(form, steps, d, dtype, ac):
    from stickbreaking_attention import sb_attn_varlen, sb_attn_varlen_fused
    lengths = [1, 32, 33, 127, 128, 129, 224, 256, 257, 550]
    H, used = 3, sum(lengths)
    T = used + 9
    q, k, v, do = (t.to(dtype) for t in orc.make_inputs((H, T, d), 40 + d))
    drem = torch.randn((H, T), generator=torch.Generator().manual_seed(d)).to(dtype)
    cu = cu_from_lengths(lengths, device=DEV)
    form(steps)
    got = gradients(sb_attn_varlen, (q, k, v), cu, max(lengths), ac, (do, drem))
    fused = gradients(sb_attn_varlen_fused, (q, k, v), cu, max(lengths), ac, (do,))
    form(1)
    fused_two = gradients(sb_attn_varlen_fused, (q, k, v), cu, max(lengths), ac, (do,))
    ref = oracle_varlen(q[:, :used], k[:, :used], v[:, :used], do[:, :used], lengths, ac, drem=drem[:, :used])[2:]
    for name, g, r, f, f2 in zip(("dq", "dk", "dv"), got, ref, fused, fused_two):
        assert not g[:, used:].any() and not f[:, used:].any()
        assert_close(name, g[:, :used], r)
        assert_close(name + " of o + rem v", f[:, :used], f2[:, :used].float())


@pytest.mark.parametrize("steps", [2, 3])
@pytest.mark.parametrize("H,lengths", [(5, [37 + 61 * i % 400 for i in range(90)]), (12, [2000, 1, 900, 4000]), (3, [4600, 700])])
def test_queues(form, steps, H, lengths):
    from stickbreaking_attention import sb_attn_varlen
    T = sum(lengths)
    tensors = orc.make_inputs((H, T, 64), T)
    drem = torch.randn((H, T), generator=torch.Generator().manual_seed(T)).to(torch.bfloat16)
    cu = cu_from_lengths(lengths, device=DEV)
    form(1)
    two = gradients(sb_attn_varlen, tensors[:3], cu, max(lengths), False, (tensors[3], drem))
    form(steps)
    first = gradients(sb_attn_varlen, tensors[:3], cu, max(lengths), False, (tensors[3], drem))
    again = gradients(sb_attn_varlen, tensors[:3], cu, max(lengths), False, (tensors[3], drem))
    for name, a, b, c in zip(("dq", "dk", "dv"), two, first, again):
        assert_close(name, b, a.float())
        assert torch.equal(b, c)


@pytest.mark.parametrize("steps,d", [(2, 128), (2, 96), (2, 64), (3, 64), (2, 32), (3, 32)])
def test_the_same_bits_from_run_to_run(form, steps, d):
    """Items of one step up to one more than the steps in flight, with product waves that have a block of dq and without."""
    from stickbreaking_attention import sb_attn_varlen
    lengths = [300, 131, 32, 161, 193, 288, 609]
    H, T = 6, sum(lengths)
    tensors = orc.make_inputs((H, T, d), 60 + d)
    drem = torch.randn((H, T), generator=torch.Generator().manual_seed(d)).to(torch.bfloat16)
    cu = cu_from_lengths(lengths, device=DEV)
    form(1)
    two = gradients(sb_attn_varlen, tensors[:3], cu, max(lengths), False, (tensors[3], drem))
    form(steps)
    runs = [gradients(sb_attn_varlen, tensors[:3], cu, max(lengths), False, (tensors[3], drem)) for _ in range(8)]
    for i, name in enumerate(("dq", "dk", "dv")):
        assert_close(name, runs[0][i], two[i].float())
        assert all(torch.equal(runs[0][i], r[i]) for r in runs[1:]), name


@pytest.mark.parametrize("H,d,lengths,declared,chained", [
    (4, 96, [2500] * 3, 2500, True),                    # 12 chains on 8 XCDs, few enough tiles to be held at once
    (12, 64, [4096], 4096, True),
    (18, 64, [3000], 3000, True), (12, 64, [4500], 4500, False),      # a third more than the mean on the worst XCD, which does not hold them: up to 4096 keys
    (16, 64, [6000, 500, 500, 500], 6000, True),        # even chains of any length
    (2, 128, [9000, 300, 200], 9000, False),            # two long ones, each on an XCD of its own
    (16, 32, [5000, 4000], 16384, True),                # declared longer than there are rows
    (18, 32, [3000], 3000, False), (20, 32, [3000], 3000, True),      # at head_dim 32 that is too much
    (2, 96, [2796] + [322] * 118, 2796, True),          # many chains come out even by their number
    (9, 96, [4881, 4881, 3341, 3186, 2728, 2219, 187, 100, 100, 100, 100, 60, 40], 4881, True),
    (2, 64, [20000] + [200] * 30, 20000, False),        # but not next to one longer than its share
])
def test_the_choice_between_one_pass_and_two(form, H, d, lengths, declared, chained):
    from stickbreaking_attention import _native as nat, sb_attn_varlen
    T = sum(lengths)
    p = nat.SbaProblem(1, d, H, 1, T, len(lengths), declared, nat.FLAG_PRODUCT_SPACE, d ** -0.5, 0x1000)
    assert (nat.load().sba_chain_scratch_bytes(ctypes.byref(p)) > 0) == chained
    gen = torch.Generator(device=DEV).manual_seed(T)
    x = [torch.randn((H, T, d), generator=gen, device=DEV).to(torch.bfloat16).requires_grad_() for _ in range(3)]
    do = torch.randn((H, T, d), generator=gen, device=DEV).to(torch.bfloat16)
    cu = cu_from_lengths(lengths, device=DEV)
    run = lambda: torch.autograd.grad(sb_attn_varlen(*x, cu, declared, zero_start=False)[0], x, do)
    got = run()
    form(1)
    for name, g, t in zip(("dq", "dk", "dv"), got, run()):
        assert_close(name, g, t.float())


@pytest.mark.parametrize("attend_current", [False, True])
@pytest.mark.parametrize("d", [128, 96])
def test_rows_streamed_past_the_l2_give_the_same_bits(form, d, attend_current):
    """The rows are streamed where an XCD has several times the L2 of them to do: 144 heads at once and a few of them alone."""
    from stickbreaking_attention import sb_attn_varlen
    from tests.helpers import kernels_of
    lengths = [300, 131, 32, 161, 193, 288, 609]
    H, T = 144, sum(lengths)
    q, k, v, do = orc.make_inputs((H, T, d), 5)
    drem = torch.randn((H, T), generator=torch.Generator().manual_seed(5)).to(torch.bfloat16)
    cu = cu_from_lengths(lengths, device=DEV)
    form(2)
    assert kernels_of(q, lengths).bwd_rows_streamed
    streamed = gradients(sb_attn_varlen, (q, k, v), cu, max(lengths), attend_current, (do, drem))
    for heads in (slice(0, 6), slice(140, 144)):
        assert not kernels_of(q[heads], lengths).bwd_rows_streamed
        kept = gradients(sb_attn_varlen, (q[heads], k[heads], v[heads]), cu, max(lengths), attend_current, (do[heads], drem[heads]))
        for name, a, b in zip(("dq", "dk", "dv"), kept, streamed):
            assert torch.equal(a, b[heads]), name


@pytest.mark.parametrize("steps,d", [(2, 128), (2, 64), (3, 64), (2, 32), (3, 32)])
def test_a_wait_that_runs_out_gives_nan_and_nothing_else(form, steps, d):
    """Every wait for the key tile before ends after one look, so that tiles go on without the partial sums they
    waited for, at whatever step they have got to.  An element that depends on a missing one has to be NaN: what is
    not NaN has to be the same bits as ever."""
    from stickbreaking_attention import sb_attn_varlen
    lengths = [2000, 128, 700, 1400, 257, 1000]
    H, T = 24, sum(lengths)
    tensors = orc.make_inputs((H, T, d), 9 + d)
    drem = torch.randn((H, T), generator=torch.Generator().manual_seed(d)).to(torch.bfloat16)
    cu = cu_from_lengths(lengths, device=DEV)
    form(steps)
    whole = gradients(sb_attn_varlen, tensors[:3], cu, max(lengths), False, (tensors[3], drem))
    form(steps | 0x100)
    cut = gradients(sb_attn_varlen, tensors[:3], cu, max(lengths), False, (tensors[3], drem))
    lost = [torch.isnan(b) for b in cut]
    for name, a, b, nan in zip(("dq", "dk", "dv"), whole, cut, lost):
        assert torch.isfinite(a).all()
        assert torch.equal(torch.where(nan, a, b), a), name
    assert lost[0].any() and lost[1].any() and not all(nan.all() for nan in lost)
    for nan in lost:      # (a row is lost as a whole)
        assert torch.equal(nan.any(-1), nan.all(-1))


@pytest.mark.parametrize("ac", [False, True])
@pytest.mark.parametrize("steps,d", [(1, 128), (2, 128), (2, 96), (1, 64), (2, 64), (3, 64), (2, 32), (3, 32)])
def test_rows_that_are_not_finite_stay_behind_the_blocks_that_hide_them(form, steps, d, ac):
    """A key that is not finite must not reach the gradients of queries that cannot see it, nor a query the gradients of
    keys it cannot see, beyond the 32-row block of its own: there, the matrix products multiply it by zero."""
    from stickbreaking_attention import sb_attn_varlen
    lengths = [300, 128, 77]
    H, T = 2, sum(lengths)
    tensors = orc.make_inputs((H, T, d), 77 + d)
    drem = torch.randn((H, T), generator=torch.Generator().manual_seed(d)).to(torch.bfloat16)
    cu = cu_from_lengths(lengths, device=DEV)
    form(steps)
    def run(x):
        return [g.cpu() for g in gradients(sb_attn_varlen, x[:3], cu, max(lengths), ac, (x[3], drem))]
    clean = run(tensors)
    for start, row in ((0, 3), (0, 40), (0, 100), (0, 127), (0, 200), (0, 299), (300, 90), (428, 33)):
        at, length = start + row, lengths[[0, 300, 428].index(start)]
        block = start + row // 32 * 32
        older, newer = range(0, block), [i for i in range(T) if i < start or i >= min(block + 32, start + length)]
        other = [i for i in range(T) if i != at]
        for which, value in ((0, float("nan")), (1, float("nan")), (1, float("-inf")), (2, float("inf")), (2, float("nan")), (3, float("inf"))):
            x = [t.clone() for t in tensors]
            x[which][:, at] = value
            dq, dk, dv = run(x)
            same = lambda a, b, rows: torch.equal(a[:, list(rows)], b[:, list(rows)])
            name = f"{'q k v do'.split()[which]}[{at}] = {value}"
            if which in (1, 2):       # a key: queries before its block
                assert same(dq, clean[0], older), name
            if which == 2:            # and its value: keys before its block, and no dv
                assert same(dk, clean[1], older) and torch.equal(dv, clean[2]), name
            if which in (0, 3):       # a query: all other queries, keys behind its block
                assert same(dq, clean[0], other), name
                assert same((dv, dk)[which // 3], clean[2 - which // 3], newer), name


@pytest.mark.parametrize("idle", [0x01, 0x20, 0xaa, 0xf7, 0xfe])
@pytest.mark.parametrize("steps,d,H,lengths", [(2, 128, 1, [500]), (2, 96, 12, [900, 31, 2000, 128]), (3, 64, 40, [1500, 700, 129])])
def test_queues_of_xcds_that_cannot_run_the_launch(form, idle, steps, d, H, lengths):
    """What a CU mask can do: some XCDs get no workgroup.  Their queues are served by the others, with the same bits."""
    from stickbreaking_attention import sb_attn_varlen
    T = sum(lengths)
    tensors = orc.make_inputs((H, T, d), 5 + d)
    drem = torch.randn((H, T), generator=torch.Generator().manual_seed(d)).to(torch.bfloat16)
    cu = cu_from_lengths(lengths, device=DEV)
    form(steps)
    whole = gradients(sb_attn_varlen, tensors[:3], cu, max(lengths), False, (tensors[3], drem))
    form(steps | idle << 16)
    some = gradients(sb_attn_varlen, tensors[:3], cu, max(lengths), False, (tensors[3], drem))
    for name, a, b in zip(("dq", "dk", "dv"), whole, some):
        assert torch.isfinite(a).all() and torch.equal(a, b), name


def test_timing_forgets_the_launches_of_another_run(form):
    """bench.py takes a dq pass without a duration for a sign of the one-pass form: what an earlier run left there must
    not be seen."""
    from stickbreaking_attention import _native, sb_attn_varlen
    lib = _native.load()
    tensors = orc.make_inputs((2, 300, 64), 1)
    cu = cu_from_lengths([300], device=DEV)
    ms = {}
    try:
        for steps in (1, 2):
            form(steps)
            lib.sba_set_timing(1)
            gradients(sb_attn_varlen, tensors[:3], cu, 300, False, (tensors[3], torch.zeros((2, 300), dtype=torch.bfloat16)))
            ms[steps] = [lib.sba_last_kernel_ms(i) for i in range(3)]
    finally:
        lib.sba_set_timing(0)
    assert min(ms[1]) > 0 and ms[2][0] > 0 and ms[2][1] == 0 and ms[2][2] > 0
