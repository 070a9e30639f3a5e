"""The backward at head_dim 129 .. 256 whose dq pass leaves p and dz in memory for the dk/dv pass (csrc/sba_wide.hip), where its steps, its
ring of three tiles and the places of its blocks can go wrong, against the passes that form the scores twice; and its scratch."""
import ctypes

import pytest
import torch

from oracle import sb_oracle as orc
from tests.helpers import assert_close, cu_from_lengths, oracle_varlen
from tests.test_abi import problem

DEV = "cuda:0"
EDGES = [1, 31, 32, 33, 96, 97, 127, 128, 129, 160, 161, 256, 257, 385]


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


@pytest.mark.gpu
@pytest.mark.parametrize("ac", [False, True])
@pytest.mark.parametrize("d,dtype", [(256, torch.bfloat16), (200, torch.float16), (192, torch.bfloat16), (136, torch.bfloat16), (256, torch.float32)])
def test_edges(form, d, dtype, ac):
    from stickbreaking_attention import sb_attn_varlen, sb_attn_varlen_fused
    H, used = 2, sum(EDGES)
    T = used + 7
    q, k, v, do = (t.to(dtype) for t in orc.make_inputs((H, T, d), 20 + d))
    drem = torch.randn((H, T), generator=torch.Generator().manual_seed(d)).to(torch.bfloat16).to(dtype)
    cu = cu_from_lengths(EDGES, device=DEV)
    got = gradients(sb_attn_varlen, (q, k, v), cu, max(EDGES), ac, (do, drem))
    again = gradients(sb_attn_varlen, (q, k, v), cu, max(EDGES), ac, (do, drem))
    fused = gradients(sb_attn_varlen_fused, (q, k, v), cu, max(EDGES), ac, (do,))
    form(1)
    twice = gradients(sb_attn_varlen, (q, k, v), cu, max(EDGES), ac, (do, drem))
    fused_twice = gradients(sb_attn_varlen_fused, (q, k, v), cu, max(EDGES), ac, (do,))
    ref = oracle_varlen(q[:, :used], k[:, :used], v[:, :used], do[:, :used], EDGES, ac, drem=drem[:, :used])[2:]
    for name, g, a, r, t, f, ft in zip(("dq", "dk", "dv"), got, again, ref, twice, fused, fused_twice):
        assert torch.equal(g, a)
        assert not g[:, used:].any() and not f[:, used:].any()
        assert_close(name, g[:, :used], r)
        # the passes that form the scores twice stay as they were
        assert_close(name + ", scores formed twice", t[:, :used], r)
        assert_close(name + " of o + rem v", f[:, :used], ft[:, :used].float())


@pytest.mark.gpu
def test_fixed_length_and_token_major(form):
    from stickbreaking_attention import sb_attn
    B, H, T, d = 2, 3, 290, 160
    gen = torch.Generator().manual_seed(3)
    x = [torch.randn((B, T, H, d), generator=gen).to(torch.bfloat16).to(DEV).transpose(1, 2).requires_grad_() for _ in range(3)]
    do = torch.randn((B, T, H, d), generator=gen).to(torch.bfloat16).to(DEV).transpose(1, 2)
    run = lambda: torch.autograd.grad(sb_attn(*x)[0], x, do)
    got = run()
    form(1)
    for name, g, t in zip(("dq", "dk", "dv"), got, run()):
        assert_close(name, g, t.float())


@pytest.mark.gpu
@pytest.mark.parametrize("fixed", [False, True])
def test_heads_in_groups(form, fixed):
    """33 heads, of which 3.75 GiB hold 29: groups of 17 and 16."""
    from stickbreaking_attention import sb_attn, sb_attn_varlen
    H, B, T, d = 33, 16, 2048, 136
    gen = torch.Generator(device=DEV).manual_seed(8)
    draw = lambda *shape: torch.randn(shape, generator=gen, device=DEV).to(torch.bfloat16)
    shape = (B, H, T, d) if fixed else (H, B * T, d)
    x, do, drem = [draw(*shape).requires_grad_() for _ in range(3)], draw(*shape), draw(*shape[:-1])
    cu = cu_from_lengths([T] * B, device=DEV)
    run = lambda: torch.autograd.grad(sb_attn(*x) if fixed else sb_attn_varlen(*x, cu, T, zero_start=False), x, (do, drem))
    got = run()
    form(1)
    for name, g, t in zip(("dq", "dk", "dv"), got, run()):
        for head in (0, 16, 17, 32):
            assert_close(name, *((t.movedim(-3, 0) if fixed else t)[head].float() for t in (g, t)))


SKEWED = [16384] + [512] * 60      # as many longest documents as fit are three times what there is


def test_the_room_goes_by_what_the_table_holds():
    """A carry table sized by the documents' lengths says how many blocks there are; the most that the declared sizes allow would be one
    head at a time, a quarter of the chip, and that is not taken."""
    from stickbreaking_attention import _native as nat, _ops
    lib = nat.load()
    def ask(heads, lengths, known):
        p = problem(head_dim=136, heads=heads, tokens=sum(lengths), n_docs=len(lengths), max_doc_len=max(lengths), flags=nat.FLAG_PRODUCT_SPACE)
        table = 4 * _ops.workspace_sizes(False, 1, heads, sum(lengths), len(lengths), max(lengths), lengths if known else None)[1]
        return lib.sba_bwd_scratch_bytes(ctypes.byref(p), table), lib.sba_chain_scratch_bytes(ctypes.byref(p))
    entries = sum(_ops.table_entries(n) for n in SKEWED)
    assert ask(8, SKEWED, True) == (4 * 128 * entries, 0)       # two groups of four
    assert ask(8, SKEWED, False) == (0, 0)
    assert ask(4, SKEWED, True)[0] == 4 * 128 * entries
    for lengths in ([2048] * 16, [4096]):                       # all alike: the table is all but the most there can be
        exact, most = ask(33, lengths, True)
        assert ask(33, lengths, False) == (most, most) and exact <= most < 1.03 * exact


@pytest.mark.gpu
def test_heads_in_groups_by_what_the_table_holds(form):
    from stickbreaking_attention import sb_attn_varlen
    H, T, d = 8, sum(SKEWED), 136
    gen = torch.Generator(device=DEV).manual_seed(10)
    draw = lambda *shape: torch.randn(shape, generator=gen, device=DEV).to(torch.bfloat16)
    x, do = [draw(H, T, d).requires_grad_() for _ in range(3)], draw(H, T, d)
    cu = cu_from_lengths(SKEWED, device=DEV)
    run = lambda: torch.autograd.grad(sb_attn_varlen(*x, cu, max(SKEWED), zero_start=False)[0], x, do)
    got = run()
    form(1)
    for name, g, t in zip(("dq", "dk", "dv"), got, run()):
        for head in (0, 3, 4, 7):
            assert_close(name, g[head].float(), t[head].float())


@pytest.mark.gpu
@pytest.mark.parametrize("native", [True, False])
def test_the_room_is_given_back_and_done_without(form, monkeypatch, native):
    """p and dz take 1.1 GiB here.  The memory is the allocator's again after the call, and where it is not to be had the
    gradients are those of the passes that form the scores twice, bit for bit."""
    from stickbreaking_attention import _ops, sb_attn_varlen
    if not native:
        monkeypatch.setattr(_ops, "VALIDATE", True)      # (takes the launchers in Python)
    _ops.release_workspaces()
    torch.cuda.empty_cache()        # (nothing of what follows lies in a large block that an earlier test left)
    H, T, d = 16, 8192, 136
    gen = torch.Generator(device=DEV).manual_seed(11)
    draw = lambda *shape: torch.randn(shape, generator=gen, device=DEV).to(torch.bfloat16)
    x, do = [draw(H, T, d).requires_grad_() for _ in range(3)], draw(H, T, d)
    cu = cu_from_lengths([4096, 4096], device=DEV)
    run = lambda: torch.autograd.grad(sb_attn_varlen(*x, cu, 4096, zero_start=False)[0], x, do)
    form(1)
    twice = run()
    form(0)
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    once = run()
    assert torch.cuda.max_memory_allocated() - before > 1 << 30
    assert torch.cuda.memory_allocated() - before < 1 << 28         # the gradients themselves
    assert not all(torch.equal(a, b) for a, b in zip(once, twice))
    del once
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    device = torch.cuda.get_device_properties(DEV)
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (1 << 29)) / device.total_memory)
        for a, b in zip(run(), twice):
            assert torch.equal(a, b)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)


@pytest.mark.gpu
def test_a_document_whose_places_pass_2_gib(form):
    """32-bit offsets from a document's first block, beyond what a signed one holds: the newest keys' blocks are the last."""
    from stickbreaking_attention import _native as nat, sb_attn_varlen
    T, d = 38000, 136
    p = problem(head_dim=d, heads=1, tokens=T, n_docs=1, max_doc_len=T, flags=nat.FLAG_PRODUCT_SPACE)
    assert nat.load().sba_chain_scratch_bytes(ctypes.byref(p)) > 1 << 31
    gen = torch.Generator(device=DEV).manual_seed(9)
    x = [torch.randn((1, T, d), generator=gen, device=DEV).to(torch.bfloat16).requires_grad_() for _ in range(3)]
    do = torch.randn((1, T, d), generator=gen, device=DEV).to(torch.bfloat16)
    cu = cu_from_lengths([T], device=DEV)
    run = lambda: torch.autograd.grad(sb_attn_varlen(*x, cu, T, zero_start=False)[0], x, do)
    got = run()
    form(1)
    for name, g, t in zip(("dq", "dk", "dv"), got, run()):
        for rows in (slice(0, 20000), slice(20000, 34000), slice(34000, T)):
            assert_close(name, g[:, rows], t[:, rows].float())


@pytest.mark.gpu
def test_a_document_longer_than_declared_gives_nan(monkeypatch):
    """Room for p and dz goes by the declared length: what does not fit is refused by the kernels, and every gradient is NaN."""
    from stickbreaking_attention import _ops, sb_attn_varlen
    monkeypatch.setattr(_ops, "SYNC_FREE", True)
    tensors = orc.make_inputs((2, 700, 256), 4)
    cu = cu_from_lengths([600, 100], device=DEV)
    for g in gradients(sb_attn_varlen, tensors[:3], cu, 128, False, (tensors[3], torch.zeros((2, 700), dtype=torch.bfloat16))):
        assert torch.isnan(g).all()


def test_scratch(form):
    from stickbreaking_attention import _native as nat
    lib = nat.load()
    p = problem(head_dim=256, heads=16, flags=nat.FLAG_PRODUCT_SPACE)
    need = lib.sba_chain_scratch_bytes(ctypes.byref(p))
    assert need == (lib.sba_table_bytes(ctypes.byref(p)) - 256) * 32      # 128 bytes for every entry of a carry table
    view = ctypes.byref(nat.SbaView(0x1000, 0, 256 * 16384, 256))
    row = ctypes.byref(nat.SbaView(0x1000, 0, 16384, 1))
    at = ctypes.c_void_p(0x1000)
    def call(problem, scratch, size):
        return lib.sba_varlen_bwd_chained(ctypes.byref(problem), at, lib.sba_schedule_bytes(ctypes.byref(problem)), view, view, view, view, row,
                                          at, 1 << 31, ctypes.c_void_p(scratch), size, view, view, view, None)
    assert call(p, 0x1000, need - 1) == -6 and call(p, 0x1004, need) == -6
    # heads that do not fit together share the room in equal groups
    shared = problem(head_dim=256, heads=33, flags=nat.FLAG_PRODUCT_SPACE)
    assert lib.sba_chain_scratch_bytes(ctypes.byref(shared)) == need // 16 * 17
    # a group too small to fill the device, a head beyond the room, and the log-space carry: the other passes
    large = problem(head_dim=256, heads=8, tokens=32768, n_docs=1, max_doc_len=32768, flags=nat.FLAG_PRODUCT_SPACE)
    longer = problem(head_dim=256, heads=8, tokens=65536, n_docs=1, max_doc_len=65536, flags=nat.FLAG_PRODUCT_SPACE)
    log = problem(head_dim=256, heads=16)
    for other in (large, longer, log):
        assert lib.sba_chain_scratch_bytes(ctypes.byref(other)) == 0
        assert call(other, 0x1000, 1 << 40) == -4
    form(1)
    assert lib.sba_chain_scratch_bytes(ctypes.byref(p)) == 0


@pytest.mark.gpu
def test_replays_from_a_hip_graph():
    """The room is the graph's own; replays with the program's own work on the same memory sizes in between."""
    from stickbreaking_attention import _ops
    H, T, d = 3, sum(EDGES), 160
    cu = cu_from_lengths(EDGES, device=DEV)

    def launch(q, k, v, do):
        o, rem, state = _ops.run_forward(q, k, v, False, cu, max(EDGES), d ** -0.5, False, need_table=True)
        return (o, rem) + _ops.run_backward(q, k, v, do, None, False, state, d ** -0.5, False)

    inputs = lambda seed: [t.to(DEV) for t in orc.make_inputs((H, T, d), seed)]
    static = inputs(300)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        launch(*static)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = launch(*static)
    for seed in (301, 302, 303):
        fresh = inputs(seed)
        for dst, src in zip(static, fresh):
            dst.copy_(src)
        graph.replay()
        torch.cuda.synchronize()
        eager = launch(*fresh)
        torch.cuda.synchronize()
        for name, a, b in zip(("o", "rem", "dq", "dk", "dv"), captured, eager):
            assert torch.equal(a, b), f"replay with seed {seed}: {name}"


@pytest.mark.gpu
def test_rows_that_are_not_finite_stay_where_they_are_seen():
    """What is not finite in a row reaches the keys before it or the queries behind it, up to the end of a block of 32: the rest of its document
    and the others keep the bits that they have without it, though a step's copies bring blocks that its queries cannot see."""
    from stickbreaking_attention import sb_attn_varlen
    lengths = [70, 300, 33]
    row, block, behind, end = 70 + 150, 70 + 128, 70 + 160, 70 + 300
    tensors = orc.make_inputs((2, sum(lengths), 136), 12)
    cu = cu_from_lengths(lengths, device=DEV)
    drem = torch.zeros(tensors[0].shape[:-1], dtype=torch.bfloat16)
    grads = lambda x: gradients(sb_attn_varlen, x[:3], cu, max(lengths), False, (x[3], drem))
    clean = grads(tensors)
    for which in range(4):
        x = [t.clone() for t in tensors]
        x[which][:, row] = float("inf")
        for name, got, want in zip(("dq", "dk", "dv"), grads(x), clean):
            same = lambda a, b: torch.equal(got[:, a:b], want[:, a:b])
            assert same(0, 70) and same(end, None), (which, name)
            if which in (0, 3):             # q or do: the keys behind it, and every other query
                assert same(behind, end), (which, name)
                assert name != "dq" or same(70, row) and same(row + 1, end), which
            elif name == "dq":              # k or v: the queries before it
                assert same(70, block), which
