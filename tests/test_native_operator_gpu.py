"""The eager operators run through a C++ autograd node (csrc/sba_torch.cpp); the autograd functions in
Python remain for tracing and graph capture.  Both call the same kernels: same bits, whatever the
element type, layout, padding and the set of inputs that want a gradient."""
import pytest
import torch

from tests.helpers import cu_from_lengths

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _inputs(shape, dtype, tokens_first, seed):
    g = torch.Generator().manual_seed(seed)
    def one(s):
        t = torch.randn(s, generator=g)
        if tokens_first:
            t = t.transpose(-3, -2).contiguous().transpose(-3, -2)
        return t.to(dtype).to(DEV)
    q, k, v, do = (one(shape) for _ in range(4))
    return q, k, v, do, torch.randn(shape[:-1], generator=g).to(dtype).to(DEV)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("d,tokens_first,wanted", [(64, False, "qkv"), (128, True, "v"), (50, True, "qkv"), (96, False, "qk")])
@pytest.mark.parametrize("fixed", [False, True])
@pytest.mark.filterwarnings("ignore::UserWarning")
def test_native_operator_equals_the_python_autograd_function(dtype, d, tokens_first, wanted, fixed):
    from stickbreaking_attention import sb_attn, sb_attn_fused, sb_attn_varlen, sb_attn_varlen_fused
    import sys
    mod_fixed, mod_varlen = (sys.modules["stickbreaking_attention." + n] for n in ("sb_attn", "sb_varlen"))
    lengths = [70, 1, 200]
    shape = (2, 3, 130, d) if fixed else (3, sum(lengths) + 3, d)
    base = _inputs(shape, dtype, tokens_first, d)
    cu = cu_from_lengths(lengths, device=DEV)
    scale = d ** -0.5

    def both_outputs(native):
        if native:
            return sb_attn(q, k, v) if fixed else sb_attn_varlen(q, k, v, cu, 200, zero_start=False)
        return (mod_fixed.StickBreakingAttention.apply(q, k, v, scale, False) if fixed
                else mod_varlen.StickBreakingAttention.apply(q, k, v, cu, 200, scale, False))

    def fused_output(native):
        if native:
            return sb_attn_fused(q, k, v) if fixed else sb_attn_varlen_fused(q, k, v, cu, 200, zero_start=False)
        return (mod_fixed.StickBreakingAttentionFused.apply(q, k, v, scale, False) if fixed
                else mod_varlen.StickBreakingAttentionFused.apply(q, k, v, cu, 200, scale, False))

    results = []
    for native in (True, False):
        q, k, v = (t.clone().requires_grad_(n in wanted) for t, n in zip(base, "qkv"))
        inputs = [t for t in (q, k, v) if t.requires_grad]
        o, rem = both_outputs(native)
        out = [o, rem] + list(torch.autograd.grad((o, rem), inputs, base[3:]))
        f = fused_output(native)
        out += [f] + list(torch.autograd.grad(f, inputs, base[3]))
        results.append(out)
    for a, b in zip(*results):
        assert a.dtype == b.dtype and a.stride() == b.stride() and torch.equal(a, b)


def test_native_backward_from_several_threads_on_their_own_streams():
    """One gradient table per stream, and a backward's two kernels are enqueued without another thread's between."""
    import threading
    from stickbreaking_attention import sb_attn
    base = [t.to(DEV) for t in _inputs((1, 4, 700, 64), torch.bfloat16, False, 5)[:4]]

    def grads():
        q, k, v = (t.detach().clone().requires_grad_() for t in base[:3])
        return torch.autograd.grad(sb_attn(q, k, v)[0], (q, k, v), base[3])

    ref = grads()
    torch.cuda.synchronize()
    bad = []

    def work(own_stream):
        with torch.cuda.stream(torch.cuda.Stream() if own_stream else torch.cuda.default_stream()):
            for _ in range(20):
                got = grads()
                torch.cuda.current_stream().synchronize()
                if not all(torch.equal(a, b) for a, b in zip(got, ref)):
                    bad.append(own_stream)
                    return

    threads = [threading.Thread(target=work, args=(i < 2,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not bad
