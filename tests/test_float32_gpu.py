"""float32 callers: operands rounded in one launch, results written as float32 by the kernels (SBA_F32_OUT).  They are
what the bfloat16 operator gives on the rounded operands, bit for bit, through every kernel that stores an output, for both token layouts, dense and sliced operands and a head_dim that still has to be padded."""
import warnings

import pytest
import torch

from oracle import sb_oracle as orc
from tests.helpers import cu_from_lengths

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("layout", ["heads", "tokens", "slices"])
@pytest.mark.parametrize("form,d", [(1, 32), (1, 64), (1, 104), (1, 128), (1, 200), (2, 64), (2, 128), (3, 64), (3, 24), (0, 20)])
def test_results_are_the_bfloat16_ones(form, d, layout):
    from stickbreaking_attention import _native, sb_attn_varlen, sb_attn_varlen_fused
    lengths = [33, 1, 129, 700]
    H, T = 3, sum(lengths) + 11
    cu = cu_from_lengths(lengths, device=DEV)
    values = [t.float() + 1e-3 * t.float().cos() for t in orc.make_inputs((H, T, d), 70 + d)]
    drem = torch.randn((H, T), generator=torch.Generator().manual_seed(d))

    def placed(t):
        if layout == "tokens":
            return t.transpose(0, 1).contiguous().to(DEV).transpose(0, 1)
        if layout == "slices":
            wide = torch.zeros((H, T, d + 8), dtype=t.dtype, device=DEV)
            wide[..., :d] = t.to(DEV)
            return wide[..., :d]
        return t.to(DEV)

    lib = _native.load()
    lib.sba_set_backward_form(form)
    try:
        got = {}
        for dt in (torch.float32, torch.bfloat16):
            q, k, v, do = (placed(t.to(dt)) for t in values)
            dr = drem.to(dt).to(DEV)
            for t in (q, k, v):
                t.requires_grad_()
            with warnings.catch_warnings():
                warnings.simplefilter("ignore")
                o, rem = sb_attn_varlen(q, k, v, cu, 700, zero_start=False)
                f = sb_attn_varlen_fused(q, k, v, cu, 700, zero_start=False)
            got[dt] = (o, rem) + torch.autograd.grad((o, rem), (q, k, v), (do, dr)) + (f,) + torch.autograd.grad(f, (q, k, v), do)
    finally:
        lib.sba_set_backward_form(0)
    names = ("o", "rem", "dq", "dk", "dv", "o + rem v", "its dq", "its dk", "its dv")
    for name, a, b in zip(names, got[torch.float32], got[torch.bfloat16]):
        assert a.dtype == torch.float32 and not a[:, sum(lengths):].any()
        assert torch.equal(a, b.float()), name
