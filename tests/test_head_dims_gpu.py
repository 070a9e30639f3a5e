"""Every head_dim that is a multiple of 8 runs on the next wider kernel without a padded copy: both sides of
each kernel's and each instantiation's width, with NaN in the columns behind the head (which belong to
the caller) and documents at tile edges, against the oracle."""
import pytest
import torch

from oracle import sb_oracle as orc
from tests.helpers import assert_close, cu_from_lengths, oracle_varlen

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("ac", [False, True])
@pytest.mark.parametrize("d", [8, 24, 40, 72, 80, 96, 104, 136, 160, 192, 200, 248])
def test_columns_behind_the_head_are_never_read(d, ac, kernels):
    from stickbreaking_attention import sb_attn_varlen, sb_attn_varlen_fused
    lengths = [33, 1, 129, 300]
    H, T = 2, sum(lengths) + 7
    q, k, v, do = orc.make_inputs((H, T, d), 900 + d)
    drem = torch.randn((H, T), generator=torch.Generator().manual_seed(d)).to(torch.bfloat16)

    def inside_nan(t):
        wide = torch.full((H, T, d + 24), float("nan"), dtype=t.dtype, device=DEV)
        wide[..., 8:8 + d] = t.to(DEV)
        return wide[..., 8:8 + d]

    qg, kg, vg = (inside_nan(t).requires_grad_() for t in (q, k, v))
    cu = cu_from_lengths(lengths, device=DEV)
    o, rem = sb_attn_varlen(qg, kg, vg, cu, 300, zero_start=False, attend_current=ac)
    dq, dk, dv = torch.autograd.grad((o, rem), (qg, kg, vg), (inside_nan(do), drem.to(DEV)))
    f = sb_attn_varlen_fused(qg, kg, vg, cu, 300, zero_start=False, attend_current=ac)
    (fdv,) = torch.autograd.grad(f, (vg,), inside_nan(do))
    torch.cuda.synchronize()
    used = sum(lengths)
    ref = oracle_varlen(q[:, :used], k[:, :used], v[:, :used], do[:, :used], lengths, ac, drem=drem[:, :used])
    for name, g, r in zip(("o", "rem", "dq", "dk", "dv"), (o, rem, dq, dk, dv), ref):
        assert g.shape[1] == T and not g[:, used:].any()
        assert_close(f"{name} (head_dim {d})", g[:, :used], r)
    assert_close("o + rem v", f[:, :used], ref[0] + ref[1][..., None] * v[:, :used].float())
    assert torch.isfinite(fdv).all()
