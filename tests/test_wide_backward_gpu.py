"""The two passes of the backward at head_dim 129 .. 256 where its step structure can go wrong: documents that end on either side of their 64-key and 128-query tiles,
32-query steps and four ring slots, columns that end inside a product wave's half; and rows that are not finite."""
import pytest
import torch

from oracle import sb_oracle as orc
from tests.helpers import assert_close, cu_from_lengths, oracle_varlen
from tests.test_head_dim_256_gpu import DEV, _need_gpu, _run  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("product_space", [False, True])
@pytest.mark.parametrize("ac", [False, True])
@pytest.mark.parametrize("d,lengths", [(256, [1, 31, 32, 33, 63, 64, 65]), (192, [95, 97, 127, 129]), (136, [160, 161, 1, 193]),
                                       (200, [225, 255, 257]), (256, [384, 385, 7])])
def test_edges(d, lengths, ac, product_space, monkeypatch):
    from stickbreaking_attention import _ops
    monkeypatch.setattr(_ops, "PRODUCT_SPACE", product_space)
    T = sum(lengths)
    q, k, v, do = orc.make_inputs((2, T, d), d + T)
    drem = torch.randn((2, T), generator=torch.Generator().manual_seed(d)).to(torch.bfloat16)
    ref = oracle_varlen(q, k, v, do, lengths, ac, drem=drem)
    for name, g, r in zip(("o", "rem", "dq", "dk", "dv"), _run(q, k, v, do, lengths, ac, drem=drem), ref):
        assert_close(name, g, r)


@pytest.mark.parametrize("ac", [False, True])
def test_rows_that_are_not_finite_stay_behind_the_blocks_that_hide_them(ac):
    lengths = [300, 77]
    T = sum(lengths)
    tensors = orc.make_inputs((2, T, 256), 9)
    _, _, clean_dq, *clean = _run(*tensors, lengths, ac)
    for at in (3, 40, 64, 100, 200, 299, 333):
        start, length = (0, 300) if at < 300 else (300, 77)
        block = start + (at - start) // 32 * 32
        newer = [i for i in range(T) if i < start or i >= min(block + 32, start + length)]
        for which in (0, 3):
            x = [t.clone() for t in tensors]
            x[which][:, at] = float("inf")
            for got, want in zip(_run(*x, lengths, ac)[3:], clean):
                assert torch.equal(got[:, newer], want[:, newer]), (at, which)
        for which in (1, 2):          # a key: queries ahead of its block
            x = [t.clone() for t in tensors]
            x[which][:, at] = float("inf")
            dq = _run(*x, lengths, ac)[2]
            assert torch.equal(dq[:, :block], clean_dq[:, :block]), (at, which)
