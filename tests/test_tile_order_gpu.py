"""In which order the query tiles of packed documents are listed, and which of them a workgroup of the forward takes."""
import random

import pytest
import torch

from stickbreaking_attention import _native as nat
from stickbreaking_attention import _ops, sb_attn_varlen
from tests import helpers
from tests.test_schedule_gpu import DEV, _schedule

pytestmark = pytest.mark.gpu
CLASS_TILES = 4
PER_CU = {32: 6, 64: 4, 128: 3, 256: 2}      # workgroups of the general forward that a compute unit holds


def _listed(lengths):
    """(length, tile) in the order of the list: classes of documents of more than three quarters of the tiles of their longest, a class tile-major;
    documents of less than CLASS_TILES tiles one by one, and those of a class of more documents than its longest has tiles."""
    lengths = sorted(lengths, reverse=True)
    tiles = [-(-n // 128) for n in lengths]
    out, r = [], 0
    while r < len(tiles):
        end = r + 1
        while tiles[r] >= CLASS_TILES and end < len(tiles) and 4 * tiles[end] > 3 * tiles[r] and tiles[end] >= CLASS_TILES:
            end += 1
        if end - r > tiles[r]:
            out += [(lengths[x], i) for x in range(r, end) for i in range(tiles[x] - 1, -1, -1)]
        else:
            for i in range(tiles[r] - 1, -1, -1):
                out += [(lengths[x], i) for x in range(r, end) if tiles[x] > i]
        r = end
    return out


@pytest.mark.parametrize("lengths", [[640] * 5 + [500] * 5, [640] * 6 + [512], [1024, 1000, 769, 768, 767, 500], [512], [385, 384, 383, 1], [4096] * 4, [100] * 30, [0, 1024, 513, 512, 511, 0, 128, 129],
                                     [2048, 1025, 1024, 897, 896, 600, 512, 385, 384, 300, 7],
                                     [random.Random(5).randint(1, 3000) for _ in range(40)],
                                     [random.Random(6).choice([200, 400, 500, 900]) for _ in range(600)]])
def test_order_of_the_list(lengths):
    _, q_tiles, _, _ = _schedule(lengths, sum(lengths), heads=1)
    assert [(t[1], t[2]) for t in q_tiles] == _listed(lengths)


@pytest.mark.parametrize("head_dim", list(PER_CU))
@pytest.mark.parametrize("lengths", [[4096] * 4, [1024, 1000, 769, 768, 767, 500], [32768] * 16])
def test_long_launches_are_listed_document_by_document(head_dim, lengths):
    """Beyond four rounds of the chip, or beyond 48 for rounds x heads where that is more, the tiles of a document follow one another."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    rounds = lambda heads: sum(lengths) // 128 * heads / (PER_CU[head_dim] * cus)
    most = max(h for h in range(1, 400) if rounds(h) <= 4 or rounds(h) * h <= 48)
    assert (rounds(most) > 4) == (len(lengths) == 16)
    by_document = [(n, i) for n in sorted(lengths, reverse=True) for i in range(-(-n // 128) - 1, -1, -1)]
    assert by_document != _listed(lengths)
    for heads, want in ((most, _listed(lengths)), (most + 1, by_document)):
        _, q_tiles, _, _ = _schedule(lengths, sum(lengths), heads=heads, head_dim=head_dim)
        assert [(t[1], t[2]) for t in q_tiles] == want


@pytest.mark.parametrize("heads,head_dim,lengths", [(12, 64, [1500, 700, 129, 2100]), (20, 32, [3000, 1, 1111]), (7, 128, [4096, 900]),
                                                    (3, 64, [97] * 200), (9, 256, [1500, 700, 129, 2100]), (31, 64, [4096, 61])])
def test_a_launch_dealt_in_turns_covers_every_tile(heads, head_dim, lengths, monkeypatch):
    """More items than compute units, all on the chip at once: the same bits as head by head, which is dealt straight."""
    monkeypatch.setattr(_ops, "FORWARD_FLAGS", nat.FLAG_GENERAL_FORWARD)
    gen = torch.Generator(device=DEV).manual_seed(3)
    q, k, v = (torch.randn(heads, sum(lengths), head_dim, generator=gen, device=DEV).to(torch.bfloat16) for _ in range(3))
    cu = helpers.cu_from_lengths(lengths, device=DEV)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert cus < sum(lengths) // 128 * heads <= PER_CU[head_dim] * cus and sum(lengths) // 128 <= cus     # (what the rule goes by)
    o, rem = sb_attn_varlen(q, k, v, cu, max(lengths), zero_start=False)
    for h in range(heads):
        o1, rem1 = sb_attn_varlen(q[h:h + 1], k[h:h + 1], v[h:h + 1], cu, max(lengths), zero_start=False)
        assert torch.equal(o[h], o1[0]) and torch.equal(rem[h], rem1[0])
