"""Large steps with few copies a token, of whose rows a thread of the pack moves one, two or four pieces of 16 bytes: rows that
end at the edges of a wavefront's, a workgroup's and a round's pieces, against the oracle."""

from dataclasses import replace

import pytest
import torch

from a2a_cases import C1, scaled
from a2a_transport import RefConfig, check, make_ref_rank, rows_for, run_gpu
from test_gpu_sources import run_and_check

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
BF16, F32, FP8 = torch.bfloat16, torch.float32, torch.float8_e4m3fn

# top-k, elements of a row, type, scales, layout of the scales, pieces a thread moves
MOVED = [
    (1, 8, BF16, None, "row", 4),            # a single piece
    (1, 2048, BF16, None, "row", 4),         # 256 pieces: one wavefront, four each
    (1, 2056, BF16, None, "row", 4),         # one piece more: two wavefronts, most of the second's pieces are not there
    (1, 5120, FP8, 40, "row", 4),
    (1, 4096, FP8, 32, "col", 4),            # scales by column beside the rows
    (2, 1016, BF16, None, "row", 2),         # 127 pieces
    (2, 4100, F32, None, "row", 4),          # 1025 pieces, the shortest rows with four of them and two copies
    (3, 4096, F32, None, "row", 2),          # 1024
    (3, 6160, FP8, 55, "row", 2),            # scales that are not asked for ahead
    (4, 2944, BF16, None, "row", 2),         # six wavefronts with a piece a thread: three
    (4, 4096, BF16, None, "row", 1),         # eight
    (4, 1024, BF16, None, "row", 2),         # the shortest ones: two
    (4, 5120, FP8, 40, "col", 1),            # scales by column in workgroups of their own
    (4, 5120, FP8, 40, "row", 2),
]
# top-k, hidden size of quantised rows, pieces
QUANTISED = [(1, 128, 4), (1, 4224, 4), (2, 2176, 2), (3, 7168, 2), (4, 5120, 2), (4, 4096, 1)]


def tokens_for(topk):
    """Three sources: just over the 16384 entries (and 2048 tokens) that one launch takes."""
    first = 16384 // topk - 700
    return [first, 0, 701]


@pytest.mark.parametrize("topk,hidden,dtype,scales,layout,pieces", MOVED, ids=[f"k{s[0]}_h{s[1]}_{s[4]}" for s in MOVED])
def test_rows_moved_as_they_are(topk, hidden, dtype, scales, layout, pieces):
    tokens = tokens_for(topk)
    print(f"topk={topk} hidden={hidden} {dtype} tokens={tokens}", flush=True)
    out = BF16 if dtype == FP8 else dtype
    cfg = RefConfig("pieces", 3, 1, max(tokens), 17, hidden, scales, topk, dtype, out, F32 if scales else None, expert_padding=4)
    world = [make_ref_rank(cfg, r, t) for r, t in enumerate(tokens)]
    rows = rows_for(cfg, world)
    routes = []
    check(cfg, world, rows, run_gpu(cfg, world, rows, DEV, split=False, scale_layout=layout, routes=routes))
    assert routes == [True]


@pytest.mark.parametrize("topk,hidden,pieces", QUANTISED)
def test_quantised_rows(topk, hidden, pieces):
    tokens = tokens_for(topk)
    print(f"topk={topk} hidden={hidden} tokens={tokens}", flush=True)
    case = replace(scaled(C1, 1), world_size=3, num_experts=18, topk=topk, hidden_dim=hidden, name="pieces", num_tokens=max(tokens),
                   seed=91 + hidden)
    run_and_check(case, tokens, two_launches=True, stray=topk == 2)
