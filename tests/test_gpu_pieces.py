"""Steps with few copies a token, of whose rows a thread of the pack moves one, two or four pieces of 16 bytes and a lane of the
gather one or two: rows that end at the edges of a wavefront's, a workgroup's and a round's pieces, against the oracle."""

from dataclasses import replace

import pytest
import torch

from a2a_cases import C1, scaled
from a2a_transport import RefConfig, check, make_ops, make_ref_rank, rows_for, run_gpu
from test_gpu_sources import run_and_check

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
BF16, F16, F32, FP8 = torch.bfloat16, torch.float16, torch.float32, torch.float8_e4m3fn

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
# top-k, ranks, experts, elements of a row, type, scales, layout of the scales, pieces: receivers of as many experts as a row
# has pieces, or a piece more
HELD = [
    (1, 3, 384, 1024, BF16, None, "row", 1),
    (1, 3, 384, 1032, BF16, None, "row", 4),
    (2, 3, 1000, 2688, FP8, 21, "col", 1),    # 168 pieces, 334 experts: by column in workgroups of their own
    (3, 2, 640, 5120, FP8, 40, "row", 1),     # 320 of each
    (4, 2, 512, 1536, BF16, None, "row", 1),
    (4, 2, 640, 2560, BF16, None, "row", 2),  # 320 of each, long copies
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


@pytest.mark.parametrize("topk,ranks,experts,hidden,dtype,scales,layout,pieces", HELD, ids=[f"k{s[0]}_h{s[3]}" for s in HELD])
def test_rows_beside_many_local_experts(topk, ranks, experts, hidden, dtype, scales, layout, pieces):
    tokens = [16384 // topk - 300, 301, 1][:ranks]
    print(f"topk={topk} experts={experts} hidden={hidden} {dtype} tokens={tokens}", flush=True)
    cfg = RefConfig("held", ranks, 1, max(tokens), experts, hidden, scales, topk, dtype, BF16, F32 if scales else None)
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


# Combines of which a wavefront moves one or two slabs of 64 pieces of a token's row: ranks, tokens, top-k, elements, type, two
GATHERS = [
    (2, 768, 1, 512, BF16, False),        # 1536 slabs: the largest step of one each
    (1, 1537, 1, 512, BF16, True),        # one more; rows that end with the first of a wavefront's two
    (3, 300, 1, 1032, BF16, True),        # three slabs, the last with one piece
    (3, 300, 2, 1528, F16, True),         # three, the last but for one piece full
    (2, 400, 2, 1024, BF16, True),        # two whole ones
    (2, 2100, 2, 516, F32, True),         # float rows, a slab and five pieces; more tokens than the sole sender's variant takes
    (2, 1100, 3, 1024, BF16, False),
]


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("ranks,tokens,topk,hidden,dtype,two", GATHERS, ids=[f"t{g[1]}_k{g[2]}_h{g[3]}" for g in GATHERS])
def test_combined_tokens(ranks, tokens, topk, hidden, dtype, two, split):
    print(f"ranks={ranks} tokens={tokens} topk={topk} hidden={hidden} {dtype} split={split}", flush=True)
    cfg = RefConfig("gather", ranks, 1, tokens, 7, hidden, None, topk, dtype, dtype, None)
    world = [make_ref_rank(cfg, r, tokens) for r in range(ranks)]
    rows = rows_for(cfg, world)
    check(cfg, world, rows, run_gpu(cfg, world, rows, DEV, split=split))


@pytest.mark.parametrize("topk", [1, 2])
@pytest.mark.parametrize("in_dtype,out_dtype", [(BF16, F32), (F32, BF16), (torch.float16, BF16)])
def test_combined_types_accumulated(topk, in_dtype, out_dtype):
    """Two slabs a wavefront onto what is there, of every width of rows and tokens; a token without copies keeps what it has."""
    ranks, tokens, hidden = 2, 900, 1048
    g = torch.Generator().manual_seed(topk)
    cfg = RefConfig("gather", ranks, 1, tokens, 6, hidden, None, topk, in_dtype, out_dtype, None)
    world = [make_ref_rank(cfg, r, tokens) for r in range(ranks)]
    rows = rows_for(cfg, world)
    ops = make_ops(cfg, DEV)
    try:
        x = [rd.dp_x.to(DEV) for rd in world]
        idx = [rd.indices.view(torch.uint32).to(DEV) for rd in world]
        w = [rd.weights.to(DEV) for rd in world]
        got_x = [torch.zeros((rows, hidden), dtype=in_dtype, device=DEV) for _ in world]
        before = [torch.randn((tokens, hidden), generator=g).to(out_dtype) for _ in world]
        out = [b.to(DEV) for b in before]
        for r in range(ranks):
            ops[r].dispatch(torch.zeros(3, dtype=torch.int32, device=DEV), got_x[r], None, x[r], None, idx[r], w[r])
        for r in range(ranks):   # (the rows come back as they went: a token's weights add up to one)
            ops[r].combine(out[r], idx[r], w[r], got_x[r], accumulate=True)
        torch.cuda.synchronize(DEV)
        assert ops[0].context.status() == 0
        ulp = 2.0 ** -8 if out_dtype == BF16 else 2.0 ** -22   # one rounding of the sum to its type
        for r in range(ranks):
            want = before[r].double() + world[r].dp_x.double()
            size = before[r].double().abs() + world[r].dp_x.double().abs()
            assert ((out[r].cpu().double() - want).abs() <= ulp * size + 1e-30).all()
    finally:
        for op in ops:
            op.destroy()
