"""Split steps whose kernels find their buffers and tables in a few packed words: the largest sizes that the words hold, tables at
their furthest distances, receivers without experts, every number of routes a group of loads is made for and its neighbours,
against the oracle."""

import pytest
import torch

from a2a_transport import RefConfig, check, make_ref_rank, rows_for, run_gpu

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
BF16, F16, F32, FP8 = torch.bfloat16, torch.float16, torch.float32, torch.float8_e4m3fn

# ranks, tokens, experts, elements of a row, scales, routes a token, types of rows and tokens, layout of the scales
STEPS = [
    (32, 3, 1024, 3840, None, 8, F32, F32, "row"),       # 960 pieces of a row, 1024 experts, tables of 32 senders
    (31, 2, 1023, 15360, 120, 64, FP8, BF16, "row"),     # 64 routes, a row of 960 pieces of one byte an element
    (16, 5, 17, 8, None, 1, BF16, BF16, "row"),          # a piece a row; seven receivers without experts
    (2, 33, 1024, 1024, 8, 2, FP8, F16, "col"),          # 512 experts a receiver
    (1, 70, 1024, 1024, 8, 3, FP8, BF16, "row"),         # all of them
    (4, 64, 12, 520, None, 4, F16, F16, "row"),
    (4, 64, 12, 520, None, 5, F16, BF16, "row"),
    (3, 50, 30, 240, 3, 9, FP8, F32, "row"),             # a group of loads and one more
    (2, 2049, 16, 256, None, 7, BF16, F16, "row"),       # more tokens than the gather leaves unbounded
    (3, 700, 64, 2048, 16, 8, FP8, BF16, "col"),         # scales by column in workgroups of their own
]


@pytest.mark.parametrize("ranks,tokens,experts,hidden,scales,topk,rows_type,out_type,layout", STEPS)
def test_split_steps(ranks, tokens, experts, hidden, scales, topk, rows_type, out_type, layout):
    print(f"ranks={ranks} tokens={tokens} experts={experts} hidden={hidden} topk={topk} {rows_type} {out_type}", flush=True)
    cfg = RefConfig("short", ranks, 1, tokens, experts, hidden, scales, topk, rows_type, out_type, F32 if scales else None,
                    expert_padding=3)
    world = [make_ref_rank(cfg, r, tokens if r % 3 != 1 else tokens // 2) for r in range(ranks)]
    rows = rows_for(cfg, world)
    check(cfg, world, rows, run_gpu(cfg, world, rows, DEV, split=True, scale_layout=layout))
