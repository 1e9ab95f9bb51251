"""Large steps of long rows without scales, whose copies are written through the L2s, and their neighbours on the other side of
each line of that rule: rows and combined tokens against the oracle."""

import pytest
import torch

from a2a_transport import RefConfig, check, make_ref_rank, rows_for, run_gpu

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
BF16, F32 = torch.bfloat16, torch.float32

# tokens, experts, top-k, hidden, type, whether they are written through: copies of 120 MB are the line.  More than 16384 copies each,
# which have a routing launch of their own and this rule behind it
STEPS = [
    ([4300, 0, 10], 24, 7, 2048, BF16, True),     # the shortest rows
    ([2900, 1], 16, 7, 3072, BF16, True),         # rows that are three quarters full: seven copies are enough
    ([3300, 1], 16, 6, 3072, BF16, False),        # six are not
    ([2900, 1], 18, 8, 3064, BF16, False),        # nor are eight of shorter ones
    ([2402, 1], 16, 7, 3568, BF16, True),         # 120.03 MB
    ([2401, 1], 16, 7, 3568, BF16, False),        # 119.98 MB
    ([2300, 500], 17, 6, 4096, BF16, True),       # an expert a receiver has not got
    ([2800, 10], 24, 6, 4088, BF16, True),        # rows that are not multiples of 2 KB: the last 4 KB nearly full
    ([1400, 1340], 32, 6, 4096, F32, True),       # 269 MB of 16 KB rows
    ([1300, 1440], 32, 6, 4352, F32, True),       # rows longer than a workgroup has threads for
    ([2799, 1], 16, 6, 5120, BF16, True),         # six copies of rows whose last 4 KB are half full: just enough
    ([2799, 1], 16, 6, 5112, BF16, False),        # and one piece less
    ([3300, 1], 12, 5, 8192, BF16, False),        # five copies a token
]
# Steps of the same sizes that one launch takes, whose stores go out at device scope always
ONE_LAUNCH = [
    ([2441, 1], 16, 6, 4096, BF16),
    ([2440, 1], 16, 6, 4096, BF16),
    ([2000, 500], 17, 6, 4096, BF16),
    ([2500, 10], 24, 6, 4088, BF16),
    ([1500, 1], 12, 5, 8192, BF16),
    ([620, 625], 32, 6, 4096, F32),
    ([560, 3], 64, 8, 7168, F32),
    ([2000, 1], 16, 6, 5120, BF16),
    ([2000, 1], 16, 6, 5112, BF16),
]


def run_and_check(tokens, experts, topk, hidden, dtype, two_launches):
    print(f"tokens={tokens} topk={topk} hidden={hidden} {dtype}", flush=True)
    cfg = RefConfig("through", len(tokens), 1, max(tokens), experts, hidden, None, topk, dtype, dtype, None, expert_padding=2)
    world = [make_ref_rank(cfg, r, t) for r, t in enumerate(tokens)]
    rows = rows_for(cfg, world)
    routes = []
    check(cfg, world, rows, run_gpu(cfg, world, rows, DEV, split=False, routes=routes))
    assert routes == [two_launches]


@pytest.mark.parametrize("tokens,experts,topk,hidden,dtype,through", STEPS, ids=[f"{s[0]}_k{s[2]}_h{s[3]}" for s in STEPS])
def test_large_steps_of_long_rows(tokens, experts, topk, hidden, dtype, through):
    run_and_check(tokens, experts, topk, hidden, dtype, two_launches=True)


@pytest.mark.parametrize("tokens,experts,topk,hidden,dtype", ONE_LAUNCH, ids=[f"{s[0]}_k{s[2]}_h{s[3]}" for s in ONE_LAUNCH])
def test_steps_of_one_launch(tokens, experts, topk, hidden, dtype):
    run_and_check(tokens, experts, topk, hidden, dtype, two_launches=False)
