"""Scales of the steps that are routed in a launch of their own (more than 16384 entries), the caller's, by row and by column,
and those of quantised rows, and of the recvs that copy by pieces of rows: at the sizes where their stores and loads change,
against the oracle bit for bit."""

from dataclasses import replace

import pytest
import torch

from a2a_cases import C1, scaled
from a2a_transport import RefConfig, check, make_ref_rank, rows_for, run_gpu
from test_gpu_sources import run_and_check

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
BF16, F32, FP8 = torch.bfloat16, torch.float32, torch.float8_e4m3fn

# tokens, world, experts, top-k, hidden, scales
GIVEN = [
    ([2100, 0], 64, 8, 3968, 31),             # below a cache line of scales
    ([2100, 1], 64, 8, 4096, 32),             # a cache line
    ([1500, 0, 700, 33], 128, 8, 6144, 48),   # the widest row whose scales are asked for ahead of it
    ([2100, 17], 33, 8, 6160, 55),            # the next wider one; an expert a receiver has not got
    ([1300, 1400], 24, 7, 256, 128),          # more scales than the row has threads
]


@pytest.mark.parametrize("layout", ["row", "col"])
@pytest.mark.parametrize("tokens,experts,topk,hidden,scales", GIVEN, ids=[f"{s[0]}_h{s[3]}_s{s[4]}" for s in GIVEN])
def test_given_scales(tokens, experts, topk, hidden, scales, layout):
    print(f"tokens={tokens} hidden={hidden} scales={scales} {layout}", flush=True)
    cfg = RefConfig("scales", len(tokens), 1, max(tokens), experts, hidden, scales, topk, FP8, BF16, F32, expert_padding=16)
    world = [make_ref_rank(cfg, r, t) for r, t in enumerate(tokens)]
    rows = rows_for(cfg, world)
    check(cfg, world, rows, run_gpu(cfg, world, rows, DEV, split=False, scale_layout=layout))


@pytest.mark.parametrize("hidden", [3968, 4096])
def test_quantised_rows(hidden):
    case = replace(scaled(C1, 1), hidden_dim=hidden, name="scales", num_tokens=2100, seed=77 + hidden)
    print(f"hidden={hidden}", flush=True)
    run_and_check(case, [2100, 0, 1, 0, 50, 0, 0, 3])


# tokens, experts, top-k, hidden, scales
RECEIVED = [
    ([300, 0], 64, 8, 2560, 20),              # few words: they travel with the rows
    ([3584, 3584], 16, 8, 512, 4),            # the smallest step whose columns have workgroups of their own
    ([3583, 3584], 16, 8, 512, 4),            # a word below it
    ([701, 3, 2650], 9, 8, 3968, 31),         # a last slice of seven columns, a last block of some rows
    ([1, 900, 900, 0], 4, 4, 4352, 136),      # one expert a rank
]


@pytest.mark.parametrize("tokens,experts,topk,hidden,scales", RECEIVED, ids=[f"{s[0]}_h{s[3]}_s{s[4]}" for s in RECEIVED])
def test_received_columns(tokens, experts, topk, hidden, scales):
    print(f"tokens={tokens} hidden={hidden} scales={scales}", flush=True)
    cfg = RefConfig("columns", len(tokens), 1, max(tokens), experts, hidden, scales, topk, FP8, BF16, F32, expert_padding=4)
    world = [make_ref_rank(cfg, r, t) for r, t in enumerate(tokens)]
    rows = rows_for(cfg, world)
    check(cfg, world, rows, run_gpu(cfg, world, rows, DEV, split=True, scale_layout="col"))
