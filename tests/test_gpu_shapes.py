"""Shapes off the beaten path: experts that do not divide evenly over the ranks, top-k other than 8
(including more routes than one scale-store round covers), hidden sizes that are not a multiple of a
wavefront's slab, the largest group, repeated experts inside a token."""

import pytest
import torch

from a2a_cases import Case, make_world
from a2a_harness import assert_combine_close, assert_dispatch_equal, rows_needed, run_gpu, run_oracle

pytestmark = pytest.mark.gpu

SHAPES = [
    Case("uneven_experts", 40, 256, 10, 4, 3, 7001),                       # Le = 3, last rank owns 1 expert
    Case("rank_without_experts", 24, 128, 5, 4, 2, 7002),                  # Le = 2, rank 3 owns none
    Case("top1", 33, 384, 6, 2, 1, 7003),
    Case("top12", 50, 1536, 48, 4, 12, 7004),                              # two rounds of scale stores
    Case("top64", 9, 128, 64, 2, 64, 7005),                                # every expert, K = 64
    Case("hidden_128", 70, 128, 16, 4, 4, 7006),                           # one scale group per token
    Case("hidden_9216", 20, 9216, 32, 4, 8, 7007, outliers=True),          # 9 slabs
    Case("world_32", 64, 256, 64, 32, 4, 7008, expert_padding=8, node_size=8),
    Case("world_1", 100, 512, 7, 1, 3, 7009, expert_padding=16),
    Case("several_chunks", 700, 256, 24, 4, 8, 7010, routing="zipf", zipf_s=1.5),   # 5600 entries: 6 chunks
    Case("many_chunks", 600, 128, 64, 2, 64, 7012),                        # 38 400 entries of one source: 38 chunks
    Case("wide_ranks", 900, 128, 90, 2, 8, 7013, expert_padding=4),        # Le = 45 experts per rank, two-launch dispatch
    Case("largest_group", 400, 128, 1024, 32, 6, 7014, expert_padding=128, node_size=16),   # 32 ranks x 1024 experts
]


@pytest.mark.parametrize("split", [False, True], ids=["group", "split"])
@pytest.mark.parametrize("case", SHAPES, ids=lambda c: c.name)
def test_shapes(case, split):
    print(f"case={case.name} split={split}", flush=True)
    device = torch.device("cuda:0")
    world = make_world(case, "ragged" if case.world_size > 1 else "all")
    rows = rows_needed(case, world)
    want = run_oracle(case, world, rows)
    got = run_gpu(case, world, rows, device, split=split)
    assert_dispatch_equal(case, got, want)
    assert_combine_close(case, got, want)


@pytest.mark.parametrize("split", [False, True], ids=["group", "split"])
def test_repeated_experts_inside_a_token(split):
    """The kernels do not require the K experts of a token to be distinct
    (a2a_dispatch_send.cu:183-190 counts entries, not tokens)."""
    case = Case("repeats", 37, 256, 6, 2, 4, 7011)
    world = make_world(case, "all")
    gen = torch.Generator().manual_seed(5)
    for rd in world:
        rd.indices.copy_(torch.randint(0, case.num_experts, rd.indices.shape, generator=gen, dtype=torch.int32))
    rows = rows_needed(case, world)
    want = run_oracle(case, world, rows)
    got = run_gpu(case, world, rows, torch.device("cuda:0"), split=split)
    assert_dispatch_equal(case, got, want)
    assert_combine_close(case, got, want)


# The combine loads its rows in groups of 1, 2, 4 or 8 (the smallest that holds K, then groups of 8), 64 chunks of
# 16 bytes per wavefront, with at most 32768 tokens to a layer of its grid.
GATHERS = [
    Case("k1", 70, 640, 8, 2, 1, 7101),
    Case("k2", 70, 1152, 8, 2, 2, 7102),
    Case("k3", 70, 512, 12, 4, 3, 7103),
    Case("k5", 70, 128, 12, 4, 5, 7104),
    Case("k7", 70, 640, 16, 4, 7, 7105),
    Case("k9", 70, 512, 16, 4, 9, 7106),
    Case("k16", 40, 640, 32, 4, 16, 7107),
    Case("second_layer", 16500, 128, 16, 2, 2, 7108),        # 33000 tokens of two ranks
    Case("uneven_layers", 16385, 128, 16, 4, 2, 7109),       # 65540 tokens in three layers, one place empty
]


@pytest.mark.parametrize("case", GATHERS, ids=lambda c: c.name)
def test_gather_groups(case):
    world = make_world(case, "all")
    rows = rows_needed(case, world)
    want = run_oracle(case, world, rows)
    got = run_gpu(case, world, rows, torch.device("cuda:0"), split=False)
    assert_combine_close(case, got, want)


# Steps whose copies go past the Infinity Cache (from 320 MB on; not two copies or fewer of rows that are not quantised),
# and whose combined tokens go past it with them or, from 84 MB on, by themselves, at row lengths that end inside a
# wavefront's slab: the group calls against the split calls, which move every row by other kernels.
# (row type, hidden, scales, experts per token, tokens of the first and third of three ranks, copies go past the cache)
STREAMED = [
    (torch.bfloat16, 1000, 0, 5, (30000, 2200), True),        # 322 MB of copies, 64 MB of tokens
    (torch.float16, 1000, 0, 3, (52000, 3001), True),         # 330 MB, 110 MB
    (torch.float32, 1004, 0, 8, (9700, 301), True),           # 321 MB, 40 MB
    (torch.float8_e4m3fn, 1152, 9, 8, (33000, 1900), True),   # 322 MB, 80 MB
    (torch.bfloat16, 1000, 0, 9, (17000, 1000), True),        # 324 MB, 36 MB: two groups of rows a token
    (torch.float32, 1004, 0, 40, (2000, 0), True),            # 321 MB, 8 MB: one sender, few enough tokens for its own gather
    (torch.bfloat16, 1000, 0, 2, (80000, 2100), False),       # 328 MB of copies that do not (two pieces a thread), 164 MB
    (torch.bfloat16, 1000, 0, 5, (29000, 2000), False),       # 310 MB, 62 MB
]


def copies_of(row, hidden, k, tokens):
    return sum(tokens) * k * hidden * row.itemsize


# The same of quantised rows, of which a thread moves several pieces: hidden, experts per token, tokens, pieces
STREAMED_QUANTISED = [
    (4224, 1, (70000, 6000), 4),      # 321 MB: 264 pieces of a row, the last of four rounds nearly empty
    (7296, 2, (20000, 2100), 2),      # 322 MB: 456
    (2176, 3, (45000, 4100), 2),      # 321 MB: 136
    (4224, 4, (17000, 2000), 2),      # 321 MB: five wavefronts with a piece a thread, three here
]


@pytest.mark.parametrize("row,hidden,scales,k,tokens,streamed", STREAMED,
                         ids=lambda v: str(v).replace("torch.", "") if isinstance(v, torch.dtype) else None)
def test_streamed_copies_and_tokens(row, hidden, scales, k, tokens, streamed):
    group_and_split_calls_agree(row, hidden, scales, k, tokens)


@pytest.mark.parametrize("hidden,k,tokens,pieces", STREAMED_QUANTISED)
def test_streamed_quantised_rows(hidden, k, tokens, pieces):
    group_and_split_calls_agree(torch.float8_e4m3fn, hidden, hidden // 128, k, tokens, quantise=True)


def group_and_split_calls_agree(row, hidden, scales, k, tokens, quantise=False):
    from pplx_garden_amd.distributed.loopback import LoopbackWorld
    from pplx_garden_amd.kernels.p2p_all_to_all import P2PAllToAll

    print(f"{row} hidden={hidden} k={k} tokens={tokens} quantise={quantise}", flush=True)
    device, N, E = torch.device("cuda:0"), 3, max(24, k + 2)
    out = torch.bfloat16 if scales else row
    world = LoopbackWorld(N, device=device)
    counts = (tokens[0], 0, tokens[1])
    rows = sum(counts) * k
    ops = [P2PAllToAll(max_num_tokens=max(counts), num_experts=E, expert_padding=1, hidden_dim=hidden,
                       hidden_dim_scale=scales or None, in_dtype=row, out_dtype=out,
                       scale_dtype=torch.float32 if scales else None, num_experts_per_token=k, device=device,
                       global_group=world.group(r)) for r in range(N)]
    gen = torch.Generator(device=device).manual_seed(hidden * k)
    data = []
    for t in counts:
        data.append(dict(
            dp_x=torch.randn((t, hidden), generator=gen, device=device).to(torch.bfloat16 if quantise else row),
            dp_x_scale=torch.rand((t, scales), generator=gen, device=device) if scales and not quantise else None,
            indices=torch.rand((t, E), generator=gen, device=device).topk(k).indices.to(torch.int32).view(torch.uint32),
            weights=torch.rand((t, k), generator=gen, device=device)))
    expert_y = [torch.randn((rows, hidden), generator=gen, device=device).to(out) for _ in range(N)]
    results = []
    for halves in ([dict()], [dict(do_recv=False), dict(do_send=False)]):
        got = [dict(out_expert_num_tokens=torch.zeros(-(-E // N), dtype=torch.int32, device=device),
                    out_expert_x=torch.zeros((rows, hidden), dtype=torch.uint8 if scales else row, device=device).view(row),
                    out_expert_x_scale=torch.zeros((rows, scales), device=device) if scales else None) for _ in range(N)]
        combined = [torch.full((t, hidden), 0.5, dtype=out, device=device) for t in counts]
        for half in halves:
            for r in range(N):
                ops[r].dispatch(**got[r], **data[r], **half)
        for half in halves:
            for r in range(N):
                ops[r].combine(out_tokens=combined[r], indices=data[r]["indices"], weights=data[r]["weights"],
                               expert_y=expert_y[r], accumulate=True, **half)
        torch.cuda.synchronize()
        assert ops[0].context.status() == 0
        results.append([g[n] for g in got for n in g if g[n] is not None] + combined)
    assert sum(int(n.sum()) for n in results[0] if n.dtype == torch.int32) == rows
    for a, b in zip(*results):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
    for op in ops:
        op.destroy()
