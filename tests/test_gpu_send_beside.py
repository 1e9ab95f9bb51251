"""The send of the split calls whose routing runs in workgroups beside those that stage the rows (8193 to 65535 entries), and
the two launches that take over above and for larger steps with a gap behind the index rows: rows, scales and routing tables
against the oracle, bit for bit, at the edges of the chunks of entries, of the teams that stage rows and of both ranges."""

from dataclasses import replace

import numpy as np
import pytest
import torch

import a2a_oracle as oracle
from a2a_cases import Case, make_rank
from a2a_harness import (RouteWatch, assert_combine_close, assert_dispatch_equal, dispatch_world_with_strays, make_ops,
                         rows_needed, run_gpu, run_oracle, with_gap)
from pplx_garden_amd.native import p2p_all_to_all as native

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")

SENDS = [
    # (tokens of every rank, hidden, experts, top-k, padding, experts may repeat inside a token)
    ([1025, 0], 256, 40, 8, 1, False),              # a wavefront a row, eight rows a workgroup
    ([1792, 1793], 2048, 64, 8, 16, True),          # whole chunks of 512 entries, and one entry row more
    ([2048, 3, 1100, 0], 7168, 256, 8, 1, False),   # seven wavefronts a row; a small send beside large ones
    ([1500], 512, 1024, 6, 1, True),                # more experts than threads
    ([700, 690], 15360, 30, 12, 4, False),          # one row of fifteen wavefronts a workgroup
    ([130], 16384, 64, 64, 1, True),                # as many routes as a token can have
    ([8191], 128, 96, 8, 1, False),                 # 65528 entries: the largest step of top-8
    ([8192, 10], 128, 96, 8, 1, True),              # 65536: routing and rows in two launches
]


def check_tables(ctx, world, experts):
    for g, rd in enumerate(world):
        if not rd.indices.shape[0]:
            continue
        count, toff, eoff = oracle.route(rd.indices.numpy(), experts)
        np.testing.assert_array_equal(ctx.read_table(g, native.TABLE_NUM_ROUTED, experts).numpy(), count)
        np.testing.assert_array_equal(ctx.read_table(g, native.TABLE_EXPERT_OFFSETS, experts).numpy(), eoff)
        np.testing.assert_array_equal(ctx.read_table(g, native.TABLE_TOKEN_OFFSET, toff.size).numpy(), toff)


@pytest.mark.parametrize("tokens,hidden,experts,topk,pad,repeats", SENDS, ids=[f"{s[0]}x{s[1]}_e{s[2]}_k{s[3]}" for s in SENDS])
def test_larger_sends(tokens, hidden, experts, topk, pad, repeats):
    print(f"tokens={tokens} hidden={hidden}", flush=True)
    case = Case("send_beside", max(tokens), hidden, experts, len(tokens), topk, 777 + hidden, expert_padding=pad)
    world = [make_rank(case, r, t) for r, t in enumerate(tokens)]
    if repeats:
        for rd in world:
            rd.indices[::3, topk - 1] = rd.indices[::3, 0]
    rows = rows_needed(case, world)
    want = run_oracle(case, world, rows)
    _, ops = make_ops(case, DEV)
    try:
        routes = []
        got = run_gpu(case, world, rows, DEV, split=True, ops=ops, routes=routes)
        assert routes == [t * topk > 65535 for t in tokens if t]
        assert_dispatch_equal(case, got, want)
        assert_combine_close(case, got, want)
        check_tables(ops[0].context, world, experts)
    finally:
        for op in ops:
            op.destroy()


@pytest.mark.parametrize("bound,strided", [(0, False), (1, False), (64, False), (1199, False), (1200, False), (700, True)])
def test_bounds_and_strided_rows(bound, strided):
    """`bound` on the device, in the first chunk of entries, at a chunk's end and in the last one; with a gap behind the index
    rows the two launches serve the step."""
    case = Case("send_beside_bound", 1200, 1024, 48, 2, 8, 4141)
    N, K, E, H = case.world_size, case.topk, case.num_experts, case.hidden_dim
    world = [make_rank(case, r, 1200 if r == 0 else 5) for r in range(N)]
    rows = rows_needed(case, world)
    inputs = [oracle.RankInput(x=rd.x.view(torch.int16).numpy().view(np.uint16), indices=rd.indices.numpy(),
                               bound_m=bound if r == 0 else None) for r, rd in enumerate(world)]
    want = oracle.dispatch_world(inputs, num_experts=E, world_size=N, node_size=N, expert_padding=1, out_rows=rows, quantize=True)
    _, ops = make_ops(case, DEV)
    try:
        watch = RouteWatch(ops[0].context)      # (of rank 0's send)
        t = []
        for r, rd in enumerate(world):
            idx = rd.indices_u32.to(DEV)
            if strided:
                idx = with_gap(idx, 1)
            t.append(dict(out_expert_num_tokens=torch.zeros(case.experts_per_rank, dtype=torch.int32, device=DEV),
                          out_expert_x=torch.zeros((rows, H), dtype=torch.uint8, device=DEV).view(torch.float8_e4m3fn),
                          out_expert_x_scale=torch.zeros((rows, H // 128), device=DEV), dp_x=rd.x.to(DEV), dp_x_scale=None,
                          indices=idx, weights=rd.weights.to(DEV),
                          bound_m=torch.tensor([bound], dtype=torch.int32, device=DEV) if r == 0 else None))
        for phase in (dict(do_send=True, do_recv=False), dict(do_send=False, do_recv=True)):
            for r in range(N):
                ops[r].dispatch(**t[r], **phase)
        torch.cuda.synchronize(DEV)
        assert watch.launched() == strided
        ctx = ops[0].context
        assert ctx.status() == 0
        for r in range(N):
            np.testing.assert_array_equal(t[r]["out_expert_num_tokens"].cpu().numpy(), want[r].num_tokens)
            wr = want[r].written
            np.testing.assert_array_equal(t[r]["out_expert_x"].view(torch.uint8).cpu().numpy()[wr], want[r].x[wr])
            np.testing.assert_array_equal(t[r]["out_expert_x_scale"].cpu().numpy()[wr].view(np.uint32),
                                          want[r].x_scale[wr].view(np.uint32))
        count, toff, _ = oracle.route(world[0].indices.numpy()[:bound], E)
        np.testing.assert_array_equal(ctx.read_table(0, native.TABLE_NUM_ROUTED, E).numpy(), count)
        if bound:
            np.testing.assert_array_equal(ctx.read_table(0, native.TABLE_TOKEN_OFFSET, bound * K).numpy(), toff)
    finally:
        for op in ops:
            op.destroy()


def test_sends_in_two_launches_one_after_the_other():
    """A send in two launches adds its counts up in one of two copies of the totals on the device and clears the other one for
    the next such send, whichever rank or step that belongs to: three steps of two ranks on one context, of different sizes and
    routings, with a step in one launch a send in between."""
    case = Case("two_launch_sends", 1300, 256, 48, 2, 8, 5151, expert_padding=4)
    _, ops = make_ops(case, DEV)
    try:
        for step, (tokens, strided) in enumerate([([1200, 1300], True), ([1250, 1029], True), ([1300, 1200], False),
                                                  ([1029, 1300], True)]):
            print(f"step {step}: tokens={tokens} strided={strided}", flush=True)
            step_case = replace(case, seed=case.seed + 17 * step, num_tokens=max(tokens))
            world = [make_rank(step_case, r, t) for r, t in enumerate(tokens)]
            rows = rows_needed(step_case, world)
            want = run_oracle(step_case, world, rows)
            routes = []
            got = run_gpu(step_case, world, rows, DEV, split=True, ops=ops, strided=strided, routes=routes if step == 0 else None)
            assert routes == ([True, True] if step == 0 else [])
            assert_dispatch_equal(step_case, got, want)
            assert_combine_close(step_case, got, want)
            check_tables(ops[0].context, world, case.num_experts)
    finally:
        for op in ops:
            op.destroy()


@pytest.mark.parametrize("strided", [False, True], ids=["one_launch", "two_launches"])
def test_experts_that_are_none(strided):
    """Ids of no expert are flagged and go nowhere; all other copies, their counts and their positions are as if those were not
    there."""
    case = Case("send_beside_strays", 1300, 512, 48, 2, 8, 6161, expert_padding=4)
    N, K, E, H = case.world_size, case.topk, case.num_experts, case.hidden_dim
    world = [make_rank(case, r, t) for r, t in enumerate([1300, 1025])]
    rows = rows_needed(case, world)
    for rd in world:
        rd.indices[::5, K - 1] = E
        rd.indices[2::9, 0] = -1      # (0xFFFFFFFF)
        rd.indices[700:770] = E + 5   # whole wavefronts of them
    inputs = [oracle.RankInput(x=rd.x.view(torch.int16).numpy().view(np.uint16), indices=rd.indices.numpy().view(np.uint32))
              for rd in world]
    want, routes = dispatch_world_with_strays(inputs, num_experts=E, world_size=N, expert_padding=4, out_rows=rows, quantize=True)
    _, ops = make_ops(case, DEV)
    try:
        ctx = ops[0].context
        t = []
        for rd in world:
            idx = rd.indices_u32.to(DEV)
            t.append(dict(out_expert_num_tokens=torch.zeros(case.experts_per_rank, dtype=torch.int32, device=DEV),
                          out_expert_x=torch.full((rows, H), 0xA5, dtype=torch.uint8, device=DEV).view(torch.float8_e4m3fn),
                          out_expert_x_scale=torch.full((rows, H // 128), -7.0, device=DEV), dp_x=rd.x.to(DEV), dp_x_scale=None,
                          indices=with_gap(idx) if strided else idx, weights=rd.weights.to(DEV)))
        watch = RouteWatch(ctx)
        for phase in (dict(do_send=True, do_recv=False), dict(do_send=False, do_recv=True)):
            for r in range(N):
                ops[r].dispatch(**t[r], **phase)
        assert watch.launched() == strided
        assert ctx.status() == native.DEV_BAD_EXPERT_ID
        for r in range(N):
            wr = want[r].written
            x, s = t[r]["out_expert_x"].view(torch.uint8).cpu().numpy(), t[r]["out_expert_x_scale"].cpu().numpy()
            np.testing.assert_array_equal(t[r]["out_expert_num_tokens"].cpu().numpy(), want[r].num_tokens)
            np.testing.assert_array_equal(x[wr], want[r].x[wr])
            np.testing.assert_array_equal(s[wr].view(np.uint32), want[r].x_scale[wr].view(np.uint32))
            assert (x[~wr] == 0xA5).all() and (s[~wr] == -7.0).all()
            count, eoff, toff, _ = routes[r]
            np.testing.assert_array_equal(ctx.read_table(r, native.TABLE_NUM_ROUTED, E).numpy(), count)
            np.testing.assert_array_equal(ctx.read_table(r, native.TABLE_EXPERT_OFFSETS, E).numpy(), eoff)
            np.testing.assert_array_equal(ctx.read_table(r, native.TABLE_TOKEN_OFFSET, toff.size).numpy(), toff)
    finally:
        for op in ops:
            op.destroy()
