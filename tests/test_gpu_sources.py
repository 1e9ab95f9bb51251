"""The one-launch dispatch of steps of several sources (and of larger steps of one) against the oracle, bit for bit: rows,
scales, counts and every routing table of every source, at the sizes where its divisions of the work can go wrong; and steps
beyond its limits, which have a routing launch of their own."""

from dataclasses import replace

import numpy as np
import pytest
import torch

import a2a_oracle as oracle
from a2a_cases import C1, bf16_codes, make_rank, scaled
from a2a_harness import SENTINEL, RouteWatch, dispatch_world_with_strays, make_ops, rows_needed, with_gap
from a2a_transport import RefConfig, check, make_ref_rank, rows_for, run_gpu
from pplx_garden_amd.native import p2p_all_to_all as native

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def run_and_check(case, tokens, bounds=None, repeats=False, strided=False, stray=False, two_launches=False):
    """One dispatch of `tokens[r]` tokens of every rank; `repeats`: every third token names its first expert twice;
    `strided`: index rows with a gap behind them (another kernel's step, the same result); `stray`: some tokens of every
    source, its first and whole wavefronts of the larger ones among them, name experts that do not exist (flagged, all other
    copies are sent as if those were not there); `two_launches`: the step has a routing launch of its own."""
    N, Le, H, Hs, K, E = (case.world_size, case.experts_per_rank, case.hidden_dim, case.hidden_dim_scale, case.topk,
                          case.num_experts)
    bounds = bounds or [None] * N
    world = [make_rank(case, r, t) for r, t in enumerate(tokens)]
    if repeats:
        for rd in world:
            rd.indices[::3, K - 1] = rd.indices[::3, 0]
    rows = rows_needed(case, world)
    if stray:
        for rd in world:
            rd.indices[::5, K - 1] = E + 3
            rd.indices[1::7, 0] = -1          # (0xFFFFFFFF)
            rd.indices[20:40] = E             # whole wavefronts of them
    inputs = [oracle.RankInput(x=bf16_codes(rd.x), indices=rd.indices.numpy().view(np.uint32), bound_m=b)
              for rd, b in zip(world, bounds)]
    if stray:
        want, routes = dispatch_world_with_strays(inputs, num_experts=E, world_size=N, expert_padding=case.expert_padding,
                                                  out_rows=rows, quantize=True)
    else:
        want = oracle.dispatch_world(inputs, num_experts=E, world_size=N, node_size=case.node_size or N,
                                     expert_padding=case.expert_padding, out_rows=rows, quantize=True)
        routes = []
        for r, rd in enumerate(world):
            n_eff = tokens[r] if bounds[r] is None else bounds[r]
            count, toff, eoff = oracle.route(rd.indices.numpy()[:n_eff], E)
            routes.append((count, eoff, toff, want[0].slots[r][:n_eff].reshape(-1)))
    _, ops = make_ops(case, DEV, max_num_tokens=max(tokens))
    try:
        t = []
        for r, rd in enumerate(world):
            idx = rd.indices_u32.to(DEV)
            t.append(dict(x=rd.x.to(DEV), idx=with_gap(idx) if strided else idx, w=rd.weights.to(DEV),
                          b=None if bounds[r] is None else torch.tensor([bounds[r]], dtype=torch.int32, device=DEV),
                          n=torch.full((Le,), -1, dtype=torch.int32, device=DEV),
                          ox=torch.full((rows, H), SENTINEL, dtype=torch.uint8, device=DEV).view(torch.float8_e4m3fn),
                          os=torch.full((rows, Hs), -7.0, dtype=torch.float32, device=DEV)))
        ctx = ops[0].context
        watch = RouteWatch(ctx)
        for r in range(N):
            ops[r].dispatch(out_expert_num_tokens=t[r]["n"], out_expert_x=t[r]["ox"], out_expert_x_scale=t[r]["os"],
                            dp_x=t[r]["x"], dp_x_scale=None, indices=t[r]["idx"], weights=t[r]["w"], bound_m=t[r]["b"])
        assert watch.launched() == two_launches
        assert ctx.status() == (native.DEV_BAD_EXPERT_ID if stray else 0)
        for r in range(N):
            n_local = max(0, min(Le, E - r * Le))
            np.testing.assert_array_equal(t[r]["n"].cpu().numpy()[:n_local], want[r].num_tokens[:n_local])
            assert (t[r]["n"].cpu().numpy()[n_local:] == -1).all()
            wr = want[r].written
            got_x, got_s = t[r]["ox"].view(torch.uint8).cpu().numpy(), t[r]["os"].cpu().numpy()
            np.testing.assert_array_equal(got_x[wr], want[r].x[wr])
            np.testing.assert_array_equal(got_s[wr].view(np.uint32), want[r].x_scale[wr].view(np.uint32))
            assert (got_x[~wr] == SENTINEL).all() and (got_s[~wr] == -7.0).all()
            count, eoff, toff, slots = routes[r]
            np.testing.assert_array_equal(ctx.read_table(r, native.TABLE_NUM_ROUTED, E).numpy(), count)
            np.testing.assert_array_equal(ctx.read_table(r, native.TABLE_EXPERT_OFFSETS, E).numpy(), eoff)
            if toff.size:
                np.testing.assert_array_equal(ctx.read_table(r, native.TABLE_TOKEN_OFFSET, toff.size).numpy(), toff)
                np.testing.assert_array_equal(ctx.read_table(r, native.TABLE_SLOT, toff.size).numpy().astype(np.uint32),
                                              slots.reshape(-1).astype(np.uint32))     # (-1: nowhere)
    finally:
        for op in ops:
            op.destroy()


BASE = scaled(C1, 1)     # 128 experts over 8 ranks, top-8, hidden 2048

STEPS = {
    "one_token_a_rank": (BASE, [1] * 8, {}),
    "one_token_of_two": (BASE, [0, 0, 1, 0, 0, 0, 1, 0], {}),
    "first_and_last_empty": (BASE, [0, 5, 0, 0, 17, 3, 0, 0], {}),
    "256_tokens_a_workgroup_each": (BASE, [32] * 8, {}),
    "257_tokens_two_a_workgroup": (BASE, [33] + [32] * 7, {}),
    "ragged_7168_pad16_two_nodes": (replace(BASE, hidden_dim=7168, expert_padding=16, node_size=4),
                                    [128, 0, 43, 1, 128, 0, 43, 1], {}),
    "65_and_64_entries_a_source": (replace(BASE, topk=1), [64, 65, 63, 0, 256, 257, 255, 1], {}),
    "top7_odd_experts_repeats": (replace(BASE, topk=7, num_experts=125), [100, 3, 77, 0, 41, 99, 1, 60], dict(repeats=True)),
    "top3_bounds": (replace(BASE, topk=3), [70, 40, 0, 9, 70, 1, 2, 55], dict(bounds=[None, 0, None, 5, 69, None, 1, 55])),
    "1024_tokens": (replace(BASE, hidden_dim=7168, num_experts=256), [128] * 8, {}),
    "2048_tokens_eight_a_workgroup": (replace(BASE, hidden_dim=7168, expert_padding=128), [250, 256, 262, 256, 256, 255, 257, 256], {}),
    "2049_tokens_the_two_launches": (BASE, [257] + [256] * 7, dict(two_launches=True)),
    "2048_tokens_of_one": (BASE, [0, 0, 0, 2048, 0, 0, 0, 0], dict(repeats=True)),
    "2048_short_rows_of_one_the_two_launches": (replace(BASE, hidden_dim=1024), [0, 0, 0, 2048, 0, 0, 0, 0],
                                                dict(repeats=True, two_launches=True)),
    "1025_tokens_of_one_bound_513": (BASE, [1025] + [0] * 7, dict(bounds=[513] + [None] * 7)),
    "16_ranks_384_experts": (replace(BASE, world_size=16, num_experts=384, hidden_dim=384), [40, 0, 7, 64] * 4, {}),
    "32_ranks_all_tables": (replace(BASE, world_size=32, num_experts=384, hidden_dim=256), [1 + 3 * (r % 5) for r in range(32)], {}),
    "32_ranks_tables_too_large": (replace(BASE, world_size=32, num_experts=512, hidden_dim=256), [9] * 32, dict(two_launches=True)),
    "two_ranks_many_experts_each": (replace(BASE, world_size=2, num_experts=300), [90, 61], {}),
    "hidden_14336_two_nodes": (replace(BASE, world_size=4, num_experts=64, hidden_dim=14336, node_size=2), [3, 20, 0, 300], {}),
    "strided_the_general_kernel": (BASE, [20] * 8, dict(strided=True)),
    "experts_that_are_none": (BASE, [5, 0, 9, 1, 30, 2, 2, 2], dict(stray=True)),
    "experts_that_are_none_eight_a_workgroup": (replace(BASE, expert_padding=4), [250, 256, 3, 255, 256, 0, 257, 700],
                                                dict(stray=True, repeats=True)),
    "experts_that_are_none_the_two_launches": (BASE, [257] + [256] * 7, dict(stray=True, two_launches=True)),
}


@pytest.mark.parametrize("name", STEPS)
def test_steps_of_several_sources(name):
    case, tokens, how = STEPS[name]
    print(f"{name} tokens={tokens}", flush=True)
    run_and_check(replace(case, name=name, num_tokens=max(tokens), seed=31_000), tokens, **how)


BF16, F16, F32, FP8 = torch.bfloat16, torch.float16, torch.float32, torch.float8_e4m3fn
# configuration, tokens, layout of the scales, whether there is a routing launch of its own
TRANSPORT = {
    "fp8_row": (RefConfig("fp8_row", 8, 1, 128, 64, 5120, 40, 8, FP8, BF16, F32), [128, 0, 42, 1, 128, 0, 42, 1], "row", False),
    "fp8_col_pad16": (RefConfig("fp8_col", 8, 1, 250, 64, 2048, 16, 8, FP8, BF16, F32, expert_padding=16), [250] * 8, "col", False),
    "fp8_col_pad16_short_rows": (RefConfig("fp8_col", 8, 1, 250, 64, 1024, 8, 8, FP8, BF16, F32, expert_padding=16), [250] * 8,
                                 "col", True),
    "bf16_no_scales": (RefConfig("bf16", 4, 1, 300, 32, 4096, None, 6, BF16, BF16, None), [300, 1, 0, 299], "row", False),
    "f32_rows_of_16_kb": (RefConfig("f32", 2, 1, 40, 16, 4096, None, 2, F32, F32, None, node_size=1), [40, 3], "row", False),
    "f16_one_chunk": (RefConfig("f16", 3, 1, 33, 9, 8, None, 3, F16, F16, None), [33, 0, 32], "row", False),
}


@pytest.mark.parametrize("name", TRANSPORT)
def test_rows_moved_as_they_are(name):
    cfg, tokens, layout, two_launches = TRANSPORT[name]
    print(f"{name} tokens={tokens}", flush=True)
    world = [make_ref_rank(cfg, r, t) for r, t in enumerate(tokens)]
    rows = rows_for(cfg, world)
    routes = []
    check(cfg, world, rows, run_gpu(cfg, world, rows, DEV, split=False, scale_layout=layout, routes=routes))
    assert routes == [two_launches]


# Steps of more tokens than a workgroup per compute unit holds, and of one source whose rows leave no wavefront beside their
# pieces: ranks' tokens, experts, top-k, elements, type, scales, layout of the scales, whether there is a routing launch
SPREAD = {
    "f32_16_kb_two_a_workgroup": ([300, 0, 301, 270], 30, 2, 4096, F32, None, "row", False),
    "f32_28_kb_of_one": ([0, 900, 0], 24, 8, 7168, F32, None, "row", False),
    "f32_16_kb_of_one": ([130, 0], 16, 8, 4096, F32, None, "row", False),
    "f32_16_kb_one_token": ([0, 0, 1], 9, 1, 4096, F32, None, "row", False),
    "bf16_2_kb_eight_a_workgroup": ([700, 0, 1, 1400], 17, 1, 1024, BF16, None, "row", False),
    "bf16_14_kb_one_copy": ([1601, 31], 10, 1, 7168, BF16, None, "row", False),
    "fp8_scales_by_column": ([1201, 1198, 2], 12, 2, 7168, FP8, 56, "col", False),
    "fp8_scales_by_row_pad": ([1300, 3, 1300], 33, 3, 2944, FP8, 23, "row", False),
    "bf16_eight_copies_of_one": ([1025, 0], 20, 8, 4096, BF16, None, "row", False),
    "f16_1500_workgroups": ([6001, 5999], 6, 1, 1024, F16, None, "row", False),
    "f16_2000_workgroups_the_two_launches": ([8001, 7999], 6, 1, 1024, F16, None, "row", True),
}


@pytest.mark.parametrize("name", SPREAD)
def test_more_workgroups_than_compute_units(name):
    tokens, experts, topk, hidden, dtype, scales, layout, two_launches = SPREAD[name]
    print(f"{name} tokens={tokens}", flush=True)
    cfg = RefConfig(name, len(tokens), 1, max(tokens), experts, hidden, scales, topk, dtype, BF16 if dtype == FP8 else dtype,
                    F32 if scales else None, expert_padding=5 if "pad" in name else 1)
    world = [make_ref_rank(cfg, r, t) for r, t in enumerate(tokens)]
    rows = rows_for(cfg, world)
    routes = []
    check(cfg, world, rows, run_gpu(cfg, world, rows, DEV, split=False, scale_layout=layout, routes=routes))
    assert routes == [two_launches]


SPREAD_QUANTISED = {
    "512_workgroups_and_the_tables": (replace(BASE, topk=4, hidden_dim=2048), [320] * 8, dict(repeats=True)),
    "two_short_copies": (replace(BASE, topk=2, hidden_dim=1024, expert_padding=16), [2049, 0, 0, 1, 300, 0, 0, 17], dict(stray=True)),
    "bounds": (replace(BASE, topk=3, hidden_dim=4096), [700, 800, 0, 5, 701, 0, 0, 9], dict(bounds=[699, 0, None, 5, None, None, None, 1])),
    "beyond_two_a_compute_unit": (replace(BASE, topk=2, hidden_dim=2048), [4080, 0, 0, 1, 0, 0, 0, 17], dict(stray=True)),
    "beyond_three_a_compute_unit": (replace(BASE, topk=2, hidden_dim=2048), [6130, 0, 0, 1, 0, 0, 0, 17], dict(two_launches=True)),
    "beyond_two_a_compute_unit_two_rounds": (replace(BASE, topk=3, hidden_dim=5120), [4000, 0, 0, 1, 90, 0, 0, 17], dict(repeats=True)),
    "eight_copies_three_a_workgroup": (BASE, [1025, 0, 1, 0, 40, 0, 0, 434], dict(repeats=True)),
}


@pytest.mark.parametrize("name", SPREAD_QUANTISED)
def test_more_workgroups_than_compute_units_quantised(name):
    case, tokens, how = SPREAD_QUANTISED[name]
    print(f"{name} tokens={tokens}", flush=True)
    run_and_check(replace(case, name=name, num_tokens=max(tokens), seed=47_000), tokens, **how)


# Steps of eight copies on both sides of the line between one workgroup a compute unit and two: tokens of a workgroup
ONE_OR_TWO = {
    "five_few_experts": (replace(BASE, num_experts=64, hidden_dim=4096), [131] + [130] * 7, dict(repeats=True)),
    "three_many_experts": (replace(BASE, num_experts=251, hidden_dim=4096, expert_padding=16), [131] + [130] * 7, dict(repeats=True)),
    "three_few_experts": (replace(BASE, num_experts=64, hidden_dim=3072), [171] + [170] * 7, dict(stray=True)),
    "seven": (replace(BASE, num_experts=256, hidden_dim=2048), [1, 700, 0, 193, 0, 0, 700, 0], dict(repeats=True)),
}


@pytest.mark.parametrize("name", ONE_OR_TWO)
def test_one_or_two_workgroups_a_compute_unit(name):
    case, tokens, how = ONE_OR_TWO[name]
    print(f"{name} tokens={tokens}", flush=True)
    run_and_check(replace(case, name=name, num_tokens=max(tokens), seed=51_000), tokens, **how)


# The same of rows moved as they are: ranks' tokens, experts, elements, type, scales
ONE_OR_TWO_MOVED = {
    "eight_2_kb": ([256] * 8, 64, 1024, BF16, None),
    "five_5_kb": ([256] * 8, 64, 2560, BF16, None),
    "eight_5_kb_scales": ([255] * 7 + [254], 64, 5120, FP8, 40),
    "five_5_kb_scales_many_experts": ([256] * 8, 256, 5120, FP8, 40),
    "five_2_kb_of_sixteen_many_experts": ([128] * 16, 384, 1024, BF16, None),
    "five_6_kb_scales": ([2047, 1], 48, 6144, FP8, 48),
    "seven_4_kb_of_sixteen": ([113] + [110] * 15, 128, 2048, BF16, None),
    "four_4_kb_of_eight": ([223] + [220] * 7, 128, 2048, BF16, None),
}


@pytest.mark.parametrize("name", ONE_OR_TWO_MOVED)
def test_one_or_two_workgroups_a_compute_unit_of_rows_as_they_are(name):
    tokens, experts, hidden, dtype, scales = ONE_OR_TWO_MOVED[name]
    print(f"{name} tokens={tokens}", flush=True)
    cfg = RefConfig(name, len(tokens), 1, max(tokens), experts, hidden, scales, 8, dtype, BF16, F32 if scales else None)
    world = [make_ref_rank(cfg, r, t) for r, t in enumerate(tokens)]
    rows = rows_for(cfg, world)
    routes = []
    check(cfg, world, rows, run_gpu(cfg, world, rows, DEV, split=False, routes=routes))
    assert routes == [False]
