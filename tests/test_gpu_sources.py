"""The one-launch dispatch of steps of several sources (and of larger steps of one) against the oracle, bit for bit: rows,
scales, counts and every routing table of every source, at the sizes where its divisions of the work can go wrong."""

from dataclasses import replace

import numpy as np
import pytest
import torch

import a2a_oracle as oracle
from a2a_cases import C1, bf16_codes, make_rank, scaled
from a2a_harness import SENTINEL, make_ops, rows_needed
from a2a_transport import RefConfig, check, make_ref_rank, rows_for, run_gpu
from pplx_garden_amd.native import p2p_all_to_all as native

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def run_and_check(case, tokens, bounds=None, repeats=False, strided=False, stray=False):
    """One dispatch of `tokens[r]` tokens of every rank; `repeats`: every third token names its first expert twice;
    `strided`: index rows with a gap behind them (another kernel's step, the same result); `stray`: the first token of
    every source names an expert that does not exist (flagged, its other copies are sent)."""
    N, Le, H, Hs, K, E = (case.world_size, case.experts_per_rank, case.hidden_dim, case.hidden_dim_scale, case.topk,
                          case.num_experts)
    bounds = bounds or [None] * N
    world = [make_rank(case, r, t) for r, t in enumerate(tokens)]
    if repeats:
        for rd in world:
            rd.indices[::3, K - 1] = rd.indices[::3, 0]
    rows = rows_needed(case, world)
    inputs = [oracle.RankInput(x=bf16_codes(rd.x), indices=rd.indices.numpy(), bound_m=b) for rd, b in zip(world, bounds)]
    want = oracle.dispatch_world(inputs, num_experts=E, world_size=N, node_size=case.node_size or N,
                                 expert_padding=case.expert_padding, out_rows=rows, quantize=True)
    _, ops = make_ops(case, DEV, max_num_tokens=max(tokens))
    try:
        t = []
        for r, rd in enumerate(world):
            idx = rd.indices.clone()
            if stray and idx.shape[0]:
                idx[0, K - 1] = E + 3
            idx = idx.view(torch.uint32).to(DEV)
            if strided and idx.shape[0]:
                wide = torch.zeros((idx.shape[0], K + 3), dtype=torch.uint32, device=DEV)
                wide[:, :K] = idx
                idx = wide[:, :K]
            t.append(dict(x=rd.x.to(DEV), idx=idx, w=rd.weights.to(DEV),
                          b=None if bounds[r] is None else torch.tensor([bounds[r]], dtype=torch.int32, device=DEV),
                          n=torch.full((Le,), -1, dtype=torch.int32, device=DEV),
                          ox=torch.full((rows, H), SENTINEL, dtype=torch.uint8, device=DEV).view(torch.float8_e4m3fn),
                          os=torch.full((rows, Hs), -7.0, dtype=torch.float32, device=DEV)))
        for r in range(N):
            ops[r].dispatch(out_expert_num_tokens=t[r]["n"], out_expert_x=t[r]["ox"], out_expert_x_scale=t[r]["os"],
                            dp_x=t[r]["x"], dp_x_scale=None, indices=t[r]["idx"], weights=t[r]["w"], bound_m=t[r]["b"])
        torch.cuda.synchronize(DEV)
        ctx = ops[0].context
        if stray:
            assert ctx.status() & 1     # A2A_DEV_BAD_EXPERT_ID
            return
        assert ctx.status() == 0
        for r in range(N):
            n_local = max(0, min(Le, E - r * Le))
            np.testing.assert_array_equal(t[r]["n"].cpu().numpy()[:n_local], want[r].num_tokens[:n_local])
            assert (t[r]["n"].cpu().numpy()[n_local:] == -1).all()
            wr = want[r].written
            got_x, got_s = t[r]["ox"].view(torch.uint8).cpu().numpy(), t[r]["os"].cpu().numpy()
            np.testing.assert_array_equal(got_x[wr], want[r].x[wr])
            np.testing.assert_array_equal(got_s[wr].view(np.uint32), want[r].x_scale[wr].view(np.uint32))
            assert (got_x[~wr] == SENTINEL).all() and (got_s[~wr] == -7.0).all()
            n_eff = tokens[r] if bounds[r] is None else bounds[r]
            count, toff, eoff = oracle.route(world[r].indices.numpy()[:n_eff], E)
            np.testing.assert_array_equal(ctx.read_table(r, native.TABLE_NUM_ROUTED, E).numpy(), count)
            np.testing.assert_array_equal(ctx.read_table(r, native.TABLE_EXPERT_OFFSETS, E).numpy(), eoff)
            if n_eff:
                np.testing.assert_array_equal(ctx.read_table(r, native.TABLE_TOKEN_OFFSET, n_eff * K).numpy(), toff)
                np.testing.assert_array_equal(ctx.read_table(r, native.TABLE_SLOT, n_eff * K).numpy(),
                                              want[0].slots[r][:n_eff].reshape(-1))
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
    "2049_tokens_the_two_launches": (BASE, [257] + [256] * 7, {}),
    "2048_tokens_of_one": (replace(BASE, hidden_dim=1024), [0, 0, 0, 2048, 0, 0, 0, 0], dict(repeats=True)),
    "1025_tokens_of_one_bound_513": (BASE, [1025] + [0] * 7, dict(bounds=[513] + [None] * 7)),
    "16_ranks_384_experts": (replace(BASE, world_size=16, num_experts=384, hidden_dim=384), [40, 0, 7, 64] * 4, {}),
    "32_ranks_all_tables": (replace(BASE, world_size=32, num_experts=384, hidden_dim=256), [1 + 3 * (r % 5) for r in range(32)], {}),
    "32_ranks_tables_too_large": (replace(BASE, world_size=32, num_experts=512, hidden_dim=256), [9] * 32, {}),
    "two_ranks_many_experts_each": (replace(BASE, world_size=2, num_experts=300), [90, 61], {}),
    "hidden_14336_two_nodes": (replace(BASE, world_size=4, num_experts=64, hidden_dim=14336, node_size=2), [3, 20, 0, 300], {}),
    "strided_the_general_kernel": (BASE, [20] * 8, dict(strided=True)),
    "expert_that_is_none": (BASE, [5, 0, 9, 1, 30, 2, 2, 2], dict(stray=True)),
}


@pytest.mark.parametrize("name", STEPS)
def test_steps_of_several_sources(name):
    case, tokens, how = STEPS[name]
    print(f"{name} tokens={tokens}", flush=True)
    run_and_check(replace(case, name=name, num_tokens=max(tokens), seed=31_000), tokens, **how)


BF16, F16, F32, FP8 = torch.bfloat16, torch.float16, torch.float32, torch.float8_e4m3fn
TRANSPORT = {
    "fp8_row": (RefConfig("fp8_row", 8, 1, 128, 64, 5120, 40, 8, FP8, BF16, F32), [128, 0, 42, 1, 128, 0, 42, 1], "row"),
    "fp8_col_pad16": (RefConfig("fp8_col", 8, 1, 250, 64, 1024, 8, 8, FP8, BF16, F32, expert_padding=16), [250] * 8, "col"),
    "bf16_no_scales": (RefConfig("bf16", 4, 1, 300, 32, 4096, None, 6, BF16, BF16, None), [300, 1, 0, 299], "row"),
    "f32_rows_of_16_kb": (RefConfig("f32", 2, 1, 40, 16, 4096, None, 2, F32, F32, None, node_size=1), [40, 3], "row"),
    "f16_one_chunk": (RefConfig("f16", 3, 1, 33, 9, 8, None, 3, F16, F16, None), [33, 0, 32], "row"),
}


@pytest.mark.parametrize("name", TRANSPORT)
def test_rows_moved_as_they_are(name):
    cfg, tokens, layout = TRANSPORT[name]
    print(f"{name} tokens={tokens}", flush=True)
    world = [make_ref_rank(cfg, r, t) for r, t in enumerate(tokens)]
    rows = rows_for(cfg, world)
    check(cfg, world, rows, run_gpu(cfg, world, rows, DEV, split=False, scale_layout=layout))
