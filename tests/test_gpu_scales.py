"""Scales of the steps that are routed in a launch of their own (more than 16384 entries), the caller's, by row and by column,
and those of quantised rows, and of the recvs that copy by pieces of rows: at the sizes where their stores and loads change,
against the oracle bit for bit."""

from dataclasses import replace

import numpy as np
import pytest
import torch

import a2a_oracle as oracle
from a2a_cases import C1, scaled
from a2a_harness import RouteWatch, dispatch_world_with_strays
from a2a_transport import RefConfig, _bytes, check, make_ops, make_ref_rank, rows_for, run_gpu
from pplx_garden_amd.native import p2p_all_to_all as native
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
    ([1300, 2500, 1], 1024, 6, 4096, 32),     # more experts than threads; a span that ends in its first chunk of entries
    ([16384, 16385, 3], 6, 1, 4096, 4),       # a copy a token: by column beside the rows
    ([2048, 2049, 3], 16, 8, 4096, 4),        # whole spans, and a token more; a single slice of columns
    ([3277, 2048, 3], 16, 5, 4096, 4),        # a last span of one entry
]


@pytest.mark.parametrize("layout", ["row", "col"])
@pytest.mark.parametrize("tokens,experts,topk,hidden,scales", GIVEN, ids=[f"{s[0]}_h{s[3]}_s{s[4]}" for s in GIVEN])
def test_given_scales(tokens, experts, topk, hidden, scales, layout):
    print(f"tokens={tokens} hidden={hidden} scales={scales} {layout}", flush=True)
    cfg = RefConfig("scales", len(tokens), 1, max(tokens), experts, hidden, scales, topk, FP8, BF16, F32, expert_padding=16)
    world = [make_ref_rank(cfg, r, t) for r, t in enumerate(tokens)]
    rows = rows_for(cfg, world)
    routes = []
    check(cfg, world, rows, run_gpu(cfg, world, rows, DEV, split=False, scale_layout=layout, routes=routes))
    assert routes == [True]


@pytest.mark.parametrize("node", [16, 4])
def test_columns_of_sixteen_sources(node):
    """Sixteen sources that send: what a receiver lays out before a source's rows is looked up for eight of them at a time, and
    the receivers of several nodes lay them out in different orders."""
    tokens = [300, 40, 0, 129, 1, 64, 260, 17, 1100, 3, 90, 0, 33, 128, 2, 255]
    print(f"node={node}", flush=True)
    cfg = RefConfig("sixteen", 16, 1, max(tokens), 96, 4096, 32, 8, FP8, BF16, F32, expert_padding=4, node_size=node)
    world = [make_ref_rank(cfg, r, t) for r, t in enumerate(tokens)]
    rows = rows_for(cfg, world)
    routes = []
    check(cfg, world, rows, run_gpu(cfg, world, rows, DEV, split=False, scale_layout="col", routes=routes))
    assert routes == [True]


@pytest.mark.parametrize("hidden", [3968, 4096])
def test_quantised_rows(hidden):
    case = replace(scaled(C1, 1), hidden_dim=hidden, name="scales", num_tokens=2100, seed=77 + hidden)
    print(f"hidden={hidden}", flush=True)
    run_and_check(case, [2100, 0, 1, 0, 50, 0, 0, 3], two_launches=True)


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


@pytest.mark.parametrize("how", ["bounds", "repeats", "strays", "too_few_rows", "unaligned", "by_column_too", "one_by_row"])
def test_columns_of_unusual_steps(how):
    """Scales by column of a step with `bounds` on the device, with experts that repeat inside a token, with experts that do not
    exist (flagged, all other copies as if those were not there), with a receive buffer that the last rows do not fit, with
    source scales that are not 16-byte pieces, with source scales that are columns themselves, and with one receiver that takes
    rows."""
    print(how, flush=True)
    tokens, bounds = [1400, 900, 0, 64], [None] * 4
    cfg = RefConfig("unusual", 4, 1, 1400, 40, 4096, 32, 8, FP8, BF16, F32, expert_padding=8)
    world = [make_ref_rank(cfg, r, t) for r, t in enumerate(tokens)]
    if how == "bounds":
        bounds = [1290, 1, None, 0]
    if how == "repeats":
        for rd in world:
            rd.indices[::3, 7] = rd.indices[::3, 0]
    fits = rows_for(cfg, world)
    rows = fits - (70 if how == "too_few_rows" else 0)
    if how == "strays":
        for rd in world:
            rd.indices[::5, 7] = 40
            rd.indices[2::9, 0] = -1          # (0xFFFFFFFF)
            rd.indices[120:250] = 45          # a whole chunk of entries and the ends of its neighbours
    inputs = [oracle.RankInput(x=_bytes(rd.dp_x), indices=rd.indices.numpy().view(np.uint32), x_scale=rd.dp_x_scale.numpy(),
                               bound_m=b) for rd, b in zip(world, bounds)]
    how_sent = dict(num_experts=40, world_size=4, expert_padding=8, out_rows=fits, quantize=False, hidden_dim_scale=32)
    if how == "strays":
        want, routes = dispatch_world_with_strays(inputs, **how_sent)
    else:
        want = oracle.dispatch_world(inputs, node_size=4, **how_sent)
    ops = make_ops(cfg, DEV)
    try:
        outs = []
        ctx = ops[0].context
        watch = RouteWatch(ctx)
        for r, rd in enumerate(world):
            xs = rd.dp_x_scale.to(DEV)
            if how == "unaligned":
                wide = torch.zeros((xs.shape[0], 36), device=DEV)
                wide[:, 1:33] = xs
                xs = wide[:, 1:33]
            if how == "by_column_too":
                xs = xs.t().contiguous().t()
            x = torch.full((rows, 4096), 0xA5, dtype=torch.uint8, device=DEV)
            s = torch.full((rows, 32) if how == "one_by_row" and r == 1 else (32, rows), -7.0, device=DEV)
            if s.shape[0] != rows:
                s = s.t()
            outs.append((x, s))
            ops[r].dispatch(out_expert_num_tokens=torch.zeros(10, dtype=torch.int32, device=DEV),
                            out_expert_x=x.view(FP8), out_expert_x_scale=s, dp_x=rd.dp_x.to(DEV), dp_x_scale=xs,
                            indices=rd.indices.view(torch.uint32).to(DEV), weights=rd.weights.to(DEV),
                            bound_m=None if bounds[r] is None else torch.tensor([bounds[r]], dtype=torch.int32, device=DEV))
        assert watch.launched()
        assert ctx.status() == {"too_few_rows": native.DEV_RECV_OVERFLOW, "strays": native.DEV_BAD_EXPERT_ID}.get(how, 0)
        if how == "strays":
            for r, (count, eoff, toff, slots) in enumerate(routes):
                np.testing.assert_array_equal(ctx.read_table(r, native.TABLE_NUM_ROUTED, 40).numpy(), count)
                np.testing.assert_array_equal(ctx.read_table(r, native.TABLE_EXPERT_OFFSETS, 40).numpy(), eoff)
                if toff.size:
                    np.testing.assert_array_equal(ctx.read_table(r, native.TABLE_TOKEN_OFFSET, toff.size).numpy(), toff)
                    np.testing.assert_array_equal(ctx.read_table(r, native.TABLE_SLOT, toff.size).numpy().astype(np.uint32),
                                                  slots.reshape(-1).astype(np.uint32))
        for (x, s), w in zip(outs, want):
            wr = w.written[:rows]
            np.testing.assert_array_equal(x.cpu().numpy()[wr], w.x[:rows][wr])
            np.testing.assert_array_equal(s.cpu().numpy()[wr].view(np.uint32), w.x_scale[:rows][wr].view(np.uint32))
            assert (x.cpu().numpy()[~wr] == 0xA5).all() and (s.cpu().numpy()[~wr] == -7.0).all()
    finally:
        for op in ops:
            op.destroy()
