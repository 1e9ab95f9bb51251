"""Split steps whose kernels find their buffers and tables in a few packed words: the largest sizes that the words hold, tables at
their furthest distances, receivers without experts, every number of routes a group of loads is made for and its neighbours,
against the oracle."""

import pytest
import torch

from a2a_transport import RefConfig, check, make_ops, make_ref_rank, rows_for, run_gpu

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


# One sender's combine in the group call: ranks, sender, tokens, experts, elements, top-k, rows' and tokens' type
SOLE = [
    (8, 0, 128, 256, 7168, 8, BF16, BF16),
    (8, 7, 1, 17, 1024, 4, F16, F32),            # receivers without experts
    (10, 3, 33, 1024, 520, 9, BF16, F16),        # the most receivers, the most experts, a group of loads and one more
    (11, 10, 33, 1023, 520, 2, F32, F32),        # a receiver more than the words hold
    (1, 0, 2048, 1024, 256, 1, F32, BF16),       # the most tokens; all experts at one rank
    (2, 1, 900, 2, 1032, 2, F16, F16),           # an expert a rank; two slabs a wavefront
    (3, 1, 5, 64, 64, 64, BF16, F32),
]


@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("ranks,sender,tokens,experts,hidden,topk,rows_type,out_type", SOLE)
def test_one_senders_combine(ranks, sender, tokens, experts, hidden, topk, rows_type, out_type, accumulate):
    """The same bits as from weights with gaps between their rows, receivers' buffers of different lengths or a bound on the
    tokens, which the general kernel serves; and what 64 bits give for them."""
    print(f"ranks={ranks} sender={sender} tokens={tokens} topk={topk} {rows_type} {out_type}", flush=True)
    cfg = RefConfig("sole", ranks, 1, tokens, experts, hidden, None, topk, rows_type, out_type, None)
    world = [make_ref_rank(cfg, r, tokens if r == sender else 0) for r in range(ranks)]
    rows, local = rows_for(cfg, world), -(-experts // ranks)
    gen = torch.Generator().manual_seed(5)
    ops = make_ops(cfg, DEV)
    try:
        idx = [rd.indices.view(torch.uint32).to(DEV) for rd in world]
        w = [rd.weights.to(DEV) for rd in world]
        for r in range(ranks):
            ops[r].dispatch(torch.zeros(local, dtype=torch.int32, device=DEV),
                            torch.zeros((rows, hidden), dtype=rows_type, device=DEV), None, world[r].dp_x.to(DEV), None, idx[r], w[r])
        y = [torch.randn((rows + 1, hidden), generator=gen).to(rows_type).to(DEV) for _ in range(ranks)]
        before = torch.randn((tokens, hidden), generator=gen).to(out_type).to(DEV)

        def combined(weights, y, bound=None):
            out = [before.clone() if r == sender else before[:0].clone() for r in range(ranks)]
            for r in range(ranks):
                ops[r].combine(out[r], idx[r], weights[r], y[r], bound_m=bound, accumulate=accumulate)
            return out[sender]

        got = combined(w, y)
        gaps = [torch.cat([t, t.new_full((t.shape[0], 3), 9.0)], dim=1)[:, :topk] for t in w]
        same = [combined(gaps, y), combined(w, [t[:rows] if r == 0 else t for r, t in enumerate(y)]),
                combined(w, y, torch.tensor([tokens], dtype=torch.int32, device=DEV))]
        torch.cuda.synchronize(DEV)
        assert ops[0].context.status() == 0
        slots = ops[0].context.read_table(sender, 3, tokens * topk).view(tokens, topk)
        for other in same:
            assert torch.equal(got.view(torch.uint8), other.view(torch.uint8))
        owner = world[sender].indices.long() // local
        taken = torch.stack([t.cpu() for t in y])[owner, slots].double()
        weights = world[sender].weights.double().unsqueeze(-1)
        want, size = (taken * weights).sum(1), (taken * weights).abs().sum(1)
        if accumulate:
            want, size = want + before.cpu().double(), size + before.cpu().double().abs()
        # topk roundings of a float sum, and one to the output's type
        unit = {BF16: 2.0 ** -8, F16: 2.0 ** -11, F32: 2.0 ** -24}[out_type]
        bound = unit * want.abs() + (topk + 1) * 2.0 ** -23 * size + (2.0 ** -24 if out_type == F16 else 0)
        assert ((got.cpu().double() - want).abs() <= bound * 1.01).all()
    finally:
        for op in ops:
            op.destroy()
