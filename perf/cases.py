"""What users of this framework run, as measurable cases: MoE dispatch + combine steps of an
expert-parallel group whose ranks live on one GPU.

One pass is one step: every rank dispatches its tokens to the experts' ranks (routing, packing, with fp8
quantisation or with the caller's rows as they are) and gets its combined tokens back.  The expert
computation in between belongs to the caller; its results (`expert_y`) are inputs here.

A case is a dict of plain values:

  api       "operator": every rank's `P2PAllToAll.dispatch` / `.combine`, both halves in one call
            "split":    the same operators with `do_send` and `do_recv` apart, all sends before the first recv
            "context":  `AllToAllContext.dispatch` / `.combine` with argument arrays packed once, as a serving
                        loop with fixed buffers calls it
  world     ranks of the group; dp: ranks that hold the same tokens
  senders   "all": every rank has `tokens` tokens; "one": rank 0 alone (one GPU's share of the group's
            work); "ragged": ranks have tokens, 0, tokens // 3, 1, tokens, ... in turn
  hidden, experts, topk, pad (rows of an expert are rounded up to it)
  rows      "quantise": bf16 tokens, dispatched as fp8 e4m3 with a float scale per 128 elements
            "fp8": fp8 tokens and scales of the caller, moved as they are; "bf16", "f16", "f32": rows without scales
  scales    "row" or "col": layout of the received scales (token-major, or element-major as grouped GEMMs read them)
  out       type of expert_y and of the combined tokens
  accumulate  combine adds to what is in the output (the shared experts' result)
  zipf      exponent of the experts' popularity, 0 for uniform routing
"""

from __future__ import annotations

import os
import sys

import torch

# the working folder is the root of the tree that is measured
_PACKAGE = os.path.join(os.getcwd(), "pplx-garden_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from pplx_garden_amd.distributed.loopback import LoopbackWorld  # noqa: E402
from pplx_garden_amd.kernels.p2p_all_to_all import P2PAllToAll  # noqa: E402
from pplx_garden_amd.native.p2p_all_to_all import A2ACombineArgs, A2ADispatchArgs  # noqa: E402

_DTYPE = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_ROW_DTYPE = {"quantise": torch.float8_e4m3fn, "fp8": torch.float8_e4m3fn, **_DTYPE}
_SCALED = ("quantise", "fp8")


def _case(name=None, **over):
    case = dict(api="operator", world=8, dp=1, senders="all", tokens=128, hidden=7168, experts=256, topk=8, pad=1,
                rows="quantise", scales="row", out="bf16", accumulate=False, zipf=0.0)
    case.update(over)
    return case if name is None else {"name": name, **case}


def listed():
    return [
        # the smallest step: eight ranks that each generate one token
        _case("decode_1x8", tokens=1),
        # a decode batch on one GPU's share of the group, from a serving loop with fixed buffers
        _case("decode_128_share", api="context", senders="one", tokens=128),
        # the same for the smaller model shape (hidden 2048, 128 experts)
        _case("decode_128_share_2048", api="context", senders="one", tokens=128, hidden=2048, experts=128),
        # a decode batch of the whole group, 128 tokens a rank
        _case("decode_128x8", tokens=128),
        # the plumbing shape: four ranks, few experts, top-4
        _case("decode_64x4_top4", world=4, tokens=64, hidden=2048, experts=32, topk=4),
        # decode through the four split calls (other work runs between the halves), bf16 rows
        _case("decode_128x8_split", api="split", tokens=128, experts=128, rows="bf16"),
        # a mixed batch of decode and prefill tokens on one GPU's share, experts padded for a grouped GEMM
        _case("mixed_1024_share", api="context", world=16, senders="one", tokens=1024, experts=384, pad=128, zipf=1.0),
        # ranks with uneven loads, rows quantised by the caller, element-major scales for a grouped GEMM
        _case("ragged_1000_fp8", senders="ragged", tokens=1000, hidden=5120, experts=128, pad=16, rows="fp8",
              scales="col", zipf=0.8),
        # a prefill chunk without fp8, top-6, combined onto the shared experts' result
        _case("prefill_1500x4_bf16_top6", world=4, tokens=1500, hidden=4096, experts=64, topk=6, rows="bf16",
              accumulate=True, zipf=0.5),
        # the headline: a prefill chunk on one GPU's share
        _case("prefill_4096_share", api="context", senders="one", tokens=4096, zipf=1.2),
        # prefill through the four split calls, rows quantised by the caller (the reference's own mode)
        _case("prefill_2048x8_split", api="split", tokens=2048, rows="fp8", zipf=0.8),
        # the largest step: a prefill chunk of the whole group
        _case("prefill_4096x8", tokens=4096, zipf=1.2),
    ]


def _log_uniform(rng, low, high):
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    """A step of the same ranges: any call style, group size, batch, row type and layout."""
    while True:
        world = rng.choice([2, 4, 8, 8, 8, 16])
        rows = rng.choice(["quantise", "quantise", "quantise", "fp8", "bf16", "f16", "f32"])
        senders = rng.choice(["one", "all", "all", "ragged"])
        hidden = rng.choice([1024, 2048, 2944, 4096, 5120, 7168])
        topk = rng.choice([1, 2, 4, 6, 8, 8, 8])
        experts = world * rng.choice([4, 8, 16, 24, 32]) - rng.choice([0, 0, 0, 1])
        accumulate = rng.random() < 0.15
        case = _case(
            api=rng.choice(["operator", "operator", "split", "context"]), world=world,
            dp=2 if not accumulate and world >= 4 and rng.random() < 0.1 else 1, senders=senders,
            tokens=_log_uniform(rng, 1, 8192 if senders == "one" else 4096), hidden=hidden, experts=experts,
            topk=topk, pad=rng.choice([1, 1, 16, 128]), rows=rows,
            scales=rng.choice(["row", "row", "col"]) if rows in _SCALED else "row",
            out=rows if rows in ("f16", "f32") else "bf16", accumulate=accumulate,
            zipf=rng.choice([0.0, 0.5, 0.8, 1.0, 1.2]))
        if experts >= 2 * topk and work(case)["bytes"] <= 0.5 * work(listed()[-1])["bytes"]:
            return case


def _tokens(case):
    """Tokens of every source (a dp group is one source)."""
    groups, t = case["world"] // case["dp"], case["tokens"]
    if case["senders"] == "one":
        return [t] + [0] * (groups - 1)
    if case["senders"] == "ragged":
        return [(t, 0, max(t // 3, 1), 1)[g % 4] for g in range(groups)]
    return [t] * groups


def _row_bytes(case):
    return case["hidden"] * _ROW_DTYPE[case["rows"]].itemsize


def _scale_bytes(case):
    return case["hidden"] // 128 * 4 if case["rows"] in _SCALED else 0


def work(case):
    tokens, k, h = sum(_tokens(case)), case["topk"], case["hidden"]
    out_row = h * _DTYPE[case["out"]].itemsize
    in_row = 2 * h if case["rows"] == "quantise" else _row_bytes(case) + _scale_bytes(case)
    dispatch = in_row + 4 * k + k * (_row_bytes(case) + _scale_bytes(case))
    combine = k * out_row + 8 * k + case["dp"] * out_row + (out_row if case["accumulate"] else 0)
    return {"bytes": tokens * (dispatch + combine), "flops": tokens * 2 * k * h * case["dp"]}


def tolerance(case):
    # Dispatched rows come back as bytes and have to be equal.  The combined tokens are sums of topk products in
    # float, rounded once to their type: in another order, or in 64 bits, those that lie near a tie round the other
    # way.  Measured against 64-bit sums over the listed cases and these types, relative 2-norm: bf16 up to 3.5e-5,
    # f16 5.8e-6, f32 6e-8; largest difference: bf16 and f16 one unit in the last place, f32 4.4e-7.
    return {"bf16": {"rel": 2e-4, "max": 0.016}, "f16": {"rel": 2.4e-5, "max": 0.002},
            "f32": {"rel": 2.4e-7, "max": 2e-6}}[case["out"]]


def _popularity(case, device):
    """Logarithm of every expert's popularity: Zipf over a fixed order of the experts."""
    gen = torch.Generator(device=device)
    gen.manual_seed(case["experts"])
    order = torch.randperm(case["experts"], generator=gen, device=device)
    return -case["zipf"] * torch.log(order.float() + 1)


def _routing(gen, tokens, experts, topk, popularity):
    """topk distinct experts a token, drawn by popularity (Gumbel keys: the largest of log p + noise)."""
    noise = torch.rand((tokens, experts), generator=gen, device=popularity.device).clamp_(1e-20, 1 - 1e-7)
    return (popularity - torch.log(-torch.log(noise))).topk(topk, dim=-1).indices.to(torch.int32)


def _capacity(case, device, popularity):
    """Rows of a rank's receive buffer: what the fullest rank can expect with a margin of 5 % and eight standard
    deviations, never more than could possibly arrive."""
    n, k, experts, pad, total = case["world"], case["topk"], case["experts"], case["pad"], sum(_tokens(case))
    local = -(-experts // n)
    gen = torch.Generator(device=device)
    gen.manual_seed(1)
    sample = _routing(gen, 16384, experts, k, popularity)
    share = torch.bincount(sample.reshape(-1).long() // local, minlength=n).max().item() / 16384
    likely = total * share * 1.05 + 8 * (total * share * k) ** 0.5 + 8 * k
    possible = total * min(k, local)
    return int(min(likely, possible)) + 1 + local * (pad - 1)


def prepare(case, seed):
    device = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=device)
    gen.manual_seed(seed)
    n, dp, h, k, experts = case["world"], case["dp"], case["hidden"], case["topk"], case["experts"]
    scaled, row_dtype, out_dtype = case["rows"] in _SCALED, _ROW_DTYPE[case["rows"]], _DTYPE[case["out"]]
    hs = h // 128 if scaled else None
    tokens = _tokens(case)
    local = -(-experts // n)

    # one operator a rank, all on one world
    world = LoopbackWorld(n, device=device)
    ops = [
        P2PAllToAll(max_num_tokens=max(tokens), num_experts=experts, expert_padding=case["pad"], hidden_dim=h,
                    hidden_dim_scale=hs, in_dtype=row_dtype, out_dtype=out_dtype,
                    scale_dtype=torch.float32 if scaled else None, num_experts_per_token=k, device=device,
                    dp_group=world.dp_group(r, dp) if dp > 1 else None, global_group=world.group(r))
        for r in range(n)
    ]

    # tokens, routing and weights of every source
    popularity = _popularity(case, device)
    sources = []
    for t in tokens:
        x = torch.randn((t, h), generator=gen, device=device)
        x_scale = None
        if case["rows"] == "quantise":     # activations: a few channels far above the rest
            x *= torch.where(torch.rand((t, h), generator=gen, device=device) < 0.01, 50.0, 1.0)
            x = x.to(torch.bfloat16)
        elif case["rows"] == "fp8":
            x = x.mul_(100).clamp_(-448, 448).to(torch.float8_e4m3fn)
            x_scale = torch.rand((t, hs), generator=gen, device=device) * 0.1 + 0.01
        else:
            x = x.to(row_dtype)
        indices = _routing(gen, t, experts, k, popularity)
        weights = torch.softmax(torch.randn((t, k), generator=gen, device=device), dim=-1)
        sources.append((x, x_scale, indices, weights))

    # receive buffers, rows that nobody writes are zero
    rows = _capacity(case, device, popularity)
    num = torch.zeros((n, local), dtype=torch.int32, device=device)
    out_x = torch.zeros((n, rows, h * row_dtype.itemsize), dtype=torch.uint8, device=device)
    out_scale = None
    if scaled:
        out_scale = torch.zeros((n, rows, hs), device=device) if case["scales"] == "row" else \
            torch.zeros((n, hs, rows), device=device).transpose(1, 2)
    expert_y = torch.empty((n, rows, h), dtype=out_dtype, device=device)
    for r in range(n):
        expert_y[r] = torch.randn((rows, h), generator=gen, device=device)
    combined = [torch.zeros((tokens[r // dp], h), dtype=out_dtype, device=device) for r in range(n)]

    ranks = []
    for r in range(n):
        x, x_scale, indices, weights = sources[r // dp]
        indices = indices.view(torch.uint32)
        ranks.append((
            ops[r],
            dict(out_expert_num_tokens=num[r], out_expert_x=out_x[r].view(row_dtype),
                 out_expert_x_scale=out_scale[r] if scaled else None, dp_x=x, dp_x_scale=x_scale, indices=indices,
                 weights=weights),
            dict(out_tokens=combined[r], indices=indices, weights=weights, expert_y=expert_y[r],
                 accumulate=case["accumulate"])))
    state = dict(api=case["api"], ranks=ranks, world=world,
                 outputs=[num, out_x, out_scale] + [c for c in combined if c.numel()])
    if case["api"] == "context":
        state.update(ctx=ops[0].context, quantise=case["rows"] == "quantise", out_dtype=out_dtype,
                     accumulate=case["accumulate"], **_packed(ops[0].context, ranks))
    return state


def _packed(ctx, ranks):
    """The argument arrays of the context's calls, for buffers that do not move."""
    dispatch, combine = [], []
    for _, d, c in ranks:
        t, x, s, os = d["dp_x"].shape[0], d["dp_x"], d["dp_x_scale"], d["out_expert_x_scale"]
        idx, w, y, out = d["indices"], d["weights"], c["expert_y"], c["out_tokens"]
        routes = dict(num_tokens=t, indices=idx.data_ptr() or None, indices_stride=idx.stride(0),
                      weights=w.data_ptr() or None, weights_stride=w.stride(0), bound_m=None)
        dispatch.append(A2ADispatchArgs(
            x_ptr=x.data_ptr() or None, x_stride=x.stride(0) * x.dtype.itemsize,
            x_scale_ptr=s.data_ptr() or None if s is not None else None,
            x_scale_stride_elem=s.stride(1) if s is not None else 0,
            x_scale_stride_token=s.stride(0) if s is not None else 0,
            out_num_tokens=d["out_expert_num_tokens"].data_ptr(), out_x=d["out_expert_x"].data_ptr(),
            out_x_stride=d["out_expert_x"].stride(0) * d["out_expert_x"].dtype.itemsize,
            out_x_rows=d["out_expert_x"].shape[0], out_x_scale=os.data_ptr() if os is not None else None,
            out_x_scale_stride_elem=os.stride(1) if os is not None else 0,
            out_x_scale_stride_token=os.stride(0) if os is not None else 0, **routes))
        combine.append(A2ACombineArgs(
            expert_y=y.data_ptr(), expert_y_stride=y.stride(0) * y.dtype.itemsize, expert_y_rows=y.shape[0],
            out_tokens=out.data_ptr() or None, out_tokens_stride=out.stride(0), **routes))
    return dict(dispatch=ctx.pack_dispatch_args(dispatch), combine=ctx.pack_combine_args(combine))


def run(state):
    ranks = state["ranks"]
    if state["api"] == "context":
        stream = torch.cuda.current_stream().cuda_stream
        state["ctx"].dispatch(state["dispatch"], state["quantise"], stream)
        state["ctx"].combine(state["combine"], state["out_dtype"], state["accumulate"], stream)
    elif state["api"] == "operator":
        for op, d, _ in ranks:
            op.dispatch(**d)
        for op, _, c in ranks:
            op.combine(**c)
    else:
        for op, d, _ in ranks:
            op.dispatch(**d, do_send=True, do_recv=False)
        for op, d, _ in ranks:
            op.dispatch(**d, do_send=False, do_recv=True)
        for op, _, c in ranks:
            op.combine(**c, do_send=True, do_recv=False)
        for op, _, c in ranks:
            op.combine(**c, do_send=False, do_recv=True)
    return state["outputs"]
