"""Run a workload through the HIP library (via the operator) and through the oracle."""

from __future__ import annotations

from dataclasses import dataclass
from typing import List, Optional, Sequence

import numpy as np
import torch

import a2a_oracle as oracle
from a2a_cases import Case, RankData, bf16_codes, rows_needed  # noqa: F401

SENTINEL = 0xA5


@dataclass
class WorldResult:
    num_tokens: List[np.ndarray]      # per rank [Le] int32
    x: List[np.ndarray]               # per rank [rows, H] uint8 (fp8 codes)
    x_scale: List[np.ndarray]         # per rank [rows, Hs] float32
    out_tokens: List[np.ndarray]      # per rank [T, H] bf16 codes (uint16)


class RouteWatch:
    """Whether the next call on `ctx` that routes its tokens does so in a launch of its own, in front of the one that moves the
    rows (KERNEL_ROUTE's events are left alone by calls that route and move in one launch)."""

    def __init__(self, ctx):
        from pplx_garden_amd.native.p2p_all_to_all import KERNEL_ROUTE

        self._events = [torch.cuda.Event(enable_timing=True) for _ in range(3)]
        for e in self._events:
            e.record()
        torch.cuda.synchronize()
        self._before = self._events[2].elapsed_time(self._events[0])
        ctx.time_next_kernel(KERNEL_ROUTE, self._events[0].cuda_event, self._events[1].cuda_event)

    def launched(self) -> bool:
        torch.cuda.synchronize()
        return self._events[2].elapsed_time(self._events[0]) != self._before


def with_gap(indices: torch.Tensor, gap: int = 3) -> torch.Tensor:
    """The same index rows with `gap` words behind each of them, which are ids of no expert."""
    if indices.shape[0] == 0:
        return indices
    wide = torch.full((indices.shape[0], indices.shape[1] + gap), -2, dtype=torch.int32, device=indices.device)
    wide[:, :indices.shape[1]] = indices.view(torch.int32)
    return wide.view(indices.dtype)[:, :indices.shape[1]]


def dispatch_world_with_strays(inputs, *, num_experts: int, world_size: int, expert_padding: int, out_rows: int, quantize: bool,
                               hidden_dim_scale: int = 0):
    """The oracle's dispatch of one node where ids of `num_experts` and above name no expert and their copies go nowhere: to the
    experts of one rank more, which has no tokens and so leaves the others' layout as it is.  Returns (outs, routes): of each
    source its counts, offsets per expert, offsets of the entries (0 for those that go nowhere) and slots (-1 for those)."""
    Le = num_experts // world_size
    assert Le * world_size == num_experts
    strays = [np.asarray(i.indices).astype(np.int64) >= num_experts for i in inputs]
    moved = [oracle.RankInput(x=i.x, indices=np.where(s, num_experts, np.asarray(i.indices).astype(np.int64)), x_scale=i.x_scale,
                              bound_m=i.bound_m) for i, s in zip(inputs, strays)]
    nobody = oracle.RankInput(x=inputs[0].x[:0], indices=moved[0].indices[:0],
                              x_scale=None if inputs[0].x_scale is None else inputs[0].x_scale[:0])
    outs = oracle.dispatch_world(moved + [nobody], num_experts=num_experts + Le, world_size=world_size + 1,
                                 node_size=world_size + 1, expert_padding=expert_padding,
                                 out_rows=out_rows + sum(int(s.sum()) for s in strays) + Le * expert_padding, quantize=quantize,
                                 hidden_dim_scale=hidden_dim_scale)
    for o in outs[:world_size]:
        assert not o.written[out_rows:].any()
        o.x, o.written = o.x[:out_rows], o.written[:out_rows]
        o.x_scale = None if o.x_scale is None else o.x_scale[:out_rows]
    routes = []
    for g, (i, s) in enumerate(zip(moved, strays)):
        n = i.indices.shape[0] if i.bound_m is None else i.bound_m
        count, toff, eoff = oracle.route(i.indices[:n], num_experts + Le)
        routes.append((count[:num_experts], eoff[:num_experts], np.where(s[:n].reshape(-1), 0, toff),
                       np.where(s, -1, outs[0].slots[g])))
    return outs[:world_size], routes


def act_numpy(q: np.ndarray, scale: np.ndarray) -> np.ndarray:
    """The 'expert' of the reference's test: 2 * dequantised row, as bf16 codes
    (tests/p2p_all_to_all/test_p2p_all_to_all.py:44-50 with the block layout of
    benchmarks/bench_all_to_all.py:40-50)."""
    deq = oracle.dequantize_block128(q, scale)
    deq = np.nan_to_num(deq, nan=0.0)
    return oracle.f32_to_bf16((deq * np.float32(2.0)).astype(np.float32))


def run_oracle(case: Case, world: Sequence[RankData], rows: int) -> WorldResult:
    inputs = [oracle.RankInput(x=bf16_codes(rd.x), indices=rd.indices.numpy()) for rd in world]
    outs = oracle.dispatch_world(
        inputs, num_experts=case.num_experts, world_size=case.world_size,
        node_size=case.node_size or case.world_size, expert_padding=case.expert_padding,
        out_rows=rows, quantize=True)
    slots = outs[0].slots
    ys = []
    for o in outs:
        y = act_numpy(o.x, o.x_scale)
        y[~o.written] = 0
        ys.append(y)
    comb = oracle.combine_world(
        ys, [rd.indices.numpy() for rd in world], [rd.weights.numpy() for rd in world], slots,
        num_experts=case.num_experts, world_size=case.world_size)
    res = WorldResult([o.num_tokens for o in outs], [o.x for o in outs], [o.x_scale for o in outs], comb)
    res.written = [o.written for o in outs]
    res.slots = slots
    res.expert_y = ys
    return res


def make_ops(case: Case, device: torch.device, max_num_tokens: Optional[int] = None, context_flags: int = 0,
             max_private_tokens: Optional[int] = None):
    from pplx_garden_amd.distributed.loopback import LoopbackWorld
    from pplx_garden_amd.kernels.p2p_all_to_all import P2PAllToAll

    world = LoopbackWorld(case.world_size, node_size=case.node_size, device=device, context_flags=context_flags)
    ops = [
        P2PAllToAll(
            max_num_tokens=max_num_tokens or max(case.num_tokens, 1), num_experts=case.num_experts,
            expert_padding=case.expert_padding, hidden_dim=case.hidden_dim,
            hidden_dim_scale=case.hidden_dim_scale, in_dtype=torch.float8_e4m3fn,
            out_dtype=torch.bfloat16, scale_dtype=torch.float32,
            num_experts_per_token=case.topk, nets_per_gpu=1, max_private_tokens=max_private_tokens, device=device,
            dp_group=None, node_group=None, global_group=world.group(r))
        for r in range(case.world_size)
    ]
    return world, ops


def run_gpu(case: Case, world_data: Sequence[RankData], rows: int, device: torch.device,
            split: bool = False, expert_y_override=None, context_flags: int = 0, ops=None,
            order: Optional[Sequence[int]] = None, strided: bool = False, routes: Optional[list] = None) -> WorldResult:
    """dispatch -> 2*dequant -> combine on the GPU through the operator API.

    split=False: every rank calls dispatch()/combine() with do_send and do_recv
    (the group calls of the library); split=True: all sends, then all recvs (the
    four split calls).  With `ops` the given operators are used (and kept): several
    steps on one context.  `order`: in which the ranks make the group calls.  `strided`: index rows with a gap behind
    them.  `routes` gets, for the group call or for every send that has tokens, whether it routed in a launch of its own."""
    N, H, Hs, Le = case.world_size, case.hidden_dim, case.hidden_dim_scale, case.experts_per_rank
    own_ops = ops is None
    if own_ops:
        _, ops = make_ops(case, device, context_flags=context_flags)
    try:
        dev = [
            dict(x=rd.x.to(device), idx=with_gap(rd.indices_u32.to(device)) if strided else rd.indices_u32.to(device),
                 w=rd.weights.to(device))
            for rd in world_data
        ]
        outs = []
        for r in range(N):
            outs.append(dict(
                n=torch.full((Le,), -1, dtype=torch.int32, device=device),
                x=torch.full((rows, H), SENTINEL, dtype=torch.uint8, device=device).view(torch.float8_e4m3fn),
                s=torch.full((rows, Hs), -7.0, dtype=torch.float32, device=device),
                o=torch.zeros((world_data[r].x.shape[0], H), dtype=torch.bfloat16, device=device)))

        def dispatch(r, **kw):
            ops[r].dispatch(out_expert_num_tokens=outs[r]["n"], out_expert_x=outs[r]["x"],
                            out_expert_x_scale=outs[r]["s"], dp_x=dev[r]["x"], dp_x_scale=None,
                            indices=dev[r]["idx"], weights=dev[r]["w"], **kw)

        watches = []

        def watch():
            if routes is not None:
                watches.append(RouteWatch(ops[0].context))

        if split:
            for r in range(N):
                if world_data[r].indices.shape[0]:
                    watch()
                dispatch(r, do_send=True, do_recv=False)
            for r in range(N):
                dispatch(r, do_send=False, do_recv=True)
        else:
            watch()
            for r in order or range(N):
                dispatch(r)
        torch.cuda.synchronize(device)
        if routes is not None:
            routes.extend(w.launched() for w in watches)
        flags = ops[0].context.status()
        assert flags == 0, f"device error flags {flags}"

        ys = []
        for r in range(N):
            q = outs[r]["x"].view(torch.uint8).cpu().numpy()
            s = outs[r]["s"].cpu().numpy()
            if expert_y_override is not None:
                y = expert_y_override[r]
            else:
                y = act_numpy(q, s)
            ys.append(torch.from_numpy(y.view(np.int16)).view(torch.bfloat16).to(device))

        def combine(r, **kw):
            ops[r].combine(out_tokens=outs[r]["o"], indices=dev[r]["idx"], weights=dev[r]["w"],
                           expert_y=ys[r], **kw)

        if split:
            for r in range(N):
                combine(r, do_send=True, do_recv=False)
            for r in range(N):
                combine(r, do_send=False, do_recv=True)
        else:
            for r in order or range(N):
                combine(r)
        torch.cuda.synchronize(device)
        flags = ops[0].context.status()
        assert flags == 0, f"device error flags {flags}"

        res = WorldResult(
            [o["n"].cpu().numpy() for o in outs],
            [o["x"].view(torch.uint8).cpu().numpy() for o in outs],
            [o["s"].cpu().numpy() for o in outs],
            [o["o"].view(torch.int16).cpu().numpy().view(np.uint16) for o in outs])
        return res
    finally:
        if own_ops:
            for op in ops:
                op.destroy()


def assert_dispatch_equal(case: Case, got: WorldResult, want: WorldResult) -> None:
    """Bit-exact: counts, fp8 bytes and scales of written rows; untouched rows keep the sentinel."""
    for r in range(case.world_size):
        n_local = max(min(case.experts_per_rank, case.num_experts - r * case.experts_per_rank), 0)
        np.testing.assert_array_equal(got.num_tokens[r][:n_local], want.num_tokens[r][:n_local],
                                      err_msg=f"rank {r} counts")
        w = want.written[r]
        np.testing.assert_array_equal(got.x[r][w], want.x[r][w], err_msg=f"rank {r} fp8 bytes")
        np.testing.assert_array_equal(got.x_scale[r][w].view(np.uint32), want.x_scale[r][w].view(np.uint32),
                                      err_msg=f"rank {r} scales")
        assert (got.x[r][~w] == SENTINEL).all(), f"rank {r}: a padding row was written"
        assert (got.x_scale[r][~w] == -7.0).all(), f"rank {r}: a padding scale row was written"


def assert_combine_close(case: Case, got: WorldResult, want: WorldResult, rtol: float = 1e-2) -> None:
    """Within 1e-2 relative (bf16), the tolerance the baseline states; in practice bit-exact
    up to float64-emulated fused multiply-add corner cases."""
    for r in range(case.world_size):
        g = oracle.bf16_to_f32(got.out_tokens[r])
        w = oracle.bf16_to_f32(want.out_tokens[r])
        assert g.shape == w.shape
        if g.size == 0:
            continue
        np.testing.assert_allclose(g, w, rtol=rtol, atol=1e-2 * max(float(np.abs(w).max()), 1e-6) * 1e-2,
                                   err_msg=f"rank {r} combine")
