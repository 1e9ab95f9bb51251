"""`P2PAllToAll`: the MoE dispatch / combine operator, one object per logical rank.

Same constructor keywords, method signatures, tensor checks and per-expert
receive counts as the reference's operator
(python/pplx_garden/kernels/p2p_all_to_all.py:50-534).  What differs:

* `global_group` is a `LoopbackGroup`: all ranks live on one GPU, so the
  constructor sets up no transport (no topology detection, RDMA registration or
  peer-memory exchange, p2p_all_to_all.py:116-278).
* a call with `do_send and do_recv` is a collective: it runs when every rank of
  the world has made it, in one launch sequence that moves every row once.
  Calls with only `do_send` or only `do_recv` run at once, rank by rank, through
  staging buffers; every send of a step must come before the first recv.
* ranks of one `dp_group` must pass the same tokens, indices and weights, as in the reference
  (only one of them sends each copy, all of them receive the combined tokens).
* `dp_x` may be bfloat16 while `in_dtype` is float8_e4m3fn and `dp_x_scale` is
  None: dispatch then quantises, one float32 scale per 128 elements
  (`hidden_dim_scale` must be `hidden_dim // 128`).  The reference only
  transports rows the caller has already quantised.
"""

from __future__ import annotations

from typing import Any, Optional

import torch

from pplx_garden_amd.distributed.loopback import LoopbackGroup
from pplx_garden_amd.kernels.all_to_all import AllToAllKernel
from pplx_garden_amd.native.p2p_all_to_all import AllToAllContext, load_extension
from pplx_garden_amd.utils.math import ceil_div, round_up


class P2PAllToAll(AllToAllKernel):
    def __init__(
        self,
        *,
        max_num_tokens: int,
        num_experts: int,
        expert_padding: int,
        hidden_dim: int,
        hidden_dim_scale: Optional[int],
        in_dtype: torch.dtype,
        out_dtype: torch.dtype,
        scale_dtype: Optional[torch.dtype],
        num_experts_per_token: int,
        nets_per_gpu: int = 1,
        max_private_tokens: Optional[int] = None,
        device: torch.device,
        dp_group: Optional[Any] = None,
        node_group: Optional[Any] = None,
        global_group: LoopbackGroup,
    ) -> None:
        del nets_per_gpu  # no NICs in loopback
        self._device = torch.device(device)
        self._global_group = global_group
        self._all_to_all: Optional[AllToAllContext] = None
        self._operator = None

        if not isinstance(global_group, LoopbackGroup):
            raise TypeError("global_group must be a LoopbackGroup (see LoopbackWorld.group)")
        # Number of ranks that hold the same tokens (p2p_all_to_all.py:80-87).
        if dp_group is not None:
            self._dp_size = dp_group.size
            if node_group is None and global_group.node_size % dp_group.size != 0:
                node_group = dp_group
        else:
            self._dp_size = 1

        rank = global_group.rank
        world_size = global_group.size
        node_size = node_group.size if node_group is not None else global_group.node_size
        if world_size % node_size != 0:
            raise ValueError(f"node size {node_size} does not divide world size {world_size}")
        self._num_local_experts = ceil_div(num_experts, world_size)

        max_private_tokens, max_recv_tokens = self.receive_capacity(
            max_num_tokens=max_num_tokens, num_experts=num_experts, expert_padding=expert_padding,
            num_experts_per_token=num_experts_per_token, world_size=world_size, dp_size=self._dp_size,
            max_private_tokens=max_private_tokens)
        self.max_recv_tokens = max_recv_tokens
        self.max_private_tokens = max_private_tokens

        if hidden_dim_scale is not None or scale_dtype is not None:
            assert scale_dtype is not None
            assert hidden_dim_scale is not None
            # the reference supports no other scale type either (p2p_all_to_all.py:164-165)
            assert scale_dtype == torch.float32

        device_index = self._device.index
        if device_index is None:
            device_index = torch.cuda.current_device()

        self._key = (
            hidden_dim, hidden_dim_scale, in_dtype, out_dtype, scale_dtype, max_num_tokens,
            max_recv_tokens, max_private_tokens, num_experts, expert_padding,
            num_experts_per_token, node_size, world_size, device_index, self._dp_size,
        )

        def make_context() -> AllToAllContext:
            return AllToAllContext.create(
                hidden_dim=hidden_dim,
                hidden_dim_scale=hidden_dim_scale,
                in_elemsize=in_dtype.itemsize,
                out_elemsize=out_dtype.itemsize,
                out_dtype=out_dtype,
                scale_elemsize=scale_dtype.itemsize if scale_dtype else None,
                max_num_tokens=max_num_tokens,
                max_recv_tokens=max_recv_tokens,
                max_private_tokens=max_private_tokens,
                num_experts=num_experts,
                expert_padding=expert_padding,
                num_experts_per_token=num_experts_per_token,
                dp_size=self._dp_size,
                node_size=node_size,
                world_size=world_size,
                device=device_index,
                flags=getattr(global_group.world, "context_flags", 0),
            )

        self._all_to_all = global_group.world.acquire_context(self._key, make_context)
        # dispatch() and combine() themselves: checks and calls in native code (a2a_torch.cpp)
        extension = load_extension()
        _call_without_a_frame(extension)
        self._operator = extension.Operator(
            self._all_to_all.shared, rank, self._dp_size, hidden_dim,
            -1 if hidden_dim_scale is None else hidden_dim_scale, self._num_local_experts, num_experts_per_token,
            in_dtype, out_dtype, scale_dtype is not None, -1 if self._device.index is None else self._device.index)

    # ------------------------------------------------------------------

    @staticmethod
    def receive_capacity(*, max_num_tokens: int, num_experts: int, expert_padding: int,
                         num_experts_per_token: int, world_size: int, dp_size: int = 1,
                         max_private_tokens: Optional[int] = None):
        """(max_private_tokens, max_recv_tokens): rows of a rank's receive region as the reference
        sizes them (p2p_all_to_all.py:94-114).  Every dp group gets a private region (by default 1.2
        times the average load of the rank's experts); on top of that come the rows all groups share:
        every copy of every group's tokens could land here, but no more than one per (token, local
        expert), and never less than one padded block per local expert."""
        groups = world_size // dp_size
        local_experts = ceil_div(num_experts, world_size)
        if max_private_tokens is None:
            average = int(ceil_div(max_num_tokens * num_experts_per_token, num_experts) * 1.2)
            max_private_tokens = average * local_experts
        assert max_private_tokens >= 0
        tokens = max_num_tokens * groups
        every_copy = tokens * num_experts_per_token + local_experts * (expert_padding - 1)
        shared = max(min(every_copy, tokens * local_experts), local_experts * expert_padding)
        return max_private_tokens, max_private_tokens * groups + round_up(shared, expert_padding)

    @property
    def num_local_experts(self) -> int:
        return self._num_local_experts

    @property
    def context(self) -> AllToAllContext:
        assert self._all_to_all is not None
        return self._all_to_all

    def dispatch(
        self,
        out_expert_num_tokens: torch.Tensor,
        out_expert_x: torch.Tensor,
        out_expert_x_scale: Optional[torch.Tensor],
        dp_x: torch.Tensor,
        dp_x_scale: Optional[torch.Tensor],
        indices: torch.Tensor,
        weights: torch.Tensor,
        bound_m: Optional[torch.Tensor] = None,
        do_send: bool = True,
        do_recv: bool = True,
    ) -> None:
        assert self._operator is not None
        self._operator.dispatch(out_expert_num_tokens, out_expert_x, out_expert_x_scale, dp_x, dp_x_scale, indices,
                                weights, bound_m, do_send, do_recv)

    def combine(
        self,
        out_tokens: torch.Tensor,
        indices: torch.Tensor,
        weights: torch.Tensor,
        expert_y: torch.Tensor,
        bound_m: Optional[torch.Tensor] = None,
        do_send: bool = True,
        do_recv: bool = True,
        accumulate: bool = False,
    ) -> None:
        assert self._operator is not None
        self._operator.combine(out_tokens, indices, weights, expert_y, bound_m, do_send, do_recv, accumulate)

    def destroy(self) -> None:
        """Release this rank's share of the context; the last rank frees it."""
        if self._all_to_all is not None:
            self._all_to_all = None
            self._operator = None
            self._global_group.world.release_context(self._key)


_DEFINED = (P2PAllToAll.dispatch, P2PAllToAll.combine)


def _call_without_a_frame(extension) -> None:
    """From the first operator on, calls of these two functions on an operator that is not destroyed run the native operator's
    methods (same names, defaults and checks) without a Python frame; the functions stay the objects they are."""
    for function in _DEFINED:
        extension.call_without_a_frame(function)
