"""``LoopbackWorld``: all simulated ranks of one world behind one object.

The per-rank ``AllToAll`` API costs one Python -> C call per rank and step.  A caller that
owns every rank anyway (a single-GPU MoE layer, a benchmark, a captured decode step) can
hand all ranks' tensors over at once; the library then makes one pass over them
(``pplx_a2a_world_dispatch`` / ``pplx_a2a_world_combine``).  The kernels, the results and
the argument checks are the same as for ``world_size`` per-rank calls.  The checks, the packing
and the launch run in compiled code: packed in Python, a step of four ranks took 33 us of host
time for 10 us of kernels (now 9 us a step), and a bound step 13 us (now 9).

``capture()`` records whatever the body enqueues on the current stream into a hipGraph
through the library's own capture entry points, so a step can be replayed without any
host-side argument handling (the reference's "CUDA graph support", ``README.md:5``).
"""

from __future__ import annotations

import contextlib
import ctypes
from collections.abc import Sequence

import torch

from . import ops
from .all_to_all import AllToAll

_launch_bound = ops._C.launch_bound
_launch_plan = ops._C.launch_plan


class Graph:
    """An instantiated hipGraph of a recorded step."""

    def __init__(self, ptr: int) -> None:
        self._ptr = ptr

    def replay(self, stream: torch.cuda.Stream | None = None) -> None:
        assert self._ptr is not None
        s = stream if stream is not None else torch.cuda.current_stream()
        ops.check_status(ops.load_library().pplx_a2a_graph_launch(self._ptr, s.cuda_stream))

    def destroy(self) -> None:
        if self._ptr is not None:
            ptr, self._ptr = self._ptr, None
            ops.check_status(ops.load_library().pplx_a2a_graph_destroy(ptr))

    def __del__(self) -> None:
        try:
            self.destroy()
        except Exception:
            pass


class BoundStep:
    """One step's arguments of all ranks, checked and packed once: ``dispatch()`` and
    ``combine()`` then cost one library call each, with no per-rank work in Python.  The eager
    alternative to :class:`Graph` for a caller whose buffers stay where they are from step to
    step (on this stack a graph replay costs more host time than two eager launches).  The
    tensors are kept alive by the object; their contents may change between calls, their
    addresses, shapes and strides may not."""

    def __init__(self, world: "LoopbackWorld", dispatch_args, combine_args, device, keep: tuple) -> None:
        # (what the launches read: packed for this world, which is named by a number of its own)
        self._keep = (dispatch_args, combine_args, keep)
        packed = ctypes.addressof(dispatch_args), ctypes.addressof(combine_args)
        # The kernels of launches on this stream read the rank tables from device memory, which the allocator gives out
        # again, to this stream, once the step is gone; launches on others, or under capture, carry the tables along.
        self._tables = plan = None
        if device.type == "cuda":
            self._tables = ops._C.step_tables(world._world_id, device.index)
        if self._tables is not None:
            plan = ops._C.bind_step(
                world._world_id, *packed, self._tables.data_ptr(), torch.cuda.current_stream(device).cuda_stream
            )
        if plan is not None:
            self._launch = _launch_plan
            self._launch_dispatch = (0, world._world_id, plan, device.index)
            self._launch_combine = (1, world._world_id, plan, device.index)
        else:
            self._launch = _launch_bound
            self._launch_dispatch = (0, world._world_id, packed[0], device.index)
            self._launch_combine = (1, world._world_id, packed[1], device.index)

    def dispatch(self, stream: torch.cuda.Stream | None = None) -> None:
        self._launch(*self._launch_dispatch, None if stream is None else stream.cuda_stream)

    def combine(self, stream: torch.cuda.Stream | None = None) -> None:
        self._launch(*self._launch_combine, None if stream is None else stream.cuda_stream)


class LoopbackWorld:
    def __init__(
        self,
        max_num_tokens: int,
        num_experts: int,
        experts_per_token: int,
        world_size: int,
        dp_size: int,
        hidden_dim: int,
        hidden_dim_bytes: int,
        hidden_dim_scale_bytes: int,
        group_name: str = "loopback",
    ) -> None:
        self.world_size = world_size
        self.dp_size = dp_size
        self.experts_per_token = experts_per_token
        self.ranks = [
            AllToAll.intranode(
                max_num_tokens,
                num_experts,
                experts_per_token,
                r,
                world_size,
                dp_size,
                hidden_dim,
                hidden_dim_bytes,
                hidden_dim_scale_bytes,
                group_name,
            )
            for r in range(world_size)
        ]
        self._world_id = ops._C.world_id(self.ranks[0]._ptr)

    def dispatch(
        self,
        out_expert_num_tokens: Sequence[torch.Tensor],
        out_expert_x: Sequence[torch.Tensor],
        out_expert_x_scale: Sequence[torch.Tensor | None],
        dp_x: Sequence[torch.Tensor],
        dp_x_scale: Sequence[torch.Tensor | None],
        indices: Sequence[torch.Tensor],
        bound_m: Sequence[torch.Tensor | None],
    ) -> None:
        """Entry ``r`` of every sequence is rank ``r``'s argument of ``AllToAll.dispatch``."""
        ops._C.world_dispatch(
            self._world_id, out_expert_num_tokens, out_expert_x, out_expert_x_scale, dp_x, dp_x_scale, indices, bound_m
        )

    def combine(
        self,
        out_tokens: Sequence[torch.Tensor],
        indices: Sequence[torch.Tensor],
        weights: Sequence[torch.Tensor],
        expert_y: Sequence[torch.Tensor],
        bound_m: Sequence[torch.Tensor | None],
    ) -> None:
        """Entry ``r`` of every sequence is rank ``r``'s argument of ``AllToAll.combine``."""
        ops._C.world_combine(self._world_id, out_tokens, indices, weights, expert_y, bound_m)

    def bind(
        self,
        out_expert_num_tokens: Sequence[torch.Tensor],
        out_expert_x: Sequence[torch.Tensor],
        out_expert_x_scale: Sequence[torch.Tensor | None],
        dp_x: Sequence[torch.Tensor],
        dp_x_scale: Sequence[torch.Tensor | None],
        indices: Sequence[torch.Tensor],
        bound_m: Sequence[torch.Tensor | None],
        out_tokens: Sequence[torch.Tensor],
        weights: Sequence[torch.Tensor],
        expert_y: Sequence[torch.Tensor],
    ) -> BoundStep:
        """Checks and packs the arguments of :meth:`dispatch` and :meth:`combine` once and
        returns a :class:`BoundStep` that launches them as often as wanted, fastest on the stream
        that is current now: the rank tables are written to device memory there (by two small kernels,
        unless the stream is captured), and the step's kernels read them.  Binding takes 18 us of the
        host for one rank, 60 for 8 and 390 for 64, 10 of them for the tables, which save about 1 us a
        step: a step that is bound for fewer than some ten launches loses by them."""
        d_args = (ops.DispatchArgs * self.world_size)()
        c_args = (ops.CombineArgs * self.world_size)()
        for r in range(self.world_size):
            ops.pack_dispatch_args(
                self.experts_per_token, out_expert_num_tokens[r], out_expert_x[r], out_expert_x_scale[r],
                dp_x[r], dp_x_scale[r], indices[r], bound_m[r], out=d_args[r],
            )  # fmt: skip
            ops.pack_combine_args(out_tokens[r], indices[r], weights[r], expert_y[r], bound_m[r], out=c_args[r])
        keep = tuple(
            list(seq)
            for seq in (out_expert_num_tokens, out_expert_x, out_expert_x_scale, dp_x, dp_x_scale, indices,
                        bound_m, out_tokens, weights, expert_y)
        )  # fmt: skip
        return BoundStep(self, d_args, c_args, indices[0].device, keep)

    def faults(self) -> int:
        """Sticky device-side fault bits since the last call (synchronises the stream):
        1 = a routed row did not fit ``out_expert_x.size(1)``, 2 = an expert index was out of
        range, 4 = combine met a slot beyond ``expert_y.size(1)``, 8 = an expert id repeated
        inside one token was dropped, 16 = a ``bound_m`` beyond ``max_num_tokens`` was clamped."""
        return ops._C.world_faults(self._world_id, torch.cuda.current_stream().cuda_stream)

    @contextlib.contextmanager
    def capture(self):
        """Records the body's launches on the current stream; yields a holder whose
        ``graph`` attribute is the instantiated :class:`Graph` after the block."""
        lib = ops.load_library()
        stream = torch.cuda.current_stream().cuda_stream
        if stream == 0:
            raise RuntimeError(
                "pplx_kernels: the default stream cannot be captured; enter "
                "`with torch.cuda.stream(torch.cuda.Stream()):` first"
            )

        class _Holder:
            graph: Graph | None = None

        holder = _Holder()
        ops.check_status(lib.pplx_a2a_graph_begin_capture(stream))
        try:
            yield holder
        finally:
            ptr = ctypes.c_void_p()
            ops.check_status(lib.pplx_a2a_graph_end_capture(stream, ctypes.byref(ptr)))
            holder.graph = Graph(ptr.value)

    def destroy(self) -> None:
        for r in self.ranks:
            r.destroy()
        self.ranks = []
