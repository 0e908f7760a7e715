"""``brt.jit``: the homo-fused expert kernel as one grouped GEMM.

The reference glues per-capacity TVM-tuned fp32 ``Linear`` kernels into one NVRTC
kernel and launches it through ``brt._C.jit.homo_invoke``
(python/brt/jit/factory.py:28-44, python/brt/jit/compiler.py:29-31,
src/jit/compiler.cu:151-246).  Here ``make_jit_kernel(..., opt_level="homo_fuse")``
returns a callable with the same shape

    kernel(shared_inputs=[x, out], standalone_inputs=[w0, (b0,) w1, ...], capacities=loads)

that runs ONE hand-written bf16 MFMA grouped GEMM over all branches; the loads
are read on the device, need not come from a menu of compiled capacities, and no
host copy or per-launch pointer shuffling happens.  Other fusion levels of the
reference (horizontal / hetero fusion, the TVM kernel database) are not part of
this build.
"""
from typing import Callable, List, Optional, Sequence, Union

import torch
import torch.nn as nn

from brainstorm_amd import _lib
from brainstorm_amd._C import router as c_router
from brainstorm_amd.runtime import deferred

__all__ = ["make_jit_kernel", "grouped_linear", "GroupedLinearKernel"]

_ACT = {None: _lib.ACT_NONE, "none": _lib.ACT_NONE, "gelu": _lib.ACT_GELU, "relu": _lib.ACT_RELU}


def grouped_linear(x: torch.Tensor, out: torch.Tensor, weight_table: torch.Tensor,
                   bias_table: Optional[torch.Tensor], loads: torch.Tensor, in_features: int,
                   out_features: int, activation: Optional[str] = None, *,
                   tags: Optional[torch.Tensor] = None, gather: bool = False,
                   scatter: bool = False, rows: Optional[int] = None,
                   row_entries: Optional[torch.Tensor] = None, entries_per_cell: int = 1,
                   row_tags_out: Optional[torch.Tensor] = None,
                   gates: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``out[s_e : s_e + loads[e]] = act(x[s_e : s_e + loads[e]] @ W_e^T + b_e)`` for every
    branch e, ``s_e = sum(loads[:e])``, in one launch.  ``weight_table`` /
    ``bias_table`` are int64 device tensors holding the branch pointers.

    With ``tags`` (the ``[cells, paths]`` tag-index matrix of
    ``generate_indices_and_loads(..., is_tag_index=True)``) the routing is folded into the
    GEMM: ``gather=True`` reads row s of branch e from ``x[tags[s, e] - 1]`` (``x`` is the
    cell-major tensor, no dispatch needed), ``scatter=True`` stores it to
    ``out[tags[s, e] - 1]`` (``out`` is cell-major and doubles as the residual; single-path
    routes only).  ``rows`` bounds ``sum(loads)``; it must be given when neither side is path-major.

    ``row_entries`` (the vector ``route_by_path`` writes: 1-based entry ``t * k + j + 1`` of every
    row of the dispatched layout, ``k = entries_per_cell``) names the rows instead of ``tags``:
    row r is cell ``(row_entries[r] - 1) // k``.

    ``out`` may be fp32 (tag-matrix and plain forms): it then receives the fp32 accumulator after
    bias and activation.  ``row_tags_out`` (``[rows]`` int32, tag-matrix form) receives the
    1-based cell behind every row of the layout, which is what a later tag-driven combine needs.

    ``gates`` (fp32, ``[cells, paths]`` beside ``tags`` or ``[cells, k]`` beside ``row_entries``) with
    ``scatter=True`` and an fp32 ``out`` folds the weighted combine of a route with several paths
    per cell into the store (route.cu:236-243): ``out[cell] += gate * bf16(row)`` by fp32 atomic
    adds, so ``out`` must hold zeros (or what the sums are added to) before the call.  Equal to
    ``combine_with_indices_and_loads`` on the separate GEMM's output: bit for bit with at most two
    paths per cell, to the last bits of an fp32 sum taken in another order with more."""
    _lib.native().grouped_linear(
        x, out, weight_table, bias_table, loads, in_features, out_features, _ACT[activation], tags, gather,
        scatter, rows, row_entries, int(entries_per_cell), row_tags_out, gates)
    return out


def _linear(x, out, weight_table, bias_table, loads, in_features, out_features, activation, *, tags=None, gather=False,
            rows=None, row_entries=None, entries_per_cell=1, row_tags_out=None) -> None:
    """:func:`grouped_linear` that takes fp32 rows of ``x`` too: they are rounded to bf16 first, by the kernel for few
    rows itself and by the cast kernel for the others."""
    _lib.native().grouped_linear_f32(
        x, out, weight_table, bias_table, loads, in_features, out_features, _ACT[activation], tags, gather,
        False, rows, row_entries, entries_per_cell, row_tags_out, None)


def _to_bf16(t: torch.Tensor) -> torch.Tensor:
    """fp32 -> bf16 (round to nearest even) with the library's cast kernel."""
    return _lib.native().cast_f32_to_bf16(t)


class _BranchOperands:
    """Device array of the branches' pointers, rebuilt only when the tensors change; fp32 branches are
    converted to bf16 copies then."""

    def __init__(self, what: str):
        self.what = what
        self.key = None
        self.table = None
        self.sources = None  # converted tensors are held, so their addresses cannot be reused unnoticed
        self.copies = None

    def get(self, operands: Sequence[torch.Tensor], first: int, step: int, used: int) -> torch.Tensor:
        fp32, key = _lib.native().branch_key(operands, first, step, used, self.what)
        if key != self.key:
            tensors = list(operands[first::step])
            sources = copies = None
            if fp32:
                sources = tensors[:used]
                tensors = copies = [_to_bf16(t.detach()) for t in sources]
            table = torch.tensor([t.data_ptr() for t in tensors], dtype=torch.int64, device=tensors[0].device)
            # all of it or nothing: a conversion that fails leaves the copies behind the old key and table alive
            self.sources, self.copies, self.table, self.key = sources, copies, table, key
        return self.table


class GroupedLinearKernel:
    """Callable returned by ``make_jit_kernel(ModuleList[Linear], ..., "homo_fuse")``.

    The reference's kernels take and give fp32 (benchmark/switch_moe/switch_expert.py:74-92
    allocates its outputs with ``torch.empty`` in the default dtype; test/python/jit_test.py:157-203
    runs fp32 throughout).  This kernel multiplies bf16 operands on the matrix units with fp32
    accumulation: fp32 shared inputs and fp32 branch parameters are converted to bf16 first (the
    parameters once, until they change), and an fp32 output tensor receives the fp32 accumulator.
    Against fp32 ``F.linear`` the result is within 1e-2 relative (bf16 operand rounding)."""

    def __init__(self, in_features: int, out_features: int, has_bias: bool,
                 activation: Optional[str] = None):
        self.in_features = in_features
        self.out_features = out_features
        self.has_bias = has_bias
        self.activation = activation
        self._weights = _BranchOperands("weights")
        self._biases = _BranchOperands("biases")

    def __call__(self, shared_inputs: List[torch.Tensor], standalone_inputs: Sequence[torch.Tensor],
                 capacities: Union[torch.Tensor, Sequence[int]] = (), *,
                 residual: Optional[torch.Tensor] = None):
        """``residual`` (an extension, for the last kernel of an expert on a route with one path
        per cell): the cell-major tensor the gather router will be given as its residual.  The
        rows are then stored straight to their cells in it -- the combine folded into the store --
        and ``out`` is NOT written; the fused combine fabric recognises the tensor and launches
        nothing.  It needs the route of the rows, which is found through ``capacities`` (the loads
        tensor of the routed GridTensor, as it came off the load stack) and must stem from a fused
        dispatch fabric built with ``compact_route=True``."""
        x, out = shared_inputs
        if not isinstance(standalone_inputs, (list, tuple)):
            standalone_inputs = list(standalone_inputs)
        if not torch.is_tensor(capacities):
            capacities = torch.tensor(list(capacities), dtype=torch.int32, device=out.device)
        step = 2 if self.has_bias else 1
        used = capacities.numel()
        if used > (len(standalone_inputs) + step - 1) // step:
            raise RuntimeError("more capacities than branches")
        weights = self._weights.get(standalone_inputs, 0, step, used)
        biases = self._biases.get(standalone_inputs, 1, step, used) if self.has_bias else None
        loads = capacities
        if loads.dtype != torch.int32 or loads.device != out.device:
            loads = loads.to(device=out.device, dtype=torch.int32)
        if residual is not None:
            return self._store_to_cells(x, weights, biases, loads, capacities, residual)
        state = deferred.pending_of(x)  # a DeferredRows, or the routed GridTensor itself
        if state is not None and not self._can_gather(state, out):
            state.materialize()
            state = None
        if state is not None:
            # the rows of a deferred dispatch: read from the cells through the route
            route = state.route
            cells = state.cells
            if isinstance(route, c_router.CompactRoute):  # rows named by the row-entry vector
                _linear(cells, out, weights, biases, loads, self.in_features, self.out_features,
                        self.activation, row_entries=route.row_entries,
                        entries_per_cell=route.k, gather=True, rows=out.shape[0])
                return
            row_tags = torch.empty((out.shape[0],), dtype=torch.int32, device=out.device)
            _linear(cells, out, weights, biases, loads, self.in_features, self.out_features,
                    self.activation, tags=route.indices, gather=True,
                    rows=out.shape[0], row_tags_out=row_tags)
            route.row_tags, route.row_tags_stride = row_tags, 0
            return
        # (a deferred buffer is filled by this read)
        _linear(x, out, weights, biases, loads, self.in_features, self.out_features, self.activation)

    def _store_to_cells(self, x, weights, biases, loads, route_loads, residual):
        """The GEMM whose rows go straight to their cells in ``residual`` (combine folded in)."""
        route = c_router.route_of_loads(route_loads) if torch.is_tensor(route_loads) else None
        if not isinstance(route, c_router.CompactRoute) or route.k != 1:
            raise RuntimeError("residual= needs the loads tensor of a route with one path per cell from a "
                               "fused dispatch fabric built with compact_route=True")
        if (residual.dtype != torch.bfloat16 or not residual.is_contiguous() or residual.dim() != 2
                or residual.shape != (route.cells, self.out_features) or not residual.is_cuda):
            raise RuntimeError("the residual must be a contiguous bf16 [cells, out_features] device tensor")
        pending = deferred.pending_of(x)
        if pending is not None:
            pending.materialize()
        if x.dtype == torch.float32:
            x = _to_bf16(x)
        if x.shape[0] != route.row_entries.numel():
            raise RuntimeError("the input does not have the rows of the dispatched layout")
        grouped_linear(x, residual, weights, biases, loads, self.in_features,
                       self.out_features, self.activation, row_entries=route.row_entries,
                       entries_per_cell=1, scatter=True, rows=x.shape[0])
        route.combined_into = residual

    def _can_gather(self, state, out: torch.Tensor) -> bool:
        cells = state.cells
        return (cells.dim() == 2 and cells.shape[1] == self.in_features and out.dim() == 2
                and out.shape[0] == state.buffer.shape[0] and out.is_contiguous()
                and cells.dtype in (torch.bfloat16, torch.float32)
                # rows that the row-entry vector names are written in bf16 only
                and (out.dtype == torch.bfloat16 or (out.dtype == torch.float32 and not isinstance(state.route, c_router.CompactRoute))))


def make_jit_kernel(modules, sample_inputs=None, method: str = "forward", opt_level=None,
                    objective_func: str = "fastest", rank=1, activation: Optional[str] = None
                    ) -> Callable[..., None]:
    """Signature of the reference (python/brt/jit/factory.py:28-44).  Only
    ``opt_level="homo_fuse"`` over ``nn.Linear`` branches of one shape is built;
    ``sample_inputs``, ``objective_func`` and ``rank`` (tuning knobs of the
    reference's kernel database) are accepted and ignored.  ``activation`` (not in
    the reference) fuses GELU / ReLU into the epilogue."""
    if opt_level != "homo_fuse" or method != "forward":
        raise NotImplementedError("only opt_level='homo_fuse', method='forward' is built")
    branches = list(modules) if isinstance(modules, (nn.ModuleList, list, tuple)) else [modules]
    if not branches or not all(isinstance(m, nn.Linear) for m in branches):
        raise NotImplementedError("homo_fuse is built for nn.Linear branches")
    shapes = {(m.in_features, m.out_features, m.bias is not None) for m in branches}
    if len(shapes) != 1:
        raise ValueError("homo_fuse needs branches of one shape")
    (in_features, out_features, has_bias), = shapes
    return GroupedLinearKernel(in_features, out_features, has_bias, activation)
