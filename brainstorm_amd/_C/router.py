"""``brt._C.router`` -- same names, arguments, defaults and error behaviour as the
pybind11 module of the reference (src/backend/torch/router.cc:479-513,
python/brt/_C/router.pyi), implemented over the C ABI of ``libbrt_hip.so``.

PyTorch is used for tensor allocation and stream handles only; every device
computation of the seat-index path is a hand-written HIP kernel.  Argument checks,
output allocation and launches live in ``csrc/native.cpp``.  Work is
enqueued on the current PyTorch stream (the reference uses the default stream,
router.cc:78; identical when no stream context is active).
"""
from __future__ import annotations

import itertools
from typing import List, Optional, Tuple

import torch

from brainstorm_amd import _lib

_DT = {torch.float32: _lib.F32, torch.float16: _lib.F16, torch.bfloat16: _lib.BF16}

__all__ = [
    "topk_hot_mask",
    "throttle_hotmask",
    "top1_to_capacity",
    "top1_route_to_capacity",
    "Route",
    "CompactRoute",
    "remember_route",
    "route_of_loads",
    "generate_route",
    "generate_indices_and_loads",
    "convert_index_format",
    "dispatch_with_indices_and_loads",
    "route_and_dispatch",
    "dispatch_rows_of_route",
    "combine_by_row_tags",
    "split_fused_cells_to_paths",
    "fuse_split_cells_from_paths",
    "combine_with_indices_and_loads",
    "combine_flows",
    "combine_with_src_indices",
    "gate_topk",
    "route_by_path",
    "dispatch_by_rows",
    "combine_by_rows",
]


# --------------------------------------------------------------------- helpers
def _check_on_device(t: torch.Tensor, name: str) -> None:
    # CHECK_ON_CUDA, src/backend/torch/torch.h:16-21
    if not t.is_cuda:
        raise RuntimeError(f"{name} must be a CUDA tensor")


def _check_int32(t: torch.Tensor, name: str) -> None:
    if t.dtype != torch.int32:  # data_ptr<int>() in the reference throws likewise
        raise RuntimeError(f"{name} must be an int32 tensor, got {t.dtype}")


def _ptr(t: Optional[torch.Tensor]):
    return None if t is None else t.data_ptr()


def _stream() -> int:
    """Raw handle of the current stream of the current device (the ops run under a guard for
    the tensors' device).  The private accessor avoids building a ``torch.cuda.Stream``."""
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


class _NoGuard:
    def __enter__(self):
        return None

    def __exit__(self, *exc):
        return False


_NO_GUARD = _NoGuard()


def _device_guard(device: torch.device):
    """``CUDAGuard`` of the reference bindings (router.cc:55,144,384); free when the tensors
    already live on the current device."""
    if device.index is None or device.index == torch._C._cuda_getDevice():
        return _NO_GUARD
    return torch.cuda.device(device)


class Route:
    """What one index-generation call knows about a route, beyond the ``(indices, loads)`` pair
    the reference returns: the true per-path counts (``loads`` may be padded), whether a cell can
    be on more than one path, and -- once a dispatch or a gathering GEMM has run -- the cell
    behind every row of the path-major layout.  Fabrics carry it next to the stacks of the routed
    GridTensor and hand it to dispatch / combine with the ``route=`` keyword; without it those ops
    take their general forms (pre-zeroed output, index-driven combine)."""

    __slots__ = ("indices", "loads", "counts", "is_tag_index", "single_path", "cells", "paths",
                 "row_tags", "row_tags_stride", "host_loads", "_versions")

    def __init__(self, indices, loads, counts, is_tag_index, single_path):
        self.indices, self.loads, self.counts = indices, loads, counts
        self.is_tag_index = bool(is_tag_index)
        self.single_path = bool(single_path)
        self.cells, self.paths = indices.shape
        self.row_tags = None        # [P] int32: 1-based cell of each row of the layout, 0 = no cell
        self.row_tags_stride = 0    # max_path_load the rows were laid out with (0 = packed)
        self.host_loads = None      # the values of loads, once a dispatch has read them
        self._versions = (indices._version, loads._version)

    def owns(self, route_indices: torch.Tensor, loads: torch.Tensor) -> bool:
        """True when the pair is the one this route was generated with, unmodified since."""
        return (route_indices is self.indices and loads is self.loads
                and self._versions == (route_indices._version, loads._version))


class CompactRoute:
    """A route kept as ``k`` path ids per cell from the gate to the combine (an extension; the
    reference carries a ``[cells, paths]`` hot mask and seat matrix, python/brt/router/fabric/fused.py:32-75):
    what ``gate_topk`` chose and ``route_by_path`` laid out.  ``seat_rows[t, j]`` is the 1-based
    row of the path-major layout that entry ``(t, j)`` owns (0: dropped), ``row_entries[r]`` the
    1-based entry ``t * k + j + 1`` behind row ``r`` (0: padding).  ``indices`` is the dense seat
    matrix the reference would have produced, generated on first read."""

    __slots__ = ("path_ids", "weights", "loads", "counts", "seat_rows", "row_entries", "k", "cells",
                 "paths", "single_path", "indices", "combined_into", "__weakref__")

    def __init__(self, path_ids, weights, loads, counts, seat_rows, row_entries, paths, indices):
        self.path_ids, self.weights = path_ids, weights
        self.loads, self.counts, self.seat_rows, self.row_entries = loads, counts, seat_rows, row_entries
        self.cells, self.k = path_ids.shape
        self.paths = int(paths)
        self.single_path = self.k == 1
        self.indices = indices       # lazily filled [cells, paths] seat indices (what the stacks carry)
        self.combined_into = None    # the tensor an expert kernel already stored the combined rows to

    def owns(self, route_indices, loads) -> bool:
        return route_indices is self.indices and loads is self.loads


# Routes by the identity of their loads tensor: an expert kernel receives the loads as its
# capacities and finds the route of its rows through them.  Both sides are held weakly: the route
# lives as long as the routed GridTensor carries it, and the entry goes when the loads tensor does.
_routes_by_loads = {}


def remember_route(loads: torch.Tensor, route) -> None:
    import weakref

    key = id(loads)

    def forget(_ref, key=key, table=_routes_by_loads):
        table.pop(key, None)

    _routes_by_loads[key] = (weakref.ref(loads, forget), weakref.ref(route))


def route_of_loads(loads: torch.Tensor):
    """The route that was generated with this very loads tensor, or None."""
    entry = _routes_by_loads.get(id(loads))
    if entry is not None and entry[0]() is loads:
        return entry[1]()
    return None


_fallback_logged = set()


def _log_general_form(op: str, why: str) -> None:
    if op not in _fallback_logged:
        _fallback_logged.add(op)
        from brainstorm_amd.runtime.log import get_logger
        get_logger(__file__).info("%s runs in its general form: %s", op, why)


def _route_for(route: Optional["Route"], route_indices, loads, op: str) -> Optional["Route"]:
    if route is None:
        _log_general_form(op, "no route object was passed (route=None)")
        return None
    if not route.owns(route_indices, loads):
        _log_general_form(op, "the route object does not describe these indices / loads any more")
        return None
    return route


# ------------------------------------------------------------------------- ops
def topk_hot_mask(score: torch.Tensor, top_k: int) -> torch.Tensor:
    """Not in the reference's extension: the hot mask of ``TopKProtocol``
    (protocol/topk.py:26-31: ``topk`` + ``zeros_like`` + ``scatter_``) in one kernel.  int32
    ``[cells, paths]`` with ones at the ``top_k`` largest scores of every row; NaN ranks
    highest, equal scores go to the lowest path."""
    return _lib.native().topk_hot_mask(score, int(top_k))


def throttle_hotmask(
    hot_mask: torch.Tensor, prefix: torch.Tensor, threshold: torch.Tensor
) -> Tuple[torch.Tensor, torch.Tensor]:
    """router.cc:15-31.  ``prefix`` is updated in place and returned."""
    return _lib.native().throttle_hotmask(hot_mask, prefix, threshold), prefix


def top1_to_capacity(score: torch.Tensor, capacity: int):
    """Not in the reference's extension: ``topk_hot_mask(score, 1)`` throttled from a zero prefix to ``capacity``
    cells of every path, and the capacity of every path as an int32 vector (swin_moe.py:101-126), in two launches; None
    where the fused kernels do not take the shape."""
    return _lib.native().top1_to_capacity(score, int(capacity))


def top1_route_to_capacity(score: torch.Tensor, capacity: int, capacity_padding: bool, path_wise_padding: bool):
    """:func:`top1_to_capacity` whose second launch also lays out the seats of the throttled mask (not in the reference):
    the same pair, and the :class:`Route` that ``generate_route`` would make of it."""
    made = _lib.native().top1_route_to_capacity(score, int(capacity), bool(capacity_padding), bool(path_wise_padding))
    if made is None:
        return None
    mask, capacities, seats, loads, counts = made
    return mask, capacities, Route(seats, loads, counts, False, True)


def generate_route(
    hot_mask: torch.Tensor,
    supported_capacities: Optional[torch.Tensor] = None,
    capacity_padding: bool = False,
    path_wise_padding: bool = False,
    is_tag_index: bool = False,
    single_path: bool = False,
) -> Route:
    """Index generation (router.cc:48-80) returning the :class:`Route`.  ``single_path`` is the
    caller's promise that no row of ``hot_mask`` has more than one nonzero; dispatch and combine
    calls that receive the route may then use the tag-driven combine (same results, one memory
    round trip less)."""
    indices, loads, counts = _lib.native().generate(
        hot_mask, supported_capacities, capacity_padding, path_wise_padding, is_tag_index)
    return Route(indices, loads, counts, is_tag_index, single_path)


def generate_indices_and_loads(
    hot_mask: torch.Tensor,
    supported_capacities: Optional[torch.Tensor] = None,
    capacity_padding: bool = False,
    path_wise_padding: bool = False,
    is_tag_index: bool = False,
) -> Tuple[torch.Tensor, torch.Tensor]:
    """router.cc:48-80."""
    route = generate_route(hot_mask, supported_capacities, capacity_padding, path_wise_padding,
                           is_tag_index)
    return route.indices, route.loads


def convert_index_format(
    origin_indices: torch.Tensor, loads: torch.Tensor, is_to_tag: bool
) -> torch.Tensor:
    """router.cc:90-110.

    As built, the reference forwards ``is_to_tag`` into the launcher's
    ``tag_to_seat`` parameter (router.cc:104-107 vs location.cu:317-333), so
    ``is_to_tag=True`` runs the tag->seat kernel.  This entry point keeps that
    behaviour; use :func:`seat_to_tag_indices` / :func:`tag_to_seat_indices` for
    the direction their names say.
    """
    return _convert(origin_indices, loads, tag_to_seat=bool(is_to_tag))


def seat_to_tag_indices(seat_indices: torch.Tensor, loads: torch.Tensor) -> torch.Tensor:
    return _convert(seat_indices, loads, tag_to_seat=False)


def tag_to_seat_indices(tag_indices: torch.Tensor, loads: torch.Tensor) -> torch.Tensor:
    return _convert(tag_indices, loads, tag_to_seat=True)


def _convert(origin_indices, loads, tag_to_seat: bool) -> torch.Tensor:
    _check_on_device(origin_indices, "origin_indices")
    _check_int32(origin_indices, "origin_indices")
    origin_indices = origin_indices.contiguous()
    T, E = origin_indices.shape
    with _device_guard(origin_indices.device):
        dev_loads = loads
        if tag_to_seat:
            _check_int32(loads, "loads")
            dev_loads = loads.to(origin_indices.device, non_blocking=True).contiguous()
        new_indices = torch.zeros_like(origin_indices)
        _lib.check(_lib.lib().brt_hip_convert_index_format(
            _ptr(origin_indices), _ptr(new_indices), _ptr(dev_loads) if tag_to_seat else None,
            T, E, int(tag_to_seat), _stream()))
    return new_indices


def dispatch_with_indices_and_loads(
    in_data: torch.Tensor,
    route_indices: torch.Tensor,
    loads: torch.Tensor,
    gates: Optional[torch.Tensor] = None,
    tag_generating: bool = False,
    tags: Optional[torch.Tensor] = None,
    max_path_padding: bool = False,
    max_path_load: int = 0,
    is_1d_routing: bool = True,
    is_tag_index: bool = False,
    *,
    route: Optional[Route] = None,
    rows: Optional[int] = None,
    host_loads: Optional[List[int]] = None,
    likely_rows: Optional[int] = None,
) -> List[torch.Tensor]:
    """router.cc:131-273.  Returns ``[out]`` or ``[out, new_tags]``.  ``route`` (keyword only,
    not in the reference): the :class:`Route` the indices came from; the kernel then zero-fills
    only the padding rows of an un-zeroed output and, for single-path routes, leaves the per-row
    tags on the route for the combine.  ``rows`` (keyword only, not in the reference): an upper
    bound of ``sum(loads)`` known to the caller; the output then has that many rows (those past
    the loads are zero) and the loads are not read back to the host (router.cc:197-201 sizes
    the output from ``loads.sum().item()``, which stalls the stream; that is what happens without
    ``rows``).  ``host_loads`` (likewise): the values of ``loads``, where the caller has just read them.
    ``likely_rows`` (likewise): as many rows as ``sum(loads)`` will hardly exceed; while the host waits for the loads, the rows
    are moved into room for that many already, of which the result is the first ``sum(loads)`` (all of them are moved
    again where the room did not do)."""
    _check_on_device(in_data, "in_data")
    _check_on_device(route_indices, "route_indices")
    _check_int32(route_indices, "route_indices")
    if in_data.size(0) == 0:
        return _dispatch_of_no_cells(in_data, route_indices, tag_generating, is_1d_routing)
    if in_data.dtype not in _DT:  # TORCH_CHECK_NOT_IMPLEMENTED, router.cc:266
        raise NotImplementedError("data type is not supported")
    counts = None
    hidden_tags = False  # the rows of a single-path route carry their tags to the combine
    if not is_tag_index:
        route = _route_for(route, route_indices, loads, "dispatch_with_indices_and_loads")
        if route is not None and not route.is_tag_index:
            counts = route.counts
            hidden_tags = route.single_path and is_1d_routing and not tag_generating
    _check_int32(loads, "loads")
    native = _lib.native()
    if (likely_rows is not None and counts is not None and is_1d_routing and not max_path_padding and rows is None
            and host_loads is None and loads.is_cuda and loads.numel() == route_indices.size(1)
            and likely_rows * (in_data.nbytes // in_data.size(0)) <= _MOST_ROOM):
        out, new_tags, route.host_loads = native.dispatch_and_read(
            in_data, route_indices, loads, counts, gates, tags if tag_generating else None,
            tag_generating or hidden_tags, likely_rows)
        if hidden_tags:
            route.row_tags, route.row_tags_stride = new_tags, 0
        return [out, new_tags] if tag_generating else [out]
    dev_loads = loads if loads.is_cuda else loads.to(in_data.device, non_blocking=True)
    # rows of the dispatched buffer (router.cc:189-202); data dependent, so one
    # host read of the loads unless a fixed per-path stride was given
    mpl = 0
    if max_path_padding:
        mpl = int(max_path_load) if max_path_load > 0 else max(native.int_list(loads))
        total = mpl * route_indices.size(1)
    elif rows is not None:
        total = int(rows)
    else:
        total = sum(native.int_list(loads) if host_loads is None else host_loads)
    # with the true counts the kernel writes every row up to sum(loads) itself; rows past that
    # (an upper bound was given) have no writer, and their tags start at zero
    clear = counts is None or (rows is not None and not max_path_padding)
    # tags None = arange(1, T+1) (router.cc:240-241), generated in the kernel
    out, new_tags = native.dispatch(in_data, route_indices, dev_loads, counts, gates,
                                    tags if tag_generating else None, tag_generating or hidden_tags,
                                    total, mpl, is_1d_routing, is_tag_index, clear)
    if hidden_tags:
        route.row_tags, route.row_tags_stride = new_tags, mpl
    return [out, new_tags] if tag_generating else [out]


# Room for rows that are moved before their number is known.  What the loads leave of it stays allocated as long as the
# result (whose storage ends with its rows), and the 4 to 7 us that it spares (1024 fp32 cells over 16 experts: scatter, FFN 512 -> 2048 and gather 67.6 -> 60.1 us, scatter and gather alone
# 46.3 -> 42.5; 2048 cells, two paths each, through the default routers 75.0 -> 71.1) are nothing beside rows of more bytes than these.
_MOST_ROOM = 1 << 26


def loads_on_host(loads: torch.Tensor) -> List[int]:
    """The values of an int32 loads vector (one wait for the stream's work so far)."""
    return _lib.native().int_list(loads)


def _dispatch_of_no_cells(in_data, route_indices, tag_generating, is_1d_routing):
    # router.cc:150-168
    shape = list(in_data.shape)
    if is_1d_routing:
        shape[0] = 0
    else:
        if len(shape) == 2:
            shape.append(1)
        shape[1] = 0
        shape = shape[1:]
    out = torch.zeros(shape, dtype=in_data.dtype, device=in_data.device)
    if tag_generating:
        return [out, torch.zeros((0,), dtype=route_indices.dtype, device=in_data.device)]
    return [out]


def route_and_dispatch(
    in_data: torch.Tensor,
    hot_mask: torch.Tensor,
    rows: int,
    supported_capacities: Optional[torch.Tensor] = None,
    capacity_padding: bool = False,
    path_wise_padding: bool = False,
    single_path: bool = False,
) -> Tuple[Route, torch.Tensor]:
    """Not in the reference: :func:`generate_route` (seat indices) and an unweighted 1-d
    :func:`dispatch_with_indices_and_loads` with ``rows=`` in one dependent step -- the second pass
    of the index scan moves the rows of its own cells (two launches instead of three, the index
    matrix is not read back).  Returns the route and the ``[rows, ...]`` path-major tensor, every
    row of it written (zeros where no cell owns the row); bit-identical to the two calls, which it
    makes itself for the shapes the fused kernel does not take."""
    rows = int(rows)
    done = _lib.native().route_and_dispatch(in_data, hot_mask, rows, supported_capacities, capacity_padding,
                                            path_wise_padding, single_path)
    if done is None:  # a shape the fused kernel does not take
        route = generate_route(hot_mask, supported_capacities, capacity_padding, path_wise_padding,
                               False, single_path)
        out = dispatch_with_indices_and_loads(in_data, route.indices, route.loads, route=route,
                                              rows=rows)[0]
        return route, out
    indices, loads, counts, out, row_tags = done
    route = Route(indices, loads, counts, False, single_path)
    if single_path:
        route.row_tags, route.row_tags_stride = row_tags, 0
    return route, out


def dispatch_rows_of_route(cells: torch.Tensor, route: Route, out: torch.Tensor) -> None:
    """The dispatch a deferred fused dispatch stands for (not in the reference): rows of ``cells``
    into the pre-allocated path-major ``out`` by the tag indices of ``route``; rows no path owns are
    zero; the row tags are left on the route."""
    if not route.is_tag_index:
        raise RuntimeError("a deferred dispatch holds tag indices")
    T = cells.size(0)
    rows = out.size(0)
    with _device_guard(cells.device):
        out.zero_()
        row_tags = torch.zeros((rows,), dtype=torch.int32, device=cells.device)
        if T > 0 and rows > 0:
            _lib.check(_lib.lib().brt_hip_dispatch(
                _ptr(cells), _ptr(out), None, _ptr(route.indices), _ptr(route.loads), None, None,
                _ptr(row_tags), T, cells.numel() // T, route.paths, rows, 0, 1, 1,
                _DT[cells.dtype], _stream()))
        route.row_tags, route.row_tags_stride = row_tags, 0


def combine_by_row_tags(in_data: torch.Tensor, row_tags: torch.Tensor, cells: int,
                        out_data: Optional[torch.Tensor] = None,
                        out_dtype: Optional[torch.dtype] = None) -> torch.Tensor:
    """Combine of a route in which no cell is on more than one path, from the per-row tags
    (not in the reference as an op; what its seat-index combine computes for such a route,
    route.cu:208-282): ``out[row_tags[p] - 1] = in_data[p]`` for every tagged row.  ``out_data``
    is updated in place (cells without a row keep their values); without it the result starts
    from zeros."""
    return _lib.native().combine_by_row_tags(in_data, row_tags, cells, out_data, out_dtype)


def split_fused_cells_to_paths(
    in_data: torch.Tensor,
    loads: torch.Tensor,
    max_path_padding: bool = False,
    is_load_split: bool = False,
    is_tag_split: bool = False,
    tags: Optional[torch.Tensor] = None,
    *,
    host_loads: Optional[List[int]] = None,
) -> List[List[torch.Tensor]]:
    """router.cc:285-335: per-path views (``narrow``) of the fused buffer.  ``host_loads`` (keyword only,
    not in the reference): the values of ``loads``, where the caller has just read them."""
    path_num = loads.numel()
    if is_tag_split:
        is_load_split = True
        if tags is None:
            raise RuntimeError("is_tag_split needs tags")
    # (where a compiler, tracer or mode looks on, the views are made by torch's own calls)
    native = None if torch.compiler.is_compiling() else _lib.native_or_none()
    if native is not None and not native.ordinary(in_data, loads, tags):
        native = None
    if max_path_padding:
        rows = [in_data.size(0) // path_num] * path_num
    elif host_loads is not None:
        rows = host_loads
    else:
        listed = native is not None and loads.dtype == torch.int32 and loads.dim() == 1
        rows = native.int_list(loads) if listed else loads.cpu().tolist()
    if native is not None:
        datas, load_list, tag_list = native.split_rows(
            in_data, rows, loads if is_load_split else None, tags if is_tag_split else None)
    else:
        starts = [0, *itertools.accumulate(rows)]
        datas = [in_data.narrow(0, s, n) for s, n in zip(starts, rows)]
        load_list = [loads.narrow(0, i, 1) for i in range(len(rows))] if is_load_split else []
        tag_list = [tags.narrow(0, s, n) for s, n in zip(starts, rows)] if is_tag_split else []
    if is_tag_split:
        return [datas, load_list, tag_list]
    if is_load_split:
        return [datas, load_list]
    return [datas]


def fuse_split_cells_from_paths(
    in_data: List[torch.Tensor],
    is_load_fuse: bool = False,
    is_tag_fuse: bool = False,
    loads: Optional[List[torch.Tensor]] = None,
    tags: Optional[List[torch.Tensor]] = None,
    *,
    tag_range: Optional[Tuple[int, int]] = None,
) -> List[torch.Tensor]:
    """router.cc:348-369.  ``tag_range`` (keyword only, not in the reference): the smallest and the largest tag, where the
    caller has just read them."""
    out_data = torch.cat(in_data, 0)
    if is_load_fuse:
        if loads is None:
            raise RuntimeError("is_load_fuse needs loads")
        return [out_data, torch.cat(loads, 0)]
    if is_tag_fuse:
        if tags is None:
            raise RuntimeError("is_tag_fuse needs tags")
        out_tags = torch.cat(tags, 0)
        new_tags, global_seat_indices = _unique_tags(out_tags, tag_range)
        return [out_data, new_tags, global_seat_indices]
    return [out_data]


_UNIQUE_WHOLE_MAX = 1 << 15  # BRT_UNIQUE_WHOLE_MAX


def _unique_tags(tags: torch.Tensor, tag_range: Optional[Tuple[int, int]] = None):
    """``torch.unique(tags, sorted=True, return_inverse=True)`` (router.cc:362-366) without the
    sort: tags are cell numbers, so a presence table over ``[min, max]`` and one prefix sum give
    the same two tensors.  Tag sets that are sparse in their range (or not a 1-d int32 / int64
    device vector) take the library call."""
    n = tags.numel()
    if not (tags.is_cuda and tags.dim() == 1 and n > 0 and tags.dtype in (torch.int32, torch.int64)):
        return torch.unique(tags, sorted=True, return_inverse=True)
    with _device_guard(tags.device):
        tags = tags.contiguous()
        if tag_range is not None:
            lo, hi = tag_range
        elif n <= _UNIQUE_WHOLE_MAX:  # one launch that finds the range itself, one read-back
            unique, inverse, lo, hi = _lib.native().unique_tags(tags)
            if unique is not None:
                return unique, inverse
        else:
            lo, hi = (int(v) for v in torch.stack(torch.aminmax(tags)).tolist())
        span = hi - lo + 1
        ws_bytes = _lib.lib().brt_hip_unique_tags_workspace_bytes(lo, hi)
        if ws_bytes == 0 or span > 16 * n + (1 << 16):
            return torch.unique(tags, sorted=True, return_inverse=True)
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device=tags.device)
        unique = torch.empty(min(n, span), dtype=tags.dtype, device=tags.device)
        inverse = torch.empty(n, dtype=torch.int64, device=tags.device)
        count = torch.empty(1, dtype=torch.int32, device=tags.device)
        _lib.check(_lib.lib().brt_hip_unique_tags(
            _ptr(tags), 32 if tags.dtype == torch.int32 else 64, n, lo, hi, _ptr(ws), ws_bytes,
            _ptr(unique), _ptr(inverse), _ptr(count), _stream()))
        return unique[:int(count.item())], inverse


def combine_with_indices_and_loads(
    in_data: torch.Tensor,
    route_indices: torch.Tensor,
    loads: Optional[torch.Tensor] = None,
    gates: Optional[torch.Tensor] = None,
    out_data: Optional[torch.Tensor] = None,
    max_path_padding: bool = False,
    ever_padded: bool = True,
    is_tag_index: bool = False,
    tags: Optional[torch.Tensor] = None,
    *,
    out_dtype: Optional[torch.dtype] = None,
    route: Optional[Route] = None,
) -> List[torch.Tensor]:
    """router.cc:372-473.

    Seat mode runs the HIP gather kernel (fp32 accumulation in ascending path
    order).  ``out_dtype`` (keyword only, not in the reference) selects an fp32
    result for 16-bit inputs; with ``out_data`` the result dtype is that of
    ``out_data``.  Tag mode is the reference's ``scatter_reduce`` formulation.
    """
    _check_on_device(in_data, "in_data")
    _check_on_device(route_indices, "route_indices")
    T = route_indices.size(0)
    if T <= 1:
        if T == 0:  # router.cc:386-397
            if not is_tag_index:
                return [out_data if out_data is not None else torch.empty_like(in_data)]
            return [torch.empty_like(in_data), torch.empty_like(tags), torch.zeros_like(tags)]
        if not is_tag_index:  # router.cc:402-412
            return [out_data + in_data if out_data is not None else in_data]
        return [in_data, tags, torch.ones_like(tags)]
    if is_tag_index:
        with _device_guard(in_data.device):
            return _combine_with_tags(in_data, route_indices, out_data, ever_padded, tags)
    if loads is None:
        raise RuntimeError("seat-index combine needs loads")
    # single-path routes whose rows still carry the tags of the paired dispatch: scatter form
    route = _route_for(route, route_indices, loads, "combine_with_indices_and_loads")
    row_tags = None
    if route is not None and route.single_path and route.row_tags is not None:
        P = in_data.size(0)
        mpl = P // route_indices.size(1) if max_path_padding else 0  # router.cc:427-430
        if route.row_tags.size(0) == P and route.row_tags_stride == mpl:
            row_tags = route.row_tags
    return [_lib.native().combine(in_data, route_indices, loads, gates, out_data, out_dtype,
                                  max_path_padding, row_tags)]


def _combine_with_tags(in_data, route_indices, out_data, ever_padded, tags):
    # router.cc:449-472
    if tags is None:
        raise RuntimeError("tag-index combine needs tags")
    tags_value = tags
    n = tags_value.size(0)
    if out_data is not None:
        _check_on_device(out_data, "out_data")
        if out_data.size(0) != n:
            raise RuntimeError("out_data must hold one row per unique tag")
        result = out_data
        # out-of-place and discarded, as in the reference (router.cc:456)
        cell = in_data.numel() // in_data.size(0)
        index = route_indices.view(-1, 1).repeat(1, cell).view_as(in_data)
        torch.scatter_reduce(result, 0, index, in_data, "sum", include_self=False)
    else:
        shape = list(in_data.shape)
        shape[0] = n
        result = _sum_rows_by_index(in_data, route_indices, n, shape)
        if ever_padded and int(tags_value[0].item()) == 0:
            result = result.narrow(0, 1, n - 1)
            tags_value = tags_value.narrow(0, 1, n - 1)
    return [result, tags_value, _lib.native().one_value(tags_value.numel(), in_data)]


def _sum_rows_by_index(in_data, index, n, shape):
    """``zeros(n, ...).scatter_reduce(0, index repeated per element, in_data, "sum")``
    (router.cc:451,459-460) as one pass over the rows: no per-element index tensor, rows added
    in ascending row order in fp32."""
    P = in_data.size(0)
    if (in_data.dtype not in _DT or index.dtype not in (torch.int32, torch.int64)
            or index.numel() != P or not index.is_cuda):
        cell = in_data.numel() // P
        expanded = index.view(-1, 1).repeat(1, cell).view_as(in_data)
        zeros = torch.zeros(shape, dtype=in_data.dtype, device=in_data.device)
        return torch.scatter_reduce(zeros, 0, expanded, in_data, "sum")
    return _lib.native().sum_rows_by_index(in_data, index, n)


def combine_flows(datas: List[torch.Tensor], tags: List[torch.Tensor], tag_range: Optional[list] = None) -> Optional[tuple]:
    """``fuse_split_cells_from_paths`` (router.cc:348-369) and the tag-mode combine (router.cc:449-472) of its result, from the
    flows where they are: ``(rows, tags, number of tags)``, bit for bit, or None where the general way is to be taken (other
    types, more than 64 flows or 8192 rows, tags too far apart, a compiler, tracer or mode that looks on).  Tags too far apart
    have been read: the smallest and the largest are appended to ``tag_range``."""
    if torch.compiler.is_compiling():
        return None
    native = _lib.native_or_none()
    made = None if native is None else native.combine_flows(datas, tags)
    if made is None or len(made) == 3:
        return made
    if tag_range is not None:
        tag_range.extend(made)
    return None


# legacy name (sample/cpp/router.ipynb:258-266) of the seat-index combine
combine_with_src_indices = combine_with_indices_and_loads


# ------------------------------------------------------- compact route format
# Not in the reference's extension.  The same route as hot mask + seat indices, held as k path
# ids per cell: ``path_ids [T, k]``, ``weights [T, k]`` (fp32), ``seat_rows [T, k]`` (1-based row of
# the dispatched buffer, 0 = dropped) and ``row_entries [P]`` (1-based entry ``t*k + j + 1`` of
# every dispatched row, 0 = padding; for ``k == 1`` these are the row tags of dispatch).
def gate_topk(score: torch.Tensor, top_k: int, softmax: bool = False,
              hot_mask: bool = False) -> Tuple[torch.Tensor, ...]:
    """``(path_ids, weights[, hot_mask])``: the ``top_k`` largest scores of every row in the order
    of ``torch.topk`` (NaN highest, lowest path among equals) and their weights -- the scores as
    fp32, or with ``softmax`` their softmax over the row (the router probabilities of
    benchmark/switch_moe/switch_transformer.py:240-253).  One kernel for what the reference does
    with ``softmax`` + ``topk`` / ``argmax`` + ``zeros`` + ``scatter_`` (protocol/topk.py:26-31)."""
    return _lib.native().gate_topk(score, top_k, softmax, hot_mask)


def route_by_path(
    path_ids: torch.Tensor,
    path_num: int,
    supported_capacities: Optional[torch.Tensor] = None,
    capacity_padding: bool = False,
    path_wise_padding: bool = False,
    max_path_load: int = 0,
    rows: Optional[int] = None,
) -> Tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor]:
    """``generate_indices_and_loads`` (router.cc:48-80) on path ids instead of a hot mask:
    ``(loads, counts, seat_rows, row_entries)``.  ``loads`` follow the same capacity rules,
    ``counts`` are the real rows per path.  ``rows`` is the length of the dispatched buffer:
    ``path_num * max_path_load`` when padding every path to ``max_path_load``, else by default
    ``cells * k``, which always holds the ``sum(loads)`` rows of a route without capacity padding
    (no read-back of the loads is needed to size it; rows behind the last path are padding)."""
    return _lib.native().route_by_path(path_ids, int(path_num), supported_capacities, capacity_padding,
                                       path_wise_padding, int(max_path_load), rows)


def dispatch_by_rows(in_data: torch.Tensor, row_entries: torch.Tensor, k: int,
                     weights: Optional[torch.Tensor] = None,
                     out: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``out[r] = in_data[(row_entries[r]-1) // k]`` (times ``weights.view(-1)[row_entries[r]-1]``,
    rounded once), zero rows where ``row_entries[r] == 0``: what ``dispatch_with_indices_and_loads``
    (router.cc:131-273) writes for the same route, every row written by the kernel."""
    return _lib.native().dispatch_by_rows(in_data, row_entries, int(k), weights, out)


def combine_by_rows(in_data: torch.Tensor, path_ids: torch.Tensor, seat_rows: torch.Tensor,
                    weights: Optional[torch.Tensor] = None, out_data: Optional[torch.Tensor] = None,
                    out_dtype: Optional[torch.dtype] = None, *,
                    gates: Optional[torch.Tensor] = None) -> torch.Tensor:
    """``out[t] = sum_j weights[t,j] * in_data[seat_rows[t,j]-1]`` over the entries that own a row,
    in ascending path id, fp32 from zero: the result of ``combine_with_indices_and_loads``
    (router.cc:372-473) for the same route, bit for bit.  With ``out_data`` the result is
    written in place and cells without a row keep their value (the residual convention).
    ``gates`` (the ``[cells, paths]`` matrix, any data type) gives the weights instead:
    ``gates[t, path_ids[t,j]]``; it has a column for every path id (the ids are not read back to check it)."""
    if gates is not None and weights is not None:
        raise RuntimeError("weights or gates, not both")
    if gates is not None and not (gates.dtype in _DT and gates.dim() == 2 and gates.size(0) == path_ids.size(0)
                                  and gates.numel() < 1 << 31):
        # what the kernel does not read in place: other types (fp64 gates), more rows than cells
        weights, gates = torch.gather(gates, 1, path_ids.long()).to(torch.float32), None
    return _lib.native().combine_by_rows(in_data, path_ids, seat_rows, weights, out_data, out_dtype, gates)
