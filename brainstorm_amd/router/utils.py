"""Small helpers shared by routers, protocols and fabrics
(reference: python/brt/router/utils.py)."""
import weakref
from typing import Any, Dict, List, Optional

import numpy as np
import torch

__all__ = ["pad_to_max", "make_kwargs", "empty_flows", "assert_compatibility", "mark_paths", "paths_per_cell"]


def pad_to_max(tensors: List[torch.Tensor], pad_value=0) -> List[torch.Tensor]:
    """Zero-pads every tensor's flattened cell to the largest cell among them."""
    sizes = [t.numel() // t.size(0) for t in tensors]
    widest = int(np.argmax(sizes))
    target, target_shape = sizes[widest], tensors[widest].shape[1:]
    out = []
    for t, size in zip(tensors, sizes):
        flat = torch.nn.functional.pad(t.view(t.size(0), -1), (0, target - size), value=pad_value)
        out.append(flat.view(t.size(0), *target_shape))
    return out


def make_kwargs(kwargs: Optional[Dict[str, Any]]) -> Dict[str, Any]:
    if kwargs is None:
        return {}
    if isinstance(kwargs, dict) and all(isinstance(k, str) for k in kwargs):
        return kwargs
    raise ValueError(f"kwargs should be a dict of str to Any, but got {kwargs}")


def empty_flows(in_flows) -> bool:
    while isinstance(in_flows, list):
        if not in_flows:
            return True
        in_flows = in_flows[0]
    return False


def assert_compatibility(instance, k, expected_v, given_v) -> None:
    assert expected_v == given_v, (
        f"compatibility check failed for {type(instance).__name__}, caused by keyword "
        f"argument {k}: expected {expected_v}, given {given_v}")


class _PathMark(tuple):
    """(the paths that a row of one mask has at most, the mask's version counter, a weak reference to it).  It holds for that
    tensor object as it stood: not for a copy, whose version counter starts anew and may agree with that of another state (a
    pickled mark comes back as an empty set)."""

    __slots__ = ()

    def __reduce__(self):
        return set, ()


def mark_paths(hot_mask: torch.Tensor, most: int) -> None:
    """Notes on a hot mask that, as it stands, no row of it has more than ``most`` nonzeros.  The note is worth nothing once the
    mask is edited in place (by a forward hook, or between protocol and fabric), so it goes with the mask's version counter; a
    tensor that has none is not marked."""
    try:
        hot_mask._brt_paths_per_cell = _PathMark((most, hot_mask._version, weakref.ref(hot_mask)))
    except RuntimeError:  # an inference tensor
        return
    if most == 1:
        hot_mask._brt_single_path = True


def paths_per_cell(hot_mask) -> int:
    """The paths that a row of the mask has at most, by a mark that still holds; 0 where that is not known."""
    mark = getattr(hot_mask, "_brt_paths_per_cell", None)
    if type(mark) is not _PathMark or mark[1] != hot_mask._version or mark[2]() is not hot_mask:
        return 0
    return mark[0]
