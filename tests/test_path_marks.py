"""What a hot mask's mark promises holds for the mask as the fabric receives it (no GPU needed)."""
import copy
import io

import pytest
import torch

from brainstorm_amd._C import router as c_router
from brainstorm_amd.router.fabric import make_fabric
from brainstorm_amd.router.protocol import make_protocol
from brainstorm_amd.router.protocol._impl import CompactHotMask, ProtocolBase, TopKProtocol
from brainstorm_amd.router.utils import paths_per_cell


class _Seen(Exception):
    pass


def _single_path_of(monkeypatch, mask, fabric_type="dispatch", **kwargs):
    """What the fabric promises index generation about this mask."""
    def generate_route(hot_mask, **kw):
        raise _Seen(kw["single_path"])

    def route_and_dispatch(*args, **kw):
        raise _Seen(kw["single_path"])

    monkeypatch.setattr(c_router, "generate_route", generate_route)
    monkeypatch.setattr(c_router, "route_and_dispatch", route_and_dispatch)
    fabric = make_fabric(fabric_type, {"flow_num": 1, **kwargs})
    with pytest.raises(_Seen) as seen:
        fabric(torch.zeros(mask.shape[0], 8), mask)
    return seen.value.args[0]


_FORMS = [("dispatch", {}), ("fused_dispatch", {}), ("fused_dispatch", {"static_rows": True}),
          ("fused_dispatch", {"defer_dispatch": True})]


@pytest.mark.parametrize("fabric_type,kwargs", _FORMS)
@pytest.mark.parametrize("edit", [lambda m: m.fill_(1), lambda m: m[:, 0].fill_(1), lambda m: m.__setitem__((3, 2), 1)])
def test_an_edit_in_place_ends_the_mark(monkeypatch, fabric_type, kwargs, edit):
    protocol = make_protocol("topk", {"top_k": 1})
    score = torch.randn(9, 4)
    mask = protocol(score)
    assert paths_per_cell(mask) == 1 and _single_path_of(monkeypatch, mask, fabric_type, **kwargs)
    protocol.register_forward_hook(lambda module, args, out: (edit(out), None)[1])
    mask = protocol(score)
    assert paths_per_cell(mask) == 0 and not _single_path_of(monkeypatch, mask, fabric_type, **kwargs)


def test_a_decision_of_a_subclass_does_not_inherit_the_promise():
    class WithSharedPath(TopKProtocol):
        def make_route_decision(self, score):
            return torch.maximum(super().make_route_decision(score), torch.tensor([1, 0, 0], dtype=torch.int32))

    class Edits(TopKProtocol):
        def make_route_decision(self, score):
            mask = super().make_route_decision(score)
            mask[:, 0] = 1
            return mask

    for protocol in (WithSharedPath(top_k=1), Edits(top_k=1)):
        assert paths_per_cell(protocol(torch.randn(5, 3))) == 0


def test_the_mark_is_that_of_the_paths_taken_at_the_call():
    protocol = make_protocol("topk", {"top_k": 1})
    protocol.top_k = 2
    assert paths_per_cell(protocol(torch.randn(5, 3))) == 2


def test_protocols_that_promise_are_marked():
    class Own(ProtocolBase):
        single_path = True

        def make_route_decision(self, score):
            return torch.ones(score.shape[0], 1, dtype=torch.int32), None

    mask, _ = Own()(torch.randn(4, 1))
    assert paths_per_cell(mask) == 1
    given = torch.eye(4, dtype=torch.int32)
    assert paths_per_cell(make_protocol("switch_top1", {"one_hot": True})(given)) == 1
    assert paths_per_cell(make_protocol("switch_top1", {})(given)) == 0 and paths_per_cell(given) == 0
    dense = CompactHotMask(torch.tensor([[1], [0]], dtype=torch.int32), torch.ones(2, 1), 3).dense()
    assert paths_per_cell(dense) == 1
    dense.fill_(1)
    assert paths_per_cell(dense) == 0


def test_masks_without_a_version_counter_are_not_marked():
    with torch.inference_mode():
        mask = make_protocol("topk", {"top_k": 1})(torch.randn(5, 3))
    assert paths_per_cell(mask) == 0 and int(mask.sum()) == 5


def _saved_and_loaded(mask):
    file = io.BytesIO()
    torch.save(mask, file)
    file.seek(0)
    return torch.load(file, weights_only=True)


@pytest.mark.parametrize("copied", [copy.copy, copy.deepcopy, _saved_and_loaded])
@pytest.mark.parametrize("edits", range(4))
def test_copies_do_not_inherit_the_mark(monkeypatch, copied, edits):
    """The version counter of a copy starts anew: what it says of the copy says nothing about what was done to the mask."""
    mask = make_protocol("topk", {"top_k": 1})(torch.randn(5, 3))
    for _ in range(edits):
        mask.fill_(1)
    other = copied(mask)
    assert torch.equal(other, mask) and paths_per_cell(other) == 0
    assert not _single_path_of(monkeypatch, other)
    assert paths_per_cell(mask) == (0 if edits else 1)


@pytest.mark.parametrize("fullgraph", [False, True])
def test_a_compiled_decision_is_marked(fullgraph):
    protocol = make_protocol("topk", {"top_k": 1})
    mask = torch.compile(protocol, backend="eager", fullgraph=fullgraph)(torch.randn(6, 4))
    assert paths_per_cell(mask) == 1
    mask[0] = 1
    assert paths_per_cell(mask) == 0


@pytest.mark.parametrize("one_hot", [False, True])
def test_protocols_saved_before_they_made_their_marks_run(one_hot):
    """A protocol object whose attributes are those of an earlier version: `single_path` where there is `one_hot` now."""
    protocol = make_protocol("switch_top1", {"one_hot": one_hot})
    del protocol.__dict__["one_hot"]
    protocol.single_path = one_hot
    assert paths_per_cell(protocol(torch.eye(4, dtype=torch.int32))) == (1 if one_hot else 0)
    protocol = make_protocol("topk", {"top_k": 1})
    protocol.single_path = True
    assert paths_per_cell(protocol(torch.randn(5, 3))) == 1
