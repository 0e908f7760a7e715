"""Routers call the protocol and the fabric that their attributes name at the call (no GPU needed)."""
import copy

import pytest
import torch.nn as nn

from brainstorm_amd.router import GatherRouter, ScatterRouter


def _mark(name):
    return lambda *args: (name, *args) if name == "protocol" else ((name, *args), None)


def test_routers_call_children_that_are_plain_callables():
    scatter, gather = ScatterRouter(), GatherRouter()
    del scatter.protocol, scatter.fabric, gather.fabric
    scatter.protocol, scatter.fabric, gather.fabric = _mark("protocol"), _mark("dispatch"), _mark("combine")
    assert scatter("flow", "score") == ("dispatch", "flow", ("protocol", "score"), None, "score")
    assert gather("flows")[0] == ("combine", "flows", None, None)


@pytest.mark.parametrize("swapped", ["protocol", "fabric"])
def test_routers_call_children_that_a_subclass_names(swapped):
    class Scatter(ScatterRouter):
        pass

    class Gather(GatherRouter):
        fabric = property(lambda self: _mark("property"), lambda self, value: None)

    setattr(Scatter, swapped, property(lambda self: _mark("protocol" if swapped == "protocol" else "property"),
                                       lambda self, value: None))
    scatter = Scatter(protocol_type="identity") if swapped == "fabric" else Scatter()
    if swapped == "protocol":
        del scatter.fabric
        scatter.fabric = _mark("dispatch")
        assert scatter("flow", "score") == ("dispatch", "flow", ("protocol", "score"), None, "score")
    else:
        assert scatter("flow", "score")[0] == "property"
    assert Gather()("flows")[0] == ("property", "flows", None, None)


def test_children_of_routers_are_ordinary_modules():
    gather = GatherRouter()
    assert [name for name, _ in gather.named_children()] == ["fabric"] and list(gather.state_dict()) == []
    other = copy.deepcopy(gather)
    assert type(other.fabric) is type(gather.fabric) and other.fabric is not gather.fabric
    gather.fabric = other.fabric
    assert gather.fabric is other.fabric and gather._modules["fabric"] is other.fabric
    gather._modules["fabric"] = nn.Identity()  # as passes that replace modules do
    assert isinstance(gather.fabric, nn.Identity)
    gather.fabric = None
    assert gather.fabric is None
    del gather.fabric
    assert not hasattr(gather, "fabric")
    with pytest.raises(AttributeError, match="'GatherRouter' object has no attribute 'fabric'"):
        gather.fabric
    gather.add_module("fabric", other.fabric)
    assert gather.fabric is other.fabric
