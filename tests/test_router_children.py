"""Routers call the protocol and the fabric that their attributes name at the call (no GPU needed)."""
import pytest

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
