"""GridTensor / Annotator / Registry behaviour (scenarios of the reference's
test/python/grid_tensor_test.py:13-71), CPU only."""
import os

import pytest
import torch
import torch.nn as nn

import brt
from brainstorm_amd import _lib
from brt.runtime.grid_tensor import GridTensor, init_grid_tensor, deinit_grid_tensor
from brt.runtime import Registry


def test_annotator_shapes_and_initial_stacks():
    x = torch.randn(2, 3, 4, 5)
    a = brt.Annotator([0])(x)
    assert isinstance(a, GridTensor) and a.shape == (2, 3, 4, 5)
    assert a.tag_stack == [None] and a.load_stack == [None] and a.stack_size == 1
    b = brt.Annotator([0, 1])(x)
    assert b.shape == (6, 4, 5)
    c = brt.Annotator([1, 3])(x)  # cell dims moved to the front, rest = cell shape
    assert c.shape == (15, 2, 4)
    assert torch.equal(c[0 * 5 + 1], x[:, 0, :, 1])
    d = brt.Annotator([0], cell_shape=[60])(x)
    assert d.shape == (2, 60)
    e = brt.Annotator([0], gridding=False)(x)
    assert not isinstance(e, GridTensor)
    assert brt.Annotator([0])(a).stack_size == 2  # annotating twice pushes a level


def test_pack_unpack_and_deep_variants():
    t = init_grid_tensor(torch.arange(6.0).view(3, 2))
    assert t.annotation_empty()
    tag, load = torch.tensor([1, 2, 3]), torch.tensor([3])
    t.pack(tag, load, extra=7)
    assert t.tag is tag and t.load is load and t.get_extra_attr("extra") == 7
    t.set_extra_attr("extra", 8)
    _, tag2, load2, extra = t.unpack("extra")
    assert tag2 is tag and load2 is load and extra == {"extra": 8} and t.annotation_empty()
    t.deep_pack([tag, None], [load, None])
    assert t.stack_size == 2
    plain, tags, loads, _ = deinit_grid_tensor(t)
    assert type(plain) is torch.Tensor and tags == [tag, None] and loads == [load, None]
    with pytest.raises(AssertionError):
        init_grid_tensor(torch.zeros(1)).unpack()


@pytest.mark.parametrize("shallow", [True, False])
def test_stacks_travel_through_torch_ops(shallow):
    old = GridTensor.SHALLOW_TRANSPORT
    GridTensor.SHALLOW_TRANSPORT = shallow
    try:
        x = brt.Annotator([0])(torch.randn(4, 10))
        tag = torch.arange(1, 5, dtype=torch.int32)
        x.tag, x.load = tag, torch.tensor([4])
        y = nn.Linear(10, 3)(x)
        z = torch.relu(y) + 1
        assert isinstance(z, GridTensor) and z.tag is tag
        assert (z.tag_stack is x.tag_stack) == shallow
        a, b = z.split(2, dim=0)
        assert isinstance(a, GridTensor) and b.tag is tag
        plain = brt.to_torch_tensor(z)
        assert type(plain) is torch.Tensor
        again = brt.to_grid_tensor(plain, *brt.to_torch_tensor(z, True)[1:])
        assert again.tag is tag
    finally:
        GridTensor.SHALLOW_TRANSPORT = old


def test_registry_names():
    from brt.router.base import RouterBase
    from brt.router.fabric import FabricBase, make_fabric
    from brt.router.protocol import ProtocolBase, make_protocol

    routers = Registry.sub_cls_registries[RouterBase]
    assert {"scatter", "gather", "swin_moe_scatter", "task_scatter"} <= set(routers)
    fabrics = Registry.sub_cls_registries[FabricBase]
    assert {"dispatch", "combine", "fused_dispatch", "fused_combine", "identity_dispatch",
            "identity_combine", "single_cell_dispatch", "single_cell_combine",
            "placeholder_combine", "distributed_fused_dispatch",
            "distributed_fused_combine"} <= set(fabrics)
    protocols = Registry.sub_cls_registries[ProtocolBase]
    assert {"topk", "switch_top1", "threshold", "residual_threshold", "binary_threshold", "hash",
            "task", "swin_moe", "label", "identity", "decoder_greedy_search"} <= set(protocols)
    assert make_protocol("topk", {"top_k": 2}).top_k == 2
    assert make_fabric("fused_combine", {"flow_num": 1}).is_tag_index is False
    assert make_fabric("combine", {"flow_num": 1}).is_tag_index is True
    with pytest.raises(ValueError):
        make_fabric("dispatch", {1: 2})
    assert brt.router.is_router(brt.router.ScatterRouter)


def test_router_defaults():
    from brt.router import GatherRouter, ScatterRouter, SwinMoEScatterRouter

    s = ScatterRouter()
    assert s.protocol_kwargs == {"top_k": 1}
    assert s.fabric_kwargs == {"flow_num": 1, "route_logic": "1d", "transform": False}
    s = ScatterRouter(dispatch_score=True, protocol_type="threshold")
    assert s.protocol_kwargs == {"threshold": 0.0, "residual_path": -1}
    assert s.fabric_kwargs == {"flow_num": 2, "route_logic": ["1d", "2d"], "transform": [False, False]}
    g = GatherRouter()
    assert g.fabric_kwargs == {"flow_num": 1, "reduction": "add", "sparse": False}
    w = SwinMoEScatterRouter(protocol_kwargs={"capacity_factor": 1.25})
    assert w.protocol.top_k == 1 and w.fabric.max_path_load == 0
    assert w.protocol.runtime_capacity(100352, 8) == 15680


def test_protocol_masks_on_cpu():
    from brt.router.protocol import make_protocol

    score = torch.tensor([[0.1, 0.7, 0.2], [0.6, 0.3, 0.1], [0.2, 0.2, 0.6]])
    assert make_protocol("topk", {"top_k": 1})(score).tolist() == [[0, 1, 0], [1, 0, 0], [0, 0, 1]]
    assert make_protocol("topk", {"top_k": 2})(score).sum(1).tolist() == [2, 2, 2]
    m = make_protocol("threshold", {"threshold": 0.5})(score)
    assert m.dtype == torch.int32 and m.tolist() == [[0, 1, 0], [1, 0, 0], [0, 0, 1]]
    m = make_protocol("threshold", {"threshold": 0.65, "residual_path": 2})(score)
    assert m.tolist() == [[0, 1, 0], [0, 0, 1], [0, 0, 1]]
    m = make_protocol("switch_top1", {})(torch.eye(3).view(1, 3, 3))
    assert m.dtype == torch.int32 and m.shape == (3, 3)
    m = make_protocol("label", {"path_num": 4})(torch.tensor([3, 0]))
    assert m.tolist() == [[0, 0, 0, 1], [1, 0, 0, 0]]
    m = make_protocol("task", {"num_tasks": 3})(torch.tensor([2, 2, 0]))
    assert m.tolist() == [[0, 0, 1], [0, 0, 1], [1, 0, 0]]
    h = make_protocol("hash", {"num_tasks": 4, "placement_aware": True})
    assert h(torch.tensor([3])).tolist() == [[1, 0, 0, 1]]
    m = make_protocol("residual_threshold", {"threshold": 0.0, "residual_path": 0})(
        torch.tensor([[-1.0, 0.0], [1.0, 0.0]]))
    assert m.tolist() == [[1, 0], [0, 1]]  # below the threshold -> path 0 (the residual path)
    m = make_protocol("binary_threshold", {"threshold": 0.9, "selected_path": 1})(
        torch.tensor([[10.0, 0.0], [0.1, 0.0]]))
    assert m.tolist() == [[0, 1], [1, 0]]  # confident rows take the selected path


def test_module_paths_of_the_reference_resolve():
    """Code written against the reference imports its classes from the modules it keeps them in
    (python/brt/router/fabric/fused.py, protocol/topk.py, ...)."""
    import importlib

    for path, attr in (("brt.router.fabric.fused", "FusedDispatchFabric"),
                       ("brt.router.fabric.generic", "DispatchFabric"),
                       ("brt.router.fabric.base", "make_fabric"),
                       ("brt.router.fabric.distributed", "DistributedFusedCombineFabric"),
                       ("brt.router.protocol.topk", "TopKProtocol"),
                       ("brt.router.protocol.swin_moe", "SwinMoEProtocol"),
                       ("brt.router.protocol.base", "make_protocol"),
                       ("brainstorm_amd.router.protocol.hashed", "HashProtocol")):
        module = importlib.import_module(path)
        assert hasattr(module, attr), path
    from brt.router.fabric.fused import FusedCombineFabric  # noqa: F401
    from brt.router.protocol.switch import SwitchTop1Protocol  # noqa: F401


def test_deferred_buffer_fills_itself_before_any_read_and_not_for_metadata():
    """Host logic of the deferred dispatch (no GPU: the dispatch itself is replaced by a counter).
    Shape, dtype, device leave the buffer alone; an operator on the plain tensor or on the
    GridTensor that wraps it fills it first, and so does anything that hands out its address
    (data_ptr, stride, storage_offset: a foreign kernel could read through them); afterwards
    nothing is deferred any more."""
    import brt
    from brainstorm_amd.runtime import deferred

    class State(deferred.DeferredState):
        __slots__ = ("fills",)

        def materialize(self):
            if not self.done:
                self.fills += 1
                self.buffer.fill_(7.0)
                self.done = True

    def make():
        cells = torch.zeros(4, 3)
        state = State(cells, route=None, buffer=torch.empty(6, 3), key="brt_deferred_0")
        state.fills = 0
        grid = brt.to_grid_tensor(state.buffer, [torch.zeros(1)], [torch.zeros(1)], {"brt_deferred_0": state})
        return state, grid

    state, grid = make()
    assert tuple(grid.shape) == (6, 3) and grid.dtype == torch.float32 and state.fills == 0
    plain, tags, loads, extra = brt.to_torch_tensor(grid, retrieve_attr=True)
    assert isinstance(plain, deferred.DeferredRows) and deferred.state_of(plain) is state
    assert plain.shape[0] == 6 and plain.device.type == "cpu" and plain.is_contiguous() and state.fills == 0
    total = plain.sum()                      # a read: the dispatch runs first
    assert state.fills == 1 and float(total) == 7.0 * 18 and deferred.state_of(plain) is None
    assert type(plain + 1) is torch.Tensor   # results are ordinary tensors
    again = brt.to_torch_tensor(grid)        # nothing pending any more: a plain tensor
    assert type(again) is torch.Tensor and state.fills == 1

    state, grid = make()
    doubled = grid * 2                       # an operator on the GridTensor fills it too
    assert state.fills == 1 and float(brt.to_torch_tensor(doubled).sum()) == 14.0 * 18
    assert isinstance(doubled, brt.GridTensor) and doubled.extra_attr_dict["brt_deferred_0"] is state

    for read in (lambda t: t.data_ptr(), lambda t: t.stride(), lambda t: t.storage_offset()):
        state, grid = make()
        read(grid)                           # the address of the GridTensor: filled first
        assert state.fills == 1
        state, grid = make()
        plain = brt.to_torch_tensor(grid)
        assert state.fills == 0
        read(plain)                          # ... and of the plain tensor
        assert state.fills == 1
    state, grid = make()
    assert deferred.pending_of(grid) is state and deferred.pending_of(brt.to_torch_tensor(grid)) is state
    assert deferred.pending_of(torch.ones(2)) is None and state.fills == 0

    state, grid = make()
    product = torch.matmul(input=grid, other=torch.ones(3, 2))  # operands passed by keyword only
    assert state.fills == 1 and float(product.sum()) == 7.0 * 3 * 12
    assert isinstance(product, brt.GridTensor) and product.extra_attr_dict["brt_deferred_0"] is state

    state, grid = make()
    other = torch.ones(6, 3)
    assert deferred.pending_state(grid.extra_attr_dict, other) is None  # another tensor is not the buffer
    assert deferred.wrap_if_pending(other, grid.extra_attr_dict) is other and state.fills == 0


@pytest.mark.parametrize("shape", [(5, 0), (0, 0), (3, 0, 2)])
def test_annotator_refuses_cells_of_no_elements(shape):
    """Their number cannot be told from the number of elements."""
    with pytest.raises(RuntimeError, match="ambiguous"):
        brt.Annotator([0])(torch.zeros(shape))


def test_annotator_takes_no_cells():
    cells = brt.Annotator([0])(torch.zeros(0, 7))
    assert tuple(cells.shape) == (0, 7) and cells.tag_stack == [None]


@pytest.mark.parametrize("built", [True, False])
def test_flows_are_wrapped_the_same_with_and_without_the_native_module(monkeypatch, built):
    """Wrapping shares storage and stacks, copies the extra attributes, keeps autograd's link, and leaves a buffer that
    is not filled yet alone -- in native code and, where that has not been built, in Python."""
    from brainstorm_amd.runtime import deferred

    if not built:
        monkeypatch.setattr(_lib, "native_or_none", lambda: None)
    elif _lib.native_or_none() is None:
        pytest.skip("the native module has not been built")
    base = torch.randn(4, 3, requires_grad=True)
    tags, loads, extra = [None], [torch.tensor([4])], {"key": 1}
    grid = init_grid_tensor(base, tags, loads, extra)
    assert type(grid).__name__ == "GridTensor" and grid.data_ptr() == base.data_ptr()
    assert grid.tag_stack is tags and grid.load_stack is loads
    assert grid.extra_attr_dict == extra and grid.extra_attr_dict is not extra
    plain, got_tags, got_loads, _ = brt.to_torch_tensor(grid, retrieve_attr=True)
    assert type(plain) is torch.Tensor and got_tags is tags and got_loads is loads
    plain.sum().backward()
    assert torch.equal(base.grad, torch.ones_like(base))
    filled = []
    lazy = deferred.lazy_tensor(torch.zeros(3), lambda b: filled.append(b.fill_(2.0)))
    assert not filled and lazy.shape == (3,)
    assert float(lazy.sum()) == 6.0 and len(filled) == 1


@pytest.mark.parametrize("sizes", [[2, 0, 3], [0, 0], [5], [1] * 7])
def test_fused_cells_are_split_the_same_with_and_without_the_native_module(monkeypatch, sizes):
    """Rows, loads and tags of every path as views: loads read or handed over, on a fixed stride, of a tensor whose gradient is
    asked for and of one that is not contiguous."""
    import brt._C.router as c_router

    if _lib.native_or_none() is None:
        pytest.skip("the native module has not been built")
    n, loads = sum(sizes), torch.tensor(sizes, dtype=torch.int32)
    tags = torch.arange(1, n + 1, dtype=torch.int32)
    for rows in (torch.randn(n, 3), torch.randn(n, 3, requires_grad=True), torch.randn(3, n).t(), torch.randn(n)):
        for kwargs in ({}, {"is_load_split": True}, {"is_tag_split": True, "tags": tags}, {"host_loads": sizes}, {"max_path_padding": True}):
            native = c_router.split_fused_cells_to_paths(rows, loads, **kwargs)
            with monkeypatch.context() as patch:
                patch.setattr(_lib, "native_or_none", lambda: None)
                plain = c_router.split_fused_cells_to_paths(rows, loads, **kwargs)
            assert [len(part) for part in native] == [len(part) for part in plain]
            for got, want in zip(sum(native, []), sum(plain, [])):
                assert torch.equal(got, want) and got.data_ptr() == want.data_ptr() and got.stride() == want.stride()
                assert got.requires_grad == want.requires_grad and type(got) is torch.Tensor


def test_loads_without_data_are_refused():
    """Fake and meta tensors have no words that a split could go by."""
    import brt._C.router as c_router
    from torch._subclasses.fake_tensor import FakeTensorMode

    loads, rows = torch.tensor([2, 0, 3], dtype=torch.int32), torch.zeros(5, 2)
    with pytest.raises(NotImplementedError):
        c_router.split_fused_cells_to_paths(rows, loads.to("meta"))
    with pytest.raises(Exception, match="_local_scalar_dense"):  # what reading a fake tensor raises
        c_router.split_fused_cells_to_paths(rows, FakeTensorMode().from_tensor(loads))
    if os.path.exists(_lib.NATIVE_PATH):
        for nothing in (loads.to("meta"), FakeTensorMode().from_tensor(loads)):
            with pytest.raises(NotImplementedError):
                _lib.native().int_list(nothing)


def _observed_passes():
    import brt._C.router as c_router
    from brainstorm_amd.runtime import deferred

    loads = torch.tensor([2, 0, 3], dtype=torch.int32)
    return {
        "annotate": lambda x: brt.to_torch_tensor(brt.Annotator([0])(x)) * 2,
        "wrap": lambda x: brt.to_torch_tensor(init_grid_tensor(x, [None], [loads], {}), retrieve_attr=True)[0] * 2,
        "lazy": lambda x: deferred.lazy_tensor(x, lambda rows: None) * 2,
        "split": lambda x: torch.cat([r * 2 for r in c_router.split_fused_cells_to_paths(x, loads)[0]]),
        "split with loads": lambda x: torch.cat(c_router.split_fused_cells_to_paths(x, loads, is_load_split=True)[0]) * 2,
    }


@pytest.mark.parametrize("name", list(_observed_passes()))
def test_flows_under_modes_and_tracers(name):
    """Wrapping and splitting work where a dispatch mode, a function mode or a tracer looks on, which see of them
    what they see without the native module."""
    from torch.fx.experimental.proxy_tensor import make_fx
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class Dispatched(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    class Called(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(getattr(func, "__name__", str(func)))
            return func(*args, **(kwargs or {}))

    run, x = _observed_passes()[name], torch.arange(10.0).view(5, 2)
    for mode in (Dispatched, Called):
        logs = []
        for native in (_lib.native_or_none, lambda: None):
            seen = []
            with pytest.MonkeyPatch.context() as patch, mode():
                patch.setattr(_lib, "native_or_none", native)
                out = run(x)
            assert torch.equal(out, 2 * x)
            logs.append(seen)
        assert logs[0] == logs[1]
    assert torch.equal(make_fx(run)(x)(x), 2 * x)


def test_split_compiles_as_one_graph():
    run = _observed_passes()["split"]
    x = torch.arange(10.0).view(5, 2)
    assert torch.equal(torch.compile(run, backend="eager", fullgraph=True)(x), 2 * x)


def test_metadata_of_unfilled_rows_is_read_without_filling_them():
    import copy

    from brainstorm_amd.runtime.deferred import DeferredRows, lazy_tensor

    fills = []
    buffer = torch.empty(3, 5, dtype=torch.bfloat16)
    rows = lazy_tensor(buffer, lambda b: fills.append(b.fill_(2)))
    assert (rows.shape, rows.dtype, rows.device) == (torch.Size([3, 5]), torch.bfloat16, buffer.device)
    assert rows.shape[0] == rows.size(0) == len(rows) and not fills
    assert torch.equal(rows + 1, torch.full((3, 5), 3, dtype=torch.bfloat16)) and len(fills) == 1
    assert rows.shape == buffer.shape and len(fills) == 1
    stateless = buffer.as_subclass(DeferredRows)  # what a copy that drops the attributes is
    assert (stateless.shape, stateless.dtype, stateless.device) == (buffer.shape, buffer.dtype, buffer.device)
    assert copy.copy(rows).shape == buffer.shape


_METADATA_READS = {
    "shape": lambda rows: torch.ones(3) * rows.shape[0],
    "dtype": lambda rows: torch.ones(3, dtype=rows.dtype),
    "device": lambda rows: torch.ones(3, device=rows.device),
}


@pytest.mark.parametrize("built", [True, False])
@pytest.mark.parametrize("name", list(_METADATA_READS))
def test_metadata_reads_of_unfilled_rows_compile_as_one_graph(monkeypatch, name, built):
    """... of rows of several sizes, of an alias without its state, and inside a function mode.  (Compiling fills the rows that it is
    handed; what is asked here is that it takes them.)"""
    from brainstorm_amd.runtime.deferred import DeferredRows, DeferredState, lazy_tensor, wrap_if_pending
    from torch.overrides import TorchFunctionMode

    class Passing(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    if not built:
        monkeypatch.setattr(_lib, "native_or_none", lambda: None)
    run = _METADATA_READS[name]
    monkeypatch.setattr(DeferredState, "materialize", lambda self: None)
    kinds = {
        "lazy": lambda buffer: lazy_tensor(buffer, lambda b: None),
        "deferred": lambda buffer: wrap_if_pending(buffer.view(buffer.shape), {"key": DeferredState(None, None, buffer, "key")}),
        "alias": lambda buffer: buffer.as_subclass(DeferredRows),
    }
    for kind, make in kinds.items():
        torch._dynamo.reset()
        compiled = torch.compile(run, backend="eager", fullgraph=True)
        for size in (4, 6, 1, 9):
            rows = make(torch.empty(size, 2, dtype=torch.bfloat16))
            assert isinstance(rows, DeferredRows)
            want = run(torch.empty(size, 2, dtype=torch.bfloat16))
            assert torch.equal(compiled(rows), want) and compiled(rows).dtype == want.dtype, (kind, size)
        with Passing():
            assert torch.equal(compiled(rows), want), kind


def test_function_modes_see_metadata_reads_of_unfilled_rows():
    from brainstorm_amd.runtime.deferred import DeferredRows, lazy_tensor
    from torch.overrides import TorchFunctionMode

    class Called(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append((func, type(args[0])))
            return func(*args, **(kwargs or {}))

    rows = lazy_tensor(torch.empty(3, 5), lambda b: seen.append("filled"))
    seen = []
    with Called():
        read = (rows.shape, rows.dtype, rows.device)
    assert read == ((3, 5), torch.float32, torch.device("cpu"))
    assert seen == [(getattr(torch.Tensor, name).__get__, DeferredRows) for name in ("shape", "dtype", "device")]
