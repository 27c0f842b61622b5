"""CPU checks of the torch.library registration (no device work): the
path's entry points are custom ops of the ``glm53`` namespace whose shape
functions give the output shapes and dtypes under FakeTensor, so
torch.compile can trace a model through them without a graph break."""

from __future__ import annotations

import pytest

from conftest import pkg, submodule

torch = pytest.importorskip("torch")


def test_ops_are_registered():
    submodule("ops")
    for name in ("block_fp8_linear", "router_topk", "moe_decode", "moe_prefill"):
        assert hasattr(torch.ops.glm53, name), name


def test_fake_shapes_and_dtypes():
    from torch._subclasses.fake_tensor import FakeTensorMode

    submodule("ops")
    with FakeTensorMode():
        x = torch.empty((2, 5, 256), dtype=torch.bfloat16)
        w = torch.empty((384, 256), dtype=torch.uint8)
        s = torch.empty((3, 2), dtype=torch.float32)
        y = torch.ops.glm53.block_fp8_linear(x, w, s, None)
        assert y.shape == (2, 5, 384) and y.dtype == torch.bfloat16
        rw = torch.empty((32, 256), dtype=torch.float32)
        rb = torch.empty((32,), dtype=torch.float32)
        ids, sc = torch.ops.glm53.router_topk(x, rw, rb, 8, 2.5, True)
        assert ids.shape == (2, 5, 8) and ids.dtype == torch.int32
        assert sc.shape == (2, 5, 8) and sc.dtype == torch.float32
        one = torch.empty((1, 1, 256), dtype=torch.bfloat16)
        assert torch.ops.glm53.moe_decode(one, 7, None, None).shape == one.shape
        assert torch.ops.glm53.moe_prefill(x, 7, ids, sc).shape == x.shape


def test_moe_direct_is_registered_with_its_shape():
    from torch._subclasses.fake_tensor import FakeTensorMode

    submodule("ops")
    with FakeTensorMode():
        x = torch.empty((2, 5, 256), dtype=torch.bfloat16)
        y = torch.ops.glm53.moe_direct(x, 7)
        assert y.shape == x.shape and y.dtype == x.dtype


def test_unknown_owner_raises():
    ops = submodule("ops")
    with pytest.raises(RuntimeError, match="no longer exists"):
        ops._owner(10 ** 9)


def test_direct_calls_only_where_the_op_would_reach_its_kernel_alone():
    """ops.direct lets an eager call skip the op; anything that acts between
    the call and the kernel goes through it."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.autograd import forward_ad
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    ops = submodule("ops")

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Subclass(torch.Tensor):
        pass

    x = torch.zeros(4)
    assert ops.direct(x, None, torch.nn.Parameter(x, requires_grad=False))
    leaf = torch.zeros(4, requires_grad=True)
    assert not ops.direct(x, leaf)
    with torch.no_grad():
        assert ops.direct(x, leaf)
    assert not ops.direct(x.as_subclass(Subclass))
    for mode in (Dispatch(), Function(), FakeTensorMode(), forward_ad.dual_level(),
                 torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU])):
        with mode:
            assert not ops.direct(x), mode
    seen = []
    torch.vmap(lambda v: seen.append(ops.direct(v)) or v)(torch.zeros(2, 3))
    torch.jit.trace(lambda v: seen.append(ops.direct(v)) or v + 1, (x,), check_trace=False)
    torch.compile(lambda v: v + 1 if ops.direct(v) else v - 1, backend="eager")(x)
    assert seen and not any(seen)
    assert torch.equal(torch.compile(lambda v: v + 1 if ops.direct(v) else v - 1, backend="eager")(x), x - 1)
    assert ops.direct(x)


@pytest.mark.parametrize("place,name", [("_C", "_get_tracing_state"), ("_C", "_len_torch_dispatch_stack"),
                                        ("_C", "_len_torch_function_stack"),
                                        ("_C._functorch", "peek_interpreter_stack"),
                                        ("autograd.forward_ad", "_current_level"),
                                        ("autograd", "_profiler_enabled")])
def test_no_direct_calls_with_a_torch_that_lacks_a_name(monkeypatch, place, name):
    """ops.direct asks private state of torch; without it every call goes
    through the op."""
    from functools import reduce

    ops, x = submodule("ops"), torch.zeros(4)
    with monkeypatch.context() as m:
        m.delattr(reduce(getattr, place.split("."), torch), name)
        probe = ops._dispatch_probe()
    monkeypatch.setattr(ops, "_dispatch_acts", probe)
    assert not ops.direct(x)


def test_stream_handle_without_the_raw_stream_name(monkeypatch):
    from types import SimpleNamespace

    N = submodule("_native")
    monkeypatch.setattr(N, "_raw_stream", None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: SimpleNamespace(cuda_stream=(device, 7)))
    assert N.stream_handle() == (None, 7) and N.stream_handle(torch.device("cuda", 3)) == (3, 7)


@pytest.fixture
def mlp_and_rows(monkeypatch):
    """A ClampedMLP and rows for it whose device addresses are never used."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    monkeypatch.setattr(submodule("ops"), "direct", lambda *tensors: True)
    with FakeTensorMode():
        yield pkg().ClampedMLP(256, 384, 2.0, device="cuda"), torch.empty((4, 256), dtype=torch.bfloat16, device="cuda")


@pytest.mark.filterwarnings("ignore:Accessing the data pointer of FakeTensor")
@pytest.mark.parametrize("name", ["gate_proj", "up_proj", "down_proj"])
@pytest.mark.parametrize("buffer", ["weight", "weight_scale_inv"])
def test_mlp_in_one_call_only_with_every_buffer_on_the_rows_device(mlp_and_rows, name, buffer):
    """glm53_mlp takes the buffers by their addresses; one on the host must
    reach the projections, which refuse it."""
    mlp, x = mlp_and_rows
    assert mlp._one_call(x)
    proj = getattr(mlp, name)
    setattr(proj, buffer, torch.empty_like(getattr(proj, buffer), device="cpu"))
    assert not mlp._one_call(x)


def _empty_linear(out_features, in_features):
    """A BlockFP8Linear of an earlier size with buffers of the sizes given."""
    proj = pkg().BlockFP8Linear(128, 128, device="cuda")
    proj.weight = torch.empty((out_features, in_features), dtype=torch.uint8, device="cuda")
    proj.weight_scale_inv = torch.empty((-(-out_features // 128), -(-in_features // 128)), device="cuda")
    return proj


@pytest.fixture
def moe_and_rows(mlp_and_rows):
    """A SortedGroupedFP8MoE with a shared expert, and a few rows for it, of
    which no device address is ever used."""
    from types import SimpleNamespace

    M = pkg()
    shared, x = mlp_and_rows
    cfg = SimpleNamespace(hidden_size=256, moe_intermediate_size=128, swiglu_limit=2.0, n_routed_experts=4,
                          num_experts_per_tok=2, n_shared_experts=1)
    put = lambda *shape, dtype=torch.uint8: M.owned_tensor(  # noqa: E731
        torch.empty(shape, dtype=dtype, device="cuda"), layout=M.TensorLayout.ROW_MAJOR_CONTIGUOUS)
    bank = M.PackedFP8ExpertBank(put(4, 256, 256), put(4, 2, 2, dtype=torch.float32), put(4, 256, 128),
                                 put(4, 2, 1, dtype=torch.float32), intermediate_size=128)
    gate = M.Float32Gate(torch.empty((4, 256), device="cuda"), torch.empty(4, device="cuda"), top_k=2)
    return M.SortedGroupedFP8MoE(bank, cfg, gate, shared), x


@pytest.mark.filterwarnings("ignore:Accessing the data pointer of FakeTensor")
def test_projections_of_another_width_than_their_attributes_run_by_their_tensors(moe_and_rows):
    """The projections go by their tensors' shapes, the C structs by
    in_features and out_features: where these differ (buffers of another size
    were assigned), neither the one-call MLP nor the few-token prefill is
    taken."""
    moe, x = moe_and_rows
    mlp = moe.shared_experts
    assert mlp._one_call(x) and moe._few_routes_on_device(x, 4)
    sizes = {"gate_proj": (384, 256), "up_proj": (384, 256), "down_proj": (256, 384)}
    for name, size in sizes.items():
        kept = getattr(mlp, name)
        setattr(mlp, name, _empty_linear(*size))
        assert not mlp._one_call(x) and not moe._few_routes_on_device(x, 4), name
        setattr(mlp, name, kept)
    assert mlp._one_call(x) and moe._few_routes_on_device(x, 4)


@pytest.mark.filterwarnings("ignore:Accessing the data pointer of FakeTensor")
@pytest.mark.parametrize("expert", [0, 1, 3])
def test_few_token_prefill_only_over_expert_views_as_the_bank_gave_them(moe_and_rows, expert):
    """The loop that the prefill stands for runs every touched expert's own
    view: an edit of any of them keeps the loop, and so do tensors of the bank
    that are no longer the views'."""
    moe, x = moe_and_rows
    view = moe._expert(expert)
    edits = [(view, "limit", 3.0), (view, "down_proj", lambda rows: rows), (view.up_proj, "row_offset", 0),
             (moe.bank, "down_scale_inv", torch.empty_like(moe.bank.down_scale_inv)), (moe, "_expert", lambda e: view)]
    for part, name, value in edits:
        moe._view_edits.clear()
        assert moe._few_routes_on_device(x, 4)
        kept = getattr(part, name)
        setattr(part, name, value)
        assert not moe._few_routes_on_device(x, 4), name
        if part is moe:
            del part._expert
        else:
            setattr(part, name, kept)
