"""ops.layer_fp8's argument handling where no GPU is: the library's entry point is replaced by one that records its arguments,
so that a call that the wrapper accepts completes, and one that it refuses raises what it raises with a GPU."""
import ctypes

import pytest
import torch

T, H, I, E, K = 3, 256, 128, 4, 2


class Lib:
    def __init__(self, real):
        self.real, self.calls = real, []
        kind = ctypes.CFUNCTYPE(ctypes.c_int, *real.moe_layer_fp8.argtypes)
        self.moe_layer_fp8 = kind(lambda *args: (self.calls.append(args), 0)[1])

    def __getattr__(self, name):
        return getattr(self.real, name)


@pytest.fixture
def road(pkg, monkeypatch):
    """(layer call, calls that reached the library)"""
    ops = pkg.ops
    lib = Lib(ops.lib)

    def address(t, name, dtype=None):
        assert isinstance(t, torch.Tensor) and t.is_contiguous() and (dtype is None or t.dtype == dtype), name
        return t.data_ptr()

    monkeypatch.setattr(ops, "lib", lib)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_dev", address)
    fp8 = torch.float8_e4m3fn
    given = dict(x=torch.zeros(T, H, dtype=torch.bfloat16), router_weight=torch.zeros(E, H, dtype=torch.bfloat16),
                 w13=torch.zeros(E, 2 * I, H, dtype=fp8), w13_scale=torch.ones(E, 2 * I // 128, H // 128),
                 w2=torch.zeros(E, H, I, dtype=fp8), w2_scale=torch.ones(E, H // 128, I // 128), top_k=K,
                 workspace=torch.empty(1 << 16, dtype=torch.uint8))
    return lambda **more: ops.layer_fp8(**{**given, **more}), lib.calls


def test_plain_call(road):
    call, calls = road
    assert call().shape == (T, H) and len(calls) == 1


def test_layer_call_under_the_jit_tracer(road):
    """A tracer records operators: one with a number as its result is not for it to see."""
    call, calls = road
    traced = torch.jit.trace(lambda x: call(x=x), (torch.zeros(T, H, dtype=torch.bfloat16),), check_trace=False)
    assert len(calls) == 1 and "_layer_fp8" not in str(traced.graph)


class Picky(torch.Tensor):
    """A subclass that declines operators that it does not know."""
    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        return NotImplemented if "my_ops" in str(func) else super().__torch_function__(func, types, args, kwargs or {})


@pytest.mark.parametrize("which", ["x", "w13_scale", "bias", "out"])
def test_operands_of_a_tensor_subclass(road, which):
    call, calls = road
    t = {"x": torch.zeros(T, H, dtype=torch.bfloat16), "w13_scale": torch.ones(E, 2 * I // 128, H // 128), "bias": torch.zeros(E),
         "out": torch.zeros(T, H, dtype=torch.bfloat16)}[which].as_subclass(Picky)
    call(**{which: t})
    assert len(calls) == 1


@pytest.mark.parametrize("renorm", [None, "x", [1]])
def test_renorm_that_is_no_number_is_refused(road, renorm):
    call, calls = road
    with pytest.raises((TypeError, ValueError)):
        call(renorm=renorm)
    assert not calls


def test_native_road_takes_renorm_as_the_other_does(road, monkeypatch):
    """A whole number's truth: 0.5 is 0, as the C argument has it."""
    call, calls = road
    seen = []

    class Op:
        default = staticmethod(lambda *args: (seen.append(args[11]), 1 << 20)[1])

    monkeypatch.setattr(torch.ops.my_ops, "_layer_fp8", Op)
    for renorm in (True, False, 2, 0, 0.5, 1.5):
        call(renorm=renorm)
    assert seen == [bool(args[11]) for args in calls] == [True, False, True, False, False, True]


@pytest.mark.parametrize("size", ["layer_workspace_bytes", "mm_workspace_bytes", "mlp_workspace_bytes"])
def test_sizes_asked_for_before_do_not_answer_other_types(pkg, size):
    """The sizes are kept by their arguments: 4.0 is refused, also once the size of 4 is known."""
    fn = getattr(pkg.ops, size)
    args = (4, 256, 128, 8, 2) if size.startswith("layer") else (4, 256, 128)
    assert fn(*args) > 0
    with pytest.raises(ctypes.ArgumentError):
        fn(float(args[0]), *args[1:])


def test_native_layer_call_declares_what_it_writes(pkg):
    schema = torch.ops.my_ops._layer_fp8.default._schema
    assert [a.name for a in schema.arguments if a.alias_info is not None and a.alias_info.is_write] == ["out", "workspace"]
