"""Repeated calls take the way of csrc/call.cpp: the signature that it reads tells apart what the one in Python does, and calls
that it does not know are left to Python."""

import ctypes
import functools
import gc
import threading
import types

import pytest
import torch

import ninetoothed_amd as ninetoothed
import ninetoothed_amd.language as ntl
from ninetoothed_amd import Tensor, programs, runtime


_FIRST_RUN = runtime.run  # (as it is before the first call)


def _signature(*args, flags=b"ttt", **kwargs):
    return runtime.call_library().signature(args, kwargs, flags)


def test_signature_tells_layouts_apart():
    a, b, c = torch.empty(4, 6), torch.empty(6, 4), torch.empty(4, 4)
    base = _signature(a, b, c)
    assert base is not None and base == _signature(torch.empty(4, 6), b, c)
    others = [
        (a.half(), b, c), (a, b.t().contiguous().t(), c), (torch.empty(4, 8)[:, :6], b, c), (torch.empty(1, 4, 6), b, c), (a, b, torch.empty(4, 5)), (a.to("meta"), b, c),
        (torch.empty(6, 4).t(), b, c),
    ]  # fmt: skip
    signatures = [_signature(*args) for args in others]
    assert None not in signatures and len({base, *signatures}) == len(others) + 1
    # (4, 6) beside (6, 4) is not (4, 6, 6) beside (4)
    assert _signature(torch.empty(4), torch.empty(6, 6, 4), c) != base


def test_signature_scalars_and_keywords():
    a = torch.empty(3)
    assert _signature(a, 1.0, 2, flags=b"tss") == _signature(a, 3.0, 5, flags=b"tss")
    assert len({_signature(a, x, 2, flags=b"tss") for x in (1.0, 1, True)}) == 3
    assert _signature(a, 1.0, 2, flags=b"tcs") != _signature(a, 3.0, 2, flags=b"tcs")
    assert _signature(a, 1, 2, flags=b"tcs") != _signature(a, 1.0, 2, flags=b"tcs")
    assert _signature(a, flags=b"t", BLOCK=1) != _signature(a, flags=b"t", BLOCK=2) != _signature(a, flags=b"t", BLOCKS=2)


def test_what_is_left_to_python():
    a, b, c = torch.empty(4, 6), torch.empty(6, 4), torch.empty(4, 4)

    class Sub(torch.Tensor):
        pass

    nested = torch.nested.nested_tensor([torch.empty(2, 6), torch.empty(3, 6)], layout=torch.jagged)
    for other in (a.as_subclass(Sub), nested, a.to_sparse(), [1.0], None, a.numpy()):
        assert _signature(other, b, c) is None
    assert _signature(a, b) is None  # a missing argument
    assert _signature(a, b, c, d=1.5) is None and _signature(a, b, c, d=True) is None
    assert _signature(a, b, 2**80, flags=b"ttc") is None
    assert torch.vmap(lambda x: x if _signature(x, b, c) is None else x + float("nan"))(torch.zeros(2, 4, 6)).isnan().sum() == 0
    assert _signature(*(torch.empty((1,) * 20) for _ in range(6)), flags=b"tttttt") is None  # longer than the buffer
    assert runtime.run({}, (a, b, c), {}, b"ttt") is None


def test_recipes_that_do_not_fit_are_refused():
    layout = runtime.ArgumentTensor.from_layout(0, (1, 1), (1, 1))
    with pytest.raises(ValueError):
        runtime.call_library().recipe("matmul", 1, (runtime.slot(0, layout),), (1, 2, 3, 4, 5), (), -1, ())
    with pytest.raises(ValueError):
        runtime.call_library().recipe("nothing", 1, (), (), (), -1, ())


@pytest.fixture
def no_gpu():
    """The native module with stand-ins for torch's current device and stream."""
    module = runtime.call_library()
    module.use(lambda: 0, lambda device: 0, runtime.check)
    yield module
    module.use(torch._C._cuda_getDevice, torch._C._cuda_getCurrentRawStream, runtime.check)


def _prepared(module, address):
    """What a softmax kernel keeps of its first call, with a function of this test as the entry point."""
    tensors = (torch.zeros(4, 6), torch.zeros(4, 6))
    slots = tuple(runtime.slot(position, runtime.ArgumentTensor.like(tensor)) for position, tensor in enumerate(tensors))
    recipe = module.recipe("softmax", address, slots, (runtime.DATA_TYPE_INDEX["fp32"], 6), (), -1, ())
    return {module.signature(tensors, {}, b"tt"): (recipe, "the plan")}, tensors


_SOFTMAX = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p, runtime.ArgumentTensor, runtime.ArgumentTensor, ctypes.c_int, ctypes.c_int)


@pytest.mark.parametrize("result", (0, 1, 2, 700))
def test_a_launch_that_fails_is_not_repeated(no_gpu, result):
    calls = []

    def entry_point(stream, input, output, dtype, block):
        calls.append((input.data, output.data, input.shape[1], output.strides[0], block))
        return result

    function = _SOFTMAX(entry_point)
    prepared, tensors = _prepared(no_gpu, ctypes.cast(function, ctypes.c_void_p).value)
    if result == 0:
        assert no_gpu.run(prepared, tensors, {}, b"tt") == "the plan"
    else:  # (a part of it may have run, or all of it with an error of an earlier launch reported here)
        with pytest.raises(runtime.KernelLaunchError) as raised:
            no_gpu.run(prepared, tensors, {}, b"tt")
        assert raised.value.error_code == result
    assert calls == [(tensors[0].data_ptr(), tensors[1].data_ptr(), 6, 6, 6)]


_LINEAR = ctypes.CFUNCTYPE(
    ctypes.c_int, ctypes.c_void_p, *(runtime.ArgumentTensor,) * 3, ctypes.c_int, ctypes.c_double, ctypes.c_double, runtime.ArgumentTensor, *(ctypes.c_int,) * 4
)


def test_linear_operands_that_are_not_taken_go_through_python(no_gpu):
    results = [0, runtime.NO_KERNEL, 700]
    function = _LINEAR(lambda *args: results.pop(0))
    tensors = tuple(torch.zeros(8, 8) for _ in range(3))
    lhs, rhs, output = (runtime.slot(position, runtime.ArgumentTensor.like(tensor)) for position, tensor in enumerate(tensors))
    recipe = no_gpu.recipe("linear", ctypes.cast(function, ctypes.c_void_p).value, (lhs, rhs, None, output), (10, 8, 0, 0, 0), (1.0, 0.0), -1, ())
    prepared = {no_gpu.signature(tensors, {}, b"ttt"): (recipe, "the plan")}
    assert no_gpu.run(prepared, tensors, {}, b"ttt") == "the plan"
    assert no_gpu.run(prepared, tensors, {}, b"ttt") is None
    with pytest.raises(runtime.KernelLaunchError):
        no_gpu.run(prepared, tensors, {}, b"ttt")
    assert not results


def test_an_exception_of_the_library_is_raised(no_gpu):
    # (libstdc++'s own function that throws std::bad_alloc stands in for the library)
    throws = ctypes.cast(ctypes.CDLL("libstdc++.so.6")._ZSt17__throw_bad_allocv, ctypes.c_void_p).value
    prepared, tensors = _prepared(no_gpu, throws)
    for _ in range(2):
        with pytest.raises(RuntimeError, match="C\\+\\+ exception"):
            no_gpu.run(prepared, tensors, {}, b"tt")


@pytest.mark.parametrize("reason", ("missing", "no library", "another torch", "no accessors"))
def test_calls_go_through_python_without_the_module(reason, tmp_path, monkeypatch):
    monkeypatch.setattr(runtime, "_call_library", None)
    monkeypatch.setattr(runtime, "_call_library_failed", False)
    monkeypatch.setattr(runtime, "run", runtime.run)  # (put back afterwards)
    monkeypatch.setattr(runtime, "run", _FIRST_RUN)
    if reason in ("missing", "no library"):
        path = tmp_path / runtime.CALL_LIBRARY_PATH.name
        if reason == "no library":
            path.write_bytes(b"text")
        monkeypatch.setattr(runtime, "CALL_LIBRARY_PATH", path)
    elif reason == "another torch":
        monkeypatch.setattr(torch, "__version__", "1.0")
    else:
        monkeypatch.delattr(torch._C, "_cuda_getDevice")
    kernel = _add()
    ran = []
    plan = types.SimpleNamespace(description="the plan", recipe=lambda: ran.append("recipe"), settled=lambda: True)
    monkeypatch.setattr(kernel, "_prepare", lambda args, kwargs: type("Plan", (types.SimpleNamespace,), {"__call__": lambda self, args: ran.append("launch")})(**vars(plan)))
    with pytest.warns(RuntimeWarning, match="through Python") as warned:
        for _ in range(3):
            kernel(torch.zeros(4), 1.0, torch.zeros(4))
    assert ran == ["launch"] * 3 and kernel.last_plan == "the plan" and len(warned) == 1


def _add():
    def arrangement(lhs, scale, output, block=ninetoothed.block_size()):
        return lhs.tile((block,)), scale, output.tile((block,))

    def application(lhs, scale, output):
        output = lhs * scale + 1  # noqa: F841

    return ninetoothed.make(arrangement, application, (Tensor(1), Tensor(0), Tensor(1)))


@pytest.mark.gpu
def test_each_entry_point_repeats_what_its_first_call_does():
    def normal(*shape):
        return torch.randn(shape, device="cuda", dtype=torch.float16)

    def linear_application(lhs, rhs, bias, output):
        accumulator = ntl.zeros(output.shape, dtype=ntl.float32)
        for k in range(lhs.shape[0]):
            accumulator += ntl.dot(lhs[k], rhs[k])
        output = ntl.maximum(accumulator + bias[None, :], 0)  # noqa: F841

    def scaled_application(lhs, rhs, bias, scale, output):
        accumulator = ntl.zeros(output.shape, dtype=ntl.float32)
        for k in range(lhs.shape[0]):
            accumulator += ntl.dot(lhs[k], rhs[k])
        output = scale * accumulator + bias[None, :]  # noqa: F841

    def linear_arrangement(lhs, rhs, bias, output, BM=ninetoothed.block_size(), BN=ninetoothed.block_size(), BK=ninetoothed.block_size()):
        lhs_arranged, rhs_arranged, output_arranged = programs.matmul.arrangement(lhs, rhs, output, BM, BN, BK)
        return lhs_arranged, rhs_arranged, bias.tile((BN,)).unsqueeze(0).expand((output_arranged.shape[0], -1)), output_arranged

    def scaled_arrangement(lhs, rhs, bias, scale, output, BM=ninetoothed.block_size(), BN=ninetoothed.block_size(), BK=ninetoothed.block_size()):
        *inputs, output_arranged = linear_arrangement(lhs, rhs, bias, output, BM, BN, BK)
        return *inputs, scale, output_arranged

    scaled_attention = ninetoothed.make(programs.attention.arrangement_with_scale, programs.attention.application_with_scale, programs.attention.tensors(True))
    attention = ninetoothed.make(programs.attention.arrangement, programs.attention.application, programs.attention.tensors())
    conv2d = ninetoothed.make(programs.conv2d.arrangement, programs.conv2d.application, programs.conv2d.tensors())
    strided = ninetoothed.make(functools.partial(programs.conv2d.arrangement, stride=(2, 2), floor_mode=True), programs.conv2d.application, programs.conv2d.tensors())
    softmax = ninetoothed.make(programs.softmax.arrangement, programs.softmax.application, programs.softmax.tensors())
    qkv = lambda: tuple(normal(1, 2, 70, 64) for _ in range(3))  # noqa: E731
    cases = [
        (ninetoothed.make(programs.matmul.arrangement, programs.matmul.application, programs.matmul.tensors()), lambda: (normal(96, 64), normal(64, 80)), (96, 80), {}),
        (ninetoothed.make(programs.addmm.arrangement, programs.addmm.application, programs.addmm.tensors()), lambda: (normal(96, 80), normal(96, 64), normal(64, 80), 0.5, 2), (96, 80), {}),
        (ninetoothed.make(linear_arrangement, linear_application, (Tensor(2), Tensor(2), Tensor(1), Tensor(2))), lambda: (normal(96, 64), normal(80, 64).t(), normal(80)), (96, 80), {}),
        (
            ninetoothed.make(scaled_arrangement, scaled_application, (Tensor(2), Tensor(2), Tensor(1), Tensor(0), Tensor(2))),
            lambda: (normal(96, 64), normal(80, 64).t(), normal(80), float(torch.rand(())) + 0.5), (96, 80), {},
        ),
        (softmax, lambda: (normal(50, 333),), (50, 333), {"BLOCK_SIZE": 333}),
        (scaled_attention, lambda: (*qkv(), True, 0.125), (1, 2, 70, 64), {}),
        (attention, lambda: (*qkv(), True), (1, 2, 70, 64), {}),
        (conv2d, lambda: (normal(2, 32, 9, 9), normal(64, 32, 3, 3)), (2, 64, 9, 9), {"padding_h": 1, "padding_w": 1}),
        (strided, lambda: (normal(2, 32, 9, 9), normal(64, 32, 3, 3)), (2, 64, 5, 5), {"padding_h": 1, "padding_w": 1}),
        (_add(), lambda: (normal(1000), 3.0), (1000,), {}),
    ]  # fmt: skip

    def fresh(shape):
        return torch.full(shape, float("nan"), device="cuda", dtype=torch.float16)

    for kernel, make_inputs, shape, options in cases:
        # each call's result through Python, then the same calls without a way back to Python
        all_inputs = [make_inputs(), make_inputs()]
        expected = []
        for inputs in all_inputs:
            expected.append(fresh(shape))
            kernel._call((*inputs, expected[-1]), options)
        assert len(kernel._prepared) == 1, kernel.kind
        assert not torch.equal(*expected) and not any(output.isnan().any() for output in expected), kernel.kind
        ((_, plan),) = kernel._prepared.values()
        for round in range(2):  # new buffers each time
            for inputs, result in zip(all_inputs, expected):
                output = fresh(shape)
                assert runtime.run(kernel._prepared, (*inputs, output), options, kernel._flags) is plan, kernel.kind
                assert torch.equal(output, result), kernel.kind
        kernel._call = None  # (a call that went through Python would raise)
        output = fresh(shape)
        stream = torch.cuda.Stream()  # a stream of its own
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            kernel(*all_inputs[0], output, **options)
        stream.synchronize()
        assert torch.equal(output, expected[0]) and kernel.last_plan == plan.description, kernel.kind
    kernel = cases[-1][0]
    values, output = normal(1000), normal(1000)
    for scale in (2.0, -1.5, 0.75):  # a scalar of this call
        kernel(values, scale, output)
        assert torch.equal(output, (values.float() * scale + 1).half())


@pytest.mark.gpu
def test_threads_share_a_kernel():
    kernel = _add()
    inputs = [torch.randn(5000, device="cuda") for _ in range(8)]
    kernel(inputs[0], 1.0, torch.empty_like(inputs[0]))
    failures = []

    def work(index):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for round in range(50):
                output = torch.empty_like(inputs[index])
                kernel(inputs[index], float(index + round), output)
                if not torch.equal(output, inputs[index] * float(index + round) + 1):
                    failures.append((index, round))

    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(index,)) for index in range(8)]
    for thread in threads:
        thread.start()
    for thread in threads:
        thread.join()
    assert not failures
    del kernel
    gc.collect()
