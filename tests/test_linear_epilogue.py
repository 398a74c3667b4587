"""A scale, a bias per column and a lower bound on a product's accumulator: one launch on every instance a product runs on,
two (the product, then a tile map) for operands and outputs that the one launch does not take."""

import pytest
import torch

import ninetoothed_amd as ninetoothed
import ninetoothed_amd.language as ntl
from ninetoothed_amd import Tensor, programs, recognition, runtime


def linear_arrangement(lhs, rhs, bias, output, BM=ninetoothed.block_size(), BN=ninetoothed.block_size(), BK=ninetoothed.block_size()):
    lhs_arranged, rhs_arranged, output_arranged = programs.matmul.arrangement(lhs, rhs, output, BM, BN, BK)
    return lhs_arranged, rhs_arranged, bias.tile((BN,)).unsqueeze(0).expand((output_arranged.shape[0], -1)), output_arranged


def linear_application(lhs, rhs, bias, output):
    accumulator = ntl.zeros(output.shape, dtype=ntl.float32)
    for k in range(lhs.shape[0]):
        accumulator += ntl.dot(lhs[k], rhs[k])
    output = ntl.maximum(accumulator + bias[None, :], 0)  # noqa: F841


def scaled_arrangement(lhs, rhs, bias, scale, output, BM=ninetoothed.block_size(), BN=ninetoothed.block_size(), BK=ninetoothed.block_size()):
    lhs_arranged, rhs_arranged, bias_arranged, output_arranged = linear_arrangement(lhs, rhs, bias, output, BM, BN, BK)
    return lhs_arranged, rhs_arranged, bias_arranged, scale, output_arranged


def scaled_application(lhs, rhs, bias, scale, output):
    accumulator = ntl.zeros(output.shape, dtype=ntl.float32)
    for k in range(lhs.shape[0]):
        accumulator += ntl.dot(lhs[k], rhs[k])
    output = bias[None, :] + scale * accumulator  # noqa: F841


def gated_application(lhs, rhs, bias, output):
    accumulator = ntl.zeros(output.shape, dtype=ntl.float32)
    for k in range(lhs.shape[0]):
        accumulator += ntl.dot(lhs[k], rhs[k])
    output = ntl.maximum(accumulator * bias[None, :], 0)  # noqa: F841


def _linear():
    return ninetoothed.make(linear_arrangement, linear_application, (Tensor(2), Tensor(2), Tensor(1), Tensor(2)))


def _scaled():
    return ninetoothed.make(scaled_arrangement, scaled_application, (Tensor(2), Tensor(2), Tensor(1), Tensor(0), Tensor(2)))


def test_recognised_parts():
    assert _linear().details["linear"] == {"scale": None, "bias": 2, "lower": 0}
    scaled = _scaled().details["linear"]
    assert scaled["bias"] == 2 and scaled["scale"].param == 3 and scaled["lower"] is None
    gated = ninetoothed.make(linear_arrangement, gated_application, (Tensor(2), Tensor(2), Tensor(1), Tensor(2)))
    assert gated.kind == "gemm_epilogue" and gated.details["linear"] is None


def test_bias_layout():
    kernel = _linear()

    def layout(bias, n):
        args = (torch.empty(64, 32), torch.empty(32, n), bias, torch.empty(64, n))
        return recognition.analyze_column_vector(kernel.types[2], kernel._environment(args, {}, check_device=False), {"n": 1}, n)

    assert layout(torch.empty(48), 48) == (0, 1)
    assert layout(torch.empty(96)[::2], 48) == (0, 2)
    assert layout(torch.empty(40), 48) is None  # columns past its end would read zeros


def _operands(m, n, k, dtype, transposed, bias_dtype=None):
    lhs = torch.randn(m, k, device="cuda").to(dtype)
    rhs = torch.randn(n, k, device="cuda").mul_(k**-0.5).to(dtype).t() if transposed else torch.randn(k, n, device="cuda").mul_(k**-0.5).to(dtype)
    return lhs, rhs, torch.randn(n, device="cuda").to(bias_dtype or dtype)


def _check(output, lhs, rhs, bias, scale=1.0, lower=None):
    expected = (lhs.double() @ rhs.double()) * scale + bias.double()
    if lower is not None:
        expected = expected.clamp_min(lower)
    # one rounding to the element type, and the fp32 sums: k roundings of at most 2^-24 of the sum of the absolute products
    epsilon = 2.0**-11 if output.dtype == torch.float16 else 2.0**-8
    bound = epsilon * expected.abs() + (lhs.shape[1] + 4) * 2.0**-24 * ((lhs.double().abs() @ rhs.double().abs()) * abs(scale) + bias.double().abs()) + 2.0**-25
    assert ((output.double() - expected).abs() <= bound).all()


# a row (skinny columns of 16), odd columns, K in parts (few rows, and a few hundred), 64 x 64 and larger tiles with and
# without tails, tile rows over whole rounds with K in parts
SIZES = (
    (1, 256, 512, True), (17, 50257, 264, True), (40, 1001, 2048, True), (8, 320, 4096, False), (200, 384, 8192, False), (300, 1003, 520, True),
    (512, 512, 512, False), (1500, 2056, 264, False), (1024, 4096, 512, True), (4352, 4096, 2048, False),
)  # fmt: skip


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", (torch.float16, torch.bfloat16))
@pytest.mark.parametrize("m, n, k, transposed", SIZES)
@pytest.mark.parametrize("tuned", ("0", "1"))
def test_bias_and_bound_in_one_launch(m, n, k, transposed, tuned, dtype, monkeypatch):
    monkeypatch.setenv("NINETOOTHED_AMD_AUTOTUNE", tuned)
    kernel = _linear()
    lhs, rhs, bias = _operands(m, n, k, dtype, transposed)
    for _ in range(2):  # (the first call is the one that times the instances)
        output = torch.full((m, n), float("nan"), dtype=dtype, device="cuda")
        kernel(lhs, rhs, bias, output)
        assert "gemm" in runtime.last_launch() and kernel.last_plan.startswith("launch_nt_linear")
        _check(output, lhs, rhs, bias, lower=0)


@pytest.mark.gpu
@pytest.mark.parametrize("block", ((64, 64, 64), (64, 64, 128), (64, 128, 64), (128, 128, 64), (128, 256, 32), (256, 256, 32), (256, 256, 64)))
@pytest.mark.parametrize("m, n, k, transposed", ((512, 512, 512, False), (512, 512, 512, True), (300, 1000, 520, False), (300, 1001, 520, True)))
def test_every_tile(m, n, k, transposed, block):
    lhs, rhs, bias = _operands(m, n, k, torch.bfloat16, transposed, torch.float32)
    output = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    arguments = [runtime.ArgumentTensor.like(tensor) for tensor in (lhs, rhs, bias, output)]
    for argument, tensor in zip(arguments, (lhs, rhs, bias, output)):
        argument.data = tensor.data_ptr()
    lhs_arg, rhs_arg, bias_arg, output_arg = arguments
    dtypes = runtime.DATA_TYPE_INDEX
    runtime.check(
        runtime.library().launch_nt_linear(runtime.current_stream(), lhs_arg, rhs_arg, bias_arg, dtypes["fp32"], 0.5, float("-inf"), output_arg, dtypes["bf16"], *block)
    )
    tile = (256, 256, 32) if block == (256, 256, 64) and k % 64 else block  # (the instance of 256 x 256 x 64 takes whole k tiles only)
    assert ": {}x{}x{} ".format(*tile) in runtime.last_launch(), runtime.last_launch()
    _check(output, lhs, rhs, bias, scale=0.5)


@pytest.mark.gpu
def test_scale_float_bias_and_not_a_number():
    kernel = _scaled()
    lhs, rhs, bias = _operands(130, 264, 512, torch.float16, True, torch.float32)
    output = torch.empty(130, 264, dtype=torch.float16, device="cuda")
    for scale in (0.125, -2):
        kernel(lhs, rhs, bias, scale, output)
        assert "gemm" in runtime.last_launch()
        _check(output, lhs, rhs, bias, scale=scale)
    lhs[7, 3] = float("nan")
    bias = bias.half()
    _linear()(lhs, rhs, bias, output)
    assert output[7].isnan().all() and not output[8].isnan().any()


@pytest.mark.gpu
def test_calls_that_stay_two_launches():
    kernel = _linear()
    for m, n, k, columns in ((96, 200, 100, False), (96, 200, 104, True)):  # K no multiple of 8; an output by columns
        lhs, rhs, bias = _operands(m, n, k, torch.bfloat16, False)
        output = torch.empty(n, m, dtype=torch.bfloat16, device="cuda").t() if columns else torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
        kernel(lhs, rhs, bias, output)
        assert "gemm" not in runtime.last_launch() and kernel.last_plan.startswith("launch_nt_matmul") and "launch_nt_map" in kernel.last_plan
        _check(output, lhs, rhs, bias, lower=0)
    lhs, rhs, bias = _operands(256, 256, 256, torch.bfloat16, False)  # an operand that is the output
    output = lhs.clone()
    kernel(output, rhs, bias, output)
    _check(output, lhs, rhs, bias, lower=0)


@pytest.mark.gpu
def test_recorded_any_stride_choice(tmp_path, monkeypatch):
    # the any-stride kernel, recorded as the fastest for the plain product, has no linear epilogue: the call stays one launch on
    # the instance of the untuned rule
    monkeypatch.setenv("NINETOOTHED_AMD_AUTOTUNE", "0")
    lhs, rhs, bias = _operands(152, 344, 200, torch.bfloat16, False)
    names, tag = runtime.gemm_config_names(), runtime.DATA_TYPE_INDEX["bf16"]
    assert names[0].startswith("128x128x32 ") and "any-stride" in names[0]
    path = tmp_path / "choices.csv"
    path.write_text(f"\n{runtime.library().nt_tune_file_format()}\n0,{tag},{tag},152,344,200,0,0\n0,128,128,32\n")
    runtime.check(runtime.library().nt_tune_cache_load(str(path).encode(), None))
    assert runtime.library().nt_tune_cache_lookup(tag, tag, 152, 344, 200, 0) == 0
    kernel = _linear()
    for _ in range(2):
        output = torch.full((152, 344), float("nan"), dtype=torch.bfloat16, device="cuda")
        kernel(lhs, rhs, bias, output)
        assert "gemm" in runtime.last_launch() and "any-stride" not in runtime.last_launch()
        _check(output, lhs, rhs, bias, lower=0)


# What a call of an untuned linear program asks of the library (a stand-in here, which only notes the entry points): `tuned` is
# what the tuner answers -- an instance it has timed, -1 during a graph capture, -2 with nothing to choose from -- and `results`
# what the linear entry point returns, call after call.
@pytest.mark.parametrize(
    "tuned, results, shared, expected",
    (
        (3, (0, 0), False, ["linear", "tune", "linear"]),  # timing wrote over the output
        (-1, (0, 0), False, ["linear", "tune"]),  # a capture records one product
        (-2, (0, 0), False, ["linear", "tune"]),
        (3, (0, 0), True, ["linear"]),  # the output lies in an operand's storage: nothing is timed
        (3, (runtime.NO_KERNEL,), False, ["linear", "tune", "matmul", "map"]),  # (the product of the two launches is tuned as well)
        (3, (0, runtime.NO_KERNEL), False, ["linear", "tune", "linear", "tune", "matmul", "map"]),
    ),
)
def test_launches_of_an_untuned_call(tuned, results, shared, expected, monkeypatch):
    import types

    from ninetoothed_amd import auto_tuner

    asked, answers = [], list(results)

    def note(name, answer=lambda: 0):
        return lambda *args: (asked.append(name), answer())[1]

    library = types.SimpleNamespace(launch_nt_linear=note("linear", lambda: answers.pop(0)), launch_nt_matmul=note("matmul"), launch_nt_map=note("map"))
    monkeypatch.setattr(runtime, "library", lambda: library)
    monkeypatch.setattr(runtime, "current_stream", lambda: None)
    monkeypatch.setattr(auto_tuner, "enabled", lambda: True)
    monkeypatch.setattr(auto_tuner, "load_once", lambda: None)
    monkeypatch.setattr(auto_tuner, "lookup", lambda *args: -1)
    monkeypatch.setattr(auto_tuner, "tune", note("tune", lambda: (tuned, 0.0)))
    storage = torch.zeros(64 * 32 + 64 * 48, dtype=torch.float16)
    output = storage[64 * 32 :].view(64, 48) if shared else torch.zeros(64, 48, dtype=torch.float16)
    args = (storage[: 64 * 32].view(64, 32), torch.zeros(32, 48, dtype=torch.float16), torch.zeros(48, dtype=torch.float16), output)
    kernel = _linear()
    plan = kernel._prepare_gemm_epilogue(args, kernel._environment(args, {}, check_device=False))
    ran = plan(args) or plan.description
    assert asked == expected
    assert ("launch_nt_linear" in ran, "launch_nt_matmul" in ran, "launch_nt_map" in ran) == ((False, True, True) if "map" in expected else (True, False, False))
    assert plan.settled() == (tuned != -1 and "map" not in expected)
