"""A matrix product followed by element-wise work on the accumulator (bias, activation, scaling,
a residual): not one of the reference's own test programs, but the obvious next thing a user of
`ninetoothed.make` writes after the README's matmul.  The product runs on the GEMM kernels into an
fp32 scratch tensor, the rest as a tile map over it."""

import pytest
import torch

import ninetoothed_amd as ninetoothed
import ninetoothed_amd.language as ntl
from ninetoothed_amd import Tensor, programs


def linear_arrangement(lhs, rhs, bias, residual, scale, output, BM=ninetoothed.block_size(), BN=ninetoothed.block_size(), BK=ninetoothed.block_size()):
    lhs_arranged, rhs_arranged, output_arranged = programs.matmul.arrangement(lhs, rhs, output, BM, BN, BK)
    bias_arranged = bias.tile((BN,)).unsqueeze(0).expand((output_arranged.shape[0], -1))
    return lhs_arranged, rhs_arranged, bias_arranged, residual.tile((BM, BN)), scale, output_arranged


def linear_application(lhs, rhs, bias, residual, scale, output):
    accumulator = ntl.zeros(output.shape, dtype=ntl.float32)
    for k in range(lhs.shape[0]):
        accumulator += ntl.dot(lhs[k], rhs[k])
    activated = ntl.maximum(accumulator * scale + bias[None, :], 0)
    output = activated + residual  # noqa: F841


def _kernel():
    return ninetoothed.make(linear_arrangement, linear_application, (Tensor(2), Tensor(2), Tensor(1), Tensor(2), Tensor(0), Tensor(2)))


def test_recognised_as_a_product_with_an_epilogue():
    kernel = _kernel()
    assert kernel.kind == "gemm_epilogue"
    assert (kernel.details["lhs"], kernel.details["rhs"], kernel.details["output"]) == (0, 1, 5)
    # the epilogue reads the accumulator as a tile of one more tensor, arranged like the output
    text = kernel.details["epilogue"].describe()
    assert "load(ref[6,1,])" in text and "dot" not in text

    def two_products(lhs, rhs, bias, residual, scale, output):
        first = ntl.zeros(output.shape, dtype=ntl.float32)
        for k in range(lhs.shape[0]):
            first += ntl.dot(lhs[k], rhs[k])
        second = ntl.zeros(output.shape, dtype=ntl.float32)
        for k in range(lhs.shape[0]):
            second += ntl.dot(lhs[k], rhs[k]) * 2
        output = first + second  # noqa: F841

    with pytest.raises(ninetoothed.UnsupportedProgram):
        ninetoothed.make(linear_arrangement, two_products, (Tensor(2), Tensor(2), Tensor(1), Tensor(2), Tensor(0), Tensor(2)))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", (torch.float16, torch.bfloat16, torch.float32))
@pytest.mark.parametrize("m, n, k", ((512, 384, 256), (300, 200, 136), (1024, 1024, 2048)))
def test_linear_with_bias_activation_and_residual(m, n, k, dtype):
    kernel = _kernel()
    lhs = torch.randn(m, k, dtype=dtype, device="cuda")
    rhs = torch.randn(k, n, dtype=dtype, device="cuda")
    bias = torch.randn(n, dtype=dtype, device="cuda")
    residual = torch.randn(m, n, dtype=dtype, device="cuda")
    scale = 0.125
    expected = (torch.relu(lhs.float() @ rhs.float() * scale + bias.float()) + residual.float()).to(dtype)
    for _ in range(2):
        output = torch.full((m, n), float("nan"), dtype=dtype, device="cuda")
        kernel(lhs, rhs, bias, residual, scale, output)
        assert "launch_nt_matmul" in kernel.last_plan and "launch_nt_map" in kernel.last_plan
        assert torch.allclose(output.float(), expected.float(), rtol=1e-2, atol=1e-2)


@pytest.mark.gpu
@pytest.mark.parametrize("form", ("whole", "odd pitch", "one row", "columns apart", "in place"))
@pytest.mark.parametrize("m, n, k", ((5, 8, 64), (129, 136, 576), (257, 264, 64), (300, 1000, 128), (2049, 1288, 96), (300, 204, 128)))
def test_addmm_inputs_at_the_edges_of_tiles(m, n, k, form):
    """The input's values are asked for before the product is done, those of rows and columns behind the output's last ones from there: NaN
    around the input would show in the output.  (The product rounds to fp16 before it is combined, the result once more: an ulp each of the largest value, and an ulp where
    the product's own rounding falls the other way.)"""
    mat1, mat2, input, output, expected, atol = _addmm_case(m, n, k, form)
    kernel = ninetoothed.make(programs.addmm.arrangement, programs.addmm.application, programs.addmm.tensors())
    kernel(input, mat1, mat2, 0.5, 2.0, output)
    assert torch.allclose(output.double(), expected, rtol=0, atol=atol)


def _addmm_case(m, n, k, form):
    mat1, mat2 = torch.randn(m, k, device="cuda").half(), (torch.randn(k, n, device="cuda") * k**-0.5).half()
    values = torch.randn(1 if form == "one row" else m, n, device="cuda").half()
    if form == "odd pitch":
        input = torch.full((m, n + 3), float("nan"), dtype=torch.float16, device="cuda")[:, 1 : 1 + n]
    elif form == "columns apart":
        input = torch.full((n, m + 1), float("nan"), dtype=torch.float16, device="cuda")[:, :m].t()
    else:
        input = torch.empty_like(values)
    input.copy_(values)
    if form == "one row":
        input = input.expand(m, n)
    output = input if form == "in place" else torch.full((m, n), float("nan"), dtype=torch.float16, device="cuda")
    product = (mat1.double() @ mat2.double()).half().double()
    expected = 0.5 * values.double() + 2.0 * product
    ulp = 2.0**-10 * float(expected.abs().max())
    return mat1, mat2, input, output, expected, 3 * ulp


@pytest.mark.gpu
@pytest.mark.parametrize("form", ("whole", "odd pitch", "one row", "columns apart", "in place"))
@pytest.mark.parametrize("tile", ("256x256x32", "128x256x32", "128x128x64 waves 2x2", "128x128x64 waves 2x4", "64x64x64", "64x64x128", "64x128x64"))
def test_addmm_inputs_on_every_tile(tile, form):
    """As above, on each instance by its index: a lane holds 2 to 16 chunks of the input, and the last rows and columns of tiles are not there."""
    from ninetoothed_amd import runtime

    (index,) = (i for i, name in enumerate(runtime.gemm_config_names()) if name.startswith(tile) and name.endswith("lds-direct tails"))
    like, tag = runtime.ArgumentTensor.from_torch_tensor, runtime.DATA_TYPE_INDEX["fp16"]
    beta, alpha = (runtime.ArgumentTensor.from_scalar(value) for value in (0.5, 2.0))
    for m, n, k in ((517, 776, 136), (250, 8, 64), (258, 264, 328)):
        mat1, mat2, input, output, expected, atol = _addmm_case(m, n, k, form)
        arguments = like(input), like(mat1), like(mat2), beta, alpha, like(output)
        runtime.check(runtime.library().launch_nt_gemm_config(runtime.current_stream(), index, *arguments, tag, tag))
        assert torch.allclose(output.double(), expected, rtol=0, atol=atol)
