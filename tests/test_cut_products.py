"""Products whose 256 x 256 tiles are more than whole rounds of the chip: the columns (or rows) of tiles that fill whole rounds in one launch,
what is left in another, with every epilogue, at ragged sizes of both parts, against products in 64 bits."""

import pytest
import torch

from ninetoothed_amd import runtime

pytestmark = pytest.mark.gpu

TAGS = runtime.DATA_TYPE_INDEX


def _operands(m, n, k, transposed, dtype):
    torch.manual_seed(m + n)
    lhs = torch.randn(m, k, device="cuda").to(dtype)
    rhs = (torch.randn(n, k, device="cuda") * k**-0.5).to(dtype).t() if transposed else (torch.randn(k, n, device="cuda") * k**-0.5).to(dtype)
    return lhs, rhs


def _check(out, expected, unit, magnitude, k, extra=0.0):
    # one rounding to the element type over fp32 sums of k products
    bound = unit * expected.abs() + (k + 4) * 2.0**-24 * magnitude + extra
    assert bool(((out.double() - expected).abs() <= bound).all())


@pytest.mark.parametrize("dtype", (torch.float16, torch.bfloat16))
@pytest.mark.parametrize(
    "m, n, k, transposed, kind",
    (
        (200, 66568, 512, False, "columns"),  # 261 tiles, 5 left, of which the last is partial
        (300, 33801, 520, True, "columns"),  # an odd number of columns, two rows of tiles
        (520, 32512, 512, True, "columns"),  # 126 left: two rounds of 128 x 128 tiles
        (33000, 304, 512, False, "rows"),
        (8500, 1800, 2048, True, "rows"),  # 272 tiles, 16 left with K in parts
        (1030, 16640, 2304, False, "columns"),  # five rows of tiles, 70 left
        (24988, 2040, 2304, True, "rows"),  # 784 tiles, 16 left with K in parts: more rounds than launch_nt_linear's own rule for last rows takes
    ),
)
def test_both_parts_with_every_epilogue(m, n, k, transposed, kind, dtype):
    name, unit = ("fp16", 2.0**-11) if dtype == torch.float16 else ("bf16", 2.0**-8)
    (index,) = (index for index, text in enumerate(runtime.gemm_config_names()) if "whole rounds" in text and f"the {kind} left" in text)
    lhs, rhs = _operands(m, n, k, transposed, dtype)
    product = lhs.double() @ rhs.double()
    magnitude = lhs.double().abs() @ rhs.double().abs()
    library, stream, null, like = runtime.library(), runtime.current_stream(), runtime.ArgumentTensor.null(), runtime.ArgumentTensor.from_torch_tensor
    pitch = (n + 7) // 8 * 8 + 8

    def output(element):
        buffer = torch.full((m + 1, pitch), 7.0, dtype=element, device="cuda")
        buffer[:m, :n] = float("nan")
        return buffer, buffer[:m, :n]

    def untouched(buffer):
        return bool((buffer[m] == 7.0).all()) and bool((buffer[:, n:] == 7.0).all())

    in_parts = (m, n) in ((8500, 1800), (24988, 2040))
    for element, tag in ((dtype, name), (torch.float32, "fp32")):
        buffer, out = output(element)
        assert library.launch_nt_gemm_config(stream, index, null, like(lhs), like(rhs), null, null, like(out), TAGS[name], TAGS[tag]) == 0
        assert ("lds-direct tails split-k" in runtime.last_launch()) == in_parts
        _check(out, product, unit if element == dtype else 2.0**-24, magnitude, k)
        assert untouched(buffer)
    bias = torch.randn(m, n, device="cuda").to(dtype)
    beta, alpha = runtime.ArgumentTensor.from_scalar(0.5), runtime.ArgumentTensor.from_scalar(2.0)
    buffer, out = output(dtype)
    assert library.launch_nt_gemm_config(stream, index, like(bias), like(lhs), like(rhs), beta, alpha, like(out), TAGS[name], TAGS[name]) == 0
    # (the product is rounded before it is doubled)
    _check(out, 0.5 * bias.double() + 2.0 * product, unit, 2.0 * magnitude, k, 2.0 * unit * product.abs() + 2.0**-14 * unit)
    assert untouched(buffer)
    column = torch.randn(n, device="cuda")
    buffer, out = output(dtype)
    runtime.check(library.launch_nt_linear(stream, like(lhs), like(rhs), like(column), TAGS["fp32"], 0.5, 0.0, like(out), TAGS[name], 0, 0, 0))
    assert "whole rounds" in runtime.last_launch() if m != 8500 else "the last rows with the k range in parts" in runtime.last_launch()
    _check(out, (0.5 * product + column.double()).clamp_min(0.0), unit, magnitude + column.double().abs(), k, 2.0**-23)
    assert untouched(buffer)


def test_which_products_are_cut():
    def served(m, n, k, blocks=(0, 0, 0)):
        lhs, rhs = _operands(m, n, k, True, torch.bfloat16)
        out = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
        arguments = [runtime.ArgumentTensor.from_torch_tensor(tensor) for tensor in (lhs, rhs, out)]
        runtime.check(runtime.library().launch_nt_matmul(runtime.current_stream(), *arguments, TAGS["bf16"], TAGS["bf16"], *blocks))
        return "whole rounds" in runtime.last_launch()

    assert served(520, 32512, 512) and not served(520, 32768, 512)  # 126 and 129 tiles left
    assert not served(256, 65536, 512)  # one whole round
    assert not served(520, 32512, 448)  # a short contraction
    assert not served(520, 32512, 512, (256, 256, 32))  # block sizes: one launch, no scratch memory
    assert not served(520, 32512, 512, (256, 0, 0)) and not served(520, 32512, 512, (0, 0, 32))  # ... also some of them
