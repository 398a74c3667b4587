"""Products whose rows begin inside cache lines: staged by whole lines, of which each k tile takes parts of two.  Every instance that has the form, at
contractions around whole tiles, rows that begin anywhere in a line, with NaN around the operands, against products in 64 bits."""

import pytest
import torch

from ninetoothed_amd import runtime

pytestmark = pytest.mark.gpu

TAGS = runtime.DATA_TYPE_INDEX
INSTANCES = ("64x64x64 waves 2x2 stages 4 lds-direct tails", "64x128x64", "128x128x64 waves 2x4", "64x64x64 waves 2x2 stages 4 lds-direct tails split-k", "128x128x64 waves 2x4 stages 4 lds-direct tails split-k")


def _instance(text):
    split = text.endswith("split-k")
    (index,) = (i for i, name in enumerate(runtime.gemm_config_names()) if name.startswith(text) and name.endswith("split-k") == split)
    return index


def _inside(rows, columns, pitch, first, scale, dtype):
    """[rows, columns] inside NaN: rows `pitch` apart, the first one `first` elements behind the beginning of a line."""
    storage = torch.full((rows * pitch + first + 64,), float("nan"), dtype=dtype, device="cuda")
    values = storage[first : first + rows * pitch].view(rows, pitch)[:, :columns]
    values.copy_(torch.randn(rows, columns, device="cuda") * scale)
    return values


@pytest.mark.parametrize("transposed", (False, True))
@pytest.mark.parametrize("text", INSTANCES)
@pytest.mark.parametrize(
    "m, n, k, apart, first",
    (
        (65, 8, 8, 0, 0),  # one chunk
        (66, 72, 56, 16, 8),  # less than a line, in two of them
        (129, 136, 64, 8, 56),  # a tile that takes two lines
        (200, 264, 72, 0, 0),
        (257, 128, 328, 24, 16),  # six tiles: the ring goes round
        (130, 520, 704, 8, 0),
        (300, 264, 2056, 0, 40),
        (70, 200, 4096, 8, 24),  # whole tiles in lines that hold parts of two
        (66, 64, 1088, 0, 32),  # rows that all begin in the middle of a line
    ),
)
def test_rows_that_begin_anywhere_in_a_line(m, n, k, apart, first, text, transposed):
    torch.manual_seed(m + n + k)
    dtype = torch.bfloat16 if k % 16 else torch.float16
    name, unit = ("fp16", 2.0**-11) if dtype == torch.float16 else ("bf16", 2.0**-8)
    lhs = _inside(m, k, k + apart, first, 1.0, dtype)
    rhs = _inside(n, k, k + apart, first, k**-0.5, dtype).t() if transposed else _inside(k, n, n + 8, 8, k**-0.5, dtype)
    buffer = torch.full((m + 1, n + 8), 7.0, dtype=dtype, device="cuda")
    out = buffer[:m, :n]
    library, stream, null, like = runtime.library(), runtime.current_stream(), runtime.ArgumentTensor.null(), runtime.ArgumentTensor.from_torch_tensor
    status = library.launch_nt_gemm_config(stream, _instance(text), null, like(lhs), like(rhs), null, null, like(out), TAGS[name], TAGS[name])
    if text.endswith("split-k") and k < 256:
        assert status != 0 or k >= 128  # (a part has two k tiles at least)
        return
    runtime.check(status)
    product, magnitude = lhs.double() @ rhs.double(), lhs.double().abs() @ rhs.double().abs()
    # one rounding to the element type over fp32 sums of k products
    assert bool(((out.double() - product).abs() <= unit * product.abs() + (k + 4) * 2.0**-24 * magnitude + 2.0**-24).all())
    assert bool((buffer[m] == 7.0).all()) and bool((buffer[:, n:] == 7.0).all())


def _store(m, n, dtype):
    buffer = torch.full((m + 1, n + 8), 7.0, dtype=dtype, device="cuda")
    return buffer, buffer[:m, :n]


@pytest.mark.parametrize("epilogue", ("plain", "fp32", "addmm"))
@pytest.mark.parametrize("transposed", (False, True))
@pytest.mark.parametrize("text", INSTANCES)
def test_every_epilogue_of_the_form_by_whole_lines(text, transposed, epilogue):
    """A size that is large enough for the form: the launch's note names it where rows begin inside lines, and not where they begin with one or for
    parts of 128 x 128 tiles with a row-major rhs, where it does not pay."""
    m, n, k = 1037, 1048, 1032
    torch.manual_seed(k)
    library, stream, null, like = runtime.library(), runtime.current_stream(), runtime.ArgumentTensor.null(), runtime.ArgumentTensor.from_torch_tensor
    bias = torch.randn(m, n, device="cuda").half()
    beta, alpha = (runtime.ArgumentTensor.from_scalar(value) for value in (0.5, 2.0))
    for apart, first in ((8, 24), (0, 0), (56, 0)):
        lhs = _inside(m, k, k + apart, first, 1.0, torch.float16)
        rhs = _inside(n, k, k + apart, first, k**-0.5, torch.float16).t() if transposed else _inside(k, n, n + 8, 8, k**-0.5, torch.float16)
        element, tag = (torch.float32, "fp32") if epilogue == "fp32" else (torch.float16, "fp16")
        buffer, out = _store(m, n, element)
        extra = (like(bias), like(lhs), like(rhs), beta, alpha) if epilogue == "addmm" else (null, like(lhs), like(rhs), null, null)
        runtime.check(library.launch_nt_gemm_config(stream, _instance(text), *extra, like(out), TAGS["fp16"], TAGS[tag]))
        by_lines = apart != 56 and (transposed or not (text.startswith("128x128") and text.endswith("split-k")))
        assert ("by whole lines" in runtime.last_launch()) == by_lines
        product, magnitude = lhs.double() @ rhs.double(), lhs.double().abs() @ rhs.double().abs()
        unit, sums = (2.0**-24 if epilogue == "fp32" else 2.0**-11), (k + 4) * 2.0**-24 * magnitude
        expected, bound = product, unit * product.abs() + sums
        if epilogue == "addmm":  # (the product is rounded before it is doubled)
            expected = 0.5 * bias.double() + 2.0 * product
            bound = unit * expected.abs() + 2.0 * (unit * product.abs() + sums) + 2.0**-24
        assert bool(((out.double() - expected).abs() <= bound).all())
        assert bool((buffer[m] == 7.0).all()) and bool((buffer[:, n:] == 7.0).all())


@pytest.mark.parametrize("transposed", (False, True))
@pytest.mark.parametrize("m, n, k, instance, in_parts", ((1037, 1048, 1032, "64x128x64", False), (600, 1048, 8200, "128x128x64", True)))
def test_the_linear_epilogue_of_the_form_by_whole_lines(m, n, k, instance, in_parts, transposed):
    torch.manual_seed(k)
    lhs = _inside(m, k, k, 8, 1.0, torch.bfloat16)
    rhs = _inside(n, k, k, 40, k**-0.5, torch.bfloat16).t() if transposed else _inside(k, n, n, 0, k**-0.5, torch.bfloat16)
    column = torch.randn(n, device="cuda")
    buffer, out = _store(m, n, torch.bfloat16)
    like = runtime.ArgumentTensor.from_torch_tensor
    runtime.check(runtime.library().launch_nt_linear(runtime.current_stream(), like(lhs), like(rhs), like(column), TAGS["fp32"], 0.5, 0.0, like(out), TAGS["bf16"], 0, 0, 0))
    note = runtime.last_launch()
    assert instance in note and ("split-k" in note) == in_parts
    assert ("by whole lines" in note) == (transposed or not in_parts)
    product, magnitude = lhs.double() @ rhs.double(), lhs.double().abs() @ rhs.double().abs()
    expected = (0.5 * product + column.double()).clamp_min(0.0)
    assert bool(((out.double() - expected).abs() <= 2.0**-8 * expected.abs() + (k + 4) * 2.0**-24 * (magnitude + column.double().abs())).all())
    assert bool((buffer[m] == 7.0).all()) and bool((buffer[:, n:] == 7.0).all())


@pytest.mark.parametrize("transposed", (False, True))
def test_a_batch_whose_products_begin_at_different_places_of_a_line(transposed):
    torch.manual_seed(0)
    batch, m, n, k = 5, 90, 72, 136
    lhs = torch.randn(batch, m * k + 8, device="cuda").half()[:, : m * k].unflatten(1, (m, k))
    rhs = torch.randn(batch, n * k + 24, device="cuda").half()[:, : n * k].unflatten(1, (n, k))
    rhs = rhs.transpose(1, 2) if transposed else rhs.reshape(batch, k, n).contiguous()
    out = torch.full((batch, m, n), float("nan"), dtype=torch.float16, device="cuda")
    like = runtime.ArgumentTensor.from_torch_tensor
    runtime.check(runtime.library().launch_nt_batched_matmul(runtime.current_stream(), like(lhs), like(rhs), like(out), TAGS["fp16"], TAGS["fp16"], 64, 64, 64))
    for i in range(batch):
        product, magnitude = lhs[i].double() @ rhs[i].double(), lhs[i].double().abs() @ rhs[i].double().abs()
        assert bool(((out[i].double() - product).abs() <= 2.0**-11 * product.abs() + (k + 4) * 2.0**-24 * magnitude).all())
