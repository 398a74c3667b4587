"""Products and convolutions whose tiles are dealt to the XCDs one by one instead of in ranges: every tile is computed once, at numbers of tiles that are no
multiple of 8, with partial last tiles, in one piece, in parts and in batches, against 64 bits."""

import pytest
import torch
import torch.nn.functional as F

from ninetoothed_amd import runtime

pytestmark = pytest.mark.gpu

TAGS = runtime.DATA_TYPE_INDEX


def _check(out, product, magnitude, k):
    # one rounding to fp16 over fp32 sums of k products
    assert bool(((out.double() - product).abs() <= 2.0**-11 * product.abs() + (k + 4) * 2.0**-24 * magnitude + 2.0**-24).all())


@pytest.mark.parametrize("transposed", (False, True))
@pytest.mark.parametrize(
    "text, m, n, k",
    (
        ("64x64x64 waves 2x2 stages 4 lds-direct tails", 64 * 8 + 3, 72, 72),  # 9 x 2
        ("64x64x64 waves 2x2 stages 4 lds-direct tails", 64 * 33 - 1, 192, 72),  # 33 x 3
        ("128x128x64 waves 2x4 stages 4 lds-direct tails", 128 * 16 + 9, 520, 136),  # 17 x 5
        ("128x256x32 waves 1x4 stages 3 lds-direct tails", 128 * 18 + 77, 768, 64),  # 19 x 3
        ("128x128x64 waves 2x4 stages 4 lds-direct tails split-k", 128 * 12 + 1, 256, 520),  # 13 x 2 in parts
        ("64x64x64 waves 2x2 stages 4 lds-direct tails split-k", 64 * 10 + 5, 328, 520),  # 11 x 6: in ranges
        ("256x256x32 waves 2x4 stages 5 lds-direct tails", 700, 776, 88),  # 3 x 4, a short contraction, ragged rows
        ("256x256x32 waves 2x4 stages 5 lds-direct tails", 257, 264, 128),
        ("256x256x32 waves 2x4 stages 5 lds-direct tails", 700, 776, 136),  # in ranges
    ),
)
def test_products_by_instance(text, m, n, k, transposed):
    (index,) = (i for i, name in enumerate(runtime.gemm_config_names()) if name == text)
    torch.manual_seed(m)
    lhs = torch.randn(m, k, device="cuda").half()
    rhs = (torch.randn(n, k, device="cuda") * k**-0.5).half().t() if transposed else (torch.randn(k, n, device="cuda") * k**-0.5).half()
    buffer = torch.full((m + 1, n + 8), 7.0, dtype=torch.float16, device="cuda")
    out = buffer[:m, :n]
    out.fill_(float("nan"))
    null, like = runtime.ArgumentTensor.null(), runtime.ArgumentTensor.from_torch_tensor
    runtime.check(runtime.library().launch_nt_gemm_config(runtime.current_stream(), index, null, like(lhs), like(rhs), null, null, like(out), TAGS["fp16"], TAGS["fp16"]))
    assert text.endswith("split-k") or "by whole lines" not in runtime.last_launch()  # (too short a contraction)
    _check(out, lhs.double() @ rhs.double(), lhs.double().abs() @ rhs.double().abs(), k)
    assert bool((buffer[m] == 7.0).all()) and bool((buffer[:, n:] == 7.0).all())


def test_a_batch_of_tall_products():
    torch.manual_seed(1)
    lhs, rhs = torch.randn(3, 64 * 12 + 5, 72, device="cuda").half(), torch.randn(3, 72, 136, device="cuda").half()  # 13 x 3 tiles each
    out = torch.full((3, lhs.shape[1], 136), float("nan"), dtype=torch.float16, device="cuda")
    like = runtime.ArgumentTensor.from_torch_tensor
    runtime.check(runtime.library().launch_nt_batched_matmul(runtime.current_stream(), like(lhs), like(rhs), like(out), TAGS["fp16"], TAGS["fp16"], 64, 64, 64))
    for i in range(3):
        _check(out[i], lhs[i].double() @ rhs[i].double(), lhs[i].double().abs() @ rhs[i].double().abs(), 72)


@pytest.mark.parametrize("stride, dilation", ((3, 1), (2, 1), (2, 2), (1, 1)))
@pytest.mark.parametrize("n, c, side, k", ((3, 48, 57, 72), (5, 16, 40, 130), (2, 64, 112, 40)))
def test_repacked_convolutions(n, c, side, k, stride, dilation):
    torch.manual_seed(side)
    x, weight = torch.randn(n, c, side, side, device="cuda").half(), (torch.randn(k, c, 3, 3, device="cuda") * (9 * c) ** -0.5).half()
    expected = F.conv2d(x.cpu().double(), weight.cpu().double(), padding=1, stride=stride, dilation=dilation)
    out = torch.full(expected.shape, float("nan"), dtype=torch.float16, device="cuda")
    arguments = [runtime.ArgumentTensor.from_torch_tensor(tensor) for tensor in (x, weight, out)]
    runtime.check(runtime.library().launch_nt_conv2d_strided(runtime.current_stream(), *arguments, TAGS["fp16"], 1, 1, stride, stride, dilation, dilation, 2, 0, 0))
    assert "conv2d_nhwc_kernel" in runtime.last_launch()
    bound = 2.0**-11 * expected.abs() + 2.0**-24 * (9 * c) ** 0.5 * 4 + 2.0**-25
    assert bool(((out.cpu().double() - expected).abs() <= bound * 1.01).all())
