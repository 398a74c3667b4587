"""The repacking convolution (implicit GEMM on channels-last copies): every tile of its main kernel, whole and with the
contraction dealt to parts, at sizes where tiles, parts and outputs end raggedly."""

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

REPACK = 2  # launch_nt_conv2d's block_size_m: the repacking path


def _outputs(shape, dtype, layout):
    """A NaN-filled output of that layout inside a guarded buffer."""
    n, k, p, q = shape
    if layout == "nchw":
        buffer = torch.full((n * k * p * q + 64,), 7.0, dtype=dtype, device="cuda")
        out = buffer[: n * k * p * q].view(n, k, p, q)
    elif layout == "channels_last":
        buffer = torch.full((n * k * p * q + 64,), 7.0, dtype=dtype, device="cuda")
        out = buffer[: n * k * p * q].view(n, p, q, k).permute(0, 3, 1, 2)
    else:  # every second column of a wider tensor
        buffer = torch.full((n, k, p, 2 * q), 7.0, dtype=dtype, device="cuda")
        out = buffer[..., ::2]
    out.fill_(float("nan"))
    return buffer, out


@pytest.mark.parametrize("layout", ("nchw", "channels_last", "sliced"))
@pytest.mark.parametrize("dtype", (torch.float16, torch.bfloat16))
@pytest.mark.parametrize(
    "n, c, size, k, window, stride, tile, parts",
    (
        (1, 320, 7, 192, 5, 2, "64x64", 32),     # 16 positions, 250 k steps: many parts
        (2, 104, 9, 60, 3, 1, "64x64", 1),       # channels padded to the k step, filters no multiple of 8
        (3, 448, 20, 64, 3, 1, "64x64", 12),
        (4, 344, 7, 152, 3, 1, "64x64", 20),     # 49 positions an image: blocks of positions span images
        (14, 200, 14, 384, 3, 1, "128x64", 1),
        (3, 192, 56, 120, 3, 2, "64x64", 1),
        (12, 128, 38, 128, 5, 1, "128x128", 3),
        (6, 64, 57, 320, 3, 1, "128x128", 1),
        (21, 192, 29, 64, 3, 1, "128x64", 1),
        (27, 72, 10, 24, 5, 1, "128x64", 11),
        (24, 32, 15, 384, 3, 1, "64x128", 1),
        (2, 192, 18, 72, 5, 1, "64x128", 22),
        (39, 32, 46, 24, 3, 1, "256x64", 1),
        (12, 104, 37, 24, 5, 1, "256x64", 6),
        (5, 3, 31, 24, 3, 1, "128x64", 1),       # k steps of several taps
        (9, 5, 61, 120, 3, 1, "128x128", 1),
        (40, 3, 45, 250, 5, 2, "128x128", 1),
        (1, 40, 7, 8, 1, 1, "64x64", 1),         # one k step and a bit
    ),
)
def test_tiles_and_parts_against_fp32(n, c, size, k, window, stride, tile, parts, dtype, layout):
    from ninetoothed_amd import runtime

    padding = window // 2
    x = torch.randn(n, c, size, size, device="cuda").to(dtype)
    weight = (torch.randn(k, c, window, window, device="cuda") * (c * window * window) ** -0.5).to(dtype)
    expected = F.conv2d(x.cpu().double(), weight.cpu().double(), padding=padding, stride=stride)
    tag = runtime.DATA_TYPE_INDEX["fp16" if dtype == torch.float16 else "bf16"]
    results = []
    for _ in range(2):  # the second call finds the scratch memory of the first
        buffer, out = _outputs(expected.shape, dtype, layout)
        tensors = [runtime.ArgumentTensor.from_torch_tensor(t) for t in (x, weight, out)]
        assert runtime.library().launch_nt_conv2d_strided(runtime.current_stream(), *tensors, tag, padding, padding, stride, stride, 1, 1, REPACK, 0, 0) == 0
        # the tile and the parts follow from times expected on 256 compute units
        assert "conv2d_repack_kernel" in runtime.last_launch() and runtime.last_launch().endswith(f"tiles of {tile}" + (f", {parts} parts" if parts > 1 else "")), runtime.last_launch()
        results.append(out.clone())
        if layout == "sliced":
            assert bool((buffer[..., 1::2] == 7.0).all())
        else:
            assert bool((buffer[-64:] == 7.0).all())
    assert torch.equal(results[0], results[1])
    # one rounding to the element type (half a unit in the last place of each value) over fp32 sums of at most 8000 products
    # (their rounding: 2^-24 times the root of the number of additions, times the sum's size)
    unit = 2.0**-11 if dtype == torch.float16 else 2.0**-8
    difference = (results[0].cpu().double() - expected).abs()
    bound = unit * expected.abs() + 2.0**-24 * 8000**0.5 * 8 * expected.pow(2).mean().sqrt()
    assert bool((difference <= bound).all())
