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
    # the tile and the number of parts for outputs that are stored in pieces of 16 bytes, and for others (element by element) where they differ
    "n, c, size, k, window, stride, whole, scattered",
    (
        (1, 320, 7, 192, 5, 2, "64x64, 32 parts", None),   # 16 positions, 250 k steps: many parts
        (2, 104, 9, 60, 3, 1, "64x64, 18 parts", None),    # channels padded to the k step, filters no multiple of 8
        (3, 448, 20, 64, 3, 1, "64x64, 12 parts", None),
        (4, 344, 7, 152, 3, 1, "64x64, 11 parts", None),   # 49 positions an image: blocks of positions span images
        (29, 32, 12, 24, 3, 2, "64x64", None),
        (14, 200, 14, 384, 3, 1, "64x128", "64x128, 3 parts"),
        (12, 104, 15, 72, 5, 1, "64x128, 4 parts", None),
        (27, 40, 39, 72, 3, 1, "64x128", None),
        (3, 192, 56, 120, 3, 2, "64x64, 3 parts", None),
        (12, 128, 38, 128, 5, 1, "128x128, 3 parts", None),
        (33, 40, 50, 72, 3, 1, "128x128", None),
        (6, 64, 57, 320, 3, 1, "128x128", "64x64"),
        (21, 192, 29, 64, 3, 1, "128x64", "64x64"),
        (28, 104, 42, 24, 3, 1, "128x64", None),
        (23, 104, 19, 24, 5, 1, "128x64, 3 parts", None),
        (19, 32, 72, 24, 3, 1, "256x64", "64x64"),
        (17, 40, 40, 264, 3, 1, "256x256", "64x128"),
        (5, 3, 31, 24, 3, 1, "128x64", None),              # k steps of several taps
        (9, 5, 61, 120, 3, 1, "128x128", None),
        (40, 3, 45, 250, 5, 2, "128x128", None),
        (1, 40, 7, 8, 1, 1, "64x64", None),                # one k step and a bit
    ),
)
def test_tiles_and_parts_against_fp32(n, c, size, k, window, stride, whole, scattered, dtype, layout):
    from ninetoothed_amd import runtime

    padding = window // 2
    positions = ((size + 2 * padding - window) // stride + 1) ** 2
    in_pieces = layout == "channels_last" or (layout == "nchw" and positions % 8 == 0)
    tile = whole if in_pieces or scattered is None else scattered  # (of the times expected on 256 compute units)
    x = torch.randn(n, c, size, size, device="cuda").to(dtype)
    weight = (torch.randn(k, c, window, window, device="cuda") * (c * window * window) ** -0.5).to(dtype)
    expected = F.conv2d(x.cpu().double(), weight.cpu().double(), padding=padding, stride=stride)
    tag = runtime.DATA_TYPE_INDEX["fp16" if dtype == torch.float16 else "bf16"]
    results = []
    for _ in range(2):  # the second call finds the scratch memory of the first
        buffer, out = _outputs(expected.shape, dtype, layout)
        tensors = [runtime.ArgumentTensor.from_torch_tensor(t) for t in (x, weight, out)]
        assert runtime.library().launch_nt_conv2d_strided(runtime.current_stream(), *tensors, tag, padding, padding, stride, stride, 1, 1, REPACK, 0, 0) == 0
        assert "conv2d_repack_kernel" in runtime.last_launch() and runtime.last_launch().endswith("tiles of " + tile), runtime.last_launch()
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
