"""The convolution with input windows in LDS: sizes where its tiles of 224 positions and 64 filters, its windows, its blocks of 32 channels and
its outputs end raggedly, against a convolution in 64 bits."""

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

WINDOW = -5  # NINETOOTHED_CONV2D_WINDOWS, launch_nt_conv2d's block_size_m: input windows in LDS


def _launch(x, weight, out, padding, stride, dilation, way):
    from ninetoothed_amd import runtime

    tensors = [runtime.ArgumentTensor.from_torch_tensor(tensor) for tensor in (x, weight, out)]
    tag = runtime.DATA_TYPE_INDEX["fp16" if x.dtype == torch.float16 else "bf16"]
    return runtime.library().launch_nt_conv2d_strided(
        runtime.current_stream(), *tensors, tag, padding, padding, stride, stride, dilation, dilation, way, 0, 0
    )


def _output(shape, dtype, layout):
    """A NaN-filled output of that layout inside a guarded buffer."""
    n, k, p, q = shape
    buffer = torch.full((n * k * p * (q + 3) + 64,), 7.0, dtype=dtype, device="cuda")
    if layout == "nchw":
        out = buffer[: n * k * p * q].view(n, k, p, q)
    elif layout == "channels_last":
        out = buffer[: n * k * p * q].view(n, p, q, k).permute(0, 3, 1, 2)
    else:  # columns of a wider tensor
        out = buffer[: n * k * p * (q + 3)].view(n, k, p, q + 3)[..., 1:-2]
    out.fill_(float("nan"))
    return buffer, out


def _check(x, weight, padding, stride, dilation, layout):
    expected = F.conv2d(x.cpu().double(), weight.cpu().double(), padding=padding, stride=stride, dilation=dilation)
    buffer, out = _output(expected.shape, x.dtype, layout)
    from ninetoothed_amd import runtime

    assert _launch(x, weight, out, padding, stride, dilation, WINDOW) == 0
    assert "conv2d_window_kernel" in runtime.last_launch()
    # one rounding of each result (half a unit in the last place) and fp32 sums of C * 9 products
    unit = 2.0**-11 if x.dtype == torch.float16 else 2.0**-8
    bound = unit * expected.abs() + 2.0**-24 * weight[0].numel() ** 0.5 * 4 + 2.0**-25
    assert bool(((out.cpu().double() - expected).abs() <= bound * 1.01).all())
    mask = torch.ones_like(buffer, dtype=torch.bool)
    out_mask = torch.as_strided(mask, out.shape, out.stride(), out.storage_offset())
    out_mask.fill_(False)
    assert bool((buffer[mask] == 7.0).all())  # nothing outside the output


@pytest.mark.parametrize("layout", ("nchw", "channels_last", "sliced"))
@pytest.mark.parametrize("dtype", (torch.float16, torch.bfloat16))
@pytest.mark.parametrize(
    "n, c, height, width, k, padding, stride, dilation",
    (
        (1, 32, 3, 4, 1, 1, 1, 1),  # less than a tile, the smallest of everything
        (4, 32, 14, 16, 64, 1, 1, 1),  # four tiles, one image each
        (2, 40, 15, 15, 65, 1, 1, 1),  # one position over a tile, one filter over a tile, 8 channels over a block
        (5, 32, 36, 8, 92, 1, 1, 1),  # a small window: what the waves exchange is larger
        (9, 72, 7, 7, 130, 1, 1, 1),  # a tile spans images of an odd number of positions
        (40, 32, 3, 4, 24, 1, 2, 1),  # ... and many of them
        (3, 64, 57, 57, 48, 1, 2, 1),
        (2, 64, 30, 112, 72, 1, 2, 1),
        (3, 96, 25, 23, 16, 0, 1, 1),  # no padding
        (3, 32, 20, 11, 33, 2, 1, 1),  # an output larger than the input
        (2, 48, 26, 19, 17, 2, 2, 2),
        (6, 32, 6, 22, 40, 1, 3, 1),
        (2, 32, 31, 17, 64, 0, 4, 1),  # steps longer than the window
        (2, 40, 7, 109, 70, 0, 2, 1),  # a window of 1526 positions, of the most that fit (1532): 132 KiB of LDS
    ),
)
def test_against_64_bits(n, c, height, width, k, padding, stride, dilation, dtype, layout):
    torch.manual_seed(n * 1000 + height)
    x = torch.randn(n, c, height, width, device="cuda").to(dtype)
    weight = (torch.randn(k, c, 3, 3, device="cuda") * (9 * c) ** -0.5).to(dtype)
    _check(x, weight, padding, stride, dilation, layout)


def test_inputs_and_filters_inside_wider_tensors():
    torch.manual_seed(3)
    wide = torch.randn(6, 80, 13, 9, device="cuda").half()
    filters = (torch.randn(90, 64, 3, 3, device="cuda") / 24).half()
    cases = ((wide[1::2, 5:69], filters[::2]), (wide[:, 16:], filters[3:20]), (wide[2:4, :64], filters[:1]), (wide[:1, :64].expand(5, 64, 13, 9), filters[::3]))
    for x, weight in cases:
        _check(x, weight, 1, 2, 1, "nchw")


def test_the_choice_follows_the_size():
    from ninetoothed_amd import runtime

    def served(n, c, size, k, stride):
        x = torch.randn(n, c, size, size, device="cuda").half()
        weight = torch.randn(k, c, 3, 3, device="cuda").half()
        out = torch.empty(n, k, (size - 1) // stride + 1, (size - 1) // stride + 1, device="cuda", dtype=torch.float16)
        assert _launch(x, weight, out, 1, stride, 1, 0) == 0
        return runtime.last_launch()

    if torch.cuda.get_device_properties(0).multi_processor_count == 256:  # (the choice counts compute units)
        assert "conv2d_window_kernel" in served(32, 64, 56, 128, 2)
        assert "conv2d_repack_kernel" in served(1, 128, 14, 64, 2)  # few workgroups: the contraction in parts
        assert "conv2d_repack_kernel" in served(32, 256, 56, 512, 2)  # several rounds of long blocks
        assert "conv2d_repack_kernel" in served(9, 328, 56, 352, 2)  # ... and one of them, with steps of 2


@pytest.mark.parametrize("stride", (1, 2))
@pytest.mark.parametrize("channels, side, way", ((16, 9, 5), (128, 14, 5), (16, 9, WINDOW)))
def test_a_block_size_of_five_and_windows_that_do_not_apply_are_left_to_the_library(channels, side, way, stride):
    """Block sizes of a program arrive where ways are named: 5 of them name none.  (Input windows take no layer of 16 channels; of 128
    channels and this few positions they are slower.)"""
    from ninetoothed_amd import runtime

    torch.manual_seed(channels)
    x, weight = torch.randn(1, channels, side, side, device="cuda").half(), (torch.randn(64, channels, 3, 3, device="cuda") * (9 * channels) ** -0.5).half()
    expected = F.conv2d(x.cpu().double(), weight.cpu().double(), padding=1, stride=stride)
    out = torch.full(expected.shape, float("nan"), dtype=torch.float16, device="cuda")
    assert _launch(x, weight, out, 1, stride, 1, way) == 0
    served = runtime.last_launch()
    assert "conv2d_window_kernel" not in served
    assert bool(((out.cpu().double() - expected).abs() <= 2.0**-11 * expected.abs() + 2.0**-24 * weight[0].numel() ** 0.5 * 4 + 2.0**-25).all())
    assert _launch(x, weight, out, 1, stride, 1, 0) == 0 and runtime.last_launch() == served


@pytest.mark.parametrize("stride", (1, 2))
def test_a_program_of_blocks_of_five_positions(stride):
    import functools

    import ninetoothed_amd as ninetoothed
    from ninetoothed_amd import programs

    torch.manual_seed(stride)
    side = 16 * stride + 3 - stride
    x, weight = torch.randn(2, 16, side, side, device="cuda").half(), (torch.randn(32, 16, 3, 3, device="cuda") / 12).half()
    expected = F.conv2d(x.cpu().double(), weight.cpu().double(), stride=stride)
    out = torch.full(expected.shape, float("nan"), dtype=torch.float16, device="cuda")
    arrangement = functools.partial(programs.conv2d.arrangement, enable_padding=False, BLOCK_SIZE_M=5, BLOCK_SIZE_N=64, BLOCK_SIZE_K=64, stride=(stride, stride), floor_mode=True)
    ninetoothed.make(arrangement, programs.conv2d.application, programs.conv2d.tensors())(x, weight, out)
    assert bool(((out.cpu().double() - expected).abs() <= 2.0**-11 * expected.abs() + 2.0**-24 * weight[0].numel() ** 0.5 * 4 + 2.0**-25).all())
