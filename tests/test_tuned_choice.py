"""Which candidate the tuner takes, from figures of this test, and what nt_tune_gemm answers."""

import ctypes
import pathlib
import shutil
import struct
import subprocess

import pytest
import torch

from ninetoothed_amd import runtime

CSRC = pathlib.Path(__file__).resolve().parent.parent / "ninetoothed_amd" / "csrc"


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    compiler = shutil.which("g++") or shutil.which("c++")
    if compiler is None:
        pytest.skip("no C++ compiler on this host")
    folder = tmp_path_factory.mktemp("choose")
    (folder / "choose.cpp").write_text(
        '#include "choose.h"\nextern "C" int choose(const float *measured, const float *counted, int count, float margin) { return nt::choose(measured, counted, count, margin); }\n'
    )
    subprocess.run([compiler, "-std=c++17", "-shared", "-fPIC", f"-I{CSRC}", str(folder / "choose.cpp"), "-o", str(folder / "choose.so")], check=True)
    function = ctypes.CDLL(str(folder / "choose.so")).choose

    def call(measured, counted=None, margin=0.02):
        array = ctypes.c_float * len(measured)
        return function(array(*measured), array(*(counted or measured)), len(measured), ctypes.c_float(margin))

    return call


def test_a_later_candidate_needs_the_margin(choose):
    assert choose([]) == -1
    assert choose([5.0, 4.95, 6.0]) == 0
    assert choose([5.0, 4.85, 4.8]) == 1  # (2 % of the one that stands)
    assert choose([5.0, 4.0], margin=0.25) == 0


def test_candidates_at_the_callers_pace(choose):
    # one launch counts for 3.5 at least, two for 6.2: positions 0 and 1 take one launch, 2 two
    def paced(*measured):
        return choose(measured, [max(ms, 6.2 if position == 2 else 3.5) for position, ms in enumerate(measured)])

    assert paced(3.4, 2.0, 9.0) == 1  # alike for the caller: the GPU's time decides
    assert paced(2.0, 3.4, 9.0) == 0
    assert paced(5.0, 8.0, 4.0) == 0  # two launches would show
    assert paced(8.0, 9.0, 4.0) == 2
    assert paced(7.0, 9.0, 6.9) == 0


@pytest.mark.gpu
@pytest.mark.parametrize(
    "m, n, k, tile",
    (
        (276, 128, 384, "64x64x64"), (1024, 1024, 1856, "64x64x64"), (1024, 1024, 1920, "64x64x128"), (384, 448, 1920, "64x64x64"),  # 10, 256 and 42 tiles of 64 x 64
        (1088, 1024, 256, "64x64x64"), (1088, 1024, 320, "64x128x64"), (1024, 2048, 2048, "64x128x64"),  # 272 of them, 136 and 256 of 64 x 128
        (1500, 2048, 512, "128x128x64"), (2048, 2048, 256, "128x128x64"),
    ),
)  # fmt: skip
def test_untuned_choice_of_tiles_that_the_chip_holds(m, n, k, tile):
    tag = runtime.DATA_TYPE_INDEX["bf16"]
    lhs, rhs = torch.randn(m, k, device="cuda", dtype=torch.bfloat16), torch.randn(k, n, device="cuda", dtype=torch.bfloat16)
    out = torch.full((m, n), float("nan"), device="cuda", dtype=torch.bfloat16)
    arguments = [runtime.ArgumentTensor.from_torch_tensor(t) for t in (lhs, rhs, out)]
    assert runtime.library().nt_tune_cache_lookup(tag, tag, m, n, k, 0) < 0
    runtime.check(runtime.library().launch_nt_matmul(runtime.current_stream(), *arguments, tag, tag, 0, 0, 0))
    assert f": {tile} " in runtime.last_launch() and "split-k" not in runtime.last_launch(), runtime.last_launch()
    expected = lhs.double() @ rhs.double()
    bound = 2.0**-8 * expected.abs() + (k + 4) * 2.0**-24 * (lhs.double().abs() @ rhs.double().abs())
    assert ((out.double() - expected).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("m, n, k", ((1024, 2560, 264), (2001, 2432, 520)))  # 160 and 304 tiles of 128 x 128
@pytest.mark.parametrize("bk", (64, 32))
def test_two_parts_of_more_tiles_than_the_chip_holds(m, n, k, bk):
    tag, library = runtime.DATA_TYPE_INDEX["bf16"], runtime.library()
    lhs, rhs = torch.randn(m, k, device="cuda", dtype=torch.bfloat16), torch.randn(k, n, device="cuda", dtype=torch.bfloat16)
    out = torch.full((m, n), float("nan"), device="cuda", dtype=torch.bfloat16)
    (index,) = (index for index, name in enumerate(runtime.gemm_config_names()) if name.startswith("128x128x64" if bk == 64 else "128x256x32") and name.endswith("split-k"))
    null, arguments = runtime.ArgumentTensor.null(), [runtime.ArgumentTensor.from_torch_tensor(t) for t in (lhs, rhs, out)]
    assert library.launch_nt_gemm_config(runtime.current_stream(), index, null, *arguments[:2], null, null, arguments[2], tag, tag) == 0
    expected = lhs.double() @ rhs.double()
    # one rounding to the element type over fp32 sums of k products
    bound = 2.0**-8 * expected.abs() + (k + 4) * 2.0**-24 * (lhs.double().abs() @ rhs.double().abs())
    assert ((out.double() - expected).abs() <= bound).all()


@pytest.mark.gpu
@pytest.mark.parametrize("m, n, k", ((64, 64, 64), (64, 256, 4096)))
def test_measured_times_come_back(m, n, k):
    # short products, timed for a caller of any pace: what comes back is a launch's time, not the pace
    tag, library = runtime.DATA_TYPE_INDEX["bf16"], runtime.library()
    lhs, rhs, out = (torch.randn(shape, device="cuda", dtype=torch.bfloat16) for shape in ((m, k), (k, n), (m, n)))
    arguments = [runtime.ArgumentTensor.null()] + [runtime.ArgumentTensor.from_torch_tensor(t) for t in (lhs, rhs)] + [runtime.ArgumentTensor.null()] * 2
    best, milliseconds = ctypes.c_int(-1), ctypes.c_float(0.0)
    answer = (ctypes.byref(best), ctypes.byref(milliseconds))
    output = runtime.ArgumentTensor.from_torch_tensor(out)
    runtime.check(library.nt_tune_gemm(runtime.current_stream(), *arguments, output, tag, tag, 5, *answer))
    for pace in (0.0036, 0.0064):  # (as 32-bit floats: no measured time is one of them but by chance)
        assert best.value >= 0 and 0 < milliseconds.value < 1 and milliseconds.value != struct.unpack("f", struct.pack("f", pace))[0]
    runtime.check(library.nt_tune_gemm_for_caller(runtime.current_stream(), *arguments, output, tag, tag, 5, 10.0, 20.0, *answer))
    assert best.value >= 0 and 0 < milliseconds.value < 1
    assert "tails split-k" not in runtime.gemm_config_names()[best.value]  # (its two launches count for twice as much there)
