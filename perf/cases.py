"""What a program written against this package has the GPU do, as a list of timed cases.

A case names one of the package's programs with its sizes, its element type and its options.  Every call goes through
the kernel that ``ninetoothed.make`` returns, on tensors that lie in GPU memory, as a model's forward pass makes it: the
handles are made once per process and kept, the outputs are written into tensors that the caller owns.

``listed()`` gives the fixed cases, ``draw(rng)`` one more case of the same ranges, ``prepare`` / ``run`` one case's inputs and
one pass over them, ``work`` what a pass cannot do without, ``tolerance`` how far two correct passes may lie apart.
"""

import functools

import torch

import ninetoothed_amd as ninetoothed
import ninetoothed_amd.language as ntl
from ninetoothed_amd import Tensor, programs

_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}

# A drawn case has at most this much to do: no more than the largest listed one (the 8192^3 product).
_MOST_FLOPS = 1.0e12
_MOST_BYTES = 1.1e9


def listed():
    return [
        # The README's matmul at its own size: the smallest call, of which a program makes many one after another.
        {"name": "matmul_512", "op": "matmul", "dtype": "fp16", "m": 512, "n": 512, "k": 512, "transposed": False},
        # One decoding step's scores over an odd vocabulary for 16 sequences: a skinny product `x @ w.T` that reads w once.
        {"name": "matmul_decode_head", "op": "matmul", "dtype": "bf16", "m": 16, "n": 50257, "k": 4096, "transposed": True},
        # The largest product, the one the package's benchmark is quoted on.
        {"name": "addmm_8192", "op": "addmm", "dtype": "fp16", "m": 8192, "n": 8192, "k": 8192},
        # A feed-forward layer over the tokens of a ragged batch: product, bias and activation in one program.
        {"name": "linear_relu_ragged", "op": "linear", "dtype": "bf16", "m": 1500, "n": 14336, "k": 4096},
        # The benchmark's row softmax: an ordinary size that memory bandwidth bounds.
        {"name": "softmax_4096", "op": "softmax", "dtype": "fp32", "rows": 4096, "cols": 4096},
        # Probabilities over an odd vocabulary for the sequences of one decoding step: few long rows, misaligned.
        {"name": "softmax_vocabulary", "op": "softmax", "dtype": "fp16", "rows": 64, "cols": 50257},
        # Prefill of long prompts, the benchmark's causal attention.
        {"name": "attention_prefill", "op": "attention", "dtype": "fp16", "batch": 4, "heads": 32, "queries": 4096, "keys": 4096, "dim": 128, "causal": True},
        # An encoder over sequences whose length fits no block.
        {"name": "attention_encoder_ragged", "op": "attention", "dtype": "bf16", "batch": 8, "heads": 16, "queries": 1000, "keys": 1000, "dim": 64, "causal": False},
        # Decoding: one query per sequence against a long cache.
        {"name": "attention_decode", "op": "attention", "dtype": "fp16", "batch": 8, "heads": 32, "queries": 1, "keys": 8192, "dim": 128, "causal": False},
        # The benchmark's convolution: a 3x3 layer over the batch of a training or inference step.
        {"name": "conv2d_3x3", "op": "conv2d", "dtype": "fp16", "batch": 32, "channels": 256, "height": 56, "width": 56, "filters": 256, "window": 3, "stride": 1},
        # A downsampling layer between two stages: smaller, strided.
        {"name": "conv2d_3x3_stride_2", "op": "conv2d", "dtype": "fp16", "batch": 32, "channels": 64, "height": 56, "width": 56, "filters": 128, "window": 3, "stride": 2},
        # The normalisation between a model's layers: a whole-row program that runs as a tile map.
        {"name": "rms_norm", "op": "rms_norm", "dtype": "bf16", "rows": 4096, "cols": 4096},
    ]


# ---- drawn cases ---------------------------------------------------------------------------------


def _log_uniform(rng, low, high):
    return int(round(low * (high / low) ** rng.random()))


def _size(rng, low, high, step):
    """A size of the range: mostly a multiple of 64 as widths and channel counts are, sometimes only one of ``step``."""
    step = 64 if rng.random() < 0.67 and low >= 64 else step
    return max(step, _log_uniform(rng, low, high) // step * step)


def _draw_product(rng, op):
    case = {"op": op, "dtype": rng.choice(("fp16", "bf16"))}
    if op == "matmul":
        case["transposed"] = rng.random() < 0.5
    # a row-major right operand has rows on 16-byte boundaries, as an aligned buffer gives them; `w.T` may have any number of rows
    any_width = op == "linear" or case.get("transposed", False)
    case["m"] = _log_uniform(rng, 1, 8192)  # tokens: any number
    case["n"] = _size(rng, 256, 16384, 1 if any_width else 8)
    case["k"] = _size(rng, 256, 16384, 8)
    return case


def _draw_softmax(rng):
    return {"op": "softmax", "dtype": rng.choice(("fp32", "fp16", "bf16")), "rows": _log_uniform(rng, 16, 32768), "cols": _size(rng, 64, 131072, 1)}


def _draw_attention(rng):
    case = {"op": "attention", "dtype": rng.choice(("fp16", "bf16")), "batch": _log_uniform(rng, 1, 16), "heads": rng.choice((8, 12, 16, 32))}
    if rng.random() < 0.4:  # decoding
        keys = _log_uniform(rng, 128, 32768)
        return dict(case, queries=1, keys=keys, dim=rng.choice((64, 128)), causal=False)
    length = _log_uniform(rng, 128, 8192)
    if rng.random() < 0.5:
        length = max(128, length // 64 * 64)
    return dict(case, queries=length, keys=length, dim=rng.choice((64, 128)), causal=rng.random() < 0.5)


def _draw_conv2d(rng):
    side = rng.choice((7, 14, 28, 56, 112, _log_uniform(rng, 7, 112)))
    return {
        "op": "conv2d", "dtype": "fp16", "batch": _log_uniform(rng, 1, 32), "channels": _size(rng, 64, 512, 8), "height": side, "width": side,
        "filters": _size(rng, 64, 512, 8), "window": rng.choice((1, 3, 3, 3, 5)), "stride": rng.choice((1, 1, 2)),
    }  # fmt: skip


def _draw_rms_norm(rng):
    return {"op": "rms_norm", "dtype": rng.choice(("fp16", "bf16", "fp32")), "rows": _log_uniform(rng, 16, 16384), "cols": _size(rng, 512, 16384, 8)}


def draw(rng):
    makers = (
        lambda: _draw_product(rng, "matmul"),
        lambda: _draw_product(rng, "matmul"),
        lambda: _draw_product(rng, "addmm"),
        lambda: _draw_product(rng, "linear"),
        lambda: _draw_softmax(rng),
        lambda: _draw_softmax(rng),
        lambda: _draw_attention(rng),
        lambda: _draw_attention(rng),
        lambda: _draw_attention(rng),
        lambda: _draw_conv2d(rng),
        lambda: _draw_conv2d(rng),
        lambda: _draw_rms_norm(rng),
    )
    maker = rng.choice(makers)
    while True:
        case = maker()
        cost = work(case)
        if cost["flops"] <= _MOST_FLOPS and cost["bytes"] <= _MOST_BYTES:
            return case


# ---- programs --------------------------------------------------------------------------------------


def _linear_arrangement(lhs, rhs, bias, output, BM=ninetoothed.block_size(), BN=ninetoothed.block_size(), BK=ninetoothed.block_size()):
    lhs_arranged, rhs_arranged, output_arranged = programs.matmul.arrangement(lhs, rhs, output, BM, BN, BK)
    bias_arranged = bias.tile((BN,)).unsqueeze(0).expand((output_arranged.shape[0], -1))
    return lhs_arranged, rhs_arranged, bias_arranged, output_arranged


def _linear_application(lhs, rhs, bias, output):
    accumulator = ntl.zeros(output.shape, dtype=ntl.float32)
    for k in range(lhs.shape[0]):
        accumulator += ntl.dot(lhs[k], rhs[k])
    output = ntl.maximum(accumulator + bias[None, :], 0)  # noqa: F841


def _rms_norm_arrangement(input, weight, output):
    def rows(tensor):
        arranged = tensor.tile((1, -1)).squeeze(1)
        arranged.dtype = arranged.dtype.squeeze(0)
        return arranged

    return rows(input), weight.tile((-1,)).expand((input.shape[0],)), rows(output)


def _rms_norm_application(input, weight, output):
    values = ntl.cast(input, ntl.float32)
    mean_square = ntl.sum(values * values) / input.shape[-1]
    output = values * ntl.rsqrt(mean_square + 1e-6) * weight  # noqa: F841


@functools.lru_cache(maxsize=None)
def _kernel(op, dtype, stride=1):
    """The handle a program makes once and keeps."""
    if op == "matmul":
        return ninetoothed.make(programs.matmul.arrangement, programs.matmul.application, programs.matmul.tensors())
    if op == "addmm":
        application = programs.addmm.application if dtype == "fp16" else programs.addmm.application_bfloat16
        return ninetoothed.make(programs.addmm.arrangement, application, programs.addmm.tensors())
    if op == "linear":
        return ninetoothed.make(_linear_arrangement, _linear_application, (Tensor(2), Tensor(2), Tensor(1), Tensor(2)))
    if op == "softmax":
        return ninetoothed.make(programs.softmax.arrangement, programs.softmax.application, programs.softmax.tensors())
    if op == "attention":
        return ninetoothed.make(programs.attention.arrangement_with_scale, programs.attention.application_with_scale, programs.attention.tensors(True))
    if op == "conv2d":
        arrangement = functools.partial(programs.conv2d.arrangement, stride=(stride, stride), floor_mode=stride > 1)
        return ninetoothed.make(arrangement, programs.conv2d.application, programs.conv2d.tensors())
    return ninetoothed.make(_rms_norm_arrangement, _rms_norm_application, (Tensor(2), Tensor(1), Tensor(2)))


def _windows(case):
    padding = case["window"] // 2
    return tuple((case[side] + 2 * padding - case["window"]) // case["stride"] + 1 for side in ("height", "width"))


# ---- one pass --------------------------------------------------------------------------------------


def prepare(case, seed):
    op, dtype = case["op"], _DTYPES[case["dtype"]]
    generator = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, scale=1.0):
        return torch.randn(shape, generator=generator, device="cuda", dtype=dtype).mul_(scale)

    def empty(*shape):
        return torch.empty(shape, dtype=dtype, device="cuda")

    kernel = _kernel(op, case["dtype"], case.get("stride", 1))
    options = {}
    if op in ("matmul", "addmm", "linear"):
        m, n, k = case["m"], case["n"], case["k"]
        lhs, output = normal(m, k), empty(m, n)
        # weights are kept as [outputs, inputs] where the layer multiplies by their transpose
        rhs = normal(n, k, scale=k**-0.5).t() if op == "linear" or case.get("transposed") else normal(k, n, scale=k**-0.5)
        if op == "addmm":
            arguments = (normal(m, n), lhs, rhs, 0.5, 1.0, output)
        else:
            arguments = (lhs, rhs, output) if op == "matmul" else (lhs, rhs, normal(n), output)
    elif op == "softmax":
        output = empty(case["rows"], case["cols"])
        arguments, options = (normal(case["rows"], case["cols"]), output), {"BLOCK_SIZE": case["cols"]}
    elif op == "attention":
        queries, keys = ((case["batch"], case["heads"], case[length], case["dim"]) for length in ("queries", "keys"))
        output = empty(*queries)
        arguments = (normal(*queries), normal(*keys), normal(*keys), case["causal"], case["dim"] ** -0.5, output)
    elif op == "conv2d":
        window, fan_in = case["window"], case["channels"] * case["window"] ** 2
        output = empty(case["batch"], case["filters"], *_windows(case))
        filters = normal(case["filters"], case["channels"], window, window, scale=fan_in**-0.5)
        arguments = (normal(case["batch"], case["channels"], case["height"], case["width"]), filters, output)
        options = {"padding_h": window // 2, "padding_w": window // 2}
    else:
        output = empty(case["rows"], case["cols"])
        arguments = (normal(case["rows"], case["cols"]), normal(case["cols"]), output)
    return kernel, arguments, options, output


def run(state):
    kernel, arguments, options, output = state
    kernel(*arguments, **options)
    return output


def work(case):
    op, itemsize = case["op"], 4 if case["dtype"] == "fp32" else 2
    if op in ("matmul", "addmm", "linear"):
        m, n, k = case["m"], case["n"], case["k"]
        elements = m * k + k * n + m * n + {"matmul": 0, "addmm": m * n, "linear": n}[op]
        return {"bytes": elements * itemsize, "flops": 2 * m * n * k}
    if op == "softmax":
        elements = case["rows"] * case["cols"]
        return {"bytes": 2 * elements * itemsize, "flops": 5 * elements}
    if op == "attention":
        pairs = case["batch"] * case["heads"]
        scores = case["queries"] * (case["queries"] + 1) // 2 if case["causal"] else case["queries"] * case["keys"]
        return {"bytes": 2 * pairs * (case["queries"] + case["keys"]) * case["dim"] * itemsize, "flops": 4 * pairs * scores * case["dim"]}
    if op == "conv2d":
        fan_in = case["channels"] * case["window"] ** 2
        positions = case["batch"] * _windows(case)[0] * _windows(case)[1]
        elements = case["batch"] * case["channels"] * case["height"] * case["width"] + case["filters"] * (fan_in + positions)
        return {"bytes": elements * itemsize, "flops": 2 * positions * case["filters"] * fan_in}
    elements = case["rows"] * case["cols"]
    return {"bytes": (2 * elements + case["cols"]) * itemsize, "flops": 4 * elements}


# About four times the distance (2-norm) between a pass and the same program in 64 bits on the same operands.  A product rounds
# once (fp16 2.1e-4, bf16 1.7e-3 measured); an addmm rounds its product as well (2.9e-4), attention its scaled queries and its
# probabilities (3.6e-4, 2.9e-3); the probabilities of a wide fp16 softmax are subnormal numbers (5.4e-4); fp32 sums differ by 1.3e-7.
def tolerance(case):
    if case["dtype"] == "fp32":
        return {"rel": 6.0e-7}
    if case["op"] == "softmax" and case["dtype"] == "fp16":
        return {"rel": 2.0e-3}
    half = {"fp16": 1.5e-3, "bf16": 1.2e-2} if case["op"] in ("attention", "addmm") else {"fp16": 9.0e-4, "bf16": 7.0e-3}
    return {"rel": half[case["dtype"]]}
