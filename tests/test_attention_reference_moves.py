"""The pipelined attention loops on scores whose row maximum keeps rising, falls from a high start, or is reached by single
keys only: the blocks in which the running reference has to move, and those in which it must not."""

import math

import pytest
import torch

from ninetoothed_amd import runtime


def _rows(pattern, keys):
    """A factor per key that the keys' common direction is scaled by."""
    position = torch.arange(keys, device="cuda", dtype=torch.float64)
    if pattern == "rising":  # every block of keys lies above the one before it, by more than any slack at the end
        return position / keys * 200
    if pattern == "falling":
        return 200 - position / keys * 200
    if pattern == "steps":  # up by a little in every block: the reference stays as long as the sums allow
        return torch.floor(position / 32) * 1.5
    spikes = torch.zeros(keys, device="cuda", dtype=torch.float64)  # single keys far above all others, the last one of all among them
    spikes[keys // 3] = 60.0
    spikes[keys - 1] = 120.0
    return spikes


@pytest.mark.gpu
@pytest.mark.parametrize("pattern", ("rising", "falling", "steps", "spikes"))
@pytest.mark.parametrize(
    "variant, heads, queries, keys, causal",
    (
        (2, 3, 300, 300, True), (2, 3, 128, 1000, False), (2, 3, 257, 33, False),
        (3, 3, 300, 300, True), (3, 3, 128, 1000, False), (3, 3, 256, 64, False), (3, 3, 257, 33, False),
        (4, 512, 130, 200, False), (4, 512, 200, 64, False),
    ),
)  # fmt: skip
@pytest.mark.parametrize("dtype", (torch.float16, torch.bfloat16))
def test_moving_reference(variant, heads, queries, keys, causal, pattern, dtype):
    shape = (1, heads, keys, 64)
    q = torch.randn(1, heads, queries, 64, device="cuda")
    q[..., 0] = 1.0  # the common direction: a key's first element is added to all of its scores
    k, v = torch.randn(shape, device="cuda"), torch.randn(shape, device="cuda")
    k[..., 0] = _rows(pattern, keys).float()
    q, k, v = (tensor.to(dtype) for tensor in (q, k, v))
    scale, output = 1.0, torch.empty_like(q)
    arguments = [runtime.ArgumentTensor.like(tensor) for tensor in (q, k, v, output)]
    for argument, tensor in zip(arguments, (q, k, v, output)):
        argument.data = tensor.data_ptr()
    query_arg, key_arg, value_arg, output_arg = arguments
    # the block sizes that lead to the variant (none, and enough heads: variant 4)
    blocks = {2: (128, 32), 3: (128, 0), 4: (0, 0)}[variant]
    runtime.check(
        runtime.library().launch_nt_attention(
            runtime.current_stream(), query_arg, key_arg, value_arg, runtime.ArgumentTensor.from_scalar(int(causal)), runtime.ArgumentTensor.from_scalar(scale), output_arg,
            runtime.DATA_TYPE_INDEX["fp16" if dtype == torch.float16 else "bf16"], *blocks,
        )
    )  # fmt: skip
    assert runtime.last_launch().startswith(f"attention variant {variant}: "), runtime.last_launch()
    # the program's own rounding: queries scaled by log2(e) and rounded, then powers of two
    scores = torch.matmul((q.float() * (scale * 1.44269504089)).to(dtype).double(), k.double().transpose(-1, -2).contiguous()) * math.log(2)
    if causal:
        scores = scores.masked_fill(torch.ones(queries, keys, device="cuda", dtype=torch.bool).triu(1), float("-inf"))
    weights = scores.softmax(-1)
    expected = torch.matmul(weights, v.double())
    # probabilities and results are rounded to the element type once each, scores carry fp32 errors of 64 products
    epsilon = 2.0**-11 if dtype == torch.float16 else 2.0**-8
    score_error = 64 * 2.0**-24 * (q.double().abs().matmul(k.double().abs().transpose(-1, -2).contiguous())).amax() * 1.45
    bound = (2 * epsilon + 2 * score_error) * weights.matmul(v.double().abs()) + epsilon * expected.abs() + 1e-6
    assert ((output.double() - expected).abs() <= bound).all()
