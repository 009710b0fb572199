"""The surrogate's dequantized operands in one kernel against the index form of
quantization.py, bit for bit, and the checks of reprogramming read from one status word."""

import pytest
import torch

from memfast_amd import Config, Nonidealities, Simulator, hip, quantization

pytestmark = pytest.mark.gpu

CASES = [
    (dict(), 5, 130, 70),
    (dict(array_size=(48, 32), rows_per_read=16, weight_bits=4, activation_bits=3), 1, 47, 33),
    (dict(array_size=(64, 64), weight_signed=False, weight_bits=7), 65, 64, 64),
    (dict(array_size=(128, 16), rows_per_read=64, weight_bits=2), 3, 300, 1),
]


def make(kwargs):
    return Config(**kwargs, nonidealities=Nonidealities(write_variation=0.0))


@pytest.mark.parametrize("kwargs,n,k,o", CASES)
def test_same_values_as_the_index_form(hip_device, kwargs, n, k, o):
    cfg = make(kwargs)
    gen = torch.Generator().manual_seed(n)
    x = torch.randn(n, k, generator=gen).to(hip_device)
    w = torch.randn(o, k, generator=gen).to(hip_device)
    if not cfg.weight_signed:
        w = w.abs()
    q, xscale = hip.input_tiles(x, cfg)
    packed, _, wscale = hip.weight_tiles(w, cfg)
    assert torch.equal(hip.dequantize_inputs(q, xscale, cfg, k),
                       quantization.dequantize_inputs(q, xscale, cfg, k))
    assert torch.equal(hip.dequantize_program(packed, wscale, cfg, k, o),
                       quantization.dequantize_program(packed, wscale, cfg, k, o))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float64])
def test_reprogramming_raises_as_before_and_changes_nothing(hip_device, dtype):
    signed, unsigned = make({}), make(dict(weight_signed=False))
    w = torch.rand(40, 70, dtype=dtype, device=hip_device)
    bias = torch.rand(40, dtype=dtype, device=hip_device)
    for cfg, bad_weight, bad_bias, message in (
            (signed, float("nan"), float("inf"), "weights must be finite"),
            (unsigned, -1.0, float("inf"), "unsigned floating weights"),
            (signed, 1.0, float("inf"), "bias must be finite and match")):
        matrix = Simulator(cfg, device=hip_device).map(w, bias=bias)
        before = [t.clone() for t in (matrix.packed, matrix.weight_scale, matrix.bias)]
        weight, shift = w.clone(), bias.clone()
        weight[3, 69] = bad_weight
        shift[39] = bad_bias
        with pytest.raises(ValueError, match=message):
            matrix._reprogram(weight, shift)
        with pytest.raises(ValueError, match="bias must be finite and match"):
            matrix._reprogram(w, bias[:39])
        for now, was in zip((matrix.packed, matrix.weight_scale, matrix.bias), before):
            assert torch.equal(now, was)
        matrix._reprogram(w * 2, bias * 2)
        fresh = Simulator(cfg, device=hip_device).map(w * 2, bias=bias * 2)
        assert matrix._same_program(fresh) and torch.equal(matrix.bias, fresh.bias)
