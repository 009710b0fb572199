"""The wide read through digits kept in LDS (k_wide_block, csrc/noisy_wide.hip) against
k_noisy_wide, which a schedule that names an LDS tier runs, bit for bit: ragged 32-vector and
128-column tiles, sixteen input slices, the read cascade's turns."""

import pytest
import torch

from memfast_amd import Config, Nonidealities, hip

pytestmark = pytest.mark.gpu

LLM = dict(activation_bits=16, weight_bits=4, input_slice=(1, 1, 2, 2, 2, 2, 2, 2, 2),
           weight_slice=(1, 1, 2), bw_e=8, adc_bits=8)
CASES = {
    "bfp16_rows64": (LLM | dict(array_size=(64, 64)),
                     dict(write_variation=0.02, read_variation=0.01, drift_coefficient=0.05,
                          drift_time=100.0)),
    "scurve_rows64": (LLM | dict(array_size=(128, 32), rows_per_read=64),
                      dict(write_variation=0.02, stuck_at_low=0.01, adc_nonlinearity=0.05)),
    "rows32": (dict(activation_bits=12, weight_bits=8, input_slice=(1, 3, 4, 4),
                    weight_slice=(1, 1, 2, 2, 2), array_size=(64, 32), rows_per_read=32,
                    adc_bits=8), dict(write_variation=0.02)),
    "sixteen_slices_scurve_rows32": (
        dict(activation_bits=16, weight_bits=4, array_size=(32, 32), adc_bits=6),
        dict(write_variation=0.02, adc_nonlinearity=0.05)),
    "sixteen_slices_rows64": (dict(activation_bits=16, weight_bits=4, adc_bits=7),
                              dict(write_variation=0.02, stuck_at_high=0.01)),
}
# (vectors, contraction, outputs): 1024 tiles and a few more.
SIZES = [(32 * 1024 - 31, 40, 100), (32 * 512 + 5, 64 * 16, 129), (32 * 342 + 1, 64 * 17, 260)]


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("name", list(CASES))
def test_same_outputs_as_the_tiered_read(hip_device, name, size):
    n, k, o = size
    kwargs, effects = CASES[name]
    cfg = Config(**kwargs, nonidealities=Nonidealities(**effects))
    gen = torch.Generator(hip_device).manual_seed(n + k)
    a = torch.randn(n, k, generator=gen, device=hip_device)
    b = torch.randn(o, k, generator=gen, device=hip_device)
    q, xs = hip.input_tiles(a, cfg)
    packed, _, ws = hip.weight_tiles(b, cfg)
    p = packed.shape[1]
    assert hip.mm_kernel(cfg, n, q.shape[1], p) == 3
    ws = ws.reshape(-1, p * cfg.array_size[1])
    want = hip.mm(q, xs, packed, None, ws, cfg, 77, 1, variant=hip.variant_word(tier=3))
    got = hip.mm(q, xs, packed, None, ws, cfg, 77, 1)
    assert torch.equal(got.view(torch.int64), want.view(torch.int64))
