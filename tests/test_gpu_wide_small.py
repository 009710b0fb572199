"""The wide read of small batches (k_wide_small, csrc/noisy_wide.hip) against k_noisy_wide, which a
schedule that names an LDS tier runs, bit for bit: batches on either side of its 32-vector tiles,
one to twenty reads (the sum's cascade turns at sixteen), a ragged last column block."""

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
    "faults_two_reads": (LLM | dict(array_size=(128, 32), rows_per_read=64),
                         dict(write_variation=0.02, stuck_at_low=0.01, stuck_at_high=0.01)),
    "rows32_scurve": (dict(activation_bits=12, weight_bits=8, input_slice=(1, 3, 4, 4),
                           weight_slice=(1, 1, 2, 2, 2), array_size=(64, 32), rows_per_read=32,
                           adc_bits=8), dict(write_variation=0.02, adc_nonlinearity=0.05)),
}
# (vectors, contraction, outputs)
SIZES = [(1, 40, 20), (31, 300, 70), (32, 64, 33), (33, 1000, 150), (70, 1280, 100)]


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("name", list(CASES))
def test_same_outputs_as_the_large_read(hip_device, name, size):
    n, k, o = size
    kwargs, effects = CASES[name]
    cfg = Config(**kwargs, nonidealities=Nonidealities(**effects))
    gen = torch.Generator().manual_seed(n + k)
    a, b = torch.randn(n, k, generator=gen), torch.randn(k, o, generator=gen)
    q, xs = hip.input_tiles(a.to(hip_device), cfg)
    packed, _, ws = hip.weight_tiles(b.T.to(hip_device), cfg)
    p = packed.shape[1]
    assert hip.mm_kernel(cfg, n, q.shape[1], p) == 3
    ws = ws.reshape(-1, p * cfg.array_size[1])
    for event in (0, 2**33 + 1):
        got, want = (hip.mm(q, xs, packed, None, ws, cfg, 77, event, variant=variant)
                     for variant in (0, hip.variant_word(tier=3)))
        assert torch.equal(got.view(torch.int64), want.view(torch.int64))
