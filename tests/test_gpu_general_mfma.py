"""The general read on FP32 MFMA (k_general_mfma32, csrc/general.hip) against k_general, which
still makes the per-pair codes: slice totals bit for bit, and the fused output the reference
epilogue of those totals.

Reads of odd and ragged lengths, of up to 64 and up to 128 rows, one to eight slices on either
side, every device effect but output-mode read noise.
"""

import pytest
import torch

from memfast_amd import Config, Nonidealities, hip
from oracle import oracle

pytestmark = pytest.mark.gpu

WRITE = dict(write_variation=0.02)
CASES = {
    "read_scurve": (dict(), WRITE | dict(read_variation=0.01, adc_nonlinearity=0.1)),
    "drift": (dict(weight_bits=4), dict(write_variation=0.0, drift_coefficient=0.05,
                                        drift_time=100.0)),
    "voltage": (dict(input_slice=(1, 1, 1, 1, 2, 2), weight_slice=(1, 1, 2, 4), adc_bits=8),
                WRITE | dict(voltage_variation=0.02)),
    "slice_pair": (dict(activation_bits=7, adc_bits=5), WRITE | dict(read_variation=0.02,
                                                                     read_mode="slice_pair")),
    "slice_pair_scurve": (dict(), WRITE | dict(read_variation=0.02, read_mode="slice_pair",
                                               adc_nonlinearity=0.05)),
    # One slice a side, 30-row reads of 40-row arrays (a short second read).
    "short": (dict(activation_bits=2, weight_bits=2, input_slice=(1, 1), weight_slice=(2,),
                   weight_signed=False, array_size=(40, 16), rows_per_read=30),
              WRITE | dict(stuck_at_low=0.01, stuck_at_high=0.01, read_variation=0.01)),
    "seven_rows": (dict(input_slice=(1, 3, 4), weight_slice=(1, 7), array_size=(20, 32),
                        rows_per_read=7, adc_bits=9), WRITE),
    "rows128": (dict(array_size=(128, 32), adc_bits=8), WRITE | dict(read_variation=0.01)),
    "rows100_voltage": (dict(input_slice=(1, 1, 2, 2, 2), weight_slice=(1, 1, 2, 2, 2),
                             array_size=(100, 64), adc_bits=8), WRITE | dict(voltage_variation=0.02)),
    "rows96_slice_pair": (dict(array_size=(96, 64), adc_bits=7),
                          WRITE | dict(read_variation=0.02, read_mode="slice_pair")),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("n,k,o", [(1, 130, 20), (33, 64, 31), (70, 300, 130)])
def test_general_mfma_read(hip_device, name, n, k, o):
    kwargs, effects = CASES[name]
    cfg = Config(**kwargs, nonidealities=Nonidealities(**effects))
    gen = torch.Generator().manual_seed(17)
    a, b = torch.randn(n, k, generator=gen), torch.randn(k, o, generator=gen)
    b = b if cfg.weight_signed else b.abs()
    q, xs = hip.input_tiles(a.to(hip_device), cfg)
    packed, packed_t, ws = hip.weight_tiles(b.T.to(hip_device), cfg)
    m, p, c = q.shape[1], packed.shape[1], cfg.array_size[1]
    assert hip.mm_kernel(cfg, n, m, p) == 0
    seed, event = 321, 5
    expected, _ = hip.partial(q, packed, cfg, None, seed, event, 0, p, codes=True)
    totals = hip.partial(q, packed, cfg, None, seed, event, 0, p)
    assert torch.equal(totals.view(torch.int32), expected.view(torch.int32))
    if p > 1:   # a chunk of tiles away from the first
        part = hip.partial(q, packed, cfg, None, seed, event, 1, p)
        assert torch.equal(part.view(torch.int32), expected[:, :, 1:].contiguous().view(torch.int32))
    restored = oracle.execute(q.cpu(), xs.cpu(), packed.cpu(), ws.cpu(), cfg, seed, event, p * c,
                              totals=expected.cpu())
    for budget in (0, None):   # unsplit, and split where the rule says so
        fused = hip.mm(q, xs, packed, packed_t, ws.reshape(-1, p * c), cfg, seed, event, k_rows=k,
                       split_budget=budget)
        assert torch.equal(fused.cpu().view(torch.int32), restored.view(torch.int32)), budget


@pytest.mark.parametrize("name", ["read_scurve", "voltage", "rows128"])
def test_conductances_beyond_finite_currents(hip_device, name):
    """Injected infinities, NaN and conductances whose currents overflow convert as on k_general."""
    kwargs, effects = CASES[name]
    cfg = Config(**kwargs, nonidealities=Nonidealities(**effects))
    p = 2
    gen = torch.Generator().manual_seed(19)
    k, o = 100, 2 * cfg.array_size[1]
    q, _ = hip.input_tiles(torch.randn(40, k, generator=gen).to(hip_device), cfg)
    packed, _, _ = hip.weight_tiles(torch.randn(o, k, generator=gen).to(hip_device), cfg)
    g = hip.restore(packed, cfg, 6, 0, 0, p)
    flat = g.view(-1)
    strange = torch.tensor([float("inf"), float("-inf"), float("nan"), 3e38, -3e38, 1e30, 0.0, -1e-5])
    at = torch.randperm(flat.numel(), generator=gen)[:flat.numel() // 50].to(hip_device)
    flat[at] = strange.to(hip_device)[torch.arange(at.numel(), device=hip_device) % 8]
    expected, _ = hip.partial(q, packed, cfg, None, 6, 0, 0, p, conductance=g, codes=True)
    got = hip.partial(q, packed, cfg, None, 6, 0, 0, p, conductance=g)
    assert torch.equal(got.view(torch.int32), expected.view(torch.int32))


@pytest.mark.parametrize("reads", [17, 256, 257, 531])
@pytest.mark.parametrize("spare", [0, 20])
def test_general_mfma_read_order_levels(hip_device, reads, spare):
    """Over 16 and 256 reads the cascade in the kernel (no room for totals: unsplit) and that of the
    split read's totals are the reference epilogue of the totals; ``spare`` reads hold padding
    alone and are not run."""
    cfg = Config(array_size=(8, 32), adc_bits=4,
                 nonidealities=Nonidealities(write_variation=0.02, read_variation=0.01))
    gen = torch.Generator().manual_seed(18)
    k, k_rows = 8 * (reads + spare), 8 * reads - 3
    a, b = torch.randn(5, k, generator=gen), torch.randn(k, 64, generator=gen)
    a[:, k_rows:] = 0.0
    q, xs = hip.input_tiles(a.to(hip_device), cfg)
    packed, packed_t, ws = hip.weight_tiles(b.T.to(hip_device), cfg)
    assert hip.mm_workspace_bytes(cfg, 5, reads + spare, 2) > 0
    totals = hip.partial(q, packed, cfg, None, 3, 0, 0, 2)
    restored = oracle.execute(q.cpu(), xs.cpu(), packed.cpu(), ws.cpu(), cfg, 3, 0, 64,
                              totals=totals.cpu())
    for budget in (0, None):
        fused = hip.mm(q, xs, packed, packed_t, ws.reshape(-1, 64), cfg, 3, 0, k_rows=k_rows,
                       split_budget=budget)
        assert torch.equal(fused.cpu().view(torch.int32), restored.view(torch.int32)), budget
