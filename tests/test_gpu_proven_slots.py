"""The proven-slot masks of ideal reads at the edges of their workgroups, bit for bit."""

import pytest
import torch

from memfast_amd import Config, Nonidealities, hip
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [60, 64 * 63, 64 * 65 - 3])
@pytest.mark.parametrize("bits", [4, 5])
def test_proven_slots_of_one_bit_slices(hip_device, k, bits):
    """64 clamp candidates per read, some proven and some not: a slot wrongly proven leaves an
    unclamped count."""
    cfg = Config(adc_bits=bits, nonidealities=Nonidealities(write_variation=0.0))
    gen = torch.Generator().manual_seed(k)
    a, b = torch.randn(70, k, generator=gen), torch.randn(k, 40, generator=gen)
    a[:20], b[:, 20:] = a[:20].sign(), b[:, 20:].sign()
    q, xscale = hip.input_tiles(a.to(hip_device), cfg)
    packed, packed_t, wscale = hip.weight_tiles(b.T.to(hip_device), cfg)
    out = hip.mm(q, xscale, packed, packed_t, wscale.reshape(-1, packed.shape[1] * 64), cfg, 1, 0)
    assert torch.equal(out[:, :40].cpu(), oracle.mm(a, b, cfg)[:, :40])
