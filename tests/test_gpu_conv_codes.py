"""Implicit im2col codes (k_conv_codes and k_conv_group_max, csrc/quantize.hip) against the
quantizer of explicit patch matrices, which divides: kernels of 1, 127 to 144 taps (the edge of the
128-column tap table), 63 to 65 rows, and values on and beside every tie of a code."""

import pytest
import torch
import torch.nn.functional as F

from memfast_amd import Config, Nonidealities, hip

pytestmark = pytest.mark.gpu

# (N, C, H, W, kernel, padding): rows per block 64, columns 128 (32 a wave).
GEOMETRIES = [
    (1, 130, 7, 9, (1, 1), (0, 0)),
    (1, 2, 21, 135, (1, 127), (0, 2)),
    (1, 3, 16, 20, (8, 16), (0, 0)),
    (2, 2, 17, 16, (12, 12), (1, 1)),
    (1, 33, 15, 7, (3, 3), (0, 0)),
]


def compare(device, x, kernel, padding, cfg, fixed):
    patches = F.unfold(x, kernel, 1, padding, 1).transpose(1, 2).flatten(0, 1)
    out = [e + 2 * p - k + 1 for e, p, k in zip(x.shape[2:], padding, kernel)]
    geom = (0, x.shape[1], kernel, (1, 1), padding, (1, 1), out)
    if fixed is not None:
        fixed = fixed.expand(1, patches.shape[1]).contiguous().to(device)
    got, got_scale = hip.conv_input_tiles(x.to(device), cfg, geom, fixed)
    want, want_scale = hip.input_tiles(patches.to(device), cfg, fixed)
    assert torch.equal(got, want)
    assert torch.equal(got_scale.view(torch.int32), want_scale.view(torch.int32))


@pytest.mark.parametrize("gran", ["fixed", (1, None), (1, 16), (1, 96), (3, 48), (None, None)],
                         ids=str)
@pytest.mark.parametrize("geometry", GEOMETRIES, ids=lambda g: "x".join(map(str, g[4])))
def test_same_codes_as_patches(hip_device, geometry, gran):
    n, c, h, w, kernel, padding = geometry
    quant = {} if gran == "fixed" else dict(input_quant_gran=gran)
    cfg = Config(array_size=(16, 32), nonidealities=Nonidealities(write_variation=0.0), **quant)
    gen = torch.Generator().manual_seed(sum(kernel))
    x = torch.randn(n, c, h, w, generator=gen)
    size = c * kernel[0] * kernel[1]
    fixed = torch.rand(1, size, generator=gen) * 0.05 + 0.005 if gran == "fixed" else None
    compare(hip_device, x, kernel, padding, cfg, fixed)


@pytest.mark.parametrize("bits", [3, 8])
@pytest.mark.parametrize("scale", [2.0**-7, 0.1, 3.0, 2.0**127, 2.0**-126, 2.0**-149, 1e-38])
def test_ties_and_extreme_scales(hip_device, scale, bits):
    """Every half code and its neighbours, beyond the largest code, zeros, the largest and smallest
    numbers: the codes that division gives, where the reciprocal overflows too."""
    s = torch.tensor(scale, dtype=torch.float32)
    half = (torch.arange(-262, 263).double() / 2 * s.double()).float()
    inf = torch.tensor(torch.inf)
    steps = [half, torch.nextafter(half, inf), torch.nextafter(half, -inf)]
    steps += [torch.nextafter(v, d) for v, d in zip(steps[1:], (inf, -inf))]
    top = torch.finfo(torch.float32).max
    values = torch.cat(steps + [torch.tensor([0.0, -0.0, top, -top, 1e-45, -1e-45, 1e30, 1.0])])
    values = values[torch.isfinite(values)]
    width = (values.numel() + 3) // 4
    x = F.pad(values, (0, 4 * width - values.numel())).reshape(1, 1, 4, width)
    cfg = Config(array_size=(32, 32), activation_bits=bits,
                 nonidealities=Nonidealities(write_variation=0.0))
    compare(hip_device, x, (2, 2), (0, 0), cfg, s.reshape(1, 1))
