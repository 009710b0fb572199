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


@pytest.mark.parametrize("gran", ["fixed", (1, None), (7, 48)], ids=str)
def test_images_beyond_32_bit_offsets(hip_device, gran):
    """One image of more than 2^29 elements, few patches of it: taps in its first and last rows and
    channels, padding on every side."""
    c, h, w, kernel, stride, padding = 4, 11601, 11603, (3, 5), (5800, 5801), (1, 2)
    assert c * h * w > 0x1FFFFFFF
    quant = {} if gran == "fixed" else dict(input_quant_gran=gran)
    cfg = Config(array_size=(16, 32), nonidealities=Nonidealities(write_variation=0.0), **quant)
    x = torch.empty(1, c, h, w, device=hip_device)
    x.normal_(generator=torch.Generator(device=hip_device).manual_seed(1))
    out = [(e + 2 * p - k) // s + 1 for e, p, k, s in zip((h, w), padding, kernel, stride)]
    rows = [[i * stride[0] - padding[0] + t for t in range(kernel[0])] for i in range(out[0])]
    columns = [[j * stride[1] - padding[1] + t for t in range(kernel[1])] for j in range(out[1])]
    assert max(map(max, rows)) >= h - 1 and max(map(max, columns)) >= w - 1
    patches = torch.zeros(out[0], out[1], c, *kernel, device=hip_device)
    for i, ys in enumerate(rows):
        for j, xs in enumerate(columns):
            for a, y in enumerate(ys):
                for b, xx in enumerate(xs):
                    if 0 <= y < h and 0 <= xx < w:
                        patches[i, j, :, a, b] = x[0, :, y, xx]
    patches = patches.reshape(out[0] * out[1], -1)
    fixed = None
    if gran == "fixed":
        fixed = (torch.rand(1, patches.shape[1]) * 0.05 + 0.005).to(hip_device)
    got, got_scale = hip.conv_input_tiles(x, cfg, (0, c, kernel, stride, padding, (1, 1), out), fixed)
    want, want_scale = hip.input_tiles(patches, cfg, fixed)
    assert torch.equal(got, want)
    assert torch.equal(got_scale.view(torch.int32), want_scale.view(torch.int32))


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
