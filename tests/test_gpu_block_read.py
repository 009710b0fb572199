"""The noisy read whose digits live in LDS (k_noisy_block, csrc/noisy_block.hip): 64-row reads
with six to eight input slices and 128-row reads, linear converters, programming noise and faults.

Sizes sit at the edges of its tiles: 32 vectors and 32 or 64 columns per wave, four waves per
workgroup, cascades of 16 and 256 reads, small batches on k_noisy_pairs.
"""

import pytest
import torch
from torch import nn

from memfast_amd import Config, Nonidealities, Simulator, hip
from memfast_amd.nn import AnalogGRU
from oracle import oracle
from parity import check_product

pytestmark = pytest.mark.gpu

WRITE = dict(write_variation=0.02)
CASES = {
    # The default configuration: 64x64 arrays, one-bit slices of eight-bit codes.
    "default": (dict(), WRITE),
    "int4_faults": (dict(weight_bits=4), WRITE | dict(stuck_at_low=0.01, stuck_at_high=0.01)),
    # Six and seven input slices, several weight slice widths, arrays of two reads.
    "six_slices": (dict(input_slice=(1, 1, 1, 1, 2, 2), weight_slice=(1, 1, 2, 4), adc_bits=8,
                        array_size=(128, 64), rows_per_read=64), WRITE),
    "seven_slices": (dict(activation_bits=7, adc_bits=5, array_size=(64, 32)), WRITE),
    # 128-row reads of one- and two-bit slices, with array columns 32 and 128.
    "rows128": (dict(array_size=(128, 128), adc_bits=8), WRITE),
    "rows128_sliced": (dict(input_slice=(1, 1, 2, 2, 2), weight_slice=(1, 1, 2, 2, 2),
                            array_size=(256, 32), rows_per_read=128, adc_bits=8), WRITE),
    "rows128_ideal": (dict(array_size=(128, 64), adc_bits=7), dict(write_variation=0.0)),
}


def case(name):
    kwargs, effects = CASES[name]
    return Config(**kwargs, nonidealities=Nonidealities(**effects))


def programmed(cfg, n, k, o, device, seed):
    gen = torch.Generator().manual_seed(seed)
    a, b = torch.randn(n, k, generator=gen), torch.randn(k, o, generator=gen)
    q, xs = hip.input_tiles(a.to(device), cfg)
    packed, packed_t, ws = hip.weight_tiles(b.T.to(device), cfg)
    return a, b, q, xs, packed, packed_t, ws.reshape(-1, packed.shape[1] * cfg.array_size[1])


@pytest.mark.parametrize("name", list(CASES))
def test_totals_with_injected_conductances(hip_device, name):
    """Slice totals equal the oracle's on the same conductances, except converter flips (the
    budget of 1e-4 of the codes)."""
    cfg = case(name)
    a, b, q, _, packed, packed_t, _ = programmed(cfg, 70, 200, 100, hip_device, 3)
    p = packed.shape[1]
    assert hip.block_read(cfg) and hip.mm_kernel(cfg, 70, q.shape[1], p) == 2
    raw, _, _ = oracle.restored(packed.cpu(), cfg, 4242, 3, 0, p)
    expected = oracle.partial(q.cpu(), packed.cpu(), cfg, 4242, 3, 0, p, conductance=raw)
    got = hip.mm_totals(q, packed_t, cfg, 4242, 3, conductance=raw.to(hip_device)).cpu()
    diff = got.double() - expected.double()
    codes = diff.numel() * len(cfg.input_layout) * len(cfg.weight_layout)
    print("[block read]", name, "totals differing", int((diff != 0).sum()), "codes", codes,
          flush=True)
    assert int((diff != 0).sum()) <= max(1, 1e-4 * codes)


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("n,k,o", [(1, 100, 32), (33, 64, 30), (32, 500, 300), (97, 300, 260)])
def test_product_and_schedules(hip_device, name, n, k, o):
    """The product is the oracle's under the flip accounting, and every read split (automatic,
    none, two and seven chunks) gives the same output bit for bit."""
    cfg = case(name)
    a, b, q, xs, packed, packed_t, ws = programmed(cfg, n, k, o, hip_device, 5)
    outputs = [hip.mm(q, xs, packed, packed_t, ws, cfg, 77, 1, variant=hip.variant_word(split=z),
                      out_cols=o, k_rows=k)[:, :o].clone() for z in (0, 1, 2, 7)]
    for output in outputs[1:]:
        assert torch.equal(output.view(torch.int32), outputs[0].view(torch.int32))
    got = Simulator(cfg, device=hip_device).mm(a.to(hip_device), b.to(hip_device))
    check_product(cfg, got, a, b, hip_device, label=f"block read {name}")


@pytest.mark.parametrize("batch,hidden", [(3, 70), (50, 768), (300, 768)])
def test_recurrent_sequence(hip_device, batch, hidden):
    """A GRU's native steps on default arrays equal its cells stepped one by one: hidden reads of
    one wave per weight slice, split over reads with the totals left to the gate kernel, and whole."""
    torch.manual_seed(13)
    source = nn.GRU(20, hidden).to(hip_device)
    layer, stepped = (AnalogGRU(source, Simulator(case("default"), device=hip_device), name="gru")
                      for _ in range(2))
    x = torch.randn(4, batch, 20, device=hip_device)
    got, _ = layer(x)
    state, states = torch.zeros(batch, hidden, device=hip_device), []
    for step in x:
        state = stepped.cells[0](step, state)
        states.append(state)
    assert torch.equal(got.view(torch.int32), torch.stack(states).view(torch.int32))
    assert layer.cells[0].hidden._event == stepped.cells[0].hidden._event == 4


SLICED = Config(input_slice=(1, 1, 2, 2, 2), weight_slice=(1, 1, 2, 2, 2), array_size=(128, 128),
                rows_per_read=32, adc_bits=7, nonidealities=Nonidealities(**WRITE))


@pytest.mark.parametrize("cfg", [case("default"), case("rows128"), case("rows128_ideal"), SLICED],
                         ids=["default", "rows128", "rows128_ideal", "sliced"])
@pytest.mark.parametrize("offset,stride", [(0, 131), (1, 132), (2, 130)])
def test_unaligned_output(hip_device, cfg, offset, stride):
    """An output view that the MFMA reads do not take (row stride, first element) gets the general
    kernel's read: the output for the conductances restored and passed in."""
    n, k, o = 33, 200, 128
    *_, q, xs, packed, packed_t, ws = programmed(cfg, n, k, o, hip_device, 9)
    g = hip.restore(packed, cfg, 5, 2, 0, packed.shape[1])
    expected = hip.mm(q, xs, packed, None, ws, cfg, 5, 2, conductance=g, k_rows=k)
    flat = torch.full((n * stride + 4,), float("nan"), device=hip_device)
    view = flat[offset:offset + n * stride].view(n, stride)
    got = hip.mm(q, xs, packed, packed_t, ws, cfg, 5, 2, out=view, k_rows=k)
    assert got is view
    assert torch.equal(got[:, :o].contiguous().view(torch.int32), expected.view(torch.int32))
    assert bool(got[:, o:].isnan().all()) and bool(flat[:offset].isnan().all())


@pytest.mark.parametrize("cfg", [case("default"), SLICED], ids=["default", "sliced"])
def test_batch_beyond_the_mfma_reads(hip_device, cfg):
    """4.2 million vectors are more than the MFMA reads' grids take: a layer's read samples the
    conductances for the general kernel."""
    k, o = cfg.array_size[0] - 1, 30
    n = (65535 - cfg.array_size[1] // 32) * 64 + 1
    gen = torch.Generator(device=hip_device).manual_seed(10)
    x = torch.randn(n, k, generator=gen, device=hip_device)
    layer = Simulator(cfg, device=hip_device).map(
        torch.randn(o, k, generator=gen, device=hip_device), name="layer")
    assert hip.mm_kernel(cfg, n, 1, 1) == 0
    got = layer(x)
    q, xs = hip.input_tiles(x[-65:], cfg)
    g = hip.restore(layer.packed, cfg, layer.seed, 0, 0, 1)
    expected = hip.mm(q, xs, layer.packed, None, layer.weight_scale.reshape(-1, layer.p * cfg.array_size[1]),
                      cfg, layer.seed, 0, conductance=g, k_rows=k)[:, :o]
    assert torch.equal(got[-65:].view(torch.int32), expected.contiguous().view(torch.int32))


def totals_in_64_bits(cfg, q, g):
    """Slice totals [N, G, p*C] of codes ``q`` [N, m, R] read through conductances ``g``
    [m, p, W, R, C], every product, sum and conversion in FP64."""
    n, m, r = q.shape
    p, c, rows = g.shape[1], g.shape[4], cfg.read_rows
    totals = torch.zeros(n, m * r // rows, p * c, dtype=torch.float64, device=q.device)
    codes = q.long()
    for read in range(totals.shape[1]):
        i, first = divmod(read * rows, r)
        for shift, mask, in_factor in cfg.input_layout:
            digits = ((codes[:, i, first:first + rows] >> shift) & mask).double()
            for w, (_, w_mask, w_factor) in enumerate(cfg.weight_layout):
                level = g[i, :, w, first:first + rows].double() - cfg.low_conductance
                current = digits @ level.permute(1, 0, 2).reshape(rows, p * c) * cfg.read_voltage
                counts = (current * (w_mask / cfg.current_unit)).clamp(0, cfg.adc_maxima[w]).round()
                totals[:, read] += counts * (in_factor * w_factor)
    return totals


@pytest.mark.parametrize("variation", [0.02, 0.1, 0.3])
@pytest.mark.parametrize("name", ["default", "int4_faults", "six_slices", "rows128",
                                  "rows128_sliced"])
def test_closer_to_64_bits_than_the_general_read(hip_device, name, variation):
    """Programming noise puts converter arguments anywhere between two counts, and the two reads
    round the closest ones differently: the block read's totals miss the 64-bit ones no more often
    than the general read's.  (Both counts are of rare independent events: four standard
    deviations of their difference.)"""
    kwargs, effects = CASES[name]
    cfg = Config(**kwargs, nonidealities=Nonidealities(**(effects | dict(write_variation=variation))))
    *_, q, _, packed, packed_t, _ = programmed(cfg, 256, 512, 256, hip_device, 12)
    n, p = q.shape[0], packed.shape[1]
    assert hip.mm_kernel(cfg, n, q.shape[1], p) == 2
    g = hip.restore(packed, cfg, 21, 0, 0, p)
    expected = totals_in_64_bits(cfg, q, g[0])
    block = hip.mm_totals(q, packed_t, cfg, 21, 0, conductance=g[0]).double().reshape_as(expected)
    general = hip.partial(q, packed, cfg, None, 21, 0, 0, p,
                          conductance=g).double().reshape_as(expected)
    missed, bound = int((block != expected).sum()), int((general != expected).sum())
    print("[block read]", name, variation, "off 64 bits:", missed, "general:", bound, "of",
          expected.numel() * len(cfg.input_layout) * len(cfg.weight_layout), flush=True)
    assert missed <= bound + 4 * (missed + bound) ** 0.5


def test_reads_between_counts_keep_the_general_kernel():
    """Read noise, drift, nonlinear converters and voltage noise: reads that have only been
    compared with 64 bits in the general kernel's order of sums."""
    for effects in (dict(read_variation=0.01), dict(adc_nonlinearity=0.1), dict(voltage_variation=0.01),
                    dict(drift_coefficient=0.05, drift_time=100.0)):
        cfg = Config(nonidealities=Nonidealities(**(WRITE | effects)))
        assert hip.mm_kernel(cfg, 100, 4, 4) == 0, effects


@pytest.mark.parametrize("name,reads", [("default", 300), ("rows128", 270), ("rows128_sliced", 17)])
def test_read_order_levels(hip_device, name, reads):
    """The fused cascade over more than 16 and 256 reads equals the split read's epilogue."""
    cfg = case(name)
    k = reads * cfg.read_rows - 5
    _, _, q, xs, packed, packed_t, ws = programmed(cfg, 40, k, 70, hip_device, 6)
    fused, split = (hip.mm(q, xs, packed, packed_t, ws, cfg, 9, 0, out_cols=70, k_rows=k,
                           variant=hip.variant_word(split=z))[:, :70] for z in (1, 4))
    assert torch.equal(fused.view(torch.int32), split.view(torch.int32))


@pytest.mark.parametrize("name,n,reads,o", [
    ("default", 700, 700, 600),          # passes of vectors
    ("int4_faults", 45, 3300, 2600),     # and of columns, the last of 13 vectors and 104 columns
    ("default", 32, 3300, 2600),         # one vector block on k_noisy_pairs
])
def test_splits_in_passes(hip_device, name, n, reads, o):
    """A split read whose totals exceed 1 GiB runs in passes; each output is the unsplit read's."""
    cfg = case(name)
    gen = torch.Generator(device=hip_device).manual_seed(7)
    k = reads * cfg.read_rows - 3
    a = torch.randn(n, k, generator=gen, device=hip_device)
    w = torch.randn(o, k, generator=gen, device=hip_device)
    q, xs = hip.input_tiles(a, cfg)
    packed, packed_t, ws = hip.weight_tiles(w, cfg)
    p = packed.shape[1]
    assert 4 * n * reads * p * cfg.array_size[1] > 1 << 30
    outputs = [hip.mm(q, xs, packed, packed_t, ws.reshape(-1, p * cfg.array_size[1]), cfg, 11, 0,
                      out_cols=o, k_rows=k, variant=hip.variant_word(split=z))[:, :o]
               for z in (1, 0, 3)]
    for output in outputs[1:]:
        assert torch.equal(output.view(torch.int32), outputs[0].view(torch.int32))


def test_tuned_read_without_samples_beyond_its_budget(hip_device, tmp_path):
    """Ideal devices need no sampled conductances: where the block read's terms exceed a tuned
    simulator's workspace budget, the general kernel reads the same counts."""
    cfg = case("rows128_ideal")
    gen = torch.Generator().manual_seed(8)
    a, b = torch.randn(40, 500, generator=gen), torch.randn(500, 200, generator=gen)
    tuned = Simulator(cfg, device=hip_device, mode="tuned", cache_dir=tmp_path, workspace_mb=0.01)
    got = tuned.mm(a.to(hip_device), b.to(hip_device))
    expected = Simulator(cfg, device=hip_device).mm(a.to(hip_device), b.to(hip_device))
    assert torch.equal(got.view(torch.int32), expected.view(torch.int32))
    assert tuned.report()["selections"][0]["selected"] is not None
    assert tuned.report()["selections"][0]["kernel"] == 0
    # A budget that only the unsplit read's scratch fits: that schedule keeps the block read.
    n, m, p = 40, 4, 4
    need = {z: hip.mm_workspace_bytes(cfg, n, m, p, hip.variant_word(split=z)) for z in (0, 1)}
    assert need[1] < need[0]
    partly = Simulator(cfg, device=hip_device, mode="tuned", cache_dir=tmp_path / "partly",
                       workspace_mb=need[1] / 1024**2)
    got = partly.mm(a.to(hip_device), b.to(hip_device))
    assert torch.equal(got.view(torch.int32), expected.view(torch.int32))
    record = partly.report()["selections"][0]
    unsplit = [c for c in record["candidates"] if c["schedule"]["split"] == 1][0]
    assert unsplit["status"] == "accepted" and unsplit["resources"]["threads"] == 256
    assert record["kernel"] == (2 if record["selected"]["split"] == 1 else 0)
