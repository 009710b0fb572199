"""Quantizers of long groups: whole rows of the inputs (k_row_groups_block) and whole columns of
the weights (k_column_peaks, k_column_scales), bit for bit against the oracle at the edges of
their waves, workgroups, chunks and tiles."""

import pytest
import torch

from memfast_amd import Config, Nonidealities, hip
from oracle import oracle

pytestmark = pytest.mark.gpu

IDEAL = Nonidealities(write_variation=0.0)


def same(a, b):
    view = torch.int32 if a.dtype == torch.float32 else torch.uint8
    return torch.equal(a.cpu().contiguous().view(view), b.contiguous().view(view))


@pytest.mark.parametrize("k,group", [(64, None), (65, None), (100, None), (784, None),
                                     (1023, None), (1025, None), (4100, None), (9001, None),
                                     (300, 128), (3000, 192), (2900, 1280)])
@pytest.mark.parametrize("n", [1, 5])
def test_row_groups(hip_device, n, k, group):
    cfg = Config(input_quant_gran=(1, group), array_size=(64, 32), nonidealities=IDEAL)
    gen = torch.Generator().manual_seed(k + n)
    a = torch.randn(n, k, generator=gen)
    a[-1] = 0.0     # a group of zeros
    q, xs = hip.input_tiles(a.to(hip_device), cfg)
    q_ref, xs_ref = oracle.input_tiles(a, cfg)
    assert same(q, q_ref) and same(xs, xs_ref)
    for value in (float("nan"), float("inf")):
        bad = a.clone()
        bad[0, k - 1] = value
        status = hip.status_word(hip_device)
        hip.input_tiles(bad.to(hip_device), cfg, status=status)
        assert int(status.item()) == hip.STATUS_INPUT


ARRAYS = {
    "default": dict(),
    "unsigned4": dict(weight_bits=4, weight_signed=False),
    "two_reads": dict(array_size=(128, 128), rows_per_read=64),
    "rows48": dict(array_size=(48, 64)),
    "short_last_read": dict(array_size=(80, 64), rows_per_read=30),
    "rows256": dict(array_size=(256, 192), rows_per_read=64),
}


@pytest.mark.parametrize("name", list(ARRAYS))
@pytest.mark.parametrize("k,o", [(65, 1), (100, 63), (128, 64), (129, 260), (513, 200), (1500, 130)])
def test_whole_column_groups(hip_device, name, k, o):
    cfg = Config(**ARRAYS[name], nonidealities=IDEAL)
    gen = torch.Generator().manual_seed(k + o)
    b = torch.randn(k, o, generator=gen)
    b[:, o // 2] = 0.0
    b = b if cfg.weight_signed else b.abs()
    packed, packed_t, ws = hip.weight_tiles(b.T.to(hip_device), cfg)
    packed_ref, ws_ref = oracle.weight_tiles(b.T, cfg)
    m, p, r, c = packed_ref.shape
    assert same(packed, packed_ref) and same(ws, ws_ref)
    assert same(packed_t, packed_ref.permute(1, 3, 0, 2).reshape(p * c, m * r))
    bad = b.clone()
    bad[k - 1, o - 1] = float("inf")
    status = hip.status_word(hip_device)
    hip.weight_tiles(bad.T.to(hip_device), cfg, status=status)
    assert int(status.item()) == hip.STATUS_WEIGHT
