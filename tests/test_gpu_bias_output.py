"""The bias of a padded read against torch's add, bit for bit, with its finiteness flag."""

import pytest
import torch

from memfast_amd import hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,o,wide", [(1, 1, 4), (5, 3, 64), (300, 64, 256), (7, 260, 260),
                                      (9, 1028, 1100), (2, 1030, 1088)])
def test_bias_of_a_padded_read(hip_device, n, o, wide):
    gen = torch.Generator().manual_seed(n + o)
    full = torch.randn(n, wide, generator=gen).to(hip_device)
    full[:, o:] = float("nan")     # columns past the layer's are never read
    bias = torch.randn(o, generator=gen).to(hip_device)
    expected = full[:, :o] + bias
    inplace = full[:, :o].clone()
    status = hip.status_word(hip_device)
    assert torch.equal(hip.bias_output(full[:, :o], bias, status), expected)
    assert int(status.item()) == 0
    assert torch.equal(hip.bias_add(inplace, bias, status), expected)
    full[n - 1, o - 1] = bias[o - 1] = torch.finfo(torch.float32).max
    hip.bias_output(full[:, :o], bias, status)
    assert int(status.item()) == hip.STATUS_OUTPUT
