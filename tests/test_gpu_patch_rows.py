"""The surrogate's patch rows against F.unfold: values and gradients, bit for bit."""

import pytest
import torch
from torch.nn import functional as F

from memfast_amd.nn.training import _PatchRows

pytestmark = pytest.mark.gpu


# (N, C, H, W), kernel, dilation, padding, stride
@pytest.mark.parametrize("shape,kernel,dilation,padding,stride", [
    ((1, 1, 1, 1), (1, 1), (1, 1), (0, 0), (1, 1)),
    ((3, 7, 9, 11), (3, 3), (1, 1), (1, 1), (1, 1)),      # 63 columns
    ((2, 13, 8, 6), (5, 1), (2, 1), (4, 0), (1, 3)),      # 65 columns
    ((1, 64, 5, 7), (1, 1), (1, 1), (2, 3), (2, 2)),      # whole rows of padding
    ((33, 5, 17, 13), (3, 5), (2, 3), (3, 6), (3, 2)),
])
def test_patch_rows(hip_device, shape, kernel, dilation, padding, stride):
    gen = torch.Generator().manual_seed(sum(shape))
    x = torch.randn(shape, generator=gen).to(hip_device)
    for image in (x, x.to(memory_format=torch.channels_last), x.transpose(2, 3).contiguous().transpose(2, 3)):
        leaf, other = (image.clone().requires_grad_() for _ in range(2))
        rows = _PatchRows.apply(leaf, kernel, dilation, padding, stride)
        expected = F.unfold(other, kernel, dilation, padding, stride).transpose(1, 2)
        assert rows.is_contiguous() and torch.equal(rows, expected)
        grad = torch.randn(rows.shape, generator=gen).to(hip_device)
        rows.backward(grad)
        expected.backward(grad)
        assert torch.equal(leaf.grad, other.grad)
