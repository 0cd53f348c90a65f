"""Padded copies of a convolution's input in planes (factors of strided or padded k x k layers): bands
of rows with a remainder, rows that do not fit into LDS, phases and columns outside of the image,
several small images to a workgroup.
Small whole numbers, so that every product and sum is exact and the factors have to be equal."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

CASES = [   # input, kernel, stride, padding, dilation, bias
    ((2, 3, 64, 80), (3, 3), (2, 2), (1, 1), (1, 1), False),       # two bands
    ((2, 2, 131, 61), (7, 7), (2, 2), (3, 3), (1, 1), False),      # bands with a remainder
    ((1, 2, 40, 4096), (3, 1), (1, 2), (1, 0), (1, 1), False),     # a band is one row
    ((1, 1, 9, 4099), (3, 3), (2, 2), (1, 1), (1, 1), True),       # a row does not fit into LDS
    ((1, 1, 70, 300), (3, 2), (14, 3), (2, 1), (1, 1), False),     # a row of all phases does not
    ((2, 2, 33, 21), (5, 3), (3, 2), (4, 2), (2, 3), True),        # dilated, wide padding
    ((1, 2, 3, 2), (5, 5), (2, 2), (4, 4), (1, 1), False),         # bands that lie in the padding
    ((2, 37, 9, 9), (1, 1), (2, 2), (0, 0), (1, 1), False),        # pointwise with a stride, one row phase
    ((3, 201, 6, 5), (1, 1), (2, 3), (0, 0), (1, 1), False),       # several images an item, with a remainder
    ((2, 53, 11, 10), (3, 3), (2, 2), (1, 1), (1, 1), True),       # ... through LDS
    ((2, 3, 70, 90), (1, 1), (3, 2), (1, 0), (1, 1), True),        # ... padded, with a bias
    ((1, 1, 400, 3), (2, 3), (2, 1), (0, 1), (1, 1), True),        # one pixel column of a stride, tall
]


@pytest.mark.parametrize('shape,kernel,stride,padding,dilation,bias', CASES)
def test_factor_equals_unfolded_product(shape, kernel, stride, padding, dilation, bias):
    from torchsso import _ops
    dev = torch.device('cuda:0')
    g = torch.Generator().manual_seed(sum(shape))
    x = torch.randint(-3, 4, shape, generator=g).float()
    m = F.unfold(x.double(), kernel, dilation, padding, stride)      # [n, c kh kw, L]
    m = m.transpose(0, 1).reshape(m.shape[1], -1)
    if bias:
        m = torch.cat([m, torch.ones_like(m[:1])])
    ref = m @ m.t()
    assert ref.abs().max().item() < 2. ** 24
    out = torch.full(tuple(ref.shape), float('nan'), device=dev)
    xd = x.to(dev)
    job = _ops.factor_job('conv_a', xd, 1., out, add_bias=bias, kernel_size=kernel, stride=stride,
                          padding=padding, dilation=dilation)
    # (a pointwise layer reads a copy in a call that makes others)
    other = torch.full((9, 9), float('nan'), device=dev)
    zeros = torch.zeros(1, 1, 5, 5, device=dev)
    _ops.factor_grouped([job, _ops.factor_job('conv_a', zeros, 1., other, kernel_size=3, stride=2)], dev)
    assert torch.equal(out.double().cpu(), ref) and not other.any().item()
    out.fill_(float('nan'))
    _ops.factor_grouped([job], dev)
    assert torch.equal(out.double().cpu(), ref)
