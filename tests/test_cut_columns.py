"""CPU: which products of a prompt leave their last strip of columns to a kernel of its own."""
import pytest
import torch


@pytest.mark.parametrize("m,n,k,cut", [(513, 22016, 4096, 256), (576, 22016, 4096, 256), (577, 22016, 4096, 0),
                                       (640, 22016, 4096, 0), (641, 22016, 4096, 256), (768, 22016, 4096, 256),
                                       (769, 22016, 4096, 0), (2900, 22016, 4096, 256), (700, 22016, 0, 0),
                                       (700, 22016, 32, 0), (700, 22016, 96, 0), (300, 28672, 4096, 0)])
def test_rule(m, n, k, cut):
    from tidaldecode_amd._kernels import _cut_columns

    assert _cut_columns(m, n, k) == cut


def test_an_empty_inner_dimension_gives_zeros():
    from tidaldecode_amd import _kernels

    with torch.no_grad():
        out = _kernels.prompt_product(torch.zeros(700, 0), torch.zeros(22016, 0))
    assert out.shape == (700, 22016) and not out.any()
