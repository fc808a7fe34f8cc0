"""GPU: the product of a strip of columns (prompt_product's last columns) against 64 bits, at the edges of its tiles,
for inner dimensions of whole and of odd numbers of stages, and the rule that cuts the strip off."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _bound(want, mag, k, dtype):
    # the result's rounding, and sums of k products in 32 bits in any order
    return 2.0 ** (-11 if dtype == torch.float16 else -8) * want.abs() + k * 2.0 ** -24 * mag


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m", [1, 63, 64, 65, 300])
@pytest.mark.parametrize("n,k", [(4, 64), (64, 128), (132, 192), (256, 448), (256, 512), (256, 576), (260, 4096)])
def test_strip(cuda, dtype, m, n, k):
    from tidaldecode_amd import _lib

    g = torch.Generator(device=cuda).manual_seed(m + n + k)
    x = torch.randn((m, k), generator=g, device=cuda).to(dtype)
    w = torch.randn((n, k), generator=g, device=cuda).to(dtype)
    out = torch.full((m, n + 4), 7.0, dtype=dtype, device=cuda)
    code = _lib.TD_F16 if dtype == torch.float16 else _lib.TD_BF16
    for _ in range(2):
        _lib.check(_lib.lib.td_gemm_strip(x.data_ptr(), w.data_ptr(), out.data_ptr(), m, n, k, n + 4, code,
                                          torch.cuda.current_stream().cuda_stream))
    want, mag = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    assert ((out[:, :n].double() - want).abs() <= _bound(want, mag, k, dtype)).all()
    assert (out[:, n:] == 7.0).all()


@pytest.mark.parametrize("m,n,k", [(513, 22016, 128), (700, 22016, 192), (958, 16640, 64), (258, 33024, 64),
                                   (700, 22272, 128), (200, 22016, 128)])
def test_prompt_product(cuda, m, n, k):
    from tidaldecode_amd import _kernels

    g = torch.Generator(device=cuda).manual_seed(m)
    x = torch.randn((m, k), generator=g, device=cuda).bfloat16()
    w = torch.randn((n, k), generator=g, device=cuda).bfloat16()
    assert _kernels._cut_columns(m, n, k) == (256 if (m, n) in ((513, 22016), (700, 22016), (958, 16640)) else 0)
    with torch.no_grad():
        out = _kernels.prompt_product(x, w)
        other = _kernels.prompt_product(x.t().contiguous().t(), w)  # a layout that stays one product
    want, mag = x.float() @ w.float().t(), x.float().abs() @ w.float().abs().t()
    assert out.shape == (m, n) and out.is_contiguous()
    for got in (out, other):
        assert ((got.float() - want).abs() <= _bound(want, 2 * mag, k, torch.bfloat16)).all()


def test_arguments_are_checked(cuda):
    from tidaldecode_amd import _lib

    t = torch.zeros((64, 64), dtype=torch.bfloat16, device=cuda)
    p, st = t.data_ptr(), torch.cuda.current_stream().cuda_stream
    for args in ((0, 64, 64, 64), (64, 6, 64, 64), (64, 64, 96, 64), (64, 64, 64, 32), (64, 64, 64, 66)):
        with pytest.raises(RuntimeError, match="td_gemm_strip"):
            _lib.check(_lib.lib.td_gemm_strip(p, p, p, *args, _lib.TD_BF16, st))
    with pytest.raises(RuntimeError, match="aligned"):
        _lib.check(_lib.lib.td_gemm_strip(p + 2, p, p, 64, 64, 64, 64, _lib.TD_BF16, st))
