"""GPU: the product of a short prompt's few rows against 64 bits, at the edges of its row tiles, for even and uneven
cuts of the inner dimension down to a step each, and the rule that takes it."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _bound(want, mag, k, dtype):
    # the result's rounding, and sums of k products in 32 bits in any order
    return 2.0 ** (-11 if dtype == torch.float16 else -8) * want.abs() + k * 2.0 ** -24 * mag


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m", [1, 16, 17, 48, 49, 80, 81, 112, 113, 138, 144, 145, 300])
@pytest.mark.parametrize("n,k,splits", [(64, 128, 1), (64, 256, 2), (192, 384, 1), (576, 896, 3), (512, 4096, 4), (128, 1408, 8)])
def test_rows(cuda, dtype, m, n, k, splits):
    from tidaldecode_amd import _lib

    g = torch.Generator(device=cuda).manual_seed(m + n + k)
    x = torch.randn((m, k), generator=g, device=cuda).to(dtype)
    w = torch.randn((n, k), generator=g, device=cuda).to(dtype)
    out = torch.full((m + 1, n), 7.0, dtype=dtype, device=cuda)
    parts = torch.full((splits, m, n), float("nan"), device=cuda)
    for _ in range(2):
        _lib.check(_lib.lib.td_gemm_rows(x.data_ptr(), w.data_ptr(), out.data_ptr(), m, n, k, splits, parts.data_ptr(),
                                         parts.numel() * 4, _lib.TD_F16 if dtype == torch.float16 else _lib.TD_BF16,
                                         torch.cuda.current_stream().cuda_stream))
    want, mag = x.double() @ w.double().t(), x.double().abs() @ w.double().abs().t()
    assert ((out[:m].double() - want).abs() <= _bound(want, mag, k, dtype)).all()
    assert (out[m] == 7.0).all()


# (sizes where the kernel is the faster one, and beside them some where it is up to 1.4 times as slow)
@pytest.mark.parametrize("m,n,k,splits", [(64, 4096, 4096, 4), (138, 6144, 4096, 2), (144, 4096, 11008, 4), (80, 6144, 4096, 0),
                                          (145, 4096, 4096, 0), (100, 12288, 4096, 0), (100, 4096, 1024, 0), (30, 4160, 4096, 0),
                                          (100, 4160, 2048, 0), (16, 4096, 4096, 0), (33, 512, 8192, 8), (100, 4160, 3584, 3),
                                          (48, 4096, 4096, 4), (49, 4096, 4096, 0), (63, 4096, 11008, 4), (120, 4096, 4096, 0),
                                          (120, 4096, 11008, 4), (128, 4096, 4096, 4), (129, 4096, 4096, 4), (32, 4096, 8192, 0),
                                          (33, 4096, 8192, 4), (90, 8192, 8192, 0), (90, 8192, 14336, 2), (90, 2048, 2048, 0),
                                          (40, 64, 4096, 0)])
def test_rule(cuda, m, n, k, splits):
    from tidaldecode_amd import _kernels

    assert _kernels._row_splits(m, n, k) == splits
    g = torch.Generator(device=cuda).manual_seed(m)
    x = torch.randn((m, k), generator=g, device=cuda).bfloat16()
    w = torch.randn((n, k), generator=g, device=cuda).bfloat16()
    with torch.no_grad():
        out = _kernels.prompt_product(x, w)
        other = _kernels.prompt_product(x.t().contiguous().t(), w)  # a layout that stays the library's
    want, mag = x.float() @ w.float().t(), x.float().abs() @ w.float().abs().t()
    for got in (out, other):
        assert got.shape == (m, n) and ((got.float() - want).abs() <= _bound(want, 2 * mag, k, torch.bfloat16)).all()


@pytest.mark.parametrize("m", [64, 16])  # a row count the kernel takes, one that is the library's anyway
def test_calls_that_are_the_librarys(cuda, m):
    """What torch's own product does, or refuses, and the kernel could not: operands on two devices, a weight of one
    dimension, vmap, tangents, traces, tensors of another class."""
    from tidaldecode_amd._kernels import _row_splits, prompt_product

    assert (_row_splits(m, 2048, 4096) > 0) == (m == 64)
    g = torch.Generator(device=cuda).manual_seed(m)
    x = torch.randn((m, 4096), generator=g, device=cuda).bfloat16()
    w = torch.randn((2048, 4096), generator=g, device=cuda).bfloat16()
    with torch.no_grad():
        with pytest.raises(RuntimeError, match="device"):
            prompt_product(x, w.cpu())
        with pytest.raises(RuntimeError, match="device"):
            prompt_product(x.cpu(), w)
        with pytest.raises(RuntimeError, match="shape"):
            prompt_product(x, w[:, :4032].contiguous())
        assert torch.equal(prompt_product(x, w[0].contiguous()), x @ w[0])
        rows = torch.stack([x, 2 * x])
        assert torch.equal(torch.func.vmap(lambda a: prompt_product(a, w))(rows), torch.func.vmap(lambda a: a @ w.t())(rows))
        with torch.autograd.forward_ad.dual_level():
            dual = torch.autograd.forward_ad.make_dual(x, x)
            assert torch.autograd.forward_ad.unpack_dual(prompt_product(dual, w)).tangent is not None
        traced = torch.jit.trace(prompt_product, (x, w), check_trace=False)
        assert torch.equal(traced(3 * x, w), (3 * x) @ w.t())

        class Watched(torch.Tensor):
            pass

        assert type(prompt_product(x.as_subclass(Watched), w)) is Watched


def test_arguments_are_checked(cuda):
    from tidaldecode_amd import _lib

    t = torch.zeros((64, 128), dtype=torch.bfloat16, device=cuda)
    p, st = t.data_ptr(), torch.cuda.current_stream().cuda_stream
    for args in ((0, 64, 128, 1), (64, 32, 128, 1), (64, 64, 64, 1), (64, 64, 128, 2), (64, 64, 128, 0)):
        with pytest.raises(RuntimeError, match="td_gemm_rows"):
            _lib.check(_lib.lib.td_gemm_rows(p, p, p, *args, p, 1 << 20, _lib.TD_BF16, st))
    with pytest.raises(RuntimeError, match="parts hold"):
        _lib.check(_lib.lib.td_gemm_rows(p, p, p, 64, 64, 256, 2, p, 64 * 64 * 4, _lib.TD_BF16, st))
