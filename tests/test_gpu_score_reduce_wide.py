"""GPU: score_reduce with four tokens a thread (large reductions of aligned rows) against one token a thread, which
rows that are not 16-byte aligned take: the same sums in the same order, so the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,n", [(8, 8, 32768), (32, 8, 32769), (33, 3, 87555), (40, 8, 40003), (9, 1, 262147),
                                      (64, 1, 262144), (17, 17, 15422)])
def test_same_bits(cuda, hq, hkv, n):
    from tidaldecode_amd import _kernels

    g = torch.Generator(device=cuda).manual_seed(n)
    wide = torch.full((hq, (n + 3) // 4 * 4), float("nan"), device=cuda)
    narrow = torch.full((hq, n + (2 if n % 2 else 1)), float("nan"), device=cuda)
    wide[:, :n] = 3 * torch.randn((hq, n), generator=g, device=cuda)
    wide[0, n // 2] = float("-inf")
    narrow[:, :n] = wide[:, :n]
    assert wide.stride(0) % 4 == 0 and narrow.stride(0) % 4 != 0
    lse = torch.logsumexp(wide[:, :n], dim=-1)
    for mode, rows in (("head_sum", 1), ("group_sum", hkv)):
        a = _kernels.score_reduce(wide, lse, hkv, n, mode)
        b = _kernels.score_reduce(narrow, lse, hkv, n, mode)
        assert a.shape == (rows, n) and torch.equal(a, b)
        want = torch.exp(wide[:, :n].double() - lse[:, None].double()).view(rows, hq // rows, n).sum(1)
        # an exponential of 2^-20 relative error (arguments up to 2^5 in 32 bits), summed in 32 bits
        assert ((a.double() - want).abs() <= 2.0 ** -16 * want + 1e-12).all()


@pytest.mark.parametrize("n", [2 ** 31 - 256, 2 ** 31 - 100, 2 ** 31 - 99])
def test_as_many_tokens_as_a_row_may_have(cuda, n):
    """More than one launch numbers; rows whose last workgroup of 256 tokens would end beyond 31 bits, and one
    that is read a token at a time."""
    from tidaldecode_amd import _kernels

    logits = torch.zeros((1, n), device=cuda)
    at = [0, 2 ** 30 - 65, 2 ** 30 - 64, 2 ** 30 + 1, n - 2, n - 1]
    for j, i in enumerate(at):
        logits[0, i] = j + 1.0
    out = torch.full((1, n), -1.0, device=cuda)
    _kernels.score_reduce(logits, torch.zeros(1, device=cuda), 1, n, "head_sum", out=out)
    del logits
    assert torch.allclose(out[0, at].cpu(), torch.arange(1.0, 7.0).exp(), rtol=1e-6)
    out[0, at] = 1.0
    assert out.amin() == 1.0 and out.amax() == 1.0
