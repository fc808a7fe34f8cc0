"""GPU parity of the prompt attention on short caches: the lengths around the edges of the staged kernel, of its
form with two key groups and of its pieces, against attention in fp32; and values behind a row, which must not
reach it from the other key group."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(cuda, hq, hkv, d, page, past, n, dtype):
    g = torch.Generator(device=cuda).manual_seed(past * 7 + n)
    total = past + n
    pages = -(-total // page)
    pool = torch.randn((pages, 2, page, hkv, d), generator=g, device=cuda).to(dtype)
    table = torch.randperm(pages, generator=g, device=cuda).int()
    q = torch.randn((n, hq, d), generator=g, device=cuda).to(dtype)
    return pool, table, q, total


def _want(pool, table, q, total, hkv, causal):
    n, hq, d = q.shape
    k = pool[table.long(), 0].reshape(-1, hkv, d)[:total].float().repeat_interleave(hq // hkv, 1).transpose(0, 1)
    v = pool[table.long(), 1].reshape(-1, hkv, d)[:total].float().repeat_interleave(hq // hkv, 1).transpose(0, 1)
    s = q.float().transpose(0, 1) @ k.transpose(1, 2).contiguous() / math.sqrt(d)
    if causal:
        pos = torch.arange(total - n, total, device=q.device)
        s = s.masked_fill(torch.arange(total, device=q.device)[None] > pos[:, None], float("-inf"))
    return (torch.softmax(s, -1) @ v).transpose(0, 1)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hq,hkv,d", [(32, 8, 128), (12, 12, 128), (7, 1, 128), (16, 4, 64)])
@pytest.mark.parametrize("past,n", [(0, 65), (0, 96), (0, 97), (0, 128), (31, 97), (0, 256), (0, 257), (200, 312),
                                    (0, 512), (1, 512), (300, 16), (600, 5), (1584, 16), (1585, 16), (470, 40)])
def test_edges(cuda, dtype, hq, hkv, d, past, n):
    from tidaldecode_amd import _kernels

    tol = 2e-3 if dtype == torch.float16 else 1e-2
    for page in (16, 5):
        pool, table, q, total = _case(cuda, hq, hkv, d, page, past, n, dtype)
        for causal in (True, False):
            got = _kernels.prefill_with_paged_kv_cache(q, pool, table, (total - 1) % page + 1, causal, 0, False, 1.0, 1e4)
            want = _want(pool, table, q, total, hkv, causal)
            # rows of a few tokens keep values of the size of v, whose 16-bit rounding is relative
            assert ((got.float() - want).abs() <= tol * want.abs().clamp(min=1.0)).all(), (page, causal)


@pytest.mark.parametrize("behind", [float("inf"), float("nan")])
def test_a_value_in_tiles_behind_a_row_does_not_reach_it(cuda, behind):
    from tidaldecode_amd import _kernels

    pool, table, q, total = _case(cuda, 4, 4, 128, 16, 0, 300, torch.bfloat16)
    flat = pool[table.long()]
    flat[-4:, 1] = behind                 # values of the last 64-odd tokens
    pool[table.long()] = flat
    got = _kernels.prefill_with_paged_kv_cache(q, pool, table, (total - 1) % 16 + 1, True, 0, False, 1.0, 1e4)
    first_bad = 16 * (pool.size(0) - 4)
    # the rows of whole 64-row tiles in front of the key tile that holds the first of them
    seen = first_bad // 64 * 64
    assert torch.isfinite(got[:seen].float()).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("kv_len,n_q,top", [(96, 96, 90), (300, 128, 100), (300, 128, 200), (500, 100, 499),
                                            (1500, 16, 1111)])
def test_a_weight_just_above_an_earlier_tile_is_not_rounded(cuda, dtype, d, kv_len, n_q, top):
    """One key outweighs all others by 2^2.1 to 2^8.4, which the tiles in front of it do not show: its weight is
    the row's reference and so exactly 1.  What is left are the roundings (u) of the result and of the small
    weights, and 1e-5 for the sums and exponentials in 32 bits."""
    from tidaldecode_amd import _kernels

    g = torch.Generator().manual_seed(d + top)
    pages = -(-kv_len // 16)
    pool = torch.zeros((pages, 2, 16, 1, d))
    pool.view(pages, 2, 16, d)[top // 16, 0, top % 16] = 1.0
    pool[:, 1] = torch.randn((pages, 16, 1, d), generator=g)
    pool = pool.to(dtype)
    q = (torch.linspace(2.1, 8.4, n_q) / (math.sqrt(d) * math.log2(math.e)))[:, None, None].expand(n_q, 1, d).to(dtype)
    got = _kernels.prefill_with_paged_kv_cache(q.contiguous().to(cuda), pool.to(cuda),
                                               torch.arange(pages, dtype=torch.int32, device=cuda),
                                               (kv_len - 1) % 16 + 1, False, 0, False, 1.0, 1e4)[:, 0].double().cpu()
    k, v = (pool[:, i].reshape(-1, d)[:kv_len].double() for i in (0, 1))
    p = (q[:, 0].double() @ k.t() / math.sqrt(d)).softmax(-1)
    want = p @ v
    p[:, top] = 0.0
    u = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    assert ((got - want).abs() <= 1.01 * u * (want.abs() + p @ v.abs()) + 1e-5).all()
