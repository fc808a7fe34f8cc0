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
