"""GPU parity: paged prefill attention (td_prefill_attn through prefill_with_paged_kv_cache)
against the CPU oracle's dense causal attention (pinned against torch SDPA in
tests/test_oracle.py).  Tolerance: max-abs 2e-3 (fp16) / 1e-2 (bf16) on identically rounded inputs,
scaled by max(1, |o|): the first rows of a prompt average one or two value rows, so |o| reaches 3-4
there and the rounding of the bf16 result alone is 8e-3 at that magnitude.
The grid follows the reference's prefill test (kernels/src/test/test_batch_prefill.cu: query
lengths against longer caches, page sizes, causal on/off, both layouts)."""
import math

import pytest
import torch

from _util import ATOL, PagedCase, randn

pytestmark = pytest.mark.gpu


def _dense(q, k, v, causal):
    """fp32 reference: q [n_q, Hq, D] are the newest n_q of the kv_len tokens in k, v [kv_len, Hkv, D]"""
    n_q, hq, d = q.shape
    kv_len, hkv, _ = k.shape
    g = hq // hkv
    kk, vv = k.repeat_interleave(g, 1), v.repeat_interleave(g, 1)
    logit = torch.einsum("qhd,khd->hqk", q, kk) / math.sqrt(d)
    if causal:
        qpos = torch.arange(kv_len - n_q, kv_len)[:, None]
        logit = logit.masked_fill(torch.arange(kv_len)[None, :] > qpos, float("-inf"))
    return torch.einsum("hqk,khd->qhd", logit.softmax(-1), vv)


def _run(cuda, case, q, causal, dtype):
    from tidaldecode_amd import _kernels

    o = _kernels.prefill_with_paged_kv_cache(
        q.to(dtype).to(cuda), case.pool.to(cuda), case.page_table.to(torch.int32).to(cuda),
        case.last_page_len, causal, case.layout, False, 1.0, 1e4)
    torch.cuda.synchronize()
    return o


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kv_len,n_q", [(1, 1), (17, 17), (70, 70), (128, 128), (129, 129),
                                        (1000, 1000), (4099, 4099), (4099, 37), (5000, 1),
                                        (777, 300), (2048, 129)])
def test_causal_prefill_matches_dense_attention(cuda, dtype, kv_len, n_q):
    hq, hkv, d, page = 8, 8, 128, 16
    case = PagedCase(kv_len, hkv, d, page, dtype, seed=kv_len + n_q)
    q = randn((n_q, hq, d), kv_len * 3 + n_q, dtype)
    want = _dense(q, case.k, case.v, True)
    # the oracle's single-query attention on the last row: the same restatement the decode tests use
    from oracle import tidal_oracle as orc

    last = orc.softmax_pv(orc.attn_logits(q[-1], case.k), case.v)
    assert (want[-1] - last).abs().max() < 1e-5
    got = _run(cuda, case, q, True, dtype)
    assert got.shape == (n_q, hq, d)
    assert ((got.float().cpu() - want).abs() <= ATOL[dtype] * want.abs().clamp(min=1.0)).all()


@pytest.mark.parametrize("hq,hkv,d,page,layout,causal", [
    (32, 8, 128, 16, 0, True), (4, 2, 64, 4, 0, True), (4, 4, 64, 16, 1, True),
    (8, 2, 128, 1, 0, True), (8, 8, 128, 8, 1, True), (6, 3, 128, 5, 0, True),
    (8, 8, 128, 16, 0, False), (4, 2, 64, 16, 1, False), (4, 2, 256, 16, 0, True),
    (2, 2, 256, 8, 1, True), (4, 1, 256, 16, 0, False)])
def test_head_layouts_page_sizes_and_non_causal(cuda, hq, hkv, d, page, layout, causal):
    dtype = torch.float16
    kv_len, n_q = 1500, 333
    case = PagedCase(kv_len, hkv, d, page, dtype, layout=layout, seed=hq * d + page)
    q = randn((n_q, hq, d), 11, dtype)
    want = _dense(q, case.k, case.v, causal)
    got = _run(cuda, case, q, causal, dtype)
    assert ((got.float().cpu() - want).abs() <= ATOL[dtype] * want.abs().clamp(min=1.0)).all()


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("page_size", [1, 8, 16])
@pytest.mark.parametrize("hq,hkv", [(32, 4), (32, 8), (32, 32), (8, 1), (8, 2), (8, 8)])
def test_reference_prefill_grid(cuda, hq, hkv, page_size, head_dim, causal):
    """The reference's prefill test grid (kernels/src/test/test_prefill.cu:408-467): its three
    families of lengths -- a few queries over a short cache (q in [1, 15), kv in [15, 257)), a fresh
    short prompt (q = kv in [1, 64)) and 63 queries over 2047 cached tokens -- with seeded draws."""
    dtype = torch.float16
    g = torch.Generator().manual_seed(hq * 1000 + hkv * 100 + page_size * 10 + head_dim + causal)
    q1 = int(torch.randint(1, 15, (1,), generator=g))
    kv1 = int(torch.randint(15, 257, (1,), generator=g))
    q2 = int(torch.randint(1, 64, (1,), generator=g))
    for n_q, kv_len in ((q1, kv1), (q2, q2), (63, 2047)):
        case = PagedCase(kv_len, hkv, head_dim, page_size, dtype, seed=kv_len + n_q + hkv)
        q = randn((n_q, hq, head_dim), n_q * 7 + kv_len, dtype)
        want = _dense(q, case.k, case.v, causal)
        got = _run(cuda, case, q, causal, dtype)
        assert ((got.float().cpu() - want).abs() <= ATOL[dtype] * want.abs().clamp(min=1.0)).all(), \
            (n_q, kv_len)


def test_prefill_at_benchmark_length(cuda):
    """32768 tokens, Llama-2-7B head shape (4 of the 32 heads, GQA 4/2): checked on sampled rows
    against the oracle's single-query attention over the row's causal prefix."""
    from oracle import tidal_oracle as orc

    dtype, n, hq, hkv, d, page = torch.bfloat16, 32768, 4, 2, 128, 16
    case = PagedCase(n, hkv, d, page, dtype, seed=5)
    q = randn((n, hq, d), 6, dtype)
    got = _run(cuda, case, q, True, dtype).float().cpu()
    for row in (0, 1, 127, 128, 4095, 20000, 32767):
        want = orc.softmax_pv(orc.attn_logits(q[row], case.k[: row + 1]), case.v[: row + 1])
        assert (got[row] - want).abs().max() <= ATOL[dtype] * max(1.0, want.abs().max().item()), row


def test_prefill_errors(cuda):
    from tidaldecode_amd import _kernels

    pool = torch.zeros((4, 2, 16, 2, 128), dtype=torch.float16, device=cuda)
    table = torch.arange(2, dtype=torch.int32, device=cuda)
    q = torch.zeros((40, 4, 128), dtype=torch.float16, device=cuda)
    with pytest.raises(RuntimeError):   # 40 queries, 20 cached tokens
        _kernels.prefill_with_paged_kv_cache(q, pool, table, 4, True, 0, False, 1.0, 1e4)
    with pytest.raises(RuntimeError):   # 3 query heads over 2 KV heads
        _kernels.prefill_with_paged_kv_cache(q[:8, :3].contiguous(), pool, table, 16, True, 0,
                                             False, 1.0, 1e4)
    with pytest.raises(RuntimeError, match="failed to dispatch"):   # head_dim without a kernel
        _kernels.prefill_with_paged_kv_cache(
            torch.zeros((4, 2, 32), dtype=torch.float16, device=cuda),
            torch.zeros((4, 2, 16, 2, 32), dtype=torch.float16, device=cuda), table, 16, True, 0,
            False, 1.0, 1e4)
    with pytest.raises(RuntimeError):   # dtype mismatch
        _kernels.prefill_with_paged_kv_cache(q[:8].bfloat16(), pool, table, 16, True, 0, False,
                                             1.0, 1e4)


@pytest.mark.parametrize("seed", range(16))
def test_random_configurations(cuda, seed):
    """Seeded random draws over head counts (incl. the 8-KV-head placement path and the eight-wave
    workgroups above 128 query rows), head_dim, page size, layout, dtype, causal, cache and query
    lengths."""
    import random

    rnd = random.Random(500 + seed)
    dtype = rnd.choice([torch.float16, torch.bfloat16])
    d = rnd.choice([64, 128, 128, 128, 256])
    hkv = rnd.choice([1, 2, 3, 8])
    hq = hkv * rnd.choice([1, 2, 4])
    page = rnd.choice([1, 3, 4, 8, 16, 16, 32])
    layout = rnd.choice([0, 1])
    causal = rnd.random() < 0.75
    kv_len = rnd.choice([1, 31, 64, 129, 257, 700, 1500, 2100])
    n_q = rnd.randint(1, kv_len)
    case = PagedCase(kv_len, hkv, d, page, dtype, layout=layout, seed=seed + 7)
    q = randn((n_q, hq, d), seed + 31, dtype)
    want = _dense(q, case.k, case.v, causal)
    got = _run(cuda, case, q, causal, dtype)
    ok = (got.float().cpu() - want).abs() <= ATOL[dtype] * want.abs().clamp(min=1.0)
    assert ok.all(), (dtype, d, hq, hkv, page, layout, causal, kv_len, n_q)


@pytest.mark.parametrize("dtype,hq,hkv,d,page,kv_len,n_q,pieces,rise", [
    # one to six key tiles around the rings of four and five, keys that end inside and on a tile
    (torch.bfloat16, 2, 2, 128, 16, 64, 64, False, 0.0), (torch.float16, 2, 2, 128, 16, 65, 65, False, 0.0),
    (torch.bfloat16, 2, 1, 128, 8, 192, 33, False, 12.0), (torch.float16, 1, 1, 64, 16, 257, 257, False, 12.0),
    (torch.bfloat16, 3, 3, 64, 5, 320, 256, False, 0.0), (torch.float16, 2, 2, 128, 1, 383, 300, False, 12.0),
    # packed rows of a group of seven: tokens cross waves and workgroup tiles
    (torch.bfloat16, 7, 1, 128, 16, 300, 37, False, 0.0), (torch.float16, 14, 2, 64, 3, 111, 74, False, 12.0),
    # keys cut into pieces: a last piece of one key, pieces past the end of the first rows, page sizes
    (torch.bfloat16, 8, 8, 128, 16, 20481, 16, True, 0.0), (torch.float16, 8, 2, 128, 16, 9000, 300, True, 12.0),
    (torch.float16, 4, 4, 64, 16, 6401, 257, True, 12.0), (torch.bfloat16, 4, 1, 128, 3, 5000, 1, True, 0.0),
    (torch.bfloat16, 2, 1, 256, 16, 4100, 70, True, 12.0), (torch.bfloat16, 4, 4, 128, 16, 2000, 2000, True, 0.0),
])
def test_row_packing_rings_and_pieces(cuda, dtype, hq, hkv, d, page, kv_len, n_q, pieces, rise):
    """The edges of the work split: key tiles of 64, rings, packed query rows, pieces and their merge.
    `rise`: queries grow to this many times their size, so that later keys exceed the first tile's by
    more than the factor of 2^8 that a row's reference point may lag, and accumulators are rescaled late.  Tolerance as above: weights are rounded
    relative to their own size whatever the reference point is."""
    from tidaldecode_amd import _kernels
    from tidaldecode_amd._lib import lib

    case = PagedCase(kv_len, hkv, d, page, dtype, seed=kv_len + n_q)
    q = randn((n_q, hq, d), kv_len * 3 + n_q, dtype)
    if rise:
        q = (q * torch.linspace(0.5, rise, n_q)[:, None, None]).to(dtype).float()
    planned = lib.td_prefill_workspace_bytes(_kernels._pool(case.pool.to(cuda), case.layout), kv_len, n_q, hq, 1)
    assert (planned > 0) == pieces
    if rise:   # some row's weights of its second to fourth key tile do exceed its first tile's by 2^8
        logit = torch.einsum("qhd,khd->hqk", q, case.k[:256].repeat_interleave(hq // hkv, 1)) / math.sqrt(d)
        logit = logit.masked_fill(torch.arange(logit.size(2)) > torch.arange(kv_len - n_q, kv_len)[:, None], -1e30)
        late = logit[..., 64:].amax(-1) - logit[..., :64].amax(-1)
        assert late.max().item() * math.log2(math.e) > 8.0
    got = _run(cuda, case, q, True, dtype).float().cpu()
    want = _dense(q, case.k, case.v, True)
    assert ((got - want).abs() <= ATOL[dtype] * want.abs().clamp(min=1.0)).all()


def _planned_bytes(case, q, causal):
    from tidaldecode_amd import _kernels
    from tidaldecode_amd._lib import lib

    # no pool: the plan depends on the geometry alone (and on whether the address is aligned)
    pool = _kernels.PagedKV(16, case.max_pages, case.hkv, case.d, case.page_size, case.layout,
                            _kernels._dtype_code(case.dtype, "pool"))
    return lib.td_prefill_workspace_bytes(pool, case.n, q.size(0), q.size(1), int(causal))


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("dtype,hq,hkv,d,past,n_q", [
    (torch.bfloat16, 8, 8, 128, 0, 4000), (torch.float16, 16, 16, 64, 0, 2900), (torch.bfloat16, 14, 2, 128, 0, 1500),
    (torch.float16, 4, 4, 128, 2048, 1000), (torch.bfloat16, 4, 2, 256, 0, 1500)])
def test_rows_that_see_no_key_of_a_piece_take_nothing_from_it(cuda, dtype, hq, hkv, d, past, n_q, bad):
    """Keys cut into pieces: everything from a key tile's first token on is infinite or NaN.  The rows
    before that token see none of it, whichever piece it lies in; their 32-token wave ends before it."""
    kv_len = past + n_q
    case = PagedCase(kv_len, hkv, d, 16, dtype, seed=kv_len)
    q = randn((n_q, hq, d), kv_len + 1, dtype)
    assert _planned_bytes(case, q, True) > 0
    want = _dense(q, case.k, case.v, True)
    q_d, pool, table = q.to(dtype).to(cuda), case.pool.to(cuda), case.page_table.to(cuda)
    from tidaldecode_amd import _kernels

    for t0 in range(kv_len // 64 * 64, past, -64):    # the clean part shrinks
        pool[table[t0 // 16:], 1] = bad
        got = _kernels.prefill_with_paged_kv_cache(q_d, pool, table.int(), case.last_page_len, True, 0, False, 1.0,
                                                   1e4)[: t0 - past].float().cpu()
        ref = want[: t0 - past]
        ok = (got - ref).abs() <= ATOL[dtype] * ref.abs().clamp(min=1.0)   # False for NaN
        assert ok.all(), (t0, (~ok).any(-1).any(-1).nonzero().flatten()[[0, -1]] + past)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("page", [1, 2, 3, 4, 5, 6, 7, 8, 12, 16])
def test_slots_outside_the_sequence_are_never_used(cuda, page, d, layout, causal):
    """The tail of the last page and every other page of the pool hold NaN, which weight 0 would not undo."""
    dtype, hq, hkv = torch.bfloat16, 4, 2
    for kv_len, n_q, pieces in ((5, 5, False), (37, 37, False), (70, 33, False), (1000, 1, True), (1001, 900, None),
                                (5000, 18, True)):
        case = PagedCase(kv_len, hkv, d, page, dtype, layout=layout, seed=kv_len + page)
        outside = torch.ones(case.max_pages * page, dtype=torch.bool)
        outside[case.slots_of(torch.arange(kv_len))] = False
        pages, entries = outside.view(-1, page).nonzero(as_tuple=True)
        view = case.pool if layout == 0 else case.pool.transpose(2, 3)   # [pages, 2, page, heads, d]
        view[pages, :, entries] = float("nan")
        q = randn((n_q, hq, d), kv_len, dtype)
        if pieces is not None:
            assert (_planned_bytes(case, q, causal) > 0) == pieces
        want = _dense(q, case.k, case.v, causal)
        got = _run(cuda, case, q, causal, dtype).float().cpu()
        assert ((got - want).abs() <= ATOL[dtype] * want.abs().clamp(min=1.0)).all(), (kv_len, n_q)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_a_weight_far_above_the_first_tile_is_not_rounded_again(cuda, dtype, d):
    """One key outweighs all others, which a row's first tile does not show: its weight is the row's
    reference and so exactly 1, up to which power of two the others are smaller.  What is left are the roundings
    (u) of the result and of the small weights."""
    n_q = kv_len = 128
    top = 100
    k = torch.zeros(kv_len, 1, d)
    k[top] = 1.0
    case = PagedCase(kv_len, 1, d, 16, dtype, seed=d, kv=(k, randn((kv_len, 1, d), d, dtype)))
    q = (torch.linspace(8.5, 13.9, n_q) / (math.sqrt(d) * math.log2(math.e)))[:, None, None].expand(n_q, 1, d)
    q = q.to(dtype).float()
    p = ((q[:, 0].double() @ k[:, 0].double().t()) / math.sqrt(d)).softmax(-1)
    v = case.v[:, 0].double()
    want = p @ v
    p[:, top] = 0.0
    u = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8     # half a unit in the last place, relative
    tol = 1.01 * u * (want.abs() + p @ v.abs()) + 1e-5          # 1e-5: sums and exponentials in 32 bits
    got = _run(cuda, case, q, False, dtype)[:, 0].double().cpu()
    assert ((got - want).abs() <= tol).all()


def test_memory_too_short_for_scratch(cuda):
    """Keys cut into pieces want 33 MB of partial results; where the allocator has 24 MB left, a call runs whole."""
    from tidaldecode_amd import _kernels

    dtype, past, n_q, h, d = torch.bfloat16, 8192, 500, 32, 128
    case = PagedCase(past + n_q, 8, d, 16, dtype, seed=3)
    q = randn((n_q, h, d), 4, dtype)
    assert _planned_bytes(case, q, True) > (24 << 20)
    want = _dense(q, case.k, case.v, True)
    q_d, pool, table = q.to(dtype).to(cuda), case.pool.to(cuda), case.page_table.int().to(cuda)
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(cuda).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (24 << 20)) / total)
    try:
        got = _kernels.prefill_with_paged_kv_cache(q_d, pool, table, case.last_page_len, True, 0, False, 1.0, 1e4)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert ((got.float().cpu() - want).abs() <= ATOL[dtype] * want.abs().clamp(min=1.0)).all()


@pytest.mark.parametrize("off", [1, 2, 4, 7])
@pytest.mark.parametrize("d,page,causal", [(64, 16, True), (64, 3, False), (128, 16, True), (128, 1, False), (256, 16, True)])
def test_pool_that_is_not_16_byte_aligned(cuda, d, page, causal, off):
    """A pool inside a wider buffer, `off` elements from its start: whole tiles and pieces."""
    from tidaldecode_amd import _kernels

    dtype, hq, hkv = torch.bfloat16, 4, 2
    for kv_len, n_q in ((37, 37), (700, 333), (5000, 18)):
        case = PagedCase(kv_len, hkv, d, page, dtype, seed=kv_len + d)
        q = randn((n_q, hq, d), kv_len + off, dtype)
        wide = torch.zeros(case.pool.numel() + 8, dtype=dtype, device=cuda)
        pool = wide[off: off + case.pool.numel()].view(case.pool.shape).copy_(case.pool)
        assert pool.data_ptr() % 16 == 2 * off
        got = _kernels.prefill_with_paged_kv_cache(q.to(dtype).to(cuda), pool, case.page_table.int().to(cuda),
                                                   case.last_page_len, causal, 0, False, 1.0, 1e4).float().cpu()
        want = _dense(q, case.k, case.v, causal)
        assert ((got - want).abs() <= ATOL[dtype] * want.abs().clamp(min=1.0)).all(), (kv_len, n_q)


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("hq,hkv,d,page", [(4, 4, 128, 16), (14, 2, 64, 3), (8, 1, 128, 1), (3, 1, 64, 32)])
def test_caches_of_one_key_tile(cuda, hq, hkv, d, page, causal):
    """Around 32 and 64 keys, where the kernel changes: fresh prompts, and a few rows on cached tokens."""
    dtype = torch.float16
    for kv_len in (1, 2, 15, 31, 32, 33, 63, 64, 65):
        case = PagedCase(kv_len, hkv, d, page, dtype, seed=kv_len)
        for n_q in {kv_len, 1, min(kv_len, 17)}:
            q = randn((n_q, hq, d), kv_len * 3 + n_q, dtype)
            got = _run(cuda, case, q, causal, dtype).float().cpu()
            want = _dense(q, case.k, case.v, causal)
            assert ((got - want).abs() <= ATOL[dtype] * want.abs().clamp(min=1.0)).all(), (kv_len, n_q)


def test_a_call_with_scratch_makes_two_allocations(cuda):
    """the result and the scratch"""
    from tidaldecode_amd import _kernels

    past, n_q, h, d = 8192, 1000, 32, 128
    case = PagedCase(past + n_q, 8, d, 16, torch.bfloat16, seed=3)
    q = randn((n_q, h, d), 4, torch.bfloat16)
    assert _planned_bytes(case, q, True) > 0
    q_d, pool, table = q.bfloat16().to(cuda), case.pool.to(cuda), case.page_table.int().to(cuda)
    made = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]
    before = made()
    _kernels.prefill_with_paged_kv_cache(q_d, pool, table, case.last_page_len, True, 0, False, 1.0, 1e4)
    assert made() - before == 2
