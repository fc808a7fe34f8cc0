"""GPU: the one launch in front of a page-estimate attention (rope_append_estimate) against the calls it stands
for, at the edges of its tiles of entries, at the first and the last token of a page, with pages and metadata
pages of other sizes, groups of heads and every head size."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hq,hkv,d,page,layout", [(32, 32, 128, 16, 0), (8, 2, 64, 4, 1), (6, 2, 256, 5, 0),
                                                  (7, 1, 128, 1, 0)])
@pytest.mark.parametrize("n_pages", [1, 2, 33, 64, 65, 130, 641])
def test_equals_the_separate_calls(cuda, dtype, hq, hkv, d, page, layout, n_pages):
    from tidaldecode_amd import _kernels

    g = torch.Generator(device=cuda).manual_seed(n_pages + d)
    shape = (lambda p: (p, 2, page, hkv, d)) if layout == 0 else (lambda p: (p, 2, hkv, page, d))
    n_meta = -(-n_pages // page)
    table = torch.randperm(n_pages + 3, generator=g, device=cuda)[:n_pages].int()
    meta_table = torch.randperm(n_meta + 2, generator=g, device=cuda)[:n_meta].int()
    pool = torch.randn(shape(n_pages + 3), generator=g, device=cuda).to(dtype)
    meta = torch.randn(shape(n_meta + 2), generator=g, device=cuda).to(dtype)
    meta_last = (n_pages - 1) % page + 1
    q, k, v = (torch.randn((1, h, d), generator=g, device=cuda).to(dtype) for h in (hq, hkv, hkv))
    indptr = torch.tensor([0, n_pages], dtype=torch.int32, device=cuda)
    meta_indptr = torch.tensor([0, n_meta], dtype=torch.int32, device=cuda)
    ulp = 2.0 ** (-10 if dtype == torch.float16 else -7)
    for last in sorted({1, (page + 1) // 2, page}):
        pos = (n_pages - 1) * page + last - 1
        cos, sin = _kernels.rope_table(torch.tensor([pos], dtype=torch.int32, device=cuda), d, 1.0, 5e5)
        p1, m1, q1, k1 = pool.clone(), meta.clone(), q.clone(), k.clone()
        _kernels.apply_rope_in_place(q1, k1, pos, 1.0, 5e5)
        _kernels.append_kv_cache_decode(k1, v, p1, table, indptr, last, int(table[-1]), m1, meta_table, meta_indptr,
                                        meta_last, int(meta_table[-1]), layout)
        e1 = torch.zeros((hq, (n_meta - 1) * page + meta_last - 1), dtype=dtype, device=cuda)
        for estimate in (True, False):
            p2, m2 = pool.clone(), meta.clone()
            q2, e2 = _kernels.rope_append_estimate(q, k, v, p2, last, int(table[-1]), m2, meta_table, meta_last,
                                                   layout, cos, sin, estimate)
            # the angles' products are contracted as the compiler likes: one rounding of the element
            assert ((q2 - q1).float().abs() <= ulp * q1.float().abs() + 1e-6).all()
            for a, b in ((p2, p1), (m2, m1)):
                assert ((a - b).float().abs() <= ulp * b.float().abs() + 1e-6).all()
            changed = (p2 != pool).any(-1).sum()
            assert int(changed) <= 2 * hkv and int((m2 != meta).any(-1).sum()) <= 2 * hkv
            if not estimate:
                assert e2 is None
                continue
            assert e2.shape == e1.shape
            if e1.numel():
                # from the same rotated q: the same sums, rounded once
                _kernels.estimate_attn_score(q2, e1, m2, meta_table, None, meta_last, int(meta_table[-1]), layout)
                assert torch.equal(e2, e1)


def test_arguments_are_checked(cuda):
    from tidaldecode_amd import _kernels

    h, d, page = 2, 64, 4
    pool = torch.zeros((3, 2, page, h, d), dtype=torch.half, device=cuda)
    meta = torch.zeros((2, 2, page, h, d), dtype=torch.half, device=cuda)
    q = torch.zeros((1, h, d), dtype=torch.half, device=cuda)
    idx = torch.zeros(1, dtype=torch.int32, device=cuda)
    cs = torch.zeros((1, d // 2), device=cuda)
    with pytest.raises(RuntimeError, match="last page"):
        _kernels.rope_append_estimate(q, q, q, pool, page + 1, 0, meta, idx, 1, 0, cs, cs)
    with pytest.raises(RuntimeError, match="last page"):
        _kernels.rope_append_estimate(q, q, q, pool, 1, 3, meta, idx, 1, 0, cs, cs)
    with pytest.raises(RuntimeError, match="disagree"):
        _kernels.rope_append_estimate(q.bfloat16(), q, q, pool, 1, 0, meta, idx, 1, 0, cs, cs)
    with pytest.raises(RuntimeError, match="cos and sin"):
        _kernels.rope_append_estimate(q, q, q, pool, 1, 0, meta, idx, 1, 0, cs[:, :8].contiguous(), cs)
