"""GPU: the short-list kernel at head_dim 64, with groups that leave head slots empty or are no power of two, on page
lists and with logits out: lengths around a wave's tile (32 or 64 tokens), a workgroup's and a split's, against the
oracle's attention over the listed tokens."""
import pytest
import torch

from _util import ATOL, PagedCase, randn, rotated, tolerance_report

pytestmark = pytest.mark.gpu
SHAPES = [(4, 4, 64), (14, 2, 64), (8, 2, 64), (4, 2, 64), (14, 2, 128), (6, 2, 128), (4, 4, 128)]


# waves of a workgroup, tokens of a split and whether it merges in the launch: as planned, and such that every wave of
# a long list takes several tiles (rows of eight lanes: of 64 tokens, else of 32)
PLANNED = (0, 0, -1)
TILES = [(4, 1024, 0), (4, 2048, 1), (8, 1024, 1), (8, 2048, 0)]


def _wrapper(hq, hkv, d, page, dtype, layout=0, shape=PLANNED):
    from tidaldecode_amd import _kernels

    w = _kernels.BatchDecodeWithPagedKVCachePyTorchWrapper(layout)
    w.begin_forward(None, hq, hkv, d, page, torch.empty(0, dtype=dtype))
    w.sparse_waves, w.chunk_tokens, w.fused_merge = shape
    assert shape == PLANNED or w.chunk_tokens >= 2 * w.sparse_waves * 4096 // d
    return w


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hq,hkv,d", SHAPES)
@pytest.mark.parametrize("per_query_head", [False, True])
@pytest.mark.parametrize("layout,shape", [(0, PLANNED), (1, PLANNED)] + [(0, x) for x in TILES])
def test_slot_lists_with_the_new_token(cuda, dtype, hq, hkv, d, per_query_head, layout, shape):
    from oracle import tidal_oracle as orc
    from tidaldecode_amd import _kernels

    page, n, theta = 16, 2700, 1e4
    rows = hq if per_query_head else hkv
    case = PagedCase(n, hkv, d, page, dtype, layout=layout, seed=hq + d)
    q, knew, vnew = randn((1, hq, d), 1, dtype), randn((1, hkv, d), 2, dtype), randn((1, hkv, d), 3, dtype)
    kk, vv = case.k.clone(), case.v.clone()
    kk[n - 1], vv[n - 1] = rotated(knew, [n - 1], dtype, theta)[0], vnew[0]
    q_rot = rotated(q, [n - 1], dtype, theta)[0]
    dev = dict(dtype=torch.int32, device=cuda)
    cos, sin = _kernels.rope_table(torch.tensor([n - 1], **dev), d, 1.0, theta)
    slot = int(case.slots_of(torch.tensor([n - 1]))[0])
    fresh = (knew.to(dtype).to(cuda), vnew.to(dtype).to(cuda), cos, sin, torch.tensor([slot], **dev))
    w = _wrapper(hq, hkv, d, page, dtype, layout, shape)
    qd = q.to(dtype).to(cuda)
    g = torch.Generator().manual_seed(hq)
    for k in (1, 31, 33, 64, 65, 129, 256, 257, 513, 1300, 2600) if shape == PLANNED else (1, 257, 513, 1300, 2600):
        pos = torch.stack([torch.randperm(n - 1, generator=g)[: k - 1] for _ in range(rows)])
        pos = torch.cat([pos, torch.full((rows, 1), n - 1)], 1)[:, torch.randperm(k, generator=g)]
        pool, o = case.pool.to(cuda), torch.full_like(qd, float("nan"))
        lse = torch.full((1, hq), float("nan"), dtype=torch.float32, device=cuda)
        for _ in range(2):  # twice: tickets and partials are reused
            w.forward(qd, o, pool, case.slots_of(pos).to(torch.int32).to(cuda).contiguous(), None, 0, 0, None,
                      index_kind="slots", lse=lse, fresh=fresh)
        assert _kernels.last_decode_kernel() == "short-list"
        torch.cuda.synchronize()
        assert tolerance_report(o[0], orc.sparse_layer_gather(q_rot, kk, vv, pos)) <= ATOL[dtype], k
        logits = torch.gather(orc.attn_logits(q_rot, kk), 1, pos[torch.arange(hq) * rows // hq])
        # (an element rotated to the other side of a rounding boundary than in float64 moves a logit by up to
        # half a storage ulp of |q| |k| / sqrt(d))
        ulp = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}[dtype]
        assert (lse[0].cpu() - torch.logsumexp(logits, -1)).abs().max() <= 1e-3 + 0.5 * ulp, k


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hq,hkv,d", SHAPES)
@pytest.mark.parametrize("page,shape", [(1, PLANNED), (16, PLANNED), (32, PLANNED)] + [(16, x) for x in TILES])
def test_pages_of_the_whole_sequence_with_logits(cuda, dtype, hq, hkv, d, page, shape):
    from oracle import tidal_oracle as orc
    from tidaldecode_amd import _kernels

    for n in (1, 33, 257, 1000, 4099):
        case = PagedCase(n, hkv, d, page, dtype, seed=n)
        q = randn((hq, d), n + 1, dtype)
        logits = orc.attn_logits(q, case.k)
        w = _wrapper(hq, hkv, d, page, dtype, shape=shape)
        qd = q.to(dtype).to(cuda).unsqueeze(0)
        for scores_dtype in (torch.float32, dtype):
            o = torch.full_like(qd, float("nan"))
            scores = torch.full((hq, case.n_pages * page), float("nan"), dtype=scores_dtype, device=cuda)
            lse = torch.empty((1, hq), dtype=torch.float32, device=cuda)
            w.forward(qd, o, case.pool.to(cuda), case.page_table[:-1].to(torch.int32).unsqueeze(0).to(cuda), None,
                      case.last_page_len, int(case.page_table[-1]), scores, lse=lse)
            assert _kernels.last_decode_kernel() == "short-list"
            torch.cuda.synchronize()
            assert tolerance_report(o[0], orc.softmax_pv(logits, case.v)) <= ATOL[dtype], n
            ulp = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[scores_dtype]
            bound = (2e-4 + ulp) * max(1.0, logits.abs().max().item())  # and the rounding of the stored logit
            assert (scores[:, :n].float().cpu() - logits).abs().max() <= bound, n
            assert torch.isnan(scores[:, n:]).all()
            assert (lse[0].cpu() - torch.logsumexp(logits, -1)).abs().max() <= 1e-3, n


@pytest.mark.parametrize("hq,hkv,d", [(4, 4, 128), (14, 2, 64)])
@pytest.mark.parametrize("shape", [PLANNED, (4, 512, 0), (4, 512, 1)])
def test_page_lists_of_a_ragged_batch(cuda, hq, hkv, d, shape):
    """Lists of pages per query head, the forced last page, counts on the device."""
    from oracle import tidal_oracle as orc
    from tidaldecode_amd import _kernels

    dtype, page = torch.bfloat16, 16
    cases = [PagedCase(n, hkv, d, page, dtype, seed=i) for i, n in enumerate((700, 40, 17))]
    base = [0]
    for c in cases[:-1]:
        base.append(base[-1] + c.max_pages)
    pool = torch.cat([c.pool for c in cases]).to(cuda)
    width, g = 24, torch.Generator().manual_seed(1)
    idx = torch.full((hq, width * len(cases)), 1 << 30)  # padding that must not be read as a page
    counts, chosen = [], []
    for i, c in enumerate(cases):
        m = min(width - 2, c.n_pages - 1)
        rows = torch.stack([torch.randperm(c.n_pages - 1, generator=g)[:m] for _ in range(hq)])
        idx[:, i * width: i * width + m] = c.page_table[rows] + base[i]
        counts.append(m)
        tail = torch.arange((c.n_pages - 1) * page, c.n).repeat(hq, 1)
        chosen.append(torch.cat([(rows[:, :, None] * page + torch.arange(page)).view(hq, -1), tail], 1))
    dev = dict(dtype=torch.int32, device=cuda)
    q = randn((len(cases), hq, d), 9, dtype)
    qd = q.to(dtype).to(cuda)
    o = torch.full_like(qd, float("nan"))
    w = _wrapper(hq, hkv, d, page, dtype, shape=shape)
    w.forward(qd, o, pool, idx.to(torch.int32).to(cuda), torch.tensor([i * width for i in range(len(cases) + 1)], **dev),
              torch.tensor([c.last_page_len for c in cases], **dev),
              torch.tensor([int(c.page_table[-1]) + b for c, b in zip(cases, base)], **dev), None,
              n_list=width, counts=torch.tensor(counts, **dev))
    assert _kernels.last_decode_kernel() == "short-list"
    torch.cuda.synchronize()
    for i, c in enumerate(cases):
        assert tolerance_report(o[i], orc.sparse_layer_gather(q[i], c.k, c.v, chosen[i])) <= ATOL[dtype], i


@pytest.mark.parametrize("batch,kernel", [(1024, "short-list"), (1025, "streaming")])
def test_batches_of_more_head_slots_than_tickets(cuda, batch, kernel):
    from tidaldecode_amd import _kernels

    hq, hkv, d, page, n, k = 14, 2, 64, 16, 3000, 130   # eight head slots a KV head
    dtype, g = torch.bfloat16, torch.Generator().manual_seed(batch)
    case = PagedCase(n, hkv, d, page, dtype, seed=4)
    pos = torch.randint(0, n, (hkv, batch * k), generator=g)
    q = randn((batch, hq, d), 9, dtype)
    qd = q.to(dtype).to(cuda)
    o = torch.full_like(qd, float("nan"))
    w = _wrapper(hq, hkv, d, page, dtype)
    starts = (torch.arange(batch + 1) * k).to(torch.int32).to(cuda)
    for _ in range(2):  # twice: tickets and partials are reused
        w.forward(qd, o, case.pool.to(cuda), case.slots_of(pos).to(torch.int32).to(cuda), starts, 0, 0, None,
                  index_kind="slots", n_list=k)
    assert _kernels.last_decode_kernel() == kernel
    for h in range(hkv):
        at = pos[h].view(batch, k)
        kk, vv, qh = case.k[at, h], case.v[at, h], q[:, h * 7:(h + 1) * 7]
        want = torch.softmax(qh @ kk.transpose(1, 2) / d ** 0.5, -1) @ vv
        assert tolerance_report(o[:, h * 7:(h + 1) * 7], want) <= ATOL[dtype]


@pytest.mark.parametrize("n,kernel", [(4608, "short-list"), (4624, "streaming")])  # either side of 72 MiB
def test_the_library_goes_by_what_a_call_reads(cuda, n, kernel):
    """Pages of a whole sequence with a plan made without the wrapper's knowledge of the call."""
    from tidaldecode_amd import _kernels, _lib

    h, d, page, dtype = 32, 128, 16, torch.float16
    g = torch.Generator(device=cuda).manual_seed(n)
    pool = torch.randn((n // page, 2, page, h, d), generator=g, device=cuda).to(dtype)
    q = torch.randn((1, h, d), generator=g, device=cuda).to(dtype)
    o = torch.full_like(q, float("nan"))
    table = torch.arange(n // page - 1, dtype=torch.int32, device=cuda)
    kv = _lib.PagedKV(pool.data_ptr(), n // page, h, d, page, _lib.TD_NHD, _lib.TD_F16)
    lst = _lib.IndexList()
    lst.idx, lst.idx_rows, lst.idx_row_stride, lst.kind = table.data_ptr(), 1, table.numel(), _lib.TD_IDX_PAGES
    lst.n_list_host, lst.last_page_len, lst.last_page_idx = table.numel(), page, n // page - 1
    plan = _lib.DecodePlan(0, 0, 0, 0, -1, 0, 0, 0)
    _lib.check(_lib.lib.td_decode_make_plan(1, h, h, d, 1, n, plan))
    assert plan.sparse_waves > 0
    ws = torch.zeros(plan.workspace_bytes, dtype=torch.uint8, device=cuda)
    _lib.check(_lib.lib.td_decode_attn(kv, lst, plan, q.data_ptr(), o.data_ptr(), 1, h, d ** -0.5, None, _lib.TD_F32, 0,
                                       None, None, ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream))
    assert _kernels.last_decode_kernel() == kernel
    k, v = (pool[:, i].reshape(n, h, d).float().transpose(0, 1).contiguous() for i in (0, 1))
    want = torch.softmax((k * q[0].float()[:, None]).sum(-1) / d ** 0.5, -1)[:, None] @ v
    assert tolerance_report(o[0], want[:, 0]) <= ATOL[dtype]
