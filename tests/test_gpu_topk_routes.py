"""GPU parity of the top-k routes that large selections take, bit-exact against the oracle's stable rule: every
register size of the kernel whose workgroups go through the whole row, and payloads, page tables, lengths and list
segments on each of the three routes.  Every call says which route it took."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _run(cuda, v, k, route, *, scratch=False, segment=None, vals=False, **kw):
    from tidaldecode_amd import _kernels

    rows = v.shape[0]
    kw = {n: t.to(cuda) if torch.is_tensor(t) else t for n, t in kw.items()}
    if segment is None:
        out = torch.full((rows, k), -1, dtype=torch.int32, device=cuda)
    else:
        groups = kw["lengths"].numel()
        out = torch.full((rows // groups, groups * segment + 3), -1, dtype=torch.int32, device=cuda)
    out_v = torch.zeros((rows, k), dtype=v.dtype, device=cuda) if vals else None
    buf = torch.zeros(_kernels.topk_workspace_bytes(rows), dtype=torch.uint8, device=cuda) if scratch else None
    in_idx = kw.pop("in_idx", None)
    _kernels.topk_filtering(v.to(cuda), in_idx, out_v, out, buf, k, segment=segment, **kw)
    assert _kernels.last_topk_route() == route
    torch.cuda.synchronize()
    return out.cpu().long(), None if out_v is None else out_v.cpu()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n", [3001, 4096, 8192, 8200, 16000, 24000, 24576, 32768, 40960, 48000, 56000, 57344, 65536, 65537, 100003])
def test_every_register_size_of_the_slices(cuda, dtype, n):
    """8 to 64 elements a thread, and rows that are read again in every pass."""
    from oracle import tidal_oracle as orc

    g = torch.Generator().manual_seed(n)
    v = torch.randn((3, n), generator=g).to(dtype)
    v[2] = torch.randint(0, 7, (n,), generator=g).to(dtype)
    lse = torch.logsumexp(v.float(), 1)
    for k in (max(n // 2, min(6700, n - 2)), n - 1):
        want = orc.stable_topk(v.float(), k)
        for bound in (None, lse):
            got, vals = _run(cuda, v, k, "slices", vals=True, upper_bound=bound)
            assert torch.equal(got, want) and torch.equal(vals, torch.gather(v, 1, want)), k


@pytest.mark.parametrize("route,n,k,page,scratch", [("one pass", 20000, 2000, 16, False), ("one pass", 100000, 3000, 5, True),
                                                    ("slices", 30000, 9000, 16, False), ("slices", 70001, 20000, 7, False),
                                                    ("shared rows", 80000, 20000, 16, True),
                                                    ("shared rows", 131077, 5000, 3, True)])
def test_payloads_tables_lengths_and_segments(cuda, route, n, k, page, scratch):
    from oracle import tidal_oracle as orc

    g = torch.Generator().manual_seed(n)
    groups, per = 3, 2
    v = torch.randn((groups * per, n), generator=g)
    want = orc.stable_topk(v, k)
    payload = torch.randint(0, 1 << 30, v.shape, generator=g, dtype=torch.int32)
    got, _ = _run(cuda, v, k, route, scratch=scratch, in_idx=payload)
    assert torch.equal(got, torch.gather(payload.long(), 1, want))
    n_pages = -(-n // page)
    tables = torch.stack([torch.randperm(n_pages + 5, generator=g)[:n_pages] for _ in range(groups)]).int()
    lens = [n, max(1, n // 2), max(1, k // 2)]
    for gi, ln in enumerate(lens):                  # what lies behind a length is larger than everything
        v[gi * per: (gi + 1) * per, ln:] = 1e9
    kw = dict(page_table=tables, page_size=page, lengths=torch.tensor(lens, dtype=torch.int32))
    plain, _ = _run(cuda, v, k, route, scratch=scratch, **kw)
    segment = k + 5
    apart, _ = _run(cuda, v, k, route, scratch=scratch, segment=segment, **kw)
    for r in range(groups * per):
        gi, ln = r // per, lens[r // per]
        pos = orc.stable_topk(v[r: r + 1, :ln], min(k, ln))[0]
        slots = tables[gi].long()[pos // page] * page + pos % page
        row = apart[r % per, gi * segment: (gi + 1) * segment]
        for got in (plain[r], row):
            assert torch.equal(got[: len(slots)], slots) and (got[len(slots):] == -1).all(), r
    assert (apart[:, groups * segment:] == -1).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,n,most32,most16", [(3, 2048, 2048, 2048), (3, 2049, 1300, 600), (256, 8192, 1300, 600),
                                                  (64, 8193, 1600, 0), (64, 32768, 3640, 1365), (65, 16384, 3276, 1024),
                                                  (256, 16384, 4096, 3036), (2, 65536, 4748, 4096), (2, 65537, 4748, 4748)])
def test_where_the_one_pass_ends(cuda, dtype, rows, n, most32, most16):
    """The largest selection that one workgroup a row takes, and the next, which goes to the slices."""
    from oracle import tidal_oracle as orc

    g = torch.Generator().manual_seed(n + rows)
    v = torch.randn((1, n), generator=g).to(dtype)
    most = most32 if dtype == torch.float32 else most16
    for k, route in ((most, "one pass"), (most + 1, "slices")):
        if 1 <= k <= n:
            got, _ = _run(cuda, v.repeat(rows, 1), k, route)
            assert torch.equal(got, orc.stable_topk(v.float(), k).expand(rows, -1)), k
