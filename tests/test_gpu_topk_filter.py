"""GPU parity of the one-pass top-k (csrc/topk_filter.cuh): rows of up to 262144 scores whose
selection fits its list.  Everything is bit-exact against the oracle's stable rule.  Every call here takes that
route; rows of some lengths do so where there are many of them, so calls are made of their rows repeated."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _run(cuda, v, k, *, bound=None, in_idx=None, table=None, page=1, lengths=None, vals=True, pad=0, skew=0):
    """v on the host; `pad` extra columns between rows and `skew` elements in front of the first row move
    the rows' addresses."""
    from tidaldecode_amd import _kernels

    given, n = v.shape
    if n > 2048 and n <= 65536 and lengths is None:
        times = -(-256 // given)
        v, bound, in_idx = (None if t is None else t.repeat(times, *([1] * (t.dim() - 1))) for t in (v, bound, in_idx))
    rows = v.shape[0]
    flat = torch.full((skew + rows * (n + pad) + 1,), float("nan"), dtype=v.dtype, device=cuda)
    dev = flat[skew: skew + rows * (n + pad)].view(rows, n + pad)[:, :n]
    dev.copy_(v)
    out = torch.full((rows, k), -1, dtype=torch.int32, device=cuda)
    out_v = torch.zeros((rows, k), dtype=v.dtype, device=cuda) if vals else None
    to = lambda t: None if t is None else t.to(cuda)
    _kernels.topk_filtering(dev, to(in_idx), out_v, out, None, k, page_table=to(table), page_size=page,
                            lengths=to(lengths), upper_bound=to(bound))
    assert _kernels.last_topk_route() == "one pass"
    torch.cuda.synchronize()
    out, out_v = out.cpu().long(), None if out_v is None else out_v.cpu()
    for first in range(given, rows, given):     # copies of the rows
        more = min(given, rows - first)
        assert torch.equal(out[first: first + more], out[:more])
    return out[:given], None if out_v is None else out_v[:given]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,k", [(1, 1), (3, 2), (255, 17), (1019, 300), (1020, 1020), (1021, 1), (2047, 2000),
                                 (2049, 511), (4099, 64), (8191, 599), (8192, 600), (8193, 900), (16383, 5),
                                 (16383, 3000), (32771, 2048), (65535, 1024), (65537, 4096), (131073, 3), (200000, 3000),
                                 (262143, 2048), (262144, 2600)])
def test_edges_of_the_sizes(cuda, dtype, n, k):
    from oracle import tidal_oracle as orc

    g = torch.Generator().manual_seed(n * 7 + k)
    v = torch.randn((3, n), generator=g).to(dtype)
    want = orc.stable_topk(v.float(), k)
    lse = torch.logsumexp(v.float(), 1)
    for bound, pad, skew in ((None, 0, 0), (lse, 1, 0), (lse, 2, 1), (None, 3, 3)):
        got, vals = _run(cuda, v, k, bound=bound, pad=pad, skew=skew)
        assert torch.equal(got, want), (pad, skew)
        assert torch.equal(vals, torch.gather(v, 1, want))


@pytest.mark.parametrize("n,k,page", [(700, 90, 16), (700, 90, 7), (5001, 600, 1), (5001, 600, 48), (40003, 2000, 5),
                                      (70001, 1500, 16)])
def test_payloads_and_lengths(cuda, n, k, page):
    from oracle import tidal_oracle as orc

    g = torch.Generator().manual_seed(n + page)
    groups, per = 3, 2
    v = torch.randn((groups * per, n), generator=g)
    lens = [n, max(1, n // 3), max(1, k // 2)]
    n_pages = -(-n // page)
    tables = torch.stack([torch.randperm(n_pages + 5, generator=g)[:n_pages] for _ in range(groups)]).int()
    got, _ = _run(cuda, v, k, table=tables, page=page, lengths=torch.tensor(lens, dtype=torch.int32), vals=False)
    for r in range(groups * per):
        ln = lens[r // per]
        pos = orc.stable_topk(v[r: r + 1, :ln], min(k, ln))[0]
        want = tables[r // per].long()[pos // page] * page + pos % page
        assert torch.equal(got[r, : len(want)], want) and (got[r, len(want):] == -1).all(), r
    payload = torch.randint(0, 1 << 30, v.shape, generator=g, dtype=torch.int32)
    got, _ = _run(cuda, v, k, in_idx=payload)
    assert torch.equal(got, torch.gather(payload.long(), 1, orc.stable_topk(v, k)))


@pytest.mark.parametrize("n,k", [(20000, 2048), (6000, 700), (100001, 4000), (262144, 2500)])
def test_samples_that_mislead(cuda, n, k):
    """The sampled elements all larger than the rest (the first threshold keeps too few), all smaller
    (it keeps everything: more than the list holds), and rows of a few values only."""
    from oracle import tidal_oracle as orc

    g = torch.Generator().manual_seed(n)
    threads = 512 if n <= 8192 else 1024
    quads, lines = threads // 4, (-(-n // 4)) >> 2
    at = (torch.arange(quads) * lines // quads)[:, None] * 16 + torch.arange(16)[None]
    at = at.flatten()
    high, low = torch.randn((2, n), generator=g), torch.randn((2, n), generator=g)
    high[:, at] += 50.0
    low[:, at] -= 50.0
    few = torch.randint(0, 3, (2, n), generator=g).float()
    one = torch.full((1, n), -2.5)
    nan = torch.randn((2, n), generator=g)
    nan[:, at[::3]] = float("nan")
    nan[1, ::5] = float("inf")
    for v in (high, low, few, one, nan):
        got, _ = _run(cuda, v, k, vals=False)
        assert torch.equal(got, orc.stable_topk(v, k))


@pytest.mark.parametrize("n", [8192, 20000, 65536, 131072])
def test_scores_just_above_the_samples_maximum(cuda, n):
    """Scores that the sample misses, a few units in the last place above the largest it has, share that one's
    bin; the selection ends between them (no bound: the sample's maximum is the reference).  The others lie so
    close together that the sample's threshold takes two levels: the survivors' window does not end with a bin."""
    from oracle import tidal_oracle as orc

    threads = 512 if n <= 8192 else 1024
    quads, lines = threads // 4, (-(-n // 4)) >> 2
    sampled = ((torch.arange(quads) * lines // quads)[:, None] * 16 + torch.arange(16)[None]).flatten()
    g = torch.Generator().manual_seed(n)
    v = 3.0 + torch.randn((8, n), generator=g) * 2e-3
    free = torch.ones(n, dtype=torch.bool)
    free[sampled] = False
    missed = torch.arange(n)[free]
    for r in range(8):
        v[r, sampled[-3]] = 4.0
        at = missed[torch.randperm(len(missed), generator=g)[: 3 + r]]
        v[r, at] = 4.0 + (1 + torch.arange(3 + r)) * 2.0 ** -21  # the spacing of floats from 4 to 8
    for k in range(2, 13):
        got, vals = _run(cuda, v, k)
        want = orc.stable_topk(v, k)
        assert torch.equal(got, want) and torch.equal(vals, torch.gather(v, 1, want)), k


def _crowded_rows(n, k, dtype, g):
    """rows whose threshold lies in or next to many equal scores"""
    pick = lambda share: torch.rand(n, generator=g) < share
    mostly = lambda share, rest: torch.where(pick(share), 1.0 + torch.rand(n, generator=g), torch.tensor(rest))
    inf = float("inf")
    return torch.stack([
        torch.full((n,), -3.5), torch.randint(0, 2, (n,), generator=g).float(), mostly(0.4 * k / n, 0.0),
        mostly(1.08 * k / n, 0.0), mostly(0.4 * k / n, -inf), torch.full((n,), inf), torch.full((n,), float("nan")),
        torch.where(pick(0.5), torch.tensor(0.0), torch.tensor(-0.0)), torch.where(pick(0.3 * k / n), inf, 2.0),
        mostly(0.5 * k / n, 0.0) - mostly(0.3 * k / n, 0.0), torch.randint(-9, 9, (n,), generator=g).float(),
    ]).to(dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("n,k", [(5000, 590), (8195, 3), (9001, 1100), (20000, 3900), (65536, 1024), (65537, 4000),
                                 (262144, 2500)])
def test_rows_of_few_values(cuda, dtype, n, k):
    """More equal scores than the list holds: those above are listed, of the equal ones the first by position
    are taken; a second crowd above or below the threshold's."""
    from oracle import tidal_oracle as orc

    g = torch.Generator().manual_seed(n + k)
    v = _crowded_rows(n, k, dtype, g)
    want = orc.stable_topk(v.float(), k)
    payload = torch.randint(0, 1 << 30, v.shape, generator=g, dtype=torch.int32)
    table = torch.randperm(-(-n // 48) + 3, generator=g).int()
    for pad, skew in ((0, 0), (1, 1)):
        got, vals = _run(cuda, v, k, pad=pad, skew=skew)
        assert torch.equal(got, want), [r for r in range(len(v)) if not torch.equal(got[r], want[r])]
        assert torch.equal(vals.nan_to_num(77.0), torch.gather(v, 1, want).nan_to_num(77.0))
        got, _ = _run(cuda, v, k, in_idx=payload, pad=pad, skew=skew)
        assert torch.equal(got, torch.gather(payload.long(), 1, want))
        got, _ = _run(cuda, v, k, table=table, page=48, vals=False, pad=pad, skew=skew)
        assert torch.equal(got, table.long()[want // 48] * 48 + want % 48)


@pytest.mark.parametrize("n,k", [(4096, 256), (32768, 2048), (102392, 4096)])
def test_rows_of_equal_scores_take_about_as_long_as_others(cuda, n, k):
    """at most eight times as long (a selection by one workgroup that queues up at one address took 4 to 34 times)"""
    from tidaldecode_amd import _kernels

    out = torch.zeros((32, k), dtype=torch.int32, device=cuda)
    took = {}
    for kind, v in (("normal", torch.randn((32, n), device=cuda)), ("equal", torch.zeros((32, n), device=cuda))):
        for _ in range(2):
            _kernels.topk_filtering(v, None, None, out, None, k)
        start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        start.record()
        for _ in range(50):
            _kernels.topk_filtering(v, None, None, out, None, k)
        end.record()
        torch.cuda.synchronize()
        took[kind] = start.elapsed_time(end)
    assert took["equal"] <= 8 * took["normal"], took
