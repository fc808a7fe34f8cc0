"""One-pass top-k of rows that 512 threads take (csrc/topk_filter.cuh): lengths around 8192 and 10240, many rows, few
and many ties at the threshold, samples after which the whole row is listed.  Bit-exact against the stable rule."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _run(cuda, v, k, bound=None, route="one pass"):
    from tidaldecode_amd import _kernels

    out = torch.full((v.shape[0], k), -1, dtype=torch.int32, device=cuda)
    _kernels.topk_filtering(v.to(cuda), None, None, out, None, k, upper_bound=None if bound is None else bound.to(cuda))
    assert _kernels.last_topk_route() == route
    return out.cpu().long()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows,n,k", [(256, 8193, 1), (256, 8193, 1200), (128, 10239, 800), (256, 10240, 1500),
                                      (257, 10240, 1201), (257, 10241, 1500), (257, 8192, 2500), (300, 2049, 2049)])
def test_edges(cuda, dtype, rows, n, k):
    from oracle import tidal_oracle as orc

    v = torch.randn((3, n), generator=torch.Generator().manual_seed(n + k)).to(dtype)
    want = orc.stable_topk(v.float(), k)
    times = -(-rows // 3)
    for bound in (None, torch.logsumexp(v.float(), 1).repeat(times)[:rows]):
        got = _run(cuda, v.repeat(times, 1)[:rows], k, bound)
        assert torch.equal(got, want.repeat(times, 1)[:rows])


@pytest.mark.parametrize("rows,n,k,ties", [(2, 300, 40, 2), (2, 1000, 90, 64), (2, 1000, 90, 65), (300, 5000, 400, 64),
                                           (300, 5000, 400, 65), (300, 9000, 400, 3), (300, 9000, 900, 5000),
                                           (300, 9000, 900, 9000), (2, 40000, 500, 63)])
def test_some_of_the_ties(cuda, rows, n, k, ties):
    """`ties` equal scores at random places, of which the selection takes the first and all but the last."""
    from oracle import tidal_oracle as orc

    g = torch.Generator().manual_seed(n + ties)
    for above in {max(k - 1, 0), max(k - ties + 1, 0)}:
        above = min(above, n - ties)
        v = torch.linspace(-3.0, -2.0, n)
        v[:above] = torch.linspace(2.0, 3.0, above)
        v[above: above + ties] = 1.0
        v = v[torch.randperm(n, generator=g)][None]
        assert torch.equal(_run(cuda, v.repeat(rows, 1), k), orc.stable_topk(v, k).expand(rows, -1)), above


def test_a_row_of_which_everything_is_listed(cuda):
    """Long list, and fewer than k elements from the ties' threshold on: the sampled elements (four vectors of each
    group of threads) descend in steps of 2^13 units, the others lie together a little below the threshold's rank."""
    from oracle import tidal_oracle as orc

    n, k, rows = 10000, 1000, 300
    tid = torch.arange(512)
    vec = (tid >> 2) * ((n // 4) >> 2) // 128 * 4 + (tid & 3)
    at = (4 * vec[:, None] + torch.arange(4)).reshape(-1).unique()
    top = torch.tensor([8.0]).view(torch.int32)
    keys = torch.full((n,), 0, dtype=torch.int32)
    keys[:] = top - 284 * 2 ** 13
    keys[at] = top - torch.arange(len(at), dtype=torch.int32) * 2 ** 13
    v = keys.view(torch.float32)[None]
    want = orc.stable_topk(v, k)
    for bound in (None, torch.full((rows,), 8.0)):
        assert torch.equal(_run(cuda, v.repeat(rows, 1), k, bound), want.expand(rows, -1))
