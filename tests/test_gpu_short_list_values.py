"""GPU: values that are no ordinary numbers, in the short-list kernel and beside it in the streaming kernel."""
import pytest
import torch

from _util import ATOL, PagedCase, randn, tolerance_report

pytestmark = pytest.mark.gpu
SHAPES = [(4, 4, 64), (4, 2, 64), (8, 2, 64), (14, 2, 64), (4, 4, 128), (4, 2, 128), (8, 2, 128), (14, 2, 128), (16, 2, 128)]


def _attend(cuda, case, q, pos=None, scores=None, lse=None, waves=0):
    """Attention of q [H, D] over the listed tokens, or over the whole sequence by its pages."""
    from tidaldecode_amd import _kernels

    hq, d = q.shape
    w = _kernels.BatchDecodeWithPagedKVCachePyTorchWrapper(case.layout)
    w.begin_forward(None, hq, case.hkv, d, case.page_size, torch.empty(0, dtype=case.dtype))
    w.sparse_waves = waves
    qd = q.to(case.dtype).to(cuda).unsqueeze(0)
    o = torch.full_like(qd, 7.0)
    if pos is not None:
        w.forward(qd, o, case.pool.to(cuda), case.slots_of(pos).to(torch.int32).to(cuda).contiguous(), None, 0, 0, None,
                  index_kind="slots", lse=lse)
    else:
        w.forward(qd, o, case.pool.to(cuda), case.page_table[:-1].to(torch.int32).unsqueeze(0).to(cuda), None,
                  case.last_page_len, int(case.page_table[-1]), scores, lse=lse)
    assert _kernels.last_decode_kernel() == ("streaming" if waves < 0 else "short-list")
    torch.cuda.synchronize()
    return o[0]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hq,hkv,d", SHAPES)
@pytest.mark.parametrize("n", [1, 40, 1300])
@pytest.mark.parametrize("pages", [False, True])
@pytest.mark.parametrize("waves", [0, -1])
def test_nan_keys_and_queries_show(cuda, dtype, hq, hkv, d, n, pages, waves):
    """A NaN key makes NaN of the outputs of its KV head's query heads and of no others, a NaN query of its own; the
    log-sum-exps, which bound the logits for the selection, are then no finite numbers."""
    from oracle import tidal_oracle as orc

    group = hq // hkv
    k, v, q = randn((n, hkv, d), n, dtype), randn((n, hkv, d), n + 1, dtype), randn((hq, d), n + 2, dtype)
    for at in {0, n // 2, n - 1}:
        for bad in ("key", "query"):
            kk, qq = k.clone(), q.clone()
            if bad == "key":
                kk[at, 0, d // 2] = float("nan")
                heads = torch.arange(hq) < group
            else:
                qq[at % hq, 1] = float("nan")
                heads = torch.arange(hq) == at % hq
            case = PagedCase(n, hkv, d, 16, dtype, seed=n, kv=(kk, v))
            scores = torch.full((hq, case.n_pages * 16), 7.0, device=cuda) if pages else None
            lse = torch.full((1, hq), 7.0, device=cuda)
            pos = None if pages else torch.randperm(n, generator=torch.Generator().manual_seed(n)).repeat(hkv, 1)
            o = _attend(cuda, case, qq, pos, scores, lse, waves).float().cpu()
            assert torch.isnan(o[heads]).all() and not torch.isfinite(lse[0].cpu()[heads]).any()
            want = orc.softmax_pv(orc.attn_logits(q, k), v)
            assert tolerance_report(o[~heads], want[~heads]) <= ATOL[dtype] if (~heads).any() else True
            assert torch.isfinite(lse[0].cpu()[~heads]).all()
            if pages:
                nans = torch.isnan(scores[:, :n].cpu())
                assert torch.equal(nans, torch.isnan(orc.attn_logits(qq, kk)))
