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


@pytest.mark.parametrize("waves,pages,dtype,hq,hkv,d", [
    (w, pages, dt, *shape) for shape in [(4, 4, 64), (4, 2, 64), (8, 2, 64), (14, 2, 64)] for w in (0, -1)
    for pages in (False, True) for dt in (torch.float16, torch.bfloat16)] + [
    (0, False, torch.float16, *shape) for shape in [(4, 4, 128), (4, 2, 128), (8, 2, 128), (16, 2, 128)]])
def test_infinite_values_stay_infinite(cuda, waves, pages, dtype, hq, hkv, d):
    """An infinite element of a value is infinite in the output of every head that reads it, not NaN, and nowhere else."""
    for n in (40, 300, 2100):
        k, v, q = randn((n, hkv, d), n, dtype), randn((n, hkv, d), n + 1, dtype), randn((hq, d), n + 2, dtype)
        v[5, 0, 3], v[n - 7, hkv - 1, 9] = float("inf"), float("-inf")
        case = PagedCase(n, hkv, d, 16, dtype, seed=n, kv=(k, v))
        o = _attend(cuda, case, q, None if pages else torch.arange(n).repeat(hkv, 1), waves=waves).float().cpu()
        want = torch.zeros_like(o)
        want[: hq // hkv, 3], want[hq - hq // hkv:, 9] = float("inf"), float("-inf")
        assert torch.equal(torch.where(torch.isfinite(o), torch.zeros_like(o), o), want), n


@pytest.mark.parametrize("hq,hkv", [(4, 2), (8, 2), (14, 2)])
@pytest.mark.parametrize("n,waves", [(4000, 0), (16000, -1)])
def test_a_flat_tail_counts(cuda, hq, hkv, n, waves):
    """One token of weight 1 and the rest of 2^-26 each, which fp16 does not hold: the sum of the rest is the output."""
    d, dtype = 64, torch.float16
    k, v, q = torch.zeros((n, hkv, d)), torch.ones((n, hkv, d)), torch.zeros((hq, d))
    v[0], q[:, 0] = 0.0, 8.0
    k[1:, :, 0] = torch.tensor(-18.02).to(dtype).float()
    case = PagedCase(n, hkv, d, 16, dtype, kv=(k, v))
    o = _attend(cuda, case, q, None if waves < 0 else torch.arange(n).repeat(hkv, 1), waves=waves).double().cpu()
    rest = (n - 1) * torch.exp(k[1, 0, 0].double())
    want = rest / (1 + rest)
    assert ((o - want).abs() <= 2.0 ** -11 * want + 2.0 ** -20 * want).all()  # the output's rounding, and the sums'


@pytest.mark.parametrize("hq,hkv", [(4, 2), (8, 2), (14, 2)])
@pytest.mark.parametrize("waves", [0, -1])
def test_weights_keep_their_bits(cuda, hq, hkv, waves):
    """Four tokens of one weight w against values that cancel 4 w to 2^-24 of it: what is left shows the weight's error.
    w is the one of bf16 logits that a bf16 value and its bf16 remainder hold worst (2^-17 of it)."""
    d, dtype = 64, torch.bfloat16
    x = torch.arange(1, 90).float() / 128  # exact in bf16
    w = torch.exp(-x.double())
    hi = w.bfloat16().double()
    lost = (w - hi - (w - hi).bfloat16().double()).abs() / w
    at = int(lost.argmax())
    assert lost[at] >= 2.0 ** -17.5
    w, values, left = w[at], [1.0] * 4, 4 * w[at]
    for _ in range(3):
        values.append(-float(left.bfloat16()))
        left = left + values[-1]
    n = len(values)
    k, v, q = torch.zeros((n, hkv, d)), torch.zeros((n, hkv, d)), torch.zeros((hq, d))
    q[:, 0] = 8.0
    k[:4, :, 0] = -x[at]
    v[:, :, :] = torch.tensor(values)[:, None, None]
    case = PagedCase(n, hkv, d, 16, dtype, kv=(k, v))
    o = _attend(cuda, case, q, torch.arange(n).repeat(hkv, 1) if waves == 0 else None, waves=waves).double().cpu()
    total = 4 * w + 3
    # the exponential and its argument, each within 2^-23, and the sums of 7 products of up to 4 in 32 bits
    bound = (4 * w * 2.0 ** -22 + n * 2.0 ** -24 * 4) / total
    assert bound < 0.5 * 4 * w * lost[at] / total
    assert ((o - left / total).abs() <= bound + 2.0 ** -8 * (left / total).abs()).all()
