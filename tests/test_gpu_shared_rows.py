"""GPU: query heads that share KV rows, scored on the matrix cores (rows of eight lanes at head_dim 64, eight
heads at head_dim 128): the fused step of a selection layer at lengths around a tile of a wave (16 or 32 tokens)
and of a workgroup (128 or 256), against the oracle's dense attention.  On the streaming kernel at every length, and on
the short-list kernel where the library prefers it (not for groups that are cut, as of 12 heads)."""
import pytest
import torch

from _util import ATOL, PagedCase, randn, rotated, tolerance_report

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hq,hkv,d", [(4, 2, 64), (8, 2, 64), (14, 2, 64), (16, 2, 64), (24, 2, 64), (14, 2, 128),
                                      (16, 2, 128)])
@pytest.mark.parametrize("n", [2, 17, 31, 33, 128, 257, 3100])
@pytest.mark.parametrize("waves", [0, -1])
def test_fused_selection_layer(cuda, dtype, hq, hkv, d, n, waves):
    from oracle import tidal_oracle as orc
    from tidaldecode_amd import _kernels

    page, theta = 16, 1e4
    case = PagedCase(n, hkv, d, page, dtype, seed=n + hq)
    q, knew, vnew = randn((1, hq, d), 1, dtype), randn((1, hkv, d), 2, dtype), randn((1, hkv, d), 3, dtype)
    kk, vv = case.k.clone(), case.v.clone()
    kk[n - 1], vv[n - 1] = rotated(knew, [n - 1], dtype, theta)[0], vnew[0]
    q_rot = rotated(q, [n - 1], dtype, theta)[0]
    logits = orc.attn_logits(q_rot, kk)
    want = orc.softmax_pv(logits, vv)
    dev = dict(dtype=torch.int32, device=cuda)
    cos, sin = _kernels.rope_table(torch.tensor([n - 1], **dev), d, 1.0, theta)
    fresh = (knew.to(dtype).to(cuda), vnew.to(dtype).to(cuda), cos, sin,
             torch.tensor([int(case.slots_of(torch.tensor([n - 1]))[0])], **dev))
    w = _kernels.BatchDecodeWithPagedKVCachePyTorchWrapper(0)
    w.begin_forward(None, hq, hkv, d, page, torch.empty(0, dtype=dtype))
    w.sparse_waves = waves
    qd = q.to(dtype).to(cuda)
    o = torch.full_like(qd, float("nan"))
    scores = torch.full((hq, case.n_pages * page), float("nan"), dtype=torch.float32, device=cuda)
    lse = torch.empty((1, hq), dtype=torch.float32, device=cuda)
    w.forward(qd, o, case.pool.to(cuda), case.page_table[:-1].to(torch.int32).unsqueeze(0).to(cuda), None,
              case.last_page_len, int(case.page_table[-1]), scores, lse=lse, fresh=fresh)
    torch.cuda.synchronize()
    assert _kernels.last_decode_kernel() == ("short-list" if waves == 0 and hq // hkv <= 8 else "streaming")
    assert tolerance_report(o[0], want) <= ATOL[dtype]
    # a rotated element on the other side of a rounding boundary than the float64 rotation: up to one storage
    # ulp of |q| |k| / sqrt(d), in the query for every token and in the key for the new one
    ulp = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}[dtype]
    bound = 2e-4 * max(1.0, logits.abs().max().item()) + 0.5 * ulp
    assert (scores[:, :n].cpu() - logits).abs().max() <= bound
    assert torch.isnan(scores[:, n:]).all()
    assert (lse[0].cpu() - torch.logsumexp(logits, -1)).abs().max() <= 1e-3 + 0.5 * ulp
