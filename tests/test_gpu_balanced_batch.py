"""GPU parity of the balanced full attention of a batch (decode_attn_balanced_kernel): workgroups dealt to the
sequences by their lengths.  Batches of very different lengths, single tokens, more sequences than a round
of workgroups holds, and beyond the 64 the kernel takes, against attention in fp32."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _lens(kind, batch, hi):
    g = torch.Generator().manual_seed(batch * 1000 + hi)
    if kind == "one long":
        return [1] * (batch - 1) + [hi]
    if kind == "equal":
        return [hi] * batch
    return torch.randint(1, hi + 1, (batch,), generator=g).tolist()


@pytest.mark.parametrize("heads,kv,d,page,dtype", [(32, 8, 128, 16, torch.bfloat16), (28, 4, 128, 16, torch.float16),
                                                   (6, 2, 64, 1, torch.float16), (16, 4, 256, 7, torch.bfloat16),
                                                   (40, 2, 128, 32, torch.bfloat16)])
@pytest.mark.parametrize("kind,batch,hi", [("mixed", 2, 700), ("mixed", 16, 3000), ("one long", 9, 5000),
                                           ("equal", 5, 129), ("mixed", 64, 300), ("mixed", 65, 300)])
def test_batches(cuda, heads, kv, d, page, dtype, kind, batch, hi):
    from tidaldecode_amd.utils import BatchInferenceController

    lens = _lens(kind, batch, hi)
    c = BatchInferenceController(1, heads, d, page, 8, hi + 1, batch, dtype, cuda, num_kv_heads=kv, page_order_seed=3)
    g = torch.Generator(device=cuda).manual_seed(hi)
    c.pool.buf.normal_(generator=g)
    c.add_sequences(lens)
    q = torch.randn((batch, heads, d), generator=g, device=cuda).to(dtype)
    pool = c.buf_layer(0)
    for step in range(2):  # the second on tickets and partials the first has used
        o = c.attend_full(q, 0, output_qk_product=True)
    rows = c.qk_product.view(batch, heads, -1)
    tol = 2e-3 if dtype == torch.float16 else 1e-2
    for b, n in enumerate(lens):
        table = c.page_table[b, : -(-n // page)].long()
        k = pool[table, 0].reshape(-1, kv, d)[:n].float().repeat_interleave(heads // kv, 1)
        v = pool[table, 1].reshape(-1, kv, d)[:n].float().repeat_interleave(heads // kv, 1)
        logits = (q[b].float()[None] * k).sum(-1).t() / math.sqrt(d)
        want = (torch.softmax(logits, 1)[..., None] * v.transpose(0, 1)).sum(1)
        assert (rows[b, :, :n] - logits).abs().max() <= 1e-4 * (1 + logits.abs().max()), b
        assert (rows[b, :, n:] == float("-inf")).all(), b
        assert (c.lse[b] - torch.logsumexp(logits, 1)).abs().max() <= 1e-4 * (1 + logits.abs().max()), b
        assert (o[b].float() - want).abs().max() <= tol, b


@pytest.mark.parametrize("batch,hi", [(3, 900), (16, 2000)])
def test_fused_step_of_a_batch(cuda, batch, hi):
    """With the new tokens folded into the launch: the same outputs, logits and cache as the separate calls."""
    from tidaldecode_amd.utils import BatchInferenceController

    heads, kv, d, page = 32, 8, 128, 16
    lens = _lens("mixed", batch, hi)
    out = []
    for fused in (False, True):
        c = BatchInferenceController(1, heads, d, page, 8, hi + 2, batch, torch.bfloat16, cuda, num_kv_heads=kv,
                                     page_order_seed=3)
        g = torch.Generator(device=cuda).manual_seed(hi)
        c.pool.buf.normal_(generator=g)
        c.add_sequences(lens)
        c.begin_step()
        q, k, v = (torch.randn((batch, h, d), generator=g, device=cuda).bfloat16() for h in (heads, kv, kv))
        if fused:
            o = c.attend_full(q, 0, output_qk_product=True, fresh=(k, v, *c.rope_table()))
        else:
            c.rope_append(q, k, v, 0)
            o = c.attend_full(q, 0, output_qk_product=True)
        out.append((o.float(), c.qk_product.clone(), c.pool.buf.float()))
    (o0, l0, p0), (o1, l1, p1) = out
    # a rotated element may differ by one bf16 step between the kernels: 2^-8 of values up to 5
    assert (p0 - p1).abs().max() <= 2 ** -8 * 8 and (o0 - o1).abs().max() <= 1e-2
    fin = torch.isfinite(l0)
    assert torch.equal(fin, torch.isfinite(l1)) and (l0[fin] - l1[fin]).abs().max() <= 0.1
