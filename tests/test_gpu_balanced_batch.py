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


@pytest.fixture(params=["planned", "balanced"])
def launch(request, monkeypatch):
    """As the planner decides, and balanced also where it takes even chunks or short lists (up to 64 sequences)."""
    from tidaldecode_amd import _kernels
    from tidaldecode_amd.utils import batch_controller

    if request.param == "planned":
        return request.param
    wrapper = _kernels.BatchDecodeWithPagedKVCachePyTorchWrapper
    planned = wrapper._plan

    def plan_of(self, batch, rows, items, short_list=True):
        plan = planned(self, batch, rows, items, False)
        heads, kv, d = self._geom[:3]
        group = next(g for g in (2, 4, 8) if heads // kv <= g or g == 8)
        hrows = kv * -(-(heads // kv) // group)
        slots = -(-batch // max(1, 256 // hrows)) * max(1, 256 // hrows)
        need = max(plan.max_splits, -(-min(slots, 64 * batch) // batch))
        part = batch * hrows * group * need
        plan.balanced, plan.max_splits = 1, need
        plan.workspace_bytes = (1 << 20) + sum(-(-part * x // 256) * 256 for x in (d * 4, 8))
        return plan

    class Declines:
        def __getattr__(self, name):
            return lambda *a: False

    monkeypatch.setattr(wrapper, "_plan", plan_of)
    for module in (_kernels, batch_controller):
        monkeypatch.setattr(module, "host_calls", Declines())
    return request.param


@pytest.mark.parametrize("heads,kv,d,page,dtype", [(32, 8, 128, 16, torch.bfloat16), (28, 4, 128, 16, torch.float16),
                                                   (6, 2, 64, 1, torch.float16), (16, 4, 256, 7, torch.bfloat16),
                                                   (40, 2, 128, 32, torch.bfloat16)])
@pytest.mark.parametrize("kind,batch,hi", [("mixed", 2, 700), ("mixed", 16, 3000), ("one long", 9, 5000),
                                           ("equal", 5, 129), ("mixed", 64, 300), ("mixed", 65, 300)])
def test_batches(cuda, launch, heads, kv, d, page, dtype, kind, batch, hi):
    from tidaldecode_amd import _kernels
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
    assert launch == "planned" or _kernels.last_decode_kernel().startswith("streaming")
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
def test_fused_step_of_a_batch(cuda, launch, batch, hi):
    """With the new tokens folded into the launch: the same outputs, logits and cache as the separate calls."""
    from tidaldecode_amd import _kernels
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
        assert launch == "planned" or _kernels.last_decode_kernel().startswith("streaming")
        out.append((o.float(), c.qk_product.clone(), c.pool.buf.float()))
    (o0, l0, p0), (o1, l1, p1) = out
    # a rotated element may differ by one bf16 step between the kernels: 2^-8 of values up to 5
    assert (p0 - p1).abs().max() <= 2 ** -8 * 8 and (o0 - o1).abs().max() <= 1e-2
    fin = torch.isfinite(l0)
    assert torch.equal(fin, torch.isfinite(l1)) and (l0[fin] - l1[fin]).abs().max() <= 0.1


def _pieces(cuda, heads, kv, d, lens, page=16, chunk=0):
    """Attention of sequences of these lengths over lists of their pages; how many partial results a head has."""
    from tidaldecode_amd import _kernels

    batch, pages = len(lens), [-(-n // page) for n in lens]
    w = _kernels.BatchDecodeWithPagedKVCachePyTorchWrapper(0)
    w.chunk_tokens = chunk
    w.begin_forward(None, heads, kv, d, page, torch.empty(0, dtype=torch.bfloat16))
    g = torch.Generator(device=cuda).manual_seed(batch)
    pool = torch.randn((sum(pages), 2, page, kv, d), generator=g, device=cuda).bfloat16()
    first = [sum(pages[:b]) for b in range(batch)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=cuda)
    table = torch.arange(sum(pages), dtype=torch.int32, device=cuda)[None]
    q = torch.randn((batch, heads, d), generator=g, device=cuda).bfloat16()
    o = torch.empty_like(q)
    args = (q, o, pool, table, i32(first + [sum(pages)]), i32([(n - 1) % page + 1 for n in lens]),
            i32([f + n - 1 for f, n in zip(first, pages)]), None)
    w.forward(*args, n_list=max(pages) - 1, counts=i32([n - 1 for n in pages]))
    for b in range(batch):
        k, v = (pool[first[b]: first[b] + pages[b], i].reshape(-1, kv, d)[: lens[b]].float()
                .repeat_interleave(heads // kv, 1).transpose(0, 1) for i in (0, 1))
        want = torch.softmax((k @ q[b].float()[..., None])[..., 0] / math.sqrt(d), 1)[:, None] @ v
        assert (o[b].float() - want[:, 0]).abs().max() <= 1e-2, b
    plan = w._plan(batch, 1, (max(pages) - 1) * page + page, False)
    partials = (w._workspace.numel() - (1 << 20)) // (4 * (d + 2) * plan.max_splits * batch) * plan.max_splits * batch
    ml = (1 << 20) + (partials * d * 4 + 255) // 256 * 256
    return int((w._workspace[ml: ml + partials * 8].view(torch.float32).view(-1, 2)[:, 1] > 0).sum()), partials // (
        plan.max_splits * batch)


@pytest.mark.parametrize("heads,kv,d,lens", [(8, 1, 128, [8192] * 16), (8, 1, 128, [40000, 50]),
                                             (16, 2, 128, [20000, 36000, 1200, 36000]), (12, 2, 128, [4096] * 16),
                                             (6, 2, 64, [6000] * 3 + [1000] * 5)])
def test_few_head_rows_fill_the_chip(cuda, heads, kv, d, lens):
    """Head rows times pieces take at least three quarters of the compute units, as far as 64 pieces of a
    sequence (what a merge takes) and tiles of 128 tokens (256 of 64 dimensions) go."""
    done, head_slots = _pieces(cuda, heads, kv, d, lens)
    hrows = kv * -(-(heads // kv) // 8)
    tile = 8 * 4 * (64 // (d // 8))
    room = hrows * sum(min(64, -(-n // tile)) for n in lens)
    assert done % head_slots == 0
    assert done // head_slots * hrows >= 0.75 * min(256, room)


def test_preset_chunks_are_kept(cuda):
    """A chunk size set by the caller cuts every sequence, however long the others are."""
    done, head_slots = _pieces(cuda, 8, 2, 128, [16384, 4096, 700], chunk=256)
    assert done // head_slots == 64 + 16 + 3
