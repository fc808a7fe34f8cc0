"""The native half of the entry points (csrc/host_calls.cpp): whatever it does not take as regular goes on in
Python with the same result or the same error, and what it takes gives the bits that Python gives."""
import ctypes

import numpy as np
import pytest
import torch

from tidaldecode_amd import _kernels, _lib
from tidaldecode_amd._lib import host_calls

_NATIVE = ("forward", "attend", "topk", "rope_table", "rope_in_place", "append", "prefill", "gemv", "score_reduce",
           "estimate")


class _Off:
    """host_calls with every function declining"""

    def __getattr__(self, name):
        assert name in _NATIVE
        return lambda *a: False


def test_wrong_argument_counts_are_type_errors():
    for name in _NATIVE:
        with pytest.raises(TypeError):
            getattr(host_calls, name)(1, 2)


def test_host_tensors_are_refused_as_before():
    q = torch.zeros(1, 4, 64)
    with pytest.raises(RuntimeError, match="q must be a CUDA tensor"):
        _kernels.apply_rope_in_place(q, q, 0, 1.0, 1e4)
    with pytest.raises(RuntimeError, match="must be a CUDA tensor"):
        _kernels.topk_filtering(torch.zeros(2, 8), None, None, torch.zeros(2, 4, dtype=torch.int32), None, 4)
    with pytest.raises(RuntimeError, match="must be a CUDA tensor"):
        _kernels.gemv(torch.zeros(4, 8), torch.zeros(8))
    assert host_calls.topk(q, None, None, q, None, 4, None, 1, None, None, None, 0, None) is False
    assert host_calls.gemv(object(), None, None, 1e-5, False, None, False, None, 0) is False


class _Recorder:
    """host_calls, with what was called and did not decline"""

    def __init__(self):
        self.served = []

    def __getattr__(self, name):
        def call(*a):
            made = getattr(host_calls, name)(*a)
            if made is not False:
                self.served.append((name, a))
            return made
        return call


def _workload(cuda, dtype, heads, kv, d, page, layout, mode):
    """A prompt and two decode steps through the public entry points; every tensor they make."""
    from tidaldecode_amd import utils as ops
    from tidaldecode_amd.utils import InferenceController

    g = torch.Generator(device=cuda).manual_seed(7)
    randn = lambda *s: torch.randn(s, generator=g, device=cuda).to(dtype)
    c = InferenceController(2, heads, d, page, 40, 400, dtype, cuda, num_kv_heads=kv, select_mode=mode,
                            kv_layout=layout, page_order_seed=5, with_metadata=True)
    c.kv_cache.pool.buf.zero_()
    c.metadata_cache.pool.buf.zero_()
    out = []
    q, k, v = randn(300, heads, d), randn(300, kv, d), randn(300, kv, d)
    c.prepare_metadata(300)
    c.begin_forward(300)
    ops.apply_rope_in_place(q, k, 0)
    for layer in range(2):
        ops.append_kv(k, v, c, layer)
        out.append(ops.prefill_forward(q, c, layer))
    for step in range(2):
        c.prepare_metadata(1)
        c.begin_forward(1)
        q, k, v = randn(1, heads, d), randn(1, kv, d), randn(1, kv, d)
        pos = torch.tensor([300 + step], dtype=torch.int32, device=cuda)
        out += list(_kernels.rope_table(pos, d, 1.0, 5e5))
        ops.apply_rope_in_place(q, k, 300 + step)
        for layer in range(2):
            ops.append_kv(k, v, c, layer)
            if layer == 0:
                out.append(ops.decode_sparse_attn(q, c, layer, c.kv_indices_without_last, True))
                ops.decode_topk(c)
                out.append(ops.decode_estimate(q, c, layer))
            else:
                out.append(ops.decode_sparse_attn(q, c, layer, c.topk_dindices_buffer, False))
        o = torch.empty_like(q)
        c._decode_handler.forward(q, o, c.kv_cache.buf_layer(0), c.kv_indices_without_last, None,
                                  c.kv_cache.last_page_len, c.kv_last_page_idx, None)
        out += [o, c.qk_product.clone(), c.lse.clone(), c.topk_dindices_buffer.clone()]
    w, x = randn(48, 64), randn(64)
    out += [_kernels.gemv(w, x), _kernels.gemv(w, x, norm_weight=randn(64), pair_gated=True),
            _kernels.gemv(w, x, residual=randn(48))]
    torch.cuda.synchronize()
    return out + [c.kv_cache.pool.buf, c.metadata_cache.pool.buf], c


_SHAPES = [(8, 8, 128, 16, "NHD", "per_head"), (8, 2, 64, 4, "HND", "group_sum"), (4, 4, 256, 7, "NHD", "per_head")]


def _use(monkeypatch, calls):
    from tidaldecode_amd import utils as ops
    from tidaldecode_amd.utils import batch_controller

    for module in (_kernels, ops, batch_controller):
        monkeypatch.setattr(module, "host_calls", calls)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", _SHAPES)
def test_same_bits_as_the_python_path(cuda, monkeypatch, dtype, shape):
    a, _ = _workload(cuda, dtype, *shape)
    _use(monkeypatch, _Off())
    b, _ = _workload(cuda, dtype, *shape)
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert x.dtype == y.dtype and x.shape == y.shape and torch.equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["per_head", "group_sum"])
@pytest.mark.parametrize("fused", [False, True])
def test_batches_are_served_natively_with_the_same_bits(cuda, monkeypatch, mode, fused):
    from tidaldecode_amd.utils import BatchInferenceController

    def workload(calls):
        _use(monkeypatch, calls)
        g = torch.Generator(device=cuda).manual_seed(3)
        c = BatchInferenceController(2, 8, 128, 16, 40, 700, 3, torch.bfloat16, cuda, num_kv_heads=2, select_mode=mode,
                                     page_order_seed=5)
        c.pool.buf.normal_(generator=g)
        c.add_sequences([600, 33, 150])
        out = []
        for _ in range(2):
            c.begin_step()
            cos, sin = c.rope_table()
            for layer in range(2):
                q, k, v = (torch.randn((3, h, 128), generator=g, device=cuda).bfloat16() for h in (8, 2, 2))
                if not fused:
                    c.rope_append(q, k, v, layer)
                fresh = (k, v, cos, sin) if fused else None
                if layer == 0:
                    out.append(c.attend_full(q, 0, output_qk_product=True, fresh=fresh))
                    c.select()
                else:
                    out.append(c.attend_sparse(q, 1, fresh=fresh))
            out += [c.qk_product.clone(), c.lse.clone(), c.topk_dindices_buffer.clone()]
        torch.cuda.synchronize()
        return out + [c.pool.buf]

    recorder = _Recorder()
    a, b = workload(recorder), workload(_Off())
    names = [name for name, _ in recorder.served]
    # (the first attention needs its workspace made)
    assert names.count("topk") == 2 and 3 <= names.count("attend") <= 4, names
    assert names.count("score_reduce") == (2 if mode == "group_sum" else 0)
    for x, y in zip(a, b):
        assert x.dtype == y.dtype and x.shape == y.shape and torch.equal(x, y)


@pytest.mark.gpu
def test_regular_calls_are_served_natively(cuda, monkeypatch):
    """No entry declines the calls it is there for (Python would give the same results, only later)."""
    calls = {}
    for shape in _SHAPES:
        recorder = _Recorder()
        _use(monkeypatch, recorder)
        _workload(cuda, torch.bfloat16, *shape)
        names = [name for name, _ in recorder.served]
        calls[shape] = {name: names.count(name) for name in _NATIVE}
    for shape, served in calls.items():
        # two steps of two layers: full attention through decode_sparse_attn needs its workspace once first
        assert served["append"] == 6 and served["rope_in_place"] == 3 and served["rope_table"] == 2, (shape, served)
        assert served["topk"] == 2 and served["estimate"] == 2 and served["gemv"] == 3, (shape, served)
        assert served["attend"] >= 2 and served["forward"] == 2, (shape, served)
        assert served["score_reduce"] == (2 if shape[-1] == "group_sum" else 0), (shape, served)
    assert max(served["prefill"] for served in calls.values()) == 2, calls  # two layers of a prompt


@pytest.mark.parametrize("mode", ["per_head", "group_sum"])
def test_slices_follow_the_tensors_they_are_of(mode):
    """Slices of a batched controller's tensors are kept while those stay: one that is exchanged, or another batch size,
    and they are made again."""
    from tidaldecode_amd.utils import batch_controller as bc

    c = bc.BatchInferenceController(1, 4, 64, 16, 8, 100, 3, torch.float16, "cpu", num_kv_heads=2, select_mode=mode)
    kinds = [bc._positions_of, bc._full_of, bc._sparse_of, bc._select_of] + ([bc._sums_of] if mode == "group_sum" else [])

    def agree():
        for of in kinds:
            kept, now = c._kept(of), of(c)
            for a, b in zip(kept if isinstance(kept, tuple) else (kept,), now if isinstance(now, tuple) else (now,)):
                assert a.data_ptr() == b.data_ptr() and a.shape == b.shape and a.stride() == b.stride(), of

    agree()
    c.add_sequences([20, 30])
    agree()
    for name in ("qk_product", "lse", "page_table", "_meta", "score_sum", "score_bound", "_table_starts", "_list_starts"):
        if getattr(c, name) is not None:
            setattr(c, name, getattr(c, name).clone())
            agree()


@pytest.mark.gpu
def test_launches_leave_the_interpreters_lock(cuda, monkeypatch):
    """Every call that was served, once more with PyGILState_Check (1 where its thread holds the lock, which
    reads as an error status) in place of the functions that launch."""
    calls, keep = _Recorder(), []
    _use(monkeypatch, calls)
    for shape in _SHAPES:
        keep.append(_workload(cuda, torch.bfloat16, *shape))
    real = {name: ctypes.cast(getattr(_lib.lib, name), ctypes.c_void_p).value for name in _lib.SIGNATURES}
    check = ctypes.cast(ctypes.pythonapi.PyGILState_Check, ctypes.c_void_p).value
    on_host = ("td_last_error", "td_decode_make_plan", "td_short_list_pays", "td_topk_workspace_bytes",
               "td_prefill_workspace_bytes")
    host_calls.bind({name: at if name in on_host else check for name, at in real.items()})
    held = set()
    try:
        for name, args in calls.served:
            try:
                assert getattr(host_calls, name)(*args) is not False, name
            except RuntimeError:
                held.add(name)
    finally:
        host_calls.bind(real)
    assert held == set()


@pytest.mark.gpu
def test_irregular_forms_still_work(cuda):
    """numpy integers, a value output, a workspace that is missing or too small, errors of the library."""
    g = torch.Generator(device=cuda).manual_seed(1)
    v = torch.randn((4, 500), generator=g, device=cuda)
    out, vals = torch.zeros((4, 30), dtype=torch.int32, device=cuda), torch.zeros((4, 30), device=cuda)
    _kernels.topk_filtering(v, None, vals, out, None, 30)
    assert torch.equal(vals, torch.gather(v, 1, out.long()))
    other = torch.zeros_like(out)
    _kernels.topk_filtering(v, None, None, other, None, np.int64(30))
    assert torch.equal(out, other)

    h, d, page, pages = 4, 128, 16, 40
    pool = torch.randn((pages, 2, page, h, d), generator=g, device=cuda).half()
    q = torch.randn((1, h, d), generator=g, device=cuda).half()
    table = torch.arange(pages - 1, dtype=torch.int32, device=cuda)[None]
    w = _kernels.BatchDecodeWithPagedKVCachePyTorchWrapper(0)
    o = torch.empty_like(q)
    with pytest.raises(RuntimeError, match="BeginForward"):
        w.forward(q, o, pool, table, None, 3, pages - 1, None)
    w.begin_forward(None, h, h, d, page, torch.empty(0, dtype=torch.half))
    first = None
    for kw in ({}, dict(n_list=np.int64(pages - 1)), dict(n_list=pages - 1)):
        w._workspace = None if first is None else torch.zeros(8, dtype=torch.uint8, device=cuda)
        w.forward(q, o, pool, table, None, 3, pages - 1, None, **kw)
        first = o.clone() if first is None else first
        assert torch.equal(o, first) and w._workspace.numel() > 8
    with pytest.raises(RuntimeError, match="o must have the shape of q"):
        w.forward(q, o[:, :2].contiguous(), pool, table, None, 3, pages - 1, None)
    with pytest.raises(RuntimeError, match="last_page_len"):
        w.forward(q, o, pool, table, None, page + 1, pages - 1, None)
