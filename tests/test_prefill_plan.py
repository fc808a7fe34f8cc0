"""CPU: the split of a prompt's work (csrc/prefill.hip, plan_prefill).

The planner adds up key tiles and pieces over all row tiles in closed form.  Here they are added up tile by
tile, with the same estimate of the time, and the bytes of scratch must agree; and a plan, which every call
makes, must not cost the host what it saves the device."""
import random
import time

import pytest

from tidaldecode_amd import _kernels
from tidaldecode_amd._lib import TD_ERR_INVALID_ARG, TD_ERR_UNSUPPORTED, PagedKV, last_error, lib

LIMIT = 256 << 20      # bytes
CUS = lib.td_num_cus()


def scratch_bytes(hq, hkv, d, kv_len, n_q, causal=1):
    pool = PagedKV(16, kv_len // 16 + 1, hkv, d, 16, 0, _kernels.TD_BF16)   # the address is not used
    return lib.td_prefill_workspace_bytes(pool, kv_len, n_q, hq, causal)


def ceil(a, b):
    return -(-a // b)


def bytes_tile_by_tile(hq, hkv, d, kv_len, n_q, causal):
    group, bn = hq // hkv, 32 if d == 256 else 64
    rows, max_tiles, best = n_q * group, ceil(kv_len, bn), None
    for bm, step, start in ((64, 1.0, 4.5),) if d == 256 else ((256, 1.0, 6.5), (128, 0.87, 4.5), (64, 0.83, 4.5)):
        ends = [kv_len - n_q + (min(r + bm, rows) - 1) // group + 1 if causal else kv_len for r in range(0, rows, bm)]
        tiles = [ceil(e, bn) for e in ends]
        for s in (1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16, 32, 64):
            chunk = ceil(max_tiles, s)
            if s > 1 and (chunk < 4 or len(tiles) * hkv >= 8 * CUS):
                break
            n = ceil(kv_len, chunk * bn)
            scratch = n * hkv * rows * (d + 2) * 4 if n > 1 else 0
            if scratch > LIMIT:
                break
            jobs = hkv * sum(ceil(t, chunk) for t in tiles)
            mean, longest = step * (hkv * sum(tiles) / jobs) + start, step * chunk + start
            slots = CUS * (2 if d == 256 else 1)
            cost = max(min(mean * jobs / slots + 0.25 * longest, ceil(jobs, slots) * mean), longest)
            if s > 1:
                cost += 2.0 + hkv * rows * d * 4e-6 * s / 4.0
            if best is None or cost < best[0] * (1 - 1e-12):
                best = (cost, scratch)
    return best[1]


@pytest.mark.parametrize("d", [64, 128, 256])
def test_closed_form_equals_the_sum_over_tiles(d):
    rng = random.Random(d)
    split = 0
    for _ in range(150):
        hkv = rng.choice([1, 2, 3, 4, 8, 16, 32])
        hq = hkv * rng.choice([1, 2, 3, 4, 7, 8])
        n_q = int(round(2 ** rng.uniform(0, 12.5)))
        past = rng.choice([0, rng.randint(1, 300), int(2 ** rng.uniform(5, 17))])
        shape = (hq, hkv, d, past + n_q, n_q, rng.choice([1, 1, 1, 0]))
        got = scratch_bytes(*shape)
        assert got == bytes_tile_by_tile(*shape), shape
        split += got > 0
    assert 30 <= split <= 120                       # both kinds are among them


@pytest.mark.parametrize("hq,hkv,d,past,n_q", [
    (32, 8, 128, 0, 2900), (28, 4, 128, 0, 4000), (32, 8, 128, 8000, 2000), (32, 8, 128, 0, 102400),
    (32, 1, 128, 0, 2000)])
def test_a_plan_takes_the_host_microseconds(hq, hkv, d, past, n_q):
    """20 to 100 us when every row tile was visited; 1 us in closed form, most of it the call through ctypes."""
    pool = PagedKV(16, (past + n_q) // 16 + 1, hkv, d, 16, 0, _kernels.TD_BF16)
    best = float("inf")
    for _ in range(20):                             # the fastest of many: the machine may be busy
        t = time.perf_counter()
        for _ in range(20):
            lib.td_prefill_workspace_bytes(pool, past + n_q, n_q, hq, 1)
        best = min(best, (time.perf_counter() - t) / 20)
    assert best < 8e-6


def test_scratch_is_bounded():
    """The largest plans: many rows of many heads on long caches."""
    rng = random.Random(0)
    used = []
    for d, hq, hkv in ((128, 40, 40), (256, 32, 32), (256, 64, 8), (64, 16, 16)):
        for _ in range(200):
            n_q = int(2 ** rng.uniform(9, 15))
            used.append(scratch_bytes(hq, hkv, d, n_q + rng.choice([0, int(2 ** rng.uniform(9, 18))]), n_q))
    assert LIMIT // 2 < max(used) <= LIMIT


def test_workspace_that_is_not_aligned_is_refused():
    """16-byte accesses to the partial results; the host refuses before anything is launched."""
    pool = PagedKV(4096, 2049, 8, 128, 16, 0, _kernels.TD_BF16)             # addresses that nothing touches
    n_bytes = lib.td_prefill_workspace_bytes(pool, 32768, 16, 32, 1)
    assert n_bytes > 0
    for off in (1, 4, 8):
        rc = lib.td_prefill_attn_split(pool, 4096, 2048, 32768, 4096, 4096, 16, 32, 0.1, 1, 4096 + off, n_bytes, None)
        assert rc == TD_ERR_INVALID_ARG and "16-byte aligned" in last_error()


def test_lengths_that_only_memory_limits():
    """2^30 tokens of one head of 64 dimensions, and 2^30 packed query rows, fit 288 GB."""
    for n in ((1 << 30) + 5, (1 << 31) - (1 << 14) - 1):
        assert scratch_bytes(4, 1, 64, n, 16) == bytes_tile_by_tile(4, 1, 64, n, 16, 1) > 0
        assert scratch_bytes(32, 32, 64, n, 1 << 16) == 0           # whole tiles
    # a head_dim without a kernel: refused for that, after the sizes were accepted and before any launch
    pool = PagedKV(4096, 1 << 22, 1, 32, 16, 0, _kernels.TD_BF16)
    rows = lib.td_prefill_attn(pool, 4096, 1 << 21, 1 << 25, 4096, 4096, 1 << 25, 32, 0.1, 1, None)
    assert rows == TD_ERR_UNSUPPORTED and "head_dim" in last_error()
