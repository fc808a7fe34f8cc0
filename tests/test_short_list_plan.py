"""Plans of the short-list kernel: they cover the list, keep to 64 splits, no split is empty, and the partials stay
within the built-in scratch wherever a single split does."""
import pytest

from tidaldecode_amd._lib import TD_ERR_INVALID_ARG, TD_ERR_UNSUPPORTED, TD_IDX_PAGES, TD_IDX_SLOTS, DecodePlan, lib


SCRATCH = 4 << 20


@pytest.mark.parametrize("hq,hkv,d", [(32, 32, 128), (32, 8, 128), (28, 4, 128), (40, 40, 64), (28, 4, 64), (8, 1, 64)])
@pytest.mark.parametrize("batch", [1, 3, 16])
def test_plans(hq, hkv, d, batch):
    for rows in {hq, hkv, 1}:
        for items in [1, 31, 32, 33, 128, 129, 255, 256, 257, 400, 777, 1300, 2048, 2500, 4096, 6001, 12000, 16384]:
            p = DecodePlan(0, 0, 0, 0, -1, 0, 0, 0)
            assert lib.td_decode_make_plan(batch, hq, hkv, d, rows, items, p) == 0
            assert p.sparse_waves in (4, 8) and p.sparse_rows == 8
            assert p.chunk_tokens % (p.sparse_waves * 4096 // d) == 0
            assert 1 <= p.max_splits <= 64 and (p.max_splits - 1) * p.chunk_tokens < items <= p.max_splits * p.chunk_tokens
            assert p.workspace_bytes <= SCRATCH or p.max_splits == 1, (rows, items, p.max_splits, p.workspace_bytes)
            # quotients by the product with 2^32 / chunk, rounded up, which the kernel forms
            magic = ((1 << 32) + p.chunk_tokens - 1) // p.chunk_tokens
            for n in (1, items // 2 + 1, items):
                x = n + p.chunk_tokens - 1
                assert (x * magic) >> 32 == x // p.chunk_tokens


@pytest.mark.parametrize("waves,rows", [(1, 0), (2, 0), (3, 8), (5, 0), (16, 0), (0, 4), (8, 12)])
def test_preset_shapes_that_no_kernel_has(waves, rows):
    """An error, not a division by the chunk that no shape gave."""
    for hq, hkv, idx_rows in [(32, 32, 32), (32, 8, 8), (32, 8, 32)]:
        p = DecodePlan(0, 0, 0, 0, -1, waves, rows, 0)
        assert lib.td_decode_make_plan(1, hq, hkv, 128, idx_rows, 2048, p) == TD_ERR_UNSUPPORTED
        assert b"no short-list kernel" in lib.td_last_error()
    for hq, hkv, d, idx_rows in [(32, 32, 64, 32), (32, 8, 64, 8), (28, 4, 128, 4), (28, 4, 128, 28)]:
        p = DecodePlan(0, 0, 0, 0, -1, waves, rows, 0)  # shapes that the short-list kernel came to later: ignored
        assert lib.td_decode_make_plan(1, hq, hkv, d, idx_rows, 2048, p) == 0 and p.sparse_waves == 0


@pytest.mark.parametrize("waves", [0, 4, 8])
@pytest.mark.parametrize("batch", [1, 4, 16, 64, 256])
def test_sixteen_rows_a_lane_keep_to_the_scratch(waves, batch):
    for items in (100, 777, 2048, 5000, 16384):
        p = DecodePlan(0, 0, 0, 0, -1, waves, 16, 0)
        assert lib.td_decode_make_plan(batch, 32, 32, 128, 32, items, p) == 0 and p.sparse_rows == 16
        assert p.workspace_bytes <= SCRATCH or p.max_splits == 1


@pytest.mark.parametrize("hq,hkv,d,slots", [(28, 4, 128, 32), (40, 8, 128, 64), (48, 8, 128, 64), (32, 8, 64, 32),
                                            (14, 2, 64, 16), (32, 8, 128, 32), (32, 32, 128, 32)])
def test_batches_beyond_a_ticket_per_head_slot_stream(hq, hkv, d, slots):
    """The short-list kernel takes a ticket per head slot (padded groups have more of them than heads), the streaming
    kernel one per head row: up to 16384 of either."""
    most = 16384 // slots
    for batch, waves in [(most, (4, 8)), (most + 1, (0,))]:
        p = DecodePlan(0, 0, 0, 0, -1, 0, 0, 0)
        rc = lib.td_decode_make_plan(batch, hq, hkv, d, hkv, 512, p)
        if hq == hkv and batch > most:
            assert rc == TD_ERR_INVALID_ARG  # a head row a head: no tickets for either
        else:
            assert rc == 0 and p.sparse_waves in waves
    hrows = hkv if hq > hkv else hq
    p = DecodePlan(0, 0, 0, 0, -1, 0, 0, 0)
    assert lib.td_decode_make_plan(16384 // hrows, hq, hkv, d, hkv, 512, p) == 0
    assert lib.td_decode_make_plan(16384 // hrows + 1, hq, hkv, d, hkv, 512, DecodePlan(0, 0, 0, 0, -1, 0, 0, 0)) == \
        TD_ERR_INVALID_ARG


@pytest.mark.parametrize("hq,hkv,d,rows", [(32, 32, 128, 32), (32, 8, 128, 8), (28, 4, 128, 4), (28, 4, 128, 28),
                                           (32, 8, 64, 1)])
def test_which_calls_are_for_the_short_list_kernel(hq, hkv, d, rows):
    def pays(kind, items, scores, batch=1):
        return lib.td_short_list_pays(batch, hq, hkv, d, rows, items, kind, scores)

    most = (72 << 20) // 4 // ((hq if rows == hq else hkv) * d)  # tokens of 72 MiB
    for kind, scores in [(TD_IDX_PAGES, 0), (TD_IDX_PAGES, 1), (TD_IDX_SLOTS, 1)]:
        assert pays(kind, most, scores) and not pays(kind, most + 1, scores)
        assert pays(kind, 500, scores, 4) and not pays(kind, 2049, scores, 2)
    assert pays(TD_IDX_SLOTS, 1 << 20, 0) and pays(TD_IDX_SLOTS, 2049, 0, 64)
