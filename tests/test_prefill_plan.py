"""The host's choices for the batched prefill's launches, on the CPU: the tests of the kernels name
sizes by what these choose."""
import ctypes

import pytest

from test_prefill_gpu import CHUNK_CASES


@pytest.fixture(scope="module")
def attention_plan(mh):
    call = ctypes.CDLL(str(mh.LIB_PATH)).muyo_prefill_attention_plan
    call.restype = None

    def plan(heads, kv_heads, head_dim, rows, pos0, workspace=True):
        """(chunks, tiles of 32 keys a chunk, keys handled at a time) of a launch."""
        out = (ctypes.c_uint32 * 3)()
        call(rows, pos0, heads, kv_heads, head_dim, int(workspace), out)
        return tuple(out)

    return plan


@pytest.mark.parametrize("shape", [(14, 2, 64), (4, 4, 64), (28, 4, 128), (8, 1, 128)])
def test_attention_chunks_cover_the_keys(attention_plan, shape):
    """At most eight chunks of whole 64-key steps, none of them empty, that hold every key; one of them
    without a workspace. At head_dim 128, where a chunk's sums run over all of it, at most 1024 keys
    or a quarter of the range (and a step)."""
    for rows in (1, 31, 32, 33, 64, 80, 100, 130, 257, 613, 1000, 2048, 4160):
        for pos0 in (0, 1, 31, 70, 700, 1000, 2015, 5003, 15000, 100000):
            tiles = (pos0 + rows - 1) // 32 + 1
            assert attention_plan(*shape, rows, pos0, workspace=False)[:2] == (1, (tiles + 1) // 2 * 2)
            chunks, length, _ = attention_plan(*shape, rows, pos0)
            assert 1 <= chunks <= 8 and length % 2 == 0 and -(-tiles // length) == chunks, (rows, pos0)
            if shape[2] == 128:
                assert length <= max(32, tiles // 4 + 2), (rows, pos0)


@pytest.mark.parametrize("rows,pos0", [(80, 0), (96, 0), (20, 70)])
@pytest.mark.parametrize("shape", [(14, 2, 64), (4, 4, 64), (28, 4, 128)])
def test_attention_of_three_key_tiles_is_one_chunk(attention_plan, shape, rows, pos0):
    """A merge costs more than a second 64-key step, also where the range is an odd number of tiles."""
    assert attention_plan(*shape, rows, pos0)[:2] == (1, 4)


def test_attention_of_short_ranges_takes_32_keys_at_a_time(attention_plan):
    """At head_dim 64 up to two tiles of 32 keys: a wave does not work through the hidden half of a
    64-key step. (At 128 it never takes 64.)"""
    for rows, pos0, keys in ((1, 0, 32), (32, 0, 32), (64, 0, 32), (20, 44, 32), (65, 0, 64), (1, 64, 64)):
        assert attention_plan(14, 2, 64, rows, pos0)[2] == keys, (rows, pos0)
        assert attention_plan(28, 4, 128, rows, pos0)[2] == 32


@pytest.mark.parametrize("rows,pos0,chunks", [(32, 100, 3), (45, 100, 3), (130, 0, 1), (250, 0, 4), (301, 100, 7)])
def test_attention_chunks_of_small_merges(attention_plan, rows, pos0, chunks):
    """14 / 2 heads of 64: three steps or more are split where the merge is small."""
    assert attention_plan(14, 2, 64, rows, pos0)[0] == chunks


@pytest.mark.parametrize("heads,kv_heads,head_dim,rows,pos0,max_seq,check,planned", CHUNK_CASES)
def test_attention_chunk_cases_are_planned_as_they_say(attention_plan, heads, kv_heads, head_dim, rows, pos0, max_seq,
                                                       check, planned):
    assert attention_plan(heads, kv_heads, head_dim, rows, pos0)[:2] == planned
