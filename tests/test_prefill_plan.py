"""The host's choices for the batched prefill's launches, on the CPU: the tests of the kernels name
sizes by what these choose."""
import ctypes

import pytest

from test_prefill_gpu import CHUNK_CASES, TILE_SHAPES


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


@pytest.fixture(scope="module")
def gemm_plan(mh):
    call = ctypes.CDLL(str(mh.LIB_PATH)).muyo_prefill_gemm_plan
    call.restype = None

    def plan(rows, n, k, splits=1):
        """(tokens, weight rows, slab columns) of the tile, token tiles per group, K splits (0: chosen)."""
        out = (ctypes.c_uint32 * 5)()
        call(rows, n, k, splits, out)
        return tuple(out[:3]), out[3], out[4]

    return plan


@pytest.mark.parametrize("rows,n,k,tile", TILE_SHAPES)
def test_gemm_tile_cases_take_the_tiles_they_say(gemm_plan, rows, n, k, tile):
    assert gemm_plan(rows, n, k)[0] == tile
    ffn = n // 8 * 4 or 4
    assert gemm_plan(rows, -(-ffn // 16) * 32, k)[0] == tile


def test_gemm_tile_cases_cover_every_tile(gemm_plan):
    covered = {case[3] for case in TILE_SHAPES}
    for rows in (1, 7, 33, 64, 100, 200, 301, 613, 900, 1300, 1500, 2048, 4096, 8192):
        for n in (64, 896, 1152, 2560, 3584, 4608, 9728, 37888, 151936):
            for k in (64, 896, 3584, 4864, 18944):
                assert gemm_plan(rows, n, k)[0] in covered, (rows, n, k)


# The fastest measured tile, or one within 2 % of it, at full prompts of both widths, an ordinary one, a
# short turn and some other large products.
@pytest.mark.parametrize("rows,n,k,tile", [
    (2048, 9728, 896, (64, 256, 64)), (4096, 9728, 896, (128, 256, 32)), (2048, 37888, 3584, (256, 256, 32)),
    (2048, 3584, 3584, (128, 256, 32)), (2048, 3584, 18944, (128, 256, 32)), (2048, 28672, 4096, (256, 256, 32)),
    (8192, 151936, 896, (256, 256, 32)), (613, 9728, 896, (128, 192, 64)), (301, 896, 4864, (32, 64, 128)),
    (45, 37888, 3584, (64, 192, 64)),
])
def test_gemm_takes_the_measured_tile(gemm_plan, rows, n, k, tile):
    assert gemm_plan(rows, n, k)[0] == tile


def test_gemm_groups_of_token_tiles(gemm_plan):
    """Over several rounds of workgroups, near the square of an XCD's resident tiles and all of about the
    same size; in one round all token tiles, or one where there are more of them than weight rows."""
    for rows, n, k, tile, group in ((8192, 28672, 4096, 256, 4), (2048, 37888, 3584, 256, 4), (2048, 9728, 896, 64, 8),
                                    (1541, 5000, 520, 64, 7), (45, 37888, 3584, 64, 1), (513, 2000, 1784, 32, 17),
                                    (1500, 896, 4864, 32, 1), (301, 9728, 896, 64, 5)):
        assert gemm_plan(rows, n, k)[0][0] == tile, (rows, n, k)
        assert gemm_plan(rows, n, k)[1] == group, (rows, n, k)


def test_gemm_splits_give_every_split_work(gemm_plan):
    """Whole 128-column units per split, none empty; at most eight up to 512 rows, four beyond, which is
    what the decoder's partial planes are sized for. The prompts of the decoder's tests meet one, a
    few and more than four splits (the norm and rope kernels sum up to one, four or eight)."""
    seen = set()
    for rows in (1, 24, 40, 96, 300, 301, 512, 513, 1024, 1990, 2048):
        for n, k in ((1152, 896), (896, 896), (896, 4864), (4608, 3584), (3584, 3584), (3584, 18944), (512, 256), (64, 8)):
            splits = gemm_plan(rows, n, k, 0)[2]
            units = -(-k // 128)
            assert 1 <= splits <= (8 if rows <= 512 else 4)
            assert -(-units // -(-units // splits)) == splits, (rows, n, k)
            if (n, k) in ((1152, 896), (896, 4864)) and rows in (96, 300):
                seen.add(splits)
    assert min(seen) <= 3 and max(seen) > 4
