"""Which kernel the launch planning picks, and its shape, at the rules'
edges, on the CPU (tests/dispatch_plan.py)."""
import pytest

import dispatch_plan as dp
from kvx_amd.abi import DType, Layout

NHD, HND, PK = Layout.BLOCK_NHD, Layout.BLOCK_HND, Layout.BLOCK_HND_PACKED
BF16, F32, E4M3, E5M2 = DType.BF16, DType.F32, DType.F8_E4M3, DType.F8_E5M2


@pytest.mark.parametrize("table,flat", [("ragged", "gather_ragged_tile"),
                                        ("offsets", "gather_indexed_flat")])
def test_wide_rows_into_f32_stay_in_the_flat_gathers(table, flat):
    for H in (33, 40, 63):  # 4224 to 8064 elements, in chunks of four
        assert dp.gather(NHD, table, E4M3, F32, 16, H, 128)["kernel"] == flat
    assert dp.gather(NHD, table, E4M3, F32, 16, 72, 128)["kernel"] == "gather_indexed"
    for io, H, kernel in ((BF16, 63, flat), (BF16, 72, "gather_indexed")):
        assert dp.gather(NHD, table, E4M3, io, 16, H, 128)["kernel"] == kernel
        assert dp.gather(NHD, table, io, io, 16, H, 128)["kernel"] == kernel


def test_four_code_chunks_in_flight():
    unroll = dp.lib().kvx_flat_unroll
    assert (unroll(4, True), unroll(4, False), unroll(8, False)) == (4, 2, 2)


@pytest.mark.parametrize("table", ["packed", "ragged", "offsets"])
def test_parts_keep_the_tile_width_of_whole_blocks(table):
    """576-byte rows: 64-byte tiles fill 8 KiB in blocks of 128 tokens and
    more; in 64-token blocks they do not."""
    for bs, tw in ((64, 144), (128, 64), (256, 64)):
        plan = dp.gather(PK, table, E4M3, BF16, bs, 1, 576)
        assert (plan["kernel"], plan["rows"], plan["tw"]) == ("gather_tiles", 64, tw)


def test_parts_of_one_byte_runs_hold_whole_lines():
    """128 rows a part of a token-innermost FP8 tensor, unless its rows are a
    whole number of KiB; the other formats and dtypes keep 64."""
    def rows(cache, table, H, D, bs, io=BF16):
        plan = dp.gather(dp.VLLM, table, cache, io, bs, H, D)
        assert plan["kernel"] == "gather_tiles" and plan["rows"] * plan["parts"] == bs
        return plan["rows"]

    for bs in (128, 256, 512):
        for H, D in ((1, 128), (2, 128), (8, 64), (8, 96), (1, 576), (12, 128)):
            assert rows(E4M3, "packed", H, D, bs) == 128
            assert rows(E5M2, "packed", H, D, bs, F32) == 128
            assert rows(E4M3, "ragged", H, D, bs) == 64
            assert rows(BF16, "packed", H, D, bs) == 64
        for H, D in ((8, 128), (16, 128), (24, 128)):
            assert rows(E4M3, "packed", H, D, bs) == 64
    assert rows(E4M3, "packed", 2, 128, 64) == 64
    assert dp.gather(PK, "packed", E4M3, BF16, 256, 2, 128)["rows"] == 64


def test_copies_of_whole_line_runs_in_big_blocks():
    """RAGGED / KV_OFFSETS copies of HND blocks of more than 64 tokens: the
    row kernel, or parts where its waves or registers do not suit the row."""
    def kernel(table, H, D, bs, dtype=BF16, io=None):
        return dp.gather(HND, table, dtype, io or dtype, bs, H, D)["kernel"]

    rows, tiles = "gather_indexed", "gather_tiles"
    for bs in (128, 256, 512):
        for H, D, dt in ((2, 128, BF16), (8, 64, BF16), (8, 128, BF16), (16, 128, BF16),
                         (6, 128, BF16), (8, 96, BF16), (2, 128, F32), (6, 128, F32)):
            assert kernel("ragged", H, D, bs, dt) == rows
            # KV_OFFSETS: a whole block whose tile fits 64 KiB goes in parts
            run = D * (4 if dt == F32 else 2)
            whole = D != 96 and bs * (run + 16) <= 65536
            assert kernel("offsets", H, D, bs, dt) == (tiles if whole else rows)
        for H, D, dt in ((3, 128, BF16), (8, 128, F32), (16, 128, F32)):
            assert kernel("ragged", H, D, bs, dt) == tiles
            assert kernel("offsets", H, D, bs, dt) == tiles
        assert kernel("ragged", 8, 128, bs, E4M3, BF16) == tiles
        assert dp.gather(PK, "ragged", BF16, BF16, bs, 8, 128)["kernel"] == tiles
    assert kernel("ragged", 8, 128, 64) == tiles
    assert kernel("packed", 3, 128, 256) == tiles


@pytest.mark.parametrize("table", ["ragged", "offsets"])
def test_short_padded_rows_into_f32_take_chunks_of_eight(table):
    def chunk(H, D, io=F32, pad=16):
        plan = dp.gather(NHD, table, E5M2, io, 16, H, D, pad=pad)
        assert plan["kernel"] == "gather_indexed"
        return plan["chunk"]

    assert [chunk(H, D) for H, D in ((4, 40), (3, 128), (7, 64))] == [8, 8, 8]
    assert [chunk(H, D) for H, D in ((4, 128), (8, 128))] == [4, 4]
    assert chunk(4, 36, pad=12) == 4  # heads that are not whole chunks of eight
    assert chunk(4, 40, BF16) == 8
    assert dp.gather(NHD, table, E5M2, F32, 16, 3, 128)["chunk"] == 4  # the flat gathers
    assert dp.gather(NHD, "packed", E5M2, F32, 16, 3, 128, pad=16)["chunk"] == 4


@pytest.mark.parametrize("bs", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("cache,io", [(BF16, BF16), (F32, F32), (E4M3, BF16), (E5M2, F32)])
def test_narrow_tiles_hold_whole_units(cache, io, bs):
    """Tiles of a token-innermost tensor have rows for a whole unit of slots
    however small the batch, and align on as much as their lanes hold."""
    seg = 16 // dp.BYTES[cache]
    for H, D in ((1, 128), (3, 128), (8, 128), (1, 576)):
        for T in (1, 64, 1000, 4000, 30000):
            plan = dp.write(dp.VLLM, cache, io, bs, H, D, T, nb=65536)
            t = plan["t"][1]
            assert (plan["kernel"], t["kind"]) == ("write_tiles", 2)
            # at most four runs a thread, unless that takes more than 256
            runs = t["rows"] * t["tw"] // t["run"]
            assert plan["threads"] == 256 or plan["threads"] * 4 >= runs
            assert t["seg"] == seg and 2 * seg <= t["rows"] <= 32
            align = min(bs, 64 // dp.BYTES[cache], t["rows"])
            assert t["align"] == align >= seg and t["tw"] >= 32


def test_narrow_tiles_that_fill_a_wave():
    """The shapes that test_gpu_write_tiles.py's WHOLE cases run: 32 rows and 32
    aligned slots, 16 KiB tiles for the larger copy."""
    for cache, io, T, tile in ((BF16, BF16, 1100, 4096), (BF16, BF16, 4200, 16384),
                               (E4M3, BF16, 2100, 4096), (E5M2, F32, 4200, 8192)):
        for bs in (32, 64, 128):
            t = dp.write(dp.VLLM, cache, io, bs, 8, 128, T)["t"][1]
            assert (t["rows"], t["align"], t["rows"] * t["tw"]) == (32, 32, tile)


def test_quantizing_writes_by_chunk():
    """The kernels and chunks that test_gpu_fp8_paths.py's CHUNKS cases run."""
    for H, D, pad, codes in ((4, 64, 8, 8), (4, 64, 4, 4), (4, 64, 2, 2), (4, 64, 1, 1),
                             (4, 40, 0, 8), (4, 12, 0, 4), (3, 6, 0, 2), (3, 7, 0, 1)):
        for io in (BF16, DType.F16, F32):
            for bs in (16, 20):
                plan = dp.write(HND, E4M3, io, bs, H, D, 90, pad=pad)
                assert (plan["kernel"], plan["chunk"]) == ("write", codes)
                plan = dp.write(NHD, E4M3, io, bs, H, D, 90, pad=pad)
                assert plan["chunk"] == codes
                assert plan["kernel"] == ("write" if pad else "write_flat")


def test_ragged_tiles_of_sparse_batches():
    """The rows per tile that test_gpu_gather_skew.py's cases run."""
    for cache, io, H, D, base in ((BF16, BF16, 1, 776, 1), (E4M3, BF16, 2, 776, 1),
                                  (E5M2, F32, 1, 1552, 1), (BF16, BF16, 1, 392, 2),
                                  (BF16, BF16, 1, 576, 2)):
        full = base * 49152
        for entries, r in ((full - 1, base), (full, 2 * base)):
            plan = dp.gather(NHD, "ragged", cache, io, 16, H, D, S=24, L=full, entries=entries)
            assert (plan["kernel"], plan["rows"]) == ("gather_ragged_tile", r)
