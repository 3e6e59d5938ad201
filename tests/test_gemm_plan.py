"""Which tiles the GEMMs of batches take (no GPU needed: the plan for 256 compute units, nothing is launched).  The GPU tests of those
tiles take their shapes from here, so that a shape that takes others after a change of the rules is noticed."""
import ctypes as C

import pytest

from llama2_rs import _lib

FP32, FP16 = _lib.PREFILL_FP32, _lib.PREFILL_MFMA

# (outputs, columns): columns of a tile, width of the tiles of what whole rounds of blocks leave over (its own: there are none), the columns
# behind the last whole tile where they have a narrower one of their own, whether a row block has whole tiles and others.
# 256 inputs, groups of 64; in the fp32 mode ...
FP32_TILES = {
    (24584, 150): (80, 80, 0, 0), (24584, 177): (64, 16, 0, 1), (24584, 192): (64, 16, 0, 1), (22008, 258): (64, 48, 0, 0),
    (22008, 300): (64, 48, 0, 0), (16640, 250): (64, 16, 0, 0), (4104, 61): (32, 32, 0, 0), (8200, 195): (64, 32, 0, 0),
    (11784, 405): (64, 32, 0, 1), (19464, 290): (80, 16, 0, 0), (14344, 385): (80, 16, 0, 1), (16392, 385): (80, 32, 0, 0),
    (18696, 385): (80, 48, 0, 0), (18696, 405): (80, 64, 0, 0)}
# ... and in the fp16 mode
FP16_TILES = {
    (21888, 300): (144, 144, 12, 0), (21888, 350): (128, 32, 0, 1), (21888, 520): (144, 48, 0, 0), (21888, 590): (128, 96, 0, 1),
    (25472, 350): (128, 32, 0, 1), (25472, 424): (128, 48, 40, 1), (15360, 180): (64, 32, 0, 0), (15360, 99): (64, 64, 0, 0),
    (22016, 440): (144, 32, 8, 1), (24832, 453): (144, 48, 21, 1), (25856, 492): (144, 64, 60, 1), (27392, 492): (144, 80, 60, 1),
    (26880, 388): (144, 32, 0, 1), (18176, 583): (144, 32, 7, 0), (24832, 570): (144, 96, 0, 0), (27392, 518): (144, 112, 0, 0),
    (27392, 570): (144, 128, 0, 0), (25088, 440): (128, 64, 56, 1), (20224, 583): (128, 80, 0, 1)}
# (inputs, outputs, group): {columns: the same}; fp32, then fp16
FP32_OF_80 = {
    (128, 22016, 64): {150: (80, 80, 0, 0), 160: (80, 80, 0, 0)}, (256, 22016, 128): {129: (80, 80, 0, 0), 150: (80, 80, 0, 0), 225: (64, 32, 0, 0)},
    (320, 22016, 64): {150: (80, 80, 0, 0)}, (384, 22016, 32): {130: (64, 16, 0, 1), 90: (64, 48, 0, 0)}, (384, 12800, 128): {230: (64, 48, 0, 0)},
    (320, 14344, 64): {385: (80, 16, 0, 1)}}
FP16_OF_144 = [(128, 22016, 32), (128, 22016, 64), (256, 22016, 128), (384, 22272, 64), (640, 22016, 32), (768, 22016, 128)]
FP16_ODD = {
    (256, 22016, 64): {200: (128, 112, 0, 0)}, (256, 20480, 128): {240: (128, 80, 0, 0), 193: (128, 80, 0, 0)},
    (384, 12800, 64): {230: (64, 48, 0, 0), 353: (128, 80, 0, 0)}, (256, 12800, 32): {225: (64, 48, 0, 0)},
    (512, 1024, 128): {33: (64, 64, 0, 0), 48: (64, 64, 0, 0), 65: (64, 64, 1, 0), 97: (64, 64, 0, 0), 113: (64, 64, 0, 0), 177: (64, 64, 0, 0)}}


def plan(n_in, out, group, columns, mode):
    p = (C.c_int32 * 8)()
    _lib.check(_lib.lib().l2_gemm_plan(n_in, (C.c_int32 * len(out))(*out), len(out), group, columns, mode, p))
    return dict(zip(("rows", "tokens", "slices", "blocks", "whole", "width", "last", "both"), p))


def tiles(n_in, n_out, group, columns, mode):
    p = plan(n_in, [n_out], group, columns, mode)
    return p["tokens"], p["width"], p["last"], p["both"]


def test_shapes_take_the_tiles_they_stand_for():
    for (n_out, columns), want in FP32_TILES.items():
        assert tiles(256, n_out, 64, columns, FP32) == want, (n_out, columns)
    for (n_out, columns), want in FP16_TILES.items():
        assert tiles(256, n_out, 64, columns, FP16) == want, (n_out, columns)
    for shapes, mode in ((FP32_OF_80, FP32), (FP16_ODD, FP16)):
        for shape, by_columns in shapes.items():
            for columns, want in by_columns.items():
                assert tiles(*shape, columns, mode) == want, (shape, columns)
    for shape in FP16_OF_144:
        assert tiles(*shape, 256, FP16) == (128, 128, 0, 0)
        for columns in (257, 273, 288):
            assert tiles(*shape, columns, FP16) == (144, 144, 0, 0), (shape, columns)


# Every output of every slice is computed once: the blocks are the whole tiles, those of what rounds leave over and the narrow last ones
@pytest.mark.parametrize("mode", [FP32, FP16])
def test_blocks_cover_the_outputs(mode):
    for n_in, group in ((256, 32), (1024, 64), (4096, 128), (28672, 64)):
        for out in ([1024], [4096, 1024, 1024], [11008, 11008], [5120], [13824, 13824], [28672, 28672], [256]):
            for columns in list(range(17, 330, 13)) + [511, 512, 640, 777, 899]:
                p = plan(n_in, out, group, columns, mode)
                units = sum(-(-n // p["rows"]) for n in out) * p["slices"]
                if p["last"]:  # of the units whose tiles are all whole
                    t_full = columns // p["tokens"]
                else:
                    t_full = -(-columns // p["tokens"])
                begun, part = (p["whole"] // t_full, p["whole"] % t_full) if t_full else (units, 0)
                assert (part > 0) == p["both"]
                rest = 0 if not part else -(-(columns - part * p["tokens"]) // p["width"])
                rest += (units - begun - (part > 0)) * -(-columns // p["width"])
                assert p["blocks"] == p["whole"] + rest + (begun if p["last"] else 0), (n_in, out, columns, p)


def test_refused():
    p, out = (C.c_int32 * 8)(), (C.c_int32 * 1)(64)
    lib = _lib.lib()
    assert lib.l2_gemm_plan(256, out, 1, 64, 64, FP32, p) == 0
    for bad in ((250, out, 1, 64, 64, FP32), (256, out, 0, 64, 64, FP32), (256, out, 1, 48, 64, FP32), (256, out, 1, 64, 0, FP32),
                (256, out, 1, 64, 64, 2), (256, out, 1, 0, 64, FP16), (192, out, 1, 64, 64, FP16), (256, None, 1, 64, 64, FP32)):
        assert lib.l2_gemm_plan(*bad, p) < 0, bad
