"""Which kernel a launch takes (csrc/launch_rules.hpp), on the CPU: the lines as they were
measured on an MI355X's 256 compute units."""
from __future__ import annotations

import ctypes
import os
import subprocess

import pytest

import test_gpu_dense as dense
import test_gpu_prefill_forms as forms

HERE = os.path.dirname(os.path.abspath(__file__))
CUS = 256
PAIRS2, PAIRS1, ROWS1X8, ROWS2X8, ROWS2X4 = range(5)
GATE_TILES, TILES16, TILES32, STREAM16, STREAM64 = range(5)


@pytest.fixture(scope="session")
def rules(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("rules") / "rules.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-Wall", "-Werror",
                    "-I" + os.path.join(HERE, "..", "llm-inference-engine_amd", "csrc"),
                    os.path.join(HERE, "launch_rules.cpp"), "-o", lib], check=True)
    return ctypes.CDLL(lib)


# rows, query heads, KV heads; the kernel with single (f16) and with hi + lo operands.
PREFILL = [
    (2, 14, 2, ROWS1X8, ROWS1X8), (288, 14, 2, ROWS1X8, ROWS1X8), (304, 14, 2, ROWS2X8, ROWS2X8),
    (1280, 14, 2, ROWS2X8, ROWS2X4), (1500, 14, 2, ROWS2X4, ROWS2X4),
    (2400, 14, 2, ROWS2X4, ROWS2X4), (2560, 14, 2, PAIRS2, ROWS2X4), (2720, 14, 2, PAIRS2, ROWS2X4),
    (2736, 14, 2, PAIRS2, PAIRS2), (4000, 14, 2, PAIRS2, PAIRS2), (5000, 14, 2, PAIRS1, PAIRS1),
    # Eight heads to a KV head, short prompts: pairs from 24 / 48 on (640 rows: 18.6 against 23.8 us)
    (512, 64, 8, ROWS2X4, ROWS2X4), (544, 64, 8, PAIRS2, ROWS2X4), (640, 64, 8, PAIRS2, PAIRS2),
    (960, 40, 5, PAIRS2, ROWS2X4), (1088, 40, 5, PAIRS2, PAIRS2),
    # Four: row blocks to two thirds, of 4 waves once 8 would leave a second round
    (512, 32, 8, ROWS2X8, ROWS2X8), (576, 32, 8, ROWS2X4, ROWS2X4), (672, 32, 8, ROWS2X4, ROWS2X4),
    (704, 32, 8, PAIRS2, PAIRS2), (1100, 16, 8, PAIRS1, PAIRS1),
    (2147483647, 14, 2, PAIRS1, PAIRS1),
]


@pytest.mark.parametrize("T,nh,nkv,single,split", PREFILL)
def test_prefill(rules, T, nh, nkv, single, split):
    assert rules.prefill_kernel(T, nh, nkv, 0, CUS) == single
    assert rules.prefill_kernel(T, nh, nkv, 1, CUS) == split


@pytest.mark.parametrize("T,nh,want", [(1, 14, ROWS1X8), (290, 14, ROWS2X8), (288, 14, ROWS1X8),
                                       (512, 14, ROWS2X8), (992, 14, ROWS2X8), (1024, 14, ROWS2X4),
                                       (2147483647, 14, ROWS2X4)])
def test_prefill_f32(rules, T, nh, want):
    assert rules.prefill_f32_kernel(T, nh, CUS) == want


def test_prefill_forms_are_reached(rules):
    """The shapes of test_gpu_prefill_forms.py take the forms that they are named after."""
    got = lambda T, nh, nkv: {rules.prefill_kernel(T, nh, nkv, split, CUS) for split in (0, 1)}
    assert all(got(*s) == {PAIRS2} for s in forms.PAIRS_TWO_TEAMS + [forms.SEGMENTS_TWO_TEAMS[1:]])
    assert all(got(*s) == {PAIRS1} for s in forms.PAIRS_ONE_TEAM + [forms.SEGMENTS_ONE_TEAM[1:]])
    assert got(*forms.ONE_TILE_OF_TWO_BLOCKS) == {ROWS2X8}
    for shapes in (forms.PAIRS_TWO_TEAMS, forms.PAIRS_ONE_TEAM):
        assert {nh // nkv for _, nh, nkv in shapes} == set(range(1, 9))


@pytest.mark.parametrize("cols,T,want", [
    (896, 1, STREAM16), (896, 16, STREAM16), (1024, 16, STREAM16), (1056, 16, TILES16),
    (864, 16, TILES16), (128, 1, TILES16), (896, 17, TILES32), (896, 32, TILES32),
    (896, 33, STREAM64), (768, 64, STREAM64), (1024, 64, STREAM64), (736, 64, TILES32),
    (128, 64, TILES32), (1056, 64, TILES32), (896, 65, TILES32)])
def test_wide(rules, cols, T, want):
    """LM heads: the weights are streamed where K fills the registers that are set aside for it."""
    assert rules.wide_kernel(0, cols, T) == want
    assert rules.wide_kernel(1, cols, T) == GATE_TILES


def test_dense_shapes_are_reached(rules):
    """test_gpu_dense.py's shapes take every tile shape and every wide form, with ragged rows."""
    wide = lambda rows: (rows + 15) // 16 >= 16 * CUS
    plain = {rules.tile(0, rows, cols, T, CUS) for T, rows, cols in dense.TILED
             if not wide(rows) and cols >= 256 and rows % 16}
    assert plain == set(range(7))
    gate = {rules.tile(1, rows, cols, T, CUS) for T, rows, cols in dense.GATE_TILED
            if not wide(rows) and cols >= 256 and rows % 16}
    assert gate == set(range(5))
    forms = {rules.wide_kernel(0, cols, T) for T, rows, cols in dense.TILED if wide(rows)}
    assert forms == {TILES16, TILES32, STREAM16, STREAM64}
    assert any(wide(rows) for _, rows, _ in dense.GATE_TILED)


@pytest.mark.parametrize("rows,tokens,cols,wbytes,fits", [
    (128, 32, 16_777_184, 2, 1), (128, 32, 16_777_216, 2, 0), (128, 32, 33_554_400, 1, 1),
    (128, 32, 33_554_432, 1, 0), (16, 16, 67_108_832, 2, 1), (16, 16, 67_108_864, 2, 0),
    (16, 16, 150_000_000, 2, 0), (16, 16, 2_147_483_616, 2, 0)])
def test_tile_offsets(rules, rows, tokens, cols, wbytes, fits):
    """The last byte of a tile's last row and token is within 32 bits of its first, or the
    launch goes to the kernel with 64-bit addresses."""
    assert rules.offsets_fit(rows, tokens, ctypes.c_int64(cols), wbytes) == fits
    assert fits == (rows * cols * wbytes < 2**32 and tokens * cols * 4 < 2**32)


def test_short_k(rules):
    """Matrices of fewer than 8 K blocks; the dense tests' shapes take both sides of the line."""
    staged = lambda T, rows, cols, norm=0: rules.short_k(
        ctypes.c_int64((rows + 15) // 16 * ((T + 15) // 16)), cols, norm, CUS)
    assert staged(600, 256, 192) and staged(4000, 64, 32) and staged(600, 896, 96, 1)
    assert not (staged(64, 896, 192) or staged(600, 64, 192) or staged(600, 896, 64, 1))
    short = [s for s in dense.TILED if s[2] < 256 and s[1] < 65000]
    assert {staged(*s) for s in short} == {0, 1}
    assert any(staged(*s) and s[2] % 256 for s in short) and any(staged(*s) for s in dense.GATE_TILED)


def test_decode_f32_waves(rules):
    got = {c: rules.decode_waves(c) for c in (16, 32, 48, 64, 80, 96, 112, 128, 144, 192, 208, 1024)}
    assert got == {16: 1, 32: 1, 48: 2, 64: 4, 80: 2, 96: 2, 112: 4, 128: 4, 144: 1, 192: 1, 208: 4,
                   1024: 4}
