"""Which kernel a launch takes (csrc/launch_rules.hpp), on the CPU: the lines as they were
measured on an MI355X's 256 compute units."""
from __future__ import annotations

import ctypes
import os
import subprocess

import pytest

import test_gpu_prefill_forms as forms

HERE = os.path.dirname(os.path.abspath(__file__))
CUS = 256
PAIRS2, PAIRS1, ROWS1X8, ROWS2X8, ROWS2X4 = range(5)


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
