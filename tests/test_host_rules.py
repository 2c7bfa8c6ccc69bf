"""Rules of the launches that no entry point tells of, compiled from moe_internal.h for the host alone."""
import ctypes as C
import os
import subprocess

import pytest

from gpt_oss_amd import build

SOURCE = """
#include "%s/moe_internal.h"
extern "C" int split_router_tokens(int E_pad, int H) { return moe::split_router_tokens(E_pad, H); }
extern "C" int bf16_wide_tiles(int T, int E, int H, int IM, int past) { return moe::bf16_wide_tiles(T, E, H, IM, past); }
extern "C" int bf16_stores_past(int gate_up, int tiles, int T, int E) { return moe::bf16_stores_past(gate_up, tiles, T, E); }
extern "C" int norm_wave_per_token(int T, int H) { return moe::norm_wave_per_token(T, H); }
""" % build.CSRC


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.hip").write_text(SOURCE)
    subprocess.run([build.HIPCC, "--offload-host-only", "-std=c++17", "-O1", "-fPIC", "-shared", "-Wno-everything",
                    str(d / "rules.hip"), "-o", str(d / "rules.so")], check=True)
    return C.CDLL(str(d / "rules.so"))


@pytest.mark.parametrize("E_pad,H,tokens", [(16, 2880, 0), (64, 2880, 0), (128, 256, 0), (128, 736, 0), (128, 768, 400),
                                            (128, 1024, 400), (128, 1440, 1024), (128, 2880, 1024), (256, 128, 200),
                                            (256, 256, 400), (256, 512, 400), (256, 2880, 1024)])
def test_router_splits_where_it_gains(rules, E_pad, H, tokens):
    """The router's first pass as a launch of its own costs small matrices more than it gains
    (times in moe_internal.h)."""
    assert rules.split_router_tokens(E_pad, H) == tokens


@pytest.mark.parametrize("T,H,wave", [(1, 32, 1), (7168, 256, 1), (1, 512, 1), (64, 544, 0), (1023, 1024, 0),
                                      (1024, 1024, 1), (7168, 1056, 0), (7168, 2880, 0)])
def test_norm_of_short_rows_takes_a_wave(rules, T, H, wave):
    """A workgroup per token of short rows is mostly idle threads (times in norm.hip)."""
    assert rules.norm_wave_per_token(T, H) == wave


@pytest.mark.parametrize("T,E,H,IM,past,wide", [
    (6144, 128, 2880, 2880, 1, 1), (2000, 128, 2880, 2880, 1, 1), (6144, 128, 2880, 2880, 0, 0),
    (256, 32, 2880, 2880, 1, 0), (1400, 32, 2880, 2880, 1, 0), (250, 8, 2880, 2880, 1, 0),
    (1028, 256, 1024, 512, 1, 1), (1028, 256, 1088, 576, 1, 1), (1028, 256, 1216, 640, 1, 1), (1028, 256, 960, 512, 1, 0)])
def test_wide_tiles_where_the_cus_take_many_rounds(rules, T, E, H, IM, past, wide):
    """Tiles of ten column blocks gain with four rounds of tiles and lose with two (times in moe_internal.h)."""
    assert rules.bf16_wide_tiles(T, E, H, IM, past) == wide


@pytest.mark.parametrize("gate_up,tiles,T,E,past", [
    (1, 368, 144, 16, 0), (1, 368, 145, 16, 1), (1, 512, 144, 16, 1), (1, 736, 150, 32, 1), (1, 256, 250, 32, 0), (1, 460, 200, 20, 1),
    (0, 192, 256, 16, 0), (0, 192, 257, 16, 1), (0, 256, 300, 32, 0), (0, 257, 300, 32, 1), (0, 384, 150, 32, 1), (0, 32, 449, 32, 0)])
def test_stores_past_the_caches_where_they_gain(rules, gate_up, tiles, T, E, past):
    """Few rows of a GEMM of a round or two are found in the caches by the next kernel (times in moe_internal.h)."""
    assert rules.bf16_stores_past(gate_up, tiles, T, E) == past
