"""How many threads share an output row in the merge kernel, from the rule the library
uses (the inline function of ``csrc/sqa_internal.h``, compiled for the host)."""

import ctypes
import subprocess

import pytest

from small_q_attention_amd import build as sqa_build


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("merge_rule")
    src, lib = tmp / "rule.cpp", tmp / "rule.so"
    src.write_text('#include "sqa_internal.h"\n'
                   'extern "C" int rule(long long rows, int per_row, int chunks, int cus) {\n'
                   "  return sqa::merge_row_threads(rows, per_row, chunks, cus);\n}\n")
    subprocess.run([sqa_build.hipcc_path(), "-x", "hip", "--offload-host-only", "-std=c++17",
                    "-fPIC", "-shared", f"-I{sqa_build.CSRC}", str(src), "-o", str(lib)],
                   check=True, capture_output=True)
    fn = ctypes.CDLL(str(lib)).rule
    fn.argtypes = [ctypes.c_longlong] + [ctypes.c_int] * 3
    return fn


@pytest.mark.parametrize("chunks", [8, 16, 32])
@pytest.mark.parametrize("cus", [32, 64, 128, 256])
def test_rows_share_a_wave_from_two_waves_per_simd_of_the_device(rule, chunks, cus):
    rows = cus * 4 * 2 * 64 // chunks
    assert rule(rows, 8, chunks, cus) == chunks
    assert rule(rows - 1, 8, chunks, cus) == (64 if rows - 1 >= 1024 else 256)
    assert rule(rows, 9, chunks, cus) == (64 if rows >= 1024 else 256)


@pytest.mark.parametrize("chunks", [8, 16, 32, 64])
def test_a_wave_per_row_where_one_round_of_loads_covers_it(rule, chunks):
    most = 8 * (64 // chunks)
    for cus in (0, 256):
        assert rule(1024, most, chunks, cus) == 64
        assert rule(1024, most + 1, chunks, cus) == 256
        assert rule(1023, 2, chunks, cus) == 256
