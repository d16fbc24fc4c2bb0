"""The rule that sends an exact per-matrix product to the row kernels or to the
tiles (moonshine_amd/csrc/k3_exact_rule.h), compiled for the CPU: products
timed on both kernels go to the faster one, and every product that the tiles
get has row offsets that fit their 32-bit counts."""
import ctypes
import pathlib
import subprocess

import pytest

CSRC = pathlib.Path(__file__).resolve().parents[1] / "moonshine_amd" / "csrc"

# (q8, tokens, rows, columns, us on the row kernels, us on the tiles)
TIMED = [(True, 3, 6144, 7168, 21.1, 25.3), (True, 5, 3584, 7168, 20.1, 22.4),
         (True, 6, 3000, 16512, 39.4, 60.0), (True, 5, 3463, 14464, 38.6, 51.6),
         (True, 5, 4427, 11392, 36.9, 60.6), (True, 2, 11390, 12288, 40.5, 58.8),
         (True, 7, 2566, 12544, 34.5, 44.9), (True, 66, 252, 9600, 23.9, 35.3),
         (True, 40, 442, 11520, 35.1, 41.3), (True, 27, 743, 12160, 38.9, 44.4),
         (False, 6, 3000, 16512, 37.9, 49.8), (False, 6, 4820, 12704, 47.3, 54.8),
         (False, 11, 1596, 9920, 26.5, 30.8),
         (True, 2, 20000, 128, 9.2, 4.9), (True, 2, 8747, 256, 5.5, 4.0),
         (True, 4, 7168, 6144, 28.5, 22.9), (True, 101, 293, 8320, 42.3, 31.5),
         (True, 18, 1183, 6528, 29.9, 23.9), (False, 8, 3072, 3584, 13.8, 12.0),
         (False, 512, 33, 8192, 32.1, 25.2), (False, 48, 512, 2048, 10.0, 8.4)]


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    (d / "rule.cpp").write_text(
        '#include "k3_exact_rule.h"\n'
        'extern "C" bool rows_form(uint32_t t, uint32_t r, uint32_t c, bool q8)\n'
        '{ return k3::dense_rows_form(t, r, c, q8); }\n'
        'extern "C" uint32_t form(uint32_t t, uint32_t r)\n'
        '{ const k3::DenseForm f = k3::dense_form(t, r); return f.rows | f.quads << 8; }\n')
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{CSRC}",
                    "-o", str(d / "rule.so"), str(d / "rule.cpp")], check=True)
    lib = ctypes.CDLL(str(d / "rule.so"))
    u = ctypes.c_uint32
    lib.rows_form.argtypes, lib.rows_form.restype = [u, u, u, ctypes.c_bool], ctypes.c_bool
    lib.form.argtypes, lib.form.restype = [u, u], u
    return lib


@pytest.mark.parametrize("q8,tokens,rows,columns,row_us,tile_us", TIMED)
def test_faster_kernel_is_chosen(rule, q8, tokens, rows, columns, row_us, tile_us):
    assert rule.rows_form(tokens, rows, columns, q8) == (row_us < tile_us)


@pytest.mark.parametrize("q8", [False, True])
def test_tiles_get_rows_within_their_offsets(rule, q8):
    # 31 rows and a stage of the last: a 32-bit byte offset
    longest = 0
    for bits in range(5, 32):
        for columns in (1 << bits, (1 << bits) + 128):
            for tokens, rows in ((2, 16384), (91, 181), (20000, 1), (3, 1 << 20)):
                if columns % 128 == 0 and not rule.rows_form(tokens, rows, columns, q8):
                    longest = max(longest, columns)
    assert longest >= 1 << 20
    assert 31 * (longest if q8 else longest // 2) + 512 < 1 << 32


def test_gpu_tests_reach_every_tile(rule):
    """The sizes that tests/test_gpu_exact.py runs as TILES take the tiles, each form among them."""
    pytest.importorskip("torch")
    import test_gpu_exact as G
    for q8 in (False, True):
        forms = set()
        for t, r, c in G.TILES:
            c = (c + 127) // 128 * 128 if q8 else c
            assert not rule.rows_form(t, r, c, q8), (t, r, c)
            f = rule.form(t, r)
            forms.add((f & 255, f >> 8, c > 8192))
        assert forms == {(b, n, long) for b, n in ((16, 1), (64, 1), (64, 2), (64, 4))
                         for long in (False, True)}
        assert all(rule.rows_form(t, r, c, q8) for t, r, c in G.SIZES)
