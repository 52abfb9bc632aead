"""elm_routes.h, the rules that pick a kernel by sizes, types and alignment, compiled by the host compiler and asked without a
GPU: each rule at the calls that were measured on both of its sides, and over the forms that it accepts."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SHIM = r"""
#include "elm_routes.h"
using namespace elmh;
extern "C" int attn(int T, int n_cap, int pos_dev, int nh, int nkv, int hd, int quant, int aligned) {
  return (int)attention_route({T, n_cap, pos_dev != 0, nh, nkv, hd, quant != 0, aligned != 0});
}
extern "C" size_t score_bytes(int T, int n_cap, int pos_dev, int nh, int nkv, int hd, int quant, int aligned) {
  return attention_global_score_bytes({T, n_cap, pos_dev != 0, nh, nkv, hd, quant != 0, aligned != 0});
}
extern "C" int split16(int q8, int sw, int tok, int ring, int nb, int T, long wgs) {
  return gemm_split16_route(q8 != 0, sw != 0, tok != 0, ring != 0, nb, T, wgs);
}
extern "C" int f32gemm(int q8, int sw, int T, int K, const int* N, int n) { return (int)f32_gemm_route(q8 != 0, sw != 0, T, K, N, n); }
extern "C" int f32tiles(long groups) { return f32_gemm_tiles_per_launch(groups); }
extern "C" int q4wide(int sw, int norm, int nb, long rows) { return f32q4_wide_route(sw != 0, norm != 0, nb, rows); }
"""
STEP, ROWS4, ROWS8, PREFILL64, PREFILL, DECODE64, WHOLE, GLOBAL = range(8)


@pytest.fixture(scope="module")
def routes(tmp_path_factory):
    d = tmp_path_factory.mktemp("routes")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "edgelm_amd", "csrc"), str(d / "shim.cpp"), "-o", str(d / "routes.so")], check=True)
    lib = C.CDLL(str(d / "routes.so"))
    lib.score_bytes.restype = C.c_size_t
    return lib


def test_attention_key_cache_off_16_bytes(routes):
    """The kernels that copy key rows to LDS 16 bytes at a time take no key cache that starts elsewhere: head sizes other
    than 64 go to attention_kernel, 64 to the kernels that it has of its own."""
    for T in (1, 2, 7, 33, 300, 2048):
        for nh, nkv in ((1, 1), (9, 3), (32, 8), (32, 32)):
            for n in (T, 300 + T, 9500 + T, 23000 + T, 40000 + T):
                for hd in (4, 20, 80, 128, 256):
                    assert routes.attn(T, n, 0, nh, nkv, hd, 0, 0) in (WHOLE, GLOBAL)
                assert routes.attn(T, n, 0, nh, nkv, 64, 0, 0) not in (STEP, ROWS4, ROWS8)
    assert routes.attn(1, 2048, 1, 32, 8, 128, 0, 0) == WHOLE
    assert routes.attn(1, 2048, 1, 32, 8, 128, 0, 1) == STEP
    assert routes.attn(256, 512, 0, 32, 8, 128, 0, 1) == ROWS8


def test_attention_score_rows_only_where_they_are_used(routes):
    """A call that keeps its score rows in LDS asks for no global ones (a step over 20 to 24 thousand positions: the step
    kernel holds them where attention_kernel would not), and one on the kernel that uses them always does."""
    assert routes.attn(1, 22000, 1, 32, 8, 128, 0, 1) == STEP and routes.score_bytes(1, 22000, 1, 32, 8, 128, 0, 1) == 0
    assert routes.attn(1, 30000, 1, 32, 8, 128, 0, 1) == GLOBAL
    assert routes.score_bytes(1, 30000, 1, 32, 8, 128, 0, 1) == 32 * 30016 * 4
    for T in (1, 2, 64, 700):
        for nh, nkv in ((9, 3), (32, 8)):
            for hd in (16, 64, 128):
                for quant in (0, 1) if T > 1 and hd == 64 else (0,):
                    for n in range(T, 50000, 997):
                        need = routes.attn(T, n, 0, nh, nkv, hd, quant, 1) == GLOBAL
                        got = routes.score_bytes(T, n, 0, nh, nkv, hd, quant, 1)
                        assert got == (T * nh * ((n + 63) // 64 * 64) * 4 if need else 0)


@pytest.mark.parametrize("nh,nkv", [(9, 3), (14, 2), (32, 8), (4, 1)])
def test_attention_short_prompts_append_inside(routes, nh, nkv):
    """Head size 64, a chunk of few (token, head) pairs without a GEMM operand (a default Session's short prompt): one launch
    with the append inside up to 128 positions, the append and the step kernel past them."""
    for T in (2, 3, 5, 8, 17, 28, 64):
        if T * nh > 256:
            continue
        for n in (T, 64, 96, 128):
            assert n < T or routes.attn(T, n, 0, nh, nkv, 64, 0, 1) == PREFILL64
        for n in (129, 144, 192, 300, 700):
            assert routes.attn(T, n, 0, nh, nkv, 64, 0, 1) == STEP
        for n in (64, 192, 300):  # with the GEMM's operand: the kernel that writes it
            assert routes.attn(T, n, 0, nh, nkv, 64, 1, 1) == PREFILL64
        assert routes.attn(T, 100, 0, nh, nkv, 128, 0, 1) == STEP  # other head sizes: always


# (rows, K, tokens, faster with K split over the waves?) by (q8, SwiGLU, per-token scale), the measured calls nearest to where
# the two kernels cross; the rows of a 16 x 16 tile grid counted in eights
SPLIT = {
    (0, 0, 0): [(4096, 14336, 16, 1), (4096, 14336, 128, 1), (4096, 14336, 256, 0), (8192, 2048, 64, 1), (8192, 2048, 65, 0),
                (1536, 1568, 320, 0), (64, 2048, 4096, 0), (256, 4096, 1536, 1), (32000, 4096, 16, 1)],
    (1, 0, 0): [(4096, 4096, 112, 1), (4096, 4096, 128, 0), (2048, 2048, 192, 1), (2048, 2048, 256, 0), (32000, 4096, 8, 0),
                (16384, 4096, 16, 1), (128, 1568, 2048, 0), (256, 2048, 1536, 0), (256, 4096, 1536, 1), (1024, 14336, 512, 0)],
    (0, 0, 1): [(1536, 1568, 192, 1), (1536, 1568, 224, 0), (8192, 2048, 64, 0), (1024, 4096, 512, 0), (4096, 14336, 128, 1),
                (32000, 4096, 16, 1)],
    (1, 0, 1): [(4096, 14336, 128, 1), (16384, 4096, 32, 0), (256, 2048, 1536, 0), (4096, 4096, 256, 0)],
    (0, 1, 0): [(14336, 4096, 16, 1), (14336, 4096, 17, 0), (576, 1568, 384, 0), (1536, 1568, 128, 1), (256, 2048, 1024, 0),
                (16384, 4096, 16, 1)],
    (1, 1, 0): [(14336, 4096, 16, 0), (14336, 4096, 5, 0), (11008, 4096, 16, 0), (6144, 4096, 16, 1), (2048, 2048, 64, 1),
                (2048, 2048, 65, 0), (4096, 4096, 32, 1), (4096, 4096, 33, 0), (1536, 1568, 48, 0), (16384, 4096, 16, 1)],
    (0, 1, 1): [(14336, 4096, 16, 1), (576, 1568, 384, 0), (1536, 1568, 160, 0), (256, 2048, 1024, 0), (4096, 4096, 64, 1)],
    (1, 1, 1): [(14336, 4096, 16, 1), (4096, 4096, 64, 1), (128, 1568, 1536, 0), (1536, 1568, 320, 0)],
}


@pytest.mark.parametrize("kind", SPLIT, ids=lambda k: f"q{8 if k[0] else 4}{'-swiglu' * k[1]}{'-token' * k[2]}")
def test_gemm_split_over_waves_where_it_is_faster(routes, kind):
    for n, k, T, split in SPLIT[kind]:
        wgs = -(-(-(-n // 16)) // 8) * 8 * -(-T // 16)
        ring = -(-n // 128) * -(-T // 64) >= 128
        assert bool(routes.split16(*kind, ring, k // 32, T, C.c_long(wgs))) == bool(split), (n, k, T)
    assert not routes.split16(*kind, 0, 48, 16, C.c_long(8))  # short rows: gemm_lds16_kernel


R64X2, R16X8, R32X16, R64X16, R64X32 = range(5)


def f32gemm(routes, rows, K, T, q8=0, sw=0):
    rows = [rows] if isinstance(rows, int) else rows
    return routes.f32gemm(q8, sw, T, K, (C.c_int * len(rows))(*rows), len(rows))


@pytest.mark.parametrize("q8", [0, 1])
@pytest.mark.parametrize("sw", [0, 1])
def test_f32_gemm_few_tokens(routes, q8, sw):
    """Two to a few tokens: pairs of tokens where the rows are many, and no tile whose waves mostly stage only."""
    for n, k, T, pairs in [(49152, 576, 2, 1), (49152, 576, 4, 1), (49152, 576, 5, 0), (49152, 576, 8, 0), (128256, 2048, 2, 1),
                           (128256, 2048, 4, 1), (128256, 2048, 5, 0), (32000, 4096, 2, 1), (32000, 4096, 3, 0), (32768, 1024, 2, 1), (24576, 576, 2, 1),
                           (16384, 1024, 2, 0), (14336, 4096, 2, 0), (12288, 576, 2, 0), (4096, 4096, 2, 0), (1536, 576, 2, 0),
                           (16384, 256, 4, 1), (576, 576, 4, 0)]:
        r = f32gemm(routes, n, k, T, q8, sw)
        assert (r == R64X2) == bool(pairs), (n, k, T)
        assert r != R64X32
        assert T > 5 or r in (R64X2, R16X8, R64X16), (n, k, T)
    assert f32gemm(routes, [4096, 1024, 1024], 4096, 2, q8, sw) == R16X8
    assert f32gemm(routes, 18432, 576, 6, q8, sw) == R16X8 and f32gemm(routes, 14336, 4096, 6, q8, sw) == R32X16


def test_f32_gemm_tiles(routes):
    for T, tile in [(256, R64X32), (128, R64X16), (64, R32X16), (32, R32X16), (16, R16X8), (2, R16X8)]:
        assert f32gemm(routes, 4096, 4096, T) == tile, T
    for T, tile in [(16, R64X16), (17, R64X32), (32, R64X32), (33, R64X32), (65, R64X32)]:
        assert f32gemm(routes, 49152, 576, T) == tile, T
    for T, tile in [(17, R64X32), (32, R64X32), (33, R64X16), (48, R64X16), (49, R64X32), (65, R64X32)]:  # q8: the last tile's fill
        assert f32gemm(routes, 49152, 576, T, q8=1) == tile, T
    assert f32gemm(routes, 1536, 576, 93, q8=1, sw=1) == R16X8 and f32gemm(routes, 4096, 4096, 64, sw=1) == R32X16
    for k, T, n, pairs in [(64, 33, 4096, 1), (64, 93, 1536, 1), (64, 64, 512, 0), (64, 256, 4096, 0), (96, 33, 4096, 0)]:
        assert (f32gemm(routes, n, k, T) == R64X2) == bool(pairs), (n, k, T)
    for T, pairs in [(9, 1), (12, 1), (16, 0), (24, 1), (32, 0), (33, 1), (48, 0)]:
        assert (f32gemm(routes, 16384, 64, T, sw=1) == R64X2) == bool(pairs), T
    assert f32gemm(routes, 65536 * 64, 32, 2) != R64X2  # more row groups than a grid's second dimension takes


# (SwiGLU, norm): (rows, K, faster with a group per thread and 8 rows each?), measured on both sides
WIDE = {
    (0, 1): [(4096, 2080, 1), (14336, 2080, 0), (14336, 2400, 0), (14336, 2720, 1), (32768, 2080, 1), (16, 4096, 1), (14336, 4096, 1)],
    (1, 1): [(256, 2080, 0), (1024, 2080, 1), (8192, 2080, 0), (256, 3072, 0), (576, 3072, 1), (256, 3584, 1), (14336, 2720, 0),
             (14336, 2752, 1), (14336, 4096, 1), (65536, 2080, 0), (32768, 2400, 1)],
    (0, 0): [(4096, 2080, 0), (65536, 2080, 0), (4096, 3072, 0), (576, 4096, 0), (1536, 4096, 1), (4096, 4096, 1), (6144, 4096, 0),
             (8192, 4096, 1), (14336, 4096, 1), (2048, 4128, 1), (3072, 4128, 0), (32768, 4128, 0), (4096, 6144, 1), (6144, 6144, 0),
             (16, 8192, 1), (14336, 8192, 1), (6144, 8224, 0), (4096, 14336, 1)],
    (1, 0): [(14336, 2080, 0), (256, 4096, 0), (1024, 4096, 1), (4096, 3072, 1), (14336, 4096, 1), (8192, 4128, 0), (32768, 4128, 0),
             (4096, 14336, 1)],
}


@pytest.mark.parametrize("kind", WIDE, ids=lambda k: f"{'swiglu' if k[0] else 'plain'}{'-norm' * k[1]}")
def test_f32_one_token_long_rows_where_they_are_faster(routes, kind):
    for n, k, wide in WIDE[kind]:
        assert bool(routes.q4wide(*kind, k // 32, C.c_long(n))) == bool(wide), (n, k)


def test_f32_gemm_launches_fit_a_grid(routes):
    """A dispatch counts threads per dimension in 32 bits: 512 a workgroup. Up to the rows that the kernel before took (65,535
    groups of 64, which are 262,140 of 16) at least one token tile fits."""
    for groups in (1, 2, 3, 511, 65535, 262140, (1 << 22) - 1, 1 << 22):
        tiles = routes.f32tiles(C.c_long(groups))
        assert tiles >= 1 and tiles * groups * 512 < 1 << 32 and (tiles + 1) * groups > 1 << 22
    for groups in (0, -5, (1 << 22) + 1, 1 << 31):
        assert routes.f32tiles(C.c_long(groups)) == 0
