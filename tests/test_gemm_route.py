"""The kernel the GEMM's dispatch takes for a shape, asked of the library on
the CPU (kr_gemm_route launches nothing; without a device it counts 256 CUs)."""

import ctypes
from collections import namedtuple

import pytest

from kernrelay_amd import libapi

LOOPS = ("simple", "ring", "deep", "staged", "wide")
Route = namedtuple("Route", "bm bn loop pieces")


def route(M, N, K, lda=None, ldb=None, relay_rows=0, ws=False, norm=False, swiglu=False):
    """None: the launch would be refused."""
    fn = libapi.lib().kr_gemm_route
    i32, i64, out = ctypes.c_int, ctypes.c_int64, ctypes.POINTER(ctypes.c_int)
    fn.argtypes = [i32, i32, i32, i64, i64, i32, i32, i32, out, out, out, out]
    v = [ctypes.c_int() for _ in range(4)]
    rc = fn(M, N, K, K if lda is None else lda, K if ldb is None else ldb, relay_rows, int(ws), 1 if norm else 2 * swiglu,
            *(ctypes.byref(x) for x in v))
    return None if rc else Route(v[0].value, v[1].value, LOOPS[v[2].value], v[3].value)


@pytest.mark.parametrize("M,N", [(5, 24), (64, 4096), (200, 1536), (1024, 1024), (2048, 2048), (4096, 1000)])
def test_one_stage_of_k_takes_the_small_tiles(M, N):
    """K = 64 is one stage: a product with a CU for every 128x128 tile runs
    them, not a 256-wide tile (2048x2048x64: 8.8 us against 5.7)."""
    r = route(M, N, 64)
    assert (r.bn, r.pieces) == (128, 1) and r.bm in (64, 128)
    assert route(M, N, 64, ws=True) == r


@pytest.mark.parametrize("M,N,K,loop", [
    (2048, 1280, 128, "ring"), (2048, 1280, 384, "ring"), (2048, 1280, 448, "deep"), (2048, 2048, 64, "ring"),
    (2048, 2048, 192, "ring"), (1024, 1024, 64, "deep"), (1024, 1024, 128, "deep"), (4096, 1000, 512, "deep")])
def test_short_k_keeps_the_two_stage_ring_of_128_row_tiles(M, N, K, loop):
    """A K of at most six stages ends before the deep ring pays (2048x2048x192:
    6.9 us against 6.3); 64 row tiles take it at any K."""
    assert route(M, N, K).loop == loop
    assert route(M, N, K, relay_rows=M // 4).loop == loop


@pytest.mark.parametrize("M", [1, 37, 64, 65, 128, 200, 640, 1024, 2048, 4097])
@pytest.mark.parametrize("N", [16, 272, 2176, 9728])
@pytest.mark.parametrize("K", [64, 72, 256, 896, 904, 4096])
def test_swiglu_tiles_have_the_epilogue(M, N, K):
    """SwiGLU on 128 columns is built for the deep ring and the 256x128 tiles;
    the simple kernel and the two-stage ring of the small tiles are built
    without it (2% of every plain launch of the simple kernel)."""
    r = route(M, N, K, swiglu=True)
    assert r.bn == 256 or r.loop == "deep" or (r.bm == 256 and r.loop != "simple")
    plain = route(M, N, K)
    if plain.bn == 256 or plain.loop == "deep":
        assert r == plain


@pytest.mark.parametrize("M,N,K,norm,loop", [
    (4096, 3584, 16384, False, "wide"), (4096, 3584, 18944, False, "staged"), (4096, 4096, 12288, False, "wide"),
    (4096, 4096, 16384, False, "staged"), (8192, 8192, 8192, False, "wide"), (8192, 8192, 14336, False, "staged"),
    (8192, 4096, 12288, False, "staged"), (4096, 24576, 4096, False, "wide"), (16384, 520, 2048, False, "staged"),
    (4096, 3584, 3584, False, "wide"), (4096, 3584, 3584, True, "staged"), (4096, 4096, 12288, True, "staged"),
    (2048, 3584, 3584, False, "wide"), (2048, 3584, 3584, True, "wide"), (2048, 4096, 18944, False, "wide")])
def test_wide_loop_where_it_is_the_faster(M, N, K, norm, loop):
    """256x256 tiles run the wide loop over operands that the Infinity Cache
    holds, with four fifths of the CUs and without the Add+RMSNorm consumer
    (4096x3584x18944: 467 us against 434 in the 8-wave loop); the smaller
    256-wide tiles run it at any K from 2048 on."""
    r = route(M, N, K, relay_rows=M // 4 if norm else 0, norm=norm)
    assert r.loop == loop and r.bm * r.bn >= 256 * 128, r


@pytest.mark.parametrize("lda,ldb,loop", [
    (4096, 4096, "wide"), (4096, (1 << 23) - 8, "wide"), (0, 4096, "wide"), (1 << 23, 4096, "staged"),
    (4096, 1 << 23, "staged"), (-4096, 4096, "staged"), (4096, -4096, "staged"), (-4096, -4096, "staged")])
def test_wide_loop_row_strides(lda, ldb, loop):
    """The wide loop's unsigned 32-bit row offsets hold neither a row that lies
    4 GB ahead nor one that lies behind the tile's first: those would be read
    out of bounds, and run the 64-bit addressing of the 8-wave loop."""
    r = route(4096, 4096, 4096, lda=lda, ldb=ldb)
    assert (r.bm, r.bn, r.loop) == (256, 256, loop)
    for M, N in ((2048, 4096), (1024, 8192)):
        r = route(M, N, 4096, lda=lda, ldb=ldb)
        assert r.bm * r.bn == 256 * 128 and r.loop == ("wide" if loop == "wide" else "ring")
