"""The GEMM's small-product kernels (deep ring, split K) and its wide loop at
the edges of their tiles and plans, against float64 and against the simple
data-parallel tiles bit for bit.

Tolerance: a 16-bit result is off its exact value by half an ulp (at most 2^-8
of the value in bf16, whose significand has 8 bits, 2^-11 in fp16, 11) plus the fp32 sum's error, at most K 2^-24 of
the sum of |a b| (far below it for these K); a bias adds one more rounding of
each of the product and the sum."""

import pytest
import torch

from kernrelay_amd import ops
from tests.conftest import announce
from tests.test_gemm_route import route

pytestmark = pytest.mark.gpu

BF, HF = torch.bfloat16, torch.float16


def make(M, N, K, dt, bias, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    # views into wider buffers: row strides beyond K, different for x and w
    x = torch.randn(M, K + 24, device="cuda", generator=g).to(dt)[:, :K]
    w = (torch.randn(N, K + 8, device="cuda", generator=g) * 0.02).to(dt)[:, :K]
    b = (torch.randn(N, device="cuda", generator=g) * 0.5).to(dt) if bias else None
    return x, w, b


def check(y, x, w, b):
    prod = x.double() @ w.double().t()
    ref = prod if b is None else prod + b.double()
    half = 2.0 ** -8 if y.dtype == BF else 2.0 ** -11
    mag = x.double().abs() @ w.double().abs().t()
    bound = half * (ref.abs() + (prod.abs() if b is not None else 0.0)) * 1.01 + x.shape[1] * 2.0 ** -24 * mag
    assert bool(((y.double() - ref).abs() <= bound).all())


# rows around the 64 and 128 row tiles, columns that are no multiple of 8 or of
# 128, K from one stage per piece up; two to sixteen pieces
@pytest.mark.parametrize("M,N,K,dt,bias", [
    (1, 8, 4096, BF, False), (37, 896, 4864, BF, True), (64, 128, 2048, HF, False), (65, 130, 2048, BF, True),
    (129, 1000, 3584, HF, True), (200, 3584, 3584, BF, False), (300, 896, 4864, BF, False),
    (200, 3584, 18944, BF, False), (1001, 896, 4864, HF, False), (1919, 520, 4096, BF, False)])
def test_split_k_small(gpu, M, N, K, dt, bias):
    announce("gemm split %dx%dx%d" % (M, N, K))
    nbytes, ncnt = ops.gemm_streamk_workspace(M, N, K)
    assert 0 < nbytes <= 16 << 20 and ncnt > 0
    x, w, b = make(M, N, K, dt, bias, 5)
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    cnt = torch.zeros(ncnt, dtype=torch.int32, device="cuda")
    pad = torch.full((M + 3, N + 16), 3.0, dtype=dt, device="cuda")
    y = pad[:M, :N]
    ops.gemm_streamk(x, w, y, ws, cnt, bias=b)
    first = y.clone()
    for _ in range(2):
        y.zero_()
        ops.gemm_streamk(x, w, y, ws, cnt, bias=b)
        assert torch.equal(y, first)
    assert int(cnt.abs().sum()) == 0
    assert torch.all(pad[M:] == 3.0) and torch.all(pad[:, N:] == 3.0)
    check(first, x, w, b)


# deep-ring tiles with fewer stages than the ring (one stage too), as many, and
# more; then larger tiles with ragged rows, on the wide loop and on the staged
# one (4097 columns: 192x256 tiles)
@pytest.mark.parametrize("M,N,K,dt,bias", [
    (5, 24, 64, BF, False), (64, 128, 128, BF, True), (65, 129, 256, HF, False), (130, 260, 320, BF, True),
    (200, 896, 384, BF, False), (1024, 3584, 448, HF, False), (1111, 6144, 4096, HF, True),
    (2040, 4097, 2048, BF, False), (515, 24576, 2048, BF, False), (4096, 3584, 2112, BF, True)])
def test_tiles_bit_exact(gpu, M, N, K, dt, bias):
    announce("gemm tiles %dx%dx%d" % (M, N, K))
    x, w, b = make(M, N, K, dt, bias, 6)
    pad = torch.full((M + 3, N + 16), 3.0, dtype=dt, device="cuda")
    y = pad[:M, :N]
    ops.gemm(x, w, y, bias=b)
    ref = torch.empty(M, N, dtype=dt, device="cuda")
    ops.gemm(x, w, ref, bias=b, bm=64)  # 64x256 tiles, two-stage ring
    assert torch.equal(y, ref)
    assert torch.all(pad[M:] == 3.0) and torch.all(pad[:, N:] == 3.0)
    check(y, x, w, b)


# the wide loop with ragged rows and columns in each of its tiles: the last tile's
# rows of A and of B past the edge re-read the last row by their 32-bit offsets
@pytest.mark.parametrize("M,N,K,dt,bias,tile", [
    (4090, 3590, 2112, BF, True, (256, 256)), (3841, 4095, 2048, HF, False, (256, 256)),
    (2041, 3465, 2112, BF, False, (256, 128)), (1793, 3969, 2048, HF, True, (256, 128)),
    (515, 24571, 2048, BF, False, (128, 256)), (513, 24449, 2112, HF, True, (128, 256))])
def test_wide_loop_ragged(gpu, M, N, K, dt, bias, tile):
    announce("gemm wide loop %dx%dx%d" % (M, N, K))
    r = route(M, N, K, lda=K + 24, ldb=K + 8)
    assert ((r.bm, r.bn), r.loop) == (tile, "wide")
    x, w, b = make(M, N, K, dt, bias, 9)
    pad = torch.full((M + 3, N + 16), 3.0, dtype=dt, device="cuda")
    y = pad[:M, :N]
    ops.gemm(x, w, y, bias=b)
    ref = torch.empty(M, N, dtype=dt, device="cuda")
    ops.gemm(x, w, ref, bias=b, bm=64)  # 64x256 tiles, two-stage ring
    assert torch.equal(y, ref)
    assert torch.all(pad[M:] == 3.0) and torch.all(pad[:, N:] == 3.0)
    check(y, x, w, b)


# the SwiGLU epilogue on 128-column tiles, and where they are built without it
# (K of one to six stages on more than 256 of the 64-row tiles, K no multiple of 64)
@pytest.mark.parametrize("M,cols,K", [(1, 8, 64), (37, 4864, 896), (200, 136, 896), (200, 12288, 4096),
                                      (1111, 1024, 256), (65, 72, 904)])
def test_swiglu_small_tiles(gpu, M, cols, K):
    announce("gemm swiglu %dx%dx%d" % (M, cols, K))
    x, w, _ = make(M, 2 * cols, K, BF, False, 7)
    gu = torch.empty(M, 2 * cols, dtype=BF, device="cuda")
    ops.gemm(x, w, gu, bm=64)
    ref, act = torch.empty(M, cols, dtype=BF, device="cuda"), torch.empty(M, cols, dtype=BF, device="cuda")
    ops.elementwise("swiglu_gu", gu, ref)
    ops.gemm_swiglu_epilogue(x, w, act)
    assert torch.equal(act, ref)


# relay tiles that no row tile divides, in one piece and split
@pytest.mark.parametrize("M,N,K,k,streamk", [
    (576, 4096, 512, 1, False), (576, 4096, 512, 3, False), (768, 3584, 512, 4, False), (192, 896, 4864, 1, True),
    (192, 896, 4864, 3, True), (768, 3584, 18944, 4, True)])
def test_relay_norm_odd_relay_tiles(gpu, M, N, K, k, streamk):
    announce("gemm+add_rmsnorm %dx%dx%d k=%d" % (M, N, K, k))
    x, w, _ = make(M, N, K, BF, False, 8)
    res, gamma = torch.randn(M, N, device="cuda").to(BF), torch.ones(N, device="cuda").to(BF)
    ws = cnt = None
    ref_c = torch.empty(M, N, dtype=BF, device="cuda")
    if streamk:
        nbytes, ncnt = ops.gemm_streamk_workspace(M, N, K)
        assert nbytes > 0
        ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
        cnt = torch.zeros(ncnt, dtype=torch.int32, device="cuda")
        ops.gemm_streamk(x, w, ref_c, ws, cnt)
    else:
        ops.gemm(x, w, ref_c)
    ref_y, ref_s, c, y, s = (torch.empty_like(ref_c) for _ in range(5))
    ops.rowop("add_rmsnorm", res, ref_y, x1=ref_c, gamma=gamma, sum_out=ref_s)
    ctrl = torch.zeros(k * ops.CTRL_WORDS, dtype=torch.int32, device="cuda")
    for run in range(1, 3):
        for t in (c, y, s):
            t.zero_()
        ops.gemm_add_rmsnorm(x, w, c, res, gamma, y, ops.make_pub(ctrl, 0, M // k), sum_out=s, ws=ws, counters=cnt)
        torch.cuda.synchronize()
        assert torch.equal(c, ref_c) and torch.equal(y, ref_y) and torch.equal(s, ref_s)
        blk = ctrl.cpu().reshape(k, ops.CTRL_WORDS)
        assert torch.all(blk[:, 0] == run) and torch.all(blk[:, 1] == run) and torch.all(blk[:, 2] == 1)
        assert torch.all(blk[:, 3:5] == 0)


def norm_case(M, N, K, k, streamk, seed):
    x, w, _ = make(M, N, K, BF, False, seed)
    g = torch.Generator(device="cuda").manual_seed(seed + 1)
    res, gamma = torch.randn(M, N, device="cuda", generator=g).to(BF), torch.ones(N, device="cuda").to(BF)
    c, y, s, ref_c, ref_y, ref_s = (torch.empty(M, N, dtype=BF, device="cuda") for _ in range(6))
    ws = cnt = None
    if streamk:
        nbytes, ncnt = ops.gemm_streamk_workspace(M, N, K)
        ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
        cnt = torch.zeros(ncnt, dtype=torch.int32, device="cuda")
        ops.gemm_streamk(x, w, ref_c, ws, cnt)
    else:
        ops.gemm(x, w, ref_c)
    ops.rowop("add_rmsnorm", res, ref_y, x1=ref_c, gamma=gamma, sum_out=ref_s)
    ctrl = torch.zeros(k * ops.CTRL_WORDS, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()

    def run(stream=None, max_spins=0):
        ops.gemm_add_rmsnorm(x, w, c, res, gamma, y, ops.make_pub(ctrl, 0, M // k), sum_out=s, ws=ws, counters=cnt,
                             max_spins=max_spins, stream=stream)

    def verify(runs, status):
        assert torch.equal(c, ref_c) and torch.equal(y, ref_y) and torch.equal(s, ref_s)
        blk = ctrl.cpu().reshape(k, ops.CTRL_WORDS)
        assert torch.all(blk[:, 0] == runs) and torch.all(blk[:, 1] == runs) and torch.all(blk[:, 3:] == 0)
        assert all(int(v) in status for v in blk[:, 2])
        for t in (c, y, s):
            t.zero_()

    return run, verify


# a spin bound of one or a few: most workgroups leave before the release and
# the one that releases the tile works their rows (whole tiles in one piece
# and two per CU, relay tiles that no row tile divides, split K in small and
# 256x256 tiles with relay tiles above and below a row block)
@pytest.mark.parametrize("M,N,K,k,streamk", [
    (1024, 3584, 512, 4, False), (2048, 2048, 192, 2, False), (576, 4096, 512, 3, False), (256, 136, 72, 4, False),
    (192, 896, 4864, 3, True), (128, 896, 4864, 2, True), (768, 3584, 18944, 4, True),
    (2048, 896, 4864, 32, True), (2048, 896, 4864, 2, True), (4096, 4096, 256, 2, False)])
def test_relay_norm_left_rows(gpu, M, N, K, k, streamk):
    announce("gemm+add_rmsnorm leaving %dx%dx%d k=%d" % (M, N, K, k))
    run, verify = norm_case(M, N, K, k, streamk, 11)
    for n, spins in enumerate((1, 3, 20), 1):
        run(max_spins=spins)
        torch.cuda.synchronize()
        verify(n, (1, 2))
    run()
    torch.cuda.synchronize()
    verify(4, (1,))


# launches on two streams that each take nearly every CU (224 workgroups, one
# per CU): neither keeps the other from its end
@pytest.mark.parametrize("M,N,K,k,streamk", [(1024, 3584, 512, 1, False), (1024, 3584, 512, 4, False),
                                             (768, 3584, 18944, 4, True)])
def test_relay_norm_two_streams(gpu, M, N, K, k, streamk):
    announce("gemm+add_rmsnorm on two streams %dx%dx%d k=%d" % (M, N, K, k))
    cases = [norm_case(M, N, K, k, streamk, seed) for seed in (12, 14)]
    streams = [ops.QueueStream() for _ in cases]
    try:
        for _ in range(4):
            for (run, _v), st in zip(cases, streams):
                run(stream=st)
        torch.cuda.synchronize()
        for _run, verify in cases:
            verify(4, (1,))
    finally:
        for st in streams:
            st.close()


# products that the shared scratch of the allocation-free entry does not cover
# (under a 256x256 tile, or fewer than two pieces of 16 stages): whole tiles, as
# kr_op_gemm, also on two streams at once
@pytest.mark.parametrize("M,N,K", [(200, 3584, 3584), (255, 896, 4864), (1000, 248, 4096), (300, 896, 1984)])
def test_noalloc_small_takes_no_scratch(gpu, M, N, K):
    announce("gemm streamk noalloc small %dx%dx%d" % (M, N, K))
    assert ops.gemm_streamk_workspace(M, N, K)[0] > 0  # with a workspace it would split
    cases = []
    for seed in (16, 17):
        x, w, b = make(M, N, K, BF, True, seed)
        ref, y = torch.empty(M, N, dtype=BF, device="cuda"), torch.empty(M, N, dtype=BF, device="cuda")
        ops.gemm(x, w, ref, bias=b)
        cases.append((x, w, b, ref, y, torch.cuda.Stream()))
    torch.cuda.synchronize()
    for _ in range(8):
        for x, w, b, _ref, y, st in cases:
            ops.gemm_streamk_noalloc(x, w, y, bias=b, stream=st)
    torch.cuda.synchronize()
    for _x, _w, _b, ref, y, _st in cases:
        assert torch.equal(y, ref)
