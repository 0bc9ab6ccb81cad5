"""Group-wise products of 17 rows and more that fit the GPU at once (the weight-streaming kernel of
more rows than one MFMA holds) against the oracle, bit for bit, on the GPU: M at the edges of its row
blocks; groups of one MFMA piece and of two, and of five, which it leaves to the tiles; K of less
than a chunk, of a partial chunk and of many; each of its forms (16 and 32 rows a workgroup, one and two
a CU, two waves where the scales of four leave no room) and sizes past them; a last workgroup with
waves past N; per-row, per-group and mixed activation scales; grouped products of
uneven row counts."""
import ctypes as C

import numpy as np
import pytest

import gworder
import rocketnpu as R
from test_gpu_stream_gw import partials

pytestmark = pytest.mark.gpu
SEED = 0x52434D80

# 16 rows a workgroup; 32, and twice a CU; more than the GPU holds (tiles)
SHAPES = [(20, 64, 64, 32), (32, 128, 64, 128), (36, 608, 2112, 32), (64, 576, 192, 64), (68, 608, 128, 32), (200, 256, 64, 64),
          (24, 2048, 320, 256), (32, 640, 64, 160), (20, 12288, 64, 32),
          (60, 832, 4224, 64), (36, 512, 8256, 256), (40, 1152, 8320, 128), (64, 4096, 8256, 32), (64, 256, 16448, 64),
          (36, 160, 16448, 32), (132, 256, 16448, 64)]


@pytest.mark.parametrize("M,K,N,group", SHAPES)
@pytest.mark.parametrize("int4", [True, False])
def test_stream_gw_mid(lib, orc, M, K, N, group, int4):
    print(f"stream gw mid int4={int4} M={M} K={K} N={N} group={group}", flush=True)
    nG, kind = K // group, "i4" if int4 else "i8"
    A = orc.gen_i8((M, K), SEED + 1)
    B = orc.gen_i8((N, K), SEED + 2, -8, 7) if int4 else orc.gen_i8((N, K), SEED + 2)
    A[0, :], B[0, :] = -128, -8 if int4 else -128
    bsc = orc.gen_uniform((N, nG), SEED + 3, 0.005, 0.02)
    row = orc.gen_uniform((M,), SEED + 4, 0.5, 1.5)
    asc = orc.gen_uniform((M, nG), SEED + 5, 0.5, 1.5)
    asc[1::3] = asc[1::3, :1]   # rows of one scale among the others
    ctx = getattr(lib, f"rocket_{kind}_ctx_create")(1)
    w = getattr(lib, f"rocket_{kind}_weights_pack_gw")(ctx, 4, K, N, R.ptr(B), group)
    assert w
    call = lambda name, *a: getattr(lib, f"rocket_matmul_int{4 if int4 else 8}_prepacked_gw{name}")(ctx, M, K, N, *a, w)  # noqa: E731
    out = np.full((M, N), np.nan, np.float32)
    assert call("_rowscale", R.ptr(A), R.ptr(row), R.ptr(bsc), R.ptr(out)) == 0
    assert np.array_equal(out, orc.matmul_gw_rowscale_f32(A, B, row, bsc, group))
    plain = out.copy()
    out[:] = np.nan
    assert call("", R.ptr(A), R.ptr(asc), R.ptr(bsc), R.ptr(out)) == 0
    assert np.array_equal(out, gworder.gw_f32(orc, A, B, asc, bsc, group))
    # the same kernels with their partials dumped: a window of rows inside the blocks
    r0, nr = (13, 6) if M > 16 else (1, M - 2)
    want = partials(A[r0:r0 + nr], B, group)
    for name, scale, first in (("_rowscale_dump", row, plain), ("_dump", asc, out.copy())):
        P = np.full((nr, nG, N), 99, np.int32)
        out[:] = np.nan
        assert getattr(lib, f"rocket_matmul_int{4 if int4 else 8}_prepacked_gw{name}")(
            ctx, M, K, N, R.ptr(A), R.ptr(scale), R.ptr(bsc), R.ptr(out), w, r0, nr, R.ptr(P)) == 0
        assert np.array_equal(out, first) and np.array_equal(P, want)
    getattr(lib, f"rocket_{kind}_weights_free")(ctx, w)
    getattr(lib, f"rocket_{kind}_ctx_free")(ctx)


@pytest.mark.parametrize("Ms,K,N,group", [([4, 0, 64, 20], 512, 96, 32), ([32, 4, 24], 1408, 2048, 32), ([20] * 18, 256, 160, 64)])
def test_stream_gw_mid_grouped(lib, orc, Ms, K, N, group):
    n, nG = len(Ms), K // group
    print(f"stream gw mid grouped Ms={Ms} K={K} N={N} group={group}", flush=True)
    ctx = lib.rocket_i8_ctx_create(1)
    Bs = [orc.gen_i8((N, K), SEED + 20 + e) for e in range(n)]
    W = [lib.rocket_i8_weights_pack_gw(ctx, 4, K, N, R.ptr(b), group) for b in Bs]
    bs = [orc.gen_uniform((N, nG), SEED + 50 + e, 0.005, 0.02) for e in range(n)]
    A = [orc.gen_i8((max(m, 4), K), SEED + 80 + e) for e, m in enumerate(Ms)]
    rs = [orc.gen_uniform((max(m, 4),), SEED + 110 + e, 0.5, 1.5) for e, m in enumerate(Ms)]
    pM, k0 = R.int_array(Ms)
    pW = C.cast((C.c_void_p * n)(*W), R.pp)
    h = [np.full((max(m, 4), N), 0x7E00, np.uint16) for m in Ms]
    (pA, k1), (pr, k2), (pb, k3), (ph, k4) = R.ptr_array(A), R.ptr_array(rs), R.ptr_array(bs), R.ptr_array(h)
    assert lib.rocket_matmul_int8_prepacked_gw_grouped_rowscale_f16out(ctx, n, pM, K, N, pA, pr, pb, ph, pW) == 0
    for e, m in enumerate(Ms):
        if m:
            want = orc.matmul_gw_rowscale_f32(np.ascontiguousarray(A[e][:m]), Bs[e], np.ascontiguousarray(rs[e][:m]), bs[e], group)
            assert np.array_equal(h[e][:m], orc.f32_to_f16_bits(want))
    del k0, k1, k2, k3, k4
    for w in W:
        lib.rocket_i8_weights_free(ctx, w)
    lib.rocket_i8_ctx_free(ctx)
