"""Group-wise products of at most 16 rows (the weight-streaming kernel) against the oracle, bit
for bit, on the GPU: M = 4 to 16 and 20, the first size past it; groups of one MFMA piece, two, and
more or odd multiples; K of less than a ring slot, of a partial slot, and of many; few columns (K
split over the waves) and many (a wave a tile, the last workgroup not full); rows quantised in
the kernel (few elements a thread) and ahead; per-row, per-group and mixed activation scales."""
import ctypes as C

import numpy as np
import pytest

import gworder
import rocketnpu as R

pytestmark = pytest.mark.gpu
SEED = 0x52434B80



def partials(A, B, group):
    """P[m][g][n]: the sums of every group, below 2^24 for groups of up to 1023 and exact in fp32."""
    a, b = A.astype(np.float32), B.astype(np.float32)
    return np.stack([a[:, k:k + group] @ b[:, k:k + group].T for k in range(0, A.shape[1], group)], 1).astype(np.int32)


SHAPES = [(4, 64, 64, 32), (4, 128, 64, 128), (8, 608, 128, 32), (16, 576, 192, 64), (20, 608, 128, 32), (12, 768, 128, 96),
          (4, 2048, 128, 256), (16, 2048, 64, 512), (16, 4096, 64, 32), (4, 8448, 64, 128), (8, 256, 8256, 32),
          (12, 1152, 8320, 128), (16, 512, 8256, 64), (4, 640, 8256, 160)]


@pytest.mark.parametrize("M,K,N,group", SHAPES)
@pytest.mark.parametrize("int4", [True, False])
def test_stream_gw(lib, orc, M, K, N, group, int4):
    print(f"stream gw int4={int4} M={M} K={K} N={N} group={group}", flush=True)
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
    x = orc.gen_normal((M, K), SEED + 6)
    x[2] = 0.0                  # a row of zeros: codes and scale 0
    q, s = orc.quant_rows(x)
    out[:] = np.nan
    assert call("_f32in", R.ptr(x), R.ptr(bsc), R.ptr(out)) == 0
    assert np.array_equal(out, orc.matmul_gw_rowscale_f32(q, B, s, bsc, group))
    getattr(lib, f"rocket_{kind}_weights_free")(ctx, w)
    getattr(lib, f"rocket_{kind}_ctx_free")(ctx)


@pytest.mark.parametrize("Ms,K,N,group", [([4, 0, 16, 8], 512, 96, 32), ([12, 4, 4], 1408, 2048, 32), ([4] * 18, 256, 160, 64),
                                          ([4, 8], 8224, 64, 32)])
def test_stream_gw_grouped(lib, orc, Ms, K, N, group):
    """Grouped products of few rows, more than a launch holds among them: fp16 results, and down
    products on gate * up rows that the kernel forms and quantises (gates in [18, 30], where SiLU
    returns its argument exactly, so the oracle's codes are the kernel's)."""
    n, nG = len(Ms), K // group
    print(f"stream gw grouped Ms={Ms} K={K} N={N} group={group}", flush=True)
    ctx = lib.rocket_i8_ctx_create(1)
    Bs = [orc.gen_i8((N, K), SEED + 20 + e) for e in range(n)]
    W = [lib.rocket_i8_weights_pack_gw(ctx, 4, K, N, R.ptr(b), group) for b in Bs]
    bs = [orc.gen_uniform((N, nG), SEED + 50 + e, 0.005, 0.02) for e in range(n)]
    A = [orc.gen_i8((max(m, 4), K), SEED + 80 + e) for e, m in enumerate(Ms)]
    rs = [orc.gen_uniform((max(m, 4),), SEED + 110 + e, 0.5, 1.5) for e, m in enumerate(Ms)]
    pM, k0 = R.int_array(Ms)
    pW = C.cast((C.c_void_p * n)(*W), R.pp)
    arr = lambda xs: R.ptr_array(xs)  # noqa: E731
    (pA, k1), (pr, k2), (pb, k3) = arr(A), arr(rs), arr(bs)
    h = [np.full((max(m, 4), N), 0x7E00, np.uint16) for m in Ms]
    ph, k4 = arr(h)
    assert lib.rocket_matmul_int8_prepacked_gw_grouped_rowscale_f16out(ctx, n, pM, K, N, pA, pr, pb, ph, pW) == 0
    for e, m in enumerate(Ms):
        if m:
            want = orc.matmul_gw_rowscale_f32(np.ascontiguousarray(A[e][:m]), Bs[e], np.ascontiguousarray(rs[e][:m]), bs[e], group)
            assert np.array_equal(h[e][:m], orc.f32_to_f16_bits(want))
    G = [orc.f32_to_f16_bits(orc.gen_uniform((max(m, 4), K), SEED + 140 + e, 18.0, 30.0)) for e, m in enumerate(Ms)]
    U = [orc.f32_to_f16_bits(orc.gen_normal((max(m, 4), K), SEED + 170 + e)) for e, m in enumerate(Ms)]
    out = [np.full((max(m, 4), N), np.nan, np.float32) for m in Ms]
    (pG, k5), (pU, k6), (po, k7) = arr(G), arr(U), arr(out)
    assert lib.rocket_matmul_int8_prepacked_gw_grouped_glu_f16in(ctx, n, pM, K, N, pG, pU, R.ROCKET_ACTIVATION_SILU, pb, po, pW) == 0
    for e, m in enumerate(Ms):
        if m:
            x = (orc.f16_bits_to_f32(G[e][:m]) * orc.f16_bits_to_f32(U[e][:m])).astype(np.float32)
            q, s = orc.quant_rows(x)
            assert np.array_equal(out[e][:m], orc.matmul_gw_rowscale_f32(q, Bs[e], s, bs[e], group))
    del k0, k1, k2, k3, k4, k5, k6, k7
    for w in W:
        lib.rocket_i8_weights_free(ctx, w)
    lib.rocket_i8_ctx_free(ctx)


@pytest.mark.parametrize("Ms,group", [([4, 0, 16, 8], 32), ([4, 20, 32], 64)])
def test_few_rows_grouped_dump(lib, orc, Ms, group):
    """Windows of some products of a grouped launch and none of the others, few rows and more."""
    K, N, n = 512, 96, len(Ms)
    print(f"few rows grouped dump Ms={Ms} group={group}", flush=True)
    nG = K // group
    ctx = lib.rocket_i8_ctx_create(1)
    Bs, A = [orc.gen_i8((N, K), SEED + 200 + e) for e in range(n)], [orc.gen_i8((max(m, 4), K), SEED + 220 + e) for e, m in enumerate(Ms)]
    W = [lib.rocket_i8_weights_pack_gw(ctx, 4, K, N, R.ptr(b), group) for b in Bs]
    bs = [orc.gen_uniform((N, nG), SEED + 240 + e, 0.005, 0.02) for e in range(n)]
    rs = [orc.gen_uniform((max(m, 4),), SEED + 260 + e, 0.5, 1.5) for e, m in enumerate(Ms)]
    out, P = [np.full((max(m, 4), N), np.nan, np.float32) for m in Ms], [np.full((3, nG, N), 99, np.int32) for _ in Ms]
    r0, nr = [1] * n, [3 if e != 0 and m else 0 for e, m in enumerate(Ms)]
    pW = C.cast((C.c_void_p * n)(*W), R.pp)
    (pM, k0), (pr0, k1), (pnr, k2) = R.int_array(Ms), R.int_array(r0), R.int_array(nr)
    (pA, k3), (pr, k4), (pb, k5), (po, k6), (pP, k7) = (R.ptr_array(x) for x in (A, rs, bs, out, P))
    assert lib.rocket_matmul_int8_prepacked_gw_grouped_rowscale_dump(ctx, n, pM, K, N, pA, pr, pb, po, pW, pr0, pnr, pP) == 0
    for e, m in enumerate(Ms):
        if m:
            assert np.array_equal(out[e][:m], orc.matmul_gw_rowscale_f32(np.ascontiguousarray(A[e][:m]), Bs[e],
                                                                         np.ascontiguousarray(rs[e][:m]), bs[e], group))
        want = partials(A[e], Bs[e], group)[1:4] if nr[e] else 99
        assert np.all(P[e] == want)
    del k0, k1, k2, k3, k4, k5, k6, k7
    for w in W:
        lib.rocket_i8_weights_free(ctx, w)
    lib.rocket_i8_ctx_free(ctx)


@pytest.mark.parametrize("M,K,N,group", [(4, 1536, 64, 128), (8, 2560, 192, 128), (4, 1536, 8256, 128), (20, 1536, 64, 128), (12, 640, 64, 64)])
@pytest.mark.parametrize("int4", [True, False])
def test_infinite_activation_scales(lib, orc, M, K, N, group, int4):
    """An infinite scale of one group (the last, where the groups are no multiple of eight; the first; one
    row's only scale) gives the chain's infinities, and no NaN where the chain has none."""
    print(f"infinite scales int4={int4} M={M} K={K} N={N} group={group}", flush=True)
    nG, kind = K // group, "i4" if int4 else "i8"
    A, B = orc.gen_i8((M, K), SEED + 300, 1, 127), orc.gen_i8((N, K), SEED + 301, 1, 7)     # partials above 0
    bsc = orc.gen_uniform((N, nG), SEED + 302, 0.005, 0.02)
    asc = orc.gen_uniform((M, nG), SEED + 303, 0.5, 1.5)
    asc[0, -1], asc[1, 0], asc[2, :] = np.inf, np.inf, np.inf
    want = gworder.gw_f32(orc, A, B, asc, bsc, group)
    assert np.isinf(want[:3]).all() and np.isfinite(want[3:]).all()
    ctx = getattr(lib, f"rocket_{kind}_ctx_create")(1)
    w = getattr(lib, f"rocket_{kind}_weights_pack_gw")(ctx, 4, K, N, R.ptr(B), group)
    out = np.full((M, N), np.nan, np.float32)
    fn = getattr(lib, f"rocket_matmul_int{4 if int4 else 8}_prepacked_gw")
    assert fn(ctx, M, K, N, R.ptr(A), R.ptr(asc), R.ptr(bsc), R.ptr(out), w) == 0
    assert np.array_equal(out, want)
    getattr(lib, f"rocket_{kind}_weights_free")(ctx, w)
    getattr(lib, f"rocket_{kind}_ctx_free")(ctx)
