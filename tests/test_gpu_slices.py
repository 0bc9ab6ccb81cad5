"""fp16, bf16 and tf32 products of 17 rows up that run in K slices of small tiles (by estimated
time), on the GPU: few rows and few columns with long K, partial tiles and a partial last slice.
Small integers make every fp32 sum exact, so the result equals float64 BLAS bit for bit whatever
the slicing; converting fp32 operands ahead of the product changes no bit of it on random values.
Plain fp16 products are not sliced by the estimate: an item of a batch, a segment of a fused call and
a row of a smaller call have the bits of the product by itself."""
import os

import numpy as np
import pytest

import rocketnpu as R

pytestmark = pytest.mark.gpu
SEED = 0x52434BC0
SHAPES = [(20, 2080, 1024), (100, 8192, 256), (300, 5984, 816), (700, 2528, 272), (64, 4096, 2064), (256, 3104, 1040), (300, 15360, 96)]


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_sliced_products_exact(lib, orc, fd, M, K, N):
    print(f"sliced M={M} K={K} N={N}", flush=True)
    A = orc.gen_i8((M, K), SEED + 1, -1, 1).astype(np.float32)
    B = orc.gen_i8((N, K), SEED + 2, -1, 1).astype(np.float32)
    want = A.astype(np.float64) @ B.astype(np.float64).T        # |sum| <= K < 2^24: exact in fp32
    out = np.empty((M, N), np.float32)
    for fn in (lib.rocket_matmul_bf16, lib.rocket_matmul_tf32):
        out[:] = np.nan
        assert fn(fd, M, K, N, R.ptr(A), R.ptr(B), R.ptr(out)) == 0
        assert np.array_equal(out, want)
    A16, B16 = orc.f32_to_f16_bits(A), orc.f32_to_f16_bits(B)
    out[:] = np.nan
    assert lib.rocket_matmul_fp16_f32out(fd, M, K, N, R.ptr(A16), R.ptr(B16), R.ptr(out)) == 0
    assert np.array_equal(out, want)
    h = np.empty((M, N), np.uint16)
    assert lib.rocket_matmul_fp16(fd, M, K, N, R.ptr(A16), R.ptr(B16), R.ptr(h)) == 0
    assert np.array_equal(h, want.astype(np.float16).view(np.uint16))


@pytest.mark.parametrize("M,K,N", [(100, 8192, 512), (700, 2528, 400), (256, 4096, 1040)])
def test_sliced_products_prepass_bits(lib, orc, fd, M, K, N, monkeypatch):
    A, B = orc.gen_normal((M, K), SEED + 3), orc.gen_normal((N, K), SEED + 4, 0, 0.02)
    for name, fn, ref, tol in (("bf16", lib.rocket_matmul_bf16, orc.matmul_bf16, 1e-5), ("tf32", lib.rocket_matmul_tf32, orc.matmul_tf32, 5e-5)):
        outs = []
        for mode in (None, "0", "1", "2"):
            if mode is None:
                monkeypatch.delenv("ROCKET_HIP_F32_PREPASS", raising=False)
            else:
                monkeypatch.setenv("ROCKET_HIP_F32_PREPASS", mode)
            out = np.full((M, N), np.nan, np.float32)
            assert fn(fd, M, K, N, R.ptr(A), R.ptr(B), R.ptr(out)) == 0
            outs.append(out)
        for o in outs[1:]:
            assert np.array_equal(o, outs[0]), name
        rows = np.r_[0:4, M - 4:M]
        assert orc.norm_err(np.ascontiguousarray(outs[0][rows]), ref(np.ascontiguousarray(A[rows]), B)) < tol


def test_sliced_products_off(lib, orc, fd, monkeypatch):
    """ROCKET_HIP_SPLITK=1 keeps one chain over K; the results agree within fp32 rounding."""
    M, K, N = 100, 8192, 256
    A, B = (orc.gen_normal(s, SEED + 5 + i) for i, s in enumerate(((M, K), (N, K))))
    one, many = np.empty((M, N), np.float32), np.empty((M, N), np.float32)
    assert lib.rocket_matmul_bf16(fd, M, K, N, R.ptr(A), R.ptr(B), R.ptr(many)) == 0
    monkeypatch.setenv("ROCKET_HIP_SPLITK", "1")
    assert lib.rocket_matmul_bf16(fd, M, K, N, R.ptr(A), R.ptr(B), R.ptr(one)) == 0
    assert os.environ["ROCKET_HIP_SPLITK"] == "1" and not np.array_equal(one, many)
    assert orc.norm_err(one, many) < 1e-5


@pytest.mark.parametrize("M,K,N,nb", [(64, 4096, 512, 3), (20, 2080, 1024, 17), (100, 8192, 96, 2)])
def test_fp16_items_and_segments_keep_their_bits(lib, orc, fd, M, K, N, nb):
    """A batch's items and a fused call's segments against the product of each by itself, at sizes whose
    fp32 counterparts run in slices; 17 items are two launches, the second of one item."""
    print(f"fp16 items M={M} K={K} N={N} nb={nb}", flush=True)
    A = [orc.f32_to_f16_bits(orc.gen_normal((M, K), SEED + 40 + i)) for i in range(nb)]
    B = [orc.f32_to_f16_bits(orc.gen_normal((N, K), SEED + 60 + i, 0, 0.02)) for i in range(nb)]
    one, out = [np.empty((M, N), np.uint16) for _ in range(nb)], [np.empty((M, N), np.uint16) for _ in range(nb)]
    for i in range(nb):
        assert lib.rocket_matmul_fp16(fd, M, K, N, R.ptr(A[i]), R.ptr(B[i]), R.ptr(one[i])) == 0
    arr = [R.ptr_array(x) for x in (A, B, out)]
    assert lib.rocket_matmul_fp16_batch(fd, M, K, N, nb, *[p for p, _ in arr]) == 0
    for i in range(nb):
        assert np.array_equal(out[i], one[i])
    s = lib.rocket_stream_create(1)
    segs = [B[0], np.ascontiguousarray(B[1][:16])]
    (pB, k0), (pN, k1) = R.ptr_array(segs), R.int_array([N, 16])
    fused = np.empty((M, N + 16), np.uint16)
    assert lib.rocket_matmul_fp16_stream_fused(s, M, K, pB, pN, 2, R.ptr(A[0]), R.ptr(fused)) == 0
    lib.rocket_stream_free(s)
    del k0, k1
    last = np.empty((M, 16), np.uint16)
    assert lib.rocket_matmul_fp16(fd, M, K, 16, R.ptr(A[0]), R.ptr(segs[1]), R.ptr(last)) == 0
    assert np.array_equal(fused[:, :N], one[0]) and np.array_equal(fused[:, N:], last)
