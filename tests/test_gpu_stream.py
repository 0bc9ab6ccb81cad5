"""Products of at most 16 rows (the weight-streaming kernel): its edges against the oracle, on
the GPU. M = 1 and 16 are the ends of its range and M = 20 the first size past it; K covers less
than a step, a partial step, slices that leave waves idle and the 16-slice form (fp32 operands
from K = 8192, the gated pair from 2048); N = 12288 + 16 runs 32-column workgroups, the last of
them half empty. fp32 sums of K products are held to 1e-5 normalised error (K 2^-24 sqrt(K) is
below 2e-6 at K = 8224), integers to equality, fp16 results to the library's 1e-2."""
import ctypes as C

import numpy as np
import pytest

import rocketnpu as R

pytestmark = pytest.mark.gpu
SEED = 0x52434B60
SHAPES = [(1, 32, 32), (4, 96, 64), (12, 544, 96), (16, 1056, 160), (20, 544, 96), (16, 8224, 64), (8, 160, 12320)]


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_stream_float(lib, orc, fd, M, K, N):
    print(f"stream float M={M} K={K} N={N}", flush=True)
    A, B = orc.gen_normal((M, K), SEED + 1), orc.gen_normal((N, K), SEED + 2, 0, 0.02)
    out = np.full((M, N), np.nan, np.float32)
    assert lib.rocket_matmul_bf16(fd, M, K, N, R.ptr(A), R.ptr(B), R.ptr(out)) == 0
    assert orc.norm_err(out, orc.matmul_bf16(A, B)) < 1e-5
    out[:] = np.nan
    assert lib.rocket_matmul_tf32(fd, M, K, N, R.ptr(A), R.ptr(B), R.ptr(out)) == 0
    assert orc.norm_err(out, orc.matmul_tf32(A, B)) < 5e-5   # the low parts' product is dropped (<= 2^-14 each)
    A16, B16 = orc.f32_to_f16_bits(A), orc.f32_to_f16_bits(B)
    out[:] = np.nan
    assert lib.rocket_matmul_fp16_f32out(fd, M, K, N, R.ptr(A16), R.ptr(B16), R.ptr(out)) == 0
    want = orc.matmul_fp16_f32out(A16, B16)
    assert orc.norm_err(out, want) < 1e-5
    h = np.full((M, N), 0x7E00, np.uint16)
    assert lib.rocket_matmul_fp16(fd, M, K, N, R.ptr(A16), R.ptr(B16), R.ptr(h)) == 0
    assert np.array_equal(h, orc.f32_to_f16_bits(out))       # the fp32 result rounded once


@pytest.mark.parametrize("M,K,N", SHAPES)
def test_stream_integer(lib, orc, fd, M, K, N):
    """int8 and int4 (N a multiple of 64) to int32, the extreme values among them."""
    print(f"stream integer M={M} K={K} N={N}", flush=True)
    N = (N + 63) // 64 * 64
    A, B, B4 = orc.gen_i8((M, K), SEED + 3), orc.gen_i8((N, K), SEED + 4), orc.gen_i8((N, K), SEED + 5, -8, 7)
    A[0, :], B[0, :], B4[0, :] = -128, -128, -8
    out = np.full((M, N), 99, np.int32)
    assert lib.rocket_matmul_int8(fd, M, K, N, R.ptr(A), R.ptr(B), R.ptr(out)) == 0
    assert np.array_equal(out, orc.matmul_int8(A, B))
    assert lib.rocket_matmul_int4(fd, M, K, N, R.ptr(A), R.ptr(B4), R.ptr(out)) == 0
    assert np.array_equal(out, orc.matmul_int8(A, B4))


@pytest.mark.parametrize("M,H,I", [(1, 32, 32), (4, 96, 160), (16, 2080, 96), (12, 544, 8192)])
def test_stream_gated(lib, orc, fd, M, H, I):
    """The FFN block on few rows: gate and up in one launch, both activations."""
    for kind in (R.ROCKET_ACTIVATION_SILU, R.ROCKET_ACTIVATION_GELU):
        print(f"stream ffn M={M} H={H} I={I} kind={kind}", flush=True)
        x, Wg, Wu, Wd = (orc.f32_to_f16_bits(orc.gen_normal(s, SEED + 6 + i, 0, d)) for i, (s, d) in
                         enumerate((((M, H), 1.0), ((I, H), H ** -0.5), ((I, H), H ** -0.5), ((H, I), I ** -0.5))))
        out = np.full((M, H), 0x7E00, np.uint16)
        assert lib.rocket_ffn_fp16(fd, M, H, I, R.ptr(x), R.ptr(Wg), R.ptr(Wu), R.ptr(Wd), kind, R.ptr(out)) == 0
        want = np.empty((M, H), np.uint16)
        lib.rocket_ffn_ref_fp16(M, H, I, R.ptr(x), R.ptr(Wg), R.ptr(Wu), R.ptr(Wd), kind, R.ptr(want))
        assert orc.norm_err(orc.f16_bits_to_f32(out), orc.f16_bits_to_f32(want)) <= 1e-2


def test_stream_batch_and_rows_keep_their_bits(lib, orc, fd):
    """A row's bits depend on its own operands: alone, among 16 rows, in a batch of products, and
    with a wider N."""
    M, K, N, nb = 16, 1056, 128, 3
    A = [orc.f32_to_f16_bits(orc.gen_normal((M, K), SEED + 20 + i)) for i in range(nb)]
    B = [orc.f32_to_f16_bits(orc.gen_normal((N, K), SEED + 30 + i, 0, 0.02)) for i in range(nb)]
    out = [np.empty((M, N), np.uint16) for _ in range(nb)]
    arr = [R.ptr_array(x) for x in (A, B, out)]
    assert lib.rocket_matmul_fp16_batch(fd, M, K, N, nb, *[p for p, _ in arr]) == 0
    for i in range(nb):
        one = np.empty((M, N), np.uint16)
        assert lib.rocket_matmul_fp16(fd, M, K, N, R.ptr(A[i]), R.ptr(B[i]), R.ptr(one)) == 0
        assert np.array_equal(one, out[i])
    row = np.empty((1, N), np.uint16)
    assert lib.rocket_matmul_fp16(fd, 1, K, N, R.ptr(np.ascontiguousarray(A[0][3:4])), R.ptr(B[0]), R.ptr(row)) == 0
    assert np.array_equal(row[0], out[0][3])
    wide = np.concatenate(B * 40)   # 15360 columns
    big = np.empty((M, wide.shape[0]), np.uint16)
    assert lib.rocket_matmul_fp16(fd, M, K, wide.shape[0], R.ptr(A[0]), R.ptr(wide), R.ptr(big)) == 0
    assert np.array_equal(big[:, :N], out[0])


def test_stream_under_capture(lib, orc):
    """The launch records into a HIP graph; each replay, with eager work between, equals the
    eager result on the inputs of that moment."""
    torch = pytest.importorskip("torch")
    M, K, N = 4, 1056, 320
    fd = lib.rocket_open()
    stream = torch.cuda.Stream()
    assert lib.rocket_hip_set_stream(fd, C.c_void_p(stream.cuda_stream)) == 0
    assert lib.rocket_hip_set_mode(fd, R.ROCKET_HIP_ASYNC | R.ROCKET_HIP_DEVICE_OPERANDS) == 0
    gen = torch.Generator().manual_seed(7)
    new = lambda *s: torch.randn(*s, generator=gen).half().cuda()  # noqa: E731
    A, B = new(M, K), new(N, K)
    out, eager = (torch.empty(M, N, dtype=torch.float16, device="cuda") for _ in range(2))
    call = lambda o: lib.rocket_matmul_fp16(fd, M, K, N, R.ptr(A), R.ptr(B), R.ptr(o))  # noqa: E731
    torch.cuda.synchronize()
    assert call(eager) == 0
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        assert call(out) == 0
    for _ in range(3):
        A.copy_(new(M, K))
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            graph.replay()
        torch.cuda.synchronize()
        assert call(eager) == 0
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
    lib.rocket_close(fd)


@pytest.mark.parametrize("K,N", [(K, N) for K in (992, 1024, 1056, 1472, 2048, 4096, 8224) for N in (16, 208)] + [(1056, 16400)])
def test_fp16_rows_have_the_bits_of_larger_calls(lib, orc, fd, K, N):
    """A plain fp16 row's sum is one chain over K: the rows of a product of 100 rows (tiles) against
    calls of its first 1, 4, 16, 20, 32 (one wave a column block) and 64 rows, with fp32 results (every
    bit of the sum) and fp16 ones; K of whole sets of loads and of a part of one, and fewer sets than a
    wave keeps in flight."""
    print(f"fp16 rows K={K} N={N}", flush=True)
    M = 100
    # magnitudes over 2^16, so that the order of the sums shows
    A = orc.f32_to_f16_bits(orc.gen_normal((M, K), SEED + 50) * np.exp2(orc.gen_uniform((M, K), SEED + 52, -8.0, 8.0)))
    B = orc.f32_to_f16_bits(orc.gen_normal((N, K), SEED + 51, 0, 0.02))
    big = np.empty((M, N), np.float32)
    assert lib.rocket_matmul_fp16_f32out(fd, M, K, N, R.ptr(A), R.ptr(B), R.ptr(big)) == 0
    assert orc.norm_err(big, orc.matmul_fp16_f32out(A, B)) < 1e-5
    for m in (1, 4, 16, 20, 32, 64):
        out, h = np.full((m, N), np.nan, np.float32), np.empty((m, N), np.uint16)
        Am = np.ascontiguousarray(A[:m])
        assert lib.rocket_matmul_fp16_f32out(fd, m, K, N, R.ptr(Am), R.ptr(B), R.ptr(out)) == 0
        assert np.array_equal(out, big[:m]), m
        assert lib.rocket_matmul_fp16(fd, m, K, N, R.ptr(Am), R.ptr(B), R.ptr(h)) == 0
        assert np.array_equal(h, orc.f32_to_f16_bits(big[:m])), m
