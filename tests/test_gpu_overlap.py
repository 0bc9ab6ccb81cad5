"""Calls whose results lie over their own rows, and calls recorded into a HIP graph on a handle that
has no scratch yet, on the GPU: rows that a pass of their own reads (quantised fp32 rows, converted
fp32 operands) are all read before the first result is stored, for few rows as for many; and a
product or an attention that would take scratch for K slices or key splits runs without them."""
import numpy as np
import pytest

import rocketnpu as R

pytestmark = pytest.mark.gpu
SEED = 0x52434F80
DEV = "cuda:0"


def _handle(lib, fd, stream):
    assert lib.rocket_hip_set_stream(fd, R.ptr(stream.cuda_stream)) == 0
    assert lib.rocket_hip_set_mode(fd, R.ROCKET_HIP_ASYNC | R.ROCKET_HIP_DEVICE_OPERANDS) == 0


@pytest.mark.parametrize("M", [4, 16, 64])
@pytest.mark.parametrize("noalloc", [False, True])
def test_quantised_rows_under_results(lib, orc, M, noalloc):
    import torch
    K = N = 1024
    group = 128
    print(f"quantised rows under results M={M} noalloc={noalloc}", flush=True)
    B = orc.gen_i8((N, K), SEED + 1, -8, 7)
    bsc = orc.gen_uniform((N, K // group), SEED + 2, 0.005, 0.02)
    x = orc.gen_normal((M, K), SEED + 3)
    ctx = lib.rocket_i4_ctx_create(1)
    w = lib.rocket_i4_weights_pack_gw(ctx, M, K, N, R.ptr(B), group)
    assert w
    fn = getattr(lib, "rocket_matmul_int4_prepacked_gw_f32in" + ("_noalloc" if noalloc else ""))
    q, s = orc.quant_rows(x)
    want = orc.matmul_gw_rowscale_f32(q, B, s, bsc, group)
    stream = torch.cuda.Stream()
    _handle(lib, lib.rocket_i4_ctx_fd(ctx), stream)
    with torch.cuda.stream(stream):
        dx, dbs = torch.from_numpy(x).to(DEV), torch.from_numpy(bsc).to(DEV)
        assert fn(ctx, M, K, N, R.ptr(dx), R.ptr(dbs), R.ptr(dx), w) == 0
        got = dx.cpu().numpy()
    assert np.array_equal(got, want)
    lib.rocket_i4_weights_free(ctx, w)
    lib.rocket_i4_ctx_free(ctx)


@pytest.mark.parametrize("M", [4, 16, 64, 300])
@pytest.mark.parametrize("math", ["bf16", "tf32"])
def test_converted_rows_under_results(lib, orc, M, math):
    import torch
    K = N = 512
    print(f"converted rows under results M={M} {math}", flush=True)
    x, B = orc.gen_normal((M, K), SEED + 4), orc.gen_normal((N, K), SEED + 5)
    fd = lib.rocket_open()
    stream = torch.cuda.Stream()
    _handle(lib, fd, stream)
    fn = getattr(lib, "rocket_matmul_" + math)
    # both operands truncated to the entry's mantissa, products exact in fp32, sums of K terms
    cut = np.uint32(0xFFFF0000 if math == "bf16" else 0xFFFFE000)
    t = lambda a: (a.view(np.uint32) & cut).view(np.float32).astype(np.float64)  # noqa: E731
    want, mag = t(x) @ t(B).T, np.abs(t(x)) @ np.abs(t(B)).T
    with torch.cuda.stream(stream):
        dx, dB = torch.from_numpy(x).to(DEV), torch.from_numpy(B).to(DEV)
        assert fn(fd, M, K, N, R.ptr(dx), R.ptr(dB), R.ptr(dx)) == 0
        got = dx.cpu().numpy().astype(np.float64)
    # three products a term at tf32: (3 K + 1) roundings of 2^-24 of the terms' magnitudes at most
    assert np.all(np.abs(got - want) <= (3 * K + 1) * 2.0 ** -24 * mag)
    lib.rocket_close(fd)


@pytest.mark.parametrize("op", ["fp16", "attn"])
def test_capture_on_a_fresh_handle(lib, orc, monkeypatch, op):
    import torch
    print(f"capture on a fresh handle {op}", flush=True)
    stream = torch.cuda.Stream()
    h = lambda shape, k, sc=1.0: torch.from_numpy((orc.gen_normal(shape, SEED + k) * sc).astype(np.float16)).to(DEV)  # noqa: E731
    if op == "fp16":
        M, K, N = 64, 4096, 1024
        a, b = h((M, K), 6), h((N, K), 7)
        out = torch.empty((M, N), dtype=torch.float16, device=DEV)
        call = lambda fd: lib.rocket_matmul_fp16(fd, M, K, N, R.ptr(a), R.ptr(b), R.ptr(out))  # noqa: E731
    else:
        H, n, d = 8, 1024, 128
        a, b, v = h((H, 1, d), 8), h((H, n, d), 9), h((H, d, n), 10)
        out = torch.empty((H, 1, d), dtype=torch.float16, device=DEV)
        call = lambda fd: lib.rocket_flash_attn_fp16(fd, 1, n, d, d, H, H, d ** -0.5, 0.0, R.ptr(a), R.ptr(b), R.ptr(v),  # noqa: E731
                                                     None, R.ptr(out))
    torch.cuda.synchronize()
    # eager first, on another handle, with slices and without: the kernels' one-time set-up
    warm = lib.rocket_open()
    _handle(lib, warm, stream)
    assert call(warm) == 0
    monkeypatch.setenv("ROCKET_HIP_SPLITK", "1")
    assert call(warm) == 0
    monkeypatch.delenv("ROCKET_HIP_SPLITK")
    stream.synchronize()
    eager = out.float().cpu().numpy()
    fd = lib.rocket_open()
    _handle(lib, fd, stream)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        rc = call(fd)
    assert rc == 0
    for _ in range(3):
        with torch.cuda.stream(stream):
            out.fill_(float("nan"))
        stream.synchronize()
        g.replay()
        stream.synchronize()
        got = out.float().cpu().numpy()
        # fp32 sums in another order (and split outputs held in fp16): a rounding or two of fp16, of the
        # largest value where terms cancel
        assert np.max(np.abs(got - eager)) <= 2.0 ** -9 * np.max(np.abs(eager))
    del g
    lib.rocket_close(warm)
    lib.rocket_close(fd)


@pytest.mark.parametrize("M,K,N", [(4, 512, 64), (16, 992, 32), (20, 1024, 64), (64, 512, 64)])
def test_one_tile_in_place(lib, orc, M, K, N):
    """Products that one 64 x 64 tile holds, with their results over their own rows or weights: int8,
    group-wise (int8 with scales per row), fp16 and bf16."""
    import torch
    print(f"one tile in place M={M} K={K} N={N}", flush=True)
    N64 = (N + 63) // 64 * 64
    A, B = orc.gen_i8((M, K), SEED + 20), orc.gen_i8((N64, K), SEED + 21)
    rs, bs = orc.gen_uniform((M,), SEED + 22, 0.5, 1.5), orc.gen_uniform((N64, K // 32), SEED + 23, 0.005, 0.02)
    x, W = orc.gen_normal((M, K), SEED + 24), orc.gen_normal((N, K), SEED + 25, 0, 0.02)
    x16, W16 = (orc.f32_to_f16_bits(v).view(np.float16) for v in (x, W))
    fd, ctx = lib.rocket_open(), lib.rocket_i8_ctx_create(1)
    stream = torch.cuda.Stream()
    for f in (fd, lib.rocket_i8_ctx_fd(ctx)):
        _handle(lib, f, stream)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
    with torch.cuda.stream(stream):
        if N == N64:
            for over in (0, 1):
                a, b = dev(A), dev(B)
                c = (a, b)[over]
                if c.numel() < M * N * 4:
                    continue
                assert lib.rocket_matmul_int8(fd, M, K, N, R.ptr(a), R.ptr(b), R.ptr(c)) == 0
                got = c.flatten()[:M * N * 4].cpu().numpy().view(np.int32).reshape(M, N)
                assert np.array_equal(got, orc.matmul_int8(A, B))
            w = lib.rocket_i8_weights_pack_gw(ctx, M, K, N, R.ptr(B), 32)
            a, r, s = dev(A), dev(rs), dev(bs)
            if M * K >= M * N * 4:
                assert lib.rocket_matmul_int8_prepacked_gw_rowscale(ctx, M, K, N, R.ptr(a), R.ptr(r), R.ptr(s), R.ptr(a), w) == 0
                got = a.flatten()[:M * N * 4].cpu().numpy().view(np.float32).reshape(M, N)
                assert np.array_equal(got, orc.matmul_gw_rowscale_f32(A, B, rs, bs, 32))
            lib.rocket_i8_weights_free(ctx, w)
        a, b = dev(x16), dev(W16)
        assert lib.rocket_matmul_fp16(fd, M, K, N, R.ptr(a), R.ptr(b), R.ptr(a)) == 0
        got = a.flatten()[:M * N].cpu().numpy().astype(np.float32).reshape(M, N)
        want = orc.matmul_fp16_f32out(x16.view(np.uint16), W16.view(np.uint16))
        assert orc.norm_err(got, want) < 1e-3        # rounded to fp16
        a, b = dev(x), dev(W)
        assert lib.rocket_matmul_bf16(fd, M, K, N, R.ptr(a), R.ptr(b), R.ptr(a)) == 0
        assert orc.norm_err(a.flatten()[:M * N].cpu().numpy().reshape(M, N), orc.matmul_bf16(x, W)) < 1e-5
    lib.rocket_i8_ctx_free(ctx)
    lib.rocket_close(fd)


def test_attention_over_its_values(lib, orc):
    """Results over V, whose ragged rows are copied first: eight heads over 100 keys."""
    import torch
    H, n, d = 8, 100, 64
    q, k, v = (orc.f32_to_f16_bits(orc.gen_normal(s, SEED + 30 + i)) for i, s in enumerate(((H, 1, d), (H, n, d), (H, d, n))))
    fd = lib.rocket_open()
    stream = torch.cuda.Stream()
    _handle(lib, fd, stream)
    with torch.cuda.stream(stream):
        dq, dk, dv = (torch.from_numpy(t.view(np.float16)).to(DEV) for t in (q, k, v))
        assert lib.rocket_flash_attn_fp16(fd, 1, n, d, d, H, H, d ** -0.5, 0.0, R.ptr(dq), R.ptr(dk), R.ptr(dv), None, R.ptr(dv)) == 0
        got = dv.flatten()[:H * d].cpu().numpy().astype(np.float32).reshape(H, 1, d)
    want = orc.f16_bits_to_f32(orc.flash_attn_f16(q, k, v, None, d ** -0.5, 0.0))
    assert np.abs(got - want).max() <= 2e-2 * np.abs(want).max()
    lib.rocket_close(fd)
