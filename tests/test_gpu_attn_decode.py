"""Attention of few query rows (at most 16 of a KV head) and V^T rows read in place, against the
oracle on the GPU: one key chunk to many splits, every remainder of a chunk and of eight keys, head
sizes that fill the compiled ones and that do not, 1 to 16 rows from tokens and grouped heads and
17, the first size past them, masks of every alignment, soft-cap, and scores that grow along the
keys (the running maximum moves in every chunk). Bar: the library's, cosine >= 0.9995 and 2e-2
normalised maximum error (fp16 results and probabilities)."""
import numpy as np
import pytest

import rocketnpu as R

pytestmark = pytest.mark.gpu
SEED = 0x52434BA0

CASES = [  # T, n_kv, dk, dv, heads, kv heads, masked, softcap
    (1, 8, 64, 64, 1, 1, False, 0.0), (1, 9, 32, 16, 2, 1, False, 0.0), (1, 31, 64, 64, 4, 4, False, 0.0),
    (1, 129, 128, 128, 8, 8, False, 0.0), (1, 3000, 256, 256, 4, 2, False, 0.0), (1, 8191, 128, 128, 4, 1, False, 0.0),
    (4, 1003, 256, 256, 4, 1, True, 0.0), (16, 333, 128, 128, 2, 2, True, 0.0), (3, 777, 96, 80, 10, 2, True, 50.0),
    (8, 2050, 192, 256, 4, 2, True, 0.0), (2, 70, 160, 224, 8, 1, True, 30.0), (17, 333, 128, 128, 2, 2, True, 0.0),
    (40, 1003, 64, 64, 2, 1, True, 0.0), (40, 1000, 128, 128, 2, 1, True, 0.0), (130, 1048, 256, 256, 2, 1, True, 0.0),
    (33, 7, 64, 64, 2, 1, False, 0.0),
]


def check(orc, got, want):
    g, w = orc.f16_bits_to_f32(got).astype(np.float64), orc.f16_bits_to_f32(want).astype(np.float64)
    assert np.isfinite(g).all()
    assert (g * w).sum() / np.sqrt((g * g).sum() * (w * w).sum()) >= 0.9995
    assert np.abs(g - w).max() / np.abs(w).max() <= 2e-2


@pytest.mark.parametrize("T,n,dk,dv,nh,kvh,masked,cap", CASES)
@pytest.mark.parametrize("grow", [False, True])
def test_attn_few_rows(lib, orc, fd, T, n, dk, dv, nh, kvh, masked, cap, grow):
    print(f"attn rows T={T} n_kv={n} dk={dk} dv={dv} heads={nh}/{kvh} mask={masked} cap={cap} grow={grow}", flush=True)
    f16 = orc.f32_to_f16_bits
    Q, K = orc.gen_normal((nh, T, dk), SEED + 1), orc.gen_normal((kvh, n, dk), SEED + 2)
    if grow:   # scores rise with the key
        Q = np.abs(Q)
        K = np.abs(K) * np.linspace(0.05, 1.0, n, dtype=np.float32)[None, :, None]
    Q, K, V = f16(Q), f16(K), f16(orc.gen_normal((kvh, dv, n), SEED + 3))
    M = None
    if masked:
        pos = n - T + np.arange(T)[:, None]
        M = f16(np.where(np.arange(n)[None, :] <= pos, orc.gen_uniform((T, n), SEED + 4, -1.0, 1.0), -np.inf).astype(np.float32))
    scale = float(dk ** -0.5)
    want = orc.flash_attn_f16(Q, K, V, M, scale, cap)
    out = np.full((nh, T, dv), 0x7E00, np.uint16)
    assert lib.rocket_flash_attn_fp16(fd, T, n, dk, dv, nh, kvh, scale, cap, R.ptr(Q), R.ptr(K), R.ptr(V), R.ptr(M), R.ptr(out)) == 0
    check(orc, out, want)


@pytest.mark.parametrize("T,n", [(1, 1000), (1, 1003), (40, 1000), (40, 1003)])
def test_attn_reads_no_other_row(lib, orc, fd, T, n):
    """V^T rows lie end to end: an infinity in one output dim's row (at its first key, where the
    row before's last chunk would read on) stays in that dim."""
    dk = dv = 64
    f16 = orc.f32_to_f16_bits
    Q, K, V = (f16(orc.gen_normal(s, SEED + 20 + i)) for i, s in enumerate(((2, T, dk), (1, n, dk), (1, dv, n))))
    out, ref = np.empty((2, T, dv), np.uint16), np.empty((2, T, dv), np.uint16)
    call = lambda v, o: lib.rocket_flash_attn_fp16(fd, T, n, dk, dv, 2, 1, 0.125, 0.0, R.ptr(Q), R.ptr(K), R.ptr(v), None, R.ptr(o))  # noqa: E731
    assert call(V, ref) == 0
    W = V.copy()
    W[0, 17, 0] = 0x7C00
    assert call(W, out) == 0
    keep = np.arange(dv) != 17
    assert np.array_equal(out[:, :, keep], ref[:, :, keep])
    assert np.isposinf(orc.f16_bits_to_f32(np.ascontiguousarray(out[:, :, 17]))).all()


@pytest.mark.parametrize("n,d,heads,kvh", [(192, 256, 16, 8), (448, 256, 16, 8), (448, 128, 32, 8), (3000, 256, 16, 8)])
def test_attn_few_rows_error(lib, orc, fd, n, d, heads, kvh):
    """The error against float64 is that of two roundings to fp16, the probabilities' and the result's,
    also where the keys are split: a rounding is 2.07e-4 (2^-11 / sqrt(3), times 0.736, the root mean
    square of 2^e / x over a log-uniform mantissa), two independent ones 2.93e-4, a third one (split
    outputs in fp16) would make 3.59e-4. Bar: 2.93e-4 and 4 %, the sampling of 4096 results. The same
    call again gives the same bits."""
    print(f"attn error n={n} d={d} heads={heads}/{kvh}", flush=True)
    Q, K, V = (orc.gen_normal(s, SEED + 30 + i).astype(np.float16) for i, s in enumerate(((heads, 1, d), (kvh, n, d), (kvh, d, n))))
    out, again = np.empty((heads, 1, d), np.uint16), np.empty((heads, 1, d), np.uint16)
    for o in (out, again):
        assert lib.rocket_flash_attn_fp16(fd, 1, n, d, d, heads, kvh, d ** -0.5, 0.0, R.ptr(Q), R.ptr(K), R.ptr(V), None, R.ptr(o)) == 0
    assert np.array_equal(out, again)
    q, k, v = (x.astype(np.float64) for x in (Q, K, V))
    k, v = np.repeat(k, heads // kvh, 0), np.repeat(v, heads // kvh, 0)
    s = np.matmul(q, k.transpose(0, 2, 1)) * d ** -0.5
    p = np.exp(s - s.max(2, keepdims=True))
    want = np.matmul(p / p.sum(2, keepdims=True), v.transpose(0, 2, 1))
    rel = np.linalg.norm(out.view(np.float16).astype(np.float64) - want) / np.linalg.norm(want)
    print(f"  rel {rel:.3e}", flush=True)
    assert rel <= 3.05e-4
