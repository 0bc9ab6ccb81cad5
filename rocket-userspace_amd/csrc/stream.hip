// stream.hip — products of at most 16 rows, plain fp16 up to 32 (decode batches): the weight-streaming
// kernels.
//
// With so few activation rows a product reads every weight once and does little with it: what
// bounds it is how many bytes of B are in flight. The tiled kernels (gemm_impl.h) walk K in LDS
// stages with a barrier each, a chain of K / 64 stages of ~0.35 us whatever M is, on as many
// CUs as N / 64 gives. Here nothing is staged. A workgroup owns 16 columns (or 32) and the
// whole of K, each of its waves a slice of K, and every lane loads its MFMA fragments straight
// from global memory: B's rows as the second operand, the activations' rows (L2 serves them to
// every workgroup) as the first, one set of steps in flight while the other's MFMAs run. The
// waves' sums meet in LDS once, at the end, added in wave order. fp32 operands are truncated or
// split in registers, so no conversion pass runs first. The K slices depend on the formats and
// K alone: a row's bits do not depend on N, on M, or on the launch's other problems where this kernel
// runs (stream_takes leaves some of many columns to the tiles). Plain
// fp16 products, whose rows have the tiled kernels' bits, take k_chain instead: one wave, all of K.
//
// Measured (three sets of operands in turn; tiled kernels before, this kernel after):
//   int8     4 x  4096 x  4096    8.0 ->  5.8 us
//   bf16     4 x  4096 x  4096   29.1 -> 13.1 us   (fp32 operands, 5.1 TB/s)
//   tf32     4 x  4096 x  4096   46.8 -> 13.4 us
//   FFN      1 x  3840 x 15360  118.3 -> 68.0 us   (two launches, 5.2 TB/s)
// A copy of 4 GB runs at 4.9 TB/s (read + write). At 32 rows the activations' own fragments
// are twice the bytes of B's through each CU's L1, and the tiled kernels win over k_stream
// (fp16 32 x 3840 x 15360: 55.5 us here, 34.3 there). B loaded non-temporally was slower
// throughout (the FFN at one row 68 -> 86 us).
#include "gemm_impl.h"

namespace rk {
namespace gk {
namespace {


// A K step as one lane loads it: row l % 16 of its 16-row block, the l / 16-th quarter of the
// step's row bytes, R chunks of 16 bytes; K elements a step.
template <Fmt F> struct Raw;
template <> struct Raw<Fmt::F16> { static constexpr int R = 1, K = 32; };
template <> struct Raw<Fmt::BF16> { static constexpr int R = 1, K = 32; };
template <> struct Raw<Fmt::F32BF16> { static constexpr int R = 2, K = 32; };
template <> struct Raw<Fmt::F32TF32> { static constexpr int R = 2, K = 32; };
template <> struct Raw<Fmt::BF16X2> { static constexpr int R = 2, K = 32; };
template <> struct Raw<Fmt::I8> { static constexpr int R = 1, K = 64; };
template <> struct Raw<Fmt::I4P> { static constexpr int R = 1, K = 128; };

// A product's step is the larger of its operands' (packed int4 columns against int8 rows: one
// chunk against two, the same K elements lane by lane).
template <Fmt FA, Fmt FB> struct Step {
    static constexpr int K = Raw<FA>::K > Raw<FB>::K ? Raw<FA>::K : Raw<FB>::K;
    static constexpr int RA = Raw<FA>::R * (K / Raw<FA>::K), RB = Raw<FB>::R * (K / Raw<FB>::K);
    static constexpr int U = RA > 1 ? 2 : 4;   // steps a set: at most 32 registers an operand and set
};

struct SArgs {
    int N, K, nsteps, per;   // per: steps a wave
    uint32_t lda, ldb;
    int epi, act;
    int shift;               // int32 results: arithmetic shift (packed int4 carries x16)
    int M[kMaxProblems];
    const void *A[kMaxProblems], *B[kMaxProblems], *B2[kMaxProblems];
    void *C[kMaxProblems];
};

template <Fmt FA, Fmt FB, class Acc>
__device__ __forceinline__ Acc mma(const i32x4 *a, const i32x4 *b, Acc acc)
{
    if constexpr (FB == Fmt::I4P) {
        const i32x4 w = b[0];
        acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[0], i32x4{nib_hi(w[0]), nib_lo(w[0]), nib_hi(w[1]), nib_lo(w[1])},
                                                    acc, 0, 0, 0);
        return __builtin_amdgcn_mfma_i32_16x16x64_i8(a[1], i32x4{nib_hi(w[2]), nib_lo(w[2]), nib_hi(w[3]), nib_lo(w[3])},
                                                     acc, 0, 0, 0);
    } else if constexpr (FA == Fmt::I8) {
        return __builtin_amdgcn_mfma_i32_16x16x64_i8(a[0], b[0], acc, 0, 0, 0);
    } else if constexpr (FA == Fmt::F16) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a[0]), __builtin_bit_cast(f16x8, b[0]), acc,
                                                      0, 0, 0);
    } else if constexpr (FA == Fmt::F32BF16 || FA == Fmt::BF16) {
        i32x4 x = a[0], y = b[0];
        if constexpr (FA == Fmt::F32BF16) x = bf16x8_of(a[0], a[1]);
        if constexpr (FB == Fmt::F32BF16) y = bf16x8_of(b[0], b[1]);
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x), __builtin_bit_cast(bf16x8, y), acc, 0,
                                                       0, 0);
    } else {
        i32x4 xh = a[0], xl = a[1], yh = b[0], yl = b[1];
        if constexpr (FA == Fmt::F32TF32) tf32x8_split(a[0], a[1], xh, xl);
        if constexpr (FB == Fmt::F32TF32) tf32x8_split(b[0], b[1], yh, yl);
        const bf16x8 ah = __builtin_bit_cast(bf16x8, xh), al = __builtin_bit_cast(bf16x8, xl);
        const bf16x8 bh = __builtin_bit_cast(bf16x8, yh), bl = __builtin_bit_cast(bf16x8, yl);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh, acc, 0, 0, 0);
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl, acc, 0, 0, 0);
    }
}

// KS waves, NB 16-column blocks of B a workgroup (GLU: block 0 the gate's, block 1 the up
// weight's rows of the same 16 output columns). Register e of lane (q, r16) of a result block is
// row 4 q + e, column r16.
template <Fmt FA, Fmt FB, int KS, int NB, bool GLU>
__global__ __launch_bounds__(KS * 64, 4) void k_stream(const SArgs a)
{
    using St = Step<FA, FB>;
    constexpr int RA = St::RA, RB = St::RB, U = St::U;
    constexpr bool INT = FA == Fmt::I8;
    using Acc = std::conditional_t<INT, i32x4, f32x4>;
    using E = std::conditional_t<INT, int, float>;
    const int tid = threadIdx.x, lane = tid & 63, r16 = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int p = blockIdx.y, M = a.M[p];
    if (M == 0) return;
    const int n0 = (int)blockIdx.x * (GLU ? 16 : 16 * NB);
    const Rsrc ra = rsrc(a.A[p], (uint32_t)M * a.lda);   // rows past M lie past the range: zeros
    Rsrc rb[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) {
        const int n = GLU ? n0 : n0 + 16 * j;
        const char *src = static_cast<const char *>(GLU && j ? a.B2[p] : a.B[p]) + (size_t)n * a.ldb;
        rb[j] = rsrc(src, n < a.N ? 16u * a.ldb : 0u);   // N is a multiple of 16: whole blocks or none
    }
    const uint32_t oa = (uint32_t)r16 * a.lda + (uint32_t)q * (16u * RA), ob = (uint32_t)r16 * a.ldb + (uint32_t)q * (16u * RB);
    const int klane = q * (St::K / 4);   // first K element of the lane's quarter
    const int s0 = wave * a.per, s1 = min(a.nsteps, s0 + a.per);

    i32x4 fa[2][U][RA], fb[2][U][NB][RB];
    Acc acc[NB];
#pragma unroll
    for (int j = 0; j < NB; j++) acc[j] = Acc{};

    auto load = [&](auto SET, int s) __attribute__((always_inline)) {
        constexpr int t = decltype(SET)::value;
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int st = s + u;
            // past the slice, or a quarter past K (a multiple of the quarter's elements): zeros
            const uint32_t z = (st < s1 && st * St::K + klane < a.K) ? 0u : kOOB;
            const uint32_t ka = (oa + (uint32_t)st * (64u * RA)) | z, kb = (ob + (uint32_t)st * (64u * RB)) | z;
#pragma unroll
            for (int j = 0; j < NB; j++)
#pragma unroll
                for (int r = 0; r < RB; r++) fb[t][u][j][r] = ld16(rb[j], kb + 16u * r);
#pragma unroll
            for (int r = 0; r < RA; r++) fa[t][u][r] = ld16(ra, ka + 16u * r);
        }
    };
    auto step = [&](auto SET) __attribute__((always_inline)) {
        constexpr int t = decltype(SET)::value;
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int j = 0; j < NB; j++) acc[j] = mma<FA, FB>(fa[t][u], fb[t][u][j], acc[j]);
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    if (s0 < s1) {
        load(I0{}, s0);
        for (int s = s0; s < s1; s += 2 * U) {
            if (s + U < s1) load(I1{}, s + U);
            step(I0{});
            if (s + U < s1) {
                if (s + 2 * U < s1) load(I0{}, s + 2 * U);
                step(I1{});
            }
        }
    }

    // thread t of 256 holds output row m, column n of a block: the registers' own order, so the
    // LDS reads and writes are contiguous
    __shared__ E red[KS][NB][256];
#pragma unroll
    for (int j = 0; j < NB; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) red[wave][j][e * 64 + lane] = acc[j][e];
    __syncthreads();
    const int t = tid & 255, j = tid >> 8, m = 4 * ((t >> 4) & 3) + (t >> 6), n = n0 + (GLU ? 0 : 16 * j) + (t & 15);
    if (j >= (GLU ? 1 : NB) || m >= M || n >= a.N) return;
    E s = red[0][j][t];
#pragma unroll
    for (int w = 1; w < KS; w++) s += red[w][j][t];
    const size_t at = (size_t)m * a.N + n;
    if constexpr (INT) {
        static_cast<int32_t *>(a.C[p])[at] = s >> a.shift;
    } else if constexpr (GLU) {
        E u = red[0][NB - 1][t];
#pragma unroll
        for (int w = 1; w < KS; w++) u += red[w][NB - 1][t];
        const float g = a.act == kActGelu ? act_k<kActGelu>(s) : act_k<kActSilu>(s);
        static_cast<_Float16 *>(a.C[p])[at] = (_Float16)(g * u);
    } else if (a.epi == (int)Epi::F32) {
        static_cast<float *>(a.C[p])[at] = s;
    } else {
        if (a.epi == (int)Epi::ACT) {
            if (a.B2[p]) s += (float)static_cast<const _Float16 *>(a.B2[p])[n];
            if (a.act == kActGelu) s = act_k<kActGelu>(s);
            else if (a.act == kActSilu) s = act_k<kActSilu>(s);
        }
        static_cast<_Float16 *>(a.C[p])[at] = (_Float16)s;
    }
}

// Plain fp16 products: one chain over K in order, so that a row has the same bits among 16 rows, among
// 20 or 128 (tiles, whose 32x32x16 MFMAs sum 32 values of K to the same bits as one 16x16x32), and in
// a batch. A wave owns 16 NB columns, MB blocks of 16 rows and all of K; lane l loads row (or column)
// l % 16, halves 8 (l / 16) .. + 8 of a step of 32. What bounds it is the loads in flight, of which a wave
// can count 63: SETS sets of four steps' operands, each set loaded again as soon as its MFMAs are issued.
// Measured (start of this kernel: K in eight slices, k_stream; tiles): 4 x 4096 x 4096 9.9 us (8.0;
// 21.4), 4 x 2048 x 4096 6.3 (5.9; 12.7), 4 x 4096 x 16384 23.9 (30.3; 31.8), 20 x 4096 x 4096 13.5 (tiles 22.1).
constexpr int kChainSteps = 4;

template <int... I, class F> __device__ __forceinline__ void each(std::integer_sequence<int, I...>, F &&f)
{
    (f(std::integral_constant<int, I>{}), ...);
}

template <int MB, int NB, int SETS, bool F16OUT>
__global__ __launch_bounds__(64) void k_chain(const SArgs a)
{
    const int lane = threadIdx.x, r = lane & 15, q = lane >> 4;
    const int p = blockIdx.y, M = a.M[p], n0 = (int)blockIdx.x * 16 * NB;
    if (M == 0) return;
    const Rsrc ra = rsrc(a.A[p], (uint32_t)M * a.lda);   // rows past M and columns past N lie past the ranges: zeros
    const Rsrc rb = rsrc(static_cast<const char *>(a.B[p]) + (size_t)n0 * a.ldb, (uint32_t)min(16 * NB, a.N - n0) * a.ldb);
    const uint32_t o = (uint32_t)r * a.lda + (uint32_t)q * 16u, blk = 16u * a.lda;   // lda == ldb
    i32x4 fa[SETS][kChainSteps][MB], fb[SETS][kChainSteps][NB];
    f32x4 acc[MB][NB];
#pragma unroll
    for (int x = 0; x < MB; x++)
#pragma unroll
        for (int y = 0; y < NB; y++) acc[x][y] = f32x4{};
    auto load = [&](auto SET, int c) __attribute__((always_inline)) {
        constexpr int t = decltype(SET)::value;
#pragma unroll
        for (int i = 0; i < kChainSteps; i++) {
            const int st = c * kChainSteps + i;   // past K: zeros, whose MFMAs add nothing
            const uint32_t off = st < a.nsteps ? o + (uint32_t)st * 64u : kOOB;
#pragma unroll
            for (int y = 0; y < NB; y++) fb[t][i][y] = ld16(rb, off + y * blk);
#pragma unroll
            for (int x = 0; x < MB; x++) fa[t][i][x] = ld16(ra, off + x * blk);
        }
    };
    auto mma = [&](auto SET) __attribute__((always_inline)) {
        constexpr int t = decltype(SET)::value;
#pragma unroll
        for (int i = 0; i < kChainSteps; i++)
#pragma unroll
            for (int y = 0; y < NB; y++)
#pragma unroll
                for (int x = 0; x < MB; x++)
                    acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, fa[t][i][x]), __builtin_bit_cast(f16x8, fb[t][i][y]),
                                                                       acc[x][y], 0, 0, 0);
    };
    const int nch = (a.nsteps + kChainSteps - 1) / kChainSteps;
    using Sets = std::make_integer_sequence<int, SETS>;
    each(Sets{}, [&](auto S) __attribute__((always_inline)) { load(S, decltype(S)::value); });
    for (int c = 0; c < nch; c += SETS)
        each(Sets{}, [&](auto S) __attribute__((always_inline)) {
            constexpr int i = decltype(S)::value;
            if (c + i < nch) {
                mma(S);
                if (c + i + SETS < nch) load(S, c + i + SETS);
            }
        });
#pragma unroll
    for (int y = 0; y < NB; y++) {
        const int n = n0 + 16 * y + r;
        if (n >= a.N) continue;
#pragma unroll
        for (int x = 0; x < MB; x++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int m = 16 * x + 4 * q + e;
                if (m >= M) continue;
                const size_t at = (size_t)m * a.N + n;
                if constexpr (F16OUT) static_cast<_Float16 *>(a.C[p])[at] = (_Float16)acc[x][y][e];
                else static_cast<float *>(a.C[p])[at] = acc[x][y][e];
            }
    }
}

hipError_t launch_chain(SArgs &a, const Launch &L, uint64_t *blocks)
{
    a.nsteps = L.K / 32;
    int maxM = 0;
    for (int i = 0; i < L.nprob; i++) maxM = std::max(maxM, L.prob[i].M);
    auto go = [&](auto MB, auto NB, auto SETS) {
        constexpr int mb = decltype(MB)::value, nb = decltype(NB)::value, sets = decltype(SETS)::value;
        const dim3 grid((unsigned)((a.N + 16 * nb - 1) / (16 * nb)), (unsigned)L.nprob);
        *blocks = (uint64_t)grid.x * grid.y;
        if (L.epi == Epi::F16) hipLaunchKernelGGL((k_chain<mb, nb, sets, true>), grid, dim3(64), 0, L.stream, a);
        else hipLaunchKernelGGL((k_chain<mb, nb, sets, false>), grid, dim3(64), 0, L.stream, a);
    };
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I5 = std::integral_constant<int, 5>;
    using I7 = std::integral_constant<int, 7>;
    // two column blocks a wave share the rows' fragments where the columns still give a CU one and a half
    // waves (16 x 3072 x 16384 23.6 -> 19.8 us; 16 x 4096 x 8192 17.2 and 18.5), but for rows of 8 KB, of
    // which 32 at a time meet in the same channels (16 x 4096 x 16384: two 38.0, one 31.4; 16 x 4096 x 40960
    // 1.09 of the tiles' rate with one, 1.31 with two)
    if (maxM > 16) go(I2{}, I1{}, I5{});
    else if (maxM > 4 && a.N > 12288 && (a.ldb != 8192 || a.N > 20480)) go(I1{}, I2{}, I5{});
    else go(I1{}, I1{}, I7{});
    return hipGetLastError();
}

template <Fmt FA, Fmt FB, int KS> hipError_t launch_ks(SArgs &a, const Launch &L, uint64_t *blocks)
{
    a.per = (a.nsteps + KS - 1) / KS;
    // 32 columns a workgroup (the activations' fragments shared by two column blocks) from one and a half
    // of them a CU. K = 3840, N = 15360: int4 16 rows 12.2 -> 9.5 us, 4 rows 8.5 -> 8.0; bf16 65.7 ->
    // 52.9 and 47.0 -> 43.7. At N = 4096, half a workgroup a CU, it loses: int4 4.9 -> 5.7 and 3.9 -> 4.9,
    // bf16 16.1 -> 22.5 and 13.0 -> 19.0. (N = 8192 and 12288 go either way, 0.86 to 1.25 times.) fp32
    // rows are twice the bytes in flight a column: tf32, which splits each of them, keeps 16 from K = 1024
    // (4 x 3840 x 15360 47.5, wide 61.0; 8 x 3840 x 32768 105, 123), with more than 8 rows from K = 2048;
    // bf16 keeps 16 at N = 12288 from K > 1024, and where its rows are a power of two of 8 KB and more, of
    // which 32 at a time meet in the same channels (8 x 2048 x 12288 1.18 of the tiles' rate, wide 0.84; 4
    // x 4096 x 20480 1.45 and 1.13; 12 x 6144 x 16384 0.89 and 1.09); it takes 32 with more than 12 rows where 16
    // columns a workgroup are more than one a CU and less than two (16 x 6400 x 5120 0.90 and 1.18; 16 x 8192 x
    // 6144 0.93 and 1.16).
    const bool glu = L.epi == Epi::GLU;
    bool wide = !glu && a.N >= 12288;
    if (FB == Fmt::F32BF16 || FB == Fmt::F32TF32) {
        int maxM = 0;
        for (int i = 0; i < L.nprob; i++) maxM = std::max(maxM, a.M[i]);
        if (FB == Fmt::F32TF32) wide = wide && a.N > 12288 && (a.K < 1024 || (a.K < 2048 && maxM > 8));
        else wide = (wide && (a.K <= 1024 || (a.N > 12288 && (a.K < 2048 || (a.K & (a.K - 1)) != 0 || maxM > 12)))) ||
                    (a.N > 4096 && a.N <= 8192 && (KS == 16 ? maxM > 8 : maxM > 12 && a.K >= 4096));
    }
    const dim3 grid((unsigned)((a.N + (wide ? 31 : 15)) / (wide ? 32 : 16)), (unsigned)L.nprob);
    *blocks = (uint64_t)grid.x * grid.y;
    if (glu) {
        if constexpr (FA == Fmt::F16) hipLaunchKernelGGL((k_stream<FA, FB, KS, 2, true>), grid, dim3(KS * 64), 0, L.stream, a);
    } else if (wide) {
        hipLaunchKernelGGL((k_stream<FA, FB, KS, 2, false>), grid, dim3(KS * 64), 0, L.stream, a);
    } else {
        hipLaunchKernelGGL((k_stream<FA, FB, KS, 1, false>), grid, dim3(KS * 64), 0, L.stream, a);
    }
    return hipGetLastError();
}

template <Fmt FA, Fmt FB> hipError_t launch_fmt(SArgs &a, const Launch &L, uint64_t *blocks)
{
    a.nsteps = (L.K + Step<FA, FB>::K - 1) / Step<FA, FB>::K;
    // Sixteen K slices where a wave's slice then still spans four sets of loads: the fp32
    // operands from K = 8192 (tf32 4 x 8192 x 4096 40.1 -> 31.7 us; at K = 4096 they lose, 13.4 ->
    // 16.2) and the gated pair from K = 2048 (K = 3840, with the down product 71.1 -> 68.0 us).
    // Else eight: fp16 4 x 8192 x 4096 (a block's second product) 12.9 us with eight, 15.8 with sixteen.
    constexpr bool F32 = FA == Fmt::F32BF16 || FA == Fmt::F32TF32 || FB == Fmt::F32BF16 || FB == Fmt::F32TF32 || FB == Fmt::BF16X2 ||
                         FB == Fmt::BF16;
    if constexpr (F32 || FA == Fmt::F16)
        if (F32 ? L.K >= 8192 : (L.epi == Epi::GLU && L.K >= 2048)) return launch_ks<FA, FB, 16>(a, L, blocks);
    return launch_ks<FA, FB, 8>(a, L, blocks);
}

}  // namespace

bool stream_takes(const Launch &L, int maxM)
{
    const bool plain = L.fmt_a == Fmt::F16 && (L.epi == Epi::F16 || L.epi == Epi::F32);
    // Below K = 1024 a plain fp16 product's chain is short, and k_small_f16 takes most such products.
    if (plain && L.K < 1024) return false;
    // Plain fp16 over columns whose 64-wide blocks nearly fill the CUs twice: more than 8 rows (16 x 5120 x 28672
    // 77.8 us, tiles 63.0; 12 x 2560 x 28672 38.6 and 33.7; 16 x 2560 x 24576 0.91 of the tiles' time), 8 of long
    // rows (8 x 5120 x 28672 1.11 of it).
    if (one_chain(L) && L.nprob == 1 && L.N > 24576 && L.N <= 32768 && L.K >= 2560 && maxM > (L.K >= 4608 ? 4 : 8)) return false;
    // Rows of 8 KB (one column block a wave, launch_chain) over columns short of a round of tiles: 16 x 4096 x
    // 14336 30.1 us, tiles 26.2; 12 rows 27.9 and 26.3.
    if (one_chain(L) && L.nprob == 1 && L.K == 4096 && L.N > 12288 && L.N < 16384 && maxM > 8) return false;
    // One chain a wave serves 32 rows too, up to a wave a CU (20 x 4096 x 4096 13.5 us, tiles 22.1; 32 rows
    // 15.4 and 22.3). Past it 20 rows, and more of short rows, until the columns give the tiles half the CUs
    // (20 rows 1.03 to 1.16 of the tiles' rate at 5120 to 7936 columns, 32 rows 1.02 to 1.16 up to K = 1536,
    // 0.97 at 2048, 0.90 at 8704; K = 12288, 20 rows 0.95).
    const long cols = (long)L.nprob * L.N;
    const int most = !one_chain(L) || cols >= 8192 ? 16 : cols <= 4096 || L.K <= 1536 ? 32 : L.K <= 8704 ? 20 : 16;
    // int8 weights: the tiles' chain is the shorter one a byte, and they win where their 64-column blocks
    // fill the CUs or rows are many and long (16 x 8192 x 16384 28.7 us, tiles 24.0; 4 x 4096 x 16384 14.5 and
    // 13.3; 16 x 8192 x 8192 16.5 and 15.2; one and a half rounds of tiles 4 x 8192 x 24576 1.16 times as
    // long, a little more than that 12 x 4224 x 25536 25.4 and 21.5; 16 x 4224 x 9216 0.94 of the tiles' rate, 12 x
    // 4224 x 40960 0.87), and on short rows from 32768 columns (4 x 512 x 32768 7.0 and 6.1; 4 x 2048 1.13 times as long).
    if (L.fmt_b == Fmt::I8 && L.fmt_a == Fmt::I8) {
        const int blocks = (L.N + 63) / 64, last = blocks % 256;
        if (L.K > 2048 && blocks >= 192 && (last == 0 || last >= 192 || (blocks > 256 && last > 128))) return false;
        if (L.K >= 256 && L.K < 2048 && blocks > 384) return false;
        if ((long)maxM * L.K > (L.N > 32768 ? 50000 : L.N > 8192 ? 65000 : 100000) && L.N > 4096) return false;
    }
    // fp32 operands over many columns: the tiles on converted rows, whose 64-column blocks nearly fill the
    // CUs there. bf16, 16 rows: from K = 2048 (16 x 3840 x 12288 49.9 us, tiles 46.9; 16 x 2048 x 14336 30.0 and
    // 25.6; 16 x 3456 x 9216 38.0 and 34.2), but for K around 3072 (16 x 3072 x 20480 0.90 of the tiles' time); 12 rows at K = 2048; K = 8192 (8 x
    // 8192 x 14336 114 and 104). tf32: at 32768 columns (16 x 3840 x 32768 129 and 97; 4 rows 94 and 96).
    if (L.fmt_b == Fmt::F32BF16 && L.nprob == 1 && L.N > 8192 && L.N <= 28672 && L.K >= 1024) {
        if (L.N > 24576) {
            if (maxM > 8) return false;
        } else if (L.K >= 2048) {
            if (maxM > 12 && !(L.K >= 2560 && L.K < 3584 && L.N > 12288)) return false;
            if (maxM > 8 && L.K < 2560 && L.N > 12288 && L.N <= 16384) return false;
        }
        if (L.K >= 8192 && L.N > 12288) return false;
    }
    if (L.fmt_b == Fmt::F32TF32 && L.nprob == 1 && L.N > 28672 && L.K >= 1024 && maxM > 4) return false;
    // one K range, results written once; operand rows are addressed with 32-bit byte offsets (64 rows',
    // the smallest tile's: longer rows are refused by the tiled kernels' own check)
    return maxM <= most && L.epi != Epi::GW && L.fmt_a != Fmt::I16 && !L.accum && L.kbeg == 0 && L.kend == L.K &&
           64 * row_bytes(L.fmt_a, L.K) < (1L << 31) && 64 * row_bytes(L.fmt_b, L.K) < (1L << 31);
}

hipError_t stream_launch(const Launch &L, uint64_t *blocks)
{
    SArgs a;
    a.N = L.epi == Epi::GLU ? L.N / 2 : L.N;
    a.K = L.K;
    a.lda = (uint32_t)row_bytes(L.fmt_a, L.K);
    a.ldb = (uint32_t)row_bytes(L.fmt_b, L.K);
    a.epi = (int)L.epi;
    a.act = L.act;
    a.shift = L.fmt_b == Fmt::I4P ? 4 : 0;
    for (int i = 0; i < kMaxProblems; i++) {
        const Problem P = i < L.nprob ? L.prob[i] : Problem{};
        a.M[i] = P.M;
        a.A[i] = P.A;
        a.B[i] = P.B;
        a.B2[i] = P.B2;
        a.C[i] = P.C;
    }
    const Fmt fa = L.fmt_a, fb = L.fmt_b;
    if (one_chain(L)) return launch_chain(a, L, blocks);
    if (fa == Fmt::F16) return launch_fmt<Fmt::F16, Fmt::F16>(a, L, blocks);
    if (fa == Fmt::I8 && fb == Fmt::I8) return launch_fmt<Fmt::I8, Fmt::I8>(a, L, blocks);
    if (fa == Fmt::I8 && fb == Fmt::I4P) return launch_fmt<Fmt::I8, Fmt::I4P>(a, L, blocks);
    if (fa == Fmt::F32BF16 && fb == fa) return launch_fmt<Fmt::F32BF16, Fmt::F32BF16>(a, L, blocks);
    if (fa == Fmt::BF16 && fb == Fmt::F32BF16) return launch_fmt<Fmt::BF16, Fmt::F32BF16>(a, L, blocks);
    if (fa == Fmt::BF16 && fb == fa) return launch_fmt<Fmt::BF16, Fmt::BF16>(a, L, blocks);
    if (fa == Fmt::F32TF32 && fb == fa) return launch_fmt<Fmt::F32TF32, Fmt::F32TF32>(a, L, blocks);
    if (fa == Fmt::BF16X2 && fb == Fmt::F32TF32) return launch_fmt<Fmt::BF16X2, Fmt::F32TF32>(a, L, blocks);
    if (fa == Fmt::BF16X2 && fb == fa) return launch_fmt<Fmt::BF16X2, Fmt::BF16X2>(a, L, blocks);
    return hipErrorInvalidValue;
}

}  // namespace gk
}  // namespace rk
