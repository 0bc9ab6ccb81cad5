// stream_gw_mid.hip — group-wise products of more rows than one MFMA holds whose workgroups fit the
// GPU at once: the weight-streaming kernel of stream_gw.hip for 17 rows and more.
//
// The same split: a wave owns 16 columns and all of K, its weights arrive by DMA in a ring of its
// own, and it folds in registers in group order. The codes of all K do not fit in LDS beside the
// rings, so they pass through it a chunk of K at a time, three chunks in turn: one read, two in
// flight, copied by the workgroup's waves together, one barrier a chunk. More rows are more
// workgroups: 16 or 32 a workgroup, 16 where those fit the CUs once.
//
// What bounds it is the serial time of a chunk (barrier, LDS reads, MFMA chain, fold) and a CU's
// load rate, not HBM. The tiled kernel's stage is 0.75 us for the same 128 of K whatever M; here
// (W4A8, rows quantised ahead, before -> after): 32 x 4096 x 4096 groups of 128 20.1 -> 9.9 us,
// 128 x 2048 x 2048 12.4 -> 6.7, 256 x 7936 x 1024 34.4 -> 16.5, 64 x 3840 x 15360 25.3 -> 15.6.
#include "gemm_impl.h"

namespace rk {
namespace gk {
namespace {

constexpr int kMD = 3;                    // chunks held (four: 0.3 us of 13 less, and a workgroup less a CU)

// Steps (KB of weights a wave) a chunk. Four halve the barriers: 16 rows, 32 x 7936 x 1024 19.3 -> 16.0 us;
// with more rows LDS would hold one workgroup a CU (32 rows, 64 x 3840 x 15360: 15.6 -> 25.9 us).
constexpr int mid_steps(int mb) { return mb == 1 ? 4 : 2; }

struct MArgs {
    int N, K, nG, nGp, nch;               // nch: chunks of K; nGp: groups of the scale tables (zeros past nG)
    int nbn, ppg, f16out;
    uint32_t ldb;
    int M[kMaxProblems];                  // problems with rows only
    const void *A[kMaxProblems], *B[kMaxProblems];
    const float *as[kMaxProblems], *bs[kMaxProblems];
    void *C[kMaxProblems];
};

// A dumping launch's arguments (as in stream_gw.hip).
struct MArgsDump : MArgs {
    FewDump dump[kMaxProblems];
};

// PK: K of an MFMA piece (32, 64 or, int4, 128); a group is PPG pieces (1, or 2 of a whole step: whole
// groups a chunk). RS: a scale a row. MB: 16-row blocks a workgroup. Two or four waves. DUMP: the
// partials of the launch's dump windows are stored too.
template <Fmt FB, int PK, int PPG, bool RS, int MB, bool DUMP>
__global__ __launch_bounds__(256, 2) void k_mid_gw(const std::conditional_t<DUMP, MArgsDump, MArgs> a)
{
    constexpr bool I4 = FB == Fmt::I4P;
    // K elements and pieces a step; code bytes of a row and chunk
    constexpr int kMS = mid_steps(MB), SK = I4 ? 128 : 64, NP = SK / PK, ROW = SK * kMS;
    constexpr int CPR = ROW / 16, ACH = 16 * MB * ROW;               // 16-byte chunks of such a row; bytes of a chunk's codes
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, r16 = lane & 15, q = lane >> 4, NT = blockDim.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), W = NT >> 6;
    const int nG = a.nG, nGp = a.nGp, K = a.K, N = a.N, nch = a.nch;
    const uint32_t ldb = a.ldb;
    const int p = __builtin_amdgcn_readfirstlane((int)blockIdx.y);
    const int m0 = (int)blockIdx.z * 16 * MB, M = min(a.M[p] - m0, 16 * MB);   // this workgroup's rows
    const int tile = (int)blockIdx.x * W + wave, n0 = tile * 16;
    if (M <= 0) return;
    const bool live = tile < a.nbn;       // a wave without columns still copies codes and meets the barriers
    // LDS: codes [chunk][row][ROW], activation scales [group][16 MB], the rows' own scales and order
    // flags, then a wave's ring and its scales [group][16]
    float *const AS = reinterpret_cast<float *>(smem + kMD * ACH);
    float *const rsl = AS + (RS ? 0 : nGp * 16 * MB);
    int *const mis = reinterpret_cast<int *>(rsl + 16 * MB);
    char *const ring = reinterpret_cast<char *>(mis + 16 * MB) + wave * (kMD * kMS * 1024 + nGp * 64);
    float *const S = reinterpret_cast<float *>(ring + kMD * kMS * 1024);

    const Rsrc sb = rsrc(a.bs[p] + (size_t)(live ? n0 : 0) * nG, live ? (uint32_t)(16 * nG) * 4u : 0u);
    constexpr int SR = 4;
    float sv[SR][4];
    auto sload = [&](int i, float (&v)[4]) __attribute__((always_inline)) { load_scales(sb, nG, r16, q, i, v); };
    auto sstore = [&](int i, const float (&v)[4]) __attribute__((always_inline)) { store_scales<I4>(S, nGp, r16, q, i, v); };
#pragma unroll
    for (int i = 0; i < SR; i++)
        if (16 * i < nGp) sload(i, sv[i]);

    // a chunk: its codes' 1 KB blocks over the waves (16-byte chunk c of row m at c ^ sw(m), so that
    // sixteen rows' reads of one chunk lie in different banks), then the wave's weights
    // (rows past M, and past K by the mask: zeros)
    const Rsrc ra = rsrc(static_cast<const char *>(a.A[p]) + (size_t)m0 * K, (uint32_t)M * (uint32_t)K);
    const Rsrc rb = rsrc(static_cast<const char *>(a.B[p]) + (size_t)(live ? n0 : 0) * ldb, live ? 16u * ldb : 0u);
    const uint32_t ob = (uint32_t)r16 * ldb + (uint32_t)q * 16u;
    const int klane = q * (SK / 4);
    constexpr int AB = ACH / 1024;         // 1 KB blocks of a chunk's codes
    const auto sw = [](int m) __attribute__((always_inline)) { return CPR >= 16 ? (m & 15) : ((m >> 1) & 7); };
    static_assert(AB % 4 == 0);            // every wave copies as many
    auto load = [&](int ch) __attribute__((always_inline)) {
#if defined(__HIP_DEVICE_COMPILE__)
        const int buf = ch % kMD;
        for (int b = wave; b < AB; b += W) {
            const int at = b * 64 + lane, m = at / CPR, c = (at % CPR) ^ sw(m), k = ch * ROW + c * 16;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (__attribute__((address_space(3))) void *)(smem + buf * ACH + b * 1024), 16,
                                                     k < K ? (uint32_t)m * (uint32_t)K + (uint32_t)k : kOOB, 0, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < kMS; u++) {
            const int st = ch * kMS + u;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (__attribute__((address_space(3))) void *)(ring + (buf * kMS + u) * 1024), 16,
                                                     st * SK + klane < K ? ob + (uint32_t)st * 64u : kOOB, 0, 0, 0);
        }
#else
        (void)ch; (void)ra; (void)rb; (void)ob; (void)klane; (void)sw;
#endif
    };
#pragma unroll
    for (int i = 0; i < kMD - 1; i++) load(i);   // (past K: zeros)
#pragma unroll
    for (int i = 0; i < SR; i++)
        if (16 * i < nGp) sstore(i, sv[i]);
    for (int i = SR; 16 * i < nGp; i++) {
        float v[4];
        sload(i, v);
        sstore(i, v);
    }
    if constexpr (!RS) {
        // a row whose scales are the same in every group folds in the row-scale order (gemm_impl.h)
        const float *as = a.as[p] + (size_t)m0 * nG;
        const bool check = nG >= 4 && nG <= 64;
        if (tid < 16 * MB) mis[tid] = check ? 0 : 1;
        lds_barrier();
        if (check)
            for (int i = tid; i < M * nG; i += NT) {
                const int m = i / nG;
                if (__float_as_int(as[i]) != __float_as_int(as[m * nG])) mis[m] = 1;
            }
        lds_barrier();
        for (int i = tid; i < 16 * MB * nGp; i += NT) {
            const int m = i / nGp, g = i - m * nGp;
            AS[g * 16 * MB + m] = m < M && g < nG ? (mis[m] ? as[m * nG + g] : 1.0f) : 0.f;
        }
        for (int i = tid; i < 16 * MB; i += NT) rsl[i] = i < M && !mis[i] ? as[i * nG] : 1.0f;
    } else {
        for (int i = tid; i < 16 * MB; i += NT) rsl[i] = i < M ? a.as[p][m0 + i] : 0.f;
    }

    f32x4 acc[MB];
    i32x4 d[MB];
#pragma unroll
    for (int i = 0; i < MB; i++) acc[i] = f32x4{};
    [[maybe_unused]] FewDump dw = {};
    if constexpr (DUMP) dw = a.dump[p];
    for (int ch = 0; ch < nch; ch++) {
        // chunk ch has arrived (only the next chunk's instructions are outstanding; none once nothing more
        // was issued), in every wave after the barrier; every wave has read chunk ch - 1, whose place
        // the next one loaded takes
        if (ch + kMD - 2 < max(kMD - 1, nch)) {
            if (W == 4) wait_vm<(kMD - 2) * (AB / 4 + kMS)>();
            else wait_vm<(kMD - 2) * (AB / 2 + kMS)>();
        } else {
            wait_vm<0>();
        }
        lds_barrier();
        if (ch + kMD - 1 < nch) load(ch + kMD - 1);
        const char *const ab = smem + (ch % kMD) * ACH, *const wb = ring + (ch % kMD) * (kMS * 1024);
#pragma unroll
        for (int u = 0; u < kMS; u++) {
            const char *const ws = wb + u * 1024;
#pragma unroll
            for (int x = 0; x < NP; x++) {
                const int y = u * NP + x;   // piece of the chunk
                i32x4 w0 = {}, w1 = {};
                long wl = 0;
                if constexpr (PK == 32) {
                    if constexpr (I4) {
                        const int w = *reinterpret_cast<const int *>(ws + (16 * x + r16) * 16 + 4 * q);
                        wl = pair64(nib_hi(w), nib_lo(w));
                    } else {
                        wl = *reinterpret_cast<const long *>(ws + (16 * (2 * x + (q >> 1)) + r16) * 16 + 8 * (q & 1));
                    }
                } else if constexpr (PK == 64) {
                    if constexpr (I4) {
                        typedef int i32x2 __attribute__((ext_vector_type(2)));
                        const i32x2 w = *reinterpret_cast<const i32x2 *>(ws + (16 * (2 * x + (q >> 1)) + r16) * 16 + 8 * (q & 1));
                        w0 = i32x4{nib_hi(w[0]), nib_lo(w[0]), nib_hi(w[1]), nib_lo(w[1])};
                    } else {
                        w0 = *reinterpret_cast<const i32x4 *>(ws + lane * 16);
                    }
                } else {
                    const i32x4 w = *reinterpret_cast<const i32x4 *>(ws + lane * 16);
                    w0 = i32x4{nib_hi(w[0]), nib_lo(w[0]), nib_hi(w[1]), nib_lo(w[1])};
                    w1 = i32x4{nib_hi(w[2]), nib_lo(w[2]), nib_hi(w[3]), nib_lo(w[3])};
                }
                const int c0 = u * (SK / 16);
#pragma unroll
                for (int i = 0; i < MB; i++) {
                    const int m = 16 * i + r16;
                    const char *const ar = ab + m * ROW;
                    const i32x4 z = y % PPG == 0 ? i32x4{} : d[i];
                    if constexpr (PK == 32) {
                        const long af = *reinterpret_cast<const long *>(ar + (((c0 + 2 * x + (q >> 1)) ^ sw(m)) << 4) + 8 * (q & 1));
                        d[i] = __builtin_amdgcn_mfma_i32_16x16x32_i8(af, wl, z, 0, 0, 0);
                    } else if constexpr (PK == 64) {
                        d[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(*reinterpret_cast<const i32x4 *>(ar + (((c0 + 4 * x + q) ^ sw(m)) << 4)),
                                                                     w0, z, 0, 0, 0);
                    } else {
                        d[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(*reinterpret_cast<const i32x4 *>(ar + (((c0 + 2 * q) ^ sw(m)) << 4)), w0,
                                                                     z, 0, 0, 0);
                        d[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(*reinterpret_cast<const i32x4 *>(ar + (((c0 + 2 * q + 1) ^ sw(m)) << 4)),
                                                                     w1, d[i], 0, 0, 0);
                    }
                }
                if ((y + 1) % PPG == 0) {
                    const int g = (ch * kMS * NP + y) / PPG;
                    const float s = S[g * 16 + r16];
#pragma unroll
                    for (int i = 0; i < MB; i++) {
                        if constexpr (DUMP) {
                            if (live && dw.p) few_dump<I4>(dw, nG, N, g, n0 + r16, m0 + 16 * i + 4 * q, d[i]);
                        }
                        if constexpr (RS) {
#pragma unroll
                            for (int e = 0; e < 4; e++) acc[i][e] = __builtin_fmaf(s, (float)d[i][e], acc[i][e]);
                        } else {
                            const f32x4 sa = *reinterpret_cast<const f32x4 *>(AS + g * 16 * MB + 16 * i + 4 * q);
#pragma unroll
                            for (int e = 0; e < 4; e++) acc[i][e] = __builtin_fmaf(sa[e] * s, (float)d[i][e], acc[i][e]);
                        }
                    }
                }
            }
        }
    }
    wait_vm<0>();
    if (!live) return;
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int m = 16 * i + 4 * q + e;
            if (m >= M) continue;
            const float v = acc[i][e] * rsl[m];
            const size_t at = (size_t)(m0 + m) * N + n0 + r16;
            if (a.f16out) static_cast<_Float16 *>(a.C[p])[at] = (_Float16)v;
            else static_cast<float *>(a.C[p])[at] = v;
        }
}

struct MPlan {
    int w, pk, np, mb, nb;
    bool dump = false;
    size_t lds;
};

// The launch's shape, or false where another kernel takes it.
bool plan_mid(const Launch &L, int maxM, MPlan &g, MArgs &a)
{
    const bool i4 = L.fmt_b == Fmt::I4P;
    const int sk = i4 ? 128 : 64;
    if (L.epi != Epi::GW || maxM <= 16 || L.kt != L.group || L.fmt_a != Fmt::I8 || L.qa) return false;
    a.nbn = L.N / 16;
    if ((long)maxM * a.nbn > 256L * 32 * 8) return false;   // past every form below, whatever the rest says
    g.np = 0;
    for (int i = 0; i < L.nprob; i++) {
        g.np += L.prob[i].M > 0;
        g.dump |= L.prob[i].dump != nullptr;
    }
    g.pk = L.group % sk == 0 ? sk : (L.group % 64 == 0 ? 64 : 32);
    a.ppg = L.group / g.pk;
    if (a.ppg > 2 || (a.ppg == 2 && g.pk != sk)) return false;
    a.nG = L.K / L.group;
    // Rows a workgroup and workgroups a CU, in the order of their times where several serve: 16 rows, one
    // (64 x 4096 x 4096, groups of 128: 10.2 us, 13.5 with 32 rows); 32 rows, one (128 x 4096 x 4096: 13.9,
    // two of 16 rows 18.1), and two (256 x 4096 x 4096: 16.7, tiles 25.8). More workgroups than the GPU
    // holds at once are the tiles' (256 x 3840 x 15360: 50, tiles 35.9). 64 rows a workgroup were
    // slower than the tiles with groups of 32 (396 x 4608 x 1344: 43.3, tiles 39.9), and so are two a CU
    // of int8 weights with such groups, four folds a step (MoE layers of 132 and 194 tokens, hidden 2880
    // and 2944: 41.6 and 43.1, tiles 38.8 and 39.0). Of int8 weights two a CU, and with groups of 32 one a
    // CU of many columns, keep ahead of the tiles on short rows alone (64 x 16384, groups of 64: K = 1024
    // 1.06 times as fast, 2048 0.98, 4096 0.89, 8192 51.0 us against 42.9; 128 x 8192, groups of 128: 1.10,
    // 0.99, 0.91, 0.86; 64 x 8192, groups of 32: 1.12, 0.98, 0.91, 0.85; at 6144 columns 1.29 to 1.17), or
    // where a tile's 64 rows are half empty (MoE layers of 64 tokens, hidden 4096, groups of 64: 56.2, tiles
    // 73.9).
    static const int form[][2] = {{1, 1}, {2, 1}, {2, 2}};
    for (const auto &f : form) {
        if (f[1] == 2 && !i4 && L.group < 64) continue;
        if (!i4 && L.K >= 2048 && ((f[1] == 2 && maxM > 32) || (f[0] == 2 && L.group < 64 && L.N >= 8192))) continue;
        g.mb = f[0];
        const int chunk = sk * mid_steps(g.mb);
        a.nch = (L.K + chunk - 1) / chunk;
        a.nGp = a.nch * (chunk / g.pk) / a.ppg;
        g.nb = (maxM + 16 * g.mb - 1) / (16 * g.mb);
        const size_t lds = 160 * 1024, tab = (size_t)a.nGp * 64;
        const size_t shared = (size_t)kMD * 16 * g.mb * chunk + (L.rowscale ? 0 : tab * g.mb) + 16 * g.mb * 8;
        for (g.w = 4; g.w >= 2; g.w /= 2) {   // two waves where four waves' scales leave no room
            g.lds = shared + g.w * (tab + (size_t)kMD * mid_steps(g.mb) * 1024);
            if (g.lds <= lds / f[1] && (long)g.np * g.nb * ((a.nbn + g.w - 1) / g.w) <= 256 * f[1]) return true;
        }
    }
    return false;
}

template <Fmt FB, int PK, int PPG, bool RS, int MB, bool DUMP> hipError_t launch_mid_k(const MArgsDump &a, const MPlan &g, hipStream_t s)
{
    auto kern = k_mid_gw<FB, PK, PPG, RS, MB, DUMP>;
    static std::atomic<uint64_t> opted{0};
    if (const hipError_t e = lds_opt_in(reinterpret_cast<const void *>(kern), 160 * 1024, opted)) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)((a.nbn + g.w - 1) / g.w), (unsigned)g.np, (unsigned)g.nb), dim3(g.w * 64), g.lds, s,
                       static_cast<const std::conditional_t<DUMP, MArgsDump, MArgs> &>(a));
    return hipGetLastError();
}

template <Fmt FB, int PK> hipError_t launch_mid_pk(const MArgsDump &a, const MPlan &g, const Launch &L)
{
    auto by = [&](auto PPG, auto RS) {
        constexpr int P = decltype(PPG)::value;
        constexpr bool R = decltype(RS)::value;
        if (g.dump)
            return g.mb == 1 ? launch_mid_k<FB, PK, P, R, 1, true>(a, g, L.stream) : launch_mid_k<FB, PK, P, R, 2, true>(a, g, L.stream);
        return g.mb == 1 ? launch_mid_k<FB, PK, P, R, 1, false>(a, g, L.stream) : launch_mid_k<FB, PK, P, R, 2, false>(a, g, L.stream);
    };
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    if constexpr (PK == (FB == Fmt::I4P ? 128 : 64))
        if (a.ppg == 2) return L.rowscale ? by(I2{}, std::true_type{}) : by(I2{}, std::false_type{});
    return L.rowscale ? by(I1{}, std::true_type{}) : by(I1{}, std::false_type{});
}

}  // namespace

bool mid_gw_takes(const Launch &L, int maxM)
{
    MPlan g;
    MArgs a;
    return plan_mid(L, maxM, g, a);
}

hipError_t mid_gw_launch(const Launch &L, int maxM, uint64_t *blocks)
{
    MPlan g;
    MArgsDump a = {};
    if (!plan_mid(L, maxM, g, a)) return hipErrorInvalidValue;
    a.N = L.N;
    a.K = L.K;
    a.ldb = (uint32_t)row_bytes(L.fmt_b, L.K);
    a.f16out = L.f16out;
    int n = 0;
    for (int i = 0; i < L.nprob; i++) {
        const Problem &P = L.prob[i];
        if (P.M == 0) continue;
        a.M[n] = P.M;
        a.A[n] = P.A;
        a.B[n] = P.B;
        a.as[n] = P.a_scale;
        a.bs[n] = P.b_scale;
        a.C[n] = P.C;
        a.dump[n] = FewDump{P.dump, P.dump_row0, P.dump_rows};
        n++;
    }
    *blocks = (uint64_t)((a.nbn + g.w - 1) / g.w) * g.np * g.nb;
    if (L.fmt_b == Fmt::I4P) {
        if (g.pk == 128) return launch_mid_pk<Fmt::I4P, 128>(a, g, L);
        return g.pk == 64 ? launch_mid_pk<Fmt::I4P, 64>(a, g, L) : launch_mid_pk<Fmt::I4P, 32>(a, g, L);
    }
    return g.pk == 64 ? launch_mid_pk<Fmt::I8, 64>(a, g, L) : launch_mid_pk<Fmt::I8, 32>(a, g, L);
}

}  // namespace gk
}  // namespace rk
