// stream_gw.hip — group-wise products of at most 16 rows (decode batches, MoE experts with few
// tokens each): the weight-streaming kernel.
//
// As in stream.hip the weights' bytes in flight bound the product, and here every output is one
// fp32 chain over its groups in order, so a wave owns 16 columns and all of K: no partial
// crosses waves and nothing but the prologue has a barrier. What keeps enough bytes in flight
// with so few waves is LDS: a wave's weights go global -> LDS by DMA into a ring of its own of
// three 4 KB slots, each step's 16 rows x 64 bytes as one instruction (lane l: row l % 16, bytes
// 16 (l / 16) .. + 16), and the ds_reads pick each group's bytes so that one MFMA covers
// exactly one group's K or a part of it: with groups of 32 a 16x16x32 MFMA whose lane quarters
// hold eight values each of the group. The activations' codes lie in LDS once a workgroup
// (copied by DMA, or quantised there from fp32 / fp16 rows, or from act(gate) * up), and so do
// the wave's scales.
//
// Measured (three sets of operands in turn; tiled kernels before, this kernel after):
//   int4 g 128   4 x  3840 x 15360   22.7 -> 10.6 us   (29.5 MB of codes, 3.0 TB/s)
//   the same on fp32 rows             25.8 -> 11.5      (quantised in the kernel)
//   int4 g 128   4 x  4096 x  4096   19.1 ->  6.0
//   int4 g 32    4 x  4096 x  4096   27.9 ->  9.5
//   MoE layer, 16 tokens, g 32       35.0 -> 27.9      (two launches instead of three)
// Other forms measured at 4 x 3840 x 15360: fragments through registers, partials exchanged in
// LDS by rounds with a barrier each, 11.8 us (MoE 33); the same with a persistent grid 14.5, and
// with its weights in an LDS ring 13.6. Rings deeper than three slots of 4 KB measured slower
// (they cost workgroups a CU).
#include "gemm_impl.h"

namespace rk {
namespace gk {
namespace {

constexpr int kCH = 4;                    // steps (KB) a ring slot

struct GArgs {
    int N, K, nG, nslots;                 // nslots: slots of kCH steps a tile
    int nGp;                              // groups of the scale tables (zeros past nG: a last slot's tail)
    int nbn;                              // 16-column tiles a problem
    int tiles;
    int depth;                            // ring slots a wave
    int spw;                              // K split over a workgroup's waves: slots of K a wave
    int ppg;                              // MFMA pieces a group
    int mb;                               // 4-row blocks of the largest problem
    int kp;                               // bytes of a row of codes in LDS (a multiple of 256)
    int f16out, act;
    uint32_t ldb;                         // bytes a row of B
    int M[kMaxProblems];                  // problems with rows only
    const void *A[kMaxProblems], *A2[kMaxProblems], *B[kMaxProblems];
    const float *as[kMaxProblems], *bs[kMaxProblems];
    void *C[kMaxProblems];
};

// A dumping launch's arguments (of their own: longer ones cost the other launches microseconds when cold).
struct GArgsDump : GArgs {
    FewDump dump[kMaxProblems];
};

// Waits until at most n vector-memory instructions of this wave are outstanding; n a multiple of
// kCH (rounded down to a count that has a case here, which waits for more).
__device__ __forceinline__ void wait_vm_le(int n)
{
    if (n >= 12 * kCH) wait_vm<12 * kCH>();
    else if (n >= 10 * kCH) wait_vm<10 * kCH>();
    else if (n >= 8 * kCH) wait_vm<8 * kCH>();
    else if (n >= 6 * kCH) wait_vm<6 * kCH>();
    else if (n >= 5 * kCH) wait_vm<5 * kCH>();
    else if (n >= 4 * kCH) wait_vm<4 * kCH>();
    else if (n >= 3 * kCH) wait_vm<3 * kCH>();
    else if (n >= 2 * kCH) wait_vm<2 * kCH>();
    else if (n >= kCH) wait_vm<kCH>();
    else wait_vm<0>();
}

// PK: K of an MFMA piece (32, 64 or, int4, 128), a divisor of the group; PPG: pieces a group (1 or
// 2: whole groups a slot, so that a slot's body has no branch and its LDS reads, MFMAs and folds
// overlap; 0: any number, counted). RS: a scale a row. QIN: 0 int8 codes in global memory, 1 / 2 fp32 / fp16 rows that each
// workgroup quantises by k_quant_rows' formula (act(A) * A2 where A2 is given). DUMP: the partials of
// the launch's dump windows are stored too (an instantiation of its own: the stores cost registers).
template <Fmt FB, int PK, int PPG, bool RS, int QIN, bool SPLIT, bool DUMP>
__global__ __launch_bounds__(512, 2) void k_stream_gw(const std::conditional_t<DUMP, GArgsDump, GArgs> a)
{
    constexpr bool I4 = FB == Fmt::I4P;
    constexpr int SK = I4 ? 128 : 64, NP = SK / PK;       // K elements and pieces a step
    constexpr int PRE = SPLIT ? 1 : 3;                    // ring slots loaded in the prologue
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, r16 = lane & 15, q = lane >> 4, NT = blockDim.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), W = NT >> 6;
    const int nG = a.nG, nGp = a.nGp, K = a.K, N = a.N, kp = a.kp, depth = a.depth, nslots = a.nslots;
    const uint32_t ldb = a.ldb;
    const int p = __builtin_amdgcn_readfirstlane((int)blockIdx.y);
    const int M = a.M[p];
    const int tile = SPLIT ? (int)blockIdx.x : (int)blockIdx.x * W + wave;   // past the last: no columns
    const int n0 = tile * 16;
    const bool live = tile < a.nbn;
    // LDS: codes [row][kp], activation scales [group][16], the rows' own scales and order flags,
    // then a wave's ring and its scales [group][16]
    char *const codes = smem;
    float *const AS = reinterpret_cast<float *>(smem + ((a.mb * 4 * kp + 1023) & ~1023));
    float *const rsl = AS + (RS ? 0 : nGp * 16);
    int *const mis = reinterpret_cast<int *>(rsl + 16);
    float *const wmax = reinterpret_cast<float *>(mis + 16);
    char *const ring = reinterpret_cast<char *>(wmax + 16) + wave * (depth * kCH * 1024 + (SPLIT ? 0 : nGp * 64));
    float *const S = reinterpret_cast<float *>(SPLIT ? reinterpret_cast<char *>(wmax + 16) + W * (depth * kCH * 1024)
                                                     : ring + depth * kCH * 1024);
    int *const P = reinterpret_cast<int *>(S + nGp * 16);  // SPLIT: partials [group][4-row block][column][row]
    // the wave's ring slots of K
    const int sl0 = SPLIT ? wave * a.spw : 0, sl1 = SPLIT ? min(nslots, sl0 + a.spw) : nslots, own = sl1 - sl0;

    // ---- prologue ----
    // the wave's b scales: lane (n, q) takes four groups of column n at a time
    const Rsrc sb = rsrc(a.bs[p] + (size_t)(live ? n0 : 0) * nG, live ? (uint32_t)(16 * nG) * 4u : 0u);
    constexpr int SR = 4;   // in registers: 64 groups; further ones after the ring's first loads
    const int i0 = SPLIT ? wave : 0, di = SPLIT ? W : 1;
    float sv[SR][4];
    auto sload = [&](int i, float (&v)[4]) __attribute__((always_inline)) { load_scales(sb, nG, r16, q, i, v); };
    auto sstore = [&](int i, const float (&v)[4]) __attribute__((always_inline)) { store_scales<I4>(S, nGp, r16, q, i, v); };
#pragma unroll
    for (int i = 0; i < SR; i++)
        if (16 * (i0 + i * di) < nGp) sload(i0 + i * di, sv[i]);
    // the codes: 16-byte chunk c of row m at chunk c ^ m, so that the sixteen rows of a fragment
    // read lie in different banks
    [[maybe_unused]] int na = 0;
    const int kc = kp >> 4;
    if constexpr (QIN == 0) {
        const Rsrc ra = rsrc(a.A[p], (uint32_t)M * (uint32_t)K);
        for (int o = wave * 64; o < M * kc; o += NT) {
#if defined(__HIP_DEVICE_COMPILE__)
            const int at = o + lane, m = at / kc, c = (at - m * kc) ^ m;
            const bool in = m < M && c * 16 < K;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (__attribute__((address_space(3))) void *)(codes + o * 16), 16,
                                                     in ? (uint32_t)m * (uint32_t)K + (uint32_t)c * 16u : kOOB, 0, 0, 0);
#else
            (void)ra;
#endif
        }
    }
    // rows quantised here: NT / Mp threads a row; its first 64 elements a thread stay in registers
    const int tpr = M <= 4 ? NT / 4 : (M <= 8 ? NT / 8 : NT / 16), qm = tid / tpr, qt = tid % tpr;
    constexpr int QC = 8;
    [[maybe_unused]] float qv[QIN ? QC : 1][8];
    auto row8q = [&](int k, float (&v)[8]) __attribute__((always_inline)) {
        load8f<QIN == 2>(a.A[p], (long)qm * K + k, v);
        if (a.A2[p]) {
            float u[8];
            load8f<QIN == 2>(a.A2[p], (long)qm * K + k, u);
            if (a.act == kActGelu) {
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = act_k<kActGelu>(v[e]) * u[e];
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = act_k<kActSilu>(v[e]) * u[e];
            }
        }
    };
    if constexpr (QIN != 0) {
#pragma unroll
        for (int c = 0; c < QC; c++) {
            const int k = (c * tpr + qt) * 8;
            if (qm < M && k < K) row8q(k, qv[c]);
        }
    }

    // ---- the ring ----
    const uint32_t ob = (uint32_t)r16 * ldb + (uint32_t)q * 16u;
    const int klane = q * (SK / 4);
    const Rsrc rb = rsrc(static_cast<const char *>(a.B[p]) + (size_t)(live ? n0 : 0) * ldb, live ? 16u * ldb : 0u);
    [[maybe_unused]] int lslot = 0, lpos = sl0;   // the next slot's place in the ring and in K
    auto load = [&]() __attribute__((always_inline)) {
#if defined(__HIP_DEVICE_COMPILE__)
        char *const d = ring + lslot * (kCH * 1024);
#pragma unroll
        for (int u = 0; u < kCH; u++) {
            const int st = lpos * kCH + u;   // past K: zeros
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (__attribute__((address_space(3))) void *)(d + u * 1024), 16,
                                                     lpos < sl1 && st * SK + klane < K ? ob + (uint32_t)st * 64u : kOOB, 0, 0, 0);
        }
#else
        (void)rb; (void)ob; (void)klane;
#endif
        lslot = lslot + 1 == depth ? 0 : lslot + 1;
        lpos++;
    };
    // (a fixed number of slots now, so that what was issued before them is waited for by count)
#pragma unroll
    for (int i = 0; i < PRE; i++) load();
    if constexpr (QIN != 0) {
        float mx = 0.f;
        if (qm < M) {
#pragma unroll
            for (int c = 0; c < QC; c++)
                if ((c * tpr + qt) * 8 < K)
#pragma unroll
                    for (int e = 0; e < 8; e++) mx = fmaxf(mx, fabsf(qv[c][e]));
            for (int k = (QC * tpr + qt) * 8; k < K; k += tpr * 8) {
                float v[8];
                row8q(k, v);
#pragma unroll
                for (int e = 0; e < 8; e++) mx = fmaxf(mx, fabsf(v[e]));
            }
        }
        for (int off = (tpr < 64 ? tpr : 64) / 2; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
        if (tpr > 64) {   // two waves a row (at most: 512 threads, rows in fours)
            if (lane == 0) wmax[wave] = mx;
            lds_barrier();
            mx = fmaxf(wmax[wave & ~1], wmax[wave | 1]);
        }
        const float s = mx > 0.f ? 127.0f / mx : 0.0f;
        auto put = [&](int k, const float (&v)[8]) __attribute__((always_inline)) {
            quant_store8(reinterpret_cast<int8_t *>(codes) + qm * kp + (((k >> 4) ^ qm) << 4) + (k & 8), v, s);
        };
        if (qm < M) {
            if (qt == 0) rsl[qm] = mx > 0.f ? mx / 127.0f : 0.0f;
#pragma unroll
            for (int c = 0; c < QC; c++)
                if ((c * tpr + qt) * 8 < K) put((c * tpr + qt) * 8, qv[c]);
            for (int k = (QC * tpr + qt) * 8; k < K; k += tpr * 8) {
                float v[8];
                row8q(k, v);
                put(k, v);
            }
        }
    } else {
        wait_vm<PRE * kCH>();   // the codes' DMA
    }
#pragma unroll
    for (int i = 0; i < SR; i++)
        if (16 * (i0 + i * di) < nGp) sstore(i0 + i * di, sv[i]);
    for (int i = i0 + SR * di; 16 * i < nGp; i += di) {
        float v[4];
        sload(i, v);
        sstore(i, v);
    }
    if constexpr (!RS) {
        // a row whose scales are the same in every group folds in the row-scale order (gemm_impl.h)
        const float *as = a.as[p];
        const bool check = nG >= 4 && nG <= 64;
        if (tid < 16) mis[tid] = check ? 0 : 1;
        __syncthreads();
        if (check)
            for (int i = tid; i < M * nG; i += NT) {
                const int m = i / nG;
                if (__float_as_int(as[i]) != __float_as_int(as[m * nG])) mis[m] = 1;
            }
        __syncthreads();
        for (int i = tid; i < 16 * nGp; i += NT) {
            const int m = i / nGp, g = i - m * nGp;
            AS[g * 16 + m] = m < M && g < nG ? (mis[m] ? as[m * nG + g] : 1.0f) : 0.f;
        }
        if (tid < 16) rsl[tid] = tid < M && !mis[tid] ? as[tid * nG] : 1.0f;
    } else if constexpr (QIN == 0) {
        if (tid < 16) rsl[tid] = tid < M ? a.as[p][tid] : 0.f;
    }
    lds_barrier();
    if (!SPLIT && !live) {
        wait_vm<0>();
        return;
    }
    for (int i = PRE; i < min(depth, own); i++) load();

    // ---- K ----
    f32x4 acc = {};
    i32x4 d = {};
    int left = a.ppg, g = 0;   // pieces left of the open group
    const int am = r16 < a.mb * 4 ? r16 : 0;               // rows past M: their results are not stored
    const char *const la = codes + am * kp;
    int slot = 0;
    const int npc = K / PK;    // pieces in all
    [[maybe_unused]] FewDump dw = {};
    if constexpr (DUMP) dw = a.dump[p];
    for (int sl = sl0; sl < sl1; sl++) {
        wait_vm_le(min(max(PRE, min(depth, own)) - 1, max(PRE, own) - 1 - (sl - sl0)) * kCH);
        asm volatile("" ::: "memory");   // no read of the slot above the wait
        const char *const wb = ring + slot * (kCH * 1024);
#pragma unroll
        for (int u = 0; u < kCH; u++) {
            const int c0 = (sl * kCH + u) * (SK / 16);     // the step's first 16-byte chunk of codes
            const char *const ws = wb + u * 1024;
#pragma unroll
            for (int x = 0; x < NP; x++) {
                if constexpr (PPG == 0)
                    if ((sl * kCH + u) * NP + x >= npc) continue;   // past K
                const int y = u * NP + x;                           // piece of the slot
                const i32x4 z = PPG != 0 && y % (PPG ? PPG : 1) == 0 ? i32x4{} : d;
                if constexpr (PK == 32) {
                    // the quarter's eight values of the group: codes 8 q .. + 8 of 32
                    const long af = *reinterpret_cast<const long *>(la + (((c0 + 2 * x + (q >> 1)) ^ am) << 4) + 8 * (q & 1));
                    if constexpr (I4) {
                        const int w = *reinterpret_cast<const int *>(ws + (16 * x + r16) * 16 + 4 * q);
                        d = __builtin_amdgcn_mfma_i32_16x16x32_i8(af, pair64(nib_hi(w), nib_lo(w)), z, 0, 0, 0);
                    } else {
                        const long w = *reinterpret_cast<const long *>(ws + (16 * (2 * x + (q >> 1)) + r16) * 16 + 8 * (q & 1));
                        d = __builtin_amdgcn_mfma_i32_16x16x32_i8(af, w, z, 0, 0, 0);
                    }
                } else if constexpr (PK == 64) {
                    const i32x4 af = *reinterpret_cast<const i32x4 *>(la + (((c0 + 4 * x + q) ^ am) << 4));
                    if constexpr (I4) {
                        typedef int i32x2 __attribute__((ext_vector_type(2)));
                        const i32x2 w = *reinterpret_cast<const i32x2 *>(ws + (16 * (2 * x + (q >> 1)) + r16) * 16 + 8 * (q & 1));
                        d = __builtin_amdgcn_mfma_i32_16x16x64_i8(af, i32x4{nib_hi(w[0]), nib_lo(w[0]), nib_hi(w[1]), nib_lo(w[1])}, z, 0,
                                                                  0, 0);
                    } else {
                        d = __builtin_amdgcn_mfma_i32_16x16x64_i8(af, *reinterpret_cast<const i32x4 *>(ws + lane * 16), z, 0, 0, 0);
                    }
                } else {
                    const i32x4 w = *reinterpret_cast<const i32x4 *>(ws + lane * 16);
                    const i32x4 a0 = *reinterpret_cast<const i32x4 *>(la + (((c0 + 2 * q) ^ am) << 4));
                    const i32x4 a1 = *reinterpret_cast<const i32x4 *>(la + (((c0 + 2 * q + 1) ^ am) << 4));
                    d = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, i32x4{nib_hi(w[0]), nib_lo(w[0]), nib_hi(w[1]), nib_lo(w[1])}, z, 0, 0, 0);
                    d = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, i32x4{nib_hi(w[2]), nib_lo(w[2]), nib_hi(w[3]), nib_lo(w[3])}, d, 0, 0, 0);
                }
                if (PPG ? (y + 1) % (PPG ? PPG : 1) == 0 : --left == 0) {
                    const int gi = PPG ? (sl * kCH * NP + y) / (PPG ? PPG : 1) : g;
                    const float s = SPLIT ? 0.f : S[gi * 16 + r16];
                    if constexpr (DUMP) {
                        if (live && dw.p) few_dump<I4>(dw, nG, N, gi, n0 + r16, 4 * q, d);
                    }
                    if constexpr (SPLIT) {
                        if (q < a.mb) *reinterpret_cast<i32x4 *>(P + ((gi * a.mb + q) * 16 + r16) * 4) = d;
                    } else if constexpr (RS) {
#pragma unroll
                        for (int e = 0; e < 4; e++) acc[e] = __builtin_fmaf(s, (float)d[e], acc[e]);
                    } else {
                        const f32x4 sa = *reinterpret_cast<const f32x4 *>(AS + gi * 16 + 4 * q);
#pragma unroll
                        for (int e = 0; e < 4; e++) acc[e] = __builtin_fmaf(sa[e] * s, (float)d[e], acc[e]);
                    }
                    if constexpr (PPG == 0) {
                        g++;
                        d = i32x4{};
                        left = a.ppg;
                    }
                }
            }
        }
        slot = slot + 1 == depth ? 0 : slot + 1;
        if (sl + depth < sl1) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the slot is read: the next loads may overwrite it
            load();
        }
    }
    wait_vm<0>();
    if constexpr (SPLIT) {
        // one thread an output folds all groups (zeros past nG) in order
        lds_barrier();
        const int fn = (tid >> 2) & 15, fm = (tid >> 6) * 4 + (tid & 3);
        if (tid >= a.mb * 64 || fm >= M) return;
        float f = 0.f;
        for (int g8 = 0; g8 < nGp; g8 += 8) {
            int pv[8];
            float s[8];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int gg = min(g8 + e, nGp - 1);
                pv[e] = P[gg * (a.mb * 64) + tid];
                s[e] = S[gg * 16 + fn];
                if constexpr (!RS) s[e] *= AS[gg * 16 + fm];
                if (g8 + e >= nGp) s[e] = 0.f;   // (the product: a last group's scale may be infinite)
            }
#pragma unroll
            for (int e = 0; e < 8; e++) f = __builtin_fmaf(s[e], (float)pv[e], f);
        }
        const float v = f * rsl[fm];
        const size_t at = (size_t)fm * N + n0 + fn;
        if (a.f16out) static_cast<_Float16 *>(a.C[p])[at] = (_Float16)v;
        else static_cast<float *>(a.C[p])[at] = v;
        return;
    }
    const int n = n0 + r16;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int m = 4 * q + e;
        if (m >= M) continue;
        const float v = acc[e] * rsl[m];
        const size_t at = (size_t)m * N + n;
        if (a.f16out) static_cast<_Float16 *>(a.C[p])[at] = (_Float16)v;
        else static_cast<float *>(a.C[p])[at] = v;
    }
}

struct GPlan {
    int w, pk, np;
    bool split = false, dump = false;
    size_t lds;
};

// The launch's shape, or false where the tiled kernels take it.
bool plan_gw(const Launch &L, int maxM, GPlan &g, GArgs &a)
{
    const bool i4 = L.fmt_b == Fmt::I4P;
    const int sk = i4 ? 128 : 64;
    if (L.epi != Epi::GW || maxM > 16 || maxM < 1 || L.kt != L.group || L.fmt_a != Fmt::I8) return false;
    if (L.qa && (!L.rowscale || (L.qa == 2 && i4) || L.prob[0].dump)) return false;   // (no entry dumps rows it quantises)
    if (64 * row_bytes(L.fmt_a, L.K) >= (1L << 31)) return false;   // (refused by the tiled kernels' own check)
    g.np = 0;
    for (int i = 0; i < L.nprob; i++) {
        g.np += L.prob[i].M > 0;
        g.dump |= L.prob[i].dump != nullptr;
    }
    g.pk = L.group % sk == 0 ? sk : (L.group % 64 == 0 ? 64 : 32);
    a.ppg = L.group / g.pk;
    a.mb = (maxM + 3) / 4;
    a.nG = L.K / L.group;
    a.nslots = ((L.K + sk - 1) / sk + kCH - 1) / kCH;
    const int per = kCH * (sk / g.pk);   // pieces a slot
    a.nGp = a.ppg <= 2 ? a.nslots * per / a.ppg : a.nG;
    a.kp = (L.K + 255) / 256 * 256;
    a.nbn = L.N / 16;
    a.tiles = g.np * a.nbn;
    const size_t slot = kCH * 1024, tab = (size_t)a.nGp * 64, lds = 160 * 1024;
    const size_t shared = (((size_t)a.mb * 4 * a.kp + 1023) & ~(size_t)1023) + (L.rowscale ? 0 : tab) + 192;
    // Few tiles: K split over a workgroup's waves, while the workgroups fit the GPU at once (4 rows,
    // 4096 x 4096: groups of 128 10.1 us a wave a tile, 6.0 split; groups of 32 15.6 and 10.6; twice
    // the columns, where they no longer do, 14.6 and 20.3).
    if (a.ppg <= 2) {
        g.w = 1;   // a power of two (the rows quantised here take whole parts of it), a thread an output
        while (g.w < std::min(8, std::max(a.mb, a.nslots))) g.w *= 2;
        a.spw = (a.nslots + g.w - 1) / g.w;
        a.depth = std::min(3, a.spw);
        g.lds = shared + tab + (size_t)a.nGp * a.mb * 256 + g.w * a.depth * slot;
        g.split = g.lds <= lds && a.tiles <= 256 * (int)(lds / g.lds);
    }
    if (!g.split) {
        // A wave a tile, W waves a workgroup that share the codes in LDS: the W of the least time, in
        // half microseconds. A batch of workgroups that LDS holds together takes 20 and one for each of
        // the busiest CU's waves (16 rows, 3840 x 15360: 11.9 us with four waves, 22.1 with two, which leave
        // one workgroup a CU; 1408 gate and up tiles of 8 rows, K = 2048: 13.5 with two, 15.2 with eight, in
        // one batch, 20.1 with four and 21.3 with one, in two; 1248 of 16, K = 1632: 11.8 with eight, 18.0 to
        // 20.4 in two batches). Rows quantised here take e elements a thread in each batch, and more where
        // they are formed from gate and up, of which 64 stay in registers (1344 tiles, 16 rows of 896: 22.4
        // us with two waves, 12.9 with four, 10.8 with eight, 12.5 quantised ahead).
        a.depth = 3;
        int best = 0, ahead = 0, waves = 0, rounds = 0;   // of the best: waves a CU, batches of workgroups
        for (int w = 8; w >= 1; w /= 2) {
            const size_t b = shared + w * (tab + a.depth * slot);
            if (b > lds || (L.qa_must && (long)maxM * L.K > 120L * w * 64)) continue;
            const int wgs = g.np * ((a.nbn + w - 1) / w), each = (wgs + 255) / 256, fit = (int)(lds / b);
            const int batches = (each + fit - 1) / fit, e = L.K * (maxM <= 4 ? 4 : maxM <= 8 ? 8 : 16) / (64 * w);
            const int plain = w * each + 20 * batches;
            const int cost = plain + (!L.qa ? 0 : L.act ? batches * (e / 7 + (e > 64 ? 12 : 0)) : batches * e / 20);
            if (!ahead || plain + 8 < ahead) ahead = plain + 8;
            if (!best || cost < best) {
                best = cost;
                g.w = w;
                g.lds = b;
                waves = w * fit;
                rounds = batches;
            }
        }
        if (!best || (L.qa && !L.qa_must && ahead <= best)) return false;   // (a pass ahead takes 4 us)
        // Long rows leave LDS for one or two waves a CU, and several batches of those take longer than
        // the tiles: int4, from more batches than waves (16 x 8192 x 16384, groups of 128, one wave, four
        // batches: 90.6 us, tiles 44.2; 16 x 8192 x 12288, groups of 256, two and two: 38.1 and 33.4; 16 x
        // 5120 x 16384, groups of 32, two and two: 39.7 and 49.5); int8, whose tiles unpack nothing, from
        // two (16 x 8192 x 16384, groups of 32: 153.7, tiles 43.4; 16 x 8192 x 16384, groups of 256, two
        // waves and two batches: 57.6 and 42.9; four waves and two batches at the least 1.06 of the tiles').
        if (i4 ? rounds > waves : rounds > 1 && waves <= 2) return false;
    }
    // Rows are quantised here while a thread has at most 120 elements of them; more of it in every
    // workgroup costs what the pass ahead does (fp32 rows, 3840 x 15360: 4 rows 15.6 -> 13.4 us, 8
    // rows, 120 elements, 15.7 -> 14.6, 16 rows 15.6 -> 24.9).
    return !L.qa || (long)maxM * L.K <= 120L * g.w * 64;
}

template <Fmt FB, int PK, int PPG, bool RS, int QIN, bool SPLIT, bool DUMP> hipError_t launch_s(const GArgsDump &a, const GPlan &g, hipStream_t s)
{
    auto kern = k_stream_gw<FB, PK, PPG, RS, QIN, SPLIT, DUMP>;
    static std::atomic<uint64_t> opted{0};
    if (const hipError_t e = lds_opt_in(reinterpret_cast<const void *>(kern), 160 * 1024, opted)) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)(SPLIT ? a.nbn : (a.nbn + g.w - 1) / g.w), (unsigned)g.np), dim3(g.w * 64), g.lds, s,
                       static_cast<const std::conditional_t<DUMP, GArgsDump, GArgs> &>(a));
    return hipGetLastError();
}

template <Fmt FB, int PK, int PPG, bool RS, int QIN> hipError_t launch_k(const GArgsDump &a, const GPlan &g, hipStream_t s)
{
    if constexpr (QIN == 0)
        if (g.dump) {
            if constexpr (PPG != 0)
                if (g.split) return launch_s<FB, PK, PPG, RS, QIN, true, true>(a, g, s);
            return launch_s<FB, PK, PPG, RS, QIN, false, true>(a, g, s);
        }
    if constexpr (PPG != 0)
        if (g.split) return launch_s<FB, PK, PPG, RS, QIN, true, false>(a, g, s);
    return launch_s<FB, PK, PPG, RS, QIN, false, false>(a, g, s);
}

template <Fmt FB, int PK, int PPG> hipError_t launch_q(const GArgsDump &a, const GPlan &g, bool rs, int qa, hipStream_t s)
{
    if (!rs) return launch_k<FB, PK, PPG, false, 0>(a, g, s);
    if (qa == 1) return launch_k<FB, PK, PPG, true, 1>(a, g, s);
    if constexpr (FB == Fmt::I8)   // fp16 rows: the grouped int8 entries
        if (qa == 2) return launch_k<FB, PK, PPG, true, 2>(a, g, s);
    return qa ? hipErrorInvalidValue : launch_k<FB, PK, PPG, true, 0>(a, g, s);
}

template <Fmt FB, int PK> hipError_t launch_pk(const GArgsDump &a, const GPlan &g, const Launch &L)
{
    const bool rs = L.rowscale != 0;
    if (a.ppg == 1) return launch_q<FB, PK, 1>(a, g, rs, L.qa, L.stream);
    if (a.ppg == 2) return launch_q<FB, PK, 2>(a, g, rs, L.qa, L.stream);
    return launch_q<FB, PK, 0>(a, g, rs, L.qa, L.stream);
}

}  // namespace

bool stream_gw_takes(const Launch &L, int maxM)
{
    GPlan g;
    GArgs a;
    return plan_gw(L, maxM, g, a);
}

hipError_t stream_gw_launch(const Launch &L, int maxM, uint64_t *blocks)
{
    GPlan g;
    GArgsDump a = {};
    if (!plan_gw(L, maxM, g, a)) return hipErrorInvalidValue;
    a.N = L.N;
    a.K = L.K;
    a.ldb = (uint32_t)row_bytes(L.fmt_b, L.K);
    a.f16out = L.f16out;
    a.act = L.act;
    int n = 0;
    for (int i = 0; i < L.nprob; i++) {
        const Problem &P = L.prob[i];
        if (P.M == 0) continue;
        a.M[n] = P.M;
        a.A[n] = P.A;
        a.A2[n] = L.qa ? P.A2 : nullptr;
        a.B[n] = P.B;
        a.as[n] = P.a_scale;
        a.bs[n] = P.b_scale;
        a.C[n] = P.C;
        a.dump[n] = FewDump{P.dump, P.dump_row0, P.dump_rows};
        n++;
    }
    *blocks = (uint64_t)(g.split ? a.nbn : (a.nbn + g.w - 1) / g.w) * g.np;
    if (L.fmt_b == Fmt::I4P) {
        if (g.pk == 128) return launch_pk<Fmt::I4P, 128>(a, g, L);
        return g.pk == 64 ? launch_pk<Fmt::I4P, 64>(a, g, L) : launch_pk<Fmt::I4P, 32>(a, g, L);
    }
    return g.pk == 64 ? launch_pk<Fmt::I8, 64>(a, g, L) : launch_pk<Fmt::I8, 32>(a, g, L);
}

}  // namespace gk
}  // namespace rk
