// attn_decode.hip — attention of few query rows (decode steps) for gfx950.
//
// A KV head's query rows, the tokens of every query head that reads it, are at most 16 here, so
// the tiled kernel's 128-query workgroups (attn.hip) would be mostly padding; what bounds the
// call is how fast K and V arrive. A workgroup owns a KV head and a range of its keys; each of
// its 4 waves takes chunks of 32 keys and loads their K rows and V^T columns straight into
// registers as MFMA fragments, 32 KB of them in flight a wave at head size 256, next chunk's K
// while this chunk's scores and outputs are formed. All of a KV head's query rows share one
// read of its keys. V^T rows of any length are read in place: no padded copy. (Rows at
// 4-byte addresses cost nothing here; an odd number of keys, rows at 2-byte ones, up to twice the time of a
// chunk.)
//
// Scores are transposed, S^T = K Q^T (v_mfma_f32_16x16x32_f16, K the first operand): lane l
// holds query l % 16. The 16 rows of K block b are keys 8 (i / 4) + 4 b + i % 4, so that lane
// quarter q ends up with keys 8 q .. 8 q + 7 of the chunk, which is what the second product's
// operand takes: O^T += V^T P^T, P rounded to fp16 in registers. The waves' outputs merge in
// LDS, the workgroups' in k_fa_merge; a short cache is one workgroup's, and has no merge.
//
// Measured (sets of operands in turn; before, with attn.hip; after):
//   1 x 3000 keys, 16 / 8 heads of 256    31.6 -> 10.8 us  (24.6 MB of K and V; 8.0 us the kernel, 3.1 TB/s)
//   1 x 4096 keys, 32 / 8 heads of 128    18.2 ->  8.8
//   8 x 3000 keys, 16 / 8 heads of 256    33.5 -> 14.2     (with a mask)
#include "attn.h"
#include "lds_optin.h"

#include <algorithm>
#include <atomic>

namespace rk {
namespace {

typedef int      i32x4  __attribute__((ext_vector_type(4)));
typedef float    f32x2  __attribute__((ext_vector_type(2)));
typedef float    f32x4  __attribute__((ext_vector_type(4)));
typedef _Float16 f16x4  __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8  __attribute__((ext_vector_type(8)));
typedef __amdgpu_buffer_rsrc_t Rsrc;
// eight halves at any 2-byte address
struct __attribute__((packed, aligned(2))) Halves8 { i32x4 v; };

constexpr int kRows = 16, kChunk = 32, kWaves = 4;
constexpr float kLog2e = 1.4426950408889634f;

__device__ __forceinline__ Rsrc rsrc(const void *base, uint32_t bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ i32x4 ld16(Rsrc r, uint32_t off)
{
    return __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}

struct RowArgs {
    const _Float16 *Q, *K, *Vt, *mask;
    _Float16 *O;
    long q_hs, q_rs, k_hs, k_rs, v_hs, v_rs, o_hs, o_rs, m_rs;
    int T, n_kv, dk, dv, gqa, n_head;
    float scale, softcap;
    int nsplit, cps;   // workgroups a KV head, chunks a workgroup
    float *part;       // [split][head][T][dv] outputs, then [split][head][T] (max, sum)
};

// Halves key .. key + 8 of a row of n (n >= 8), zeros past the row: the last eight are loaded
// and shifted where the row ends inside. No branch: one around each of a chunk's loads made them wait
// for each other (1 x 255 keys in one workgroup a head, heads of 256: 20.8 -> 18.8 us).
__device__ __forceinline__ i32x4 row8(const _Float16 *row, int key, int n)
{
    const i32x4 v = reinterpret_cast<const Halves8 *>(row + min(key, n - 8))->v;
    const int past = max(key + 8 - n, 0), s = 16 * (past & 3);   // halves past the row's end
    unsigned long lo = (unsigned)v[0] | ((unsigned long)(unsigned)v[1] << 32);
    unsigned long hi = (unsigned)v[2] | ((unsigned long)(unsigned)v[3] << 32);
    lo = past >= 8 ? 0 : (past >= 4 ? hi : lo);
    hi = past >= 4 ? 0 : hi;
    lo = (lo >> s) | ((hi << 1) << (63 - s));
    hi >>= s;
    return i32x4{(int)(unsigned)lo, (int)(lo >> 32), (int)(unsigned)hi, (int)(hi >> 32)};
}

// Merges the splits, one (head, token) row a workgroup: out = sum_s w_s On_s / sum_s w_s with
// w_s = 2^(m_s - m) l_s, for up to 64 splits. The outputs are fp32, as one workgroup without splits
// holds them: caches from 257 keys on are split here, and a rounding of each split's output to fp16
// beside those of the probabilities and of the result would cost a quarter more error (448 keys, heads
// of 256: 2.5e-4 of the result, with it 3.2e-4). The splits spread over
// the workgroup's 256 threads (dv / 8 threads a split), whose sums add in LDS. (A merge by each KV
// head's last workgroup instead of this launch, on an arrival counter, measured 15.5 against 11.1
// us at 3000 keys: the counter's release and acquire write back and invalidate the XCD's L2, and
// one workgroup walks all rows.)
__global__ __launch_bounds__(256) void k_fa_merge(const float *__restrict__ part, _Float16 *__restrict__ O, long o_hs, long o_rs,
                                                  int n_head, int T, int dv, int nsplit)
{
    __shared__ float wt[64], sum[8 * 256];
    const int tid = threadIdx.x, row = blockIdx.x, h = row / T, t = row - h * T;
    const size_t rows = (size_t)n_head * T;
    const int dq = dv / 8, sg = tid / dq, d0 = (tid - sg * dq) * 8, ng = min(8, 256 / dq);   // dv <= 256: 8
    f32x4 os[8][2];
    if (sg < ng)
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int s = sg + i * ng;
            if (s < nsplit)
#pragma unroll
                for (int j = 0; j < 2; j++) os[i][j] = reinterpret_cast<const f32x4 *>(part + ((size_t)s * rows + row) * dv + d0)[j];
        }
    if (tid < 64) {
        const f32x2 x = tid < nsplit ? reinterpret_cast<const f32x2 *>(part + (size_t)nsplit * rows * dv)[(size_t)tid * rows + row]
                                     : f32x2{-INFINITY, 0.f};
        float m = x[0];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
        const float w = __builtin_amdgcn_exp2f(x[0] - m) * x[1];
        float l = w;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o, 64);
        wt[tid] = l > 0.f ? w / l : 0.f;
    }
    __syncthreads();
    if (sg < ng) {
        float acc[8] = {};
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int s = sg + i * ng;
            if (s < nsplit)
#pragma unroll
                for (int e = 0; e < 8; e++) acc[e] += wt[s] * os[i][e >> 2][e & 3];
        }
#pragma unroll
        for (int e = 0; e < 8; e++) sum[sg * dv + d0 + e] = acc[e];
    }
    __syncthreads();
    for (int d = tid; d < dv; d += 256) {
        float o = 0.f;
        for (int s = 0; s < ng; s++) o += sum[s * dv + d];
        O[(size_t)h * o_hs + (size_t)t * o_rs + d] = (_Float16)o;
    }
}

// D: head sizes up to this (64, 128, 256); dk a multiple of 32, dv of 16. FULL: both are D, so
// that no load or product carries a test of its dims.
template <int D, bool CAP, bool FULL>
__global__ __launch_bounds__(kWaves * 64) void k_fa_rows(const RowArgs a)
{
    constexpr int KS = D / 32, VB = D / 16, LROW = D + 4;   // score steps, output blocks, LDS row (floats)
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, q = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int hk = blockIdx.x, zs = blockIdx.y;
    const int R = a.gqa * a.T;
    const int hg = c / a.T, t = c - hg * a.T;               // this lane's query: head hk gqa + hg, token t
    const bool qok = c < R;

    i32x4 qf[KS];
    {
        const _Float16 *qrow = a.Q + (size_t)(hk * a.gqa + (qok ? hg : 0)) * a.q_hs + (size_t)(qok ? t : 0) * a.q_rs;
#pragma unroll
        for (int s = 0; s < KS; s++)
            qf[s] = (qok && (FULL || 32 * s < a.dk)) ? *reinterpret_cast<const i32x4 *>(qrow + 32 * s + 8 * q) : i32x4{0, 0, 0, 0};
    }
    const Rsrc rk = rsrc(a.K + (size_t)hk * a.k_hs, (uint32_t)((long)a.n_kv * a.k_rs * 2));   // keys past n_kv: zeros
    const _Float16 *const Vh = a.Vt + (size_t)hk * a.v_hs + (size_t)c * a.v_rs;              // rows 16 j + c
    const _Float16 *const mrow = a.mask ? a.mask + (size_t)t * a.m_rs : nullptr;

    i32x4 kf[2][KS], vf[VB];
    const uint32_t ko = (uint32_t)((8 * (c >> 2) + (c & 3)) * a.k_rs + 8 * q) * 2u, k4 = (uint32_t)(4 * a.k_rs) * 2u;
    auto load_k = [&](int key0) __attribute__((always_inline)) {
        const uint32_t o = ko + (uint32_t)((long)key0 * a.k_rs * 2);
#pragma unroll
        for (int s = 0; s < KS; s++)
            if (FULL || 32 * s < a.dk) {
                kf[0][s] = ld16(rk, o + 64u * s);
                kf[1][s] = ld16(rk, o + k4 + 64u * s);
            }
    };
    auto load_v = [&](int key0) __attribute__((always_inline)) {
        const int key = key0 + 8 * q;
        if (key0 + kChunk <= a.n_kv) {   // uniform: whole chunks
#pragma unroll
            for (int j = 0; j < VB; j++)
                if (FULL || 16 * j < a.dv) vf[j] = reinterpret_cast<const Halves8 *>(Vh + (size_t)(16 * j) * a.v_rs + key)->v;
        } else {
#pragma unroll
            for (int j = 0; j < VB; j++)
                if (FULL || 16 * j < a.dv) vf[j] = row8(Vh + (size_t)(16 * j) * a.v_rs, key, a.n_kv);
        }
    };

    float m_run = -INFINITY, l_run = 0.f;
    f32x4 O[VB];
#pragma unroll
    for (int j = 0; j < VB; j++) O[j] = f32x4{};
    const int chunks = (a.n_kv + kChunk - 1) / kChunk;
    const int c1 = min(chunks, (zs + 1) * a.cps);
    int ch = zs * a.cps + wave;
    if (ch < c1) {
        load_k(ch * kChunk);
        load_v(ch * kChunk);
    }
    for (; ch < c1; ch += kWaves) {
        const int key0 = ch * kChunk;
        f32x4 S[2] = {};
#pragma unroll
        for (int s = 0; s < KS; s++)
            if (FULL || 32 * s < a.dk) {
#pragma unroll
                for (int b = 0; b < 2; b++)
                    S[b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, kf[b][s]), __builtin_bit_cast(f16x8, qf[s]),
                                                                  S[b], 0, 0, 0);
            }
        const bool more = ch + kWaves < c1;
        if (more) load_k(key0 + kWaves * kChunk);
        // the reference's score steps in log2 units; lane holds keys key0 + 8 q + 4 b + e
        i32x4 mw = {0, 0, 0, 0};
        if (mrow) mw = row8(mrow, key0 + 8 * q, a.n_kv);
        const f16x8 mv = __builtin_bit_cast(f16x8, mw);
        float v[8], mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float x = S[i >> 2][i & 3];
            if constexpr (CAP) v[i] = fmaxf(a.softcap * tanhf(x * a.scale / a.softcap) + (float)mv[i], -30000.f) * kLog2e;
            else v[i] = fmaxf(fmaf((float)mv[i], kLog2e, x * (a.scale * kLog2e)), -30000.f * kLog2e);
            if (key0 + 8 * q + i >= a.n_kv) v[i] = -INFINITY;   // weighs 0
            mx = fmaxf(mx, v[i]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        if (__any(mx > m_run)) {   // (a chunk has a key below n_kv, so the new maximum is finite)
            const float m_new = fmaxf(m_run, mx), alpha = __builtin_amdgcn_exp2f(m_run - m_new);
            m_run = m_new;
            l_run *= alpha;
#pragma unroll
            for (int j = 0; j < VB; j++) O[j] *= alpha;
        }
        f16x8 p;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float e = __builtin_amdgcn_exp2f(v[i] - m_run);
            l_run += e;
            p[i] = (_Float16)e;
        }
#pragma unroll
        for (int j = 0; j < VB; j++)
            if (FULL || 16 * j < a.dv) O[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, vf[j]), p, O[j], 0, 0, 0);
        if (more) load_v(key0 + kWaves * kChunk);
    }
    l_run += __shfl_xor(l_run, 16, 64);
    l_run += __shfl_xor(l_run, 32, 64);

    // merge the waves: [wave][row][LROW] outputs, then [wave][row] (max, sum)
    float *const Ol = reinterpret_cast<float *>(smem);
    f32x2 *const ml = reinterpret_cast<f32x2 *>(Ol + kWaves * R * LROW);
    if (qok) {
#pragma unroll
        for (int j = 0; j < VB; j++)
            if (FULL || 16 * j < a.dv) *reinterpret_cast<f32x4 *>(Ol + (wave * R + c) * LROW + 16 * j + 4 * q) = O[j];
        if (q == 0) ml[wave * R + c] = f32x2{m_run, l_run};
    }
    __syncthreads();
    const int dq = a.dv / 4;
    for (int i = tid; i < R * dq; i += kWaves * 64) {
        const int r = i / dq, d0 = (i - r * dq) * 4;
        float m = -INFINITY;
#pragma unroll
        for (int w = 0; w < kWaves; w++) m = fmaxf(m, ml[w * R + r][0]);
        float l = 0.f;
        f32x4 o = {};
#pragma unroll
        for (int w = 0; w < kWaves; w++) {
            const f32x2 x = ml[w * R + r];
            // (a wave without keys: 2^-inf = 0)
            const float f = __builtin_amdgcn_exp2f(x[0] - m);
            l += f * x[1];
            o += f * *reinterpret_cast<const f32x4 *>(Ol + (w * R + r) * LROW + d0);
        }
        const float inv = l > 0.f ? 1.f / l : 0.f;
        const int g = r / a.T, tt = r - g * a.T, h = hk * a.gqa + g;
        if (a.nsplit > 1) {
            const size_t row = ((size_t)zs * a.n_head + h) * a.T + tt;
            *reinterpret_cast<f32x4 *>(a.part + row * a.dv + d0) = o * inv;
            if (d0 == 0) reinterpret_cast<f32x2 *>(a.part + (size_t)a.nsplit * a.n_head * a.T * a.dv)[row] = f32x2{m, l};
        } else {
            f16x4 out;
#pragma unroll
            for (int e = 0; e < 4; e++) out[e] = (_Float16)(o[e] * inv);
            *reinterpret_cast<f16x4 *>(a.O + (size_t)h * a.o_hs + (size_t)tt * a.o_rs + d0) = out;
        }
    }
}

template <int D, bool CAP, bool FULL> hipError_t launch_rows_f(const RowArgs &a, int kv_heads, hipStream_t s)
{
    auto kern = k_fa_rows<D, CAP, FULL>;
    const int R = a.gqa * a.T;
    const size_t lds = (size_t)kWaves * R * ((D + 4) * 4 + 8);
    if (lds > 64 * 1024) {
        static std::atomic<uint64_t> opted{0};
        if (const hipError_t e = lds_opt_in(reinterpret_cast<const void *>(kern), 80 * 1024, opted)) return e;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)kv_heads, (unsigned)a.nsplit), dim3(kWaves * 64), lds, s, a);
    return hipGetLastError();
}

template <int D> hipError_t launch_rows(const RowArgs &a, int kv_heads, hipStream_t s)
{
    const bool cap = a.softcap != 0.f;
    if (a.dk == D && a.dv == D) return cap ? launch_rows_f<D, true, true>(a, kv_heads, s) : launch_rows_f<D, false, true>(a, kv_heads, s);
    return cap ? launch_rows_f<D, true, false>(a, kv_heads, s) : launch_rows_f<D, false, false>(a, kv_heads, s);
}

// Workgroups a KV head: one chunk a wave while the workgroups stay near three a CU; one workgroup for
// short caches, where the merge's launch costs more than the waves' further chunks (one token, 32 heads
// of 64, 192 keys 4.3 us, split 7.0; 512 keys 6.4 and 7.1; heads of 128, 320 keys 7.5 and 8.3, 384 keys
// 8.1 and 8.3; heads of 256, 256 keys 10.2 and 10.5, 320 keys 12.2 and 10.5); fewer chunks with an odd
// number of keys, whose loads take longer (heads of 64, 319 keys 7.7 and 8.1, 383 keys 8.7 and 8.3; heads of
// 128, 255 keys 10.6 and 10.4, 319 keys 12.6 and 10.2; heads of 256, 159 keys 9.8 and 10.6, 191 keys 15.0
// and 12.8, 255 keys 18.8 and 14.6).
void split_of(const FaLaunch &L, int *nsplit, int *cps)
{
    const int kvh = L.n_head / L.gqa, chunks = (L.n_kv + kChunk - 1) / kChunk;
    const int d = std::max(L.dk, L.dv), odd = L.n_kv & 1;
    const int whole = d <= 64 ? (odd ? 10 : 16) : d <= 128 ? (odd ? 8 : 10) : odd ? 5 : 8;
    const int n = chunks <= whole ? 1 : std::min({(chunks + kWaves - 1) / kWaves, std::max(1, 768 / kvh), 64});
    *cps = (chunks + n - 1) / n;
    *nsplit = (chunks + *cps - 1) / *cps;
}

}  // namespace

bool flash_attn_few_rows(const FaLaunch &L)
{
    if ((long)L.gqa * L.T > kRows || L.n_kv < 8 || L.dk % 32 || L.dv % 16) return false;
    // One query head a KV head and long caches: the tiled kernel reads V^T in whole 128-byte lines (64
    // keys a tile, 32 here), and where its workgroups fill the CUs and nothing has to be padded it is the
    // faster one while the cache is not far larger than the memory-side cache (heads of 256, 16 x 8192
    // keys 28.9 us, here 33.0; 32 x 8192 54.8 and 62.8, 32 x 32768 212 and 200; heads of 128, 32 x 8192 28.3
    // and 30.7; 24 heads, whose 264 workgroups are two rounds, 8192 keys 69 and 48.6).
    const int d = std::max(L.dk, L.dv);
    const size_t kv = (size_t)L.n_head / L.gqa * L.n_kv * (L.dk + L.dv) * sizeof(_Float16);
    return !(L.gqa == 1 && d > 64 && L.n_kv % 8 == 0 && kv >= ((size_t)(d > 128 ? 64 : 96) << 20) && kv <= ((size_t)512 << 20) &&
             flash_attn_tiles_fill(L));
}

size_t flash_attn_rows_ws(const FaLaunch &L)
{
    int n, cps;
    split_of(L, &n, &cps);
    return n > 1 ? (size_t)n * L.n_head * L.T * (L.dv + 2) * sizeof(float) : 0;
}

hipError_t flash_attn_rows(const FaLaunch &L, hipStream_t s, uint64_t *blocks)
{
    RowArgs a;
    a.Q = L.Q; a.K = L.K; a.Vt = L.Vt; a.mask = L.mask; a.O = L.O;
    a.q_hs = L.q_hs; a.q_rs = L.q_rs; a.k_hs = L.k_hs; a.k_rs = L.k_rs; a.v_hs = L.v_hs; a.v_rs = L.v_rs;
    a.o_hs = L.o_hs; a.o_rs = L.o_rs; a.m_rs = L.m_rs;
    a.T = L.T; a.n_kv = L.n_kv; a.dk = L.dk; a.dv = L.dv; a.gqa = L.gqa; a.n_head = L.n_head;
    a.scale = L.scale; a.softcap = L.softcap;
    split_of(L, &a.nsplit, &a.cps);
    if (a.nsplit > 1 && (!L.ws || L.ws_bytes < flash_attn_rows_ws(L))) {
        a.nsplit = 1;
        a.cps = (L.n_kv + kChunk - 1) / kChunk;
    }
    a.part = L.ws;
    const int kvh = L.n_head / L.gqa;
    const int d = std::max(L.dk, L.dv);
    const hipError_t e = d <= 64 ? launch_rows<64>(a, kvh, s) : d <= 128 ? launch_rows<128>(a, kvh, s) : launch_rows<256>(a, kvh, s);
    if (blocks) *blocks = (uint64_t)kvh * a.nsplit;
    if (e != hipSuccess || a.nsplit == 1) return e;
    const unsigned rows = (unsigned)(L.n_head * L.T);
    hipLaunchKernelGGL(k_fa_merge, dim3(rows), dim3(256), 0, s, a.part, L.O, L.o_hs, L.o_rs, L.n_head, L.T, L.dv, a.nsplit);
    if (blocks) *blocks += rows;
    return hipGetLastError();
}

}  // namespace rk
