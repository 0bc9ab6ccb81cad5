// matmul.cpp — the one-shot matmul entries of rocket_matmul.h and their planners.
//
// Each entry keeps the reference's validation and return codes (reference
// src/rocket_matmul.c; lines cited per entry) and runs one gfx950 kernel launch
// (gemm.hip) on the handle's stream through rk::run.
#include "ops.h"
#include "rocket_hip.h"
#include "rocket_hw_profile.h"
#include "rocket_matmul.h"

#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <memory>
#include <new>
#include <vector>

namespace rk {

size_t fmt_row_bytes(Fmt f, int K)
{
    switch (f) {
    case Fmt::I8: return (size_t)K;
    case Fmt::I4P: return (size_t)K / 2;
    case Fmt::I16: case Fmt::F16: case Fmt::BF16: return 2 * (size_t)K;
    case Fmt::F32BF16: case Fmt::F32TF32: case Fmt::BF16X2: return 4 * (size_t)K;
    }
    return 0;
}

size_t epi_elem_bytes(Epi e)
{
    switch (e) {
    case Epi::I32: return 4;
    case Epi::I64: return 8;
    case Epi::F16: case Epi::GLU: case Epi::ACT: return 2;
    case Epi::F32: case Epi::GW: return 4;
    }
    return 0;
}

// n fp32 values at device address src (and n2 at src2, when src2 is given) converted into
// arena scratch in one launch; false on failure (the Call then carries the error).
static bool convert(Call &c, const void *src, size_t n, Fmt to, const void **out, const void *src2 = nullptr,
                    size_t n2 = 0, const void **out2 = nullptr)
{
    const size_t el = to == Fmt::BF16X2 ? 4 : 2;
    void *dst = c.scratch(n * el);
    void *dst2 = src2 ? c.scratch(n2 * el) : nullptr;
    if (!dst || (src2 && !dst2)) return false;
    if (convert_f32(static_cast<const float *>(src), dst, (long)n, to, c.stream(), static_cast<const float *>(src2),
                    dst2, src2 ? (long)n2 : 0) != hipSuccess) {
        (void)hipGetLastError();
        ROCKET_LOGE("%s: fp32 conversion launch failed\n", c.who());
        return false;
    }
    count_launch((uint64_t)((n / 8 + (src2 ? n2 / 8 : 0) + 255) / 256));
    *out = dst;
    if (src2) *out2 = dst2;
    return true;
}

int gw_period(int group)
{
    if (group <= 65536) return group;
    for (int d = 65536 / 32 * 32; d >= 32; d -= 32)
        if (group % d == 0) return d;
    return 32;
}

// Whether a result of the call lies over rows (A, A2) of it. The ranges are walked in the order of
// their starts: one that starts below the furthest end so far of the other kind lies over it (pair by
// pair, 256 products took 196 us).
bool results_overlap_rows(const Req &r, size_t a_row, size_t c_elem)
{
    struct Range {
        uintptr_t at, end;
        bool result;
        bool operator<(const Range &o) const { return at < o.at; }
    };
    constexpr int kFew = 24;
    Range few[kFew];
    std::unique_ptr<Range[]> many;
    Range *v = few;
    if (r.nprob > kFew / 3) {
        many.reset(new (std::nothrow) Range[(size_t)r.nprob * 3]);
        if (!(v = many.get())) return true;   // (no host memory: as if they did, which is right for all)
    }
    size_t n = 0;
    for (int p = 0; p < r.nprob; p++) {
        const size_t na = (size_t)r.M[p] * a_row, nc = (size_t)r.M[p] * r.N * c_elem;
        if (!na || !nc) continue;
        const auto add = [&](const void *x, size_t bytes, bool result) { v[n++] = {(uintptr_t)x, (uintptr_t)x + bytes, result}; };
        add(r.A[p], na, false);
        if (r.A2) add(r.A2[p], na, false);
        add(r.C[p], nc, true);
    }
    // (mostly the rows lie together and the results lie together)
    uintptr_t lo[2] = {~(uintptr_t)0, ~(uintptr_t)0}, hi[2] = {0, 0};
    for (size_t i = 0; i < n; i++) {
        lo[v[i].result] = std::min(lo[v[i].result], v[i].at);
        hi[v[i].result] = std::max(hi[v[i].result], v[i].end);
    }
    if (n == 0 || hi[0] <= lo[1] || hi[1] <= lo[0]) return false;
    std::sort(v, v + n);
    uintptr_t end[2] = {0, 0};   // furthest end of the rows, of the results
    for (size_t i = 0; i < n; i++) {
        if (v[i].at < end[!v[i].result]) return true;
        end[v[i].result] = std::max(end[v[i].result], v[i].end);
    }
    return false;
}

// fp32 operands (bf16 / tf32 entries) are either converted as the GEMM loads them, or
// converted first in one streaming pass into the handle's arena (bf16: half the bytes;
// tf32: hi/lo pairs), so the GEMM moves half the bytes through L2 (bf16) and spends no VALU
// on the conversion. The pass costs one extra read + write of the operand, so it pays for
// an operand whose rows many tiles re-read: A (read once per 128-column tile) from N >= 384,
// B (read once per 256-row tile) from M >= 2048 (measured on MI355X: A alone is 5-25%
// faster than neither from M = 64 up; both are 1.4-2.3x faster from M = 2048 up, A alone
// up to M = 1024). Returns 0 (no pass), 1 (both operands) or 2 (A only).
// ROCKET_HIP_F32_PREPASS = 0 / 1 / 2 forces a choice (read per call). All give identical bits.
int f32_prepass(const Req &r)
{
    if (r.fa != Fmt::F32BF16 && r.fa != Fmt::F32TF32) return 0;
    if (const char *e = getenv("ROCKET_HIP_F32_PREPASS")) {
        if (e[0] >= '0' && e[0] <= '2' && e[1] == 0) return e[0] - '0';
    }
    int maxM = 0;
    for (int p = 0; p < r.nprob; p++) maxM = std::max(maxM, r.M[p]);
    // (with few columns, or few values, the pass's own launch costs more than it saves: tf32 700 x
    // 2528 x 272 25.6 us with it, 20.3 without; 128 x 2048 x 2048 17.5 and 16.0; 128 x 4096 x 4096
    // 30.6 and 33.4. Few values that many columns' tiles read again are worth it all the same: tf32 256 x
    // 1024 x 8192 25.1 with it, 27.7 without; 2044 x 128 x 8192 35.7 and 42.2; 20 x 2048 x 16384 39.1 and
    // 48.3; 64 x 2048 x 8192 22 and 21.2; bf16, whose conversion in the loads is cheaper, 512 x 512 x
    // 16384 24.8 and 27.7; 64 x 4096 x 8192 35.0 and 45.5; 256 x 512 x 8192 13 and 12. tf32: where the
    // tiles nearly fill the CUs no K slices shorten their chain, and the conversion is in it (20 x 3840 x
    // 14336 67.4 us with it, 85.8 without, 100 x 3840 x 10240 71.2 and 87.2; in slices 20 x 3840 x 12288 is 1.06
    // times as long with it); likewise where they are more than the CUs (1040 x 256 x 7792 36.5 and 42.3, 944 x
    // 128 x 5312 19.8 and 21.9; 512 x 128 x 7792, in one round, 1.04 times as long with it). bf16, few
    // rows: 20 x 3072 x 10240 31.0 and 36.6, 20 x 3840 x 20480 76.6 and 84.4, 100 x 1536 x 20480 32.1 and 39.2, 20 x
    // 512 x 32768 21.6 and 23.6; 20 x 1024 x 24576 1.01 times as long with it)
    const long mk = (long)maxM * r.K, N = r.N, K = r.K;
    bool pays = N >= 384 && mk >= 400000;
    Launch L;   // the product on unconverted rows
    L.fmt_a = r.fa; L.fmt_b = r.fb; L.epi = r.epi; L.N = r.N; L.K = L.kend = r.K;
    L.nprob = 1;
    L.prob[0].M = maxM;
    if (r.fa == Fmt::F32TF32)
        pays = pays || (K >= 64 && (long)((maxM + 127) / 128) * ((N + 127) / 128) > 256) ||
               (N >= 4096 && maxM >= 128 && mk * N >= 900000000L) || (K >= 256 && N > 16384) ||
               (N >= 6144 && K >= 512 && maxM > 128) ||
               (((N >= 8192 && K >= 512) || (N >= 3072 && K >= 1024)) && gemm_ws_bytes(L) == 0);
    else
        pays = pays || (N >= 384 && mk * N >= 2600000000L) || (N > 28672 && K >= 512) || (N > 32768 && K >= 256) || (N > 16384 && K >= 1536) ||
               (N > 8192 && N < 16384 && K >= (N > 12288 ? 2048 : 1536)) ||
               (N >= 4096 && N <= 8192 && (K >= 2560 || (K >= 2048 && mk >= 80000)));
    if (pays) pays = !gemm_streams(L);   // few rows: the weight-streaming kernel converts as it loads
    // (results stored over the rows: with the pass every row has been read before the first of them)
    if (!pays) return r.N >= 256 && results_overlap_rows(r, (size_t)r.K * 4, 4) ? 2 : 0;
    return (maxM >= 2048 && r.N >= 2048) ? 1 : 2;
}

int run(int fd, const Req &r)
{
    Locked L(fd);
    if (!L.ok()) {
        ROCKET_LOGE("%s: fd %d is not an open rocket handle\n", r.who, fd);
        return ROCKET_E_DEVICE;
    }
    if (r.nprob < 1) return ROCKET_E_SHAPE;
    const int nG = r.group ? r.K / r.group : 0;
    const bool gw = (r.epi == Epi::GW);
    // B as it arrives from the caller: int8 per value when we pack it ourselves
    const size_t brow_in = r.pack_b_int4 ? (size_t)r.K : fmt_row_bytes(r.fb, r.K);
    int prepass = f32_prepass(r);
    const Fmt cvt = r.fa == Fmt::F32TF32 ? Fmt::BF16X2 : Fmt::BF16;
    // (a capture cannot grow the arena for converted rows: the product converts them as it loads them, the
    // same bits, unless its results lie over them)
    if (prepass == 2) {
        size_t rows = 0;
        for (int p = 0; p < r.nprob; p++) rows += ((size_t)std::max(r.M[p], 0) * fmt_row_bytes(cvt, r.K) + 255) & ~(size_t)255;
        if (rows > L.h->arena_cap && stream_capturing(L.h->stream) && !results_overlap_rows(r, (size_t)r.K * 4, 4)) prepass = 0;
    }
    const Fmt fa_dev = prepass ? cvt : r.fa;
    const Fmt fb_dev = r.pack_b_int4 ? Fmt::I4P : (prepass == 1 ? cvt : r.fb);

    // quantised-on-device activations: bytes per source element, and the pre-pass plan
    const size_t qa_bytes = r.quant_a == 1 ? 4 : (r.quant_a == 2 ? 2 : 0);
    if (qa_bytes && (!gw || !r.rowscale || r.fa != Fmt::I8 || r.K % 8)) return ROCKET_E_SHAPE;
    const bool glu_in = r.act != 0;
    if (glu_in && (!qa_bytes || !r.A2)) return ROCKET_E_SHAPE;
    if (r.f16out && !gw) return ROCKET_E_SHAPE;
    const size_t c_elem = r.f16out ? 2 : epi_elem_bytes(r.epi);
    const size_t a_row_in = qa_bytes ? qa_bytes * r.K : fmt_row_bytes(r.fa, r.K);

    // few rows: the product quantises them itself (every launch of the call, or none)
    // (where that is the shorter way, or a capture cannot grow the arena for the codes)
    size_t codes = 0;
    for (int p = 0; p < r.nprob; p++) codes += (size_t)std::max(r.M[p], 0) * (r.K + sizeof(float));
    const int must = qa_bytes && codes > L.h->arena_cap && stream_capturing(L.h->stream);
    bool fuse = qa_bytes != 0;
    for (int p0 = 0; fuse && p0 < r.nprob; p0 += kMaxProblems) {
        Launch Lq;
        Lq.fmt_a = r.fa; Lq.fmt_b = fb_dev; Lq.epi = r.epi; Lq.N = r.N; Lq.K = Lq.kend = r.K;
        Lq.group = r.group; Lq.kt = gw_period(r.group); Lq.rowscale = 1; Lq.qa = r.quant_a; Lq.act = r.act;
        Lq.qa_must = must;
        Lq.nprob = std::min(kMaxProblems, r.nprob - p0);
        int rows = 0;
        for (int q = 0; q < Lq.nprob; q++) rows += Lq.prob[q].M = r.M[p0 + q];
        fuse = rows == 0 || gemm_quantises(Lq);
    }
    // (a pass of its own has read every row before the first result is stored)
    if (fuse && results_overlap_rows(r, a_row_in, c_elem)) fuse = false;

    Call c(L.h, r.who);
    for (int p = 0; p < r.nprob; p++) {
        const size_t M = (size_t)r.M[p];
        if (M == 0) continue;
        c.want(r.A[p], M * a_row_in);
        if (glu_in) c.want(r.A2[p], M * a_row_in);
        if (qa_bytes && !fuse) {
            c.want_scratch(M * r.K);
            c.want_scratch(M * sizeof(float));
        }
        c.want(r.B[p], (size_t)r.N * brow_in);
        c.want(r.C[p], M * r.N * c_elem);
        if (gw) {
            if (!qa_bytes) c.want(r.a_scale[p], M * (r.rowscale ? 1 : nG) * sizeof(float));
            c.want(r.b_scale[p], (size_t)r.N * nG * sizeof(float));
        }
        if (r.pack_b_int4) c.want_scratch((size_t)r.N * r.K / 2);
        if (prepass) c.want_scratch(M * fmt_row_bytes(fa_dev, r.K));
        if (prepass == 1) c.want_scratch((size_t)r.N * fmt_row_bytes(fb_dev, r.K));
    }
    auto dump_of = [&](int p) -> int32_t * { return (r.dump && r.dump_rows[p] > 0) ? r.dump[p] : nullptr; };
    auto dump_bytes = [&](int p) { return (size_t)r.dump_rows[p] * nG * r.N * sizeof(int32_t); };
    for (int p = 0; p < r.nprob; p++)
        if (dump_of(p) && r.M[p]) c.want(dump_of(p), dump_bytes(p));
    // split-K workspace (plain int32, fp16 and fp32 results): the largest any launch of the
    // call needs; successive launches reuse it in stream order
    size_t ws = 0;
    if (r.epi == Epi::I32 || r.epi == Epi::F16 || r.epi == Epi::F32) {
        for (int p0 = 0; p0 < r.nprob; p0 += kMaxProblems) {
            Launch Lp;
            Lp.fmt_a = fa_dev; Lp.fmt_b = fb_dev; Lp.epi = r.epi; Lp.N = r.N; Lp.K = r.K;
            Lp.nprob = std::min(kMaxProblems, r.nprob - p0);
            for (int q = 0; q < Lp.nprob; q++) Lp.prob[q].M = r.M[p0 + q];
            Lp.kbeg = 0;
            Lp.kend = (r.kchunk > 0 && r.K > r.kchunk) ? r.kchunk : r.K;
            ws = std::max(ws, gemm_ws_bytes(Lp));
        }
        // (bf16 / tf32 products of few columns, which convert no rows ahead, hold no scratch in a graph)
        ws = c.want_optional(ws, r.fa == Fmt::F16 || r.N >= 256);
    }
    if (int rc = c.begin()) return rc;
    int32_t *wsp = static_cast<int32_t *>(c.optional(ws));

    // launches hold up to kMaxProblems problems each
    for (int p0 = 0; p0 < r.nprob; p0 += kMaxProblems) {
        // the launch's activations quantised per row first (one pre-pass launch)
        QuantRows qr;
        if (qa_bytes && !fuse) {
            qr.n = std::min(kMaxProblems, r.nprob - p0);
            qr.K = r.K;
            qr.f16 = r.quant_a == 2;
            qr.act = r.act;
            for (int i = 0; i < qr.n; i++) {
                const int p = p0 + i;
                qr.M[i] = r.M[p];
                if (!qr.M[i]) continue;
                qr.A[i] = c.in(r.A[p], (size_t)qr.M[i] * a_row_in);
                if (glu_in) {
                    qr.A2[i] = c.in(r.A2[p], (size_t)qr.M[i] * a_row_in);
                    if (!qr.A2[i]) return c.finish();
                }
                qr.Aq[i] = static_cast<int8_t *>(c.scratch((size_t)qr.M[i] * r.K));
                qr.row_scale[i] = static_cast<float *>(c.scratch((size_t)qr.M[i] * sizeof(float)));
                if (!qr.A[i] || !qr.Aq[i] || !qr.row_scale[i]) return c.finish();
            }
            uint64_t qb = 0;
            if (quant_rows(qr, c.stream(), &qb) != hipSuccess) {
                (void)hipGetLastError();
                ROCKET_LOGE("%s: activation quantisation launch rejected\n", r.who);
                (void)c.finish();
                return ROCKET_E_DEVICE;
            }
            count_launch(qb);
        }
        Launch Lc;
        Lc.fmt_a = fa_dev;
        Lc.fmt_b = fb_dev;
        Lc.epi = r.epi;
        Lc.N = r.N;
        Lc.K = r.K;
        Lc.group = r.group;
        Lc.rowscale = r.rowscale;
        Lc.f16out = r.f16out ? 1 : 0;
        Lc.qa = fuse ? r.quant_a : 0;
        Lc.qa_must = must;
        Lc.act = fuse ? r.act : 0;
        Lc.kt = gw ? gw_period(r.group) : 0;
        Lc.ws = wsp;
        Lc.ws_bytes = wsp ? ws : 0;
        Lc.nprob = std::min(kMaxProblems, r.nprob - p0);
        for (int q = 0; q < Lc.nprob; q++) {
            const int p = p0 + q;
            Problem &P = Lc.prob[q];
            P.M = r.M[p];
            P.B2 = nullptr;
            if (P.M == 0) { P.A = P.B = nullptr; P.C = nullptr; P.a_scale = P.b_scale = nullptr; continue; }
            P.A = qa_bytes && !fuse ? qr.Aq[q] : c.in(r.A[p], (size_t)P.M * a_row_in);
            if (fuse && glu_in) {
                P.A2 = c.in(r.A2[p], (size_t)P.M * a_row_in);
                if (!P.A2) return c.finish();
            }
            const void *b = c.in(r.B[p], (size_t)r.N * brow_in);
            if (r.pack_b_int4 && b) {
                void *packed = c.scratch((size_t)r.N * r.K / 2);
                if (packed) {
                    if (pack_int4(static_cast<const int8_t *>(b), static_cast<uint8_t *>(packed), r.N, r.K,
                                  c.stream()) != hipSuccess) {
                        (void)hipGetLastError();
                        ROCKET_LOGE("%s: int4 pack launch failed\n", r.who);
                        return ROCKET_E_DEVICE;
                    }
                    count_launch((uint64_t)(((size_t)r.N * r.K / 8 + 255) / 256));
                }
                b = packed;
            }
            P.B = b;
            if (prepass && P.A && P.B) {
                const bool ok = prepass == 1
                                    ? convert(c, P.A, (size_t)P.M * r.K, fa_dev, &P.A, P.B, (size_t)r.N * r.K, &P.B)
                                    : convert(c, P.A, (size_t)P.M * r.K, fa_dev, &P.A);
                if (!ok) {
                    const int e = c.finish();
                    return e ? e : ROCKET_E_DEVICE;
                }
            }
            P.C = c.out(r.C[p], (size_t)P.M * r.N * c_elem);
            P.a_scale = !gw || fuse ? nullptr
                        : qa_bytes ? qr.row_scale[q]
                                   : static_cast<const float *>(
                                         c.in(r.a_scale[p], (size_t)P.M * (r.rowscale ? 1 : nG) * sizeof(float)));
            P.b_scale = gw ? static_cast<const float *>(c.in(r.b_scale[p], (size_t)r.N * nG * sizeof(float))) : nullptr;
            if (!P.A || !P.B || !P.C || (gw && ((!P.a_scale && !fuse) || !P.b_scale))) return c.finish();
            if (dump_of(p)) {
                P.dump = static_cast<int32_t *>(c.out(dump_of(p), dump_bytes(p)));
                P.dump_row0 = r.dump_row0[p];
                P.dump_rows = r.dump_rows[p];
                if (!P.dump) return c.finish();
            }
        }
        if (r.kchunk > 0 && r.K > r.kchunk) {
            for (int k0 = 0; k0 < r.K; k0 += r.kchunk) {
                Lc.kbeg = k0;
                Lc.kend = std::min(r.K, k0 + r.kchunk);
                Lc.accum = k0 > 0;
                if (c.launch(Lc)) return c.finish();
            }
        } else {
            Lc.kbeg = 0;
            Lc.kend = r.K;
            if (c.launch(Lc)) return c.finish();
        }
    }
    return c.finish();
}

}  // namespace rk

using namespace rk;

namespace {

bool dims_ok(int M, int K, int N)
{
    return M > 0 && K > 0 && N > 0 && M <= kDimMax && K <= kDimMax && N <= kDimMax;
}

// Shared planner body: the reference's alignment test, then the MI355X workgroup tiling.
int plan(int M, int K, int N, int kal, int nal, Fmt fa, Epi epi, int kt, int *pMt, int *pKt, int *pNt)
{
    if (!dims_ok(M, K, N) || K % kal || N % nal || M % 4) return ROCKET_E_SHAPE;
    int bm, bn;
    gemm_tile(fa, epi, M, N, &bm, &bn);
    const long count = (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn);
    if (count > 0x7FFFFFFFL) return ROCKET_E_SHAPE;
    if (pMt) *pMt = std::min(M, bm);
    if (pNt) *pNt = std::min(N, bn);
    if (pKt) *pKt = kt ? kt : K;
    return (int)count;
}

// M==1 is accepted by the one-shot entries (the reference pads it to a 4-row tile,
// rocket_matmul.c:258-267; the kernels here take any M, so the single row is computed
// directly and equals row 0 of the padded product). Other M go through the planner.
int oneshot_shape(int M, int K, int N, int kal, int nal)
{
    if (M == 1) return (dims_ok(1, K, N) && K % kal == 0 && N % nal == 0) ? 0 : ROCKET_E_SHAPE;
    return plan(M, K, N, kal, nal, Fmt::I8, Epi::I32, 0, nullptr, nullptr, nullptr) < 0 ? ROCKET_E_SHAPE : 0;
}

bool dtype_ok(int precision)
{
    return rocket_hw_dtype_supported(rocket_hw_current(), precision);
}

int single(int fd, const char *who, Fmt fa, Fmt fb, Epi epi, int M, int K, int N,
           const void *A, const void *B, void *C)
{
    if (!A || !B || !C) {
        ROCKET_LOGE("%s: NULL operand\n", who);
        return ROCKET_E_SHAPE;
    }
    Req r;
    r.who = who; r.fa = fa; r.fb = fb; r.epi = epi; r.K = K; r.N = N;
    r.M = &M; r.A = &A; r.B = &B; r.C = &C;
    return run(fd, r);
}

}  // namespace

extern "C" {

// ---- planners ----------------------------------------------------------------------
int rocket_matmul_plan(int M, int K, int N, int *Mt, int *Kt, int *Nt)
{   // reference rocket_matmul.c:498-568: K%32, N%16, M%4, 0 < dims <= 2^24
    return plan(M, K, N, 32, 16, Fmt::F16, Epi::F16, 0, Mt, Kt, Nt);
}

int rocket_matmul_plan_int8(int M, int K, int N, int *Mt, int *Kt, int *Nt)
{   // reference rocket_matmul.c:2383-2437: K%32, N%32, M%4
    return plan(M, K, N, 32, 32, Fmt::I8, Epi::I32, 0, Mt, Kt, Nt);
}

int rocket_matmul_plan_int8_gw(int M, int K, int N, int group, int *Mt, int *Kt, int *Nt)
{   // reference rocket_matmul.c:2671-2714: + group >= 32, group%32, K%group; Kt | group
    if (!dims_ok(M, K, N) || K % 32 || N % 32 || M % 4) return ROCKET_E_SHAPE;
    if (group < 32 || group % 32 || K % group) return ROCKET_E_SHAPE;
    return plan(M, K, N, 32, 32, Fmt::I8, Epi::GW, gw_period(group), Mt, Kt, Nt);
}

int rocket_matmul_plan_int4(int M, int K, int N, int *Mt, int *Kt, int *Nt)
{   // reference rocket_matmul.c:2917-2956: K%32, N%64, M%4
    return plan(M, K, N, 32, 64, Fmt::I8, Epi::I32, 0, Mt, Kt, Nt);
}

int rocket_matmul_plan_int16(int M, int K, int N, int *Mt, int *Kt, int *Nt)
{   // reference rocket_matmul.c:3320-3359: K%32, N%16, M%4
    return plan(M, K, N, 32, 16, Fmt::I16, Epi::I64, 0, Mt, Kt, Nt);
}

int rocket_matmul_plan_bf16(int M, int K, int N, int *Mt, int *Kt, int *Nt)
{   // reference rocket_matmul.c:3448-3452: the int16 geometry and alignment
    return plan(M, K, N, 32, 16, Fmt::F32BF16, Epi::F32, 0, Mt, Kt, Nt);
}

int rocket_matmul_plan_tf32(int M, int K, int N, int *Mt, int *Kt, int *Nt)
{   // reference rocket_matmul.c:3797-3838: K%16, N%16, M%4
    return plan(M, K, N, 16, 16, Fmt::F32TF32, Epi::F32, 0, Mt, Kt, Nt);
}

// ---- fp16 ----------------------------------------------------------------------------
int rocket_matmul_fp16(int fd, int M, int K, int N, const _Float16 *A, const _Float16 *B, _Float16 *C)
{   // reference rocket_matmul.c:1945-1998
    if (!dtype_ok(precision_float16)) return ROCKET_E_UNSUPPORTED;
    if (oneshot_shape(M, K, N, 32, 16)) {
        ROCKET_LOGE("rocket_matmul_fp16: unsupported shape M=%d K=%d N=%d (need K%%32, N%%16, M%%4||1)\n", M, K, N);
        return ROCKET_E_SHAPE;
    }
    return single(fd, "rocket_matmul_fp16", Fmt::F16, Fmt::F16, Epi::F16, M, K, N, A, B, C);
}

int rocket_matmul_fp16_f32out(int fd, int M, int K, int N, const _Float16 *A, const _Float16 *B, float *C)
{   // reference rocket_matmul.c:3620-3758
    if (!dtype_ok(precision_float16)) return ROCKET_E_UNSUPPORTED;
    if (oneshot_shape(M, K, N, 32, 16)) {
        ROCKET_LOGE("rocket_matmul_fp16_f32out: unsupported shape M=%d K=%d N=%d (need K%%32, N%%16, M%%4||1)\n", M, K, N);
        return ROCKET_E_SHAPE;
    }
    return single(fd, "rocket_matmul_fp16_f32out", Fmt::F16, Fmt::F16, Epi::F32, M, K, N, A, B, C);
}

int rocket_matmul_fp16_batch(int fd, int M, int K, int N, int nbatch,
                             const _Float16 *const *A, const _Float16 *const *B, _Float16 *const *C)
{   // reference rocket_matmul.c:2042-2310: M%4, K%32, N%16; nbatch==1 -> rocket_matmul_fp16
    if (nbatch < 1 || !A || !B || !C) return ROCKET_E_SHAPE;
    if (nbatch == 1) return rocket_matmul_fp16(fd, M, K, N, A[0], B[0], C[0]);
    if (plan(M, K, N, 32, 16, Fmt::F16, Epi::F16, 0, nullptr, nullptr, nullptr) < 0) {
        ROCKET_LOGE("rocket_matmul_fp16_batch: unsupported shape M=%d K=%d N=%d (need M%%4, K%%32, N%%16)\n", M, K, N);
        return ROCKET_E_SHAPE;
    }
    for (int i = 0; i < nbatch; i++)
        if (!A[i] || !B[i] || !C[i]) return ROCKET_E_SHAPE;
    std::vector<int> Ms(nbatch, M);
    Req r;
    r.who = "rocket_matmul_fp16_batch"; r.fa = r.fb = Fmt::F16; r.epi = Epi::F16;
    r.K = K; r.N = N; r.nprob = nbatch; r.M = Ms.data();
    r.A = reinterpret_cast<const void *const *>(A);
    r.B = reinterpret_cast<const void *const *>(B);
    r.C = reinterpret_cast<void *const *>(C);
    return run(fd, r);
}

// ---- int8 ----------------------------------------------------------------------------
int rocket_matmul_int8(int fd, int M, int K, int N, const int8_t *A, const int8_t *B, int32_t *C)
{   // reference rocket_matmul.c:2439-2627
    if (!dtype_ok(precision_int8)) return ROCKET_E_UNSUPPORTED;
    if (oneshot_shape(M, K, N, 32, 32)) {
        ROCKET_LOGE("rocket_matmul_int8: unsupported shape M=%d K=%d N=%d (need K%%32, N%%32, M%%4||1)\n", M, K, N);
        return ROCKET_E_SHAPE;
    }
    return single(fd, "rocket_matmul_int8", Fmt::I8, Fmt::I8, Epi::I32, M, K, N, A, B, C);
}

static int gw_common(int fd, const char *who, bool b_int4, int M, int K, int N,
                     const int8_t *A, const int8_t *B, const float *as, const float *bs,
                     float *Cf, int group, int32_t *dump, int row0, int nrows, bool rowscale = false)
{
    if (!A || !B || !as || !bs || !Cf) { ROCKET_LOGE("%s: NULL operand\n", who); return ROCKET_E_SHAPE; }
    Req r;
    const void *a = A, *b = B;
    void *c = Cf;
    r.who = who; r.fa = Fmt::I8; r.fb = b_int4 ? Fmt::I4P : Fmt::I8; r.pack_b_int4 = b_int4;
    r.epi = Epi::GW; r.K = K; r.N = N; r.M = &M; r.A = &a; r.B = &b; r.C = &c;
    r.a_scale = &as; r.b_scale = &bs; r.group = group;
    r.dump = &dump; r.dump_row0 = &row0; r.dump_rows = &nrows;
    r.rowscale = rowscale;
    return run(fd, r);
}

int rocket_matmul_int8_groupwise(int fd, int M, int K, int N, const int8_t *A, const int8_t *B,
                                 const float *a_scale, const float *b_scale, float *Cf, int group)
{   // reference rocket_matmul.c:2716-2871 (no M==1 pad: M%4)
    if (!dtype_ok(precision_int8)) return ROCKET_E_UNSUPPORTED;
    if (rocket_matmul_plan_int8_gw(M, K, N, group, nullptr, nullptr, nullptr) < 0) {
        ROCKET_LOGE("rocket_matmul_int8_groupwise: unsupported shape M=%d K=%d N=%d group=%d "
                    "(need K%%32, N%%32, M%%4, group%%32, group|K)\n", M, K, N, group);
        return ROCKET_E_SHAPE;
    }
    return gw_common(fd, "rocket_matmul_int8_groupwise", false, M, K, N, A, B, a_scale, b_scale, Cf,
                     group, nullptr, 0, 0);
}

// ---- int4 ----------------------------------------------------------------------------
int rocket_matmul_int4_ex(int fd, int M, int K, int N, const int8_t *A, const int8_t *B, int32_t *C, int kt_cap)
{   // reference rocket_matmul.c:2958-3114. kt_cap bounded the NPU's int16 K-tile readback;
    // the int32 accumulation here is exact for every kt_cap, so it does not change C.
    (void)kt_cap;
    if (!dtype_ok(precision_int4)) return ROCKET_E_UNSUPPORTED;
    if (oneshot_shape(M, K, N, 32, 64)) {
        ROCKET_LOGE("rocket_matmul_int4: unsupported shape M=%d K=%d N=%d (need K%%32, N%%64, M%%4||1)\n", M, K, N);
        return ROCKET_E_SHAPE;
    }
    if (!A || !B || !C) return ROCKET_E_SHAPE;
    Req r;
    const void *a = A, *b = B;
    void *c = C;
    r.who = "rocket_matmul_int4"; r.fa = Fmt::I8; r.fb = Fmt::I4P; r.pack_b_int4 = true;
    r.epi = Epi::I32; r.K = K; r.N = N; r.M = &M; r.A = &a; r.B = &b; r.C = &c;
    r.kchunk = 65536;   // the x16 int4 accumulators stay exact below 2^17 products of int8 x int4
    return run(fd, r);
}

int rocket_matmul_int4(int fd, int M, int K, int N, const int8_t *A, const int8_t *B, int32_t *C)
{
    return rocket_matmul_int4_ex(fd, M, K, N, A, B, C, 0);
}

int rocket_matmul_int4_groupwise(int fd, int M, int K, int N, const int8_t *A, const int8_t *B,
                                 const float *a_scale, const float *b_scale, float *Cf, int group)
{   // reference rocket_matmul.c:3132-3282
    if (!dtype_ok(precision_int4)) return ROCKET_E_UNSUPPORTED;
    if (group < 32 || group % 32 || K % group || M % 4 || 49 * group >= 32767) {
        ROCKET_LOGE("rocket_matmul_int4_groupwise: bad group=%d (need %%32, |K, 49*group<32767, M%%4) K=%d M=%d\n",
                    group, K, M);
        return ROCKET_E_SHAPE;
    }
    if (rocket_matmul_plan_int4(M, K, N, nullptr, nullptr, nullptr) < 0) {
        ROCKET_LOGE("rocket_matmul_int4_groupwise: unsupported shape M=%d K=%d N=%d\n", M, K, N);
        return ROCKET_E_SHAPE;
    }
    return gw_common(fd, "rocket_matmul_int4_groupwise", true, M, K, N, A, B, a_scale, b_scale, Cf,
                     group, nullptr, 0, 0);
}

// ---- per-row activation scales (rocket_hip.h) ------------------------------------------
int rocket_matmul_int8_groupwise_rowscale(int fd, int M, int K, int N, const int8_t *A, const int8_t *B,
                                          const float *a_row_scale, const float *b_scale, float *Cf, int group)
{   // validation of rocket_matmul_int8_groupwise
    if (!dtype_ok(precision_int8)) return ROCKET_E_UNSUPPORTED;
    if (rocket_matmul_plan_int8_gw(M, K, N, group, nullptr, nullptr, nullptr) < 0) {
        ROCKET_LOGE("rocket_matmul_int8_groupwise_rowscale: unsupported shape M=%d K=%d N=%d group=%d\n", M, K, N,
                    group);
        return ROCKET_E_SHAPE;
    }
    return gw_common(fd, "rocket_matmul_int8_groupwise_rowscale", false, M, K, N, A, B, a_row_scale, b_scale, Cf,
                     group, nullptr, 0, 0, true);
}

int rocket_matmul_int4_groupwise_rowscale(int fd, int M, int K, int N, const int8_t *A, const int8_t *B,
                                          const float *a_row_scale, const float *b_scale, float *Cf, int group)
{   // validation of rocket_matmul_int4_groupwise
    if (!dtype_ok(precision_int4)) return ROCKET_E_UNSUPPORTED;
    if (group < 32 || group % 32 || K % group || M % 4 || 49 * group >= 32767 ||
        rocket_matmul_plan_int4(M, K, N, nullptr, nullptr, nullptr) < 0) {
        ROCKET_LOGE("rocket_matmul_int4_groupwise_rowscale: unsupported shape M=%d K=%d N=%d group=%d\n", M, K, N,
                    group);
        return ROCKET_E_SHAPE;
    }
    return gw_common(fd, "rocket_matmul_int4_groupwise_rowscale", true, M, K, N, A, B, a_row_scale, b_scale, Cf,
                     group, nullptr, 0, 0, true);
}

// ---- int16 exact ---------------------------------------------------------------------
int rocket_matmul_int16_exact(int fd, int M, int K, int N, const int16_t *A, const int16_t *B, int64_t *C)
{   // reference rocket_matmul.c:3377-3421 (int8 alignment: K%32, N%32, M%4||1)
    if (!dtype_ok(precision_int8)) return ROCKET_E_UNSUPPORTED;
    if (oneshot_shape(M, K, N, 32, 32)) {
        ROCKET_LOGE("rocket_matmul_int16_exact: unsupported shape M=%d K=%d N=%d (need K%%32, N%%32, M%%4||1)\n", M, K, N);
        return ROCKET_E_SHAPE;
    }
    if (!A || !B || !C) return ROCKET_E_SHAPE;
    Req r;
    const void *a = A, *b = B;
    void *c = C;
    r.who = "rocket_matmul_int16_exact"; r.fa = r.fb = Fmt::I16; r.epi = Epi::I64;
    r.K = K; r.N = N; r.M = &M; r.A = &a; r.B = &b; r.C = &c;
    r.kchunk = 32768;   // every int32 byte-plane accumulator stays below 2^31
    return run(fd, r);
}

// ---- bf16 / tf32 ---------------------------------------------------------------------
int rocket_matmul_bf16(int fd, int M, int K, int N, const float *A, const float *B, float *C)
{   // reference rocket_matmul.c:3454-3596
    if (!dtype_ok(precision_bfloat16)) return ROCKET_E_UNSUPPORTED;
    if (oneshot_shape(M, K, N, 32, 16)) {
        ROCKET_LOGE("rocket_matmul_bf16: unsupported shape M=%d K=%d N=%d (need K%%32, N%%16, M%%4||1)\n", M, K, N);
        return ROCKET_E_SHAPE;
    }
    return single(fd, "rocket_matmul_bf16", Fmt::F32BF16, Fmt::F32BF16, Epi::F32, M, K, N, A, B, C);
}

int rocket_matmul_tf32(int fd, int M, int K, int N, const float *A, const float *B, float *C)
{   // reference rocket_matmul.c:3840-3982
    if (!dtype_ok(precision_tf32)) return ROCKET_E_UNSUPPORTED;
    if (oneshot_shape(M, K, N, 16, 16)) {
        ROCKET_LOGE("rocket_matmul_tf32: unsupported shape M=%d K=%d N=%d (need K%%16, N%%16, M%%4||1)\n", M, K, N);
        return ROCKET_E_SHAPE;
    }
    return single(fd, "rocket_matmul_tf32", Fmt::F32TF32, Fmt::F32TF32, Epi::F32, M, K, N, A, B, C);
}

// ---- RK3576 entries: a different chip's requantising contract -------------------------
int rocket_matmul_plan_int8_rk3576(int M, int K, int N, int *Mt, int *Kt, int *Nt)
{
    (void)M; (void)K; (void)N; (void)Mt; (void)Kt; (void)Nt;
    return ROCKET_E_UNSUPPORTED;
}
int rocket_matmul_int8_rk3576(int fd, int M, int K, int N, const int8_t *A, const int8_t *B,
                              const int32_t *bias, float scale, int8_t *C)
{
    (void)fd; (void)M; (void)K; (void)N; (void)A; (void)B; (void)bias; (void)scale; (void)C;
    return ROCKET_E_UNSUPPORTED;
}
int rocket_matmul_int8_rk3576_perc(int fd, int M, int K, int N, const int8_t *A, const int8_t *B,
                                   const int32_t *bias, const float *scale_n, int8_t *C, double *worst_rel_err)
{
    (void)fd; (void)M; (void)K; (void)N; (void)A; (void)B; (void)bias; (void)scale_n; (void)C; (void)worst_rel_err;
    return ROCKET_E_UNSUPPORTED;
}
int rocket_matmul_int8_rk3576_perc_sa(int fd, int M, int K, int N, const int8_t *A, const int8_t *B,
                                      const int32_t *bias, const float *scale_n, const int64_t *sum_abs_w,
                                      int8_t *C, double *worst_rel_err)
{
    (void)fd; (void)M; (void)K; (void)N; (void)A; (void)B; (void)bias; (void)scale_n; (void)sum_abs_w;
    (void)C; (void)worst_rel_err;
    return ROCKET_E_UNSUPPORTED;
}
int rocket_rk3576_wbo_create(int fd, int K, int N, const int8_t *B, struct rocket_rk3576_wbo **out)
{
    (void)fd; (void)K; (void)N; (void)B;
    if (out) *out = nullptr;
    return ROCKET_E_UNSUPPORTED;
}
void rocket_rk3576_wbo_free(int fd, struct rocket_rk3576_wbo *w) { (void)fd; (void)w; }
int rocket_matmul_int8_rk3576_perc_wbo(int fd, int M, int K, int N, const int8_t *A,
                                       const struct rocket_rk3576_wbo *wbo, const int32_t *bias,
                                       const float *scale_n, const int64_t *sum_abs_w, int8_t *C,
                                       double *worst_rel_err)
{
    (void)fd; (void)M; (void)K; (void)N; (void)A; (void)wbo; (void)bias; (void)scale_n; (void)sum_abs_w;
    (void)C; (void)worst_rel_err;
    return ROCKET_E_UNSUPPORTED;
}
void rocket_rk3576_bo_pool_drain(int fd) { (void)fd; }
int rocket_matmul_int8_rk3576_i32(int fd, int M, int K, int N, const int8_t *A, const int8_t *B,
                                  const int32_t *bias, int32_t *C)
{
    (void)fd; (void)M; (void)K; (void)N; (void)A; (void)B; (void)bias; (void)C;
    return ROCKET_E_UNSUPPORTED;
}
void rocket_rk3576_i32_last_stats(rocket_rk3576_i32_stats *out)
{
    if (out) memset(out, 0, sizeof(*out));
}

}  // extern "C"
