// arena_check.cpp — what the library's calls launch and do with a handle's scratch, on the fake runtime
// of fake_hip.h: which kernels a call launches where the arena may not grow (a captured stream), what a
// captured call's graph may still replay on after the arena has grown, and what is freed when the
// handle closes. Built and run by tests/test_arena.py. Exit status 0 when every check passes.
#include "fake_hip.h"

#include <stdio.h>

#include <stdlib.h>

#include <algorithm>
#include <chrono>
#include <new>
#include <random>

#include "ops.h"
#include "rocket_attn.h"
#include "rocket_ffn.h"
#include "rocket_hip.h"
#include "rocket_matmul.h"
#include "rocket_npu.h"

// Host allocations of at least g_refuse bytes fail (0: none does).
static size_t g_refuse = 0;
void *operator new(size_t n)
{
    void *const p = g_refuse && n >= g_refuse ? nullptr : malloc(n ? n : 1);
    if (!p) throw std::bad_alloc();
    return p;
}
void *operator new(size_t n, const std::nothrow_t &) noexcept { return g_refuse && n >= g_refuse ? nullptr : malloc(n ? n : 1); }
void *operator new[](size_t n) { return operator new(n); }
void *operator new[](size_t n, const std::nothrow_t &t) noexcept { return operator new(n, t); }
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }
void operator delete[](void *p) noexcept { free(p); }
void operator delete[](void *p, size_t) noexcept { free(p); }

static int g_fail = 0;
#define CHECK(c)                                                                                       \
    do {                                                                                               \
        if (!(c)) {                                                                                    \
            fprintf(stderr, "arena_check: %s:%d: CHECK(%s) failed\n", __FILE__, __LINE__, #c);         \
            g_fail++;                                                                                  \
        }                                                                                              \
    } while (0)

static int open_async()
{
    const int fd = rocket_open();
    CHECK(fd >= 0);
    CHECK(rocket_hip_set_mode(fd, ROCKET_HIP_ASYNC | ROCKET_HIP_DEVICE_OPERANDS) == 0);
    fake::st().launches.clear();
    return fd;
}

// Operands: addresses that no kernel reads here.
static float *const X = reinterpret_cast<float *>(0x100000);
static float *const W = reinterpret_cast<float *>(0x10000000);
static float *const Y = reinterpret_cast<float *>(0x20000000);
static _Float16 *h(float *p) { return reinterpret_cast<_Float16 *>(p); }

static int bf16(int fd, int M, int K, int N) { return rocket_matmul_bf16(fd, M, K, N, X, W, Y); }
static int fp16(int fd, int M, int K, int N) { return rocket_matmul_fp16(fd, M, K, N, h(X), h(W), h(Y)); }
static int attn(int fd, int T, int n)
{
    return rocket_flash_attn_fp16(fd, T, n, 128, 128, 8, 8, 0.1f, 0.f, h(X), h(W), h(W), nullptr, h(Y));
}

// Recorded while the stream is captured: the names of its launches.
template <class F> static std::vector<std::string> captured(F call, int want_rc = 0)
{
    auto &f = fake::st();
    f.launches.clear();
    f.capturing = true;
    const int syncs = f.syncs;
    const int rc = call();
    f.capturing = false;
    CHECK(rc == want_rc);
    if (rc == 0) CHECK(f.syncs == syncs);
    return f.launches;
}

// A captured call's arena outlives its growth, and goes with the handle.
static void arena_kept_for_graphs()
{
    auto &f = fake::st();
    const int live0 = (int)f.live.size();
    const int fd = open_async();
    CHECK(attn(fd, 1, 4096) == 0);                       // eager: the arena
    CHECK((int)f.live.size() == live0 + 1);
    CHECK(captured([&] { return attn(fd, 1, 4096); }).size() == 2);   // keys split, and the merge
    const int frees = f.frees;
    CHECK(rocket_ffn_fp16(fd, 512, 1024, 8192, h(X), h(W), h(W), h(W), ROCKET_ACTIVATION_SILU, h(Y)) == 0);   // a larger arena
    CHECK(f.frees == frees && (int)f.live.size() == live0 + 2);
    // one that no graph holds is freed when it grows
    CHECK(rocket_ffn_fp16(fd, 512, 1024, 16384, h(X), h(W), h(W), h(W), ROCKET_ACTIVATION_SILU, h(Y)) == 0);
    CHECK(f.frees == frees + 1 && (int)f.live.size() == live0 + 2);
    rocket_close(fd);
    CHECK((int)f.live.size() == live0);
}

// Calls that can do without scratch hold none in a graph, on a handle that has some.
static void small_calls_hold_no_scratch()
{
    const int fd = open_async();
    CHECK(rocket_ffn_fp16(fd, 512, 1024, 8192, h(X), h(W), h(W), h(W), ROCKET_ACTIVATION_SILU, h(Y)) == 0);
    fake::st().launches.clear();
    CHECK(bf16(fd, 300, 15360, 96) == 0);
    CHECK(fake::count("k_sum_slices") == 1);             // eager: K slices
    CHECK(captured([&] { return bf16(fd, 300, 15360, 96); }).size() == 1);
    CHECK(captured([&] { return attn(fd, 1, 448); }).size() == 1);
    CHECK(captured([&] { return attn(fd, 1, 1000); }).size() == 2);
    CHECK(captured([&] { return fp16(fd, 64, 4096, 4096); }).size() == 1);
    CHECK(captured([&] { return fp16(fd, 4, 4096, 4096); }).size() == 1);
    // a call that converts its rows ahead holds scratch anyway
    captured([&] { return bf16(fd, 128, 8192, 512); });
    CHECK(fake::count("k_cvt") == 1 && fake::count("k_sum_slices") == 1);
    rocket_close(fd);
}

// fp32 rows that are converted ahead are converted in the product where a captured call has no arena for them.
static void rows_converted_without_an_arena()
{
    const int fd = open_async();
    auto tf32 = [&] { return rocket_matmul_tf32(fd, 20, 3840, 14336, X, W, Y); };
    auto bf = [&] { return bf16(fd, 16, 3840, 12288); };
    CHECK(captured(tf32).size() == 1);
    CHECK(captured(bf).size() == 1);
    CHECK(captured([&] { return bf16(fd, 20, 3072, 10240); }).size() == 1);
    fake::st().launches.clear();
    CHECK(tf32() == 0 && fake::count("k_cvt") == 1);
    CHECK(captured(tf32).size() == 2);
    rocket_close(fd);
}

// Rows that are quantised ahead are quantised in the product where a captured call has no arena for the codes.
static void rows_quantised_without_an_arena()
{
    const int fd = open_async();
    const std::vector<int> M(8, 12);
    const std::vector<const void *> A(8, X), A2(8, X + 500000), B(8, W);
    const std::vector<const float *> S(8, W + 10000000);
    std::vector<void *> C;
    for (int i = 0; i < 8; i++) C.push_back(Y + 100000 * i);
    rk::Req r;
    r.epi = rk::Epi::GW;
    r.K = 1344;
    r.N = 2560;
    r.nprob = 8;
    r.M = M.data();
    r.A = A.data();
    r.A2 = A2.data();
    r.B = B.data();
    r.C = C.data();
    r.b_scale = S.data();
    r.group = 32;
    r.rowscale = true;
    r.quant_a = 1;
    r.act = rk::kActSilu;
    for (int n = 1024; n <= 6144; n += 512) {   // (fused by the estimate, or not)
        r.N = n;
        CHECK(captured([&] { return rk::run(fd, r); }).size() == 1);
    }
    rocket_close(fd);
}

// A block's second product runs without its K slices where the arena holds the hidden rows alone.
static void blocks_on_a_small_arena()
{
    const int M = 64, H = 3840, I = 15360;
    auto ffn = [&](int fd) { return rocket_ffn_fp16(fd, M, H, I, h(X), h(W), h(W), h(W), ROCKET_ACTIVATION_SILU, h(Y)); };
    auto mlp = [&](int fd) { return rocket_mlp_fp16_fused(fd, M, H, I, H, h(X), h(W), nullptr, h(W), ROCKET_ACTIVATION_GELU, h(Y)); };
    for (int which = 0; which < 2; which++) {
        auto call = [&](int fd) { return which ? mlp(fd) : ffn(fd); };
        const int fd = open_async();
        setenv("ROCKET_HIP_SPLITK", "1", 1);
        CHECK(call(fd) == 0);
        unsetenv("ROCKET_HIP_SPLITK");
        CHECK(captured([&] { return call(fd); }).size() == 2);
        fake::st().launches.clear();
        CHECK(call(fd) == 0);
        CHECK(fake::count("k_sum_slices") == 1);                  // eager: the arena grows
        CHECK(captured([&] { return call(fd); }).size() == 3);    // and then holds the slices too
        rocket_close(fd);
    }
}

// Memory for what a call can do without may be short: the call then runs without it.
static void short_of_memory()
{
    auto &f = fake::st();
    const int fd = open_async();
    f.limit = 100000;
    CHECK(bf16(fd, 300, 15360, 96) == 0);                // no K slices' planes
    CHECK(f.launches.size() == 1);
    CHECK(attn(fd, 1, 4096) == 0);                       // no key splits
    CHECK(f.launches.size() == 2);
    CHECK(bf16(fd, 128, 8192, 512) == ROCKET_E_NOMEM);   // converted rows it needs
    // V's rows padded, the mask read as it is
    const int T = 512, n = 3001, np = 3008, d = 64, kvh = 2;
    auto masked = [&] { return rocket_flash_attn_fp16(fd, T, n, d, d, 2, kvh, 0.125f, 0.f, h(X), h(W), h(W), h(X), h(Y)); };
    f.limit = (size_t)kvh * d * np * 2 * 5 / 4 + 4096;
    f.launches.clear();
    CHECK(masked() == 0);
    CHECK(fake::count("k_pad_cols") == 1 && fake::count("k_flash_attn") == 1);
    f.limit = (size_t)-1;
    rocket_close(fd);
}

// A dump's partials come from the kernel that the call without it runs.
static void dumps_run_the_same_kernel()
{
    auto &f = fake::st();
    const int fd = open_async();
    int8_t *const A = reinterpret_cast<int8_t *>(X), *const B = reinterpret_cast<int8_t *>(W);
    for (int M : {4, 16, 20, 64, 512})
        for (int N : {64, 4096}) {
            auto base = [&] {
                // the name up to its template arguments (the last of which is the dump)
                CHECK(f.launches.size() == 1);
                std::string n = f.launches.empty() ? "" : f.launches[0];
                const size_t at = n.find("k_");
                return at == std::string::npos ? n : n.substr(at, n.find('I', at) - at);
            };
            f.launches.clear();
            CHECK(rocket_matmul_int8_groupwise(fd, M, 1024, N, A, B, X, W, Y, 128) == 0);
            const std::string plain = base();
            f.launches.clear();
            CHECK(rocket_matmul_int8_groupwise_dump(fd, M, 1024, N, A, B, X, W, Y, 128, 0, 4, reinterpret_cast<int32_t *>(Y)) == 0);
            CHECK(base() == plain && !plain.empty());
        }
    rocket_close(fd);
}

// Results over rows, against every pair; and in a time that grows with the products, not their square.
static void overlaps()
{
    std::mt19937 rng(7);
    std::vector<int> M;
    std::vector<const void *> A, A2;
    std::vector<void *> C;
    rk::Req r;
    auto make = [&](int n, int spread) {
        M.resize(n), A.resize(n), A2.resize(n), C.resize(n);
        for (int i = 0; i < n; i++) {
            M[i] = (int)(rng() % 4) * 4;
            A[i] = (const void *)(uintptr_t)(4096 + rng() % spread * 16);
            A2[i] = (const void *)(uintptr_t)(4096 + rng() % spread * 16);
            C[i] = (void *)(uintptr_t)(4096 + rng() % spread * 16);
        }
        r.nprob = n;
        r.N = 32;
        r.M = M.data(), r.A = A.data(), r.C = C.data();
        r.A2 = rng() % 2 ? A2.data() : nullptr;
    };
    int hits = 0;
    for (int t = 0; t < 4000; t++) {
        make(1 + (int)(rng() % 20), 40 << (rng() % 10));
        bool any = false;
        const size_t row = 64, el = 4;
        for (int p = 0; p < r.nprob; p++)
            for (int q = 0; q < r.nprob; q++)
                for (const void *a : {A[p], r.A2 ? A2[p] : A[p]}) {
                    const uintptr_t x = (uintptr_t)a, y = (uintptr_t)C[q];
                    if (M[p] && M[q] && x < y + (size_t)M[q] * r.N * el && y < x + M[p] * row) any = true;
                }
        CHECK(rk::results_overlap_rows(r, row, el) == any);
        hits += any;
    }
    CHECK(hits > 400 && hits < 3600);
    auto time = [&](int n) {   // rows and results in turn in memory, none over another
        make(n, 1);
        for (int i = 0; i < n; i++) {
            M[i] = 4;
            A[i] = A2[i] = (const void *)(uintptr_t)(4096 + 4096 * (size_t)(2 * i));
            C[i] = (void *)(uintptr_t)(4096 + 4096 * (size_t)(2 * i + 1));
        }
        double best = 1e9;
        for (int k = 0; k < 9; k++) {
            const auto t0 = std::chrono::steady_clock::now();
            CHECK(!rk::results_overlap_rows(r, 64, 4));
            best = std::min(best, std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count());
        }
        return best;
    };
    CHECK(time(4096) < 100 * time(128));   // 32 times the products: their square takes 1024 times as long
}

// The kernels that sizes on both sides of a dispatch rule's line run.
static void routes()
{
    const int fd = open_async();
    int8_t *const A = reinterpret_cast<int8_t *>(X), *const B = reinterpret_cast<int8_t *>(W);
    auto ran = [&](const char *kernel) {
        const bool r = fake::count(kernel) == 1;
        if (!r)
            for (const auto &l : fake::st().launches) fprintf(stderr, "  launched %s\n", l.c_str());
        fake::st().launches.clear();
        return r;
    };
    auto gw8 = [&](int M, int K, int N, int g) { return rocket_matmul_int8_groupwise(fd, M, K, N, A, B, X, W, Y, g) == 0; };
    auto gw4 = [&](int M, int K, int N, int g) { return rocket_matmul_int4_groupwise(fd, M, K, N, A, B, X, W, Y, g) == 0; };
    auto int8 = [&](int M, int K, int N) { return rocket_matmul_int8(fd, M, K, N, A, B, reinterpret_cast<int32_t *>(Y)) == 0; };
    auto tf32 = [&](int M, int K, int N) { return rocket_matmul_tf32(fd, M, K, N, X, W, Y) == 0; };
    auto fa = [&](int T, int n, int d, int heads, int kv) {
        return rocket_flash_attn_fp16(fd, T, n, d, d, heads, kv, 0.1f, 0.f, h(X), h(W), h(W), nullptr, h(Y)) == 0;
    };
    (void)gw8, (void)gw4, (void)int8, (void)tf32, (void)fa;
    // rows so long that LDS holds a wave or two a CU
    CHECK(gw4(16, 8192, 4096, 128) && ran("k_stream_gw"));
    CHECK(gw4(16, 8192, 16384, 128) && ran("k_gemm"));
    CHECK(gw8(16, 4096, 16384, 32) && ran("k_stream_gw"));
    CHECK(gw8(16, 8192, 16384, 32) && ran("k_gemm"));
    CHECK(gw8(16, 8192, 8192, 64) && ran("k_gemm"));
    // int8 weights, 17 rows and more, long rows
    CHECK(gw8(64, 1024, 16384, 64) && ran("k_mid_gw"));
    CHECK(gw8(64, 2048, 16384, 64) && ran("k_gemm"));
    CHECK(gw8(64, 2048, 8192, 32) && ran("k_gemm"));
    CHECK(gw8(64, 8192, 16384, 64) && ran("k_gemm"));
    CHECK(gw8(48, 8192, 6144, 32) && ran("k_mid_gw"));
    CHECK(gw8(48, 8192, 8192, 32) && ran("k_gemm"));
    // int8 to int32, few rows
    CHECK(int8(16, 8192, 4096) && ran("k_stream"));
    CHECK(int8(16, 8192, 8192) && ran("k_gemm"));
    CHECK(int8(4, 8192, 8192) && ran("k_stream"));
    CHECK(int8(4, 4096, 16384) && ran("k_gemm"));
    CHECK(int8(4, 4096, 24576) && ran("k_stream"));
    CHECK(int8(4, 512, 16384) && ran("k_stream"));
    CHECK(int8(4, 512, 32768) && ran("k_gemm"));
    // fp32 rows converted ahead
    CHECK(tf32(128, 2048, 2048) && !ran("k_cvt"));
    CHECK(tf32(128, 4096, 4096) && ran("k_cvt"));
    CHECK(tf32(256, 1024, 8192) && ran("k_cvt"));
    CHECK(tf32(2044, 128, 8192) && ran("k_cvt"));
    CHECK(tf32(20, 2048, 16384) && ran("k_cvt"));
    CHECK(tf32(64, 2048, 8192) && !ran("k_cvt"));
    // attention of few query rows: short caches, and long ones of one query head a KV head
    CHECK(fa(1, 192, 128, 8, 8) && fake::st().launches.size() == 1 && ran("k_fa_rows"));
    CHECK(fa(1, 512, 64, 8, 8) && fake::st().launches.size() == 1 && ran("k_fa_rows"));
    CHECK(fa(1, 512, 128, 8, 8) && fake::st().launches.size() == 2 && ran("k_fa_rows"));
    CHECK(fa(1, 256, 256, 8, 8) && fake::st().launches.size() == 1 && ran("k_fa_rows"));
    CHECK(fa(1, 255, 256, 8, 8) && fake::st().launches.size() == 2 && ran("k_fa_rows"));
    CHECK(fa(1, 159, 256, 8, 8) && fake::st().launches.size() == 1 && ran("k_fa_rows"));
    CHECK(fa(1, 319, 128, 8, 8) && fake::st().launches.size() == 2 && ran("k_fa_rows"));
    CHECK(fa(1, 511, 64, 8, 8) && fake::st().launches.size() == 2 && ran("k_fa_rows"));
    CHECK(fa(1, 8192, 256, 32, 32) && ran("k_flash_attn"));
    CHECK(fa(1, 8191, 256, 32, 32) && ran("k_fa_rows"));
    CHECK(fa(1, 8192, 256, 64, 32) && ran("k_fa_rows"));
    CHECK(fa(1, 8192, 256, 24, 24) && ran("k_fa_rows"));
    CHECK(fa(1, 8192, 64, 32, 32) && ran("k_fa_rows"));
    // results over their own operands: one workgroup, which has read all of them first
    CHECK(int8(4, 512, 64) && ran("k_stream"));
    CHECK(rocket_matmul_int8(fd, 4, 512, 64, A, B, reinterpret_cast<int32_t *>(A)) == 0 && ran("k_gemm"));
    CHECK(rocket_matmul_int8_groupwise(fd, 4, 512, 64, A, B, Y, W, reinterpret_cast<float *>(A), 64) == 0 && ran("k_gemm"));
    CHECK(rocket_matmul_int8_groupwise(fd, 20, 512, 64, A, B, Y, W, reinterpret_cast<float *>(B), 64) == 0 && ran("k_gemm"));
    CHECK(rocket_matmul_fp16(fd, 4, 1024, 64, h(X), h(W), h(X)) == 0 && ran("k_gemm"));
    // attention's results over V: V is copied first where its rows are no multiple of a tile
    CHECK(fa(1, 100, 64, 8, 8) && !ran("k_pad_cols"));
    CHECK(rocket_flash_attn_fp16(fd, 1, 100, 64, 64, 8, 8, 0.1f, 0.f, h(X), h(W), h(Y), nullptr, h(Y)) == 0 && ran("k_pad_cols"));
    // plain fp16 over many columns, and 17 to 32 rows over more than a wave a CU
    CHECK(fp16(fd, 16, 5120, 28672) == 0 && ran("k_gemm"));
    CHECK(fp16(fd, 12, 2560, 28672) == 0 && ran("k_gemm"));
    CHECK(fp16(fd, 8, 2560, 28672) == 0 && ran("k_chain"));
    CHECK(fp16(fd, 16, 2560, 24576) == 0 && ran("k_chain"));
    CHECK(fp16(fd, 16, 4096, 14336) == 0 && ran("k_gemm"));
    CHECK(fp16(fd, 16, 4096, 16384) == 0 && ran("k_chain"));
    CHECK(fp16(fd, 32, 4096, 4096) == 0 && ran("k_chain"));
    CHECK(fp16(fd, 32, 8704, 7808) == 0 && ran("k_gemm"));
    CHECK(fp16(fd, 20, 8704, 7808) == 0 && ran("k_chain"));
    CHECK(fp16(fd, 20, 12288, 5120) == 0 && ran("k_gemm"));
    CHECK(fp16(fd, 32, 1536, 5120) == 0 && ran("k_chain"));
    // int8 to int32 over a little more than whole rounds of tiles, and of many long rows
    CHECK(int8(12, 4224, 25536) && ran("k_gemm"));
    CHECK(int8(4, 4224, 22528) && ran("k_stream"));
    CHECK(int8(16, 4224, 9216) && ran("k_gemm"));
    CHECK(int8(12, 4224, 9216) && ran("k_stream"));
    CHECK(int8(12, 4224, 40960) && ran("k_gemm"));
    CHECK(int8(4, 4224, 40960) && ran("k_stream"));
    // bf16 products that K slices of large tiles do not shorten
    CHECK(bf16(fd, 652, 3328, 1728) == 0 && !ran("k_sum_slices"));
    CHECK(bf16(fd, 320, 3776, 3536) == 0 && !ran("k_sum_slices"));
    CHECK(bf16(fd, 384, 9408, 2048) == 0 && ran("k_sum_slices"));
    // fp32 operands, few rows over many columns
    CHECK(bf16(fd, 16, 3840, 12288) == 0 && ran("k_gemm"));
    CHECK(bf16(fd, 12, 3840, 12288) == 0 && ran("k_stream"));
    CHECK(bf16(fd, 16, 3456, 9216) == 0 && ran("k_gemm"));
    CHECK(bf16(fd, 16, 3072, 20480) == 0 && ran("k_stream"));
    CHECK(bf16(fd, 12, 2048, 14336) == 0 && ran("k_gemm"));
    CHECK(bf16(fd, 8, 8192, 14336) == 0 && ran("k_gemm"));
    CHECK(tf32(16, 3840, 32768) && ran("k_gemm"));
    CHECK(tf32(4, 3840, 32768) && ran("k_stream"));
    // and their rows, converted ahead where tiles without K slices read them
    CHECK(tf32(20, 3840, 14336) && ran("k_cvt"));
    CHECK(tf32(100, 3840, 10240) && ran("k_cvt"));
    CHECK(tf32(20, 1536, 7168) && ran("k_cvt"));
    CHECK(tf32(1040, 256, 7792) && ran("k_cvt"));
    CHECK(tf32(944, 128, 5312) && ran("k_cvt"));
    CHECK(tf32(512, 128, 7792) && !ran("k_cvt"));
    CHECK(bf16(fd, 20, 3072, 10240) == 0 && ran("k_cvt"));
    CHECK(bf16(fd, 20, 512, 32768) == 0 && ran("k_cvt"));
    // few-row group-wise launches of many tiles: as many waves a workgroup as make one batch of them, and
    // rows quantised there only where that takes less than a pass ahead
    auto moe = [&](int np, int M, int K, int N, int g, int qa) {
        rk::Launch L;
        L.fmt_a = L.fmt_b = rk::Fmt::I8; L.epi = rk::Epi::GW; L.N = N; L.K = L.kend = K;
        L.group = L.kt = g; L.rowscale = 1; L.qa = qa; L.act = qa ? rk::kActSilu : 0;
        L.nprob = np;
        for (int i = 0; i < np; i++) L.prob[i] = rk::Problem{M, A, B, Y + 4096L * 4096 * i, X, W, nullptr};
        for (int i = 0; qa && i < np; i++) L.prob[i].A2 = A;
        uint64_t blocks = 0;
        if (qa && !rk::gemm_quantises(L)) return uint64_t{0};
        CHECK(rk::gemm_launch(L, &blocks) == hipSuccess);
        fake::st().launches.clear();
        return blocks;
    };
    CHECK(moe(16, 16, 1632, 1248, 32, 0) == 16 * 10);
    CHECK(moe(16, 12, 3328, 1280, 128, 0) == 16 * 10);
    CHECK(moe(16, 8, 2048, 1408, 32, 0) == 16 * 44);
    CHECK(moe(8, 16, 896, 2688, 128, 2) == 8 * 21);
    CHECK(moe(8, 12, 576, 2176, 32, 2) == 8 * 17);
    CHECK(moe(8, 8, 1408, 2048, 32, 2) == 8 * 32);
    CHECK(moe(8, 16, 1856, 3872, 32, 2) == 0);
    // fp16, 17 to 32 rows of short K
    CHECK(fp16(fd, 32, 992, 32768) == 0 && ran("k_small_f16"));
    CHECK(fp16(fd, 32, 992, 65536) == 0 && ran("k_gemm"));
    rocket_close(fd);
}

// No host memory for the lists that a growing arena and the overlap check keep: an error code, or the
// answer that is right for all; no exception leaves a C entry.
static void short_of_host_memory()
{
    auto &f = fake::st();
    const int fd = open_async();
    CHECK(bf16(fd, 128, 8192, 512) == 0);
    captured([&] { return bf16(fd, 128, 8192, 512); });
    const int frees = f.frees;
    g_refuse = 1;
    int rc = 1;
    try {
        rc = rocket_matmul_bf16(fd, 512, 8192, 512, X, W, Y);
    } catch (...) {
    }
    g_refuse = 0;
    CHECK(rc == ROCKET_E_NOMEM);
    CHECK(f.frees == frees);
    CHECK(bf16(fd, 512, 8192, 512) == 0);
    CHECK(f.frees == frees);
    rocket_close(fd);

    std::vector<int> M(64, 4);
    std::vector<const void *> A(64, X);
    std::vector<void *> C(64, Y);
    rk::Req r;
    r.nprob = 64;
    r.M = M.data();
    r.A = A.data();
    r.C = C.data();
    r.N = 64;
    CHECK(!rk::results_overlap_rows(r, 64, 4));
    g_refuse = 1;
    bool over = false;
    try {
        over = rk::results_overlap_rows(r, 64, 4);
    } catch (...) {
    }
    g_refuse = 0;
    CHECK(over);
}

int main()
{
    arena_kept_for_graphs();
    small_calls_hold_no_scratch();
    rows_converted_without_an_arena();
    rows_quantised_without_an_arena();
    blocks_on_a_small_arena();
    short_of_memory();
    dumps_run_the_same_kernel();
    overlaps();
    routes();
    short_of_host_memory();
    if (g_fail) {
        fprintf(stderr, "arena_check: %d check(s) failed\n", g_fail);
        return 1;
    }
    printf("arena_check: all checks passed\n");
    return 0;
}
