// pgemm_lab — tiling / ring-depth sweep of the prefill GEMM (csrc/prefill.h pgemm_kernel) on the Llama-2-7B
// projection shapes at a 256-row chunk: device time per launch (HIP events, 20 launches), issued MFMA
// TFLOP/s (hi + lo: 4 N K M), and a spot check of 64 outputs against a host fp64 sum.
//   hipcc -O3 -std=c++17 --offload-arch=gfx950 -I simplellminference_amd/csrc tools/pgemm_lab.hip -o tools/pgemm_lab
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "prefill.h"

using namespace sli;

#define CK(x)                                                                          \
    do {                                                                               \
        hipError_t e_ = (x);                                                           \
        if (e_ != hipSuccess) {                                                        \
            fprintf(stderr, "%s:%d %s: %s\n", __FILE__, __LINE__, #x, hipGetErrorString(e_)); \
            exit(1);                                                                   \
        }                                                                              \
    } while (0)

static uint32_t rng(uint64_t& s) {
    s = s * 6364136223846793005ull + 1442695040888963407ull;
    return (uint32_t)(s >> 33);
}

struct Shape {
    const char* name;
    int N, K;
};

template <typename WT>
struct Bufs {
    WT* W;
    std::vector<WT*> Wc;  // the timing loop rotates over copies (none MALL-resident: weights stream from HBM as in
                          // the engine, where a layer's weights are read once per chunk)
    __half *hi, *lo;
    float* y;
    std::vector<WT> hW;
    std::vector<__half> hhi, hlo;
};

static float h2f(__half h) { return __half2float(h); }

template <typename WT>
static void make(Bufs<WT>& b, int N, int K, int M) {
    uint64_t s = 12345 + N + K;
    b.hW.resize((size_t)N * K);
    for (auto& w : b.hW) {
        if constexpr (sizeof(WT) == 1)
            w = (int8_t)((int)(rng(s) % 255) - 127);
        else
            w = __float2half(((int)(rng(s) % 2001) - 1000) * 1e-3f * 0.05f);
    }
    b.hhi.resize((size_t)M * K);
    b.hlo.resize((size_t)M * K);
    for (size_t i = 0; i < b.hhi.size(); ++i) {
        const float v = ((int)(rng(s) % 200001) - 100000) * 1e-5f;
        b.hhi[i] = __float2half(v);
        b.hlo[i] = __float2half(v - __half2float(b.hhi[i]));
    }
    CK(hipMalloc(&b.W, sizeof(WT) * b.hW.size()));
    CK(hipMalloc(&b.hi, 2 * b.hhi.size()));
    CK(hipMalloc(&b.lo, 2 * b.hlo.size()));
    CK(hipMalloc(&b.y, sizeof(float) * (size_t)M * N));
    CK(hipMemcpy(b.W, b.hW.data(), sizeof(WT) * b.hW.size(), hipMemcpyHostToDevice));
    const int ncopy = getenv("LAB_HOT") ? 1 : 4;
    b.Wc.assign(1, b.W);
    for (int c = 1; c < ncopy; ++c) {
        WT* p;
        CK(hipMalloc(&p, sizeof(WT) * b.hW.size()));
        CK(hipMemcpy(p, b.W, sizeof(WT) * b.hW.size(), hipMemcpyDeviceToDevice));
        b.Wc.push_back(p);
    }
    CK(hipMemcpy(b.hi, b.hhi.data(), 2 * b.hhi.size(), hipMemcpyHostToDevice));
    CK(hipMemcpy(b.lo, b.hlo.data(), 2 * b.hlo.size(), hipMemcpyHostToDevice));
}

template <typename WT>
static void release(Bufs<WT>& b) {
    for (auto* p : b.Wc) CK(hipFree(p));
    CK(hipFree(b.hi));
    CK(hipFree(b.lo));
    CK(hipFree(b.y));
}

static float* g_ws;
static unsigned* g_cnt;
// force: splits of every tile (0: the plan)
template <class Cfg, typename WT>
static void run(const char* name, Bufs<WT>& b, const Shape& sh, int M, int force = 0) {
    using Geo = PgGeo<Cfg, WT>;
    if (M % Geo::BM) return;
    PgPlan pl = pg_plan<Cfg, WT>(sh.N, sh.K, M, 256, true);
    if (force) {
        const int nx = ((sh.N + Geo::BN - 1) / Geo::BN + 7) / 8 * (M / Geo::BM), f = nx / (32 * (160 * 1024 / Geo::LDS)) * (32 * (160 * 1024 / Geo::LDS));
        if (force == 1) pl.full = 0x7fffffff, pl.splits = 1, pl.slots = nx;
        else pl.full = f, pl.splits = force, pl.slots = f + (nx - f) * force;
        if ((size_t)8 * (nx - f) * force * 16 * Geo::AT * Geo::WPT * Geo::THREADS > kPgWsBytes || (sh.K + Geo::KS - 1) / Geo::KS < force) return;
        if (force > 1 && nx == f) return;
    }
    char tag[96];
    snprintf(tag, sizeof tag, "%s full %d S %d", name, pl.full > 100000 ? -1 : pl.full, pl.splits);
    CK((pgemm_allow_lds<PgEpiResid, Cfg, WT>()));
    PgIn<WT> in{b.W, b.hi, b.lo, sh.N, sh.K, M};
    in.full = pl.full, in.splits = pl.splits, in.ws = g_ws, in.cnt = g_cnt;
    PgEpiResid e{b.y, nullptr, nullptr, sh.N, sh.N};
    CK(hipMemset(b.y, 0, sizeof(float) * (size_t)M * sh.N));
    CK((launch_pgemm<PgEpiResid, Cfg, WT>(in, e, PfState{0, M, M, 1}, 0)));
    CK(hipDeviceSynchronize());
    // spot check (y[m][row] = sum_k W[row][k] (hi + lo)[m][k])
    std::vector<float> y((size_t)M * sh.N);
    CK(hipMemcpy(y.data(), b.y, sizeof(float) * y.size(), hipMemcpyDeviceToHost));
    double maxrel = 0.0;
    uint64_t s = 777;
    for (int i = 0; i < 64; ++i) {
        const int m = rng(s) % M, row = rng(s) % sh.N;
        double ref = 0.0, mag = 0.0;
        for (int k = 0; k < sh.K; ++k) {
            double w;
            if constexpr (sizeof(WT) == 1)
                w = (double)b.hW[(size_t)row * sh.K + k];
            else
                w = (double)h2f(b.hW[(size_t)row * sh.K + k]);
            const double x = (double)h2f(b.hhi[(size_t)m * sh.K + k]) + (Cfg::NB == 2 ? (double)h2f(b.hlo[(size_t)m * sh.K + k]) : 0.0);
            ref += w * x;
            mag += fabs(w * x);
        }
        maxrel = fmax(maxrel, fabs(y[(size_t)m * sh.N + row] - ref) / (mag + 1e-30));
    }
    hipEvent_t e0, e1;
    CK(hipEventCreate(&e0));
    CK(hipEventCreate(&e1));
    const int iters = 20;
    CK(hipEventRecord(e0, 0));
    for (int i = 0; i < iters; ++i) {
        PgIn<WT> ic = in;
        ic.W = b.Wc[i % b.Wc.size()];
        CK((launch_pgemm<PgEpiResid, Cfg, WT>(ic, e, PfState{0, M, M, 1}, 0)));
    }
    CK(hipEventRecord(e1, 0));
    CK(hipEventSynchronize(e1));
    float ms = 0.0f;
    CK(hipEventElapsedTime(&ms, e0, e1));
    const double us = 1000.0 * ms / iters;
    const double tf = 2.0 * Cfg::NB * sh.N * sh.K * (double)M / (us * 1e-6) / 1e12;
    const double wgbs = (double)sh.N * sh.K * sizeof(WT) / (us * 1e-6) / 1e9;
    const int nrb = (sh.N + Geo::BN - 1) / Geo::BN;
    printf("%-5s %-6s %-22s grid %5d lds %6zu  %8.1f us  %6.1f TF issued  W %6.0f GB/s  relerr %.1e\n", sh.name,
           sizeof(WT) == 1 ? "i8" : "f16", tag, nrb * (M / Geo::BM), Geo::LDS, us, tf, wgbs, maxrel);
    fflush(stdout);
    CK(hipEventDestroy(e0));
    CK(hipEventDestroy(e1));
}

#define RUN(BM, WR, S, AT, SA)                                                            \
    for (int f : forces) run<PgCfg<BM, WR, S, AT, SA>, WT>("BM" #BM " WR" #WR " S" #S " AT" #AT " SA" #SA, b, sh, M, f)

// LAB_ONE: one fp16 image (block-stack models)
#define RUN1(BM, WR, S, AT)                                                               \
    for (int f : forces) run<PgCfg<BM, WR, S, AT, 0, 1>, WT>("BM" #BM " WR" #WR " S" #S " AT" #AT " NB1", b, sh, M, f)

template <typename WT>
static void sweep(const Shape& sh, int M, const std::vector<int>& forces) {
    Bufs<WT> b;
    make(b, sh.N, sh.K, M);
    if (getenv("LAB_ONE")) {
        if constexpr (sizeof(WT) == 2) {
            RUN1(256, 4, 2, 4);
            RUN1(128, 4, 2, 4);
            RUN1(128, 4, 3, 4);
            RUN1(128, 4, 2, 2);
            RUN1(128, 2, 3, 4);
            RUN1(64, 4, 3, 4);
            RUN1(64, 4, 4, 2);
            RUN1(64, 2, 4, 2);
            RUN1(32, 2, 4, 2);
            RUN1(32, 2, 4, 4);
        }
        release(b);
        return;
    }
    if constexpr (sizeof(WT) == 2) {
        if (M <= 32) {
            RUN(32, 2, 4, 2, 0);
            RUN(32, 4, 4, 2, 0);
            RUN(32, 4, 3, 4, 0);
            RUN(32, 2, 3, 2, 0);
            RUN(32, 4, 4, 3, 0);
        } else if (M <= 64) {
            RUN(64, 2, 4, 2, 0);
            RUN(64, 4, 4, 2, 0);
            RUN(64, 4, 3, 4, 0);
            RUN(64, 2, 3, 2, 0);
            RUN(64, 4, 3, 3, 0);
            RUN(64, 4, 2, 2, 0);
        } else if (M <= 96) {
            RUN(96, 4, 2, 2, 4);
            RUN(96, 4, 2, 4, 3);
            RUN(96, 4, 2, 3, 4);
            RUN(96, 4, 3, 2, 0);
            RUN(32, 4, 4, 2, 0);
        } else {
            RUN(64, 4, 3, 2, 0);
            RUN(128, 4, 2, 2, 4);
            RUN(128, 4, 2, 4, 3);
            RUN(128, 4, 2, 4, 0);
        }
    } else {
        if (M <= 32) {
            RUN(32, 2, 4, 2, 0);
            RUN(32, 4, 4, 2, 0);
            RUN(32, 2, 3, 2, 0);
            RUN(32, 4, 3, 4, 0);
        } else if (M <= 64) {
            RUN(64, 4, 2, 2, 0);
            RUN(64, 4, 3, 2, 0);
            RUN(64, 4, 2, 4, 0);
            RUN(64, 4, 2, 3, 0);
            RUN(64, 2, 2, 2, 0);
        } else if (M <= 96) {
            RUN(96, 4, 2, 2, 0);
            RUN(96, 2, 2, 2, 0);
            RUN(32, 4, 4, 2, 0);
        } else {
            RUN(64, 4, 3, 2, 0);
            RUN(128, 4, 2, 2, 0);
        }
    }
    release(b);
}

// pgemm_lab M [splits ...]: splits 0 = the plan, 1 = none, n = the last round's tiles cut into n
int main(int argc, char** argv) {
    const int M = argc > 1 ? atoi(argv[1]) : 256;
    std::vector<int> forces;
    for (int i = 2; i < argc; ++i) forces.push_back(atoi(argv[i]));
    if (forces.empty()) forces = {0, 1};
    CK(hipMalloc(&g_ws, kPgWsBytes));
    CK(hipMalloc(&g_cnt, sizeof(unsigned) * kPgWsTiles));
    CK(hipMemset(g_cnt, 0, sizeof(unsigned) * kPgWsTiles));
    std::vector<Shape> shapes = {{"qkv", 12288, 4096}, {"gu", 22016, 4096}, {"wo", 4096, 4096}, {"down", 4096, 11008}};
    if (getenv("LAB_ONE")) shapes = {{"in7b", 34304, 4096}, {"out7b", 4096, 15104}, {"in1b", 22528, 2048}, {"out1b", 2048, 10240}};
    if (!getenv("LAB_I8"))
        for (const Shape& sh : shapes) sweep<__half>(sh, M, forces);
    else
        for (const Shape& sh : shapes) sweep<int8_t>(sh, M, forces);
    return 0;
}
