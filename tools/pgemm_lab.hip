// pgemm_lab — the tilings of the prompt GEMM (csrc/prefill.h pg_tilings, pg_row_tilings):
//   pgemm_lab M [splits ...]  device time per launch at M rows of the 7B projections (HIP events, 20 launches, weights
//                             streamed from HBM), issued MFMA TFLOP/s, a spot check of 64 outputs against a host fp64 sum.
//                             splits 0 = the plan, 1 = whole tiles, n = the last round's tiles cut into n. Each projection
//                             ends with the tiling that the engine takes, its time and the fastest
//   pgemm_lab stages          time of one stage of every tiling with the chip full of whole tiles (two rounds over a depth
//                             of 8192), weights read once (one position block) and shared by eight, beside the listed one
// LAB_W: f16 (default), i8, f32, or one (a single fp16 image: the block stacks' tilings).
//   hipcc -O3 -std=c++17 --offload-arch=gfx950 -Xclang -target-feature -Xclang -packed-fp32-ops
//         -I simplellminference_amd/csrc -I include tools/pgemm_lab.hip -o tools/pgemm_lab
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
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

// what a GEMM reads beside WT weights
template <typename WT>
struct XOf {
    typedef __half type;
};
template <>
struct XOf<float> {
    typedef float type;
};

template <typename WT>
struct Bufs {
    typedef typename XOf<WT>::type X;
    WT* W;
    std::vector<WT*> Wc;  // the timing loop rotates over copies (none MALL-resident: weights stream from HBM as in
                          // the engine, where a layer's weights are read once per chunk)
    X *hi, *lo;
    float* y;
    std::vector<WT> hW;
    std::vector<X> hhi, hlo;
};

static float h2f(__half h) { return __half2float(h); }
static float h2f(float v) { return v; }
static void put(__half& h, float v) { h = __float2half(v); }
static void put(float& h, float v) { h = v; }

template <typename WT>
static void make(Bufs<WT>& b, int N, int K, int M) {
    uint64_t s = 12345 + N + K;
    b.hW.resize((size_t)N * K);
    for (auto& w : b.hW) {
        if constexpr (sizeof(WT) == 1)
            w = (int8_t)((int)(rng(s) % 255) - 127);
        else
            put(w, ((int)(rng(s) % 2001) - 1000) * 1e-3f * 0.05f);
    }
    b.hhi.resize((size_t)M * K);
    b.hlo.resize((size_t)M * K);
    for (size_t i = 0; i < b.hhi.size(); ++i) {
        const float v = ((int)(rng(s) % 200001) - 100000) * 1e-5f;
        put(b.hhi[i], v);
        put(b.hlo[i], v - h2f(b.hhi[i]));
    }
    CK(hipMalloc(&b.W, sizeof(WT) * b.hW.size()));
    CK(hipMalloc(&b.hi, sizeof(b.hhi[0]) * b.hhi.size()));
    CK(hipMalloc(&b.lo, sizeof(b.hlo[0]) * b.hlo.size()));
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
    CK(hipMemcpy(b.hi, b.hhi.data(), sizeof(b.hhi[0]) * b.hhi.size(), hipMemcpyHostToDevice));
    CK(hipMemcpy(b.lo, b.hlo.data(), sizeof(b.hlo[0]) * b.hlo.size(), hipMemcpyHostToDevice));
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
struct Timed {
    std::string tag;
    double us = 1e30;
};
// rows are padded to the tiling's; force: splits of the last round's tiles (0: the plan); returns the time and what it is of
template <class Cfg, typename WT>
static Timed run(const char* name, Bufs<WT>& b, const Shape& sh, int rows, int force, float stage) {
    using Geo = PgGeo<Cfg, WT>;
    const int M = (rows + Geo::BM - 1) / Geo::BM * Geo::BM;
    PgPlan pl = pg_plan<Cfg, WT>(sh.N, sh.K, M, 256, true, stage);
    if (force) {
        const int nx = ((sh.N + Geo::BN - 1) / Geo::BN + 7) / 8 * (M / Geo::BM), f = nx / (32 * (160 * 1024 / Geo::LDS)) * (32 * (160 * 1024 / Geo::LDS));
        if (force == 1) pl.full = 0x7fffffff, pl.splits = 1, pl.slots = nx;
        else pl.full = f, pl.splits = force, pl.slots = f + (nx - f) * force;
        if ((size_t)8 * (nx - f) * force * 16 * Geo::AT * Geo::WPT * Geo::THREADS > kPgWsBytes || (sh.K + Geo::KS - 1) / Geo::KS < force) return {};
        if (force > 1 && nx == f) return {};
    }
    char tag[96];
    snprintf(tag, sizeof tag, "%s full %d S %d", name, pl.full > 100000 ? -1 : pl.full, pl.splits);
    CK((pgemm_allow_lds<PgEpiResid, Cfg, WT>()));
    PgIn<WT> in{b.W, (const __half*)b.hi, (const __half*)b.lo, sh.N, sh.K, M};
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
        const int m = rng(s) % rows, row = rng(s) % sh.N;
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
           sizeof(WT) == 1 ? "i8" : sizeof(WT) == 4 ? "f32" : "f16", tag, nrb * (M / Geo::BM), Geo::LDS, us, tf, wgbs, maxrel);
    fflush(stdout);
    CK(hipEventDestroy(e0));
    CK(hipEventDestroy(e1));
    return {tag, us};
}

template <class Cfg>
static std::string name_of(Cfg) {
    char t[96];
    snprintf(t, sizeof t, "BM%d WR%d S%d AT%d SA%d%s%s", Cfg::BM, Cfg::WR, Cfg::S, Cfg::AT, Cfg::SA, Cfg::NB == 1 ? " NB1" : "",
             Cfg::FO ? " FO" : "");
    return t;
}
template <typename WT, class F>
static void each(bool one, int M, F&& f) {
    if constexpr (sizeof(WT) == 2)
        if (one) return M ? pg_row_tilings(M, false, f) : (pg_row_tilings(32, false, f), pg_row_tilings(256, false, f));
    pg_tilings<WT>(f);
}

template <typename WT>
static void sweep(const Shape& sh, int M, const std::vector<int>& forces, bool one) {
    Bufs<WT> b;
    make(b, sh.N, sh.K, M + 128);
    Timed pick, best;
    float least = INFINITY;
    each<WT>(one, M, [&](auto cfg, float us) {
        using Cfg = decltype(cfg);
        for (int f : forces) {
            const Timed t = run<Cfg, WT>(name_of(cfg).c_str(), b, sh, M, f, us);
            if (!one && PgGeo<Cfg, WT>::FOLD == 0 && !pg_one_chain(sh.N, sh.K, M)) continue;  // (listed, not taken)
            if (t.us < best.us) best = t;
            const float p = pg_plan<Cfg, WT>(sh.N, sh.K, (M + Cfg::BM - 1) / Cfg::BM * Cfg::BM, 256, true, us).us;
            if (f == 0 && p < least) least = p, pick = t;
        }
    });
    printf("%-5s taken: %s %.1f us (%.1f planned); fastest: %s %.1f us\n", sh.name, pick.tag.c_str(), pick.us, least, best.tag.c_str(), best.us);
    release(b);
}

__global__ void fill(unsigned* p, size_t n, unsigned mask, unsigned bias) {  // (fp16 / fp32: small values of either sign)
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        unsigned h = (unsigned)i * 2654435761u;
        h ^= h >> 15, h *= 0x85ebca6bu, h ^= h >> 13;
        p[i] = (h & mask) | bias;
    }
}
template <typename WT>
static void stages(bool one) {
    constexpr unsigned mask = sizeof(WT) == 1 ? 0xffffffffu : sizeof(WT) == 2 ? 0x83ff83ffu : 0x807fffffu;
    constexpr unsigned bias = sizeof(WT) == 1 ? 0u : sizeof(WT) == 2 ? 0x28002800u : 0x3d000000u;
    const int K = 8192;
    each<WT>(one, 0, [&](auto cfg, float us) {
        using Cfg = decltype(cfg);
        using Geo = PgGeo<Cfg, WT>;
        typedef typename XOf<WT>::type X;
        CK((pgemm_allow_lds<PgEpiResid, Cfg, WT>()));
        const int occ = 160 * 1024 / Geo::LDS;
        printf("%-4s %-26s BN %3d occ %d listed %.2f us a stage |", one ? "one" : sizeof(WT) == 1 ? "i8" : sizeof(WT) == 4 ? "f32" : "f16",
               name_of(cfg).c_str(), Geo::BN, occ, us);
        for (int PB : {1, 8}) {
            const int N = 8 * Geo::BN * (2 * 32 * occ / PB), M = PB * Geo::BM;
            WT* W;
            X *hi, *lo;
            float* y;
            const size_t nw = sizeof(WT) * (size_t)N * K, nx = sizeof(X) * (size_t)M * K;
            CK(hipMalloc(&W, nw));
            CK(hipMalloc(&hi, nx));
            CK(hipMalloc(&lo, nx));
            CK(hipMalloc(&y, sizeof(float) * (size_t)M * N));
            hipLaunchKernelGGL(fill, dim3(4096), dim3(256), 0, 0, (unsigned*)W, nw / 4, mask, bias);
            const unsigned xm = sizeof(X) == 2 ? 0x83ff83ffu : 0x807fffffu;
            hipLaunchKernelGGL(fill, dim3(1024), dim3(256), 0, 0, (unsigned*)hi, nx / 4, xm, sizeof(X) == 2 ? 0x38003800u : 0x3f000000u);
            hipLaunchKernelGGL(fill, dim3(1024), dim3(256), 0, 0, (unsigned*)lo, nx / 4, xm, sizeof(X) == 2 ? 0x0c000c00u : 0x3f000000u);
            PgIn<WT> in{W, (const __half*)hi, (const __half*)lo, N, K, M};
            PgEpiResid e{y, nullptr, nullptr, N, N};
            hipEvent_t e0, e1;
            CK(hipEventCreate(&e0));
            CK(hipEventCreate(&e1));
            for (int i = 0; i < 2; ++i) CK((launch_pgemm<PgEpiResid, Cfg, WT>(in, e, PfState{0, M, M, 1}, 0)));
            CK(hipEventRecord(e0, 0));
            for (int i = 0; i < 5; ++i) CK((launch_pgemm<PgEpiResid, Cfg, WT>(in, e, PfState{0, M, M, 1}, 0)));
            CK(hipEventRecord(e1, 0));
            CK(hipEventSynchronize(e1));
            float ms = 0.0f;
            CK(hipEventElapsedTime(&ms, e0, e1));
            printf(" %d block%s %.2f", PB, PB > 1 ? "s" : "", 1000.0 * ms / 5 / 2 / (K / Geo::KS + 5));
            fflush(stdout);
            CK(hipEventDestroy(e0));
            CK(hipEventDestroy(e1));
            CK(hipFree(W));
            CK(hipFree(hi));
            CK(hipFree(lo));
            CK(hipFree(y));
        }
        printf("\n");
        fflush(stdout);
    });
}

template <typename WT>
static void all(int argc, char** argv, bool one) {
    if (argc > 1 && !strcmp(argv[1], "stages")) return stages<WT>(one);
    const int M = argc > 1 ? atoi(argv[1]) : 256;
    std::vector<int> forces;
    for (int i = 2; i < argc; ++i) forces.push_back(atoi(argv[i]));
    if (forces.empty()) forces = {0, 1};
    std::vector<Shape> shapes = {{"qkv", 12288, 4096}, {"gu", 22016, 4096}, {"wo", 4096, 4096}, {"down", 4096, 11008}};
    if (one) shapes = {{"in7b", 34304, 4096}, {"out7b", 4096, 15104}, {"in1b", 22528, 2048}, {"out1b", 2048, 10240}};
    for (const Shape& sh : shapes) sweep<WT>(sh, M, forces, one);
}

int main(int argc, char** argv) {
    const std::string w = getenv("LAB_W") ? getenv("LAB_W") : "f16";
    CK(hipMalloc(&g_ws, kPgWsBytes));
    CK(hipMalloc(&g_cnt, sizeof(unsigned) * kPgWsTiles));
    CK(hipMemset(g_cnt, 0, sizeof(unsigned) * kPgWsTiles));
    if (w == "i8")
        all<int8_t>(argc, argv, false);
    else if (w == "f32")
        all<float>(argc, argv, false);
    else
        all<__half>(argc, argv, w == "one");
    return 0;
}
