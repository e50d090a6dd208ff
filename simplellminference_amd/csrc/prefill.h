// prefill.h — prompt prefill as real GEMMs over the prompt (the reference teacher-forces the
// prompt one token per forward, source/model/model.cpp:157-165, so every weight is streamed once per prompt
// token). Here a chunk of up to kPfMaxChunk prompt positions runs through each layer together:
//
//   1. pf_norm_split_kernel: per position RMSNorm (rms_kernel.cpp:5-23, fp32) and the split of the fp32
//      result into fp16 hi + lo (hi = fp16(h), lo = fp16(h - hi): h to ~2^-22 relative);
//   2. pgemm_kernel: Y[pos][row] = sum_k W[row][k] * H[pos][k] on MFMA (v_mfma_f32_16x16x32_f16), A = a 16-row
//      weight tile, B = 16 positions' hi columns, then the same tile with the lo columns into the same fp32
//      accumulator (W * (hi + lo)); a workgroup owns 16 AT WR weight rows x BM positions (PgCfg), so a weight row
//      is read from HBM once per BM positions (the decode step reads it once per position). Operands are staged
//      through an S-deep LDS ring by LDS-DMA (global_load_lds_dwordx4: one 1-KiB fragment image per
//      wave-instruction, read back conflict-free by ds_read_b128), S - 1 stages in flight behind a counted
//      vmcnt and a raw s_barrier, or the weight images
//      in a deeper ring of their own (PgCfg::SA); the fragment reads of the next k-block and the next stage's DMA are
//      spread between the current k-block's MFMAs. Fused epilogues:
//      RoPE + K/V cache rows + q (model.cpp:52-67), residual add (:86-90, :124-128), SwiGLU (:111-115,
//      written straight as the down projection's hi/lo operand);
//   3. pf_flash_kernel (fp16 KV): block-causal attention against the cache rows 0 .. position (mha_kernel.cpp:36-77
//      per query: s_t = q.k_t * scale, softmax, sum p_t v_t): S = K q^T on MFMA with q in two fp16 terms (batches:
//      three), online softmax in fp32, P V on MFMA with V read transposed (ds_read_b64_tr_b16) from LDS-DMA'd K/V tiles; pf_attn_kernel, the
//      VALU form (fp32, 64-position query blocks, K/V tiles of 64 positions in LDS), serves fp32 KV caches and fp32 weights.
// fp32 weights: the same GEMM on v_mfma_f32_16x16x4_f32 with fp32 activations (one image, stages of 32 k).
// int8 weights: stages of 128 k; a depth that is 64 mod 128 (e.g. Llama-2-7B int8 down at TP 4, 2752) ends with
// a half stage (pgemm_kernel).
// The launches of a chunk go to the stream one by one (its start position and valid count are kernel arguments): at the
// widths of a 7B model each runs longer than it takes to enqueue, and a captured graph would add its capture to a model's
// first prompt.
#pragma once
#include <algorithm>
#include <type_traits>
#include <utility>

#include "common.h"
#include "step_state.h"

namespace sli {

// Prompt positions per weight pass. The activations of a chunk (at 4096 rows of a 7B model 0.4 GB) are small beside the
// weights, and every chunk pays a partial last round of tiles per GEMM (pg_plan) and reads the weights once. Where that does
// not fit beside the model, chunks are smaller (engine.hip pf_ready).
constexpr int kPfMaxChunk = 4096;
constexpr int kPgGroup = 8;        // position blocks that an XCD takes through its row blocks together

// nseq sequences (cache slots in order) of rps chunk rows each, rps a multiple of 16 (fp32 cache: 64): row i of a sequence
// is its position p0 + i.
struct PfState {
    int32_t p0 = 0;
    int32_t nv = 0;  // valid rows of a sequence (the rest is padding: computed, never written to the cache)
    int32_t rps = 1, nseq = 1;
};

typedef _Float16 pf_half8 __attribute__((ext_vector_type(8)));
typedef float pf_float4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ pf_float4 pf_mfma(const u32x4& a, const u32x4& b, pf_float4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(pf_half8, a), __builtin_bit_cast(pf_half8, b), c,
                                                  0, 0, 0);
}

// fp32 -> fp16 hi + fp16 lo
__device__ __forceinline__ void pf_split(float v, __half& hi, __half& lo) {
    hi = __float2half_rn(v);
    lo = __float2half_rn(v - __half2float(hi));
}

// v as N fp16 terms, each the rounding of what the ones before leave: 2 carry 22 to 23 bits, 3 all 24 (down to the fp16
// subnormal step 2^-24)
template <int N>
__device__ __forceinline__ void pf_terms(float v, __half (&t)[N][8], int e) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
        t[i][e] = __float2half_rn(v);
        v -= __half2float(t[i][e]);
    }
}

// What a GEMM reads: fp16 hi + lo, or fp32 (beside fp32 weights)
struct PfOut {
    __half *hi = nullptr, *lo = nullptr;
    float* f = nullptr;
    template <int N>
    __device__ __forceinline__ void store(size_t i, const float* v) const {  // N = 2 or 4 values, i a multiple of N
        if (f) {
            if constexpr (N == 4)
                *reinterpret_cast<float4*>(f + i) = make_float4(v[0], v[1], v[2], v[3]);
            else
                *reinterpret_cast<float2*>(f + i) = make_float2(v[0], v[1]);
            return;
        }
        __half hh[N], hl[N];
#pragma unroll
        for (int e = 0; e < N; ++e) pf_split(v[e], hh[e], hl[e]);
        typedef typename std::conditional<N == 4, uint2, unsigned>::type T;
        *reinterpret_cast<T*>(hi + i) = *reinterpret_cast<const T*>(hh);
        *reinterpret_cast<T*>(lo + i) = *reinterpret_cast<const T*>(hl);
    }
};

// ---------------------------------------------------------------- 1. embedding + RMSNorm / split
// x[m] = emb[prompt[p0 + i]] of the row's sequence (emb_kernel.cpp:4-21; padding rows repeat the last valid token)
template <typename WT>
__global__ void __launch_bounds__(256) pf_embed_kernel(PfState ps, const int32_t* __restrict__ prompt,
                                                      int prompt_ld, const WT* __restrict__ emb,
                                                      const float* __restrict__ emb_s, float* __restrict__ x, int D) {
    const int m = blockIdx.x;
    const int b = min(m / ps.rps, ps.nseq - 1);
    const int tok = prompt[(size_t)b * prompt_ld + ps.p0 + min(m - b * ps.rps, ps.nv - 1)];
    const float s = emb_s ? emb_s[tok] : 1.0f;
    for (int i = threadIdx.x; i < D; i += 256) x[(size_t)m * D + i] = to_f32(emb[(size_t)tok * D + i]) * s;
}

// y[b] = the residual row of sequence b's last valid position in the chunk
static __global__ void __launch_bounds__(256) pf_last_rows_kernel(PfState ps, const float* __restrict__ x, float* __restrict__ y, int D) {
    const float* r = x + ((size_t)blockIdx.x * ps.rps + ps.nv - 1) * D;
    for (int i = threadIdx.x; i < D; i += 256) y[(size_t)blockIdx.x * D + i] = r[i];
}

// Partial sums of a GEMM that the next norm adds up (PgIn::defer): x += (part[0] + .. + part[n - 1]) * rscale, in x
struct PfPart {
    const float* part = nullptr;  // [n][rows][D]
    int n = 0;
    size_t stride = 0;  // rows D
    const float* rscale = nullptr;
};

// one workgroup per chunk row: h = (x * 1/rms) * w (rms_kernel.cpp:12-22) or plain x (w == nullptr), as hi/lo.
// The row is held in registers (a float4 per thread and pass; D % 4 == 0, D <= 8192): one read of x, 8-byte
// hi / lo stores. 512 threads a row for few rows (pp: more loads in flight: 45 rows 1 us less), 256 else.
template <int THREADS>
__global__ void __launch_bounds__(THREADS) pf_norm_split_kernel(float* __restrict__ x, const float* __restrict__ w, PfOut out,
                                                                int D, float eps, PfPart pp) {
    constexpr int MAXV = 8192 / 4 / THREADS;  // float4 per thread: D <= 8192
    constexpr int PB = 8;                     // partial sums in flight
    const int m = blockIdx.x;
    float* xr = x + (size_t)m * D;
    const int n4 = D / 4;
    float4 v[MAXV], wv[MAXV];
    float ss = 0.0f;
    // the norm weights are loaded with x, not after the reduction: one memory round trip fewer
    const float4* w4 = reinterpret_cast<const float4*>(w ? w : xr);
#pragma unroll
    for (int j = 0; j < MAXV; ++j) {
        const int i = j * THREADS + (int)threadIdx.x;
        if (i < n4) {
            v[j] = reinterpret_cast<const float4*>(xr)[i];
            wv[j] = w4[i];
            if (pp.n) {
                const float4* p4 = reinterpret_cast<const float4*>(pp.part + (size_t)m * D) + i;
                const float4 sc = pp.rscale ? reinterpret_cast<const float4*>(pp.rscale)[i] : make_float4(1.0f, 1.0f, 1.0f, 1.0f);
                float4 s = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                for (int q0 = 0; q0 < pp.n; q0 += PB) {
                    float4 t[PB];
#pragma unroll
                    for (int q = 0; q < PB; ++q) t[q] = p4[(size_t)min(q0 + q, pp.n - 1) * (pp.stride / 4)];
#pragma unroll
                    for (int q = 0; q < PB; ++q)
                        if (q0 + q < pp.n) s.x += t[q].x, s.y += t[q].y, s.z += t[q].z, s.w += t[q].w;
                }
                if (pp.rscale) s.x *= sc.x, s.y *= sc.y, s.z *= sc.z, s.w *= sc.w;
                v[j].x += s.x, v[j].y += s.y, v[j].z += s.z, v[j].w += s.w;
                reinterpret_cast<float4*>(xr)[i] = v[j];
            }
            ss += v[j].x * v[j].x + v[j].y * v[j].y + v[j].z * v[j].z + v[j].w * v[j].w;
        }
    }
    float inv = 1.0f;
    if (w) {
        ss = wave_sum(ss);
        __shared__ float red[THREADS / 64];
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
        __syncthreads();
        float t = red[0];
#pragma unroll
        for (int k = 1; k < THREADS / 64; ++k) t += red[k];
        const float tep = t / (float)D;      // rms_kernel.cpp:17
        const float rms = sqrtf(tep + eps);  // :18
        inv = 1.0f / rms;                    // :19
    }
#pragma unroll
    for (int j = 0; j < MAXV; ++j)
        if (j * THREADS + (int)threadIdx.x < n4) {
            const int i = (j * THREADS + threadIdx.x) * 4;
            const float f[4] = {v[j].x, v[j].y, v[j].z, v[j].w}, g[4] = {wv[j].x, wv[j].y, wv[j].z, wv[j].w};
            float y[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = w ? (f[e] * inv) * g[e] : f[e];  // :20-22
            out.store<4>((size_t)m * D + i, y);
        }
}

// ---------------------------------------------------------------- 2. the GEMM
// LDS-DMA of one 1-KiB fragment image: lane i's 16 bytes at gsrc land at LDS byte lds + 16 i (inline asm: the
// compiler neither counts nor drains it; the kernel counts its own vmcnt). m0 is named as written, so the compiler sets it
// anew for its own uses.
__device__ __forceinline__ void pf_dma(const void* gsrc, unsigned lds) {
    asm volatile(
        "s_mov_b32 m0, %1\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %0, off"
        :
        : "v"(gsrc), "s"(lds)
        : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void pf_wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Grouped form (PgCfg::GR): row block pb of BM output rows multiplies its own weight matrix. tiles[pb] = {weight group,
// first input row}; input row i of the block is rowmap[pb * BM + i] where a row map is given, else tiles[pb].y + i.
// Blocks from *ntiles on (a device count; the grid is sized for the most there can be) return at once.
struct PgGroups {
    const int2* tiles = nullptr;
    const int32_t* ntiles = nullptr;
    const int32_t* rowmap = nullptr;
    size_t wstride = 0;  // elements between two groups' weights
};

template <typename WT>
struct PgIn {
    const WT* W;        // [N][K] fp32, fp16 or int8 (row-major, PyTorch [out][in]; int8 row scales in the epilogue)
    const __half* Bhi;  // [M][K] activations, fp16 hi (fp32 weights: fp32)
    const __half* Blo;  // [M][K] fp16 lo
    int N, K, M;        // rows, depth, chunk rows (a multiple of BM)
    // weight rows from row_b2 on (a multiple of the tiling's BN) read their activations from Bhi2 (one image only)
    const __half* Bhi2 = nullptr;
    int row_b2 = 0x7fffffff;
    PgGroups grp;
    // The launch's slots, per XCD (pg_plan): the first `full` own a whole tile each, the tiles after them are cut into
    // `splits` depth ranges (partial sums in ws [tail tile][split], arrival counters in cnt, zero between launches).
    int full = 0x7fffffff, splits = 1;
    float* ws = nullptr;
    unsigned* cnt = nullptr;
    // (epilogues with kDefer, where every tile is cut) the sums stay partial: ws [split][M][N], for the launch that reads them
    bool defer = false;
    int valid = 0x7fffffff;  // chunk rows from here on are padding: a wave that holds only such rows multiplies nothing
};

// Tiling: a workgroup of 2 WR waves owns BN = 32 WR weight rows x BM chunk rows; wave w holds the 2 x BM/32
// accumulator tiles of rows 32 (w % WR) .. +32 and position half w / WR. A stage covers KS depth: 64 for fp16
// weights, 128 for int8, so a weight row's slice is one whole 128-byte line (a chunk row's fp16 hi / lo slice
// one or two lines). Each LDS-DMA wave-instruction moves 1 KiB of whole lines (8 rows x 128 B or 4 x 256 B;
// fragment-shaped pieces of 16 rows x 64 B fetched every line twice and capped the ingest at ~29 GB/s per
// CU, tools/pgemm_lab); the 16-byte chunks of a row are XOR-swizzled by the row so the fragment reads
// (16 rows x 16 B per lane group) stay conflict-free. S stages in the LDS ring, S - 1 of them in flight.
// Epilogue contract: row(t, i) = weight row of 16-row tile t's row i (i < 16, always valid); store(t, i0, m, v)
// gets the fp32 sums of tile rows i0 .. i0+3 (i0 % 4 == 0) for chunk row m.
// AT_: 16-row weight tiles per wave (2: a wave's 32 rows; 4: 64 rows, so every B fragment read from LDS feeds twice
// the MFMAs). The fragment reads of k-block j + 1 run beside the MFMAs of k-block j (two register sets), across the stage
// barrier too.
// SA_ > 0: the weight (A) images get a ring of their own, SA_ stages deep (SA_ - 1 issued ahead), and
// the activation (B) images a 2-stage ring (one ahead): the A bytes come from HBM (read once per chunk), the B bytes
// from L2, so only A needs the longer prefetch, and B, the larger image, does not pay for it in LDS. Loads are waited for in
// order and every stage's activations are waited for, so a weight stage has two iterations to land whatever SA_ is: a fourth
// slot holds a stage that has landed.
// NB_: activation images per position: 2 (fp16 hi + lo, two MFMAs per product) or 1 (fp16 activations).
// GR_: row blocks with weights of their own (PgGroups; one image).
// FO_: short chains (PgGeo::FOLD) for a 64 x 64 wave tile too.
template <int BM_, int WR_, int S_, int AT_ = 2, int SA_ = 0, int NB_ = 2, bool GR_ = false, bool FO_ = false>
struct PgCfg {
    static_assert(NB_ == 2 || NB_ == 1, "activation images");
    static_assert(!GR_ || NB_ == 1, "grouped: one image");
    static constexpr bool GR = GR_, FO = FO_;
    static constexpr int BM = BM_, WR = WR_, S = S_, AT = AT_, SA = SA_, NB = NB_;
};

template <class Cfg, typename WT>
struct PgGeo {
    static constexpr int BM = Cfg::BM, WR = Cfg::WR, S = Cfg::S, AT = Cfg::AT, NB = Cfg::NB;
    static constexpr int WAVES = 2 * WR, THREADS = 64 * WAVES, BN = 16 * AT * WR;
    static constexpr bool F32 = sizeof(WT) == 4;
    static constexpr int KS = sizeof(WT) == 1 ? 128 : F32 ? 32 : 64;  // depth per stage
    static constexpr int KBS = KS / (F32 ? 16 : 32);       // k-blocks per stage: an MFMA per tile, fp32 four
    static constexpr int A_ROW = KS * (int)sizeof(WT);     // 128 B
    static constexpr int B_ROW = KS * (F32 ? 4 : 2);       // 128 or 256 B
    static constexpr int A_IMG = 16 * A_ROW, B_IMG = 16 * B_ROW;
    static constexpr int PT = BM / 16;  // position tiles per workgroup
    static constexpr int WPT = PT / 2;  // per wave
    static constexpr int NA = AT * WR;  // weight row tiles
    static constexpr int A_BYTES = NA * A_IMG;
    static constexpr int STAGE = A_BYTES + NB * PT * B_IMG;
    static constexpr int NDMA = STAGE / 1024;  // wave-instructions per stage
    // depth after which a wave's sums go into a second set of accumulators (0: one chain over the whole depth). hi + lo
    // activations keep 2^-23 of a value, one fp32 chain over 4096 k loses more: with it the logits after 100 tokens of
    // Llama-3-8B are 1.2e-4 from float64, with chains of 256 9.0e-5 (the decode step's: 8.9e-5). Up to 12 tiles a wave it
    // costs nothing; a 64 x 64 wave tile (16) 3 to 8 % of a GEMM, so there only where the caller's other route has them.
    // fp32: every 4 k are a sum of their own (mfmas), chained up to 512 k: no longer than the chains of the decode step's
    // lanes.
    static constexpr int FOLD = F32 ? 512 : NB == 2 && (AT * WPT <= 12 || Cfg::FO) ? 256 : 0;
    static_assert(!F32 || NB == 1, "fp32: one image");
    static constexpr int DPW = NDMA / WAVES;   // per wave
    static constexpr int SA = Cfg::SA;         // split rings (PgCfg): A pieces per wave DPA, B pieces DPB
    static constexpr int B_BYTES = STAGE - A_BYTES;
    static constexpr int DPA = SA ? A_BYTES / 1024 / WAVES : 0, DPB = SA ? B_BYTES / 1024 / WAVES : 0;
    static constexpr size_t LDS = SA ? (size_t)SA * A_BYTES + (size_t)S * B_BYTES : (size_t)S * STAGE;
    static_assert(A_ROW == 128 && WPT >= 1 && NDMA % WAVES == 0, "tiling");
    static_assert(S >= 2 && (S - 1) * DPW <= 63, "ring depth (vmcnt counts 63 loads)");
    // (SA > S: A(s) must be issued in an earlier iteration than B(s), the wait below counts on it; SA == S computed
    // wrong sums in tools/pgemm_lab)
    static_assert(SA == 0 || (S == 2 && SA > S && (A_BYTES / 1024) % WAVES == 0 &&
                              (B_BYTES / 1024) % WAVES == 0 && (SA - 1) * DPA + DPB <= 63), "split rings");
    static_assert(LDS <= 160 * 1024, "LDS");
};

// 16-byte chunk swizzle of an image row (conflict-free fragment reads): rows of 128 B pair up in one 256-B
// bank span, so the chunk index is XORed with row / 2; rows of 256 B with the row
__device__ __forceinline__ int pg_swz(int row, int row_bytes) { return row_bytes == 128 ? (row >> 1) & 7 : row & 15; }

// 8 int8 weights -> 8 fp16 (exact): fp16 bits 0x6400 | (b ^ 0x80) = 1024 + b + 128, minus 1152
__device__ __forceinline__ u32x4 pg_i8_to_f16(uint2 w) {
    u32x4 r;
    const unsigned x[2] = {w.x ^ 0x80808080u, w.y ^ 0x80808080u};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        // bytes b0 b1 -> halves (0x64 b0), (0x64 b1) via byte permutes
        const unsigned lo = __builtin_amdgcn_perm(0x64646464u, x[h], 0x05010400u);  // {b0, 0x64, b1, 0x64}
        const unsigned hi = __builtin_amdgcn_perm(0x64646464u, x[h], 0x07030602u);  // {b2, 0x64, b3, 0x64}
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        const h2 k = {(_Float16)1152.0f, (_Float16)1152.0f};
        r[2 * h] = __builtin_bit_cast(unsigned, __builtin_bit_cast(h2, lo) - k);
        r[2 * h + 1] = __builtin_bit_cast(unsigned, __builtin_bit_cast(h2, hi) - k);
    }
    return r;
}

// wait until at most `later` stages of DPW images each are still in flight (later: 0 .. 6)
template <int DPW>
__device__ __forceinline__ void pg_wait_stages(int later) {
    switch (later) {
        case 0: pf_wait_vm<0>(); break;
        case 1: pf_wait_vm<1 * DPW>(); break;
        case 2: pf_wait_vm<(2 * DPW > 63 ? 63 : 2 * DPW)>(); break;
        case 3: pf_wait_vm<(3 * DPW > 63 ? 63 : 3 * DPW)>(); break;
        case 4: pf_wait_vm<(4 * DPW > 63 ? 63 : 4 * DPW)>(); break;
        case 5: pf_wait_vm<(5 * DPW > 63 ? 63 : 5 * DPW)>(); break;
        default: pf_wait_vm<(6 * DPW > 63 ? 63 : 6 * DPW)>(); break;
    }
}

// f(std::integral_constant<int, 0>{}) .. f(<N - 1>): indices that are constants whatever the unroller makes of a loop
template <int N, class F, int... I>
__device__ __forceinline__ void pg_for_seq(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void pg_for(F&& f) {
    pg_for_seq<N>(f, std::make_integer_sequence<int, N>{});
}
#define PG_INLINE __attribute__((always_inline))

// Epilogues with a member kDefer = true may leave a cut round's sums partial (PgIn::defer): row i of tile t is t * 16 + i
template <class Epi, class = void>
struct PgDefers : std::false_type {};
template <class Epi>
struct PgDefers<Epi, std::enable_if_t<Epi::kDefer>> : std::true_type {};

// Epilogues with a member kRolled = true are too large to be unrolled over a wave's tiles: they are looped over its weight tiles.
// What a chunk row's stores need of it, row_of(m), is asked for once and for all of a wave's rows together; store(t, i0, m, v, r)
// gets it. Waves whose weight tiles t0 .. t0 + n - 1 are all flat(t0, n) are not looped: flat_store<n>(t0, lane group, m, v[n], r).
template <class Epi, class = void>
struct PgRolled : std::false_type {};
template <class Epi>
struct PgRolled<Epi, std::enable_if_t<Epi::kRolled>> : std::true_type {};

template <class Epi, class Cfg, typename WT>
__global__ void __launch_bounds__(128 * Cfg::WR) pgemm_kernel(PgIn<WT> in, Epi epi, PfState ps) {
    using Geo = PgGeo<Cfg, WT>;
    constexpr int KBS = Geo::KBS, BM = Geo::BM, WR = Geo::WR, S = Geo::S;
    extern __shared__ __attribute__((aligned(1024))) char pg_smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int wr = wave % WR, wp = wave / WR;  // row pair, position half
    const int PB = in.M / BM;
    const int nrb = (in.N + Geo::BN - 1) / Geo::BN;
    // Row block rb runs on XCD rb % 8 (blocks b and b + 8 share one under round-robin placement; speed only). An XCD
    // walks its row blocks in groups of kPgGroup position blocks, so that what runs on its CUs together is a block of
    // tiles that shares both operands in its L2.
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int nsp = slot < in.full ? 1 : in.splits;
    const int ti = nsp == 1 ? slot : in.full + (slot - in.full) / nsp, sp = nsp == 1 ? 0 : (slot - in.full) % nsp;
    const int nr8 = (nrb + 7) / 8, grp0 = ti / (nr8 * kPgGroup) * kPgGroup, gw = min(kPgGroup, PB - grp0);
    const int tg = ti - grp0 * nr8, rb = tg / gw * 8 + xcd, pb = grp0 + tg % gw;
    if (rb >= nrb) return;  // (uniform) padding of the grid to a multiple of 8 row blocks
    int2 tile = make_int2(0, 0);
    if constexpr (Cfg::GR) {
        if (pb >= *in.grp.ntiles) return;
        tile = in.grp.tiles[pb];
        in.W += (size_t)tile.x * in.grp.wstride;
    }
    // stages: K is a multiple of 64, so with int8 weights (KS 128) the last stage may be a half stage. Its DMA
    // pieces past the row's end reload the stage's first half instead (in bounds; never read), and only its
    // first KBS / 2 k-blocks are multiplied.
    // A split's stages are s0 .. s0 + ns - 1 (every split has one: pg_plan).
    const int nsk = (in.K + Geo::KS - 1) / Geo::KS;
    const int s0 = nsp == 1 ? 0 : nsk * sp / nsp, ns = (nsp == 1 ? nsk : nsk * (sp + 1) / nsp) - s0;
    constexpr bool HALF = sizeof(WT) == 1;
    const bool half_tail = HALF && (in.K % Geo::KS) != 0 && s0 + ns == nsk;
    const int nt = in.N >> 4;       // row tiles
    // Row blocks start their walk of the depth at different stages, rot on, and wrap around: workgroups that all walk from the
    // same column reach less of the memory's rate where rows of fp16 weights lie a multiple of 8 KiB apart (likely a few
    // channels at a time), of 4 KiB with one activation image. 22016 x 4096 at 32 | 64 | 96 rows 47.3 | 51.1 | 53.9 -> 36.7 |
    // 41.5 | 45.8 us, a stack's 22528 x 2048 at 32 rows 23.4 -> 21.1; other distances lose by it: 27648 x 5120 at 96 rows 78.8
    // -> 82.2, 16384 x 2048 (two images) at 64 19.6 -> 20.7, a stack's 25600 x 3072 at 128 42.5 -> 43.8. Where one row block's
    // weights are read once (a chunk of one position block): with more, their activations no longer fit the L2 side by side
    // (256 rows, gate/up 92.7 -> 94.7); up to two splits, more of them start apart already (down at 96 rows 34.8 -> 38.9); 128
    // weight rows and more (tiles of 64, two on a CU, 28672 x 4096 at 32 rows 52.4 -> 60.1). int8 rows are half as long and
    // their walk is not bound by memory: 39.2 -> 39.1.
    constexpr bool ROT = sizeof(WT) == 2 && !Cfg::GR && BM <= 128 && Geo::BN >= 128;
    const bool apart = in.K % (Geo::NB == 2 ? 4096 : 2048) == 0;
    const int rot = ROT && PB == 1 && nsp <= 2 && apart ? rb % ns : 0, wrap = ns - 1 - rot;  // stage t: (t + rot) % ns of the range
    const unsigned ring = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) char*)pg_smem;

    // this wave's DMA instructions d in [wave*DPW, (wave+1)*DPW): stage bytes [1024 d, 1024 (d + 1)). Lane i
    // lands at byte 16 i of it: image row i / cpr, physical chunk i % cpr (cpr = 16-B chunks per image row),
    // so it loads the row's logical chunk (i % cpr) ^ swizzle(row).
    // (src walks on with every issue; adv, back: int8 only, elsewhere both operands advance 128 bytes and every stage is whole)
    const char* src[Geo::DPW];
    [[maybe_unused]] int adv[HALF ? Geo::DPW : 1];   // bytes per stage
    [[maybe_unused]] int back[HALF ? Geo::DPW : 1];  // bytes to step back in a half last stage (logical chunk in the stage's second half)
    static_assert(HALF || Geo::A_ROW == Geo::B_ROW, "one advance");
#pragma unroll
    for (int j = 0; j < Geo::DPW; ++j) {
        // split rings: the wave's DPA pieces of the A images, then its DPB pieces of the B images
        const int off = Geo::SA ? (j < Geo::DPA ? (wave * Geo::DPA + j) * 1024
                                                : Geo::A_BYTES + (wave * Geo::DPB + j - Geo::DPA) * 1024)
                                : (wave * Geo::DPW + j) * 1024;
        if (off < Geo::A_BYTES) {
            const int t = rb * Geo::NA + off / Geo::A_IMG;
            const int r = (off % Geo::A_IMG) / Geo::A_ROW + lane / 8;
            const int c = (lane % 8) ^ pg_swz(r, Geo::A_ROW);
            const int row = epi.row(min(t, nt - 1), r);
            src[j] = reinterpret_cast<const char*>(in.W) + (size_t)row * in.K * sizeof(WT) + c * 16 + (size_t)(s0 + rot) * Geo::A_ROW;
            if constexpr (HALF) adv[j] = Geo::A_ROW, back[j] = c >= 4 ? Geo::A_ROW / 2 : 0;
        } else {
            constexpr int cpr = Geo::B_ROW / 16;
            const int o2 = off - Geo::A_BYTES;
            const int u = o2 / Geo::B_IMG, pt = Geo::NB == 2 ? u >> 1 : u;
            const int r = (o2 % Geo::B_IMG) / Geo::B_ROW + lane / cpr;
            const int c = (lane % cpr) ^ pg_swz(r, Geo::B_ROW);
            const __half* B = Geo::NB == 2 ? ((u & 1) ? in.Blo : in.Bhi) : rb * Geo::BN >= in.row_b2 ? in.Bhi2 : in.Bhi;
            int m = pb * BM + pt * 16 + r;
            if constexpr (Cfg::GR) m = in.grp.rowmap ? in.grp.rowmap[m] : tile.y + pt * 16 + r;
            src[j] = reinterpret_cast<const char*>(B) + (size_t)m * in.K * (Geo::F32 ? 4 : 2) + c * 16 + (size_t)(s0 + rot) * Geo::B_ROW;
            if constexpr (HALF) adv[j] = Geo::B_ROW, back[j] = c >= cpr / 2 ? Geo::B_ROW / 2 : 0;
        }
    }
    auto piece = [&](int j, unsigned dst, int t) PG_INLINE {  // of stage t
        if constexpr (HALF) {
            pf_dma(src[j] - (half_tail && t == ns - 1 ? back[j] : 0), dst);
            src[j] += adv[j];
        } else {
            pf_dma(src[j], dst);
            src[j] += ROT && t == wrap ? Geo::A_ROW - ns * Geo::A_ROW : Geo::A_ROW;
        }
    };
    // One ring: stage s in slot s % S. Split rings: A stage s in slot s % SA at ring, B stage s in slot s % 2 behind the A ring.
    const unsigned ring_b = ring + (unsigned)(Geo::SA * Geo::A_BYTES);
    // piece j of what iteration s issues: stage s + S - 1, or A stage s + SA - 1 (j < DPA) and B stage s + 1. Issue order:
    // B pieces first (j counts from them).
    constexpr int SAN = Geo::SA ? Geo::SA : 1;
    auto dma = [&](int j, int s) PG_INLINE {
        if constexpr (Geo::SA == 0) {
            const int t = s + S - 1;
            piece(j, ring + (unsigned)((t % S) * Geo::STAGE + (wave * Geo::DPW + j) * 1024), t);
        } else if (j < Geo::DPB) {
            const int t = s + 1;
            piece(Geo::DPA + j, ring_b + (unsigned)((t & 1) * Geo::B_BYTES + (wave * Geo::DPB + j) * 1024), t);
        } else {
            const int t = s + SAN - 1;
            piece(j - Geo::DPB, ring + (unsigned)((t % SAN) * Geo::A_BYTES + (wave * Geo::DPA + j - Geo::DPB) * 1024), t);
        }
    };
    constexpr int AT = Geo::AT;
    pf_float4 acc[AT][Geo::WPT];
#pragma unroll
    for (int a = 0; a < AT; ++a)
#pragma unroll
        for (int b = 0; b < Geo::WPT; ++b) acc[a][b] = pf_float4{0.0f, 0.0f, 0.0f, 0.0f};

    // fragment read offsets: lane l reads row / column r = l & 15, k group kg = l >> 4 of each 32-k block
    const int kg = lane >> 4, r16 = lane & 15;
    const int sa = pg_swz(r16, Geo::A_ROW), sb = pg_swz(r16, Geo::B_ROW);
    if constexpr (Geo::SA == 0) {
#pragma unroll
        for (int i = 1 - S; i < 0; ++i)
            if (i + S - 1 < ns) {
#pragma unroll
                for (int j = 0; j < Geo::DPW; ++j) dma(j, i);
            }
    } else {  // the schedule of iterations -(SA - 1) .. -1: B(i + 1), then A(i + SA - 1)
#pragma unroll
        for (int i = 1 - Geo::SA; i < 0; ++i) {
            if (i + 1 >= 0 && i + 1 < ns) {
#pragma unroll
                for (int j = 0; j < Geo::DPB; ++j) dma(j, i);
            }
            if (i + Geo::SA - 1 < ns) {
#pragma unroll
                for (int j = Geo::DPB; j < Geo::DPW; ++j) dma(j, i);
            }
        }
    }
    // Fragments of a k-block: AT of the weights, NB WPT of the activations
    struct Frags {
        u32x4 a[AT], b[Geo::WPT][Geo::NB];
    };
    // read r of k-block kb of stage buffer st (A images at st, B images at stb): the weights' first
    auto read_frag = [&](int r, const char* st, const char* stb, int kb, Frags& f) PG_INLINE {
        if (r < AT) {
            const char* img = st + (wr * AT + r) * Geo::A_IMG + r16 * Geo::A_ROW;
            if constexpr (sizeof(WT) != 1) {
                f.a[r] = *reinterpret_cast<const u32x4*>(img + ((4 * kb + kg) ^ sa) * 16);
            } else {
                const int off = ((2 * kb + (kg >> 1)) ^ sa) * 16 + 8 * (kg & 1);
                f.a[r] = pg_i8_to_f16(*reinterpret_cast<const uint2*>(img + off));
            }
        } else {
            const int u = r - AT, b = u / Geo::NB, t = u % Geo::NB;
            const int pt = wp * Geo::WPT + b;
            const char* img = stb + (Geo::NB * pt + t) * Geo::B_IMG + r16 * Geo::B_ROW + ((4 * kb + kg) ^ sb) * 16;
            f.b[b][t] = *reinterpret_cast<const u32x4*>(img);
        }
    };
    constexpr int NR = AT + Geo::NB * Geo::WPT;   // reads of a k-block
    constexpr int NSL = Geo::NB * Geo::WPT;       // slices of a k-block: AT MFMAs each
    auto slice_mfma = [&](int i, const Frags& f) PG_INLINE {
        const int b = i / Geo::NB, t = i % Geo::NB;
        if constexpr (Geo::F32) {
#pragma unroll
            for (int a = 0; a < AT; ++a) {
                pf_float4 p[4];
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    p[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(f.a[a][e]), __uint_as_float(f.b[b][t][e]),
                                                                pf_float4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                acc[a][b] += (p[0] + p[1]) + (p[2] + p[3]);
            }
        } else {
#pragma unroll
            for (int a = 0; a < AT; ++a) acc[a][b] = pf_mfma(f.a[a], f.b[b][t], acc[a][b]);
        }
    };
    // MFMAs of fragments f in slices of AT (one activation fragment each), between them the reads of the next k-block into n
    // and DMA pieces j0 .. j1 - 1 of iteration s: a wave issues them in the 12 cycles that an MFMA holds the matrix pipe
    // after its issue. The order is fixed (sched_barrier, every 4 MFMAs or, of slices of 3, every 3): left to itself the
    // compiler gathered a set's reads behind the MFMAs they should run beside, each wait for LDS then stood open, and the 16
    // DMA pieces stood in front. 128 x 192 tiles, 7B q/k/v | gate/up at 512 rows 92 | 188 -> 83 | 166 us; 128 x 256, gate/up
    // at 2048 rows 754 -> 670 (1260 TFLOP/s). The clock then falls from 2.0 to 1.66 GHz (MFMAs on random data alone hold 1.74
    // PFLOP/s): more waves, s_setprio and 128-row wave tiles measured the same.
    // PAIR: where a second workgroup runs on the CU and the ring has two stages, the order is the compiler's and the DMA goes
    // first: the other workgroup's MFMAs run beside the reads, and the next stage needs all of the time there is to land
    // (128 x 128 of a stack, 5120 x 18944 at 1536 rows: 315 -> 283 us).
    constexpr bool PAIR = Geo::SA == 0 && S == 2 && 2 * Geo::LDS <= 160 * 1024;
    auto phase = [&](const Frags& f, Frags& n, const char* st, const char* stb, auto KB, auto J0, auto J1, int s) PG_INLINE {
        constexpr int RS = NSL > 1 ? NSL - 1 : 1;  // slices with reads
        constexpr int kb = decltype(KB)::value, j0 = decltype(J0)::value, j1 = decltype(J1)::value;
        pg_for<NSL>([&](auto I) PG_INLINE {
            constexpr int i = decltype(I)::value;
            if constexpr (kb >= 0 && i < RS) {
                constexpr int r0 = NR * i / RS, r1 = NR * (i + 1) / RS;
                pg_for<r1 - r0>([&](auto R) PG_INLINE { read_frag(r0 + R, st, stb, kb, n); });
            }
            constexpr int d0 = j0 + (j1 - j0) * i / NSL, d1 = j0 + (j1 - j0) * (i + 1) / NSL;
            slice_mfma(i, f);
            pg_for<d1 - d0>([&](auto J) PG_INLINE { dma(d0 + J, s); });
            if constexpr (!PAIR && ((i + 1) % (AT < 4 ? 4 / AT : 1) == 0 || i == NSL - 1)) __builtin_amdgcn_sched_barrier(0);
        });
    };
    constexpr bool TWO = Geo::FOLD > 0;
    pf_float4 tot[TWO ? AT : 1][TWO ? Geo::WPT : 1] = {};
    auto fold = [&](auto& to, auto& from) PG_INLINE {
#pragma unroll
        for (int a = 0; a < AT; ++a)
#pragma unroll
            for (int b = 0; b < Geo::WPT; ++b) {
                to[a][b] += from[a][b];
                from[a][b] = pf_float4{0.0f, 0.0f, 0.0f, 0.0f};
            }
    };
    const bool live = Cfg::GR || pb * BM + wp * Geo::WPT * 16 < in.valid;  // (wave-uniform)
    // before iteration s: stage s landed, every wave is done with the buffers that iteration s issues into
    auto stage_begin = [&](int s) {
        if constexpr (Geo::SA == 0) {
            pg_wait_stages<Geo::DPW>(min(S - 2, ns - 1 - s));
        } else {
            // B(s) was the first load of iteration s - 1; only that iteration's A pieces (if it issued any) were
            // issued after it, and A(s) before it
            if (s + Geo::SA - 2 < ns)
                pf_wait_vm<Geo::DPA>();
            else
                pf_wait_vm<0>();
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
    };
    // pieces that iteration s issues
    auto pieces = [&](int s) {
        if constexpr (Geo::SA == 0)
            return s + S - 1 < ns ? Geo::DPW : 0;
        else
            return s + Geo::SA - 1 < ns ? Geo::DPW : s + 1 < ns ? Geo::DPB : 0;
    };
    auto bufs = [&](int s, const char*& st, const char*& stb) {
        if constexpr (Geo::SA == 0) {
            st = pg_smem + (size_t)(s % S) * Geo::STAGE;
            stb = st + Geo::A_BYTES;
        } else {
            st = pg_smem + (size_t)(s % Geo::SA) * Geo::A_BYTES;
            stb = pg_smem + (size_t)Geo::SA * Geo::A_BYTES + (size_t)(s & 1) * Geo::B_BYTES;
        }
    };
    static_assert(KBS % 2 == 0, "k-blocks per stage");
    if (!live) {
        for (int s = 0; s < ns; ++s) {
            stage_begin(s);
            const int np = pieces(s);
#pragma unroll
            for (int j = 0; j < Geo::DPW; ++j)
                if (j < np) dma(j, s);
        }
    } else {
        // Set X holds even k-blocks, set Y odd ones (an int8 half stage has KBS / 2 = 2): per stage MFMA(Y: the previous
        // stage's last k-block) beside read(0) -> X, MFMA(X) beside read(1) -> Y, ... The stage barrier follows this wave's
        // lgkmcnt(0), so the previous stage's buffer is free for the DMA issued after it while its last fragments wait in
        // registers.
        Frags X, Y;
        // Of an iteration's np pieces, those issued before phase i. What must land within the stage that issues it goes out
        // early: a split ring's activations in the first phase, all of a two-stage ring in the first half. Spread over the whole
        // stage the last of them were waited for at its end (96 x 128 tiles of fp16, 4096 x 11008 at 384 rows: 84.5 -> 79.4 us;
        // 256 x 256 of a stack, 34304 x 4096 at 2048 rows: 550 -> 530).
        constexpr auto due = [](int i, int np) constexpr {
            const int early = np < Geo::DPB ? np : Geo::DPB;
            if (PAIR || i == 0) return PAIR ? np : 0;
            if (Geo::SA) return early + i * (np - early) / KBS;
            return S > 2 ? i * np / KBS : 2 * i < KBS ? (2 * i * np + KBS - 1) / KBS : np;
        };
        // one iteration; P: pieces it issues
        auto iter = [&](int s, auto P, auto first) PG_INLINE {
            constexpr int NP = decltype(P)::value;
            constexpr bool FIRST = decltype(first)::value;
            const char *st, *stb;
            stage_begin(s);
            bufs(s, st, stb);
            constexpr std::integral_constant<int, due(0, NP)> q0;
            constexpr std::integral_constant<int, due(1, NP)> q1;
            constexpr std::integral_constant<int, due(2, NP)> q2;
            if constexpr (PAIR) pg_for<NP>([&](auto J) PG_INLINE { dma(J, s); });
            if constexpr (FIRST) {
                pg_for<NR>([&](auto R) PG_INLINE { read_frag(R, st, stb, 0, X); });
                pg_for<q1 - q0>([&](auto J) PG_INLINE { dma(q0 + J, s); });
                __builtin_amdgcn_sched_barrier(0);
            } else {
                phase(Y, X, st, stb, std::integral_constant<int, 0>{}, q0, q1, s);
            }
            phase(X, Y, st, stb, std::integral_constant<int, 1>{}, q1, q2, s);
            if constexpr (KBS == 4) {
                constexpr std::integral_constant<int, due(3, NP)> q3;
                if (NP > 0 || !(half_tail && s == ns - 1)) {
                    phase(Y, X, st, stb, std::integral_constant<int, 2>{}, q2, q3, s);
                    phase(X, Y, st, stb, std::integral_constant<int, 3>{}, q3, std::integral_constant<int, NP>{}, s);
                }
            }
            if constexpr (TWO)
                if (s % (Geo::FOLD / Geo::KS) == Geo::FOLD / Geo::KS - 1) fold(tot, acc);
        };
        constexpr std::integral_constant<int, Geo::DPW> full;
        constexpr std::integral_constant<int, Geo::SA ? Geo::DPB : 0> part;
        constexpr std::integral_constant<int, 0> none;
        constexpr int AHEAD = Geo::SA ? Geo::SA - 1 : S - 1;
        constexpr std::true_type yes;
        constexpr std::false_type no;
        int s = 0;
        if (AHEAD < ns) iter(s++, full, yes);
        else if (part.value && 1 < ns) iter(s++, part, yes);
        else iter(s++, none, yes);
        for (; s + AHEAD < ns; ++s) iter(s, full, no);
        if constexpr (part.value > 0)
            for (; s + 1 < ns; ++s) iter(s, part, no);
        for (; s < ns; ++s) iter(s, none, no);
        phase(Y, X, nullptr, nullptr, std::integral_constant<int, -1>{}, none, none, 0);
        if constexpr (TWO) fold(acc, tot);
    }
    const int i0 = 4 * (lane >> 4);  // C[i][n] of a 16x16 tile: lane l holds rows 4 (l >> 4) + r, column l & 15
    if constexpr (PgDefers<Epi>::value) {
        if (nsp > 1 && in.defer) {
            if (!live) return;
#pragma unroll
            for (int a = 0; a < AT; ++a) {
                const int t = rb * Geo::NA + wr * AT + a;
                if (t >= nt) continue;
#pragma unroll
                for (int b = 0; b < Geo::WPT; ++b) {
                    const int m = pb * BM + (wp * Geo::WPT + b) * 16 + r16;
                    *reinterpret_cast<pf_float4*>(in.ws + ((size_t)sp * in.M + m) * in.N + t * 16 + i0) = acc[a][b];
                }
            }
            return;
        }
    }
    if (nsp > 1) {
        // Partial sums go out write-through (sc1); the tile's last workgroup to arrive adds them in split order (the
        // same sum whichever arrives last) and runs the epilogue.
        constexpr int NV = AT * Geo::WPT, TILE = NV * Geo::THREADS;  // float4s per split
        const unsigned tail = (unsigned)(ti - in.full) * 8 + xcd, bytes = 16u * TILE;
        float* tw = in.ws + (size_t)tail * nsp * TILE * 4;
        const auto own = __builtin_amdgcn_make_buffer_rsrc(tw + (size_t)sp * TILE * 4, 0, bytes, 0x00020000);
#pragma unroll
        for (int a = 0; a < AT; ++a)
#pragma unroll
            for (int b = 0; b < Geo::WPT; ++b)
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[a][b]), own,
                                                       16u * ((a * Geo::WPT + b) * Geo::THREADS + threadIdx.x), 0, 16 /* sc1 */);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every storing wave drains before the arrival
        __syncthreads();
        unsigned* flag = reinterpret_cast<unsigned*>(pg_smem);
        if (threadIdx.x == 0) {
            const unsigned prev = __hip_atomic_fetch_add(in.cnt + tail, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *flag = prev == (unsigned)(nsp - 1);
            if (*flag) __hip_atomic_store(in.cnt + tail, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        if (*flag == 0) return;  // uniform
#pragma unroll
        for (int a = 0; a < AT; ++a)
#pragma unroll
            for (int b = 0; b < Geo::WPT; ++b) acc[a][b] = pf_float4{0.0f, 0.0f, 0.0f, 0.0f};
        // A split's partials come from memory: several splits' loads are in flight together (16 float4 of a thread), or the
        // merge takes a round trip each. 45 tokens of an int8 7B prompt 1.013 -> 1.023 times as fast as one by one.
        if constexpr (NV <= 16) {
            constexpr int QB = 16 / NV;
            const auto rs = __builtin_amdgcn_make_buffer_rsrc(tw, 0, bytes * nsp, 0x00020000);
            for (int q0 = 0; q0 < nsp; q0 += QB) {
                u32x4 p[QB][NV];
#pragma unroll
                for (int i = 0; i < QB; ++i)
#pragma unroll
                    for (int j = 0; j < NV; ++j)
                        p[i][j] = __builtin_amdgcn_raw_buffer_load_b128(rs, 16u * threadIdx.x + 16u * Geo::THREADS * j,
                                                                        bytes * min(q0 + i, nsp - 1), 16);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < QB; ++i)
                    if (q0 + i < nsp) {
#pragma unroll
                        for (int j = 0; j < NV; ++j) acc[j / Geo::WPT][j % Geo::WPT] += __builtin_bit_cast(pf_float4, p[i][j]);
                    }
            }
        } else {
            for (int q = 0; q < nsp; ++q) {
                const auto rs = __builtin_amdgcn_make_buffer_rsrc(tw + (size_t)q * TILE * 4, 0, bytes, 0x00020000);
#pragma unroll
                for (int a = 0; a < AT; ++a) {
#pragma unroll
                    for (int b = 0; b < Geo::WPT; ++b)
                        acc[a][b] += __builtin_bit_cast(
                            pf_float4, __builtin_amdgcn_raw_buffer_load_b128(
                                           rs, 16u * ((a * Geo::WPT + b) * Geo::THREADS + threadIdx.x), 0, 16));
                    asm volatile("" ::: "memory");  // (one tile row's loads in flight: more would spill at 256 columns)
                }
            }
        }
    }
    if constexpr (PgRolled<Epi>::value) {
        // A loop over the weight tiles, their sums indexed in the ring's LDS (indexed registers would live in scratch), unrolled
        // over the chunk rows: one tile at a time, each with its own look at its row, waited for memory and LDS in turn, 0.7 us
        // a tile.
        constexpr int W = AT * Geo::WPT * 16 * Geo::THREADS <= Geo::LDS ? Geo::WPT : Geo::WPT / 2;  // chunk row tiles at a time
        static_assert(AT * W * 16 * Geo::THREADS <= Geo::LDS && Geo::WPT % W == 0, "sums in the ring");
        const int t0 = rb * Geo::NA + wr * AT, m0 = pb * BM + wp * Geo::WPT * 16 + r16;
        decltype(epi.row_of(0)) rr[Geo::WPT];
#pragma unroll
        for (int b = 0; b < Geo::WPT; ++b) rr[b] = epi.row_of(m0 + 16 * b);
        __syncthreads();  // every wave is done with its fragments
        if (!live) return;
        if (t0 + AT <= nt && epi.flat(t0, AT)) {
#pragma unroll
            for (int b = 0; b < Geo::WPT; ++b) {
                pf_float4 v[AT];
#pragma unroll
                for (int a = 0; a < AT; ++a) v[a] = acc[a][b];
                epi.template flat_store<AT>(t0, kg, m0 + 16 * b, v, rr[b]);
            }
            return;
        }
        pf_float4* mine = reinterpret_cast<pf_float4*>(pg_smem) + threadIdx.x;  // (each thread reads what it wrote)
        pg_for<Geo::WPT / W>([&](auto B0) PG_INLINE {
            constexpr int b0 = decltype(B0)::value * W;
#pragma unroll
            for (int j = 0; j < AT * W; ++j) mine[j * Geo::THREADS] = acc[j / W][b0 + j % W];
#pragma unroll 1
            for (int a = 0; a < AT; ++a) {
                if (t0 + a >= nt) break;
                pg_for<W>([&](auto B) PG_INLINE {
                    constexpr int b = decltype(B)::value;
                    const pf_float4 o = mine[(a * W + b) * Geo::THREADS];
                    const float v[4] = {o[0], o[1], o[2], o[3]};
                    epi.store(t0 + a, i0, m0 + 16 * (b0 + b), v, rr[b0 + b]);
                });
            }
        });
    } else {
        if (!live) return;
#pragma unroll
        for (int a = 0; a < AT; ++a) {
            const int t = rb * Geo::NA + wr * AT + a;
            if (t >= nt) continue;
#pragma unroll
            for (int b = 0; b < Geo::WPT; ++b) {
                const int m = pb * BM + (wp * Geo::WPT + b) * 16 + r16;
                const float v[4] = {acc[a][b][0], acc[a][b][1], acc[a][b][2], acc[a][b][3]};
                epi.store(t, i0, m, v, ps);
            }
        }
    }
}

// ---- epilogues. Tiles hold 4-row groups {first(u), first(u + 1), second(u), second(u + 1)} where a pair is a
// RoPE pair {d, d + hd/2} (q/k/v) or {gate u, up u}, so each lane's 4 rows are 2 complete pairs.
template <typename KT>
struct PgEpiQKV {  // model.cpp:52-67: q (fp32 [M][hq*hd]), rotated k / v rows of the cache at p0 + m
    float* q;
    KT* kc;  // this layer's cache base [sequence][hkv][T][hd]
    KT* vc;
    const float* rscale;  // int8 row scales (nullable)
    const float* sin_t;
    const float* cos_t;
    int hq, hkv, hd, T;
    __device__ int row(int t, int i) const {
        const int half = hd >> 1;
        const int u = t * 8 + (i >> 2) * 2 + (i & 1);
        const int uh = u / half, d = u - uh * half;
        return uh * hd + d + ((i & 2) ? half : 0);
    }
    __device__ void store(int t, int i0, int m, const float* v, const PfState& ps) const {
        // units u, u + 1 (u even): d, d + 1 of one head (hd / 2 is even), so every store is a pair
        const int b = ps.nseq == 1 ? 0 : m / ps.rps, i = m - b * ps.rps, pos = ps.p0 + i;
        const bool keep = i < ps.nv && b < ps.nseq && pos < T;
        const int half = hd >> 1;
        const int u = t * 8 + (i0 >> 2) * 2;
        const int uh = u / half, d = u - uh * half;
        float a0[2] = {v[0], v[1]}, a1[2] = {v[2], v[3]};  // first / second element of the pairs of u, u + 1
        if (rscale) {
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                a0[e] *= rscale[uh * hd + d + e];
                a1[e] *= rscale[uh * hd + d + e + half];
            }
        }
        if (uh < hq + hkv) {  // rope_kernel.cpp:30-38
            const int pp = min(pos, T - 1);
            float r0[2], r1[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const float fci = sin_t[pp * half + d + e], fcr = cos_t[pp * half + d + e];
                r0[e] = a0[e] * fcr - a1[e] * fci;
                r1[e] = a1[e] * fcr + a0[e] * fci;
            }
            if (uh < hq) {
                float* qr = q + (size_t)m * hq * hd + (size_t)uh * hd;
                *reinterpret_cast<float2*>(qr + d) = make_float2(r0[0], r0[1]);
                *reinterpret_cast<float2*>(qr + d + half) = make_float2(r1[0], r1[1]);
            } else if (keep) {
                KT* kr = kc + (((size_t)b * hkv + uh - hq) * T + pos) * hd;
                store2(kr + d, r0);
                store2(kr + d + half, r1);
            }
        } else if (keep) {
            KT* vr = vc + (((size_t)b * hkv + uh - hq - hkv) * T + pos) * hd;
            store2(vr + d, a0);
            store2(vr + d + half, a1);
        }
    }
    __device__ static void store2(KT* p, const float* f) {
        if constexpr (sizeof(KT) == 2) {
            __half h[2] = {__float2half_rn(f[0]), __float2half_rn(f[1])};
            *reinterpret_cast<unsigned*>(p) = *reinterpret_cast<const unsigned*>(h);
        } else {
            *reinterpret_cast<float2*>(p) = make_float2(f[0], f[1]);
        }
    }
};

struct PgEpiSwiGLU {  // model.cpp:99-115: act = sigmoid(g) * u (or SiLU), stored as the down GEMM's input
    PfOut out;
    const float* rscale;
    int inter, silu;
    __device__ int row(int t, int i) const { return t * 8 + (i >> 2) * 2 + (i & 1) + ((i & 2) ? inter : 0); }
    __device__ void store(int t, int i0, int m, const float* v, const PfState&) const {
        const int u = t * 8 + (i0 >> 2) * 2;  // units u, u + 1: stored together
        float y[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            float g = v[e], up = v[2 + e];
            if (rscale) {
                g *= rscale[u + e];
                up *= rscale[inter + u + e];
            }
            float sg = 1.0f / (1.0f + expf(-g));  // swiglu_kernel.cpp:12
            if (silu) sg = g * sg;
            y[e] = sg * up;  // :13
        }
        out.store<2>((size_t)m * inter + u, y);
    }
};

struct PgEpiResid {  // y[m][row] = resid[m][row] + sum * row scale (matmul_kernel.cpp:26 + add_kernel.cpp:5-14)
    float* y;        // [M][ld]: the residual stream (in place), or this rank's partial under TP
    const float* resid;  // the residual stream (tensor-parallel ranks > 0: null, their partial has none)
    const float* rscale;
    int nrows, ld;
    static constexpr bool kDefer = true;
    __device__ int row(int t, int i) const { return min(t * 16 + i, nrows - 1); }
    __device__ void store(int t, int i0, int m, const float* v, const PfState&) const {
        const int row = t * 16 + i0;  // rows row .. row + 3 (nrows % 16 == 0: the host's check)
        const size_t i = (size_t)m * ld + row;
        float4 p = make_float4(v[0], v[1], v[2], v[3]);
        if (rscale) {
            const float4 sc = *reinterpret_cast<const float4*>(rscale + row);
            p = make_float4(p.x * sc.x, p.y * sc.y, p.z * sc.z, p.w * sc.w);
        }
        if (resid) {
            const float4 r = *reinterpret_cast<const float4*>(resid + i);
            p = make_float4(r.x + p.x, r.y + p.y, r.z + p.z, r.w + p.w);
        }
        *reinterpret_cast<float4*>(y + i) = p;
    }
};

// How a GEMM's tiles fill the chip: whole rounds of one tile per resident workgroup, and the tiles of the last, partial
// round cut into `splits` depth ranges each, so that it is short and all CUs share it.
struct PgPlan {
    int full = 0x7fffffff, splits = 1;  // PgIn
    int slots = 0;                      // per XCD
    float us = 0.0f;
};
constexpr size_t kPgWsBytes = 64u << 20;  // partial sums of a launch at most
constexpr int kPgWsTiles = 4096;          // tiles cut at most (counters)
// stage: us of a stage of the tiling (pg_tilings). Around its walk of the depth a workgroup takes 2 us and 6 for 128 KiB of sums
// (a 128 x 256 tile): dispatch, the ring's first stages, the epilogue; a cut round 2 us, 0.6 for each split and 1.5 for each
// split's and two more 128 KiB: the partial sums' way out and back. These and the stage times are fitted together, so that the
// plan that costs least is the fastest one, and are no times of their own (a large product's stages last longer: the clock
// falls). Over 600 sizes of fp16 (1024 to 28672 outputs, 9 to 4096 rows) the plan taken lasts 1.1 % longer than the fastest, of
// int8 0.4, of fp32 0.8, of block stacks 2 % (tools/pgemm_lab prints both).
// rolled: a looped epilogue (kRolled) is priced by the tiles a wave loops over: 0.7 us each, shared by the workgroups of a CU. That was
// fitted to a stack's 25600 x 3072 at 384 rows, 100.6 us in 128 x 256 tiles (16 a wave) and 95.9 in 128 x 128 (8); a plain epilogue 84
// and 90. It takes about half of that by now, and the price stays all the same: it sets where the depth is cut, so the order of a prompt's
// sums. (0.35, and rows to spare as the output GEMM has, pick other tiles or cuts at 10 of 36 row counts of a 2048-wide stack's two inputs and would
// take 4.43 ms for 4.61 at 1280 rows, 4.03 for 4.09 at 1025.)
template <class Cfg, typename WT>
PgPlan pg_plan(int N, int K, int M, int cus, bool ws, float stage, bool rolled = false) {
    using Geo = PgGeo<Cfg, WT>;
    const int nrb = (N + Geo::BN - 1) / Geo::BN, nx = (nrb + 7) / 8 * (M / Geo::BM);
    const int ns = (K + Geo::KS - 1) / Geo::KS;
    const int occ = (int)((160 * 1024) / Geo::LDS), cpx = std::max(1, cus / 8) * occ;
    constexpr float kTile = 16.0f * Geo::AT * Geo::WPT * Geo::THREADS / 131072.0f, kEdge = 2.0f + 6.0f * kTile;
    const float epi = rolled ? 0.7f * Geo::AT * Geo::WPT / (float)occ : 0.0f;
    PgPlan best;
    best.slots = nx;
    best.us = (float)((nx + cpx - 1) / cpx) * ((float)ns * stage + kEdge + epi);
    const int full = nx / cpx * cpx, tail = nx - full;
    for (int S : {2, 3, 4, 5, 6, 8, 10, 12, 16}) {
        if (!ws || tail == 0 || ns < 4 * S || 8 * tail > kPgWsTiles ||
            (size_t)8 * tail * S * 16 * Geo::AT * Geo::WPT * Geo::THREADS > kPgWsBytes)
            break;
        const float us = (float)(full / cpx) * ((float)ns * stage + kEdge + epi) +
                         (float)((tail * S + cpx - 1) / cpx) * ((float)(ns + S - 1) / (float)S * stage + kEdge) + 2.0f +
                         0.6f * (float)S + 1.5f * kTile * (float)(S + 2) + epi;
        if (us < best.us) best = PgPlan{full, S, full + tail * S, us};
    }
    return best;
}

template <class Epi, class Cfg, typename WT>
hipError_t launch_pgemm(const PgIn<WT>& in, const Epi& epi, const PfState& ps, hipStream_t s) {
    using Geo = PgGeo<Cfg, WT>;
    if (in.M % Geo::BM != 0) return hipErrorInvalidValue;  // rows past the last whole tile would be skipped
    const int nx = ((in.N + Geo::BN - 1) / Geo::BN + 7) / 8 * (in.M / Geo::BM);
    if (in.full < nx && (!in.ws || !in.cnt || in.splits < 2)) return hipErrorInvalidValue;
    const int slots = in.full < nx ? in.full + (nx - in.full) * in.splits : nx;
    hipLaunchKernelGGL((pgemm_kernel<Epi, Cfg, WT>), dim3(8 * slots), dim3(Geo::THREADS), Geo::LDS, s, in, epi, ps);
    return hipGetLastError();
}

template <class Epi, class Cfg, typename WT>
hipError_t pgemm_allow_lds() {
    return hipFuncSetAttribute(reinterpret_cast<const void*>(&pgemm_kernel<Epi, Cfg, WT>),
                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)PgGeo<Cfg, WT>::LDS);
}

// Where a prompt's GEMM may sum in one chain over its depth or split (PgGeo::FOLD 0: the 128 x 256 tiling, 4 % faster than with
// short chains): what long prompts spend their time on, gate/up from 769 rows and depths of 8192 and more from 1537. Llama-2-7B,
// relative error of the logits against float64, so | wherever it is the fastest: 512 tokens 4.4e-5 | 4.9e-5, 700 4.1e-5 |
// 5.8e-5, 1025 4.0e-5 | 4.8e-5, 2000 4.5e-5 | 4.5e-5.
inline bool pg_one_chain(int N, int K, int rows) { return (N >= 16384 && rows > 768) || (K >= 8192 && rows > 1536); }

// The tilings of the Llama prompts, f(PgCfg<...>{}, us): us is a stage of the tiling as pg_plan counts it. A launch takes the
// tiling whose plan costs least (rounds over the rows padded to its BM, the last round's tiles cut over the depth).
// Llama-2-7B, q/k/v | gate/up | wo | down, us, what the plan takes against the best tiling in whole tiles
// (profiles/pgemm_tilings.txt): 512 rows 86 | 187 | 38 | 88 against 86 | 183 | 40 | 110; 64 rows 28 | 42 | 13 | 28 against 39 |
// 46 | 19 | 56; int8 64 rows 24 | 36 | 15 | 24 against 32 | 41 | 26 | 65; fp32 96 rows 157 | 248 | 56 | 137 against 194 | 335 |
// 98 | 260. In the engine (profiles/prompt_7b_f16_512_kernel_stats.csv) 512 rows take 97 | 184 | 44 | 95.
// The int8 tilings with a weight ring of their own (SA 3) have two stages of the weights in flight instead of one (a wave waits
// for its loads in order, so for all weights issued before the activations it needs: a deeper ring holds stages that have
// landed); 64 rows: gate/up 39.1 -> 36.2, q/k/v 24.8 -> 24.4, down 25.2 -> 23.7; 192 rows: q/k/v of 96 x 128 tiles 54.8 ->
// 50.6; 32 rows: q/k/v 17.8 us with 3 slots, 19.5 with 5, gate/up 25.3 and 26.4. 256 x 32 in one ring stays for very wide
// outputs: 28672 x 4096 at 9 rows 27.6, the next 30.4.
template <typename WT, class F>
void pg_tilings(F&& f) {
    if constexpr (std::is_same<WT, float>::value) {
        f(PgCfg<128, 4, 4, 2, 0, 1>{}, 2.29f), f(PgCfg<96, 2, 4, 2, 0, 1>{}, 2.22f), f(PgCfg<64, 4, 4, 2, 0, 1>{}, 1.22f);
        f(PgCfg<32, 2, 6, 2, 0, 1>{}, 1.08f), f(PgCfg<32, 2, 4, 4, 0, 1>{}, 1.53f);
    } else if constexpr (std::is_same<WT, int8_t>::value) {
        f(PgCfg<128, 4, 2, 2>{}, 1.57f), f(PgCfg<96, 4, 2, 3>{}, 1.64f), f(PgCfg<96, 4, 2, 2, 3>{}, 1.18f);
        f(PgCfg<64, 4, 2, 3, 3>{}, 1.32f), f(PgCfg<64, 4, 2, 2, 3>{}, 1.01f);
        f(PgCfg<32, 4, 3, 4>{}, 1.33f), f(PgCfg<32, 4, 4, 2>{}, 0.99f), f(PgCfg<32, 4, 2, 3, 3>{}, 1.02f), f(PgCfg<32, 2, 4, 2>{}, 1.03f);
    } else {
        f(PgCfg<128, 4, 2, 4, 3>{}, 0.95f), f(PgCfg<128, 4, 2, 4, 3, 2, false, true>{}, 0.98f);
        f(PgCfg<128, 4, 2, 3, 4>{}, 0.88f), f(PgCfg<128, 4, 2, 2, 4>{}, 0.67f);
        f(PgCfg<96, 4, 2, 3, 4>{}, 0.76f), f(PgCfg<96, 4, 2, 2, 4>{}, 0.64f);
        f(PgCfg<64, 4, 3, 3>{}, 0.58f), f(PgCfg<64, 4, 3, 2>{}, 0.5f);
        f(PgCfg<32, 4, 4, 3>{}, 0.44f), f(PgCfg<32, 2, 4, 2>{}, 0.42f);
    }
}

// The tilings of block-stack prompts (one fp16 image; their row count divides M). 34304 x 4096 and 4096 x 15104,
// us, as above: 1024 rows 321 | 138 against 352 | 147; 256 rows 108 | 53 against 120 | 73; 64 rows 64 | 34 against 75 | 74.
// Two workgroups of 128 x 128 on a CU are the fastest where tiles twice as wide leave half a round empty: 3072 x 11264 at 768
// rows 75, the others 86 and more; 11264 x 1024 at 1408 rows 40, the others 46. The 32-row tiles read weights and little else,
// whatever a stage takes alone: theirs are the values that pick the faster one at 32 rows. With a looped epilogue (rolled) pairs
// of 128 x 128 gain less: 22528 x 2048 at 768 rows 117 us where 128 x 256 takes 106.
template <class F>
void pg_row_tilings(int M, bool rolled, F&& f) {
    if (M % 256 == 0) f(PgCfg<256, 4, 2, 4, 0, 1>{}, 1.3f);
    if (M % 128 == 0) f(PgCfg<128, 4, 3, 4, 0, 1>{}, 0.76f), f(PgCfg<128, 2, 3, 4, 0, 1>{}, 0.52f);
    if (M % 128 == 0) f(PgCfg<128, 4, 2, 2, 0, 1>{}, rolled ? 1.3f : 1.05f);
    if (M % 64 == 0) f(PgCfg<64, 2, 4, 2, 0, 1>{}, 0.46f);
    if (M < 64) f(PgCfg<32, 2, 4, 2, 0, 1>{}, 0.42f);
    if (M % 64 != 0) f(PgCfg<32, 2, 4, 4, 0, 1>{}, 0.4f);
}

// ---------------------------------------------------------------- 3. block-causal attention
// grid (rows / 64, hq); 4 waves x 16 queries; lane l: query l & 15 of the wave, dims [c * HD/4, (c+1) * HD/4) with
// c = l >> 4. Scores: the 4 lanes of a query add their quarter dot products (xor 16 / 32 exchanges); every lane
// of a query keeps the same online-softmax state (m, l) and its quarter of o. Output attn / l as hi / lo.
constexpr int kPaQB = 64;  // queries per workgroup
constexpr int kPaKT = 64;  // keys per LDS tile

template <typename KT>
struct PfAttnArgs {
    const float* q;    // [M][hq*hd]
    const KT* kc;      // layer base [sequence][hkv][T][hd]
    const KT* vc;
    PfOut out;         // [M][hq*hd]
    int hq, hkv, T;
    float scale;       // 1/sqrt(hd) (mha_kernel.cpp:41)
};

template <typename KT, int HD>
__global__ void __launch_bounds__(256) pf_attn_kernel(PfAttnArgs<KT> a, PfState ps) {
    constexpr int QD = HD / 4;  // dims per lane
    __shared__ __attribute__((aligned(16))) KT ks[kPaKT][HD];
    __shared__ __attribute__((aligned(16))) KT vs[kPaKT][HD];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int h = blockIdx.y, G = a.hq / a.hkv, kvh = h / G;
    const int seq = blockIdx.x * kPaQB / ps.rps, row0 = seq * ps.rps, p0 = ps.p0 - row0;
    if (seq >= ps.nseq) return;                                   // (uniform)
    const int mi = blockIdx.x * kPaQB + wave * 16 + (lane & 15);  // this lane's query (chunk row)
    const int c = lane >> 4;
    const int pos = p0 + mi;                                      // its position
    const int end = min((int)blockIdx.x * kPaQB + kPaQB, row0 + ps.nv);
    if (end <= (int)blockIdx.x * kPaQB) return;                   // (uniform) only padding rows
    // The block's last valid position. Rows past it are loaded as this one: their p is 0, but what the cache still holds
    // there may be no number.
    const int last = min(p0 + end - 1, a.T - 1);
    const int nt = last / kPaKT + 1;                              // key tiles
    float qv[QD], o[QD];
#pragma unroll
    for (int e = 0; e < QD; ++e) {
        qv[e] = a.q[(size_t)mi * a.hq * HD + (size_t)h * HD + c * QD + e];
        o[e] = 0.0f;
    }
    float mx = -INFINITY, l = 0.0f;
    const KT* kb = a.kc + ((size_t)seq * a.hkv + kvh) * a.T * HD;
    const KT* vb = a.vc + ((size_t)seq * a.hkv + kvh) * a.T * HD;
    constexpr int V16 = 16 / (int)sizeof(KT);  // elements per 16-byte vector
    for (int tt = 0; tt < nt; ++tt) {
        const int t0 = tt * kPaKT;
        __syncthreads();
        for (int i = threadIdx.x; i < kPaKT * HD / V16; i += 256) {  // the tile's K and V rows
            const int r = i / (HD / V16), cc = i - r * (HD / V16);
            const int t = min(t0 + r, last);
            reinterpret_cast<u32x4*>(&ks[r][0])[cc] = reinterpret_cast<const u32x4*>(kb + (size_t)t * HD)[cc];
            reinterpret_cast<u32x4*>(&vs[r][0])[cc] = reinterpret_cast<const u32x4*>(vb + (size_t)t * HD)[cc];
        }
        __syncthreads();
        float s[kPaKT];
        float tmax = -INFINITY;
#pragma unroll
        for (int j = 0; j < kPaKT; ++j) {
            float d = 0.0f;
#pragma unroll
            for (int e = 0; e < QD; ++e) d = fmaf(qv[e], to_f32(ks[j][c * QD + e]), d);
            d = sum_xor16(d);
            d = sum_xor32(d);
            s[j] = (t0 + j <= pos) ? d * a.scale : -INFINITY;  // mha_kernel.cpp:51-60 (sum * scale), causal
            tmax = fmaxf(tmax, s[j]);
        }
        const float mn = fmaxf(mx, tmax);
        const float corr = mn == -INFINITY ? 1.0f : expf(mx - mn);
        l *= corr;
#pragma unroll
        for (int e = 0; e < QD; ++e) o[e] *= corr;
        mx = mn;
#pragma unroll
        for (int j = 0; j < kPaKT; ++j) {
            const float p = (t0 + j <= pos) ? expf(s[j] - mx) : 0.0f;
            l += p;
#pragma unroll
            for (int e = 0; e < QD; ++e) o[e] = fmaf(p, to_f32(vs[j][c * QD + e]), o[e]);
        }
    }
#pragma unroll
    for (int e = 0; e < QD; e += 4) {
        const float y[4] = {o[e] / l, o[e + 1] / l, o[e + 2] / l, o[e + 3] / l};
        a.out.template store<4>((size_t)mi * a.hq * HD + (size_t)h * HD + c * QD + e, y);
    }
}

// ---- 3b. block stacks' packed portions by 16 rows (PfRowsArgs): passes of few rows (pf_rows_by_16), and windowed attention over
// expanded keys of the latent attention, on MFMA. A workgroup = 16 rows (queries) of one head; its 4 waves split the key range
// into 32-key tiles (wave w takes tiles w, w + 4, ...) and merge their (max, sum, o) through LDS at the end; per tile as
// pf_flash_kernel, with K and V in the wave's own images.
template <int HD>
struct PaGeo {
    static constexpr int ROWB = HD * 2;          // bytes per image row
    static constexpr int IMG = 32 * ROWB;        // one 32-key image
    static constexpr int WAVE = 2 * IMG;         // K + V
    static constexpr int PIECES = WAVE / 1024;   // DMA instructions per tile
    static constexpr int CPR = ROWB / 16;        // 16-B chunks per row
};
__device__ __forceinline__ int pa_swz_k(int r, int rowb) { return rowb == 256 ? r & 15 : (r >> 1) & 7; }
__device__ __forceinline__ int pa_swz_v(int r, int rowb) { return rowb == 256 ? (r & 7) << 1 : ((r >> 1) & 3) << 1; }

__device__ __forceinline__ uint2 pa_tr_read(unsigned lds_addr) {
    uint2 v;
    asm volatile("ds_read_b64_tr_b16 %0, %1" : "=v"(v) : "v"(lds_addr) : "memory");
    return v;
}

// the transposed reads landed: their registers are named in the wait, so the MFMAs that use them stay below it (as in
// attn_mfma.h; an asm load's outputs count as written at its end)
__device__ __forceinline__ void pa_tr_wait(uint2 (&x1)[8], uint2 (&x2)[8]) {
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(x1[0]), "+v"(x1[1]), "+v"(x1[2]), "+v"(x1[3]), "+v"(x1[4]), "+v"(x1[5]), "+v"(x1[6]),
                   "+v"(x1[7]), "+v"(x2[0]), "+v"(x2[1]), "+v"(x2[2]), "+v"(x2[3]), "+v"(x2[4]), "+v"(x2[5]),
                   "+v"(x2[6]), "+v"(x2[7])
                 :
                 : "memory");
}
__device__ __forceinline__ void pa_tr_wait(uint2 (&x1)[4], uint2 (&x2)[4]) {
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(x1[0]), "+v"(x1[1]), "+v"(x1[2]), "+v"(x1[3]), "+v"(x2[0]), "+v"(x2[1]), "+v"(x2[2]),
                   "+v"(x2[3])
                 :
                 : "memory");
}

// ---- 3a. the same over an fp16 cache, on MFMA. A workgroup = 4 waves over one kv head: GW of its query heads x 4 / GW
// blocks of 16 QT query positions, a wave each (GQA: 4 heads read one tile; MHA: 4 position blocks do). K and V tiles of
// 64 keys reach LDS by DMA, double-buffered, one barrier per tile: every key row is fetched once per 64 QT query rows.
// Per tile a wave computes
//   - Sᵀ = K Qᵀ: C[key][query] on v_mfma_f32_16x16x32_f16, A = K rows (exact fp16), B = Qᵀ as TERMS fp16 images;
//   - online softmax in base 2 (p = 2^(s c - m), one fma and one v_exp per score, its rounding that of the exponent);
//     the row maximum over the 4 lane groups of a query, the row sum only at the end. p carries a factor 2^8, which
//     divides out with the row sum: the lo halves of p >= 2^-21 stay normal fp16 numbers;
//   - Oᵀ += Vᵀ Pᵀ: B = Pᵀ straight from the Sᵀ accumulators (lane l holds query l & 15, keys {4g .. 4g+3, 16+4g ..
//     16+4g+3}, g = l >> 4 — the k order of the B operand), P as TERMS images; A = Vᵀ by ds_read_b64_tr_b16, whose 4-row
//     blocks are exactly those keys.
// The latest (longest) position blocks are dispatched first. mha_kernel.cpp:36-77 per query. Bound by the matrix cores and
// the softmax between them: Llama-3-8B, 3776 rows, 299 us a layer (785 TFLOP/s with hi + lo), where a workgroup per 16 rows
// and head, each key tile waited for as it was issued, took 651; Llama-2-7B, 511 rows, 18.7 us against 28.
template <int HD>
struct PfFlash {
    static constexpr int KT = 64, ROWB = HD * 2, IMG = KT * ROWB, CPR = ROWB / 16, PIECES = IMG / 1024;
};
// ROWS: the rows are packed portions of several sequences (step_state.h SegRef; the caches hold one [hkv][T][HD] block per
// sequence slot), with a distance bias and a sink per head (attn_rows.h) and one fp16 output [M][ldo] of vdim dims per head.
// 1025 rows of 32 heads of 128: 85 us as a workgroup per 16 rows and head, 51 here.
struct PfPortions {
    const SegRef* segs = nullptr;
    const int32_t* nsegs = nullptr;
    const float *r1 = nullptr, *r2 = nullptr, *sink = nullptr;  // [hq]
    int ldo = 0, vdim = 0;
};
template <int HD, int QT, int TERMS, bool ROWS = false>
__global__ void __launch_bounds__(256, 2) pf_flash_kernel(PfAttnArgs<__half> a, PfState ps, int GW, PfPortions x) {
    using F = PfFlash<HD>;
    constexpr int ND = HD / 32, NT = HD / 16, NK = F::KT / 16, PPW = 2 * F::PIECES / 4;
    __shared__ __attribute__((aligned(1024))) char sm[2 * 2 * F::IMG];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int g = lane >> 4, i16 = lane & 15;
    const int G = a.hq / a.hkv, ng = G / GW, kvh = blockIdx.y / ng;
    const int h = kvh * G + (blockIdx.y - kvh * ng) * GW + wave % GW;
    const int RB = (4 / GW) * 16 * QT;  // query positions per workgroup
    const int bx = gridDim.x - 1 - blockIdx.x;
    int blk, seq, row0;
    if constexpr (ROWS) {  // block bx of the portions' blocks
        int i = 0;
        const int n = *x.nsegs;
        for (blk = bx; i < n; ++i) {
            const int nb = (x.segs[i].n + RB - 1) / RB;
            if (blk < nb) break;
            blk -= nb;
        }
        if (i >= n) return;  // (uniform)
        const SegRef sg = x.segs[i];
        seq = sg.slot, row0 = sg.row0, ps.p0 = sg.pos0, ps.nv = ps.rps = sg.n;
    } else {
        blk = bx / ps.nseq, seq = bx - blk * ps.nseq, row0 = seq * ps.rps;
    }
    if (blk * RB >= ps.nv) return;  // (uniform) only padding rows
    const int i0 = blk * RB + (wave / GW) * 16 * QT;
    const int last = min(ps.p0 + min(blk * RB + RB, ps.nv) - 1, a.T - 1);                   // the workgroup's
    const int wlast = i0 < ps.nv ? min(ps.p0 + min(i0 + 16 * QT, ps.nv) - 1, a.T - 1) : -1;  // the wave's
    const size_t qs = (size_t)a.hq * HD;
    u32x4 qf[TERMS][QT][ND];
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        const int row = row0 + min(i0 + t * 16 + i16, ps.rps - 1);
#pragma unroll
        for (int db = 0; db < ND; ++db) {
            const float4* qp = reinterpret_cast<const float4*>(a.q + (size_t)row * qs + (size_t)h * HD + db * 32 + g * 8);
            const float4 v0 = qp[0], v1 = qp[1];
            const float f[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
            __half ht[TERMS][8];
#pragma unroll
            for (int e = 0; e < 8; ++e) pf_terms(f[e], ht, e);
#pragma unroll
            for (int i = 0; i < TERMS; ++i) qf[i][t][db] = *reinterpret_cast<const u32x4*>(ht[i]);
        }
    }
    pf_float4 o[QT][NT];
    float mx[QT], l[QT];
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        mx[t] = -INFINITY, l[t] = 0.0f;
#pragma unroll
        for (int d = 0; d < NT; ++d) o[t][d] = pf_float4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    const unsigned base = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) char*)sm;
    const size_t head = ((size_t)seq * a.hkv + kvh) * a.T * HD;
    // this wave's DMA pieces of a tile: piece p < PIECES of K, then of V; lane i of a piece: row (piece rows) + i / CPR,
    // physical chunk i % CPR <- logical chunk (i % CPR) ^ swizzle(row)
    auto issue = [&](int tt) {
#pragma unroll
        for (int j = 0; j < PPW; ++j) {
            const int p = wave * PPW + j;
            const bool isv = p >= F::PIECES;
            const int r = (isv ? p - F::PIECES : p) * (1024 / F::ROWB) + lane / F::CPR;
            const int c = (lane % F::CPR) ^ (isv ? pa_swz_v(r, F::ROWB) : pa_swz_k(r, F::ROWB));
            pf_dma((isv ? a.vc : a.kc) + head + (size_t)min(tt * F::KT + r, last) * HD + c * 8,
                   base + (unsigned)((tt & 1) * 2 * F::IMG + p * 1024));
        }
    };
    const float c2 = a.scale * 1.44269504088896340736f;
    const int nt = last / F::KT + 1;
    const float bias1 = ROWS ? x.r1[h] : 0.0f, bias2 = ROWS ? x.r2[h] : 0.0f;
    issue(0);
    for (int tt = 0; tt < nt; ++tt) {
        pf_wait_vm<0>();
        __builtin_amdgcn_s_barrier();  // every wave's pieces of tile tt landed; every wave is done with tile tt - 1
        if (tt + 1 < nt) issue(tt + 1);
        const int t0 = tt * F::KT;
        if (t0 > wlast) continue;  // (wave-uniform) nothing of this tile is seen
        const char* kimg = sm + (tt & 1) * 2 * F::IMG;
        const unsigned vbase = base + (unsigned)((tt & 1) * 2 * F::IMG + F::IMG);
        // Sᵀ[key][query] for keys t0 + 16 kt + (0..15)
        pf_float4 s[NK][QT];
#pragma unroll
        for (int kt = 0; kt < NK; ++kt)
#pragma unroll
            for (int t = 0; t < QT; ++t) s[kt][t] = pf_float4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int db = 0; db < ND; ++db) {
            u32x4 kf[NK];
#pragma unroll
            for (int kt = 0; kt < NK; ++kt) {
                const int r = kt * 16 + i16;
                kf[kt] = *reinterpret_cast<const u32x4*>(kimg + r * F::ROWB + ((4 * db + g) ^ pa_swz_k(r, F::ROWB)) * 16);
            }
#pragma unroll
            for (int i = 0; i < TERMS; ++i)
#pragma unroll
                for (int kt = 0; kt < NK; ++kt)
#pragma unroll
                    for (int t = 0; t < QT; ++t) s[kt][t] = pf_mfma(kf[kt], qf[i][t][db], s[kt][t]);
        }
        // lane holds keys t0 + 16 kt + 4 g + r of query i0 + 16 t + i16
        u32x4 pf[TERMS][QT][NK / 2];
#pragma unroll
        for (int t = 0; t < QT; ++t) {
            const int pos = ps.p0 + i0 + t * 16 + i16;
            if constexpr (ROWS) {  // the scores in base 2, less the bias of their distance (keys past the query: any number)
#pragma unroll
                for (int kt = 0; kt < NK; ++kt) s[kt][t] *= c2;
                if (bias1 != 0.0f) {
#pragma unroll
                    for (int kt = 0; kt < NK; ++kt)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const float dist = (float)max(pos - (t0 + kt * 16 + 4 * g + r), 0);
                            s[kt][t][r] -= bias1 * __builtin_amdgcn_logf(fmaf(bias2, dist, 1.0f));  // (log2)
                        }
                }
            }
            if (t0 + F::KT - 1 > ps.p0 + i0 + t * 16) {  // (wave-uniform) the diagonal
#pragma unroll
                for (int kt = 0; kt < NK; ++kt)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (t0 + kt * 16 + 4 * g + r > pos) s[kt][t][r] = -INFINITY;
            }
            float cmax = -INFINITY;
#pragma unroll
            for (int kt = 0; kt < NK; ++kt)
                cmax = fmaxf(cmax, fmaxf(fmaxf(s[kt][t][0], s[kt][t][1]), fmaxf(s[kt][t][2], s[kt][t][3])));
            cmax = max_xor32(max_xor16(cmax)) * (ROWS ? 1.0f : c2);
            const float mn = fmaxf(mx[t], cmax);
            if (__any(mn > mx[t])) {  // (key 0 is seen by every row: the maximum is finite from the first tile on)
                const float corr = __builtin_amdgcn_exp2f(mx[t] - mn);
                l[t] *= corr;
#pragma unroll
                for (int d = 0; d < NT; ++d) o[t][d] *= corr;
                mx[t] = mn;
            }
#pragma unroll
            for (int kb = 0; kb < NK / 2; ++kb) {
                __half ht[TERMS][8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float p = __builtin_amdgcn_exp2f(ROWS ? s[2 * kb + (e >> 2)][t][e & 3] - mx[t]
                                                                : fmaf(s[2 * kb + (e >> 2)][t][e & 3], c2, -mx[t])) * 256.0f;
                    l[t] += p;
                    pf_terms(p, ht, e);
                }
#pragma unroll
                for (int i = 0; i < TERMS; ++i) pf[i][t][kb] = *reinterpret_cast<const u32x4*>(ht[i]);
            }
        }
        // Vᵀ 16-d tile d: lane 16 g + 4 q + p addresses row (4 g + q) [+16] of the 32-key block, d 16 d + 4 p .. +3
        const int q4 = (lane & 15) >> 2, p4 = lane & 3;
#pragma unroll
        for (int kb = 0; kb < NK / 2; ++kb) {
            const int r1 = kb * 32 + 4 * g + q4, r2 = r1 + 16;
            const unsigned a1 = vbase + r1 * F::ROWB + 8 * (p4 & 1), a2 = vbase + r2 * F::ROWB + 8 * (p4 & 1);
            const int s1 = pa_swz_v(r1, F::ROWB), s2 = pa_swz_v(r2, F::ROWB);
            uint2 x1[NT], x2[NT];
#pragma unroll
            for (int d = 0; d < NT; ++d) {
                const int c = 2 * d + (p4 >> 1);
                x1[d] = pa_tr_read(a1 + ((c ^ s1) * 16));
                x2[d] = pa_tr_read(a2 + ((c ^ s2) * 16));
            }
            pa_tr_wait(x1, x2);
#pragma unroll
            for (int i = 0; i < TERMS; ++i)
#pragma unroll
                for (int d = 0; d < NT; ++d)
#pragma unroll
                    for (int t = 0; t < QT; ++t)
                        o[t][d] = pf_mfma(u32x4{x1[d].x, x1[d].y, x2[d].x, x2[d].y}, pf[i][t][kb], o[t][d]);
        }
    }
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        const int i = i0 + t * 16 + i16;
        const float ls = sum_xor32(sum_xor16(l[t]));
        if constexpr (ROWS) {
            const float sk = x.sink[h] * 1.44269504088896340736f, M = fmaxf(mx[t], sk), f = __builtin_amdgcn_exp2f(mx[t] - M);
            const float inv = f / (ls * f + 256.0f * __builtin_amdgcn_exp2f(sk - M));
            if (i >= ps.nv) continue;
            __half* dst = a.out.hi + (size_t)(row0 + i) * x.ldo + (size_t)h * x.vdim;
#pragma unroll
            for (int d = 0; d < NT; ++d) {
                const int d0 = d * 16 + 4 * g;
                const __half y[4] = {__float2half_rn(o[t][d][0] * inv), __float2half_rn(o[t][d][1] * inv),
                                     __float2half_rn(o[t][d][2] * inv), __float2half_rn(o[t][d][3] * inv)};
                if (x.vdim % 4 == 0 && d0 < x.vdim) {
                    *reinterpret_cast<uint2*>(dst + d0) = *reinterpret_cast<const uint2*>(y);
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (d0 + r < x.vdim) dst[d0 + r] = y[r];
                }
            }
            continue;
        }
        const float inv = 1.0f / ls;
        if (i >= ps.nv) continue;
#pragma unroll
        for (int d = 0; d < NT; ++d) {  // lane holds d = 16 d + 4 g + r of query i
            const size_t idx = (size_t)(seq * ps.rps + i) * qs + (size_t)h * HD + d * 16 + 4 * g;
            const float y[4] = {o[t][d][0] * inv, o[t][d][1] * inv, o[t][d][2] * inv, o[t][d][3] * inv};
            a.out.template store<4>(idx, y);
        }
    }
}

// Batches take three terms of q and p, as their steps do (attn_mfma.h); one sequence's prefill takes two. Heads and positions
// per workgroup and wave: 32 query positions per wave where that still gives every CU two workgroups, 16 (twice as many
// workgroups, each key row read twice as often) below (511 rows of 32 heads: 256 workgroups, not 128) and with three terms
// at head_dim 128, where 32 spill 48 registers (8 prompts of 2000 of Llama-3-8B 480 ms, with 16 461; two terms 456).
template <int HD>
hipError_t launch_pf_flash(const PfAttnArgs<__half>& a, const PfState& ps, int cus, hipStream_t s) {
    const int G = a.hq / a.hkv, GW = G < 4 ? G : 4;
    const int ny = a.hkv * (G / GW);
    auto blocks = [&](int qt) { return (ps.nv + (4 / GW) * 16 * qt - 1) / ((4 / GW) * 16 * qt) * ps.nseq; };
    const bool wide = blocks(2) * ny >= 2 * cus;
    auto go = [&](auto kernel, int qt) { hipLaunchKernelGGL(kernel, dim3(blocks(qt), ny), dim3(256), 0, s, a, ps, GW, PfPortions{}); };
    if (ps.nseq > 1)
        HD == 64 && wide ? go(pf_flash_kernel<HD, HD == 64 ? 2 : 1, 3>, 2) : go(pf_flash_kernel<HD, 1, 3>, 1);
    else
        wide ? go(pf_flash_kernel<HD, 2, 2>, 2) : go(pf_flash_kernel<HD, 1, 2>, 1);
    return hipGetLastError();
}

// The portions of a pass of M rows, msegs of them at most
template <int HD>
hipError_t launch_pf_flash_rows(const PfAttnArgs<__half>& a, const PfPortions& x, int M, int msegs, int cus, hipStream_t s) {
    const int G = a.hq / a.hkv, GW = G % 4 == 0 ? 4 : G % 2 == 0 ? 2 : 1, ny = a.hkv * (G / GW);
    auto blocks = [&](int qt) { return M / ((4 / GW) * 16 * qt) + msegs; };
    if ((M / ((4 / GW) * 32)) * ny >= 2 * cus)
        hipLaunchKernelGGL((pf_flash_kernel<HD, 2, 2, true>), dim3(blocks(2), ny), dim3(256), 0, s, a, PfState{}, GW, x);
    else
        hipLaunchKernelGGL((pf_flash_kernel<HD, 1, 2, true>), dim3(blocks(1), ny), dim3(256), 0, s, a, PfState{}, GW, x);
    return hipGetLastError();
}

// Where the portions take pf_attn_mfma_kernel instead: `groups` live groups of 16 rows in a pass, whose workgroups (heads of 128:
// 2 a CU, of 64: 4) run side by side, each wave with a quarter of the keys, where a flash workgroup walks all of them. A block of
// a 256-wide stack without feed-forward, by 16 rows | flash: 17 rows from position 15000 on, 8 query and 1 kv heads of 128, 233 | 384
// us; 32 and 32 heads of 128, 256 rows from 4000, 134 | 151; 32 and 8 heads of 64, 512 rows from 2000, 96 | 103. With twice the rows
// flash leads: 512 of the 32 of 128 227 | 211, 1024 of the 32 of 64 180 | 144. Over 1932 shapes (1 to 8 portions of 2 to 1024 rows,
// from position 0 to 15000, 8 to 64 heads) no pass was slower by this rule than by 16 rows throughout.
inline bool pf_rows_by_16(long groups, int heads, int hd, int cus) { return groups * heads <= (hd > 64 ? 2L : 4L) * cus; }

// The rows are packed portions (step_state.h RowRef; a 16-row group belongs to one portion, its valid rows first); one fp16
// output row [M][ldo] of vdim dims per head.
// WINDOWED false: as pf_flash_kernel's ROWS: bias, sink, one [hkv][T][HD] cache block per sequence slot.
// WINDOWED true: a query sees the last `window` positions up to its own, position t's K and V are row t + koff[row / 32] of one
// [hkv][T][HD] block (latent.h expands them), and the output is multiplied by gate [M][hq vdim].
struct PfRowsArgs {
    const RowRef* rows = nullptr;
    const float *r1 = nullptr, *r2 = nullptr, *sink = nullptr;  // [hq]
    int ldo = 0, vdim = 0;
    int window = 0;
    const int32_t* koff = nullptr;
    const float* gate = nullptr;
};
template <int HD, bool WINDOWED>
__global__ void __launch_bounds__(256) pf_attn_mfma_kernel(PfAttnArgs<__half> a, PfRowsArgs x) {
    using G = PaGeo<HD>;
    constexpr int ND = HD / 32, NT = HD / 16;  // 32-d blocks (S), 16-d tiles (O)
    __shared__ __attribute__((aligned(1024))) char sm[4 * G::WAVE];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int g = lane >> 4, i16 = lane & 15;
    const int h = blockIdx.y, kvh = h / (a.hq / a.hkv);
    const int mq = blockIdx.x * 16 + i16;  // this lane's query (chunk row)
    const RowRef r0 = x.rows[blockIdx.x * 16];
    if (r0.slot < 0) return;  // (uniform) a group of padding rows
    const bool live = x.rows[mq].slot >= 0;
    const int pos = r0.pos + i16;
    const int last = r0.pos + (int)__popcll(__ballot(live)) / 4 - 1;  // the group's last query (a row is the query of 4 lanes)
    const int kmin = WINDOWED ? max(0, r0.pos - x.window + 1) : 0;  // the first key any row of the group sees
    const int koff = WINDOWED ? x.koff[blockIdx.x >> 1] : 0, tile0 = kmin / 32;
    const float bias1 = WINDOWED ? 0.0f : x.r1[h], bias2 = WINDOWED ? 0.0f : x.r2[h];
    const int kmax = last;  // cache rows past it are read as this one (their scores are masked)
    const int ntiles = last / 32 + 1;
    const size_t qs = (size_t)a.hq * HD;
    // Qᵀ as the B operand: lane l = query l & 15, d = 32 db + 8 g .. +8, fp32 -> hi + lo
    u32x4 qh[ND], ql[ND];
#pragma unroll
    for (int db = 0; db < ND; ++db) {
        const float4* qp = reinterpret_cast<const float4*>(a.q + (size_t)mq * qs + (size_t)h * HD + db * 32 + g * 8);
        const float4 v0 = qp[0], v1 = qp[1];
        const float f[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
        __half hh[8], hl[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) pf_split(f[e], hh[e], hl[e]);
        qh[db] = *reinterpret_cast<const u32x4*>(hh);
        ql[db] = *reinterpret_cast<const u32x4*>(hl);
    }
    pf_float4 o[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) o[t] = pf_float4{0.0f, 0.0f, 0.0f, 0.0f};
    float mx = -INFINITY, l = 0.0f;
    char* kimg = sm + wave * G::WAVE;
    const unsigned kbase = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) char*)kimg;
    const unsigned vbase = kbase + G::IMG;
    const size_t head = ((size_t)(WINDOWED ? 0 : r0.slot) * a.hkv + kvh) * a.T * HD;
    const __half *kc = a.kc + head, *vc = a.vc + head;
    for (int tt = tile0 + wave; tt < ntiles; tt += 4) {
        const int t0 = tt * 32;
        // K pieces 0 .. P/2-1, V pieces P/2 .. P-1; lane i of a piece: row (piece rows) + i / CPR, physical
        // chunk i % CPR <- logical chunk (i % CPR) ^ swizzle(row)
#pragma unroll
        for (int j = 0; j < G::PIECES; ++j) {
            const bool isv = j >= G::PIECES / 2;
            const int jj = isv ? j - G::PIECES / 2 : j;
            const int r = jj * (1024 / G::ROWB) + lane / G::CPR;
            const int c = (lane % G::CPR) ^ (isv ? pa_swz_v(r, G::ROWB) : pa_swz_k(r, G::ROWB));
            const int kr = max(min(t0 + r, kmax), kmin) + koff;
            const __half* src = (isv ? vc : kc) + (size_t)kr * HD + c * 8;
            pf_dma(src, (isv ? vbase : kbase) + (unsigned)(jj * 1024));
        }
        pf_wait_vm<0>();
        // Sᵀ[key][query] for keys t0 + 16 kt + (0..15)
        pf_float4 sacc[2];
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
            sacc[kt] = pf_float4{0.0f, 0.0f, 0.0f, 0.0f};
            const int r = kt * 16 + i16;
            const char* krow = kimg + r * G::ROWB;
#pragma unroll
            for (int db = 0; db < ND; ++db) {
                const u32x4 kf = *reinterpret_cast<const u32x4*>(krow + ((4 * db + g) ^ pa_swz_k(r, G::ROWB)) * 16);
                sacc[kt] = pf_mfma(kf, qh[db], sacc[kt]);
                sacc[kt] = pf_mfma(kf, ql[db], sacc[kt]);
            }
        }
        // lane holds keys t0 + 16 kt + 4 g + r of query mq
        float sv[8];
        float cmax = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int key = t0 + kt * 16 + 4 * g + r;
                float sc = sacc[kt][r] * a.scale;
                if constexpr (!WINDOWED) sc -= bias1 * __logf(1.0f + bias2 * (float)(pos - key));
                const bool see = key <= pos && (!WINDOWED || key > pos - x.window);
                const float v = see ? sc : -INFINITY;
                sv[kt * 4 + r] = v;
                cmax = fmaxf(cmax, v);
            }
        cmax = fmaxf(cmax, __shfl_xor(cmax, 16));
        cmax = fmaxf(cmax, __shfl_xor(cmax, 32));
        const float mn = fmaxf(mx, cmax);
        const float corr = mn == -INFINITY ? 1.0f : expf(mx - mn);
        float pv[8], psum = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            pv[e] = sv[e] == -INFINITY ? 0.0f : expf(sv[e] - mn);
            psum += pv[e];
        }
        psum += __shfl_xor(psum, 16);
        psum += __shfl_xor(psum, 32);
        l = l * corr + psum;
        mx = mn;
        __half ph[8], pl[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) pf_split(pv[e], ph[e], pl[e]);
        const u32x4 pfh = *reinterpret_cast<const u32x4*>(ph);
        const u32x4 pfl = *reinterpret_cast<const u32x4*>(pl);
        // Vᵀ 16-d tile dt: lane 16 g + 4 q + p addresses row (4 g + q) [+16], d 16 dt + 4 p .. +3
        const int q4 = (lane & 15) >> 2, p4 = lane & 3;
        const int r1 = 4 * g + q4, r2 = 16 + 4 * g + q4;
        const unsigned a1 = vbase + r1 * G::ROWB + 8 * (p4 & 1), a2 = vbase + r2 * G::ROWB + 8 * (p4 & 1);
        const int s1 = pa_swz_v(r1, G::ROWB), s2 = pa_swz_v(r2, G::ROWB);
        uint2 x1[NT], x2[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int c = 2 * t + (p4 >> 1);
            x1[t] = pa_tr_read(a1 + ((c ^ s1) * 16));
            x2[t] = pa_tr_read(a2 + ((c ^ s2) * 16));
        }
        pa_tr_wait(x1, x2);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            o[t] *= corr;
            const u32x4 vf = u32x4{x1[t].x, x1[t].y, x2[t].x, x2[t].y};
            o[t] = pf_mfma(vf, pfh, o[t]);
            o[t] = pf_mfma(vf, pfl, o[t]);
        }
    }
    // merge the 4 key splits: wave w publishes (mx, l, o) and merges 16-d tiles t = w, w + 4, ...
    __syncthreads();
    float* fo = reinterpret_cast<float*>(sm);                         // [wave][NT][64 lanes][4]
    float* fm = fo + 4 * NT * 64 * 4;                                 // [wave][64]
    float* fl = fm + 4 * 64;
#pragma unroll
    for (int t = 0; t < NT; ++t)
        *reinterpret_cast<pf_float4*>(fo + ((wave * NT + t) * 64 + lane) * 4) = o[t];
    fm[wave * 64 + lane] = mx;
    fl[wave * 64 + lane] = l;
    __syncthreads();
    float m4[4], w4[4], M = -INFINITY;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        m4[w] = fm[w * 64 + lane];
        M = fmaxf(M, m4[w]);
    }
    float L = 0.0f;
    if constexpr (!WINDOWED) {
        M = fmaxf(M, x.sink[h]);
        L = expf(x.sink[h] - M);
    }
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        w4[w] = m4[w] == -INFINITY ? 0.0f : expf(m4[w] - M);
        L += fl[w * 64 + lane] * w4[w];
    }
    const float inv = 1.0f / L;
    for (int t = wave; t < NT; t += 4) {
        pf_float4 acc = pf_float4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int w = 0; w < 4; ++w) acc += *reinterpret_cast<const pf_float4*>(fo + ((w * NT + t) * 64 + lane) * 4) * w4[w];
        // lane holds d = 16 t + 4 g + r of query mq
        const int d0 = t * 16 + 4 * g;
        __half* dst = a.out.hi + (size_t)mq * x.ldo + (size_t)h * x.vdim + d0;
        if (!live) continue;
        if constexpr (WINDOWED) {
            const float* gt = x.gate + ((size_t)mq * a.hq + h) * x.vdim + d0;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (d0 + r < x.vdim) acc[r] *= gt[r];
        }
        if (x.vdim % 4 == 0 && d0 < x.vdim) {
            const __half hv[4] = {__float2half_rn(acc[0] * inv), __float2half_rn(acc[1] * inv),
                                  __float2half_rn(acc[2] * inv), __float2half_rn(acc[3] * inv)};
            *reinterpret_cast<uint2*>(dst) = *reinterpret_cast<const uint2*>(hv);
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (d0 + r < x.vdim) dst[r] = __float2half_rn(acc[r] * inv);
        }
    }
}

}  // namespace sli
