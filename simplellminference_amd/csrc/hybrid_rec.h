// hybrid_rec.h — recording a projection over M rows for block-stack models (hybrid.h): which kernel runs it, by the row
// count and the element type. Base of the recorders of the two arrangements.
#pragma once
#include <type_traits>

#include "hybrid_kernels.h"
#include "hybrid_stack.h"

namespace sli {

template <typename WT>
struct HyProj {
    BlockStack* s;
    int M;      // rows of the launches
    bool one;   // one row per sequence (decode)
    int msegs;  // portions at most
    int key_tiles = 0;  // sequential arrangement: expansion tiles at most
    hipStream_t st() const { return s->stream; }

    // How a projection over M rows runs: the batch-1 GEMV, the batched MFMA projection (fp16, 2 .. 8 rows; one row past
    // the GEMV's LDS stage), the prompt GEMM (fp16, more rows), or the plain kernel (fp32, more rows or wider).
    enum Path { GV, BG, PG, RG };
    static constexpr bool F16 = std::is_same<WT, __half>::value;
    static Path path(int M, int K) {
        if (M == 1 && K <= kGemvMaxCols) return GV;
        if (!F16) return RG;
        return M <= kBgMaxBatch ? BG : PG;
    }
    // rows of the launches for n rows
    static int rows_for(int n) { return F16 && n > kBgMaxBatch ? pad_to(n, kHyTile) : n; }

    template <class Epi>
    int project(const void* W, const void* X, int K, int npairs, int u0, const Epi& e, const void* Wt = nullptr) const {
        const WT* w = (const WT*)W + (size_t)2 * u0 * K;
        const Path p = path(M, K);
        if (p == GV) {
            GemvIn in{(const float*)X, nullptr, 0.0f, K};
            SLI_HIP((launch_gemv_u<WT, 2, 4, true>(w, in, GvPair<Epi>{e, npairs, u0}, npairs, st())));
            return SLI_OK;
        }
        if constexpr (F16) {
            if (p == BG) {
                BgIn in{};
                in.x = (const float*)X;
                in.K = K;
                in.B = M;
                in.ws = s->bg_ws;
                in.counters = s->bg_cnt;
                const BgPlan pl = bg_plan((npairs + 7) / 8, K, M, false, gemv_max_blocks(), true);
                in.tiled = Wt != nullptr;  // (Wt: the copy from pair u0 on)
                SLI_HIP((launch_bgemm(Wt ? (const WT*)Wt : w, in, BgPair<Epi>{e, npairs, u0}, pl, st())));
                return SLI_OK;
            }
            if (p == PG) return pgemm(w, (const __half*)X, nullptr, 0, K, npairs, u0, e);
        }
        SLI_HIP((launch_rows_gemm<WT, Epi>(w, (const float*)X, K, npairs, u0, M, e, st())));
        return SLI_OK;
    }
    // 2 .. 8 rows: pairs [0, n1) of X and [u1, u1 + n2) of X2 in one launch. 6 rows of 2048 columns, a block's 9728 and 11264
    // pairs in the mean: two launches 25.6 us, one 22.8; a decode pass of 16 blocks for 2 | 3 | 5 | 8 sequences 1020 | 1084 | 1220 |
    // 1413 us -> 982 | 1045 | 1187 | 1375.
    template <class Epi>
    int project2(const void* W, const void* X, const void* X2, int K, int n1, int u1, int n2, const Epi& e, const void* Wt) const {
        if constexpr (F16) {
            BgIn in{};
            in.x = (const float*)X, in.x2 = (const float*)X2;
            in.K = K, in.B = M;
            in.ws = s->bg_ws, in.counters = s->bg_cnt;
            const int nt1 = (n1 + 7) / 8, nt2 = (n2 + 7) / 8;
            in.tiled = Wt != nullptr;
            SLI_HIP((launch_bgemm((const WT*)(Wt ? Wt : W), in, BgPair2<Epi>{e, n1, n2, u1, nt1},
                                  bg_plan(nt1 + nt2, K, M, false, gemv_max_blocks(), true, nt1), st())));
            return SLI_OK;
        } else {
            return fail(SLI_ERR_ARG, "batched projection: fp16 weights");
        }
    }
    // pairs [0, split) read X, pairs [split, npairs) X2 (split: a multiple of kHySection; X2 null: one input)
    template <class Epi>
    int pgemm(const WT* w, const __half* X, const __half* X2, int split, int K, int npairs, int u0, const Epi& e, int spare = 0,
              int valid = 0x7fffffff) const {
        if constexpr (F16) {
            PgIn<__half> in{w, X, nullptr, pad_to(2 * npairs, 16), K, M};
            in.valid = valid;
            if (X2) in.Bhi2 = X2, in.row_b2 = 2 * split;
            in.ws = s->pg_ws, in.cnt = s->pg_cnt;
            float best = INFINITY;
            int pick = 0;
            constexpr bool rolled = PgRolled<PgPair<Epi>>::value;
            // spare: rows there are. Tiles of 256 rows over more rows than there are to do may be faster than tiles of 128: 4096 x
            // 15104 at 1152 rows 191 us, at 1280 rows 169.
            // valid: waves whose rows are all padding past it multiply nothing (that 4096 x 15104 at 1025 rows 173 -> 169).
            for (int m : {M, pad_to(M, 256)}) {
                int i = 0;
                if (m > M && m > spare) break;
                pg_row_tilings(m, rolled, [&](auto cfg, float us) {
                    const PgPlan p = pg_plan<decltype(cfg), __half>(in.N, K, m, device_cus(), true, us, rolled);
                    if (p.us < best) best = p.us, pick = i, in.full = p.full, in.splits = p.splits, in.M = m;
                    ++i;
                });
            }
            hipError_t err = hipSuccess;
            int i = 0;
            pg_row_tilings(in.M, rolled, [&](auto cfg, float) {
                if (i++ == pick) err = launch_pgemm<PgPair<Epi>, decltype(cfg), __half>(in, PgPair<Epi>{e, npairs, u0}, PfState{}, st());
            });
            SLI_HIP(err);
            return SLI_OK;
        } else {
            return fail(SLI_ERR_ARG, "prompt GEMM: fp16 weights");
        }
    }
    template <class Epi>
    static int allow() {
        if constexpr (F16) {
            hipError_t err = hipSuccess;
            for (int M : {32, 256})
                pg_row_tilings(M, false, [&](auto cfg, float) {
                    const hipError_t e = pgemm_allow_lds<PgPair<Epi>, decltype(cfg), __half>();
                    if (e != hipSuccess) err = e;
                });
            SLI_HIP(err);
            SLI_HIP((bg_allow_lds<BgPair<Epi>, false>()));
        }
        return SLI_OK;
    }

    // Row blocks with weights of their own (prefill.h PgGroups): X fp16 for fp16 weights, else fp32
    static constexpr int group_rows(int pairs_per_group) {
        return !F16 ? kRowsGemmTile : pairs_per_group >= 192 ? 128 : pairs_per_group >= 48 ? 64 : 32;
    }
    template <class Epi>
    int grouped(const void* W, const void* X, int K, int npairs, const PgGroups& g, int bm, int maxtiles, const Epi& e) const {
        if constexpr (F16) {
            PgIn<__half> in{(const __half*)W, (const __half*)X, nullptr, pad_to(2 * npairs, 16), K, maxtiles * bm};
            in.grp = g;
            return pg_group_pick(bm, [&](auto cfg) -> int {
                SLI_HIP((launch_pgemm<PgPair<Epi>, decltype(cfg), __half>(in, PgPair<Epi>{e, npairs, 0}, PfState{}, st())));
                return SLI_OK;
            });
        } else {
            SLI_HIP((launch_rows_gemm_grouped<WT, Epi>((const WT*)W, (const float*)X, K, npairs, g, maxtiles, e, st())));
            return SLI_OK;
        }
    }
    template <class F>
    static int pg_group_pick(int bm, F&& f) {
        if (bm == 128) return f(PgCfg<128, 2, 3, 4, 0, 1, true>{});
        if (bm == 64) return f(PgCfg<64, 4, 4, 2, 0, 1, true>{});
        return f(PgCfg<32, 2, 4, 2, 0, 1, true>{});
    }
    template <class Epi>
    static int allow_grouped() {
        if constexpr (F16)
            for (int bm : {32, 64, 128})
                HY_TRY(pg_group_pick(bm, [&](auto cfg) -> int {
                    SLI_HIP((pgemm_allow_lds<PgPair<Epi>, decltype(cfg), __half>()));
                    return SLI_OK;
                }));
        return SLI_OK;
    }
};

}  // namespace sli
