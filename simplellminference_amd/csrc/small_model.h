// small_model.h — the greedy loop of a small model (batch 1, fp32 or fp16 weights) as ONE launch: n steps of
// LlamaModel::predict (source/model/model.cpp:150-187), each the layer loop of forward (:50-129), the LM head, the argmax and
// the next token, with every dependency inside the launch.
//
// Why: a step of the 256-wide two-layer preset reads 7 MB (1 us), and its 13 graph launches of 2 to 8 us take 69. Here a step
// has four all-to-all edges a layer and one for the token, each a store and a load and what a workgroup does between them: 19.4 us a step
// on half of one XCD, 25 over all eight, 36 greedy tokens in 0.70 and 0.90 ms instead of 2.5. The edges bound it (and, with large
// vocabularies, the head's rows: small_launch.h small_lost_us), and within an edge the instructions: on one XCD a granule is handed on
// in 0.3 of an edge's 1.8 us, the rest is some 200 instructions of 4 waves a SIMD. So sums end in one lane (sm_sum63), the norm's
// factor is applied to finished sums, beside which its squares are added up, LDS is read by LDS loads only, and each wave asks for its
// rows by 5 instructions a KiB (as 64-bit addresses and flat loads, each of them waited for, the same step took 28 us over all XCDs and 26
// on one).
//
// Structure: hq J workgroups, all resident (ONE: of 16 waves on half of one XCD's CUs; else of 8 waves, twice the workgroups, over all
// XCDs: engine.hip small_on_one); every workgroup holds the whole residual row and runs every op on its share of the rows. An edge is 8-byte {value, tag} granules as in tp_layers.h: one store each, no flag, no drain;
// readers sweep them with sc1 loads until the tags are this edge's. Between XCDs the stores are sc1 too; on one they end in its L2,
// where sc1 loads look. Tags count (launch, step, layer, edge), so one array an
// edge serves every layer: before a workgroup writes an edge's granules again it has read a later edge to which every
// workgroup contributes, so nobody still reads them.
//   q, k, v rows -> the workgroups of head h: its q, its kv head's k and v
//   attention of head h over the whole context, by each of its J workgroups; at once their D / J rows of wo over that head's
//   columns -> partial sums [hq][D] -> every workgroup: x1 = x + the heads' partials in head order
//   gate/up units -> act -> every workgroup: down rows + x1 -> x
//   the workgroups' argmax keys -> every workgroup: the next token
// A wave asks for its weight rows of the next op (LDS-DMA, its share of 64 KiB) when that of the op at hand has its input. K and V rows
// of earlier steps are read with sc1 loads: other CUs wrote them.
// Every wait is bounded: one that gives up sets DevState::error kSmErrWait, the workgroup skips every later wait, the others'
// waits give up too and the grid drains; the host then launches the loop over all XCDs, or runs the steps, and so every later call of
// the model's.
#pragma once
#include "common.h"
#include "prefill.h"
#include "small_launch.h"
#include "step_state.h"

namespace sli {

template <int WAVES>
struct alignas(16) SmSmem {
    float x[kSmMaxD], x1[kSmMaxD];  // the residual row before and after wo; zeros from D on (so are xg and act)
    float xg[kSmMaxD];              // x or x1 times the norm weights of the op that reads it
    float act[kSmMaxI];
    float qkv[3 * 128];
    float part[WAVES][128];      // a wave's o of the attention
    float ml[2][WAVES];          // its m and l
    float o[128];                   // the head's output
    unsigned long long key[WAVES];
    int dead, next;
};
template <int WAVES>
struct SmGeo {
    static constexpr int BYTES = kSmRowBytes / WAVES;  // rows of an op that a wave holds
    static constexpr size_t PRE = (sizeof(SmSmem<WAVES>) + 1023) / 1024 * 1024, LDS = PRE + 2 * kSmRowBytes;
    static_assert(LDS <= 160 * 1024, "LDS");
};
typedef int sm_i4 __attribute__((ext_vector_type(4)));

template <bool ONE>
__device__ __forceinline__ void sm_put(const SmArgs& a, int i, float v, unsigned tag) {
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(a.g, 0, 0x7fffffff, 0x00020000);
    __builtin_amdgcn_raw_buffer_store_b64(sm_u2{__float_as_uint(v), tag}, rs, 8u * (unsigned)i, 0, ONE ? 0 : 16 /* sc1 */);
}
// N granules at element offsets off[], of a thread, until all carry `tag`
template <int N, class Smem>
__device__ __forceinline__ void sm_wait(const int (&off)[N], unsigned tag, float (&out)[N], Smem& sm,
                                        const SmArgs& a) {
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(a.g, 0, 0x7fffffff, 0x00020000);
    for (unsigned pass = 0;; ++pass) {
        sm_u2 v[N];
#pragma unroll
        for (int j = 0; j < N; ++j) v[j] = __builtin_amdgcn_raw_buffer_load_b64(rs, 8u * (unsigned)off[j], 0, 16 /* sc1 */);
        bool miss = false;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            miss |= v[j].y != tag;
            out[j] = __uint_as_float(v[j].x);
        }
        if (!__any(miss) || sm.dead) return;
        if ((pass & a.look) == a.look) {
            const bool peer = (__hip_atomic_load(&a.st->error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & kSmErrWait) != 0;
            if (peer || pass >= a.spin) {
                __hip_atomic_fetch_or(&a.st->error, kSmErrWait, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                sm.dead = 1;
                return;
            }
        }
    }
}

// a matrix (or any array) as a buffer: loads past `bytes` read nothing and give zeros
__device__ __forceinline__ sm_i4 sm_buf(const void* p, unsigned bytes) {
    const unsigned long long u = (unsigned long long)p;
    auto uniform = [](unsigned v) { return (int)__builtin_amdgcn_readfirstlane((int)v); };
    return sm_i4{uniform((unsigned)u), uniform((unsigned)(u >> 32) & 0xffff), uniform(bytes), 0x00020000};
}
// 1 KiB from byte `off` on: lane i's 16 bytes at LDS byte lds + 16 i (counted by sm_landed only, as pf_dma)
__device__ __forceinline__ void sm_dma(const sm_i4& b, unsigned off, unsigned lds) {
    asm volatile(
        "s_mov_b32 m0, %2\n\t"
        "s_nop 0\n\t"
        "buffer_load_dwordx4 %0, %1, 0 offen lds"
        :
        : "v"(off), "s"(b), "s"(lds)
        : "memory", "m0");
}

// A wave's rows of an op: R rows of each of n items, row k of item i from byte off(i) + k second of W on, C columns (a multiple of 8)
// and `each` 1-KiB pieces a row (what follows a row's end in its last piece is never used). The rows of the first `held` items lie in
// the wave's half of LDS, in order; the others are loaded when they are used. These are two loops: one pointer to either memory would be a
// flat load, each waited for by itself.
template <typename WT, int R, int WBYTES, bool P1>
struct SmRows {
    static constexpr int E = 16 / (int)sizeof(WT);
    const WT* W;
    unsigned bytes, second;
    int C, n, each_, held;
    __device__ int each() const { return P1 ? 1 : each_; }
    __device__ SmRows(const void* w, unsigned nrows, int c, int n_, unsigned sec = 0)
        : W((const WT*)w), bytes(nrows * (unsigned)c * (unsigned)sizeof(WT)), second(sec * (unsigned)c * (unsigned)sizeof(WT)), C(c), n(n_),
          each_((c * (int)sizeof(WT) + 1023) / 1024), held(min(n_, WBYTES / 1024 / (R * each()))) {}
    template <class Off>
    __device__ void ask(unsigned lds, int lane, const Off& off) const {
        const sm_i4 b = sm_buf(W, bytes);
#pragma unroll 1
        for (int i = 0; i < held; ++i) {
            const unsigned o = off(i);
#pragma unroll
            for (int k = 0; k < R; ++k)
#pragma unroll 1
                for (int p = 0; p < each(); ++p, lds += 1024) sm_dma(b, o + k * second + p * 1024 + 16 * lane, lds);
        }
    }
    // piece p of NI items from i0 on times x (LDS, zeros past C), added to s
    template <int NI, bool HELD, class Off>
    __device__ void piece(const char* mine, int lane, const float* x, int i0, int p, const Off& off, float (&s)[NI * R]) const {
        const int c = (p * 64 + lane) * E;
        const bool on = c < C;
        float xv[E];
#pragma unroll
        for (int e = 0; e < E; e += 4) *reinterpret_cast<float4*>(&xv[e]) = *reinterpret_cast<const float4*>(x + (on ? c : 0) + e);
        u32x4 v[NI * R];
#pragma unroll
        for (int j = 0; j < NI * R; ++j) {
            if constexpr (HELD)
                v[j] = *reinterpret_cast<const u32x4*>(mine + ((i0 * R + j) * each() + p) * 1024 + lane * 16);
            else
                v[j] = *reinterpret_cast<const u32x4*>((const char*)W + off(i0 + j / R) + (j % R) * second + (on ? c : 0) * sizeof(WT));
        }
#pragma unroll
        for (int j = 0; j < NI * R; ++j) {
            float f[E], t = 0.0f;
            Vec16<WT>::unpack(v[j], f);
#pragma unroll
            for (int e = 0; e < E; ++e) t = fmaf(f[e], xv[e], t);
            s[j] += on ? t : 0.0f;
        }
    }
    // items i0 .. i0 + NI - 1: this lane's part of their rows times x
    template <int NI, class Off>
    __device__ void dot(const char* mine, int lane, const float* x, int i0, const Off& off, float (&s)[NI * R]) const {
#pragma unroll
        for (int j = 0; j < NI * R; ++j) s[j] = 0.0f;
        if (i0 + NI <= held) {
            if (P1) {
                piece<NI, true>(mine, lane, x, i0, 0, off, s);
            } else {
#pragma unroll 1
                for (int p = 0; p < each(); ++p) piece<NI, true>(mine, lane, x, i0, p, off, s);
            }
        } else {
#pragma unroll 1
            for (int p = 0; p < each(); ++p) piece<NI, false>(mine, lane, x, i0, p, off, s);
        }
    }
};

// a lane's part of the sum of squares of a row (zeros past its end): added up beside the dots it scales
__device__ __forceinline__ float sm_squares(const float* x, int lane) {
    static_assert(kSmMaxD == 512, "two float4 a lane");
    const float4 u = *reinterpret_cast<const float4*>(x + 4 * lane), v = *reinterpret_cast<const float4*>(x + 256 + 4 * lane);
    return ((u.x * u.x + u.y * u.y) + (u.z * u.z + u.w * u.w)) + ((v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w));
}
// The wave's sum, in lane 63: six instructions (four shifts inside the rows of 16, two broadcasts of a row's last lane), where a
// sum in every lane takes a dozen. What a step's ops cost beside their edges is instructions: 4 waves share a SIMD.
__device__ __forceinline__ float sm_sum63(float v) {
    auto step = [](float x, auto ctrl, auto rows) {
        return x + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(ctrl)::value, decltype(rows)::value, 0xF, true));
    };
    typedef std::integral_constant<int, 0xF> all;
    v = step(v, std::integral_constant<int, 0x111>{}, all{});  // row_shr 1, 2, 4, 8
    v = step(v, std::integral_constant<int, 0x112>{}, all{});
    v = step(v, std::integral_constant<int, 0x114>{}, all{});
    v = step(v, std::integral_constant<int, 0x118>{}, all{});
    v = step(v, std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xA>{});  // row_bcast 15
    v = step(v, std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xC>{});  // row_bcast 31
    asm volatile("" : "+v"(v));  // (made here, where all lanes are on: sunk into a branch on the lane the shifts would read zeros)
    return v;
}
__device__ __forceinline__ float sm_lane63(float v) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63)); }
// 1 / sqrt(ss / D + eps) (rms_kernel.cpp:12-19) of lane 63's sum, in every lane. v_rsq_f32 is good to 1 ulp, as a correctly rounded
// root and quotient together; it takes no subnormal numbers.
__device__ __forceinline__ float sm_inv(float ss, float inv_d, float eps) {
    const float m = fmaf(sm_lane63(ss), inv_d, eps);
    return m >= 1e-30f ? __builtin_amdgcn_rsqf(m) : 1.0f / sqrtf(m);
}
// f over the lanes a multiple of LK apart (8, 16 or 32), in every lane
template <int LK, class F>
__device__ __forceinline__ float sm_over(float v, F f) {
    static_assert(LK == 8 || LK == 16 || LK == 32, "lanes a key row");
    if constexpr (LK <= 8) v = f(v, dpp_f<kDppRor8>(v));
    if constexpr (LK <= 16) {
        const LanePair p = lanes_xor16(v);
        v = f(p.a, p.b);
    }
    const LanePair p = lanes_xor32(v);
    return f(p.a, p.b);
}
// the wave's largest argmax key: the values' halves first, then the lowest index among their equals (two 32-bit maxima over DPP; as
// 64-bit exchanges through LDS it took 0.4 us)
__device__ __forceinline__ unsigned long long sm_key_max(unsigned long long k) {
    auto umax = [](unsigned v) {
        auto step = [](unsigned x, unsigned y) { return x > y ? x : y; };
        v = step(v, (unsigned)__builtin_amdgcn_mov_dpp((int)v, kDppXor1, 0xF, 0xF, true));
        v = step(v, (unsigned)__builtin_amdgcn_mov_dpp((int)v, kDppXor2, 0xF, 0xF, true));
        v = step(v, (unsigned)__builtin_amdgcn_mov_dpp((int)v, kDppHalfMirror, 0xF, 0xF, true));
        v = step(v, (unsigned)__builtin_amdgcn_mov_dpp((int)v, kDppMirror, 0xF, 0xF, true));
        const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
        v = step(r[0], r[1]);
        const auto t = __builtin_amdgcn_permlane32_swap(v, v, false, false);
        return step(t[0], t[1]);
    };
    const unsigned hi = umax((unsigned)(k >> 32));
    const unsigned lo = umax((unsigned)(k >> 32) == hi ? (unsigned)k : 0u);
    return (unsigned long long)hi << 32 | lo;
}
__device__ __forceinline__ void sm_landed() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

template <typename WT, typename KT, int HD, int WAVES, bool ONE, bool D1>
__global__ void __launch_bounds__(64 * WAVES) small_predict_kernel(SmArgs a) {
    using Geo = SmGeo<WAVES>;
    constexpr int THREADS = 64 * WAVES, WBYTES = Geo::BYTES;
    extern __shared__ __attribute__((aligned(1024))) char sm_raw[];
    SmSmem<WAVES>& sm = *reinterpret_cast<SmSmem<WAVES>*>(sm_raw);
    int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int wg = blockIdx.x;
    if constexpr (ONE) {
        unsigned xcc;
        asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
        if ((int)(xcc & 15) != a.xcd) return;
        if (tid == 0) sm.dead = (int)__hip_atomic_fetch_add(a.ticket + a.turn, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        wg = __builtin_amdgcn_readfirstlane(sm.dead);
        __syncthreads();
        if (wg >= a.nwg) return;
        if (wg == 0 && tid == 0) __hip_atomic_store(a.ticket + 1 - a.turn, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    const int J = a.nwg / a.hq, h = wg / J, hj = wg - h * J, kvh = h / (a.hq / a.hkv);
    const int D = a.D, I = a.I, half = HD / 2;
    const float inv_d = 1.0f / (float)D;
    // The wave's two halves of LDS: an op's rows lie in one, the next op's are asked for into the other as soon as the op's input is
    // there. (Asked for just before a wait they would come back ahead of its granules: loads return in order.)
    char* const base = sm_raw + Geo::PRE + wave * 2 * WBYTES;
    const unsigned lds0 = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) char*)base;
    int side = 0;  // of the op at hand
    auto mine = [&] { return base + side * WBYTES; };
    auto next_lds = [&] { return lds0 + (unsigned)((side ^ 1) * WBYTES); };
    if (tid == 0) sm.dead = 0;
    int token = a.st->token, pos = a.st->pos, next = 0;
    const int advance = a.st->advance, forced = a.st->n_forced;
    // this wave's share of every op: items wg + nwg (wave + 8 i)
    auto count = [&](int n) { return max(0, n <= wg ? 0 : ((n - wg + a.nwg - 1) / a.nwg - wave + WAVES - 1) / WAVES); };
    auto item = [&](int i) { return wg + a.nwg * (wave + WAVES * i); };
    const int npair = count((a.hq + 2 * a.hkv) * half), nunit = count(I), ndown = count(D), nhead = count(a.V);
    auto off_qkv = [&](int i) { const int u = item(i), uh = u / half; return (unsigned)(uh * HD + (u - uh * half)) * (unsigned)(D * (int)sizeof(WT)); };
    auto off_d = [&](int i) { return (unsigned)item(i) * (unsigned)(D * (int)sizeof(WT)); };
    auto off_i = [&](int i) { return (unsigned)item(i) * (unsigned)(I * (int)sizeof(WT)); };
    // wo: this workgroup's rows hj + J i, over head h's columns; LW lanes a row, RW rows a piece
    constexpr int EW = 16 / (int)sizeof(WT), LW = HD / EW, RW = 64 / LW;
    const int nwo = (D - hj + J - 1) / J;  // rows of the workgroup; wave w has pieces w, w + 8, ..
    const int pwo = max(0, ((nwo + RW - 1) / RW - wave + WAVES - 1) / WAVES);
    auto wo_at = [&](int p) {  // (bytes)
        const int i = min((wave + WAVES * p) * RW + lane / LW, nwo - 1);
        return (unsigned)((hj + J * i) * a.hq * HD + h * HD + (lane % LW) * EW) * (unsigned)sizeof(WT);
    };
    // (the table is constant: scalar loads)
    auto weights = [&](int l, int k) { return (const void*)((const __attribute__((address_space(4))) unsigned long long*)a.w)[4 * l + k]; };
    auto rows_qkv = [&](int l) { return SmRows<WT, 2, WBYTES, D1>(weights(l, 0), (a.hq + 2 * a.hkv) * HD, D, npair, half); };
    auto rows_up = [&](int l) { return SmRows<WT, 2, WBYTES, D1>(weights(l, 2), 2 * I, D, nunit, I); };
    auto rows_down = [&](int l) { return SmRows<WT, 1, WBYTES, false>(weights(l, 3), D, I, ndown); };
    auto rows_head = [&] { return SmRows<WT, 1, WBYTES, D1>(a.emb, a.V, D, nhead); };
    // norm weights of the thread's value of the residual row, loaded an op ahead
    const int di = min(tid, D - 1);
    float gw = a.norms[di];
    rows_qkv(0).ask(lds0, lane, off_qkv);
    for (int i = tid; i < kSmMaxD; i += THREADS) sm.x[i] = 0.0f, sm.x1[i] = 0.0f, sm.xg[i] = 0.0f;
    for (int i = tid; i < kSmMaxI; i += THREADS) sm.act[i] = 0.0f;
    for (int i = tid; i < WAVES * 128; i += THREADS) (&sm.part[0][0])[i] = 0.0f;
    if (tid < WAVES) sm.ml[0][tid] = -INFINITY, sm.ml[1][tid] = 0.0f;
    __syncthreads();
    for (int step = 0; step < a.n; ++step) {
        const int after = a.prompt[min(pos + 1, a.T)];  // the prompt's next token, where there is one
        auto turn = [&](const float* t, int i) { return t[pos * half + item(i) % half]; };
        const float fci0 = npair ? turn(a.sin_t, 0) : 0.0f, fcr0 = npair ? turn(a.cos_t, 0) : 0.0f;  // of the first pair
        const bool ok = token >= 0 && token < a.V;  // (as embedding_kernel: zeros for a token that is none)
        if (tid < D) {
            const float v = ok ? to_f32(((const WT*)a.emb)[(size_t)token * D + tid]) : 0.0f;
            sm.x[tid] = v;
            sm.xg[tid] = v * gw;
        }
        __syncthreads();
        for (int l = 0; l < a.L; ++l) {
            // (what follows from these is computed where it is used: kept over the loop it would be spilled, a mask at two lane
            // reads a use)
            asm volatile("" : "+v"(tid), "+v"(lane), "+s"(wave), "+s"(wg));
            const unsigned tag = a.tag0 + (unsigned)(step * (a.L + 1) + l) * 4;
            KT* kc = (KT*)a.kc + (size_t)l * a.hkv * a.T * HD;
            KT* vc = (KT*)a.vc + (size_t)l * a.hkv * a.T * HD;
            const void* wo = weights(l, 1);
            {  // q, k, v (model.cpp:52-67)
                const auto r = rows_qkv(l);
                sm_landed();
                gw = a.norms[(2 * l + 1) * D + di];
                const sm_i4 wob = sm_buf(wo, (unsigned)(D * a.hq * HD) * (unsigned)sizeof(WT));
                for (int p = 0; p < pwo && (p + 1) * 1024 <= WBYTES; ++p) sm_dma(wob, wo_at(p), next_lds() + p * 1024);
                float ss = sm_squares(sm.x, lane), inv = 0.0f;
                for (int i = 0; i < npair; ++i) {
                    float v2[2];
                    r.template dot<1>(mine(), lane, sm.xg, i, off_qkv, v2);
                    v2[0] = sm_sum63(v2[0]), v2[1] = sm_sum63(v2[1]);
                    if (i == 0) inv = sm_inv(sm_sum63(ss), inv_d, a.eps);
                    v2[0] = sm_lane63(v2[0]) * inv, v2[1] = sm_lane63(v2[1]) * inv;
                    const int u = item(i), uh = u / half, d = u - uh * half;
                    if (uh < a.hq + a.hkv) {  // rope_kernel.cpp:30-38
                        const float fci = i ? turn(a.sin_t, i) : fci0, fcr = i ? turn(a.cos_t, i) : fcr0;
                        const float r0 = v2[0] * fcr - v2[1] * fci, r1 = v2[1] * fcr + v2[0] * fci;
                        v2[0] = r0, v2[1] = r1;
                    }
                    if (lane < 2) {
                        const float v = lane ? v2[1] : v2[0];
                        const int e = d + lane * half;
                        const int kh = uh - a.hq, vh = kh - a.hkv;
                        const KT kv = from_f32<KT>(v);
                        // (k and v as the cache holds them)
                        sm_put<ONE>(a, uh * HD + e, kh >= 0 ? to_f32<KT>(kv) : v, tag);
                        if (kh >= 0) {
                            KT* to = (vh >= 0 ? vc + ((size_t)vh * a.T + pos) * HD : kc + ((size_t)kh * a.T + pos) * HD) + e;
                            if constexpr (sizeof(KT) == 4)
                                __hip_atomic_store((unsigned*)to, __builtin_bit_cast(unsigned, kv), __ATOMIC_RELAXED, ONE ? __HIP_MEMORY_SCOPE_WORKGROUP : __HIP_MEMORY_SCOPE_AGENT);
                            else
                                __hip_atomic_store((unsigned short*)to, __builtin_bit_cast(unsigned short, kv), __ATOMIC_RELAXED, ONE ? __HIP_MEMORY_SCOPE_WORKGROUP : __HIP_MEMORY_SCOPE_AGENT);
                        }
                    }
                }
                side ^= 1;
            }
            // ---- attention of head h (mha_kernel.cpp:36-77) and its columns of wo
            constexpr int EK = 16 / (int)sizeof(KT), LK = HD / EK, NG = THREADS / LK;  // lanes a key row, keys a pass
            const int grp = tid / LK, c0 = (lane % LK) * EK;
            const auto rk = __builtin_amdgcn_make_buffer_rsrc(kc + (size_t)kvh * a.T * HD, 0, 0x7fffffff, 0x00020000);
            const auto rv = __builtin_amdgcn_make_buffer_rsrc(vc + (size_t)kvh * a.T * HD, 0, 0x7fffffff, 0x00020000);
            auto key_at = [&](int t) { return (unsigned)((min(t, pos) * HD + c0) * (int)sizeof(KT)); };
            u32x4 kn = __builtin_amdgcn_raw_buffer_load_b128(rk, key_at(grp), 0, 16), vn = __builtin_amdgcn_raw_buffer_load_b128(rv, key_at(grp), 0, 16);
            if (wave * 64 < 3 * HD) {
                const int i = min(tid, 3 * HD - 1);
                const int off[1] = {i < HD ? h * HD + i : i < 2 * HD ? (a.hq + kvh) * HD + i - HD : (a.hq + a.hkv + kvh) * HD + i - 2 * HD};
                float v[1];
                sm_wait<1>(off, tag, v, sm, a);
                sm.qkv[i] = v[0];
            }
            __syncthreads();
            const auto ru = rows_up(l);
            float q[EK], o[EK], mx = -INFINITY, lsum = 0.0f;
#pragma unroll
            for (int e = 0; e < EK; ++e) q[e] = sm.qkv[c0 + e], o[e] = 0.0f;
            for (int t0 = 0; t0 + wave * (64 / LK) <= pos; t0 += NG) {  // (passes in which the wave has a key)
                const int t = t0 + grp;
                float kf[EK], vf[EK];
                Vec16<KT>::unpack(kn, kf);
                Vec16<KT>::unpack(vn, vf);
                if (t0 + NG <= pos) {
                    kn = __builtin_amdgcn_raw_buffer_load_b128(rk, key_at(t + NG), 0, 16);
                    vn = __builtin_amdgcn_raw_buffer_load_b128(rv, key_at(t + NG), 0, 16);
                }
                if (t == pos) {  // this step's own row
#pragma unroll
                    for (int e = 0; e < EK; ++e) kf[e] = sm.qkv[HD + c0 + e], vf[e] = sm.qkv[2 * HD + c0 + e];
                }
                float s = 0.0f;
#pragma unroll
                for (int e = 0; e < EK; ++e) s = fmaf(q[e], kf[e], s);
                s = group_sum<LK>(s) * a.scale;
                if (t <= pos) {
                    const float mn = fmaxf(mx, s), c = expf(mx - mn), p = expf(s - mn);
                    lsum = lsum * c + p;
#pragma unroll
                    for (int e = 0; e < EK; ++e) o[e] = fmaf(p, vf[e], o[e] * c);
                    mx = mn;
                }
            }
            // the wave's groups, then the waves: HD / 64 of them merge all parts
            if (wave * (64 / LK) <= pos) {
                const float M = sm_over<LK>(mx, [](float x, float y) { return fmaxf(x, y); });
                const float f = mx == -INFINITY ? 0.0f : expf(mx - M);
                auto add = [](float x, float y) { return x + y; };
                lsum = sm_over<LK>(lsum * f, add);
#pragma unroll
                for (int e = 0; e < EK; ++e) o[e] = sm_over<LK>(o[e] * f, add);
                if (lane < LK) {
#pragma unroll
                    for (int e = 0; e < EK; e += 4)
                        *reinterpret_cast<float4*>(&sm.part[wave][c0 + e]) = make_float4(o[e], o[e + 1], o[e + 2], o[e + 3]);
                }
                if (lane == 0) sm.ml[0][wave] = M, sm.ml[1][wave] = lsum;
            }
            __syncthreads();
            sm_landed();  // (wo's pieces; the K / V row of this step is out before wo's sums: the steps after read it behind a later edge)
            // the next op's rows, where the q, k, v rows lay (not before the keys: what is left of their loads is waited for with all
            // that came after them)
            ru.ask(next_lds(), lane, off_d);
            if (wave * 64 < HD) {  // lane v: wave v's factor
                // (a wave without a key yet: -inf, 0 and zeros, as they were set at the start)
                const float m8 = sm.ml[0][lane % WAVES], l8 = sm.ml[1][lane % WAVES];
                float s = 0.0f, p8[WAVES];
#pragma unroll
                for (int v = 0; v < WAVES; ++v) p8[v] = sm.part[v][tid];
                const float f8 = expf(m8 - group_max<WAVES>(m8)), fi = f8 * (1.0f / group_sum<WAVES>(l8 * f8));
#pragma unroll
                for (int v = 0; v < WAVES; ++v) s = fmaf(p8[v], __int_as_float(__builtin_amdgcn_readlane(__float_as_int(fi), v)), s);
                sm.o[tid] = s;
            }
            __syncthreads();
            for (int p = 0; p < pwo; ++p) {
                float wf[EW], s = 0.0f;
                if ((p + 1) * 1024 <= WBYTES)
                    Vec16<WT>::unpack(*reinterpret_cast<const u32x4*>(mine() + p * 1024 + lane * 16), wf);
                else
                    Vec16<WT>::unpack(*reinterpret_cast<const u32x4*>((const char*)wo + wo_at(p)), wf);
#pragma unroll
                for (int e = 0; e < EW; ++e) s = fmaf(wf[e], sm.o[(lane % LW) * EW + e], s);
                s = group_sum<LW>(s);
                const int i = (wave + WAVES * p) * RW + lane / LW;
                if (lane % LW == 0 && i < nwo) sm_put<ONE>(a, a.g_wo + h * D + hj + J * i, s, tag + 1);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (wo's rows are read)
            side ^= 1;
            // ---- x1 = x + wo, then gate/up (model.cpp:86-115)
            for (int i0 = wave * 64; i0 < D; i0 += THREADS) {
                const int i = min(i0 + lane, D - 1);
                float s = 0.0f;
                for (int h0 = 0; h0 < a.hq; h0 += 4) {
                    int off[4];
                    float v[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) off[j] = a.g_wo + min(h0 + j, a.hq - 1) * D + i;
                    sm_wait<4>(off, tag + 1, v, sm, a);
#pragma unroll
                    for (int j = 0; j < 4; ++j) s += h0 + j < a.hq ? v[j] : 0.0f;
                }
                s += sm.x[i];
                sm.x1[i] = s;
                sm.xg[i] = s * gw;
            }
            __syncthreads();
            const auto rd = rows_down(l);
            {
                sm_landed();
                gw = a.norms[(2 * l + 2) * D + di];
                rd.ask(next_lds(), lane, off_i);
                float ss = sm_squares(sm.x1, lane), inv = 0.0f;
                auto put = [&](int i, int n, float g, float u) {  // lanes 0 .. n - 1: units i .. i + n - 1
                    g *= inv, u *= inv;
                    float sg = 1.0f / (1.0f + expf(-g));  // swiglu_kernel.cpp:12
                    if (a.act_mode) sg = g * sg;
                    if (lane < n) sm_put<ONE>(a, a.g_act + item(i + lane), sg * u, tag + 2);
                };
                int i = 0;
                for (; i + 1 < nunit; i += 2) {
                    float v[4];
                    ru.template dot<2>(mine(), lane, sm.xg, i, off_d, v);
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[j] = sm_lane63(sm_sum63(v[j]));
                    if (i == 0) inv = sm_inv(sm_sum63(ss), inv_d, a.eps);
                    put(i, 2, lane == 0 ? v[0] : v[2], lane == 0 ? v[1] : v[3]);
                }
                if (i < nunit) {
                    float v[2];
                    ru.template dot<1>(mine(), lane, sm.xg, i, off_d, v);
                    v[0] = sm_sum63(v[0]), v[1] = sm_sum63(v[1]);
                    if (i == 0) inv = sm_inv(sm_sum63(ss), inv_d, a.eps);
                    put(i, 1, sm_lane63(v[0]), sm_lane63(v[1]));
                }
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                side ^= 1;
            }
            // ---- down (model.cpp:118-128)
            for (int i0 = wave * 64; i0 < I; i0 += 2 * THREADS) {
                const int u0 = min(i0 + lane, I - 1), u1 = min(i0 + THREADS + lane, I - 1), off[2] = {a.g_act + u0, a.g_act + u1};
                float v[2];
                sm_wait<2>(off, tag + 2, v, sm, a);
                sm.act[u0] = v[0], sm.act[u1] = v[1];
            }
            __syncthreads();
            sm_landed();
            if (l + 1 < a.L)
                rows_qkv(l + 1).ask(next_lds(), lane, off_qkv);
            else
                rows_head().ask(next_lds(), lane, off_d);
            for (int i = 0; i < ndown; ++i) {
                float s[1];
                rd.template dot<1>(mine(), lane, sm.act, i, off_i, s);
                s[0] = sm_sum63(s[0]);
                if (lane == 63) sm_put<ONE>(a, a.g_x + item(i), sm.x1[item(i)] + s[0], tag + 3);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            side ^= 1;
            for (int i0 = wave * 64; i0 < D; i0 += THREADS) {
                const int d = min(i0 + lane, D - 1), off[1] = {a.g_x + d};
                float v[1];
                sm_wait<1>(off, tag + 3, v, sm, a);
                sm.x[d] = v[0];
                sm.xg[d] = v[0] * gw;
            }
            __syncthreads();
        }
        // ---- final norm, LM head, argmax (model.cpp:131-148, argmax.cpp:11), next token (:157-183)
        const unsigned tag = a.tag0 + (unsigned)(step * (a.L + 1) + a.L) * 4;
        unsigned long long best = 0;
        {
            const auto rh = rows_head();
            sm_landed();
            gw = a.norms[di];
            rows_qkv(0).ask(next_lds(), lane, off_qkv);  // of the next step
            float ss = sm_squares(sm.x, lane), inv = 0.0f;
            auto take = [&](int i, float v) {  // (lane 63's)
                v *= inv;
                if (lane == 63) a.logits[item(i)] = v;
                const unsigned long long k = argmax_key(v, (unsigned)item(i));
                best = k > best ? k : best;
            };
            int i = 0;
            for (; i + 1 < nhead; i += 2) {
                float v[2];
                rh.template dot<2>(mine(), lane, sm.xg, i, off_d, v);
                v[0] = sm_sum63(v[0]), v[1] = sm_sum63(v[1]);
                if (i == 0) inv = sm_inv(sm_sum63(ss), inv_d, a.eps);
                take(i, v[0]);
                take(i + 1, v[1]);
            }
            if (i < nhead) {
                float v[1];
                rh.template dot<1>(mine(), lane, sm.xg, i, off_d, v);
                v[0] = sm_sum63(v[0]);
                if (i == 0) inv = sm_inv(sm_sum63(ss), inv_d, a.eps);
                take(i, v[0]);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            side ^= 1;
        }
        if (lane == 63) sm.key[wave] = best;
        __syncthreads();
        if (wave == 0) {
            const unsigned long long k = sm_key_max(sm.key[lane % WAVES]);
            if (lane < 2) sm_put<ONE>(a, a.g_key + 2 * wg + lane, __uint_as_float(lane ? (unsigned)(k >> 32) : (unsigned)k), tag);
            best = 0;
            for (int i0 = 0; i0 < a.nwg; i0 += 64) {
                const int i = min(i0 + lane, a.nwg - 1);
                const int off[2] = {a.g_key + 2 * i, a.g_key + 2 * i + 1};
                float v[2];
                sm_wait<2>(off, tag, v, sm, a);
                const unsigned long long k = (unsigned long long)__float_as_uint(v[1]) << 32 | __float_as_uint(v[0]);
                best = k > best ? k : best;
            }
            best = sm_key_max(best);
            if (lane == 0) sm.next = (int)argmax_key_index(best);
        }
        __syncthreads();
        next = __builtin_amdgcn_readfirstlane(sm.next);
        if (advance && pos + 1 < a.T) {
            ++pos;
            token = pos < forced ? after : next;
            if (wg == 0 && tid == 0) a.hist[pos] = token;
        }
    }
    sm_landed();  // (no DMA into this LDS is left when the workgroup ends)
    if (wg == 0 && tid == 0) {
        a.st->last_argmax = next;
        a.st->key = 0;
        a.st->pos = pos;
        a.st->token = token;
    }
}

}  // namespace sli
