// small_model.h — the greedy loop of a small model (batch 1, fp32 or fp16 weights) as ONE launch: n steps of
// LlamaModel::predict (source/model/model.cpp:150-187), each the layer loop of forward (:50-129), the LM head, the argmax and
// the next token, with every dependency inside the launch.
//
// Why: a step of the 256-wide two-layer preset reads 7 MB (1 us), and its 13 graph launches of 2 to 8 us take 69. Here a step
// has four all-to-all edges a layer and one for the token, each a store and a load through memory and what a workgroup does
// between them, 3 us: 28 us a step, 36 greedy tokens in 1.0 ms instead of 2.5. The edges bound it (and, with large
// vocabularies, the head's rows: small_launch.h small_lost_us).
//
// Structure: hq J workgroups of 8 waves, all resident; every workgroup holds the whole residual row and runs every op on its
// share of the rows. An edge is 8-byte {value, tag} granules as in tp_layers.h: one sc1 store each, no flag, no drain;
// readers sweep them with sc1 loads until the tags are this edge's. Tags count (launch, step, layer, edge), so one array an
// edge serves every layer: before a workgroup writes an edge's granules again it has read a later edge to which every
// workgroup contributes (small_nwg), so nobody still reads them.
//   q, k, v rows -> the workgroups of head h: its q, its kv head's k and v
//   attention of head h over the whole context, by each of its J workgroups; at once their D / J rows of wo over that head's
//   columns -> partial sums [hq][D] -> every workgroup: x1 = x + the heads' partials in head order
//   gate/up units -> act -> every workgroup: down rows + x1 -> x
//   the workgroups' argmax keys -> every workgroup: the next token
// A wave asks for its weight rows of the next op (LDS-DMA, its own 8 KiB) before it waits for that op's input. K and V rows of
// earlier steps are read with sc1 loads: other XCDs wrote them.
// Every wait is bounded: one that gives up sets DevState::error kSmErrWait, the workgroup skips every later wait, the others'
// waits give up too and the grid drains; the host then runs the steps as launches, and every later call of the model's.
#pragma once
#include "common.h"
#include "prefill.h"
#include "small_launch.h"
#include "step_state.h"

namespace sli {

struct alignas(16) SmSmem {
    float x[kSmMaxD], x1[kSmMaxD], act[kSmMaxI];
    float qkv[3 * 128];
    float part[kSmWaves][2 + 128];  // a wave's m, l, o of the attention
    float o[kSmWaves][128];         // the head's output, a copy a wave
    unsigned long long key[kSmWaves];
    int dead;
};
constexpr size_t kSmPre = (sizeof(SmSmem) + 1023) / 1024 * 1024;
constexpr size_t kSmLds = kSmPre + (size_t)kSmWaves * kSmWaveBytes;

__device__ __forceinline__ void sm_put(sm_u2* g, int i, float v, unsigned tag) {
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(g, 0, 0x7fffffff, 0x00020000);
    __builtin_amdgcn_raw_buffer_store_b64(sm_u2{__float_as_uint(v), tag}, rs, 8u * (unsigned)i, 0, 16 /* sc1 */);
}
// N granules at element offsets off[], of a thread, until all carry `tag` (of lanes with !on: whatever they hold)
template <int N>
__device__ __forceinline__ void sm_wait(const sm_u2* g, const int (&off)[N], bool on, unsigned tag, float (&out)[N], SmSmem& sm,
                                        const SmArgs& a) {
    const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<sm_u2*>(g), 0, 0x7fffffff, 0x00020000);
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
        if (!__any(on && miss) || sm.dead) return;
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

// A wave's rows of an op: row(i), i < n, of C columns (a multiple of 8), `each` 1-KiB pieces a row; the norm weights before them (nw:
// D floats, or null). Row i's piece p lies at byte (lead + i each + p) 1024 of the wave's LDS where that is below kSmWaveBytes;
// what does not fit is loaded when it is used.
template <typename WT>
struct SmRows {
    static constexpr int E = 16 / (int)sizeof(WT);
    const WT* W;
    const float* nw;
    int C, n, each, lead;
    __device__ SmRows(const void* w, const float* nw_, int c, int n_)
        : W((const WT*)w), nw(nw_), C(c), n(n_), each((c * (int)sizeof(WT) + 1023) / 1024), lead(nw_ ? (c * 4 + 1023) / 1024 : 0) {}
    __device__ bool held(int i, int p) const { return (lead + i * each + p + 1) * 1024 <= kSmWaveBytes; }
    template <class Row>
    __device__ void ask(unsigned lds, int lane, const Row& row) const {  // (lds: the wave's)
        for (int p = 0; p < lead; ++p) pf_dma(nw + min((p * 64 + lane) * 4, C - 4), lds + p * 1024);
        for (int i = 0; i < n; ++i)
            for (int p = 0; p < each; ++p)
                if (held(i, p)) pf_dma(W + (size_t)row(i) * C + min((p * 64 + lane) * E, C - E), lds + (lead + i * each + p) * 1024);
    }
    // rows i0 .. i0 + N - 1 times x (LDS), of RMSNorm'd x where there are norm weights: (x inv) nw
    template <int N, class Row>
    __device__ void dot(const char* mine, int lane, const float* x, float inv, int i0, const Row& row, float (&s)[N]) const {
#pragma unroll
        for (int j = 0; j < N; ++j) s[j] = 0.0f;
        for (int p = 0; p < each; ++p) {
            const int c = (p * 64 + lane) * E;
            if (c >= C) continue;
            float xv[E];
#pragma unroll
            for (int e = 0; e < E; e += 4) *reinterpret_cast<float4*>(xv + e) = *reinterpret_cast<const float4*>(x + c + e);
            if (lead) {
#pragma unroll
                for (int e = 0; e < E; e += 4) {
                    const float4 g = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(mine) + c + e);
                    xv[e] = (xv[e] * inv) * g.x, xv[e + 1] = (xv[e + 1] * inv) * g.y;
                    xv[e + 2] = (xv[e + 2] * inv) * g.z, xv[e + 3] = (xv[e + 3] * inv) * g.w;
                }
            }
#pragma unroll
            for (int j = 0; j < N; ++j) {
                const u32x4 v = held(i0 + j, p) ? *reinterpret_cast<const u32x4*>(mine + (lead + (i0 + j) * each + p) * 1024 + lane * 16)
                                                : *reinterpret_cast<const u32x4*>(W + (size_t)row(i0 + j) * C + c);
                float f[E];
                Vec16<WT>::unpack(v, f);
#pragma unroll
                for (int e = 0; e < E; ++e) s[j] = fmaf(f[e], xv[e], s[j]);
            }
        }
#pragma unroll
        for (int j = 0; j < N; ++j) s[j] = wave_sum(s[j]);
    }
};

__device__ __forceinline__ float sm_rms(const float* x, int D, float eps, int lane) {  // 1 / rms (rms_kernel.cpp:12-19)
    float ss = 0.0f;
    for (int i = lane; i < D; i += 64) ss = fmaf(x[i], x[i], ss);
    ss = wave_sum(ss);
    return 1.0f / sqrtf(ss / (float)D + eps);
}
__device__ __forceinline__ void sm_landed() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

template <typename WT, typename KT, int HD>
__global__ void __launch_bounds__(kSmThreads) small_predict_kernel(SmArgs a) {
    extern __shared__ __attribute__((aligned(1024))) char sm_raw[];
    SmSmem& sm = *reinterpret_cast<SmSmem*>(sm_raw);
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wg = blockIdx.x, J = a.nwg / a.hq, h = wg / J, hj = wg - h * J, kvh = h / (a.hq / a.hkv);
    const int D = a.D, I = a.I, half = HD / 2;
    char* mine = sm_raw + kSmPre + wave * kSmWaveBytes;
    const unsigned lds = (unsigned)(uintptr_t)(const __attribute__((address_space(3))) char*)mine;
    if (tid == 0) sm.dead = 0;
    int token = a.st->token, pos = a.st->pos, next = 0;
    const int advance = a.st->advance, forced = a.st->n_forced;
    // this wave's share of every op: items wg + nwg (wave + 8 i)
    auto count = [&](int n) { return n <= wg ? 0 : ((n - wg + a.nwg - 1) / a.nwg - wave + kSmWaves - 1) / kSmWaves; };
    auto item = [&](int i) { return wg + a.nwg * (wave + kSmWaves * i); };
    const int npair = max(0, count((a.hq + 2 * a.hkv) * half)), nunit = max(0, count(I)), ndown = max(0, count(D)),
              nhead = max(0, count(a.V));
    auto pair_row = [&](int r) { const int u = item(r >> 1), uh = u / half; return uh * HD + (u - uh * half) + (r & 1) * half; };
    auto unit_row = [&](int r) { return item(r >> 1) + (r & 1) * I; };
    auto plain_row = [&](int r) { return item(r); };
    // wo: this workgroup's rows hj + J i, over head h's columns; LW lanes a row, RW rows a piece
    constexpr int EW = 16 / (int)sizeof(WT), LW = HD / EW, RW = 64 / LW;
    const int nwo = (D - hj + J - 1) / J;  // rows of the workgroup; wave w has pieces w, w + 8, ..
    const int pwo = max(0, ((nwo + RW - 1) / RW - wave + kSmWaves - 1) / kSmWaves);
    auto wo_at = [&](const void* W, int p) {
        const int i = min((wave + kSmWaves * p) * RW + lane / LW, nwo - 1);
        return (const WT*)W + (size_t)(hj + J * i) * a.hq * HD + h * HD + (lane % LW) * EW;
    };
    for (int step = 0; step < a.n; ++step) {
        const int after = a.prompt[min(pos + 1, a.T)];  // the prompt's next token, where there is one
        const bool ok = token >= 0 && token < a.V;  // (as embedding_kernel: zeros for a token that is none)
        for (int i = tid; i < D; i += kSmThreads) sm.x[i] = ok ? to_f32(((const WT*)a.emb)[(size_t)token * D + i]) : 0.0f;
        __syncthreads();
        for (int l = 0; l < a.L; ++l) {
            const unsigned tag = a.tag0 + (unsigned)(step * (a.L + 1) + l) * 4;
            const void* const* w = a.w + 4 * l;
            KT* kc = (KT*)a.kc + (size_t)l * a.hkv * a.T * HD;
            KT* vc = (KT*)a.vc + (size_t)l * a.hkv * a.T * HD;
            {  // q, k, v (model.cpp:52-67)
                const SmRows<WT> r(w[0], a.norms + (size_t)(2 * l) * D, D, 2 * npair);
                r.ask(lds, lane, pair_row);
                auto turn = [&](const float* t, int i) { const int u = item(i); return t[pos * half + u % half]; };
                float fci = npair ? turn(a.sin_t, 0) : 0.0f, fcr = npair ? turn(a.cos_t, 0) : 0.0f;
                const float inv = sm_rms(sm.x, D, a.eps, lane);
                sm_landed();
                for (int i = 0; i < npair; ++i) {
                    float v2[2];
                    r.template dot<2>(mine, lane, sm.x, inv, 2 * i, pair_row, v2);
                    const int u = item(i), uh = u / half, d = u - uh * half;
                    if (uh < a.hq + a.hkv) {  // rope_kernel.cpp:30-38
                        const float r0 = v2[0] * fcr - v2[1] * fci, r1 = v2[1] * fcr + v2[0] * fci;
                        v2[0] = r0, v2[1] = r1;
                    }
                    if (i + 1 < npair) fci = turn(a.sin_t, i + 1), fcr = turn(a.cos_t, i + 1);
                    if (lane < 2) {
                        const float v = lane ? v2[1] : v2[0];
                        const int e = d + lane * half;
                        const int kh = uh - a.hq, vh = kh - a.hkv;
                        const KT kv = from_f32<KT>(v);
                        if (kh >= 0) {
                            KT* to = (vh >= 0 ? vc + ((size_t)vh * a.T + pos) * HD : kc + ((size_t)kh * a.T + pos) * HD) + e;
                            if constexpr (sizeof(KT) == 4)
                                __hip_atomic_store((unsigned*)to, __builtin_bit_cast(unsigned, kv), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            else
                                __hip_atomic_store((unsigned short*)to, __builtin_bit_cast(unsigned short, kv), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        }
                        // (k and v as the cache holds them)
                        sm_put(a.g_qkv, uh * HD + e, kh >= 0 ? to_f32<KT>(kv) : v, tag);
                    }
                }
            }
            // ---- attention of head h (mha_kernel.cpp:36-77) and its columns of wo
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (the last op's rows are read)
            for (int p = 0; p < pwo; ++p)
                if ((p + 1) * 1024 <= kSmWaveBytes) pf_dma(wo_at(w[1], p), lds + p * 1024);
            constexpr int EK = 16 / (int)sizeof(KT), LK = HD / EK, NG = kSmThreads / LK;  // lanes a key row, keys a pass
            const int grp = tid / LK, c0 = (lane % LK) * EK;
            const auto rk = __builtin_amdgcn_make_buffer_rsrc(kc + (size_t)kvh * a.T * HD, 0, 0x7fffffff, 0x00020000);
            const auto rv = __builtin_amdgcn_make_buffer_rsrc(vc + (size_t)kvh * a.T * HD, 0, 0x7fffffff, 0x00020000);
            auto key_at = [&](int t) { return (unsigned)((min(t, pos) * HD + c0) * (int)sizeof(KT)); };
            u32x4 kn = __builtin_amdgcn_raw_buffer_load_b128(rk, key_at(grp), 0, 16), vn = __builtin_amdgcn_raw_buffer_load_b128(rv, key_at(grp), 0, 16);
            if (tid < 3 * HD || HD == 128) {
                const int i = min(tid, 3 * HD - 1);
                const int off[1] = {i < HD ? h * HD + i : i < 2 * HD ? (a.hq + kvh) * HD + i - HD : (a.hq + a.hkv + kvh) * HD + i - 2 * HD};
                float v[1];
                sm_wait<1>(a.g_qkv, off, true, tag, v, sm, a);
                sm.qkv[i] = v[0];
            }
            __syncthreads();
            float q[EK], o[EK], mx = -INFINITY, lsum = 0.0f;
#pragma unroll
            for (int e = 0; e < EK; ++e) q[e] = sm.qkv[c0 + e], o[e] = 0.0f;
            for (int t0 = 0; t0 <= pos; t0 += NG) {
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
            // the wave's groups, then the waves
            float M = mx;
#pragma unroll
            for (int x = LK; x < 64; x <<= 1) M = fmaxf(M, __shfl_xor(M, x));
            const float f = mx == -INFINITY ? 0.0f : expf(mx - M);
            lsum *= f;
#pragma unroll
            for (int x = LK; x < 64; x <<= 1) lsum += __shfl_xor(lsum, x);
#pragma unroll
            for (int e = 0; e < EK; ++e) {
                o[e] *= f;
#pragma unroll
                for (int x = LK; x < 64; x <<= 1) o[e] += __shfl_xor(o[e], x);
            }
            if (lane < LK) {
#pragma unroll
                for (int e = 0; e < EK; ++e) sm.part[wave][2 + c0 + e] = o[e];
            }
            if (lane == 0) sm.part[wave][0] = M, sm.part[wave][1] = lsum;
            __syncthreads();
            {
                float mw = -INFINITY, lw = 0.0f, f8[kSmWaves];
#pragma unroll
                for (int v = 0; v < kSmWaves; ++v) mw = fmaxf(mw, sm.part[v][0]);
#pragma unroll
                for (int v = 0; v < kSmWaves; ++v) {
                    f8[v] = sm.part[v][0] == -INFINITY ? 0.0f : expf(sm.part[v][0] - mw);
                    lw = fmaf(sm.part[v][1], f8[v], lw);
                }
                const float inv = 1.0f / lw;
#pragma unroll
                for (int d = lane; d < HD; d += 64) {
                    float s = 0.0f;
#pragma unroll
                    for (int v = 0; v < kSmWaves; ++v) s = fmaf(sm.part[v][2 + d], f8[v], s);
                    sm.o[wave][d] = s * inv;
                }
            }
            sm_landed();  // (wo's pieces; the K / V row of this step is out too, for the steps after)
            for (int p = 0; p < pwo; ++p) {
                const u32x4 v = (p + 1) * 1024 <= kSmWaveBytes ? *reinterpret_cast<const u32x4*>(mine + p * 1024 + lane * 16)
                                                               : *reinterpret_cast<const u32x4*>(wo_at(w[1], p));
                float wf[EW], s = 0.0f;
                Vec16<WT>::unpack(v, wf);
#pragma unroll
                for (int e = 0; e < EW; ++e) s = fmaf(wf[e], sm.o[wave][(lane % LW) * EW + e], s);
                s = group_sum<LW>(s);
                const int i = (wave + kSmWaves * p) * RW + lane / LW;
                if (lane % LW == 0 && i < nwo) sm_put(a.g_wo, h * D + hj + J * i, s, tag + 1);
            }
            // ---- x1 = x + wo, then gate/up (model.cpp:86-115)
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            const SmRows<WT> ru(w[2], a.norms + (size_t)(2 * l + 1) * D, D, 2 * nunit);
            ru.ask(lds, lane, unit_row);
            for (int i0 = 0; i0 < D; i0 += kSmThreads) {
                const int i = min(i0 + tid, D - 1);
                float s = 0.0f;
                for (int h0 = 0; h0 < a.hq; h0 += 4) {
                    int off[4];
                    float v[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) off[j] = min(h0 + j, a.hq - 1) * D + i;
                    sm_wait<4>(a.g_wo, off, true, tag + 1, v, sm, a);
#pragma unroll
                    for (int j = 0; j < 4; ++j) s += h0 + j < a.hq ? v[j] : 0.0f;
                }
                sm.x1[i] = sm.x[i] + s;
            }
            __syncthreads();
            {
                const float inv = sm_rms(sm.x1, D, a.eps, lane);
                sm_landed();
                for (int i = 0; i < nunit; ++i) {
                    float gu[2];
                    ru.template dot<2>(mine, lane, sm.x1, inv, 2 * i, unit_row, gu);
                    float sg = 1.0f / (1.0f + expf(-gu[0]));  // swiglu_kernel.cpp:12
                    if (a.act_mode) sg = gu[0] * sg;
                    if (lane == 0) sm_put(a.g_act, item(i), sg * gu[1], tag + 2);
                }
            }
            // ---- down (model.cpp:118-128)
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            const SmRows<WT> rd(w[3], nullptr, I, ndown);
            rd.ask(lds, lane, plain_row);
            for (int i0 = 0; i0 < I; i0 += 2 * kSmThreads) {
                const int off[2] = {min(i0 + tid, I - 1), min(i0 + kSmThreads + tid, I - 1)};
                float v[2];
                sm_wait<2>(a.g_act, off, true, tag + 2, v, sm, a);
                sm.act[off[0]] = v[0], sm.act[off[1]] = v[1];
            }
            __syncthreads();
            sm_landed();
            for (int i = 0; i < ndown; ++i) {
                float s[1];
                rd.template dot<1>(mine, lane, sm.act, 1.0f, i, plain_row, s);
                if (lane == 0) sm_put(a.g_x, item(i), sm.x1[item(i)] + s[0], tag + 3);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            for (int i0 = 0; i0 < D; i0 += kSmThreads) {
                const int off[1] = {min(i0 + tid, D - 1)};
                float v[1];
                sm_wait<1>(a.g_x, off, true, tag + 3, v, sm, a);
                sm.x[off[0]] = v[0];
            }
            __syncthreads();
        }
        // ---- final norm, LM head, argmax (model.cpp:131-148, argmax.cpp:11), next token (:157-183)
        const unsigned tag = a.tag0 + (unsigned)(step * (a.L + 1) + a.L) * 4;
        unsigned long long best = 0;
        {
            const SmRows<WT> r(a.emb, a.norms + (size_t)(2 * a.L) * D, D, nhead);
            r.ask(lds, lane, plain_row);
            const float inv = sm_rms(sm.x, D, a.eps, lane);
            sm_landed();
            for (int i = 0; i < nhead; ++i) {
                float v[1];
                r.template dot<1>(mine, lane, sm.x, inv, i, plain_row, v);
                if (lane == 0) a.logits[item(i)] = v[0];
                const unsigned long long k = argmax_key(v[0], (unsigned)item(i));
                best = k > best ? k : best;
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        if (lane == 0) sm.key[wave] = best;
        __syncthreads();
        if (tid < 2) {
#pragma unroll
            for (int v = 0; v < kSmWaves; ++v) best = sm.key[v] > best ? sm.key[v] : best;
            sm_put(a.g_key, 2 * wg + tid, __uint_as_float(tid ? (unsigned)(best >> 32) : (unsigned)best), tag);
        }
        best = 0;
        for (int i0 = 0; i0 < a.nwg; i0 += 64) {  // (every wave for itself)
            const int i = min(i0 + lane, a.nwg - 1);
            const int off[2] = {2 * i, 2 * i + 1};
            float v[2];
            sm_wait<2>(a.g_key, off, true, tag, v, sm, a);
            const unsigned long long k = (unsigned long long)__float_as_uint(v[1]) << 32 | __float_as_uint(v[0]);
            best = k > best ? k : best;
        }
        next = (int)argmax_key_index(wave_max_u64(best));
        if (advance && pos + 1 < a.T) {
            ++pos;
            token = pos < forced ? after : next;
            if (wg == 0 && tid == 0) a.hist[pos] = token;
        }
    }
    if (wg == 0 && tid == 0) {
        a.st->last_argmax = next;
        a.st->key = 0;
        a.st->pos = pos;
        a.st->token = token;
    }
}

}  // namespace sli
