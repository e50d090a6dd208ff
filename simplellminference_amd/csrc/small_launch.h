// small_launch.h — what the engine and the small models' greedy loop (small_model.h, small_model.hip) share.
#pragma once
#include "common.h"
#include "step_state.h"

namespace sli {

constexpr int kSmMaxD = 512, kSmMaxI = 2048;   // model and FFN width
constexpr int kSmWaves = 8, kSmOneWaves = 16;   // waves of a workgroup, over all XCDs and on one
constexpr int kSmRowBytes = 65536;              // weights of an op that a workgroup asks for ahead
constexpr int kSmErrWait = 64;                 // DevState::error
constexpr unsigned kSmSpin = 1u << 20;         // sweeps of one wait before it gives up
typedef unsigned sm_u2 __attribute__((ext_vector_type(2)));

struct SmArgs {
    int D, hq, hkv, hd, I, L, T, V, nwg, act_mode, n;
    float eps, scale;
    const void* const* w;  // [L][4] device table: qkv [(hq + 2 hkv) hd][D], wo [D][hq hd], gu [2 I][D], down [D][I]
    const void* emb;       // [V][D], the LM head too
    const float* norms;    // [2 L + 1][D]
    void *kc, *vc;         // [L][hkv][T][hd]
    const float *sin_t, *cos_t;  // [T][hd / 2]
    DevState* st;
    const int32_t* prompt;
    int32_t* hist;
    float* logits;
    sm_u2* g;                         // granules of q, k, v, (hq + 2 hkv) hd; then, from these on,
    int g_wo, g_act, g_x, g_key;      // hq D, I, D and 2 nwg
    unsigned spin, look;   // kSmSpin; a wait looks up from its sweeps every look + 1 of them (a power of two)
    // xcd >= 0: the launch runs on this XCD alone, its workgroups take their numbers from ticket[turn], and ticket[1 - turn] is left
    // zero for the next one
    int xcd, turn;
    unsigned* ticket;
    unsigned tag0;         // the launch's tags are tag0 + (step (L + 1) + layer) 4 + edge (never one that was used before)
};

// us a step that the launch loses to rows which a wave cannot ask for ahead: it waits for each in turn, a head row of `each` KiB
// 0.5 + 0.4 each, a gate/up pair 2.9. 256-wide fp32, two layers, us a step as launches | here: 512 tokens of vocabulary 69 | 26, 16384
// 72 | 44, 32000 74 | 71, 128256 94 | 205; 512-wide 69 | 31, 75 | 67, 79 | 100, 109 | 371; 320-wide with 2048 units, 3 layers 92 | 96
// (the KiB of the norm weights off what is asked for ahead: the fit).
inline float small_lost_us(int D, int I, int L, int V, int wbytes, int nwg) {
    const int each = (D * wbytes + 1023) / 1024, ahead = kSmRowBytes / kSmWaves / 1024 - (D * 4 + 1023) / 1024, waves = nwg * kSmWaves;
    auto late = [&](int items, int rows) {
        const int n = (items + waves - 1) / waves - ahead / (rows * each);
        return (float)(n > 0 ? n : 0);
    };
    return late(V, 1) * (0.5f + 0.4f * each) + L * 2.9f * late(I, 2);
}

// dtypes: SLI_DT_F32 or SLI_DT_F16 of the weights and of the cache. small_allow: once a process and device, before a launch.
hipError_t small_allow(int wd, int kd, int hd);
hipError_t small_launch(const SmArgs& a, int wd, int kd, int hd, hipStream_t s);
// The current device's XCDs that take every eighth workgroup of a launch, `per` of 8 per workgroups each (their XCC_IDs as a mask; 0:
// it is not so). Asked of the device once for each `per`.
unsigned small_xcds(int per);

}  // namespace sli
