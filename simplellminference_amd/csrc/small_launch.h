// small_launch.h — what the engine and the small models' greedy loop (small_model.h, small_model.hip) share.
#pragma once
#include "common.h"
#include "step_state.h"

namespace sli {

constexpr int kSmMaxD = 512, kSmMaxI = 2048;   // model and FFN width
constexpr int kSmErrWait = 64;                 // DevState::error
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
    sm_u2 *g_qkv, *g_wo, *g_act, *g_x, *g_key;  // granules: (hq + 2 hkv) hd, hq D, I, D, 2 nwg
    unsigned tag0;         // the launch's tags are tag0 + (step (L + 1) + layer) 4 + edge (never one that was used before)
};

// dtypes: SLI_DT_F32 or SLI_DT_F16 of the weights and of the cache. small_allow: once a process and device, before a launch.
hipError_t small_allow(int wd, int kd, int hd);
hipError_t small_launch(const SmArgs& a, int wd, int kd, int hd, hipStream_t s);

}  // namespace sli
