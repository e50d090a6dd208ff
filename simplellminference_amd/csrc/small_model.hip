// small_model.hip — launches of the small models' greedy loop (small_model.h).
#include "small_model.h"

#include "../../include/sli.h"

namespace sli {

template <typename WT, typename KT, int HD>
static hipError_t go(const SmArgs* a, hipStream_t s) {
    auto* k = &small_predict_kernel<WT, KT, HD>;
    if (!a) return hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kSmLds);
    hipLaunchKernelGGL(k, dim3(a->nwg), dim3(kSmThreads), kSmLds, s, *a);
    return hipGetLastError();
}
template <typename WT, typename KT>
static hipError_t go_hd(const SmArgs* a, int hd, hipStream_t s) {
    return hd == 128 ? go<WT, KT, 128>(a, s) : go<WT, KT, 64>(a, s);
}
template <typename WT>
static hipError_t go_kv(const SmArgs* a, int kd, int hd, hipStream_t s) {
    return kd == SLI_DT_F32 ? go_hd<WT, float>(a, hd, s) : go_hd<WT, __half>(a, hd, s);
}
static hipError_t dispatch(const SmArgs* a, int wd, int kd, int hd, hipStream_t s) {
    return wd == SLI_DT_F32 ? go_kv<float>(a, kd, hd, s) : go_kv<__half>(a, kd, hd, s);
}
hipError_t small_allow(int wd, int kd, int hd) { return dispatch(nullptr, wd, kd, hd, nullptr); }
hipError_t small_launch(const SmArgs& a, int wd, int kd, int hd, hipStream_t s) { return dispatch(&a, wd, kd, hd, s); }

}  // namespace sli
