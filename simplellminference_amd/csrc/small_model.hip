// small_model.hip — launches of the small models' greedy loop (small_model.h).
#include "small_model.h"

#include <map>
#include <mutex>

#include "../../include/sli.h"

namespace sli {

template <typename WT, typename KT, int HD, int WAVES, bool ONE, bool D1>
static hipError_t run(const SmArgs* a, hipStream_t s) {
    auto* k = &small_predict_kernel<WT, KT, HD, WAVES, ONE, D1>;
    constexpr size_t lds = SmGeo<WAVES>::LDS;
    if (!a) return hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(k, dim3(ONE ? 8 * a->nwg : a->nwg), dim3(64 * WAVES), lds, s, *a);
    return hipGetLastError();
}
// (rows of the model's width in one KiB, or not: fp32 past 256, over all XCDs only)
template <typename WT, typename KT, int HD>
static hipError_t go(const SmArgs* a, hipStream_t s) {
    constexpr bool wide = sizeof(WT) * kSmMaxD > 1024;
    if (a) {
        if (a->xcd >= 0) return run<WT, KT, HD, kSmOneWaves, true, true>(a, s);
        return wide && a->D * sizeof(WT) > 1024 ? run<WT, KT, HD, kSmWaves, false, !wide>(a, s) : run<WT, KT, HD, kSmWaves, false, true>(a, s);
    }
    hipError_t e = run<WT, KT, HD, kSmWaves, false, true>(a, s);
    if (e == hipSuccess && wide) e = run<WT, KT, HD, kSmWaves, false, !wide>(a, s);
    return e == hipSuccess ? run<WT, KT, HD, kSmOneWaves, true, true>(a, s) : e;
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


static __global__ void xcd_kernel(unsigned* count) {  // workgroups by XCC_ID
    unsigned xcc;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
    if (threadIdx.x == 0) atomicAdd(count + (xcc & 15), 1u);
}
unsigned small_xcds(int per) {
    static std::mutex mu;
    static std::map<std::pair<int, int>, unsigned> known;  // by device and per
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    std::lock_guard<std::mutex> lock(mu);
    const auto it = known.find({dev, per});
    if (it != known.end()) return it->second;
    unsigned *n = nullptr, h[16] = {}, mask = 0;
    bool asked = false;
    if (hipMalloc(&n, sizeof(h)) == hipSuccess && hipMemset(n, 0, sizeof(h)) == hipSuccess) {
        hipLaunchKernelGGL(xcd_kernel, dim3(8 * per), dim3(64), 0, nullptr, n);
        asked = hipGetLastError() == hipSuccess && hipMemcpy(h, n, sizeof(h), hipMemcpyDeviceToHost) == hipSuccess;
        for (int i = 0; asked && i < 16; ++i) mask |= h[i] == (unsigned)per ? 1u << i : 0u;
        for (int i = 0; i < 16; ++i)
            if (h[i] && h[i] != (unsigned)per) mask = 0;
    }
    if (n) (void)hipFree(n);
    (void)hipGetLastError();
    if (asked) known[{dev, per}] = mask;  // (memory that was not there may be there for the next model)
    return mask;
}

}  // namespace sli
