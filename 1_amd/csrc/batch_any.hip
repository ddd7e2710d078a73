// The batched engine's length-dispatch kernels.  build.py compiles this file in
// parts: 0 the Z forward, 1 the Z inverse of the inner stages, 2 of the last
// stages, 3 the Y and X passes.
#include <hip/hip_runtime.h>

#include <mutex>

#include "batch_dev.h"

namespace gk {

template <typename F> static void any_attr(F* f) {
    GK_CHECK(hipFuncSetAttribute((const void*)f, hipFuncAttributeMaxDynamicSharedMemorySize, kAnyLds));
}
#define GK_ANY_LAUNCH(kern) kern<<<b.blocks, b.nt, b.lds, b.s>>>(b.sims, b.map, sg)

#if GK_PART == 0

template <int NK>
__global__ __launch_bounds__(1024) void kb_zfwd_any(const BSim* sims, const int2* map,
                                                    BStage sg) {
    extern __shared__ float2 dyn[];
    const BBlock bb = bblock(sims, map);
    const BSim& d = *bb.d;
    if (bskip(d, sg)) return;
    switch (d.Q - 1) {
#define GK_CASE(m)                                    \
    case m: {                                         \
        constexpr int TR = z_rows_c<m>();             \
        if (threadIdx.x >= TR * RegFFT<m>::G) return; \
        bz_fwd<m, TR, NK>(d, bb.lb, sg, d.twM, d.twP, \
                          dyn);                       \
        break;                                        \
    }
        GK_ANY_M(GK_CASE)
#undef GK_CASE
    }
}

void any_zfwd(const BLaunch& b, const BStage& sg) {
    switch (zfwd_nk(sg.nk)) {
    case 0: GK_ANY_LAUNCH(kb_zfwd_any<0>); break;
    case 1: GK_ANY_LAUNCH(kb_zfwd_any<1>); break;
    case 2: GK_ANY_LAUNCH(kb_zfwd_any<2>); break;
    case 3: GK_ANY_LAUNCH(kb_zfwd_any<3>); break;
    default: GK_ANY_LAUNCH(kb_zfwd_any<5>); break;
    }
}
void any_attr_zfwd() {
    any_attr(kb_zfwd_any<0>);
    any_attr(kb_zfwd_any<1>);
    any_attr(kb_zfwd_any<2>);
    any_attr(kb_zfwd_any<3>);
    any_attr(kb_zfwd_any<5>);
}

#elif GK_PART <= 2

// (96 registers, 5 waves per SIMD; the last stage of an adaptive tableau, with six
// earlier stages and their FP64 errors, would spill: 91 us, 136 with the bound)
template <int NU, int FIN>
__global__ __launch_bounds__(768) __attribute__((amdgpu_waves_per_eu(FIN == 2 ? 1 : 5))) void kb_zinv_any(
    const BSim* sims, const int2* map, BStage sg) {
    extern __shared__ float2 dyn[];
    const BBlock bb = bblock(sims, map);
    const BSim& d = *bb.d;
    if (bskip(d, sg)) return;
    switch (d.Q - 1) {
#define GK_CASE(m)                                                                   \
    case m: {                                                                        \
        constexpr int TR = epi_rows_any<m>(), NT = 3 * TR * RegFFT<m>::G;            \
        if (threadIdx.x >= NT) return;                                               \
        float* hext_s = reinterpret_cast<float*>(dyn + zinv_epi_lds<m, TR>());       \
        bz_inv<m, TR, NU, FIN>(d, bb.lb, sg, d.twM, d.twP, dyn, hext_s, hext_s + 4); \
        break;                                                                       \
    }
        GK_ANY_M(GK_CASE)
#undef GK_CASE
    }
}

#if GK_PART == 1
void any_zinv(const BLaunch& b, const BStage& sg) {
    if (sg.nu == 0) GK_ANY_LAUNCH((kb_zinv_any<0, 0>));
    else if (sg.nu == 1) GK_ANY_LAUNCH((kb_zinv_any<1, 0>));
    else if (sg.nu <= 3) GK_ANY_LAUNCH((kb_zinv_any<3, 0>));
    else GK_ANY_LAUNCH((kb_zinv_any<6, 0>));
}
void any_attr_zinv() {
    any_attr(kb_zinv_any<0, 0>);
    any_attr(kb_zinv_any<1, 0>);
    any_attr(kb_zinv_any<3, 0>);
    any_attr(kb_zinv_any<6, 0>);
}
#else
void any_zinv_fin(const BLaunch& b, const BStage& sg) {
    if (sg.fin == 1) {
        if (sg.nu <= 1) GK_ANY_LAUNCH((kb_zinv_any<1, 1>));
        else GK_ANY_LAUNCH((kb_zinv_any<3, 1>));
    } else {
        if (sg.nu <= 3) GK_ANY_LAUNCH((kb_zinv_any<3, 2>));
        else GK_ANY_LAUNCH((kb_zinv_any<6, 2>));
    }
}
void any_attr_zinv_fin() {
    any_attr(kb_zinv_any<1, 1>);
    any_attr(kb_zinv_any<3, 1>);
    any_attr(kb_zinv_any<3, 2>);
    any_attr(kb_zinv_any<6, 2>);
}
#endif

#else

__global__ __launch_bounds__(kYxyThreads) void kb_yxy_any(const BSim* sims, const int2* map,
                                                          BStage sg) {
    extern __shared__ float2 dyn[];
    const BBlock bb = bblock(sims, map);
    const BSim& d = *bb.d;
    if (bskip(d, sg)) return;
    if (d.PX == 4) {
        switch (d.PY) {
#define GK_CASE(py)     case py: if constexpr (yxy_fits(4, py)) b_yxy<py, 4>(d, bb.lb, d.twY, d.twX, dyn); break;
            GK_ANY_Y(GK_CASE)
#undef GK_CASE
        }
    } else {
        switch (d.PY) {
#define GK_CASE(py)     case py: if constexpr (yxy_fits(8, py)) b_yxy<py, 8>(d, bb.lb, d.twY, d.twX, dyn); break;
            GK_ANY_Y(GK_CASE)
#undef GK_CASE
        }
    }
}

__global__ __launch_bounds__(Y2<1024>::NT) void kb_y2r_any(const BSim* sims, const int2* map,
                                                  BStage sg) {
    extern __shared__ float2 dyn[];
    const BBlock bb = bblock(sims, map);
    const BSim& d = *bb.d;
    if (bskip(d, sg)) return;
    switch (d.PY) {
#define GK_CASE(py)                                 \
    case py:                                        \
        if (threadIdx.x >= Y2<py>::NT) return;      \
        b_y2r<py>(d, bb.lb, d.twY, dyn);            \
        break;
        GK_ANY_Y(GK_CASE)
#undef GK_CASE
    }
}

template <bool FWD>
__global__ __launch_bounds__(kNT) void kb_ypass_any(const BSim* sims, const int2* map,
                                                    BStage sg) {
    extern __shared__ float2 dyn[];
    const BBlock bb = bblock(sims, map);
    const BSim& d = *bb.d;
    if (bskip(d, sg)) return;
    switch (d.PY) {
#define GK_CASE(py) \
    case py: b_ypass<py, FWD>(d, bb.lb, d.twY, dyn); break;
        GK_ANY_Y(GK_CASE)
#undef GK_CASE
    }
}

__global__ __launch_bounds__(kNT) void kb_xmul_any(const BSim* sims, const int2* map,
                                                   BStage sg) {
    extern __shared__ float2 dyn[];
    const BBlock bb = bblock(sims, map);
    const BSim& d = *bb.d;
    if (bskip(d, sg)) return;
    switch (d.PX) {
#define GK_CASE(px) \
    case px: b_xmul<px>(d, bb.lb, d.twX, dyn); break;
        GK_ANY_X(GK_CASE)
#undef GK_CASE
    }
}

void any_y2r(const BLaunch& b, const BStage& sg) { GK_ANY_LAUNCH(kb_y2r_any); }
void any_yxy(const BLaunch& b, const BStage& sg) { GK_ANY_LAUNCH(kb_yxy_any); }
void any_ypass(const BLaunch& b, const BStage& sg, bool fwd) {
    if (fwd) GK_ANY_LAUNCH(kb_ypass_any<true>);
    else GK_ANY_LAUNCH(kb_ypass_any<false>);
}
void any_xmul(const BLaunch& b, const BStage& sg) { GK_ANY_LAUNCH(kb_xmul_any); }
void any_attr_y() {
    any_attr(kb_yxy_any);
    any_attr(kb_y2r_any);
    any_attr(kb_ypass_any<true>);
    any_attr(kb_ypass_any<false>);
    any_attr(kb_xmul_any);
}

#endif

}  // namespace gk
