// The Z passes of the single-simulation convolution for the lengths of part
// GK_PART of GK_LEN_M (build.py compiles this file once per part).
#include <hip/hip_runtime.h>

#include "conv_z.h"

#define GK_CAT2(a, b) a##b
#define GK_CAT(a, b) GK_CAT2(a, b)
#define GK_LEN_M_HERE GK_CAT(GK_LEN_M_PART, GK_PART)

namespace gk {

template <int M, int TR>
static void zfwd_launch(const ConvPlan& cp, const StageIn& si, int NKp, const float2* twM, const float2* twP,
                        hipStream_t s) {
    const int Nx = cp.N[0], Ny = cp.N[1], Nz = cp.N[2];
    const dim3 g(div_up(Ny, TR), Nx, 3);
    constexpr int nt = TR * RegFFT<M>::G;
    switch (NKp) {
    case 0: k_zfwd<M, TR, 0><<<g, nt, 0, s>>>(si, cp.B1, twM, twP, Nx, Ny, Nz); break;
    case 1: k_zfwd<M, TR, 1><<<g, nt, 0, s>>>(si, cp.B1, twM, twP, Nx, Ny, Nz); break;
    case 2: k_zfwd<M, TR, 2><<<g, nt, 0, s>>>(si, cp.B1, twM, twP, Nx, Ny, Nz); break;
    case 3: k_zfwd<M, TR, 3><<<g, nt, 0, s>>>(si, cp.B1, twM, twP, Nx, Ny, Nz); break;
    default: k_zfwd<M, TR, 5><<<g, nt, 0, s>>>(si, cp.B1, twM, twP, Nx, Ny, Nz); break;
    }
}

template <int M, int TR>
static void zinv_epi_launch(const ConvPlan& cp, const EpiArgs& e, const EngineState* st, const float2* twM,
                            const float2* twP, hipStream_t s) {
    const int Nx = cp.N[0], Ny = cp.N[1], Nz = cp.N[2], nu = e.nu;
    const dim3 g(div_up(Ny, TR), Nx), b(3 * TR * RegFFT<M>::G);
    if constexpr (z_fwd_fused(M))
        if (e.nx >= 0) {
#define GK_ZX(NU, FIN, NX) k_zinv_epi<M, TR, NU, FIN, NX><<<g, b, 0, s>>>(cp.B1, e, twM, twP, st, Nx, Ny, Nz)
            if (e.fin == 1) {
                if (nu <= 1) GK_ZX(1, 1, 0);
                else GK_ZX(3, 1, 0);
            } else if (nu == 0) {
                if (e.nx == 0) GK_ZX(0, 0, 0);
                else GK_ZX(0, 0, 4);
            } else {
                if (e.nx == 0) GK_ZX(1, 0, 0);
                else if (e.nx == 1) GK_ZX(1, 0, 1);
                else GK_ZX(1, 0, 4);
            }
#undef GK_ZX
            return;
        }
    if (e.fin == 1) {
        if (nu <= 1) k_zinv_epi<M, TR, 1, 1><<<g, b, 0, s>>>(cp.B1, e, twM, twP, st, Nx, Ny, Nz);
        else k_zinv_epi<M, TR, 3, 1><<<g, b, 0, s>>>(cp.B1, e, twM, twP, st, Nx, Ny, Nz);
    } else if (e.fin == 2) {
        if (nu <= 3) k_zinv_epi<M, TR, 3, 2><<<g, b, 0, s>>>(cp.B1, e, twM, twP, st, Nx, Ny, Nz);
        else k_zinv_epi<M, TR, 6, 2><<<g, b, 0, s>>>(cp.B1, e, twM, twP, st, Nx, Ny, Nz);
    } else {
        if (nu == 0) k_zinv_epi<M, TR, 0, 0><<<g, b, 0, s>>>(cp.B1, e, twM, twP, st, Nx, Ny, Nz);
        else if (nu == 1) k_zinv_epi<M, TR, 1, 0><<<g, b, 0, s>>>(cp.B1, e, twM, twP, st, Nx, Ny, Nz);
        else if (nu <= 3) k_zinv_epi<M, TR, 3, 0><<<g, b, 0, s>>>(cp.B1, e, twM, twP, st, Nx, Ny, Nz);
        else k_zinv_epi<M, TR, 6, 0><<<g, b, 0, s>>>(cp.B1, e, twM, twP, st, Nx, Ny, Nz);
    }
}

template <int M>
void zfwd_run(const ConvPlan& cp, const StageIn& si, int NKp, const float2* twM, const float2* twP, hipStream_t s) {
    if (cp.zr() == 1) zfwd_launch<M, z_rows_v<M>(1)>(cp, si, NKp, twM, twP, s);
    else if (cp.zr() == 2) zfwd_launch<M, z_rows_v<M>(2)>(cp, si, NKp, twM, twP, s);
    else if (cp.zr() == 3) zfwd_launch<M, z_rows_v<M>(3)>(cp, si, NKp, twM, twP, s);
    else zfwd_launch<M, z_rows_v<M>(0)>(cp, si, NKp, twM, twP, s);
}

template <int M>
void zinv_run(const ConvPlan& cp, float* h, const EngineState* st, const float2* twM, const float2* twP, hipStream_t s) {
    constexpr int TR = z_rows<M>();
    const int Nx = cp.N[0], Ny = cp.N[1], Nz = cp.N[2];
    k_zinv<M, TR><<<dim3(div_up(Ny, TR), Nx, 3), TR * RegFFT<M>::G, 0, s>>>(cp.B1, h, twM, twP, st, Nx, Ny, Nz);
}

template <int M>
void zinv_epi_run(const ConvPlan& cp, const EpiArgs& e, const EngineState* st, const float2* twM, const float2* twP,
                  hipStream_t s) {
    if (cp.er() == 1) zinv_epi_launch<M, epi_rows_v<M>(1)>(cp, e, st, twM, twP, s);
    else if (cp.er() == 2) zinv_epi_launch<M, epi_rows_v<M>(2)>(cp, e, st, twM, twP, s);
    else zinv_epi_launch<M, epi_rows_v<M>(0)>(cp, e, st, twM, twP, s);
}

#define GK_CASE(n)                                                                                            \
    template void zfwd_run<n>(const ConvPlan&, const StageIn&, int, const float2*, const float2*, hipStream_t); \
    template void zinv_run<n>(const ConvPlan&, float*, const EngineState*, const float2*, const float2*,        \
                              hipStream_t);                                                                   \
    template void zinv_epi_run<n>(const ConvPlan&, const EpiArgs&, const EngineState*, const float2*,          \
                                  const float2*, hipStream_t);
GK_LEN_M_HERE(GK_CASE)
#undef GK_CASE

}  // namespace gk
