// The batched Z passes for the lengths of part GK_PART of GK_LEN_M (build.py
// compiles this file once per part).
#include <hip/hip_runtime.h>

#include "batch_dev.h"

#define GK_CAT2(a, b) a##b
#define GK_CAT(a, b) GK_CAT2(a, b)
#define GK_LEN_M_HERE GK_CAT(GK_LEN_M_PART, GK_PART)

namespace gk {

template <int M> void bz_fwd_run(const BLaunch& b, const BStage& sg, const float2* twM, const float2* twP) {
    constexpr int TR = z_rows_c<M>(), nt = TR * RegFFT<M>::G;
    switch (zfwd_nk(sg.nk)) {
    case 0: kb_zfwd<M, TR, 0><<<b.blocks, nt, 0, b.s>>>(b.sims, b.map, sg, twM, twP); break;
    case 1: kb_zfwd<M, TR, 1><<<b.blocks, nt, 0, b.s>>>(b.sims, b.map, sg, twM, twP); break;
    case 2: kb_zfwd<M, TR, 2><<<b.blocks, nt, 0, b.s>>>(b.sims, b.map, sg, twM, twP); break;
    case 3: kb_zfwd<M, TR, 3><<<b.blocks, nt, 0, b.s>>>(b.sims, b.map, sg, twM, twP); break;
    default: kb_zfwd<M, TR, 5><<<b.blocks, nt, 0, b.s>>>(b.sims, b.map, sg, twM, twP); break;
    }
}

template <int M, int NU, int FIN>
static void epi_launch(const BLaunch& b, const BStage& sg, const float2* twM, const float2* twP) {
    constexpr int TR = epi_rows_c<M>(), nt = 3 * TR * RegFFT<M>::G;
    kb_zinv_epi<M, TR, NU, FIN><<<b.blocks, nt, 0, b.s>>>(b.sims, b.map, sg, twM, twP);
}
template <int M> void bz_epi_run(const BLaunch& b, const BStage& sg, const float2* twM, const float2* twP) {
    if (sg.fin == 1) {
        if (sg.nu <= 1) epi_launch<M, 1, 1>(b, sg, twM, twP);
        else epi_launch<M, 3, 1>(b, sg, twM, twP);
    } else if (sg.fin == 2) {
        if (sg.nu <= 3) epi_launch<M, 3, 2>(b, sg, twM, twP);
        else epi_launch<M, 6, 2>(b, sg, twM, twP);
    } else {
        if (sg.nu == 0) epi_launch<M, 0, 0>(b, sg, twM, twP);
        else if (sg.nu == 1) epi_launch<M, 1, 0>(b, sg, twM, twP);
        else if (sg.nu <= 3) epi_launch<M, 3, 0>(b, sg, twM, twP);
        else epi_launch<M, 6, 0>(b, sg, twM, twP);
    }
}

#define GK_CASE(n)                                                                            \
    template void bz_fwd_run<n>(const BLaunch&, const BStage&, const float2*, const float2*); \
    template void bz_epi_run<n>(const BLaunch&, const BStage&, const float2*, const float2*);
GK_LEN_M_HERE(GK_CASE)
#undef GK_CASE

}  // namespace gk
