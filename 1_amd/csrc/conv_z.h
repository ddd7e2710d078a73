// Block shapes of the Z passes and the launchers of their kernels, which are
// compiled in parts (conv_z.hip: one translation unit per GK_LEN_M_PART*).
#pragma once
#include "engine.h"
#include "passes.h"

namespace gk {

// rows per Z block: enough consecutive y for 64-128 B transposed segments, at most 1024 threads
template <int M> constexpr int z_rows() {
    constexpr int G = RegFFT<M>::G;
    int tr = 1024 / G;
    if (tr > 16) tr = 16;
    while (tr > 1 && tr * (M + 1) * 8 > 72 * 1024) tr /= 2;
    return tr;
}

// rows per Z forward block of shape variant v: 0 and 4 the length's own, 1 half of
// them, 2 double (while the block stays within 1024 threads and 80 KB of LDS), 3 a
// quarter.  Short rows (M < 32) have one shape; a variant that does not exist gives
// the length's own.  (A plan's variant 0 is the one grid_rows chose, conv.hip; 4 and
// the Z inverse's 3 ask for the length's own rows on any grid.)
template <int M> constexpr int z_rows_v(int v) {
    constexpr int d = z_rows<M>();
    if (M < 32) return d;
    if (v == 1) return d > 1 ? d / 2 : d;
    if (v == 2) {
        const int t = 2 * d;
        const int fft = t * RegFFT<M>::LDS, tile = (M + 1) * (t + 1);
        return (t * RegFFT<M>::G <= 1024 && (fft > tile ? fft : tile) * 8 <= 80 * 1024) ? t : d;
    }
    if (v == 3) return d >= 16 ? d / 4 : d;  // small grids: more blocks
    return d;
}

// rows per block of the fused Z inverse: 3 x TR lane groups <= 1024 threads, its
// LDS (transposed tiles, FFT exchange buffers) within 80 KB (two blocks per CU)
template <int M> constexpr int epi_rows() {
    constexpr int G = RegFFT<M>::G;
    int tr = 1024 / (3 * G);
    if (tr > 16) tr = 16;
    int p = 1;
    while (p * 2 <= tr) p *= 2;
    tr = p;
    // two blocks per CU (80 KB of LDS), except for long rows that this would leave
    // with two rows per block and 16 B runs of B1
    const int cap = M >= 1024 ? 150 * 1024 : 80 * 1024;
    while (tr > 1 && zinv_epi_lds_elems(M, tr) * 8 > cap) tr /= 2;
    return tr;
}

// rows per fused Z inverse block of shape variant v: 0 and 3 the length's own, 1
// half of them, 2 two rows (where that is less than half; small grids: more blocks)
template <int M> constexpr int epi_rows_v(int v) {
    constexpr int d = epi_rows<M>();
    if (M < 32) return d;
    if (v == 2) return d > 4 ? 2 : d;
    return (v == 1 && d > 1) ? d / 2 : d;
}

// lengths whose fused Z inverse can end with the next stage's Z forward (a block of
// longer rows has two of them, whose 16 B runs of B1 would make the stores partial lines)
constexpr bool z_fwd_fused(int M) { return M >= 2 && M <= 1024; }

template <int M>
void zfwd_run(const ConvPlan& cp, const StageIn& si, int NKp, const float2* twM, const float2* twP, hipStream_t s);
template <int M>
void zinv_run(const ConvPlan& cp, float* h, const EngineState* st, const float2* twM, const float2* twP, hipStream_t s);
template <int M>
void zinv_epi_run(const ConvPlan& cp, const EpiArgs& e, const EngineState* st, const float2* twM, const float2* twP,
                  hipStream_t s);

}  // namespace gk
