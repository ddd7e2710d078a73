// Device table and kernels of the batched engine (batch.hip), shared by the
// translation units its kernels are compiled in (batch_z.hip, batch_any.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "engine.h"
#include "passes.h"

namespace gk {

// one simulation of a batch, as the batched kernels see it (device table)
struct BSim {
    int Nx, Ny, Nz, Q, PY, PX;
    long N;
    float* m;
    float* mi;  // stage input stored by the Z forward pass (BStage::use_mi)
    float* k[7];
    float* mtmp;
    float2* B1;
    float2* B2;
    const float* Kc;
    EngineState* st;
    float* part;  // 3 x npart: |k0|, |k_last|, error
    int npart;
    int nfin;     // blocks of the RK final (error partials)
    TorqueArgs t; // c and part are set per stage
    CtrlParams cp;
    // twiddle tables of the simulation's lengths (the length-dispatch kernels)
    const float2* twM;  // Z half length M
    const float2* twP;  // Z padded length 2M
    const float2* twY;  // padded Y
    const float2* twX;  // padded X
    FastDiv dx, dq;     // by Nx and Q (3-D Y passes)
};

// one RK stage, the same for every simulation of the batch
struct BStage {
    int i;
    int fsal0;  // stage 0 of an FSAL tableau: simulations holding an FSAL k skip the convolution
    int nk;
    int kj[6];
    float a[6];
    int nu;
    int uj[6];
    float ua[6], ub[6];
    float bs;
    int fin;             // epilogue mode (zinv_epi_tile's FIN)
    int use_mi;          // the Z forward pass stores m_i, the epilogue reads it (nu = 0)
    double ce[6], ce_self;  // fin == 2: b2_j - b_j of the slots and of this stage
    float c, cmax;
    int partslot;  // -1: none, 0: |k0|, 1: |k_last|
};

// The simulation of this block and the block's index within it, from the launch's
// table of one int2 per block.  (A binary search over the simulations' first
// blocks took log2(n) dependent loads at the start of every block, of a few
// hundred ns each, where the pass itself takes a few us: a 40-member
// sweep of Dormand-Prince steps 6694 us, 6625 with the table.)
struct BBlock {
    const BSim* d;
    int lb;
};
__device__ __forceinline__ BBlock bblock(const BSim* sims, const int2* map) {
    const int2 e = map[blockIdx.x];
    return BBlock{sims + e.x, e.y};
}
__device__ __forceinline__ bool bskip(const BSim& d, const BStage& sg) {
    return !d.st->trial_active || (sg.fsal0 && d.st->fsal_init);
}

// ------------------------------------------------------------------ passes
// The bodies of the batched passes: block lb of simulation d.  The per-length
// kernels (kb_*) and the length-dispatch kernels (kb_*_any, one launch for
// many length classes) both run them, with the same block shapes.
template <int M, int TR, int NK>
__device__ __forceinline__ void bz_fwd(const BSim& d, int lb, const BStage& sg, const float2* __restrict__ twM,
                                       const float2* __restrict__ twP, float2* lds) {
    const int nyb = (d.Ny + TR - 1) / TR;
    const int yb = lb % nyb, r = lb / nyb, x = r % d.Nx, c = r / d.Nx;
    StageIn si{};
    si.m = d.m;
    si.st = d.st;
    si.nk = sg.nk;
    si.mout = sg.use_mi ? d.mi : nullptr;
    for (int j = 0; j < 6; j++) {
        si.k[j] = j < sg.nk ? d.k[sg.kj[j]] : d.m;
        si.a[j] = sg.a[j];
    }
    zfwd_tile<M, TR, NK>(si, d.B1, twM, twP, d.Nx, d.Ny, d.Nz, c, x, yb * TR, lds);
}

template <int M, int TR, int NK>
__global__ __launch_bounds__(TR * RegFFT<M>::G) void kb_zfwd(const BSim* sims, const int2* map, BStage sg,
                                                             const float2* __restrict__ twM,
                                                             const float2* __restrict__ twP) {
    __shared__ float2 lds[zfwd_lds<M, TR>()];
    const BBlock bb = bblock(sims, map);
    const BSim& d = *bb.d;
    if (bskip(d, sg)) return;
    bz_fwd<M, TR, NK>(d, bb.lb, sg, twM, twP, lds);
}

// 3-D Y passes: lds holds the exchange buffers and then the twiddle copy
template <int PY> constexpr int ypass_lds() {
    return (kNT / RegFFT<PY>::G) * RegFFT<PY>::LDS + (PY <= 1024 ? PY : 1);
}
template <int PY, bool FWD>
__device__ __forceinline__ void b_ypass(const BSim& d, int lb, const float2* __restrict__ tw, float2* lds) {
    using F = RegFFT<PY>;
    constexpr int E = F::E, G = F::G, LPB = kNT / G;
    constexpr bool TWL = PY <= 1024;
    float2* twl = lds + LPB * F::LDS;
    if constexpr (TWL)
        for (int i = threadIdx.x; i < PY; i += kNT) twl[i] = tw[i];
    const int li = threadIdx.x / G, g = threadIdx.x % G;
    const unsigned nlines = 3u * d.Nx * d.Q, line = (unsigned)lb * LPB + li;
    const YLine ln = ypass_line(line < nlines ? line : 0, d.dx, d.dq, d.Ny, PY);
    float2 v[E];
    ypass_load<PY, FWD>(v, FWD ? d.B1 : d.B2, ln, line < nlines, d.Ny, g);
    __syncthreads();  // twiddle table
    reg_fft<float, PY, FWD ? -1 : +1>(v, g, lds + li * F::LDS, TWL ? twl : tw);
    if (line < nlines) ypass_store<PY, FWD>(v, FWD ? d.B2 : d.B1, ln, d.Ny, g);
}

template <int PY, bool FWD>
__global__ __launch_bounds__(kNT) void kb_ypass(const BSim* sims, const int2* map, BStage sg,
                                                const float2* __restrict__ tw) {
    __shared__ float2 lds[ypass_lds<PY>()];
    const BBlock bb = bblock(sims, map);
    const BSim& d = *bb.d;
    if (bskip(d, sg)) return;
    b_ypass<PY, FWD>(d, bb.lb, tw, lds);
}

// 3-D X . K . X: lds holds the exchange buffers and then the twiddle copy
template <int PX> constexpr int xmul_lds() { return (kNT / RegFFT<PX>::G) * RegFFT<PX>::LDS + PX; }
template <int PX>
__device__ __forceinline__ void b_xmul(const BSim& d, int lb, const float2* __restrict__ tw, float2* lds) {
    using F = RegFFT<PX>;
    constexpr int E = F::E, G = F::G, LPB = kNT / G;
    float2* twl = lds + LPB * F::LDS;
    for (int i = threadIdx.x; i < PX; i += kNT) twl[i] = tw[i];
    const int li = threadIdx.x / G, g = threadIdx.x % G;
    const int lpr = LPB < d.PY ? LPB : d.PY;
    const int rows = (d.PY + lpr - 1) / lpr;
    int kz, ky;
    xmul_column(lb, (unsigned)d.Q * rows, rows, lpr, li, d.PY, kz, ky);
    float2 v[3][E];
    xmul_load<PX>(v, d.B2, kz, ky, d.Nx, d.PY, d.Q, g);
    __syncthreads();  // twiddle table
#pragma unroll
    for (int c = 0; c < 3; c++) reg_fft<float, PX, -1>(v[c], g, lds + li * F::LDS, twl);
    if (ky >= 0) xmul_kernel<PX>(v, d.Kc, kz, ky, d.PY, g);
#pragma unroll
    for (int c = 0; c < 3; c++) reg_fft<float, PX, +1>(v[c], g, lds + li * F::LDS, twl);
    if (ky >= 0) xmul_store<PX>(v, d.B2, kz, ky, d.Nx, d.PY, d.Q, g);
}

template <int PX>
__global__ __launch_bounds__(kNT) void kb_xmul(const BSim* sims, const int2* map, BStage sg,
                                               const float2* __restrict__ tw) {
    __shared__ float2 lds[xmul_lds<PX>()];
    const BBlock bb = bblock(sims, map);
    const BSim& d = *bb.d;
    if (bskip(d, sg)) return;
    b_xmul<PX>(d, bb.lb, tw, lds);
}

template <int PY, int PX>
__device__ __forceinline__ void b_yxy(const BSim& d, int lb, const float2* __restrict__ twY,
                                      const float2* __restrict__ twX, float2* lds) {
    using Y = Yxy<PY, PX>;
    float2 wx[PX];
#pragma unroll
    for (int j = 0; j < PX; j++) wx[j] = twX[j];
    float2 v[Y::RMAX][Y::E];
    yxy_load<PY, PX>(v, d.B1, d.Nx, d.Ny, d.Q, lb);
    yxy_plane<PY, PX>(v, d.B1, d.Kc, twY, wx, d.Nx, d.Ny, d.Q, lb, lds);
}

template <int PY, int PX>
__global__ __launch_bounds__(kYxyThreads) void kb_yxy(const BSim* sims, const int2* map,
                                                       BStage sg, const float2* __restrict__ twY,
                                                       const float2* __restrict__ twX) {
    __shared__ float2 lds[yxy_lds<PY, PX>()];
    const BBlock bb = bblock(sims, map);
    const BSim& d = *bb.d;
    if (bskip(d, sg)) return;
    b_yxy<PY, PX>(d, bb.lb, twY, twX, lds);
}

// 2-D: the columns of block lb
template <int PY>
__device__ __forceinline__ void b_y2r(const BSim& d, int lb, const float2* __restrict__ tw, float2* lds) {
    y2_columns<PY>(d.B1, d.Kc, tw, (long)lb * Y2<PY>::COLS, d.Ny, d.Q, lds);
}

template <int PY>
__global__ __launch_bounds__(Y2<PY>::NT) void kb_y2r(const BSim* sims, const int2* map,
                                                     BStage sg, const float2* __restrict__ tw) {
    __shared__ float2 lds[Y2<PY>::LDS];
    const BBlock bb = bblock(sims, map);
    const BSim& d = *bb.d;
    if (bskip(d, sg)) return;
    b_y2r<PY>(d, bb.lb, tw, lds);
}

template <int M, int TR, int NU, int FIN>
__device__ __forceinline__ void bz_inv(const BSim& d, int lb, const BStage& sg, const float2* __restrict__ twM,
                                       const float2* __restrict__ twP, float2* lds, float* hext_s, float* red) {
    const int nyb = (d.Ny + TR - 1) / TR;
    const int yb = lb % nyb, x = lb / nyb;
    EpiArgs ea{};
    ea.nx = -1;
    ea.m = sg.use_mi ? d.mi : d.m;
    ea.out = FIN == 1 ? d.m : d.k[sg.i];
    for (int j = 0; j < 6; j++) {
        const bool u = j < sg.nu;
        ea.k[j] = u ? d.k[sg.uj[j]] : d.m;  // unused slots: m with zero coefficients
        ea.a[j] = u ? sg.ua[j] : 0.f;
        ea.b[j] = u ? sg.ub[j] : 0.f;
        ea.ce[j] = u ? sg.ce[j] : 0.0;
    }
    ea.ce_self = sg.ce_self;
    ea.mhigh = d.mtmp;
    ea.part_err = d.part + 2L * d.npart;
    ea.bs = sg.bs;
    ea.nu = sg.nu;
    ea.fin = sg.fin;
    ea.t = d.t;
    ea.t.c = sg.c;
    ea.t.cmax = sg.cmax;
    ea.t.part = sg.partslot < 0 ? nullptr : d.part + (long)sg.partslot * d.npart;
    zinv_epi_tile<M, TR, NU, FIN>(d.B1, ea, twM, twP, d.st, d.Nx, d.Ny, d.Nz, x, yb * TR, lb, lds, hext_s, red);
}

template <int M, int TR, int NU, int FIN>
__global__ __launch_bounds__(3 * TR * RegFFT<M>::G) void kb_zinv_epi(const BSim* sims, const int2* map, BStage sg,
                                                                       const float2* __restrict__ twM,
                                                                       const float2* __restrict__ twP) {
    __shared__ float2 lds[zinv_epi_lds<M, TR>()];
    __shared__ float hext_s[3];
    __shared__ float red[3 * TR * RegFFT<M>::G];
    const BBlock bb = bblock(sims, map);
    const BSim& d = *bb.d;
    if (bskip(d, sg)) return;
    bz_inv<M, TR, NU, FIN>(d, bb.lb, sg, twM, twP, lds, hext_s, red);
}

// rows per Z block of a batch
template <int M> constexpr int z_rows_c() {
    constexpr int G = RegFFT<M>::G;
    int tr = 1024 / G;
    if (tr > 16) tr = 16;
    while (tr > 1 && tr * (M + 1) * 8 > 72 * 1024) tr /= 2;
    return tr;
}
template <int M> constexpr int epi_rows_c() {
    constexpr int G = RegFFT<M>::G;
    int tr = 1024 / (3 * G);
    if (tr > 16) tr = 16;
    int p = 1;
    while (p * 2 <= tr) p *= 2;
    tr = p;
    while (tr > 1 && zinv_epi_lds_elems(M, tr) * 8 > 80 * 1024) tr /= 2;
    return tr;
}
// rows of a dispatch launch's block: it has the LDS of the launch's largest length,
// so at 80 KB all of them ran two to a CU; three by their LDS (40-member sweep, the
// launch of the short lengths 44.4 us, now 38.1).  A launch of one length keeps its
// rows: half of them made 24 members of 256 x 256 3.8 % slower, of 256 x 256 x 4 3.1 %.
template <int M> constexpr int epi_rows_any() {
    int tr = epi_rows_c<M>();
    while (tr > 4 && zinv_epi_lds_elems(M, tr) * 8 > 48 * 1024) tr /= 2;
    return tr;
}

// ---------------------------------------------------------------- length-dispatch kernels
// One launch for the small length classes of a pass: each block reads its
// simulation's lengths and runs the body of that length, with the block shape
// of the per-length kernel (threads beyond it leave at once) and its LDS carved
// from dynamic shared memory sized for the launch's largest class.  A batch of
// many small simulations of different sizes then issues a few launches per
// stage instead of one per length class and pass.
constexpr int kAnyLds = 96 * 1024;
#define GK_ANY_M(X) X(8) X(12) X(16) X(24) X(32) X(48) X(64) X(96) X(128) X(192) X(256) X(384) X(512)
#define GK_ANY_Y(X) X(16) X(24) X(32) X(48) X(64) X(96) X(128) X(192) X(256) X(384) X(512) X(768) X(1024)
inline bool any_m(int M) {
    switch (M) {
#define GK_CASE(n) case n:
        GK_ANY_M(GK_CASE)
#undef GK_CASE
        return true;
    }
    return false;
}
inline bool any_y(int PY) {
    switch (PY) {
#define GK_CASE(n) case n:
        GK_ANY_Y(GK_CASE)
#undef GK_CASE
        return true;
    }
    return false;
}
inline bool any_yx(int PY, int PX) { return any_y(PY) && (PX == 4 || PX == 8) && yxy_fits(PX, PY); }

#define GK_ANY_X(X) X(4) X(8) X(16) X(32)
inline bool any_x(int PX) { return PX == 4 || PX == 8 || PX == 16 || PX == 32; }

template <int M> constexpr int zinv_any_bytes() {
    constexpr int TR = epi_rows_any<M>(), NR = TR * RegFFT<M>::G;
    return zinv_epi_lds<M, TR>() * 8 + 16 + 3 * NR * 4;
}

// the batch's table, the blocks of a launch and its geometry
struct BLaunch {
    const BSim* sims;
    const int2* map;  // per block: simulation, block within it
    int blocks;
    int nt, lds;  // dispatch launch: threads per block and dynamic LDS bytes
    hipStream_t s;
};
// per-length launches (batch_z.hip) and dispatch launches (batch_any.hip)
template <int M> void bz_fwd_run(const BLaunch& b, const BStage& sg, const float2* twM, const float2* twP);
template <int M> void bz_epi_run(const BLaunch& b, const BStage& sg, const float2* twM, const float2* twP);
void any_zfwd(const BLaunch& b, const BStage& sg);
void any_zinv(const BLaunch& b, const BStage& sg);
void any_zinv_fin(const BLaunch& b, const BStage& sg);
void any_y2r(const BLaunch& b, const BStage& sg);
void any_yxy(const BLaunch& b, const BStage& sg);
void any_ypass(const BLaunch& b, const BStage& sg, bool fwd);
void any_xmul(const BLaunch& b, const BStage& sg);
// raise the dispatch kernels' dynamic LDS limit (before any graph capture)
void any_attr_zfwd();
void any_attr_zinv();
void any_attr_zinv_fin();
void any_attr_y();

}  // namespace gk
