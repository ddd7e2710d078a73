// Device code of the convolution passes, shared by the single-simulation
// kernels (conv.hip) and the batched kernels (batch.hip): each pass is a
// __device__ body over one tile / line / column set, wrapped by kernels that
// only decide which tile a block works on.
#pragma once
#include <hip/hip_runtime.h>

#include "engine.h"
#include "fft_device.h"

// Lengths the engine's register-FFT passes are built for (2^a and 3 * 2^a):
// M = half the padded Z length, PY the padded Y length, PX the padded X length.
#define GK_LEN_M(X)                                                                                              \
    X(1) X(2) X(3) X(4) X(6) X(8) X(12) X(16) X(24) X(32) X(48) X(64) X(96) X(128) X(192) X(256) X(384) X(512) \
        X(768) X(1024) X(1536) X(2048)
// the same list in parts: the Z kernels are compiled one part per translation
// unit (conv_z.hip, batch_z.hip; build.py), since they are most of the build time
#define GK_LEN_M_PART0(X) X(1) X(2) X(3) X(4) X(6) X(8) X(12) X(16) X(24) X(32)
#define GK_LEN_M_PART1(X) X(48) X(64)
#define GK_LEN_M_PART2(X) X(96) X(128)
#define GK_LEN_M_PART3(X) X(192) X(256)
#define GK_LEN_M_PART4(X) X(384) X(512)
#define GK_LEN_M_PART5(X) X(768) X(1024)
#define GK_LEN_M_PART6(X) X(1536) X(2048)
#define GK_LEN_Y(X)                                                                                              \
    X(2) X(4) X(6) X(8) X(12) X(16) X(24) X(32) X(48) X(64) X(96) X(128) X(192) X(256) X(384) X(512) X(768)    \
        X(1024) X(1536) X(2048) X(3072) X(4096)
#define GK_LEN_X(X)                                                                                              \
    X(2) X(4) X(6) X(8) X(12) X(16) X(24) X(32) X(48) X(64) X(96) X(128) X(192) X(256) X(384) X(512) X(768)    \
        X(1024)

namespace gk {

// =============================================================== passes
constexpr int kNT = 256;

// Workgroups are dispatched to the 8 XCDs round-robin (block b runs on XCD b % 8),
// and each XCD has its own L2.  Renumber so that every XCD gets one contiguous
// range of logical blocks: neighbouring blocks, which share cache lines (and
// mirrored kernel rows), then meet in the same L2.
__device__ __forceinline__ int xcd_block(int b, int nb) {
    constexpr int kXcd = 8;
    if (nb % kXcd) return b;
    return (b % kXcd) * (nb / kXcd) + b / kXcd;
}

// shuffle of a complex value within groups of W lanes
template <int W> __device__ __forceinline__ float2 shfl2(float2 v, int src) {
    return make_float2(__shfl(v.x, src, W), __shfl(v.y, src, W));
}

// Z forward.  TR rows (y0..y0+TR) of one (c, x) plane; each row is a group of G
// lanes holding the packed complex row z[n] = x[2n] + i x[2n+1] (RK stage build
// m + sum dt a_ij k_j applied while loading), transformed in registers; the
// r2c split takes Z[M-k] from the partner lane by a shuffle, and the spectrum is
// transposed through a padded LDS tile into B1[c][x][kz][y] (TR consecutive y).
//
// The pass is bound by instruction issue as much as by memory (a wave takes 4
// cycles per instruction, and small grids leave one or two waves per SIMD), so
// index arithmetic is kept out of the loops: a thread's tile elements are a
// fixed row r and kz = k0 + G u, one addition apart.  All of a lane's loads
// (m, the earlier k_j, the twiddles of the split) are issued together, and the
// transform's twiddles come from LDS.
constexpr bool z_twl(int M) { return M > 1 && M <= 512; }  // longer tables stay in global memory
template <int M, int TR> constexpr int zfwd_core() {
    constexpr int FFT_LDS = TR * RegFFT<M>::LDS, TILE_LDS = (M + 1) * (TR + 1);
    return FFT_LDS > TILE_LDS ? FFT_LDS : TILE_LDS;
}
template <int M, int TR> constexpr int zfwd_lds() { return zfwd_core<M, TR>() + (z_twl(M) ? M : 0); }

// body: component c, plane x, rows y0..y0+TR; lds holds zfwd_lds<M,TR>() complex.
// NK earlier stages enter the stage build (a compile-time count, so every load
// of a lane is issued before the first is used; unused slots hold m with a
// zero coefficient).
constexpr int zfwd_nk(int nk) { return nk <= 3 ? nk : 5; }
template <int M, int TR, int NK>
__device__ __forceinline__ void zfwd_tile(const StageIn& si, float2* __restrict__ B1, const float2* __restrict__ twM,
                                          const float2* __restrict__ twP, int Nx, int Ny, int Nz, int c, int x,
                                          int y0, float2* lds) {
    using F = RegFFT<M>;
    constexpr int E = F::E, G = F::G, NT = TR * G, Q = M + 1, TS = TR + 1;
    const int row = threadIdx.x / G, g = threadIdx.x % G;
    const int nrows = min(TR, Ny - y0);
    const bool ok = row < nrows;
    const long N = (long)Nx * Ny * Nz;
    const long rbase = c * N + ((long)x * Ny + y0 + row) * Nz;
    float2 v[E], wp[E];
    if ((Nz & 1) == 0) {
        // pairs (2n, 2n+1) as float2: rows start at an even float offset
        float2 kv[NK > 0 ? NK : 1][E];
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int n = g + G * e;
            const bool in = !pad_half<M>(e) && ok && 2 * n < Nz;
            v[e] = in ? *reinterpret_cast<const float2*>(si.m + rbase + 2 * n) : make_float2(0.f, 0.f);
#pragma unroll
            for (int j = 0; j < NK; j++)
                kv[j][e] = in ? *reinterpret_cast<const float2*>(si.k[j] + rbase + 2 * n) : make_float2(0.f, 0.f);
        }
#pragma unroll
        for (int e = 0; e < E; e++) wp[e] = twP[g + G * e];
        const float dt = si.st ? si.st->dt_used : 0.f;
        const bool store = si.mout != nullptr;
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int n = g + G * e;
#pragma unroll
            for (int j = 0; j < NK; j++) {
                v[e].x = fmaf(dt * si.a[j], kv[j][e].x, v[e].x);
                v[e].y = fmaf(dt * si.a[j], kv[j][e].y, v[e].y);
            }
            if (store && !pad_half<M>(e) && ok && 2 * n < Nz) *reinterpret_cast<float2*>(si.mout + rbase + 2 * n) = v[e];
        }
    } else {
        float ks[NK > 0 ? NK : 1][E][2], ms[E][2];
#pragma unroll
        for (int e = 0; e < E; e++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int i = 2 * (g + G * e) + h;
                const bool in = !pad_half<M>(e) && ok && i < Nz;
                ms[e][h] = in ? si.m[rbase + i] : 0.f;
#pragma unroll
                for (int j = 0; j < NK; j++) ks[j][e][h] = in ? si.k[j][rbase + i] : 0.f;
            }
#pragma unroll
        for (int e = 0; e < E; e++) wp[e] = twP[g + G * e];
        const float dt = si.st ? si.st->dt_used : 0.f;
        const bool store = si.mout != nullptr;
#pragma unroll
        for (int e = 0; e < E; e++) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int i = 2 * (g + G * e) + h;
#pragma unroll
                for (int j = 0; j < NK; j++) ms[e][h] = fmaf(dt * si.a[j], ks[j][e][h], ms[e][h]);
                if (store && !pad_half<M>(e) && ok && i < Nz) si.mout[rbase + i] = ms[e][h];
            }
            v[e] = make_float2(ms[e][0], ms[e][1]);
        }
    }
    const float2* tw = twM;
    if constexpr (z_twl(M)) {
        float2* twl = lds + zfwd_core<M, TR>();
        for (int i = threadIdx.x; i < M; i += NT) twl[i] = twM[i];
        tw = twl;
    }
    if constexpr (z_twl(M)) __syncthreads();
    reg_fft<float, M, -1>(v, g, lds + row * F::LDS, tw);
    // r2c split: lane g holds Z[k], k = g + G e; Z[M-k] is in lane (G-g) % G at e' = E-1-e
    // (or, for g = 0, in this lane at e' = (E-e) % E)
    const int partner = (G - g) % G;
    float2 X[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
        const float2 t = shfl2<G>(v[E - 1 - e], partner);
        const float2 zmk = g == 0 ? v[(E - e) % E] : t;
        X[e] = r2c_split<float>(v[e], zmk, wp[e]);
    }
    const float2 nyq = make_float2(v[0].x - v[0].y, 0.f);  // X[M], valid in lane 0
    __syncthreads();  // the FFT exchange buffer becomes the transpose tile
#pragma unroll
    for (int e = 0; e < E; e++) lds[(g + G * e) * TS + row] = X[e];
    if (g == 0) lds[M * TS + row] = nyq;
    __syncthreads();
    const int r = threadIdx.x % TR, k0 = threadIdx.x / TR;  // kz = k0 + G u (and kz = M)
    float2* dst = B1 + ((long)c * Nx + x) * Q * Ny + y0 + (k0 * Ny + r);
    const float2* tile = lds + k0 * TS + r;
    if (r < nrows) {
#pragma unroll
        for (int u = 0; u < E; u++) dst[(long)(u * G * Ny)] = tile[u * G * TS];
        if (k0 == 0) dst[(long)(M * Ny)] = tile[M * TS];
    }
}

template <int M, int TR, int NK>
__global__ __launch_bounds__(TR * RegFFT<M>::G) void k_zfwd(StageIn si, float2* __restrict__ B1,
                                                              const float2* __restrict__ twM,
                                                              const float2* __restrict__ twP, int Nx, int Ny, int Nz) {
    __shared__ float2 lds[zfwd_lds<M, TR>()];
    if (si.st && !si.st->trial_active) return;
    zfwd_tile<M, TR, NK>(si, B1, twM, twP, Nx, Ny, Nz, blockIdx.z, blockIdx.y, blockIdx.x * TR, lds);
}

// A plane's spectra B1[kz][y0..y0+TR) (src, row pitch Ny) into the padded tile
// [kz][TS]: thread t of the component's TR G threads takes row t % TR and kz =
// t / TR + G u, loads issued 8 at a time.
template <int M, int TR>
__device__ __forceinline__ void zinv_load_tile(const float2* __restrict__ src, int Ny, int nrows, int t, float2* tile) {
    constexpr int E = RegFFT<M>::E, G = RegFFT<M>::G, TS = TR + 1;
    const int r = t % TR, k0 = t / TR;
    const bool in = r < nrows;
    src += k0 * Ny + (in ? r : 0);
    tile += k0 * TS + r;
    float2 last = make_float2(0.f, 0.f);
    if (in && k0 == 0) last = src[(long)(M * Ny)];
#pragma unroll
    for (int u0 = 0; u0 < E; u0 += kUnroll) {
        float2 w[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; u++)
            if (u0 + u < E) w[u] = in ? src[(long)((u0 + u) * G * Ny)] : make_float2(0.f, 0.f);
#pragma unroll
        for (int u = 0; u < kUnroll; u++)
            if (u0 + u < E) tile[(u0 + u) * G * TS] = w[u];
    }
    if (k0 == 0) tile[M * TS] = last;
}

// Z inverse: B1[c][x][kz][y0..y0+TR) -> rows of h.  The spectrum is read through
// a padded LDS tile (TR consecutive y per kz), merged (c2r) in registers and
// transformed back; each lane writes its (2n, 2n+1) pairs as float2.
template <int M, int TR>
__global__ __launch_bounds__(TR * RegFFT<M>::G) void k_zinv(const float2* __restrict__ B1, float* __restrict__ h,
                                                              const float2* __restrict__ twM,
                                                              const float2* __restrict__ twP, const EngineState* st,
                                                              int Nx, int Ny, int Nz) {
    using F = RegFFT<M>;
    constexpr int E = F::E, G = F::G, NT = TR * G, Q = M + 1, TS = TR + 1;
    __shared__ float2 lds[zfwd_lds<M, TR>()];
    if (st && !st->trial_active) return;
    const int row = threadIdx.x / G, g = threadIdx.x % G;
    const int c = blockIdx.z, x = blockIdx.y, y0 = blockIdx.x * TR;
    const int nrows = min(TR, Ny - y0);
    const float2* src = B1 + ((long)c * Nx + x) * Q * Ny + y0;
    zinv_load_tile<M, TR>(src, Ny, nrows, threadIdx.x, lds);
    const float2* tw = twM;
    if constexpr (z_twl(M)) {
        float2* twl = lds + zfwd_core<M, TR>();
        for (int i = threadIdx.x; i < M; i += NT) twl[i] = twM[i];
        tw = twl;
    }
    __syncthreads();
    float2 v[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int k = g + G * e;
        v[e] = c2r_merge<float>(lds[k * TS + row], lds[(M - k) * TS + row], twP[k]);
    }
    __syncthreads();  // the tile becomes the FFT exchange buffer
    reg_fft<float, M, +1>(v, g, lds + row * F::LDS, tw);
    if (row < nrows) {
        const long N = (long)Nx * Ny * Nz;
        float* dst = h + c * N + ((long)x * Ny + y0 + row) * Nz;
        if ((Nz & 1) == 0) {
#pragma unroll
            for (int e = 0; e < E; e++) {
                const int n = g + G * e;
                if (!pad_half<M>(e) && 2 * n < Nz) *reinterpret_cast<float2*>(dst + 2 * n) = v[e];
            }
        } else {
#pragma unroll
            for (int e = 0; e < E; e++) {
                const int n = g + G * e;
                if (!pad_half<M>(e) && 2 * n < Nz) dst[2 * n] = v[e].x;
                if (!pad_half<M>(e) && 2 * n + 1 < Nz) dst[2 * n + 1] = v[e].y;
            }
        }
    }
}

// Fused Z inverse + RK stage epilogue.  One block: TR rows (y0..y0+TR) of one x
// plane for all 3 components (3 x TR lane groups).  The 3 spectra are read
// through transposed LDS tiles, merged and transformed back in registers, and
// the fields are exchanged through LDS so that every thread sees h of all 3
// components for its cells.  The epilogue (EpiArgs) rebuilds the stage input
// m_i from m and the earlier k_j (the same fmaf sequence as the forward pass's
// stage build), evaluates the torque, and stores k_i (with the per-block max
// |k_i|) or, for the last stage of a fixed-step tableau, the normalised new m.
// h itself never leaves the chip.  NU bounds the number of earlier stages read
// (the launcher points unused slots at m with zero coefficients, which leaves
// every fmaf chain unchanged), so all loads are unconditional.
__host__ __device__ constexpr int zinv_epi_lds_elems(int M, int TR) {
    const int Q = M + 1, TS = TR + 1, HS = (M + 1) / 2;
    const int TILE = 3 * Q * TS, FFTB = 3 * TR * (M + M / 8), HB = 3 * TR * HS;  // RegFFT<M>::LDS = M + M/8
    return TILE > FFTB ? (TILE > HB ? TILE : HB) : (FFTB > HB ? FFTB : HB);
}
template <int M, int TR> constexpr int zinv_epi_lds() {
    static_assert(RegFFT<M>::LDS == M + M / 8, "exchange buffer size");
    return zinv_epi_lds_elems(M, TR) + (z_twl(M) ? M : 0);  // + the twiddle table
}

// body: plane x, rows y0..y0+TR, all 3 components; the per-block max |k| goes to
// ea.t.part[pidx]; lds / hext_s / red: zinv_epi_lds<M,TR>() complex, 3 and
// 3 TR G floats
// FIN: 0 torque only; 1 last stage of a fixed-step tableau (m <- normalise(m +
// dt sum b_j k_j)); 2 last stage of an adaptive FSAL tableau, whose stage input
// is the high-order solution (a_Sj = b_j): it is stored to ea.mhigh and the
// error dt sum (b2_j - b_j) k_j, this stage's k included, is reduced per block
// into ea.part_err (rk.go:381-403), in place of a separate final pass.
// NX >= 0: the next stage's Z forward follows in the same block.  Everything of it
// is local to the rows: its input is formed from this stage's k in registers (NX
// earlier stages besides, padded as above), exchanged through LDS, transformed
// and stored over the spectra the block has read.  A stage of a film is then two
// launches instead of three, and the forward pass's read of m and of this stage's
// k is gone: 128 x 32 film, Z inverse 6.0 and Z forward 4.4 us, together 8.8 us (and
// one launch gap); 301 x 180 film 8.5 and 9.7 us, together 16.2 us.
// Where few earlier stages enter (NU <= 1) the cells' m and k_j are loaded with the
// spectra, before the transform.  As in the forward pass, a thread's tile
// elements, cells and twiddles need no division or 64-bit product per element
// (the copy's, 16 per thread, and the cells' had cost more instructions than the
// transform).
template <int M, int TR, int NU, int FIN, int NX = -1>
__device__ __forceinline__ void zinv_epi_tile(float2* B1, const EpiArgs& ea,
                                              const float2* __restrict__ twM, const float2* __restrict__ twP,
                                              const EngineState* st, int Nx, int Ny, int Nz, int x, int y0, int pidx,
                                              float2* lds, float* hext_s, float* red) {
    using F = RegFFT<M>;
    constexpr int E = F::E, G = F::G, NR = TR * G, NT = 3 * NR, Q = M + 1, TS = TR + 1;
    constexpr int HS = (M + 1) / 2;  // float2 per h row (z pairs); Nz <= M
    const int c = threadIdx.x / NR, rem = threadIdx.x - c * NR, row = rem / G, g = rem % G;
    const int nrows = min(TR, Ny - y0);
    if (threadIdx.x == 0) stage_field(ea.t, st, hext_s);
    zinv_load_tile<M, TR>(B1 + ((long)c * Nx + x) * Q * Ny + y0, Ny, nrows, rem, lds + c * Q * TS);
    const float2* tw = twM;
    if constexpr (z_twl(M)) {
        float2* twl = lds + zinv_epi_lds_elems(M, TR);
        for (int i = threadIdx.x; i < M; i += NT) twl[i] = twM[i];
        tw = twl;
    }
    const float dt = st->dt_used;
    float ca[NU > 0 ? NU : 1], cb[NU > 0 ? NU : 1];
#pragma unroll
    for (int j = 0; j < NU; j++) {
        ca[j] = dt * ea.a[j];
        cb[j] = dt * ea.b[j];
    }
    const float cbs = dt * ea.bs;
    double ce[NU > 0 ? NU : 1];
#pragma unroll
    for (int j = 0; j < NU; j++) ce[j] = FIN == 2 ? ea.ce[j] * (double)dt : 0.0;
    const double ce_self = FIN == 2 ? ea.ce_self * (double)dt : 0.0;
    const long N = (long)Nx * Ny * Nz;
    const long rowbase = ((long)x * Ny + y0) * Nz;
    // A thread's cells: pairs (2n, 2n+1) as float2 where rows start at an even
    // float (VW = 2), else single cells.  The stage input mi (and the final sum hi,
    // or the error of the earlier stages er) is accumulated from m and the k_j.
    constexpr int IT2 = (TR * HS + NT - 1) / NT, IT1 = (2 * TR * HS + NT - 1) / NT;
    struct Cells {
        float mi[IT1][3], hi[FIN == 1 ? IT1 : 1][3];
        double er[FIN == 2 ? IT1 : 1][3];
    };
    const bool pairs = (Nz & 1) == 0;
    // cell index of slot it of this thread, -1 if none; row r and column z of the tile
    auto cell1 = [&](int it, int& r, int& z) -> long {
        const int p = threadIdx.x + it * NT;
        r = p / (2 * HS);
        z = p % (2 * HS);
        return r < nrows && z < Nz ? rowbase + (r * Nz + z) : -1;
    };
    auto cell2 = [&](int it, int& r, int& n) -> long {
        const int p = threadIdx.x + it * NT;
        r = p / HS;
        n = p % HS;
        return r < nrows && 2 * n < Nz ? rowbase + (r * Nz + 2 * n) : -1;
    };
    float2 ai[IT2][3], af[IT2][3];
    double ex[FIN == 2 ? IT2 : 1][3], ey[FIN == 2 ? IT2 : 1][3];
    auto build2 = [&]() {
#pragma unroll
        for (int it = 0; it < IT2; it++) {
            int r, n;
            const long gi = cell2(it, r, n);
            if (gi >= 0) {
#pragma unroll
                for (int q = 0; q < 3; q++) ai[it][q] = af[it][q] = *reinterpret_cast<const float2*>(ea.m + q * N + gi);
                if constexpr (FIN == 2)
#pragma unroll
                    for (int q = 0; q < 3; q++) ex[it][q] = ey[it][q] = 0.0;
#pragma unroll
                for (int j = 0; j < NU; j++)
#pragma unroll
                    for (int q = 0; q < 3; q++) {
                        const float2 kv = *reinterpret_cast<const float2*>(ea.k[j] + q * N + gi);
                        ai[it][q].x = fmaf(ca[j], kv.x, ai[it][q].x);
                        ai[it][q].y = fmaf(ca[j], kv.y, ai[it][q].y);
                        if constexpr (FIN == 1) {
                            af[it][q].x = fmaf(cb[j], kv.x, af[it][q].x);
                            af[it][q].y = fmaf(cb[j], kv.y, af[it][q].y);
                        }
                        if constexpr (FIN == 2) {
                            ex[it][q] = fma(ce[j], (double)kv.x, ex[it][q]);
                            ey[it][q] = fma(ce[j], (double)kv.y, ey[it][q]);
                        }
                    }
            }
        }
    };
    constexpr bool PRE = NU <= 1 && FIN != 2 && E <= 12;
    if constexpr (PRE)
        if (pairs) build2();
    float2 wp[E];
#pragma unroll
    for (int e = 0; e < E; e++) wp[e] = twP[g + G * e];
    __syncthreads();
    float2 v[E];
    {
        const float2* tile = lds + c * Q * TS;
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int k = g + G * e;
            v[e] = c2r_merge<float>(tile[k * TS + row], tile[(M - k) * TS + row], wp[e]);
        }
    }
    __syncthreads();  // the tiles become the FFT exchange buffers
    reg_fft<float, M, +1>(v, g, lds + (c * TR + row) * F::LDS, tw);
    __syncthreads();  // ... and then the h rows
    const int nh = (Nz + 1) >> 1;
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int n = g + G * e;
        if (!pad_half<M>(e) && n < nh) lds[(c * TR + row) * HS + n] = v[e];
    }
    __syncthreads();

    const float hext[3] = {hext_s[0], hext_s[1], hext_s[2]};
    float lmax = 0.f, emax = 0.f;
    double esum = 0.0;
    const bool want_e = ea.epart != nullptr;
    // one cell from the accumulated stage input mi (and final sum hi, or the
    // error of the earlier stages er) and the field h
    auto finish = [&](long ci, const float mi[3], const float hi[3], const double er[3], const float h[3],
                      float o[3]) {
        if (want_e) {
            // phi = -1/2 m.H_conv - m.B_ext - 1/2 k (m.u)^2 (field.go:64-71, gpu_local_contr3.cu:238-256)
            const double mx = mi[0], my = mi[1], mz = mi[2];
            double phi = -0.5 * (mx * h[0] + my * h[1] + mz * h[2]);
            phi -= mx * hext[0] + my * hext[1] + mz * hext[2];
            if (ea.t.anisType == 1) {
                const double mu = mx * ea.t.u[0] + my * ea.t.u[1] + mz * ea.t.u[2];
                phi -= 0.5 * ea.t.kAnis * mu * mu;
            }
            esum += phi;
        }
        float k[3], ht[3] = {h[0], h[1], h[2]};
        add_thermal(ea.t, st, ci, ht);  // not in the energy density (field.go:64-80)
        llg_torque_cell(ea.t, cell_alpha(ea.t, ci), hext, mi[0], mi[1], mi[2], ht[0], ht[1], ht[2], k);
        lmax = fmaxf(lmax, fmaxf(abs_keep_nan(k[0]), fmaxf(abs_keep_nan(k[1]), abs_keep_nan(k[2]))));
        if constexpr (FIN == 2) {
#pragma unroll
            for (int q = 0; q < 3; q++) emax = fmaxf(emax, abs_keep_nan((float)fma(ce_self, (double)k[q], er[q])));
        }
        if constexpr (FIN == 1) {
            float f[3];
#pragma unroll
            for (int q = 0; q < 3; q++) f[q] = fmaf(cbs, k[q], hi[q]);
            const float sc = norm_scale(f[0], f[1], f[2], ea.t.normMap, ci);
#pragma unroll
            for (int q = 0; q < 3; q++) o[q] = f[q] * sc;
        } else {
#pragma unroll
            for (int q = 0; q < 3; q++) o[q] = k[q];
        }
    };
    // the next stage's input from xm and the earlier stages (this stage's k is added below)
    const float xs = NX >= 0 ? dt * ea.xself : 0.f;
    if (pairs) {
        if constexpr (!PRE) build2();
        float2 xn[NX >= 0 && FIN != 1 ? IT2 : 1][3];
        if constexpr (NX >= 0 && FIN != 1) {
#pragma unroll
            for (int it = 0; it < IT2; it++) {
                int r, n;
                const long gi = cell2(it, r, n);
                if (gi >= 0) {
#pragma unroll
                    for (int q = 0; q < 3; q++) {
                        xn[it][q] = *reinterpret_cast<const float2*>(ea.xm + q * N + gi);
#pragma unroll
                        for (int j = 0; j < NX; j++) {
                            const float2 kv = *reinterpret_cast<const float2*>(ea.xk[j] + q * N + gi);
                            xn[it][q].x = fmaf(dt * ea.xa[j], kv.x, xn[it][q].x);
                            xn[it][q].y = fmaf(dt * ea.xa[j], kv.y, xn[it][q].y);
                        }
                    }
                }
            }
        }
#pragma unroll
        for (int it = 0; it < IT2; it++) {
            int r, n;
            const long gi = cell2(it, r, n);
            if (gi >= 0) {
                float2 hv[3];
#pragma unroll
                for (int q = 0; q < 3; q++) hv[q] = lds[(q * TR + r) * HS + n];
                float mi[3], hi[3], h[3], o0[3], o1[3];
                double er[3] = {0.0, 0.0, 0.0};
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    mi[q] = ai[it][q].x;
                    hi[q] = af[it][q].x;
                    h[q] = hv[q].x;
                    if constexpr (FIN == 2) er[q] = ex[it][q];
                }
                finish(gi, mi, hi, er, h, o0);
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    mi[q] = ai[it][q].y;
                    hi[q] = af[it][q].y;
                    h[q] = hv[q].y;
                    if constexpr (FIN == 2) er[q] = ey[it][q];
                }
                finish(gi + 1, mi, hi, er, h, o1);
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    *reinterpret_cast<float2*>(ea.out + q * N + gi) = make_float2(o0[q], o1[q]);
                    if constexpr (FIN == 2)
                        *reinterpret_cast<float2*>(ea.mhigh + q * N + gi) = ai[it][q];
                    if constexpr (NX >= 0) {
                        float2 z = make_float2(o0[q], o1[q]);
                        if constexpr (FIN != 1) z = make_float2(fmaf(xs, o0[q], xn[it][q].x), fmaf(xs, o1[q], xn[it][q].y));
                        if (ea.xmi) *reinterpret_cast<float2*>(ea.xmi + q * N + gi) = z;
                        lds[(q * TR + r) * HS + n] = z;  // this thread's own h slot
                    }
                }
            }
        }
    } else {
        // rows of odd length: single cells, all of a thread's loads issued first
        float* hf = reinterpret_cast<float*>(lds);
        Cells a;
        float xn[NX >= 0 && FIN != 1 ? IT1 : 1][3];
        if constexpr (NX >= 0 && FIN != 1) {
#pragma unroll
            for (int it = 0; it < IT1; it++) {
                int r, z;
                const long gi = cell1(it, r, z);
                if (gi >= 0) {
#pragma unroll
                    for (int q = 0; q < 3; q++) {
                        xn[it][q] = ea.xm[q * N + gi];
#pragma unroll
                        for (int j = 0; j < NX; j++) xn[it][q] = fmaf(dt * ea.xa[j], ea.xk[j][q * N + gi], xn[it][q]);
                    }
                }
            }
        }
#pragma unroll
        for (int it = 0; it < IT1; it++) {
            int r, z;
            const long gi = cell1(it, r, z);
            if (gi >= 0) {
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    float mi = ea.m[q * N + gi], hi = mi;
                    double er = 0.0;
#pragma unroll
                    for (int j = 0; j < NU; j++) {
                        const float kv = ea.k[j][q * N + gi];
                        mi = fmaf(ca[j], kv, mi);
                        if constexpr (FIN == 1) hi = fmaf(cb[j], kv, hi);
                        if constexpr (FIN == 2) er = fma(ce[j], (double)kv, er);
                    }
                    a.mi[it][q] = mi;
                    if constexpr (FIN == 1) a.hi[it][q] = hi;
                    if constexpr (FIN == 2) a.er[it][q] = er;
                }
            }
        }
#pragma unroll
        for (int it = 0; it < IT1; it++) {
            int r, z;
            const long gi = cell1(it, r, z);
            if (gi >= 0) {
                float h[3], o[3];
#pragma unroll
                for (int q = 0; q < 3; q++) h[q] = hf[(q * TR + r) * 2 * HS + z];
                finish(gi, a.mi[it], a.hi[FIN == 1 ? it : 0], a.er[FIN == 2 ? it : 0], h, o);
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    ea.out[q * N + gi] = o[q];
                    if constexpr (FIN == 2) ea.mhigh[q * N + gi] = a.mi[it][q];
                    if constexpr (NX >= 0) {
                        float x = o[q];
                        if constexpr (FIN != 1) x = fmaf(xs, o[q], xn[it][q]);
                        if (ea.xmi) ea.xmi[q * N + gi] = x;
                        hf[(q * TR + r) * 2 * HS + z] = x;
                    }
                }
            }
        }
    }
    if constexpr (NX >= 0) {
        // Z forward of the rows (as zfwd_tile, all 3 components in this block)
        __syncthreads();
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int n = g + G * e;
            v[e] = make_float2(0.f, 0.f);
            if (!pad_half<M>(e) && row < nrows && 2 * n < Nz) {
                v[e] = lds[(c * TR + row) * HS + n];
                if (2 * n + 1 >= Nz) v[e].y = 0.f;
            }
        }
        __syncthreads();  // the input rows become the FFT exchange buffers
        reg_fft<float, M, -1>(v, g, lds + (c * TR + row) * F::LDS, tw);
        const int partner = (G - g) % G;
        float2 X[E];
#pragma unroll
        for (int e = 0; e < E; e++) {
            const float2 u = shfl2<G>(v[E - 1 - e], partner);
            const float2 zmk = g == 0 ? v[(E - e) % E] : u;
            X[e] = r2c_split<float>(v[e], zmk, twP[g + G * e]);
        }
        const float2 nyq = make_float2(v[0].x - v[0].y, 0.f);
        __syncthreads();  // ... and then the transpose tiles
        float2* tile = lds + c * Q * TS;
#pragma unroll
        for (int e = 0; e < E; e++) tile[(g + G * e) * TS + row] = X[e];
        if (g == 0) tile[M * TS + row] = nyq;
        __syncthreads();
        const int r = rem % TR, k0 = rem / TR;
        if (r < nrows) {
            float2* dst = B1 + ((long)c * Nx + x) * Q * Ny + y0 + (k0 * Ny + r);
            const float2* src = tile + k0 * TS + r;
#pragma unroll
            for (int u = 0; u < E; u++) dst[(long)(u * G * Ny)] = src[u * G * TS];
            if (k0 == 0) dst[(long)(M * Ny)] = src[M * TS];
        }
    }
    if (want_e) {
        // one slot per thread in the tile buffer (3 (M+1)(TR+1) >= NT complex; the h rows are done)
        __syncthreads();
        double* dred = reinterpret_cast<double*>(lds);
        dred[threadIdx.x] = esum;
        __syncthreads();
        if (threadIdx.x == 0) {
            double e = 0.0;
            for (int i = 0; i < NT; i++) e += dred[i];
            ea.epart[pidx] = e;
        }
    }
    // per-block maximum of v (>= 0) into out[pidx]
    auto block_max = [&](float v, float* out) {
        __syncthreads();
        red[threadIdx.x] = v;
        __syncthreads();
        if constexpr (NT >= 64) {
            if (threadIdx.x < 64) {
                float vm = 0.f;
                for (int i = threadIdx.x; i < NT; i += 64) vm = fmaxf(vm, red[i]);
                for (int off = 32; off > 0; off >>= 1) vm = fmaxf(vm, __shfl_xor(vm, off, 64));
                if (threadIdx.x == 0) out[pidx] = vm;
            }
        } else {
            if (threadIdx.x == 0) {
                float vm = 0.f;
                for (int i = 0; i < NT; i++) vm = fmaxf(vm, red[i]);
                out[pidx] = vm;
            }
        }
    };
    if (ea.t.part) block_max(lmax, ea.t.part);
    if constexpr (FIN == 2) block_max(emax, ea.part_err);
}

template <int M, int TR, int NU, int FIN, int NX = -1>
__global__ __launch_bounds__(3 * TR * RegFFT<M>::G) void k_zinv_epi(float2* B1, EpiArgs ea,
                                                                      const float2* __restrict__ twM,
                                                                      const float2* __restrict__ twP,
                                                                      const EngineState* st, int Nx, int Ny, int Nz) {
    __shared__ float2 lds[zinv_epi_lds<M, TR>()];
    __shared__ float hext_s[3];
    __shared__ float red[3 * TR * RegFFT<M>::G];
    if (!st->trial_active) return;
    const int lb = xcd_block(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
    zinv_epi_tile<M, TR, NU, FIN, NX>(B1, ea, twM, twP, st, Nx, Ny, Nz, lb / gridDim.x, (lb % gridDim.x) * TR,
                                  blockIdx.y * gridDim.x + blockIdx.x, lds, hext_s, red);
}

// Division of n < 2^31 by a runtime constant d >= 1 as a product: a pass's lines
// cost two of these instead of four 64-bit divisions (about 100 instructions each,
// twice the line's transform).  With 2^(shift - 31) >= d, mul = ceil(2^shift / d) is
// over 2^shift / d by less than 1, the quotient by less than n / 2^shift < 1 / d: the
// floor is exact.  mul is below 2^32 (2^31 for d = 1 and powers of two, more for others:
// it needs all 32 bits), the product below 2^63.
struct FastDiv {
    unsigned d, mul, shift;
    FastDiv() = default;
    constexpr explicit FastDiv(unsigned dv) : d(dv), mul(0), shift(31) {
        while ((1ull << (shift - 31)) < dv) shift++;
        mul = (unsigned)(((1ull << shift) + dv - 1) / dv);
    }
    __host__ __device__ __forceinline__ constexpr unsigned div(unsigned n) const {
        return (unsigned)(((unsigned long long)n * mul) >> shift);
    }
};
// 3-D Y passes, software-pipelined.  One line per lane group and iteration:
//   forward  B1[c][x][kz][0..Ny) -> B2[c][kz][x][0..Py)   (zero padded)
//   inverse  B2[c][kz][x][0..Py) -> B1[c][x][kz][0..Ny)   (rows >= Ny dropped)
// Lines are numbered with x fastest (a block touches consecutive B2 lines).
// Each lane group walks `nit` lines strided by the grid and loads line i+1
// before transforming line i, so the memory of one line overlaps the FFT of
// the previous one; twiddles come from LDS, so no global load sits between a
// prefetch and its use.
// offsets of B1 line (c, x, kz) and B2 line (c, kz, x) of a Y-pass line number (x fastest)
struct YLine {
    long b1, b2;
};
__device__ __forceinline__ YLine ypass_line(unsigned ln, FastDiv dx, FastDiv dq, int Ny, int PY) {
    const unsigned r = dx.div(ln), x = ln - r * dx.d;
    const unsigned c = dq.div(r), kz = r - c * dq.d;
    return YLine{(long)((c * dx.d + x) * dq.d + kz) * Ny, (long)((c * dq.d + kz) * dx.d + x) * PY};
}
// one line into the lane-strided registers of lane g (zeros when !ok)
template <int PY, bool FWD>
__device__ __forceinline__ void ypass_load(float2* v, const float2* __restrict__ src, const YLine& ln, bool ok, int Ny,
                                           int g) {
    using F = RegFFT<PY>;
    const float2* p = src + (FWD ? ln.b1 : ln.b2) + g;
#pragma unroll
    for (int e = 0; e < F::E; e++) {
        if constexpr (FWD) v[e] = (!pad_half<PY>(e) && ok && g + F::G * e < Ny) ? p[F::G * e] : make_float2(0.f, 0.f);
        else v[e] = ok ? p[F::G * e] : make_float2(0.f, 0.f);
    }
}
template <int PY, bool FWD>
__device__ __forceinline__ void ypass_store(const float2* v, float2* __restrict__ dst, const YLine& ln, int Ny, int g) {
    using F = RegFFT<PY>;
    float2* p = dst + (FWD ? ln.b2 : ln.b1) + g;
#pragma unroll
    for (int e = 0; e < F::E; e++) {
        if constexpr (FWD) p[F::G * e] = v[e];
        else if (!pad_half<PY>(e) && g + F::G * e < Ny) p[F::G * e] = v[e];
    }
}

template <int PY, bool FWD>
__global__ __launch_bounds__(kNT) void k_ypass(const float2* __restrict__ src, float2* __restrict__ dst,
                                               const float2* __restrict__ tw, const EngineState* st, FastDiv dx,
                                               FastDiv dq, int Ny, int nit) {
    using F = RegFFT<PY>;
    constexpr int E = F::E, G = F::G, LPB = kNT / G;
    constexpr bool TWL = PY <= 1024;  // twiddle table in LDS (longer lines keep it in global memory)
    __shared__ float2 lds[LPB * F::LDS];
    __shared__ float2 twl[TWL ? PY : 1];
    if (st && !st->trial_active) return;
    if constexpr (TWL)
        for (int i = threadIdx.x; i < PY; i += kNT) twl[i] = tw[i];
    const int li = threadIdx.x / G, g = threadIdx.x % G;
    const unsigned nlines = 3 * dx.d * dq.d, stride = gridDim.x * LPB;
    unsigned line = blockIdx.x * LPB + li;
    constexpr bool PIPE = E <= 16;  // registers for a second line (longer lines load in place)
    float2 nxt[PIPE ? E : 1];
    YLine ln = ypass_line(line < nlines ? line : 0, dx, dq, Ny, PY);
    if constexpr (PIPE) ypass_load<PY, FWD>(nxt, src, ln, line < nlines, Ny, g);
    __syncthreads();  // twiddle table
    for (int it = 0; it < nit; it++, line += stride) {
        float2 v[E];
        const YLine cur = ln;
        const unsigned next = line + stride;
        if (it + 1 < nit) ln = ypass_line(next < nlines ? next : 0, dx, dq, Ny, PY);
        if constexpr (PIPE) {
#pragma unroll
            for (int e = 0; e < E; e++) v[e] = nxt[e];
            if (it + 1 < nit) ypass_load<PY, FWD>(nxt, src, ln, next < nlines, Ny, g);
        } else {
            ypass_load<PY, FWD>(v, src, cur, line < nlines, Ny, g);
        }
        reg_fft<float, PY, FWD ? -1 : +1>(v, g, lds + li * F::LDS, TWL ? twl : tw);
        if (line < nlines) ypass_store<PY, FWD>(v, dst, cur, Ny, g);
    }
}

// 3-D X forward . kernel . X inverse.  One (kz, ky) column
// per group of G lanes, all 3 components in registers (lane-strided x = g + G e):
// the loads and stores touch G rows of consecutive ky per instruction, the
// 6-component symmetric multiply is lane-local, and each transform needs one
// LDS exchange per radix pass.  A block item is one kz and a run of lpr
// consecutive ky.  Items are ordered so that the runs ky and Py - ky (which read the
// same kernel rows) follow each other.
// the 3 components of column (kz, ky) into lane g's registers (ky < 0: zeros)
template <int PX>
__device__ __forceinline__ void xmul_load(float2 (*v)[RegFFT<PX>::E], const float2* __restrict__ B2, int kz, int ky,
                                          int Nx, int PY, int Q, int g) {
    using F = RegFFT<PX>;
    const long cstride = (long)Q * Nx * PY;
    const float2* base = B2 + (long)kz * Nx * PY + (ky < 0 ? 0 : ky);
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
        for (int e = 0; e < F::E; e++) {
            const int x = g + F::G * e;
            v[c][e] = (!pad_half<PX>(e) && ky >= 0 && x < Nx) ? base[c * cstride + (long)x * PY] : make_float2(0.f, 0.f);
        }
}
template <int PX>
__device__ __forceinline__ void xmul_store(float2 (*v)[RegFFT<PX>::E], float2* __restrict__ B2, int kz, int ky,
                                           int Nx, int PY, int Q, int g) {
    using F = RegFFT<PX>;
    const long cstride = (long)Q * Nx * PY;
    float2* base = B2 + (long)kz * Nx * PY + ky;
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
        for (int e = 0; e < F::E; e++) {
            const int x = g + F::G * e;
            if (!pad_half<PX>(e) && x < Nx) base[c * cstride + (long)x * PY] = v[c][e];
        }
}
// H = K M on the spectrum of column (kz, ky): the symmetric 6-component kernel,
// stored for kx <= PX/2, ky <= PY/2, with the parity signs restored
template <int PX>
__device__ __forceinline__ void xmul_kernel(float2 (*v)[RegFFT<PX>::E], const float* __restrict__ Kc, int kz, int ky,
                                            int PY, int g) {
    GK_FFT_FP
    using F = RegFFT<PX>;
    const int hx = PX / 2 + 1, hy = PY / 2 + 1;
    const bool fy = ky > PY / 2;
    const int kyp = fy ? PY - ky : ky;
    const float* kb = Kc + ((long)kz * hy + kyp) * hx * 6;
#pragma unroll
    for (int e = 0; e < F::E; e++) {
        const int kx = g + F::G * e;
        const bool fx = kx > PX / 2;
        const int kxp = fx ? PX - kx : kx;
        const float2* kk = reinterpret_cast<const float2*>(kb + kxp * 6);
        const float2 k01 = kk[0], k23 = kk[1], k45 = kk[2];
        const float kxx = k01.x, kyy = k01.y, kzz = k23.x;
        float kyz = k23.y, kxz = k45.x, kxy = k45.y;
        if (fy) kyz = -kyz;
        if (fx) kxz = -kxz;
        if (fx != fy) kxy = -kxy;
        const float2 a = v[0][e], b = v[1][e], c = v[2][e];
        v[0][e] = make_float2(a.x * kxx + b.x * kxy + c.x * kxz, a.y * kxx + b.y * kxy + c.y * kxz);
        v[1][e] = make_float2(a.x * kxy + b.x * kyy + c.x * kyz, a.y * kxy + b.y * kyy + c.y * kyz);
        v[2][e] = make_float2(a.x * kxz + b.x * kyz + c.x * kzz, a.y * kxz + b.y * kyz + c.y * kzz);
    }
}
// column of item t for lane group li: items are (kz, run of lpr ky), with the
// runs ky and PY - ky adjacent; ky < 0 when the lane group has no column
__device__ __forceinline__ void xmul_column(unsigned t, unsigned items, unsigned rows, int lpr, int li, int PY,
                                            int& kz, int& ky) {
    kz = (int)(t / rows);
    const int rr = (int)(t - kz * rows);
    const int r = (rr & 1) ? rows - 1 - (rr >> 1) : (rr >> 1);
    ky = (t < items && li < lpr && r * lpr + li < PY) ? r * lpr + li : -1;
}

// Variants of the X . K . X pass whose blocks walk `nit` consecutive items: EE
// elements per lane, RegFFT<PX>::E or half of it over twice the lanes (fewer live
// registers, one more LDS exchange per transform), and PIPE, the next item's
// columns loaded before the current one is transformed (twice the data
// registers) or after.  Lane g of a line holds x = g + (PX / EE) e.  Halves are
// TuneParams::xv 2 (PIPE) and 3; padded X 192 takes the whole with PIPE: its 180
// registers allow two waves per SIMD, the prefetch's 233 as many, so there it costs
// none.  With it / walking items without it / an item per block: 75 x 270 x 74 136 / 163 /
// 158 us a launch, 100 x 45 x 78 32 / 36 / 36, 90 x 90 x 90 51 / 59 / 50.  (At 384, where it
// costs none either, 323 x 11 x 133 59 / 64 / 52 and 90 x 90 x 180 117 / 125 / 111: an item per
// block.)
constexpr bool xmul_walks(int PX) { return PX == 192; }
template <int PX, int EE>
__device__ __forceinline__ void xmul_load_e(float2 (*v)[EE], const float2* __restrict__ B2, int kz, int ky, int Nx,
                                            int PY, int Q, int g) {
    constexpr int G = PX / EE;
    const long cstride = (long)Q * Nx * PY;
    const float2* base = B2 + (long)kz * Nx * PY + (ky < 0 ? 0 : ky);
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
        for (int e = 0; e < EE; e++) {
            const int x = g + G * e;
            const bool pad = EE >= 2 && EE % 2 == 0 && e >= EE / 2;  // x >= PX / 2 >= Nx
            v[c][e] = (!pad && ky >= 0 && x < Nx) ? base[c * cstride + (long)x * PY] : make_float2(0.f, 0.f);
        }
}
template <int PX, int EE>
__device__ __forceinline__ void xmul_store_e(float2 (*v)[EE], float2* __restrict__ B2, int kz, int ky, int Nx, int PY,
                                             int Q, int g) {
    constexpr int G = PX / EE;
    const long cstride = (long)Q * Nx * PY;
    float2* base = B2 + (long)kz * Nx * PY + ky;
#pragma unroll
    for (int c = 0; c < 3; c++)
#pragma unroll
        for (int e = 0; e < EE; e++) {
            const int x = g + G * e;
            const bool pad = EE >= 2 && EE % 2 == 0 && e >= EE / 2;
            if (!pad && x < Nx) base[c * cstride + (long)x * PY] = v[c][e];
        }
}
template <int PX, int EE>
__device__ __forceinline__ void xmul_kernel_e(float2 (*v)[EE], const float* __restrict__ Kc, int kz, int ky, int PY,
                                              int g) {
    GK_FFT_FP
    constexpr int G = PX / EE;
    const int hx = PX / 2 + 1, hy = PY / 2 + 1;
    const bool fy = ky > PY / 2;
    const int kyp = fy ? PY - ky : ky;
    const float* kb = Kc + ((long)kz * hy + kyp) * hx * 6;
#pragma unroll
    for (int e = 0; e < EE; e++) {
        const int kx = g + G * e;
        const bool fx = kx > PX / 2;
        const int kxp = fx ? PX - kx : kx;
        const float2* kk = reinterpret_cast<const float2*>(kb + kxp * 6);
        const float2 k01 = kk[0], k23 = kk[1], k45 = kk[2];
        const float kxx = k01.x, kyy = k01.y, kzz = k23.x;
        float kyz = k23.y, kxz = k45.x, kxy = k45.y;
        if (fy) kyz = -kyz;
        if (fx) kxz = -kxz;
        if (fx != fy) kxy = -kxy;
        const float2 a = v[0][e], b = v[1][e], c = v[2][e];
        v[0][e] = make_float2(a.x * kxx + b.x * kxy + c.x * kxz, a.y * kxx + b.y * kxy + c.y * kxz);
        v[1][e] = make_float2(a.x * kxy + b.x * kyy + c.x * kyz, a.y * kxy + b.y * kyy + c.y * kyz);
        v[2][e] = make_float2(a.x * kxz + b.x * kyz + c.x * kzz, a.y * kxz + b.y * kyz + c.y * kzz);
    }
}
template <int PX, int EE, bool PIPE>
__global__ __launch_bounds__(kNT) void k_xmul_v(float2* __restrict__ B2, const float* __restrict__ Kc,
                                                const float2* __restrict__ tw, const EngineState* st, int Nx, int PY,
                                                int Q, int nit) {
    constexpr int E = EE, G = PX / EE, LPB = kNT / G, LDS = RegFFT<PX>::LDS;
    __shared__ float2 lds[LPB * LDS];
    __shared__ float2 twl[PX];
    if (st && !st->trial_active) return;
    for (int i = threadIdx.x; i < PX; i += kNT) twl[i] = tw[i];
    const int li = threadIdx.x / G, g = threadIdx.x % G;
    const int lpr = LPB < PY ? LPB : PY;
    const int rows = (PY + lpr - 1) / lpr;
    const unsigned items = (unsigned)Q * rows, t0 = blockIdx.x * nit;
    float2 nxt[3][E];
    if constexpr (PIPE) {
        int kz, ky;
        xmul_column(t0, items, rows, lpr, li, PY, kz, ky);
        xmul_load_e<PX, E>(nxt, B2, kz, ky, Nx, PY, Q, g);
    }
    __syncthreads();  // twiddle table
    for (int it = 0; it < nit; it++) {
        const unsigned t = t0 + it;
        int kz, ky;
        xmul_column(t, items, rows, lpr, li, PY, kz, ky);
        float2 v[3][E];
        if constexpr (PIPE) {
#pragma unroll
            for (int c = 0; c < 3; c++)
#pragma unroll
                for (int e = 0; e < E; e++) v[c][e] = nxt[c][e];
            if (it + 1 < nit) {
                int kz1, ky1;
                xmul_column(t + 1, items, rows, lpr, li, PY, kz1, ky1);
                xmul_load_e<PX, E>(nxt, B2, kz1, ky1, Nx, PY, Q, g);
            }
        } else {
            xmul_load_e<PX, E>(v, B2, kz, ky, Nx, PY, Q, g);
        }
#pragma unroll
        for (int c = 0; c < 3; c++) reg_fft<float, PX, -1, 1, E>(v[c], g, lds + li * LDS, twl);
        if (ky >= 0) xmul_kernel_e<PX, E>(v, Kc, kz, ky, PY, g);
#pragma unroll
        for (int c = 0; c < 3; c++) reg_fft<float, PX, +1, 1, E>(v[c], g, lds + li * LDS, twl);
        if (ky >= 0) xmul_store_e<PX, E>(v, B2, kz, ky, Nx, PY, Q, g);
    }
}

// every other length, and the default: RegFFT<PX>::E elements per lane, an item per
// block.  A prefetch of the next item doubles the data registers, and the waves it
// costs hide more latency than it does; and without one, a block that walks items
// only makes later ones wait: 70 x 60 x 51 (padded X 128) 21.2 us a launch with the
// prefetch and 4 blocks per CU, 18.0 an item per block; 256 x 256 x 16 36.8, walking items
// without it 33.8, an item per block 31.0 us; 300 x 300 x 24 148, 135 and 113 us.
// (The launch gives nit = 1; written without the loop, the compiler's schedule was up
// to 12 % faster in the pass on its own, but 64 x 64 x 64 steps went 164 -> 167 us.)
template <int PX>
__global__ __launch_bounds__(kNT) void k_xmul(float2* __restrict__ B2, const float* __restrict__ Kc,
                                              const float2* __restrict__ tw, const EngineState* st, int Nx, int PY,
                                              int Q, int nit) {
    using F = RegFFT<PX>;
    constexpr int E = F::E, G = F::G, LPB = kNT / G;
    __shared__ float2 lds[LPB * F::LDS];
    __shared__ float2 twl[PX];
    if (st && !st->trial_active) return;
    for (int i = threadIdx.x; i < PX; i += kNT) twl[i] = tw[i];
    const int li = threadIdx.x / G, g = threadIdx.x % G;
    const int lpr = LPB < PY ? LPB : PY;  // columns per item
    const int rows = (PY + lpr - 1) / lpr;  // items per kz plane (the last may be partial)
    const unsigned items = (unsigned)Q * rows, t0 = blockIdx.x * nit;
    __syncthreads();  // twiddle table
    for (int it = 0; it < nit; it++) {
        int kz, ky;
        xmul_column(t0 + it, items, rows, lpr, li, PY, kz, ky);
        float2 v[3][E];
        xmul_load<PX>(v, B2, kz, ky, Nx, PY, Q, g);
#pragma unroll
        for (int c = 0; c < 3; c++) reg_fft<float, PX, -1>(v[c], g, lds + li * F::LDS, twl);
        if (ky >= 0) xmul_kernel<PX>(v, Kc, kz, ky, PY, g);
#pragma unroll
        for (int c = 0; c < 3; c++) reg_fft<float, PX, +1>(v[c], g, lds + li * F::LDS, twl);
        if (ky >= 0) xmul_store<PX>(v, B2, kz, ky, Nx, PY, Q, g);
    }
}

// 3-D Y forward . X.K.X . Y inverse of one kz plane in one pass, for padded
// Y = 512 and padded X = 16 or 32 (Nx <= PX/2, Ny <= 256): per field
// evaluation B1 is read and written once and the Y-padded B2 is not used
// (48 A1 + kernel bytes instead of 48 A1 + 96 A2 + kernel for the three
// separate passes).
//
// The length-512 Y transform of a line of 256 inputs splits by the parity p of
// ky: Y(2k + p) = FFT_256(y[n] w^(p n))[k], w = exp(-2 pi i / 512), and the
// inverse, keeping n < 256, is h[n] = sum_p w^(-p n) IFFT_256(H_p)[n].  The
// two parities are independent through the X.K.X stage (a column ky only
// meets the kernel at its own ky), so a block does them one after the other
// and adds the two inverse halves.  Wave x (x < Nx) holds the 3 component
// lines of x (a 256-line is one wave, 4 elements per lane, n or k = g + 64 e);
// each round's spectra go to an LDS staging tile [k][c][x], whose columns the
// block takes through X forward, the kernel multiply and X inverse 128 at a
// time (8 lanes per column, 4 elements per lane), and come back.
//
// Block 0 packs the two real planes kz = 0 and kz = M (= Q - 1; their Z
// spectra are real) as P = A + i B.  After the Y transform, A = (P(k) +
// conj P(-k)) / 2 and B = (P(k) - conj P(-k)) / 2i (-k within the same
// parity round: a lane shuffle), and only the columns k <= its Hermitian
// partner are needed: K_A of A (kernel plane 0) and K_A of B (kernel plane M).
// Coming back, H_P = H_A + i H_B, with the partner's conjugate for the other
// half, and the real and imaginary parts go to planes 0 and M.  So Q planes
// take M = Q - 1 blocks: 256 for the 256x256x16 cuboid, one per CU.
constexpr int kPlaneThreads = 1024;
constexpr int kPlanePY = 512;
__host__ __device__ constexpr bool plane3_fits(int PX, int PY, int Nx) {
    return PY == kPlanePY && (PX == 16 || PX == 32) && Nx >= 1 && 2 * Nx <= PX;
}
template <int PX> struct Plane3 {
    static constexpr int L = kPlanePY / 2;             // half-length Y transform (256)
    static constexpr int YE = 4;                       // elements per lane of a 256-line (64 lanes)
    static constexpr int XE = 4, XG = PX / XE;         // X layout: elements / lanes per column
    static constexpr int SUB = kPlaneThreads / XG;     // columns in the X layout at once
    static constexpr int HX = PX / 2;                  // x slots of a column (Nx <= HX)
    static constexpr int SQ = 3 * HX + 1;              // staging stride per column, padded
    static constexpr int SLOTS = L + 2;                // columns of a round (block 0, even: 2 x 129)
    static constexpr int STAGE = SLOTS * SQ;
    static constexpr int XEXCH = SUB * (PX + PX / 8);
    static constexpr int YEXCH = (kPlaneThreads / 64) * (L + L / 8);
    static constexpr int EXCH = XEXCH > YEXCH ? XEXCH : YEXCH;
    static constexpr int LDS = STAGE + EXCH + L + kPlanePY + PX;  // + twiddle tables
};

template <int PX>
__global__ __launch_bounds__(kPlaneThreads) void k_plane3(float2* __restrict__ B1, const float* __restrict__ Kc,
                                                          const float2* __restrict__ twLg,
                                                          const float2* __restrict__ twPg,
                                                          const float2* __restrict__ twXg, const EngineState* st,
                                                          int Nx, int Ny, int Q) {
    GK_FFT_FP
    using P3 = Plane3<PX>;
    constexpr int L = P3::L, YE = P3::YE, XE = P3::XE, XG = P3::XG, SQ = P3::SQ, HX = P3::HX, SUB = P3::SUB;
    constexpr int PY = kPlanePY;
    __shared__ float2 lds[P3::LDS];
    if (st && !st->trial_active) return;
    float2* stage = lds;                      // [SLOTS][SQ]
    float2* exch = lds + P3::STAGE;           // Y (per wave) or X (per column) exchange buffers
    float2* twL = exch + P3::EXCH;            // exp(-2 pi i j / 256)
    float2* twP = twL + L;                    // exp(-2 pi i j / 512)
    float2* twX = twP + PY;                   // exp(-2 pi i j / PX)
    for (int i = threadIdx.x; i < L; i += kPlaneThreads) twL[i] = twLg[i];
    for (int i = threadIdx.x; i < PY; i += kPlaneThreads) twP[i] = twPg[i];
    if (threadIdx.x < PX) twX[threadIdx.x] = twXg[threadIdx.x];
    const int M = Q - 1;
    const bool packed = blockIdx.x == 0;
    const int kz = blockIdx.x;  // plane of an unpacked block
    const int x = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), g = threadIdx.x % 64;  // wave x, lane g
    const bool xok = x < Nx;
    const long cs = (long)Nx * Q * Ny;
    const long row = ((long)(xok ? x : 0) * Q + kz) * Ny;
    const long rowM = ((long)(xok ? x : 0) * Q + M) * Ny;
    __syncthreads();  // twiddle tables
    const int q = threadIdx.x / XG, gx = threadIdx.x % XG;  // X layout: column q of a sub-round, lane gx
    const int hx = PX / 2 + 1, hy = PY / 2 + 1;
    float2 half0[3][YE];  // the even round's inverse half of the lines
#pragma unroll
    for (int p = 0; p < 2; p++) {
        // columns of block 0: A for k < KA, B for KA <= slot < 2 KA (KA = 129 even, 128 odd)
        const int KA = p ? L / 2 : L / 2 + 1;
        const int nslots = packed ? 2 * KA : L;
        // ---- the plane's lines (read again for the odd round rather than held in
        // registers through the even one), then Y forward of this parity:
        // FFT_256(y[n] w^(p n)); loads from clamped indices and a select, so no
        // divergent branch sits around them
        float2 u[3][YE];
        if (packed) {
#pragma unroll
            for (int c = 0; c < 3; c++)
#pragma unroll
                for (int e = 0; e < YE; e++) {
                    const int n = g + 64 * e, nn = n < Ny ? n : Ny - 1;
                    const float2 a = B1[c * cs + row + nn], b = B1[c * cs + rowM + nn];
                    u[c][e] = (xok && n < Ny) ? make_float2(a.x, b.x) : make_float2(0.f, 0.f);
                }
        } else {
#pragma unroll
            for (int c = 0; c < 3; c++)
#pragma unroll
                for (int e = 0; e < YE; e++) {
                    const int n = g + 64 * e, nn = n < Ny ? n : Ny - 1;
                    const float2 a = B1[c * cs + row + nn];
                    u[c][e] = (xok && n < Ny) ? a : make_float2(0.f, 0.f);
                }
        }
        if (p && xok) {
            // the even round's half of h parks in B1 (its inputs are read): registers stay free for the odd round
#pragma unroll
            for (int c = 0; c < 3; c++)
#pragma unroll
                for (int e = 0; e < YE; e++) {
                    const int n = g + 64 * e;
                    if (n < Ny) B1[c * cs + row + n] = half0[c][e];
                }
        }
#pragma unroll
        for (int c = 0; c < 3; c++) {
            if (p)
#pragma unroll
                for (int e = 0; e < YE; e++) u[c][e] = cmul<float>(u[c][e], twP[g + 64 * e]);
            reg_fft<float, L, -1, 1, YE, true>(u[c], g, exch + x * (L + L / 8), twL);
        }
        // ---- into the staging tile
        if (xok) {
            if (!packed) {
#pragma unroll
                for (int e = 0; e < YE; e++)
#pragma unroll
                    for (int c = 0; c < 3; c++) stage[(g + 64 * e) * SQ + c * HX + x] = u[c][e];
            } else {
                // partner -k of k = g + 64 e: lane (64 - g) % 64 (even) or 63 - g (odd), element 3 - e;
                // for g = 0 of the even round, this lane's element (4 - e) % 4
                const int src = p ? 63 - g : (64 - g) & 63;
#pragma unroll
                for (int c = 0; c < 3; c++)
#pragma unroll
                    for (int e = 0; e < YE; e++) {
                        const float2 ta = shfl2<64>(u[c][YE - 1 - e], src);
                        const float2 pm = (p == 0 && g == 0) ? u[c][(YE - e) % YE] : ta;
                        const int k = g + 64 * e;
                        if (k < KA) {
                            const float2 a = u[c][e];
                            stage[k * SQ + c * HX + x] = make_float2((a.x + pm.x) * 0.5f, (a.y - pm.y) * 0.5f);
                            stage[(KA + k) * SQ + c * HX + x] =
                                make_float2((a.y + pm.y) * 0.5f, (pm.x - a.x) * 0.5f);
                        }
                    }
            }
        }
        __syncthreads();  // the Y exchange buffers become the X ones
        // ---- X . K . X of every column, SUB at a time
        for (int j = 0; j * SUB < nslots; j++) {
            const int slot = j * SUB + q;
            const bool ok = slot < nslots;
            float2* col = stage + (ok ? slot : 0) * SQ;
            // kernel plane and ky of the column
            const bool bcol = packed && slot >= KA;
            const int kzk = packed ? (bcol ? M : 0) : kz;
            const int ky = 2 * (bcol ? slot - KA : slot) + p;
            float2 xv[3][XE];
#pragma unroll
            for (int c = 0; c < 3; c++)
#pragma unroll
                for (int e = 0; e < XE; e++) {
                    const int xx = gx + XG * e;
                    xv[c][e] = (ok && 2 * e < XE && xx < Nx) ? col[c * HX + xx] : make_float2(0.f, 0.f);
                }
#pragma unroll
            for (int c = 0; c < 3; c++) reg_fft<float, PX, -1, 1, XE, true>(xv[c], gx, exch + q * (PX + PX / 8), twX);
            if (ok) {
                // H = K M with the compressed kernel's parity signs restored (as xmul_kernel)
                const bool fy = ky > PY / 2;
                const float* kb = Kc + ((long)kzk * hy + (fy ? PY - ky : ky)) * hx * 6;
#pragma unroll
                for (int e = 0; e < XE; e++) {
                    const int kx = gx + XG * e;
                    const bool fx = kx > PX / 2;
                    const float2* kk = reinterpret_cast<const float2*>(kb + (fx ? PX - kx : kx) * 6);
                    const float2 k01 = kk[0], k23 = kk[1], k45 = kk[2];
                    const float kxx = k01.x, kyy = k01.y, kzz = k23.x;
                    const float kyz = fy ? -k23.y : k23.y, kxz = fx ? -k45.x : k45.x;
                    const float kxy = (fx != fy) ? -k45.y : k45.y;
                    const float2 a = xv[0][e], b = xv[1][e], cc = xv[2][e];
                    xv[0][e] = make_float2(a.x * kxx + b.x * kxy + cc.x * kxz, a.y * kxx + b.y * kxy + cc.y * kxz);
                    xv[1][e] = make_float2(a.x * kxy + b.x * kyy + cc.x * kyz, a.y * kxy + b.y * kyy + cc.y * kyz);
                    xv[2][e] = make_float2(a.x * kxz + b.x * kyz + cc.x * kzz, a.y * kxz + b.y * kyz + cc.y * kzz);
                }
            }
#pragma unroll
            for (int c = 0; c < 3; c++) reg_fft<float, PX, +1, 1, XE, true>(xv[c], gx, exch + q * (PX + PX / 8), twX);
            if (ok)
#pragma unroll
                for (int c = 0; c < 3; c++)
#pragma unroll
                    for (int e = 0; e < XE; e++) {
                        const int xx = gx + XG * e;
                        if (2 * e < XE && xx < Nx) col[c * HX + xx] = xv[c][e];
                    }
        }
        __syncthreads();  // the staging tile is complete; the X exchange buffers become the Y ones
        // ---- back into the lines and Y inverse of this parity
#pragma unroll
        for (int e = 0; e < YE; e++) {
            const int k = g + 64 * e;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                float2 h = make_float2(0.f, 0.f);
                if (xok) {
                    if (!packed) {
                        h = stage[k * SQ + c * HX + x];
                    } else {
                        // H_P = H_A + i H_B; beyond KA from the Hermitian partner, conjugated
                        const bool low = k < KA;
                        const int kk = low ? k : (p ? L - 1 - k : L - k);
                        float2 ha = stage[kk * SQ + c * HX + x], hb = stage[(KA + kk) * SQ + c * HX + x];
                        if (!low) {
                            ha.y = -ha.y;
                            hb.y = -hb.y;
                        }
                        h = make_float2(ha.x - hb.y, ha.y + hb.x);
                    }
                }
                u[c][e] = h;
            }
        }
#pragma unroll
        for (int c = 0; c < 3; c++) {
            reg_fft<float, L, +1, 1, YE, true>(u[c], g, exch + x * (L + L / 8), twL);
            if (p) {
#pragma unroll
                for (int e = 0; e < YE; e++) {
                    float2 w = twP[g + 64 * e];
                    w.y = -w.y;
                    u[c][e] = cmul<float>(u[c][e], w);
                }
            }
        }
        if (p == 0) {
#pragma unroll
            for (int c = 0; c < 3; c++)
#pragma unroll
                for (int e = 0; e < YE; e++) half0[c][e] = u[c][e];
        } else if (xok) {
            // h = even half (parked in B1 by this lane) + odd half
#pragma unroll
            for (int c = 0; c < 3; c++)
#pragma unroll
                for (int e = 0; e < YE; e++) {
                    const int n = g + 64 * e;
                    if (n < Ny) {
                        const float2 h0 = B1[c * cs + row + n];
                        const float2 h = make_float2(h0.x + u[c][e].x, h0.y + u[c][e].y);
                        if (packed) {
                            B1[c * cs + row + n] = make_float2(h.x, 0.f);
                            B1[c * cs + rowM + n] = make_float2(h.y, 0.f);
                        } else {
                            B1[c * cs + row + n] = h;
                        }
                    }
                }
        }
        __syncthreads();  // the staging tile and exchange buffers are free for the next round
    }
}

// Thin 3-D grids (padded X of 4 to 16): Y forward, X . K . X and Y inverse of
// one kz plane in one pass.  The plane of Y spectra [3][Nx][PY] stays in LDS,
// so per field evaluation the pass reads and writes B1 once, where the three
// separate passes move B1 twice and the Y-padded B2 four times.  The X
// transforms of length PX (Nx <= PX/2 nonzero inputs, Nx outputs kept) are
// register butterflies with the table exp(-2 pi i j / PX).
constexpr int kYxyThreads = 256;
constexpr int kYxyLdsBytes = 80 * 1024;
// Which plans take the plane pass: a plane of 3 (PX/2) lines plus separate
// FFT exchange buffers within 80 KB (the sizes its registers were sized for).
__host__ __device__ constexpr bool yxy_fits(int PX, int PY) {
    return PX >= 4 && PX <= 16 && reg_fft_length(PY) &&
           (3 * (PX / 2) * PY + (kYxyThreads / reg_fft_G(PY)) * (PY + PY / 8)) * 8 <= kYxyLdsBytes;
}
// LDS of the pass: the plane's rows l = r LPB + li at l PY; the FFT exchange
// buffers overlay the rows of the last round of lines (r = RMAX - 1), which are
// written only after every lane group's last forward FFT and read back before
// any inverse FFT (yxy_plane), so the two share memory: ~50 KB instead of
// ~66 KB for PY = 512, PX = 8, three blocks per CU instead of two.
__host__ __device__ constexpr int yxy_lds_elems(int PX, int PY) {
    return (3 * (PX / 2) * PY) >
                   ((3 * (PX / 2) + kYxyThreads / reg_fft_G(PY) - 1) / (kYxyThreads / reg_fft_G(PY)) - 1) *
                           (kYxyThreads / reg_fft_G(PY)) * PY +
                       (kYxyThreads / reg_fft_G(PY)) * (PY + PY / 8)
               ? 3 * (PX / 2) * PY
               : ((3 * (PX / 2) + kYxyThreads / reg_fft_G(PY) - 1) / (kYxyThreads / reg_fft_G(PY)) - 1) *
                         (kYxyThreads / reg_fft_G(PY)) * PY +
                     (kYxyThreads / reg_fft_G(PY)) * (PY + PY / 8);
}
template <int PY, int PX> constexpr int yxy_lds() { return yxy_lds_elems(PX, PY); }
template <int PY, int PX> struct Yxy {
    using F = RegFFT<PY>;
    static constexpr int E = F::E, G = F::G, LPB = kYxyThreads / G;
    static constexpr int RMAX = (3 * (PX / 2) + LPB - 1) / LPB;  // rounds of lines per lane group, at most
};

// the 3 Nx lines (l = c Nx + x) of plane kz into the lane group's registers
template <int PY, int PX>
__device__ __forceinline__ void yxy_load(float2 (*v)[RegFFT<PY>::E], const float2* __restrict__ B1, int Nx, int Ny,
                                         int Q, int kz) {
    using Y = Yxy<PY, PX>;
    const int li = threadIdx.x / Y::G, g = threadIdx.x % Y::G;
#pragma unroll
    for (int r = 0; r < Y::RMAX; r++) {
        const int l = r * Y::LPB + li;
        const bool ok = l < 3 * Nx;
        const float2* src = B1 + ((long)(ok ? l : 0) * Q + kz) * Ny;  // B1[c][x][kz][y], (c, x) = line l
#pragma unroll
        for (int e = 0; e < Y::E; e++) {
            const int i = g + Y::G * e;
            v[r][e] = (!pad_half<PY>(e) && ok && i < Ny) ? src[i] : make_float2(0.f, 0.f);
        }
    }
}

// the plane pass on loaded lines (called by every thread of the block)
template <int PY, int PX>
__device__ __forceinline__ void yxy_plane(float2 (*v)[RegFFT<PY>::E], float2* __restrict__ B1,
                                          const float* __restrict__ Kc, const float2* twY, const float2* wx, int Nx,
                                          int Ny, int Q, int kz, float2* lds) {
    using Y = Yxy<PY, PX>;
    using F = RegFFT<PY>;
    constexpr int E = Y::E, G = Y::G, NT = kYxyThreads, LPB = Y::LPB, RMAX = Y::RMAX;
    constexpr int hx = PX / 2 + 1, hy = PY / 2 + 1;
    float2* plane = lds;                                  // [3 Nx][PY]
    float2* exch = lds + (long)(RMAX - 1) * LPB * PY;     // LPB exchange buffers over the last round's rows
    static_assert((RMAX - 1) * LPB * PY + LPB * F::LDS <= yxy_lds<PY, PX>(), "LDS layout");
    const int li = threadIdx.x / G, g = threadIdx.x % G;
    const int nl = 3 * Nx;
    // Y forward
#pragma unroll
    for (int r = 0; r < RMAX; r++) {
        const int l = r * LPB + li;
        if (r * LPB < nl) {  // uniform: some lane group has a line in this round
            reg_fft<float, PY, -1>(v[r], g, exch + li * F::LDS, twY);
            // the last round's rows hold the exchange buffers until every lane group is through
            if (r == RMAX - 1) __syncthreads();
            if (l < nl)
#pragma unroll
                for (int e = 0; e < E; e++) plane[(long)l * PY + g + G * e] = v[r][e];
        }
    }
    __syncthreads();
    // X . K . X for every ky of the plane
    for (int ky = threadIdx.x; ky < PY; ky += NT) {
        GK_FFT_FP
        // radix-4 / radix-8 butterflies, or two factors for 6, 12 and 16 (the direct sums
        // these replace took 3 x PX^2 / 2 complex products a transform, more than
        // everything else in the pass: 150 x 91 x 3, PX 6, 7.9 us a launch, now 7.5;
        // 128 x 128 x 8, PX 16, 21.8 us, now 14.0)
        constexpr bool R48 = PX == 4 || PX == 8;
        float2 a[3][PX];
#pragma unroll
        for (int c = 0; c < 3; c++)
#pragma unroll
            for (int kx = 0; kx < PX; kx++) a[c][kx] = make_float2(0.f, 0.f);
#pragma unroll
        for (int x = 0; x < PX / 2; x++)
            if (x < Nx)
#pragma unroll
                for (int c = 0; c < 3; c++) a[c][x] = plane[(long)(c * Nx + x) * PY + ky];
#pragma unroll
        for (int c = 0; c < 3; c++) {
            if constexpr (R48) dft<float, PX, -1>(a[c]);
            else dft_small<float, PX, -1>(a[c], wx);
        }
        // kernel layout of plane-pass plans: [kz][component][kx <= PX/2][ky <= PY/2], so that
        // consecutive ky (threads) read consecutive floats
        const bool fy = ky > PY / 2;
        const int kyp = fy ? PY - ky : ky;
        const float* kb = Kc + (long)kz * 6 * hx * hy + kyp;
#pragma unroll
        for (int kx = 0; kx < PX; kx++) {
            const bool fx = kx > PX / 2;
            const float* kk = kb + (fx ? PX - kx : kx) * hy;
            constexpr int cs = hx * hy;
            const float kxx = kk[0], kyy = kk[cs], kzz = kk[2 * cs];
            const float kyz = fy ? -kk[3 * cs] : kk[3 * cs], kxz = fx ? -kk[4 * cs] : kk[4 * cs];
            const float kxy = (fx != fy) ? -kk[5 * cs] : kk[5 * cs];
            const float2 p = a[0][kx], q = a[1][kx], w = a[2][kx];
            a[0][kx] = make_float2(p.x * kxx + q.x * kxy + w.x * kxz, p.y * kxx + q.y * kxy + w.y * kxz);
            a[1][kx] = make_float2(p.x * kxy + q.x * kyy + w.x * kyz, p.y * kxy + q.y * kyy + w.y * kyz);
            a[2][kx] = make_float2(p.x * kxz + q.x * kyz + w.x * kzz, p.y * kxz + q.y * kyz + w.y * kzz);
        }
#pragma unroll
        for (int c = 0; c < 3; c++) {
            if constexpr (R48) dft<float, PX, +1>(a[c]);
            else dft_small<float, PX, +1>(a[c], wx);
        }
#pragma unroll
        for (int x = 0; x < PX / 2; x++)
            if (x < Nx)
#pragma unroll
                for (int c = 0; c < 3; c++) plane[(long)(c * Nx + x) * PY + ky] = a[c][x];
    }
    __syncthreads();
    // Y inverse, first Ny kept; the last round first, whose rows the exchange
    // buffers take over once every lane group has read them
#pragma unroll
    for (int r = RMAX - 1; r >= 0; r--) {
        if (r * LPB >= nl) continue;  // uniform
        const int l = r * LPB + li;
        const bool ok = l < nl;
        float2 w[E];
#pragma unroll
        for (int e = 0; e < E; e++) w[e] = ok ? plane[(long)l * PY + g + G * e] : make_float2(0.f, 0.f);
        if (r == RMAX - 1) __syncthreads();
        reg_fft<float, PY, +1>(w, g, exch + li * F::LDS, twY);
        if (ok) {
            float2* dst = B1 + ((long)l * Q + kz) * Ny;
#pragma unroll
            for (int e = 0; e < E; e++) {
                const int i = g + G * e;
                if (!pad_half<PY>(e) && i < Ny) dst[i] = w[e];
            }
        }
    }
}

// single simulation: one block per kz plane
template <int PY, int PX>
__global__ __launch_bounds__(kYxyThreads) void k_yxy(float2* __restrict__ B1, const float* __restrict__ Kc,
                                                      const float2* __restrict__ twY, const float2* __restrict__ twX,
                                                      const EngineState* st, int Nx, int Ny, int Q) {
    using Y = Yxy<PY, PX>;
    __shared__ float2 lds[yxy_lds<PY, PX>()];
    if (st && !st->trial_active) return;
    float2 wx[PX];
#pragma unroll
    for (int j = 0; j < PX; j++) wx[j] = twX[j];
    float2 v[Y::RMAX][Y::E];
    yxy_load<PY, PX>(v, B1, Nx, Ny, Q, blockIdx.x);
    yxy_plane<PY, PX>(v, B1, Kc, twY, wx, Nx, Ny, Q, blockIdx.x, lds);
}

// 2-D: Y forward . kernel . Y inverse of kz columns, in place in B1[c][0][kz][y].
// Each component of a column has lanes of its own (block = 3 x W threads, W =
// max(64, G), thread group c; W / G columns per block), so a column's six
// transforms run as two after one another; only y and z meet, through LDS, at the
// kernel multiply (the 4 stored components xx, yy, zz, yz for ky <= PY/2, the yz
// sign restored beyond).  A lane holds up to 8 (12 for 3 * 2^a) elements, so long
// lines span several waves, with block barriers in their exchanges.  The kernel
// values are loaded with the line, before the transforms (of long lines after the
// forward transform: 80 registers, so that two blocks of 768 threads share a CU).
//
// The form this replaces held the 3 components in one lane group with L/64
// elements per lane: one wave per SIMD, 4 cycles per instruction and nothing to
// overlap.  Measured per launch (before / now): 1025 columns of 2048 (film 1024 x
// 1024) 75 / 43 us; 385 of 384 (301 x 180) 15 / 8.2 us; 129 of 64 (128 x 32) 6.0 /
// 4.4 us.
constexpr int y2_E(int L) { return L % 3 == 0 ? (L < 12 ? L : 12) : (L < 8 ? L : (L <= 2048 ? 8 : 16)); }
template <int PY> struct Y2 {
    static constexpr int E = y2_E(PY), G = PY / E;
    static constexpr int W = G > 64 ? G : 64;     // threads per component
    static constexpr int NT = 3 * W, COLS = W / G;  // threads and columns per block
    static constexpr int LINE = PY + PY / 8;      // exchange buffer of one line
    static constexpr bool TWL = PY <= 2048;       // twiddle table in LDS
    static constexpr int LDS = 3 * COLS * LINE + (TWL ? PY : 1);
};
// inputs / outputs at index >= PY/2 are padding (compile time, lane-strided i = g + G e)
template <int PY> __device__ constexpr bool y2_pad(int e) { return Y2<PY>::E % 2 == 0 && e >= Y2<PY>::E / 2; }

// columns kz0 .. kz0 + COLS of the block; every thread of the block calls it
template <int PY>
__device__ __forceinline__ void y2_columns(float2* __restrict__ B1, const float* __restrict__ Kc,
                                           const float2* __restrict__ tw, long kz0, int Ny, int Q, float2* lds) {
    using Y = Y2<PY>;
    constexpr int E = Y::E, G = Y::G, hy = PY / 2 + 1;
    constexpr bool WS = G <= 64;
    const int c = threadIdx.x / Y::W, r = threadIdx.x % Y::W, li = r / G, g = r % G;
    const long kz = kz0 + li;
    const bool ok = kz < Q;
    float2* p = B1 + ((long)c * Q + (ok ? kz : 0)) * Ny;
    float2* line = lds + (c * Y::COLS + li) * Y::LINE;
    float2 v[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int i = g + G * e;
        v[e] = (!y2_pad<PY>(e) && ok && i < Ny) ? p[i] : make_float2(0.f, 0.f);
    }
    // this component's diagonal value and, for y and z, kyz
    float kd[E], ko[E];
    auto load_kernel = [&]() {
        const float* K = Kc + (ok ? kz : 0) * hy;
        const long cs = (long)Q * hy;
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int ky = g + G * e, kyp = ky > PY / 2 ? PY - ky : ky;
            kd[e] = K[c * cs + kyp];
            ko[e] = c ? K[3 * cs + kyp] : 0.f;
        }
    };
    if constexpr (WS) load_kernel();
    const float2* t = tw;
    if constexpr (Y::TWL) {
        float2* twl = lds + 3 * Y::COLS * Y::LINE;
        for (int i = threadIdx.x; i < PY; i += Y::NT) twl[i] = tw[i];
        t = twl;
        __syncthreads();
    }
    reg_fft<float, PY, -1, 1, E, WS>(v, g, line, t);
    if (c) {
#pragma unroll
        for (int e = 0; e < E; e++) line[g + G * e] = v[e];
    }
    if constexpr (!WS) load_kernel();
    __syncthreads();
    {
        GK_FFT_FP
        const float2* other = lds + ((3 - c) * Y::COLS + li) * Y::LINE;  // the z line for y, the y line for z
#pragma unroll
        for (int e = 0; e < E; e++) {
            const float k = kd[e], kyz = g + G * e > PY / 2 ? -ko[e] : ko[e];
            const float2 a = v[e];
            if (c == 0) {
                v[e] = make_float2(a.x * k, a.y * k);
            } else {
                const float2 o = other[g + G * e];
                if (c == 1) v[e] = make_float2(a.x * k + o.x * kyz, a.y * k + o.y * kyz);
                else v[e] = make_float2(o.x * kyz + a.x * k, o.y * kyz + a.y * k);
            }
        }
    }
    __syncthreads();  // the y and z lines become exchange buffers again
    reg_fft<float, PY, +1, 1, E, WS>(v, g, line, t);
    if (ok)
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int i = g + G * e;
            if (!y2_pad<PY>(e) && i < Ny) p[i] = v[e];
        }
}

// single simulation: a block walks nit column sets strided by the grid
template <int PY>
__global__ __launch_bounds__(Y2<PY>::NT) __attribute__((amdgpu_waves_per_eu(Y2<PY>::G > 128 ? 6 : 1))) void k_y2r(
    float2* __restrict__ B1, const float* __restrict__ Kc, const float2* __restrict__ tw, const EngineState* st, int Ny,
    int Q, int nit) {
    __shared__ float2 lds[Y2<PY>::LDS];
    if (st && !st->trial_active) return;
    for (int it = 0; it < nit; it++) {
        if (it) __syncthreads();
        y2_columns<PY>(B1, Kc, tw, ((long)it * gridDim.x + blockIdx.x) * Y2<PY>::COLS, Ny, Q, lds);
    }
}

}  // namespace gk
