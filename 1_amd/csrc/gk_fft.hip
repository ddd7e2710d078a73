// Padded real FFT plan (drop-in for gpu_fft0.cu:30-112) and the generic
// line-transform kernels it is built from.
//
// The reference runs cuFFT over the whole zero-padded volume after zeroing it
// (gpu_fft0.cu:96-101).  Here the transform is split per axis and only lines
// that can be non-zero are transformed:
//   forward: Z real->complex on the Nx*Ny input rows (padding done while
//            loading), Y on the Nx planes (rows >= Ny are known zeros),
//            X on every (ky,kz) column (planes >= Nx are known zeros);
//   inverse: X on every column, Y on the Nx planes only, Z complex->real on
//            the Nx*Ny output rows only (the unpad is the store).
// No scratch zeroing and no separate pad/unpad launches are needed.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../include/gpukern.h"
#include "fft_device.h"
#include "gk_enqueue.h"
#include "gk_fft.h"

namespace gk {

// ----------------------------------------------------------------------------
// generic line transform: line l starts at (l / n_inner)*outer + (l % n_inner)*inner,
// elements at stride `estride`.  A block handles NL consecutive lines.  Only the
// first `nvalid` inputs are read (the rest are zero padding) and only the first
// `nkeep` outputs are stored.
template <typename T, int L, int DIR, int NL, int NT>
__global__ __launch_bounds__(NT) void k_fft_lines(C2<T>* __restrict__ data, const C2<T>* __restrict__ tw,
                                                  long nlines, long n_inner, long inner, long outer, long estride,
                                                  int nvalid, int nkeep) {
    constexpr int LS = L + 1;
    __shared__ C2<T> lds[NL * LS];
    const long l0 = (long)blockIdx.x * NL;
    const bool col = estride != 1;
    auto pos = [&](int t, int n, int& i, int& e) {
        if (col) {
            i = t % NL;
            e = t / NL;
        } else {
            i = t / n;
            e = t % n;
        }
    };
    batched_copy<C2<T>, NT>(
        NL * nvalid,
        [&](int t) {
            int i, e;
            pos(t, nvalid, i, e);
            const long l = l0 + i;
            return l < nlines ? data[(l / n_inner) * outer + (l % n_inner) * inner + e * estride] : mk<T>(0, 0);
        },
        [&](int t, C2<T> v) {
            int i, e;
            pos(t, nvalid, i, e);
            lds[i * LS + e] = v;
        });
    __syncthreads();
    fft_lds<T, L, DIR, NL, NT>(lds, LS, tw, nvalid);
    for (int t = threadIdx.x; t < NL * nkeep; t += NT) {
        int i, e;
        if (col) {
            i = t % NL;
            e = t / NL;
        } else {
            i = t / nkeep;
            e = t % nkeep;
        }
        const long l = l0 + i;
        if (l < nlines) data[(l / n_inner) * outer + (l % n_inner) * inner + e * estride] = lds[i * LS + e];
    }
}

// ----------------------------------------------------------------------------
// Register transforms (FP32, 2^a and 3 * 2^a).  A line is held by G lanes with
// up to 8 (2^a) or 12 (3 * 2^a) elements each, so a lane keeps 16-24 data
// registers whatever the length, and the radix passes exchange through LDS.
//
// Strided lines (Y and X of the drop-in layout): 2^sh neighbouring lines per
// block, line index fastest over the lanes, so a load touches runs of 2^sh x 8 B;
// the exchange buffers are interleaved the same way.  Contiguous rows: lane
// index fastest.  All of a lane's loads and the block's copy of the twiddle
// table are issued together, one memory latency for the whole kernel (the LDS
// Stockham kernels these replace read the table from global memory in every
// pass).  Strided lines go 16 (short lengths more) to a block, whole 128 B cache
// lines: with 4, for more blocks, neighbours on other XCDs wrote parts of the same
// line.  Threads and LDS allow that up to length 384: 8 lines at 512, 4 at 768 and
// 1024, 2 at 1536 and 2048, one at 3072 and 4096 share parts of cache lines.  Rows go
// as many to a block as leave about two blocks per CU: small transforms are
// latency-bound and need the CUs, not the occupancy.
// Measured per launch (before / now): 2064 lines of 256 12.9 / 6.9 us (4 lines a
// block 9.0), 33024 of 32 8.0 / 5.5 us, 2048 rows of 256 reals 8.9 / 4.3 us; 64 rows
// of 512 12.4 / 4.0 us.
constexpr int line_E(int L) { return L % 3 == 0 ? (L < 12 ? L : 12) : (L < 8 ? L : 8); }
constexpr int line_G(int L) { return L / line_E(L); }
constexpr int line_buf(int L) { return L + L / 8 + 1; }

template <int L, int DIR>
__global__ __launch_bounds__(1024) void k_lines_reg(float2* __restrict__ data, const float2* __restrict__ tw,
                                                    LineArgs a, int sh) {
    constexpr int E = line_E(L), G = line_G(L);
    extern __shared__ float2 dyn_lines[];
    float2* twl = dyn_lines;
    float2* buf = dyn_lines + L;
    const int i = threadIdx.x & ((1 << sh) - 1), g = threadIdx.x >> sh;
    const unsigned l = (blockIdx.x << sh) + i;
    const bool ok = l < a.nlines;
    float2* p = data + blockIdx.y * a.cstride + a.start(ok ? l : 0);
    float2 v[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int n = g + G * e;
        v[e] = (ok && n < a.nvalid) ? p[n * a.estride] : make_float2(0.f, 0.f);
    }
    for (int t = threadIdx.x; t < L; t += G << sh) twl[t] = tw[t];
    __syncthreads();
    reg_fft<float, L, DIR, 1, E, false>(v, g, StridedBuf{buf + i, sh}, twl);
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int n = g + G * e;
        if (ok && n < a.nkeep) p[n * a.estride] = v[e];
    }
}

// rows of n_real floats -> M+1 complex (real transform of length P = 2M, zero padded)
template <int M>
__global__ __launch_bounds__(1024) void k_rows_r2c_reg(const float* __restrict__ in, float2* __restrict__ out,
                                                       const float2* __restrict__ twM, const float2* __restrict__ twP,
                                                       RowArgs a, int nr) {
    constexpr int E = line_E(M), G = line_G(M);
    extern __shared__ float2 dyn_lines[];
    float2* twl = dyn_lines;
    const int g = threadIdx.x % G, row = threadIdx.x / G;
    float2* buf = dyn_lines + M + row * line_buf(M);
    const unsigned r = blockIdx.x * nr + row;
    const bool ok = r < a.nrows;
    const float* src = in + blockIdx.y * a.real_comp + a.real_at(ok ? r : 0);
    float2 v[E], wp[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int n = g + G * e;
        float2 x = make_float2(0.f, 0.f);
        if (a.vec) {
            if (ok && 2 * n < a.n_real) x = *reinterpret_cast<const float2*>(src + 2 * n);
        } else {
            if (ok && 2 * n < a.n_real) x.x = src[2 * n];
            if (ok && 2 * n + 1 < a.n_real) x.y = src[2 * n + 1];
        }
        v[e] = x;
        wp[e] = twP[n];
    }
    for (int t = threadIdx.x; t < M; t += G * nr) twl[t] = twM[t];
    __syncthreads();
    reg_fft<float, M, -1, 1, E, false>(v, g, buf, twl);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < E; e++) buf[g + G * e] = v[e];
    __syncthreads();
    if (!ok) return;
    float2* dst = out + blockIdx.y * a.cplx_comp + a.cplx_at(r);
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int k = g + G * e;
        dst[k] = r2c_split<float>(v[e], buf[k ? M - k : 0], wp[e]);
    }
    if (g == 0) dst[M] = make_float2(v[0].x - v[0].y, 0.f);
}

// M+1 complex per row -> first n_real floats of the length-2M real inverse transform
template <int M>
__global__ __launch_bounds__(1024) void k_rows_c2r_reg(const float2* __restrict__ in, float* __restrict__ out,
                                                       const float2* __restrict__ twM, const float2* __restrict__ twP,
                                                       RowArgs a, int nr) {
    constexpr int E = line_E(M), G = line_G(M);
    extern __shared__ float2 dyn_lines[];
    float2* twl = dyn_lines;
    const int g = threadIdx.x % G, row = threadIdx.x / G;
    float2* buf = dyn_lines + M + row * line_buf(M);
    const unsigned r = blockIdx.x * nr + row;
    const bool ok = r < a.nrows;
    const float2* src = in + blockIdx.y * a.cplx_comp + a.cplx_at(ok ? r : 0);
    float2 v[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int k = g + G * e;
        v[e] = c2r_merge<float>(src[k], src[M - k], twP[k]);
    }
    for (int t = threadIdx.x; t < M; t += G * nr) twl[t] = twM[t];
    __syncthreads();
    reg_fft<float, M, +1, 1, E, false>(v, g, buf, twl);
    if (!ok) return;
    float* dst = out + blockIdx.y * a.real_comp + a.real_at(r);
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int n = g + G * e;
        if (a.vec) {
            if (2 * n < a.n_real) *reinterpret_cast<float2*>(dst + 2 * n) = v[e];
        } else {
            if (2 * n < a.n_real) dst[2 * n] = v[e].x;
            if (2 * n + 1 < a.n_real) dst[2 * n + 1] = v[e].y;
        }
    }
}

// ----------------------------------------------------------------------------
// dispatch over the supported compile-time lengths
constexpr int kFFTThreads = 256;
constexpr int pow2floor(int v) {
    int p = 1;
    while (p * 2 <= v) p *= 2;
    return p;
}
template <typename T> constexpr int lines_per_block(int L) {
    int n = 71680 / ((L + 1) * (int)sizeof(C2<T>));
    n = n < 1 ? 1 : (n > 16 ? 16 : n);
    return pow2floor(n);
}

#define GK_FOR_EACH_POW2(X) X(1) X(2) X(4) X(8) X(16) X(32) X(64) X(128) X(256) X(512) X(1024) X(2048) X(4096)

bool fft_length_supported(int L) {
    switch (L) {
#define GK_CASE(n) case n:
        GK_FOR_EACH_POW2(GK_CASE)
#undef GK_CASE
        return true;
    default: return false;
    }
}

template <typename T, int DIR>
void fft_lines(C2<T>* data, int L, long nlines, long n_inner, long inner, long outer, long estride, int nvalid,
               int nkeep, hipStream_t s) {
    if (nlines <= 0) return;
    const C2<T>* tw;
    if constexpr (sizeof(T) == 4) tw = twiddle_f32(L);
    else tw = twiddle_f64(L);
    switch (L) {
#define GK_CASE(n)                                                                                              \
    case n: {                                                                                                   \
        constexpr int NL = lines_per_block<T>(n);                                                               \
        k_fft_lines<T, n, DIR, NL, kFFTThreads><<<div_up(nlines, NL), kFFTThreads, 0, s>>>(                     \
            data, tw, nlines, n_inner, inner, outer, estride, nvalid, nkeep);                                   \
        break;                                                                                                  \
    }
        GK_FOR_EACH_POW2(GK_CASE)
#undef GK_CASE
    default: fprintf(stderr, "libgpukern: FFT length %d is not supported\n", L); abort();
    }
    GK_LAUNCH_CHECK();
}

template void fft_lines<double, -1>(double2*, int, long, long, long, long, long, int, int, hipStream_t);
template void fft_lines<double, +1>(double2*, int, long, long, long, long, long, int, int, hipStream_t);

// 2^a up to 4096 and 3 * 2^a up to 3072
#define GK_FOR_EACH_REG(X) GK_FOR_EACH_POW2(X) X(3) X(6) X(12) X(24) X(48) X(96) X(192) X(384) X(768) X(1536) X(3072)

bool fft_reg_length(int L) {
    switch (L) {
#define GK_CASE(n) case n:
        GK_FOR_EACH_REG(GK_CASE)
#undef GK_CASE
        return true;
    default: return false;
    }
}

// log2 of the lines per block: 16 (128 B runs, a cache line) or as many more as 256
// threads take, fewer where they pass 1024 threads or 60 KB of LDS (8 at length 512
// down to one at 3072 and at 4096, whose line takes 70 KB), and down to 4 (32 B runs)
// while the launch has under 64 blocks of more than a wave
static int lines_shift(int L, int G, unsigned nlines) {
    int sh = 4;
    while ((G << (sh + 1)) <= 256) sh++;
    while (sh > 0 && ((G << sh) > 1024 || (((line_buf(L) << sh) + L) * 8) > 60 * 1024)) sh--;
    while (sh > 2 && (G << (sh - 1)) >= 64 && (nlines >> sh) < 64) sh--;
    return sh;
}
// rows per block: 256 threads, fewer while the launch has under 512 blocks and a block a whole wave
static int rows_per_launch_block(int M, int G, unsigned nrows) {
    int nr = 1;
    while (2 * nr * G <= 256 && (2 * nr * line_buf(M) + M) * 8 <= 60 * 1024) nr *= 2;
    while (nr > 1 && nr / 2 * G >= 64 && nrows / nr < 512) nr /= 2;
    return nr;
}

template <int DIR> void fft_lines_reg(float2* data, int L, const LineArgs& a, hipStream_t s) {
    if (a.nlines == 0) return;
    const float2* tw = twiddle_f32(L);
    switch (L) {
#define GK_CASE(n)                                                                                              \
    case n: {                                                                                                   \
        const int sh = lines_shift(n, line_G(n), a.nlines * a.ncomp);                                                     \
        k_lines_reg<n, DIR><<<dim3(div_up(a.nlines, 1L << sh), a.ncomp), line_G(n) << sh, ((line_buf(n) << sh) + n) * 8, s>>>( \
            data, tw, a, sh);                                                                                   \
        break;                                                                                                  \
    }
        GK_FOR_EACH_REG(GK_CASE)
#undef GK_CASE
    default: fprintf(stderr, "libgpukern: FFT length %d is not supported\n", L); abort();
    }
    GK_LAUNCH_CHECK();
}
template void fft_lines_reg<-1>(float2*, int, const LineArgs&, hipStream_t);
template void fft_lines_reg<+1>(float2*, int, const LineArgs&, hipStream_t);

void fft_rows_r2c_reg(const float* in, float2* out, int P, const RowArgs& a, hipStream_t s) {
    const int M = P / 2;
    const float2* twM = twiddle_f32(M);
    const float2* twP = twiddle_f32(P);
    switch (M) {
#define GK_CASE(n)                                                                                       \
    case n: {                                                                                            \
        const int nr = rows_per_launch_block(n, line_G(n), a.nrows * a.ncomp);                                     \
        k_rows_r2c_reg<n><<<dim3(div_up(a.nrows, nr), a.ncomp), line_G(n) * nr, (line_buf(n) * nr + n) * 8, s>>>(       \
            in, out, twM, twP, a, nr);                                                                   \
        break;                                                                                           \
    }
        GK_FOR_EACH_REG(GK_CASE)
#undef GK_CASE
    default: fprintf(stderr, "libgpukern: real FFT length %d is not supported\n", P); abort();
    }
    GK_LAUNCH_CHECK();
}

void fft_rows_c2r_reg(const float2* in, float* out, int P, const RowArgs& a, hipStream_t s) {
    const int M = P / 2;
    const float2* twM = twiddle_f32(M);
    const float2* twP = twiddle_f32(P);
    switch (M) {
#define GK_CASE(n)                                                                                       \
    case n: {                                                                                            \
        const int nr = rows_per_launch_block(n, line_G(n), a.nrows * a.ncomp);                                     \
        k_rows_c2r_reg<n><<<dim3(div_up(a.nrows, nr), a.ncomp), line_G(n) * nr, (line_buf(n) * nr + n) * 8, s>>>(       \
            in, out, twM, twP, a, nr);                                                                   \
        break;                                                                                           \
    }
        GK_FOR_EACH_REG(GK_CASE)
#undef GK_CASE
    default: fprintf(stderr, "libgpukern: real FFT length %d is not supported\n", P); abort();
    }
    GK_LAUNCH_CHECK();
}

// 3-D complex FFT of [n0][n1][n2] in FP64 (kernel setup), all lines.
void fft3_c2c_f64(double2* d, const int n[3], int dir, hipStream_t s) {
    const long n12 = (long)n[1] * n[2];
    if (dir < 0) {
        if (n[2] > 1) fft_lines_any<double, -1>(d, n[2], (long)n[0] * n[1], (long)n[0] * n[1], n[2], 0, 1, n[2], n[2], s);
        if (n[1] > 1) fft_lines_any<double, -1>(d, n[1], (long)n[0] * n[2], n[2], 1, n12, n[2], n[1], n[1], s);
        if (n[0] > 1) fft_lines_any<double, -1>(d, n[0], n12, n12, 1, 0, n12, n[0], n[0], s);
    } else {
        if (n[2] > 1) fft_lines_any<double, +1>(d, n[2], (long)n[0] * n[1], (long)n[0] * n[1], n[2], 0, 1, n[2], n[2], s);
        if (n[1] > 1) fft_lines_any<double, +1>(d, n[1], (long)n[0] * n[2], n[2], 1, n12, n[2], n[1], n[1], s);
        if (n[0] > 1) fft_lines_any<double, +1>(d, n[0], n12, n12, 1, 0, n12, n[0], n[0], s);
    }
}

}  // namespace gk

// ----------------------------------------------------------------------------
// drop-in plan
using namespace gk;

// gpuFFT3dPlan_forward_noalloc refuses plans above this many elements of what
// its contract counts (forward_scratch_elems).
constexpr size_t kFFTScratchElems = size_t(4) << 20;

struct gpuFFT3dPlan {
    int size[3];
    int padded[3];
    int pzc;
};

namespace gk {
// rows, then columns; twiddle and chirp tables come from the plan's construction
void enq_fft_forward(gpuFFT3dPlan* p, const float* real, long real_stride, float* cplx, long cplx_stride, int nc) {
    const int N0 = p->size[0], N1 = p->size[1], N2 = p->size[2];
    const int P0 = p->padded[0], P1 = p->padded[1], P2 = p->padded[2], Q = p->pzc;
    float2* out = (float2*)cplx;
    const long cs = cplx_stride / 2;
    hipStream_t s = stream();
    // Z: real rows (x<N0, y<N1) -> out[x][y][0..Q)
    fft_rows_r2c_any(real, out, P2, (long)N0 * N1, N1, N2, (long)N1 * N2, Q, (long)P1 * Q, N2, s, nc, real_stride, cs);
    // Y: columns (x<N0, kz) over y; rows y>=N1 are zero padding and not read
    if (P1 > 1) fft_lines_any<float, -1>(out, P1, (long)N0 * Q, Q, 1, (long)P1 * Q, Q, N1, P1, s, nc, cs);
    // X: every (ky,kz) column; planes x>=N0 are zero padding and not read
    if (P0 > 1) fft_lines_any<float, -1>(out, P0, (long)P1 * Q, (long)P1 * Q, 1, 0, (long)P1 * Q, N0, P0, s, nc, cs);
}
void enq_fft_inverse(gpuFFT3dPlan* p, float* cplx, long cplx_stride, float* real, long real_stride, int nc) {
    const int N0 = p->size[0], N1 = p->size[1], N2 = p->size[2];
    const int P0 = p->padded[0], P1 = p->padded[1], P2 = p->padded[2], Q = p->pzc;
    float2* in = (float2*)cplx;
    const long cs = cplx_stride / 2;
    hipStream_t s = stream();
    // X: all columns, only planes x<N0 are kept
    if (P0 > 1) fft_lines_any<float, +1>(in, P0, (long)P1 * Q, (long)P1 * Q, 1, 0, (long)P1 * Q, P0, N0, s, nc, cs);
    // Y: columns of the kept planes, only rows y<N1 are kept
    if (P1 > 1) fft_lines_any<float, +1>(in, P1, (long)N0 * Q, Q, 1, (long)P1 * Q, Q, P1, N1, s, nc, cs);
    // Z: complex rows (x<N0, y<N1) -> first N2 reals
    fft_rows_c2r_any(in, real, P2, (long)N0 * N1, N1, Q, (long)P1 * Q, N2, (long)N1 * N2, N2, s, nc, cs, real_stride);
}
}  // namespace gk

extern "C" {

gpuFFT3dPlan* new_gpuFFT3dPlan_padded(int* size, int* paddedSize) {
    GK_ASSERT(paddedSize[0] > 0 && paddedSize[1] > 0 && paddedSize[2] > 1,
              "new_gpuFFT3dPlan_padded: padded size %d x %d x %d", paddedSize[0], paddedSize[1], paddedSize[2]);
    for (int i = 0; i < 3; i++)
        GK_ASSERT(size[i] > 0 && size[i] <= paddedSize[i], "new_gpuFFT3dPlan_padded: size[%d]=%d padded=%d", i,
                  size[i], paddedSize[i]);
    gpuFFT3dPlan* p = new gpuFFT3dPlan;
    for (int i = 0; i < 3; i++) {
        p->size[i] = size[i];
        p->padded[i] = paddedSize[i];
    }
    p->pzc = paddedSize[2] / 2 + 1;
    // the twiddle and chirp tables of both directions are built here, once, so
    // that no transform call has to allocate them (without a device they are
    // built by the first transform instead)
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) == hipSuccess && ndev > 0) {
        for (int dir = -1; dir <= 1; dir += 2) {
            fft_rows_any_tables(paddedSize[2], dir);
            if (paddedSize[1] > 1) fft_lines_any_tables(paddedSize[1], dir);
            if (paddedSize[0] > 1) fft_lines_any_tables(paddedSize[0], dir);
        }
    }
    return p;
}

void delete_gpuFFT3dPlan(gpuFFT3dPlan* plan) { delete plan; }

int gpuFFT3dPlan_normalization(gpuFFT3dPlan* p) { return p->padded[0] * p->padded[1] * p->padded[2]; }

// The no-allocation transform's size limit counts, for the largest pass, the
// packed rows and padded lines of lengths that are no power of two (the transforms
// themselves use registers and LDS only, for every plan).
static size_t forward_scratch_elems(const gpuFFT3dPlan* p) {
    const long N0 = p->size[0], N1 = p->size[1];
    const int P0 = p->padded[0], P1 = p->padded[1], P2 = p->padded[2], Q = p->pzc;
    const int H = P2 % 2 == 0 ? P2 / 2 : P2;
    size_t need = 0;
    if (P2 % 2 || !fft_length_supported(H)) need = (size_t)(N0 * N1) * (H + fft_blue_length(H));
    if (P1 > 1) need = std::max(need, (size_t)(N0 * Q) * fft_blue_length(P1));
    if (P0 > 1) need = std::max(need, (size_t)P1 * Q * fft_blue_length(P0));
    return need;
}

// The row pass reads rows of one length and stores rows of another, block by
// block in any order, so real data that share memory with the spectrum go
// through an array of their own (from the engine's cache of device memory).
static float* aside_if_shared(const gpuFFT3dPlan* p, const float* real, const float* cplx) {
    const long n = (long)p->size[0] * p->size[1] * p->size[2], nc = (long)p->padded[0] * p->padded[1] * p->pzc * 2;
    return real < cplx + nc && cplx < real + n ? (float*)cached_malloc(n * sizeof(float)) : nullptr;
}
static size_t real_bytes(const gpuFFT3dPlan* p) { return (size_t)p->size[0] * p->size[1] * p->size[2] * sizeof(float); }
static float* enq_forward_any(gpuFFT3dPlan* p, const float* input, float* output) {
    float* aside = aside_if_shared(p, input, output);
    if (aside) GK_CHECK(hipMemcpyAsync(aside, input, real_bytes(p), hipMemcpyDeviceToDevice, stream()));
    enq_fft_forward(p, aside ? aside : input, 0, output, 0, 1);
    return aside;
}

void gpuFFT3dPlan_forward(gpuFFT3dPlan* p, float* input, float* output) {
    float* aside = enq_forward_any(p, input, output);
    sync();
    cached_free(aside);
}

void gpuFFT3dPlan_forward_noalloc(gpuFFT3dPlan* p, float* input, float* output) {
    const size_t need = forward_scratch_elems(p);
    GK_ASSERT(need <= kFFTScratchElems,
              "gpuFFT3dPlan_forward_noalloc: padded size %d x %d x %d needs %zu scratch elements (8 bytes each); "
              "the maximum is %zu (use gpuFFT3dPlan_forward)",
              p->padded[0], p->padded[1], p->padded[2], need, kFFTScratchElems);
    tables_frozen(true);
    float* aside = enq_forward_any(p, input, output);
    tables_frozen(false);
    sync();
    cached_free(aside);
}

void gpuFFT3dPlan_inverse(gpuFFT3dPlan* p, float* input, float* output) {
    float* aside = aside_if_shared(p, output, input);
    enq_fft_inverse(p, input, 0, aside ? aside : output, 0, 1);
    if (aside) GK_CHECK(hipMemcpyAsync(output, aside, real_bytes(p), hipMemcpyDeviceToDevice, stream()));
    sync();
    cached_free(aside);
}

}  // extern "C"
