// Transforms of any length for the drop-in plan (gpu_fft0.cu:30-112 accepts
// every size cuFFT does; the Go driver pads each axis to 2N, kernel.go:80-90,
// so lengths such as 2^a 3^b 5^c 7^d and 2p for a prime p all occur).
//
// Lengths whose factors are 2, 3, 5 and 7 (beyond the register lengths of
// gk_fft.hip) run as Stockham passes in LDS with a runtime list of radices (8, 4,
// 2, 3, 5, 7), up to 8 neighbouring lines per block.  Any other length uses
// Bluestein's chirp-z identity nk = (n^2 + k^2 - (k-n)^2)/2:
//   X[k] = w[k] sum_n (x[n] w[n]) conj(w)[k-n],   w[n] = exp(DIR pi i n^2 / L),
// i.e. a circular convolution of length Lp >= 2L-1 (a power of two), both of whose
// transforms run in registers in one kernel; the chirp and the transformed filter
// are computed on the host in long double.  Real rows of even length P use the
// half-length complex transform (same split / merge as the power-of-two path);
// odd P (a periodic axis) uses the full complex transform of length P.
#include <hip/hip_runtime.h>

#include <cmath>
#include <complex>
#include <map>
#include <mutex>
#include <vector>

#include "fft_device.h"
#include "gk_common.h"
#include "gk_fft.h"

namespace gk {

struct RadixList {
    int n;
    int r[32];
};

static bool factor_radices(int L, RadixList& rl) {
    rl.n = 0;
    int rem = L;
    while (rem > 1) {
        const int R = rem % 8 == 0 ? 8 : rem % 4 == 0 ? 4 : rem % 2 == 0 ? 2 : rem % 3 == 0 ? 3 : rem % 5 == 0 ? 5
                                                                                                 : rem % 7 == 0 ? 7
                                                                                                                : 0;
        if (!R || rl.n == 32) return false;
        rl.r[rl.n++] = R;
        rem /= R;
    }
    return true;
}

// one Stockham pass of radix RR over 2^sh lines of L held interleaved in LDS
// (element i of line q at (i << sh) + q, src -> dst)
template <typename T, int DIR, int RR>
__device__ __forceinline__ void stockham_pass_rt(const C2<T>* src, C2<T>* dst, unsigned L, unsigned NS, int sh,
                                                 const C2<T>* __restrict__ tw) {
    const unsigned nb = L / RR, mask = (1u << sh) - 1;
    for (unsigned b = threadIdx.x; b < (nb << sh); b += blockDim.x) {
        const unsigned q = b & mask, j = b >> sh, jq = j / NS, k = j - jq * NS;
        C2<T> v[RR];
#pragma unroll
        for (unsigned r = 0; r < RR; r++) v[r] = src[((j + r * nb) << sh) + q];
        if (NS > 1) {
            const unsigned step = L / (NS * RR);
#pragma unroll
            for (unsigned r = 1; r < RR; r++) v[r] = cmul<T>(v[r], twid<T, DIR>(tw, r * k * step));
        }
        dft<T, RR, DIR>(v);
        const unsigned base = jq * NS * RR + k;
#pragma unroll
        for (unsigned r = 0; r < RR; r++) dst[((base + r * NS) << sh) + q] = v[r];
    }
}
// all passes; returns the buffer holding the result (every thread of the block calls it)
template <typename T, int DIR>
__device__ __forceinline__ C2<T>* stockham_rt(C2<T>* a, C2<T>* b, int L, const RadixList& rl, int sh,
                                              const C2<T>* __restrict__ tw) {
    int NS = 1;
    for (int p = 0; p < rl.n; p++) {
        const int R = rl.r[p];
        switch (R) {
        case 8: stockham_pass_rt<T, DIR, 8>(a, b, L, NS, sh, tw); break;
        case 4: stockham_pass_rt<T, DIR, 4>(a, b, L, NS, sh, tw); break;
        case 2: stockham_pass_rt<T, DIR, 2>(a, b, L, NS, sh, tw); break;
        case 3: stockham_pass_rt<T, DIR, 3>(a, b, L, NS, sh, tw); break;
        case 5: stockham_pass_rt<T, DIR, 5>(a, b, L, NS, sh, tw); break;
        default: stockham_pass_rt<T, DIR, 7>(a, b, L, NS, sh, tw); break;
        }
        __syncthreads();
        C2<T>* t = a;
        a = b;
        b = t;
        NS *= R;
    }
    return a;
}

// Lines (LineArgs), 2^sh neighbours per block: strided lines load and store runs
// of 2^sh elements, contiguous ones (estride 1) along the line.  One line per
// block, the form this replaces, moved 8 B (16 B in FP64) per 64 B of memory: 1070
// lines of 150 11.2 us, now 7.7 us.
template <typename T, int DIR>
__global__ __launch_bounds__(256) void k_fft_lines_rt(C2<T>* __restrict__ data, const C2<T>* __restrict__ tw, int L,
                                                      RadixList rl, LineArgs la, int sh) {
    extern __shared__ __align__(16) unsigned char smem_rt[];
    C2<T>* a = reinterpret_cast<C2<T>*>(smem_rt);
    C2<T>* b = a + ((long)L << sh);
    const unsigned l0 = blockIdx.x << sh, mask = (1u << sh) - 1, nl = min(la.nlines - l0, 1u << sh);
    const bool col = la.estride != 1;
    data += blockIdx.y * la.cstride;
    for (unsigned t = threadIdx.x; t < ((unsigned)L << sh); t += blockDim.x) {
        const unsigned q = col ? t & mask : t / L, n = col ? t >> sh : t - q * L;
        const bool in = q < nl && (int)n < la.nvalid;
        a[(n << sh) + q] = in ? data[la.start(l0 + q) + (long)n * la.estride] : mk<T>(0, 0);
    }
    __syncthreads();
    a = stockham_rt<T, DIR>(a, b, L, rl, sh, tw);
    for (unsigned t = threadIdx.x; t < ((unsigned)la.nkeep << sh); t += blockDim.x) {
        const unsigned q = col ? t & mask : t / la.nkeep, n = col ? t >> sh : t - q * la.nkeep;
        if (q < nl) data[la.start(l0 + q) + (long)n * la.estride] = a[(n << sh) + q];
    }
}

// Real rows of length P: even P through the packed transform of H = P/2 and
// the split, odd P as H = P complex numbers
__global__ __launch_bounds__(256) void k_rows_r2c_rt(const float* __restrict__ in, float2* __restrict__ out,
                                                     const float2* __restrict__ tw, const float2* __restrict__ twP,
                                                     int H, int even, RadixList rl, RowArgs ra, int sh) {
    extern __shared__ __align__(16) unsigned char smem_rt[];
    float2* a = reinterpret_cast<float2*>(smem_rt);
    float2* b = a + ((long)H << sh);
    const unsigned r0 = blockIdx.x << sh, nr = min(ra.nrows - r0, 1u << sh);
    in += blockIdx.y * ra.real_comp;
    out += blockIdx.y * ra.cplx_comp;
    for (unsigned t = threadIdx.x; t < ((unsigned)H << sh); t += blockDim.x) {
        const unsigned q = t / H, n = t - q * H;
        float2 v = make_float2(0.f, 0.f);
        if (q < nr) {
            const float* row = in + ra.real_at(r0 + q);
            if (even) {
                if (2 * (int)n < ra.n_real) v.x = row[2 * n];
                if (2 * (int)n + 1 < ra.n_real) v.y = row[2 * n + 1];
            } else if ((int)n < ra.n_real) {
                v.x = row[n];
            }
        }
        a[(n << sh) + q] = v;
    }
    __syncthreads();
    a = stockham_rt<float, -1>(a, b, H, rl, sh, tw);
    const unsigned Q = even ? H + 1 : H / 2 + 1;
    for (unsigned t = threadIdx.x; t < (Q << sh); t += blockDim.x) {
        const unsigned q = t / Q, k = t - q * Q;
        if (q >= nr) continue;
        const float2 zk = a[((k == (unsigned)H ? 0 : k) << sh) + q];
        float2 X = zk;
        if (even) {
            if (k == (unsigned)H) X = make_float2(zk.x - zk.y, 0.f);
            else X = r2c_split<float>(zk, a[((k ? H - k : 0) << sh) + q], twP[k]);
        }
        out[ra.cplx_at(r0 + q) + k] = X;
    }
}

__global__ __launch_bounds__(256) void k_rows_c2r_rt(const float2* __restrict__ in, float* __restrict__ out,
                                                     const float2* __restrict__ tw, const float2* __restrict__ twP,
                                                     int H, int even, RadixList rl, RowArgs ra, int sh) {
    extern __shared__ __align__(16) unsigned char smem_rt[];
    float2* a = reinterpret_cast<float2*>(smem_rt);
    float2* b = a + ((long)H << sh);
    const unsigned r0 = blockIdx.x << sh, nr = min(ra.nrows - r0, 1u << sh);
    in += blockIdx.y * ra.cplx_comp;
    out += blockIdx.y * ra.real_comp;
    for (unsigned t = threadIdx.x; t < ((unsigned)H << sh); t += blockDim.x) {
        const unsigned q = t / H, k = t - q * H;
        float2 v = make_float2(0.f, 0.f);
        if (q < nr) {
            const float2* X = in + ra.cplx_at(r0 + q);
            if (even) v = c2r_merge<float>(X[k], X[H - k], twP[k]);
            else v = (int)k <= H / 2 ? X[k] : cconj<float>(X[H - k]);
        }
        a[(k << sh) + q] = v;
    }
    __syncthreads();
    a = stockham_rt<float, +1>(a, b, H, rl, sh, tw);
    const unsigned n_real = ra.n_real;
    for (unsigned t = threadIdx.x; t < (n_real << sh); t += blockDim.x) {
        const unsigned q = t / n_real, i = t - q * n_real;
        if (q >= nr) continue;
        const float2 y = a[((even ? i >> 1 : i) << sh) + q];
        out[ra.real_at(r0 + q) + i] = even && (i & 1) ? y.y : y.x;
    }
}

// log2 of the lines per block: 8 (64 B runs of float2), fewer where both buffers
// pass 48 KB or, down to 4, where the launch has under 512 blocks, and one where it
// has under 16 (9 lines of 210: the transform padded to 210 x 1 x 16 23.2 us with 4, 20.7 with one)
template <typename T> static int rt_shift(int L, unsigned nlines) {
    int sh = 3;
    while (sh > 0 && (2L * L * (long)sizeof(C2<T>) << sh) > 48 * 1024) sh--;
    while (sh > 2 && (nlines >> sh) < 512) sh--;
    while (sh > 0 && (nlines >> sh) < 16) sh--;
    return sh;
}

// ---------------------------------------------------------------- Bluestein
struct BlueTables {
    int L = 0, Lp = 0;
    float2* w = nullptr;  // chirp, L entries
    float2* B = nullptr;  // Lp-point transform of the conjugate chirp filter, divided by Lp
};

static void host_fft_pow2(std::vector<std::complex<long double>>& a, int sign) {
    const size_t n = a.size();
    for (size_t i = 1, j = 0; i < n; i++) {
        size_t bit = n >> 1;
        for (; j & bit; bit >>= 1) j ^= bit;
        j ^= bit;
        if (i < j) std::swap(a[i], a[j]);
    }
    const long double pi = 3.141592653589793238462643383279502884L;
    for (size_t len = 2; len <= n; len <<= 1) {
        for (size_t i = 0; i < n; i += len)
            for (size_t k = 0; k < len / 2; k++) {
                const long double ang = sign * 2 * pi * (long double)k / (long double)len;
                const std::complex<long double> w(cosl(ang), sinl(ang));
                const std::complex<long double> u = a[i + k], v = a[i + k + len / 2] * w;
                a[i + k] = u + v;
                a[i + k + len / 2] = u - v;
            }
    }
}

static const BlueTables& blue_tables(int L, int dir) {
    static std::mutex mu;
    static std::map<std::pair<int, int>, BlueTables> cache;
    std::lock_guard<std::mutex> lock(mu);
    auto it = cache.find({L, dir});
    if (it != cache.end()) return it->second;
    GK_ASSERT(!tables_frozen(), "chirp table of length %d is missing in a call that may not allocate", L);
    BlueTables t;
    t.L = L;
    t.Lp = 1;
    while (t.Lp < 2 * L - 1) t.Lp *= 2;
    const long double pi = 3.141592653589793238462643383279502884L;
    std::vector<std::complex<long double>> w(L), b(t.Lp, 0);
    for (int n = 0; n < L; n++) {
        const long long n2 = ((long long)n * n) % (2LL * L);  // exp(i pi n^2 / L) has period 2L in n^2
        const long double ang = dir * pi * (long double)n2 / (long double)L;
        w[n] = std::complex<long double>(cosl(ang), sinl(ang));
    }
    for (int m = 0; m < L; m++) {
        b[m] = std::conj(w[m]);
        if (m) b[t.Lp - m] = std::conj(w[m]);
    }
    host_fft_pow2(b, -1);
    std::vector<float2> hw(L), hB(t.Lp);
    for (int n = 0; n < L; n++) hw[n] = make_float2((float)w[n].real(), (float)w[n].imag());
    for (int k = 0; k < t.Lp; k++)
        hB[k] = make_float2((float)(b[k].real() / t.Lp), (float)(b[k].imag() / t.Lp));
    GK_CHECK(hipMalloc(&t.w, L * sizeof(float2)));
    GK_CHECK(hipMalloc(&t.B, t.Lp * sizeof(float2)));
    GK_CHECK(hipMemcpy(t.w, hw.data(), L * sizeof(float2), hipMemcpyHostToDevice));
    GK_CHECK(hipMemcpy(t.B, hB.data(), t.Lp * sizeof(float2), hipMemcpyHostToDevice));
    return cache.emplace(std::make_pair(L, dir), t).first->second;
}

// One kernel per transform: the chirped inputs go through the length-Lp forward
// transform, the filter, the inverse transform and the second chirp in registers
// (fft_device.h; E elements per lane, G lanes per line), and real rows are packed,
// split or merged at its ends.  L <= Lp / 2, so the upper half of each lane's
// inputs is zero and of its outputs dead at compile time.  The separate kernels
// this replaces (pack, chirp, transform, multiply, transform, chirp, split) moved
// the Lp-padded lines through memory eight times and allocated them per call:
// 750 rows of 212 reals (H = 106, Lp = 256) took 49 us and seven launches, now 6.3 us.
enum { BLUE_LINES = 0, BLUE_R2C = 1, BLUE_C2R = 2 };
constexpr int blue_G(int Lp) { return Lp / 8; }
constexpr int blue_buf(int Lp) { return Lp + Lp / 8 + 1; }

template <int Lp, int DIR>
__device__ __forceinline__ void blue_transform(float2* v, int g, StridedBuf buf, const float2* __restrict__ w,
                                               const float2* __restrict__ B, const float2* tw, int L) {
    constexpr int G = blue_G(Lp);
    float2 c[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int n = g + G * e;
        c[e] = n < L ? w[n] : make_float2(0.f, 0.f);
        v[e] = cmul<float>(v[e], c[e]);
        v[e + 4] = make_float2(0.f, 0.f);
    }
    reg_fft<float, Lp, -1, 1, 8, false>(v, g, buf, tw);
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = cmul<float>(v[e], B[g + G * e]);
    reg_fft<float, Lp, +1, 1, 8, false>(v, g, buf, tw);
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = cmul<float>(v[e], c[e]);
}

// strided lines: 2^sh neighbours per block, line index fastest (as k_lines_reg)
template <int Lp, int DIR>
__global__ __launch_bounds__(1024) void k_lines_blue(float2* __restrict__ data, const float2* __restrict__ w,
                                                     const float2* __restrict__ B, const float2* __restrict__ tw,
                                                     int L, LineArgs a, int sh) {
    constexpr int G = blue_G(Lp);
    extern __shared__ float2 dyn_blue[];
    float2* twl = dyn_blue;
    const int i = threadIdx.x & ((1 << sh) - 1), g = threadIdx.x >> sh;
    const unsigned l = (blockIdx.x << sh) + i;
    const bool ok = l < a.nlines;
    float2* p = data + blockIdx.y * a.cstride + a.start(ok ? l : 0);
    float2 v[8];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int n = g + G * e;
        v[e] = (ok && n < a.nvalid && n < L) ? p[n * a.estride] : make_float2(0.f, 0.f);
    }
    for (int t = threadIdx.x; t < Lp; t += G << sh) twl[t] = tw[t];
    __syncthreads();
    blue_transform<Lp, DIR>(v, g, StridedBuf{dyn_blue + Lp + i, sh}, w, B, twl, L);
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int n = g + G * e;
        if (ok && n < a.nkeep) p[n * a.estride] = v[e];
    }
}

// real rows through a transform of H = P/2 (even P) or H = P (odd) complex numbers
template <int Lp, int MODE>
__global__ __launch_bounds__(1024) void k_rows_blue(const float* __restrict__ rin, float* __restrict__ rout,
                                                    const float2* __restrict__ cin, float2* __restrict__ cout,
                                                    const float2* __restrict__ w, const float2* __restrict__ B,
                                                    const float2* __restrict__ tw, const float2* __restrict__ twP,
                                                    int H, int even, RowArgs a, int nr) {
    constexpr int G = blue_G(Lp);
    extern __shared__ float2 dyn_blue[];
    float2* twl = dyn_blue;
    const int g = threadIdx.x % G, row = threadIdx.x / G;
    float2* buf = dyn_blue + Lp + row * blue_buf(Lp);
    const unsigned r = blockIdx.x * nr + row;
    const bool ok = r < a.nrows;
    float2 v[8];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int n = g + G * e;
        float2 x = make_float2(0.f, 0.f);
        if (ok && n < H) {
            if constexpr (MODE == BLUE_R2C) {
                const float* src = rin + blockIdx.y * a.real_comp + a.real_at(r);
                if (even) {
                    if (2 * n < a.n_real) x.x = src[2 * n];
                    if (2 * n + 1 < a.n_real) x.y = src[2 * n + 1];
                } else if (n < a.n_real) {
                    x.x = src[n];
                }
            } else {
                const float2* X = cin + blockIdx.y * a.cplx_comp + a.cplx_at(r);
                if (even) x = c2r_merge<float>(X[n], X[H - n], twP[n]);
                else x = n <= H / 2 ? X[n] : cconj<float>(X[H - n]);
            }
        }
        v[e] = x;
    }
    for (int t = threadIdx.x; t < Lp; t += G * nr) twl[t] = tw[t];
    __syncthreads();
    blue_transform<Lp, MODE == BLUE_R2C ? -1 : +1>(v, g, StridedBuf{buf, 0}, w, B, twl, H);
    if constexpr (MODE == BLUE_R2C) {
        if (even) {  // uniform over the launch
            __syncthreads();
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (g + G * e < H) buf[g + G * e] = v[e];
            __syncthreads();
        }
        if (!ok) return;
        float2* dst = cout + blockIdx.y * a.cplx_comp + a.cplx_at(r);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int k = g + G * e;
            if (even) {
                if (k < H) dst[k] = r2c_split<float>(v[e], buf[k ? H - k : 0], twP[k]);
                if (k == 0) dst[H] = make_float2(v[e].x - v[e].y, 0.f);
            } else if (k <= H / 2) {
                dst[k] = v[e];
            }
        }
    } else {
        if (!ok) return;
        float* dst = rout + blockIdx.y * a.real_comp + a.real_at(r);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int n = g + G * e;
            if (n >= H) continue;
            if (even) {
                if (2 * n < a.n_real) dst[2 * n] = v[e].x;
                if (2 * n + 1 < a.n_real) dst[2 * n + 1] = v[e].y;
            } else if (n < a.n_real) {
                dst[n] = v[e].x;
            }
        }
    }
}

#define GK_FOR_EACH_BLUE(X) X(32) X(64) X(128) X(256) X(512) X(1024) X(2048) X(4096)

int fft_blue_length(int L) {
    RadixList rl;
    if (fft_length_supported(L) || factor_radices(L, rl)) return 0;
    int Lp = 1;
    while (Lp < 2 * L - 1) Lp *= 2;
    return Lp;
}

// lines (log2) and rows per block: the choices of k_lines_reg and k_rows_r2c_reg
static int blue_shift(int Lp, unsigned nlines) {
    const int G = Lp / 8;
    int sh = 3;
    while ((G << (sh + 1)) <= 256) sh++;
    while (sh > 0 && ((G << sh) > 1024 || (((blue_buf(Lp) << sh) + Lp) * 8) > 60 * 1024)) sh--;
    while (sh > 2 && (G << (sh - 1)) >= 64 && (nlines >> sh) < 512) sh--;
    return sh;
}
static int blue_rows(int Lp, unsigned nrows) {
    const int G = Lp / 8;
    int nr = 1;
    while (2 * nr * G <= 256 && (2 * nr * blue_buf(Lp) + Lp) * 8 <= 60 * 1024) nr *= 2;
    while (nr > 1 && nr / 2 * G >= 64 && nrows / nr < 512) nr /= 2;
    return nr;
}
template <int DIR> static void lines_blue(float2* data, int L, const LineArgs& a, hipStream_t s) {
    const BlueTables& bt = blue_tables(L, DIR);
    const float2* tw = twiddle_f32(bt.Lp);
    const int sh = blue_shift(bt.Lp, a.nlines * a.ncomp);
    switch (bt.Lp) {
#define GK_CASE(n)                                                                                               \
    case n:                                                                                                      \
        k_lines_blue<n, DIR><<<dim3(div_up(a.nlines, 1L << sh), a.ncomp), blue_G(n) << sh, ((blue_buf(n) << sh) + n) * 8, s>>>( \
            data, bt.w, bt.B, tw, L, a, sh);                                                                     \
        break;
        GK_FOR_EACH_BLUE(GK_CASE)
#undef GK_CASE
    default: GK_ASSERT(false, "FFT length %d is not supported", L);
    }
    GK_LAUNCH_CHECK();
}
template <int MODE>
static void rows_blue(const float* rin, float* rout, const float2* cin, float2* cout, int P, const RowArgs& a,
                      hipStream_t s) {
    const int even = P % 2 == 0, H = even ? P / 2 : P;
    const BlueTables& bt = blue_tables(H, MODE == BLUE_R2C ? -1 : +1);
    const float2* tw = twiddle_f32(bt.Lp);
    const float2* twP = even ? twiddle_f32(P) : nullptr;
    const int nr = blue_rows(bt.Lp, a.nrows * a.ncomp);
    switch (bt.Lp) {
#define GK_CASE(n)                                                                                                \
    case n:                                                                                                       \
        k_rows_blue<n, MODE><<<dim3(div_up(a.nrows, nr), a.ncomp), blue_G(n) * nr, (blue_buf(n) * nr + n) * 8, s>>>(             \
            rin, rout, cin, cout, bt.w, bt.B, tw, twP, H, even, a, nr);                                           \
        break;
        GK_FOR_EACH_BLUE(GK_CASE)
#undef GK_CASE
    default: GK_ASSERT(false, "FFT length %d is not supported", P);
    }
    GK_LAUNCH_CHECK();
}

// ---------------------------------------------------------------- any length
void fft_lines_any_tables(int L, int dir) {
    RadixList rl;
    if (fft_length_supported(L) || factor_radices(L, rl)) {
        twiddle_f32(L);
        return;
    }
    blue_tables(L, dir);
    twiddle_f32(fft_blue_length(L));
}

template <typename T, int DIR>
void fft_lines_any(C2<T>* data, int L, long nlines, long n_inner, long inner, long outer, long estride, int nvalid,
                   int nkeep, hipStream_t s, int ncomp, long cstride) {
    if (nlines <= 0) return;
    if constexpr (sizeof(T) == 8) {
        GK_ASSERT(ncomp == 1, "one FP64 transform per call");
        if (fft_length_supported(L)) {
            fft_lines<T, DIR>(data, L, nlines, n_inner, inner, outer, estride, nvalid, nkeep, s);
            return;
        }
    }
    GK_ASSERT(nlines < (1L << 31) && n_inner < (1L << 31), "FFT of %ld lines", nlines);
    const LineArgs a{(unsigned)nlines, (unsigned)n_inner, inner, outer, estride, nvalid, nkeep, ncomp, cstride};
    if constexpr (sizeof(T) == 4) {
        if (fft_reg_length(L)) {
            fft_lines_reg<DIR>(data, L, a, s);
            return;
        }
    }
    RadixList rl;
    if (factor_radices(L, rl)) {
        // FP64: up to 3072 (96 KB, one block per CU), which the engine pads 1025..1536 cells to
        constexpr int max_lds = sizeof(T) == 8 ? 96 * 1024 : 64 * 1024;
        GK_ASSERT(2L * L * (long)sizeof(C2<T>) <= max_lds, "FFT length %d is too long for one block", L);
        const C2<T>* tw;
        if constexpr (sizeof(T) == 4) {
            tw = twiddle_f32(L);
        } else {
            tw = twiddle_f64(L);
            GK_CHECK(hipFuncSetAttribute((const void*)k_fft_lines_rt<T, DIR>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                         max_lds));
        }
        const int sh = rt_shift<T>(L, a.nlines * ncomp);
        k_fft_lines_rt<T, DIR><<<dim3(div_up(nlines, 1L << sh), ncomp), 256, (2 * L * sizeof(C2<T>)) << sh, s>>>(data, tw, L, rl, a, sh);
        GK_LAUNCH_CHECK();
        return;
    }
    if constexpr (sizeof(T) == 4) lines_blue<DIR>(data, L, a, s);
    else GK_ASSERT(false, "FP64 FFT length %d is not supported", L);
}

template void fft_lines_any<float, -1>(float2*, int, long, long, long, long, long, int, int, hipStream_t, int,
                                        long);
template void fft_lines_any<float, +1>(float2*, int, long, long, long, long, long, int, int, hipStream_t, int,
                                        long);
template void fft_lines_any<double, -1>(double2*, int, long, long, long, long, long, int, int, hipStream_t, int,
                                        long);
template void fft_lines_any<double, +1>(double2*, int, long, long, long, long, long, int, int, hipStream_t, int,
                                        long);

void fft_rows_any_tables(int P, int dir) {
    const int H = P % 2 == 0 ? P / 2 : P;
    if (P % 2 == 0) twiddle_f32(P);
    fft_lines_any_tables(H, dir);
}

static RowArgs row_args(const void* real, long nrows, long n_inner, long real_inner, long real_outer, long cplx_inner,
                        long cplx_outer, int n_real, int ncomp, long real_comp, long cplx_comp) {
    GK_ASSERT(nrows < (1L << 31) && n_inner < (1L << 31), "FFT of %ld rows", nrows);
    const int vec = n_real % 2 == 0 && real_inner % 2 == 0 && real_outer % 2 == 0 && real_comp % 2 == 0 &&
                    (uintptr_t)real % 8 == 0;
    return RowArgs{(unsigned)nrows, (unsigned)n_inner, real_inner, real_outer, cplx_inner, cplx_outer, n_real, vec, ncomp,
                   real_comp, cplx_comp};
}

void fft_rows_r2c_any(const float* in, float2* out, int P, long nrows, long n_inner, long in_inner, long in_outer,
                      long out_inner, long out_outer, int n_real, hipStream_t s, int ncomp, long in_comp,
                      long out_comp) {
    if (nrows <= 0) return;
    GK_ASSERT(n_real <= P, "real FFT length %d (data %d)", P, n_real);
    const RowArgs a = row_args(in, nrows, n_inner, in_inner, in_outer, out_inner, out_outer, n_real, ncomp, in_comp,
                               out_comp);
    const int even = P % 2 == 0, H = even ? P / 2 : P;
    RadixList rl;
    if (even && fft_reg_length(H)) {
        fft_rows_r2c_reg(in, out, P, a, s);
    } else if (factor_radices(H, rl)) {
        GK_ASSERT(2L * H * 8 <= 65536, "FFT length %d is too long for one block", H);
        const int sh = rt_shift<float>(H, a.nrows * ncomp);
        k_rows_r2c_rt<<<dim3(div_up(nrows, 1L << sh), ncomp), 256, (2 * H * 8) << sh, s>>>(
            in, out, twiddle_f32(H), even ? twiddle_f32(P) : nullptr, H, even, rl, a, sh);
        GK_LAUNCH_CHECK();
    } else {
        rows_blue<BLUE_R2C>(in, nullptr, nullptr, out, P, a, s);
    }
}

void fft_rows_c2r_any(const float2* in, float* out, int P, long nrows, long n_inner, long in_inner, long in_outer,
                      long out_inner, long out_outer, int n_real, hipStream_t s, int ncomp, long in_comp,
                      long out_comp) {
    if (nrows <= 0) return;
    GK_ASSERT(n_real <= P, "real FFT length %d (data %d)", P, n_real);
    const RowArgs a = row_args(out, nrows, n_inner, out_inner, out_outer, in_inner, in_outer, n_real, ncomp, out_comp,
                               in_comp);
    const int even = P % 2 == 0, H = even ? P / 2 : P;
    RadixList rl;
    if (even && fft_reg_length(H)) {
        fft_rows_c2r_reg(in, out, P, a, s);
    } else if (factor_radices(H, rl)) {
        GK_ASSERT(2L * H * 8 <= 65536, "FFT length %d is too long for one block", H);
        const int sh = rt_shift<float>(H, a.nrows * ncomp);
        k_rows_c2r_rt<<<dim3(div_up(nrows, 1L << sh), ncomp), 256, (2 * H * 8) << sh, s>>>(
            in, out, twiddle_f32(H), even ? twiddle_f32(P) : nullptr, H, even, rl, a, sh);
        GK_LAUNCH_CHECK();
    } else {
        rows_blue<BLUE_C2R>(nullptr, out, in, nullptr, P, a, s);
    }
}

}  // namespace gk
