// Host-side launchers of the FFT kernels (gk_fft.hip), shared by the
// drop-in plan and the engine.
#pragma once
#include <hip/hip_runtime.h>

#include "fft_device.h"

namespace gk {

bool fft_length_supported(int L);

// Lines of length L: line l starts at (l / n_inner)*outer + (l % n_inner)*inner,
// elements at stride estride (in complex elements).  Reads the first nvalid
// elements (the rest are zero padding), stores the first nkeep.
template <typename T, int DIR>
void fft_lines(C2<T>* data, int L, long nlines,
               long n_inner, long inner, long outer, long estride, int nvalid, int nkeep, hipStream_t s);

// Batched FP32 transforms in registers for 2^a and 3 * 2^a lengths (gk_fft.hip)
// and in LDS or through Bluestein's chirp-z convolution for the others
// (gk_fft_any.hip).  None needs device memory beyond its operands and tables.
struct LineArgs {
    unsigned nlines, n_inner;   // line l starts at (l / n_inner) outer + (l % n_inner) inner
    long inner, outer, estride;  // elements at stride estride
    int nvalid, nkeep;           // inputs read (the rest are zeros), outputs stored
    int ncomp;                   // transforms of the same shape, one per blockIdx.y ...
    long cstride;                // ... at this distance
    __device__ __forceinline__ long start(unsigned l) const { return (long)(l / n_inner) * outer + (long)(l % n_inner) * inner; }
};
// Rows of n_real floats (row r at (r / n_inner)*real_outer + (r % n_inner)*real_inner)
// and their P/2+1 complex numbers (same indexing, complex units).  vec: every row
// starts at an even float of an 8-byte aligned array, so pairs load as float2.
struct RowArgs {
    unsigned nrows, n_inner;
    long real_inner, real_outer, cplx_inner, cplx_outer;
    int n_real, vec;
    int ncomp;                // transforms of the same shape, one per blockIdx.y
    long real_comp, cplx_comp;
    __device__ __forceinline__ long real_at(unsigned r) const {
        return (long)(r / n_inner) * real_outer + (long)(r % n_inner) * real_inner;
    }
    __device__ __forceinline__ long cplx_at(unsigned r) const {
        return (long)(r / n_inner) * cplx_outer + (long)(r % n_inner) * cplx_inner;
    }
};
bool fft_reg_length(int L);  // the register transforms take this length
template <int DIR> void fft_lines_reg(float2* data, int L, const LineArgs& a, hipStream_t s);
void fft_rows_r2c_reg(const float* in, float2* out, int P, const RowArgs& a, hipStream_t s);
void fft_rows_c2r_reg(const float2* in, float* out, int P, const RowArgs& a, hipStream_t s);

// Any length: 2^a and 3 * 2^a go to the register kernels (FP64: 2^a to the
// LDS kernel above), lengths with factors 2, 3, 5, 7 to LDS Stockham passes with
// a runtime radix list, others through Bluestein's chirp-z convolution.
template <typename T, int DIR>
void fft_lines_any(C2<T>* data, int L, long nlines, long n_inner, long inner, long outer, long estride, int nvalid,
                   int nkeep, hipStream_t s, int ncomp = 1, long cstride = 0);
// rows: n_real floats -> P/2+1 complex, and the unnormalised inverse
void fft_rows_r2c_any(const float* in, float2* out, int P, long nrows, long n_inner, long in_inner, long in_outer,
                      long out_inner, long out_outer, int n_real, hipStream_t s, int ncomp = 1, long in_comp = 0,
                      long out_comp = 0);
void fft_rows_c2r_any(const float2* in, float* out, int P, long nrows, long n_inner, long in_inner, long in_outer,
                      long out_inner, long out_outer, int n_real, hipStream_t s, int ncomp = 1, long in_comp = 0,
                      long out_comp = 0);
// Build (once, cached) every twiddle / chirp table the FP32 transforms of this
// length and direction read, so that a later call finds them all.
void fft_lines_any_tables(int L, int dir);
void fft_rows_any_tables(int P, int dir);
// length of the padded convolution Bluestein's identity needs for length L, 0 if L does not go through it
int fft_blue_length(int L);

// in-place 3-D complex FFT in FP64 of [n0][n1][n2] (dir -1 forward, +1 inverse)
void fft3_c2c_f64(double2* d, const int n[3], int dir, hipStream_t s);

}  // namespace gk
