// The drop-in operations without their wait: what a gpu_* entry point enqueues
// on the library stream before it synchronises.  The engine's replay of the
// reference's call sequence (sim.hip) uses them, since nothing on the host reads
// a result before the step's reduction.
#pragma once
#include "../../include/gpukern.h"

namespace gk {

void enq_copy(const float* src, float* dst, int n);
// dst = src + sum_j c[j] k[j], each term one multiply-add in order (the copy and the gpu_madd calls it stands for)
struct CombineTerms {
    const float* k[7];
    float c[7];
    int n;
};
void enq_combine(float* dst, const float* src, const CombineTerms& t, int n);
void enq_linear_combination(float* a, float* b, float wa, float wb, int n);
void enq_normalize(float* m, float* map, int N);  // map null: uniform
void enq_deltaM(float* m, float* h, float alpha_mul, float* alpha_map, float dt_gilb, int N);
void enq_spintorque_deltaM(float* m, float* h, float alpha, float beta, float eps, const float* u, float* jmap,
                           float dt_gilb, int N0, int N1, int N2);
void enq_add_local_fields(float* m, float* h, int N, const float* Hext, float* hmap, int anisType, const float* anisK,
                          const float* anisAxes);
void enq_anal_fw_step(float dt, float alpha, int N, float* m_in, float* m_out, float* h);
void enq_kernelmul6(float* mx, float* my, float* mz, float* kxx, float* kyy, float* kzz, float* kyz, float* kxz,
                    float* kxy, int nReal);
void enq_kernelmul4(float* mx, float* my, float* mz, float* kxx, float* kyy, float* kzz, float* kyz, int nReal);
// ncomp transforms at once, component c at real + c real_stride and cplx + c cplx_stride (floats)
void enq_fft_forward(gpuFFT3dPlan* p, const float* real, long real_stride, float* cplx, long cplx_stride, int ncomp);
void enq_fft_inverse(gpuFFT3dPlan* p, float* cplx, long cplx_stride, float* real, long real_stride, int ncomp);

}  // namespace gk
