// Batched engine: many independent simulations (same Runge-Kutta tableau, any
// sizes and materials) advanced together, one launch per pass and length
// class per RK stage for the whole batch.
//
// Each simulation keeps its own device state exactly as in the single-simulation
// engine (sim.hip): m, k_i, spectra B1/B2, kernel spectrum, EngineState, trial
// log.  A batched kernel covers every simulation whose padded length matches its
// template: a table per launch maps each of its blocks to (simulation, local
// block), after which the kernel runs the same device body
// as the single-simulation kernel (passes.h, rk_dev.h).  So a simulation gets
// bit-identical arithmetic alone and in a batch; only its scheduling differs.
//
// Step control stays per simulation on the device (own dt, error, accept /
// reject, FSAL state, stop time), so a batched trial is a fixed launch
// sequence, captured once into a HIP graph and replayed.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <cmath>
#include <cstring>
#include <functional>
#include <map>
#include <vector>

#include "../../include/mumax_engine.h"
#include "batch_dev.h"
#include "engine.h"
#include "passes.h"
#include "rk_dev.h"
#include "sim.h"

namespace gk {

// ------------------------------------------------------------------ RK pointwise and control
__global__ __launch_bounds__(256) void kb_rk_final(const BSim* sims, const int2* map,
                                                   FinalArgs fa) {
    const BBlock bb = bblock(sims, map);
    const BSim& d = *bb.d;
    if (!d.st->trial_active) return;
    KPtrs kp;
    for (int s = 0; s < 7; s++) kp.k[s] = d.k[s] ? d.k[s] : d.k[0];
    FinalArgs a = fa;
    a.part_err = d.part + 2L * d.npart;
    a.normMap = d.t.normMap;
    rk_final_body(d.m, kp, d.mtmp, d.st, a, (int)d.N, bb.lb, d.nfin);
}

// last: the FSAL tableau's last stage, 0 for the others
__global__ __launch_bounds__(256) void kb_commit(const BSim* sims, const int2* map, int last) {
    const BBlock bb = bblock(sims, map);
    const BSim& d = *bb.d;
    commit_body(d.m, d.mtmp, last ? d.k[0] : nullptr, d.k[last], d.st, d.t.normMap, (int)d.N, bb.lb, d.nfin);
}

// one thread per simulation
__global__ void kb_ctrl_begin(const BSim* sims, int n) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < n) ctrl_begin_body(sims[j].st);
}
// one wave per simulation
__global__ __launch_bounds__(64) void kb_ctrl_after_k0(const BSim* sims, int fsal) {
    const BSim& d = sims[blockIdx.x];
    if (!d.st->trial_active || d.cp.fold_k0) return;
    ctrl_after_k0_body(d.st, fsal && d.st->fsal_init, d.cp);
}
__global__ __launch_bounds__(64) void kb_ctrl_end(const BSim* sims) {
    const BSim& d = sims[blockIdx.x];
    ctrl_end_body(d.st, d.cp);
}
// status flags (0 running, 1 done, 2 stopped on a NaN dt or a non-finite torque or
// error, i.e. failed); with rem, each running simulation's remaining trials at its
// current dt, (stop - time) / dt, or its remaining steps under a step target
__global__ void kb_done(const BSim* sims, int n, int* done, float* rem) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const EngineState* st = sims[j].st;
    done[j] = st->done ? (st->nan_dt || st->nonfinite ? 2 : 1) : 0;
    if (rem) {
        double r = 0.0;
        if (!st->done)
            r = st->stop < INFINITY ? (st->stop - st->time) / fmax((double)st->dt, 1e-30)
                                    : (double)(st->steps_target - st->steps);
        rem[j] = (float)fmin(r, 1e30);
    }
}

// one simulation of a launch: the table entries of its blocks
struct BlockRun {
    int first, sim, n;
};
// The launches' block tables (batch_dev.h, BBlock), one wave per run.  Filled on the
// device: filling them on the host and copying 8 bytes per block, a batch of 400
// simulations of a sweep took 315 us to build, from the runs 155 us (64: 61 and 45 us).
__global__ __launch_bounds__(64) void kb_block_tables(const BlockRun* runs, int2* __restrict__ table) {
    const BlockRun r = runs[blockIdx.x];
    for (int i = threadIdx.x; i < r.n; i += 64) table[r.first + i] = make_int2(r.sim, i);
}

}  // namespace gk

using namespace gk;

// ------------------------------------------------------------------ host
namespace {

// blocks of one pass for one simulation, per padded length class
struct LaunchSet {
    int L = 0;       // template length of the class
    int cnt = 0;     // simulations
    int blocks = 0;  // total blocks
    int2* map = nullptr;          // device, per block: simulation, block within it
    int map_first = 0;            // its first entry in the batch's block tables (set-up)
    std::vector<int> hidx, hst;   // the simulations and their first blocks (set-up)
    int any = 0;                        // 1: small length classes merged, launched by a dispatch kernel
    int nt = 0, lds = 0;                // dispatch launch: threads per block and dynamic LDS bytes
};

// Host image of a batch's device tables, uploaded with one copy on the batch's
// stream: a synchronous hipMemcpy per table would wait for other batches'
// queued work.
struct TableImage {
    std::vector<char> bytes;
    size_t put(const void* src, size_t n) {
        const size_t off = (bytes.size() + 255) & ~(size_t)255;
        bytes.resize(off + n);
        memcpy(bytes.data() + off, src, n);
        return off;
    }
};

int epi_rows_host(int M, bool any);
int z_rows_host(int M);

}  // namespace

struct mmBatch {
    std::vector<mmSim*> sims;
    Tableau tb;
    hipStream_t s = nullptr;
    BSim* dsims = nullptr;
    int* ddone = nullptr;
    float* drem = nullptr;      // remaining trials per simulation (kb_done)
    std::vector<void*> owned;  // device allocations of the tables
    TableImage image;          // set-up only: the tables before upload
    // per pass: one LaunchSet per length class
    std::vector<LaunchSet> zf, y3, xm, y2, yx, zi, fin;
    int useGraph = 1;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    long long trials = 0;
    int* hdone = nullptr;       // pinned host copy of the done flags (mm_batch_enqueue)
    float* hrem = nullptr;      // pinned host copy of drem
    hipEvent_t ev = nullptr;    // end of the last enqueued work
};

namespace {

int z_rows_host(int M) {
    switch (M) {
#define GK_CASE(n) \
    case n: return z_rows_c<n>();
        GK_LEN_M(GK_CASE)
#undef GK_CASE
    }
    abort();
}
int epi_rows_host(int M, bool any) {
    switch (M) {
#define GK_CASE(n) \
    case n: return any ? epi_rows_any<n>() : epi_rows_c<n>();
        GK_LEN_M(GK_CASE)
#undef GK_CASE
    }
    abort();
}
int lanes_host(int L) { return reg_fft_G(L); }  // RegFFT<L>::G
int y2_cols_host(int L) { return std::max(1, 64 / (L / y2_E(L))); }  // Y2<L>::COLS

// per length: threads and dynamic LDS bytes of a block in the dispatch kernels
struct AnyShape {
    int nt, lds;
};
AnyShape any_shape(int pass, int L) {
    switch (pass) {
    case 0:  // Z forward, L = M
        switch (L) {
#define GK_CASE(n) case n: return {z_rows_c<n>() * RegFFT<n>::G, zfwd_lds<n, z_rows_c<n>()>() * 8};
            GK_ANY_M(GK_CASE)
#undef GK_CASE
        }
        break;
    case 1:  // Z inverse + epilogue, L = M
        switch (L) {
#define GK_CASE(n) case n: return {3 * epi_rows_any<n>() * RegFFT<n>::G, zinv_any_bytes<n>()};
            GK_ANY_M(GK_CASE)
#undef GK_CASE
        }
        break;
    case 2: {  // thin plane, L = PY * 64 + PX
        const int PY = L / 64, PX = L % 64;
        switch (PY) {
#define GK_CASE(n)     case n: return {kYxyThreads, PX == 4 ? yxy_lds_elems(4, n) * 8 : yxy_lds_elems(8, n) * 8};
            GK_ANY_Y(GK_CASE)
#undef GK_CASE
        }
        break;
    }
    case 3:  // 2-D, L = PY
        switch (L) {
#define GK_CASE(n) case n: return {Y2<n>::NT, Y2<n>::LDS * 8};
            GK_ANY_Y(GK_CASE)
#undef GK_CASE
        }
        break;
    case 4:  // 3-D Y passes, L = PY
        switch (L) {
#define GK_CASE(n) case n: return {kNT, ypass_lds<n>() * 8};
            GK_ANY_Y(GK_CASE)
#undef GK_CASE
        }
        break;
    case 5:  // 3-D X . K . X, L = PX
        switch (L) {
#define GK_CASE(n) case n: return {kNT, xmul_lds<n>() * 8};
            GK_ANY_X(GK_CASE)
#undef GK_CASE
        }
        break;
    }
    abort();
}
void any_kernel_attributes() {
    static std::once_flag once;
    std::call_once(once, [] {
        any_attr_zfwd();
        any_attr_zinv();
        any_attr_zinv_fin();
        any_attr_y();
    });
}

void* balloc(mmBatch* b, size_t bytes) {
    void* p = cached_malloc(bytes);
    b->owned.push_back(p);
    return p;
}

// group simulations by a length key; blocks(sim) gives each simulation's block count
template <typename Key, typename Blocks>
std::vector<LaunchSet> make_sets(mmBatch* b, const std::vector<int>& members, Key key, Blocks blocks) {
    std::map<int, std::vector<int>> groups;
    for (int j : members) groups[key(b->sims[j])].push_back(j);
    std::vector<LaunchSet> out;
    for (auto& kv : groups) {
        LaunchSet ls;
        ls.L = kv.first;
        ls.cnt = (int)kv.second.size();
        std::vector<int> st(ls.cnt + 1, 0);
        for (int i = 0; i < ls.cnt; i++) st[i + 1] = st[i] + blocks(b->sims[kv.second[i]]);
        ls.blocks = st[ls.cnt];
        ls.hidx = kv.second;
        ls.hst = st;
        if (ls.blocks > 0) out.push_back(ls);
    }
    return out;
}

// Length classes of a pass (0 Z forward, 1 Z inverse, 2 thin plane, 3 2-D, 4 3-D
// Y forward or inverse, 5 3-D X . K . X) with
// fewer blocks than this are merged into one dispatch launch when two or more
// of them are small and have a body in the dispatch kernel.
std::atomic<int> g_merge_blocks{1024};
// any_blocks(j), if given: simulation j's blocks in the dispatch launch (else the same).
std::vector<LaunchSet> merge_small(std::vector<LaunchSet> sets, int pass,
                                   const std::function<int(int)>& any_blocks = nullptr) {
    std::vector<LaunchSet> out, small;
    const int limit = g_merge_blocks.load();
    for (auto& ls : sets) {
        const bool has = pass <= 1   ? any_m(ls.L)
                         : pass == 2 ? any_yx(ls.L / 64, ls.L % 64)
                         : pass == 5 ? any_x(ls.L)
                                     : any_y(ls.L);
        (has && ls.blocks < limit ? small : out).push_back(std::move(ls));
    }
    if (small.size() < 2) {
        for (auto& ls : small) out.push_back(std::move(ls));
        return out;
    }
    LaunchSet m;
    m.any = 1;
    m.L = -1;
    m.hst.push_back(0);
    for (auto& ls : small) {
        const AnyShape a = any_shape(pass, ls.L);
        m.nt = std::max(m.nt, a.nt);
        m.lds = std::max(m.lds, a.lds);
        for (int i = 0; i < ls.cnt; i++) {
            m.hidx.push_back(ls.hidx[i]);
            m.hst.push_back(m.hst.back() + (any_blocks ? any_blocks(ls.hidx[i]) : ls.hst[i + 1] - ls.hst[i]));
        }
        m.cnt += ls.cnt;
    }
    m.blocks = m.hst.back();
    GK_ASSERT(m.lds <= kAnyLds && m.nt <= 1024, "dispatch launch: %d threads, %d bytes of LDS", m.nt, m.lds);
    out.push_back(std::move(m));
    return out;
}

// the runs of the launch sets' block tables, which follow each other from entry `entries` on
void stage_sets(std::vector<LaunchSet>& sets, std::vector<BlockRun>& runs, int& entries) {
    for (auto& ls : sets) {
        ls.map_first = entries;
        for (int i = 0; i < ls.cnt; i++)
            runs.push_back({entries + ls.hst[i], ls.hidx[i], ls.hst[i + 1] - ls.hst[i]});
        entries += ls.blocks;
    }
}

int fin_blocks(const mmSim* s) { return std::max(1, std::min(kRedBlocks, div_up(s->N, 256))); }

// ---------------------------------------------------------------- launchers (one length class each)
BLaunch bl(const mmBatch* b, const LaunchSet& ls) {
    return BLaunch{b->dsims, ls.map, ls.blocks, ls.nt, ls.lds, b->s};
}
void bl_zfwd(mmBatch* b, const LaunchSet& ls, const BStage& sg) {
    if (ls.any) {
        any_zfwd(bl(b, ls), sg);
        GK_LAUNCH_CHECK();
        return;
    }
    const float2* twM = twiddle_f32(ls.L);
    const float2* twP = twiddle_f32(2 * ls.L);
    switch (ls.L) {
#define GK_CASE(n) \
    case n: bz_fwd_run<n>(bl(b, ls), sg, twM, twP); break;
        GK_LEN_M(GK_CASE)
#undef GK_CASE
    default: abort();
    }
    GK_LAUNCH_CHECK();
}
void bl_ypass(mmBatch* b, const LaunchSet& ls, const BStage& sg, bool fwd) {
    if (ls.any) {
        any_ypass(bl(b, ls), sg, fwd);
        GK_LAUNCH_CHECK();
        return;
    }
    const float2* tw = twiddle_f32(ls.L);
    switch (ls.L) {
#define GK_CASE(n)                                                                                       \
    case n:                                                                                              \
        if (fwd) kb_ypass<n, true><<<ls.blocks, kNT, 0, b->s>>>(b->dsims, ls.map, sg, tw);  \
        else kb_ypass<n, false><<<ls.blocks, kNT, 0, b->s>>>(b->dsims, ls.map, sg, tw);     \
        break;
        GK_LEN_Y(GK_CASE)
#undef GK_CASE
    default: abort();
    }
    GK_LAUNCH_CHECK();
}
void bl_xmul(mmBatch* b, const LaunchSet& ls, const BStage& sg) {
    if (ls.any) {
        any_xmul(bl(b, ls), sg);
        GK_LAUNCH_CHECK();
        return;
    }
    const float2* tw = twiddle_f32(ls.L);
    switch (ls.L) {
#define GK_CASE(n)                                                                            \
    case n: kb_xmul<n><<<ls.blocks, kNT, 0, b->s>>>(b->dsims, ls.map, sg, tw); break;
        GK_LEN_X(GK_CASE)
#undef GK_CASE
    default: abort();
    }
    GK_LAUNCH_CHECK();
}
// thin 3-D plane pass; the class key is PY * 64 + PX
void bl_yxy(mmBatch* b, const LaunchSet& ls, const BStage& sg) {
    if (ls.any) {
        any_yxy(bl(b, ls), sg);
        GK_LAUNCH_CHECK();
        return;
    }
    const int PY = ls.L / 64, PX = ls.L % 64;
    const float2* twY = twiddle_f32(PY);
    const float2* twX = twiddle_f32(PX);
    switch (PY) {
#define GK_YX(n, px)                                                                                              \
    case px:                                                                                                      \
        if constexpr (yxy_fits(px, n))                                                                            \
            kb_yxy<n, px><<<ls.blocks, kYxyThreads, 0, b->s>>>(b->dsims, ls.map, sg, twY, twX); \
        else                                                                                                      \
            abort();                                                                                              \
        break;
#define GK_CASE(n)                                                                                                \
    case n:                                                                                                       \
        switch (PX) {                                                                                             \
            GK_YX(n, 4) GK_YX(n, 6) GK_YX(n, 8) GK_YX(n, 12) GK_YX(n, 16)                                         \
        default: abort();                                                                                         \
        }                                                                                                         \
        break;
        GK_LEN_Y(GK_CASE)
#undef GK_CASE
#undef GK_YX
    default: abort();
    }
    GK_LAUNCH_CHECK();
}
void bl_y2d(mmBatch* b, const LaunchSet& ls, const BStage& sg) {
    if (ls.any) {
        any_y2r(bl(b, ls), sg);
        GK_LAUNCH_CHECK();
        return;
    }
    const float2* tw = twiddle_f32(ls.L);
    switch (ls.L) {
#define GK_CASE(n)                                                                                           \
    case n: kb_y2r<n><<<ls.blocks, Y2<n>::NT, 0, b->s>>>(b->dsims, ls.map, sg, tw); \
        break;
        GK_LEN_Y(GK_CASE)
#undef GK_CASE
    default: abort();
    }
    GK_LAUNCH_CHECK();
}
void bl_zinv_epi(mmBatch* b, const LaunchSet& ls, const BStage& sg) {
    if (ls.any) {
        if (sg.fin) any_zinv_fin(bl(b, ls), sg);
        else any_zinv(bl(b, ls), sg);
        GK_LAUNCH_CHECK();
        return;
    }
    const float2* twM = twiddle_f32(ls.L);
    const float2* twP = twiddle_f32(2 * ls.L);
    switch (ls.L) {
#define GK_CASE(n) \
    case n: bz_epi_run<n>(bl(b, ls), sg, twM, twP); break;
        GK_LEN_M(GK_CASE)
#undef GK_CASE
    default: abort();
    }
    GK_LAUNCH_CHECK();
}

// ---------------------------------------------------------------- one batched trial
void enqueue_btrial(mmBatch* b) {
    const Tableau& t = b->tb;
    const int n = (int)b->sims.size();
    kb_ctrl_begin<<<div_up(n, 64), 64, 0, b->s>>>(b->dsims, n);
    GK_LAUNCH_CHECK();
    for (int i = 0; i < t.S; i++) {
        BStage sg{};
        sg.i = i;
        sg.fsal0 = (i == 0 && t.fsal) ? 1 : 0;
        for (int j = 0; j < t.S; j++)
            if (t.a[i][j] != 0.f) {
                sg.kj[sg.nk] = j;
                sg.a[sg.nk] = t.a[i][j];
                sg.nk++;
            }
        const bool fin = !t.adaptive && i == t.S - 1;
        const bool efin = t.fsal_final() && i == t.S - 1;
        for (int j = 0; j < i; j++)
            if (t.a[i][j] != 0.f || (fin && t.b[j] != 0.f) || (efin && t.b2[j] != t.b[j])) {
                sg.uj[sg.nu] = j;
                sg.ua[sg.nu] = t.a[i][j];
                sg.ub[sg.nu] = fin ? t.b[j] : 0.f;
                sg.ce[sg.nu] = efin ? (double)t.b2[j] - (double)t.b[j] : 0.0;
                sg.nu++;
            }
        sg.fin = fin ? 1 : efin ? 2 : 0;
        sg.ce_self = efin ? (double)t.b2[i] - (double)t.b[i] : 0.0;
        sg.use_mi = (!fin && !efin && sg.nu >= 2) ? 1 : 0;
        if (sg.use_mi) sg.nu = 0;
        sg.bs = fin ? t.b[i] : 0.f;
        sg.c = t.c[i];
        sg.cmax = t.cmax(i);
        sg.partslot = i == 0 ? 0 : (t.fsal && i == t.S - 1) ? 1 : -1;
        for (auto& ls : b->zf) bl_zfwd(b, ls, sg);
        for (auto& ls : b->y3) bl_ypass(b, ls, sg, true);
        for (auto& ls : b->xm) bl_xmul(b, ls, sg);
        for (auto& ls : b->y3) bl_ypass(b, ls, sg, false);
        for (auto& ls : b->y2) bl_y2d(b, ls, sg);
        for (auto& ls : b->yx) bl_yxy(b, ls, sg);
        for (auto& ls : b->zi) bl_zinv_epi(b, ls, sg);
        if (i == 0) {
            kb_ctrl_after_k0<<<n, 64, 0, b->s>>>(b->dsims, t.fsal);
            GK_LAUNCH_CHECK();
        }
    }
    if (t.adaptive && !t.fsal_final()) {
        FinalArgs fa{};
        fa.S = t.S;
        for (int i = 0; i < 7; i++) {
            fa.b[i] = t.b[i];
            fa.b2[i] = t.b2[i];
        }
        fa.adaptive = 1;
        for (auto& ls : b->fin) {
            kb_rk_final<<<ls.blocks, 256, 0, b->s>>>(b->dsims, ls.map, fa);
            GK_LAUNCH_CHECK();
        }
    }
    kb_ctrl_end<<<n, 64, 0, b->s>>>(b->dsims);
    GK_LAUNCH_CHECK();
    if (t.adaptive)
        for (auto& ls : b->fin) {
            kb_commit<<<ls.blocks, 256, 0, b->s>>>(b->dsims, ls.map, t.fsal ? t.S - 1 : 0);
            GK_LAUNCH_CHECK();
        }
}

}  // namespace

extern "C" {

mmBatch* mm_batch_new(mmSim* const* sims, int n) {
    GK_ASSERT(n > 0 && sims, "mm_batch_new: empty batch");
    mmBatch* b = new mmBatch();
    b->sims.assign(sims, sims + n);
    b->tb = sims[0]->tb;
    for (int j = 0; j < n; j++) {
        const mmSim* s = sims[j];
        GK_ASSERT(s->mode == MM_MODE_FUSED && s->conv, "mm_batch_new: simulation %d is not a fused-mode engine", j);
        GK_ASSERT(s->p.solver == sims[0]->p.solver, "mm_batch_new: simulations must share the solver");
    }
    b->s = cached_stream();
    // simulation table
    std::vector<BSim> h(n);
    for (int j = 0; j < n; j++) {
        mmSim* s = sims[j];
        BSim& d = h[j];
        d = BSim{};
        d.Nx = s->cp.N[0];
        d.Ny = s->cp.N[1];
        d.Nz = s->cp.N[2];
        d.Q = s->cp.Q;
        d.PY = s->cp.P[1];
        d.PX = s->cp.P[0];
        d.N = s->N;
        d.m = s->m;
        d.mi = s->mi;
        for (int i = 0; i < 7; i++) d.k[i] = s->k[i];
        d.mtmp = s->mtmp;
        d.B1 = s->cp.B1;
        d.B2 = s->cp.B2;
        d.Kc = s->cp.Kc;
        d.st = s->st;
        d.part = s->part;
        d.npart = s->npart;
        d.nfin = fin_blocks(s);
        d.t = torque_args(s, 0.f, nullptr);
        if (s->field.n >= 2) {
            // the batch keeps its own copy of the pointwise field table, so the
            // simulation can replace its table in place (mm_sim_set_field)
            const int nf = s->field.n;
            double* ft = (double*)balloc(b, nf * sizeof(double));
            float* fbv = (float*)balloc(b, 3 * nf * sizeof(float));
            GK_CHECK(hipMemcpyAsync(ft, s->field.t, nf * sizeof(double), hipMemcpyDeviceToDevice, b->s));
            GK_CHECK(hipMemcpyAsync(fbv, s->field.b, 3 * nf * sizeof(float), hipMemcpyDeviceToDevice, b->s));
            d.t.field.t = ft;
            d.t.field.b = fbv;
        }
        d.twM = twiddle_f32(s->cp.M);
        d.twP = twiddle_f32(s->cp.P[2]);
        d.twY = s->cp.P[1] > 1 ? twiddle_f32(s->cp.P[1]) : nullptr;
        d.twX = s->cp.P[0] > 1 ? twiddle_f32(s->cp.P[0]) : nullptr;
        d.dx = FastDiv(s->cp.N[0]);
        d.dq = FastDiv(s->cp.Q);
        d.cp = ctrl_params(s);
        d.cp.part_e = nullptr;  // the batched epilogue computes no energy
    }
    b->ddone = (int*)balloc(b, n * sizeof(int));
    b->drem = (float*)balloc(b, n * sizeof(float));
    // launch sets per pass and length class
    std::vector<int> all(n), d3, d2, dt;
    for (int j = 0; j < n; j++) {
        all[j] = j;
        (sims[j]->cp.P[0] == 1 ? d2 : sims[j]->cp.yxy ? dt : d3).push_back(j);
    }
    auto M = [](const mmSim* s) { return s->cp.M; };
    auto PY = [](const mmSim* s) { return s->cp.P[1]; };
    auto PX = [](const mmSim* s) { return s->cp.P[0]; };
    b->zf = make_sets(b, all, M, [](const mmSim* s) { return div_up(s->cp.N[1], z_rows_host(s->cp.M)) * s->cp.N[0] * 3; });
    auto zinv_blocks = [](const mmSim* s, bool any) { return div_up(s->cp.N[1], epi_rows_host(s->cp.M, any)) * s->cp.N[0]; };
    b->zi = make_sets(b, all, M, [&](const mmSim* s) { return zinv_blocks(s, false); });
    auto ylines = [](const mmSim* s) { return div_up(3L * s->cp.N[0] * s->cp.Q, 256 / lanes_host(s->cp.P[1])); };
    b->y3 = make_sets(b, d3, PY, ylines);
    b->xm = make_sets(b, d3, PX, [](const mmSim* s) {
        const int lpb = 256 / lanes_host(s->cp.P[0]);
        const int lpr = std::min(lpb, s->cp.P[1]);
        return s->cp.Q * div_up(s->cp.P[1], lpr);
    });
    b->y2 = make_sets(b, d2, PY, [](const mmSim* s) { return div_up(s->cp.Q, y2_cols_host(s->cp.P[1])); });
    b->yx = make_sets(b, dt, [](const mmSim* s) { return s->cp.P[1] * 64 + s->cp.P[0]; },
                      [](const mmSim* s) { return s->cp.Q; });
    b->fin = make_sets(b, all, [](const mmSim*) { return 0; }, [](const mmSim* s) { return fin_blocks(s); });
    // small length classes of each pass: one dispatch launch per pass
    any_kernel_attributes();
    b->zf = merge_small(std::move(b->zf), 0);
    b->zi = merge_small(std::move(b->zi), 1, [&](int j) { return zinv_blocks(sims[j], true); });
    b->yx = merge_small(std::move(b->yx), 2);
    b->y2 = merge_small(std::move(b->y2), 3);
    b->y3 = merge_small(std::move(b->y3), 4);
    b->xm = merge_small(std::move(b->xm), 5);
    // per-block maxima as this batch's Z inverse writes them: one per block of its launch
    for (const LaunchSet& ls : b->zi)
        for (int i = 0; i < ls.cnt; i++) {
            BSim& d = h[ls.hidx[i]];
            d.cp.n_k = ls.hst[i + 1] - ls.hst[i];
            d.cp.n_err = b->tb.fsal_final() ? d.cp.n_k : d.nfin;
        }
    const size_t sims_off = b->image.put(h.data(), n * sizeof(BSim));
    std::vector<BlockRun> runs;
    int entries = 0;
    for (auto* sets : {&b->zf, &b->zi, &b->y3, &b->xm, &b->y2, &b->yx, &b->fin})
        stage_sets(*sets, runs, entries);
    const size_t runs_off = b->image.put(runs.data(), runs.size() * sizeof(BlockRun));
    // upload the tables: one block, one copy on the batch's stream from pinned memory
    {
        const size_t nb = b->image.bytes.size();
        char* dev = (char*)balloc(b, nb);
        char* host = (char*)cached_host_malloc(nb);
        memcpy(host, b->image.bytes.data(), nb);
        GK_CHECK(hipMemcpyAsync(dev, host, nb, hipMemcpyHostToDevice, b->s));
        int2* tables = (int2*)balloc(b, (size_t)entries * sizeof(int2));
        kb_block_tables<<<(unsigned)runs.size(), 64, 0, b->s>>>((const BlockRun*)(dev + runs_off), tables);
        GK_LAUNCH_CHECK();
        GK_CHECK(hipStreamSynchronize(b->s));
        cached_host_free(host);
        b->dsims = (BSim*)(dev + sims_off);
        for (auto* sets : {&b->zf, &b->zi, &b->y3, &b->xm, &b->y2, &b->yx, &b->fin})
            for (LaunchSet& ls : *sets) ls.map = tables + ls.map_first;
        b->image = TableImage{};
    }
    // twiddle tables are created on first use: make them now, outside any graph capture
    for (int j = 0; j < n; j++) {
        const ConvPlan& cp = sims[j]->cp;
        (void)twiddle_f32(cp.M);
        (void)twiddle_f32(cp.P[2]);
        if (cp.P[1] > 1) (void)twiddle_f32(cp.P[1]);
        if (cp.P[0] > 1) (void)twiddle_f32(cp.P[0]);
    }
    // tables above were copied synchronously; other batches' streams keep running
    GK_CHECK(hipStreamSynchronize(b->s));
    return b;
}

void mm_batch_free(mmBatch* b) {
    if (!b) return;
    if (b->s) (void)hipStreamSynchronize(b->s);
    cached_host_free(b->hdone);
    cached_host_free(b->hrem);
    if (b->ev) (void)hipEventDestroy(b->ev);
    if (b->exec) (void)hipGraphExecDestroy(b->exec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    for (void* p : b->owned) cached_free(p);
    cached_stream_release(b->s);
    delete b;
}

void mm_batch_set_graph(mmBatch* b, int on) { b->useGraph = on; }

int mm_batch_set_merge_blocks(int blocks) {
    GK_ASSERT(blocks >= 0, "mm_batch_set_merge_blocks: %d", blocks);
    return g_merge_blocks.exchange(blocks);
}

int mm_batch_size(mmBatch* b) { return (int)b->sims.size(); }

// Run(): every simulation j gets the stop time time_j + seconds[j] and is
// normalised first (simrun.go:19-24); Steps() (seconds null): steps[j] steps,
// no normalisation (simrun.go:85-92).
void mm_batch_start(mmBatch* b, const double* seconds, const long long* steps) {
    for (size_t j = 0; j < b->sims.size(); j++) {
        mmSim* s = b->sims[j];
        GK_CHECK(hipStreamSynchronize(s->s));
        EngineState h = read_state(s);
        const double stop = seconds ? h.time + seconds[j] / s->unitTime : INFINITY;
        if (seconds) launch_normalize_active(s->m, nullptr, s->normMap, s->N, b->s);
        launch_set_target(s->st, steps ? steps[j] : -1, stop, nullptr, b->s);
    }
    GK_CHECK(hipStreamSynchronize(b->s));
}

// enqueue n batched trials and wait; returns the number of simulations not done
void mm_batch_enqueue(mmBatch* b, int n) {
    if (b->useGraph) {
        if (!b->exec) {
            GK_CHECK(hipStreamBeginCapture(b->s, hipStreamCaptureModeRelaxed));
            enqueue_btrial(b);
            GK_CHECK(hipStreamEndCapture(b->s, &b->graph));
            GK_CHECK(hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0));
        }
        for (int i = 0; i < n; i++) GK_CHECK(hipGraphLaunch(b->exec, b->s));
    } else {
        for (int i = 0; i < n; i++) enqueue_btrial(b);
    }
    b->trials += n;
    const int ns = (int)b->sims.size();
    kb_done<<<div_up(ns, 64), 64, 0, b->s>>>(b->dsims, ns, b->ddone, b->drem);
    GK_LAUNCH_CHECK();
    if (!b->hdone) {
        b->hdone = (int*)cached_host_malloc(ns * sizeof(int));
        b->hrem = (float*)cached_host_malloc(ns * sizeof(float));
        GK_CHECK(hipEventCreateWithFlags(&b->ev, hipEventDisableTiming));
    }
    GK_CHECK(hipMemcpyAsync(b->hdone, b->ddone, ns * sizeof(int), hipMemcpyDeviceToHost, b->s));
    GK_CHECK(hipMemcpyAsync(b->hrem, b->drem, ns * sizeof(float), hipMemcpyDeviceToHost, b->s));
    GK_CHECK(hipEventRecord(b->ev, b->s));
}

int mm_batch_ready(mmBatch* b) {
    if (!b->ev) return 1;
    const hipError_t e = hipEventQuery(b->ev);
    if (e == hipErrorNotReady) return 0;
    GK_CHECK(e);
    return 1;
}

int mm_batch_flags(mmBatch* b, int* done) {
    GK_ASSERT(b->ev != nullptr, "mm_batch_flags before mm_batch_enqueue");
    GK_CHECK(hipEventSynchronize(b->ev));
    const int ns = (int)b->sims.size();
    int active = 0;
    for (int i = 0; i < ns; i++) {
        if (done) done[i] = b->hdone[i];
        active += !b->hdone[i];
    }
    return active;
}

int mm_batch_remaining(mmBatch* b, float* rem) {
    GK_ASSERT(b->ev != nullptr, "mm_batch_remaining before mm_batch_enqueue");
    GK_CHECK(hipEventSynchronize(b->ev));
    const int ns = (int)b->sims.size();
    for (int i = 0; i < ns; i++) rem[i] = b->hrem[i];
    return ns;
}

int mm_batch_trials(mmBatch* b, int n) {
    mm_batch_enqueue(b, n);
    return mm_batch_flags(b, nullptr);
}

// status of every simulation (0 running, 1 reached its stop time / step target, 2 failed)
void mm_batch_done(mmBatch* b, int* done) {
    const int ns = (int)b->sims.size();
    kb_done<<<div_up(ns, 64), 64, 0, b->s>>>(b->dsims, ns, b->ddone, nullptr);
    GK_LAUNCH_CHECK();
    GK_CHECK(hipMemcpyAsync(done, b->ddone, ns * sizeof(int), hipMemcpyDeviceToHost, b->s));
    GK_CHECK(hipStreamSynchronize(b->s));
}

// run until every simulation is done, polling every `poll` trials; returns batched trials
long long mm_batch_run(mmBatch* b, const double* seconds, int poll) {
    mm_batch_start(b, seconds, nullptr);
    long long n = 0;
    if (poll < 1) poll = 16;
    while (true) {
        const int active = mm_batch_trials(b, poll);
        n += poll;
        if (!active) break;
    }
    return n;
}

}  // extern "C"
