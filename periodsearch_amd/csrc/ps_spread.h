// ps_spread.h -- fits and evaluations whose passes are spread over many workgroups, included by
// ps_device.hip after ps_fit2.h.
//
// The J-free kernels give a fit to one workgroup, which walks the passes of every evaluation one after
// the other: right when there are more fits than resident workgroups, but ten fits (one trial period)
// or a hundred (a round of the convexity-weight search) leave most of the chip idle, and so do the last
// fits of a longer list.  Here an LM iteration is two launches:
//   spread_eval  one workgroup per task, a few passes of one fit's trial point: curv and the pole matrices
//                (each task forms its own), then the passes; the Gram blocks of every pass go to memory;
//   spread_step  one workgroup per fit: adds the passes' blocks in their order (mrqcof2's order, so a fit's
//                bits do not depend on the form), accepts or rejects, does the driver's bookkeeping, and
//                solves for the next trial point.
// Launches on one stream order the two; no workgroup waits for another inside a kernel.  The fit's state
// lives in memory between them.  A finished fit's tasks and step return at once.
//
// What bounds it: the latency of one task, of the sum and solve, and two launches per iteration (10 fits of 20
// passes: 50 + 29 us of kernels in 92 us an iteration; 100 fits 185 + 32).  Measured, 6 iterations, one
// workgroup each / spread: Lmax 6, 288 facets, 20 passes: 10 fits 3.27 / 0.63 ms, 100 fits 3.29 / 1.53, 256
// fits 3.31 / 2.92, 300 fits 4.68 / 3.59, 384 fits 4.71 / 4.37, 448 fits 4.72 / 5.53; Lmax 3, 288 facets, 5
// passes: 10 fits 0.71 / 0.39, 100 fits 0.72 / 0.46, 256 fits 0.72 / 0.64, 300 fits 0.92 / 0.94.  Fewer
// passes: spread_pays in ps_device.hip, which chooses.
#pragma once

#include "ps_fit2.h"

namespace psk {

enum : int { kSpreadNew, kSpreadInit, kSpreadTrial, kSpreadDone };

struct SpreadState {
    double a[64];   // the point under evaluation
    double cg[64];  // accepted parameters
    LmState lm;
    int phase;
};

struct SpreadJob {
    const DevProblem *P;
    double freq, conw_r;
    int pole, layout;  // the initial pole; the OrbitModel's Lmax
    int out;           // result index
    int part0, npass;  // the job's passes in the buffer of Gram blocks
    int pad;
};

struct SpreadTask {
    int job;
    int k0, k1;  // passes [k0, k1)
};

// Device buffers: per pass the Gram blocks (kStashPerSlot doubles), per job the accepted and the trial
// normal equations and two area arrays (written by the task of the first and of the last pass).
struct SpreadBuf {
    SpreadState *state;
    double *part, *alpha, *beta, *area;
    size_t a_stride, b_stride, f_stride;
    int *done;  // number of finished jobs
};

template <class Model, bool LS, int NFM>
__device__ __forceinline__ void spread_passes(const DevProblem &P, Shared2<NFM> &sh, const SpreadJob &job, const SpreadTask &t,
                                              double *part, double *area, double *raw_y, double *raw_dyda) {
    const double wqc = conv_weight(job.conw_r);
    const int nb = (P.mfit + 16) >> 4;
    const int k0 = __builtin_amdgcn_readfirstlane(t.k0), k1 = __builtin_amdgcn_readfirstlane(t.k1);
    // the first task's areas serve the step's convexity check, the last one's its own convexity rows
    double *ar = k0 == 0 ? area : k1 == P.npass ? area + P.nf : nullptr;
    Model::template curv<LS>(P, sh.a, sh, ar);
    blmatrix_lds(sh.a[P.nc], sh.a[P.nc + 1], sh);
    __syncthreads();
    for (int k = k0; k < k1; ++k) {
        Prec<false>::V4 acc[kOwn];
        const int ow = eval_pass<Model, LS>(P, sh, wqc, k, nb, ar, raw_y, raw_dyda, acc);
        stash_io(nb, ow, acc, part + size_t(job.part0 + k) * kStashPerSlot, true);
        __syncthreads();
    }
}

// One task.  avec: the parameter vectors of ps_eval's jobs (job j's at j * ma), nullptr: the fits' states.
template <bool LS>
__global__ __launch_bounds__(kWG2, 2) void spread_eval(const SpreadJob *jobs, const SpreadTask *tasks, SpreadBuf B,
                                                       const double *avec, double *raw_y, double *raw_dyda) {
    __shared__ Shared2<kMaxFac> sh;
    const SpreadTask t = tasks[blockIdx.x];
    const int j = __builtin_amdgcn_readfirstlane(t.job);
    if (!avec && __builtin_amdgcn_readfirstlane(B.state[j].phase) == kSpreadDone) return;
    const SpreadJob job = jobs[j];
    const DevProblem &P = *uniform_ptr(job.P);
    if (int(threadIdx.x) < P.ma) sh.a[threadIdx.x] = avec ? avec[size_t(j) * P.ma + threadIdx.x] : B.state[j].a[threadIdx.x];
    if (__builtin_amdgcn_readfirstlane(t.k1) == P.npass) load_facets2(P, sh);  // the convexity rows' normals
    __syncthreads();
    double *ry = raw_y ? raw_y + size_t(j) * P.npts : nullptr, *rd = raw_dyda ? raw_dyda + size_t(j) * P.npts * P.ma : nullptr;
    double *area = B.area + B.f_stride * (2 * size_t(j));
    switch (__builtin_amdgcn_readfirstlane(job.layout)) {
        case 3: spread_passes<OrbitModel<3>, LS>(P, sh, job, t, B.part, area, ry, rd); break;
        case 4: spread_passes<OrbitModel<4>, LS>(P, sh, job, t, B.part, area, ry, rd); break;
        case 5: spread_passes<OrbitModel<5>, LS>(P, sh, job, t, B.part, area, ry, rd); break;
        default: spread_passes<OrbitModel<6>, LS>(P, sh, job, t, B.part, area, ry, rd); break;
    }
}

// All jobs new, none finished.
__global__ void spread_reset(SpreadBuf B, int njobs) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < njobs) B.state[j].phase = kSpreadNew;
    if (j == 0) *B.done = 0;
}

// The Gram blocks of a job's passes, added in their order, into alpha, beta and sh.scal[0] (chi2).
template <int NFM>
__device__ __forceinline__ void spread_sum_passes(const DevProblem &P, Shared2<NFM> &sh, const double *part, int npass,
                                                  double *alpha, double *beta) {
    const int nb = (P.mfit + 16) >> 4, ow = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = own_blocks(nb, ow).n;
    const d4 *p = reinterpret_cast<const d4 *>(part) + size_t(ow) * kOwn * 64 + (threadIdx.x & 63);
    constexpr size_t kStep = kStashPerSlot / 4;
    Prec<false>::V4 acc[kOwn];
#pragma unroll
    for (int b = 0; b < kOwn; ++b) acc[b] = b < n ? p[b * 64] : Prec<false>::zero();
    int k = 1;
    for (; k + 4 <= npass; k += 4) {  // four passes' reads in flight, added in order
        d4 v[4][kOwn];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int b = 0; b < kOwn; ++b)
                if (b < n) v[u][b] = p[(k + u) * kStep + b * 64];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int b = 0; b < kOwn; ++b)
                if (b < n) acc[b] = acc[b] + v[u][b];
    }
    for (; k < npass; ++k)
#pragma unroll
        for (int b = 0; b < kOwn; ++b)
            if (b < n) acc[b] = acc[b] + p[k * kStep + b * 64];
    gram_store(nb, P, sh, ow, acc, alpha, beta);
}

// ps_eval: the outputs of one vector from its passes.
__global__ __launch_bounds__(kWG2, 2) void spread_sum(const SpreadJob *jobs, SpreadBuf B, double *alpha, double *beta,
                                                      double *chisq) {
    __shared__ Shared2<kMaxFac> sh;
    const int j = blockIdx.x;
    const SpreadJob job = jobs[j];
    const DevProblem &P = *uniform_ptr(job.P);
    const int mfit = P.mfit;
    double *al = alpha ? alpha + size_t(j) * mfit * mfit : B.alpha + B.a_stride * (2 * size_t(j));
    double *be = beta ? beta + size_t(j) * mfit : B.beta + B.b_stride * (2 * size_t(j));
    spread_sum_passes(P, sh, B.part + size_t(job.part0) * kStashPerSlot, job.npass, al, be);
    __syncthreads();
    if (threadIdx.x == 0 && chisq) chisq[j] = sh.scal[0];
}

// One job between two evaluations: fit_one's loop (ps_fit2.h) from the evaluated point to the next one.
__global__ __launch_bounds__(kWG2, 2) void spread_step(const SpreadJob *jobs, SpreadBuf B, ps_fit_result *out) {
    __shared__ Shared2<kMaxFac> sh;
    const int tid = threadIdx.x, j = blockIdx.x;
    SpreadState &st = B.state[j];
    const int phase = __builtin_amdgcn_readfirstlane(st.phase);
    if (phase == kSpreadDone) return;
    const SpreadJob job = jobs[j];
    const DevProblem &P = *uniform_ptr(job.P);
    const int ma = P.ma;
    if (phase == kSpreadNew) {
        if (tid < ma) {
            const double v = initial_param(P, tid, job.freq, job.pole);
            st.cg[tid] = v;
            st.a[tid] = v;
        }
        if (tid == 0) {
            LmState lm;
            lm.alamda = P.alamda_start;
            st.lm = lm;
            st.phase = kSpreadInit;
        }
        return;
    }
    double *al[2] = {B.alpha + B.a_stride * (2 * size_t(j)), B.alpha + B.a_stride * (2 * size_t(j) + 1)};
    double *be[2] = {B.beta + B.b_stride * (2 * size_t(j)), B.beta + B.b_stride * (2 * size_t(j) + 1)};
    double *area = B.area + B.f_stride * (2 * size_t(j));
    LmState lm = st.lm;
    lm.settle();
    if (tid < ma) {
        sh.cg[tid] = st.cg[tid];
        sh.atry[tid] = st.a[tid];
    }
    load_facets2(P, sh);
    const bool init = phase == kSpreadInit;
    const int to = __builtin_amdgcn_readfirstlane(lm.cur ^ int(!init));
    spread_sum_passes(P, sh, B.part + size_t(job.part0) * kStashPerSlot, job.npass, to ? al[1] : al[0], to ? be[1] : be[0]);
    __syncthreads();
    const double chi = uniform_double(sh.scal[0]);
    bool fresh = false, eval = true;
    if (init)
        lm.start(chi);
    else if (lm.judge(chi, P)) {
        fresh = true;
        if (tid < ma) sh.cg[tid] = sh.atry[tid];
    }
    __syncthreads();
    // the bookkeeping of the iteration just evaluated, then solves until one succeeds or the fit ends
    bool counted = !init;
    for (;;) {
        lm.settle();
        if (counted) {
            ++lm.niter;
            if (lm.niter == 1 || lm.chisq < lm.ochisq) {
                lm.ochisq = lm.chisq;
                if (!__builtin_amdgcn_readfirstlane(fresh)) {  // curv(cg); else the evaluation's areas are cg's
                    for (int i = tid; i < P.nf; i += kWG2) area[i] = gload(P.darea, i) * exp(facet_shape_sum(P, sh.cg, i));
                    __syncthreads();
                }
                if (__builtin_amdgcn_readfirstlane(tid >> 6) == 0) {
                    double sn[3];
                    facet_sums_n(area, sh.nx, sh.ny, sh.nz, P.nf, sn);
                    if (tid == 0) {
                        sh.scal[1] = sn[0];
                        sh.scal[2] = sn[1];
                        sh.scal[3] = sn[2];
                    }
                }
                __syncthreads();
                const double sn[3] = {uniform_double(sh.scal[1]), uniform_double(sh.scal[2]), uniform_double(sh.scal[3])};
                lm.convexity(sn, job.conw_r);
                __syncthreads();
            }
            lm.settle();
            lm.rms(P);
            fresh = false;
        }
        lm.settle();
        if (!lm.more(P)) {
            eval = false;
            break;
        }
        const int err = lm_solve(P, sh, lm, lm.cur ? al[1] : al[0], lm.cur ? be[1] : be[0]);
        lm.err = __builtin_amdgcn_readfirstlane(err);
        if (lm.err == 0) break;
        ++lm.nfail;
        counted = true;
    }
    __syncthreads();
    if (eval) {
        if (tid < ma) {
            st.cg[tid] = sh.cg[tid];
            st.a[tid] = sh.a[tid];
        }
        if (tid == 0) {
            st.lm = lm;
            st.phase = kSpreadTrial;
        }
    } else if (__builtin_amdgcn_readfirstlane(tid >> 6) == 0) {
        const double totarea = facet_sum(area, nullptr, P.nf);
        if (tid == 0) {
            out[job.out] = lm.result(sh.cg, P.nc, totarea);
            st.phase = kSpreadDone;
            atomicAdd(B.done, 1);
        }
    }
}

}  // namespace psk
