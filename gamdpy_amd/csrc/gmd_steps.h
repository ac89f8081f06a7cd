// gmd_steps.h -- the step kernels as templates over (pair function, cutoff,
// integrator, list kind): included by gmd_core.hip, which declares them
// extern, and by gmd_steps_inst.hip, which instantiates one group of them per
// compilation.
#pragma once
#include "gmd_kernels.h"

// ============================================================================
// Drivers
// ============================================================================
// Every step of a run inside one launch; the blocks of one system meet at a
// software barrier after each step, and the last to arrive runs the tail.
template <int BASE, int CUT, int INTEG, int KIND>
__device__ __forceinline__ void persistent_body(const DP *Pp, const BlockCtx &B) {
    extern __shared__ __align__(16) char lds[];
    PairP *pp = (PairP *)(lds + Pp->lds_pp);
    double *red = (double *)(lds + Pp->lds_red);
    char *build = lds + Pp->lds_build;
    load_pair_table(*Pp, pp);
    __syncthreads();
    const int nsteps = Pp->ctrl->nsteps;
    for (int s = 0; s <= nsteps; ++s) {
        const DP &P = *Pp;
        const bool rebuild = ld_flag(P.rebuild_flag + s) != 0;
        const StepInfo I = step_info(P, s, INTEG, rebuild);
        float acc[GMD_NRED];
#pragma unroll
        for (int c = 0; c < GMD_NRED; ++c) acc[c] = 0.f;
        step_body<BASE, CUT, INTEG, KIND>(P, B, I, pp, build, acc);
        const unsigned mask = red_mask(I.need_ksum, I.need_mom, I.need_save, I.need_wsum);
        if (mask) block_partials(P, B, acc, red, P.partial, mask);
        grid_barrier(P.ctrl, B.nb, [&]() { step_tail(P, I, red, B.nb); });
    }
}

// One step, s_base + k: the rebuild decision is the flag the previous step
// raised, and the previous step's tail runs in every block of the system here
// (folded_tail); the partial sums alternate between two buffers.
//
// BATCH (a replica of a batch; B.bid: the block among those of its rebuild
// steps): a rebuild step is split over rebuild_grid blocks, a list step works
// in the first step_grid of them and the others leave at once.  A rebuild's
// time is the number of cells (or particles) its wavefronts take one after
// another, and in a batch most steps have some replica rebuilding while the
// others wait for it.  The sums of a step are grouped by the wavefronts of
// step_grid blocks, split or not, so that they keep their bits: a split step
// leaves each particle's kinetic energy in P.kcell, and k_batch_ksum adds them
// up in that grouping.  A step that needs other sums (momentum reset, saver
// row, virial) is not split.
template <int BASE, int CUT, int INTEG, int KIND, bool BATCH>
__device__ __forceinline__ void step_once(const DP &P, BlockCtx B, int k) {
    extern __shared__ __align__(16) char lds[];
    const int s = P.ctrl->s_base + k;
    if (s > P.ctrl->nsteps) return;
    bool rebuild = ld_flag(P.rebuild_flag + s) != 0;
    if (BATCH) {
        // (visibly uniform: the grid and the loops over it stay in scalar registers)
        rebuild = __builtin_amdgcn_readfirstlane(rebuild ? 1 : 0) != 0;
        B.nb = P.step_grid;
        if (!rebuild && B.bid >= B.nb) return;
    }
    PairP *pp = (PairP *)(lds + P.lds_pp);
    double *red = (double *)(lds + P.lds_red);
    char *build = lds + P.lds_build;
    StepInfo I = step_info(P, s, INTEG, rebuild, true);
    unsigned mask = red_mask(I.need_ksum, I.need_mom, I.need_save, I.need_wsum);
    if (BATCH && rebuild) {
        // split: a step that needs no sums, or the kinetic sum and has room for its parts
        if (P.rebuild_grid > P.step_grid && (mask == 0u || (mask == (1u << RED_K) && P.kcell != nullptr))) {
            B.nb = P.rebuild_grid;
            I.ksplit = mask != 0u;
            mask = 0u;
        }
        if (B.bid >= B.nb) return;
    }
    // the previous step's sums (only the components its tail needs) and the
    // pair table, then the step itself
    const unsigned qmask = folded_tail_mask<INTEG>(P, I);
    if (INTEG == 2 && !rebuild && !I.scal && qmask == (1u << RED_K) &&
        P.step_grid <= RED_PRE * (int)blockDim.x) {
        // a Nose-Hoover list step whose tail needs only the kinetic sum: the
        // partials go to LDS by DMA now and are summed after the first
        // particle's pair sums (deferred_tail), so their latency and the
        // reduction's barriers overlap the list loop instead of preceding it
        const int q = s - 1;
        const GMEM float *kp = P.partial + (size_t)(q & 1) * GMD_NRED * P.pstride + (size_t)RED_K * P.pstride;
        LDSMEM float *kst = tail_stage(P);
        const int wbase = __builtin_amdgcn_readfirstlane((int)(threadIdx.x & ~63u));
#pragma unroll
        for (int u = 0; u < RED_PRE; ++u) {
            const int b = (int)threadIdx.x + u * (int)blockDim.x;
            if (b < P.step_grid)
                __builtin_amdgcn_global_load_lds((const GMEM void *)(kp + b),
                                                 (LDSMEM void *)(kst + u * (int)blockDim.x + wbase), 4, 0, 0);
        }
        const float xi_q = P.ctrl->xib[q & 1];
        I.apply_shift = false;
        load_pair_table(P, pp);
        __syncthreads();
        float acc[GMD_NRED];
#pragma unroll
        for (int c = 0; c < GMD_NRED; ++c) acc[c] = 0.f;
        // the folded tail's K-only sum, in its order (thread t: blocks t,
        // t + 256, ... in double; the wavefronts in index order): the same
        // thermostat variable bit for bit
        auto hook = [&](StepInfo &J) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            double a = 0.0;
#pragma unroll
            for (int u = 0; u < RED_PRE; ++u) {
                const int b = (int)threadIdx.x + u * (int)blockDim.x;
                a += b < P.step_grid ? (double)kst[u * (int)blockDim.x + (int)threadIdx.x] : 0.0;
            }
            const double x = wave_sum_d(a);
            const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
            if (lane == 0) red[wid * GMD_NRED + RED_K] = x;
            __syncthreads();
            double tot = 0.0;
            for (int w = 0; w < nw; ++w) tot += red[w * GMD_NRED + RED_K];
            __syncthreads();
            J.xi = uniform_f(thermostat_next(P, xi_q, (float)tot, J.t0, q));
            if (B.bid == 0 && threadIdx.x == 0) {
                GMEM Ctrl *C = P.ctrl;
                C->xib[J.s & 1] = J.xi;
                C->xi = J.xi;
                C->ksum = 0.0f;
            }
        };
        if (P.nb16)
            particle_loop_deferred<BASE, CUT, INTEG, 1>(P, B, I, pp, acc, hook);
        else
            particle_loop_deferred<BASE, CUT, INTEG, 2>(P, B, I, pp, acc, hook);
        step_cells_clear(P, B, I);
        if (mask) block_partials(P, B, acc, red, P.partial + (size_t)(s & 1) * GMD_NRED * P.pstride, mask);
        return;
    }
    float pv[RED_PRE][GMD_NRED];
    if ((qmask & ~(1u << RED_K)) == 0u) {
        folded_tail_load<INTEG, 1u << RED_K>(P, I, qmask, pv);
        load_pair_table(P, pp);
        folded_tail<INTEG, 1u << RED_K>(P, B, I, red, qmask, pv);
    } else {
        folded_tail_load<INTEG, RED_ALL>(P, I, qmask, pv);
        load_pair_table(P, pp);
        folded_tail<INTEG, RED_ALL>(P, B, I, red, qmask, pv);
    }
    __syncthreads();
    float acc[GMD_NRED];
#pragma unroll
    for (int c = 0; c < GMD_NRED; ++c) acc[c] = 0.f;
    step_body<BASE, CUT, INTEG, KIND>(P, B, I, pp, build, acc);
    if (mask) block_partials(P, B, acc, red, P.partial + (size_t)(s & 1) * GMD_NRED * P.pstride, mask);
    if (rebuild && B.bid == 0 && threadIdx.x == 0) P.ctrl->nbflag[2] += 1;
}

// The blocks of a launch go to the 8 XCDs in turn (block b to XCD b % 8).
// The logical block index gives each XCD a contiguous eighth of the
// particles of a list step (and of every stride of cells of a rebuild), so
// each XCD's L2 holds one region's positions instead of the whole system's.
__device__ __forceinline__ BlockCtx xcd_block(int b, int nb) {
    if ((nb & 7) == 0) b = (b & 7) * (nb >> 3) + (b >> 3);
    return BlockCtx{b, nb};
}

template <int BASE, int CUT, int INTEG, int KIND>
__global__ void __launch_bounds__(256) k_persistent(const DP *__restrict__ Pp) {
    persistent_body<BASE, CUT, INTEG, KIND>(Pp, xcd_block((int)blockIdx.x, (int)gridDim.x));
}

// One step per launch (step s_base + k).  The cross-block work of a step
// (sums, thermostat, momentum shift, saver row) runs at the start of the
// next step's launch in every block (folded_tail): no one-block tail launch
// between steps, and no last-block-done scheme, which would need an
// agent-scope release per block (a write-back of the XCD's L2 under the
// blocks still running).
template <int BASE, int CUT, int INTEG, int KIND>
__global__ void __launch_bounds__(256, 4) k_step(const DP *__restrict__ Pp, int k) {
    step_once<BASE, CUT, INTEG, KIND, false>(*Pp, xcd_block((int)blockIdx.x, (int)gridDim.x), k);
}

// Batched replicas: block b of the grid works for replica blk[b].rep as its
// block blk[b].bid of blk[b].nb.  Replicas never wait for each other: the
// persistent form synchronises only the blocks of one replica.
struct BatchBlk {
    int rep, bid, nb, pad;
};

template <int BASE, int CUT, int INTEG>
__global__ void __launch_bounds__(256) k_batch_persistent(const DP *__restrict__ Ps, const BatchBlk *blks) {
    const BatchBlk a = blks[blockIdx.x];
    const int rep = __builtin_amdgcn_readfirstlane(a.rep);
    if (rep < 0) return;
    const BlockCtx B = {__builtin_amdgcn_readfirstlane(a.bid), __builtin_amdgcn_readfirstlane(a.nb)};
    persistent_body<BASE, CUT, INTEG, 2>(Ps + rep, B);
}

// One step of every replica, with the previous step's tails folded in as in
// k_step.  The replicas' descriptors lie one after another behind one
// restrict pointer, as k_step's does: read through a table of pointers they
// took vector loads and the kernel 168 VGPRs; now scalar loads and 128, four
// wavefronts per SIMD instead of three (64 KA replicas of 1000 to 8000, with
// the tails no longer a launch of their own: 290 -> 236 us a step).
template <int BASE, int CUT, int INTEG>
__global__ void __launch_bounds__(256, 4) k_batch_step(const DP *__restrict__ Ps, const BatchBlk *blks, int k) {
    const BatchBlk a = blks[blockIdx.x];
    const int rep = __builtin_amdgcn_readfirstlane(a.rep);
    if (rep < 0) return;
    step_once<BASE, CUT, INTEG, 2, true>(Ps[rep], BlockCtx{__builtin_amdgcn_readfirstlane(a.bid), 0}, k);
}


// explicit instantiation (EXT empty) or declaration (EXT extern) of the step
// kernels of one (base, cutoff, integrator)
#define GMD_STEP_KERNELS(EXT, B, C, I)                                                          \
    EXT template __global__ void k_persistent<B, C, I, 0>(const DP *);                           \
    EXT template __global__ void k_persistent<B, C, I, 1>(const DP *);                           \
    EXT template __global__ void k_step<B, C, I, 0>(const DP *, int);                            \
    EXT template __global__ void k_step<B, C, I, 1>(const DP *, int);                            \
    EXT template __global__ void k_batch_persistent<B, C, I>(const DP *, const BatchBlk *); \
    EXT template __global__ void k_batch_step<B, C, I>(const DP *, const BatchBlk *, int);
#define GMD_STEP_KERNELS_CUT(EXT, B, C) \
    GMD_STEP_KERNELS(EXT, B, C, 0)      \
    GMD_STEP_KERNELS(EXT, B, C, 1)      \
    GMD_STEP_KERNELS(EXT, B, C, 2)      \
    GMD_STEP_KERNELS(EXT, B, C, 3)
#define GMD_STEP_KERNELS_BASE(EXT, B) \
    GMD_STEP_KERNELS_CUT(EXT, B, 0)   \
    GMD_STEP_KERNELS_CUT(EXT, B, 1)   \
    GMD_STEP_KERNELS_CUT(EXT, B, 2)
// NPT_Atomic (integrator 4) of one base, in files of their own
#define GMD_STEP_KERNELS_NPT(EXT, B) \
    GMD_STEP_KERNELS(EXT, B, 0, 4)   \
    GMD_STEP_KERNELS(EXT, B, 1, 4)   \
    GMD_STEP_KERNELS(EXT, B, 2, 4)
