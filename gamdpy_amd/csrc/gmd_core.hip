// gmd_core.hip -- kernels, launch drivers and the C ABI of gamdpy_amd.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdlib>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "gamdpy_amd.h"
#include "gmd_kernels.h"

#include "gmd_steps.h"

// the step kernels are instantiated by gmd_steps_inst.hip, a group per compilation
GMD_STEP_KERNELS_BASE(extern, 0)
GMD_STEP_KERNELS_BASE(extern, 1)
GMD_STEP_KERNELS_BASE(extern, 2)
GMD_STEP_KERNELS_BASE(extern, 3)
GMD_STEP_KERNELS_NPT(extern, 0)
GMD_STEP_KERNELS_NPT(extern, 1)
GMD_STEP_KERNELS_NPT(extern, 2)
GMD_STEP_KERNELS_NPT(extern, 3)

// end of a captured group of steps: the next group starts 'n' steps later
__global__ void k_advance(Ctrl *Cp, int n) {
    GMEM Ctrl *C = (GMEM Ctrl *)Cp;
    if (threadIdx.x == 0 && blockIdx.x == 0) C->s_base += n;
}

// the same for every replica of a batch
__global__ void __launch_bounds__(256) k_batch_advance(const DP *__restrict__ Ps, int nrep, int n) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < nrep) Ps[r].ctrl->s_base += n;
}

// The kinetic sums of the replicas whose step was a split rebuild (step_once),
// in the grouping of an unsplit one, bit for bit: block b's wavefront w adds up
// cell after cell (particle after particle) of those it would have taken.  It
// follows every step of a split NVT batch, whether some replica rebuilds or
// not, and takes 7.6 us of a step of 216 (64 replicas, 3.5 %).
__global__ void __launch_bounds__(256) k_batch_ksum(const DP *__restrict__ Ps, int k) {
    const DP &P = Ps[blockIdx.y];
    const int s = P.ctrl->s_base + k;
    if (P.rebuild_grid <= P.step_grid || s >= P.ctrl->nsteps || ld_flag(P.rebuild_flag + s) == 0) return;
    const StepInfo I = step_info(P, s, GMD_NVT, true, true);
    if (red_mask(I.need_ksum, I.need_mom, I.need_save, I.need_wsum) != (1u << RED_K)) return;
    __shared__ double red[4 * GMD_NRED];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, wpb = blockDim.x >> 6;
    const int nb = P.step_grid, stride = nb * wpb;
    for (int b = blockIdx.x; b < nb; b += gridDim.x) {
        float acc[GMD_NRED];
#pragma unroll
        for (int c = 0; c < GMD_NRED; ++c) acc[c] = 0.f;
        constexpr int U = 8;   // loads in flight
        if (P.nblist_kind == 1) {
            for (int c = b * wpb + wid; c < P.ncells; c += U * stride) {
                float v[U];
#pragma unroll
                for (int u = 0; u < U; ++u)
                    v[u] = c + u * stride < P.ncells && lane < P.ccap ? P.kcell[(size_t)(c + u * stride) * P.ccap + lane]
                                                                      : 0.f;
#pragma unroll
                for (int u = 0; u < U; ++u) acc[RED_K] += v[u];
            }
        } else {
            // 64 rounds at a time, added up in lane 0
            for (int i0 = b * wpb + wid; i0 < P.N; i0 += 64 * stride) {
                const float v = i0 + lane * stride < P.N ? P.kcell[i0 + lane * stride] : 0.f;
                for (int u = 0; u < 64; ++u) {
                    const float x = lane_f(v, u);
                    if (lane == 0) acc[RED_K] += x;
                }
            }
        }
        block_partials(P, BlockCtx{b, nb}, acc, red, P.partial + (size_t)(s & 1) * GMD_NRED * P.pstride, 1u << RED_K);
    }
}

// ---- run set-up: cell grid of the starting positions and the skin test ----
// Kernel parameters are generic pointers (an address-space qualifier would
// change the kernel's mangled name between the host and device passes).
//
// What a run starts from, in one launch: the control block, the rebuild flags
// (that of step 0 set where a rebuild is pending), the saver's rows and the
// three cell buffers cleared.  For small systems a launch costs more than its
// work, so the clears share one (before: two memsets, a copy and two
// kernels); block 0 of the x grid writes the control block.
struct RunStart {
    int buf0, need_rebuild;
    long long lstep;
};

__device__ __forceinline__ void run_begin(const DP &P, int nsteps, float t0, const RunStart R) {
    GMEM Ctrl *C = P.ctrl;
    const int t = blockIdx.x * blockDim.x + threadIdx.x, nt = gridDim.x * blockDim.x;
    if (t == 0) {
        // NPT_Atomic: the last run left the state of its final step at
        // npt[nsteps & 1]; this run's step 0 reads npt[0]
        if (C->nsteps & 1)
            for (int k = 0; k < 6; ++k) C->npt[0][k] = C->npt[1][k];
        C->npt_grid_bad = 0;
        C->nsteps = nsteps;
        C->t0 = t0;
        C->buf0 = R.buf0;
        C->lstep0 = R.lstep;
        C->s_base = 0;
        C->red_count = 0;
        C->bar_count = 0;
        C->cell_overflow = 0;
        C->unwrapped = 0;
    }
    for (int k = t; k < nsteps + 2; k += nt) P.rebuild_flag[k] = k == 0 ? R.need_rebuild : 0;
    if (P.save_every > 0)
        for (int k = t; k < P.saves_per_block * 6; k += nt) P.saver_out[k] = 0.f;
    if (P.nblist_kind == 1)
        for (int k = t; k < 3 * P.ncells; k += nt) P.ccount[k] = 0;
}

__global__ void __launch_bounds__(256) k_run_begin(const DP *__restrict__ Pp, int nsteps, float t0, RunStart R) {
    run_begin(*Pp, nsteps, t0, R);
}

// the same for the replicas of a batch (one per y of the grid)
__global__ void __launch_bounds__(256) k_batch_begin(const DP *__restrict__ Ps, int nsteps, float t0, const RunStart *R) {
    run_begin(Ps[blockIdx.y], nsteps, t0, R[blockIdx.y]);
}

// skin test of the starting positions (nblist.py:58-86 at step 0) and, for
// linked lists, insertion into cell buffer 0
__device__ __forceinline__ void run_setup(const DP &P) {
    cpos_t pos = P.ctrl->buf0 ? P.pos1 : P.pos0;
    // the box of step 0 (NPT_Atomic: of its state)
    const float L0 = P.npt ? P.ctrl->npt[0][3] : P.box0, L1 = P.npt ? P.ctrl->npt[0][4] : P.box1,
                L2 = P.npt ? P.ctrl->npt[0][5] : P.box2;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < P.N; i += gridDim.x * blockDim.x) {
        const float4 r = pos[i], rr = P.rref[i];
        float dx, dy, dz;
        if (dist_sq_mic(r.x, r.y, r.z, rr.x, rr.y, rr.z, L0, L1, L2, dx, dy, dz) > P.skin2q)
            P.rebuild_flag[0] = 1;
        // a position outside the box (as a caller may upload it): the run
        // takes the minimum image of every pair (an integration step wraps
        // each particle into [-L/2, L/2], where it then stays)
        if (fabsf(r.x) * 2.0f > L0 || fabsf(r.y) * 2.0f > L1 || fabsf(r.z) * 2.0f > L2)
            P.ctrl->unwrapped = 1;
        if (P.nblist_kind == 1) cell_insert(P, 0, i, r.x, r.y, r.z, L0, L1, L2, 1.0f / L0, 1.0f / L1, 1.0f / L2);
    }
}

__global__ void __launch_bounds__(256) k_run_setup(const DP *__restrict__ Pp) { run_setup(*Pp); }

__global__ void __launch_bounds__(256) k_batch_setup(const DP *__restrict__ Ps) { run_setup(Ps[blockIdx.y]); }

// the prepared pair table of the context (once)
__global__ void k_pair_table(const DP *__restrict__ Pp) {
    const DP &P = *Pp;
    const int nt2 = P.ntypes * P.ntypes;
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < nt2; t += gridDim.x * blockDim.x) {
        PairP q;
        prepare_pair(P, t, q);
        P.ptab[t] = q;
    }
}

// ---- what the host reads after a run, into pinned memory: the control block
// and the saver's rows (a kernel's stores instead of a copy per read) ----
__device__ __forceinline__ void run_publish(const DP &P) {
    const GMEM int *c = (const GMEM int *)P.ctrl;
    const int nc = (int)(sizeof(Ctrl) / 4);
    for (int k = threadIdx.x; k < nc; k += blockDim.x) P.pub[k] = c[k];
    if (P.save_every > 0)
        for (int k = threadIdx.x; k < P.saves_per_block * 6; k += blockDim.x)
            P.pub[nc + k] = __float_as_int(P.saver_out[k]);
}

__global__ void __launch_bounds__(256) k_run_publish(const DP *__restrict__ Pp) { run_publish(*Pp); }

__global__ void __launch_bounds__(256) k_batch_publish(const DP *__restrict__ Ps) { run_publish(Ps[blockIdx.x]); }

// ---- the host's arrays to and from the device layout ----
// One kernel gathers every array into the packed buffer (unpack) or takes it
// apart (pack), in the caller's numbering, and one copy moves the buffer: a
// copy and a host loop per array cost about 15 us each of round trips and,
// at N = 50021, 0.6 ms of host time.  Up to XFER_DIRECT particles the kernels
// read and write the pinned buffer themselves (one launch less; N = 500: an
// upload, evaluation and download take 74 us, 203 us with the copies per
// array); above, where the 12-byte rows would make poor use of the bus, a
// linear copy kernel moves it, or from XFER_DMA words (1 MB, where its launch
// no longer matters) the copy engine: 66 us for the 3.4 MB of N = 50021.  The
// kernels themselves take 6 us there and are bound by latency.
#define XFER_DIRECT 1024
#define XFER_DMA (1 << 18)
#define XFER_CHUNK (640 << 10)   // words of a half of the pinned buffer of a large system

__device__ __forceinline__ void unpack_state(const DP &P, int cur, unsigned what, int *dst_p, int i) {
    GMEM int *dst = (GMEM int *)dst_p;
    const XferSeg X((size_t)P.N, (size_t)P.nscal);
    const size_t N = P.N, o = P.perm[i];
    auto put3 = [&](size_t at, float x, float y, float z) {
        dst[at + 3 * o] = __float_as_int(x);
        dst[at + 3 * o + 1] = __float_as_int(y);
        dst[at + 3 * o + 2] = __float_as_int(z);
    };
    if (what & (XF_R | XF_T)) {
        const float4 r = cur ? P.pos1[i] : P.pos0[i];
        if (what & XF_R) put3(X.r, r.x, r.y, r.z);
        if (what & XF_T) dst[X.t + o] = __float_as_int(r.w);
    }
    if (what & (XF_V | XF_S)) {
        const float4 v = P.vel[i];
        if (what & XF_V) put3(X.v, v.x, v.y, v.z);
        if (what & XF_S) {
            GMEM int *row = dst + X.s + o * P.nscal;
            if (P.sid_u >= 0) row[P.sid_u] = __float_as_int(P.sc[SC_U * N + i]);
            if (P.sid_w >= 0) row[P.sid_w] = __float_as_int(P.sc[SC_W * N + i]);
            if (P.sid_lap >= 0) row[P.sid_lap] = __float_as_int(P.sc[SC_LAP * N + i]);
            if (P.sid_k >= 0) row[P.sid_k] = __float_as_int(P.sc[SC_K * N + i]);
            if (P.sid_fsq >= 0) row[P.sid_fsq] = __float_as_int(P.sc[SC_FSQ * N + i]);
            if (P.sid_m >= 0) row[P.sid_m] = __float_as_int(v.w);
        }
    }
    if (what & XF_F) {
        const float4 f = P.frc[i];
        put3(X.f, f.x, f.y, f.z);
    }
    if (what & XF_IM)
        for (int k = 0; k < 3; ++k) dst[X.im + 3 * o + k] = P.rim[(size_t)k * N + i];
}

__global__ void __launch_bounds__(256) k_unpack(const DP *__restrict__ Pp, int cur, unsigned what, int *dst) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < Pp->N; i += gridDim.x * blockDim.x)
        unpack_state(*Pp, cur, what, dst, i);
}

// every replica of a batch into its own packed buffer in device memory
__global__ void __launch_bounds__(256) k_batch_unpack(const DP *__restrict__ Ps, const RunStart *R) {
    const DP &P = Ps[blockIdx.y];
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < P.N; i += gridDim.x * blockDim.x)
        unpack_state(P, R[blockIdx.y].buf0, XF_ALL, (int *)P.xdev, i);
}

__device__ __forceinline__ void copy_words(const int *src_p, int *dst_p, size_t n) {
    const GMEM int4 *src = (const GMEM int4 *)src_p;
    GMEM int4 *dst = (GMEM int4 *)dst_p;
    const size_t t = blockIdx.x * (size_t)blockDim.x + threadIdx.x, nt = (size_t)gridDim.x * blockDim.x;
    for (size_t k = t; k < n / 4; k += nt) dst[k] = src[k];
    for (size_t k = n / 4 * 4 + t; k < n; k += nt) ((GMEM int *)dst_p)[k] = ((const GMEM int *)src_p)[k];
}

// n words between two 16-byte aligned buffers
__global__ void __launch_bounds__(256) k_copy_words(const int *src, int *dst, size_t n) { copy_words(src, dst, n); }

__global__ void __launch_bounds__(256) k_batch_fetch(const DP *__restrict__ Ps) {
    const DP &P = Ps[blockIdx.y];
    copy_words((const int *)P.xdev, P.xhost, XferSeg((size_t)P.N, (size_t)P.nscal).end);
}

// the packed arrays named by what, in the identity numbering, into the device
// layout; positions go to pos0.  Positions and types share pos, velocities
// and masses share vel: a field that is not given keeps its value
__global__ void __launch_bounds__(256) k_pack(const DP *__restrict__ Pp, int cur, unsigned what, const int *src_p) {
    const DP &P = *Pp;
    const GMEM int *src = (const GMEM int *)src_p;
    const GMEM float *fs = (const GMEM float *)src_p;
    const size_t N = P.N;
    const XferSeg X(N, (size_t)P.nscal);
    const bool new_m = (what & XF_S) && P.sid_m >= 0;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < N; i += (size_t)gridDim.x * blockDim.x) {
        const GMEM float *row = fs + X.s + i * P.nscal;
        if (what & (XF_R | XF_T)) {
            float4 r = make_float4(0.f, 0.f, 0.f, 0.f);
            if (!(what & XF_R) || !(what & XF_T)) r = cur ? P.pos1[i] : P.pos0[i];
            if (what & XF_R) {
                r.x = fs[X.r + 3 * i];
                r.y = fs[X.r + 3 * i + 1];
                r.z = fs[X.r + 3 * i + 2];
            }
            if (what & XF_T) r.w = __int_as_float(src[X.t + i]);
            P.pos0[i] = r;
        }
        if ((what & XF_V) || new_m) {
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (!(what & XF_V) || !new_m) v = P.vel[i];
            if (what & XF_V) {
                v.x = fs[X.v + 3 * i];
                v.y = fs[X.v + 3 * i + 1];
                v.z = fs[X.v + 3 * i + 2];
            }
            if (new_m) v.w = row[P.sid_m];
            P.vel[i] = v;
        }
        if (what & XF_F) P.frc[i] = make_float4(fs[X.f + 3 * i], fs[X.f + 3 * i + 1], fs[X.f + 3 * i + 2], 0.f);
        if (what & XF_S) {
            P.sc[SC_U * N + i] = P.sid_u >= 0 ? row[P.sid_u] : 0.f;
            P.sc[SC_W * N + i] = P.sid_w >= 0 ? row[P.sid_w] : 0.f;
            P.sc[SC_LAP * N + i] = P.sid_lap >= 0 ? row[P.sid_lap] : 0.f;
            P.sc[SC_K * N + i] = P.sid_k >= 0 ? row[P.sid_k] : 0.f;
            P.sc[SC_FSQ * N + i] = P.sid_fsq >= 0 ? row[P.sid_fsq] : 0.f;
        }
        if (what & XF_IM)
            for (int k = 0; k < 3; ++k) P.rim[(size_t)k * N + i] = src[X.im + 3 * i + k];
    }
}

// ============================================================================
// Radial distribution (calculator_radial_distribution.py:76-109)
// ============================================================================
#define RDF_CHUNK 64     // particles per chunk: the i of a wavefront, one a lane
#define RDF_GROUP 16     // particles per group: the j a chunk is tested and counted against at a time
#define RDF_PAD 1e30f    // coordinate of the places past the last particle (-: in the role of i)
#define RDF_LDS_SPARE (4096 + 64)   // of 64 KB a block: beyond the histogram and thresholds
#define RDF_MAX_CELL 32  // sorting cells per dimension

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
// constant for the kernel, so that an address the same in every lane becomes
// a scalar load
typedef const __attribute__((address_space(4))) f32x16 *rdf_quad_t;

struct RdfP {
    int N, nt, bins, nchunks;
    int unit, nrow, nper;      // groups a wavefront tests at a time; row pairs; units a row pair
    float L0, L1, L2, rL0, rL1, rL2;   // box and 1 / box
    float inv_bw, edge;        // bin estimate and the fraction from which it is settled by the threshold
    // per group g: [4g] centre and [4g+1] half extents of its box in the
    // minimum-image frame of its first particle, [4g+2] / [4g+3] lower and
    // upper corners of its raw coordinates; per chunk the same in cbox
    const GMEM float4 *gbox, *cbox;
    float skip2;               // chunk-group pairs whose distance lower bound exceeds this are skipped
    cpos_t pos;                // sorted and padded to whole chunks; w: byte offset of the type's histogram
    const GMEM float *thr;     // thr[k] k = 0..bins: smallest d^2 of bin >= k (thr[bins]: first excluded)
    GMEM unsigned *part;       // [gridDim][nt][nt][bins]
};

// ---- sorting -----------------------------------------------------------------
// The histogram does not depend on the numbering, its cost does: particles
// sorted along a Hilbert curve through coarse cells (Skilling's transform, AIP
// Conf. Proc. 707, 381 (2004)) make chunks and groups compact,
// so that more of their pairs are skipped whole and few need the per-pair
// minimum image.  k_rdf_count gives each particle its cell and its place among
// the cell's particles (in any order), k_rdf_starts the cells' first places,
// k_rdf_place writes the sorted positions.
struct RdfSort {
    int N, ncell, npad, nt_bytes;   // npad: N up to whole chunks; nt_bytes: histogram bytes a type
    float rL0, rL1, rL2;
    const float4 *pos;              // x, y, z, type bits; or null:
    const float *r;                 // (N, 3) as the host gave them, with
    const int *ptype;               // their types (also instead of pos.w if given)
    int *count;                     // [ncell^3], zero on entry
    int2 *key;                      // [N] cell and place
    float4 *out;                    // [npad]
};

__device__ __forceinline__ float4 rdf_read(const RdfSort &S, int i) {
    if (!S.pos) {
        const GMEM float *r = (const GMEM float *)S.r;
        return make_float4(r[3 * i], r[3 * i + 1], r[3 * i + 2], __int_as_float(((const GMEM int *)S.ptype)[i]));
    }
    float4 p = ((cpos_t)S.pos)[i];
    if (S.ptype) p.w = __int_as_float(((const GMEM int *)S.ptype)[i]);
    return p;
}

// bits of v (up to five) three apart
__device__ __forceinline__ int rdf_spread(int v) {
    v = (v | (v << 8)) & 0x100f;
    v = (v | (v << 4)) & 0x10c3;
    return (v | (v << 2)) & 0x1249;
}

__global__ void __launch_bounds__(256) k_rdf_count(RdfSort S) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= S.N) return;
    const float4 p = rdf_read(S, i);
    // any position gets some cell: not a number and infinities the first
    auto cell = [&](float x, float rL) {
        float u = x * rL;
        u = (u - floorf(u)) * (float)S.ncell;
        return u > 0.f ? min((int)fminf(u, 1e6f), S.ncell - 1) : 0;
    };
    int c[3] = {cell(p.x, S.rL0), cell(p.y, S.rL1), cell(p.z, S.rL2)};
    // transpose of the Hilbert index, from the most significant bit down:
    // each bit of a coordinate reflects or exchanges the lower bits of the first
    for (int b = S.ncell >> 1; b > 1; b >>= 1) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const int t = c[d] & b ? b - 1 : (c[0] ^ c[d]) & (b - 1);
            if (!(c[d] & b)) c[d] ^= t;
            c[0] ^= t;
        }
    }
    c[1] ^= c[0];
    c[2] ^= c[1];
    int t = 0;
    for (int b = S.ncell >> 1; b > 1; b >>= 1)
        if (c[2] & b) t ^= b - 1;
    const int k = rdf_spread(c[0] ^ t) << 2 | rdf_spread(c[1] ^ t) << 1 | rdf_spread(c[2] ^ t);
    ((GMEM int2 *)S.key)[i] = make_int2(k, atomicAdd(S.count + k, 1));
}

// exclusive prefix sum of n counts in place, one block of 1024
__global__ void __launch_bounds__(1024) k_rdf_starts(int *count_p, int n) {
    GMEM int *count = (GMEM int *)count_p;
    __shared__ int wsum[16];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int per = (n + 1023) / 1024, k0 = threadIdx.x * per;
    int s = 0;
    for (int k = k0; k < min(n, k0 + per); ++k) s += count[k];
    int inc = s;
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(inc, o, 64);
        if (lane >= o) inc += y;
    }
    if (lane == 63) wsum[wid] = inc;
    __syncthreads();
    int base = inc - s;
    for (int x = 0; x < wid; ++x) base += wsum[x];
    for (int k = k0; k < min(n, k0 + per); ++k) {
        const int c = count[k];
        count[k] = base;
        base += c;
    }
}

// the position and histogram offset of particle i, or what fills a last chunk
__device__ __forceinline__ float4 rdf_entry(const RdfSort &S, int i) {
    float4 p = make_float4(RDF_PAD, RDF_PAD, RDF_PAD, 0.f);
    if (i < S.N) {
        p = rdf_read(S, i);
        p.w = __int_as_float(__float_as_int(p.w) * S.nt_bytes);
    }
    return p;
}

__global__ void __launch_bounds__(256) k_rdf_place(RdfSort S) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= S.npad) return;
    const float4 p = rdf_entry(S, i);
    int to = i;
    if (i < S.N) {
        const int2 k = ((const GMEM int2 *)S.key)[i];
        to = ((const GMEM int *)S.count)[k.x] + k.y;
    }
    ((GMEM float4 *)S.out)[to] = p;
}

// Boxes of each group and chunk (a wavefront a chunk): centre and half
// extents in the minimum-image frame of its first particle (tight for one
// that straddles the periodic boundary), with a rounding margin, and the raw
// coordinate bounds.  A group without particles gets a negative extent.
// place: not sorted, so the positions are laid out here.
__global__ void __launch_bounds__(256) k_rdf_boxes(RdfSort S, int place, float L0, float L1, float L2,
                                                   float4 *gbox_p, float4 *cbox_p) {
    const int c = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, N = S.N;
    const int i0 = c * RDF_CHUNK, i = i0 + lane;
    if (i >= S.npad) return;
    GMEM float4 *pos = (GMEM float4 *)S.out;
    const float4 own = place ? rdf_entry(S, i) : pos[i];
    if (place) pos[i] = own;
    for (int level = 0; level < 2; ++level) {
        const int w = level ? RDF_CHUNK : RDF_GROUP;
        const int b0 = i0 + (lane & ~(w - 1)), l0 = min(b0, N - 1) - i0;   // (a chunk has a particle)
        const float4 r0 = make_float4(__shfl(own.x, l0, 64), __shfl(own.y, l0, 64), __shfl(own.z, l0, 64), 0.f);
        const float4 r = i < N ? own : r0;
        float lo[3] = {mic1(r.x - r0.x, L0), mic1(r.y - r0.y, L1), mic1(r.z - r0.z, L2)};
        float hi[3] = {lo[0], lo[1], lo[2]};
        float rlo[3] = {r.x, r.y, r.z};
        float rhi[3] = {r.x, r.y, r.z};
        for (int k = 0; k < 3; ++k) {
            for (int o = w / 2; o > 0; o >>= 1) {
                lo[k] = fminf(lo[k], __shfl_xor(lo[k], o, 64));
                hi[k] = fmaxf(hi[k], __shfl_xor(hi[k], o, 64));
                rlo[k] = fminf(rlo[k], __shfl_xor(rlo[k], o, 64));
                rhi[k] = fmaxf(rhi[k], __shfl_xor(rhi[k], o, 64));
            }
        }
        if ((lane & (w - 1)) == 0) {
            float cc[3], h[3];
            for (int k = 0; k < 3; ++k) {
                h[k] = 0.5f * (hi[k] - lo[k]) * 1.0001f + 1e-4f;   // rounding margin
                cc[k] = 0.5f * (lo[k] + hi[k]);
            }
            GMEM float4 *box = level ? (GMEM float4 *)cbox_p + 4 * c : (GMEM float4 *)gbox_p + 4 * (b0 / RDF_GROUP);
            box[0] = make_float4(r0.x + cc[0], r0.y + cc[1], r0.z + cc[2], 0.f);
            box[1] = b0 < N ? make_float4(h[0], h[1], h[2], 0.f) : make_float4(-1.f, -1.f, -1.f, 0.f);
            box[2] = make_float4(rlo[0], rlo[1], rlo[2], 0.f);
            box[3] = make_float4(rhi[0], rhi[1], rhi[2], 0.f);
        }
    }
}

// ---- counting ----------------------------------------------------------------
// Image of every pair of a chunk and a group in one dimension.  fl(xj - xi)
// lies in [fl(jlo - ihi), fl(jhi - ilo)] because rounding is monotone, so the
// minimum-image rule |d| > L/2 -> d - copysign(L, d) takes one branch for
// all of them, or they are mixed: 0 = no wrap, 1 = d - L, 2 = d + L,
// 3 = mixed.
__device__ __forceinline__ int rdf_dim_code(float ilo, float ihi, float jlo, float jhi, float L) {
#pragma clang fp contract(off)
    const float a = jlo - ihi, b = jhi - ilo, h = 0.5f * L;
    if (a >= -h && b <= h) return 0;
    if (a > h) return 1;
    if (b < -h) return 2;
    return 3;
}

// lower bound of the minimum-image distance between two boxes in a dimension
__device__ __forceinline__ float rdf_gap(float ci, float hi, float cj, float hj, float L, float rL) {
    const float d = ci - cj;
    return fmaxf(0.f, fabsf(d - L * __builtin_rintf(d * rL)) - (hi + hj) - 4e-7f * L);
}

// Pairs of lane i with the RDF_GROUP particles of one group, read as scalars.
// CX, CY, CZ: 0 no image, 1 the one the shift s = L or -L gives for the whole
// group, fl(fl(xj - xi) - s), which is what mic1 returns, bit for bit, 2 the
// per-pair minimum image.  after: only the j past this one (of the lane's own
// chunk; -1: all).  The bin: the estimate b = sqrt(d2) * inv_bw with inv_bw
// scaled down by more than the rounding of v_sqrt_f32, of the product and of
// the exact rule can raise it, so floor(b) is the exact bin or one below it,
// and one below only if the fraction of b is past R.edge; those few are settled
// by the exact threshold thr[k + 1].  Excluded pairs (d2 >= thr[bins], i.e.
// d >= L/2) are masked off: an atomic of theirs would land on one word per
// type pair.
template <int CX, int CY, int CZ>
__device__ __forceinline__ void rdf_group(const RdfP &R, rdf_quad_t pj, int after, float xi, float yi, float zi,
                                          float sx, float sy, float sz, float out_thr, const float *thr,
                                          char *hist_i) {
#pragma clang fp contract(off)
    f32x16 q = pj[0];
#pragma unroll
    for (int u0 = 0; u0 < RDF_GROUP; u0 += 4) {
        f32x16 nxt = q;
        if (u0 + 4 < RDF_GROUP) nxt = pj[u0 / 4 + 1];
        float d2[4], b[4], f = 0.f;
        bool ok[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            float dx = q[4 * u] - xi, dy = q[4 * u + 1] - yi, dz = q[4 * u + 2] - zi;
            if (CX == 1) dx = dx - sx;
            if (CX == 2) dx = mic1(dx, R.L0);
            if (CY == 1) dy = dy - sy;
            if (CY == 2) dy = mic1(dy, R.L1);
            if (CZ == 1) dz = dz - sz;
            if (CZ == 2) dz = mic1(dz, R.L2);
            d2[u] = dx * dx;
            d2[u] = d2[u] + dy * dy;
            d2[u] = d2[u] + dz * dz;
            ok[u] = d2[u] < out_thr;
            if (CX + CY + CZ == 6) ok[u] &= u0 + u > after;
        }
        // four excluded in every lane skip the binning
        if (ok[0] | ok[1] | ok[2] | ok[3]) {
            int k[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                b[u] = __builtin_amdgcn_sqrtf(d2[u]) * R.inv_bw;
                k[u] = (int)b[u];
                f = fmaxf(f, __builtin_amdgcn_fractf(b[u]));
            }
            if (f >= R.edge) {
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (ok[u] && d2[u] >= thr[k[u] + 1]) ++k[u];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (ok[u]) atomicAdd((unsigned *)(hist_i + __float_as_int(q[4 * u + 3]) + 4 * k[u]), 1u);
        }
        q = nxt;
    }
}

// Unordered pairs i < j are visited once and counted in the slot of the
// ordered type pair (type of the row particle i, type of j); the host adds
// the (a, b) and (b, a) slots.  Chunk I meets the groups of the chunks J >= I;
// rows I and nchunks-1-I together hold nchunks + 1 chunks, so the work is cut
// into units of R.unit <= 64 groups of such a row pair, taken by turns by the
// wavefronts of the grid.  Each lane tests one group of the unit (skipped when
// no pair can be closer than L/2) and finds its image codes; the groups left
// are counted one after the other, their positions in scalar registers.
// Bound by the issue of VALU instructions, about 19 a visited pair and lane,
// one of them a square root at a quarter of the rate (five cycles an
// instruction and SIMD measured; LDS is busy a quarter of the time).  N = 65536,
// 1000 bins, 2 types, in random order: 1.16 ms, against 1.76 for blocks that
// staged tiles of 256 j in LDS, read the threshold of every pair and took the
// particles in the caller's order (sorting adds 0.02; along a Morton curve
// instead 1.22, counting excluded pairs in a spare word instead of masking
// them off 1.18).
__global__ void __launch_bounds__(256) k_rdf(RdfP R) {
    extern __shared__ __align__(16) char lds[];
    const int nh = R.nt * R.nt * R.bins;
    unsigned *hist = (unsigned *)lds;
    float *thr = (float *)(lds + (((size_t)nh * 4 + 15) & ~(size_t)15));
    for (int x = threadIdx.x; x < nh; x += blockDim.x) hist[x] = 0u;
    for (int x = threadIdx.x; x <= R.bins; x += blockDim.x) thr[x] = R.thr[x];
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)));
    const int waves = (int)(gridDim.x * (blockDim.x >> 6));
    const float out_thr = R.thr[R.bins];
    const int n = R.nchunks;
    // unit u of row pair q, advanced by 'waves' units without a division a turn
    int q = wave / R.nper, u = wave - q * R.nper;
    const int dq = waves / R.nper, du = waves - dq * R.nper;
    float xi = 0.f, yi = 0.f, zi = 0.f;
    char *hist_i = nullptr;
    int Icur = -1;
    while (q < R.nrow) {
        // group x of the row pair: chunk J and row I
        const int first = (n - q) * (RDF_CHUNK / RDF_GROUP);
        const int rows = (2 * q == n - 1) ? first : (n + 1) * (RDF_CHUNK / RDF_GROUP);
        const int x = u * R.unit + lane;
        int code = -1, I = 0, g = 0;
        if (lane < R.unit && x < rows) {
            I = x < first ? q : n - 1 - q;
            g = x < first ? q * (RDF_CHUNK / RDF_GROUP) + x : I * (RDF_CHUNK / RDF_GROUP) + x - first;
            const float4 bi = R.cbox[4 * I], hi = R.cbox[4 * I + 1], bj = R.gbox[4 * (size_t)g],
                         hj = R.gbox[4 * (size_t)g + 1];
            const float4 li = R.cbox[4 * I + 2], ui = R.cbox[4 * I + 3], lj = R.gbox[4 * (size_t)g + 2],
                         uj = R.gbox[4 * (size_t)g + 3];
            const float gx = rdf_gap(bi.x, hi.x, bj.x, hj.x, R.L0, R.rL0);
            const float gy = rdf_gap(bi.y, hi.y, bj.y, hj.y, R.L1, R.rL1);
            const float gz = rdf_gap(bi.z, hi.z, bj.z, hj.z, R.L2, R.rL2);
            // (a box around a position that is not finite is not a number: never skipped)
            if (!(hj.x < 0.f) && !(gx * gx + gy * gy + gz * gz > R.skip2))
                code = rdf_dim_code(li.x, ui.x, lj.x, uj.x, R.L0) | (rdf_dim_code(li.y, ui.y, lj.y, uj.y, R.L1) << 2) |
                       (rdf_dim_code(li.z, ui.z, lj.z, uj.z, R.L2) << 4);
            if (code >= 0 && g / (RDF_CHUNK / RDF_GROUP) == I) code = 0x3f;   // its own chunk: the form with 'after'
        }
        unsigned long long live = __ballot(code >= 0);
        while (live) {
            const int l = __builtin_ctzll(live);
            live &= live - 1;
            const int cd = __builtin_amdgcn_readlane(code, l), gj = __builtin_amdgcn_readlane(g, l),
                      Ij = __builtin_amdgcn_readlane(I, l);
            if (Ij != Icur) {
                Icur = Ij;
                float4 ri = R.pos[(size_t)Ij * RDF_CHUNK + lane];
                if (Ij * RDF_CHUNK + lane >= R.N) ri.x = -RDF_PAD;
                xi = ri.x;
                yi = ri.y;
                zi = ri.z;
                hist_i = (char *)hist + (size_t)__float_as_int(ri.w) * R.nt;
            }
            const int own = gj - Ij * (RDF_CHUNK / RDF_GROUP);   // below 4: a group of the chunk itself
            const int after = own < RDF_CHUNK / RDF_GROUP ? lane - own * RDF_GROUP : -1;
            const int cx = cd & 3, cy = (cd >> 2) & 3, cz = (cd >> 4) & 3;
            const float sx = cx == 2 ? -R.L0 : R.L0, sy = cy == 2 ? -R.L1 : R.L1, sz = cz == 2 ? -R.L2 : R.L2;
            const rdf_quad_t pj = (rdf_quad_t)(size_t)(R.pos + (size_t)gj * RDF_GROUP);
            const int form = (cx == 0 ? 0 : cx == 3 ? 2 : 1) * 9 + (cy == 0 ? 0 : cy == 3 ? 2 : 1) * 3 +
                             (cz == 0 ? 0 : cz == 3 ? 2 : 1);
#define RDF_FORM(F)                                                                                              \
    case F:                                                                                                      \
        rdf_group<(F) / 9, (F) / 3 % 3, (F) % 3>(R, pj, after, xi, yi, zi, sx, sy, sz, out_thr, thr, hist_i);          \
        break;
#define RDF_FORMS3(F) RDF_FORM(F) RDF_FORM(F + 1) RDF_FORM(F + 2)
#define RDF_FORMS9(F) RDF_FORMS3(F) RDF_FORMS3(F + 3) RDF_FORMS3(F + 6)
            switch (form) { RDF_FORMS9(0) RDF_FORMS9(9) RDF_FORMS9(18) }
#undef RDF_FORMS9
#undef RDF_FORMS3
#undef RDF_FORM
        }
        q += dq;
        u += du;
        if (u >= R.nper) {
            u -= R.nper;
            ++q;
        }
    }
    __syncthreads();
    GMEM unsigned *dst = R.part + (size_t)blockIdx.x * nh;
    for (int x = threadIdx.x; x < nh; x += blockDim.x) dst[x] = hist[x];
}

// Independent FMA chains (8 per lane) for gmd_fma_probe: 16 flop per lane and
// iteration, the sums stored so nothing is optimised away.
__global__ void __launch_bounds__(256) k_fma(int iters, float *out_p) {
    GMEM float *out = (GMEM float *)out_p;
    float a[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) a[k] = (float)(threadIdx.x + k) * 1e-3f;
    const float m = 0.999f, c = 1e-4f;
    for (int it = 0; it < iters; ++it) {
#pragma unroll
        for (int k = 0; k < 8; ++k) a[k] = fmaf(a[k], m, c);
    }
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) s += a[k];
    out[blockIdx.x * blockDim.x + threadIdx.x] = s;
}

// zero n floats (a fill kernel, not a memset)
__global__ void __launch_bounds__(256) k_fill_f32(float *p_p, size_t n) {
    GMEM float *p = (GMEM float *)p_p;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] = 0.f;
}

// Plain streaming copy (n float4), the known-size HBM workload of gmd_copy_probe:
// each thread keeps four 16-byte loads in flight (elements one grid stride
// apart), then stores them.
__global__ void __launch_bounds__(256) k_copy(const float4 *src_p, float4 *dst_p, size_t n) {
    const GMEM float4 *src = (const GMEM float4 *)src_p;
    GMEM float4 *dst = (GMEM float4 *)dst_p;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    for (; i + 3 * stride < n; i += 4 * stride) {
        float4 a[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) a[u] = src[i + u * stride];
#pragma unroll
        for (int u = 0; u < 4; ++u) dst[i + u * stride] = a[u];
    }
    for (; i < n; i += stride) dst[i] = src[i];
}

// ---------------------------------------------------------------------------
// The radial distribution of host positions without device allocations
// (gmd_rdf_compute_host_noalloc): every device buffer of the histogram lives
// in one file-scope array, 'scratch', of a fixed size.  Each device holds its
// own copy; the host reaches it through the address hipGetSymbolAddress gives
// on that device (the array's name in host code is not a device address).
// ---------------------------------------------------------------------------
#define NOALLOC_RDF_MAX_N 65536      // particles
#define NOALLOC_RDF_MAX_HIST 4096    // ntypes * ntypes * bins
#define NOALLOC_RDF_GRID 512         // histogram blocks (per-block partial histograms)
// byte offsets of the buffers inside 'scratch' (each 256-byte aligned)
#define NOALLOC_OFF_R 0                                                           // float [3 N]
#define NOALLOC_OFF_T (NOALLOC_OFF_R + 3 * 4 * NOALLOC_RDF_MAX_N)                // int [N]
#define NOALLOC_OFF_POS (NOALLOC_OFF_T + 4 * NOALLOC_RDF_MAX_N)                  // float4 [N]
#define NOALLOC_OFF_GBOX (NOALLOC_OFF_POS + 16 * NOALLOC_RDF_MAX_N)              // float4 [4 groups]
#define NOALLOC_OFF_CBOX (NOALLOC_OFF_GBOX + 16 * 4 * (NOALLOC_RDF_MAX_N / RDF_GROUP))   // float4 [4 chunks]
#define NOALLOC_OFF_KEY (NOALLOC_OFF_CBOX + 16 * 4 * (NOALLOC_RDF_MAX_N / RDF_CHUNK))    // int2 [N]
#define NOALLOC_OFF_CELL (NOALLOC_OFF_KEY + 8 * NOALLOC_RDF_MAX_N)               // int [cells]
#define NOALLOC_OFF_THR (NOALLOC_OFF_CELL + 4 * RDF_MAX_CELL * RDF_MAX_CELL * RDF_MAX_CELL)   // float [bins + 1]
#define NOALLOC_OFF_PART (NOALLOC_OFF_THR + ((4 * (NOALLOC_RDF_MAX_HIST + 1) + 255) / 256) * 256)   // u32 [grid][hist]
#define NOALLOC_OFF_OUT (NOALLOC_OFF_PART + 4 * NOALLOC_RDF_GRID * NOALLOC_RDF_MAX_HIST)   // u64 [hist]
#define NOALLOC_BYTES (NOALLOC_OFF_OUT + 8 * NOALLOC_RDF_MAX_HIST)

static __device__ __align__(256) unsigned char scratch[NOALLOC_BYTES];

// a fill kernel instead of a memset, so the clear can sit in a captured graph
__global__ void __launch_bounds__(256) k_fill_u64(unsigned long long *p_p, int n) {
    GMEM unsigned long long *p = (GMEM unsigned long long *)p_p;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0ull;
}

// Sum the per-block histograms: thread (x, chunk) adds 'per' blocks of bin x.
__global__ void k_rdf_reduce(const unsigned *part_p, int nblocks, int nh, int per, unsigned long long *out_p) {
    const GMEM unsigned *part = (const GMEM unsigned *)part_p;
    GMEM unsigned long long *out = (GMEM unsigned long long *)out_p;
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    if (x >= nh) return;
    const int b0 = blockIdx.y * per, b1 = min(nblocks, b0 + per);
    unsigned long long s = 0;
    for (int b = b0; b < b1; ++b) s += part[(size_t)b * nh + x];
    if (s) atomicAdd(gen_ptr(out + x), s);
}

// ============================================================================
// Renumbering of the particles in cell order (gather locality for the step,
// rebuild and histogram kernels).  Deterministic: cells in index order,
// particles of a cell in their previous order.
// ============================================================================
// Morton code of a cell's coordinates (bits interleaved x, y, z): cells close
// in space get close keys, so a run of consecutive particles is a compact
// block of cells
__device__ __forceinline__ unsigned spread3(unsigned v) {
    v &= 0x3ffu;
    v = (v | (v << 16)) & 0x030000ffu;
    v = (v | (v << 8)) & 0x0300f00fu;
    v = (v | (v << 4)) & 0x030c30c3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

__global__ void __launch_bounds__(256) k_sort_count(const DP *__restrict__ Pp, int cur, int *key, int *cnt) {
    const DP &P = *Pp;
    cpos_t pos = cur ? P.pos1 : P.pos0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < P.N; i += gridDim.x * blockDim.x) {
        const float4 r = pos[i];
        const int c = cell_of(P, r.x, r.y, r.z);
        const unsigned cz = c % P.ncz, cy = (c / P.ncz) % P.ncy, cx = c / (P.ncz * P.ncy);
        const int k = (int)((spread3(cx) << 2) | (spread3(cy) << 1) | spread3(cz));
        key[i] = k;
        atomicAdd(cnt + k, 1);
    }
}

// Exclusive prefix sum of the key counts in place: the sums of chunks of
// SCAN_CHUNK counts, then each block scans its chunk on top of the sums before
// it.  (One block over all counts read each thread's run of counts alone, one
// load after another: LJ N = 1048576, 2097152 keys, 3650 us a renumbering.)
#define SCAN_CHUNK 4096
__device__ __forceinline__ int scan_block_sum(int v, int *red) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    v = red[0] + red[1] + red[2] + red[3];
    __syncthreads();
    return v;
}

__global__ void __launch_bounds__(256) k_scan_sums(const int *a, int n, int *sums) {
    __shared__ int red[4];
    const int b = blockIdx.x * SCAN_CHUNK;
    int s = 0;
#pragma unroll
    for (int u = 0; u < SCAN_CHUNK / 256; ++u) {
        const int k = b + u * 256 + (int)threadIdx.x;
        if (k < n) s += a[k];
    }
    s = scan_block_sum(s, red);
    if (threadIdx.x == 0) sums[blockIdx.x] = s;
}

__global__ void __launch_bounds__(256) k_scan(int *a, int n, const int *sums) {
    __shared__ int red[4];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    int before = 0;
    for (int k = threadIdx.x; k < (int)blockIdx.x; k += 256) before += sums[k];
    before = scan_block_sum(before, red);
    // a thread's run of counts
    constexpr int R = SCAN_CHUNK / 256;
    const int k0 = blockIdx.x * SCAN_CHUNK + (int)threadIdx.x * R;
    int v[R], s = 0;
#pragma unroll
    for (int u = 0; u < R; ++u) {
        v[u] = k0 + u < n ? a[k0 + u] : 0;
        s += v[u];
    }
    int inc = s;
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(inc, o, 64);
        if (lane >= o) inc += y;
    }
    if (lane == 63) red[wid] = inc;
    __syncthreads();
    int base = before + inc - s;
    for (int x = 0; x < wid; ++x) base += red[x];
#pragma unroll
    for (int u = 0; u < R; ++u) {
        if (k0 + u < n) a[k0 + u] = base;
        base += v[u];
    }
}

__global__ void __launch_bounds__(256) k_sort_scatter(int N, const int *key, int *cursor, int *order) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x)
        order[atomicAdd(cursor + key[i], 1)] = i;
}

// particles of one cell in ascending previous index
__global__ void __launch_bounds__(256) k_sort_cells(const int *start, int ncells, int N, int *order) {
    for (int c = blockIdx.x * blockDim.x + threadIdx.x; c < ncells; c += gridDim.x * blockDim.x) {
        const int b = start[c], e = (c + 1 < ncells) ? start[c + 1] : N;
        for (int x = b + 1; x < e; ++x) {
            const int v = order[x];
            int y = x - 1;
            while (y >= b && order[y] > v) {
                order[y + 1] = order[y];
                --y;
            }
            order[y + 1] = v;
        }
    }
}

// new[k] = old[order[k]] for every per-particle array; the positions go to
// the other ping-pong buffer (the caller flips buf0)
struct PermBufs {
    float4 *vel, *frc, *rref, *obeta;
    float *sc;
    int *rim, *perm;
};

__global__ void __launch_bounds__(256) k_permute(const DP *__restrict__ Pp, int cur, const int *order, PermBufs T) {
    const DP &P = *Pp;
    const int N = P.N;
    cpos_t src = cur ? P.pos1 : P.pos0;
    pos_t dst = cur ? P.pos0 : P.pos1;
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < N; k += gridDim.x * blockDim.x) {
        const int o = order[k];
        dst[k] = src[o];
        T.vel[k] = P.vel[o];
        T.frc[k] = P.frc[o];
        T.rref[k] = P.rref[o];
        T.obeta[k] = P.obeta[o];
        for (int c = 0; c < 5; ++c) T.sc[(size_t)c * N + k] = P.sc[(size_t)c * N + o];
        for (int c = 0; c < 3; ++c) T.rim[(size_t)c * N + k] = P.rim[(size_t)c * N + o];
        T.perm[k] = P.perm[o];
    }
}

// inverse of the permutation: order[perm[i]] = i (the caller's order back)
__global__ void __launch_bounds__(256) k_perm_inverse(const DP *__restrict__ Pp, int *order) {
    const DP &P = *Pp;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < P.N; i += gridDim.x * blockDim.x) order[P.perm[i]] = i;
}

// ============================================================================
// Host side
// ============================================================================
namespace {

thread_local std::string g_err;

int fail(const char *fmt, ...) {
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    g_err = buf;
    return -1;
}

#define HIPCHECK(x)                                                                        \
    do {                                                                                   \
        hipError_t e_ = (x);                                                               \
        if (e_ != hipSuccess) return fail("%s: %s (%s:%d)", #x, hipGetErrorString(e_), __FILE__, __LINE__); \
    } while (0)

template <typename T>
int dalloc(T **p, size_t n) {
    *p = nullptr;
    if (n == 0) n = 1;
    HIPCHECK(hipMalloc((void **)p, n * sizeof(T)));
    return 0;
}

// Device buffers of one owner in one allocation (an allocation costs about as
// much as a small system's step): pointers are registered with their sizes,
// those to be cleared first, then allocated together
struct Arena {
    struct Want {
        void **p;
        size_t bytes;
    };
    std::vector<Want> zeroed, plain;
    char *base = nullptr;

    template <typename T>
    void add(T **p, size_t n, bool zero = false) {
        *p = nullptr;
        (zero ? zeroed : plain).push_back(Want{(void **)p, std::max<size_t>(n, 1) * sizeof(T)});
    }
    static size_t padded(size_t bytes) { return (bytes + 255) / 256 * 256; }

    int allocate() {
        size_t total = 0, clear = 0;
        for (const Want &w : zeroed) clear += padded(w.bytes);
        total = clear;
        for (const Want &w : plain) total += padded(w.bytes);
        HIPCHECK(hipMalloc((void **)&base, total));
        HIPCHECK(hipMemset(base, 0, clear));
        size_t at = 0;
        for (const std::vector<Want> *v : {&zeroed, &plain})
            for (const Want &w : *v) {
                *w.p = base + at;
                at += padded(w.bytes);
            }
        return 0;
    }
};

typedef void (*kfun)(const DP *);
typedef void (*sfun)(const DP *, int);
typedef void (*bfun)(const DP *, const BatchBlk *);
typedef void (*bsfun)(const DP *, const BatchBlk *, int);

// the kernel instances of one (pair function, cutoff, integrator) combination
// and list kind
struct Kernels {
    kfun pers;
    sfun step;
    bfun bpers;
    bsfun bstep;
};

template <int BASE, int CUT, int INTEG>
Kernels pick(int kind) {
    return Kernels{kind == 1 ? k_persistent<BASE, CUT, INTEG, 1> : k_persistent<BASE, CUT, INTEG, 0>,
                   kind == 1 ? k_step<BASE, CUT, INTEG, 1> : k_step<BASE, CUT, INTEG, 0>,
                   k_batch_persistent<BASE, CUT, INTEG>, k_batch_step<BASE, CUT, INTEG>};
}

template <int BASE, int CUT>
Kernels pick_integ(int integ, int kind) {
    switch (integ) {
        case 0: return pick<BASE, CUT, 0>(kind);
        case 1: return pick<BASE, CUT, 1>(kind);
        case 2: return pick<BASE, CUT, 2>(kind);
        case 3: return pick<BASE, CUT, 3>(kind);
        default: return pick<BASE, CUT, 4>(kind);
    }
}

template <int BASE>
Kernels pick_cut(int cut, int integ, int kind) {
    switch (cut) {
        case 0: return pick_integ<BASE, 0>(integ, kind);
        case 1: return pick_integ<BASE, 1>(integ, kind);
        default: return pick_integ<BASE, 2>(integ, kind);
    }
}

// pair functions 2..5 share one instance (a uniform switch on the kind
// inside), and so do 6..7 (parameter rows)
Kernels pick_kernels(int base, int cut, int integ, int kind) {
    return base == 0   ? pick_cut<0>(cut, integ, kind)
           : base == 1 ? pick_cut<1>(cut, integ, kind)
           : base <= 5 ? pick_cut<2>(cut, integ, kind)
                       : pick_cut<3>(cut, integ, kind);
}

// One host array's place in the packed buffer: words [at, at + n)
struct HostSeg {
    void *host;
    size_t at, n;
};

// Words [lo, hi) of the packed buffer, held at buf, to or from the host
// arrays they belong to (one thread: a core copies tens of GB/s here, and
// starting another costs 25 us)
void host_move(int *buf, size_t lo, size_t hi, const std::vector<HostSeg> &segs, bool into) {
    for (const HostSeg &s : segs) {
        const size_t b = std::max(lo, s.at), e = std::min(hi, s.at + s.n);
        if (b >= e) continue;
        char *h = (char *)s.host + (b - s.at) * 4, *p = (char *)(buf + (b - lo));
        memcpy(into ? p : h, into ? h : p, (e - b) * 4);
    }
}

bool is_pow2(int x) { return x > 0 && (x & (x - 1)) == 0; }

int ilog2(int x) {
    int s = 0;
    while ((1 << s) < x) ++s;
    return s;
}

}  // namespace

static const int GRAPH_STEPS = 20;
static const double NPT_GRID_SHRINK = 0.95;   // smallest box (per side, relative) an NPT cell grid admits

struct gmd_ctx {
    gmd_desc d;
    std::vector<float> params;
    std::vector<int> excl;
    std::vector<int> boff;       // bonds per particle (CSR offsets, N + 1; empty: no bonds)
    std::vector<int2> bnd;       // (partner, bond type) per entry
    std::vector<float2> bpar;    // (r0, k) per bond type
    char *arena = nullptr;       // every device buffer but rebuild_flag
    hipEvent_t xev[2] = {nullptr, nullptr};   // a half of xhost is free again / has arrived
    size_t xcap = 0;             // words of xhost
    int *pinned = nullptr;       // pinned host memory: the published control block and saver rows, then xhost
    int *xhost = nullptr, *xdev = nullptr;   // packed host arrays (XferSeg), in pinned and in device memory
    Ctrl *pub = nullptr;         // the control block as of the end of the last run
    bool pub_valid = false;      // nothing has changed the device's control block since pub was written
    bool fetched = false;        // xhost holds the current state (gmd_batch_fetch)
    bool all_cols = true;        // every column of the host's scalar rows has a device array
    hipStream_t stream = nullptr;
    bool own_stream = true;   // false: a replica of a gmd_batch (the batch owns the stream and the context)
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    int cus = 0;
    // device
    float4 *pos0 = nullptr, *pos1 = nullptr, *vel = nullptr, *frc = nullptr, *rref = nullptr, *obeta = nullptr;
    float *sc = nullptr;
    int *rim = nullptr, *nbl = nullptr, *nbc = nullptr;
    int *ccount = nullptr, *cmem = nullptr;   // cell grid, three rotating buffers
    int *d_excl = nullptr;
    int *d_boff = nullptr;
    int2 *d_bnd = nullptr;
    float2 *d_bpar = nullptr;
    float *d_params = nullptr;
    Ctrl *ctrl = nullptr;
    float *partial = nullptr;
    int *rebuild_flag = nullptr;
    int rebuild_cap = 0;
    float *saver_out = nullptr;
    float *conf_out = nullptr;   // ConfigurationSaver array (conf_saves_per_block > 0)
    float cur_box[3] = {0.f, 0.f, 0.f};   // the box after the last run (NPT_Atomic changes it)
    PairP *ptab = nullptr;       // prepared pair table
    bool ptab_ready = false;
    size_t nbl_len = 0;          // words of the neighbour list
    bool nb16 = false;           // 16-bit list entries
    // renumbering in cell order
    int *perm = nullptr, *skey = nullptr, *sorder = nullptr, *scnt = nullptr, *scur = nullptr, *ssum = nullptr;
    PermBufs tb = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
    int nkeys = 0;                // Morton key space of the renumbering
    int reorder_every = 0;        // steps between renumberings (0: never)
    long long since_reorder = 0;  // steps since the last renumbering
    bool permuted = false;        // perm is not the identity
    long long renumberings = 0;   // renumberings done so far
    // state
    int buf0 = 0;
    long long lstep = 0;
    bool need_rebuild = true;   // forced rebuild pending (first build, gmd_force_rebuild)
    float last_ms = 0.f;
    // launch
    DP P;
    DP *d_P = nullptr;            // device copy of P (kernels take a pointer)
    Kernels kern = {nullptr, nullptr, nullptr, nullptr};
    int block = 256, grid_pers = 1, grid_step = 1, grid_aux = 1;
    size_t lds_pers = 0, lds_step = 0, lds_build = 0;
    hipGraphExec_t gexec = nullptr;
    hipGraph_t graph = nullptr;
};

// Positions and types of the host go to the device in one copy up to this many
// particles: a copy waits for its end, about 15 us, which is more than bringing
// them together takes (whole updates with two copies and with one: N = 300 77
// and 67 us, 4000 98 and 79, 8000 111 and 101, 30000 376 and 374).
#define RDF_ONE_COPY 32768

struct gmd_rdf {
    int N, nt, bins, nchunks;
    float4 *pos = nullptr;    // snapshot of a context's positions; (N, 3) positions of the host
    float4 *sorted = nullptr; // what the kernels read: cell order, whole chunks
    float4 *gbox = nullptr, *cbox = nullptr;   // group and chunk boxes, 4 each
    int2 *key = nullptr;
    int *ptype = nullptr;
    std::vector<int> h_in;    // the host's positions and types, for one copy of both (RDF_ONE_COPY)
    float *d_thr = nullptr;
    unsigned *part = nullptr;
    unsigned long long *d_out = nullptr;   // the counts, and after them the sorting cells (cleared together)
    int grid = 0;      // histogram blocks of a launch whose result is awaited at once
    int grid_bg = 0;   // fewer blocks for a launch that runs beside the simulation's steps
    float box[3] = {0, 0, 0};
    std::vector<float> thr;
    hipStream_t stream = nullptr;
    hipEvent_t snap = nullptr, done = nullptr;   // snapshot taken on the context's stream; result on the host
    unsigned long long *h_out = nullptr;         // pinned: the reduced counts of the last launch
    bool pending = false;                        // a launched update not collected yet
};

extern "C" {

int gmd_abi_version(void) { return GMD_ABI_VERSION; }

int gmd_desc_size(void) { return (int)sizeof(gmd_desc); }

const char *gmd_last_error(void) { return g_err.c_str(); }

int gmd_get_device_info(gmd_device_info *out) {
    if (!out) return fail("gmd_get_device_info: null output");
    int dev = 0;
    HIPCHECK(hipGetDevice(&dev));
    hipDeviceProp_t p;
    HIPCHECK(hipGetDeviceProperties(&p, dev));
    out->compute_units = p.multiProcessorCount;
    out->wavefront_size = p.warpSize;
    out->max_threads_per_block = p.maxThreadsPerBlock;
    out->total_mem = (long long)p.totalGlobalMem;
    snprintf(out->name, sizeof out->name, "%s", p.name);
    snprintf(out->arch, sizeof out->arch, "%s", p.gcnArchName);
    return 0;
}

static int ctx_free(gmd_ctx *c) {
    if (!c) return 0;
    if (c->gexec) hipGraphExecDestroy(c->gexec);
    if (c->graph) hipGraphDestroy(c->graph);
    if (c->arena) hipFree(c->arena);
    if (c->rebuild_flag) hipFree(c->rebuild_flag);
    for (hipEvent_t e : c->xev)
        if (e) hipEventDestroy(e);
    if (c->pinned) hipHostFree(c->pinned);
    if (c->ev0) hipEventDestroy(c->ev0);
    if (c->ev1) hipEventDestroy(c->ev1);
    if (c->stream && c->own_stream) hipStreamDestroy(c->stream);
    delete c;
    return 0;
}

static int ctx_create(const gmd_desc *desc, gmd_ctx **out, hipStream_t shared_stream);
static int unpermute(gmd_ctx *c);
static int host_perm(gmd_ctx *c, std::vector<int> &perm);

int gmd_create(const gmd_desc *desc, gmd_ctx **out) { return ctx_create(desc, out, nullptr); }

// shared_stream != nullptr: the context works on the caller's stream (a batch
// of replicas) instead of creating its own
static int ctx_create(const gmd_desc *desc, gmd_ctx **out, hipStream_t shared_stream) {
    if (!desc || !out) return fail("gmd_create: null argument");
    *out = nullptr;
    const gmd_desc &d = *desc;
    if (d.abi_version != GMD_ABI_VERSION)
        return fail("gmd_create: ABI version %d, library expects %d", d.abi_version, GMD_ABI_VERSION);
    if (d.D != 3) return fail("gmd_create: only D=3 is supported (got D=%d)", d.D);
    if (d.N < 1) return fail("gmd_create: N must be positive (got %d)", d.N);
    if (d.ntypes < 1 || d.ntypes > MAX_TYPES) return fail("gmd_create: ntypes must be in [1,%d]", MAX_TYPES);
    if (d.pair_base < 0 || d.pair_base > GMD_PAIR_SUM) return fail("gmd_create: unknown pair function %d", d.pair_base);
    const bool param_rows = d.pair_base >= GMD_SAAP;   // SAAP, sums: parameter rows
    if (param_rows) {
        if (d.nparams < 2 || d.nparams > 9)
            return fail("gmd_create: nparams must be in [2, 9] for parameter rows (got %d)", d.nparams);
        const int nterms = d.pair_base == GMD_SAAP ? 1 : d.nterms;
        if (nterms < 1 || nterms > 2) return fail("gmd_create: a sum of pair functions has 1 or 2 terms (got %d)", nterms);
        for (int k = 0; k < nterms; ++k) {
            const int kind = d.pair_base == GMD_SAAP ? GMD_SAAP : d.term_kind[k];
            const int first = d.pair_base == GMD_SAAP ? 0 : d.term_first[k];
            if (kind < 0 || kind > GMD_SAAP) return fail("gmd_create: unknown term function %d", kind);
            const int need = kind == GMD_SAAP ? 8 : kind == GMD_HERTZIAN ? 3 : kind == GMD_IPL_N ? 1 : 2;
            if (first < 0 || first + need > d.nparams - 1)
                return fail("gmd_create: term %d reads parameters %d..%d of a row of %d before the cut", k, first,
                            first + need - 1, d.nparams - 1);
            const float *ex = d.term_exps + 2 * k;
            if ((kind == GMD_IPL_N || kind == GMD_LJ_M_N) && !(ex[0] > 0.0f))
                return fail("gmd_create: the exponent of an IPL_n / LJ_m_n term must be positive");
            if (kind == GMD_LJ_M_N && !(ex[1] > 0.0f))
                return fail("gmd_create: the exponents of an LJ_m_n term must be positive");
        }
    }
    if ((d.pair_base == GMD_IPL_N || d.pair_base == GMD_LJ_M_N) && !(d.pair_exps[0] > 0.0f))
        return fail("gmd_create: the exponent of IPL_n / LJ_m_n must be positive");
    if (d.pair_base == GMD_LJ_M_N && !(d.pair_exps[1] > 0.0f))
        return fail("gmd_create: the exponents of LJ_m_n must be positive");
    if (d.pair_base == GMD_HERTZIAN && !(d.pair_exps[0] > 0.0f))
        return fail("gmd_create: the hertzian exponent alpha must be positive");
    if (d.cutoff < 0 || d.cutoff > 2) return fail("gmd_create: unknown cutoff wrapper %d", d.cutoff);
    if (d.nblist_kind < 0 || d.nblist_kind > 1) return fail("gmd_create: unknown nblist kind %d", d.nblist_kind);
    if (d.integrator < 0 || d.integrator > GMD_NPT_ATOMIC) return fail("gmd_create: unknown integrator %d", d.integrator);
    if (d.integrator == GMD_NPT_ATOMIC) {
        if (!d.compute_w) return fail("gmd_create: NPT_Atomic requires virial (compute_w)");
        if (!(d.mass_t > 0.f) || !(d.mass_p > 0.f) || d.degrees < 2)
            return fail("gmd_create: NPT_Atomic needs positive thermostat and barostat masses and N D - D >= 2");
        if (d.pfunc < 0 || d.pfunc > 2) return fail("gmd_create: unknown pressure schedule %d", d.pfunc);
    }
    if (d.max_nbs < 1) return fail("gmd_create: max_nbs must be positive");
    if (!d.params) return fail("gmd_create: params missing");
    if (!is_pow2(d.tp) || d.tp > 64) return fail("gmd_create: tp must be a power of two <= 64 (got %d)", d.tp);
    if (d.pb < 1) return fail("gmd_create: pb must be positive");
    for (int k = 0; k < 3; ++k)
        if (!(d.box[k] > 0.f)) return fail("gmd_create: box lengths must be positive");
    if (d.scalar_save_every > 0 && d.scalar_saves_per_block < 1)
        return fail("gmd_create: scalar_saves_per_block must be positive");
    if (d.nbonds < 0) return fail("gmd_create: nbonds must not be negative");
    if (d.nbonds > 0) {
        if (!d.bonds || !d.bond_params || d.nbond_types < 1)
            return fail("gmd_create: bonds need their index rows and at least one bond type");
        for (int b = 0; b < d.nbonds; ++b) {
            const int *e = d.bonds + 3 * (size_t)b;
            if (e[0] < 0 || e[0] >= d.N || e[1] < 0 || e[1] >= d.N || e[0] == e[1])
                return fail("gmd_create: bond %d joins particles %d and %d (N = %d)", b, e[0], e[1], d.N);
            if (e[2] < 0 || e[2] >= d.nbond_types)
                return fail("gmd_create: bond %d has type %d, outside [0, %d)", b, e[2], d.nbond_types);
        }
    }

    gmd_ctx *c = new gmd_ctx();
    c->d = d;
    const int N = d.N;
    const int nparams = param_rows ? d.nparams : 3;
    c->params.assign(d.params, d.params + (size_t)d.ntypes * d.ntypes * nparams);
    if (d.exclusions && d.exclusions_cols > 0) c->excl.assign(d.exclusions, d.exclusions + (size_t)N * d.exclusions_cols);
    if (d.nbonds > 0) {
        // each bond under both its ends, in bond order
        c->boff.assign((size_t)N + 1, 0);
        for (int b = 0; b < d.nbonds; ++b) {
            ++c->boff[(size_t)d.bonds[3 * (size_t)b] + 1];
            ++c->boff[(size_t)d.bonds[3 * (size_t)b + 1] + 1];
        }
        for (int i = 0; i < N; ++i) c->boff[(size_t)i + 1] += c->boff[i];
        std::vector<int> fill(c->boff.begin(), c->boff.end() - 1);
        c->bnd.resize((size_t)2 * d.nbonds);
        for (int b = 0; b < d.nbonds; ++b) {
            const int *e = d.bonds + 3 * (size_t)b;
            c->bnd[(size_t)fill[e[0]]++] = make_int2(e[1], e[2]);
            c->bnd[(size_t)fill[e[1]]++] = make_int2(e[0], e[2]);
        }
        for (int t = 0; t < d.nbond_types; ++t)
            c->bpar.push_back(make_float2(d.bond_params[2 * t], d.bond_params[2 * t + 1]));
    }
    c->d.params = nullptr;
    c->d.exclusions = nullptr;
    c->d.bonds = nullptr;
    c->d.bond_params = nullptr;

    int rc = 0;
#define TRY(x)                 \
    do {                       \
        if ((rc = (x)) != 0) { \
            ctx_free(c);       \
            return rc;         \
        }                      \
    } while (0)
#define HTRY(x)                                                                 \
    do {                                                                        \
        hipError_t e_ = (x);                                                    \
        if (e_ != hipSuccess) {                                                 \
            ctx_free(c);                                                        \
            return fail("%s: %s", #x, hipGetErrorString(e_));                   \
        }                                                                       \
    } while (0)

    int dev = 0;
    HTRY(hipGetDevice(&dev));
    HTRY(hipDeviceGetAttribute(&c->cus, hipDeviceAttributeMultiprocessorCount, dev));
    if (shared_stream) {
        c->stream = shared_stream;
        c->own_stream = false;
    } else {
        HTRY(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
    }
    HTRY(hipEventCreate(&c->ev0));
    HTRY(hipEventCreate(&c->ev1));

    // ---- cell grid (nblist_linked_lists.py:36-42) ----
    int ncx = 1, ncy = 1, ncz = 1;
    // NPT_Atomic: the grid stays valid while the box is at least 95% of its
    // starting lengths (the cells no smaller than (rc + skin) / 2)
    const double grid_scale = d.integrator == GMD_NPT_ATOMIC ? NPT_GRID_SHRINK : 1.0;
    if (d.nblist_kind == GMD_NBLIST_LINKED_LISTS) {
        double min_size = ((double)d.max_cut + (double)d.skin) / 2.0;
        ncx = (int)((double)d.box[0] * grid_scale / min_size);
        ncy = (int)((double)d.box[1] * grid_scale / min_size);
        ncz = (int)((double)d.box[2] * grid_scale / min_size);
        if (ncx <= 6 || ncy <= 4 || ncz <= 4) {
            ctx_free(c);
            return fail("linked lists need more than 6 cells in x and more than 4 in y and z "
                        "(box/((max_cut+skin)/2) gives %d x %d x %d); use 'N squared'", ncx, ncy, ncz);
        }
    }
    const int ncells = ncx * ncy * ncz;
    if (d.nblist_kind == GMD_NBLIST_LINKED_LISTS && N >= LL_MAX_N) {
        ctx_free(c);
        return fail("linked lists support at most %d particles (got %d)", LL_MAX_N - 1, N);
    }

    // ---- launch geometry ----
    const int tp = d.tp;
    int block = d.pb * tp;
    if (block % 64) block = ((block + 63) / 64) * 64;
    if (block > 256) block = 256;
    c->block = block;
    const int slots = block / tp;
    c->grid_step = (N + slots - 1) / slots;
    c->grid_aux = std::max(1, std::min((N + block - 1) / block, c->cus * 16));
    const int wpb = block / 64;
    // dynamic LDS: pair table | reduction scratch (one row of sums per wave) |
    // rebuild scratch; sized so that four blocks of 256 fit in a CU's 160 KB
    const size_t lds_cells = (d.nblist_kind == GMD_NBLIST_LINKED_LISTS) ? (size_t)wpb * LL_WAVE_LDS : 0;
    // N squared: two tiles of positions (16 B each) and the accepted slots of a wave's particles
    // (a list step stages each wave's velocities and reference positions in
    // the same region: 2 KB a wave)
    // (and a deferred Nose-Hoover tail stages the previous step's kinetic
    // partials after them: RED_PRE floats a thread)
    const size_t lds_nsq = (size_t)block * 32 + (size_t)wpb * NSQ_PP * NSQ_CAP * 2;
    c->lds_build = std::max(std::max(lds_cells, lds_nsq), (size_t)wpb * 2048 + (size_t)RED_PRE * block * 4);
    const size_t lds_pp = 0;
    const size_t lds_red = ((size_t)d.ntypes * d.ntypes * sizeof(PairP) + 15) / 16 * 16;
    const size_t lds_b = lds_red + (size_t)wpb * GMD_NRED * sizeof(double);
    c->lds_step = lds_b + c->lds_build;
    c->lds_pers = c->lds_step;
    // cell capacity: room for 4x the mean occupancy, at least 16, at most 64
    int ccap = 16;
    if (d.nblist_kind == GMD_NBLIST_LINKED_LISTS) {
        const double mean = (double)N / ncells;
        while (ccap < 4.0 * mean + 8.0 && ccap < LL_OWNCAP) ccap *= 2;
        if (4.0 * mean + 8.0 > LL_OWNCAP) {
            ctx_free(c);
            return fail("linked lists: %.1f particles per cell on average exceeds the cell capacity %d", mean, LL_OWNCAP);
        }
    }

    // ---- buffers ----
    // list slots per particle: max_nbs, or with UtilizeNIII twice that, as the
    // full list is kept and max_nbs bounds the half list (nblist.py:112-116)
    const int slots_nb = d.utilize_niii ? 2 * d.max_nbs : d.max_nbs;
    // at least 8 rows: the force loop requests the first 8 rows before the
    // count arrives; with 16-bit entries (N <= 65536) two rows share a word
    c->nb16 = N <= 65536;
    size_t rows = std::max((size_t)(slots_nb + tp - 1) / tp, (size_t)8);
    if (c->nb16) rows = (rows + 1) & ~(size_t)1;
    c->nbl_len = (c->nb16 ? rows / 2 : rows) * (size_t)N * tp;
    Arena A;
    A.add(&c->pos0, N);
    A.add(&c->pos1, N);
    A.add(&c->vel, N);
    A.add(&c->frc, N, true);
    A.add(&c->rref, N, true);
    A.add(&c->obeta, N, true);
    A.add(&c->sc, (size_t)5 * N, true);
    A.add(&c->rim, (size_t)3 * N, true);
    A.add(&c->nbl, c->nbl_len, true);   // entries past a count stay valid indices
    A.add(&c->nbc, N, true);
    A.add(&c->ccount, (size_t)3 * ncells, true);
    A.add(&c->cmem, (size_t)3 * ncells * ccap, true);
    A.add(&c->d_params, c->params.size());
    A.add(&c->ptab, (size_t)d.ntypes * d.ntypes);
    A.add(&c->ctrl, 1);
    const int max_grid = std::max(c->grid_step, c->cus * 32);
    A.add(&c->partial, (size_t)2 * max_grid * GMD_NRED);   // two buffers: steps alternate (folded tail)
    A.add(&c->saver_out, (size_t)std::max(1, d.scalar_saves_per_block) * 6, true);
    if (d.conf_saves_per_block > 0) A.add(&c->conf_out, (size_t)d.conf_saves_per_block * 6 * N, true);
    A.add(&c->perm, N);
    int side = 1;
    while (side < std::max(ncx, std::max(ncy, ncz))) side *= 2;
    if (d.nblist_kind == GMD_NBLIST_LINKED_LISTS && c->excl.empty() && c->boff.empty() && !d.utilize_niii &&
        side <= 256) {
        // renumbering buffers (the exclusion and bond tables are indexed by
        // particle, and the NIII half-list rule by the caller's index, so
        // systems with exclusions, bonds or UtilizeNIII keep the caller's
        // numbering)
        A.add(&c->skey, N);
        A.add(&c->sorder, N);
        c->nkeys = side * side * side;
        A.add(&c->scnt, (size_t)c->nkeys);
        A.add(&c->scur, (size_t)c->nkeys);
        A.add(&c->ssum, (size_t)(c->nkeys + SCAN_CHUNK - 1) / SCAN_CHUNK);   // key counts of each chunk
        A.add(&c->tb.vel, N);
        A.add(&c->tb.frc, N);
        A.add(&c->tb.rref, N);
        A.add(&c->tb.obeta, N);
        A.add(&c->tb.sc, (size_t)5 * N);
        A.add(&c->tb.rim, (size_t)3 * N);
        A.add(&c->tb.perm, N);
        c->reorder_every = 400;
        c->since_reorder = 1LL << 40;
    }
    if (!c->excl.empty()) A.add(&c->d_excl, c->excl.size());
    if (!c->boff.empty()) {
        A.add(&c->d_boff, c->boff.size());
        A.add(&c->d_bnd, c->bnd.size());
        A.add(&c->d_bpar, c->bpar.size());
    }
    const XferSeg X((size_t)N, (size_t)std::max(0, d.nscalars));
    A.add(&c->xdev, X.end);
    A.add(&c->d_P, 1);
    rc = A.allocate();
    c->arena = A.base;
    TRY(rc);
    {
        std::vector<int> iota(N);
        for (int i = 0; i < N; ++i) iota[i] = i;
        HTRY(hipMemcpy(c->perm, iota.data(), (size_t)N * sizeof(int), hipMemcpyHostToDevice));
    }
    if (!c->excl.empty())
        HTRY(hipMemcpy(c->d_excl, c->excl.data(), c->excl.size() * sizeof(int), hipMemcpyHostToDevice));
    if (!c->boff.empty()) {
        HTRY(hipMemcpy(c->d_boff, c->boff.data(), c->boff.size() * sizeof(int), hipMemcpyHostToDevice));
        HTRY(hipMemcpy(c->d_bnd, c->bnd.data(), c->bnd.size() * sizeof(int2), hipMemcpyHostToDevice));
        HTRY(hipMemcpy(c->d_bpar, c->bpar.data(), c->bpar.size() * sizeof(float2), hipMemcpyHostToDevice));
    }
    HTRY(hipMemcpy(c->d_params, c->params.data(), c->params.size() * sizeof(float), hipMemcpyHostToDevice));
    Ctrl h_ctrl;
    memset(&h_ctrl, 0, sizeof h_ctrl);
    h_ctrl.shift_step = -1;
    for (int b = 0; b < 2; ++b) {   // NPT_Atomic: zero rates, the descriptor's box and its volume
        h_ctrl.npt[b][2] = d.box[0] * d.box[1] * d.box[2];
        for (int k = 0; k < 3; ++k) h_ctrl.npt[b][3 + k] = d.box[k];
    }
    HTRY(hipMemcpy(c->ctrl, &h_ctrl, sizeof h_ctrl, hipMemcpyHostToDevice));
    for (int k = 0; k < 3; ++k) c->cur_box[k] = d.box[k];
    {
        // the whole of a small system's arrays; a large one's go through it in
        // two halves by turns (pinning costs about 0.25 ms a MB)
        c->xcap = std::min(X.end, (size_t)2 * XFER_CHUNK);
        if (c->xcap < X.end)
            for (hipEvent_t &e : c->xev) HTRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        const size_t pub_words = (sizeof(Ctrl) / 4 + (size_t)std::max(1, d.scalar_saves_per_block) * 6 + 63) / 64 * 64;
        HTRY(hipHostMalloc((void **)&c->pinned, (pub_words + c->xcap) * 4, hipHostMallocDefault));
        c->pub = (Ctrl *)c->pinned;
        c->xhost = c->pinned + pub_words;
    }

    // ---- device parameter block ----
    DP &P = c->P;
    memset(&P, 0, sizeof P);
    P.N = N;
    P.ntypes = d.ntypes;
    P.tp = tp;
    P.tp_shift = ilog2(tp);
    P.max_nbs = slots_nb;
    P.nblist_kind = d.nblist_kind;
    P.niii = d.utilize_niii ? 1 : 0;
    P.max_half = d.max_nbs;
    P.box0 = d.box[0];
    P.box1 = d.box[1];
    P.box2 = d.box[2];
    P.ibox0 = 1.0f / d.box[0];
    P.ibox1 = 1.0f / d.box[1];
    P.ibox2 = 1.0f / d.box[2];
    {
        float cps = d.max_cut + d.skin;
        P.cps2 = cps * cps;
        P.skin2q = (d.skin * d.skin) * 0.25f;
        // A listed pair was closer than max_cut + skin at the rebuild and each
        // particle has moved less than skin / 2 since, so it is closer than
        // R = max_cut + 2 skin now; a particle with |x_d| <= L_d / 2 - R then
        // has every listed neighbour inside the box in its own image in
        // dimension d (rounding margin: 1e-4 relative plus 1e-3)
        const double R = ((double)d.max_cut + 2.0 * d.skin) * 1.0001 + 1e-3;
        P.mic_edge0 = (float)std::max(0.0, 0.5 * d.box[0] - R);
        P.mic_edge1 = (float)std::max(0.0, 0.5 * d.box[1] - R);
        P.mic_edge2 = (float)std::max(0.0, 0.5 * d.box[2] - R);
    }
    P.nrows = (int)rows;
    P.nb16 = c->nb16 ? 1 : 0;
    P.nwrows = (int)(c->nb16 ? rows / 2 : rows);
    P.pos0 = (GMEM float4 *)c->pos0;
    P.pos1 = (GMEM float4 *)c->pos1;
    P.vel = (GMEM float4 *)c->vel;
    P.frc = (GMEM float4 *)c->frc;
    P.rref = (GMEM float4 *)c->rref;
    P.obeta = (GMEM float4 *)c->obeta;
    P.sc = (GMEM float *)c->sc;
    P.rim = (GMEM int *)c->rim;
    P.nbl = (GMEM int *)c->nbl;
    P.nbc = (GMEM int *)c->nbc;
    P.ncx = ncx;
    P.ncy = ncy;
    P.ncz = ncz;
    P.ncells = ncells;
    P.ccap = ccap;
    P.ccount = (GMEM int *)c->ccount;
    P.cmem = (GMEM int *)c->cmem;
    P.excl = (const GMEM int *)c->d_excl;
    P.excl_cols = d.exclusions_cols;
    P.boff = (const GMEM int *)c->d_boff;
    P.bnd = (const GMEM int2 *)c->d_bnd;
    P.bpar = (const GMEM float2 *)c->d_bpar;
    P.raw_params = (const GMEM float *)c->d_params;
    P.ptab = (GMEM PairP *)c->ptab;
    P.nparams = nparams;
    if (d.pair_base == GMD_SAAP) {
        P.nterms = 1;
        P.term_kind[0] = GMD_SAAP;
        P.term_first[0] = 0;
        P.term_kind[1] = -1;
        P.term_first[1] = 0;
        for (int k = 0; k < 4; ++k) P.term_exps[k] = 0.0f;
    } else if (param_rows) {
        P.nterms = d.nterms;
        for (int k = 0; k < 2; ++k) {
            P.term_kind[k] = k < d.nterms ? d.term_kind[k] : -1;
            P.term_first[k] = k < d.nterms ? d.term_first[k] : 0;
        }
        for (int k = 0; k < 4; ++k) P.term_exps[k] = d.term_exps[k];
    }
    P.pair_base = d.pair_base;
    P.cutoff = d.cutoff;
    P.pexp0 = d.pair_exps[0];
    P.pexp1 = d.pair_exps[1];
    P.dt = d.dt;
    P.omega2 = d.omega2;
    P.alpha = d.alpha;
    P.degrees = (double)d.degrees;
    P.seed = d.seed;
    P.tfunc = d.tfunc;
    P.tpar0 = d.tparams[0];
    P.tpar1 = d.tparams[1];
    P.tpar2 = d.tparams[2];
    P.tpar3 = d.tparams[3];
    P.npt = d.integrator == GMD_NPT_ATOMIC ? 1 : 0;
    P.mass_t = d.mass_t;
    P.mass_p = d.mass_p;
    P.pfunc = d.pfunc;
    P.ppar0 = d.pparams[0];
    P.ppar1 = d.pparams[1];
    P.ppar2 = d.pparams[2];
    P.ppar3 = d.pparams[3];
    P.cell_min = (float)(((double)d.max_cut + (double)d.skin) / 2.0);
    P.compute_u = d.compute_u;
    P.compute_w = d.compute_w;
    P.compute_lap = d.compute_lap;
    P.compute_k = d.compute_k;
    P.compute_fsq = d.compute_fsq;
    P.mom_every = d.momentum_reset_every;
    P.save_every = d.scalar_save_every;
    P.saves_per_block = d.scalar_saves_per_block;
    P.ctrl = (GMEM Ctrl *)c->ctrl;
    P.partial = (GMEM float *)c->partial;
    P.pstride = max_grid;
    P.saver_out = (GMEM float *)c->saver_out;
    P.conf_saves = d.conf_saves_per_block > 0 ? d.conf_saves_per_block : 0;
    P.conf_out = (GMEM float *)c->conf_out;
    P.lds_pp = (int)lds_pp;
    P.lds_red = (int)lds_red;
    P.lds_build = (int)lds_b;
    P.step_grid = P.rebuild_grid = c->grid_step;
    P.perm = (const GMEM int *)c->perm;
    P.xdev = (GMEM int *)c->xdev;
    P.xhost = c->xhost;
    P.pub = c->pinned;
    // the scalar columns: a column outside the host's rows is absent (the
    // packing kernels index the rows with it), and two quantities may share one
    P.nscal = std::max(0, d.nscalars);
    std::vector<char> covered(P.nscal, 0);
    auto column = [&](int sid) {
        if (sid < 0 || sid >= P.nscal) return -1;
        covered[sid] = 1;
        return sid;
    };
    P.sid_u = column(d.sid_u);
    P.sid_w = column(d.sid_w);
    P.sid_lap = column(d.sid_lap);
    P.sid_k = column(d.sid_k);
    P.sid_fsq = column(d.sid_fsq);
    P.sid_m = column(d.sid_m);
    c->all_cols = std::count(covered.begin(), covered.end(), (char)1) == P.nscal;

    HTRY(hipMemcpy(c->d_P, &P, sizeof(DP), hipMemcpyHostToDevice));
    c->kern = pick_kernels(d.pair_base, d.cutoff, d.integrator, d.nblist_kind);

    // ---- cooperative grid: all blocks must be co-resident ----
    if (d.gridsync) {
        int nb = 0;
        HTRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, (const void *)c->kern.pers, block, c->lds_pers));
        if (nb < 1) {
            ctx_free(c);
            return fail("gridsync: persistent kernel cannot be resident with %d threads per block", block);
        }
        // at most eight wavefronts a CU: what the barrier after every step costs
        // grows with its blocks, and a third block a CU hides less than that
        // (NVE, linked lists, tp = 8, two and three blocks a CU: N = 20000 58 and
        // 70 us a step, N = 60000 74 and 101)
        nb = std::min(nb, std::max(1, 512 / block));
        c->grid_pers = std::max(1, std::min(c->grid_step, nb * c->cus));
    }
    *out = c;
    return 0;
#undef TRY
#undef HTRY
}

int gmd_destroy(gmd_ctx *ctx) {
    if (ctx && !ctx->own_stream) return fail("gmd_destroy: this context belongs to a batch; use gmd_batch_destroy");
    return ctx_free(ctx);
}

// blocks of a packing kernel
static dim3 xfer_grid(const gmd_ctx *c, size_t n) {
    return dim3((unsigned)std::max<size_t>(1, std::min<size_t>((n + 255) / 256, (size_t)c->cus * 8)));
}

// words of a packed buffer between host and device, on the context's stream
static int xfer_copy(gmd_ctx *c, const int *src, int *dst, size_t n, hipMemcpyKind kind) {
    if (n >= XFER_DMA)
        HIPCHECK(hipMemcpyAsync(dst, src, n * 4, kind, c->stream));
    else
        hipLaunchKernelGGL(k_copy_words, xfer_grid(c, n / 4), dim3(256), 0, c->stream, src, dst, n);
    return 0;
}

int gmd_upload(gmd_ctx *c, const float *r, const float *v, const float *f, const float *scalars, const int *ptype,
               const int *r_im) {
    if (!c) return fail("gmd_upload: null context");
    // work queued on the context's stream (a run, an RDF snapshot of the
    // positions) finishes before any of its buffers is overwritten
    HIPCHECK(hipStreamSynchronize(c->stream));
    const size_t N = c->d.N;
    const gmd_desc &d = c->d;
    if (ptype)
        for (size_t i = 0; i < N; ++i)
            if (ptype[i] < 0 || ptype[i] >= d.ntypes)
                return fail("gmd_upload: particle %d has type %d outside [0,%d)", (int)i, ptype[i], d.ntypes);
    if (unpermute(c)) return -1;   // host arrays come in the caller's numbering
    c->fetched = false;
    const XferSeg X(N, (size_t)std::max(0, d.nscalars));
    unsigned what = 0;
    size_t lo = X.end, hi = 0;
    std::vector<HostSeg> segs;
    auto take = [&](unsigned bit, const void *src, size_t at, size_t n) {
        if (!src || n == 0) return;
        what |= bit;
        lo = std::min(lo, at);
        hi = std::max(hi, at + n);
        segs.push_back(HostSeg{const_cast<void *>(src), at, n});
    };
    take(XF_R, r, X.r, 3 * N);
    take(XF_V, v, X.v, 3 * N);
    take(XF_F, f, X.f, 3 * N);
    take(XF_S, scalars, X.s, N * (size_t)std::max(0, d.nscalars));
    take(XF_T, ptype, X.t, N);
    take(XF_IM, r_im, X.im, 3 * N);
    if (!what) return 0;
    const int *src = c->xhost;
    if (c->xcap >= X.end) {
        host_move(c->xhost, 0, X.end, segs, true);
        if (N > XFER_DIRECT) {
            lo = lo / 4 * 4;   // (16-byte aligned in both buffers)
            if (xfer_copy(c, c->xhost + lo, c->xdev + lo, hi - lo, hipMemcpyHostToDevice)) return -1;
            src = c->xdev;
        }
    } else {
        // by halves: the host fills one while the other is on its way
        int half = 0, turn = 0;
        for (size_t at = lo; at < hi; at += XFER_CHUNK, half ^= 1, ++turn) {
            const size_t n = std::min((size_t)XFER_CHUNK, hi - at);
            int *buf = c->xhost + (size_t)half * XFER_CHUNK;
            if (turn >= 2) HIPCHECK(hipEventSynchronize(c->xev[half]));
            host_move(buf, at, at + n, segs, true);
            HIPCHECK(hipMemcpyAsync(c->xdev + at, buf, n * 4, hipMemcpyHostToDevice, c->stream));
            HIPCHECK(hipEventRecord(c->xev[half], c->stream));
        }
        src = c->xdev;
    }
    hipLaunchKernelGGL(k_pack, xfer_grid(c, N), dim3(256), 0, c->stream, (const DP *)c->d_P, c->buf0, what, src);
    HIPCHECK(hipGetLastError());
    // the current buffer becomes pos0; whether the list is still valid is
    // decided by the skin test at the start of the next run
    if (r || ptype) c->buf0 = 0;
    return 0;
}

int gmd_download(gmd_ctx *c, float *r, float *v, float *f, float *scalars, int *ptype, int *r_im) {
    if (!c) return fail("gmd_download: null context");
    const size_t N = c->d.N;
    const gmd_desc &d = c->d;
    const size_t ns = (size_t)std::max(0, d.nscalars);
    const XferSeg X(N, ns);
    unsigned what = 0;
    size_t lo = X.end, hi = 0;
    auto want = [&](unsigned bit, const void *dst, size_t at, size_t n) {
        if (!dst || n == 0) return;
        what |= bit;
        lo = std::min(lo, at);
        hi = std::max(hi, at + n);
    };
    want(XF_R, r, X.r, 3 * N);
    want(XF_V, v, X.v, 3 * N);
    want(XF_F, f, X.f, 3 * N);
    want(XF_S, scalars, X.s, N * ns);
    want(XF_T, ptype, X.t, N);
    want(XF_IM, r_im, X.im, 3 * N);
    const bool whole = c->xcap >= X.end;
    if (!c->fetched && what) {
        const bool direct = whole && N <= XFER_DIRECT && !c->permuted;
        hipLaunchKernelGGL(k_unpack, xfer_grid(c, N), dim3(256), 0, c->stream, (const DP *)c->d_P, c->buf0, what,
                           direct ? c->xhost : c->xdev);
        HIPCHECK(hipGetLastError());
        if (whole && !direct) {
            const size_t at = lo / 4 * 4;
            if (xfer_copy(c, c->xdev + at, c->xhost + at, hi - at, hipMemcpyDeviceToHost)) return -1;
        }
    }
    c->fetched = false;
    std::vector<HostSeg> segs;
    auto put = [&](void *dst, size_t at, size_t n) {
        if (dst && n) segs.push_back(HostSeg{dst, at, n});
    };
    put(r, X.r, 3 * N);
    put(v, X.v, 3 * N);
    put(f, X.f, 3 * N);
    put(ptype, X.t, N);
    put(r_im, X.im, 3 * N);
    std::vector<float> rows;   // columns without a device array stay as the caller has them
    if (scalars && !c->all_cols) rows.resize(N * ns);
    put(c->all_cols ? (void *)scalars : (void *)rows.data(), X.s, scalars ? N * ns : 0);
    if (whole) {
        HIPCHECK(hipStreamSynchronize(c->stream));
        host_move(c->xhost, 0, X.end, segs, false);
    } else if (what) {
        // by halves: the host empties one while the other is on its way
        auto start = [&](size_t at, int half) {
            const size_t n = std::min((size_t)XFER_CHUNK, hi - at);
            HIPCHECK(hipMemcpyAsync(c->xhost + (size_t)half * XFER_CHUNK, c->xdev + at, n * 4, hipMemcpyDeviceToHost,
                                    c->stream));
            HIPCHECK(hipEventRecord(c->xev[half], c->stream));
            return 0;
        };
        if (start(lo, 0)) return -1;
        int half = 0;
        for (size_t at = lo; at < hi; at += XFER_CHUNK, half ^= 1) {
            if (at + XFER_CHUNK < hi && start(at + XFER_CHUNK, half ^ 1)) return -1;
            HIPCHECK(hipEventSynchronize(c->xev[half]));
            host_move(c->xhost + (size_t)half * XFER_CHUNK, at, std::min(at + XFER_CHUNK, hi), segs, false);
        }
    }
    if (!rows.empty())
        for (int sid : {c->P.sid_u, c->P.sid_w, c->P.sid_lap, c->P.sid_k, c->P.sid_fsq, c->P.sid_m})
            if (sid >= 0)
                for (size_t i = 0; i < N; ++i) scalars[i * ns + sid] = rows[i * ns + sid];
    return 0;
}

static int ensure_flags(gmd_ctx *c, int steps) {
    if (c->rebuild_cap < steps + 2) {
        if (c->rebuild_flag) HIPCHECK(hipFree(c->rebuild_flag));
        c->rebuild_flag = nullptr;
        int cap = std::max(steps + 2, 1024);
        if (dalloc(&c->rebuild_flag, cap)) return -1;
        c->rebuild_cap = cap;
        c->P.rebuild_flag = (GMEM int *)c->rebuild_flag;
        HIPCHECK(hipMemcpy(c->d_P, &c->P, sizeof(DP), hipMemcpyHostToDevice));
        if (c->gexec) {
            hipGraphExecDestroy(c->gexec);
            c->gexec = nullptr;
        }
        if (c->graph) {
            hipGraphDestroy(c->graph);
            c->graph = nullptr;
        }
    }
    return 0;
}

// Renumber the particles by applying 'order' (new k = old order[k]) to every
// per-particle array; the positions move to the other ping-pong buffer.
static int apply_order(gmd_ctx *c, const int *order) {
    hipStream_t st = c->stream;
    const int N = c->d.N;
    const int grid = std::max(1, std::min((N + 255) / 256, c->cus * 8));
    hipLaunchKernelGGL(k_permute, dim3(grid), dim3(256), 0, st, (const DP *)c->d_P, c->buf0, order, c->tb);
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipMemcpyAsync(c->vel, c->tb.vel, (size_t)N * sizeof(float4), hipMemcpyDeviceToDevice, st));
    HIPCHECK(hipMemcpyAsync(c->frc, c->tb.frc, (size_t)N * sizeof(float4), hipMemcpyDeviceToDevice, st));
    HIPCHECK(hipMemcpyAsync(c->rref, c->tb.rref, (size_t)N * sizeof(float4), hipMemcpyDeviceToDevice, st));
    HIPCHECK(hipMemcpyAsync(c->obeta, c->tb.obeta, (size_t)N * sizeof(float4), hipMemcpyDeviceToDevice, st));
    HIPCHECK(hipMemcpyAsync(c->sc, c->tb.sc, (size_t)5 * N * sizeof(float), hipMemcpyDeviceToDevice, st));
    HIPCHECK(hipMemcpyAsync(c->rim, c->tb.rim, (size_t)3 * N * sizeof(int), hipMemcpyDeviceToDevice, st));
    HIPCHECK(hipMemcpyAsync(c->perm, c->tb.perm, (size_t)N * sizeof(int), hipMemcpyDeviceToDevice, st));
    c->buf0 ^= 1;
    c->need_rebuild = true;   // list indices refer to the old numbering
    return 0;
}

// cell order of the current positions
static int reorder(gmd_ctx *c) {
    hipStream_t st = c->stream;
    const int N = c->d.N, nc = c->nkeys;
    const int grid = std::max(1, std::min((N + 255) / 256, c->cus * 8));
    const int gridc = std::max(1, std::min((nc + 255) / 256, c->cus * 8));
    HIPCHECK(hipMemsetAsync(c->scnt, 0, (size_t)nc * sizeof(int), st));
    hipLaunchKernelGGL(k_sort_count, dim3(grid), dim3(256), 0, st, (const DP *)c->d_P, c->buf0, c->skey, c->scnt);
    const int chunks = (nc + SCAN_CHUNK - 1) / SCAN_CHUNK;
    hipLaunchKernelGGL(k_scan_sums, dim3(chunks), dim3(256), 0, st, (const int *)c->scnt, nc, c->ssum);
    hipLaunchKernelGGL(k_scan, dim3(chunks), dim3(256), 0, st, c->scnt, nc, (const int *)c->ssum);
    HIPCHECK(hipMemcpyAsync(c->scur, c->scnt, (size_t)nc * sizeof(int), hipMemcpyDeviceToDevice, st));
    hipLaunchKernelGGL(k_sort_scatter, dim3(grid), dim3(256), 0, st, N, (const int *)c->skey, c->scur, c->sorder);
    hipLaunchKernelGGL(k_sort_cells, dim3(gridc), dim3(256), 0, st, (const int *)c->scnt, nc, N, c->sorder);
    HIPCHECK(hipGetLastError());
    if (apply_order(c, c->sorder)) return -1;
    c->permuted = true;
    c->since_reorder = 0;
    ++c->renumberings;
    return 0;
}

// back to the caller's numbering (before host data arrive in that order)
static int unpermute(gmd_ctx *c) {
    if (!c->permuted) return 0;
    const int N = c->d.N;
    const int grid = std::max(1, std::min((N + 255) / 256, c->cus * 8));
    hipLaunchKernelGGL(k_perm_inverse, dim3(grid), dim3(256), 0, c->stream, (const DP *)c->d_P, c->sorder);
    HIPCHECK(hipGetLastError());
    if (apply_order(c, c->sorder)) return -1;
    HIPCHECK(hipStreamSynchronize(c->stream));
    c->permuted = false;
    // the next run with steps renumbers again instead of running in the
    // caller's order until reorder_every more steps have passed
    c->since_reorder = c->reorder_every;
    return 0;
}

// the permutation on the host (internal index -> caller's index), or empty
static int host_perm(gmd_ctx *c, std::vector<int> &perm) {
    perm.clear();
    if (!c->permuted) return 0;
    perm.resize(c->d.N);
    HIPCHECK(hipMemcpy(perm.data(), c->perm, (size_t)c->d.N * sizeof(int), hipMemcpyDeviceToHost));
    return 0;
}

// per-run set-up of one system on its stream: control block, rebuild flags,
// saver rows, the cell grid of the starting positions and the skin test
// (launch = false: the caller launches that for all its replicas)
static RunStart run_start(const gmd_ctx *c) { return RunStart{c->buf0, c->need_rebuild ? 1 : 0, c->lstep}; }

// blocks of the clears at the start of a run
static unsigned run_begin_blocks(const gmd_ctx *c, int steps) {
    const int cells = c->d.nblist_kind == GMD_NBLIST_LINKED_LISTS ? 3 * c->P.ncells : 0;
    const int rows = c->d.scalar_save_every > 0 ? c->d.scalar_saves_per_block * 6 : 0;
    return (unsigned)std::max(1, std::min((std::max(steps + 2, std::max(cells, rows)) + 255) / 256, c->cus * 8));
}

static int run_prepare(gmd_ctx *c, float t0, int steps, bool launch = true) {
    if (steps < 0) return fail("gmd_run: steps must be non-negative");
    if (ensure_flags(c, steps)) return -1;
    if (c->reorder_every > 0 && steps > 0 && c->since_reorder >= c->reorder_every)
        if (reorder(c)) return -1;
    c->pub_valid = false;
    c->fetched = false;
    if (!c->ptab_ready) {
        hipLaunchKernelGGL(k_pair_table, dim3(1), dim3(64), 0, c->stream, (const DP *)c->d_P);
        c->ptab_ready = true;
    }
    if (!launch) return 0;
    hipStream_t st = c->stream;
    const DP *dP = c->d_P;
    hipLaunchKernelGGL(k_run_begin, dim3(run_begin_blocks(c, steps)), dim3(256), 0, st, dP, steps, t0,
                       run_start(c));
    hipLaunchKernelGGL(k_run_setup, dim3(c->grid_aux), dim3(c->block), 0, st, dP);
    HIPCHECK(hipGetLastError());
    return 0;
}

// after the stream has drained: host-side state of the run and its errors
static int run_complete(gmd_ctx *c, int steps) {
    c->buf0 ^= (steps & 1);
    c->lstep += steps;
    c->since_reorder += steps;
    c->need_rebuild = false;
    const Ctrl &h = *c->pub;   // published by the run (k_run_publish), on the host since the stream drained
    c->pub_valid = true;
    if (c->P.npt)
        for (int k = 0; k < 3; ++k) c->cur_box[k] = h.npt[h.nsteps & 1][3 + k];
    if (h.cell_overflow > 0)
        return fail("linked lists: %d particles fell into one cell, more than the cell capacity %d "
                    "(use 'N squared' or a larger skin)", h.cell_overflow, c->P.ccap);
    if (h.npt_grid_bad)
        return fail("NPT_Atomic: the box shrank below %.0f%% of the lengths the linked-list cell grid was laid out "
                    "for; create a new Simulation from the current configuration or use 'N squared'",
                    100.0 * NPT_GRID_SHRINK);
    return 0;
}

static int run_impl(gmd_ctx *c, float t0, int steps) {
    if (run_prepare(c, t0, steps)) return -1;
    hipStream_t st = c->stream;
    const DP *dP = c->d_P;
    HIPCHECK(hipEventRecord(c->ev0, st));
    if (c->d.gridsync) {
        void *args[] = {(void *)&dP};
        HIPCHECK(hipLaunchCooperativeKernel((const void *)c->kern.pers, dim3(c->grid_pers), dim3(c->block), args,
                                            (unsigned)c->lds_pers, st));
    } else if (c->d.use_graph) {
        if (!c->gexec) {
            HIPCHECK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
            for (int k = 0; k < GRAPH_STEPS; ++k)
                hipLaunchKernelGGL(c->kern.step, dim3(c->grid_step), dim3(c->block), c->lds_step, st, dP, k);
            hipLaunchKernelGGL(k_advance, dim3(1), dim3(64), 0, st, c->ctrl, GRAPH_STEPS);
            HIPCHECK(hipStreamEndCapture(st, &c->graph));
            HIPCHECK(hipGraphInstantiate(&c->gexec, c->graph, nullptr, nullptr, 0));
        }
        // whole groups of GRAPH_STEPS steps from the graph, the rest as plain
        // launches (k counts from the step after the last group)
        const int groups = (steps + 1) / GRAPH_STEPS, rest = (steps + 1) % GRAPH_STEPS;
        for (int g = 0; g < groups; ++g) HIPCHECK(hipGraphLaunch(c->gexec, st));
        for (int k = 0; k < rest; ++k)
            hipLaunchKernelGGL(c->kern.step, dim3(c->grid_step), dim3(c->block), c->lds_step, st, dP, k);
        HIPCHECK(hipGetLastError());
    } else {
        for (int s = 0; s <= steps; ++s)
            hipLaunchKernelGGL(c->kern.step, dim3(c->grid_step), dim3(c->block), c->lds_step, st, dP, s);
        HIPCHECK(hipGetLastError());
    }
    HIPCHECK(hipEventRecord(c->ev1, st));
    hipLaunchKernelGGL(k_run_publish, dim3(1), dim3(256), 0, st, dP);
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipStreamSynchronize(st));
    HIPCHECK(hipEventElapsedTime(&c->last_ms, c->ev0, c->ev1));
    return run_complete(c, steps);
}

int gmd_run(gmd_ctx *c, float time_zero, int steps) {
    if (!c) return fail("gmd_run: null context");
    if (!c->own_stream) return fail("gmd_run: this context is a replica of a batch; use gmd_batch_run");
    if (c->d.integrator == GMD_INTEGRATOR_NONE && steps > 0)
        return fail("gmd_run: context has no integrator; only steps=0 (evaluation) is possible");
    return run_impl(c, time_zero, steps);
}

int gmd_evaluate(gmd_ctx *c) {
    if (!c) return fail("gmd_evaluate: null context");
    if (!c->own_stream) return fail("gmd_evaluate: this context is a replica of a batch");
    return run_impl(c, 0.0f, 0);
}

int gmd_profile_steps(gmd_ctx *c, float time_zero, int steps, float *step_ms, float *tail_ms) {
    if (!c || !step_ms || !tail_ms) return fail("gmd_profile_steps: null argument");
    if (!c->own_stream) return fail("gmd_profile_steps: this context is a replica of a batch");
    if (c->d.gridsync) return fail("gmd_profile_steps: the persistent driver runs every step in one launch");
    if (c->d.integrator == GMD_INTEGRATOR_NONE && steps > 0) return fail("gmd_profile_steps: no integrator");
    if (run_prepare(c, time_zero, steps)) return -1;
    hipStream_t st = c->stream;
    const DP *dP = c->d_P;
    const int n = steps + 1;
    std::vector<hipEvent_t> ev(2, nullptr);
    int rc = 0;
    for (auto &e : ev)
        if (hipEventCreate(&e) != hipSuccess) {
            rc = fail("gmd_profile_steps: hipEventCreate failed");
            break;
        }
    if (rc == 0) {
        // back-to-back launches between two events: the mean includes the
        // dispatch gap between consecutive kernels, nothing else
        hipEventRecord(ev[0], st);
        for (int s = 0; s < n; ++s)
            hipLaunchKernelGGL(c->kern.step, dim3(c->grid_step), dim3(c->block), c->lds_step, st, dP, s);
        hipEventRecord(ev[1], st);
        hipLaunchKernelGGL(k_run_publish, dim3(1), dim3(256), 0, st, dP);
        if (hipGetLastError() != hipSuccess || hipStreamSynchronize(st) != hipSuccess)
            rc = fail("gmd_profile_steps: launch failed");
    }
    if (rc == 0) {
        float x = 0.f;
        hipEventElapsedTime(&x, ev[0], ev[1]);
        *step_ms = x / n;
        *tail_ms = 0.0f;   // the tail of each step runs inside the next step kernel
    }
    for (auto &e : ev)
        if (e) hipEventDestroy(e);
    if (rc) return rc;
    return run_complete(c, steps);
}

int gmd_last_run_ms(gmd_ctx *c, float *ms) {
    if (!c || !ms) return fail("gmd_last_run_ms: null argument");
    *ms = c->last_ms;
    return 0;
}

// the control block: as the last run published it, or from the device
static int read_ctrl(gmd_ctx *c, Ctrl &h) {
    if (c->pub_valid) {
        h = *c->pub;
        return 0;
    }
    HIPCHECK(hipStreamSynchronize(c->stream));
    HIPCHECK(hipMemcpy(&h, c->ctrl, sizeof h, hipMemcpyDeviceToHost));
    return 0;
}

int gmd_read_nbflag(gmd_ctx *c, int nbflag[3]) {
    if (!c || !nbflag) return fail("gmd_read_nbflag: null argument");
    Ctrl h;
    if (read_ctrl(c, h)) return -1;
    for (int k = 0; k < 3; ++k) nbflag[k] = h.nbflag[k];
    return 0;
}

int gmd_read_nblist(gmd_ctx *c, int *out) {
    if (!c || !out) return fail("gmd_read_nblist: null argument");
    HIPCHECK(hipStreamSynchronize(c->stream));
    const int N = c->d.N, M = c->d.max_nbs, tp = c->d.tp, cap = c->P.max_nbs;
    std::vector<int> nbl(c->nbl_len), nbc(N);
    HIPCHECK(hipMemcpy(nbl.data(), c->nbl, nbl.size() * sizeof(int), hipMemcpyDeviceToHost));
    HIPCHECK(hipMemcpy(nbc.data(), c->nbc, (size_t)N * sizeof(int), hipMemcpyDeviceToHost));
    std::vector<int> perm;
    if (host_perm(c, perm)) return -1;
    auto at = [&](int i) { return perm.empty() ? i : perm[i]; };
    for (int i = 0; i < N; ++i) {
        int *row = out + (size_t)at(i) * (M + 1);
        const int n = std::min(nbc[i], cap);
        int w = 0;
        for (int k = 0; k < n; ++k) {
            const size_t m = (size_t)(k / tp), t = (size_t)(k % tp);
            const int raw = c->nb16 ? (int)((const unsigned short *)nbl.data())[2 * (((m / 2) * N + i) * tp + t) + (m & 1)]
                                    : nbl[(m * N + i) * tp + t];
            const int j = at(raw);
            if (c->d.utilize_niii) {
                // the reference's half list (nblist.py:112-116); an NIII
                // context keeps the caller's numbering
                const int two_dn = 2 * (j - at(i));
                if (!((two_dn > 0 && two_dn <= N) || (two_dn < -N))) continue;
            }
            if (w < M) row[w] = j;
            ++w;
        }
        for (int k = std::min(w, M); k < M; ++k) row[k] = 0;
        row[M] = c->d.utilize_niii ? w : nbc[i];
    }
    return 0;
}

int gmd_reorder_stats(gmd_ctx *c, int *permuted, long long *renumberings) {
    if (!c || !permuted || !renumberings) return fail("gmd_reorder_stats: null argument");
    *permuted = c->permuted ? 1 : 0;
    *renumberings = c->renumberings;
    return 0;
}

int gmd_set_reorder_interval(gmd_ctx *c, int steps) {
    if (!c) return fail("gmd_set_reorder_interval: null context");
    if (steps < 0) return fail("gmd_set_reorder_interval: steps must be non-negative");
    if (steps > 0 && !c->sorder)
        return fail("gmd_set_reorder_interval: renumbering needs linked lists, no exclusions, no bonds and UtilizeNIII off");
    c->reorder_every = steps;
    return 0;
}

int gmd_copy_probe(unsigned long long bytes, int reps, float *ms_per_copy) {
    if (!ms_per_copy) return fail("gmd_copy_probe: null argument");
    if (bytes == 0 || bytes % 16 || reps < 1) return fail("gmd_copy_probe: bytes must be a positive multiple of 16");
    float4 *src = nullptr, *dst = nullptr;
    hipStream_t st = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int rc = 0;
    if (hipMalloc(&src, bytes) != hipSuccess || hipMalloc(&dst, bytes) != hipSuccess) {
        rc = fail("gmd_copy_probe: out of device memory");
    } else if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess ||
               hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
        rc = fail("gmd_copy_probe: stream or event creation failed");
    } else {
        const size_t n = bytes / 16;
        int dev = 0, cus = 0;
        hipGetDevice(&dev);
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        const unsigned grid = (unsigned)std::max<size_t>(1, std::min<size_t>((n + 255) / 256, (size_t)cus * 16));
        bool ok = hipMemsetAsync(src, 0, bytes, st) == hipSuccess;
        hipLaunchKernelGGL(k_copy, dim3(grid), dim3(256), 0, st, (const float4 *)src, dst, n);
        ok = ok && hipEventRecord(e0, st) == hipSuccess;
        for (int r = 0; r < reps; ++r) hipLaunchKernelGGL(k_copy, dim3(grid), dim3(256), 0, st, (const float4 *)src, dst, n);
        ok = ok && hipGetLastError() == hipSuccess && hipEventRecord(e1, st) == hipSuccess &&
             hipEventSynchronize(e1) == hipSuccess;
        float ms = 0.f;
        if (!ok || hipEventElapsedTime(&ms, e0, e1) != hipSuccess) rc = fail("gmd_copy_probe: launch failed");
        else *ms_per_copy = ms / reps;
    }
    if (e0) hipEventDestroy(e0);
    if (e1) hipEventDestroy(e1);
    if (st) hipStreamDestroy(st);
    if (src) hipFree(src);
    if (dst) hipFree(dst);
    return rc;
}

int gmd_fma_probe(int iters, float *tflops) {
    if (!tflops || iters < 1) return fail("gmd_fma_probe: bad argument");
    int dev = 0, cus = 0;
    HIPCHECK(hipGetDevice(&dev));
    HIPCHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const int grid = cus * 8, block = 256;
    float *out = nullptr;
    hipStream_t st = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int rc = 0;
    if (hipMalloc(&out, (size_t)grid * block * sizeof(float)) != hipSuccess) {
        rc = fail("gmd_fma_probe: out of device memory");
    } else if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess ||
               hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
        rc = fail("gmd_fma_probe: stream or event creation failed");
    } else {
        hipLaunchKernelGGL(k_fma, dim3(grid), dim3(block), 0, st, iters, out);   // warm-up
        bool ok = hipEventRecord(e0, st) == hipSuccess;
        hipLaunchKernelGGL(k_fma, dim3(grid), dim3(block), 0, st, iters, out);
        ok = ok && hipGetLastError() == hipSuccess && hipEventRecord(e1, st) == hipSuccess &&
             hipEventSynchronize(e1) == hipSuccess;
        float ms = 0.f;
        if (!ok || hipEventElapsedTime(&ms, e0, e1) != hipSuccess) rc = fail("gmd_fma_probe: launch failed");
        else *tflops = (float)(16.0 * iters * (double)grid * block / (ms * 1e-3) / 1e12);
    }
    if (e0) hipEventDestroy(e0);
    if (e1) hipEventDestroy(e1);
    if (st) hipStreamDestroy(st);
    if (out) hipFree(out);
    return rc;
}

int gmd_force_rebuild(gmd_ctx *c) {
    if (!c) return fail("gmd_force_rebuild: null context");
    c->need_rebuild = true;
    return 0;
}

int gmd_get_thermostat(gmd_ctx *c, float state[2]) {
    if (!c || !state) return fail("gmd_get_thermostat: null argument");
    Ctrl h;
    if (read_ctrl(c, h)) return -1;
    state[0] = h.xi;
    state[1] = h.ksum;
    return 0;
}

int gmd_set_thermostat(gmd_ctx *c, const float state[2]) {
    if (!c || !state) return fail("gmd_set_thermostat: null argument");
    HIPCHECK(hipStreamSynchronize(c->stream));
    HIPCHECK(hipMemcpy(&c->ctrl->xi, state, 2 * sizeof(float), hipMemcpyHostToDevice));
    c->pub_valid = false;
    return 0;
}

int gmd_get_npt_state(gmd_ctx *c, float state[6]) {
    if (!c || !state) return fail("gmd_get_npt_state: null argument");
    if (!c->P.npt) return fail("gmd_get_npt_state: the context does not run NPT_Atomic");
    Ctrl h;
    if (read_ctrl(c, h)) return -1;
    for (int k = 0; k < 6; ++k) state[k] = h.npt[h.nsteps & 1][k];
    return 0;
}

int gmd_set_npt_state(gmd_ctx *c, const float state[6]) {
    if (!c || !state) return fail("gmd_set_npt_state: null argument");
    if (!c->P.npt) return fail("gmd_set_npt_state: the context does not run NPT_Atomic");
    for (int k = 0; k < 3; ++k)
        if (!(state[3 + k] > 0.f)) return fail("gmd_set_npt_state: box lengths must be positive");
    if (!(state[2] > 0.f)) return fail("gmd_set_npt_state: the volume must be positive");
    HIPCHECK(hipStreamSynchronize(c->stream));
    float both[2][6];
    for (int b = 0; b < 2; ++b)
        for (int k = 0; k < 6; ++k) both[b][k] = state[k];
    HIPCHECK(hipMemcpy(&c->ctrl->npt[0][0], both, sizeof both, hipMemcpyHostToDevice));
    c->pub_valid = false;
    for (int k = 0; k < 3; ++k) c->cur_box[k] = state[3 + k];
    return 0;
}

int gmd_read_scalar_output(gmd_ctx *c, float *out) {
    if (!c || !out) return fail("gmd_read_scalar_output: null argument");
    if (c->d.scalar_save_every <= 0) return fail("gmd_read_scalar_output: no scalar saver configured");
    const size_t bytes = (size_t)c->d.scalar_saves_per_block * 6 * sizeof(float);
    if (c->pub_valid)
        memcpy(out, c->pub + 1, bytes);   // published after the control block
    else
        HIPCHECK(hipMemcpy(out, c->saver_out, bytes, hipMemcpyDeviceToHost));
    return 0;
}

int gmd_read_conf_output(gmd_ctx *c, float *out) {
    if (!c || !out) return fail("gmd_read_conf_output: null argument");
    if (c->d.conf_saves_per_block <= 0) return fail("gmd_read_conf_output: no configuration saver configured");
    HIPCHECK(hipStreamSynchronize(c->stream));
    const size_t n = (size_t)c->d.conf_saves_per_block * 6 * c->d.N;
    HIPCHECK(hipMemcpy(out, c->conf_out, n * sizeof(float), hipMemcpyDeviceToHost));
    // cleared for the next block (configuration_saver.py:88, the zero kernel)
    hipLaunchKernelGGL(k_fill_f32, dim3((unsigned)std::min<size_t>((n + 255) / 256, (size_t)c->cus * 8)), dim3(256), 0,
                       c->stream, c->conf_out, n);
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipStreamSynchronize(c->stream));
    return 0;
}

// ---------------------------------------------------------------------------
// RDF
// ---------------------------------------------------------------------------
static int rdf_bin_host(float x, double half, double bw, int bins) {
    // calculator_radial_distribution.py:101-104 with numba's float64 promotion
    if (!((double)x < half * half)) return bins;
    float dd = std::sqrt(x);
    if (!((double)dd < half)) return bins;
    int b = (int)std::floor((double)dd / bw);
    return std::min(b, bins);
}

// thr[0 .. bins+1]: thr[k] = the smallest float32 d^2 whose bin is >= k
// (thr[bins]: the first excluded), thr[bins + 1] = infinity
static void rdf_thresholds(const float box[3], int bins, float *thr) {
    float mn = std::min(box[0], std::min(box[1], box[2]));
    double half = (double)mn / 2.0;
    double bw = half / bins;
    thr[0] = 0.f;
    thr[bins + 1] = INFINITY;
    for (int k = 1; k <= bins; ++k) {
        // smallest non-negative float x with bin(x) >= k (bin is monotone in x)
        uint32_t lo = 0, hi = 0x7f800000u;  // +inf
        while (lo < hi) {
            uint32_t mid = lo + (hi - lo) / 2;
            float x;
            memcpy(&x, &mid, 4);
            if (rdf_bin_host(x, half, bw, bins) >= k)
                hi = mid;
            else
                lo = mid + 1;
        }
        float x;
        memcpy(&x, &lo, 4);
        thr[k] = x;
    }
}

static void rdf_thresholds(const float box[3], int bins, std::vector<float> &thr) {
    thr.assign(bins + 2, 0.f);
    rdf_thresholds(box, bins, thr.data());
}

static size_t rdf_hist_size(int nt, int bins) { return (size_t)nt * nt * bins; }

static size_t rdf_lds_bytes(int nt, int bins) {
    const size_t nh = rdf_hist_size(nt, bins);
    return ((nh * 4 + 15) & ~(size_t)15) + (((size_t)(bins + 1) * 4 + 15) & ~(size_t)15);
}

// Mean share of the box that 64 consecutive positions and 'pad' around them
// span, of n runs spread over the numbering
static double chunk_share(const float *r, int N, const float box[3], float pad, int n) {
    const int chunks = (N + 63) / 64;
    n = std::min(n, chunks);
    double sum = 0.0;
    for (int k = 0; k < n; ++k) {
        const int b = (int)((long long)k * chunks / n) * 64, e = std::min(N, b + 64);
        float lo[3], hi[3];
        for (int c = 0; c < 3; ++c) lo[c] = hi[c] = r[3 * (size_t)b + c];
        for (int i = b + 1; i < e; ++i)   // six independent chains
            for (int c = 0; c < 3; ++c) {
                lo[c] = std::min(lo[c], r[3 * (size_t)i + c]);
                hi[c] = std::max(hi[c], r[3 * (size_t)i + c]);
            }
        double share = 1.0;
        for (int c = 0; c < 3; ++c) share *= std::min(1.0, (double)(hi[c] - lo[c] + pad) / box[c]);
        sum += share;
    }
    return sum / n;
}

// Whether the numbering keeps particles together without a sort, asked where
// rdf_cells does (in lattice order a run of 64 spans some hundredths of the
// box, in no order 0.9 of it)
static bool rdf_in_order(const float *r, int N, const float box[3]) {
    return N >= 8192 && N < 65536 && chunk_share(r, N, box, 0.f, 8) < 0.25;
}

// Sorting cells per dimension: some 16 particles a cell; 1 (none) where the
// sort's three launches (20 us with their gaps) are what it saves or more.
// In no order, without and with the sort: N = 8000 106 and 109 us, 12000 143
// and 139, 16000 191 and 180, 30000 453 and 383; in lattice order 8000 101 and
// 111, 16000 168 and 182, 30000 374 and 388, 131072 4630 and 4590.
static int rdf_cells(int N, bool in_order) {
    if (N < 8192 || (in_order && N < 65536)) return 1;
    return N < 32768 ? 8 : N < 262144 ? 16 : RDF_MAX_CELL;
}

// The launches of one histogram on a stream: sort, boxes, counts, sum over
// blocks.  S.pos (or S.r) / S.ptype: the input; out and the cell counts are
// zero; grid: blocks of k_rdf, at most what R.part holds.
static int rdf_kernels(RdfP R, RdfSort S, const float box[3], int grid, bool in_order, float4 *gbox, float4 *cbox,
                       unsigned long long *out, hipStream_t st) {
    const int N = R.N;
    R.L0 = box[0];
    R.L1 = box[1];
    R.L2 = box[2];
    R.rL0 = S.rL0 = 1.0f / box[0];
    R.rL1 = S.rL1 = 1.0f / box[1];
    R.rL2 = S.rL2 = 1.0f / box[2];
    const float mn = std::min(box[0], std::min(box[1], box[2]));
    const double bw = ((double)mn / 2.0) / R.bins;
    // relative errors of the estimate against the exact rule: square root
    // 2^-23 here and 2^-24 there, product and constant 2^-24 each, 0.625 2^-21
    // in all; so scaled by 1 - 0.75 2^-21 it is never above, and below by less
    // than 1.375 2^-21 of at most 'bins'
    R.inv_bw = (float)((1.0 / bw) * (1.0 - 0.75 / 2097152.0));
    R.edge = (float)(1.0 - 1.5 / 2097152.0 * R.bins);
    R.nchunks = (N + RDF_CHUNK - 1) / RDF_CHUNK;
    R.nrow = (R.nchunks + 1) / 2;
    const long long row = (long long)(R.nchunks + 1) * (RDF_CHUNK / RDF_GROUP);
    // as many groups a unit as leave a wavefront some eight units
    R.unit = (int)std::max(1LL, std::min(64LL, R.nrow * row / (8LL * 4 * grid)));
    R.nper = (int)((row + R.unit - 1) / R.unit);
    R.cbox = (const GMEM float4 *)cbox;
    R.gbox = (const GMEM float4 *)gbox;
    R.pos = (cpos_t)S.out;
    S.N = N;
    S.npad = R.nchunks * RDF_CHUNK;
    S.nt_bytes = R.bins * 4;
    S.ncell = rdf_cells(N, in_order);
    const unsigned nb = (unsigned)((N + 255) / 256);
    if (S.ncell > 1) {
        hipLaunchKernelGGL(k_rdf_count, dim3(nb), dim3(256), 0, st, S);
        hipLaunchKernelGGL(k_rdf_starts, dim3(1), dim3(1024), 0, st, S.count, S.ncell * S.ncell * S.ncell);
        hipLaunchKernelGGL(k_rdf_place, dim3((unsigned)((S.npad + 255) / 256)), dim3(256), 0, st, S);
    }
    hipLaunchKernelGGL(k_rdf_boxes, dim3((unsigned)((R.nchunks + 3) / 4)), dim3(256), 0, st, S, S.ncell > 1 ? 0 : 1,
                       box[0], box[1], box[2], gbox, cbox);
    hipLaunchKernelGGL(k_rdf, dim3(grid), dim3(256), rdf_lds_bytes(R.nt, R.bins), st, R);
    HIPCHECK(hipGetLastError());
    const int nh = (int)rdf_hist_size(R.nt, R.bins), per = 16;
    hipLaunchKernelGGL(k_rdf_reduce, dim3((unsigned)((nh + 255) / 256), (unsigned)((grid + per - 1) / per)),
                       dim3(256), 0, st, (const unsigned *)R.part, grid, nh, per, out);
    HIPCHECK(hipGetLastError());
    return 0;
}

int gmd_rdf_create(int N, int ntypes, int bins, gmd_rdf **out) {
    if (!out) return fail("gmd_rdf_create: null output");
    *out = nullptr;
    if (N < 1 || ntypes < 1 || ntypes > MAX_TYPES || bins < 1) return fail("gmd_rdf_create: bad sizes");
    gmd_rdf *r = new gmd_rdf();
    r->N = N;
    r->nt = ntypes;
    r->bins = bins;
    r->nchunks = (N + RDF_CHUNK - 1) / RDF_CHUNK;
    const size_t nh = rdf_hist_size(ntypes, bins);
    if (rdf_lds_bytes(ntypes, bins) > 64 * 1024 - RDF_LDS_SPARE) {
        delete r;
        return fail("gmd_rdf_create: %d x %d type pairs x %d bins do not fit the LDS histogram", ntypes, ntypes,
                    bins);
    }
    int dev = 0, cus = 0;
    HIPCHECK(hipGetDevice(&dev));
    HIPCHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    // blocks of four wavefronts that have a group each
    const long long npairs = ((long long)r->nchunks * (r->nchunks + 1) / 2 * (RDF_CHUNK / RDF_GROUP) + 3) / 4;
    // a block's 32-bit counters see at most 2^31 pairs
    const long long need = (long long)(((double)N * (double)N / 2.0) / 2147483648.0) + 1;
    r->grid = (int)std::max(1LL, std::min(npairs, std::max((long long)cus * 4, need)));
    // beside the step kernels, 2 blocks per CU take fewer of their slots and
    // still finish within a block of steps
    r->grid_bg = (int)std::max(1LL, std::min(npairs, std::max((long long)cus * 2, need)));
    const size_t ng = (size_t)r->nchunks * (RDF_CHUNK / RDF_GROUP), cells = rdf_cells(N, false);
    if (hipMalloc(&r->pos, (size_t)N * sizeof(float4)) != hipSuccess ||
        hipMalloc(&r->sorted, (size_t)r->nchunks * RDF_CHUNK * sizeof(float4)) != hipSuccess ||
        hipMalloc(&r->cbox, (size_t)4 * r->nchunks * sizeof(float4)) != hipSuccess ||
        hipMalloc(&r->gbox, 4 * ng * sizeof(float4)) != hipSuccess ||
        hipMalloc(&r->key, (size_t)N * sizeof(int2)) != hipSuccess ||
        hipMalloc(&r->ptype, (size_t)N * sizeof(int)) != hipSuccess ||
        hipMalloc(&r->d_thr, (size_t)(bins + 1) * sizeof(float)) != hipSuccess ||
        hipMalloc(&r->part, (size_t)r->grid * nh * sizeof(unsigned)) != hipSuccess ||
        hipMalloc(&r->d_out, nh * sizeof(unsigned long long) + cells * cells * cells * sizeof(int)) != hipSuccess) {
        gmd_rdf_destroy(r);
        return fail("gmd_rdf_create: out of device memory");
    }
    if (hipStreamCreateWithFlags(&r->stream, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&r->snap, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&r->done, hipEventDisableTiming) != hipSuccess) {
        gmd_rdf_destroy(r);
        return fail("gmd_rdf_create: stream or event creation failed");
    }
    if (hipHostMalloc((void **)&r->h_out, nh * sizeof(unsigned long long), hipHostMallocDefault) != hipSuccess) {
        r->h_out = nullptr;
        gmd_rdf_destroy(r);
        return fail("gmd_rdf_create: out of pinned host memory");
    }
    *out = r;
    return 0;
}

int gmd_rdf_destroy(gmd_rdf *r) {
    if (!r) return 0;
    void *ptrs[] = {r->pos, r->sorted, r->cbox, r->gbox, r->key, r->ptype, r->d_thr, r->part, r->d_out};
    for (void *p : ptrs)
        if (p) hipFree(p);
    if (r->pending && r->done) hipEventSynchronize(r->done);
    if (r->stream) hipStreamDestroy(r->stream);
    if (r->snap) hipEventDestroy(r->snap);
    if (r->done) hipEventDestroy(r->done);
    if (r->h_out) hipHostFree(r->h_out);
    delete r;
    return 0;
}

// Enqueue one histogram on the calculator's stream (pos: positions with types,
// or null: the host's in r->pos; d_ptype: their types, with pos instead of its
// own; in_order: they need no sort), ending in an asynchronous copy of the
// counts to pinned host memory.
static int rdf_launch(gmd_rdf *r, const float4 *pos, const int *d_ptype, const float box[3], int grid, bool in_order) {
    if (box[0] != r->box[0] || box[1] != r->box[1] || box[2] != r->box[2] || r->thr.empty()) {
        rdf_thresholds(box, r->bins, r->thr);
        HIPCHECK(hipMemcpy(r->d_thr, r->thr.data(), (size_t)(r->bins + 1) * sizeof(float), hipMemcpyHostToDevice));
        memcpy(r->box, box, sizeof r->box);
    }
    const size_t nh = rdf_hist_size(r->nt, r->bins), cells = rdf_cells(r->N, false);
    RdfP R = {};
    R.N = r->N;
    R.nt = r->nt;
    R.bins = r->bins;
    R.thr = (const GMEM float *)r->d_thr;
    R.part = (GMEM unsigned *)r->part;
    R.skip2 = r->thr[r->bins];
    RdfSort S = {};
    S.pos = pos;
    S.r = (const float *)r->pos;
    S.ptype = d_ptype;
    S.count = (int *)(r->d_out + nh);
    S.key = r->key;
    S.out = r->sorted;
    HIPCHECK(hipMemsetAsync(r->d_out, 0, nh * sizeof(unsigned long long) + cells * cells * cells * sizeof(int),
                            r->stream));
    if (rdf_kernels(R, S, box, grid, in_order, r->gbox, r->cbox, r->d_out, r->stream)) return -1;
    HIPCHECK(hipMemcpyAsync(r->h_out, r->d_out, nh * sizeof(unsigned long long), hipMemcpyDeviceToHost, r->stream));
    HIPCHECK(hipEventRecord(r->done, r->stream));
    r->pending = true;
    return 0;
}

// Wait for the launched histogram and fold it into ordered-pair counts.
static int rdf_collect(gmd_rdf *r, unsigned long long *counts) {
    if (!r->pending) return fail("gmd_rdf_collect: no update is pending");
    HIPCHECK(hipEventSynchronize(r->done));
    r->pending = false;
    const unsigned long long *h = r->h_out;
    // unordered pair counts in ordered-type slots -> ordered pair counts
    const int nt = r->nt, bins = r->bins;
    for (int a = 0; a < nt; ++a)
        for (int b = 0; b < nt; ++b)
            for (int k = 0; k < bins; ++k) {
                const unsigned long long ab = h[((size_t)a * nt + b) * bins + k];
                const unsigned long long ba = h[((size_t)b * nt + a) * bins + k];
                counts[((size_t)a * nt + b) * bins + k] = (a == b) ? 2 * ab : ab + ba;
            }
    return 0;
}

static int rdf_launch_ctx(gmd_rdf *r, gmd_ctx *c, const int *ptype, int grid) {
    if (!r || !c) return fail("gmd_rdf_launch_ctx: null argument");
    if (c->d.N != r->N) return fail("gmd_rdf_launch_ctx: N mismatch (%d vs %d)", c->d.N, r->N);
    if (r->pending) return fail("gmd_rdf_launch_ctx: the previous update is not collected");
    const int *dp = nullptr;
    if (ptype) {
        for (int i = 0; i < r->N; ++i)
            if (ptype[i] < 0 || ptype[i] >= r->nt) return fail("gmd_rdf_launch_ctx: type out of range");
        std::vector<int> perm, pt(ptype, ptype + r->N);
        if (host_perm(c, perm)) return -1;
        if (!perm.empty())
            for (int i = 0; i < r->N; ++i) pt[i] = ptype[perm[i]];   // types in the context's numbering
        HIPCHECK(hipMemcpy(r->ptype, pt.data(), (size_t)r->N * sizeof(int), hipMemcpyHostToDevice));
        dp = r->ptype;
    } else if (c->d.ntypes > r->nt) {
        return fail("gmd_rdf_launch_ctx: context has %d types, calculator %d", c->d.ntypes, r->nt);
    }
    // snapshot of the current positions, ordered after the context's work so
    // far; the context's later steps may overwrite its buffers meanwhile
    HIPCHECK(hipMemcpyAsync(r->pos, c->buf0 ? c->pos1 : c->pos0, (size_t)r->N * sizeof(float4),
                            hipMemcpyDeviceToDevice, c->stream));
    HIPCHECK(hipEventRecord(r->snap, c->stream));
    HIPCHECK(hipStreamWaitEvent(r->stream, r->snap, 0));
    return rdf_launch(r, r->pos, dp, c->cur_box, grid, c->permuted);   // (renumbered: in cell order)
}

int gmd_rdf_launch_ctx(gmd_rdf *r, gmd_ctx *c, const int *ptype) {
    if (!r) return fail("gmd_rdf_launch_ctx: null argument");
    return rdf_launch_ctx(r, c, ptype, r->grid_bg);
}

int gmd_rdf_collect(gmd_rdf *r, unsigned long long *counts) {
    if (!r || !counts) return fail("gmd_rdf_collect: null argument");
    return rdf_collect(r, counts);
}

int gmd_rdf_compute_ctx(gmd_rdf *r, gmd_ctx *c, const int *ptype, unsigned long long *counts) {
    if (!r || !c || !counts) return fail("gmd_rdf_compute_ctx: null argument");
    if (rdf_launch_ctx(r, c, ptype, r->grid)) return -1;
    return rdf_collect(r, counts);
}

int gmd_rdf_compute_host(gmd_rdf *r, const float *pos, const int *ptype, const float box[3],
                         unsigned long long *counts) {
    if (!r || !pos || !ptype || !box || !counts) return fail("gmd_rdf_compute_host: null argument");
    for (int i = 0; i < r->N; ++i)
        if (ptype[i] < 0 || ptype[i] >= r->nt) return fail("gmd_rdf_compute_host: type out of range");
    if (r->pending) return fail("gmd_rdf_compute_host: a launched update is not collected");
    const bool in_order = rdf_in_order(pos, r->N, box);
    if (r->N <= RDF_ONE_COPY) {
        const size_t N = r->N;
        r->h_in.resize(4 * N);
        memcpy(r->h_in.data(), pos, 3 * N * sizeof(float));
        memcpy(r->h_in.data() + 3 * N, ptype, N * sizeof(int));
        HIPCHECK(hipMemcpy(r->pos, r->h_in.data(), 4 * N * sizeof(int), hipMemcpyHostToDevice));
        if (rdf_launch(r, nullptr, (const int *)r->pos + 3 * N, box, r->grid, in_order)) return -1;
        return rdf_collect(r, counts);
    }
    HIPCHECK(hipMemcpy(r->pos, pos, (size_t)r->N * 3 * sizeof(float), hipMemcpyHostToDevice));
    HIPCHECK(hipMemcpy(r->ptype, ptype, (size_t)r->N * sizeof(int), hipMemcpyHostToDevice));
    if (rdf_launch(r, nullptr, r->ptype, box, r->grid, in_order)) return -1;
    return rdf_collect(r, counts);
}


// Device address of 'scratch' on each device, looked up once per device with
// that device current.
static std::mutex g_noalloc_mu;
static unsigned char *g_noalloc_ptr[64] = {nullptr};

static int noalloc_scratch(unsigned char **out) {
    int dev = 0;
    HIPCHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) return fail("gmd_rdf_compute_host_noalloc: device %d out of range", dev);
    std::lock_guard<std::mutex> lock(g_noalloc_mu);
    if (!g_noalloc_ptr[dev]) {
        void *ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr)
            return fail("gmd_rdf_compute_host_noalloc: hipGetSymbolAddress(scratch) failed on device %d: %s", dev,
                        hipGetErrorString(e));
        g_noalloc_ptr[dev] = (unsigned char *)ptr;
    }
    *out = g_noalloc_ptr[dev];
    return 0;
}

int gmd_rdf_compute_host_noalloc(int N, int ntypes, int bins, const float *pos, const int *ptype, const float box[3],
                                 unsigned long long *counts) {
    if (!pos || !ptype || !box || !counts) return fail("gmd_rdf_compute_host_noalloc: null argument");
    if (N < 1 || ntypes < 1 || ntypes > MAX_TYPES || bins < 1)
        return fail("gmd_rdf_compute_host_noalloc: bad sizes (N %d, ntypes %d, bins %d)", N, ntypes, bins);
    if (N > NOALLOC_RDF_MAX_N)
        return fail("gmd_rdf_compute_host_noalloc: N = %d exceeds the maximum %d of the static buffer", N,
                    NOALLOC_RDF_MAX_N);
    const size_t nh = rdf_hist_size(ntypes, bins);
    if (nh > NOALLOC_RDF_MAX_HIST)
        return fail("gmd_rdf_compute_host_noalloc: %d x %d type pairs x %d bins = %zu exceeds the maximum %d of the "
                    "static buffer", ntypes, ntypes, bins, nh, NOALLOC_RDF_MAX_HIST);
    for (int k = 0; k < 3; ++k)
        if (!(box[k] > 0.f)) return fail("gmd_rdf_compute_host_noalloc: box lengths must be positive");
    for (int i = 0; i < N; ++i)
        if (ptype[i] < 0 || ptype[i] >= ntypes) return fail("gmd_rdf_compute_host_noalloc: type out of range");
    unsigned char *base = nullptr;
    if (noalloc_scratch(&base)) return -1;
    float *d_r = (float *)(base + NOALLOC_OFF_R);
    int *d_t = (int *)(base + NOALLOC_OFF_T);
    float4 *d_pos = (float4 *)(base + NOALLOC_OFF_POS);
    float *d_thr = (float *)(base + NOALLOC_OFF_THR);
    unsigned *d_part = (unsigned *)(base + NOALLOC_OFF_PART);
    unsigned long long *d_out = (unsigned long long *)(base + NOALLOC_OFF_OUT);
    // host-side staging on the stack (no heap): thresholds and raw counts
    float thr[NOALLOC_RDF_MAX_HIST + 2];
    unsigned long long raw[NOALLOC_RDF_MAX_HIST];
    rdf_thresholds(box, bins, thr);
    const hipStream_t st = 0;   // the null stream: no stream is created
    HIPCHECK(hipMemcpy(d_r, pos, (size_t)N * 3 * sizeof(float), hipMemcpyHostToDevice));
    HIPCHECK(hipMemcpy(d_t, ptype, (size_t)N * sizeof(int), hipMemcpyHostToDevice));
    HIPCHECK(hipMemcpy(d_thr, thr, (size_t)(bins + 1) * sizeof(float), hipMemcpyHostToDevice));
    RdfP R = {};
    R.N = N;
    R.nt = ntypes;
    R.bins = bins;
    R.thr = (const GMEM float *)d_thr;
    R.part = (GMEM unsigned *)d_part;
    R.skip2 = thr[bins];
    RdfSort S = {};
    S.r = d_r;
    S.ptype = d_t;
    S.count = (int *)(base + NOALLOC_OFF_CELL);
    S.key = (int2 *)(base + NOALLOC_OFF_KEY);
    S.out = d_pos;
    // at most NOALLOC_RDF_MAX_N^2 / 2 = 2^31 pairs in total, so even a single
    // block's 32-bit counters cannot overflow
    const long long nc = (N + RDF_CHUNK - 1) / RDF_CHUNK;
    const int grid = (int)std::min(nc * (nc + 1) / 2, (long long)NOALLOC_RDF_GRID);
    hipLaunchKernelGGL(k_fill_u64, dim3((unsigned)((nh + 255) / 256)), dim3(256), 0, st, d_out, (int)nh);
    const int cells = rdf_cells(N, false) * rdf_cells(N, false) * rdf_cells(N, false);
    hipLaunchKernelGGL(k_fill_u64, dim3((unsigned)(((cells + 1) / 2 + 255) / 256)), dim3(256), 0, st,
                       (unsigned long long *)S.count, (cells + 1) / 2);
    if (rdf_kernels(R, S, box, grid, rdf_in_order(pos, N, box), (float4 *)(base + NOALLOC_OFF_GBOX), (float4 *)(base + NOALLOC_OFF_CBOX), d_out,
                    st))
        return -1;
    HIPCHECK(hipMemcpy(raw, d_out, nh * sizeof(unsigned long long), hipMemcpyDeviceToHost));
    // unordered pair counts in ordered-type slots -> ordered pair counts
    for (int a = 0; a < ntypes; ++a)
        for (int b = 0; b < ntypes; ++b)
            for (int k = 0; k < bins; ++k) {
                const unsigned long long ab = raw[((size_t)a * ntypes + b) * bins + k];
                const unsigned long long ba = raw[((size_t)b * ntypes + a) * bins + k];
                counts[((size_t)a * ntypes + b) * bins + k] = (a == b) ? 2 * ab : ab + ba;
            }
    return 0;
}

// ============================================================================
// Batches of independent replicas
// ============================================================================
struct gmd_batch {
    std::vector<gmd_ctx *> reps;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    int driver = GMD_BATCH_PERSISTENT, integrator = 0, block = 256, grid = 0, cus = 0;
    size_t lds = 0;
    Kernels kern = {nullptr, nullptr, nullptr, nullptr};
    std::vector<BatchBlk> h_blk;
    RunStart *h_start = nullptr;   // pinned: what each replica's run starts from (read by the kernels)
    BatchBlk *d_blk = nullptr;
    DP *d_Ps = nullptr;            // the replicas' DP, one after another (each context's d_P points here)
    float *d_kcell = nullptr;      // the replicas' DP::kcell
    int gk = 1;                    // blocks a replica of k_batch_ksum
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
    float last_ms = 0.f;
};

static int batch_free(gmd_batch *b) {
    if (!b) return 0;
    if (b->stream) hipStreamSynchronize(b->stream);
    if (b->gexec) hipGraphExecDestroy(b->gexec);
    if (b->graph) hipGraphDestroy(b->graph);
    for (gmd_ctx *c : b->reps) ctx_free(c);
    if (b->h_start) hipHostFree(b->h_start);
    if (b->d_blk) hipFree(b->d_blk);
    if (b->d_Ps) hipFree(b->d_Ps);
    if (b->d_kcell) hipFree(b->d_kcell);
    if (b->ev0) hipEventDestroy(b->ev0);
    if (b->ev1) hipEventDestroy(b->ev1);
    if (b->stream) hipStreamDestroy(b->stream);
    delete b;
    return 0;
}

// Grid layout of a batch.  Consecutive workgroups of a launch go to the
// device's 8 XCDs in turn, so grid slot k*8 + x runs on XCD x.  The blocks
// are packed into 8 bins of T = ceil(total/8) slots, largest replica first,
// each into the fullest bin that still holds it whole (its positions and
// lists then live in one XCD's L2); a replica that fits no bin whole is
// spread over the emptiest bins.  At most 7 slots stay idle (rep = -1).
// Within a bin the blocks past a replica's list steps (nlist) come first: they
// work on rebuild steps only, the longest a block has, and start with the
// launch.
static void batch_layout(const std::vector<int> &nb, const std::vector<int> &nlist, std::vector<BatchBlk> &out) {
    const int NX = 8;
    long long total = 0;
    for (int n : nb) total += n;
    const long long T = (total + NX - 1) / NX;
    std::vector<int> order(nb.size());
    for (size_t r = 0; r < nb.size(); ++r) order[r] = (int)r;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b2) { return nb[a] > nb[b2]; });
    std::vector<std::vector<BatchBlk>> bins(NX);
    for (int r : order) {
        int best = -1;
        for (int x = 0; x < NX; ++x) {
            const long long room = T - (long long)bins[x].size();
            if (room >= nb[r] && (best < 0 || room < T - (long long)bins[best].size())) best = x;
        }
        if (best >= 0) {
            for (int k = 0; k < nb[r]; ++k) bins[best].push_back(BatchBlk{r, k, nb[r], 0});
            continue;
        }
        int k = 0;
        while (k < nb[r]) {
            int x = 0;
            for (int y = 1; y < NX; ++y)
                if (bins[y].size() < bins[x].size()) x = y;
            while (k < nb[r] && (long long)bins[x].size() < T) bins[x].push_back(BatchBlk{r, k++, nb[r], 0});
        }
    }
    for (std::vector<BatchBlk> &bin : bins)
        std::stable_partition(bin.begin(), bin.end(), [&](const BatchBlk &a) { return a.bid >= nlist[a.rep]; });
    out.assign((size_t)T * NX, BatchBlk{-1, 0, 0, 0});
    for (int x = 0; x < NX; ++x)
        for (size_t k = 0; k < bins[x].size(); ++k) out[k * NX + x] = bins[x][k];
}

// Blocks of a replica's split rebuild steps: a wavefront for every cell (or
// NSQ_PP particles of an N-squared list) where the batch leaves the device that
// room, else for every two.  Before and after the split: 64 KA replicas of 1000
// to 8000 particles, tp = 2 (8 to 63 blocks a list step), 20.8 -> 18.0 ms for
// 64 steps; a batch of few replicas 8.9 -> 4.3 ms.  (The steps alone, with a
// wavefront for every cell of the 64 12.9 ms, for two 12.6, for three 13.0.)
static int rebuild_blocks(const gmd_ctx *c, int nrep) {
    const int wpb = c->block / 64;
    const int units = c->d.nblist_kind == GMD_NBLIST_LINKED_LISTS ? c->P.ncells : (c->d.N + NSQ_PP - 1) / NSQ_PP;
    const int every = (units + wpb - 1) / wpb;
    return std::min(std::min(every, std::max((every + 1) / 2, c->cus * 4 / nrep)), c->cus * 4);
}

int gmd_batch_create(const gmd_desc *descs, int nrep, const int *blocks, int driver, gmd_batch **out) {
    if (!descs || !out) return fail("gmd_batch_create: null argument");
    *out = nullptr;
    if (nrep < 1) return fail("gmd_batch_create: need at least one replica");
    if (driver != GMD_BATCH_PERSISTENT && driver != GMD_BATCH_GRAPH)
        return fail("gmd_batch_create: unknown driver %d", driver);
    const gmd_desc &d0 = descs[0];
    for (int r = 1; r < nrep; ++r) {
        const gmd_desc &d = descs[r];
        if (d.pair_base != d0.pair_base || d.cutoff != d0.cutoff || d.integrator != d0.integrator ||
            d.ntypes != d0.ntypes || d.tp != d0.tp || d.pb != d0.pb)
            return fail("gmd_batch_create: replica %d differs from replica 0 in pair function, cutoff, integrator, "
                        "number of types, tp or pb (one kernel runs every replica)", r);
    }
    if (d0.integrator == GMD_INTEGRATOR_NONE) return fail("gmd_batch_create: replicas need an integrator");
    gmd_batch *b = new gmd_batch();
    b->driver = driver;
    b->integrator = d0.integrator;
#define BTRY(x)                                                             \
    do {                                                                    \
        hipError_t e_ = (x);                                                \
        if (e_ != hipSuccess) {                                             \
            batch_free(b);                                                  \
            return fail("gmd_batch_create: %s: %s", #x, hipGetErrorString(e_)); \
        }                                                                   \
    } while (0)
    BTRY(hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking));
    BTRY(hipEventCreate(&b->ev0));
    BTRY(hipEventCreate(&b->ev1));
    BTRY(hipMalloc((void **)&b->d_Ps, nrep * sizeof(DP)));
    std::vector<int> nb(nrep);
    for (int r = 0; r < nrep; ++r) {
        gmd_desc d = descs[r];
        d.gridsync = 0;
        d.use_graph = 0;
        gmd_ctx *c = nullptr;
        if (ctx_create(&d, &c, b->stream)) {
            std::string msg = g_err;
            batch_free(b);
            return fail("gmd_batch_create: replica %d: %s", r, msg.c_str());
        }
        b->reps.push_back(c);
        nb[r] = blocks ? blocks[r] : c->grid_step;
        const int cap = std::max(c->grid_step, c->cus * 32);
        if (nb[r] < 1 || nb[r] > cap) {
            batch_free(b);
            return fail("gmd_batch_create: replica %d: %d blocks requested, allowed 1..%d", r, nb[r], cap);
        }
        c->P.step_grid = c->P.rebuild_grid = nb[r];
        c->d_P = b->d_Ps + r;
        b->lds = std::max(b->lds, c->lds_step);
        b->block = c->block;
        b->cus = c->cus;
    }
    b->kern = b->reps[0]->kern;
    // Rebuild steps are split where the list steps of all replicas fill the
    // device at most three times over (16 wavefronts a CU): a step then waits
    // for its rebuilding replicas.  In more rounds than that their time is
    // hidden behind the others' and the extra blocks only cost (gains and
    // losses of the steps' time, tp = 2: 2200 list blocks 18 %, 2800 29 %;
    // 5000 -4 %, 18000 -6 %).
    long long blocks_all = 0;
    for (int n : nb) blocks_all += n;
    const std::vector<int> nlist = nb;
    if (driver == GMD_BATCH_GRAPH && blocks_all <= 3LL * 4 * b->cus) {
        std::vector<size_t> kat(nrep, 0);
        size_t kn = 0;
        for (int r = 0; r < nrep; ++r) {
            DP &P = b->reps[r]->P;
            P.rebuild_grid = std::max(nb[r], rebuild_blocks(b->reps[r], nrep));
            b->gk = std::max(b->gk, std::min(P.step_grid, 16));
            kat[r] = kn;
            kn += P.nblist_kind == 1 ? (size_t)P.ncells * P.ccap : (size_t)P.N;
        }
        if (b->integrator == GMD_NVT) {
            BTRY(hipMalloc((void **)&b->d_kcell, kn * sizeof(float)));
            for (int r = 0; r < nrep; ++r) b->reps[r]->P.kcell = (GMEM float *)(b->d_kcell + kat[r]);
        }
    }
    for (int r = 0; r < nrep; ++r) {
        gmd_ctx *c = b->reps[r];
        nb[r] = c->P.rebuild_grid;
        BTRY(hipMemcpy(c->d_P, &c->P, sizeof(DP), hipMemcpyHostToDevice));
    }
    batch_layout(nb, nlist, b->h_blk);
    b->grid = (int)b->h_blk.size();
    if (driver == GMD_BATCH_PERSISTENT) {
        int per_cu = 0;
        BTRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)b->kern.bpers, b->block, b->lds));
        if (per_cu * b->cus < b->grid) {
            const int g = b->grid, room = per_cu * b->cus, bs = b->block;
            batch_free(b);
            return fail("gmd_batch_create: the persistent batch needs %d co-resident blocks of %d threads, the device "
                        "holds %d; assign fewer blocks per replica", g, bs, room);
        }
    }
    BTRY(hipMalloc((void **)&b->d_blk, b->h_blk.size() * sizeof(BatchBlk)));
    BTRY(hipMemcpy(b->d_blk, b->h_blk.data(), b->h_blk.size() * sizeof(BatchBlk), hipMemcpyHostToDevice));
    BTRY(hipHostMalloc((void **)&b->h_start, (size_t)nrep * sizeof(RunStart), hipHostMallocDefault));
#undef BTRY
    *out = b;
    return 0;
}

int gmd_batch_destroy(gmd_batch *b) { return batch_free(b); }

int gmd_batch_size(gmd_batch *b, int *nrep, int *grid) {
    if (!b) return fail("gmd_batch_size: null batch");
    if (nrep) *nrep = (int)b->reps.size();
    if (grid) *grid = b->grid;
    return 0;
}

int gmd_batch_context(gmd_batch *b, int rep, gmd_ctx **out) {
    if (!b || !out) return fail("gmd_batch_context: null argument");
    if (rep < 0 || rep >= (int)b->reps.size()) return fail("gmd_batch_context: replica %d out of range", rep);
    *out = b->reps[rep];
    return 0;
}

int gmd_batch_run(gmd_batch *b, float time_zero, int steps) {
    if (!b) return fail("gmd_batch_run: null batch");
    const unsigned nrep = (unsigned)b->reps.size();
    unsigned gx = 1, gs = 1;
    for (size_t r = 0; r < b->reps.size(); ++r) {
        gmd_ctx *c = b->reps[r];
        if (run_prepare(c, time_zero, steps, false)) {
            std::string msg = g_err;
            return fail("gmd_batch_run: replica %d: %s", (int)r, msg.c_str());
        }
        b->h_start[r] = run_start(c);
        gx = std::max(gx, run_begin_blocks(c, steps));
        gs = std::max(gs, (unsigned)c->grid_aux);
    }
    // the rebuild-flag arrays may have been reallocated by the preparation;
    // the set-up of all replicas in two launches
    hipStream_t st = b->stream;
    const DP *Ps = b->d_Ps;
    const BatchBlk *blk = b->d_blk;
    hipLaunchKernelGGL(k_batch_begin, dim3(gx, nrep), dim3(256), 0, st, Ps, steps, time_zero,
                       (const RunStart *)b->h_start);
    hipLaunchKernelGGL(k_batch_setup, dim3(gs, nrep), dim3(256), 0, st, Ps);
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipEventRecord(b->ev0, st));
    if (b->driver == GMD_BATCH_PERSISTENT) {
        void *args[] = {(void *)&Ps, (void *)&blk};
        HIPCHECK(hipLaunchCooperativeKernel((const void *)b->kern.bpers, dim3(b->grid), dim3(b->block), args,
                                            (unsigned)b->lds, st));
    } else {
        auto step = [&](int k) {
            hipLaunchKernelGGL(b->kern.bstep, dim3(b->grid), dim3(b->block), b->lds, st, Ps, blk, k);
            if (b->d_kcell) hipLaunchKernelGGL(k_batch_ksum, dim3(b->gk, nrep), dim3(b->block), 0, st, Ps, k);
        };
        if (!b->gexec) {
            HIPCHECK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
            for (int k = 0; k < GRAPH_STEPS; ++k) step(k);
            hipLaunchKernelGGL(k_batch_advance, dim3((nrep + 255) / 256), dim3(256), 0, st, Ps, (int)nrep, GRAPH_STEPS);
            HIPCHECK(hipStreamEndCapture(st, &b->graph));
            HIPCHECK(hipGraphInstantiate(&b->gexec, b->graph, nullptr, nullptr, 0));
        }
        // as in run_impl: whole groups of steps, then the rest
        const int groups = (steps + 1) / GRAPH_STEPS, rest = (steps + 1) % GRAPH_STEPS;
        for (int g = 0; g < groups; ++g) HIPCHECK(hipGraphLaunch(b->gexec, st));
        for (int k = 0; k < rest; ++k) step(k);
        HIPCHECK(hipGetLastError());
    }
    HIPCHECK(hipEventRecord(b->ev1, st));
    hipLaunchKernelGGL(k_batch_publish, dim3(nrep), dim3(256), 0, st, Ps);
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipStreamSynchronize(st));
    HIPCHECK(hipEventElapsedTime(&b->last_ms, b->ev0, b->ev1));
    for (size_t r = 0; r < b->reps.size(); ++r)
        if (run_complete(b->reps[r], steps)) {
            std::string msg = g_err;
            return fail("gmd_batch_run: replica %d: %s", (int)r, msg.c_str());
        }
    return 0;
}

int gmd_batch_fetch(gmd_batch *b) {
    if (!b) return fail("gmd_batch_fetch: null batch");
    // (replicas on one stream: earlier work is done when these run)
    HIPCHECK(hipStreamSynchronize(b->stream));
    const unsigned nrep = (unsigned)b->reps.size();
    unsigned gx = 1;
    for (size_t r = 0; r < b->reps.size(); ++r) {
        b->h_start[r].buf0 = b->reps[r]->buf0;   // the buffer that holds the positions
        gx = std::max(gx, xfer_grid(b->reps[r], b->reps[r]->d.N).x);
    }
    for (const gmd_ctx *c : b->reps)
        if (c->xcap < XferSeg((size_t)c->d.N, (size_t)std::max(0, c->d.nscalars)).end)
            return 0;   // a large replica: each is brought by its own gmd_download
    hipLaunchKernelGGL(k_batch_unpack, dim3(gx, nrep), dim3(256), 0, b->stream, (const DP *)b->d_Ps,
                       (const RunStart *)b->h_start);
    hipLaunchKernelGGL(k_batch_fetch, dim3(gx, nrep), dim3(256), 0, b->stream, (const DP *)b->d_Ps);
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipStreamSynchronize(b->stream));
    for (gmd_ctx *c : b->reps) c->fetched = true;
    return 0;
}

int gmd_batch_last_run_ms(gmd_batch *b, float *ms) {
    if (!b || !ms) return fail("gmd_batch_last_run_ms: null argument");
    *ms = b->last_ms;
    return 0;
}

}  // extern "C"

#include "gmd_adjoint.h"
