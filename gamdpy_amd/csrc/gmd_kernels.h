// gmd_kernels.h -- the per-timestep work as device functions.
//
// One MD step is ONE kernel (k_step), or one iteration of the persistent
// cooperative kernel.  The step body is:
//
//   rebuild step (skin test failed at the end of the previous step):
//     linked lists: one wavefront per cell walks the 5x5x5 stencil
//       (nblist_linked_lists.py:133-193), writes the lists of the cell's
//       particles, then computes their forces and integrates them;
//     N squared: LDS-tiled scan of all j (nblist.py:89-143), then forces;
//   other steps: forces from the neighbour lists, tp lanes per particle
//     (pair_potential.py:185-246), then the integrator update of the same
//     particle (NVE.py / NVT.py / NVT_Langevin.py).
//
// Positions are double-buffered (read pos[cur], write pos[cur^1]), so a
// particle can be integrated as soon as its own force is known.  After the
// update each particle inserts itself into the cell grid of the next step
// (three rotating buffers), so a rebuild never needs an extra pass or a grid
// barrier.  The step's tail finishes the deterministic reductions
// (thermostat, momentum reset, scalar saver): in the persistent kernel one
// block runs it after the grid barrier; in the kernel-per-step path every
// block of the next step (of its replica, in a batch) runs it (folded_tail).
#pragma once
#include "gmd_device.h"
#include <type_traits>

#define LL_PER 8                 // candidates per lane and pass of the cell walk
#define LL_IDXCAP (64 * LL_PER)  // stencil members per wave and pass
#define LL_OWNCAP 64             // particles of the centre cell (cell capacity limit)
#define LL_WAVE_LDS (LL_OWNCAP * 4 + LL_IDXCAP * 16 + LL_IDXCAP * 2)
#define LL_MAX_N (1 << 24)       // candidate tags pack index | type << 24

typedef const GMEM float4 *cpos_t;
typedef GMEM float4 *pos_t;

// The blocks that share one system's step: this block's index among them and
// their count (the whole grid for one system; a slice of it for a batch).
struct BlockCtx {
    int bid, nb;
};

// store j as list entry k of the particle whose lanes' words start at row
// (nbl + i tp): local entry m = k >> tsh of lane k & (tp - 1), in the layout
// of nb16 (rs: words between rows)
__device__ __forceinline__ void nbl_put(GMEM int *row, int k, int j, int tsh, int tp, size_t rs, bool nb16) {
    const unsigned m = (unsigned)k >> tsh, t = (unsigned)k & (unsigned)(tp - 1);
    if (nb16)
        ((GMEM unsigned short *)row)[2 * ((size_t)(m >> 1) * rs + t) + (m & 1u)] = (unsigned short)j;
    else
        row[(size_t)m * rs + t] = j;
}

// list entry u (0 .. PS_UNR-1) of a batch from the words the lane loaded:
// 16-bit entries two a word (low half first), or one 32-bit entry a word
__device__ __forceinline__ int nbl_entry(const unsigned *raw, int u, bool nb16) {
    const unsigned h = (u & 1) ? (raw[u >> 1] >> 16) : (raw[u >> 1] & 0xffffu);
    return (int)(nb16 ? h : raw[u]);
}

template <typename T>
__device__ __forceinline__ T *gen_ptr(GMEM T *p) {
    return (T *)p;
}

__device__ __forceinline__ int ld_flag(const GMEM int *p) {
    return __hip_atomic_load(gen_ptr(const_cast<GMEM int *>(p)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// nblist.py:112-116: the pair (i, j) is in i's half list (UtilizeNIII)
__device__ __forceinline__ bool niii_owns(int i, int j, int N) {
    const int two_dn = 2 * (j - i);
    return (two_dn > 0 && two_dn <= N) || (two_dn < -N);
}

// A list longer than its slots (nblist.py:126-129 records the largest count);
// with UtilizeNIII the limit the caller set applies to the half list
__device__ __forceinline__ void list_overflow(const DP &P, int count, int half) {
    if (count > P.max_nbs) atomicMax(gen_ptr(&P.ctrl->nbflag[1]), count);
    if (P.niii && half > P.max_half) atomicMax(gen_ptr(&P.ctrl->nbflag[1]), half);
}

__device__ __forceinline__ bool excluded(const DP &P, int i, int j) {
    if (P.excl == nullptr) return false;
    const GMEM int *row = P.excl + (size_t)i * P.excl_cols;
    int n = row[P.excl_cols - 1];
    for (int k = 0; k < n; ++k)
        if (row[k] == j) return true;
    return false;
}

// The pair table entry of type pair t from the parameter table (once per
// run, k_pair_table)
__device__ inline void prepare_pair(const DP &P, int t, PairP &q) {
    const GMEM float *row = P.raw_params + (size_t)P.nparams * t;
    if (P.pair_base >= 6) {
        float r[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) r[k] = k < P.nparams - 1 ? row[k] : 0.0f;
        make_pairp_rows(P.pair_base, P.cutoff, r, P.nparams - 1, row[P.nparams - 1], P.term_kind, P.term_first,
                        P.term_exps, P.nterms, q);
    } else {
        make_pairp(P.pair_base, P.cutoff, row[0], row[1], row[2], q, P.pexp0, P.pexp1);
    }
}

// The prepared table into LDS, word by word
__device__ inline void load_pair_table(const DP &P, PairP *pp) {
    const int nw = P.ntypes * P.ntypes * (int)(sizeof(PairP) / 4);
    const GMEM int *src = (const GMEM int *)P.ptab;
    int *dst = (int *)pp;
    for (int w = threadIdx.x; w < nw; w += blockDim.x) dst[w] = src[w];
}

// Entry t of a pair table row in LDS, the address formed in 32 bits
__device__ __forceinline__ const LDSMEM PairP *lds_pair(const LDSMEM PairP *row, int t) {
    return (const LDSMEM PairP *)(uintptr_t)((unsigned)(uintptr_t)row + (unsigned)t * (unsigned)sizeof(PairP));
}

__device__ __forceinline__ void wave_sync_lds() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A barrier of the block over its LDS only: __syncthreads also waits for the
// wavefront's global loads and stores, here the next tile's positions and
// the list entries, which no other wavefront of the block reads
__device__ __forceinline__ void block_sync_lds() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// ---------------------------------------------------------------------------
// Cell grid: nblist_linked_lists.py:125-131, cell index evaluated in float64
// (numba promotes r + 0.5*L to float64): floor((r + L/2) n / L) mod n.
// ---------------------------------------------------------------------------
// floor(...) mod n with Python's sign rule; a wrapped position gives a value
// in [0, n], so the modulo is one compare in the common case
__device__ __forceinline__ int cell_mod(double f, int n) {
    int c = (int)f;
    if ((unsigned)c >= (unsigned)n) {
        c %= n;
        if (c < 0) c += n;
    }
    return c;
}

// floor(((x + L/2) n) / L) mod n without the division (three float64 divides
// took a fifth of a rebuild's integrations, 28600 -> 22400 cycles a wavefront
// at KA N = 65536): with iL the inverse of L to an ulp or two, the quotient is
// off by at most one up to 2^21 cells, and the sign of the remainder, one exact
// fma, says which way
__device__ __forceinline__ int cell_dim(float x, double L, float iL, int n) {
    const double a = ((double)x + 0.5 * L) * (double)n;
    double q = floor(a * (double)iL);
    const double r = fma(-q, L, a);
    if (r < 0.0) q -= 1.0;
    if (r >= L) q += 1.0;
    return cell_mod(q, n);
}

__device__ __forceinline__ int cell_of_box(const DP &P, float x, float y, float z, float Lx, float Ly, float Lz,
                                           float iLx, float iLy, float iLz) {
    const int cx = cell_dim(x, (double)Lx, iLx, P.ncx);
    const int cy = cell_dim(y, (double)Ly, iLy, P.ncy);
    const int cz = cell_dim(z, (double)Lz, iLz, P.ncz);
    return (cx * P.ncy + cy) * P.ncz + cz;
}

__device__ __forceinline__ int cell_of(const DP &P, float x, float y, float z) {
    return cell_of_box(P, x, y, z, P.box0, P.box1, P.box2, P.ibox0, P.ibox1, P.ibox2);
}

// insertion into cell buffer buf of the grid over the box (Lx, Ly, Lz)
__device__ __forceinline__ void cell_insert(const DP &P, int buf, int i, float x, float y, float z, float Lx, float Ly,
                                            float Lz, float iLx, float iLy, float iLz) {
    const int c = cell_of_box(P, x, y, z, Lx, Ly, Lz, iLx, iLy, iLz);
    const size_t cc = (size_t)buf * P.ncells + c;
    const int slot = atomicAdd(gen_ptr(P.ccount + cc), 1);
    if (slot < P.ccap)
        P.cmem[cc * P.ccap + slot] = i;
    else
        atomicMax(gen_ptr(&P.ctrl->cell_overflow), slot + 1);
}

// ---------------------------------------------------------------------------
// Step description shared by all threads of a step
// ---------------------------------------------------------------------------
struct StepInfo {
    int s;
    int cur;                   // position buffer read this step
    int cbuf, cbuf_next, cbuf_clear;
    bool integrate, rebuild;
    bool need_ksum, need_mom, need_save;
    bool npt;                  // NPT_Atomic: the step also needs the W sum (need_wsum)
    bool need_wsum;
    bool scal;                 // U, W, lapU of this evaluation are wanted (saver step or no integration)
    int conf_idx;              // ConfigurationSaver save index of this step (-1: none)
    bool ksplit;               // each particle's kinetic energy goes to P.kcell (a split rebuild step)
    bool wrapped;              // every position of the run lies in [-L/2, L/2] (else: minimum image always)
    bool apply_shift;
    float sh0, sh1, sh2;
    float xi;
    // NPT_Atomic: the box of this step's interactions (L), its inverse, the
    // box after this step's integration (Ln), the state of this step and
    // the coefficients it implies (friction factors, dilation rate, length
    // factor)
    float L0, L1, L2, iL0, iL1, iL2, Ln0, Ln1, Ln2;
    float np_t0, np_b0, np_vol;
    float np_plus, np_minus, np_rf;
    double np_sf;
    float lang_amp;
    float t0;
    int nsteps;
    long long lstep;
};

// the same value in every lane, made visibly uniform (a scalar register)
__device__ __forceinline__ float uniform_f(float x) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
}

// the NPT_Atomic fields of a StepInfo computed alike in every lane, kept in
// scalar registers
__device__ __forceinline__ void npt_uniform(StepInfo &I) {
    I.np_t0 = uniform_f(I.np_t0);
    I.np_b0 = uniform_f(I.np_b0);
    I.np_vol = uniform_f(I.np_vol);
    I.L0 = uniform_f(I.L0);
    I.L1 = uniform_f(I.L1);
    I.L2 = uniform_f(I.L2);
    I.iL0 = uniform_f(I.iL0);
    I.iL1 = uniform_f(I.iL1);
    I.iL2 = uniform_f(I.iL2);
    I.Ln0 = uniform_f(I.Ln0);
    I.Ln1 = uniform_f(I.Ln1);
    I.Ln2 = uniform_f(I.Ln2);
    I.np_plus = uniform_f(I.np_plus);
    I.np_minus = uniform_f(I.np_minus);
    I.np_rf = uniform_f(I.np_rf);
    const unsigned long long b = (unsigned long long)__double_as_longlong(I.np_sf);
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)b);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(b >> 32));
    I.np_sf = __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// NPT_Atomic.py:108-114,162-170: the friction factors, the dilation rate and
// the length factor of a step from its state (float64 where numba promotes),
// and the box after the step
__device__ inline void npt_coeffs(const DP &P, StepInfo &I) {
#pragma clang fp contract(off)
    const double deg = P.degrees;
    const double factor = (double)(0.5f * P.dt) * ((1.0 + 3.0 / deg) * (double)I.np_b0 + (double)I.np_t0);
    I.np_plus = 1.0f / (float)(1.0 + factor);
    I.np_minus = (float)(1.0 - factor);
    I.np_rf = I.np_b0 * P.dt;
    const double sf3 = 1.0 + (double)P.dt * 3.0 * (double)I.np_b0;
    I.np_sf = pow(sf3, 1.0 / 3.0);
    I.iL0 = 1.0f / I.L0;
    I.iL1 = 1.0f / I.L1;
    I.iL2 = 1.0f / I.L2;
    I.Ln0 = (float)((double)I.L0 * I.np_sf);
    I.Ln1 = (float)((double)I.L1 * I.np_sf);
    I.Ln2 = (float)((double)I.L2 * I.np_sf);
}

// update_thermostat_barostat_state (NPT_Atomic.py:148-187): the state of the
// step after one (at time t) whose kinetic energies sum to K and virials to
// W: volume and box scaled, then the thermostat and barostat rates
__device__ inline void npt_advance(const DP &P, StepInfo &I, float K, float W, double t) {
#pragma clang fp contract(off)
    const double deg = P.degrees;
    const double T = 2.0 * (double)K / deg;
    const double sf3 = 1.0 + (double)P.dt * 3.0 * (double)I.np_b0;
    const double mt = (double)P.mass_t * T, mp = (double)P.mass_p * T;
    const float vol = (float)((double)I.np_vol * sf3);
    const double sf = pow(sf3, 1.0 / 3.0);
    I.L0 = (float)((double)I.L0 * sf);
    I.L1 = (float)((double)I.L1 * sf);
    I.L2 = (float)((double)I.L2 * sf);
    const double tT = target_temperature(P, t), tP = target_pressure(P, t);
    const double ip = (T * (double)P.N + (double)W) / (double)vol;
    const float b0 = I.np_b0;
    const double ke = ((double)(2.0f * K) + (double)(b0 * b0) * mp) / ((deg + 1.0) * tT) - 1.0;
    const double pd = 3.0 * ((double)vol * (ip - tP) + (double)(0.5f * K) / deg);
    const float t0n = (float)((double)I.np_t0 + (double)P.dt * ke * (deg + 1.0) * tT / mt);
    I.np_b0 = (float)((double)b0 + (double)P.dt * (pd / mp + (double)(t0n * b0)));
    I.np_t0 = t0n;
    I.np_vol = vol;
}

// fold: the folded-tail path, where the state of step s is computed from
// that of step s - 1 by the step's own tail (folded_tail)
__device__ __forceinline__ StepInfo step_info(const DP &P, int s, int integrator, bool rebuild, bool fold = false) {
    StepInfo I;
    const GMEM Ctrl *C = P.ctrl;
    I.s = s;
    I.cur = C->buf0 ^ (s & 1);
    I.cbuf = s % 3;
    I.cbuf_next = (s + 1) % 3;
    I.cbuf_clear = (s + 2) % 3;
    I.rebuild = rebuild;
    I.nsteps = C->nsteps;
    I.t0 = C->t0;
    I.integrate = (s < I.nsteps) && integrator != 0;
    I.npt = integrator == 4;
    I.need_ksum = I.integrate && (integrator == 2 || I.npt);
    I.need_wsum = I.integrate && I.npt;
    I.need_mom = I.integrate && P.mom_every > 0 && (s % P.mom_every) == 0;
    I.need_save = I.integrate && P.save_every > 0 && (s % P.save_every) == 0 && (s / P.save_every) < P.saves_per_block;
    // an evaluation's U, W, lapU are read only by its saver row or, after the
    // last evaluation of a run (which does not integrate), by the host
    I.scal = I.need_save || !I.integrate || I.npt;   // NPT_Atomic: W every step
    // configuration_saver.py:118-127: block-local step 0 -> save 0, step 2^b -> save b + 1
    I.ksplit = false;
    I.conf_idx = -1;
    if (P.conf_saves > 0) {
        if (s == 0)
            I.conf_idx = 0;
        else if ((s & (s - 1)) == 0 && 32 - __clz(s) < P.conf_saves)
            I.conf_idx = 32 - __clz(s);   // log2(s) + 1
    }
    I.apply_shift = (C->shift_step == s);
    // NPT_Atomic: a scaled position may lie an ulp outside the scaled box,
    // so every pair takes the minimum image
    I.wrapped = C->unwrapped == 0 && !I.npt;
    I.sh0 = C->shift[0];
    I.sh1 = C->shift[1];
    I.sh2 = C->shift[2];
    I.xi = C->xi;
    I.lstep = C->lstep0 + s;
    if (I.npt) {
        const int b = (fold && s > 0) ? ((s - 1) & 1) : (s & 1);
        I.np_t0 = C->npt[b][0];
        I.np_b0 = C->npt[b][1];
        I.np_vol = C->npt[b][2];
        I.L0 = C->npt[b][3];
        I.L1 = C->npt[b][4];
        I.L2 = C->npt[b][5];
        if (!(fold && s > 0)) {
            npt_coeffs(P, I);
            npt_uniform(I);
        }
    }
    I.lang_amp = 0.f;
    if (integrator == 3) {
        double t = (double)I.t0 + (double)s * (double)P.dt;
        float T = (float)target_temperature(P, t);
        {
#pragma clang fp contract(off)
            I.lang_amp = sqrtf(((2.0f * P.alpha) * T) * P.dt);
        }
    }
    return I;
}

__device__ __forceinline__ void wrap_pbc(float &r, int &dim_img, float L) {
#pragma clang fp contract(off)
    if (r * 2.0f > L) {
        r = r - L;
        dim_img += 1;
    }
    if (r * 2.0f < -L) {
        r = r + L;
        dim_img -= 1;
    }
}

// ---------------------------------------------------------------------------
// Integrator update of particle i once its force (fx, fy, fz) and its
// interaction scalars are known (NVE.py:59-105 / NVT.py:188-224 /
// NVT_Langevin.py:342-385), PBC wrap, skin test of the next evaluation and
// insertion into the next cell grid.  Only 'writer' lanes store.
// ---------------------------------------------------------------------------
template <int INTEG>
__device__ __forceinline__ void particle_finish(const DP &P, const StepInfo &I, const int i, const float4 ri,
                                                float4 v4, const float4 rr, const float fx, const float fy,
                                                const float fz, const float uu, const float ww, const float ll,
                                                const bool writer, float acc[GMD_NRED]) {
    const int N = P.N;
    // the box of this step (NPT_Atomic: of its state)
    const float L0 = INTEG == 4 ? I.L0 : P.box0, L1 = INTEG == 4 ? I.L1 : P.box1, L2 = INTEG == 4 ? I.L2 : P.box2;
    if (I.conf_idx >= 0 && writer) {
        // the configuration at the start of the step, after its interactions
        // (the reference's prestep action), in the caller's numbering
        const int ic = P.perm[i];
        GMEM float *o = P.conf_out + (size_t)I.conf_idx * 6 * N;
        o[3 * ic] = ri.x;
        o[3 * ic + 1] = ri.y;
        o[3 * ic + 2] = ri.z;
        o[3 * ((size_t)N + ic)] = (float)P.rim[i];
        o[3 * ((size_t)N + ic) + 1] = (float)P.rim[(size_t)N + i];
        o[3 * ((size_t)N + ic) + 2] = (float)P.rim[(size_t)2 * N + i];
    }
    if (I.apply_shift) {
#pragma clang fp contract(off)
        v4.x = v4.x - I.sh0;
        v4.y = v4.y - I.sh1;
        v4.z = v4.z - I.sh2;
    }
    if (writer) {
        P.frc[i] = make_float4(fx, fy, fz, 0.f);
        if (I.scal) {
            if (P.compute_u) P.sc[(size_t)SC_U * N + i] = uu;
            if (P.compute_w) P.sc[(size_t)SC_W * N + i] = ww;
            if (P.compute_lap) P.sc[(size_t)SC_LAP * N + i] = ll;
        }
        acc[RED_U] += uu;
        acc[RED_W] += ww;
        acc[RED_LAP] += ll;
    }
    if (!I.integrate) {
        if (writer && I.apply_shift) P.vel[i] = v4;
        return;
    }
    float rx = ri.x, ry = ri.y, rz = ri.z;
    float vx = v4.x, vy = v4.y, vz = v4.z;
    const float m = v4.w;
    const float dt = P.dt;
    float K, fsq;
    {
#pragma clang fp contract(off)
        fsq = fx * fx;
        fsq = fsq + fy * fy;
        fsq = fsq + fz * fz;
        if (INTEG == 1) {  // NVE.py:78-97
            float vo, vm;
            vo = vx; vx = vx + (fx / m) * dt; vm = (vo + vx) / 2.0f; K = ((0.5f * m) * vm) * vm; rx = rx + vx * dt;
            vo = vy; vy = vy + (fy / m) * dt; vm = (vo + vy) / 2.0f; K = K + ((0.5f * m) * vm) * vm; ry = ry + vy * dt;
            vo = vz; vz = vz + (fz / m) * dt; vm = (vo + vz) / 2.0f; K = K + ((0.5f * m) * vm) * vm; rz = rz + vz * dt;
        } else if (INTEG == 2) {  // NVT.py:196-215
            const float factor = (0.5f * I.xi) * dt;
            const float plus = 1.0f / (1.0f + factor);
            const float minus = 1.0f - factor;
            vx = plus * (minus * vx + (fx / m) * dt); K = ((0.5f * m) * vx) * vx; rx = rx + vx * dt;
            vy = plus * (minus * vy + (fy / m) * dt); K = K + ((0.5f * m) * vy) * vy; ry = ry + vy * dt;
            vz = plus * (minus * vz + (fz / m) * dt); K = K + ((0.5f * m) * vz) * vz; rz = rz + vz * dt;
        } else if (INTEG == 4) {  // NPT_Atomic.py:126-138: friction of both rates, dilation of r
            const float plus = I.np_plus, minus = I.np_minus, rf = I.np_rf;
            vx = plus * (minus * vx + (fx / m) * dt); K = ((0.5f * m) * vx) * vx; rx = rx + (vx * dt + rf * rx);
            vy = plus * (minus * vy + (fy / m) * dt); K = K + ((0.5f * m) * vy) * vy; ry = ry + (vy * dt + rf * ry);
            vz = plus * (minus * vz + (fz / m) * dt); K = K + ((0.5f * m) * vz) * vz; rz = rz + (vz * dt + rf * rz);
        } else {  // NVT_Langevin.py:363-378
            float z0, z1, z2;
            normal3(P.seed, I.lstep, P.perm[i], z0, z1, z2);   // keyed by the caller's particle index
            float4 ob = P.obeta[i];
            const float num = 2.0f * m - P.alpha * dt;
            const float den = 2.0f * m + P.alpha * dt;
            const float a = num / den;
            const float bom = 2.0f / den;
            float b;
            b = I.lang_amp * z0; K = ((0.5f * m) * vx) * vx;
            vx = (a * vx + (bom * fx) * dt) + (bom * 0.5f) * (b + ob.x); ob.x = b; rx = rx + vx * dt;
            b = I.lang_amp * z1; K = K + ((0.5f * m) * vy) * vy;
            vy = (a * vy + (bom * fy) * dt) + (bom * 0.5f) * (b + ob.y); ob.y = b; ry = ry + vy * dt;
            b = I.lang_amp * z2; K = K + ((0.5f * m) * vz) * vz;
            vz = (a * vz + (bom * fz) * dt) + (bom * 0.5f) * (b + ob.z); ob.z = b; rz = rz + vz * dt;
            if (writer) P.obeta[i] = ob;
        }
    }
    int imx = 0, imy = 0, imz = 0;
    wrap_pbc(rx, imx, L0);
    wrap_pbc(ry, imy, L1);
    wrap_pbc(rz, imz, L2);
    // the box after this step: NPT_Atomic scales the wrapped positions with
    // it (scale_box, NPT_Atomic.py:162-171)
    float Ln0 = L0, Ln1 = L1, Ln2 = L2;
    if (INTEG == 4) {
        rx = (float)(I.np_sf * (double)rx);
        ry = (float)(I.np_sf * (double)ry);
        rz = (float)(I.np_sf * (double)rz);
        Ln0 = I.Ln0;
        Ln1 = I.Ln1;
        Ln2 = I.Ln2;
    }
    if (writer) {
        pos_t posn = I.cur ? P.pos0 : P.pos1;
        posn[i] = make_float4(rx, ry, rz, ri.w);
        P.vel[i] = make_float4(vx, vy, vz, m);
        if (P.compute_k) P.sc[(size_t)SC_K * N + i] = K;
        if (P.compute_fsq) P.sc[(size_t)SC_FSQ * N + i] = fsq;
        if (imx | imy | imz) {
            P.rim[i] += imx;
            P.rim[(size_t)N + i] += imy;
            P.rim[(size_t)2 * N + i] += imz;
        }
        // skin test for the next interaction evaluation (nblist.py:71-73)
        float dx, dy, dz;
        const float d2 = dist_sq_mic(rx, ry, rz, rr.x, rr.y, rr.z, Ln0, Ln1, Ln2, dx, dy, dz);
        if (d2 > P.skin2q) P.rebuild_flag[I.s + 1] = 1;
        if (P.nblist_kind == 1) {
            // (the context's box read here, not held from above: fewer live registers)
            if (INTEG == 4)
                cell_insert(P, I.cbuf_next, i, rx, ry, rz, Ln0, Ln1, Ln2, uniform_f(__builtin_amdgcn_rcpf(Ln0)),
                            uniform_f(__builtin_amdgcn_rcpf(Ln1)), uniform_f(__builtin_amdgcn_rcpf(Ln2)));
            else
                cell_insert(P, I.cbuf_next, i, rx, ry, rz, P.box0, P.box1, P.box2, P.ibox0, P.ibox1, P.ibox2);
        }
        acc[RED_K] += K;
        acc[RED_FSQ] += fsq;
        {
#pragma clang fp contract(off)
            acc[RED_PX] += m * vx;
            acc[RED_PX + 1] += m * vy;
            acc[RED_PX + 2] += m * vz;
        }
        acc[RED_M] += m;
    }
}

// Bond terms of particle i (bonds.py:91-123 with the harmonic bond,
// harmonic_bond_function.py:37-44): u = k (r - r0)^2 / 2, s = -k (r - r0) / r.
// Each end of a bond computes its own share from dr = r_partner - r_i (the
// minimum image), which is the other end's dr negated bit for bit, so both
// ends get the reference's force, f_i -= dr s.  u, r^2 s and (1 - D) s + k
// go to the sums that particle_finish halves and scales like the pair sums:
// each end gets u / 2 and r^2 s / (2 D).
__device__ __forceinline__ void bond_terms(const DP &P, cpos_t pos, const int i, const float4 ri, const float L0,
                                           const float L1, const float L2, float &fx, float &fy, float &fz, float &uu,
                                           float &ww, float &ll) {
    const int b1 = P.boff[i + 1];
    for (int b = P.boff[i]; b < b1; ++b) {
#pragma clang fp contract(off)
        const int2 e = P.bnd[b];
        const float4 rj = pos[e.x];
        const float2 q = P.bpar[e.y];
        float dx, dy, dz;
        const float d2 = dist_sq_mic(rj.x, rj.y, rj.z, ri.x, ri.y, ri.z, L0, L1, L2, dx, dy, dz);
        const float dist = sqrtf(d2);
        const float del = dist - q.x;
        const float u = (0.5f * q.y) * (del * del);
        const float s = ((-q.y) * del) / dist;
        fx = fx - dx * s;
        fy = fy - dy * s;
        fz = fz - dz * s;
        uu = uu + u;
        ww = ww + d2 * s;
        ll = ll + (-2.0f * s + q.y);
    }
}

// Pair term of the full-list calculator (pair_potential.py:162-178),
// accumulated as sums over pairs: f -= dr s, W += r^2 s, U += u, lap += u'' - 2 s
template <int BASE, int CUT>
__device__ __forceinline__ void pair_accum(const float d2, const float dx, const float dy, const float dz,
                                           const PairP &q, float &fx, float &fy, float &fz, float &uu, float &ww,
                                           float &ll, const bool lap) {
    float u_, sv, umm;
    pair_fast<BASE, CUT>(d2, q, u_, sv, umm, lap);
    fx -= dx * sv;
    fy -= dy * sv;
    fz -= dz * sv;
    ww += d2 * sv;
    uu += u_;
    if (lap) ll += umm - 2.0f * sv;  // (1 - D) s + u'' with D = 3
}

// The same with the pair's scalars weighted for UtilizeNIII
// (pair_potential.py:141-160): wgt = 2 when the pair is in this particle's
// half list (it then carries the whole u, r^2 s / D and 2 ((1 - D) s + u'')),
// 0 when it is in the other particle's.  The force is unchanged.
template <int BASE, int CUT>
__device__ __forceinline__ void pair_accum_w(const float d2, const float dx, const float dy, const float dz,
                                             const PairP &q, float &fx, float &fy, float &fz, float &uu, float &ww,
                                             float &ll, const bool lap, const float wgt) {
    float u_, sv, umm;
    pair_fast<BASE, CUT>(d2, q, u_, sv, umm, lap);
    fx -= dx * sv;
    fy -= dy * sv;
    fz -= dz * sv;
    ww += wgt * (d2 * sv);
    uu += wgt * u_;
    if (lap) ll += wgt * (umm - 2.0f * sv);
}

// ---------------------------------------------------------------------------
// Interactions from the neighbour list + integration of particle i by the tp
// lanes of its group (lane t).  All tp lanes must call it together.
//
// SCAL: this evaluation's U, W (and lapU when LAP) are wanted (a saver step,
// or the run's last evaluation, whose scalars the host reads); on the other
// steps only the forces are summed.  mic: bit d set when some particle of the
// wavefront is within rc + 2 skin of a box face in dimension d; otherwise
// every listed neighbour lies inside the box in the particle's own image, the
// minimum image of fl(xj - xi) is fl(xj - xi) itself, and that dimension
// skips it (a uniform branch per batch, not per pair).
// ---------------------------------------------------------------------------
#define PS_UNR 8   // list entries a lane gathers at a time

// What a particle's lanes load before its list loop: the words of the first
// PS_UNR list entries of the lane (requested before the count arrives: the
// list is zero-initialised and holds only particle indices, so an entry past
// the count is a valid index, its pair masked off), the position and the
// count.
// The velocity and the reference position, needed only after the loop, go
// by LDS DMA (global_load_lds, 16 bytes a lane) into the wave's slot of the
// rebuild scratch region, which a list step does not otherwise use: they
// arrive during the loop without holding registers through it.
struct PState {
    unsigned raw[PS_UNR];   // list words: PS_UNR / 2 of them with 16-bit entries
    float4 ri;
    int cnt;
};

// the wave's velocity and reference-position stage: 64 float4 each
__device__ __forceinline__ LDSMEM float4 *finish_stage(const DP &P) {
    extern __shared__ __align__(16) char lds[];
    const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    return (LDSMEM float4 *)((LDSMEM char *)lds + P.lds_build + wid * 2048);
}

// NBF: the list format, 1 = 16-bit entries, 2 = 32-bit, 0 = P.nb16 at run time
template <int NBF>
__device__ __forceinline__ bool list_nb16(const DP &P) {
    return NBF == 1 ? true : (NBF == 2 ? false : P.nb16 != 0);
}

// the block's stage of a deferred tail's partial sums: RED_PRE floats a
// thread, after the wavefronts' finish stages
__device__ __forceinline__ LDSMEM float *tail_stage(const DP &P) {
    extern __shared__ __align__(16) char lds[];
    return (LDSMEM float *)((LDSMEM char *)lds + P.lds_build + (blockDim.x >> 6) * 2048);
}

template <int NBF>
__device__ __forceinline__ void particle_issue(const DP &P, const StepInfo &I, const int i, const int t,
                                               PState &st) {
    cpos_t pos = I.cur ? P.pos1 : P.pos0;
    const GMEM unsigned *nbrow = (const GMEM unsigned *)P.nbl + (size_t)i * P.tp + t;
    const size_t rs = (size_t)P.N * P.tp;
    const int nw = list_nb16<NBF>(P) ? PS_UNR / 2 : PS_UNR;
#pragma unroll
    for (int u = 0; u < PS_UNR; ++u)
        if (u < nw) st.raw[u] = __builtin_nontemporal_load(nbrow + (size_t)u * rs);
    st.ri = pos[i];
    st.cnt = P.nbc[i];
    LDSMEM float4 *fs = finish_stage(P);
    __builtin_amdgcn_global_load_lds((const GMEM void *)(P.vel + i), (LDSMEM void *)fs, 16, 0, 0);
    __builtin_amdgcn_global_load_lds((const GMEM void *)(P.rref + i), (LDSMEM void *)(fs + 64), 16, 0, 0);
}

// The pair sums of particle i over its list (and its bonds): f6 = fx, fy,
// fz, and the U, W, lapU sums before their 1/2 and 1/(2 D) factors.
template <int BASE, int CUT, int INTEG, bool LAP, bool NIII, bool SCAL, int NBF>
__device__ __forceinline__ void particle_forces(const DP &P, const StepInfo &I, const PairP *pp, const int i,
                                                const int t, const PState &st, float f6[6]) {
    const int tp = P.tp;
    const int N = P.N;
    cpos_t pos = I.cur ? P.pos1 : P.pos0;
    const float L0 = INTEG == 4 ? I.L0 : P.box0, L1 = INTEG == 4 ? I.L1 : P.box1, L2 = INTEG == 4 ? I.L2 : P.box2;
    const float iL0 = INTEG == 4 ? I.iL0 : P.ibox0, iL1 = INTEG == 4 ? I.iL1 : P.ibox1,
                iL2 = INTEG == 4 ? I.iL2 : P.ibox2;
    const GMEM unsigned *nbrow = (const GMEM unsigned *)P.nbl + (size_t)i * tp + t;
    const size_t rs = (size_t)N * tp;
    const bool nb16 = list_nb16<NBF>(P);
    const int wlast = P.nwrows - 1;
    constexpr int UNR = PS_UNR;
    unsigned raw[UNR];
#pragma unroll
    for (int u = 0; u < UNR; ++u) raw[u] = st.raw[u];
    const float4 ri = st.ri;
    const int cnt = min(st.cnt, P.max_nbs);
    const int ti = __float_as_int(ri.w);
    // the dimensions in which some particle of the wavefront is within
    // rc + 2 skin of a face (every lane of the wavefront that has a particle
    // takes part; all positions of the run must lie in the box)
    unsigned mic = 7u;
    if (I.wrapped)
        mic = (__ballot(fabsf(ri.x) > P.mic_edge0) != 0ull ? 1u : 0u) |
              (__ballot(fabsf(ri.y) > P.mic_edge1) != 0ull ? 2u : 0u) |
              (__ballot(fabsf(ri.z) > P.mic_edge2) != 0ull ? 4u : 0u);
    // the pair table row of i's type, addressed in LDS with 32-bit offsets
    const LDSMEM PairP *ppi = lds_pair((const LDSMEM PairP *)pp, ti * P.ntypes);
    float fx = 0.f, fy = 0.f, fz = 0.f, uu = 0.f, ww = 0.f, ll = 0.f;
    // this lane handles entries t, t+tp, ...; UNR gathers in flight, the next
    // batch of list entries (rows clamped to the list) requested while the
    // current batch is used; every pair term is computed and masked, so the
    // batch has no branches
    const int nloc = (cnt > t) ? (cnt - t + tp - 1) / tp : 0;
    for (int m = 0; m < nloc; m += UNR) {
        float4 rj[UNR];
        int jc[UNR];   // NIII: the indices of this batch, for the half-list owner test
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            const int j = nbl_entry(raw, u, nb16);
            rj[u] = pos[j];
            if (NIII && SCAL) jc[u] = j;
        }
        if (m + UNR < nloc) {
            // the next batch's words (rows of words clamped to the list)
            if (nb16) {
#pragma unroll
                for (int u = 0; u < UNR / 2; ++u)
                    raw[u] = __builtin_nontemporal_load(nbrow + (size_t)min((m + UNR) / 2 + u, wlast) * rs);
            } else {
#pragma unroll
                for (int u = 0; u < UNR; ++u)
                    raw[u] = __builtin_nontemporal_load(nbrow + (size_t)min(m + UNR + u, wlast) * rs);
            }
        }
        float dx[UNR], dy[UNR], dz[UNR];
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            dx[u] = rj[u].x - ri.x;
            dy[u] = rj[u].y - ri.y;
            dz[u] = rj[u].z - ri.z;
        }
        if (mic & 1u) {
#pragma unroll
            for (int u = 0; u < UNR; ++u) dx[u] = mic_list(dx[u], L0, iL0);
        }
        if (mic & 2u) {
#pragma unroll
            for (int u = 0; u < UNR; ++u) dy[u] = mic_list(dy[u], L1, iL1);
        }
        if (mic & 4u) {
#pragma unroll
            for (int u = 0; u < UNR; ++u) dz[u] = mic_list(dz[u], L2, iL2);
        }
#pragma unroll
        for (int u = 0; u < UNR; ++u) {
            float d2;
            {
#pragma clang fp contract(off)
                d2 = dx[u] * dx[u];
                d2 = d2 + dy[u] * dy[u];
                d2 = d2 + dz[u] * dz[u];
            }
            PairP q;
            if (!SCAL && BASE <= 1 && CUT != 2) {
                // a, c, cut2, d in one read
                const float4 qv = *(const LDSMEM float4 *)lds_pair(ppi, __float_as_int(rj[u].w));
                q.a = qv.x;
                q.c = qv.y;
                q.cut2 = qv.z;
                q.d = qv.w;
                q.b = q.ucut = q.scut = q.cut = q.e0 = q.e1 = 0.f;
                q.kind = q.pad = 0;
            } else {
                q = *lds_pair(ppi, __float_as_int(rj[u].w));
            }
            const bool ok = (m + u < nloc) & (d2 < q.cut2);
            float u_, sv, umm;
            pair_fast<BASE, CUT>(d2, q, u_, sv, umm, LAP && SCAL);
            sv = ok ? sv : 0.f;
            fx -= dx[u] * sv;
            fy -= dy[u] * sv;
            fz -= dz[u] * sv;
            if (SCAL) {
                // full list: u / 2 and r^2 s / (2 D) per pair (applied after
                // the sums); NIII: the whole term to the owner of the pair
                float wgt = 1.0f;
                if (NIII) wgt = niii_owns(i, jc[u], N) ? 2.0f : 0.0f;
                u_ = ok ? u_ : 0.f;
                ww += wgt * (d2 * sv);
                uu += wgt * u_;
                if (LAP) ll += wgt * (ok ? umm - 2.0f * sv : 0.f);   // (1 - D) s + u'' with D = 3
            }
        }
    }
    fx = group_sum(fx, tp);
    fy = group_sum(fy, tp);
    fz = group_sum(fz, tp);
    if (SCAL) {
        uu = group_sum(uu, tp);
        ww = group_sum(ww, tp);
        if (LAP) ll = group_sum(ll, tp);
    }
    if (P.boff) bond_terms(P, pos, i, ri, L0, L1, L2, fx, fy, fz, uu, ww, ll);
    f6[0] = fx;
    f6[1] = fy;
    f6[2] = fz;
    f6[3] = uu;
    f6[4] = ww;
    f6[5] = ll;
}

// The integration of particle i from its sums, with the velocity and
// reference position its particle_issue staged.
template <int INTEG>
__device__ __forceinline__ void particle_end(const DP &P, const StepInfo &I, const int i, const int t,
                                             const float4 ri, const float f6[6], float acc[GMD_NRED]) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const LDSMEM float4 *fs = finish_stage(P);
    const int lane = threadIdx.x & 63;
    const float4 v4 = fs[lane];
    const float4 rr = fs[64 + lane];
    particle_finish<INTEG>(P, I, i, ri, v4, rr, f6[0], f6[1], f6[2], f6[3] * 0.5f, f6[4] * (0.5f / 3.0f), f6[5],
                           t == 0, acc);
}

template <int BASE, int CUT, int INTEG, bool LAP, bool NIII, bool SCAL, int NBF>
__device__ __forceinline__ void particle_step(const DP &P, const StepInfo &I, const PairP *pp, const int i,
                                              const int t, const PState &st, float acc[GMD_NRED]) {
    float f6[6];
    particle_forces<BASE, CUT, INTEG, LAP, NIII, SCAL, NBF>(P, I, pp, i, t, st, f6);
    particle_end<INTEG>(P, I, i, t, st.ri, f6, acc);
}

// ---------------------------------------------------------------------------
// Steps without a rebuild: tp lanes per particle, grid-stride over particles
// ---------------------------------------------------------------------------
template <int BASE, int CUT, int INTEG, bool LAP, bool NIII, bool SCAL, int NBF>
__device__ __forceinline__ void particle_loop(const DP &P, const BlockCtx &B, const StepInfo &I, const PairP *pp,
                                              float acc[GMD_NRED]) {
    const int t = threadIdx.x & (P.tp - 1);
    const int slots = blockDim.x >> P.tp_shift;
    for (int i = B.bid * slots + (int)(threadIdx.x >> P.tp_shift); i < P.N; i += B.nb * slots) {
        PState st;
        particle_issue<NBF>(P, I, i, t, st);
        particle_step<BASE, CUT, INTEG, LAP, NIII, SCAL, NBF>(P, I, pp, i, t, st, acc);
    }
}

template <int BASE, int CUT, int INTEG>
__device__ __forceinline__ void step_lists(const DP &P, const BlockCtx &B, const StepInfo &I, const PairP *pp,
                                  float acc[GMD_NRED]) {
    // loops of their own: without the scalars (most steps; one per list
    // format), with them, with the laplacian, with the NIII split of the
    // scalars (these read the format at run time)
    if (!I.scal) {
        if (P.nb16)
            particle_loop<BASE, CUT, INTEG, false, false, false, 1>(P, B, I, pp, acc);
        else
            particle_loop<BASE, CUT, INTEG, false, false, false, 2>(P, B, I, pp, acc);
    } else if (P.niii) {
        if (P.compute_lap)
            particle_loop<BASE, CUT, INTEG, true, true, true, 0>(P, B, I, pp, acc);
        else
            particle_loop<BASE, CUT, INTEG, false, true, true, 0>(P, B, I, pp, acc);
    } else if (P.compute_lap) {
        particle_loop<BASE, CUT, INTEG, true, false, true, 0>(P, B, I, pp, acc);
    } else {
        particle_loop<BASE, CUT, INTEG, false, false, true, 0>(P, B, I, pp, acc);
    }
}

// A list step whose folded tail (the previous step's kinetic sum, the
// thermostat update) is deferred: every wavefront computes its first
// particle's pair sums, then runs hook(I) once, at uniform control flow (it
// holds block barriers), then integrates; further particles (a grid smaller
// than N) follow as usual.  The scalars are not summed (no saver, not the
// last evaluation).
template <int BASE, int CUT, int INTEG, int NBF, class Hook>
__device__ __forceinline__ void particle_loop_deferred(const DP &P, const BlockCtx &B, StepInfo &I, const PairP *pp,
                                                       float acc[GMD_NRED], Hook &hook) {
    const int t = threadIdx.x & (P.tp - 1);
    const int slots = blockDim.x >> P.tp_shift;
    const int stride = B.nb * slots;
    int i = B.bid * slots + (int)(threadIdx.x >> P.tp_shift);
    const bool has = i < P.N;
    float f6[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    PState st;
    if (has) {
        particle_issue<NBF>(P, I, i, t, st);
        particle_forces<BASE, CUT, INTEG, false, false, false, NBF>(P, I, pp, i, t, st, f6);
    }
    hook(I);
    if (has) particle_end<INTEG>(P, I, i, t, st.ri, f6, acc);
    for (i += stride; i < P.N; i += stride) {
        PState s2;
        particle_issue<NBF>(P, I, i, t, s2);
        particle_step<BASE, CUT, INTEG, false, false, false, NBF>(P, I, pp, i, t, s2, acc);
    }
}

// ---------------------------------------------------------------------------
// Rebuild step, linked lists: one wavefront per cell.  The wavefront stages
// the members of the 125 stencil cells (cell >= (rc+skin)/2,
// nblist_linked_lists.py:151-182) in LDS, then for each particle of its cell
// tests them 64 at a time: accepted neighbours are appended to the list in
// ballot order (stencil order, then particle index: deterministic) and those
// inside the pair cutoff contribute to the force in the same pass.  Lane q
// finally holds the totals of particle q and integrates it.
// ---------------------------------------------------------------------------
// The value of lane l (l wave-uniform) in every lane, via a scalar register.
__device__ __forceinline__ int lane_i(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ float lane_f(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// Sums of six per-lane values over the wavefront.  The first three exchange
// levels halve the set of values a lane carries (eight slots, the last two
// zero): after them lane l holds a partial of slot l >> 3 over the eight
// lanes that differ from it in bits 3-5, and three more levels complete it.
// The total of slot c is then in lanes 8c .. 8c + 7 (10 exchanges instead of
// 36 for six separate reductions; the swaps across halves and rows are a
// level's exchange and selection in one).
__device__ __forceinline__ float wave_sum6(float a0, float a1, float a2, float a3, float a4, float a5) {
    const bool h3 = (threadIdx.x & 8) != 0;
    // sum of x in the lower half or even rows, of y in the others
    auto halve = [](auto m, float x, float y) {
        int a = __float_as_int(x), b = __float_as_int(y);
        lane_swap<decltype(m)::value>(a, b);
        return __int_as_float(a) + __int_as_float(b);
    };
    constexpr std::integral_constant<int, 32> half{};
    constexpr std::integral_constant<int, 16> row{};
    // level 32: lanes below 32 keep slots 0-3, the others slots 4-7
    const float y0 = halve(half, a0, a4), y1 = halve(half, a1, a5);
    const float y2 = halve(half, a2, 0.f), y3 = halve(half, a3, 0.f);
    // level 16: keep two of the four
    const float z0 = halve(row, y0, y2), z1 = halve(row, y1, y3);
    // level 8: keep one
    const int give = __float_as_int(h3 ? z0 : z1);
    float w = (h3 ? z1 : z0) + __int_as_float(row_xor_i<8>(give));
    w = xor_sum<4>(w);
    w = xor_sum<2>(w);
    return xor_sum<1>(w);
}

// Test the staged candidates cand[0, ce) against each particle of the cell:
// cand holds (x, y, z, index | type << 24) per candidate.  For particle q the
// 64 lanes first filter the candidates (the list test only, compacted in
// ballot order into the slot list accs); then, over the accepted ones only,
// every lane busy, they write q's list entries and evaluate its pair terms,
// instead of carrying both through the filter where most lanes of a
// 64-candidate batch hold rejected pairs.  Particles go two at a time: one
// read of each candidate serves both filters, whose ballot chains are
// independent, and the two pair passes share a loop; each keeps up to
// LL_IDXCAP / 2 accepted slots in its half of accs, and a particle with more
// is done again on its own with the whole of accs (same results: the slot
// lists and the sums do not depend on the pairing).
struct CellQ {           // particle q of the cell, wave-uniform
    int iq, tq, cnt0, nacc, nhalf;
    float rx, ry, rz;
};

template <int BASE, int CUT, int INTEG, bool EXCL>
__device__ __forceinline__ void cell_test(const DP &P, const StepInfo &I, const PairP *pp, const float4 *cand,
                                          unsigned short *accs, const int ce, const int np, const int myi,
                                          const float4 myr, int &mycount, int &myhalf, float q6[6],
                                          const unsigned micm) {
    const int lane = threadIdx.x & 63;
    const unsigned long long lt_mask = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const float L0 = INTEG == 4 ? I.L0 : P.box0, L1 = INTEG == 4 ? I.L1 : P.box1, L2 = INTEG == 4 ? I.L2 : P.box2;
    const float iL0 = INTEG == 4 ? I.iL0 : P.ibox0, iL1 = INTEG == 4 ? I.iL1 : P.ibox1,
                iL2 = INTEG == 4 ? I.iL2 : P.ibox2;
    const bool lap = P.compute_lap != 0;
    // the descriptor fields the filter needs, held in registers (the list
    // stores would otherwise make the compiler reload them every batch)
    const int N = P.N, tp = P.tp, tsh = P.tp_shift, maxnb = P.max_nbs;
    const bool niii = P.niii != 0;
    const bool nb16 = P.nb16 != 0;
    const float cps2 = P.cps2;
    GMEM int *const nbl = P.nbl;
    const size_t rs = (size_t)N * (size_t)tp;   // list row stride
    // q's values, read from lane q into scalar registers
    auto load_q = [&](int q) {
        CellQ c;
        c.iq = lane_i(myi, q);
        c.rx = lane_f(myr.x, q);
        c.ry = lane_f(myr.y, q);
        c.rz = lane_f(myr.z, q);
        c.tq = lane_i(__float_as_int(myr.w), q);
        c.cnt0 = lane_i(mycount, q);   // q's list entries before this pass
        c.nacc = 0;
        c.nhalf = 0;
        return c;
    };
    // the list test of candidate cj (slot k0 + lane) against q, appended to
    // q's slot list sl while it has room (cap); list minimum image only in
    // the dimensions mm where the cell's stencil wraps (exact for every pair
    // closer than L/2, and the stencil needs L >= 2.5 (rc + skin))
    auto test = [&](CellQ &c, unsigned short *sl, const int cap, const float4 cj, const int k0, const unsigned mm) {
        const int j = __float_as_int(cj.w) & 0xffffff;
        float dx, dy, dz;
        const float d2 = dist_sq_masked(cj.x, cj.y, cj.z, c.rx, c.ry, c.rz, L0, L1, L2, iL0, iL1, iL2, mm, dx, dy, dz);
        bool ok = (k0 + lane < ce) & (j != c.iq) & (d2 < cps2);
        if (EXCL) {
            if (ok) ok = !excluded(P, c.iq, j);
        }
        const unsigned long long mask = __ballot(ok);
        const int at = c.nacc + __popcll(mask & lt_mask);
        if (ok && at < cap) sl[at] = (unsigned short)(k0 + lane);
        c.nacc += __popcll(mask);
        if (niii) c.nhalf += __popcll(__ballot(ok && niii_owns(c.iq, j, N)));
    };
    // accepted candidate cj as list slot cnt0 + e of q, and its pair terms
    auto pair = [&](const CellQ &c, const float4 cj, const int e, float &fx, float &fy, float &fz, float &uu,
                    float &ww, float &ll) {
        const int slot = c.cnt0 + e;
        if (slot < maxnb) nbl_put(nbl + (size_t)c.iq * tp, slot, __float_as_int(cj.w) & 0xffffff, tsh, tp, rs, nb16);
        float dx, dy, dz;
        const float d2 = dist_sq_masked(cj.x, cj.y, cj.z, c.rx, c.ry, c.rz, L0, L1, L2, iL0, iL1, iL2, micm, dx, dy, dz);
        const PairP &qq = pp[c.tq * P.ntypes + (__float_as_int(cj.w) >> 24)];
        if (d2 < qq.cut2) {
            if (niii)
                pair_accum_w<BASE, CUT>(d2, dx, dy, dz, qq, fx, fy, fz, uu, ww, ll, lap,
                                        niii_owns(c.iq, __float_as_int(cj.w) & 0xffffff, N) ? 2.0f : 0.0f);
            else
                pair_accum<BASE, CUT>(d2, dx, dy, dz, qq, fx, fy, fz, uu, ww, ll, lap);
        }
    };
    // q's six sums over the wavefront, added to lane q's totals
    auto finish = [&](int q, const CellQ &c, float fx, float fy, float fz, float uu, float ww, float ll) {
        const int w = __float_as_int(wave_sum6(fx, fy, fz, uu, ww, ll));
        float t[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) t[k] = __int_as_float(__builtin_amdgcn_readlane(w, 8 * k));
        if (lane == q) {
            mycount = c.cnt0 + c.nacc;
            myhalf += c.nhalf;
#pragma unroll
            for (int k = 0; k < 6; ++k) q6[k] += t[k];
        }
    };
    // one particle with the whole of accs: the filter 128 candidates an
    // iteration (both reads issued before the first test; kk + 64 + lane <
    // LL_IDXCAP, so the reads stay inside the staging buffer; lanes past ce
    // are masked), in a form without the minimum image for cells whose
    // stencil does not wrap, then the pair pass over the accepted slots
    auto single = [&](int q) {
        CellQ c = load_q(q);
        auto filter = [&](auto nomic) {
            constexpr bool NM = decltype(nomic)::value;
            const unsigned mm = NM ? 0u : micm;
            for (int kk = 0; kk < ce; kk += 128) {
                const float4 c0 = cand[kk + lane];
                const float4 c1 = cand[kk + 64 + lane];
                test(c, accs, LL_IDXCAP, c0, kk, mm);
                if (kk + 64 < ce) test(c, accs, LL_IDXCAP, c1, kk + 64, mm);
            }
        };
        if (micm == 0u)
            filter(std::integral_constant<bool, true>{});
        else
            filter(std::integral_constant<bool, false>{});
        wave_sync_lds();
        float fx = 0.f, fy = 0.f, fz = 0.f, uu = 0.f, ww = 0.f, ll = 0.f;
        int anext = lane < c.nacc ? accs[lane] : 0;   // the next iteration's slot, read ahead
        for (int e = lane; e < c.nacc; e += 64) {
            const float4 cj = cand[anext];
            if (e + 64 < c.nacc) anext = accs[e + 64];
            pair(c, cj, e, fx, fy, fz, uu, ww, ll);
        }
        wave_sync_lds();   // accs is rewritten for the next particle
        finish(q, c, fx, fy, fz, uu, ww, ll);
    };
    int q = 0;
    for (; q + 1 < np; q += 2) {
        constexpr int HC = LL_IDXCAP / 2;   // slots of each half of accs
        unsigned short *sa = accs, *sb = accs + HC;
        CellQ a = load_q(q), b = load_q(q + 1);
        auto filter2 = [&](auto nomic) {
            constexpr bool NM = decltype(nomic)::value;
            const unsigned mm = NM ? 0u : micm;
            for (int kk = 0; kk < ce; kk += 128) {
                const float4 c0 = cand[kk + lane];
                const float4 c1 = cand[kk + 64 + lane];
                test(a, sa, HC, c0, kk, mm);
                test(b, sb, HC, c0, kk, mm);
                if (kk + 64 < ce) {
                    test(a, sa, HC, c1, kk + 64, mm);
                    test(b, sb, HC, c1, kk + 64, mm);
                }
            }
        };
        if (micm == 0u)
            filter2(std::integral_constant<bool, true>{});
        else
            filter2(std::integral_constant<bool, false>{});
        wave_sync_lds();
        // a particle whose slot list overflowed its half is done on its own below
        const bool oka = a.nacc <= HC, okb = b.nacc <= HC;
        const int na = oka ? a.nacc : 0, nbb = okb ? b.nacc : 0;
        float fxa = 0.f, fya = 0.f, fza = 0.f, uua = 0.f, wwa = 0.f, lla = 0.f;
        float fxb = 0.f, fyb = 0.f, fzb = 0.f, uub = 0.f, wwb = 0.f, llb = 0.f;
        for (int e = lane; e < max(na, nbb); e += 64) {
            const bool ea = e < na, eb = e < nbb;
            const float4 cja = cand[ea ? sa[e] : 0];
            const float4 cjb = cand[eb ? sb[e] : 0];
            if (ea) pair(a, cja, e, fxa, fya, fza, uua, wwa, lla);
            if (eb) pair(b, cjb, e, fxb, fyb, fzb, uub, wwb, llb);
        }
        wave_sync_lds();   // accs is rewritten for the next particles
        if (oka) finish(q, a, fxa, fya, fza, uua, wwa, lla);
        if (okb) finish(q + 1, b, fxb, fyb, fzb, uub, wwb, llb);
        if (!oka) single(q);
        if (!okb) single(q + 1);
    }
    if (q < np) single(q);
}

__device__ __forceinline__ void lds_sort_segment(int *a, int b, int e) {
    for (int x = b + 1; x < e; ++x) {
        int v = a[x], y = x - 1;
        while (y >= b && a[y] > v) {
            a[y + 1] = a[y];
            --y;
        }
        a[y + 1] = v;
    }
}

// stencil cell sc (0..124) of cell (cx, cy, cz): offsets in [-2, 2] and at
// least 5 cells per dimension, so each coordinate wraps at most once
__device__ __forceinline__ int stencil_cell(const DP &P, int cx, int cy, int cz, int sc) {
    const int ix = sc / 25 - 2, iy = (sc / 5) % 5 - 2, iz = sc % 5 - 2;
    int ox = cx + ix, oy = cy + iy, oz = cz + iz;
    ox += ox < 0 ? P.ncx : 0;
    ox -= ox >= P.ncx ? P.ncx : 0;
    oy += oy < 0 ? P.ncy : 0;
    oy -= oy >= P.ncy ? P.ncy : 0;
    oz += oz < 0 ? P.ncz : 0;
    oz -= oz >= P.ncz ? P.ncz : 0;
    return (ox * P.ncy + oy) * P.ncz + oz;
}

// stage the members of one stencil cell in LDS at dst (n <= ccap, rows of
// ccap >= 16 ints, 64-byte aligned), in index order.  Up to 8 members: read
// in two vector loads, put in order by a network of 19 compare-exchanges in
// registers (an insertion sort in LDS is a chain of some n^2/4 dependent LDS
// accesses).  A lane stores its own cell's slots only: the order of stores of
// different lanes to one slot is not the program's.  (KA N = 65536, cycles a
// wavefront of 4.8 cells spends here: 46400 -> 18400 of 200000.)
__device__ __forceinline__ void stage_cell_members(const GMEM int *row, int n, int *dst) {
    const GMEM int4 *r4 = (const GMEM int4 *)row;
    const int4 m0 = r4[0], m1 = r4[1];
    int v[8] = {m0.x, m0.y, m0.z, m0.w, m1.x, m1.y, m1.z, m1.w};
#pragma unroll
    for (int k = 1; k < 8; ++k) v[k] = k < n ? v[k] : 0x7fffffff;
    constexpr int ex[19][2] = {{0, 1}, {2, 3}, {4, 5}, {6, 7}, {0, 2}, {1, 3}, {4, 6}, {5, 7}, {1, 2}, {5, 6},
                               {0, 4}, {1, 5}, {2, 6}, {3, 7}, {2, 4}, {3, 5}, {1, 2}, {3, 4}, {5, 6}};
#pragma unroll
    for (int k = 0; k < 19; ++k) {
        const int lo = min(v[ex[k][0]], v[ex[k][1]]), hi = max(v[ex[k][0]], v[ex[k][1]]);
        v[ex[k][0]] = lo;
        v[ex[k][1]] = hi;
    }
#pragma unroll
    for (int k = 0; k < 8; ++k)
        if (k < n) dst[k] = v[k];
}

// the members of a fuller cell (more than 8): inserted one after another
__device__ __forceinline__ void stage_cell_more(const GMEM int *row, int n, int *dst) {
    const GMEM int4 *r4 = (const GMEM int4 *)row;
    for (int k = 0; k < n; k += 4) {
        const int4 m = r4[k >> 2];
        const int w[4] = {m.x, m.y, m.z, m.w};
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (k + t < n) dst[k + t] = w[t];
    }
    lds_sort_segment(dst, 0, n);
}

template <int BASE, int CUT, int INTEG>
__device__ __forceinline__ void step_ll_rebuild(const DP &P, const BlockCtx &B, const StepInfo &I, const PairP *pp, char *lds,
                                       float acc[GMD_NRED]) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int wpb = blockDim.x >> 6;
    // per wave: own[LL_OWNCAP] | cand[LL_IDXCAP] float4 | accs[LL_IDXCAP] u16; the sorted member
    // indices of a pass are staged at the start of cand, then overwritten by
    // the candidates themselves
    int *own = (int *)(lds + (size_t)wid * LL_WAVE_LDS);
    float4 *cand = (float4 *)(own + LL_OWNCAP);
    unsigned short *accs = (unsigned short *)(cand + LL_IDXCAP);
    int *idx = (int *)cand;
    cpos_t pos = I.cur ? P.pos1 : P.pos0;
    const GMEM int *ccount = P.ccount + (size_t)I.cbuf * P.ncells;
    const GMEM int *cmem = P.cmem + (size_t)I.cbuf * P.ncells * P.ccap;
    const int sb = lane + 64;
    // counts of all 125 stencil cells (lane owns stencil cells lane and
    // lane + 64) and the unsorted row of the cell itself (stencil cell 62);
    // the next cell's are requested before this cell is worked on
    struct CellHead {
        int nca, ncb, na, nb, ownm;
        unsigned micm;
    };
    // dimensions in which a cell's 5x5x5 stencil needs the minimum image:
    // unless it spans only cells 1 .. n-1 of that dimension without wrapping
    // (cell 0 may hold a particle at exactly +L/2) and 3 cells are less than
    // L/2, so every candidate pair lies within the box in the same image
    const int ncx_ = P.ncx, ncy_ = P.ncy, ncz_ = P.ncz;
    auto mic_mask = [&](int cx, int cy, int cz) {
        unsigned m = 0u;
        if (!(ncx_ >= 7 && cx >= 3 && cx <= ncx_ - 3)) m |= 1u;
        if (!(ncy_ >= 7 && cy >= 3 && cy <= ncy_ - 3)) m |= 2u;
        if (!(ncz_ >= 7 && cz >= 3 && cz <= ncz_ - 3)) m |= 4u;
        return m;
    };
    auto head = [&](int c, int cx, int cy, int cz, CellHead &h) {
        h.micm = mic_mask(cx, cy, cz);
        h.nca = stencil_cell(P, cx, cy, cz, lane);
        h.ncb = (sb < 125) ? stencil_cell(P, cx, cy, cz, sb) : 0;
        h.na = ccount[h.nca];
        h.nb = (sb < 125) ? ccount[h.ncb] : 0;
        h.ownm = (lane < P.ccap) ? cmem[(size_t)c * P.ccap + lane] : 0;
    };
    const int cstride = B.nb * wpb;
    const int ncz = P.ncz, ncy = P.ncy;
    const int c_first = __builtin_amdgcn_readfirstlane(B.bid * wpb + wid);
    const int stz = cstride % ncz, sty = (cstride / ncz) % ncy, stx = cstride / (ncz * ncy);
    int hz = c_first % ncz, hy = (c_first / ncz) % ncy, hx = c_first / (ncz * ncy);   // cell of the next head
    CellHead nxt;
    if (c_first < P.ncells) head(c_first, hx, hy, hz, nxt);
    for (int c = c_first; c < P.ncells; c += cstride) {
        const CellHead cur = nxt;
        hz += stz;
        hy += sty;
        hx += stx;
        if (hz >= ncz) {
            hz -= ncz;
            ++hy;
        }
        if (hy >= ncy) {
            hy -= ncy;
            ++hx;
        }
        if (c + cstride < P.ncells) head(c + cstride, hx, hy, hz, nxt);
        const int nca = cur.nca, ncb = cur.ncb, ownm = cur.ownm;
        const unsigned micm = I.wrapped ? __builtin_amdgcn_readfirstlane(cur.micm) : 7u;
        const int na = min(cur.na, P.ccap);
        const int nb = (sb < 125) ? min(cur.nb, P.ccap) : 0;
        const int np = lane_i(na, 62);
        if (np == 0) {
            if (I.ksplit && lane < P.ccap) P.kcell[(size_t)c * P.ccap + lane] = 0.f;
            continue;
        }
        // the cell's own particles in index order: lane q takes the q-th
        int rank = 0;
        for (int q = 0; q < np; ++q) rank += (lane_i(ownm, q) < ownm) ? 1 : 0;
        wave_sync_lds();
        if (lane < np) own[rank] = ownm;
        wave_sync_lds();
        const int myi = (lane < np) ? own[lane] : -1;
        float4 myr = make_float4(0.f, 0.f, 0.f, 0.f), myv = make_float4(0.f, 0.f, 0.f, 1.f);
        if (myi >= 0) {
            myr = pos[myi];
            myv = P.vel[myi];
        }
        // stencil-order offsets of every cell's members
        const int ia = wave_prefix(na);
        int ib = wave_prefix(nb);
        const int totA = lane_i(ia, 63);
        ib += totA;
        const int M = lane_i(ib, 63);
        const int offa = ia - na, offb = ib - nb;
        int mycount = 0, myhalf = 0;
        float q6[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        // passes over consecutive stencil cells holding at most LL_IDXCAP members
        // (a cell holds at most ccap <= LL_OWNCAP members, so every pass advances)
        for (int done = 0; done < M;) {
            const bool ina = offa >= done && ia - done <= LL_IDXCAP;
            const bool inb = sb < 125 && offb >= done && ib - done <= LL_IDXCAP;
            // the members up to the last cell of the pass: all of them as a
            // rule, else the largest prefix sum of its cells
            int pe = M;
            if (M - done > LL_IDXCAP) {
                pe = max(ina ? ia : done, inb ? ib : done);
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) pe = max(pe, __shfl_xor(pe, o, 64));
            }
            const int ce = pe - done;
            wave_sync_lds();
            if (ina && na > 0) stage_cell_members(cmem + (size_t)nca * P.ccap, na, idx + (offa - done));
            if (inb && nb > 0) stage_cell_members(cmem + (size_t)ncb * P.ccap, nb, idx + (offb - done));
            if (ina && na > 8) stage_cell_more(cmem + (size_t)nca * P.ccap, na, idx + (offa - done));
            if (inb && nb > 8) stage_cell_more(cmem + (size_t)ncb * P.ccap, nb, idx + (offb - done));
            wave_sync_lds();
            int jj[LL_PER];
#pragma unroll
            for (int u = 0; u < LL_PER; ++u) jj[u] = (lane + 64 * u < ce) ? idx[lane + 64 * u] : 0;
            wave_sync_lds();
            // the gathers in flight four at a time (an index past ce is 0, a
            // valid particle), then the LDS writes
#pragma unroll
            for (int u0 = 0; u0 < LL_PER; u0 += 4) {
                if (64 * u0 >= ce) break;
                float4 rg[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) rg[u] = pos[jj[u0 + u]];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int tag = jj[u0 + u] | (__float_as_int(rg[u].w) << 24);
                    if (lane + 64 * (u0 + u) < ce)
                        cand[lane + 64 * (u0 + u)] = make_float4(rg[u].x, rg[u].y, rg[u].z, __int_as_float(tag));
                }
            }
            wave_sync_lds();
            // exclusions in a variant of their own: the common case keeps its
            // filter free of the exclusion-row scan
            if (P.excl)
                cell_test<BASE, CUT, INTEG, true>(P, I, pp, cand, accs, ce, np, myi, myr, mycount, myhalf, q6, micm);
            else
                cell_test<BASE, CUT, INTEG, false>(P, I, pp, cand, accs, ce, np, myi, myr, mycount, myhalf, q6,
                                                   micm);
            done = pe;
        }
        if (I.ksplit) acc[RED_K] = 0.f;
        if (myi >= 0) {
            P.nbc[myi] = mycount;
            P.rref[myi] = myr;
            list_overflow(P, mycount, myhalf);
            if (P.boff)
                bond_terms(P, pos, myi, myr, INTEG == 4 ? I.L0 : P.box0, INTEG == 4 ? I.L1 : P.box1,
                           INTEG == 4 ? I.L2 : P.box2, q6[0], q6[1], q6[2], q6[3], q6[4], q6[5]);
            particle_finish<INTEG>(P, I, myi, myr, myv, myr, q6[0], q6[1], q6[2], q6[3] * 0.5f,
                                   q6[4] * (0.5f / 3.0f), q6[5], true, acc);
        }
        if (I.ksplit && lane < P.ccap) P.kcell[(size_t)c * P.ccap + lane] = acc[RED_K];
    }
}

// ---------------------------------------------------------------------------
// Rebuild step, N squared (nblist.py:89-143): PP particles per wavefront at a
// time, four or one (step_nsq_rebuild).  The block stages tiles of blockDim.x
// positions in LDS (two buffers, the next tile's load in flight during the
// current one: one block barrier a tile).  A wavefront reads 64 positions of
// the tile once and tests them against its particles, compacting each
// particle's accepted tile slots with a ballot; then every particle's 64 / PP
// lanes write its list entries (ascending j) and add its pair terms, the
// particles side by side.  The first lane of each group integrates its
// particle.
//
// The kernel is bound by the latency of each wavefront's chain (tile read,
// test, ballot, compaction): a system that takes the N-squared list leaves a
// SIMD one wavefront or less, so the particles of a wavefront are its only
// independent work, and one at a time left most of the chain exposed.
// Measured with one and with four at a time (and the rebuild in a kernel
// without the linked-list walk): a rebuild step of LJ N = 2048 (512
// wavefronts) 56.5 -> 33.6 us, of KA N = 4000 101 -> 57.6 us.  A wavefront
// then spends about 5100 cycles a tile on the tests and 2850 on the pairs,
// an instruction about every 10 cycles.
//
// The sums keep the order of a wavefront that gives each accepted pair of a
// tile the lane of its rank mod 64 and adds the lanes pairwise (32, 16, ...,
// 1 apart), for every PP: rank 16 k + l of one of four particles is added to
// its sum k in lane l of its group, and sums 0 + 2 and 1 + 3 are those two
// levels.
// ---------------------------------------------------------------------------
#define NSQ_PP 4                 // particles a wavefront takes at a time, at most
#define NSQ_CAP 256              // accepted slots of one particle and tile (a tile holds at most 256 positions)

template <int BASE, int CUT, int INTEG, int PP>
__device__ __forceinline__ void nsq_rebuild(const DP &P, const BlockCtx &B, const StepInfo &I, const PairP *pp,
                                            float4 *tiles, const int rounds, float acc[GMD_NRED]) {
    static_assert(PP == 4 || PP == 1, "lanes of a group: 16 or 64");
    constexpr int LPP = 64 / PP;   // lanes of a particle
    const int bd = blockDim.x;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, wpb = bd >> 6;
    const int g = lane / LPP, lp = lane & (LPP - 1);
    const float L0 = INTEG == 4 ? I.L0 : P.box0, L1 = INTEG == 4 ? I.L1 : P.box1, L2 = INTEG == 4 ? I.L2 : P.box2;
    cpos_t pos = I.cur ? P.pos1 : P.pos0;
    const bool lap = P.compute_lap != 0;
    const int N = P.N, maxnb = P.max_nbs;
    const bool niii = P.niii != 0, has_excl = P.excl != nullptr;
    const float cps2 = P.cps2;
    // held in registers (the list stores would otherwise make the compiler
    // read the descriptor again every tile)
    const int tp = P.tp, tsh = P.tp_shift;
    const bool nb16 = P.nb16 != 0;
    GMEM int *const nbl = P.nbl;
    const size_t rs = (size_t)N * (size_t)tp;
    const float iL0 = P.ibox0, iL1 = P.ibox1, iL2 = P.ibox2;
    // With every position in the box and the list radius below half of it,
    // the three-instruction image gives the same bits for every pair inside
    // the radius (mic_list differs from mic1 only where |d| is L/2 to within
    // a few ulp, and such a pair is outside)
    const float hmin = 0.5f * fminf(L0, fminf(L1, L2));
    const bool near = I.wrapped && cps2 < 0.9999f * (hmin * hmin);
    // this wave's accepted tile slots, NSQ_CAP a particle
    unsigned short *accs = (unsigned short *)(tiles + 2 * bd) + wid * (PP * NSQ_CAP);
    for (int rd = 0; rd < rounds; rd += PP) {
        // particle k of the wavefront: round rd + k, held by lanes LPP k and on
        const int iq = ((rd + g) * B.nb + B.bid) * wpb + wid;
        const bool mine = iq < N && rd + g < rounds;
        float4 rq = make_float4(0.f, 0.f, 0.f, 0.f), vq = make_float4(0.f, 0.f, 0.f, 1.f);
        if (mine) {
            rq = pos[iq];
            vq = P.vel[iq];
        }
        int ik[PP], cnt[PP], nhalf[PP];
        float xk[PP], yk[PP], zk[PP];
#pragma unroll
        for (int k = 0; k < PP; ++k) {
            // a round past the last, or an index past N, takes no pair
            ik[k] = lane_i(mine ? iq : -1, LPP * k);
            xk[k] = lane_f(rq.x, LPP * k);
            yk[k] = lane_f(rq.y, LPP * k);
            zk[k] = lane_f(rq.z, LPP * k);
            cnt[k] = 0;
            nhalf[k] = 0;
        }
        const PairP *ppi = pp + __float_as_int(rq.w) * P.ntypes;
        float fx[PP], fy[PP], fz[PP], uu[PP], ww[PP], ll[PP];
#pragma unroll
        for (int u = 0; u < PP; ++u) fx[u] = fy[u] = fz[u] = uu[u] = ww[u] = ll[u] = 0.f;
        auto rotate = [&]() {
            auto turn1 = [](float (&v)[PP]) {
                if constexpr (PP == 4) {
                    const float t = v[0];
                    v[0] = v[1];
                    v[1] = v[2];
                    v[2] = v[3];
                    v[3] = t;
                }
            };
            turn1(fx);
            turn1(fy);
            turn1(fz);
            turn1(uu);
            turn1(ww);
            turn1(ll);
        };
        // the value of the lane's own particle
        auto own = [&](const int (&v)[PP]) {
            if constexpr (PP == 4)
                return g == 0 ? v[0] : g == 1 ? v[1] : g == 2 ? v[2] : v[3];
            else
                return v[0];
        };
        int buf = 0;
        float4 nxt = pos[min((int)threadIdx.x, N - 1)];
        if (rd > 0) block_sync_lds();   // the last tiles of the previous round have been read
        for (int t0 = 0; t0 < N; t0 += bd) {
            float4 *tile = tiles + buf * bd;
            buf ^= 1;
            tile[threadIdx.x] = nxt;
            block_sync_lds();
            if (t0 + bd < N) nxt = pos[min(t0 + bd + (int)threadIdx.x, N - 1)];
            const int tn = min(bd, N - t0);
            // the list test of 64 positions against each particle.  PLAIN: a
            // full tile that holds none of the particles themselves, no
            // exclusions, no half lists
            int nacc[PP];
            bool plain = tn == bd && !has_excl && !niii;
#pragma unroll
            for (int k = 0; k < PP; ++k) {
                nacc[k] = 0;
                plain = plain && ik[k] >= 0 && (unsigned)(ik[k] - t0) >= (unsigned)bd;
            }
            float4 cj[4];   // the tile's positions (at most 256), read together
#pragma unroll
            for (int u = 0; u < 4; ++u) cj[u] = tile[64 * u < bd ? 64 * u + lane : lane];
            auto filter = [&](auto img, auto full) {
                constexpr bool NEAR = decltype(img)::value, PLAIN = decltype(full)::value;
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if (64 * u >= tn) break;   // the same for every lane
                    const int c0 = 64 * u, left = tn - c0;
                    // the distances of all the particles before the first
                    // compaction: independent chains
                    float d2[PP];
#pragma unroll
                    for (int k = 0; k < PP; ++k) {
                        float dx, dy, dz;
                        d2[k] = NEAR ? dist_sq_list(cj[u].x, cj[u].y, cj[u].z, xk[k], yk[k], zk[k], L0, L1, L2, iL0,
                                                    iL1, iL2, dx, dy, dz)
                                     : dist_sq_mic(cj[u].x, cj[u].y, cj[u].z, xk[k], yk[k], zk[k], L0, L1, L2, dx, dy,
                                                   dz);
                    }
#pragma unroll
                    for (int k = 0; k < PP; ++k) {
                        bool ok = d2[k] < cps2;
                        unsigned long long mask = __ballot(ok);
                        if (!PLAIN) {
                            mask &= left >= 64 ? ~0ull : (1ull << left) - 1ull;
                            const unsigned self = (unsigned)(ik[k] - (t0 + c0));   // the particle itself
                            if (self < 64u) mask &= ~(1ull << self);
                            if (ik[k] < 0) mask = 0ull;
                            ok = (mask >> lane) & 1ull;
                            if (has_excl) {
                                if (ok) ok = !excluded(P, ik[k], t0 + c0 + lane);
                                mask = __ballot(ok);
                            }
                            if (niii) nhalf[k] += __popcll(__ballot(ok && niii_owns(ik[k], t0 + c0 + lane, N)));
                        }
                        const int at = nacc[k] + __builtin_amdgcn_mbcnt_hi(
                                                     (unsigned)(mask >> 32),
                                                     __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
                        if (ok) accs[k * NSQ_CAP + at] = (unsigned short)(c0 + lane);
                        nacc[k] += __popcll(mask);
                    }
                }
            };
            if (near && plain)
                filter(std::integral_constant<bool, true>{}, std::integral_constant<bool, true>{});
            else if (near)
                filter(std::integral_constant<bool, true>{}, std::integral_constant<bool, false>{});
            else
                filter(std::integral_constant<bool, false>{}, std::integral_constant<bool, false>{});
            wave_sync_lds();
            // the accepted pairs of the tile, each particle on its lanes: list
            // entries (slots cnt + rank, tile order) and pair terms
            const int na = own(nacc), c_q = own(cnt);
            int amax = nacc[0];
            if constexpr (PP == 4) amax = max(max(nacc[0], nacc[1]), max(nacc[2], nacc[3]));
            const unsigned short *mya = accs + g * NSQ_CAP;
            auto pair = [&](const int a, float &ax, float &ay, float &az, float &au, float &aw, float &al) {
                if (a >= na) return;
                const int e = mya[a];
                const float4 rj = tile[e];
                const int slot = c_q + a;
                if (slot < maxnb) nbl_put(nbl + (size_t)iq * tp, slot, t0 + e, tsh, tp, rs, nb16);
                float dx, dy, dz;
                const float d2 = dist_sq_mic(rj.x, rj.y, rj.z, rq.x, rq.y, rq.z, L0, L1, L2, dx, dy, dz);
                const PairP &q = ppi[__float_as_int(rj.w)];
                if (!(d2 < q.cut2)) return;   // (a cut that is not a number has no pairs)
                if (niii)
                    pair_accum_w<BASE, CUT>(d2, dx, dy, dz, q, ax, ay, az, au, aw, al, lap,
                                            niii_owns(iq, t0 + e, N) ? 2.0f : 0.0f);
                else
                    pair_accum<BASE, CUT>(d2, dx, dy, dz, q, ax, ay, az, au, aw, al, lap);
            };
            // (the sums take turns by rotation, so the pair function is there
            // once: the families of the later bases are long)
            int turn = 0;
#pragma unroll 1
            for (int a0 = 0; a0 < amax; a0 += LPP, ++turn) {
                pair(a0 + lp, fx[0], fy[0], fz[0], uu[0], ww[0], ll[0]);
                rotate();
            }
#pragma unroll 1
            for (; turn & (PP - 1); ++turn) rotate();
#pragma unroll
            for (int k = 0; k < PP; ++k) cnt[k] += nacc[k];
            wave_sync_lds();   // accs is rewritten for the next tile
        }
        auto total = [&](const float (&v)[PP]) {
            float t;
            if constexpr (PP == 4)
                t = (v[0] + v[2]) + (v[1] + v[3]);
            else
                t = xor_sum<16>(xor_sum<32>(v[0]));
            t = xor_sum<8>(t);
            t = xor_sum<4>(t);
            t = xor_sum<2>(t);
            return xor_sum<1>(t);
        };
        float sx = total(fx), sy = total(fy), sz = total(fz), su = total(uu), sw = total(ww);
        float sl = lap ? total(ll) : 0.f;
        float part[GMD_NRED];
#pragma unroll
        for (int c = 0; c < GMD_NRED; ++c) part[c] = 0.f;
        if (mine) {
            const int n = own(cnt), nh = own(nhalf);
            if (lp == 0) {
                P.nbc[iq] = n;
                P.rref[iq] = rq;
                list_overflow(P, n, nh);
            }
            if (P.boff) bond_terms(P, pos, iq, rq, L0, L1, L2, sx, sy, sz, su, sw, sl);
            particle_finish<INTEG>(P, I, iq, rq, vq, rq, sx, sy, sz, su * 0.5f, sw * (0.5f / 3.0f), sl, lp == 0,
                                   part);
            if (I.ksplit && lp == 0) P.kcell[iq] = part[RED_K];
        }
        // the step's sums in lane 0, particle after particle
#pragma unroll
        for (int k = 0; k < PP; ++k)
#pragma unroll
            for (int c = 0; c < GMD_NRED; ++c) {
                const float v = lane_f(part[c], LPP * k);
                if (lane == 0) acc[c] += v;
            }
    }
}

// One particle at a time where a wavefront has no more than two, each with all
// lanes: the other slots of the four would be tested for nothing, and a
// particle's pairs take a quarter of the lanes.  Rebuild steps of LJ N = 2048
// at tp = 64, 32 and 16 (one, two and four particles): four at a time 35, 36
// and 32 us, one at a time 13, 19 and 49.
template <int BASE, int CUT, int INTEG>
__device__ __forceinline__ void step_nsq_rebuild(const DP &P, const BlockCtx &B, const StepInfo &I, const PairP *pp,
                                                 float4 *tiles, float acc[GMD_NRED]) {
    const int per_round = B.nb * (int)(blockDim.x >> 6);
    const int rounds = (P.N + per_round - 1) / per_round;
    if (rounds <= 2)
        nsq_rebuild<BASE, CUT, INTEG, 1>(P, B, I, pp, tiles, rounds, acc);
    else
        nsq_rebuild<BASE, CUT, INTEG, NSQ_PP>(P, B, I, pp, tiles, rounds, acc);
}

// linked lists: clear the cell buffer that step s+2 will fill
__device__ __forceinline__ void step_cells_clear(const DP &P, const BlockCtx &B, const StepInfo &I) {
    if (P.nblist_kind == 1 && I.integrate) {
        GMEM int *clr = P.ccount + (size_t)I.cbuf_clear * P.ncells;
        for (int c = B.bid * blockDim.x + threadIdx.x; c < P.ncells; c += B.nb * blockDim.x) clr[c] = 0;
    }
}

// One full step body (everything but the cross-block tail).  KIND: the list
// kind the kernel is for (0 N squared, 1 linked lists), or 2 for a kernel
// that runs replicas of either: a kernel that holds one rebuild only keeps
// its registers and its instructions
template <int BASE, int CUT, int INTEG, int KIND>
__device__ __forceinline__ void step_body(const DP &P, const BlockCtx &B, const StepInfo &I, const PairP *pp, char *build,
                                 float acc[GMD_NRED]) {
    if (I.rebuild) {
        if (KIND == 1 || (KIND == 2 && P.nblist_kind == 1))
            step_ll_rebuild<BASE, CUT, INTEG>(P, B, I, pp, build, acc);
        else
            step_nsq_rebuild<BASE, CUT, INTEG>(P, B, I, pp, (float4 *)build, acc);
    } else {
        step_lists<BASE, CUT, INTEG>(P, B, I, pp, acc);
    }
    step_cells_clear(P, B, I);
}

// The partial-sum components a step's tail reads: K for the thermostat (and
// with W the barostat), momentum and mass for the momentum reset, the
// saver's five sums.
__device__ __forceinline__ unsigned red_mask(bool ksum, bool mom, bool save, bool wsum) {
    unsigned m = 0u;
    if (ksum) m |= 1u << RED_K;
    if (wsum) m |= 1u << RED_W;
    if (mom) m |= (7u << RED_PX) | (1u << RED_M);
    if (save) m |= (1u << RED_U) | (1u << RED_W) | (1u << RED_LAP) | (1u << RED_K) | (1u << RED_FSQ);
    return m;
}

// Block-level reduction of the per-thread sums of the components in 'mask'
// into part[block] (fixed order).
__device__ __forceinline__ void block_partials(const DP &P, const BlockCtx &B, float acc[GMD_NRED], double *red,
                                               GMEM float *part, unsigned mask) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
    for (int c = 0; c < GMD_NRED; ++c) {
        if (!((mask >> c) & 1u)) continue;
        float v = wave_sum_f(acc[c]);
        if (lane == 0) red[wid * GMD_NRED + c] = (double)v;
    }
    __syncthreads();
    if (threadIdx.x < GMD_NRED && ((mask >> threadIdx.x) & 1u)) {
        double sum = 0.0;
        for (int w = 0; w < nw; ++w) sum += red[w * GMD_NRED + threadIdx.x];
        part[(size_t)threadIdx.x * P.pstride + B.bid] = (float)sum;
    }
    __syncthreads();
}

// A thread's first four per-block partials (blocks t, t+256, t+512, t+768)
// of the components in 'mask', loaded together: one memory round trip for a
// grid of up to 1024 blocks.  CM: the components the caller may ask for (a
// compile-time set, so the registers of the others are not allocated).
#define RED_PRE 4
#define RED_ALL ((1u << GMD_NRED) - 1u)
template <unsigned CM = RED_ALL>
__device__ __forceinline__ void load_partials(const DP &P, const GMEM float *part, const int nblocks, unsigned mask,
                                              float v[RED_PRE][GMD_NRED]) {
#pragma unroll
    for (int u = 0; u < RED_PRE; ++u) {
        const int b = threadIdx.x + u * blockDim.x;
#pragma unroll
        for (int c = 0; c < GMD_NRED; ++c)
            if ((CM >> c) & 1u) v[u][c] = (((mask >> c) & 1u) && b < nblocks) ? part[(size_t)c * P.pstride + b] : 0.f;
    }
}

// Sum of the per-block partials of the components in 'mask' over nblocks
// blocks, in a fixed order (thread t: blocks t, t+256, ... in double; then
// the wavefronts in index order): tot[c] in the threads that 'all' names
// (every thread, or thread 0 only).  Every caller with the same data gets
// the same bits.  v holds what load_partials returned.
template <unsigned CM = RED_ALL>
__device__ __forceinline__ void sum_partials(const DP &P, const GMEM float *part, const int nblocks, unsigned mask,
                                             bool all, double *red, const float v[RED_PRE][GMD_NRED],
                                             double tot[GMD_NRED]) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = blockDim.x >> 6;
    mask &= CM;
    if (mask) {
        double acc[GMD_NRED];
#pragma unroll
        for (int c = 0; c < GMD_NRED; ++c) acc[c] = 0.0;
#pragma unroll
        for (int u = 0; u < RED_PRE; ++u)
#pragma unroll
            for (int c = 0; c < GMD_NRED; ++c)
                if ((CM >> c) & 1u) acc[c] += (double)v[u][c];
        for (int b = threadIdx.x + RED_PRE * blockDim.x; b < nblocks; b += blockDim.x) {
#pragma unroll
            for (int c = 0; c < GMD_NRED; ++c)
                if (((CM >> c) & 1u) && ((mask >> c) & 1u)) acc[c] += (double)part[(size_t)c * P.pstride + b];
        }
#pragma unroll
        for (int c = 0; c < GMD_NRED; ++c) {
            if (!((CM >> c) & 1u) || !((mask >> c) & 1u)) continue;
            double x = wave_sum_d(acc[c]);
            if (lane == 0) red[wid * GMD_NRED + c] = x;
        }
    }
    __syncthreads();
    if (all || threadIdx.x == 0) {
#pragma unroll
        for (int c = 0; c < GMD_NRED; ++c) {
            tot[c] = 0.0;
            if (((CM >> c) & 1u) && ((mask >> c) & 1u))
                for (int w = 0; w < nw; ++w) tot[c] += red[w * GMD_NRED + c];
        }
    }
    __syncthreads();
}

// NVT.py:226-237: the thermostat variable after a step with kinetic sum ksum.
__device__ __forceinline__ float thermostat_next(const DP &P, float xi, float ksum, float t0, int s) {
    const double t = (double)t0 + (double)s * (double)P.dt;
    const double T = target_temperature(P, t);
    const double dev = (double)(2.0f * ksum) / (P.degrees * T) - 1.0;
    const double inc = (double)(P.dt * P.omega2) * dev;
    return (float)((double)xi + inc);
}

// scalar_saver.py:374-408 output row of step s; vol: the volume of the box
// after the step (the saver runs after the integrator, which may scale it)
__device__ __forceinline__ void saver_row(const DP &P, int s, const double tot[GMD_NRED], const float vol) {
    GMEM float *row = P.saver_out + (size_t)(s / P.save_every) * 6;
    row[0] = (float)tot[RED_U];
    row[1] = (float)tot[RED_W];
    row[2] = (float)tot[RED_LAP];
    row[3] = (float)tot[RED_K];
    row[4] = (float)tot[RED_FSQ];
    row[5] = vol;
}

// the context's box volume (volume_function, orthorhombic.py), float32
__device__ __forceinline__ float box_volume(const DP &P) { return P.box0 * P.box1 * P.box2; }

// NPT_Atomic: publish the state of step s (block 0, one thread) and flag a
// box that has become too small for the linked-list cell grid
__device__ __forceinline__ void npt_publish(const DP &P, const StepInfo &J, int s) {
    GMEM Ctrl *C = P.ctrl;
    GMEM float *st = C->npt[s & 1];
    st[0] = J.np_t0;
    st[1] = J.np_b0;
    st[2] = J.np_vol;
    st[3] = J.L0;
    st[4] = J.L1;
    st[5] = J.L2;
    if (P.nblist_kind == 1 && (J.L0 < P.cell_min * (float)P.ncx || J.L1 < P.cell_min * (float)P.ncy ||
                               J.L2 < P.cell_min * (float)P.ncz))
        C->npt_grid_bad = 1;
}

// The tail of a step of the persistent driver, executed by its last block:
// final sums over all blocks, then the one-thread updates of the reference
// (NVT.py:226-237 thermostat, momentum_reset.py:166-186 shift,
// scalar_saver.py:374-408 output row; NPT_Atomic.py:148-187).
__device__ inline void step_tail(const DP &P, const StepInfo &I, double *red, const int nblocks) {
    GMEM Ctrl *C = P.ctrl;
    const unsigned mask = red_mask(I.need_ksum, I.need_mom, I.need_save, I.need_wsum);
    float v[RED_PRE][GMD_NRED];
    load_partials(P, P.partial, nblocks, mask, v);
    double tot[GMD_NRED];
    sum_partials(P, P.partial, nblocks, mask, false, red, v, tot);
    if (threadIdx.x == 0) {
        float vol = box_volume(P);
        if (I.need_wsum) {
            // NPT_Atomic: the state of the next step
            StepInfo J = I;
            npt_advance(P, J, (float)tot[RED_K], (float)tot[RED_W], (double)I.t0 + (double)I.s * (double)P.dt);
            npt_publish(P, J, I.s + 1);
            vol = J.L0 * J.L1 * J.L2;
        } else if (I.need_ksum) {
            C->xi = thermostat_next(P, I.xi, (float)tot[RED_K], I.t0, I.s);
            C->ksum = 0.0f;
        }
        if (I.need_mom) {
            const float mt = (float)tot[RED_M];
            C->shift[0] = (float)tot[RED_PX] / mt;
            C->shift[1] = (float)tot[RED_PX + 1] / mt;
            C->shift[2] = (float)tot[RED_PX + 2] / mt;
            C->shift_step = I.s + 1;
        }
        if (I.need_save) saver_row(P, I.s, tot, vol);
        if (I.rebuild) C->nbflag[2] += 1;
    }
    __syncthreads();
}

// The tail of step q = I.s - 1 folded into step I.s (kernel-per-step path of
// one system): every block sums step q's partials (buffer q & 1) itself, in
// the order step_tail uses, so all blocks hold the same thermostat variable
// and momentum shift, bit for bit, without a separate one-block launch and
// its round trips through memory.  Block 0 publishes what the host reads
// (thermostat state, pending shift, saver row of step q).
// folded_tail_mask names the components step q's tail needs;
// folded_tail_load issues their loads (before the pair table is staged, so
// the two overlap); folded_tail finishes.  CM as in load_partials.
template <int INTEG>
__device__ __forceinline__ unsigned folded_tail_mask(const DP &P, const StepInfo &I) {
    if (I.s == 0) return 0u;
    const int q = I.s - 1;   // q < nsteps: step q integrated
    const bool integ_q = INTEG != 0;
    return red_mask(integ_q && (INTEG == 2 || INTEG == 4), integ_q && P.mom_every > 0 && (q % P.mom_every) == 0,
                    integ_q && P.save_every > 0 && (q % P.save_every) == 0 && (q / P.save_every) < P.saves_per_block,
                    integ_q && INTEG == 4);
}

template <int INTEG, unsigned CM>
__device__ __forceinline__ void folded_tail_load(const DP &P, const StepInfo &I, unsigned mask,
                                                 float v[RED_PRE][GMD_NRED]) {
    if (I.s > 0) {
        const int q = I.s - 1;
        load_partials<CM>(P, P.partial + (size_t)(q & 1) * GMD_NRED * P.pstride, P.step_grid, mask, v);
    }
}

template <int INTEG, unsigned CM>
__device__ __forceinline__ void folded_tail(const DP &P, const BlockCtx &B, StepInfo &I, double *red, unsigned mask,
                                            const float v[RED_PRE][GMD_NRED]) {
    GMEM Ctrl *C = P.ctrl;
    const bool pub = B.bid == 0 && threadIdx.x == 0;
    if (I.s == 0) {
        // xi of step 0 is the run's starting state; no shift is pending
        I.apply_shift = false;
        if (pub) C->xib[0] = I.xi;
        return;
    }
    const int q = I.s - 1;
    const bool ksum_q = (mask >> RED_K) & 1u && INTEG == 2;
    const bool mom_q = (mask >> RED_M) & 1u;
    const bool save_q = (mask >> RED_FSQ) & 1u;
    const float xi_q = C->xib[q & 1];
    double tot[GMD_NRED];
    sum_partials<CM>(P, P.partial + (size_t)(q & 1) * GMD_NRED * P.pstride, P.step_grid, mask, true, red, v, tot);
    // the same value in every lane: kept in scalar registers over the step
    I.xi = uniform_f(ksum_q ? thermostat_next(P, xi_q, (float)tot[RED_K], I.t0, q) : xi_q);
    I.apply_shift = mom_q;
    if (mom_q) {
        const float mt = (float)tot[RED_M];
        I.sh0 = uniform_f((float)tot[RED_PX] / mt);
        I.sh1 = uniform_f((float)tot[RED_PX + 1] / mt);
        I.sh2 = uniform_f((float)tot[RED_PX + 2] / mt);
    }
    if (INTEG == 4) {
        // step_info loaded the state of step q: advance it to this step's
        npt_advance(P, I, (float)tot[RED_K], (float)tot[RED_W], (double)I.t0 + (double)q * (double)P.dt);
        npt_coeffs(P, I);
        npt_uniform(I);
    }
    if (pub) {
        if (INTEG == 4) npt_publish(P, I, I.s);
        C->xib[I.s & 1] = I.xi;
        C->xi = I.xi;
        if (ksum_q) C->ksum = 0.0f;
        if (mom_q) {
            C->shift[0] = I.sh0;
            C->shift[1] = I.sh1;
            C->shift[2] = I.sh2;
            C->shift_step = I.s;
        }
        if (save_q) saver_row(P, q, tot, INTEG == 4 ? I.L0 * I.L1 * I.L2 : box_volume(P));
    }
}

// Software grid barrier for the cooperative (co-resident) launch.  The last
// block to arrive runs the tail before releasing the others.
template <typename Tail>
__device__ inline void grid_barrier(GMEM Ctrl *C, const int nb, Tail tail) {
    __shared__ int s_last;
    __shared__ unsigned s_gen;
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned gen = __hip_atomic_load(gen_ptr(&C->bar_gen), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // release this block's writes, acquire everybody's when last
        const unsigned arrived =
            __hip_atomic_fetch_add(gen_ptr(&C->bar_count), 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        s_last = (arrived == (unsigned)nb - 1u);
        s_gen = gen;
    }
    __syncthreads();
    if (s_last) {
        tail();
        __syncthreads();
        if (threadIdx.x == 0) {
            __hip_atomic_store(gen_ptr(&C->bar_count), 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(gen_ptr(&C->bar_gen), s_gen + 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
        }
    } else if (threadIdx.x == 0) {
        // spin without invalidating caches; one acquire fence once released
        while (__hip_atomic_load(gen_ptr(&C->bar_gen), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == s_gen)
            __builtin_amdgcn_s_sleep(1);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    __syncthreads();
}
