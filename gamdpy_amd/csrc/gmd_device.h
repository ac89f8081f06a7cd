// gmd_device.h -- device-side building blocks shared by the MD kernels.
//
// State layout in HBM (one context = one system of N particles):
//   pos[2]  float4 (x, y, z, type bits)      ping-pong: step s reads pos[buf0^(s&1)]
//   vel     float4 (vx, vy, vz, mass)
//   frc     float4 (fx, fy, fz, 0)
//   sc      float  [5][N]  U, W, lapU, K, Fsq   (column-major, coalesced)
//   rim     int    [3][N]  image counters (touched only when a particle wraps)
//   rref    float4 positions at the last neighbour-list rebuild
//   nbl     neighbour list; entry k of particle i is local entry m = k/tp of
//           lane t = k%tp.  N <= 65536: 16-bit indices, entries m and m+1
//           (m even) in the low and high halves of word ((m/2)*N + i)*tp + t;
//           otherwise 32-bit indices, entry m in word (m*N + i)*tp + t
//   nbc     int    neighbour count (true count; entries beyond max_nbs are dropped)
//   perm    int    internal index -> caller's index; the particles are renumbered
//                  in cell order at run starts (gather locality), every array
//                  above is in internal order and the C ABI converts on upload /
//                  download
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define GMD_NRED 10   // per-block partial sums: K U W lap Fsq px py pz m (unused)
#define RED_K 0
#define RED_U 1
#define RED_W 2
#define RED_LAP 3
#define RED_FSQ 4
#define RED_PX 5
#define RED_M 8

#define SC_U 0
#define SC_W 1
#define SC_LAP 2
#define SC_K 3
#define SC_FSQ 4

#define MAX_TYPES 8

// Pointers into device memory are declared in the global address space in
// device code, so the compiler emits global_load/store rather than flat ones.
#if defined(__HIP_DEVICE_COMPILE__)
#define GMEM __attribute__((address_space(1)))
#else
#define GMEM
#endif

// Control block kept in device memory for the lifetime of a context.
struct Ctrl {
    float xi, ksum;            // NVT thermostat_state (NVT.py:143)
    float shift[3];            // pending momentum-reset shift (momentum_reset.py:186)
    int shift_step;            // step at which the pending shift is applied (-1 = none)
    int nbflag[3];             // nblist.py:9 [update pending, overflow, #rebuilds]
    unsigned red_count;        // last-block counter (kernel-per-phase path)
    unsigned bar_count;        // grid barrier arrival counter
    unsigned bar_gen;          // grid barrier generation
    int nsteps;
    int buf0;                  // position buffer holding r at step 0 of the run
    float t0;
    int cell_overflow;         // largest cell occupancy seen beyond the cell capacity
    long long lstep0;          // Langevin counter of step 0 of the run
    float xib[2];              // xi used by step s at xib[s & 1] (folded-tail path)
    int s_base;                // step of launch argument k = 0 (folded-tail path)
    int unwrapped;             // some position of the run's start lies outside [-L/2, L/2]
    // NPT_Atomic state of step s at npt[s & 1]: thermostat rate p_xi/Q,
    // barostat rate p_eps/W, volume, box lengths (NPT_Atomic.py:38-39; the
    // accumulators of each step are the step's K and W sums)
    float npt[2][6];
    int npt_grid_bad;          // the box shrank below the cell grid's smallest admissible cell
};

// Per-type-pair constants, prepared in LDS at kernel start.
//   LJ sigma/epsilon: a = sigma^2, b = 4 eps, c = 24 eps
//   LJ 12-6:          a = A12, b = A6, c = 12 A12, d = 6 A6
//   IPL_n:            a = A_n, c = n A_n, e0 = n
//   LJ_m_n:           a = A_m, b = A_n, c = m A_m, d = n A_n, e0 = m, e1 = n
//   harmonic:         a = eps, b = sigma
//   hertzian:         a = eps, b = sigma, e0 = alpha
// The first four fields are what the force-only list loop of the LJ forms
// needs (one 16-byte LDS read per pair).
struct PairP {
    float a, c, cut2, d;
    float b, ucut, scut, cut;
    float e0, e1;
    int kind, pad;
    // functions read from parameter rows (kind 6 SAAP, 7 a sum of two terms):
    // the row before the cut, and per term its function, first parameter and
    // exponents (t2 < 0: one term)
    float p[8];
    int t1, t2, o1, o2;
    float x1a, x1b, x2a, x2b;
};

// Pointers into LDS, declared in the local address space in device code so
// their arithmetic is 32-bit
#if defined(__HIP_DEVICE_COMPILE__)
#define LDSMEM __attribute__((address_space(3)))
#else
#define LDSMEM
#endif

struct DP {
    int N, ntypes, tp, tp_shift, max_nbs;   // max_nbs: list slots per particle
    int nblist_kind;
    int niii;                  // compute_plan['UtilizeNIII']: the full list is kept, and each pair's
                               // U, W, lapU go to the particle whose half list holds it
    int max_half;              // NIII: the caller's max_nbs, the limit on that half list
    float box0, box1, box2;
    float ibox0, ibox1, ibox2;   // 1 / box lengths
    int nrows;                 // rows of the neighbour list (entries per lane of a particle)
    int nb16;                  // 16-bit list entries, two rows a word (N <= 65536)
    int nwrows;                // rows of words: nrows / 2 with nb16, else nrows
    float mic_edge0, mic_edge1, mic_edge2;   // |x_d| beyond which a listed pair may need the minimum image
    float cps2;                // fl32(max_cut + skin)^2 (nblist.py:119)
    float skin2q;              // skin*skin*0.25 (orthorhombic.py:131)
    GMEM float4 *pos0, *pos1, *vel, *frc, *rref, *obeta;
    GMEM float *sc;
    GMEM int *rim;
    GMEM int *nbl, *nbc;
    // cell grid (linked lists): three buffers, step s reads buffer s%3
    int ncx, ncy, ncz, ncells, ccap;
    GMEM int *ccount;          // [3][ncells]
    GMEM int *cmem;            // [3][ncells*ccap]
    const GMEM int *excl;
    int excl_cols;
    // bonds (bonds.py): each bond listed under both its ends, boff[i] ..
    // boff[i + 1] - 1 the entries of particle i as (partner, bond type);
    // harmonic (r0, k) per bond type; boff == nullptr: no bonds
    const GMEM int *boff;
    const GMEM int2 *bnd;
    const GMEM float2 *bpar;
    const GMEM float *raw_params;   // ntypes*ntypes rows of nparams (3: p0, p1, cut)
    GMEM PairP *ptab;          // the prepared pair table (k_pair_table), copied to LDS by every block
    int nparams;
    int nterms, term_kind[2], term_first[2];
    float term_exps[4];
    int pair_base, cutoff;
    float pexp0, pexp1;        // exponents fixed by the pair function (IPL n; LJ_m_n m, n; hertzian alpha)
    // integrator
    float dt, omega2, alpha;
    double degrees;
    unsigned long long seed;
    int tfunc;
    float tpar0, tpar1, tpar2, tpar3;
    // NPT_Atomic (NPT_Atomic.py:45-56): thermostat and barostat masses
    // without their temperature factor, pressure schedule
    int npt;
    float mass_t, mass_p;
    int pfunc;
    float ppar0, ppar1, ppar2, ppar3;
    float cell_min;            // (max_cut + skin) / 2: smallest cell of a valid linked-list grid
    int compute_u, compute_w, compute_lap, compute_k, compute_fsq;
    int mom_every, save_every, saves_per_block;
    int conf_saves;            // ConfigurationSaver saves per block (0 = off)
    GMEM float *conf_out;      // [conf_saves][2][N][3]: r and r_im (float32), caller's numbering
    GMEM Ctrl *ctrl;
    GMEM float *partial;       // [GMD_NRED][pstride]: sum c of block b at c * pstride + b
    int pstride;
    GMEM int *rebuild_flag;    // [nsteps+2]
    GMEM float *saver_out;     // [saves_per_block][6]
    int lds_pp, lds_red, lds_build;   // byte offsets into dynamic LDS
    int step_grid;             // blocks of the step kernel (partial sums to reduce)
    int rebuild_grid;          // replicas of a batch: blocks of a split rebuild step (step_once)
    // the kinetic energies of such a step, [ncells][ccap] or [N] for N-squared
    // lists; null: a rebuild whose kinetic sum is wanted is not split (it is set
    // where rebuild_grid exceeds step_grid and the integrator is NVT)
    GMEM float *kcell;
    const GMEM int *perm;      // internal index -> index in the caller's order (particles are kept in cell order)
    // the host's arrays: a packed copy of them in device memory (xdev) and in
    // pinned host memory (xhost), the words of each array one after another
    // (XferSeg), and the run's control block and saver rows as the host reads
    // them (pub, pinned)
    GMEM int *xdev;
    int *xhost, *pub;
    int nscal, sid_u, sid_w, sid_lap, sid_k, sid_fsq, sid_m;   // scalar columns of the host's rows (-1: none)
};

// The host arrays as segments of a packed buffer of 4-byte words: r, v, f
// (N, 3), scalars (N, nscal), types (N), images (N, 3)
enum { XF_R = 1, XF_V = 2, XF_F = 4, XF_S = 8, XF_T = 16, XF_IM = 32, XF_ALL = 63 };
struct XferSeg {
    size_t r, v, f, s, t, im, end;
    __host__ __device__ XferSeg(size_t N, size_t ns)
        : r(0), v(3 * N), f(6 * N), s(9 * N), t((9 + ns) * N), im((10 + ns) * N), end((13 + ns) * N) {}
};

// ---------------------------------------------------------------------------
// Orthorhombic box (simulation_boxes/orthorhombic.py:43-132).  The exact
// float32 operation order matters for neighbour sets and histogram bins, so
// contraction into FMA is switched off here.
// ---------------------------------------------------------------------------
// Reference rule: d -= L if 2d > L, d += L if 2d < -L.  Doubling is exact,
// so this is |d| > L/2 -> d - copysign(L, d): the same result bit for bit,
// in four instructions (L/2 is loop-invariant).
__device__ __forceinline__ float mic1(float d, float L) {
#pragma clang fp contract(off)
    return (fabsf(d) > 0.5f * L) ? d - copysignf(L, d) : d;
}

// Minimum image of a list pair: d - L rint(d / L), exact (the product L k is
// exact for k in {-1, 0, 1}, so the fma rounds once, as mic1's subtraction
// does).  It equals mic1 bit for bit except within a few ulp of |d| = L/2,
// where both images are equally near; three instructions instead of five.
__device__ __forceinline__ float mic_list(float d, float L, float invL) {
    return fmaf(-L, __builtin_rintf(d * invL), d);
}

__device__ __forceinline__ float dist_sq_list(float ax, float ay, float az, float bx, float by, float bz, float L0,
                                              float L1, float L2, float iL0, float iL1, float iL2, float &dx,
                                              float &dy, float &dz) {
#pragma clang fp contract(off)
    dx = mic_list(ax - bx, L0, iL0);
    dy = mic_list(ay - by, L1, iL1);
    dz = mic_list(az - bz, L2, iL2);
    float d2 = dx * dx;
    d2 = d2 + dy * dy;
    d2 = d2 + dz * dz;
    return d2;
}

// dist_sq_list where the minimum image is taken only in the dimensions whose
// bit is set in mic (a uniform mask): in the others every pair lies within
// the box in the same image, fl(a - b) is its own minimum image, and the
// result equals dist_sq_list's bit for bit.
__device__ __forceinline__ float dist_sq_masked(float ax, float ay, float az, float bx, float by, float bz,
                                                float L0, float L1, float L2, float iL0, float iL1, float iL2,
                                                unsigned mic, float &dx, float &dy, float &dz) {
#pragma clang fp contract(off)
    dx = ax - bx;
    dy = ay - by;
    dz = az - bz;
    if (mic & 1u) dx = mic_list(dx, L0, iL0);
    if (mic & 2u) dy = mic_list(dy, L1, iL1);
    if (mic & 4u) dz = mic_list(dz, L2, iL2);
    float d2 = dx * dx;
    d2 = d2 + dy * dy;
    d2 = d2 + dz * dz;
    return d2;
}

__device__ __forceinline__ float dist_sq_mic(float ax, float ay, float az, float bx, float by, float bz,
                                             float L0, float L1, float L2, float &dx, float &dy, float &dz) {
#pragma clang fp contract(off)
    dx = mic1(ax - bx, L0);
    dy = mic1(ay - by, L1);
    dz = mic1(az - bz, L2);
    float d2 = dx * dx;
    d2 = d2 + dy * dy;
    d2 = d2 + dz * dz;
    return d2;
}

// ---------------------------------------------------------------------------
// Pair functions in the reference's float32 operation order
// (LJ_12_6_sigma_epsilon.py:25-36, LJ_12_6.py:34-41), used for the cutoff
// constants u(rc), s(rc) so they equal the oracle's bit for bit.
// ---------------------------------------------------------------------------
// r^-n for n > 0: by multiplication when n is a whole number up to 32, else
// exp2(-n log2 r)
__device__ __forceinline__ float inv_pow(float inv_r, float n) {
    const int k = (int)n;
    if ((float)k == n && k >= 0 && k <= 32) {
        float p = 1.0f, x = inv_r;
        for (int e = k; e > 0; e >>= 1) {
            if (e & 1) p *= x;
            x *= x;
        }
        return p;
    }
    return exp2f(n * log2f(inv_r));
}

// x^a for x >= 0, a > 0 (hertzian): exp2(a log2 x), 0 at x = 0
__device__ __forceinline__ float pos_pow(float x, float a) {
    return x > 0.0f ? exp2f(a * log2f(x)) : 0.0f;
}

// The pair functions of the family kind 2..5 at distance dist
// (make_IPL_n.py:26-34, make_LJ_m_n.py:24-35, harmonic_repulsion.py:22-33,
// hertzian.py:24-37); e0, e1 = the function's exponents.
__device__ inline void pair_family(int kind, float dist, float p0, float p1, float e0, float e1, float &u, float &s,
                                   float &umm) {
    const float inv = 1.0f / dist;
    if (kind == 2) {            // u = A r^-n
        const float pn = inv_pow(inv, e0), pn2 = pn * inv * inv;
        u = p0 * pn;
        s = e0 * p0 * pn2;
        umm = (e0 * (e0 + 1.0f)) * p0 * pn2;
    } else if (kind == 3) {     // u = A_m r^-m + A_n r^-n
        const float pm = inv_pow(inv, e0), pn = inv_pow(inv, e1), i2 = inv * inv;
        u = p0 * pm + p1 * pn;
        s = e0 * p0 * pm * i2 + e1 * p1 * pn * i2;
        umm = (e0 * (e0 + 1.0f)) * p0 * pm * i2 + (e1 * (e1 + 1.0f)) * p1 * pn * i2;
    } else if (kind == 4) {     // u = eps (1 - r/sigma)^2 / 2
        const float is = 1.0f / p1, delta = 1.0f - dist * is;
        u = 0.5f * p0 * delta * delta;
        s = p0 * delta * is / dist;
        umm = p0 * is * is;
    } else {                    // u = eps (1 - r/sigma)^alpha
        const float is = 1.0f / p1, delta = 1.0f - dist * is;
        u = p0 * pos_pow(delta, e0);
        s = p0 * e0 * pos_pow(delta, e0 - 1.0f) * is / dist;
        umm = p0 * e0 * (e0 - 1.0f) * pos_pow(delta, e0 - 2.0f) * is * is;
    }
}

// SAAP.py:4-84: u(x = r/sigma) = eps (a0 e^{a1 x}/x + a2 e^{a3 x} + a4) / D,
// D = 1 + a5 x^6; p = a0..a5, sigma, eps.  s = -u'(r)/r and u''(r) from
// the quotient rule in x, then the chain rule for r = sigma x.
__device__ __noinline__ void pair_saap(float dist, const float *p, float &u, float &s, float &umm) {
#pragma clang fp contract(off)
    const float a0 = p[0], a1 = p[1], a2 = p[2], a3 = p[3], a4 = p[4], a5 = p[5], sigma = p[6], eps = p[7];
    const float x = dist / sigma;
    const float e1 = expf(a1 * x), e3 = expf(a3 * x);
    const float ix = 1.0f / x;
    const float g = a0 * e1 * ix + a2 * e3 + a4;
    const float dg = a0 * e1 * (a1 * ix - ix * ix) + a2 * a3 * e3;
    const float ddg = a0 * e1 * (a1 * a1 * ix - 2.0f * a1 * ix * ix + 2.0f * ix * ix * ix) + a2 * a3 * a3 * e3;
    const float x2 = x * x, x4 = x2 * x2;
    const float den = 1.0f + a5 * x4 * x2;
    const float dden = 6.0f * a5 * x4 * x;
    const float ddden = 30.0f * a5 * x4;
    const float iden = 1.0f / den;
    u = eps * g * iden;
    const float du = eps * (dg - g * dden * iden) * iden;
    const float d2u = eps * (ddg - (2.0f * dg * dden + g * ddden) * iden + 2.0f * g * dden * dden * iden * iden) * iden;
    s = -du / (x * sigma * sigma);
    umm = d2u / (sigma * sigma);
}

__device__ inline void pair_ref(int base, float dist, float p0, float p1, float &u, float &s, float &umm,
                                float e0 = 0.f, float e1 = 0.f);

// One term of a function read from a parameter row: the pair function kind
// (GMD_* 0..6) with its parameters from p on; hertzian reads eps, alpha,
// sigma, SAAP a0..a5, sigma, eps.
__device__ inline void pair_term(int kind, float dist, const float *p, float e0, float e1, float &u, float &s,
                                 float &umm) {
    if (kind == 6)
        pair_saap(dist, p, u, s, umm);
    else if (kind == 5)
        pair_family(5, dist, p[0], p[2], p[1], 0.0f, u, s, umm);
    else
        pair_ref(kind, dist, p[0], p[1], u, s, umm, e0, e1);
}

// add_potential_functions.py:24-30: u1 + u2, s1 + s2, u''1 + u''2.  Not
// inlined: the row functions are a rare path, and inlining them into every
// step-kernel instance multiplies the build time.
__device__ __noinline__ void pair_rows(const PairP &q, float dist, float &u, float &s, float &umm) {
    pair_term(q.t1, dist, q.p + q.o1, q.x1a, q.x1b, u, s, umm);
    if (q.t2 >= 0) {
        float u2, s2, umm2;
        pair_term(q.t2, dist, q.p + q.o2, q.x2a, q.x2b, u2, s2, umm2);
        u = u + u2;
        s = s + s2;
        umm = umm + umm2;
    }
}

__device__ inline void pair_ref(int base, float dist, float p0, float p1, float &u, float &s, float &umm,
                                float e0, float e1) {
#pragma clang fp contract(off)
    if (base >= 2) {
        pair_family(base, dist, p0, p1, e0, e1, u, s, umm);
    } else if (base == 0) {
        float od = 1.0f / dist;
        float x = p0 * od;
        float x2 = x * x;
        float x6 = x2 * x2 * x2;
        float x12 = x6 * x6;
        float od2 = od * od;
        u = (4.0f * p1) * (x12 - x6);
        s = ((24.0f * p1) * (2.0f * x12 - x6)) * od2;
        umm = ((24.0f * p1) * (26.0f * x12 - 7.0f * x6)) * od2;
    } else {
        float inv = 1.0f / dist;
        float p2 = inv * inv;
        float p6 = p2 * p2 * p2;
        float p12 = p6 * p6;
        float p8 = p6 * p2;
        float p14 = p12 * p2;
        u = p0 * p12 + p1 * p6;
        s = (12.0f * p0) * p14 + (6.0f * p1) * p8;
        umm = (156.0f * p0) * p14 + (42.0f * p1) * p8;
    }
}

// The pair table entry of a function read from a parameter row (kinds 6, 7):
// row = the nparams - 1 parameters before the cut; the cutoff constants from
// the same evaluation as the force loop's
__device__ inline void make_pairp_rows(int base, int cutoff, const float *row, int nrow, float cut, const int tk[2],
                                       const int tf[2], const float tx[4], int nterms, PairP &q) {
    q.kind = base;
    q.a = q.b = q.c = q.d = 0.0f;
    q.e0 = q.e1 = 0.0f;
    q.pad = 0;
    for (int k = 0; k < 8; ++k) q.p[k] = k < nrow ? row[k] : 0.0f;
    q.t1 = tk[0];
    q.o1 = tf[0];
    q.x1a = tx[0];
    q.x1b = tx[1];
    q.t2 = nterms > 1 ? tk[1] : -1;
    q.o2 = nterms > 1 ? tf[1] : 0;
    q.x2a = tx[2];
    q.x2b = tx[3];
    q.cut = cut;
    {
#pragma clang fp contract(off)
        q.cut2 = cut * cut;
    }
    float u, s, umm;
    pair_rows(q, cut, u, s, umm);
    q.ucut = (cutoff == 0) ? 0.0f : u;
    q.scut = (cutoff == 2) ? s : 0.0f;
}

__device__ inline void make_pairp(int base, int cutoff, float p0, float p1, float cut, PairP &q, float e0 = 0.f,
                                  float e1 = 0.f) {
    q.kind = base;
    q.e0 = e0;
    q.e1 = e1;
    q.pad = 0;
    for (int k = 0; k < 8; ++k) q.p[k] = 0.0f;
    q.t1 = q.t2 = -1;
    q.o1 = q.o2 = 0;
    q.x1a = q.x1b = q.x2a = q.x2b = 0.0f;
    if (base == 2) {
        q.a = p0;
        q.b = 0.0f;
        q.c = e0 * p0;
        q.d = 0.0f;
    } else if (base == 3) {
        q.a = p0;
        q.b = p1;
        q.c = e0 * p0;
        q.d = e1 * p1;
    } else if (base >= 4) {
        q.a = p0;
        q.b = p1;
        q.c = 0.0f;
        q.d = 0.0f;
    } else if (base == 0) {
        q.a = p0 * p0;
        q.b = 4.0f * p1;
        q.c = 24.0f * p1;
        q.d = 0.0f;
    } else {
        q.a = p0;
        q.b = p1;
        q.c = 12.0f * p0;
        q.d = 6.0f * p1;
    }
    q.cut = cut;
    {
#pragma clang fp contract(off)
        q.cut2 = cut * cut;
    }
    float u, s, umm;
    pair_ref(base, cut, p0, p1, u, s, umm, e0, e1);
    q.ucut = (cutoff == 0) ? 0.0f : u;
    q.scut = (cutoff == 2) ? s : 0.0f;
}

// Fast evaluation inside the force loop: from d2 directly, one reciprocal.
template <int BASE, int CUT>
__device__ __forceinline__ void pair_fast(float d2, const PairP &q, float &u, float &s, float &umm, bool lap) {
    float ir2 = __builtin_amdgcn_rcpf(d2);
    umm = 0.f;
    if (BASE == 2) {
        // the family IPL_n / LJ_m_n / harmonic / hertzian: a uniform switch on
        // the kind (one per PairPotential), evaluated from the distance
        const float dist = d2 * __builtin_amdgcn_rsqf(d2);
        pair_family(q.kind, dist, q.a, q.b, q.e0, q.e1, u, s, umm);
        if (!lap) umm = 0.f;
    } else if (BASE == 3) {
        // functions read from parameter rows (SAAP, sums of two terms): a
        // call, kept out of the family's instance so that instance needs no
        // registers saved around it
        const float dist = d2 * __builtin_amdgcn_rsqf(d2);
        pair_rows(q, dist, u, s, umm);
        if (!lap) umm = 0.f;
    } else if (BASE == 0) {
        float x2 = q.a * ir2;
        float x6 = x2 * x2 * x2;
        float x12 = x6 * x6;
        u = q.b * (x12 - x6);
        s = q.c * (2.0f * x12 - x6) * ir2;
        if (lap) umm = q.c * (26.0f * x12 - 7.0f * x6) * ir2;
    } else {
        float p6 = ir2 * ir2 * ir2;
        float p12 = p6 * p6;
        u = q.a * p12 + q.b * p6;
        s = (q.c * p12 + q.d * p6) * ir2;
        if (lap) umm = (13.0f * q.c * p12 + 7.0f * q.d * p6) * ir2;
    }
    if (CUT == 1) {
        u = u - q.ucut;
    } else if (CUT == 2) {
        float r = d2 * __builtin_amdgcn_rsqf(d2);
        u = u - (q.ucut - q.scut * q.cut * (r - q.cut));
        s = s - q.scut;
    }
}

// ---------------------------------------------------------------------------
// Counter-based normal variates: Philox-4x32-10 (Salmon et al., SC'11) and
// the Box-Muller transform.  counter = (id, step lo, step hi, 0).
// ---------------------------------------------------------------------------
__device__ __forceinline__ void philox4x32_10(uint32_t c[4], uint32_t k0, uint32_t k1) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        uint64_t p0 = (uint64_t)0xD2511F53u * c[0];
        uint64_t p1 = (uint64_t)0xCD9E8D57u * c[2];
        uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0;
        uint32_t hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
        uint32_t n0 = hi1 ^ c[1] ^ k0;
        uint32_t n2 = hi0 ^ c[3] ^ k1;
        c[0] = n0;
        c[1] = lo1;
        c[2] = n2;
        c[3] = lo0;
        if (r < 9) {
            k0 += 0x9E3779B9u;
            k1 += 0xBB67AE85u;
        }
    }
}

__device__ __forceinline__ void normal3(unsigned long long seed, long long step, int id, float &z0, float &z1,
                                        float &z2) {
    uint32_t c[4] = {(uint32_t)id, (uint32_t)((unsigned long long)step & 0xFFFFFFFFull),
                     (uint32_t)((unsigned long long)step >> 32), 0u};
    philox4x32_10(c, (uint32_t)(seed & 0xFFFFFFFFull), (uint32_t)(seed >> 32));
    const float inv24 = 5.9604644775390625e-08f;  // 2^-24
    float u0 = (float)((c[0] >> 8) + 1u) * inv24;
    float u1 = (float)((c[1] >> 8) + 1u) * inv24;
    float u2 = (float)((c[2] >> 8) + 1u) * inv24;
    float u3 = (float)((c[3] >> 8) + 1u) * inv24;
    const float two_pi = 6.283185307179586f;
    float r0 = sqrtf(-2.0f * logf(u0));
    float r1 = sqrtf(-2.0f * logf(u2));
    float sn, cs;
    sincosf(two_pi * u1, &sn, &cs);
    z0 = r0 * cs;
    z1 = r0 * sn;
    z2 = r1 * cosf(two_pi * u3);
}

// ---------------------------------------------------------------------------
// Reductions.  The cross-lane exchanges are data-parallel moves (DPP) inside a
// row of 16 lanes and gfx950's row and half swaps across rows: a vector
// instruction each, where a shuffle goes through the LDS crossbar and waits
// some 120 cycles for it.  A reduction is a chain of up to six of them, and
// the end of every step is such chains: a step (rebuilds included) of KA
// N = 4000 14.25 -> 13.70 us, of N = 65536 26.8 -> 25.8 us, of LJ N = 10976
// in NPT 18.2 -> 17.5 us.  Sums pair the lanes 32, 16, 8, 4, 2, 1 apart
// (a + b = b + a: every lane holds the same bits).
// ---------------------------------------------------------------------------
// v of lane (lane ^ M) for M = 1, 2, 4, 8 (within a row of 16 lanes)
template <int M>
__device__ __forceinline__ int row_xor_i(int v) {
    static_assert(M == 1 || M == 2 || M == 4 || M == 8, "lanes of one row");
    if (M == 1) return __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, true);    // quad_perm [1,0,3,2]
    if (M == 2) return __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xf, 0xf, true);    // quad_perm [2,3,0,1]
    if (M == 8) return __builtin_amdgcn_update_dpp(0, v, 0x128, 0xf, 0xf, true);   // row_ror:8
    // 4 = 7 ^ 3: row_half_mirror, then quad_perm [3,2,1,0]
    const int h = __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, true);
    return __builtin_amdgcn_update_dpp(0, h, 0x1B, 0xf, 0xf, true);
}

// a and b with a's upper half (M = 32) or odd rows (M = 16) and b's lower
// half or even rows exchanged
template <int M>
__device__ __forceinline__ void lane_swap(int &a, int &b) {
    static_assert(M == 16 || M == 32, "rows or halves");
    if (M == 32) {
        const auto r = __builtin_amdgcn_permlane32_swap((unsigned)a, (unsigned)b, false, false);
        a = (int)r[0];
        b = (int)r[1];
    } else {
        const auto r = __builtin_amdgcn_permlane16_swap((unsigned)a, (unsigned)b, false, false);
        a = (int)r[0];
        b = (int)r[1];
    }
}

// v + (v of lane ^ M)
template <int M>
__device__ __forceinline__ float xor_sum(float v) {
    if constexpr (M >= 16) {
        int a = __float_as_int(v), b = a;
        lane_swap<M>(a, b);
        return __int_as_float(a) + __int_as_float(b);
    } else {
        return v + __int_as_float(row_xor_i<M>(__float_as_int(v)));
    }
}

template <int M>
__device__ __forceinline__ double xor_sum(double v) {
    const unsigned long long bits = (unsigned long long)__double_as_longlong(v);
    int lo = (int)bits, hi = (int)(bits >> 32);
    auto join = [](int l, int h) {
        return __longlong_as_double((long long)(((unsigned long long)(unsigned)h << 32) | (unsigned)l));
    };
    if constexpr (M >= 16) {
        int lo2 = lo, hi2 = hi;
        lane_swap<M>(lo, lo2);
        lane_swap<M>(hi, hi2);
        return join(lo, hi) + join(lo2, hi2);
    } else {
        return v + join(row_xor_i<M>(lo), row_xor_i<M>(hi));
    }
}

// sum over the lanes that differ in the bits below n (a power of two, the
// same for every lane): pairs 1, 2, 4, ... lanes apart
__device__ __forceinline__ float group_sum(float v, int n) {
    if (n > 1) v = xor_sum<1>(v);
    if (n > 2) v = xor_sum<2>(v);
    if (n > 4) v = xor_sum<4>(v);
    if (n > 8) v = xor_sum<8>(v);
    if (n > 16) v = xor_sum<16>(v);
    if (n > 32) v = xor_sum<32>(v);
    return v;
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
    v = xor_sum<32>(v);
    v = xor_sum<16>(v);
    v = xor_sum<8>(v);
    v = xor_sum<4>(v);
    v = xor_sum<2>(v);
    return xor_sum<1>(v);
}

__device__ __forceinline__ float wave_sum_f(float v) { return wave_sum(v); }

__device__ __forceinline__ double wave_sum_d(double v) { return wave_sum(v); }

// inclusive prefix sum over the wavefront: within rows by shifts, then the
// row totals carried to the rows above
__device__ __forceinline__ int wave_prefix(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);   // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);   // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);   // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);   // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   // row_bcast:15 into rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);   // row_bcast:31 into rows 2 and 3
    return v;
}

// Schedules of misc/make_function.py (temperature, pressure), evaluated in
// float64 like numba does once the time (float32 + int64*float32) has become
// float64.
__device__ inline double schedule_value(int kind, float p0, float p1, float p2, float p3, double t) {
    if (kind == 0) return (double)p0;
    if (kind == 1) {  // ramp(value0, x0, value1, x1)
        double v0 = p0, x0 = p1, v1 = p2, x1 = p3;
        float alpha = (p2 - p0) / (p3 - p1);
        if (t < x0) return v0;
        if (t < x1) return v0 + (t - x0) * (double)alpha;
        return v1;
    }
    // sin(period, amplitude, offset)
    double period = p0, amp = p1, off = p2;
    return off + amp * sin(2.0 * 3.141592653589793 * t / period);
}

__device__ inline double target_temperature(const DP &P, double t) {
    return schedule_value(P.tfunc, P.tpar0, P.tpar1, P.tpar2, P.tpar3, t);
}

__device__ inline double target_pressure(const DP &P, double t) {
    return schedule_value(P.pfunc, P.ppar0, P.ppar1, P.ppar2, P.ppar3, t);
}
