// gmd_adjoint.h -- differentiable NVE trajectory: float32 forward whose
// positions stay in memory (or checkpoints of them), hand-written adjoint
// (force Jacobian-vector products and gradients with respect to the per-type
// LJ sigma / epsilon), and a Gaussian-smoothed partial radial distribution as
// the observable.
//
// Included once into gmd_core.hip (shares its error channel and helpers).
//
// Model: LJ_12_6_sigma_epsilon with the shifted-force cutoff as gamdpy
// defines it (apply_shifted_force_cutoff.py:29-37: s(r) - s(rc)), at a cut
// held fixed while sigma and epsilon vary; leap-frog NVE as NVE.py:59-105
// (v += f/m dt; r += v dt; wrap).
//
// Forward, for n = 0 .. S-1 (state x_n = (r_n, v_{n-1/2})):
//   F_n = F(r_n),  v_{n+1/2} = v_{n-1/2} + F_n/m dt,  r_{n+1} = r_n + v_{n+1/2} dt
// Observable: H[c][k] = sum over frames n (n % rdf_every == 0) and unordered
// pairs of class c of K(d_ij - r_k), K(x) = max(0, exp(-x^2/2w^2) - exp(-12.5))
// for |x| < 5w, r_k = (k + 1/2) rmax / bins.
// Adjoint (lambda_r = dL/dr_n, lambda_v = dL/dv_{n-1/2}), n = S-1 .. 0:
//   lambda_v <- lambda_v + dt lambda_r(n+1);  w = dt/m lambda_v
//   lambda_r(n) = lambda_r(n+1) + J(r_n) w + dL/dr_n|frame
//   dL/dtheta  += w . dF(r_n)/dtheta
// with J = dF/dr symmetric: (J w)_i = sum_j A_ij (w_i - w_j) + B_ij d_ij (d_ij . (w_i - w_j)),
// A = s(r), B = (ds/dr)/r, d_ij = r_i - r_j (minimum image).
//
// The force and J w sums run over neighbour lists (radius max cut + skin, N
// squared build, rebuilt when a particle has moved more than skin/2 and every
// ckpt_every steps, so a segment recomputed from its checkpoint repeats the
// forward bit for bit and both layouts give the same bits); the observable and its
// gradient run over a list of radius rmax + 5 w built afresh (no skin) at
// each frame, one frame every rdf_every steps.
//
// A step of either pass is ONE kernel: the rebuild of the lists of a block's
// own particles where the last step's skin check asks for it (in a launch of
// its own for large systems), the sums, the update of the particle and the skin
// check of its next positions.  The systems are small (a step of N = 4096 is
// some microseconds of work spread over the device), so a step is bound by its
// launches and by the latency of each lane's chain of list entry, neighbour and
// pair term; the separate check, build, sum and update kernels of a step were
// three to four launches, most of the builds finding nothing to do.  Forward
// and backward pass of KA N = 4096, 200 steps: 11.7 ms with them apart, 7.5
// with one kernel a step, 5.9 with the trajectory kept, 5.65 with builds that
// test boxes only where that saves something (N = 500, 40 steps: 2.1, 1.2, 0.95
// and 0.96 ms); a forward step is 5.3 us, a backward step 9.3, a rebuild inside
// one 31 us more.
#pragma once

#define ADJ_MAX_TYPES 3
#define ADJ_MAX_CLS 6            // ADJ_MAX_TYPES (ADJ_MAX_TYPES + 1) / 2
#define ADJ_MAX_BINS 512
#define ADJ_SKIN 0.5f             // neighbour-list skin of the force and J w sums

struct AdjPairC {                // one ordered type pair
    float sig, sig2, eps, eps24; // sigma, sigma^2, epsilon, 24 epsilon
    float cut2, sc, dsc_dsig;    // cut^2, s(rc), ds(rc)/dsigma at fixed rc
    int cls;                     // unordered class index
};

struct AdjK {
    int N, nt, ncls;
    float L0, L1, L2;
    float dt;
    // neighbour lists of the force and J w sums
    float cps2;                  // (max cut + skin)^2
    float skin2q;                // (skin / 2)^2
    int maxnb;                   // list slots per particle (row-major [i][slot])
    int tp, tpsh;                // lanes per particle of the list sums
    int boxes;                   // the builds of those lists test chunks by their boxes first (adj_boxes)
    AdjPairC pc[ADJ_MAX_TYPES * ADJ_MAX_TYPES];
    // observable
    int bins;
    float rmax, dr, wid, inv_w2, kfloor, rcut2;   // rcut = rmax + 5 w
    float hup;                   // fixed point of the frame histograms: units of 2^-32 / hup (adj_weight_scale)
};

__device__ __forceinline__ int adj_type(float4 r) { return __float_as_int(r.w); }

// s(r) - s(rc) of the LJ pair function, and the pieces the adjoint needs
struct AdjPairEval {
    float s, B, ds_deps, ds_dsig;
};

__device__ __forceinline__ AdjPairEval adj_pair(const AdjPairC &q, float d2) {
    const float inv_r2 = 1.0f / d2;
    const float x = q.sig2 * inv_r2;
    const float x3 = x * x * x;
    const float x6 = x3 * x3;
    AdjPairEval e;
    const float s_lj = q.eps24 * (2.0f * x6 - x3) * inv_r2;
    e.s = s_lj - q.sc;
    e.B = q.eps24 * (8.0f * x3 - 28.0f * x6) * inv_r2 * inv_r2;
    e.ds_deps = e.s / q.eps;
    e.ds_dsig = (q.eps24 / q.sig) * (24.0f * x6 - 6.0f * x3) * inv_r2 - q.dsc_dsig;
    return e;
}

// the pair constants of a kernel's arguments into LDS (an index that differs
// between lanes would otherwise be a load from the argument segment per pair);
// the caller synchronises the block
__device__ __forceinline__ void adj_stage_pairs(const AdjK &K, AdjPairC *pc) {
    const int n = K.nt * K.nt * (int)(sizeof(AdjPairC) / 4);
    if ((int)threadIdx.x < n) ((int *)pc)[threadIdx.x] = ((const int *)K.pc)[threadIdx.x];
}

// smallest (MAXI: largest) value over the wavefront, in every lane
template <bool MAXI>
__device__ __forceinline__ float wave_extreme(float v) {
    auto pick = [](float a, float b) { return MAXI ? fmaxf(a, b) : fminf(a, b); };
    int a = __float_as_int(v), b = a;
    lane_swap<32>(a, b);
    v = pick(__int_as_float(a), __int_as_float(b));
    a = b = __float_as_int(v);
    lane_swap<16>(a, b);
    v = pick(__int_as_float(a), __int_as_float(b));
    v = pick(v, __int_as_float(row_xor_i<8>(__float_as_int(v))));
    v = pick(v, __int_as_float(row_xor_i<4>(__float_as_int(v))));
    v = pick(v, __int_as_float(row_xor_i<2>(__float_as_int(v))));
    return pick(v, __int_as_float(row_xor_i<1>(__float_as_int(v))));
}

// centre and half extents (with a rounding margin) of the box around a
// wavefront's positions
__device__ __forceinline__ void wave_box(const float4 r, float4 &c, float4 &h) {
    const float x0 = wave_extreme<false>(r.x), x1 = wave_extreme<true>(r.x);
    const float y0 = wave_extreme<false>(r.y), y1 = wave_extreme<true>(r.y);
    const float z0 = wave_extreme<false>(r.z), z1 = wave_extreme<true>(r.z);
    c = make_float4(0.5f * (x0 + x1), 0.5f * (y0 + y1), 0.5f * (z0 + z1), 0.f);
    h = make_float4(0.5001f * (x1 - x0) + 1e-3f, 0.5001f * (y1 - y0) + 1e-3f, 0.5001f * (z1 - z0) + 1e-3f, 0.f);
}

// whether some position of a box (centre c, half extents h) may be within
// sqrt(r2) of r in some image: the distance to the centre's nearest image less
// the half extent bounds the distance to every position from below (4e-7 L
// and the last factor cover the rounding of positions, centre and difference)
__device__ __forceinline__ bool box_near(const AdjK &K, const float4 r, const float4 c, const float4 h, float r2) {
    auto gap = [](float d, float L, float e) {
        return fmaxf(0.f, fabsf(d - L * __builtin_rintf(d * __builtin_amdgcn_rcpf(L))) - fmaf(L, 4e-7f, e));
    };
    const float x = gap(r.x - c.x, K.L0, h.x), y = gap(r.y - c.y, K.L1, h.y), z = gap(r.z - c.z, K.L2, h.z);
    return x * x + y * y + z * z <= 1.0001f * r2;
}

// N-squared list build of radius^2 r2 into nbl (maxnb slots a particle): one
// wavefront per particle, 16 a block, the block's tiles of ADJ_BT positions
// staged in LDS, the accepted j compacted with a ballot (ascending j; HALF:
// each pair in one of its particles' lists, evenly, as niii_owns says); rref
// (if given) receives the positions and *over records the longest list beyond
// maxnb (HALF: the longest there would be with every j, so that a system whose
// gradient needs longer lists than there is room for is refused by the forward
// pass already).  The tests are most of the work, so a tile comes with the boxes of
// its chunks of 64 positions (a wavefront each) and a particle tests only the
// chunks whose box is near it, where the numbering keeps chunks together
// (boxes; adj_boxes).  Without, a chunk that has no neighbour is one test and
// a branch.  The particle itself and the slots past the last are taken out of
// the wavefront's mask, not tested per lane.  when (if given): build only if
// that flag is set.
#define ADJ_BT 1024   // threads of a build block, positions of its tile
template <bool HALF>
__global__ void __launch_bounds__(ADJ_BT) k_adj_build(AdjK K, const float4 *pos_p, float4 *rref_p, int *nbl_p,
                                                      int *nbc_p, int maxnb, float r2, int boxes, const int *when,
                                                      int *over) {
    if (when && *when == 0) return;
    __shared__ float4 tile[ADJ_BT], box_c[ADJ_BT / 64], box_h[ADJ_BT / 64];
    cpos_t pos = (cpos_t)pos_p;
    GMEM int *nbl = (GMEM int *)nbl_p;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int i = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (ADJ_BT / 64)) + wid);
    const bool valid = i < K.N;
    float4 ri = make_float4(0.f, 0.f, 0.f, 0.f);
    if (valid) ri = pos[i];
    int cnt = 0, all = 0;
    float4 nxt = pos[min((int)threadIdx.x, K.N - 1)];
    for (int t0 = 0; t0 < K.N; t0 += ADJ_BT) {
        float4 bc, bh;
        if (boxes) wave_box(nxt, bc, bh);   // (a slot past the last holds the last position)
        if (t0 > 0) __syncthreads();
        tile[threadIdx.x] = nxt;
        if (boxes && lane == 0) {
            box_c[wid] = bc;
            box_h[wid] = bh;
        }
        __syncthreads();
        if (t0 + ADJ_BT < K.N) nxt = pos[min(t0 + ADJ_BT + (int)threadIdx.x, K.N - 1)];
        if (!valid) continue;
        const int tn = min(ADJ_BT, K.N - t0);
        // PLAIN: 64 positions, none of them the particle's own
        auto chunk = [&](const int c0, auto whole) {
            constexpr bool PLAIN = decltype(whole)::value;
            const float4 rj = tile[c0 + lane];
            float dx, dy, dz;
            const float d2 = dist_sq_mic(ri.x, ri.y, ri.z, rj.x, rj.y, rj.z, K.L0, K.L1, K.L2, dx, dy, dz);
            unsigned long long m = __ballot(d2 < r2);
            if (!PLAIN) {
                if (tn - c0 < 64) m &= (1ull << (tn - c0)) - 1ull;
                const unsigned self = (unsigned)(i - t0 - c0);   // the particle's own lane of these 64
                if (self < 64u) m &= ~(1ull << self);
            }
            if (m == 0ull) return;
            if (HALF) {
                all += __popcll(m);
                m &= __ballot(niii_owns(i, t0 + c0 + lane, K.N));
            }
            const int slot = cnt + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                             __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
            if (__builtin_amdgcn_inverse_ballot_w64(m) && slot < maxnb) nbl[(size_t)i * maxnb + slot] = t0 + c0 + lane;
            cnt += __popcll(m);
        };
        if (boxes) {
            unsigned long long live =
                __ballot(lane < (tn + 63) / 64 && box_near(K, ri, box_c[lane & 15], box_h[lane & 15], r2));
            while (live) {
                chunk(64 * __builtin_ctzll(live), std::integral_constant<bool, false>{});
                live &= live - 1;
            }
        } else if (tn == ADJ_BT && (unsigned)(i - t0) >= (unsigned)ADJ_BT) {
#pragma unroll 4
            for (int c0 = 0; c0 < ADJ_BT; c0 += 64) chunk(c0, std::integral_constant<bool, true>{});
        } else {
            for (int c0 = 0; c0 < tn; c0 += 64) chunk(c0, std::integral_constant<bool, false>{});
        }
    }
    if (!HALF) all = cnt;
    if (valid && lane == 0) {
        nbc_p[i] = cnt;
        if (rref_p) rref_p[i] = ri;
        if (all > maxnb) atomicMax(over, all);
    }
}

// The same list for the particles of one block of a step kernel (256 threads,
// 256 / tp particles), rebuilt in place when the skin check asked for it: rare
// enough (a list lasts some ten steps) that the block's few wavefronts may take
// longer than k_adj_build would, as long as the build is short.  From
// ADJ_APART_N particles on the launch of its own before every step costs less.
// Forward + backward, in place and apart, 40 steps: in lattice order N = 4000
// (100 steps) 2362 and 2510 us, 8000 1604 and 1560, 16384 3406 and 3060; in no
// order 4000 2691 and 2899, 8000 2060 and 2064, 16384 5532 and 4550.
__device__ __forceinline__ void adj_relist(const AdjK &K, cpos_t pos, GMEM float4 *rref, GMEM int *nbl, GMEM int *nbc,
                                        GMEM int *over) {
    __shared__ float4 tile[256], own[64], box_c[4], box_h[4];
    __shared__ int count[64];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int np = 256 >> K.tpsh, i0 = (int)blockIdx.x * np;   // tp >= 4: at most 64
    if ((int)threadIdx.x < np) {
        count[threadIdx.x] = 0;
        own[threadIdx.x] = pos[min(i0 + (int)threadIdx.x, K.N - 1)];
    }
    float4 nxt = pos[min((int)threadIdx.x, K.N - 1)];
    for (int t0 = 0; t0 < K.N; t0 += 256) {
        float4 bc, bh;
        if (K.boxes) wave_box(nxt, bc, bh);
        __syncthreads();
        tile[threadIdx.x] = nxt;
        if (K.boxes && lane == 0) {
            box_c[wid] = bc;
            box_h[wid] = bh;
        }
        __syncthreads();
        if (t0 + 256 < K.N) nxt = pos[min(t0 + 256 + (int)threadIdx.x, K.N - 1)];
        const int tn = min(256, K.N - t0);
        for (int p = wid; p < np; p += 4) {
            const int i = __builtin_amdgcn_readfirstlane(i0 + p);
            if (i >= K.N) break;
            const float4 ri = own[p];
            int cnt = count[p];
            auto chunk = [&](const int c0) {
                const float4 rj = tile[c0 + lane];
                float dx, dy, dz;
                const float d2 = dist_sq_mic(ri.x, ri.y, ri.z, rj.x, rj.y, rj.z, K.L0, K.L1, K.L2, dx, dy, dz);
                unsigned long long m = __ballot(d2 < K.cps2);
                if (tn - c0 < 64) m &= (1ull << (tn - c0)) - 1ull;
                const unsigned self = (unsigned)(i - t0 - c0);
                if (self < 64u) m &= ~(1ull << self);
                const int slot = cnt + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                                 __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
                if (__builtin_amdgcn_inverse_ballot_w64(m) && slot < K.maxnb)
                    nbl[(size_t)i * K.maxnb + slot] = t0 + c0 + lane;
                cnt += __popcll(m);
            };
            if (K.boxes) {
                unsigned long long live =
                    __ballot(lane < (tn + 63) / 64 && box_near(K, ri, box_c[lane & 3], box_h[lane & 3], K.cps2));
                while (live) {
                    chunk(64 * __builtin_ctzll(live));
                    live &= live - 1;
                }
            } else {
                for (int c0 = 0; c0 < tn; c0 += 64) chunk(c0);
            }
            if (lane == 0) count[p] = cnt;
        }
    }
    __syncthreads();
    if ((int)threadIdx.x < np && i0 + (int)threadIdx.x < K.N) {
        const int i = i0 + (int)threadIdx.x, cnt = count[threadIdx.x];
        nbc[i] = cnt;
        rref[i] = own[threadIdx.x];
        if (cnt > K.maxnb) atomicMax(gen_ptr(over), cnt);
    }
    __syncthreads();
}

// flag[b] = 1 when r has moved more than skin/2 from its reference
__device__ __forceinline__ void adj_skin_flag(const AdjK &K, const float4 r, const float4 q, GMEM int *flag, int b) {
    float dx, dy, dz;
    if (dist_sq_mic(r.x, r.y, r.z, q.x, q.y, q.z, K.L0, K.L1, K.L2, dx, dy, dz) > K.skin2q) flag[b] = 1;
}

// What the step kernels share: the lists, and the skin flags of three steps
// by turns (a step reads flag[b], raises flag[b + 1] for the next and clears
// flag[b + 2]); built: the lists were built for these positions just before
// (a checkpoint), whatever the flag says
struct AdjLists {
    int *nbl, *nbc, *flag, *over;
    float4 *rref;
    int b, built;
};

#define ADJ_APART_N 8000
#define ADJ_UNR 4   // list entries a lane gathers at a time

// The pairs of particle i (lane t of its tp) in list order: ADJ_UNR entries,
// their positions and (W) their w are requested together, then each pair is
// handed to body(w_j, dx, dy, dz, d2, type of j, inside the list).  Entries
// past the count stand for the particle itself.
template <bool W, class Body>
__device__ __forceinline__ void adj_pairs(const AdjK &K, cpos_t pos, cpos_t w, const GMEM int *row, int cnt, int i,
                                          int t, const float4 ri, Body body) {
    const int tp = K.tp;
    int j[ADJ_UNR];
#pragma unroll
    for (int u = 0; u < ADJ_UNR; ++u) j[u] = t + u * tp < cnt ? row[t + u * tp] : i;
    for (int k0 = t; k0 < cnt; k0 += ADJ_UNR * tp) {
        float4 rj[ADJ_UNR], wj[ADJ_UNR];
#pragma unroll
        for (int u = 0; u < ADJ_UNR; ++u) rj[u] = pos[j[u]];
        if (W) {
#pragma unroll
            for (int u = 0; u < ADJ_UNR; ++u) wj[u] = w[j[u]];
        }
#pragma unroll
        for (int u = 0; u < ADJ_UNR; ++u) {
            const int k = k0 + (ADJ_UNR + u) * tp;
            j[u] = k < cnt ? row[k] : i;
        }
#pragma unroll
        for (int u = 0; u < ADJ_UNR; ++u) {
            float dx, dy, dz;
            const float d2 = dist_sq_mic(ri.x, ri.y, ri.z, rj[u].x, rj[u].y, rj[u].z, K.L0, K.L1, K.L2, dx, dy, dz);
            body(wj[u], dx, dy, dz, d2, adj_type(rj[u]), k0 + u * tp < cnt);
        }
    }
}

// One forward step from the positions r to rn (F_n = F(r_n), leap-frog,
// wrap), K.tp lanes per particle (the lanes' sums added by a butterfly, a
// fixed order); the new positions take the next step's skin check.
__global__ void __launch_bounds__(256) k_adj_fstep(AdjK K, const float4 *r_p, float4 *rn_p, float4 *vel_p,
                                                   AdjLists A) {
    cpos_t pos = (cpos_t)r_p;
    GMEM int *flag = (GMEM int *)A.flag;
    GMEM float4 *rref = (GMEM float4 *)A.rref;
    __shared__ AdjPairC pc[ADJ_MAX_TYPES * ADJ_MAX_TYPES];
    adj_stage_pairs(K, pc);
    const bool relist = !A.built && flag[A.b] != 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) flag[(A.b + 2) % 3] = 0;
    if (relist) adj_relist(K, pos, rref, (GMEM int *)A.nbl, (GMEM int *)A.nbc, (GMEM int *)A.over);
    const int i = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> K.tpsh);
    const int t = threadIdx.x & (K.tp - 1);
    const bool valid = i < K.N;
    block_sync_lds();   // pc
    float fx = 0.f, fy = 0.f, fz = 0.f;
    float4 ri = make_float4(0.f, 0.f, 0.f, 0.f), v = ri, q0 = ri;
    if (valid) {
        ri = pos[i];
        const int cnt = min(((const GMEM int *)A.nbc)[i], K.maxnb);
        if (t == 0) {   // needed after the sums: on their way meanwhile
            v = ((const GMEM float4 *)vel_p)[i];
            q0 = rref[i];
        }
        const int ti = adj_type(ri) * K.nt;
        adj_pairs<false>(K, pos, pos, (const GMEM int *)A.nbl + (size_t)i * K.maxnb, cnt, i, t, ri,
                  [&](const float4 &, float dx, float dy, float dz, float d2, int tj, bool in) {
                      const AdjPairC &q = pc[ti + tj];
                      const bool ok = in & (d2 < q.cut2);
                      AdjPairEval e = adj_pair(q, d2);
                      const float sv = ok ? e.s : 0.f;
                      fx += sv * dx;
                      fy += sv * dy;
                      fz += sv * dz;
                  });
    }
    fx = group_sum(fx, K.tp);
    fy = group_sum(fy, K.tp);
    fz = group_sum(fz, K.tp);
    if (!valid || t != 0) return;
    float4 r = ri;
    {
#pragma clang fp contract(off)
        const float inv_m = 1.0f / v.w;
        v.x = v.x + fx * inv_m * K.dt;
        v.y = v.y + fy * inv_m * K.dt;
        v.z = v.z + fz * inv_m * K.dt;
        r.x = r.x + v.x * K.dt;
        r.y = r.y + v.y * K.dt;
        r.z = r.z + v.z * K.dt;
    }
    int im = 0;
    wrap_pbc(r.x, im, K.L0);
    wrap_pbc(r.y, im, K.L1);
    wrap_pbc(r.z, im, K.L2);
    ((GMEM float4 *)vel_p)[i] = v;
    ((GMEM float4 *)rn_p)[i] = r;
    adj_skin_flag(K, r, q0, flag, (A.b + 1) % 3);
}

// One backward step n at the positions r_n: J w over the lists,
//   sum_j A (w_i - w_j) + B d (d . (w_i - w_j)),
// lambda_r += J w (+ the frame's gradient rpart); then, unless n == 0
// (advance), lambda_v += dt lambda_r and wn = dt/m lambda_v for step n - 1
// (another buffer: the neighbours of this step still read w).  The block's
// parameter gradients sum_i w_i . d ds/d{sigma, epsilon} are added to its
// slot pgl[block][2c + {0, 1}].  rnext: the positions of step n - 1 take
// their skin check here (null: the next list is built anyway).
__global__ void __launch_bounds__(256) k_adj_bstep(AdjK K, const float4 *r_p, const float4 *w_p, float4 *wn_p,
                                                   const float4 *vel_p, float4 *lr_p, float4 *lv_p,
                                                   const float4 *rpart_p, int advance, double *pgl_p,
                                                   const float4 *rnext_p, AdjLists A) {
    __shared__ float red[4][2 * ADJ_MAX_CLS];
    cpos_t pos = (cpos_t)r_p, w = (cpos_t)w_p;
    GMEM int *flag = (GMEM int *)A.flag;
    GMEM float4 *rref = (GMEM float4 *)A.rref;
    __shared__ AdjPairC pc[ADJ_MAX_TYPES * ADJ_MAX_TYPES];
    adj_stage_pairs(K, pc);
    const bool relist = !A.built && flag[A.b] != 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) flag[(A.b + 2) % 3] = 0;
    if (relist) adj_relist(K, pos, rref, (GMEM int *)A.nbl, (GMEM int *)A.nbc, (GMEM int *)A.over);
    const int i = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> K.tpsh);
    const int t = threadIdx.x & (K.tp - 1);
    const bool valid = i < K.N;
    block_sync_lds();   // pc
    float ax = 0.f, ay = 0.f, az = 0.f;
    float g[2 * ADJ_MAX_CLS];
#pragma unroll
    for (int c = 0; c < 2 * ADJ_MAX_CLS; ++c) g[c] = 0.f;
    float4 a0 = make_float4(0.f, 0.f, 0.f, 0.f), b0 = a0, p0 = a0, q0 = a0, rx = a0;
    float mass = 1.f;
    if (valid) {
        const float4 ri = pos[i];
        const float4 wi = w[i];
        const int cnt = min(((const GMEM int *)A.nbc)[i], K.maxnb);
        if (t == 0) {   // needed after the sums: on their way meanwhile
            a0 = ((const GMEM float4 *)lr_p)[i];
            if (rpart_p) p0 = ((const GMEM float4 *)rpart_p)[i];
            if (advance) {
                b0 = ((const GMEM float4 *)lv_p)[i];
                mass = ((const GMEM float4 *)vel_p)[i].w;
            }
            if (rnext_p) {
                q0 = rref[i];
                rx = ((cpos_t)rnext_p)[i];
            }
        }
        const int ti = adj_type(ri) * K.nt;
        adj_pairs<true>(K, pos, w, (const GMEM int *)A.nbl + (size_t)i * K.maxnb, cnt, i, t, ri,
                  [&](const float4 &wj, float dx, float dy, float dz, float d2, int tj, bool in) {
                      const AdjPairC &q = pc[ti + tj];
                      if (!(in & (d2 < q.cut2))) return;
                      const AdjPairEval e = adj_pair(q, d2);
                      const float ux = wi.x - wj.x, uy = wi.y - wj.y, uz = wi.z - wj.z;
                      const float du = dx * ux + dy * uy + dz * uz;
                      ax += e.s * ux + e.B * dx * du;
                      ay += e.s * uy + e.B * dy * du;
                      az += e.s * uz + e.B * dz * du;
                      const float wd = wi.x * dx + wi.y * dy + wi.z * dz;
#pragma unroll
                      for (int c = 0; c < ADJ_MAX_CLS; ++c)
                          if (c == q.cls) {
                              g[2 * c] += wd * e.ds_dsig;
                              g[2 * c + 1] += wd * e.ds_deps;
                          }
                  });
    }
    ax = group_sum(ax, K.tp);
    ay = group_sum(ay, K.tp);
    az = group_sum(az, K.tp);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nc = 2 * K.ncls;
#pragma unroll
    for (int c = 0; c < 2 * ADJ_MAX_CLS; ++c) {
        if (c >= nc) continue;
        const float v = wave_sum_f(g[c]);
        if (lane == 0) red[wid][c] = v;
    }
    if (valid && t == 0) {
        float4 a = a0;
        a.x += ax;
        a.y += ay;
        a.z += az;
        if (rpart_p) {
            a.x += p0.x;
            a.y += p0.y;
            a.z += p0.z;
        }
        ((GMEM float4 *)lr_p)[i] = a;
        if (advance) {
            float4 b = b0;
            b.x += K.dt * a.x;
            b.y += K.dt * a.y;
            b.z += K.dt * a.z;
            ((GMEM float4 *)lv_p)[i] = b;
            const float f = K.dt / mass;
            ((GMEM float4 *)wn_p)[i] = make_float4(f * b.x, f * b.y, f * b.z, 0.f);
        }
        if (rnext_p) adj_skin_flag(K, rx, q0, flag, (A.b + 1) % 3);
    }
    __syncthreads();
    if ((int)threadIdx.x < nc) {
        double s = 0.0;
        for (int k = 0; k < (int)(blockDim.x >> 6); ++k) s += (double)red[k][threadIdx.x];
        ((GMEM double *)pgl_p)[(size_t)blockIdx.x * (2 * ADJ_MAX_CLS) + threadIdx.x] += s;
    }
}

// smoothed pair histogram of one frame over its half list (each pair once) of radius
// rmax + 5 w, K.tp lanes per particle, one LDS histogram per block added to
// hacc[block][ncls * bins].  The histogram is in 64-bit fixed point: float
// atomics on LDS run at a third of a lane a cycle and CU here, 32-bit integer
// ones at eight, and the sum of whole numbers is the same in every order.
// KA N = 4096, rmax 4, 200 bins: 57 -> 16 us a frame.  A weight is the
// difference of two floats of at least kfloor > 2^-19, so a whole number of
// 2^-42: at hup = 2^10 it is added with all its bits.
__global__ void __launch_bounds__(256) k_adj_rdf_list(AdjK K, const float4 *pos_p, const int *nbl_p, const int *nbc_p,
                                                      int maxnb, double *hacc_p) {
    __shared__ unsigned long long h[ADJ_MAX_CLS * ADJ_MAX_BINS];
    const int nh = K.ncls * K.bins;
    __shared__ AdjPairC pc[ADJ_MAX_TYPES * ADJ_MAX_TYPES];
    adj_stage_pairs(K, pc);
    for (int t = threadIdx.x; t < nh; t += blockDim.x) h[t] = 0ull;
    __syncthreads();
    cpos_t pos = (cpos_t)pos_p;
    const int i = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> K.tpsh);
    const int tl = threadIdx.x & (K.tp - 1);
    if (i < K.N) {
        const float4 ri = pos[i];
        const int ti = adj_type(ri) * K.nt;
        adj_pairs<false>(K, pos, pos, (const GMEM int *)nbl_p + (size_t)i * maxnb,
                         min(((const GMEM int *)nbc_p)[i], maxnb), i, tl, ri,
                  [&](const float4 &, float, float, float, float d2, int tj, bool in) {
                      if (!(in & (d2 < K.rcut2))) return;
                      const float d = sqrtf(d2);
                      const int c = pc[ti + tj].cls;
                      const int k0 = max(0, (int)floorf((d - 5.0f * K.wid) / K.dr - 0.5f));
                      const int k1 = min(K.bins - 1, (int)ceilf((d + 5.0f * K.wid) / K.dr - 0.5f));
                      for (int kb = k0; kb <= k1; ++kb) {
                          const float x = d - ((float)kb + 0.5f) * K.dr;
                          const float kv = __expf(-0.5f * x * x * K.inv_w2) - K.kfloor;
                          if (kv > 0.f) {
                              const float a = kv * K.hup;
                              const unsigned long long hi = (unsigned)a;
                              const unsigned lo = (unsigned)(__builtin_amdgcn_fractf(a) * 0x1p32f);
                              atomicAdd(&h[c * K.bins + kb], hi << 32 | lo);
                          }
                      }
                  });
    }
    __syncthreads();
    GMEM double *dst = (GMEM double *)hacc_p + (size_t)blockIdx.x * nh;
    const double unit = 0x1p-32 / (double)K.hup;
    for (int t = threadIdx.x; t < nh; t += blockDim.x) dst[t] += (double)h[t] * unit;
}

// dL/dr_i of one frame given G = dL/dH over the frame's list (all j of i):
// sum_j (sum_k G[c][k] K'(d - r_k)) d_ij / d, K.tp lanes per particle
__global__ void __launch_bounds__(256) k_adj_rdf_grad_list(AdjK K, const float4 *pos_p, const float *G,
                                                           const int *nbl_p, const int *nbc_p, int maxnb,
                                                           float4 *out) {
    __shared__ float sg[ADJ_MAX_CLS * ADJ_MAX_BINS];
    const int nh = K.ncls * K.bins;
    __shared__ AdjPairC pc[ADJ_MAX_TYPES * ADJ_MAX_TYPES];
    adj_stage_pairs(K, pc);
    for (int t = threadIdx.x; t < nh; t += blockDim.x) sg[t] = G[t];
    __syncthreads();
    cpos_t pos = (cpos_t)pos_p;
    const int i = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> K.tpsh);
    const int tl = threadIdx.x & (K.tp - 1);
    float ax = 0.f, ay = 0.f, az = 0.f;
    if (i < K.N) {
        const float4 ri = pos[i];
        const int ti = adj_type(ri);
        adj_pairs<false>(K, pos, pos, (const GMEM int *)nbl_p + (size_t)i * maxnb,
                         min(((const GMEM int *)nbc_p)[i], maxnb), i, tl, ri,
                  [&](const float4 &, float dx, float dy, float dz, float d2, int tj, bool in) {
                      if (!(in & (d2 < K.rcut2))) return;
                      const float d = sqrtf(d2);
                      const int c = pc[ti * K.nt + tj].cls;
                      const int k0 = max(0, (int)floorf((d - 5.0f * K.wid) / K.dr - 0.5f));
                      const int k1 = min(K.bins - 1, (int)ceilf((d + 5.0f * K.wid) / K.dr - 0.5f));
                      float dLdd = 0.f;
                      for (int kb = k0; kb <= k1; ++kb) {
                          const float x = d - ((float)kb + 0.5f) * K.dr;
                          const float e = __expf(-0.5f * x * x * K.inv_w2);
                          if (e - K.kfloor > 0.f) dLdd += sg[c * K.bins + kb] * (-x * K.inv_w2) * e;
                      }
                      const float sc = dLdd / d;
                      ax += sc * dx;
                      ay += sc * dy;
                      az += sc * dz;
                  });
    }
    ax = group_sum(ax, K.tp);
    ay = group_sum(ay, K.tp);
    az = group_sum(az, K.tp);
    if (i < K.N && tl == 0) out[i] = make_float4(ax, ay, az, 0.f);
}

// fixed-order float64 sum over a block of 256 threads of one value each
__device__ __forceinline__ double adj_block_sum(double v, double *sred) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    v = wave_sum_d(v);
    __syncthreads();
    if (lane == 0) sred[wid] = v;
    __syncthreads();
    double s = 0.0;
    for (int k = 0; k < (int)(blockDim.x >> 6); ++k) s += sred[k];
    return s;
}

// out[k] = sum over the blocks' slots in[block][stride], one block of 256
// threads per k (each thread the slots t, t + 256, ..., then a fixed-order
// block sum)
__global__ void __launch_bounds__(256) k_adj_sum(const double *in, int nblocks, int stride, double *out) {
    __shared__ double sred[4];
    const int k = blockIdx.x;
    double s = 0.0;
    for (int b = threadIdx.x; b < nblocks; b += blockDim.x) s += in[(size_t)b * stride + k];
    s = adj_block_sum(s, sred);
    if (threadIdx.x == 0) out[k] = s;
}

// start of the adjoint at r_S: lambda_r = the frame's gradient (if r_S is a
// frame), lambda_v = dt lambda_r, w = dt/m lambda_v of step S - 1
__global__ void __launch_bounds__(256) k_adj_start(AdjK K, const float4 *vel, float4 *lr, float4 *lv, float4 *w,
                                                   const float4 *rpart) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= K.N) return;
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
    if (rpart) {
        const float4 p = rpart[i];
        a.x += p.x;
        a.y += p.y;
        a.z += p.z;
    }
    lr[i] = a;
    b.x += K.dt * a.x;
    b.y += K.dt * a.y;
    b.z += K.dt * a.z;
    lv[i] = b;
    const float f = K.dt / vel[i].w;
    w[i] = make_float4(f * b.x, f * b.y, f * b.z, 0.f);
}

// ============================================================================
// Host side
// ============================================================================
struct gmd_adj {
    gmd_adj_desc d;
    AdjK K;
    std::vector<int> ptype;
    std::vector<float> mass;
    int nck = 0;
    int gl = 0;                  // blocks of the list sums
    int rmaxnb = 0;              // slots per particle of the frame list
    int fboxes = 0;              // K.boxes for the frame lists
    bool apart = false;          // list builds between checkpoints in launches of their own (ADJ_APART_N)
    int chk = 0;                 // steps of a pass so far (the turn of the skin flags)
    size_t nbl_cap = 0;          // allocated list slots
    hipStream_t stream = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    float fwd_ms = 0.f, bwd_ms = 0.f;
    bool have_forward = false;
    // device
    float4 *pos = nullptr, *pos2 = nullptr, *vel = nullptr, *rpart = nullptr, *rref = nullptr;
    int *nbl = nullptr, *nbc = nullptr, *flag = nullptr;
    int *rnbl = nullptr, *rnbc = nullptr;   // list of one frame (radius rmax + 5 w)
    // the positions of every step (traj), or the checkpoints and one segment
    // recomputed from its checkpoint (adj_storage)
    float4 *traj = nullptr;
    float4 *ck_r = nullptr, *ck_v = nullptr, *seg = nullptr;
    float4 *lr = nullptr, *lv = nullptr, *w = nullptr, *w2 = nullptr;
    double *pgl = nullptr, *pgrad_tot = nullptr, *H = nullptr, *hacc = nullptr;
    float *G = nullptr;
};

static int adj_free(gmd_adj *a) {
    if (!a) return 0;
    void *ptrs[] = {a->pos, a->pos2, a->vel, a->rpart, a->rref, a->nbl, a->nbc, a->flag, a->rnbl, a->rnbc,
                    a->traj, a->ck_r, a->ck_v, a->seg, a->lr, a->lv, a->w, a->w2, a->pgl, a->pgrad_tot, a->H, a->hacc, a->G};
    for (void *p : ptrs)
        if (p) hipFree(p);
    if (a->e0) hipEventDestroy(a->e0);
    if (a->e1) hipEventDestroy(a->e1);
    if (a->stream) hipStreamDestroy(a->stream);
    delete a;
    return 0;
}

static int adj_cls(int a, int b, int nt) {
    if (a > b) std::swap(a, b);
    return a * nt - a * (a - 1) / 2 + (b - a);
}

// The upper word's scale of the frame histograms: 2^10, or the largest power
// of two at which a block's 64-bit counters hold every pair of its lists (only
// lists of more than 65536 entries leave less)
static float adj_weight_scale(double pairs) {
    float up = 1024.0f;
    while (up > 1.0f && pairs * up >= 4294967296.0) up *= 0.5f;
    return up;
}

// The storage the backward pass reads the positions from.  A trajectory of up
// to ADJ_TRAJ_BYTES stays in memory as the forward pass writes it: one buffer
// of step after step, nothing copied and no step computed twice (N = 4096, 200
// steps: 13 MB, and the backward pass 200 forward steps and ten list builds
// shorter).  A longer one, one the device has no room for beside everything
// else, or any one where the caller asks for it, keeps a checkpoint of
// positions and velocities every ckpt_every steps and recomputes a segment at
// a time.  On an error the handle is left without storage.
#define ADJ_TRAJ_BYTES ((size_t)4 << 30)
static hipError_t adj_storage(gmd_adj *a, bool whole) {
    auto release = [a]() {
        for (float4 **p : {&a->traj, &a->pos, &a->pos2, &a->ck_r, &a->ck_v, &a->seg}) {
            if (*p) hipFree(*p);
            *p = nullptr;
        }
    };
    auto get = [](float4 **p, size_t n) {
        const hipError_t e = hipMalloc((void **)p, n * sizeof(float4));
        if (e != hipSuccess) {
            *p = nullptr;
            (void)hipGetLastError();
        }
        return e;
    };
    release();
    a->have_forward = false;
    const size_t N = a->d.N;
    if (whole && get(&a->traj, ((size_t)a->d.nsteps + 1) * N) == hipSuccess) return hipSuccess;
    hipError_t e = get(&a->pos, N);
    if (e == hipSuccess) e = get(&a->pos2, N);
    if (e == hipSuccess) e = get(&a->ck_r, (size_t)a->nck * N);
    if (e == hipSuccess) e = get(&a->ck_v, (size_t)a->nck * N);
    if (e == hipSuccess) e = get(&a->seg, (size_t)(a->d.ckpt_every + 1) * N);
    if (e != hipSuccess) release();
    return e;
}

// Whether the builds of lists of this radius test a chunk's box before its 64
// positions: a question of the caller's numbering.  The share of chunks whose
// box is near a particle is estimated from 16 of the start's chunks; the boxes
// pay where it is below about 0.3.  Ordered along a lattice, rho = 1.2, 40
// steps, forward + backward without and with boxes: N = 2000 (0.47) 814 and
// 838 us, 4000 (0.30; 100 steps) 2340 and 2362, 8000 (0.16) 1687 and 1560,
// 65536 (0.05) 38.7 and 25.5 ms.  In no order (1.0), where every box is tested
// for nothing: 8000 2064 and 2523 us, 65536 42.9 and 71.1 ms.
static int adj_boxes(const gmd_adj *a, const float *r, float radius) {
    return chunk_share(r, a->d.N, a->d.box, 2.0f * radius, 16) < 0.3 ? 1 : 0;
}

// pair constants from (sigma, epsilon, cut) per ordered type pair
static int adj_set_params(gmd_adj *a, const float *params) {
    const int nt = a->d.ntypes;
    for (int ti = 0; ti < nt; ++ti)
        for (int tj = 0; tj < nt; ++tj) {
            const float *p = params + 3 * (ti * nt + tj);
            const float *q = params + 3 * (tj * nt + ti);
            if (p[0] != q[0] || p[1] != q[1] || p[2] != q[2])
                return fail("gmd_adj: parameters of types (%d,%d) and (%d,%d) differ", ti, tj, tj, ti);
            if (!(p[0] > 0.f) || !(p[2] > 0.f)) return fail("gmd_adj: sigma and cut must be positive");
            const float half = 0.5f * std::min(a->d.box[0], std::min(a->d.box[1], a->d.box[2]));
            if (!(p[2] < half))
                return fail("gmd_adj: cut %g of types (%d,%d) must be below half the box (%g)", p[2], ti, tj, half);
            AdjPairC &c = a->K.pc[ti * nt + tj];
            const double sig = p[0], eps = p[1], rc = p[2];
            c.sig = (float)sig;
            c.sig2 = (float)(sig * sig);
            c.eps = (float)eps;
            c.eps24 = (float)(24.0 * eps);
            c.cut2 = (float)(rc * rc);
            const double x6c = std::pow(sig / rc, 6.0), x12c = x6c * x6c;
            c.sc = (float)(24.0 * eps * (2.0 * x12c - x6c) / (rc * rc));
            c.dsc_dsig = (float)(24.0 * eps / sig * (24.0 * x12c - 6.0 * x6c) / (rc * rc));
            c.cls = adj_cls(ti, tj, nt);
        }
    // neighbour lists: radius max cut + skin, capacity about twice the mean
    // length at the system's density
    double maxcut = 0.0;
    for (int k = 0; k < nt * nt; ++k) maxcut = std::max(maxcut, std::sqrt((double)a->K.pc[k].cut2));
    const double rl = maxcut + ADJ_SKIN;
    const double half = 0.5 * std::min(a->d.box[0], std::min(a->d.box[1], a->d.box[2]));
    if (!(rl < half)) return fail("gmd_adj: max cut + skin (%g) must be below half the box (%g)", rl, half);
    a->K.cps2 = (float)(rl * rl);
    a->K.skin2q = 0.25f * ADJ_SKIN * ADJ_SKIN;
    const double vol = (double)a->d.box[0] * a->d.box[1] * a->d.box[2];
    const double nbar = a->d.N / vol * 4.18879020478639 * rl * rl * rl;
    const int maxnb = ((int)(2.0 * nbar) + 64 + 31) / 32 * 32;
    const size_t need = (size_t)a->d.N * maxnb;
    if (need > a->nbl_cap) {
        if (a->nbl) hipFree(a->nbl);
        a->nbl = nullptr;
        a->nbl_cap = 0;
        hipError_t e = hipMalloc((void **)&a->nbl, need * sizeof(int));
        if (e != hipSuccess && a->traj) {
            // the lists come first: the trajectory makes room
            (void)hipGetLastError();
            e = adj_storage(a, false);
            if (e == hipSuccess) e = hipMalloc((void **)&a->nbl, need * sizeof(int));
        }
        if (e != hipSuccess) {
            a->nbl = nullptr;
            return fail("gmd_adj: list allocation");
        }
        a->nbl_cap = need;
    }
    a->K.maxnb = maxnb;
    return 0;
}

extern "C" {

int gmd_adj_create(const gmd_adj_desc *desc, const int *ptype, const float *mass, gmd_adj **out) {
    if (!desc || !ptype || !mass || !out) return fail("gmd_adj_create: null argument");
    *out = nullptr;
    const gmd_adj_desc &d = *desc;
    if (d.N < 2) return fail("gmd_adj_create: N must be at least 2");
    if (d.ntypes < 1 || d.ntypes > ADJ_MAX_TYPES) return fail("gmd_adj_create: ntypes must be in [1,%d]", ADJ_MAX_TYPES);
    if (d.nsteps < 1 || d.ckpt_every < 1) return fail("gmd_adj_create: nsteps and ckpt_every must be positive");
    if (d.rdf_every < 1 || d.rdf_bins < 1 || !(d.rdf_rmax > 0.f) || !(d.rdf_width > 0.f))
        return fail("gmd_adj_create: bad RDF settings");
    const int ncls = d.ntypes * (d.ntypes + 1) / 2;
    if (ncls * d.rdf_bins > ADJ_MAX_CLS * ADJ_MAX_BINS)
        return fail("gmd_adj_create: %d classes x %d bins exceed the LDS histogram (%d)", ncls, d.rdf_bins,
                    ADJ_MAX_CLS * ADJ_MAX_BINS);
    for (int k = 0; k < 3; ++k)
        if (!(d.box[k] > 0.f)) return fail("gmd_adj_create: box lengths must be positive");
    const float half = 0.5f * std::min(d.box[0], std::min(d.box[1], d.box[2]));
    if (d.rdf_rmax + 5.0f * d.rdf_width > half)
        return fail("gmd_adj_create: rdf_rmax + 5 width (%g) must stay below half the box (%g)",
                    d.rdf_rmax + 5.0f * d.rdf_width, half);
    gmd_adj *a = new gmd_adj();
    a->d = d;
    a->ptype.assign(ptype, ptype + d.N);
    a->mass.assign(mass, mass + d.N);
    for (int i = 0; i < d.N; ++i) {
        if (ptype[i] < 0 || ptype[i] >= d.ntypes) {
            adj_free(a);
            return fail("gmd_adj_create: particle %d has type %d", i, ptype[i]);
        }
        if (!(mass[i] > 0.f)) {
            adj_free(a);
            return fail("gmd_adj_create: particle %d has mass %g", i, mass[i]);
        }
    }
    AdjK &K = a->K;
    memset(&K, 0, sizeof K);
    K.N = d.N;
    K.nt = d.ntypes;
    K.ncls = ncls;
    K.L0 = d.box[0];
    K.L1 = d.box[1];
    K.L2 = d.box[2];
    K.dt = d.dt;
    K.bins = d.rdf_bins;
    K.rmax = d.rdf_rmax;
    K.dr = d.rdf_rmax / d.rdf_bins;
    K.wid = d.rdf_width;
    K.inv_w2 = 1.0f / (d.rdf_width * d.rdf_width);
    K.kfloor = std::exp(-12.5f);
    const float rc = d.rdf_rmax + 5.0f * d.rdf_width;
    K.rcut2 = rc * rc;
    // lanes per particle of the list sums: enough wavefronts to fill the device
    K.tp = 4;
    while (K.tp < 32 && (size_t)d.N * K.tp < 131072) K.tp *= 2;
    K.tpsh = 0;
    while ((1 << K.tpsh) < K.tp) ++K.tpsh;
    a->gl = (int)(((size_t)d.N * K.tp + 255) / 256);
    // frame list: capacity about twice the mean count within rmax + 5 w
    {
        const double vol = (double)d.box[0] * d.box[1] * d.box[2];
        const double nbar = d.N / vol * 4.18879020478639 * (double)rc * rc * rc;
        a->rmaxnb = (int)std::min<double>((2.0 * nbar + 64.0 + 31.0) / 32.0 * 32.0, (double)d.N + 31.0);
        a->rmaxnb = a->rmaxnb / 32 * 32;
    }
    K.hup = adj_weight_scale((double)(256 / K.tp) * a->rmaxnb);
    a->nck = (d.nsteps + d.ckpt_every - 1) / d.ckpt_every;
    a->apart = d.N >= ADJ_APART_N;
    const size_t N = d.N;
#define ATRY(x)                                                               \
    do {                                                                      \
        hipError_t e_ = (x);                                                  \
        if (e_ != hipSuccess) {                                               \
            adj_free(a);                                                      \
            return fail("gmd_adj_create: %s: %s", #x, hipGetErrorString(e_)); \
        }                                                                     \
    } while (0)
    ATRY(hipStreamCreateWithFlags(&a->stream, hipStreamNonBlocking));
    ATRY(hipEventCreate(&a->e0));
    ATRY(hipEventCreate(&a->e1));
    ATRY(hipMalloc((void **)&a->vel, N * sizeof(float4)));
    ATRY(hipMalloc((void **)&a->rpart, N * sizeof(float4)));
    ATRY(hipMalloc((void **)&a->rnbl, N * (size_t)a->rmaxnb * sizeof(int)));
    ATRY(hipMalloc((void **)&a->rnbc, N * sizeof(int)));
    ATRY(hipMalloc((void **)&a->rref, N * sizeof(float4)));
    ATRY(hipMalloc((void **)&a->nbc, N * sizeof(int)));
    ATRY(hipMalloc((void **)&a->flag, 5 * sizeof(int)));   // skin flags of three steps, list overflows
    ATRY(hipMalloc((void **)&a->lr, N * sizeof(float4)));
    ATRY(hipMalloc((void **)&a->lv, N * sizeof(float4)));
    ATRY(hipMalloc((void **)&a->w, N * sizeof(float4)));
    ATRY(hipMalloc((void **)&a->w2, N * sizeof(float4)));
    ATRY(hipMalloc((void **)&a->pgl, (size_t)a->gl * 2 * ADJ_MAX_CLS * sizeof(double)));
    ATRY(hipMalloc((void **)&a->pgrad_tot, 2 * ADJ_MAX_CLS * sizeof(double)));
    ATRY(hipMalloc((void **)&a->H, (size_t)ncls * d.rdf_bins * sizeof(double)));
    ATRY(hipMalloc((void **)&a->hacc, (size_t)a->gl * ncls * d.rdf_bins * sizeof(double)));
    ATRY(hipMalloc((void **)&a->G, (size_t)ncls * d.rdf_bins * sizeof(float)));
    ATRY(adj_storage(a, ((size_t)d.nsteps + 1) * N * sizeof(float4) <= ADJ_TRAJ_BYTES));   // (what is left for it)
#undef ATRY
    *out = a;
    return 0;
}

int gmd_adj_destroy(gmd_adj *a) { return adj_free(a); }

int gmd_adj_use_checkpoints(gmd_adj *a) {
    if (!a) return fail("gmd_adj_use_checkpoints: null handle");
    HIPCHECK(hipStreamSynchronize(a->stream));
    const bool whole = a->traj != nullptr;
    const hipError_t e = adj_storage(a, false);
    if (e == hipSuccess) return 0;
    if (whole) (void)adj_storage(a, true);   // as it was
    return fail("gmd_adj_use_checkpoints: %s", hipGetErrorString(e));
}

// blocks of a list build: ADJ_BT / 64 particles each
static dim3 adj_build_grid(const gmd_adj *a) { return dim3((a->K.N + ADJ_BT / 64 - 1) / (ADJ_BT / 64)); }

// the smoothed histogram of the frame at pos (its half list: each pair once)
static void adj_rdf_frame(gmd_adj *a, const float4 *pos) {
    hipLaunchKernelGGL(k_adj_build<true>, adj_build_grid(a), dim3(ADJ_BT), 0, a->stream, a->K, pos,
                       (float4 *)nullptr, a->rnbl, a->rnbc, a->rmaxnb, a->K.rcut2, a->fboxes, (const int *)nullptr, a->flag + 4);
    hipLaunchKernelGGL(k_adj_rdf_list, dim3(a->gl), dim3(256), 0, a->stream, a->K, pos, (const int *)a->rnbl,
                       (const int *)a->rnbc, a->rmaxnb, a->hacc);
}

// dL/dr of the frame at pos into a->rpart
static void adj_rdf_grad(gmd_adj *a, const float4 *pos) {
    hipLaunchKernelGGL(k_adj_build<false>, adj_build_grid(a), dim3(ADJ_BT), 0, a->stream, a->K, pos,
                       (float4 *)nullptr, a->rnbl, a->rnbc, a->rmaxnb, a->K.rcut2, a->fboxes, (const int *)nullptr, a->flag + 4);
    hipLaunchKernelGGL(k_adj_rdf_grad_list, dim3(a->gl), dim3(256), 0, a->stream, a->K, pos, (const float *)a->G,
                       (const int *)a->rnbl, (const int *)a->rnbc, a->rmaxnb, a->rpart);
}

// the lists of the next step kernel, at the positions pos: built here when
// the step needs them afresh (a checkpoint), else by the step itself where
// the last step's skin check asks for it
static AdjLists adj_lists(gmd_adj *a, const float4 *pos, bool build) {
    const int b = a->chk++ % 3;
    const bool apart = build || a->apart;
    if (apart)
        hipLaunchKernelGGL(k_adj_build<false>, adj_build_grid(a), dim3(ADJ_BT), 0, a->stream, a->K, pos, a->rref,
                           a->nbl, a->nbc, a->K.maxnb, a->K.cps2, a->K.boxes,
                           (const int *)(build ? nullptr : a->flag + b), a->flag + 3);
    return AdjLists{a->nbl, a->nbc, a->flag, a->flag + 3, a->rref, b, apart ? 1 : 0};
}

static int adj_reset_lists(gmd_adj *a) {
    a->chk = 0;
    HIPCHECK(hipMemsetAsync(a->flag, 0, 5 * sizeof(int), a->stream));
    return 0;
}

static int adj_check_lists(gmd_adj *a) {
    int f[5];
    HIPCHECK(hipMemcpy(f, a->flag, sizeof f, hipMemcpyDeviceToHost));
    if (f[3] > 0)
        return fail("gmd_adj: a neighbour list of %d entries exceeds its %d slots", f[3], a->K.maxnb);
    if (f[4] > 0)
        return fail("gmd_adj: a frame list of %d entries exceeds its %d slots", f[4], a->rmaxnb);
    return 0;
}

// one forward step from the positions r to rn
static void adj_step(gmd_adj *a, const float4 *r, float4 *rn, bool build) {
    const AdjLists A = adj_lists(a, r, build);
    hipLaunchKernelGGL(k_adj_fstep, dim3(a->gl), dim3(256), 0, a->stream, a->K, r, rn, a->vel, A);
}

int gmd_adj_forward(gmd_adj *a, const float *params, const float *r0, const float *v0, double *H, float *r_end,
                    float *v_end) {
    if (!a || !params || !r0 || !v0 || !H) return fail("gmd_adj_forward: null argument");
    // the stored pair constants and positions are overwritten from here on: a
    // pass that fails leaves nothing to differentiate
    a->have_forward = false;
    if (adj_set_params(a, params)) return -1;
    if (!a->traj && !a->seg) return fail("gmd_adj_forward: no memory for the trajectory or its checkpoints");
    const int N = a->d.N, S = a->d.nsteps, C = a->d.ckpt_every, E = a->d.rdf_every;
    a->K.boxes = adj_boxes(a, r0, std::sqrt(a->K.cps2));
    a->fboxes = adj_boxes(a, r0, std::sqrt(a->K.rcut2));
    std::vector<float4> hr(N), hv(N);
    for (int i = 0; i < N; ++i) {
        int t = a->ptype[i];
        float tf;
        memcpy(&tf, &t, 4);
        hr[i] = make_float4(r0[3 * i], r0[3 * i + 1], r0[3 * i + 2], tf);
        hv[i] = make_float4(v0[3 * i], v0[3 * i + 1], v0[3 * i + 2], a->mass[i]);
    }
    hipStream_t st = a->stream;
    float4 *cur = a->traj ? a->traj : a->pos, *nxt = a->traj ? a->traj + N : a->pos2;
    HIPCHECK(hipMemcpyAsync(cur, hr.data(), N * sizeof(float4), hipMemcpyHostToDevice, st));
    HIPCHECK(hipMemcpyAsync(a->vel, hv.data(), N * sizeof(float4), hipMemcpyHostToDevice, st));
    const int nh = a->K.ncls * a->K.bins;
    HIPCHECK(hipMemsetAsync(a->hacc, 0, (size_t)a->gl * nh * sizeof(double), st));
    if (adj_reset_lists(a)) return -1;
    HIPCHECK(hipEventRecord(a->e0, st));
    for (int n = 0; n < S; ++n) {
        if (!a->traj && n % C == 0) {
            HIPCHECK(hipMemcpyAsync(a->ck_r + (size_t)(n / C) * N, cur, N * sizeof(float4),
                                    hipMemcpyDeviceToDevice, st));
            HIPCHECK(hipMemcpyAsync(a->ck_v + (size_t)(n / C) * N, a->vel, N * sizeof(float4),
                                    hipMemcpyDeviceToDevice, st));
        }
        if (n % E == 0) adj_rdf_frame(a, cur);
        adj_step(a, cur, nxt, n % C == 0);
        if (a->traj) {
            cur = nxt;
            nxt += N;
        } else {
            std::swap(cur, nxt);
        }
    }
    if (S % E == 0) adj_rdf_frame(a, cur);
    hipLaunchKernelGGL(k_adj_sum, dim3(nh), dim3(256), 0, st, (const double *)a->hacc, a->gl, nh, a->H);
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipEventRecord(a->e1, st));
    HIPCHECK(hipEventSynchronize(a->e1));
    HIPCHECK(hipEventElapsedTime(&a->fwd_ms, a->e0, a->e1));
    HIPCHECK(hipMemcpy(H, a->H, nh * sizeof(double), hipMemcpyDeviceToHost));
    if (adj_check_lists(a)) return -1;
    if (r_end || v_end) {
        HIPCHECK(hipMemcpy(hr.data(), cur, N * sizeof(float4), hipMemcpyDeviceToHost));
        HIPCHECK(hipMemcpy(hv.data(), a->vel, N * sizeof(float4), hipMemcpyDeviceToHost));
        for (int i = 0; i < N; ++i) {
            if (r_end) {
                r_end[3 * i] = hr[i].x;
                r_end[3 * i + 1] = hr[i].y;
                r_end[3 * i + 2] = hr[i].z;
            }
            if (v_end) {
                v_end[3 * i] = hv[i].x;
                v_end[3 * i + 1] = hv[i].y;
                v_end[3 * i + 2] = hv[i].z;
            }
        }
    }
    a->have_forward = true;
    return 0;
}

int gmd_adj_backward(gmd_adj *a, const double *dLdH, double *grad_params, float *grad_r0, float *grad_v0) {
    if (!a || !dLdH || !grad_params || !grad_r0) return fail("gmd_adj_backward: null argument");
    if (!a->have_forward) return fail("gmd_adj_backward: no forward pass to differentiate");
    const int N = a->d.N, S = a->d.nsteps, C = a->d.ckpt_every, E = a->d.rdf_every;
    const int nh = a->K.ncls * a->K.bins;
    hipStream_t st = a->stream;
    std::vector<float> g(nh);
    for (int k = 0; k < nh; ++k) g[k] = (float)dLdH[k];
    HIPCHECK(hipMemcpyAsync(a->G, g.data(), nh * sizeof(float), hipMemcpyHostToDevice, st));
    HIPCHECK(hipMemsetAsync(a->pgl, 0, (size_t)a->gl * 2 * ADJ_MAX_CLS * sizeof(double), st));
    if (adj_reset_lists(a)) return -1;
    HIPCHECK(hipEventRecord(a->e0, st));
    const dim3 gu((N + 255) / 256);
    // lambda_r(S) = dL/dr_S, then lambda_v, w of step S-1; the last segment also provides r_S
    const int last = a->nck - 1;
    float4 *w = a->w, *wn = a->w2;
    for (int sgm = last; sgm >= 0; --sgm) {
        const int n0 = sgm * C, n1 = std::min(S, n0 + C);
        const float4 *seg = a->traj ? a->traj + (size_t)n0 * N : a->seg;   // r_n0 .. r_n1
        if (!a->traj) {
            HIPCHECK(hipMemcpyAsync(a->vel, a->ck_v + (size_t)sgm * N, N * sizeof(float4), hipMemcpyDeviceToDevice,
                                    st));
            HIPCHECK(hipMemcpyAsync(a->seg, a->ck_r + (size_t)sgm * N, N * sizeof(float4), hipMemcpyDeviceToDevice,
                                    st));
            // the segment's steps repeat the forward's: the list is rebuilt at
            // the checkpoint as it was there
            for (int k = 0; k < n1 - n0; ++k)
                adj_step(a, a->seg + (size_t)k * N, a->seg + (size_t)(k + 1) * N, k == 0);
        }
        if (sgm == last) {
            // start of the adjoint: frame gradient at r_S, then lambda_v and w of step S-1
            const float4 *rS = seg + (size_t)(n1 - n0) * N;
            if (S % E == 0) adj_rdf_grad(a, rS);
            hipLaunchKernelGGL(k_adj_start, gu, dim3(256), 0, st, a->K, (const float4 *)a->vel, a->lr, a->lv, w,
                               (const float4 *)(S % E == 0 ? a->rpart : nullptr));
        }
        for (int n = n1 - 1; n >= n0; --n) {
            const float4 *rn = seg + (size_t)(n - n0) * N;
            const AdjLists A = adj_lists(a, rn, n == n1 - 1);
            if (n % E == 0) adj_rdf_grad(a, rn);
            // the positions of step n-1 (same segment) take their skin check here
            hipLaunchKernelGGL(k_adj_bstep, dim3(a->gl), dim3(256), 0, st, a->K, rn, (const float4 *)w, wn,
                               (const float4 *)a->vel, a->lr, a->lv,
                               (const float4 *)(n % E == 0 ? a->rpart : nullptr), n > 0 ? 1 : 0, a->pgl,
                               n > n0 ? rn - N : (const float4 *)nullptr, A);
            std::swap(w, wn);
        }
    }
    hipLaunchKernelGGL(k_adj_sum, dim3(2 * a->K.ncls), dim3(256), 0, st, (const double *)a->pgl, a->gl,
                       2 * ADJ_MAX_CLS, a->pgrad_tot);
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipEventRecord(a->e1, st));
    HIPCHECK(hipEventSynchronize(a->e1));
    HIPCHECK(hipEventElapsedTime(&a->bwd_ms, a->e0, a->e1));
    if (adj_check_lists(a)) return -1;
    // gradient per unordered class: (d/dsigma, d/depsilon)
    double pg[2 * ADJ_MAX_CLS];
    HIPCHECK(hipMemcpy(pg, a->pgrad_tot, sizeof pg, hipMemcpyDeviceToHost));
    for (int c = 0; c < 2 * a->K.ncls; ++c) grad_params[c] = pg[c];
    std::vector<float4> h(N);
    HIPCHECK(hipMemcpy(h.data(), a->lr, N * sizeof(float4), hipMemcpyDeviceToHost));
    for (int i = 0; i < N; ++i) {
        grad_r0[3 * i] = h[i].x;
        grad_r0[3 * i + 1] = h[i].y;
        grad_r0[3 * i + 2] = h[i].z;
    }
    if (grad_v0) {
        HIPCHECK(hipMemcpy(h.data(), a->lv, N * sizeof(float4), hipMemcpyDeviceToHost));
        for (int i = 0; i < N; ++i) {
            grad_v0[3 * i] = h[i].x;
            grad_v0[3 * i + 1] = h[i].y;
            grad_v0[3 * i + 2] = h[i].z;
        }
    }
    return 0;
}

int gmd_adj_last_ms(gmd_adj *a, float *fwd_ms, float *bwd_ms) {
    if (!a) return fail("gmd_adj_last_ms: null handle");
    if (fwd_ms) *fwd_ms = a->fwd_ms;
    if (bwd_ms) *bwd_ms = a->bwd_ms;
    return 0;
}

}  // extern "C"
