// gmd_adjoint.h -- differentiable NVE trajectory: float32 forward with
// checkpoints, hand-written adjoint (force Jacobian-vector products and
// gradients with respect to the per-type LJ sigma / epsilon), and a
// Gaussian-smoothed partial radial distribution as the observable.
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
// squared build with one wavefront per particle, rebuilt when a particle has
// moved more than skin/2 and at every checkpoint, so a segment recomputed
// from its checkpoint in the backward pass repeats the forward bit for bit);
// the observable and its gradient run over a list of radius rmax + 5 w built
// afresh (same N-squared build, no skin) at each frame, one frame every
// rdf_every steps.
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
    AdjPairC pc[ADJ_MAX_TYPES * ADJ_MAX_TYPES];
    // observable
    int bins;
    float rmax, dr, wid, inv_w2, kfloor, rcut2;   // rcut = rmax + 5 w
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

// list check: flag[b] = 1 when some particle has moved more than skin/2
// from its position at the last build
__global__ void __launch_bounds__(256) k_adj_check(AdjK K, const float4 *pos, const float4 *rref, int *flag, int b) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= K.N) return;
    const float4 r = pos[i], q = rref[i];
    float dx, dy, dz;
    if (dist_sq_mic(r.x, r.y, r.z, q.x, q.y, q.z, K.L0, K.L1, K.L2, dx, dy, dz) > K.skin2q) flag[b] = 1;
}

// N-squared list build of radius^2 r2 into nbl (maxnb slots a particle)
// when flag[b] is set or force: one wavefront per particle, 16 a block (a
// launch that finds no build needed dispatches few blocks), the block's
// tiles of ADJ_BT positions staged in LDS, the accepted j compacted with a
// ballot (ascending j); flag[b ^ 1] is cleared for the next check (b >= 0),
// rref (if given) receives the positions and *over records the longest list
// beyond maxnb
#define ADJ_BT 1024   // threads of a build block, positions of its tile
__global__ void __launch_bounds__(ADJ_BT) k_adj_build(AdjK K, const float4 *pos, float4 *rref, int *nbl, int *nbc,
                                                      int maxnb, float r2, int *flag, int b, int force, int *over) {
    __shared__ float4 tile[ADJ_BT];
    if (b >= 0 && blockIdx.x == 0 && threadIdx.x == 0) flag[b ^ 1] = 0;
    if (!force && flag[b] == 0) return;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int i = blockIdx.x * (ADJ_BT / 64) + wid;
    const bool valid = i < K.N;
    const float4 ri = valid ? pos[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    const unsigned long long lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    int cnt = 0;
    for (int t0 = 0; t0 < K.N; t0 += ADJ_BT) {
        __syncthreads();
        if (t0 + (int)threadIdx.x < K.N) tile[threadIdx.x] = pos[t0 + threadIdx.x];
        __syncthreads();
        if (!valid) continue;
        const int tn = min(ADJ_BT, K.N - t0);
        for (int c0 = 0; c0 < tn; c0 += 64) {
            const int e = c0 + lane;
            const float4 rj = tile[e];
            float dx, dy, dz;
            const float d2 = dist_sq_mic(ri.x, ri.y, ri.z, rj.x, rj.y, rj.z, K.L0, K.L1, K.L2, dx, dy, dz);
            const bool ok = (e < tn) & (t0 + e != i) & (d2 < r2);
            const unsigned long long m = __ballot(ok);
            const int slot = cnt + __popcll(m & lt);
            if (ok && slot < maxnb) nbl[(size_t)i * maxnb + slot] = t0 + e;
            cnt += __popcll(m);
        }
    }
    if (valid && lane == 0) {
        nbc[i] = cnt;
        if (rref) rref[i] = ri;
        if (cnt > maxnb) atomicMax(over, cnt);
    }
}

// Pair sums over the neighbour lists, K.tp lanes per particle (the lanes'
// sums added by a butterfly, a fixed order):
//   MODE 0: force      out[i] = sum_j s d_ij
//   MODE 1: J w        out[i] = sum_j A (w_i - w_j) + B d (d.(w_i - w_j)),
//                      pgrad[block][2c + {0,1}] = sum_i w_i . d ds/d{sigma,epsilon}
template <int MODE>
__global__ void __launch_bounds__(256) k_adj_pairs_list(AdjK K, const float4 *pos, const float4 *w, const int *nbl,
                                                        const int *nbc, float4 *out, double *pgrad) {
    __shared__ float red[4][2 * ADJ_MAX_CLS];
    const int tp = K.tp;
    const int i = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> K.tpsh);
    const int t = threadIdx.x & (tp - 1);
    const bool valid = i < K.N;
    float ax = 0.f, ay = 0.f, az = 0.f;
    float g[2 * ADJ_MAX_CLS];
#pragma unroll
    for (int c = 0; c < 2 * ADJ_MAX_CLS; ++c) g[c] = 0.f;
    if (valid) {
        const float4 ri = pos[i];
        const int ti = adj_type(ri);
        float4 wi = make_float4(0.f, 0.f, 0.f, 0.f);
        if (MODE == 1) wi = w[i];
        const int cnt = min(nbc[i], K.maxnb);
        const int *row = nbl + (size_t)i * K.maxnb;
        for (int k = t; k < cnt; k += tp) {
            const int j = row[k];
            const float4 rj = pos[j];
            float dx, dy, dz;
            const float d2 = dist_sq_mic(ri.x, ri.y, ri.z, rj.x, rj.y, rj.z, K.L0, K.L1, K.L2, dx, dy, dz);
            const AdjPairC &q = K.pc[ti * K.nt + adj_type(rj)];
            if (d2 >= q.cut2) continue;
            const AdjPairEval e = adj_pair(q, d2);
            if (MODE == 0) {
                ax += e.s * dx;
                ay += e.s * dy;
                az += e.s * dz;
            } else {
                const float4 wj = w[j];
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
            }
        }
    }
    for (int mm = 1; mm < tp; mm <<= 1) {
        ax += __shfl_xor(ax, mm, 64);
        ay += __shfl_xor(ay, mm, 64);
        az += __shfl_xor(az, mm, 64);
    }
    if (valid && t == 0) out[i] = make_float4(ax, ay, az, 0.f);
    if (MODE == 1) {
        const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
        for (int c = 0; c < 2 * ADJ_MAX_CLS; ++c) {
            const float v = wave_sum_f(g[c]);
            if (lane == 0) red[wid][c] = v;
        }
        __syncthreads();
        if (threadIdx.x < 2 * ADJ_MAX_CLS) {
            double s = 0.0;
            for (int k = 0; k < (int)(blockDim.x >> 6); ++k) s += (double)red[k][threadIdx.x];
            pgrad[(size_t)blockIdx.x * (2 * ADJ_MAX_CLS) + threadIdx.x] = s;
        }
    }
}

// the list check of k_adj_check for one particle, folded into the kernel
// that produces (or precedes) the positions the next list is wanted for:
// flag[b] = 1 when r has moved more than skin/2 from its reference
__device__ __forceinline__ void adj_skin_flag(const AdjK &K, const float4 r, const float4 q, int *flag, int b) {
    float dx, dy, dz;
    if (dist_sq_mic(r.x, r.y, r.z, q.x, q.y, q.z, K.L0, K.L1, K.L2, dx, dy, dz) > K.skin2q) flag[b] = 1;
}

// forward leap-frog step of particle i from its force (nparts partial sums);
// rec (optional) receives the new position; with bnext >= 0 the new position
// also takes the next step's list check (flag[bnext] against rref)
__global__ void __launch_bounds__(256) k_adj_step(AdjK K, float4 *pos, float4 *vel, const float4 *part, int nparts,
                                                  float4 *rec, const float4 *rref, int *flag, int bnext) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= K.N) return;
    float fx = 0.f, fy = 0.f, fz = 0.f;
    for (int c = 0; c < nparts; ++c) {
        const float4 p = part[(size_t)c * K.N + i];
        fx += p.x;
        fy += p.y;
        fz += p.z;
    }
    float4 v = vel[i], r = pos[i];
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
    vel[i] = v;
    pos[i] = r;
    if (rec) rec[i] = r;
    if (bnext >= 0) adj_skin_flag(K, r, rref[i], flag, bnext);
}

// smoothed pair histogram of one frame over its list of radius rmax + 5 w
// (unordered pairs: j > i), K.tp lanes per particle, one LDS histogram per
// block written to hpart[block][ncls * bins]
__global__ void __launch_bounds__(256) k_adj_rdf_list(AdjK K, const float4 *pos, const int *nbl, const int *nbc,
                                                      int maxnb, float *hpart) {
    __shared__ float h[ADJ_MAX_CLS * ADJ_MAX_BINS];
    const int nh = K.ncls * K.bins;
    for (int t = threadIdx.x; t < nh; t += blockDim.x) h[t] = 0.f;
    __syncthreads();
    const int i = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> K.tpsh);
    const int tl = threadIdx.x & (K.tp - 1);
    if (i < K.N) {
        const float4 ri = pos[i];
        const int ti = adj_type(ri);
        const int cnt = min(nbc[i], maxnb);
        const int *row = nbl + (size_t)i * maxnb;
        for (int k = tl; k < cnt; k += K.tp) {
            const int j = row[k];
            if (j <= i) continue;
            const float4 rj = pos[j];
            float dx, dy, dz;
            const float d2 = dist_sq_mic(ri.x, ri.y, ri.z, rj.x, rj.y, rj.z, K.L0, K.L1, K.L2, dx, dy, dz);
            if (d2 >= K.rcut2) continue;
            const float d = sqrtf(d2);
            const int c = K.pc[ti * K.nt + adj_type(rj)].cls;
            const int k0 = max(0, (int)floorf((d - 5.0f * K.wid) / K.dr - 0.5f));
            const int k1 = min(K.bins - 1, (int)ceilf((d + 5.0f * K.wid) / K.dr - 0.5f));
            for (int kb = k0; kb <= k1; ++kb) {
                const float x = d - ((float)kb + 0.5f) * K.dr;
                const float kv = __expf(-0.5f * x * x * K.inv_w2) - K.kfloor;
                if (kv > 0.f) atomicAdd(&h[c * K.bins + kb], kv);
            }
        }
    }
    __syncthreads();
    float *dst = hpart + (size_t)blockIdx.x * nh;
    for (int t = threadIdx.x; t < nh; t += blockDim.x) dst[t] = h[t];
}

// dL/dr_i of one frame given G = dL/dH over the frame's list (all j of i):
// sum_j (sum_k G[c][k] K'(d - r_k)) d_ij / d, K.tp lanes per particle
__global__ void __launch_bounds__(256) k_adj_rdf_grad_list(AdjK K, const float4 *pos, const float *G, const int *nbl,
                                                           const int *nbc, int maxnb, float4 *out) {
    __shared__ float sg[ADJ_MAX_CLS * ADJ_MAX_BINS];
    const int nh = K.ncls * K.bins;
    for (int t = threadIdx.x; t < nh; t += blockDim.x) sg[t] = G[t];
    __syncthreads();
    const int i = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> K.tpsh);
    const int tl = threadIdx.x & (K.tp - 1);
    float ax = 0.f, ay = 0.f, az = 0.f;
    if (i < K.N) {
        const float4 ri = pos[i];
        const int ti = adj_type(ri);
        const int cnt = min(nbc[i], maxnb);
        const int *row = nbl + (size_t)i * maxnb;
        for (int k = tl; k < cnt; k += K.tp) {
            const float4 rj = pos[row[k]];
            float dx, dy, dz;
            const float d2 = dist_sq_mic(ri.x, ri.y, ri.z, rj.x, rj.y, rj.z, K.L0, K.L1, K.L2, dx, dy, dz);
            if (d2 >= K.rcut2) continue;
            const float d = sqrtf(d2);
            const int c = K.pc[ti * K.nt + adj_type(rj)].cls;
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
        }
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

// H[k] += sum over block partials, one block of 256 threads per bin k
// (each thread the partials t, t + 256, ..., then a fixed-order block sum)
__global__ void __launch_bounds__(256) k_adj_rdf_reduce(const float *hpart, int nblocks, int nh, double *H) {
    __shared__ double sred[4];
    const int k = blockIdx.x;
    double s = 0.0;
    for (int b = threadIdx.x; b < nblocks; b += blockDim.x) s += (double)hpart[(size_t)b * nh + k];
    s = adj_block_sum(s, sred);
    if (threadIdx.x == 0) H[k] += s;
}

// backward step n: lambda_r += J w (nparts partial sums) (+ frame gradient);
// then, unless n == 0, lambda_v += dt lambda_r and w = dt/m lambda_v for step
// n-1.  Block 0 also adds this step's parameter-gradient block partials
// (fixed order).  With rnext, the positions of step n-1 take their list
// check (flag[bnext] against rref).
__global__ void __launch_bounds__(256) k_adj_back(AdjK K, const float4 *vel, float4 *lr, float4 *lv, float4 *w,
                                                  const float4 *part, int nparts, const float4 *rpart, int advance,
                                                  const double *pgrad, int npg, double *pgrad_tot,
                                                  const float4 *rnext, const float4 *rref, int *flag, int bnext) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (blockIdx.x == 0 && pgrad) {
        // the step's parameter-gradient block partials: thread t the blocks
        // t, t + 256, ... of every component, then per component the wave
        // sums and the waves in index order (one barrier for all of them)
        __shared__ double sred[4 * 2 * ADJ_MAX_CLS];
        const int nc = 2 * K.ncls;
        const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
        double v[2 * ADJ_MAX_CLS];
#pragma unroll
        for (int c = 0; c < 2 * ADJ_MAX_CLS; ++c) v[c] = 0.0;
        for (int b = threadIdx.x; b < npg; b += blockDim.x)
#pragma unroll
            for (int c = 0; c < 2 * ADJ_MAX_CLS; ++c)
                if (c < nc) v[c] += pgrad[(size_t)b * (2 * ADJ_MAX_CLS) + c];
#pragma unroll
        for (int c = 0; c < 2 * ADJ_MAX_CLS; ++c) {
            if (c >= nc) continue;
            const double x = wave_sum_d(v[c]);
            if (lane == 0) sred[wid * (2 * ADJ_MAX_CLS) + c] = x;
        }
        __syncthreads();
        if ((int)threadIdx.x < nc) {
            double sc = 0.0;
            for (int k = 0; k < (int)(blockDim.x >> 6); ++k) sc += sred[k * (2 * ADJ_MAX_CLS) + threadIdx.x];
            pgrad_tot[threadIdx.x] += sc;
        }
    }
    if (i >= K.N) return;
    float4 a = lr[i];
    if (part)
        for (int c = 0; c < nparts; ++c) {
            const float4 p = part[(size_t)c * K.N + i];
            a.x += p.x;
            a.y += p.y;
            a.z += p.z;
        }
    if (rpart) {
        const float4 p = rpart[i];
        a.x += p.x;
        a.y += p.y;
        a.z += p.z;
    }
    lr[i] = a;
    if (advance) {
        float4 b = lv[i];
        b.x += K.dt * a.x;
        b.y += K.dt * a.y;
        b.z += K.dt * a.z;
        lv[i] = b;
        const float f = K.dt / vel[i].w;
        w[i] = make_float4(f * b.x, f * b.y, f * b.z, 0.f);
    }
    if (rnext) adj_skin_flag(K, rnext[i], rref[i], flag, bnext);
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
    int chk = 0;                 // list checks so far (flag parity)
    bool prechecked = false;     // the next list's check ran in the kernel before it
    size_t nbl_cap = 0;          // allocated list slots
    hipStream_t stream = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    float fwd_ms = 0.f, bwd_ms = 0.f;
    bool have_forward = false;
    // device
    float4 *pos = nullptr, *vel = nullptr, *fpart = nullptr, *rpart = nullptr, *rref = nullptr;
    int *nbl = nullptr, *nbc = nullptr, *flag = nullptr;
    int *rnbl = nullptr, *rnbc = nullptr;   // list of one frame (radius rmax + 5 w)
    float4 *ck_r = nullptr, *ck_v = nullptr, *seg = nullptr;
    float4 *lr = nullptr, *lv = nullptr, *w = nullptr;
    double *pgl = nullptr, *pgrad_tot = nullptr, *H = nullptr;
    float *hpart = nullptr, *G = nullptr;
};

static int adj_free(gmd_adj *a) {
    if (!a) return 0;
    void *ptrs[] = {a->pos, a->vel, a->fpart, a->rpart, a->rref, a->nbl, a->nbc, a->flag, a->rnbl, a->rnbc,
                    a->ck_r, a->ck_v, a->seg, a->lr, a->lv, a->w, a->pgl, a->pgrad_tot, a->H, a->hpart, a->G};
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
        if (hipMalloc((void **)&a->nbl, need * sizeof(int)) != hipSuccess) return fail("gmd_adj: list allocation");
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
    a->nck = (d.nsteps + d.ckpt_every - 1) / d.ckpt_every;
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
    ATRY(hipMalloc((void **)&a->pos, N * sizeof(float4)));
    ATRY(hipMalloc((void **)&a->vel, N * sizeof(float4)));
    ATRY(hipMalloc((void **)&a->fpart, N * sizeof(float4)));
    ATRY(hipMalloc((void **)&a->rpart, N * sizeof(float4)));
    ATRY(hipMalloc((void **)&a->rnbl, N * (size_t)a->rmaxnb * sizeof(int)));
    ATRY(hipMalloc((void **)&a->rnbc, N * sizeof(int)));
    ATRY(hipMalloc((void **)&a->rref, N * sizeof(float4)));
    ATRY(hipMalloc((void **)&a->nbc, N * sizeof(int)));
    ATRY(hipMalloc((void **)&a->flag, 4 * sizeof(int)));
    ATRY(hipMalloc((void **)&a->ck_r, (size_t)a->nck * N * sizeof(float4)));
    ATRY(hipMalloc((void **)&a->ck_v, (size_t)a->nck * N * sizeof(float4)));
    ATRY(hipMalloc((void **)&a->seg, (size_t)(d.ckpt_every + 1) * N * sizeof(float4)));
    ATRY(hipMalloc((void **)&a->lr, N * sizeof(float4)));
    ATRY(hipMalloc((void **)&a->lv, N * sizeof(float4)));
    ATRY(hipMalloc((void **)&a->w, N * sizeof(float4)));
    ATRY(hipMalloc((void **)&a->pgl, (size_t)a->gl * 2 * ADJ_MAX_CLS * sizeof(double)));
    ATRY(hipMalloc((void **)&a->pgrad_tot, 2 * ADJ_MAX_CLS * sizeof(double)));
    ATRY(hipMalloc((void **)&a->H, (size_t)ncls * d.rdf_bins * sizeof(double)));
    ATRY(hipMalloc((void **)&a->hpart, (size_t)a->gl * ncls * d.rdf_bins * sizeof(float)));
    ATRY(hipMalloc((void **)&a->G, (size_t)ncls * d.rdf_bins * sizeof(float)));
#undef ATRY
    *out = a;
    return 0;
}

int gmd_adj_destroy(gmd_adj *a) { return adj_free(a); }

// blocks of a list build: ADJ_BT / 64 particles each
static dim3 adj_build_grid(const gmd_adj *a) { return dim3((a->K.N + ADJ_BT / 64 - 1) / (ADJ_BT / 64)); }

// the list of one frame (radius rmax + 5 w) at the positions pos; list
// overflow is recorded in flag[3]
static void adj_frame_list(gmd_adj *a, const float4 *pos) {
    hipLaunchKernelGGL(k_adj_build, adj_build_grid(a), dim3(ADJ_BT), 0, a->stream, a->K, pos, (float4 *)nullptr,
                       a->rnbl, a->rnbc, a->rmaxnb, a->K.rcut2, a->flag, -1, 1, a->flag + 3);
}

static void adj_rdf_frame(gmd_adj *a, const float4 *pos) {
    const int nh = a->K.ncls * a->K.bins;
    adj_frame_list(a, pos);
    hipLaunchKernelGGL(k_adj_rdf_list, dim3(a->gl), dim3(256), 0, a->stream, a->K, pos, (const int *)a->rnbl,
                       (const int *)a->rnbc, a->rmaxnb, a->hpart);
    hipLaunchKernelGGL(k_adj_rdf_reduce, dim3(nh), dim3(256), 0, a->stream, a->hpart, a->gl, nh, a->H);
}

// dL/dr of the frame at pos into a->rpart
static void adj_rdf_grad(gmd_adj *a, const float4 *pos) {
    adj_frame_list(a, pos);
    hipLaunchKernelGGL(k_adj_rdf_grad_list, dim3(a->gl), dim3(256), 0, a->stream, a->K, pos, (const float *)a->G,
                       (const int *)a->rnbl, (const int *)a->rnbc, a->rmaxnb, a->rpart);
}

// a neighbour list valid for the positions pos: the skin check (unless a
// build is forced), then the build where it is needed
static void adj_list(gmd_adj *a, const float4 *pos, bool force) {
    const int b = a->chk & 1;
    if (!force && !a->prechecked)
        hipLaunchKernelGGL(k_adj_check, dim3((a->K.N + 255) / 256), dim3(256), 0, a->stream, a->K, pos,
                           (const float4 *)a->rref, a->flag, b);
    a->prechecked = false;
    hipLaunchKernelGGL(k_adj_build, adj_build_grid(a), dim3(ADJ_BT), 0, a->stream, a->K, pos, a->rref, a->nbl,
                       a->nbc, a->K.maxnb, a->K.cps2, a->flag, b, force ? 1 : 0, a->flag + 2);
    ++a->chk;
}

static int adj_reset_lists(gmd_adj *a) {
    a->chk = 0;
    a->prechecked = false;
    HIPCHECK(hipMemsetAsync(a->flag, 0, 4 * sizeof(int), a->stream));
    return 0;
}

static int adj_check_lists(gmd_adj *a) {
    int f[4];
    HIPCHECK(hipMemcpy(f, a->flag, sizeof f, hipMemcpyDeviceToHost));
    if (f[2] > 0)
        return fail("gmd_adj: a neighbour list of %d entries exceeds its %d slots", f[2], a->K.maxnb);
    if (f[3] > 0)
        return fail("gmd_adj: a frame list of %d entries exceeds its %d slots", f[3], a->rmaxnb);
    return 0;
}

// one forward step from (pos, vel); rec receives r_{n+1} when not null; the
// list is rebuilt when force (a checkpoint) or when the skin check asks
static void adj_step(gmd_adj *a, float4 *rec, bool force) {
    adj_list(a, a->pos, force);
    hipLaunchKernelGGL(k_adj_pairs_list<0>, dim3(a->gl), dim3(256), 0, a->stream, a->K, (const float4 *)a->pos,
                       (const float4 *)nullptr, (const int *)a->nbl, (const int *)a->nbc, a->fpart,
                       (double *)nullptr);
    // the new positions take the next step's list check here
    hipLaunchKernelGGL(k_adj_step, dim3((a->K.N + 255) / 256), dim3(256), 0, a->stream, a->K, a->pos, a->vel,
                       (const float4 *)a->fpart, 1, rec, (const float4 *)a->rref, a->flag, a->chk & 1);
    a->prechecked = true;
}

int gmd_adj_forward(gmd_adj *a, const float *params, const float *r0, const float *v0, double *H, float *r_end,
                    float *v_end) {
    if (!a || !params || !r0 || !v0 || !H) return fail("gmd_adj_forward: null argument");
    if (adj_set_params(a, params)) return -1;
    const int N = a->d.N, S = a->d.nsteps, C = a->d.ckpt_every, E = a->d.rdf_every;
    std::vector<float4> hr(N), hv(N);
    for (int i = 0; i < N; ++i) {
        int t = a->ptype[i];
        float tf;
        memcpy(&tf, &t, 4);
        hr[i] = make_float4(r0[3 * i], r0[3 * i + 1], r0[3 * i + 2], tf);
        hv[i] = make_float4(v0[3 * i], v0[3 * i + 1], v0[3 * i + 2], a->mass[i]);
    }
    hipStream_t st = a->stream;
    HIPCHECK(hipMemcpyAsync(a->pos, hr.data(), N * sizeof(float4), hipMemcpyHostToDevice, st));
    HIPCHECK(hipMemcpyAsync(a->vel, hv.data(), N * sizeof(float4), hipMemcpyHostToDevice, st));
    const int nh = a->K.ncls * a->K.bins;
    HIPCHECK(hipMemsetAsync(a->H, 0, nh * sizeof(double), st));
    if (adj_reset_lists(a)) return -1;
    HIPCHECK(hipEventRecord(a->e0, st));
    for (int n = 0; n < S; ++n) {
        if (n % C == 0) {
            HIPCHECK(hipMemcpyAsync(a->ck_r + (size_t)(n / C) * N, a->pos, N * sizeof(float4),
                                    hipMemcpyDeviceToDevice, st));
            HIPCHECK(hipMemcpyAsync(a->ck_v + (size_t)(n / C) * N, a->vel, N * sizeof(float4),
                                    hipMemcpyDeviceToDevice, st));
        }
        if (n % E == 0) adj_rdf_frame(a, a->pos);
        adj_step(a, nullptr, n % C == 0);
    }
    if (S % E == 0) adj_rdf_frame(a, a->pos);
    HIPCHECK(hipGetLastError());
    HIPCHECK(hipEventRecord(a->e1, st));
    HIPCHECK(hipEventSynchronize(a->e1));
    HIPCHECK(hipEventElapsedTime(&a->fwd_ms, a->e0, a->e1));
    HIPCHECK(hipMemcpy(H, a->H, nh * sizeof(double), hipMemcpyDeviceToHost));
    if (adj_check_lists(a)) return -1;
    if (r_end || v_end) {
        HIPCHECK(hipMemcpy(hr.data(), a->pos, N * sizeof(float4), hipMemcpyDeviceToHost));
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
    HIPCHECK(hipMemsetAsync(a->lr, 0, N * sizeof(float4), st));
    HIPCHECK(hipMemsetAsync(a->lv, 0, N * sizeof(float4), st));
    HIPCHECK(hipMemsetAsync(a->pgrad_tot, 0, 2 * ADJ_MAX_CLS * sizeof(double), st));
    if (adj_reset_lists(a)) return -1;
    HIPCHECK(hipEventRecord(a->e0, st));
    const dim3 gu((N + 255) / 256);
    // lambda_r(S) = dL/dr_S, then lambda_v, w of step S-1; recompute r_S from the last checkpoint first
    const int last = a->nck - 1;
    // recompute the last segment (it also provides r_S)
    bool have_seg = false;
    int seg_n0 = -1;
    for (int sgm = last; sgm >= 0; --sgm) {
        const int n0 = sgm * C, n1 = std::min(S, n0 + C);
        HIPCHECK(hipMemcpyAsync(a->pos, a->ck_r + (size_t)sgm * N, N * sizeof(float4), hipMemcpyDeviceToDevice, st));
        HIPCHECK(hipMemcpyAsync(a->vel, a->ck_v + (size_t)sgm * N, N * sizeof(float4), hipMemcpyDeviceToDevice, st));
        HIPCHECK(hipMemcpyAsync(a->seg, a->pos, N * sizeof(float4), hipMemcpyDeviceToDevice, st));
        // the segment's steps repeat the forward's: the list is rebuilt at the
        // checkpoint as it was there
        for (int k = 0; k < n1 - n0; ++k) adj_step(a, a->seg + (size_t)(k + 1) * N, k == 0);
        if (!have_seg) {
            // start of the adjoint: frame gradient at r_S, then lambda_v and w of step S-1
            const float4 *rS = a->seg + (size_t)(n1 - n0) * N;
            const float4 *rp = nullptr;
            if (S % E == 0) {
                adj_rdf_grad(a, rS);
                rp = a->rpart;
            }
            hipLaunchKernelGGL(k_adj_back, gu, dim3(256), 0, st, a->K, a->vel, a->lr, a->lv, a->w,
                               (const float4 *)nullptr, 0, rp, 1, (const double *)nullptr, 0, a->pgrad_tot,
                               (const float4 *)nullptr, (const float4 *)nullptr, a->flag, -1);
            have_seg = true;
        }
        seg_n0 = n0;
        for (int n = n1 - 1; n >= n0; --n) {
            const float4 *rn = a->seg + (size_t)(n - seg_n0) * N;
            adj_list(a, rn, n == n1 - 1);
            hipLaunchKernelGGL(k_adj_pairs_list<1>, dim3(a->gl), dim3(256), 0, st, a->K, rn, (const float4 *)a->w,
                               (const int *)a->nbl, (const int *)a->nbc, a->fpart, a->pgl);
            const float4 *rp = nullptr;
            if (n % E == 0) {
                adj_rdf_grad(a, rn);
                rp = a->rpart;
            }
            // the positions of step n-1 (same segment) take their list check here
            const float4 *rnext = n > seg_n0 ? rn - N : nullptr;
            hipLaunchKernelGGL(k_adj_back, gu, dim3(256), 0, st, a->K, a->vel, a->lr, a->lv, a->w,
                               (const float4 *)a->fpart, 1, rp, n > 0 ? 1 : 0, (const double *)a->pgl, a->gl,
                               a->pgrad_tot, rnext, (const float4 *)a->rref, a->flag, a->chk & 1);
            a->prechecked = rnext != nullptr;
        }
    }
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
