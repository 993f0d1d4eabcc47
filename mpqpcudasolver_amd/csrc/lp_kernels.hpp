// lp_kernels.hpp — the LP kernels (gfx950).
//
//   feas_kernel  one workgroup per candidate: the feasibility LP
//                (replaces simplex_gpu_feasibility, batched_simplex.cu:
//                990-1258, and its kernels a3/a4/a10-a15/a22/a23/a27).
//   opt_kernel_t one workgroup per feasible candidate (or a persistent grid
//                drawing candidates from a work counter): phase-1 dual
//                simplex, drive-out, phase-2 primal simplex, in FP64 or in
//                FP32 with FP64 certification (opt_kernel.hpp; replaces
//                dual_simplex_gpu_optimality, batched_simplex.cu:1260-1721).
#pragma once
#include "lp_engine.hpp"

// ---------------------------------------------------------------------
// Candidate-level arguments
// ---------------------------------------------------------------------
struct FeasArgs {
    DevProb P;
    DevOpts O;
    int n, level, kw;
    const int *sets;    // n x kw ascending constraint ids, -1 padded
    const int *parent;  // n: row of the parent in fstore_prev, -1 = cold
    const unsigned char *fstore_prev;
    unsigned char *fstore_cur;
    long long fstride;
    int store;
    DevRecord *rec;     // n
    int *fbasis;        // n x M1 or null
    const int *licq_fail;  // n: 1 = S failed the LICQ screen (no LP), or null
};

struct OptArgs {
    DevProb P;
    DevOpts O;
    int n, level, kw;
    const int *list;      // candidate ids to solve: n of them, or *n_dev
    const int *n_dev;     // device-side length of list, or null
    int *counter;         // work counter of a persistent launch (starts at 0), or
                          // null: workgroup b solves list[b]
    const int *sets;      // by candidate
    const int *p1parent;  // by candidate: parent row in ostore_prev, -1 = cold
    const unsigned char *ostore_prev;
    unsigned char *ostore_cur;
    long long ostride;
    int store;            // keep clean phase-1 states for the next level
    int store32;          // FP64 kernel: keep them rounded to FP32 (mixed runs)
    int force_cold;       // ignore p1parent (FP64 re-solve of the mixed path)
    DevRecord *rec;       // by candidate
    int *b1, *b2;         // by candidate x M2, or null
    int *fb_list;         // mixed: candidates whose FP32 result failed
    int *fb_count;        //        certification (appended), and their count
    long long *prof;      // phase cycle counts, 16 per workgroup (MPQP_PROFILE builds), or null
    unsigned char *gtab;  // split tableaus: rows [split_rows, M2) of each workgroup's in global
    long long gtab_stride;  // memory (the tableau does not fit in LDS), or null
    int split_rows;       // rows of a split tableau held in LDS (even), with the cost row
    int stage_passes;     // register tableau: passes that stage its rows through LDS
};

// Byte layout of one stored state: T (rows x cols doubles, contiguous) then
// basis (M ints) then nonbasic (K ints).
__host__ __device__ inline long long state_bytes(int rows, int cols, int M, int K) {
    long long b = (long long)rows * cols * 8 + (long long)(M + K) * 4;
    return (b + 255) & ~255LL;
}

// ---------------------------------------------------------------------
// Feasibility LP
// ---------------------------------------------------------------------
// dst[0..n) = src[0..n) (doubles; both 16-byte aligned) by the workgroup:
// 16-byte vectors, eight in flight per thread, then the odd tail.
template <int NT>
__device__ __forceinline__ void copy_doubles(double *dst, const double *src, int n) {
    const int nv = n / 2, tid = threadIdx.x;
    const int4 *s4 = reinterpret_cast<const int4 *>(src);
    int4 *d4 = reinterpret_cast<int4 *>(dst);
    constexpr int UL = 8;
    int e0 = tid;
    for (; e0 + (UL - 1) * NT < nv; e0 += NT * UL) {
        int4 vv[UL];
#pragma unroll
        for (int u = 0; u < UL; ++u) vv[u] = s4[e0 + u * NT];
#pragma unroll
        for (int u = 0; u < UL; ++u) d4[e0 + u * NT] = vv[u];
    }
    for (int e = e0; e < nv; e += NT) d4[e] = s4[e];
    if ((n & 1) && tid == 0) dst[n - 1] = src[n - 1];
}

__host__ __device__ inline long long feas_lds_bytes(int M, int K, int n_c) {
    const int ld = K + 1;
    long long b = (long long)(M + 1) * ld * 8 + (long long)(M + 1) * 8 + (long long)(M + K) * 4 +
                  (long long)((n_c + 31) / 32) * 4;
    return (b + 15) & ~15LL;
}

// the feasibility LP's part of a candidate's record, the rest cleared (one
// thread)
__device__ __forceinline__ void feas_record(DevRecord &R, int level, int status, int iters, int feasible, double z) {
    R.level = level;
    R.feas_status = status;
    R.feas_iters = iters;
    R.feasible = feasible;
    R.z_feas = z;
    R.p1_status = R.p1_iters = R.kkt_feasible = R.p1_warm = 0;
    R.p2_status = R.p2_iters = R.final_set = 0;
    R.z1 = R.z2 = 0.0;
    R.repivots = 0;
    R.p1_clean = 0;
}

// rows of S linearly dependent (LICQ screen): no LP, no children
template <int NT>
__device__ __forceinline__ void feas_dependent(const FeasArgs &a, int c) {
    if (threadIdx.x == 0) feas_record(a.rec[c], a.level, ST_SINGULAR, 0, 0, 0.0);
    if (a.fbasis)
        for (int i = threadIdx.x; i < a.P.M1; i += NT) a.fbasis[(long long)c * a.P.M1 + i] = -1;
}

template <int NT>
__global__ __launch_bounds__(NT) void feas_kernel(FeasArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    __shared__ int sh_r, sh_q, sh_done, sh_feas;
    __shared__ double sh_z;
    const DevProb &P = a.P;
    const DevOpts &O = a.O;
    const int M = P.M1, K = P.K1, ld = K + 1;
    const int c = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & (MPQP_WAVE - 1);
    double *T = reinterpret_cast<double *>(smem);
    double *colq = T + (M + 1) * ld;
    int *basis = reinterpret_cast<int *>(colq + (M + 1));
    int *nonb = basis + M;
    unsigned *inS = reinterpret_cast<unsigned *>(nonb + K);
    const int nw = (P.n_c + 31) / 32;
    const DevTol tl = dev_tol64(O);

    if (a.licq_fail && a.licq_fail[c]) {
        feas_dependent<NT>(a, c);
        return;
    }
    for (int w = tid; w < nw; w += NT) inS[w] = 0u;
    __syncthreads();
    for (int t = tid; t < a.level; t += NT) {  // the members of S
        const int s = a.sets[(long long)c * a.kw + t];
        atomicOr(&inS[s >> 5], 1u << (s & 31));
    }
    const int par = a.parent[c];
    if (par >= 0 && O.warm) {
        const unsigned char *src = a.fstore_prev + (long long)par * a.fstride;
        const double *sT = reinterpret_cast<const double *>(src);
        copy_doubles<NT>(T, sT, M * ld);
        const int *sb = reinterpret_cast<const int *>(sT + M * ld);
        for (int i = tid; i < M; i += NT) basis[i] = sb[i];
        for (int k = tid; k < K; k += NT) nonb[k] = sb[M + k];
    } else {
        for (int e = tid; e < M * ld; e += NT) {
            const int i = e / ld, k = e - i * ld;
            T[e] = (k < K) ? P.A1[(long long)k * M + i] : P.xb1[i];
        }
        for (int i = tid; i < M; i += NT) basis[i] = K + i;
        for (int k = tid; k < K; k += NT) nonb[k] = k;
    }
    __syncthreads();

    auto cvar = [&](int var) -> double {
        const int s = var - K;
        return (s >= 0 && s < P.n_c && ((inS[s >> 5] >> (s & 31)) & 1u)) ? 1.0 : 0.0;
    };
    for (int i = tid; i < M; i += NT) colq[i] = cvar(basis[i]);
    __syncthreads();
    cost_row_cb<NT, double>(T, ld, M, K + 1, colq, [&](int j) { return j < K ? cvar(nonb[j]) : 0.0; });

    int status = ST_ITER_CAP, iters = 0, feasible = 0;
    double z = 0.0;
    for (int it = 0; it < O.max_iter_feas; ++it) {
        if (tid < MPQP_WAVE) { MPQP_PRIO_HI();
            // Dantzig pricing, lowest variable id on ties (min_idx_kernel :256-316)
            double v = 0.0;
            int key = -1, aux = -1;
            for (int k = lane; k < K; k += MPQP_WAVE) {
                const double d = T[M * ld + k];
                const int var = nonb[k];
                if (key < 0 || d < v || (d == v && var < key)) { v = d; key = var; aux = k; }
            }
            lex_min(v, key, aux);
            int done = 0, r = -1, fe = 0;
            double zz = 0.0;
            if (v > O.tol_minus_1) {
                double zs[MPQP_MAXS];
#pragma unroll
                for (int s = 0; s < MPQP_MAXS; ++s) {
                    const int i = lane + MPQP_WAVE * s;
                    zs[s] = (i < M) ? cvar(basis[i]) * T[i * ld + K] : 0.0;
                }
                zz = tree_sum(zs, M, lane);
                fe = (zz >= -O.feas_z_tol && zz <= O.feas_z_tol) ? 1 : 0;
                done = 1 + ST_OPTIMAL;
            } else {
                // ratio test, lowest row on ties (pivot_kernel_1_2 :901-942)
                r = primal_ratio_wave(flat_tab(T, ld), M, aux, K, tl);
                if (r < 0) done = 1 + ST_UNBOUNDED;
            }
            if (lane == 0) {
                sh_r = r;
                sh_q = aux;
                sh_done = done;
                sh_z = zz;
                sh_feas = fe;
            }
        }
        MPQP_PRIO_LO(); __syncthreads();
        if (sh_done) {
            status = sh_done - 1;
            z = sh_z;
            feasible = sh_feas;
            break;
        }
        const int r = sh_r, q = sh_q;
        pivot_rows_narrow<NT>(T, ld, M + 1, K + 1, r, q, colq, [&] {
            const int t = basis[r];
            basis[r] = nonb[q];
            nonb[q] = t;
        });
        ++iters;
    }

    if (tid == 0) feas_record(a.rec[c], a.level, status, iters, feasible, z);
    if (a.fbasis)
        for (int i = tid; i < M; i += NT) a.fbasis[(long long)c * M + i] = basis[i];
    if (a.store && feasible) {
        unsigned char *dst = a.fstore_cur + (long long)c * a.fstride;
        double *dT = reinterpret_cast<double *>(dst);
        copy_doubles<NT>(dT, T, M * ld);
        int *db = reinterpret_cast<int *>(dT + M * ld);
        for (int i = tid; i < M; i += NT) db[i] = basis[i];
        for (int k = tid; k < K; k += NT) db[M + k] = nonb[k];
    }
}

// ---------------------------------------------------------------------
// Optimality LP
// ---------------------------------------------------------------------
// slots per lane a reduction over n elements needs on one wave
__host__ __device__ inline int red_slots(int n) {
    const int s = (n + 63) / 64;
    return s <= 4 ? (s < 1 ? 1 : s) : (s <= 6 ? 6 : 8);
}

__device__ __forceinline__ double lam_entry(const DevProb &P, int j, int row) {
    if (row == P.M2 - P.n_c + j) return 0.0;
    return P.A2[(long long)(P.n_x + P.n_t + j) * P.M2 + row];
}

__device__ __forceinline__ int rfl(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ double rfl_d(double x) {
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readfirstlane((int)(unsigned)(b & 0xffffffffLL));
    const int hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// Combine predicates of the reference's reductions, branch-free (see
// tree_argmin).  Each returns "slot t takes slot u".
struct DminPred {  // dual_min_idx_kernel, batched_simplex.cu:177-198
    int mode_b;
    double stop_tol;
    __device__ bool operator()(double vt, int, int ct, double vu, int, int cu) const {
        const bool a = (vt > vu) | ((vt > vu - 1e-10) & (ct > cu));
        const bool b = ((vt > vu + 1e-10) & (ct > cu - 10)) | ((vt > vu) & (ct > cu - 5)) |
                       ((vu < stop_tol) & (vt < stop_tol) & (ct > cu + 10));
        return mode_b ? b : a;
    }
};

struct DratioPred {  // dual_pivot_kernel_1, batched_simplex.cu:841-866
    int mode;
    __device__ bool operator()(double vt, int it, int ct, double vu, int iu, int cu) const {
        const bool c0 = vt > vu;
        const bool c1 = c0 | ((vt >= vu - 1e-12) & (ct > cu + 2));
        const bool c2 = (vt >= vu - 1e-10) & (ct > cu + 5);
        const bool core = mode == 0 ? c0 : (mode == 1 ? c1 : c2);
        return (iu >= 0) & ((it < 0) | core);
    }
};

struct P2Pred {  // min_idx_kernel_optimal, batched_simplex.cu:343-344
    __device__ bool operator()(double vt, int, int ct, double vu, int, int cu) const {
        return (vt > vu) | ((ct > cu) & (vu < -1e-10));
    }
};

#include "opt_kernel.hpp"
#include "reg_kernel.hpp"
#include "feas_reg.hpp"
