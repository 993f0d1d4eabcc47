// kernels.hpp — the gfx950 kernels of libmpqp_hip.so: those of the LPs
// (lp_kernels.hpp, all that the kernels' own translation units include) and
// those of a call around them: the lists of a level, the LICQ screen and the
// root tableau.
//
//   root_kernel  once per problem: Gauss-Jordan build of the S = {} KKT basis
//                tableau of the optimality LP (replaces get_B_kernel_2 +
//                getrf of batched_simplex.cu:715-726,1435,1478 for the cold
//                start).
#pragma once
#include "lp_kernels.hpp"

// ---------------------------------------------------------------------
// Level-wise enumeration on the device: after the feasibility LPs the list
// of the feasible candidates and their children's offsets (S + {j} for j
// above max S, in parent order, j ascending), after the optimality LPs the
// work sums and the final sets, in order.  Counts that the host needs go
// into a host-visible mailbox, read when the chunk is done (and before its
// optimality launch where that is sized by the list).  With scans, lists and
// sums as launches of their own, and a copy and a wait for each count, small
// calls spent their time there: n=10 m=20 p=2 |S|<=2 in FP64 890 -> 418 us,
// n=20 m=40 p=4 |S|<=2 without allocation 1429 -> 909 us.  Each kernel here
// takes 3 to 5 us, most of it the launch.
//
// LEVEL_TILE candidates per block.  With more than one block, level_count
// writes each block's sums first and a block adds up those before it.
// ---------------------------------------------------------------------
#define LEVEL_NT 256
#define LEVEL_TILE 1024
// Ints of final sets that fit in the mailbox; more take a copy and a wait of
// their own, 70 us (n=10 m=20 p=2: 0.40 -> 0.47 ms a call).  1,024, 4,096 and
// 65,536 gave the same times as 16,384 from 211 to 39,774 candidates.
#define LEVEL_MAIL_ROWS 16384

struct LevelMail {
    long long children;          // of the chunk's feasible candidates
    int nf, final, fb, pad;      // feasible candidates, final sets, failed certifications
    unsigned long long sums[6];  // see level_sums
    int rows[LEVEL_MAIL_ROWS];   // the final sets (kw ints each), if they fit
};

struct LevelArgs {
    const DevRecord *rec;
    const int *sets;
    int n, kw, level, n_c, emit;  // emit: collect the final sets
    int2 *bsum;                   // per block: feasible and children, or final sets
    int *list, *off;              // feasible candidates; first child of each candidate
    int *ctr;                     // 4 counters of the optimality launches, [3]: length of the list
    unsigned long long *sums;     // 6
    int *rows;                    // final sets, kw ints each
    LevelMail *mail;
};

// max S + 1 .. n_c - 1 extend a feasible candidate of this level
__device__ __forceinline__ int child_first(const int *sets, int c, int kw, int level) {
    return level > 0 ? sets[(long long)c * kw + level - 1] + 1 : 0;
}

__device__ __forceinline__ int2 level_flags(const LevelArgs &a, int c, bool fin) {
    if (c >= a.n) return make_int2(0, 0);
    if (fin) return make_int2(a.emit && a.rec[c].final_set ? 1 : 0, 0);
    const int f = a.rec[c].feasible ? 1 : 0;
    return make_int2(f, f ? a.n_c - child_first(a.sets, c, a.kw, a.level) : 0);
}

// Work sums for the statistics: [0] feasibility pivots; [1] phase-1 / [2]
// phase-2 pivots of the optimality LPs kept in the first precision; [3] / [4]
// those of the LPs re-solved in FP64; [5] re-solves.
__device__ __forceinline__ void level_sums(const LevelArgs &a, int c, unsigned long long (&s)[6]) {
    if (c >= a.n) return;
    const DevRecord &r = a.rec[c];
    const bool rs = r.repivots != 0;
    s[0] += (unsigned long long)r.feas_iters;
    s[1] += (unsigned long long)(rs ? 0 : r.p1_iters);
    s[2] += (unsigned long long)(rs ? 0 : r.p2_iters);
    s[3] += (unsigned long long)(rs ? r.p1_iters : 0);
    s[4] += (unsigned long long)(rs ? r.p2_iters : 0);
    s[5] += (unsigned long long)r.repivots;
}

// the block's sums, added to out (LDS, cleared before)
__device__ __forceinline__ void level_sums_add(unsigned long long (&v)[6], unsigned long long *out) {
#pragma unroll
    for (int i = 0; i < 6; ++i) {
#pragma unroll
        for (int d = MPQP_WAVE / 2; d > 0; d >>= 1) v[i] += __shfl_xor(v[i], d, MPQP_WAVE);
        if (threadIdx.x % MPQP_WAVE == 0 && v[i]) atomicAdd(&out[i], v[i]);
    }
    __syncthreads();
}

// Exclusive prefix of v over the block's threads, the block's total in tot.
__device__ __forceinline__ int2 block_prefix(int2 v, int2 &tot) {
    __shared__ int2 ws[LEVEL_NT / MPQP_WAVE];
    const int lane = threadIdx.x % MPQP_WAVE, wave = threadIdx.x / MPQP_WAVE;
    int2 x = v;
#pragma unroll
    for (int d = 1; d < MPQP_WAVE; d <<= 1) {
        const int ox = __shfl_up(x.x, d, MPQP_WAVE), oy = __shfl_up(x.y, d, MPQP_WAVE);
        if (lane >= d) {
            x.x += ox;
            x.y += oy;
        }
    }
    __syncthreads();
    if (lane == MPQP_WAVE - 1) ws[wave] = x;
    __syncthreads();
    int2 base = make_int2(0, 0);
    tot = make_int2(0, 0);
#pragma unroll
    for (int w = 0; w < LEVEL_NT / MPQP_WAVE; ++w) {
        if (w < wave) {
            base.x += ws[w].x;
            base.y += ws[w].y;
        }
        tot.x += ws[w].x;
        tot.y += ws[w].y;
    }
    return make_int2(base.x + x.x - v.x, base.y + x.y - v.y);
}

// FIN: the final sets and the work sums, else the feasible candidates.
template <bool FIN>
__global__ __launch_bounds__(LEVEL_NT) void level_count(LevelArgs a) {
    __shared__ unsigned long long s[6];
    if (FIN && threadIdx.x < 6) s[threadIdx.x] = 0ull;
    __syncthreads();
    unsigned long long w[6] = {};
    int2 v = make_int2(0, 0);
    for (int u = threadIdx.x; u < LEVEL_TILE; u += LEVEL_NT) {
        const int c = blockIdx.x * LEVEL_TILE + u;
        const int2 f = level_flags(a, c, FIN);
        v.x += f.x;
        v.y += f.y;
        if (FIN) level_sums(a, c, w);
    }
    int2 tot;
    block_prefix(v, tot);
    if (FIN) level_sums_add(w, s);
    if (threadIdx.x == 0) a.bsum[blockIdx.x] = tot;
    if (FIN && threadIdx.x < 6) atomicAdd(&a.sums[threadIdx.x], s[threadIdx.x]);
}

template <bool FIN>
__global__ __launch_bounds__(LEVEL_NT) void level_write(LevelArgs a) {
    __shared__ unsigned long long s[6];
    __shared__ long long before[2];
    const bool one = gridDim.x == 1;
    if (threadIdx.x < 6) s[threadIdx.x] = 0ull;
    if (threadIdx.x < 2) before[threadIdx.x] = 0;
    __syncthreads();
    long long px = 0, py = 0;
    for (int b = threadIdx.x; b < (int)blockIdx.x; b += LEVEL_NT) {
        px += a.bsum[b].x;
        py += a.bsum[b].y;
    }
    if (px) atomicAdd((unsigned long long *)&before[0], (unsigned long long)px);
    if (py) atomicAdd((unsigned long long *)&before[1], (unsigned long long)py);
    __syncthreads();
    px = before[0];
    py = before[1];
    unsigned long long w[6] = {};
    for (int u = 0; u < LEVEL_TILE; u += LEVEL_NT) {
        const int c = blockIdx.x * LEVEL_TILE + u + threadIdx.x;
        if (blockIdx.x * LEVEL_TILE + u >= a.n) break;
        const int2 f = level_flags(a, c, FIN);
        if (FIN && one) level_sums(a, c, w);
        int2 tot;
        const int2 e = block_prefix(f, tot);
        const int pos = (int)(px + e.x);
        if constexpr (!FIN) {
            if (c < a.n) a.off[c] = (int)(py + e.y);
            if (f.x) a.list[pos] = c;
        } else if (f.x) {
            const int *S = a.sets + (long long)c * a.kw;
            for (int t = 0; t < a.kw; ++t) {
                const long long at = (long long)pos * a.kw + t;
                a.rows[at] = S[t];
                if (at < LEVEL_MAIL_ROWS) a.mail->rows[at] = S[t];
            }
        }
        px += tot.x;
        py += tot.y;
    }
    if (FIN && one) level_sums_add(w, s);
    if (blockIdx.x != gridDim.x - 1) return;
    if constexpr (!FIN) {
        if (threadIdx.x < 6) a.sums[threadIdx.x] = 0ull;
        if (threadIdx.x == 0) {
            a.ctr[0] = a.ctr[1] = a.ctr[2] = 0;
            a.ctr[3] = (int)px;
            a.mail->nf = (int)px;
            a.mail->children = py;
        }
    } else {
        if (threadIdx.x < 6) a.mail->sums[threadIdx.x] = one ? s[threadIdx.x] : a.sums[threadIdx.x];
        if (threadIdx.x == 0) {
            a.mail->final = (int)px;
            a.mail->fb = a.ctr[1];
        }
    }
}

// Children of parents [p0, p0 + pn) of a chunk: parent p0 + t's first child
// is row off[t] of the range; par holds chunk-wide parent indices
// (their rows in the parent chunk's state stores), p1par the parent whenever
// its phase 1 ended optimal (its phase-1 state warm-starts the child), else
// -1.  CHILD_LANES lanes per parent, a child each: 4, 16 and 64 take the same
// time, one lane 1 to 2% of a call more (n=30 m=62 p=8 |S|<=2 2.26 -> 2.30 ms).
#define CHILD_LANES 16
static __global__ __launch_bounds__(256) void child_write(const DevRecord *prec, const int *psets, const int *off, int p0, int pn,
                                                          int kw, int level, int n_c, int *sets, int *par, int *p1par) {
    const int t = (blockIdx.x * 256 + threadIdx.x) / CHILD_LANES, g = threadIdx.x % CHILD_LANES;
    if (t >= pn) return;
    const int pi = p0 + t;
    if (!prec[pi].feasible) return;
    const int *ps = psets + (long long)pi * kw;
    const int j0 = child_first(psets, pi, kw, level - 1);
    const int warm = prec[pi].p1_status == ST_OPTIMAL ? pi : -1;
    const int o = off[t];
    for (int j = j0 + g; j < n_c; j += CHILD_LANES) {
        const int ch = o + (j - j0);
        int *cs = sets + (long long)ch * kw;
        for (int u = 0; u < kw; ++u) cs[u] = u < level - 1 ? ps[u] : (u == level - 1 ? j : -1);
        par[ch] = pi;
        p1par[ch] = warm;
    }
}

// level 0: the empty set, without a parent
static __global__ void level0_write(int *sets, int kw, int *par, int *p1par) {
    for (int u = threadIdx.x; u < kw; u += blockDim.x) sets[u] = -1;
    if (threadIdx.x == 0) *par = *p1par = -1;
}

// [Q | A^T] of gram_solve from A2 (its stationarity rows, columns x', each
// row restored to the sign of its positive diagonal entry: main.py:108-116
// negates the rows whose right-hand side is negative) and A (n_c x n_x).
static __global__ __launch_bounds__(256) void gram_pack(const double *A2, int M2, int n_c, int n_x, const double *A,
                                                        double *W) {
    const int ld = n_x + n_c, r4 = M2 - n_c - n_x;
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= n_x * ld) return;
    const int i = e / ld, c = e - i * ld;
    double v;
    if (c < n_x) {
        v = A2[(long long)c * M2 + r4 + i];
        if (A2[(long long)i * M2 + r4 + i] < 0.0) v = -v;
    } else {
        v = A[(long long)(c - n_x) * n_x + i];
    }
    W[e] = v;
}

// ---------------------------------------------------------------------
// LICQ screen.  G = A Q^-1 A^T (n_c x n_c) is built once per problem:
// gram_solve turns W = [Q | A^T] (n_x x (n_x + n_c), row-major) into
// [I | Q^-1 A^T] by Gauss-Jordan with diagonal pivots (Q is symmetric
// positive definite), gram_mfma multiplies A by Q^-1 A^T on the FP64
// matrix cores.  licq_screen then factors G_SS (rows of S ascending) per
// candidate.
// ---------------------------------------------------------------------
// The matrix is worked on in LDS when it fits there (in_lds; colq then
// follows it): one workgroup's pivots wait on each access, and global memory
// made them 9 us each at n_x = 60, ncols = 180 (0.55 ms; 0.12 ms in LDS).
template <int NT>
__global__ __launch_bounds__(NT) void gram_solve(double *W, int n_x, int ld, int ncols, double *colq, int in_lds) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    if (!in_lds) {
        for (int i = 0; i < n_x; ++i) pivot_team<NT, double>(W, ld, n_x, ncols, i, i, colq);
        return;
    }
    double *T = reinterpret_cast<double *>(smem);
    for (int e = threadIdx.x; e < n_x * ld; e += NT) T[e] = W[e];
    __syncthreads();
    for (int i = 0; i < n_x; ++i) pivot_team<NT, double>(T, ld, n_x, ncols, i, i, T + n_x * ld);
    for (int e = threadIdx.x; e < n_x * ld; e += NT) W[e] = T[e];
}

// G (n_c x n_c, row-major) = A (n_c x n_x, row-major) x Y (n_x x n_c, rows
// of stride ldy): one wave per 16 x 16 tile of G, v_mfma_f64_16x16x4f64
// over n_x in steps of 4 (operands outside the matrices read as 0).
// Lane l supplies A[i0 + l % 16][k + l / 16] and Y[k + l / 16][j0 + l % 16]
// and receives G[i0 + 4 r + l / 16][j0 + l % 16] in result register r = 0..3
// (the result layout of this instruction, measured on gfx950).
static __global__ __launch_bounds__(64) void gram_mfma(const double *A, const double *Y, int n_c, int n_x, int ldy,
                                                 double *G) {
    typedef double v4d __attribute__((ext_vector_type(4)));
    const int tiles = (n_c + 15) / 16;
    const int ti = blockIdx.x / tiles, tj = blockIdx.x % tiles;
    const int l = threadIdx.x, lr = l % 16, lk = l / 16;
    const int i = ti * 16 + lr, j = tj * 16 + lr;
    v4d acc = {0.0, 0.0, 0.0, 0.0};
    for (int k0 = 0; k0 < n_x; k0 += 4) {
        const int k = k0 + lk;
        const double a = (i < n_c && k < n_x) ? A[(long long)i * n_x + k] : 0.0;
        const double b = (j < n_c && k < n_x) ? Y[(long long)k * ldy + j] : 0.0;
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int gi = ti * 16 + 4 * r + lk, gj = tj * 16 + lr;
        if (gi < n_c && gj < n_c) G[(long long)gi * n_c + gj] = acc[r];
    }
}

// One group of GS lanes per candidate (GS >= level, a power of two <= 64):
// lane r of the group holds row r of the Cholesky factor of G_SS in LDS and
// reads the other rows' column entries by lane exchange.  fail[c] = 1 when a
// pivot d_t <= tol * G_tt (G_tt the original diagonal entry); d_t is the
// squared distance of row t of A (Q^-1 metric) to the span of the rows
// before it, relative to its squared length.
template <int GS>
__global__ __launch_bounds__(64) void licq_screen(const double *G, int n_c, const int *sets, int n, int kw, int level,
                                                   double tol, int *fail) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    constexpr int PER = 64 / GS;
    double *Lrow = reinterpret_cast<double *>(smem) + (long long)threadIdx.x * level;
    const int g = threadIdx.x / GS, r = threadIdx.x % GS;
    const int c = blockIdx.x * PER + g;
    const bool live = c < n;
    const int *S = sets + (long long)(live ? c : 0) * kw;
    const int sr = (live && r < level) ? S[r] : 0;
    for (int q = 0; q < level; ++q) Lrow[q] = (live && r < level) ? G[(long long)sr * n_c + S[q]] : 0.0;
    bool bad = false;
    for (int t = 0; t < level; ++t) {
        const double gtt = __shfl(Lrow[t], t, GS);  // row t's current pivot entry
        const double dtt = G[(long long)(live ? S[t] : 0) * n_c + (live ? S[t] : 0)];
        bad |= !(gtt > tol * dtt);
        const double sq = sqrt(gtt > 0.0 ? gtt : 1.0);
        const double lt = (r > t && r < level) ? Lrow[t] / sq : 0.0;
        if (r > t && r < level) Lrow[t] = lt;
        for (int q = t + 1; q < level; ++q) {
            const double lq = __shfl(lt, q, GS);
            if (r >= q && r < level) Lrow[q] = fma(-lt, lq, Lrow[q]);
        }
    }
    if (live && r == 0) fail[c] = bad ? 1 : 0;
}

// ---------------------------------------------------------------------
// Root: S = {} KKT basis tableau (one workgroup, tableau in global memory)
// ---------------------------------------------------------------------
struct RootArgs {
    DevProb P;
    DevOpts O;
    double *G;        // M2 x (K2+2) scratch (root_w: by columns)
    double *F, *p;    // n_x factor columns of M2, n_x pivots
    int *prow, *pos;  // n_x pivot rows; the position of each row
    int *rowvar;      // M2
    int *slotvar;     // K2
    int *rowof;       // N2
    int *slotof;      // N2
    double *root;     // M2 x (K2+2)
    float *root32;    // the same in FP32, as a stored phase-1 state, or null
    int *root_basis;  // M2
    int *root_nonb;   // K2
    int *root_ok;
};

// The root by columns.  The pivots are known in advance but for the rows of
// the x pivots, so a column can go through all of them by itself, in one
// wave's registers (lane = row), given each pivot's factor column:
//   root_w  the n_c pivots (row of w_j, column w_j): their factor columns are
//           the columns w_j of A2 as they stand, since no other w pivot's row
//           has an entry there (the host has checked that this block of A2 is
//           diagonal with usable entries);
//   root_x  the n_x pivots on the columns x_i alone, one workgroup in LDS:
//           the pivot rows and the factor columns;
//   root_y  those pivots on every column, and the root's layout.
// Every entry goes through pivot_team's operations (a row with a zero factor
// keeps its entry, as there).  root_kernel below, one workgroup pivoting the
// whole matrix in global memory, took 9.0 ms at n=60 m=120 p=12 (326 x 196)
// and remains for a w block that is not diagonal; these three take 0.27 ms.
#define MPQP_ROOT_R 8  // rows per lane: M2 <= 512

// row r of a column held by lane (uniform r)
__device__ __forceinline__ double root_row(const double (&col)[MPQP_ROOT_R], int r) {
    double v = col[0];
#pragma unroll
    for (int s = 1; s < MPQP_ROOT_R; ++s) v = r / MPQP_WAVE == s ? col[s] : v;
    return __shfl(v, r % MPQP_WAVE, MPQP_WAVE);
}

// One pivot (row r, entry p, factor column f) on a column; own: the pivot
// column itself.
__device__ __forceinline__ void root_pivot(double (&col)[MPQP_ROOT_R], int M, int r, double p, const double *f,
                                           bool own) {
    const int lane = threadIdx.x;
    double fr[MPQP_ROOT_R];
#pragma unroll
    for (int s = 0; s < MPQP_ROOT_R; ++s) {
        const int i = lane + MPQP_WAVE * s;
        fr[s] = i < M ? f[i] : 0.0;
    }
    const double prj = (own ? 1.0 : root_row(col, r)) / p;
#pragma unroll
    for (int s = 0; s < MPQP_ROOT_R; ++s) {
        const int i = lane + MPQP_WAVE * s;
        const double t = own ? 0.0 : col[s];
        const double u = prj != 0.0 ? fma(-fr[s], prj, t) : t;
        col[s] = i == r ? prj : u;
    }
}

// entry (r, v) of the optimality LP's first K columns without the S-only
// entries of the w columns, the rhs (v = K) and the perturbation (K + 1)
__device__ __forceinline__ double root_entry(const DevProb &P, double step, int r, int v) {
    if (v == P.K2) return P.xb2[r];
    if (v > P.K2) return (double)(r + 1) * step;
    const int w = v - P.n_x - P.n_t;
    if (w >= 0 && w < P.n_c && r >= P.M2 - P.n_c - P.n_x && r < P.M2 - P.n_c) return 0.0;
    return P.A2[(long long)v * P.M2 + r];
}

static __global__ __launch_bounds__(64) void root_w(RootArgs a) {
    const DevProb &P = a.P;
    const int M = P.M2, v = blockIdx.x, lane = threadIdx.x;
    const int w0 = P.n_x + P.n_t;
    double col[MPQP_ROOT_R];
#pragma unroll
    for (int s = 0; s < MPQP_ROOT_R; ++s) {
        const int i = lane + MPQP_WAVE * s;
        col[s] = i < M ? root_entry(P, a.O.perturb_step, i, v) : 0.0;
    }
    // rows of w_j: no w pivot but its own changes them.  The factors of the
    // next pivot are read while this one is applied.
    auto factors = [&](double (&f)[MPQP_ROOT_R], int j) {
#pragma unroll
        for (int s = 0; s < MPQP_ROOT_R; ++s) {
            const int i = lane + MPQP_WAVE * s;
            f[s] = root_entry(P, 0.0, i < M ? i : 0, w0 + j);
        }
    };
    double fn[MPQP_ROOT_R];
    factors(fn, 0);
    for (int j = 0; j < P.n_c; ++j) {
        const int r = M - P.n_c + j;
        const bool own = v == w0 + j;
        double fr[MPQP_ROOT_R];
#pragma unroll
        for (int s = 0; s < MPQP_ROOT_R; ++s) fr[s] = fn[s];
        factors(fn, j + 1 < P.n_c ? j + 1 : j);
        const double t = root_row(col, r);
        if (!own && t == 0.0) continue;
        const double prj = (own ? 1.0 : t) / root_row(fr, r);
#pragma unroll
        for (int s = 0; s < MPQP_ROOT_R; ++s) {
            const int i = lane + MPQP_WAVE * s;
            col[s] = i == r ? prj : fma(-fr[s], prj, own ? 0.0 : col[s]);
        }
    }
#pragma unroll
    for (int s = 0; s < MPQP_ROOT_R; ++s) {
        const int i = lane + MPQP_WAVE * s;
        if (i < M) a.G[(long long)v * M + i] = col[s];
    }
}

// a.F: the factor columns (n_x x M); a.p: the pivots; a.prow: their rows;
// a.pos: the position of each row.  LDS: the x columns fit there.
template <int NT, bool LDS>
__global__ __launch_bounds__(NT) void root_x(RootArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    __shared__ int sh_r;
    __shared__ double sh_pr[512];  // the divided pivot row: n_x <= 512
    __shared__ int sh_row[512];    // the pivot rows
    const DevProb &P = a.P;
    const int M = P.M2, n_x = P.n_x, n_c = P.n_c, n_t = P.n_t, r4 = M - n_c - n_x;
    const int tid = threadIdx.x, lane = tid % MPQP_WAVE, wave = tid / MPQP_WAVE;
    double *X;  // column i at X + i * M
    if constexpr (LDS) X = reinterpret_cast<double *>(smem);
    else X = a.G;
    if constexpr (LDS)
        for (int e = tid; e < n_x * M; e += NT) X[e] = a.G[e];
    for (int r = tid; r < M; r += NT) a.pos[r] = r >= M - n_c ? n_x + (r - (M - n_c)) : (r < r4 ? n_x + n_c + r : -1);
    unsigned used = 0u;  // wave 0: bit s of a lane: row r4 + lane + 64 s is taken
    __syncthreads();
    int ok = 1;
    for (int i = 0; i < n_x; ++i) {
        double *Xi = X + (long long)i * M;
        if (wave == 0) {
            // largest |entry| of the free rows, the lowest on ties
            double v = 0.0;
            int key = -1, aux = 0;
            for (int t = lane, s = 0; t < n_x; t += MPQP_WAVE, ++s) {
                const double av = fabs(Xi[r4 + t]);
                if (!((used >> s) & 1u) && av == av && (key < 0 || -av < v)) {
                    v = -av;
                    key = t;
                }
            }
            lex_min(v, key, aux);
            if (key >= 0 && key % MPQP_WAVE == lane) used |= 1u << (key / MPQP_WAVE);
            if (lane == 0) sh_r = key >= 0 && -v > a.O.licq_tol ? r4 + key : -1;
        }
        __syncthreads();
        const int r = sh_r;
        if (r < 0) {
            ok = 0;
            break;
        }
        const double p = Xi[r];
        if (tid == 0) sh_row[i] = r;
        for (int c = i + 1 + tid; c < n_x; c += NT) sh_pr[c] = X[(long long)c * M + r] / p;
        __syncthreads();
        for (int c = i + 1 + wave; c < n_x; c += NT / MPQP_WAVE) {
            double *Xc = X + (long long)c * M;
            const double prj = sh_pr[c];
            double t[MPQP_ROOT_R], f[MPQP_ROOT_R];
#pragma unroll
            for (int s = 0; s < MPQP_ROOT_R; ++s) {
                const int k = lane + MPQP_WAVE * s;
                t[s] = Xc[k < M ? k : 0];
                f[s] = Xi[k < M ? k : 0];
            }
#pragma unroll
            for (int s = 0; s < MPQP_ROOT_R; ++s) {
                const int k = lane + MPQP_WAVE * s;
                if (k < M) Xc[k] = k == r ? prj : (prj != 0.0 ? fma(-f[s], prj, t[s]) : t[s]);
            }
        }
        __syncthreads();
    }
    // column i is left as it was at its pivot: the factors (written once,
    // since a barrier in the loop would wait for stores to global memory)
    __syncthreads();
    for (int e = tid; ok && e < n_x * M; e += NT) a.F[e] = X[e];
    for (int i = tid; ok && i < n_x; i += NT) {
        const int r = sh_row[i];
        a.p[i] = X[(long long)i * M + r];
        a.prow[i] = r;
        a.pos[r] = i;
    }
    // basis and nonbasic: fixed but for the order of the e_r of the x rows
    const int N2 = P.N2, K = P.K2;
    for (int t = tid; t < M; t += NT)
        a.root_basis[t] = t < n_x ? t : (t < n_x + n_c ? n_x + n_t + (t - n_x) : N2 - M + (t - n_x - n_c));
    for (int t = tid; t < K; t += NT)
        a.root_nonb[t] = t < n_t ? n_x + t : (t < n_t + 2 ? n_x + n_t + n_c + (t - n_t) : N2 - M + r4 + (t - n_t - 2));
    if (a.root32) {
        int *db = reinterpret_cast<int *>(a.root32 + (long long)opt_tw<float>(M, K));
        __syncthreads();
        for (int t = tid; t < M; t += NT) db[t] = a.root_basis[t];
        for (int t = tid; t < K; t += NT) db[M + t] = a.root_nonb[t];
    }
    if (tid == 0) *a.root_ok = ok;
}

static __global__ __launch_bounds__(64) void root_y(RootArgs a) {
    if (!*a.root_ok) return;
    const DevProb &P = a.P;
    const int M = P.M2, K = P.K2, n_x = P.n_x, n_t = P.n_t, n_c = P.n_c, r4 = M - n_c - n_x;
    const int v = blockIdx.x, lane = threadIdx.x;
    double col[MPQP_ROOT_R];
#pragma unroll
    for (int s = 0; s < MPQP_ROOT_R; ++s) {
        const int i = lane + MPQP_WAVE * s;
        col[s] = i < M && v >= n_x ? a.G[(long long)v * M + i] : 0.0;
    }
    // a column x_v begins with its own pivot
    for (int i = v < n_x ? v : 0; i < n_x; ++i)
        root_pivot(col, M, a.prow[i], a.p[i], a.F + (long long)i * M, i == v);
    // its slot: theta', eps, u, then the e of the x rows and of the w rows
    const int w0 = n_x + n_t;
    const int kk = v < n_x ? n_t + 2 + a.prow[v] - r4
                           : (v < w0 ? v - n_x : (v < w0 + n_c ? n_t + 2 + n_x + (v - w0) : (v < K ? n_t + (v - w0 - n_c) : v)));
#pragma unroll
    for (int s = 0; s < MPQP_ROOT_R; ++s) {
        const int i = lane + MPQP_WAVE * s;
        if (i < M) {
            a.root[(long long)a.pos[i] * (K + 2) + kk] = col[s];
            if (a.root32) a.root32[(long long)a.pos[i] * opt_ld<float>(K) + kk] = (float)col[s];
        }
    }
}

template <int NT>
__global__ __launch_bounds__(NT) void root_kernel(RootArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    __shared__ int sh_r, sh_ok;
    const DevProb &P = a.P;
    const int M = P.M2, K = P.K2, N2 = P.N2, ld = K + 2;
    const int n_x = P.n_x, n_t = P.n_t, n_c = P.n_c;
    const int tid = threadIdx.x;
    double *colq = reinterpret_cast<double *>(smem);
    double *G = a.G;
    const int r4 = M - n_c - n_x;
    for (int e = tid; e < M * ld; e += NT) {
        const int r = e / ld, kk = e - r * ld;
        double v;
        if (kk < K) {
            const bool is_w = kk >= n_x + n_t && kk < n_x + n_t + n_c;
            v = P.A2[(long long)kk * M + r];
            if (is_w && r >= r4 && r < M - n_c) v = 0.0;
        } else if (kk == K) {
            v = P.xb2[r];
        } else {
            v = (double)(r + 1) * a.O.perturb_step;
        }
        G[e] = v;
    }
    for (int r = tid; r < M; r += NT) a.rowvar[r] = N2 - M + r;
    for (int kk = tid; kk < K; kk += NT) a.slotvar[kk] = kk;
    if (tid == 0) sh_ok = 1;
    __syncthreads();
    for (int j = 0; j < n_c; ++j) {
        const int r = M - n_c + j, q = n_x + n_t + j;
        if (!(fabs(G[r * ld + q]) > a.O.licq_tol)) {
            if (tid == 0) sh_ok = 0;
            break;
        }
        pivot_team<NT, double>(G, ld, M, K + 2, r, q, colq);
        if (tid == 0) {
            const int t = a.rowvar[r];
            a.rowvar[r] = a.slotvar[q];
            a.slotvar[q] = t;
        }
        __syncthreads();
    }
    __syncthreads();
    int *used = reinterpret_cast<int *>(colq + M + 1);
    for (int r = tid; r < M; r += NT) used[r] = 0;
    __syncthreads();
    for (int i = 0; i < n_x && sh_ok; ++i) {
        if (tid == 0) {
            int r = -1;
            double best = -1.0;
            for (int rr = r4; rr < r4 + n_x; ++rr) {
                if (used[rr]) continue;
                const double av = fabs(G[rr * ld + i]);
                if (av > best) { best = av; r = rr; }
            }
            if (r < 0 || !(best > a.O.licq_tol)) sh_ok = 0;
            sh_r = r;
        }
        __syncthreads();
        if (!sh_ok) break;
        const int r = sh_r;
        pivot_team<NT, double>(G, ld, M, K + 2, r, i, colq);
        if (tid == 0) {
            used[r] = 1;
            const int t = a.rowvar[r];
            a.rowvar[r] = a.slotvar[i];
            a.slotvar[i] = t;
        }
        __syncthreads();
    }
    __syncthreads();
    if (tid == 0) {
        int ok = sh_ok;
        for (int v = 0; v < N2; ++v) a.rowof[v] = a.slotof[v] = -1;
        for (int r = 0; r < M; ++r) a.rowof[a.rowvar[r]] = r;
        for (int kk = 0; kk < K; ++kk) a.slotof[a.slotvar[kk]] = kk;
        int p = 0;
        for (int i = 0; i < n_x; ++i) a.root_basis[p++] = i;
        for (int j = 0; j < n_c; ++j) a.root_basis[p++] = n_x + n_t + j;
        for (int t = 0; t < M - P.n_eqs; ++t) a.root_basis[p++] = N2 - M + t;
        int k2 = 0;
        for (int v = 0; v < N2; ++v)
            if (a.rowof[v] < 0) {
                if (k2 < K) a.root_nonb[k2] = v;
                ++k2;
            }
        if (p != M || k2 != K) ok = 0;
        for (int pp = 0; pp < M && ok; ++pp)
            if (a.rowof[a.root_basis[pp]] < 0) ok = 0;
        for (int kk = 0; kk < K && ok; ++kk)
            if (a.slotof[a.root_nonb[kk]] < 0) ok = 0;
        sh_ok = ok;
    }
    __syncthreads();
    if (sh_ok) {
        for (int e = tid; e < M * ld; e += NT) {
            const int pp = e / ld, kk = e - pp * ld;
            const int src = a.rowof[a.root_basis[pp]];
            const int sc = kk < K ? a.slotof[a.root_nonb[kk]] : kk;
            const double v = G[src * ld + sc];
            a.root[e] = v;
            if (a.root32) a.root32[pp * opt_ld<float>(K) + kk] = (float)v;
        }
        if (a.root32) {
            int *db = reinterpret_cast<int *>(a.root32 + (long long)opt_tw<float>(M, K));
            for (int i = tid; i < M; i += NT) db[i] = a.root_basis[i];
            for (int kk = tid; kk < K; kk += NT) db[M + kk] = a.root_nonb[kk];
        }
    }
    if (tid == 0) *a.root_ok = sh_ok;
}
