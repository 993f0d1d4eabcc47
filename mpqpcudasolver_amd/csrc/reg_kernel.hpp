// reg_kernel.hpp — the optimality LP with its tableau in registers: FP32
// (mixed precision) pivoted by the matrix cores, FP64 by the vector unit.
//
// FP32.  One LP per workgroup of NW waves.  Wave w holds the rows w * RW ..
// w * RW + RW - 1 of the condensed tableau, lane l of slot s the column
// l + 64 s (CS slots): a block of four rows of a slot is the accumulator of
// v_mfma_f32_4x4x1_16b_f32 with its A operand broadcast from one block (16
// blocks of 4 x 4, K = 1: result register i of lane l is row i, column l).  A
// pivot is then one such instruction per block and slot,
//   T[4b + i][l] = fma(-f[4b + i], pr[l], T[4b + i][l]),
// A = the wave's factors by lane (lane 4b + i = row 4b + i), B = the divided
// pivot row by lane.  This instruction rounds as fmaf does, denormals and
// cancellations included (compared bit for bit on 4 M random operands), so
// the entries go through the operations of opt_kernel.hpp in the same order;
// a column whose pivot-row entry is zero changes at most in the sign of a
// zero.  The tableau needs no LDS and no global memory while it is pivoted,
// and 256 FMA a clock and CU instead of the vector unit's 64.
//
// The right-hand side and the perturbation column are held by row (lane i =
// row i of the wave), with copies in LDS; the cost row is held by every
// wave.  Each wave knows its smallest basic value after a pivot, so the
// leaving row costs one exchange of NW values; the wave that holds it runs
// the ratio test on its registers and publishes the divided row in LDS.
//
// FP64.  The same layout with a register pair per entry; of a wave's rows the
// last LW may lie in its part of LDS, lane = column as well (336 x 196 doubles
// are 512 KB: all of a CU's registers, or 3/4 of them and 132 KB of LDS).
// The matrix unit has no FP64 form with a broadcast operand and no higher FP64
// rate, so a pivot takes column q out of the pivot lane into scalar registers
// (two lane reads a row) and is one v_fma_f64 per row and slot.
//
// What bounds both: with the tableau out of LDS and of global memory, the
// chain of a pivot - leaving row, entering column, division, factors - at two
// waves per SIMD, about 9,000 cycles in FP64 and 10,000 in FP32 at
// n=60 m=120 p=12.  The LDS and split kernels (opt_kernel.hpp) spend the same
// chain and a pass over the tableau: n=60 m=120 p=12 |S|<=3 mixed 822 -> 571 ms
// with the FP32 tableau and -> 486 ms with the re-solves' FP64 too; FP64
// |S|<=2 at that size 57 -> 24.5 ms of kernel time, n=30 m=62 p=8 |S|<=3 18.4
// -> 7.8 ms, n=6 m=28 p=4 |S|<=6 6.4 -> 2.9 ms.  An FP64 update takes 2,800
// cycles at 171 x 102 and 5,500 at 325 x 194, where the vector unit's issue
// bounds it (two waves per SIMD, four cycles an instruction).
#pragma once
#include <type_traits>
#include <utility>

typedef float v4f __attribute__((ext_vector_type(4)));

// f(integral_constant<i>) for every i in [0, N): the tableau's registers are
// named by constants from the start (an array that a loop indexes is placed
// in memory before the loop is unrolled, and stays there)
template <typename F, int... I>
__device__ __forceinline__ void reg_for_seq(F &f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void reg_for(F &&f) {
    reg_for_seq(f, std::make_integer_sequence<int, N>{});
}
#define MPQP_INL __attribute__((always_inline))

// f(integral_constant<i>) for the (wave-uniform) i in [LO, HI) by scalar
// branches.  The empty asm (its operand differs from branch to branch) keeps
// the branches' last accesses from being merged into one with a variable
// index, which would place the tableau in memory.
template <int LO, int HI, typename F>
__device__ __forceinline__ void reg_pick(int i, F &&f) {
    if constexpr (HI - LO == 1) {
        f(std::integral_constant<int, LO>{});
        asm volatile("" ::"n"(LO));
    } else {
        constexpr int MID = (LO + HI) / 2;
        if (i < MID) reg_pick<LO, MID>(i, f);
        else reg_pick<MID, HI>(i, f);
    }
}

// x (uniform) as a value that the compiler knows nothing about: the one test
// of a loop's end is not split up into exits of its own
__device__ __forceinline__ int opaque(int x) {
    x = rfl(x);
    asm volatile("" : "+s"(x));
    return x;
}

// lane l's value (uniform)
__device__ __forceinline__ float lane_get(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ double lane_get(double v, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}
// v with lane l's value replaced by the uniform x (the compiler has no
// builtin of the instruction's name: its intrinsic, by name)
extern "C" __device__ __attribute__((const)) int mpqp_writelane(int x, int l, int v) __asm("llvm.amdgcn.writelane.i32");
__device__ __forceinline__ double lane_set(double v, int l, double x) {
    return __hiloint2double(mpqp_writelane(__double2hiint(x), l, __double2hiint(v)),
                            mpqp_writelane(__double2loint(x), l, __double2loint(v)));
}

// Minimum over the wave of values that are not NaN, known to every lane:
// v_min with DPP row shifts, then the row broadcasts of lanes 15 and 31, into
// lane 63 (six dependent instructions; lane shifts with compare and select
// took four times as long).
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_get(float old, float v) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(v), CTRL, ROWS, 0xf, false));
}
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_get(double old, double v) {
    return __hiloint2double(
        __builtin_amdgcn_update_dpp(__double2hiint(old), __double2hiint(v), CTRL, ROWS, 0xf, false),
        __builtin_amdgcn_update_dpp(__double2loint(old), __double2loint(v), CTRL, ROWS, 0xf, false));
}
__device__ __forceinline__ float min_r(float a, float b) { return fminf(a, b); }
__device__ __forceinline__ float max_r(float a, float b) { return fmaxf(a, b); }
__device__ __forceinline__ double min_r(double a, double b) { return fmin(a, b); }
__device__ __forceinline__ double max_r(double a, double b) { return fmax(a, b); }
__device__ __forceinline__ unsigned min_r(unsigned a, unsigned b) { return a < b ? a : b; }
template <int CTRL, int ROWS>
__device__ __forceinline__ unsigned dpp_get(unsigned old, unsigned v) {
    return (unsigned)__builtin_amdgcn_update_dpp((int)old, (int)v, CTRL, ROWS, 0xf, false);
}
__device__ __forceinline__ unsigned lane_get(unsigned v, int l) { return (unsigned)__builtin_amdgcn_readlane((int)v, l); }
template <int CTRL, int ROWS, typename Re>
__device__ __forceinline__ Re dpp_min(Re v) {
    return min_r(v, dpp_get<CTRL, ROWS>(v, v));
}
template <typename Re>
__device__ __forceinline__ Re row8_min(Re v) {  // into lane 7, of lanes 0 .. 7
    v = dpp_min<0x111, 0xf>(v);
    v = dpp_min<0x112, 0xf>(v);
    return dpp_min<0x114, 0xf>(v);
}
template <typename Re>
__device__ __forceinline__ Re wave_min(Re v) {
    v = row8_min(v);
    v = dpp_min<0x118, 0xf>(v);
    v = dpp_min<0x142, 0xa>(v);
    v = dpp_min<0x143, 0xc>(v);
    return lane_get(v, 63);
}

// The reference tree (tree_argmin_s) over float values with an id below 1024
// and a count packed into one word (count << 10 | id; negative: no element):
// two lane shifts a step instead of four.
template <int I, typename Pred>
__device__ __forceinline__ void tree32_step(float &v, int &pk, int n, int lane, Pred pred) {
    const float ov = lane_down_f<I>(v);
    const int op = lane_down_i<I>(pk);
    const bool take = (lane < I) & (lane + I < n) & pred(v, pk, ov, op);
    v = take ? ov : v;
    pk = take ? op : pk;
}
template <int S, typename Pred>
__device__ __forceinline__ int tree32(float (&v)[S], int (&pk)[S], int n, int lane, Pred pred) {
    const int half = half_pow2(n);
#pragma unroll
    for (int lvl = 2; lvl >= 0; --lvl) {
        const int i = 64 << lvl, ds = 1 << lvl;
        if (i <= half) {
#pragma unroll
            for (int s = 0; s < ds; ++s)
                if (s + ds < S) {
                    const bool take = (lane + 64 * (s + ds) < n) & pred(v[s], pk[s], v[s + ds], pk[s + ds]);
                    v[s] = take ? v[s + ds] : v[s];
                    pk[s] = take ? pk[s + ds] : pk[s];
                }
        }
    }
    if (half >= 32) tree32_step<32>(v[0], pk[0], n, lane, pred);
    if (half >= 16) tree32_step<16>(v[0], pk[0], n, lane, pred);
    if (half >= 8) tree32_step<8>(v[0], pk[0], n, lane, pred);
    if (half >= 4) tree32_step<4>(v[0], pk[0], n, lane, pred);
    if (half >= 2) tree32_step<2>(v[0], pk[0], n, lane, pred);
    if (half >= 1) tree32_step<1>(v[0], pk[0], n, lane, pred);
    return rfl(pk[0]);
}

// The reference tree over values of either type: id of the element it keeps
// (ids below 1024, negative: no element), its value in v[0] of lane 0.
template <int S, typename Pred>
__device__ __forceinline__ int reg_tree(float (&v)[S], int (&id)[S], int (&cn)[S], int n, int lane, Pred pred) {
    int pk[S];
    reg_for<S>([&](auto s) MPQP_INL { pk[s] = id[s] < 0 ? -1 : cn[s] << 10 | id[s]; });
    const int w = tree32<S>(v, pk, n, lane, [&](float vt, int pt, float vu, int pu) {
        return pred((double)vt, pt, pt >> 10, (double)vu, pu, pu >> 10);
    });
    return w < 0 ? -1 : w & 1023;
}
template <int S, typename Pred>
__device__ __forceinline__ int reg_tree(double (&v)[S], int (&id)[S], int (&cn)[S], int n, int lane, Pred pred) {
    tree_argmin_s<S>(v, id, cn, n, lane, pred);
    return rfl(id[0]);
}

// Of the elements (lane + 64 s, s < S) whose lanes are set in hit[s], the one
// that a reference tree keeps when it replaces an element only by a strictly
// smaller one and these are the minima: the combines run from the largest
// stride to 1, and each keeps its lower half, so the last one decides first:
// lowest bit 0 of the index clear, then bit 1, ... (-1: none).
template <int S>
__device__ __forceinline__ int tree_first(const unsigned long long (&hit)[S]) {
    unsigned long long m = 0ull;
#pragma unroll
    for (int s = 0; s < S; ++s) m |= hit[s];
    if (m == 0ull) return -1;
    constexpr unsigned long long half[6] = {0x5555555555555555ull, 0x3333333333333333ull, 0x0f0f0f0f0f0f0f0full,
                                            0x00ff00ff00ff00ffull, 0x0000ffff0000ffffull, 0x00000000ffffffffull};
#pragma unroll
    for (int b = 0; b < 6; ++b) m = (m & half[b]) ? m & half[b] : m;
    const int lane = __ffsll((long long)m) - 1;
    unsigned sl = 0u;
#pragma unroll
    for (int s = 0; s < S; ++s) sl |= (unsigned)((hit[s] >> lane) & 1ull) << s;
    sl = (sl & 0x55u) ? sl & 0x55u : sl;
    sl = (sl & 0x33u) ? sl & 0x33u : sl;
    sl = (sl & 0x0fu) ? sl & 0x0fu : sl;
    return lane + 64 * (__ffs((int)sl) - 1);
}

// The columns past 64 CS, if no more than EX, are held by row like the rhs
// (a whole slot for two columns would cost a quarter of the registers and of
// the matrix instructions at n=60 m=120 p=12, whose 194 columns are three
// slots and two); in a decision they are lanes 0 .. EX - 1 of one more slot.
// Rows past M repeat row M - 1, and the columns of a slot past K repeat
// column 0: nothing reads them, and no entry depends on another row or column
// than its own.
//
// FP64: the same, with the vector unit (T = fma(-f, pr, T) with the row's
// factor in scalar registers) and, of a wave's RW rows, the last LW in its
// part of LDS, lane = column as well.
template <typename Re, int NW, int RW, int CS, int EX, int LW>
struct RegTab {
    static_assert(RW <= MPQP_WAVE, "one lane per row");
    static_assert(sizeof(Re) == 8 || (RW % 4 == 0 && LW == 0), "FP32: blocks of four rows");
    static constexpr int RR = RW - LW;
    static constexpr int NS = CS + (EX > 0 ? 1 : 0);  // slots of a decision
    typedef std::conditional_t<sizeof(Re) == 4, v4f, Re> cell;
    cell t[sizeof(Re) == 4 ? RW / 4 : RR][CS];
    int cb;         // by row: use count of the basic variable (phase 1)
    Re d[NS];       // cost row (the same in every wave)
    Re xs[EX + 2];  // by row (lanes < RW): the extra columns, the rhs, the perturbation
    Re *lt;         // this lane's column of the wave's LDS rows
    __device__ __forceinline__ Re x() const { return xs[EX]; }
    __device__ __forceinline__ Re xp() const { return xs[EX + 1]; }
    template <int I, int S>
    __device__ __forceinline__ Re get() const {
        if constexpr (sizeof(Re) == 4) return t[I / 4][S][I % 4];
        else if constexpr (I < RR) return t[I][S];
        else return lt[((I - RR) * CS + S) * MPQP_WAVE];
    }
    template <int I, int S>
    __device__ __forceinline__ void set(Re v) {
        if constexpr (sizeof(Re) == 4) t[I / 4][S][I % 4] = v;
        else if constexpr (I < RR) t[I][S] = v;
        else lt[((I - RR) * CS + S) * MPQP_WAVE] = v;
    }
};

// Per-wave results of the distributed decisions.
template <typename Re>
struct RegMin {
    Re m1;     // smallest x_B of the wave
    int at;    // its row: of several, the one that the reference tree keeps
    int cnt;   // use count of the values within the tree's band of m1, if
    int flag;  // it is the same; 1: it is not, 2: a NaN among the values,
               // 4: no row
};
template <typename Re, int NW>
struct RegShared {
    __attribute__((aligned(16))) RegMin<Re> min[NW];
    Re cmax[NW], rv[NW];
    int rk[NW];
};

// LDS of one workgroup: the divided pivot row (with its rhs and perturbation
// entries), copies of the rhs, perturbation and one column by row, the cost
// row by column; the bookkeeping of OptLds; for certification x, r and the
// nonbasic e-list; a stage of `rp` rows for the steps that read the tableau
// against its layout (lambda swap, certification): np passes of NW / np
// waves' rows each.
__host__ __device__ inline long long reg_lds_bytes(int nw, int rw, int cs, int M, int K, int N2, int np) {
    const long long mr = (long long)nw * rw, kc = 64LL * (cs + 1);
    long long b = (2 * kc + 3 * mr) * (long long)sizeof(float);
    b = (b + 15) & ~15LL;
    b += (3LL * N2 + 2 * M + K) * 4;
    b = ((b + 7) & ~7LL) + 2LL * M * 8 + 2LL * (M + 1) * 4;
    b = (b + 15) & ~15LL;
    b += mr / np * (K | 1) * (long long)sizeof(float);
    return (b + 15) & ~15LL;
}
// FP64: no certification and no stage; the LDS rows
__host__ __device__ inline long long reg64_lds_bytes(int nw, int rw, int cs, int lw, int M, int K, int N2) {
    const long long mr = (long long)nw * rw, kc = 64LL * (cs + 1);
    long long b = ((long long)nw * lw * cs * 64 + 2 * kc + 3 * mr) * (long long)sizeof(double);
    b += (3LL * N2 + 2 * M + K) * 4;
    return (b + 15) & ~15LL;
}

template <typename Re, int NW, int RW, int CS, int EX, int LW>
struct RegLds {
    static constexpr int MR = NW * RW, KC = MPQP_WAVE * (CS + 1);
    Re *ep, *gx, *gp, *colx, *dl, *rows_lds;
    float *stage;
    int *basis, *nonb, *where, *bcnt, *nbcnt, *rows;
    double *cx, *cr, *xv;
    int *elr, *els;
    int sld, np, rp;
    __device__ void carve(unsigned char *smem, int M, int K, int N2, int np_) {
        constexpr size_t LT = (size_t)NW * LW * CS * MPQP_WAVE;
        np = np_;
        rp = sizeof(Re) == 4 ? MR / np : 0;
        sld = K | 1;
        rows_lds = reinterpret_cast<Re *>(smem);
        ep = rows_lds + LT;
        gx = ep + KC;
        gp = gx + MR;
        colx = gp + MR;
        dl = colx + MR;
        size_t b = (LT + 2 * KC + 3 * MR) * sizeof(Re);
        b = (b + 15) & ~(size_t)15;
        bcnt = reinterpret_cast<int *>(smem + b);
        nbcnt = bcnt + N2;
        where = nbcnt + N2;
        basis = where + N2;
        rows = basis + M;
        nonb = rows + M;
        b += (size_t)(3 * N2 + 2 * M + K) * 4;
        cx = cr = nullptr;
        elr = els = nullptr;
        xv = reinterpret_cast<double *>(bcnt);
        stage = nullptr;
        if constexpr (sizeof(Re) == 4) {
            b = (b + 7) & ~(size_t)7;
            cx = reinterpret_cast<double *>(smem + b);
            cr = cx + M;
            elr = reinterpret_cast<int *>(cr + M);
            els = elr + M + 1;
            b += (size_t)2 * M * 8 + (size_t)2 * (M + 1) * 4;
            b = (b + 15) & ~(size_t)15;
            stage = reinterpret_cast<float *>(smem + b);
        }
    }
    __device__ __forceinline__ Re rhs_of(int i) const { return gx[i]; }
    __device__ __forceinline__ unsigned col(const DevProb &P, int v) const { return P.csc_col[v]; }
    __device__ __forceinline__ Re cost_of(int k) const { return dl[k]; }
};

__device__ __forceinline__ int wave_id() { return rfl((int)(threadIdx.x / MPQP_WAVE)); }

// The wave's rows into the stage, pass h (waves [h, h + 1) * NW / np); the
// caller's barriers surround it.
template <typename Re, int NW, int RW, int CS, int EX, int LW>
__device__ __forceinline__ void reg_dump(const RegTab<Re, NW, RW, CS, EX, LW> &R, const RegLds<Re, NW, RW, CS, EX, LW> &L, int K, int h) {
    const int wave = wave_id(), lane = fresh_lane();
    const int w0 = h * (NW / L.np);
    if (wave >= w0 && wave < w0 + NW / L.np) {
        float *dst = L.stage + (wave - w0) * RW * L.sld;
        reg_for<CS>([&](auto s) MPQP_INL {
            const int c = lane + MPQP_WAVE * s;
            if (c < K) {
                float *dc = dst + c;
                reg_for<RW>([&](auto i) MPQP_INL {
                    *dc = R.template get<decltype(i)::value, decltype(s)::value>();
                    dc += L.sld;
                });
            }
        });
        if (lane < RW)
            reg_for<EX>([&](auto e) MPQP_INL {
                if (MPQP_WAVE * CS + e < K) dst[lane * L.sld + MPQP_WAVE * CS + e] = R.xs[e];
            });
    }
}

// T -= f (by row) x v (by column) in slot s, every block of rows
template <int S, int NW, int RW, int CS, int EX>
__device__ __forceinline__ void reg_rank1(RegTab<float, NW, RW, CS, EX, 0> &R, float nf, float v) {
    reg_for<RW / 4>([&](auto b) MPQP_INL {
        R.t[b][S] = __builtin_amdgcn_mfma_f32_4x4x1f32(nf, v, R.t[b][S], 4, decltype(b)::value, 0);
    });
}

// The LDS rows' entries of column q < 64 CS by lane (lane = row; 0 elsewhere)
template <int NW, int RW, int CS, int EX, int LW>
__device__ __forceinline__ double reg_lds_col(const RegTab<double, NW, RW, CS, EX, LW> &R, int q) {
    const int lane = fresh_lane(), g = lane - (RW - LW);
    const bool in = (unsigned)g < (unsigned)LW && q < MPQP_WAVE * CS;
    const double v = R.lt[(in ? (g * CS + q / MPQP_WAVE) * MPQP_WAVE + q % MPQP_WAVE : 0) - lane];
    return in ? v : 0.0;
}

// Column q of the wave's rows by lane, through the wave's part of L.colx (a
// wave's LDS operations stay in order).  CLEAR: the column is left zero
// (T - f * 1 in its lane), if `on`.
// FP64: lane by lane through scalar registers (CLEAR is left to reg_apply).
template <bool CLEAR, typename Re, int NW, int RW, int CS, int EX, int LW, typename RT>
__device__ __forceinline__ Re reg_col_op(RT &R, const RegLds<Re, NW, RW, CS, EX, LW> &L, int q, bool on) {
    const int lane = fresh_lane(), lq = q % MPQP_WAVE;
    Re v = 0;
    if constexpr (sizeof(Re) == 8) {
        if constexpr (LW > 0) v = reg_lds_col(R, q);
        reg_for<CS>([&](auto s) MPQP_INL {
            if (q / MPQP_WAVE == s)
                reg_for<RW - LW>([&](auto i) MPQP_INL { v = lane_set(v, i, lane_get(R.t[i][s], lq)); });
        });
        reg_for<EX>([&](auto e) MPQP_INL { v = q == MPQP_WAVE * CS + e ? R.xs[e] : v; });
        return v;
    } else {
        float *cx = L.colx + wave_id() * RW;
        reg_for<CS>([&](auto s) MPQP_INL {
            if (q / MPQP_WAVE == s) {
                if (lane == lq)
                    reg_for<RW / 4>([&](auto b) MPQP_INL { *reinterpret_cast<v4f *>(cx + 4 * b) = R.t[b][s]; });
                __builtin_amdgcn_wave_barrier();
                v = cx[lane < RW ? lane : 0];
                if constexpr (CLEAR) reg_rank1<decltype(s)::value>(R, on ? -v : 0.f, lane == lq ? 1.f : 0.f);
            }
        });
        reg_for<EX>([&](auto e) MPQP_INL {
            const bool at = q == MPQP_WAVE * CS + e;
            v = at ? R.xs[e] : v;
            if constexpr (CLEAR) R.xs[e] = at && on ? 0.f : R.xs[e];
        });
        __builtin_amdgcn_wave_barrier();
        return v;
    }
}
template <typename Re, int NW, int RW, int CS, int EX, int LW>
__device__ __forceinline__ Re reg_col(const RegTab<Re, NW, RW, CS, EX, LW> &R, const RegLds<Re, NW, RW, CS, EX, LW> &L, int q) {
    return reg_col_op<false>(R, L, q, false);
}

// Row `lr` of the wave; al[CS]: its extra columns, rhs and perturbation entry
// in the first lanes.
template <typename Re, int NW, int RW, int CS, int EX, int LW>
__device__ __forceinline__ void reg_row(const RegTab<Re, NW, RW, CS, EX, LW> &R, int lr, Re (&al)[CS + 1]) {
    if constexpr (sizeof(Re) == 8) {
        constexpr int RR = RW - LW;
        if (LW > 0 && lr >= RR)
            reg_for<CS>([&](auto s) MPQP_INL { al[s] = R.lt[((lr - RR) * CS + s) * MPQP_WAVE]; });
        else
            reg_pick<0, RR>(lr, [&](auto i) MPQP_INL {
                reg_for<CS>([&](auto s) MPQP_INL { al[s] = R.t[i][s]; });
            });
    } else {
        const int u = lr % 4;
        reg_pick<0, RW / 4>(lr / 4, [&](auto b) MPQP_INL {
            reg_for<CS>([&](auto s) MPQP_INL {
                const v4f v = R.t[b][s];
                al[s] = u < 2 ? (u == 0 ? v[0] : v[1]) : (u == 2 ? v[2] : v[3]);
            });
        });
    }
    const int lane = fresh_lane();
    al[CS] = 0;
    reg_for<EX + 2>([&](auto e) MPQP_INL { al[CS] = lane == e ? lane_get(R.xs[e], lr) : al[CS]; });
}

// Row `lr` of the wave (its entries al) made zero: T - 1 * al.
template <int NW, int RW, int CS, int EX>
__device__ __forceinline__ void reg_clear_row(RegTab<float, NW, RW, CS, EX, 0> &R, int lr, const float (&al)[CS + 1]) {
    const float a = fresh_lane() == lr ? -1.f : 0.f;
    // (one test after the other: the branches of a tree would meet with a
    // tableau changed in different places)
    reg_for<RW / 4>([&](auto b) MPQP_INL {
        if (lr / 4 == b)
            reg_for<CS>([&](auto s) MPQP_INL {
                R.t[b][s] = __builtin_amdgcn_mfma_f32_4x4x1f32(a, al[s], R.t[b][s], 4, decltype(b)::value, 0);
            });
    });
}

// FP64: row `lr` of the wave := al (blocks of rows for fewer tests)
template <int NW, int RW, int CS, int EX, int LW>
__device__ __forceinline__ void reg_set_row(RegTab<double, NW, RW, CS, EX, LW> &R, int lr, const double (&al)[CS + 1]) {
    constexpr int RR = RW - LW, B = 4;
    if (LW > 0 && lr >= RR)
        reg_for<CS>([&](auto s) MPQP_INL { R.lt[((lr - RR) * CS + s) * MPQP_WAVE] = al[s]; });
    reg_for<(RR + B - 1) / B>([&](auto b) MPQP_INL {
        if (lr / B == b)
            reg_for<B>([&](auto u) MPQP_INL {
                constexpr int i = decltype(b)::value * B + decltype(u)::value;
                if constexpr (i < RR) reg_for<CS>([&](auto s) MPQP_INL { R.t[i][s] = lr == i ? al[s] : R.t[i][s]; });
            });
    });
}

// The pivot row's wave: row lr (al) divided by p into L.ep (1 / p at column
// q, if any), with its rhs and perturbation entries; the row itself is left
// zero for reg_apply (FP32).
template <typename Re, int NW, int RW, int CS, int EX, int LW>
__device__ __forceinline__ void reg_divide(RegTab<Re, NW, RW, CS, EX, LW> &R, const RegLds<Re, NW, RW, CS, EX, LW> &L, const Re (&al)[CS + 1],
                                           int lr, int q, Re p) {
    const int lane = fresh_lane();
    reg_for<CS + 1>([&](auto s) MPQP_INL {
        const int c = lane + MPQP_WAVE * s;
        L.ep[c] = (c == q ? (Re)1 : al[s]) / p;
    });
    if constexpr (sizeof(Re) == 4) reg_clear_row(R, lr, al);
}

template <typename Re, int NW, int RW, int CS, int EX, int LW>
__device__ __forceinline__ void reg_publish(RegTab<Re, NW, RW, CS, EX, LW> &R, const RegLds<Re, NW, RW, CS, EX, LW> &L, const Re (&al)[CS + 1],
                                            int lr, int q) {
    Re v = al[0];
    reg_for<RegTab<Re, NW, RW, CS, EX, LW>::NS>([&](auto s) MPQP_INL { v = q / MPQP_WAVE == s ? al[s] : v; });
    reg_divide(R, L, al, lr, q, lane_get(v, q % MPQP_WAVE));
}

// The rank-1 update of the wave's rows by the divided pivot row pr (pr[CS]:
// extra columns, rhs, perturbation) with the factors fv by lane.  FP32: the
// wave that holds the pivot row r finds it zero: its factor -1 puts pr there.
// FP64: a column whose entry of pr is zero keeps its entries, column q (any,
// or -1) starts from zero, and the pivot row is put in place.
template <bool COL = false, typename Re, int NW, int RW, int CS, int EX, int LW>
__device__ __forceinline__ void reg_apply(RegTab<Re, NW, RW, CS, EX, LW> &R, const RegLds<Re, NW, RW, CS, EX, LW> &L,
                                          const Re (&pr)[CS + 1], Re fv, int r, int q) {
    const int lane = fresh_lane(), wave = wave_id(), lr = r - wave * RW;
    if constexpr (sizeof(Re) == 8) {
        constexpr int CH = 16;  // rows whose factors are in scalar registers at a time
        const int lq = q % MPQP_WAVE;
        // (COL: the factors are column q, taken a chunk at a time: its lane's
        // entries of one slot, or the extra column that fv already is)
        constexpr int RR = RW - LW;
        if constexpr (LW > 0) {
            if (COL && q < MPQP_WAVE * CS) fv = reg_lds_col(R, q < 0 ? 0 : q);
        }
        reg_for<(RR + CH - 1) / CH>([&](auto h) MPQP_INL {
            constexpr int i0 = decltype(h)::value * CH, n = RR - i0 < CH ? RR - i0 : CH;
            Re f[n];
            if (!COL || (EX > 0 && q >= MPQP_WAVE * CS)) {
                reg_for<n>([&](auto i) MPQP_INL { f[i] = lane_get(fv, i0 + decltype(i)::value); });
            }
            if constexpr (COL)
                reg_for<CS>([&](auto s) MPQP_INL {
                    if (q / MPQP_WAVE == s)
                        reg_for<n>([&](auto i) MPQP_INL {
                            constexpr int I = i0 + decltype(i)::value;
                            f[i] = lane_get(R.t[I][s], lq);
                            fv = lane_set(fv, I, f[i]);
                        });
                });
            reg_for<CS>([&](auto s) MPQP_INL {
                constexpr int S = decltype(s)::value;
                const bool at = lane + MPQP_WAVE * S == q;
                if (pr[S] != (Re)0 && !at)
                    reg_for<n>([&](auto i) MPQP_INL {
                        constexpr int I = i0 + decltype(i)::value;
                        R.t[I][S] = fma(-f[i], pr[S], R.t[I][S]);
                    });
                if (at)
                    reg_for<n>([&](auto i) MPQP_INL {
                        constexpr int I = i0 + decltype(i)::value;
                        R.t[I][S] = fma(-f[i], pr[S], (Re)0);
                    });
            });
        });
        // the LDS rows, G of them in flight
        constexpr int G = 4;
        reg_for<(LW + G - 1) / G>([&](auto h) MPQP_INL {
            constexpr int g0 = decltype(h)::value * G, n = LW - g0 < G ? LW - g0 : G;
            Re f[n];
            reg_for<n>([&](auto i) MPQP_INL { f[i] = lane_get(fv, RR + g0 + i); });
            reg_for<CS>([&](auto s) MPQP_INL {
                Re x[n];
                reg_for<n>([&](auto i) MPQP_INL { x[i] = R.lt[((g0 + i) * CS + s) * MPQP_WAVE]; });
                const bool at = lane + MPQP_WAVE * s == q;
                reg_for<n>([&](auto i) MPQP_INL {
                    x[i] = fma(-f[i], pr[s], at ? (Re)0 : x[i]);
                });
                if (pr[s] != (Re)0)
                    reg_for<n>([&](auto i) MPQP_INL { R.lt[((g0 + i) * CS + s) * MPQP_WAVE] = x[i]; });
            });
        });
        if ((unsigned)lr < (unsigned)RW) reg_set_row(R, lr, pr);
        reg_for<EX + 2>([&](auto e) MPQP_INL {
            const Re p = lane_get(pr[CS], e), x0 = q == MPQP_WAVE * CS + e && e < EX ? (Re)0 : R.xs[e];
            const Re xn = p != (Re)0 ? fma(-fv, p, x0) : x0;
            R.xs[e] = lane == lr ? p : xn;
        });
    } else {
        const float nf = lane == lr ? 1.f : -fv;
        reg_for<CS>([&](auto s) MPQP_INL { reg_rank1<decltype(s)::value>(R, nf, pr[s]); });
        reg_for<EX + 2>([&](auto e) MPQP_INL { R.xs[e] = fma(nf, lane_get(pr[CS], e), lane == lr ? 0.f : R.xs[e]); });
    }
    if (lane < RW) {
        L.gx[wave * RW + lane] = R.x();
        L.gp[wave * RW + lane] = R.xp();
    }
}

// The pivot on (r, q) from the divided row in L.ep, by every wave, cost row
// included.  Barriers before (L.ep written) and after belong to the caller.
// MAYBE: r < 0 leaves everything as it is (a branch around the update would
// give the tableau's registers two states to be merged).
template <bool MAYBE = false, typename Re, int NW, int RW, int CS, int EX, int LW>
__device__ __forceinline__ void reg_update(RegTab<Re, NW, RW, CS, EX, LW> &R, const RegLds<Re, NW, RW, CS, EX, LW> &L, int r, int q) {
    const int lane = fresh_lane();
    const bool off = MAYBE && r < 0;
    Re fv = 0;
    if constexpr (sizeof(Re) == 4) fv = reg_col_op<true>(R, L, q, !off);
    else reg_for<EX>([&](auto e) MPQP_INL { fv = q == MPQP_WAVE * CS + e ? R.xs[e] : fv; });
    Re pr[CS + 1], dv = 0;
    reg_for<CS + 1>([&](auto s) MPQP_INL {
        pr[s] = L.ep[lane + MPQP_WAVE * s];
        if constexpr (MAYBE) pr[s] = off ? (Re)0 : pr[s];
    });
    if constexpr (MAYBE) fv = off ? (Re)0 : fv;
    constexpr int NS = RegTab<Re, NW, RW, CS, EX, LW>::NS;
    reg_for<NS>([&](auto s) MPQP_INL { dv = q / MPQP_WAVE == s ? R.d[s] : dv; });
    const Re fd = lane_get(dv, q % MPQP_WAVE);
    reg_for<NS>([&](auto s) MPQP_INL {
        const Re d0 = lane + MPQP_WAVE * s == q && !off ? (Re)0 : R.d[s];
        R.d[s] = pr[s] != (Re)0 ? fma(-fd, pr[s], d0) : d0;
    });
    reg_apply<true>(R, L, pr, fv, off ? -MPQP_WAVE * NW : r, off ? -1 : q);
}

// Cost row d = init(column) - c * (sum of the rows whose basic variable
// satisfies sel), rows ascending: the waves that hold such rows continue the
// chain one after the other through L.dl.
template <typename Re, int NW, int RW, int CS, int EX, int LW, typename SelF, typename InitF>
__device__ __forceinline__ void reg_cost(RegTab<Re, NW, RW, CS, EX, LW> &R, const RegLds<Re, NW, RW, CS, EX, LW> &L, int M, int K,
                                         Re c, SelF sel, InitF init) {
    constexpr int NS = RegTab<Re, NW, RW, CS, EX, LW>::NS;
    const int lane = fresh_lane(), wave = wave_id();
    reg_for<NS>([&](auto s) MPQP_INL {
        const int col = lane + MPQP_WAVE * s;
        R.d[s] = col < K ? (Re)init(col) : (Re)0;
    });
    bool started = false;
    for (int w = 0; w < NW; ++w) {
        const int row = w * RW + lane;
        const unsigned long long m = __ballot(lane < RW && row < M && sel(L.basis[row < M ? row : 0]));
        if (m == 0ull) continue;
        if (wave == w) {
            if (started)
                reg_for<NS>([&](auto s) MPQP_INL { R.d[s] = L.dl[lane + MPQP_WAVE * s]; });
            reg_for<RW>([&](auto i) MPQP_INL {
                if ((m >> i) & 1ull) {
                    reg_for<CS>([&](auto s) MPQP_INL { R.d[s] = fma(-c, R.template get<decltype(i)::value, decltype(s)::value>(), R.d[s]); });
                    if constexpr (EX > 0) {
                        Re v = 0;
                        reg_for<EX>([&](auto e) MPQP_INL { v = lane == e ? lane_get(R.xs[e], i) : v; });
                        R.d[CS] = fma(-c, v, R.d[CS]);
                    }
                }
            });
            reg_for<NS>([&](auto s) MPQP_INL { L.dl[lane + MPQP_WAVE * s] = R.d[s]; });
        }
        started = true;
        __syncthreads();
    }
    if (started) {
        reg_for<NS>([&](auto s) MPQP_INL { R.d[s] = L.dl[lane + MPQP_WAVE * s]; });
        __syncthreads();
    }
}

// d into L.dl (wave 0)
template <typename Re, int NW, int RW, int CS, int EX, int LW>
__device__ __forceinline__ void reg_cost_out(const RegTab<Re, NW, RW, CS, EX, LW> &R, const RegLds<Re, NW, RW, CS, EX, LW> &L) {
    if (wave_id() == 0) {
        const int lane = fresh_lane();
        reg_for<RegTab<Re, NW, RW, CS, EX, LW>::NS>([&](auto s) MPQP_INL { L.dl[lane + MPQP_WAVE * s] = R.d[s]; });
    }
}

// The wave's smallest basic value (perturbed: x + xp) for the choice of the
// leaving row.  The reference tree keeps, of equal values with equal counts,
// the index whose lowest bits are clear first (see tree_first): the smallest
// index with its bits reversed.
template <typename Re, int NW, int RW, int CS, int EX, int LW>
__device__ __forceinline__ void reg_min_out(const RegTab<Re, NW, RW, CS, EX, LW> &R, RegShared<Re, NW> &ws, int M,
                                            bool pert) {
    const int lane = fresh_lane(), wave = wave_id(), row = wave * RW + lane;
    const bool valid = lane < RW && row < M;
    const Re x = pert ? R.x() + R.xp() : R.x();
    const bool nan = valid && x != x;
    const Re v = (valid && !nan) ? x : (Re)INFINITY;
    const Re m1 = wave_min(v);
    const unsigned long long hit = __ballot(v == m1 && valid);
    const unsigned long long near = hit | __ballot(valid && !((double)m1 <= (double)v - 1e-10));
    int f = __ffsll((long long)hit) - 1, flag = 0;
    const int cnt = __builtin_amdgcn_readlane(R.cb, f < 0 ? 0 : f);
    if ((near & (near - 1)) != 0ull) {
        flag = (near & ~__ballot(R.cb == cnt)) != 0ull ? 1 : 0;
        const unsigned k = wave_min((hit >> lane) & 1ull ? __brev((unsigned)row) : ~0u);
        f = hit ? (int)__brev(k) - wave * RW : f;
    }
    if (__any(nan)) flag |= 2;
    if (hit == 0ull) flag |= 4;
    if (lane == 0) {
        ws.min[wave] = RegMin<Re>{m1, wave * RW + f, cnt, flag};
    }
}

// primal_ratio_wave over the register tableau, by the whole workgroup: every
// wave returns the row.  Two barriers.
template <typename Re, int NW, int RW, int CS, int EX, int LW>
__device__ __forceinline__ int reg_ratio(const RegTab<Re, NW, RW, CS, EX, LW> &R, const RegLds<Re, NW, RW, CS, EX, LW> &L, RegShared<Re, NW> &ws,
                                         int M, int q, const DevTol &tl) {
    const int lane = fresh_lane(), wave = wave_id();
    const bool valid = lane < RW && wave * RW + lane < M;
    const Re a = reg_col(R, L, q);
    Re lim = (Re)tl.tol_plus;
    if (tl.pivot_rel > 0.0) {
        const Re fa = fabs(a);
        const Re cw = -wave_min((valid && fa > (Re)0) ? -fa : (Re)0);
        if (lane == 0) ws.cmax[wave] = cw;
        __syncthreads();
        const Re cm = -lane_get(row8_min(-ws.cmax[lane % NW]), 7);
        const Re rl = (Re)tl.pivot_rel * cm;
        lim = rl > lim ? rl : lim;
    }
    // the wave's smallest ratio, its lowest row
    const bool take = valid && a > lim;
    const Re rt = take ? R.x() / a : (Re)0;
    const bool num = take && rt == rt;
    const Re m = wave_min(num ? rt : (Re)INFINITY);
    const unsigned long long hit = __ballot(num && rt == m), any = __ballot(take);
    const int f = __ffsll((long long)(hit ? hit : any)) - 1;
    if (lane == 0) {
        ws.rv[wave] = m;
        ws.rk[wave] = f < 0 ? -1 : wave * RW + f;
    }
    __syncthreads();
    const int k = ws.rk[lane % NW];
    const Re v = k >= 0 ? ws.rv[lane % NW] : (Re)INFINITY;
    const Re mm = lane_get(row8_min(v), 7);
    const unsigned long long has = __ballot(lane < NW && k >= 0), best = __ballot(lane < NW && k >= 0 && v == mm);
    const int w = __ffsll((long long)(best ? best : has)) - 1;
    return w < 0 ? -1 : __builtin_amdgcn_readlane(k, w);
}

// A pivot on (r, q) that every wave knows: the row's wave divides and
// publishes it, every wave updates; `between` is run by one thread while the
// update runs (the basis bookkeeping).  Two barriers.
template <typename Re, int NW, int RW, int CS, int EX, int LW, typename F>
__device__ __forceinline__ void reg_pivot(RegTab<Re, NW, RW, CS, EX, LW> &R, const RegLds<Re, NW, RW, CS, EX, LW> &L, int r, int q,
                                          F between) {
    const int wave = wave_id(), lr = r - wave * RW;
    if ((unsigned)lr < (unsigned)RW) {
        Re al[CS + 1];
        reg_row(R, lr, al);
        reg_publish(R, L, al, lr, q);
    }
    __syncthreads();
    if (threadIdx.x == (NW - 1) * MPQP_WAVE) between();
    reg_update(R, L, r, q);
    __syncthreads();
}

template <typename LT>
__device__ __forceinline__ void reg_swap(const LT &L, int r, int q) {
    const int t = L.basis[r], v = L.nonb[q];
    L.basis[r] = v;
    L.nonb[q] = t;
    L.where[v] = r;
    L.where[t] = -(q + 1);
}

// ---------------------------------------------------------------------
// start
// ---------------------------------------------------------------------
template <typename Re, int NW, int RW, int CS, int EX, int LW, typename Src>
__device__ __forceinline__ void reg_load(RegTab<Re, NW, RW, CS, EX, LW> &R, const RegLds<Re, NW, RW, CS, EX, LW> &L,
                                         const DevProb &P, const Src *sT, int src_ld, const int *sb, const int *sn) {
    const int M = P.M2, K = P.K2;
    const int lane = fresh_lane(), wave = wave_id();
    unsigned cc[CS];
    reg_for<CS>([&](auto s) MPQP_INL {
        const int c = lane + MPQP_WAVE * s;
        cc[s] = c < K ? c : 0;
    });
    reg_for<RW>([&](auto i) MPQP_INL {
        const int row = min(wave * RW + i, M - 1);
        const Src *rp = sT + (long long)row * src_ld;
        reg_for<CS>([&](auto s) MPQP_INL { R.template set<decltype(i)::value, decltype(s)::value>((Re)rp[cc[s]]); });
    });
    const int row = wave * RW + lane;
    const bool valid = lane < RW && row < M;
    const Src *rr = sT + (long long)(valid ? row : 0) * src_ld;
    reg_for<EX>([&](auto e) MPQP_INL {
        const int c = MPQP_WAVE * CS + e;
        R.xs[e] = (valid && c < K) ? (Re)rr[c] : (Re)0;
    });
    R.xs[EX] = valid ? (Re)rr[K] : (Re)0;
    R.xs[EX + 1] = valid ? (Re)rr[K + 1] : (Re)0;
    for (int i = threadIdx.x; i < M; i += NW * MPQP_WAVE) {
        const int b = sb[i];
        L.basis[i] = b;
        L.where[b] = i;
    }
    for (int kk = threadIdx.x; kk < K; kk += NW * MPQP_WAVE) {
        const int v = sn[kk];
        L.nonb[kk] = v;
        L.where[v] = -(kk + 1);
    }
    __syncthreads();
}

// opt_lambda: the lambda swaps of S[j0 .. j1), a row's terms in ascending t,
// zeros skipped.  A thread walks its row's e-columns: in FP32 the rows are
// staged in LDS; in FP64 the first swap reads them from the state that was
// just loaded (sT, still as it was), and later ones, of a cold start, take
// the columns out of the registers one after the other.
template <typename Re, int NW, int RW, int CS, int EX, int LW>
__device__ __forceinline__ int reg_lambda(RegTab<Re, NW, RW, CS, EX, LW> &R, const RegLds<Re, NW, RW, CS, EX, LW> &L,
                                          const DevProb &P, const DevTol &tl, const int *Sset, int j0, int j1,
                                          const Re *sT, int src_ld) {
    const int M = P.M2, K = P.K2, N2 = P.N2;
    const int r4 = M - P.n_c - P.n_x, nt = P.n_x + 1;
    const int tid = threadIdx.x;
    Re *lam = L.ep;
    int *wl = L.bcnt;
    auto walk = [&](const Re *Ti, int row) {
        // loads of U terms in flight
        constexpr int U = sizeof(Re) == 4 ? 4 : 8;
        Re acc = 0;
        for (int t0 = 0; t0 < nt; t0 += U) {
            Re av[U], tv[U];
            int w[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int t = t0 + u < nt ? t0 + u : nt - 1;
                av[u] = t0 + u < nt ? lam[t] : (Re)0;
                w[u] = wl[t];
            }
#pragma unroll
            for (int u = 0; u < U; ++u) tv[u] = Ti[w[u] >= 0 ? 0 : -w[u] - 1];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const Re f1 = fma(av[u], (Re)1, acc);
                const Re f2 = fma(av[u], tv[u], acc);
                const Re na = w[u] >= 0 ? (row == w[u] ? f1 : acc) : f2;
                acc = av[u] == (Re)0 ? acc : na;
            }
        }
        L.colx[row] = acc;
    };
    for (int jj = j0; jj < j1; ++jj) {
        const int j = Sset[jj];
        for (int t = tid; t < nt; t += NW * MPQP_WAVE) {
            const int rho = t == 0 ? j : r4 + t - 1;
            lam[t] = (Re)lam_entry(P, j, rho);
            wl[t] = L.where[N2 - M + rho];
        }
        if constexpr (sizeof(Re) == 4) {
            for (int h = 0; h < L.np; ++h) {
                reg_dump(R, L, K, h);
                __syncthreads();
                for (int i = tid; i < L.rp && h * L.rp + i < M; i += NW * MPQP_WAVE)
                    walk(L.stage + i * L.sld, h * L.rp + i);
                __syncthreads();
            }
        } else {
            __syncthreads();
            if (jj == j0) {
                for (int i = tid; i < M; i += NW * MPQP_WAVE) walk(sT + (long long)i * src_ld, i);
            } else {
                const int lane = fresh_lane(), row = wave_id() * RW + lane;
                Re acc = 0;
                for (int t = 0; t < nt; ++t) {
                    const Re av = lane_get(lam[t], 0);
                    const int w = rfl(wl[t]);
                    const Re tv = reg_col(R, L, w >= 0 ? 0 : -w - 1);
                    const Re f1 = fma(av, (Re)1, acc);
                    const Re f2 = fma(av, tv, acc);
                    const Re na = w >= 0 ? (row == w ? f1 : acc) : f2;
                    acc = av == (Re)0 ? acc : na;
                }
                if (lane < RW && row < M) L.colx[row] = acc;
            }
            __syncthreads();
        }
        const int p = rfl(L.where[P.n_x + P.n_t + j]);
        const int lane = fresh_lane(), wave = wave_id();
        const int row = wave * RW + lane;
        const Re fv = (lane < RW && row < M) ? L.colx[row] : (Re)0;
        // w_j basic at position p: a pivot on row p with the column vcol held
        // outside the tableau; w_j nonbasic in column kk: the column
        // replaced (T - column * 1, then + vcol * 1, in its lane)
        const Re pv = lane_get(L.colx[p >= 0 ? p : 0], 0);
        if (p >= 0 && !(fabs((double)pv) > tl.licq)) return 0;
        const int kk = p >= 0 ? -1 : -p - 1, lr = p - wave * RW;
        if (p >= 0 && (unsigned)lr < (unsigned)RW) {
            Re al[CS + 1];
            reg_row(R, lr, al);
            reg_divide(R, L, al, lr, -1, pv);
        }
        __syncthreads();
        if constexpr (sizeof(Re) == 4) reg_col_op<true>(R, L, kk < 0 ? 0 : kk, kk >= 0);
        Re pr[CS + 1];
        reg_for<CS + 1>([&](auto s) MPQP_INL {
            const int col = lane + MPQP_WAVE * s;
            pr[s] = kk < 0 ? L.ep[col] : (col == kk ? (Re)1 : (Re)0);
        });
        reg_apply(R, L, pr, kk < 0 ? fv : -fv, kk < 0 ? p : -MPQP_WAVE * NW, kk);
        __syncthreads();
    }
    return 1;
}

// ---------------------------------------------------------------------
// phase 1 (opt_phase1's decisions)
// ---------------------------------------------------------------------
template <typename Re, int NW, int RW, int CS, int EX, int LW>
__device__ __forceinline__ P1Result reg_phase1(RegTab<Re, NW, RW, CS, EX, LW> &R, const RegLds<Re, NW, RW, CS, EX, LW> &L,
                                               const DevProb &P, const DevOpts &O, const DevTol &tl, OptShared &sh,
                                               RegShared<Re, NW> &ws) {
    constexpr int SM = (NW * RW + MPQP_WAVE - 1) / MPQP_WAVE, NS = RegTab<Re, NW, RW, CS, EX, LW>::NS;
    const int M = P.M2, K = P.K2, N2 = P.N2, Nn = P.Nn;
    const int wave = wave_id();
    reg_cost(R, L, M, K, (Re)1, [&](int b) { return b >= Nn; },
             [&](int col) { return L.nonb[col] >= Nn ? 1.f : 0.f; });
    for (int v = threadIdx.x; v < N2; v += NW * MPQP_WAVE) { L.bcnt[v] = 0; L.nbcnt[v] = 0; }
    {
        const int lane = fresh_lane();
        if (lane < RW) {
            L.gx[wave * RW + lane] = R.x();
            L.gp[wave * RW + lane] = R.xp();
        }
    }
    P1Result res{ST_ITER_CAP, 0, 0, 0.0};
    int n_same = 0, no_pert = 0;
    double best_p = -INFINITY;
    int it = 0;
    bool stopped = false;  // uniform, as every condition around the pivots must be
    R.cb = 0;
    reg_min_out(R, ws, M, n_same >= O.stall_perturb);
    __syncthreads();
    // One exit and one way back, so that the tableau has one place: what
    // ends the loop is noted and acted on before the update.
    bool stall = false;
    for (;;) {
        int r = -1, q = -1, act = ACT_PIVOT;
        int ec = 0;  // the leaving row's wave: use count of the entering variable
        bool pert = false;
        for (;;) {
            if (stall) { act = ACT_STOP; res.status = ST_STALL; break; }
            if (it >= O.max_iter_p1) { act = ACT_STOP; break; }
            pert = !no_pert && n_same >= O.stall_perturb;
            const int lane = fresh_lane();
            // Leaving row, by every wave.  Without counter preference the
            // predicate lets a value give way to a smaller one, and within
            // its 1e-10 band to one of a smaller count: where the counts of
            // the values within that band of the minimum are all the same
            // (and none is NaN), the minima win every combine, and of them
            // the first in the tree's order remains (FP64 values of a
            // degenerate basis tie exactly, three decisions of four).
            // Anything else runs the tree.
            const RegMin<Re> w = ws.min[lane % NW];
            const Re m = lane_get(row8_min(lane < NW ? w.m1 : (Re)INFINITY), 7);
            const bool go_on = (double)m < tl.dual_stop_tol;
            const int mode_b = (n_same % 20) >= 10 ? 1 : 0;
            const unsigned long long wh = __ballot(lane < NW && w.m1 == m && !(w.flag & 4));
            const bool wn = lane < NW && !((double)m <= (double)w.m1 - 1e-10);
            const int f = __ffsll((long long)wh) - 1;
            r = __builtin_amdgcn_readlane(w.at, f < 0 ? 0 : f);
            const int c0 = __builtin_amdgcn_readlane(w.cnt, f < 0 ? 0 : f);
            const bool mixed_counts = wn && ((w.flag & 1) || w.cnt != c0);
            if ((wh & (wh - 1)) != 0ull)
                r = (int)__brev(lane_get(row8_min((wh >> lane) & 1ull ? __brev((unsigned)w.at) : ~0u), 7));
            if (rfl((mode_b || f < 0 || __any(mixed_counts || (lane < NW && (w.flag & 2)))) ? 1 : 0)) {
                Re v[SM];
                int id[SM], cn[SM];
#pragma unroll
                for (int s = 0; s < SM; ++s) {
                    const int i = lane + MPQP_WAVE * s;
                    const bool valid = i < M;
                    const int ic = valid ? i : 0;
                    const Re x0 = L.gx[ic], xp = L.gp[ic];
                    v[s] = valid ? (pert ? x0 + xp : x0) : (Re)0;
                    id[s] = ic;
                    cn[s] = L.bcnt[L.basis[ic]];
                }
                r = reg_tree<SM>(v, id, cn, M, lane, DminPred{mode_b, tl.dual_stop_tol});
            }
            r = rfl(r);
            if (rfl(go_on ? 1 : 0)) break;
            act = ACT_STOP;
            if (pert) {
                bool inf = false;
                for (int i = lane; i < M; i += MPQP_WAVE) inf |= (double)L.gx[i] < tl.dual_stop_tol;
                if (__any(inf)) act = ACT_UNPERT;
            }
            if (rfl(act) == ACT_STOP) { stopped = true; break; }
            act = ACT_PIVOT;
            no_pert = 1;
            n_same = 0;
            best_p = -INFINITY;
            __syncthreads();
            if (threadIdx.x == 0) L.bcnt[L.basis[r]] += 1;
            R.cb += lane == r - wave * RW ? 1 : 0;
            reg_min_out(R, ws, M, false);
            __syncthreads();
            ++it;
        }
        if (rfl(act) == ACT_PIVOT) {
            const int lane = fresh_lane();
            const int wo = r / RW, lr = r - wo * RW;
            if (wave == wo) { MPQP_PRIO_HI();
                // entering column, by the wave that holds the leaving row
                // (the use counts only matter to the trees; read ahead)
                int cnt_of[NS];
                reg_for<NS>([&](auto s) MPQP_INL {
                    const int kk = lane + MPQP_WAVE * s;
                    cnt_of[s] = L.nbcnt[L.nonb[kk < K ? kk : 0]];
                });
                Re al[CS + 1];
                reg_row(R, lr, al);
                Re dlim = (Re)tl.tol_minus;
                if (tl.pivot_rel > 0.0) {
                    Re am = 0;
                    reg_for<NS>([&](auto s) MPQP_INL {
                        const Re a = lane + MPQP_WAVE * s < K ? (Re)fabs(al[s]) : (Re)0;
                        am = a > am ? a : am;
                    });
                    const Re rl = -(Re)tl.pivot_rel * -wave_min(-am);
                    dlim = rl < dlim ? rl : dlim;
                }
                const int mode = n_same < 10 ? 0 : (n_same < 100 ? 1 : 2);
                Re v[NS];
                bool tk[NS];
                Re ml = (Re)INFINITY;
                bool nn = false, any_t = false;
                reg_for<NS>([&](auto s) MPQP_INL {
                    tk[s] = lane + MPQP_WAVE * s < K && al[s] < dlim;
                    v[s] = -R.d[s] / al[s];
                    any_t |= tk[s];
                    nn |= tk[s] && v[s] != v[s];
                    ml = (tk[s] && v[s] < ml) ? v[s] : ml;
                });
                int qk = -2;
                if (!__any(any_t)) {
                    qk = -1;
                } else if (mode < 2 && !__any(nn)) {
                    // The reference tree without its values.  mode 0 replaces
                    // an entry only by a strictly smaller one: the first of the
                    // minima in the tree's order.  mode 1 also where a count
                    // exceeds the other's by more than 2 and the values are
                    // within 1e-12: if no other value lies within that band
                    // of the minimum, the minima are compared by their counts
                    // alone, and any of them beats everything else.
                    const Re m = wave_min(ml);
                    unsigned long long hit[NS];
                    bool near = false;
                    int cnt = 0;
                    reg_for<NS>([&](auto s) MPQP_INL {
                        hit[s] = __ballot(tk[s] && v[s] == m);
                        near |= tk[s] && v[s] != m && (double)m >= (double)v[s] - 1e-12;
                        cnt += __popcll(hit[s]);
                    });
                    if (mode == 0 || (cnt == 1 && !__any(near))) {
                        qk = tree_first<NS>(hit);
                    } else if (!__any(near)) {
                        int id[NS];
                        reg_for<NS>([&](auto s) MPQP_INL { id[s] = tk[s] && v[s] == m ? lane + MPQP_WAVE * s : -1; });
                        qk = reg_tree<NS>(v, id, cnt_of, K, lane, [](double, int it, int ct, double, int iu, int cu) {
                            return (iu >= 0) & ((it < 0) | (ct > cu + 2));
                        });
                    }
                }
                if (qk == -2) {
                    int id[NS];
                    reg_for<NS>([&](auto s) MPQP_INL {
                        id[s] = tk[s] ? lane + MPQP_WAVE * s : -1;
                        v[s] = tk[s] ? v[s] : (Re)100000;
                    });
                    qk = reg_tree<NS>(v, id, cnt_of, K, lane, DratioPred{mode});
                }
                qk = rfl(qk);
                if (qk >= 0) {
                    // read before the barrier: behind it the last wave's first
                    // thread writes the bookkeeping, whenever it gets there
                    const int nv = L.nonb[qk];
                    reg_publish(R, L, al, lr, qk);
                    ec = L.bcnt[nv];
                }
                if (lane == 0) sh.q = qk;
                MPQP_PRIO_LO();
            }
            if (wave == (wo + 1) % NW) {
                // meanwhile: the sum of the negative x_B for the stall counter
                Re ps[SM];
    #pragma unroll
                for (int s = 0; s < SM; ++s) {
                    const int i = lane + MPQP_WAVE * s;
                    const int ic = i < M ? i : 0;
                    const Re x0 = L.gx[ic], xp = L.gp[ic];
                    const Re x = (pert && i < M) ? x0 + xp : x0;
                    ps[s] = (i < M && x < (Re)0) ? x : (Re)0;
                }
                tree_sum_lane0<SM, Re>(ps, M, lane);
                if (lane == 0) sh.pinf = (double)ps[0];
            }
            __syncthreads();
            q = rfl(sh.q);
            if (q < 0) res.status = ST_UNBOUNDED;
            OPT_PROF(sh, 1);
        }
        if (opaque(q) < 0) break;
        const double pinf = rfl_d(sh.pinf);
        if (pinf > best_p) {
            best_p = pinf;
            n_same = 0;
        } else {
            ++n_same;
        }
        stall = n_same > O.stall_exit;
        // Up to the closing barrier the bookkeeping is one thread's alone; its
        // reads pass while the tableau is updated.
        const bool keeper = threadIdx.x == (NW - 1) * MPQP_WAVE;
        int bv = 0, nv = 0, bc = 0, nc = 0;
        if (keeper) {
            bv = L.basis[r];
            nv = L.nonb[q];
            bc = L.bcnt[bv];
            nc = L.nbcnt[nv];
        }
        reg_update(R, L, r, q);
        R.cb = fresh_lane() == r - wave * RW ? ec : R.cb;
        if (keeper) {
            L.bcnt[bv] = bc + 1;
            L.nbcnt[nv] = nc + 1;
            L.basis[r] = nv;
            L.nonb[q] = bv;
            L.where[nv] = r;
            L.where[bv] = -(q + 1);
        }
        reg_min_out(R, ws, M, !no_pert && n_same >= O.stall_perturb);
        ++res.iters;
        ++it;
        __syncthreads();
        OPT_PROF(sh, 2);
    }
    __syncthreads();
    if (!stopped) return res;

    // dual-feasibility cleanup (see opt_phase1)
    int end = 0;  // 1: dual feasible (or accepted), 2: unbounded, 3: iteration cap
    for (;;) {
        int r = -1, aux = -1;
        if (it >= O.max_iter_p1) {
            end = 3;
        } else {
            const int lane = fresh_lane();
            Re dl = (Re)INFINITY;
            bool nn = false;
            reg_for<NS>([&](auto s) MPQP_INL {
                const bool in = lane + MPQP_WAVE * s < K;
                nn |= in && R.d[s] != R.d[s];
                dl = (in && R.d[s] < dl) ? R.d[s] : dl;
            });
            const Re dm = wave_min(dl);
            double dv = (double)dm;
            int cnt = 0;
            reg_for<NS>([&](auto s) MPQP_INL {
                const unsigned long long hit = __ballot(lane + MPQP_WAVE * s < K && R.d[s] == dm);
                cnt += __popcll(hit);
                aux = hit ? __ffsll((long long)hit) - 1 + MPQP_WAVE * s : aux;
            });
            if (!(dv > tl.tol_minus) && (cnt != 1 || __any(nn))) {
                // lowest variable on ties
                int key = -1;
                aux = -1;
                dv = 0.0;
                reg_for<NS>([&](auto s) MPQP_INL {
                    const int kk = lane + MPQP_WAVE * s;
                    const double dd = (double)R.d[s];
                    const int var = L.nonb[kk < K ? kk : 0];
                    if (kk < K && (key < 0 || dd < dv || (dd == dv && var < key))) { dv = dd; key = var; aux = kk; }
                });
                lex_min(dv, key, aux);
            }
            if (dv > tl.tol_minus) {
                end = 1;
            } else {
                r = reg_ratio(R, L, ws, M, aux, tl);
                if (r < 0) end = tl.cleanup_accept ? 1 : 2;
            }
        }
        if (opaque(end)) break;
        reg_pivot(R, L, r, aux, [&] { reg_swap(L, r, aux); });
        ++res.iters;
        ++it;
    }
    if (end == 2) res.status = ST_UNBOUNDED;
    if (end != 1) return res;
    if (wave == 0) {
        const int lane = fresh_lane();
        Re zs[SM];
#pragma unroll
        for (int s = 0; s < SM; ++s) {
            const int i = lane + MPQP_WAVE * s;
            zs[s] = (i < M) ? (L.basis[i] >= Nn ? (Re)1 : (Re)0) * L.gx[i] : (Re)0;
        }
        const double zz = (double)tree_sum_s<SM, Re>(zs, M, lane);
        if (lane == 0) sh.z = zz;
    }
    reg_cost_out(R, L);
    __syncthreads();
    res.status = ST_OPTIMAL;
    res.z1 = rfl_d(sh.z);
    res.kkt = (res.z1 > -tl.dual_feas_tol && res.z1 < tl.dual_feas_tol) ? 1 : 0;
    return res;
}

// opt_drive_out (on = 0: nothing to do)
template <typename Re, int NW, int RW, int CS, int EX, int LW>
__device__ __forceinline__ int reg_drive_out(RegTab<Re, NW, RW, CS, EX, LW> &R, const RegLds<Re, NW, RW, CS, EX, LW> &L, const DevProb &P,
                                             const DevTol &tl, OptShared &sh, int on) {
    constexpr int SM = (NW * RW + MPQP_WAVE - 1) / MPQP_WAVE, NS = RegTab<Re, NW, RW, CS, EX, LW>::NS;
    const int M = P.M2, K = P.K2, Nn = P.Nn;
    rows_where<SM>(L.rows, M, sh, [&](int i) { return L.basis[i] >= Nn; });
    const int n = on ? rfl(sh.nrows) : 0, wave = wave_id();
    int clean = 1;
    for (int t = 0; t < n; ++t) {
        const int i = rfl(L.rows[t]), lr = i - wave * RW;
        if ((unsigned)lr < (unsigned)RW) {
            const int lane = fresh_lane();
            Re al[CS + 1];
            reg_row(R, lr, al);
            double v = 0.0;
            int key = -1, aux = 0;
            reg_for<NS>([&](auto s) MPQP_INL {
                const int kk = lane + MPQP_WAVE * s;
                if (kk < K && L.nonb[kk] < Nn) {
                    const double a = fabs((double)al[s]);
                    if (a > tl.tol_plus && (key < 0 || -a < v)) { v = -a; key = kk; }
                }
            });
            lex_min(v, key, aux);
            if (key >= 0) reg_publish(R, L, al, lr, key);
            if (lane == 0) sh.best = key;
        }
        __syncthreads();
        const int best = rfl(sh.best);
        clean = best < 0 ? 0 : clean;
        if (threadIdx.x == (NW - 1) * MPQP_WAVE && best >= 0) reg_swap(L, i, best);
        reg_update<true>(R, L, best < 0 ? -1 : i, best < 0 ? 0 : best);
        __syncthreads();
    }
    return clean;
}

// ---------------------------------------------------------------------
// phase 2 (opt_phase2's decisions); SN slots of 64 cover the Nn variables
// ---------------------------------------------------------------------
template <int SN, typename Re, int NW, int RW, int CS, int EX, int LW>
__device__ __forceinline__ P2Result reg_phase2(RegTab<Re, NW, RW, CS, EX, LW> &R, const RegLds<Re, NW, RW, CS, EX, LW> &L,
                                               const DevProb &P, const DevOpts &O, const DevTol &tl, OptShared &sh,
                                               RegShared<Re, NW> &ws) {
    constexpr int SM = (NW * RW + MPQP_WAVE - 1) / MPQP_WAVE;
    const int M = P.M2, K = P.K2, N2 = P.N2, Nn = P.Nn;
    const int EPS = P.n_x + P.n_t + P.n_c;
    const int wave = wave_id();
    reg_cost(R, L, M, K, (Re)-1, [&](int b) { return b == EPS; },
             [&](int col) { return L.nonb[col] == EPS ? -1.f : 0.f; });
    for (int v = threadIdx.x; v < N2; v += NW * MPQP_WAVE) L.bcnt[v] = 0;
    reg_cost_out(R, L);
    __syncthreads();
    P2Result res{ST_ITER_CAP, 0, 0, 0.0};
    for (int it = 0;; ++it) {
        int r = -1, q = -1;
        if (it < O.max_iter_p2) {
            if (wave == 0) { MPQP_PRIO_HI();
                const int lane = fresh_lane();
                Re v[SN];
                int id[SN], cn[SN];
                Re ml = (Re)INFINITY;
                bool tree = false;
#pragma unroll
                for (int s = 0; s < SN; ++s) {
                    const int var = lane + MPQP_WAVE * s;
                    v[s] = 0;
                    id[s] = var;
                    cn[s] = 0;
                    if (var < Nn) {
                        const int w = L.where[var];
                        cn[s] = L.bcnt[var];
                        v[s] = w >= 0 ? (Re)100000 : L.dl[-w - 1];
                        tree |= v[s] != v[s] || (cn[s] != 0 && (double)v[s] < -1e-10);
                        ml = v[s] < ml ? v[s] : ml;
                    }
                }
                // The counts only matter to the reference tree where they
                // differ among the improving variables: with none of them
                // chosen before, the first of the minima in its order.
                int wv;
                Re dm;
                if (!__any(tree)) {
                    dm = wave_min(ml);
                    unsigned long long hit[SN];
#pragma unroll
                    for (int s = 0; s < SN; ++s) hit[s] = __ballot(lane + MPQP_WAVE * s < Nn && v[s] == dm);
                    wv = tree_first<SN>(hit);
                } else {
                    wv = reg_tree<SN>(v, id, cn, Nn, lane, P2Pred{});
                    dm = lane_get(v[0], 0);
                }
                const double dmin = (double)dm;
                if (lane == 0) L.bcnt[wv] += 1;
                int q = -1;
                double zz = 0.0;
                if (dmin > tl.tol_minus_opt) {
                    Re zs[SM];
    #pragma unroll
                    for (int s = 0; s < SM; ++s) {
                        const int i = lane + MPQP_WAVE * s;
                        zs[s] = (i < M) ? (L.basis[i] == EPS ? (Re)-1 : (Re)0) * L.gx[i] : (Re)0;
                    }
                    zz = (double)tree_sum_s<SM, Re>(zs, M, lane);
                } else {
                    q = -L.where[wv] - 1;
                }
                if (lane == 0) {
                    sh.q = q;
                    sh.action = dmin > tl.tol_minus_opt ? ACT_STOP : ACT_PIVOT;
                    sh.z = zz;
                }
                MPQP_PRIO_LO();
            }
            __syncthreads();
            q = rfl(sh.q);
            if (rfl(sh.action) == ACT_STOP) {
                res.status = ST_OPTIMAL;
                res.z2 = rfl_d(sh.z);
            } else {
                // (q < 0 only from NaN costs: no column to enter)
                if (q >= 0) r = reg_ratio(R, L, ws, M, q, tl);
                if (r < 0) res.status = ST_UNBOUNDED;
            }
        }
        if (opaque(r) < 0) break;
        reg_pivot(R, L, r, q, [&] { reg_swap(L, r, q); });
        // (the pivot's second barrier precedes this copy of the cost row,
        // which wave 0 alone writes and reads)
        reg_cost_out(R, L);
        ++res.iters;
    }
    __syncthreads();
    res.final_set = (res.status == ST_OPTIMAL && -res.z2 > tl.final_tol) ? 1 : 0;
    return res;
}

// ---------------------------------------------------------------------
// the certificate's corrections over the staged rows
// ---------------------------------------------------------------------
// x += B32^-1 r (see cert_primal): the team of row i over its e-columns
template <typename Re, int NW, int RW, int CS, int EX, int LW>
__device__ __forceinline__ void reg_primal_corr(const RegTab<Re, NW, RW, CS, EX, LW> &R, const RegLds<Re, NW, RW, CS, EX, LW> &L,
                                                const DevProb &P, int ne) {
    const int M = P.M2, K = P.K2, e0 = P.N2 - M;
    double *x = L.cx, *r = L.cr;
    for (int h = 0; h < L.np; ++h) {
        reg_dump(R, L, K, h);
        __syncthreads();
        const int nr = min(L.rp, M - h * L.rp);
        for (int q = threadIdx.x; q < nr * MPQP_GB; q += NW * MPQP_WAVE) {
            const int li = q / MPQP_GB, g = q % MPQP_GB, i = h * L.rp + li;
            const float *Ti = L.stage + li * L.sld;
            const int bv = L.basis[i];
            double acc = (g == 0 && bv >= e0) ? r[bv - e0] : 0.0;
            int k = g;
            for (; k + (MPQP_CBL - 1) * MPQP_GB < ne; k += MPQP_CBL * MPQP_GB) {
                int rk[MPQP_CBL], sk[MPQP_CBL];
                double rv[MPQP_CBL], tv[MPQP_CBL];
#pragma unroll
                for (int u = 0; u < MPQP_CBL; ++u) {
                    rk[u] = L.elr[k + u * MPQP_GB];
                    sk[u] = L.els[k + u * MPQP_GB];
                }
#pragma unroll
                for (int u = 0; u < MPQP_CBL; ++u) {
                    rv[u] = r[rk[u]];
                    tv[u] = (double)Ti[sk[u]];
                }
#pragma unroll
                for (int u = 0; u < MPQP_CBL; ++u) acc = fma(rv[u], tv[u], acc);
            }
            for (; k < ne; k += MPQP_GB) acc = fma(r[L.elr[k]], (double)Ti[L.els[k]], acc);
            acc = team_add<MPQP_GB>(acc);
            if (g == 0) {
                const double xn = x[i] + acc;
                x[i] = xn;
                L.xv[bv] = xn == xn ? xn : INFINITY;
            }
        }
        __syncthreads();
    }
}

// y += B32^-T r (see cert_dual): the team of an e-column down the positions,
// its partial sums kept across the passes
template <typename Re, int NW, int RW, int CS, int EX, int LW>
__device__ __forceinline__ void reg_dual_corr(const RegTab<Re, NW, RW, CS, EX, LW> &R, const RegLds<Re, NW, RW, CS, EX, LW> &L,
                                              const DevProb &P, int ne) {
    constexpr int NT = NW * MPQP_WAVE;
    constexpr int NI = ((MPQP_WAVE * CS + EX) * MPQP_GT + NT - 1) / NT;
    static_assert(RW % MPQP_GT == 0, "the teams' positions start over with each pass");
    const int M = P.M2, K = P.K2, e0 = P.N2 - M;
    double *y = L.cx, *r = L.cr;
    double acc[NI];
#pragma unroll
    for (int u = 0; u < NI; ++u) acc[u] = 0.0;
    for (int h = 0; h < L.np; ++h) {
        reg_dump(R, L, K, h);
        __syncthreads();
        const int i0 = h * L.rp, nr = min(L.rp, M - i0);
#pragma unroll
        for (int u = 0; u < NI; ++u) {
            const int q = threadIdx.x + u * NT;
            if (q < ne * MPQP_GT) {
                const int k = q / MPQP_GT, g = q % MPQP_GT;
                const float *Tc = L.stage + L.els[k];
                double a = acc[u];
                int i = g;
                for (; i + (MPQP_CBL - 1) * MPQP_GT < nr; i += MPQP_CBL * MPQP_GT) {
                    double rv[MPQP_CBL], tv[MPQP_CBL];
#pragma unroll
                    for (int w = 0; w < MPQP_CBL; ++w) {
                        rv[w] = r[i0 + i + w * MPQP_GT];
                        tv[w] = (double)Tc[(i + w * MPQP_GT) * L.sld];
                    }
#pragma unroll
                    for (int w = 0; w < MPQP_CBL; ++w) a = fma(rv[w], tv[w], a);
                }
                for (; i < nr; i += MPQP_GT) a = fma(r[i0 + i], (double)Tc[i * L.sld], a);
                acc[u] = a;
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < NI; ++u) {
        const int q = threadIdx.x + u * NT;
        if (q < ne * MPQP_GT) {
            const double a = team_add<MPQP_GT>(acc[u]);
            const int rho = L.elr[q / MPQP_GT];
            if (q % MPQP_GT == 0) y[rho] = y[rho] + a;
        }
    }
    for (int i = threadIdx.x; i < M; i += NT) {
        const int bv = L.basis[i];
        if (bv >= e0) y[bv - e0] = y[bv - e0] + r[i];
    }
    __syncthreads();
}

// The phase-1 state into the store of the next level (rows of opt_ld).
template <typename Dst, typename Re, int NW, int RW, int CS, int EX, int LW>
__device__ __forceinline__ void reg_store(const RegTab<Re, NW, RW, CS, EX, LW> &R, const RegLds<Re, NW, RW, CS, EX, LW> &L, int M, int K,
                                          unsigned char *dst) {
    const int ld = opt_ld<Dst>(K), wave = wave_id(), lane = fresh_lane();
    Dst *dT = reinterpret_cast<Dst *>(dst);
    reg_for<CS>([&](auto s) MPQP_INL {
        const unsigned c = lane + MPQP_WAVE * s;
        if (c < (unsigned)K)
            reg_for<RW>([&](auto i) MPQP_INL {
                const int row = wave * RW + i;
                if (row < M) (dT + (long long)row * ld)[c] = (Dst)R.template get<decltype(i)::value, decltype(s)::value>();
            });
    });
    if (lane < RW && wave * RW + lane < M) {
        Dst *dr = dT + (long long)(wave * RW + lane) * ld;
        reg_for<EX>([&](auto e) MPQP_INL {
            if (MPQP_WAVE * CS + e < K) dr[MPQP_WAVE * CS + e] = (Dst)R.xs[e];
        });
        dr[K] = (Dst)R.x();
        dr[K + 1] = (Dst)R.xp();
    }
    int *db = reinterpret_cast<int *>(dT + (long long)opt_tw<Dst>(M, K));
    for (int i = threadIdx.x; i < M; i += NW * MPQP_WAVE) db[i] = L.basis[i];
    for (int kk = threadIdx.x; kk < K; kk += NW * MPQP_WAVE) db[M + kk] = L.nonb[kk];
}

// opt_body over a register tableau.
template <typename Re, int NW, int RW, int CS, int EX, int LW, int SN>
__device__ __forceinline__ void reg_body(const OptArgs &a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    __shared__ OptShared sh;
    __shared__ RegShared<Re, NW> ws;
    __shared__ unsigned inS[8];
    __shared__ double red[NW];
    constexpr bool MIXED = sizeof(Re) == 4;
    constexpr int NT = NW * MPQP_WAVE, SM = (NW * RW + MPQP_WAVE - 1) / MPQP_WAVE;
    const DevProb &P = a.P;
    const DevOpts &O = a.O;
    const int M = P.M2, K = P.K2, N2 = P.N2;
    const int tid = threadIdx.x;
    const int k = a.level;
    const int n = a.n_dev ? *a.n_dev : a.n;
    RegTab<Re, NW, RW, CS, EX, LW> R;
    RegLds<Re, NW, RW, CS, EX, LW> L;
    L.carve(smem, M, K, N2, a.stage_passes);
    R.lt = L.rows_lds + wave_id() * (LW * CS * MPQP_WAVE) + fresh_lane();
    const DevTol tl = MIXED ? dev_tol32(O) : dev_tol64(O);
    if (a.counter) {
        if (tid == 0) sh.item = atomicAdd(a.counter, 1);
    }
    for (int iter = 0;; ++iter) {
        int item;
        if (a.counter) {
            __syncthreads();
            item = sh.item;
        } else {
            item = iter == 0 ? (int)blockIdx.x : n;
        }
        if (item >= n) break;
        const int c = a.list[item];
        const int *Sset = a.sets + (long long)c * a.kw;
        DevRecord &Rc = a.rec[c];
#ifdef MPQP_PROFILE
        if (tid == 0) {
            sh.prof = a.prof ? a.prof + (long long)blockIdx.x * 16 : nullptr;
            sh.t0 = (long long)__builtin_amdgcn_s_memtime();
        }
#endif
        if (tid < 8) inS[tid] = 0u;
        const bool try_warm = !a.force_cold && O.warm && k > 0;
        const int par = try_warm ? a.p1parent[c] : -1;
        const int root_ok = *P.root_ok;
        const int sj = tid < k ? Sset[tid] : 0;
        __syncthreads();  // inS cleared; every thread has read sh.item
        if (a.counter && tid == 0) sh.item = atomicAdd(a.counter, 1);
        if (tid < k) atomicOr(&inS[sj >> 5], 1u << (sj & 31));
        if (root_ok == 0) {
            if (tid == 0) Rc.p1_status = ST_SINGULAR;
            continue;
        }
        P1Result p1{ST_NOT_RUN, 0, 0, 0.0};
        P2Result p2{ST_NOT_RUN, 0, 0, 0.0};
        int clean = 0, warm = par >= 0 ? 1 : 0;
        auto pcorr = [&](int ne) {
            if constexpr (MIXED) reg_primal_corr(R, L, P, ne);
        };
        auto dcorr = [&](int ne) {
            if constexpr (MIXED) reg_dual_corr(R, L, P, ne);
        };
        (void)pcorr;
        (void)dcorr;
        auto solve = [&]() MPQP_INL -> bool {
            // start: the parent's state + the lambda swap of S[k-1]; else
            // (or if that basis is singular) the root's + those of all of S
            for (;;) {
                const Re *sT;
                const int *sb, *sn;
                int sld = opt_ld<Re>(K);
                if constexpr (MIXED) {
                    sT = warm ? reinterpret_cast<const Re *>(a.ostore_prev + (long long)par * a.ostride) : P.root32;
                    sb = reinterpret_cast<const int *>(sT + (long long)opt_tw<Re>(M, K));
                    sn = sb + M;
                } else {
                    sT = warm ? reinterpret_cast<const Re *>(a.ostore_prev + (long long)par * a.ostride) : P.root;
                    sb = warm ? reinterpret_cast<const int *>(sT + (long long)opt_tw<Re>(M, K)) : P.root_basis;
                    sn = warm ? sb + M : P.root_nonb;
                    sld = warm ? sld : K + 2;
                }
                reg_load(R, L, P, sT, sld, sb, sn);
                const int ok = reg_lambda(R, L, P, tl, Sset, warm ? k - 1 : 0, k, sT, sld);
                __syncthreads();
                if (ok) break;
                if (!warm) return false;
                warm = 0;
            }
            OPT_PROF(sh, 0);
            p1 = reg_phase1(R, L, P, O, tl, sh, ws);
            OPT_PROF(sh, 3);
            if constexpr (MIXED) {
                if (!cert_phase1<NT, SM>(L, P, O, inS, red, sh, Sset, k, p1, pcorr, dcorr)) return false;
            }
            OPT_PROF(sh, 4);
            p1.kkt = rfl(p1.kkt);
            clean = reg_drive_out(R, L, P, tl, sh, p1.kkt);
            if (a.b1)
                for (int i = tid; i < M; i += NT) a.b1[(long long)c * M + i] = L.basis[i];
            if (a.store && (MIXED || p1.status == ST_OPTIMAL)) {
                unsigned char *dst = a.ostore_cur + (long long)c * a.ostride;
                if (MIXED || a.store32) reg_store<float>(R, L, M, K, dst);
                else reg_store<Re>(R, L, M, K, dst);
            }
            if (p1.kkt) {
                __syncthreads();
                OPT_PROF(sh, 5);
                p2 = reg_phase2<SN>(R, L, P, O, tl, sh, ws);
                OPT_PROF(sh, 6);
                if constexpr (MIXED) {
                    if (!cert_phase2<NT, SM>(L, P, O, inS, red, sh, Sset, k, p2, pcorr, dcorr)) return false;
                }
                if (a.b2)
                    for (int i = tid; i < M; i += NT) a.b2[(long long)c * M + i] = L.basis[i];
            }
            return true;
        };
        const bool fail = !solve();
        if (fail) {
            if constexpr (MIXED) {
                // handed to the FP64 re-solve
                if (a.b1)
                    for (int i = tid; i < M; i += NT) a.b1[(long long)c * M + i] = -1;
                if (tid == 0) {
                    Rc.repivots = 1;
                    a.fb_list[atomicAdd(a.fb_count, 1)] = c;
                }
            } else {
                if (tid == 0) Rc.p1_status = ST_SINGULAR;
            }
            continue;
        }
        if (tid == 0) opt_record(Rc, p1, p2, warm, clean);
        OPT_PROF(sh, 7);
    }
}

// EU: waves per SIMD the register budget is for (512 / EU vector registers)
template <int NW, int RW, int CS, int EX, int SN, int EU>
__global__ __launch_bounds__(NW *MPQP_WAVE) __attribute__((amdgpu_waves_per_eu(EU, EU))) void reg_kernel32(OptArgs a) {
    reg_body<float, NW, RW, CS, EX, 0, SN>(a);
}
template <int NW, int RW, int CS, int EX, int LW, int SN, int EU>
__global__ __launch_bounds__(NW *MPQP_WAVE) __attribute__((amdgpu_waves_per_eu(EU, EU))) void reg_kernel64(OptArgs a) {
    reg_body<double, NW, RW, CS, EX, LW, SN>(a);
}
