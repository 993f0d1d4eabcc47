// reg_kernel.hpp — the FP32 optimality LP (mixed precision) with its tableau
// in registers, pivoted by the matrix cores.
//
// One LP per workgroup of NW waves.  Wave w holds the rows w * RW ..
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

// Minimum over the wave of values that are not NaN, known to every lane:
// v_min with DPP row shifts, then the row broadcasts of lanes 15 and 31, into
// lane 63 (six dependent instructions; lane shifts with compare and select
// took four times as long).
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_min(float v) {
    const int i = __float_as_int(v);
    return fminf(v, __int_as_float(__builtin_amdgcn_update_dpp(i, i, CTRL, ROWS, 0xf, false)));
}
__device__ __forceinline__ float row8_min_f(float v) {  // into lane 7, of lanes 0 .. 7
    v = dpp_min<0x111, 0xf>(v);
    v = dpp_min<0x112, 0xf>(v);
    return dpp_min<0x114, 0xf>(v);
}
__device__ __forceinline__ float wave_min_f(float v) {
    v = row8_min_f(v);
    v = dpp_min<0x118, 0xf>(v);
    v = dpp_min<0x142, 0xa>(v);
    v = dpp_min<0x143, 0xc>(v);
    return lane_get(v, 63);
}

// The two smallest of the wave's values (not NaN; equal ones count twice),
// known to every lane, in one pass.
template <int CTRL, int ROWS>
__device__ __forceinline__ void dpp_min2(float &a, float &b) {
    const int inf = 0x7f800000;
    const float oa = __int_as_float(__builtin_amdgcn_update_dpp(inf, __float_as_int(a), CTRL, ROWS, 0xf, false));
    const float ob = __int_as_float(__builtin_amdgcn_update_dpp(inf, __float_as_int(b), CTRL, ROWS, 0xf, false));
    b = fminf(fminf(b, ob), fmaxf(a, oa));
    a = fminf(a, oa);
}
__device__ __forceinline__ void row8_min2_f(float &a, float &b) {  // into lane 7, of lanes 0 .. 7
    dpp_min2<0x111, 0xf>(a, b);
    dpp_min2<0x112, 0xf>(a, b);
    dpp_min2<0x114, 0xf>(a, b);
}
__device__ __forceinline__ void wave_min2_f(float &a, float &b) {
    row8_min2_f(a, b);
    dpp_min2<0x118, 0xf>(a, b);
    dpp_min2<0x142, 0xa>(a, b);
    dpp_min2<0x143, 0xc>(a, b);
    a = lane_get(a, 63);
    b = lane_get(b, 63);
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
template <int NW, int RW, int CS, int EX>
struct RegTab {
    static_assert(RW % 4 == 0 && RW <= MPQP_WAVE, "blocks of four rows, one lane per row");
    static constexpr int NB = RW / 4;
    static constexpr int NS = CS + (EX > 0 ? 1 : 0);  // slots of a decision
    v4f t[NB][CS];
    float d[NS];       // cost row (the same in every wave)
    float xs[EX + 2];  // by row (lanes < RW): the extra columns, the rhs, the perturbation
    __device__ __forceinline__ float x() const { return xs[EX]; }
    __device__ __forceinline__ float xp() const { return xs[EX + 1]; }
};

// Per-wave results of the distributed decisions.
struct RegMin {
    float m1, m2;  // smallest and second smallest x_B of the wave
    int at, nan;   // row of the smallest; a NaN among them
};
template <int NW>
struct RegShared {
    __attribute__((aligned(16))) RegMin min[NW];
    float cmax[NW], rv[NW];
    int rk[NW];
};

// LDS of one workgroup: the divided pivot row (with its rhs and perturbation
// entries), copies of the rhs, perturbation and one column by row, the cost
// row by column; the bookkeeping of OptLds; for certification x, r and the
// nonbasic e-list; a stage of `rp` rows for the steps that read the tableau
// against its layout (lambda swap, certification): np passes of NW / np
// waves' rows each.
__host__ __device__ inline long long reg_lds_bytes(int nw, int rw, int cs, int M, int K, int N2, bool cert, int np) {
    const long long mr = (long long)nw * rw, kc = 64LL * (cs + 1);
    long long b = (2 * kc + 3 * mr) * (long long)sizeof(float);
    b = (b + 15) & ~15LL;
    b += (3LL * N2 + 2 * M + K) * 4;
    if (cert) b = ((b + 7) & ~7LL) + 2LL * M * 8 + 2LL * (M + 1) * 4;
    b = (b + 15) & ~15LL;
    b += mr / np * (K | 1) * (long long)sizeof(float);
    return (b + 15) & ~15LL;
}

template <int NW, int RW, int CS, int EX>
struct RegLds {
    static constexpr int MR = NW * RW, KC = MPQP_WAVE * (CS + 1);
    float *ep, *gx, *gp, *colx, *dl, *stage;
    int *basis, *nonb, *where, *bcnt, *nbcnt, *rows;
    double *cx, *cr, *xv;
    int *elr, *els;
    int sld, np, rp;
    __device__ void carve(unsigned char *smem, int M, int K, int N2, bool cert, int np_) {
        np = np_;
        rp = MR / np;
        sld = K | 1;
        ep = reinterpret_cast<float *>(smem);
        gx = ep + KC;
        gp = gx + MR;
        colx = gp + MR;
        dl = colx + MR;
        size_t b = (size_t)(2 * KC + 3 * MR) * sizeof(float);
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
        if (cert) {
            b = (b + 7) & ~(size_t)7;
            cx = reinterpret_cast<double *>(smem + b);
            cr = cx + M;
            elr = reinterpret_cast<int *>(cr + M);
            els = elr + M + 1;
            b += (size_t)2 * M * 8 + (size_t)2 * (M + 1) * 4;
        }
        b = (b + 15) & ~(size_t)15;
        stage = reinterpret_cast<float *>(smem + b);
    }
    __device__ __forceinline__ float rhs_of(int i) const { return gx[i]; }
    __device__ __forceinline__ float cost_of(int k) const { return dl[k]; }
};

__device__ __forceinline__ int wave_id() { return rfl((int)(threadIdx.x / MPQP_WAVE)); }

// The wave's rows into the stage, pass h (waves [h, h + 1) * NW / np); the
// caller's barriers surround it.
template <int NW, int RW, int CS, int EX>
__device__ __forceinline__ void reg_dump(const RegTab<NW, RW, CS, EX> &R, const RegLds<NW, RW, CS, EX> &L, int K, int h) {
    const int wave = wave_id(), lane = fresh_lane();
    const int w0 = h * (NW / L.np);
    if (wave >= w0 && wave < w0 + NW / L.np) {
        float *dst = L.stage + (wave - w0) * RW * L.sld;
        reg_for<CS>([&](auto s) MPQP_INL {
            const int c = lane + MPQP_WAVE * s;
            if (c < K) {
                float *dc = dst + c;
                reg_for<RW>([&](auto i) MPQP_INL {
                    *dc = R.t[i / 4][s][i % 4];
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
__device__ __forceinline__ void reg_rank1(RegTab<NW, RW, CS, EX> &R, float nf, float v) {
    reg_for<RW / 4>([&](auto b) MPQP_INL {
        R.t[b][S] = __builtin_amdgcn_mfma_f32_4x4x1f32(nf, v, R.t[b][S], 4, decltype(b)::value, 0);
    });
}

// Column q of the wave's rows by lane, through the wave's part of L.colx (a
// wave's LDS operations stay in order).  CLEAR: the column is left zero
// (T - f * 1 in its lane), if `on`.
template <bool CLEAR, int NW, int RW, int CS, int EX, typename RT>
__device__ __forceinline__ float reg_col_op(RT &R, const RegLds<NW, RW, CS, EX> &L, int q, bool on) {
    const int lane = fresh_lane(), lq = q % MPQP_WAVE;
    float *cx = L.colx + wave_id() * RW;
    float v = 0.f;
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
template <int NW, int RW, int CS, int EX>
__device__ __forceinline__ float reg_col(const RegTab<NW, RW, CS, EX> &R, const RegLds<NW, RW, CS, EX> &L, int q) {
    return reg_col_op<false>(R, L, q, false);
}

// Row `lr` of the wave; al[CS]: its extra columns, rhs and perturbation entry
// in the first lanes.
template <int NW, int RW, int CS, int EX>
__device__ __forceinline__ void reg_row(const RegTab<NW, RW, CS, EX> &R, int lr, float (&al)[CS + 1]) {
    const int u = lr % 4;
    reg_pick<0, RW / 4>(lr / 4, [&](auto b) MPQP_INL {
        reg_for<CS>([&](auto s) MPQP_INL {
            const v4f v = R.t[b][s];
            al[s] = u < 2 ? (u == 0 ? v[0] : v[1]) : (u == 2 ? v[2] : v[3]);
        });
    });
    const int lane = fresh_lane();
    al[CS] = 0.f;
    reg_for<EX + 2>([&](auto e) MPQP_INL { al[CS] = lane == e ? lane_get(R.xs[e], lr) : al[CS]; });
}

// Row `lr` of the wave (its entries al) made zero: T - 1 * al.
template <int NW, int RW, int CS, int EX>
__device__ __forceinline__ void reg_clear_row(RegTab<NW, RW, CS, EX> &R, int lr, const float (&al)[CS + 1]) {
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

// The pivot row's wave: row lr (al) divided by p into L.ep (1 / p at column
// q, if any), with its rhs and perturbation entries; the row itself is left
// zero for reg_apply.
template <int NW, int RW, int CS, int EX>
__device__ __forceinline__ void reg_divide(RegTab<NW, RW, CS, EX> &R, const RegLds<NW, RW, CS, EX> &L, const float (&al)[CS + 1],
                                           int lr, int q, float p) {
    const int lane = fresh_lane();
    reg_for<CS + 1>([&](auto s) MPQP_INL {
        const int c = lane + MPQP_WAVE * s;
        L.ep[c] = (c == q ? 1.f : al[s]) / p;
    });
    reg_clear_row(R, lr, al);
}

template <int NW, int RW, int CS, int EX>
__device__ __forceinline__ void reg_publish(RegTab<NW, RW, CS, EX> &R, const RegLds<NW, RW, CS, EX> &L, const float (&al)[CS + 1],
                                            int lr, int q) {
    float v = al[0];
    reg_for<RegTab<NW, RW, CS, EX>::NS>([&](auto s) MPQP_INL { v = q / MPQP_WAVE == s ? al[s] : v; });
    reg_divide(R, L, al, lr, q, lane_get(v, q % MPQP_WAVE));
}

// The rank-1 update of the wave's rows by the divided pivot row pr (pr[CS]:
// extra columns, rhs, perturbation) with the factors fv by lane.  The wave
// that holds the pivot row r finds it zero: its factor -1 puts pr there.
template <int NW, int RW, int CS, int EX>
__device__ __forceinline__ void reg_apply(RegTab<NW, RW, CS, EX> &R, const RegLds<NW, RW, CS, EX> &L,
                                          const float (&pr)[CS + 1], float fv, int r) {
    const int lane = fresh_lane(), wave = wave_id(), lr = r - wave * RW;
    const float nf = lane == lr ? 1.f : -fv;
    reg_for<CS>([&](auto s) MPQP_INL { reg_rank1<decltype(s)::value>(R, nf, pr[s]); });
    reg_for<EX + 2>([&](auto e) MPQP_INL { R.xs[e] = fma(nf, lane_get(pr[CS], e), lane == lr ? 0.f : R.xs[e]); });
    if (lane < RW) {
        L.gx[wave * RW + lane] = R.x();
        L.gp[wave * RW + lane] = R.xp();
    }
}

// The pivot on (r, q) from the divided row in L.ep, by every wave, cost row
// included.  Barriers before (L.ep written) and after belong to the caller.
// MAYBE: r < 0 leaves everything as it is (a branch around the update would
// give the tableau's registers two states to be merged).
template <bool MAYBE = false, int NW, int RW, int CS, int EX>
__device__ __forceinline__ void reg_update(RegTab<NW, RW, CS, EX> &R, const RegLds<NW, RW, CS, EX> &L, int r, int q) {
    const int lane = fresh_lane();
    const bool off = MAYBE && r < 0;
    float fv = reg_col_op<true>(R, L, q, !off);
    float pr[CS + 1], dv = 0.f;
    reg_for<CS + 1>([&](auto s) MPQP_INL {
        pr[s] = L.ep[lane + MPQP_WAVE * s];
        if constexpr (MAYBE) pr[s] = off ? 0.f : pr[s];
    });
    if constexpr (MAYBE) fv = off ? 0.f : fv;
    constexpr int NS = RegTab<NW, RW, CS, EX>::NS;
    reg_for<NS>([&](auto s) MPQP_INL { dv = q / MPQP_WAVE == s ? R.d[s] : dv; });
    const float fd = lane_get(dv, q % MPQP_WAVE);
    reg_for<NS>([&](auto s) MPQP_INL {
        const float d0 = lane + MPQP_WAVE * s == q && !off ? 0.f : R.d[s];
        R.d[s] = pr[s] != 0.f ? fma(-fd, pr[s], d0) : d0;
    });
    reg_apply(R, L, pr, fv, off ? -MPQP_WAVE * NW : r);
}

// Cost row d = init(column) - c * (sum of the rows whose basic variable
// satisfies sel), rows ascending: the waves that hold such rows continue the
// chain one after the other through L.dl.
template <int NW, int RW, int CS, int EX, typename SelF, typename InitF>
__device__ __forceinline__ void reg_cost(RegTab<NW, RW, CS, EX> &R, const RegLds<NW, RW, CS, EX> &L, int M, int K,
                                         float c, SelF sel, InitF init) {
    constexpr int NS = RegTab<NW, RW, CS, EX>::NS;
    const int lane = fresh_lane(), wave = wave_id();
    reg_for<NS>([&](auto s) MPQP_INL {
        const int col = lane + MPQP_WAVE * s;
        R.d[s] = col < K ? init(col) : 0.f;
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
                    reg_for<CS>([&](auto s) MPQP_INL { R.d[s] = fma(-c, R.t[i / 4][s][i % 4], R.d[s]); });
                    if constexpr (EX > 0) {
                        float v = 0.f;
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
template <int NW, int RW, int CS, int EX>
__device__ __forceinline__ void reg_cost_out(const RegTab<NW, RW, CS, EX> &R, const RegLds<NW, RW, CS, EX> &L) {
    if (wave_id() == 0) {
        const int lane = fresh_lane();
        reg_for<RegTab<NW, RW, CS, EX>::NS>([&](auto s) MPQP_INL { L.dl[lane + MPQP_WAVE * s] = R.d[s]; });
    }
}

// The wave's two smallest basic values (perturbed: x + xp) for the choice of
// the leaving row.
template <int NW, int RW, int CS, int EX>
__device__ __forceinline__ void reg_min_out(const RegTab<NW, RW, CS, EX> &R, RegShared<NW> &ws, int M,
                                            bool pert) {
    const int lane = fresh_lane(), wave = wave_id();
    const bool valid = lane < RW && wave * RW + lane < M;
    const float x = pert ? R.x() + R.xp() : R.x();
    const bool nan = valid && x != x;
    const float v = (valid && !nan) ? x : INFINITY;
    float m1 = v, m2 = INFINITY;
    wave_min2_f(m1, m2);
    const int f = __ffsll((long long)__ballot(v == m1)) - 1;
    const int an = __any(nan) ? 1 : 0;
    if (lane == 0) {
        ws.min[wave] = RegMin{m1, m2, wave * RW + f, an};
    }
}

// primal_ratio_wave over the register tableau, by the whole workgroup: every
// wave returns the row.  Two barriers.
template <int NW, int RW, int CS, int EX>
__device__ __forceinline__ int reg_ratio(const RegTab<NW, RW, CS, EX> &R, const RegLds<NW, RW, CS, EX> &L, RegShared<NW> &ws,
                                         int M, int q, const DevTol &tl) {
    const int lane = fresh_lane(), wave = wave_id();
    const bool valid = lane < RW && wave * RW + lane < M;
    const float a = reg_col(R, L, q);
    float lim = (float)tl.tol_plus;
    if (tl.pivot_rel > 0.0) {
        const float fa = fabsf(a);
        const float cw = -wave_min_f((valid && fa > 0.f) ? -fa : 0.f);
        if (lane == 0) ws.cmax[wave] = cw;
        __syncthreads();
        const float cm = -lane_get(row8_min_f(-ws.cmax[lane % NW]), 7);
        const float rl = (float)tl.pivot_rel * cm;
        lim = rl > lim ? rl : lim;
    }
    // the wave's smallest ratio, its lowest row
    const bool take = valid && a > lim;
    const float rt = take ? R.x() / a : 0.f;
    const bool num = take && rt == rt;
    const float m = wave_min_f(num ? rt : INFINITY);
    const unsigned long long hit = __ballot(num && rt == m), any = __ballot(take);
    const int f = __ffsll((long long)(hit ? hit : any)) - 1;
    if (lane == 0) {
        ws.rv[wave] = m;
        ws.rk[wave] = f < 0 ? -1 : wave * RW + f;
    }
    __syncthreads();
    const int k = ws.rk[lane % NW];
    const float v = k >= 0 ? ws.rv[lane % NW] : INFINITY;
    const float mm = lane_get(row8_min_f(v), 7);
    const unsigned long long has = __ballot(lane < NW && k >= 0), best = __ballot(lane < NW && k >= 0 && v == mm);
    const int w = __ffsll((long long)(best ? best : has)) - 1;
    return w < 0 ? -1 : __builtin_amdgcn_readlane(k, w);
}

// A pivot on (r, q) that every wave knows: the row's wave divides and
// publishes it, every wave updates; `between` is run by one thread while the
// update runs (the basis bookkeeping).  Two barriers.
template <int NW, int RW, int CS, int EX, typename F>
__device__ __forceinline__ void reg_pivot(RegTab<NW, RW, CS, EX> &R, const RegLds<NW, RW, CS, EX> &L, int r, int q,
                                          F between) {
    const int wave = wave_id(), lr = r - wave * RW;
    if ((unsigned)lr < (unsigned)RW) {
        float al[CS + 1];
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
template <int NW, int RW, int CS, int EX, typename Src>
__device__ __forceinline__ void reg_load(RegTab<NW, RW, CS, EX> &R, const RegLds<NW, RW, CS, EX> &L,
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
        reg_for<CS>([&](auto s) MPQP_INL { R.t[i / 4][s][i % 4] = (float)rp[cc[s]]; });
    });
    const int row = wave * RW + lane;
    const bool valid = lane < RW && row < M;
    const Src *rr = sT + (long long)(valid ? row : 0) * src_ld;
    reg_for<EX>([&](auto e) MPQP_INL {
        const int c = MPQP_WAVE * CS + e;
        R.xs[e] = (valid && c < K) ? (float)rr[c] : 0.f;
    });
    R.xs[EX] = valid ? (float)rr[K] : 0.f;
    R.xs[EX + 1] = valid ? (float)rr[K + 1] : 0.f;
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

// opt_lambda: the lambda swaps of S[j0 .. j1); the rows are staged in LDS so
// that a thread can walk its row's e-columns in the order of the terms.
template <int NW, int RW, int CS, int EX>
__device__ __forceinline__ int reg_lambda(RegTab<NW, RW, CS, EX> &R, const RegLds<NW, RW, CS, EX> &L,
                                          const DevProb &P, const DevTol &tl, const int *Sset, int j0, int j1) {
    const int M = P.M2, K = P.K2, N2 = P.N2;
    const int r4 = M - P.n_c - P.n_x, nt = P.n_x + 1;
    const int tid = threadIdx.x;
    float *lam = L.ep;
    int *wl = L.bcnt;
    for (int jj = j0; jj < j1; ++jj) {
        const int j = Sset[jj];
        for (int t = tid; t < nt; t += NW * MPQP_WAVE) {
            const int rho = t == 0 ? j : r4 + t - 1;
            lam[t] = (float)lam_entry(P, j, rho);
            wl[t] = L.where[N2 - M + rho];
        }
        for (int h = 0; h < L.np; ++h) {
            reg_dump(R, L, K, h);
            __syncthreads();
            for (int i = tid; i < L.rp && h * L.rp + i < M; i += NW * MPQP_WAVE) {
                const int row = h * L.rp + i;
                const float *Ti = L.stage + i * L.sld;
                // terms in ascending t, zeros skipped; loads of 4 in flight
                float acc = 0.f;
                for (int t0 = 0; t0 < nt; t0 += 4) {
                    float av[4], tv[4];
                    int w[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const int t = t0 + u < nt ? t0 + u : nt - 1;
                        av[u] = t0 + u < nt ? lam[t] : 0.f;
                        w[u] = wl[t];
                    }
#pragma unroll
                    for (int u = 0; u < 4; ++u) tv[u] = Ti[w[u] >= 0 ? 0 : -w[u] - 1];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const float f1 = fma(av[u], 1.f, acc);
                        const float f2 = fma(av[u], tv[u], acc);
                        const float na = w[u] >= 0 ? (row == w[u] ? f1 : acc) : f2;
                        acc = av[u] == 0.f ? acc : na;
                    }
                }
                L.colx[row] = acc;
            }
            __syncthreads();
        }
        const int p = rfl(L.where[P.n_x + P.n_t + j]);
        const int lane = fresh_lane(), wave = wave_id();
        const int row = wave * RW + lane;
        const float fv = (lane < RW && row < M) ? L.colx[row] : 0.f;
        // w_j basic at position p: a pivot on row p with the column vcol held
        // outside the tableau; w_j nonbasic in column kk: the column
        // replaced (T - column * 1, then + vcol * 1, in its lane)
        const float pv = lane_get(L.colx[p >= 0 ? p : 0], 0);
        if (p >= 0 && !(fabs((double)pv) > tl.licq)) return 0;
        const int kk = p >= 0 ? -1 : -p - 1, lr = p - wave * RW;
        if (p >= 0 && (unsigned)lr < (unsigned)RW) {
            float al[CS + 1];
            reg_row(R, lr, al);
            reg_divide(R, L, al, lr, -1, pv);
        }
        __syncthreads();
        reg_col_op<true>(R, L, kk < 0 ? 0 : kk, kk >= 0);
        float pr[CS + 1];
        reg_for<CS + 1>([&](auto s) MPQP_INL {
            const int col = lane + MPQP_WAVE * s;
            pr[s] = kk < 0 ? L.ep[col] : (col == kk ? 1.f : 0.f);
        });
        reg_apply(R, L, pr, kk < 0 ? fv : -fv, kk < 0 ? p : -MPQP_WAVE * NW);
        __syncthreads();
    }
    return 1;
}

// ---------------------------------------------------------------------
// phase 1 (opt_phase1's decisions)
// ---------------------------------------------------------------------
template <int NW, int RW, int CS, int EX>
__device__ __forceinline__ P1Result reg_phase1(RegTab<NW, RW, CS, EX> &R, const RegLds<NW, RW, CS, EX> &L,
                                               const DevProb &P, const DevOpts &O, const DevTol &tl, OptShared &sh,
                                               RegShared<NW> &ws) {
    constexpr int SM = (NW * RW + MPQP_WAVE - 1) / MPQP_WAVE, NS = RegTab<NW, RW, CS, EX>::NS;
    const int M = P.M2, K = P.K2, N2 = P.N2, Nn = P.Nn;
    const int wave = wave_id();
    reg_cost(R, L, M, K, 1.f, [&](int b) { return b >= Nn; },
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
    reg_min_out(R, ws, M, n_same >= O.stall_perturb);
    __syncthreads();
    // One exit and one way back, so that the tableau has one place: what
    // ends the loop is noted and acted on before the update.
    bool stall = false;
    for (;;) {
        int r = -1, q = -1, act = ACT_PIVOT;
        bool pert = false;
        for (;;) {
            if (stall) { act = ACT_STOP; res.status = ST_STALL; break; }
            if (it >= O.max_iter_p1) { act = ACT_STOP; break; }
            pert = !no_pert && n_same >= O.stall_perturb;
            const int lane = fresh_lane();
            // Leaving row, by every wave: a unique minimum (no NaN, no other
            // value within the tree's 1e-10 band, no counter preference) wins
            // every combine of the reference tree; anything else runs the tree.
            const RegMin w = ws.min[lane % NW];
            float m = lane < NW ? w.m1 : INFINITY, m2 = lane < NW ? w.m2 : INFINITY;
            row8_min2_f(m, m2);
            m = lane_get(m, 7);
            m2 = lane_get(m2, 7);
            const int f = __ffsll((long long)__ballot(w.m1 == m)) - 1;
            r = __builtin_amdgcn_readlane(w.at, f);
            const bool tie = m2 == m || (double)m > (double)m2 - 1e-10;
            const bool go_on = (double)m < tl.dual_stop_tol;
            const int mode_b = (n_same % 20) >= 10 ? 1 : 0;
            if (rfl((mode_b || tie || __any(w.nan)) ? 1 : 0)) {
                float v[SM];
                int pk[SM];
#pragma unroll
                for (int s = 0; s < SM; ++s) {
                    const int i = lane + MPQP_WAVE * s;
                    const bool valid = i < M;
                    const int ic = valid ? i : 0;
                    const float x0 = L.gx[ic], xp = L.gp[ic];
                    v[s] = valid ? (pert ? x0 + xp : x0) : 0.f;
                    pk[s] = L.bcnt[L.basis[ic]] << 10 | ic;
                }
                const DminPred pred{mode_b, tl.dual_stop_tol};
                r = tree32<SM>(v, pk, M, lane, [&](float vt, int pt, float vu, int pu) {
                    return pred((double)vt, 0, pt >> 10, (double)vu, 0, pu >> 10);
                }) & 1023;
            }
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
                float al[CS + 1];
                reg_row(R, lr, al);
                float dlim = (float)tl.tol_minus;
                if (tl.pivot_rel > 0.0) {
                    float am = 0.f;
                    reg_for<NS>([&](auto s) MPQP_INL {
                        const float a = lane + MPQP_WAVE * s < K ? fabsf(al[s]) : 0.f;
                        am = a > am ? a : am;
                    });
                    const float rl = -(float)tl.pivot_rel * -wave_min_f(-am);
                    dlim = rl < dlim ? rl : dlim;
                }
                const int mode = n_same < 10 ? 0 : (n_same < 100 ? 1 : 2);
                float v[NS];
                bool tk[NS];
                float ml = INFINITY;
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
                    const float m = wave_min_f(ml);
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
                        int pk[NS];
                        reg_for<NS>([&](auto s) MPQP_INL {
                            const bool h = tk[s] && v[s] == m;
                            pk[s] = h ? cnt_of[s] << 10 | (lane + MPQP_WAVE * s) : -1;
                        });
                        qk = tree32<NS>(v, pk, K, lane, [](float, int pt, float, int pu) {
                            return (pu >= 0) & ((pt < 0) | ((pt >> 10) > (pu >> 10) + 2));
                        }) & 1023;
                    }
                }
                if (qk == -2) {
                    int pk[NS];
                    reg_for<NS>([&](auto s) MPQP_INL {
                        pk[s] = tk[s] ? cnt_of[s] << 10 | (lane + MPQP_WAVE * s) : -1;
                        v[s] = tk[s] ? v[s] : 100000.f;
                    });
                    const DratioPred pred{mode};
                    const int w = tree32<NS>(v, pk, K, lane, [&](float vt, int pt, float vu, int pu) {
                        return pred((double)vt, pt, pt >> 10, (double)vu, pu, pu >> 10);
                    });
                    qk = w < 0 ? -1 : w & 1023;
                }
                qk = rfl(qk);
                if (qk >= 0) reg_publish(R, L, al, lr, qk);
                if (lane == 0) sh.q = qk;
                MPQP_PRIO_LO();
            }
            if (wave == (wo + 1) % NW) {
                // meanwhile: the sum of the negative x_B for the stall counter
                float ps[SM];
    #pragma unroll
                for (int s = 0; s < SM; ++s) {
                    const int i = lane + MPQP_WAVE * s;
                    const int ic = i < M ? i : 0;
                    const float x0 = L.gx[ic], xp = L.gp[ic];
                    const float x = (pert && i < M) ? x0 + xp : x0;
                    ps[s] = (i < M && x < 0.f) ? x : 0.f;
                }
                tree_sum_lane0<SM, float>(ps, M, lane);
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
        // the bookkeeping's reads pass while the tableau is updated
        int bv = 0, nv = 0, bc = 0, nc = 0;
        if (wave == NW - 1) {
            bv = L.basis[r];
            nv = L.nonb[q];
            bc = L.bcnt[bv];
            nc = L.nbcnt[nv];
        }
        reg_update(R, L, r, q);
        if (threadIdx.x == (NW - 1) * MPQP_WAVE) {
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
            float dl = INFINITY;
            bool nn = false;
            reg_for<NS>([&](auto s) MPQP_INL {
                const bool in = lane + MPQP_WAVE * s < K;
                nn |= in && R.d[s] != R.d[s];
                dl = (in && R.d[s] < dl) ? R.d[s] : dl;
            });
            const float dm = wave_min_f(dl);
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
        float zs[SM];
#pragma unroll
        for (int s = 0; s < SM; ++s) {
            const int i = lane + MPQP_WAVE * s;
            zs[s] = (i < M) ? (L.basis[i] >= Nn ? 1.f : 0.f) * L.gx[i] : 0.f;
        }
        const double zz = (double)tree_sum_s<SM, float>(zs, M, lane);
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
template <int NW, int RW, int CS, int EX>
__device__ __forceinline__ int reg_drive_out(RegTab<NW, RW, CS, EX> &R, const RegLds<NW, RW, CS, EX> &L, const DevProb &P,
                                             const DevTol &tl, OptShared &sh, int on) {
    constexpr int SM = (NW * RW + MPQP_WAVE - 1) / MPQP_WAVE, NS = RegTab<NW, RW, CS, EX>::NS;
    const int M = P.M2, K = P.K2, Nn = P.Nn;
    rows_where<SM>(L.rows, M, sh, [&](int i) { return L.basis[i] >= Nn; });
    const int n = on ? rfl(sh.nrows) : 0, wave = wave_id();
    int clean = 1;
    for (int t = 0; t < n; ++t) {
        const int i = rfl(L.rows[t]), lr = i - wave * RW;
        if ((unsigned)lr < (unsigned)RW) {
            const int lane = fresh_lane();
            float al[CS + 1];
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
template <int SN, int NW, int RW, int CS, int EX>
__device__ __forceinline__ P2Result reg_phase2(RegTab<NW, RW, CS, EX> &R, const RegLds<NW, RW, CS, EX> &L,
                                               const DevProb &P, const DevOpts &O, const DevTol &tl, OptShared &sh,
                                               RegShared<NW> &ws) {
    constexpr int SM = (NW * RW + MPQP_WAVE - 1) / MPQP_WAVE;
    const int M = P.M2, K = P.K2, N2 = P.N2, Nn = P.Nn;
    const int EPS = P.n_x + P.n_t + P.n_c;
    const int wave = wave_id();
    reg_cost(R, L, M, K, -1.f, [&](int b) { return b == EPS; },
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
                float v[SN];
                int pk[SN];
                float ml = INFINITY;
                bool tree = false;
#pragma unroll
                for (int s = 0; s < SN; ++s) {
                    const int var = lane + MPQP_WAVE * s;
                    v[s] = 0.f;
                    pk[s] = var;
                    if (var < Nn) {
                        const int w = L.where[var], cn = L.bcnt[var];
                        v[s] = w >= 0 ? 100000.f : L.dl[-w - 1];
                        pk[s] = cn << 10 | var;
                        tree |= v[s] != v[s] || (cn != 0 && (double)v[s] < -1e-10);
                        ml = v[s] < ml ? v[s] : ml;
                    }
                }
                // The counts only matter to the reference tree where they
                // differ among the improving variables: with none of them
                // chosen before, the first of the minima in its order.
                int wv;
                float dm;
                if (!__any(tree)) {
                    dm = wave_min_f(ml);
                    unsigned long long hit[SN];
#pragma unroll
                    for (int s = 0; s < SN; ++s) hit[s] = __ballot(lane + MPQP_WAVE * s < Nn && v[s] == dm);
                    wv = tree_first<SN>(hit);
                } else {
                    wv = tree32<SN>(v, pk, Nn, lane, [](float vt, int pt, float vu, int pu) {
                        return P2Pred{}((double)vt, 0, pt >> 10, (double)vu, 0, pu >> 10);
                    }) & 1023;
                    dm = lane_get(v[0], 0);
                }
                const double dmin = (double)dm;
                if (lane == 0) L.bcnt[wv] += 1;
                int q = -1;
                double zz = 0.0;
                if (dmin > tl.tol_minus_opt) {
                    float zs[SM];
    #pragma unroll
                    for (int s = 0; s < SM; ++s) {
                        const int i = lane + MPQP_WAVE * s;
                        zs[s] = (i < M) ? (L.basis[i] == EPS ? -1.f : 0.f) * L.gx[i] : 0.f;
                    }
                    zz = (double)tree_sum_s<SM, float>(zs, M, lane);
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
template <int NW, int RW, int CS, int EX>
__device__ __forceinline__ void reg_primal_corr(const RegTab<NW, RW, CS, EX> &R, const RegLds<NW, RW, CS, EX> &L,
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
template <int NW, int RW, int CS, int EX>
__device__ __forceinline__ void reg_dual_corr(const RegTab<NW, RW, CS, EX> &R, const RegLds<NW, RW, CS, EX> &L,
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
template <int NW, int RW, int CS, int EX>
__device__ __forceinline__ void reg_store(const RegTab<NW, RW, CS, EX> &R, const RegLds<NW, RW, CS, EX> &L, int M, int K,
                                          unsigned char *dst) {
    const int ld = opt_ld<float>(K), wave = wave_id(), lane = fresh_lane();
    float *dT = reinterpret_cast<float *>(dst);
    reg_for<CS>([&](auto s) MPQP_INL {
        const unsigned c = lane + MPQP_WAVE * s;
        if (c < (unsigned)K)
            reg_for<RW>([&](auto i) MPQP_INL {
                const int row = wave * RW + i;
                if (row < M) (dT + (long long)row * ld)[c] = R.t[i / 4][s][i % 4];
            });
    });
    if (lane < RW && wave * RW + lane < M) {
        float *dr = dT + (long long)(wave * RW + lane) * ld;
        reg_for<EX>([&](auto e) MPQP_INL {
            if (MPQP_WAVE * CS + e < K) dr[MPQP_WAVE * CS + e] = R.xs[e];
        });
        dr[K] = R.x();
        dr[K + 1] = R.xp();
    }
    int *db = reinterpret_cast<int *>(dT + (long long)opt_tw<float>(M, K));
    for (int i = threadIdx.x; i < M; i += NW * MPQP_WAVE) db[i] = L.basis[i];
    for (int kk = threadIdx.x; kk < K; kk += NW * MPQP_WAVE) db[M + kk] = L.nonb[kk];
}

// The FP32 opt_body over a register tableau.
template <int NW, int RW, int CS, int EX, int SN>
__device__ __forceinline__ void reg_body(const OptArgs &a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    __shared__ OptShared sh;
    __shared__ RegShared<NW> ws;
    __shared__ unsigned inS[8];
    __shared__ double red[NW];
    constexpr int NT = NW * MPQP_WAVE, SM = (NW * RW + MPQP_WAVE - 1) / MPQP_WAVE;
    const DevProb &P = a.P;
    const DevOpts &O = a.O;
    const int M = P.M2, K = P.K2, N2 = P.N2;
    const int tid = threadIdx.x;
    const int k = a.level;
    const int n = a.n_dev ? *a.n_dev : a.n;
    RegTab<NW, RW, CS, EX> R;
    RegLds<NW, RW, CS, EX> L;
    L.carve(smem, M, K, N2, true, a.stage_passes);
    const DevTol tl = dev_tol32(O);
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
        auto pcorr = [&](int ne) { reg_primal_corr(R, L, P, ne); };
        auto dcorr = [&](int ne) { reg_dual_corr(R, L, P, ne); };
        auto solve = [&]() MPQP_INL -> bool {
            // start: the parent's state + the lambda swap of S[k-1]; else
            // (or if that basis is singular) the root's + those of all of S
            for (;;) {
                const float *sT = warm ? reinterpret_cast<const float *>(a.ostore_prev + (long long)par * a.ostride)
                                       : P.root32;
                const int *sb = reinterpret_cast<const int *>(sT + (long long)opt_tw<float>(M, K));
                reg_load(R, L, P, sT, opt_ld<float>(K), sb, sb + M);
                const int ok = reg_lambda(R, L, P, tl, Sset, warm ? k - 1 : 0, k);
                __syncthreads();
                if (ok) break;
                if (!warm) return false;
                warm = 0;
            }
            OPT_PROF(sh, 0);
            p1 = reg_phase1(R, L, P, O, tl, sh, ws);
            OPT_PROF(sh, 3);
            if (!cert_phase1<NT, SM>(L, P, O, inS, red, sh, Sset, k, p1, pcorr, dcorr)) return false;
            OPT_PROF(sh, 4);
            p1.kkt = rfl(p1.kkt);
            clean = reg_drive_out(R, L, P, tl, sh, p1.kkt);
            if (a.b1)
                for (int i = tid; i < M; i += NT) a.b1[(long long)c * M + i] = L.basis[i];
            if (a.store) reg_store(R, L, M, K, a.ostore_cur + (long long)c * a.ostride);
            if (p1.kkt) {
                __syncthreads();
                OPT_PROF(sh, 5);
                p2 = reg_phase2<SN>(R, L, P, O, tl, sh, ws);
                OPT_PROF(sh, 6);
                if (!cert_phase2<NT, SM>(L, P, O, inS, red, sh, Sset, k, p2, pcorr, dcorr)) return false;
                if (a.b2)
                    for (int i = tid; i < M; i += NT) a.b2[(long long)c * M + i] = L.basis[i];
            }
            return true;
        };
        const bool fail = !solve();
        if (fail) {
            if (a.b1)
                for (int i = tid; i < M; i += NT) a.b1[(long long)c * M + i] = -1;
            if (tid == 0) {
                Rc.repivots = 1;
                a.fb_list[atomicAdd(a.fb_count, 1)] = c;
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
    reg_body<NW, RW, CS, EX, SN>(a);
}
