// feas_reg.hpp — the feasibility LP with its tableau in registers (the layout
// and the pivot of the FP64 LPs in reg_kernel.hpp, no perturbation column).
//
// feas_kernel keeps the tableau in LDS and decides in one wave: at n=60 m=120
// p=12 (144 x 73) its 90 KB leave one LP per CU, whose other waves wait for
// the decision.  Here every wave prices the cost row, which all of them hold,
// and the ratio test is one exchange; three LPs share a CU: 67.3 -> 24.8 ms for
// 288,101 LPs.  What bounds it now is the chain of a pivot, as in the other
// register kernels.
#pragma once

template <int NW, int RW, int CS, int EX, int EU>
__global__ __launch_bounds__(NW *MPQP_WAVE) __attribute__((amdgpu_waves_per_eu(EU, EU))) void feas_reg(FeasArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    __shared__ RegShared<double, NW> ws;
    __shared__ unsigned inS[16];
    __shared__ double sh_z;
    typedef RegTab<double, NW, RW, CS, EX, 0> Tab;
    constexpr int NT = NW * MPQP_WAVE, SM = (NW * RW + MPQP_WAVE - 1) / MPQP_WAVE, NS = Tab::NS;
    const DevProb &P = a.P;
    const DevOpts &O = a.O;
    const int M = P.M1, K = P.K1, ld = K + 1;
    const int c = blockIdx.x, tid = threadIdx.x, wave = wave_id(), lane = fresh_lane();
    const DevTol tl = dev_tol64(O);
    if (a.licq_fail && a.licq_fail[c]) {
        feas_dependent<NT>(a, c);
        return;
    }
    Tab R;
    RegLds<double, NW, RW, CS, EX, 0> L;
    L.carve(smem, M, K, M + K, 1);
    R.lt = L.rows_lds;
    const int par = a.parent[c];
    if (tid < 16) inS[tid] = 0u;
    __syncthreads();
    for (int t = tid; t < a.level; t += NT) {  // the members of S
        const int s = a.sets[(long long)c * a.kw + t];
        atomicOr(&inS[s >> 5], 1u << (s & 31));
    }
    const int row = wave * RW + lane;
    const bool valid = lane < RW && row < M;
    const bool warm = par >= 0 && O.warm;
    // the parent's rows, or A1 by columns
    const double *sT = warm ? reinterpret_cast<const double *>(a.fstore_prev + (long long)par * a.fstride) : P.A1;
    const int rs = warm ? ld : 1, cs = warm ? 1 : M;
    reg_for<RW>([&](auto i) MPQP_INL {
        const double *rp = sT + (long long)min(wave * RW + i, M - 1) * rs;
        reg_for<CS>([&](auto s) MPQP_INL {
            const int col = lane + MPQP_WAVE * s;
            R.t[i][s] = rp[(long long)(col < K ? col : 0) * cs];
        });
    });
    const double *rr = sT + (long long)(valid ? row : 0) * rs;
    reg_for<EX>([&](auto e) MPQP_INL {
        const int col = MPQP_WAVE * CS + e;
        const double v = rr[(long long)(col < K ? col : 0) * cs];
        R.xs[e] = (valid && col < K) ? v : 0.0;
    });
    const double b = warm ? rr[K] : P.xb1[valid ? row : 0];
    R.xs[EX] = valid ? b : 0.0;
    R.xs[EX + 1] = 0.0;
    if (lane < RW) L.gx[row] = R.x();
    const int *sb = reinterpret_cast<const int *>(sT + (long long)M * ld);
    for (int i = tid; i < M; i += NT) L.basis[i] = warm ? sb[i] : K + i;
    for (int k = tid; k < K; k += NT) L.nonb[k] = warm ? sb[M + k] : k;
    __syncthreads();
    auto member = [&](int var) -> bool {
        const int s = var - K;
        return s >= 0 && s < P.n_c && ((inS[s >> 5] >> (s & 31)) & 1u);
    };
    reg_cost(R, L, M, K, 1.0, member, [&](int col) { return member(L.nonb[col]) ? 1.0 : 0.0; });

    int end = 0, it = 0, status = ST_ITER_CAP;  // end: 1 optimal, 2 unbounded, 3 iteration cap
    for (;;) {
        int r = -1, aux = -1;
        if (it >= O.max_iter_feas) {
            end = 3;
        } else {
            // Dantzig pricing, lowest variable id on ties (min_idx_kernel :256-316)
            const int lane = fresh_lane();
            double dl = INFINITY;
            bool nn = false;
            reg_for<NS>([&](auto s) MPQP_INL {
                const bool in = lane + MPQP_WAVE * s < K;
                nn |= in && R.d[s] != R.d[s];
                dl = (in && R.d[s] < dl) ? R.d[s] : dl;
            });
            double dv = wave_min(dl);
            int cnt = 0;
            reg_for<NS>([&](auto s) MPQP_INL {
                const unsigned long long hit = __ballot(lane + MPQP_WAVE * s < K && R.d[s] == dv);
                cnt += __popcll(hit);
                aux = hit ? __ffsll((long long)hit) - 1 + MPQP_WAVE * s : aux;
            });
            if (__any(nn)) {
                int key = -1;
                aux = -1;
                dv = 0.0;
                reg_for<NS>([&](auto s) MPQP_INL {
                    const int kk = lane + MPQP_WAVE * s;
                    const double d = R.d[s];
                    const int var = L.nonb[kk < K ? kk : 0];
                    if (kk < K && (key < 0 || d < dv || (d == dv && var < key))) { dv = d; key = var; aux = kk; }
                });
                lex_min(dv, key, aux);
            } else if (cnt > 1) {
                unsigned key = ~0u;
                reg_for<NS>([&](auto s) MPQP_INL {
                    const int kk = lane + MPQP_WAVE * s;
                    const unsigned k = (unsigned)L.nonb[kk < K ? kk : 0] << 10 | (unsigned)kk;
                    key = (kk < K && R.d[s] == dv) ? min_r(key, k) : key;
                });
                aux = (int)(wave_min(key) & 1023u);
            }
            aux = rfl(aux);
            if (dv > O.tol_minus_1) {
                end = 1;
            } else {
                // ratio test, lowest row on ties (pivot_kernel_1_2 :901-942)
                r = reg_ratio(R, L, ws, M, aux, tl);
                if (r < 0) end = 2;
            }
        }
        if (opaque(end)) break;
        reg_pivot(R, L, r, aux, [&] {
            const int t = L.basis[r];
            L.basis[r] = L.nonb[aux];
            L.nonb[aux] = t;
        });
        ++it;
    }
    if (wave == 0) {
        double zs[SM];
#pragma unroll
        for (int s = 0; s < SM; ++s) {
            const int i = lane + MPQP_WAVE * s;
            zs[s] = i < M ? (member(L.basis[i]) ? 1.0 : 0.0) * L.gx[i] : 0.0;
        }
        const double zz = tree_sum_s<SM, double>(zs, M, lane);
        if (lane == 0) sh_z = zz;
    }
    __syncthreads();
    const double z = end == 1 ? sh_z : 0.0;
    const int feasible = rfl((end == 1 && z >= -O.feas_z_tol && z <= O.feas_z_tol) ? 1 : 0);
    status = end == 1 ? ST_OPTIMAL : (end == 2 ? ST_UNBOUNDED : ST_ITER_CAP);
    if (tid == 0) feas_record(a.rec[c], a.level, status, it, feasible, z);
    if (a.fbasis)
        for (int i = tid; i < M; i += NT) a.fbasis[(long long)c * M + i] = L.basis[i];
    if (a.store && feasible) {
        double *dT = reinterpret_cast<double *>(a.fstore_cur + (long long)c * a.fstride);
        reg_for<CS>([&](auto s) MPQP_INL {
            const int col = lane + MPQP_WAVE * s;
            if (col < K)
                reg_for<RW>([&](auto i) MPQP_INL {
                    const int ri = wave * RW + i;
                    if (ri < M) dT[(long long)ri * ld + col] = R.t[i][s];
                });
        });
        if (valid) {
            double *dr = dT + (long long)row * ld;
            reg_for<EX>([&](auto e) MPQP_INL {
                if (MPQP_WAVE * CS + e < K) dr[MPQP_WAVE * CS + e] = R.xs[e];
            });
            dr[K] = R.x();
        }
        int *db = reinterpret_cast<int *>(dT + (long long)M * ld);
        for (int i = tid; i < M; i += NT) db[i] = L.basis[i];
        for (int k = tid; k < K; k += NT) db[M + k] = L.nonb[k];
    }
}
