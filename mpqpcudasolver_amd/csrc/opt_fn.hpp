// opt_fn.hpp — the optimality kernels by shape.  Their instantiations are most
// of the build, so each group is a translation unit of its own (opt_fn.hip
// compiled with MPQP_PART = its number), compiled side by side.
#pragma once

// Groups: threads per workgroup, FP32 pivots with certification or FP64, the
// tableau in LDS or split between LDS and global memory; S the slots of a
// reduction.
#define MPQP_OPT_PARTS(X)          \
    X(0, 256, true, false)         \
    X(1, 512, true, false)         \
    X(2, 512, true, true)          \
    X(3, 1024, true, true)         \
    X(4, 256, false, false)        \
    X(5, 512, false, false)        \
    X(6, 512, false, true)         \
    X(7, 1024, false, true)

#define MPQP_DECL(part, nt, fp32, gt) __attribute__((visibility("hidden"))) const void *opt_fn_part##part(int S);
MPQP_OPT_PARTS(MPQP_DECL)
#undef MPQP_DECL

// Kernels with the tableau in registers (parts 8 ..): FP32 or FP64, waves per
// workgroup, rows per wave, of these in LDS (FP64), column slots, extra
// columns, reduction slots over the Nn variables, waves per SIMD of the
// register budget (512 / that many registers a lane).
#define MPQP_REG_PARTS(X)                  \
    X(8, true, 2, 44, 0, 1, 4, 3, 4)       \
    X(9, true, 2, 64, 0, 1, 8, 4, 3)       \
    X(10, true, 4, 44, 0, 2, 0, 4, 3)      \
    X(11, true, 4, 64, 0, 2, 8, 6, 2)      \
    X(12, true, 8, 44, 0, 3, 4, 6, 2)      \
    X(13, true, 8, 44, 0, 4, 0, 6, 2)      \
    X(14, false, 2, 24, 0, 1, 0, 3, 4)     \
    X(15, false, 2, 40, 0, 1, 0, 3, 3)     \
    X(16, false, 4, 32, 0, 1, 8, 4, 3)     \
    X(17, false, 4, 44, 0, 2, 0, 4, 2)     \
    X(18, false, 8, 32, 0, 2, 8, 6, 2)     \
    X(19, false, 8, 42, 11, 3, 4, 6, 2)

// Feasibility LPs with the tableau in registers (parts 20 ..): waves, rows
// per wave, column slots, extra columns, waves per SIMD.
#define MPQP_FEAS_PARTS(X)   \
    X(20, 4, 32, 1, 0, 4)    \
    X(21, 4, 40, 1, 12, 3)   \
    X(22, 4, 40, 2, 0, 2)

struct FeasConfig {
    int nw, rw, cs, ex, eu;
    void (*fn)(FeasArgs);
    int rows() const { return nw * rw; }
    int columns() const { return 64 * cs + ex; }
    int threads() const { return nw * 64; }
};

#define MPQP_DECL(part, ...) __attribute__((visibility("hidden"))) FeasConfig feas_config_part##part();
MPQP_FEAS_PARTS(MPQP_DECL)
#undef MPQP_DECL

struct RegConfig {
    bool fp32;
    int nw, rw, lw, cs, ex, sn, eu;
    const void *fn;
    int rows() const { return nw * rw; }
    int columns() const { return 64 * cs + ex; }
    int threads() const { return nw * 64; }
    int wgs() const { return eu * 4 / nw; }  // workgroups per CU of the budget
};

#define MPQP_DECL(part, ...) __attribute__((visibility("hidden"))) RegConfig reg_config_part##part();
MPQP_REG_PARTS(MPQP_DECL)
#undef MPQP_DECL
