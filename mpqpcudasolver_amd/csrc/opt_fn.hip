// opt_fn.hip — one group of optimality kernels (see opt_fn.hpp).
#include <hip/hip_runtime.h>

#include "lp_kernels.hpp"
#include "opt_fn.hpp"

#define MPQP_CAT_(a, b) a##b
#define MPQP_CAT(a, b) MPQP_CAT_(a, b)

#if MPQP_PART >= 20

template <int P>
struct Part;
#define MPQP_PICK(part, nw_, rw_, cs_, ex_, eu_)                                    \
    template <>                                                                     \
    struct Part<part> {                                                             \
        static constexpr int nw = nw_, rw = rw_, cs = cs_, ex = ex_, eu = eu_;      \
    };
MPQP_FEAS_PARTS(MPQP_PICK)

FeasConfig MPQP_CAT(feas_config_part, MPQP_PART)() {
    typedef Part<MPQP_PART> P;
    return FeasConfig{P::nw, P::rw, P::cs, P::ex, P::eu, &feas_reg<P::nw, P::rw, P::cs, P::ex, P::eu>};
}

#elif MPQP_PART >= 8

template <int P>
struct Part;
#define MPQP_PICK(part, fp32_, nw_, rw_, lw_, cs_, ex_, sn_, eu_)                                      \
    template <>                                                                                        \
    struct Part<part> {                                                                                \
        static constexpr bool fp32 = fp32_;                                                            \
        static constexpr int nw = nw_, rw = rw_, lw = lw_, cs = cs_, ex = ex_, sn = sn_, eu = eu_;     \
    };
MPQP_REG_PARTS(MPQP_PICK)

template <typename P>
static const void *reg_fn() {
    if constexpr (P::fp32)
        return reinterpret_cast<const void *>(&reg_kernel32<P::nw, P::rw, P::cs, P::ex, P::sn, P::eu>);
    else
        return reinterpret_cast<const void *>(&reg_kernel64<P::nw, P::rw, P::cs, P::ex, P::lw, P::sn, P::eu>);
}

RegConfig MPQP_CAT(reg_config_part, MPQP_PART)() {
    typedef Part<MPQP_PART> P;
    return RegConfig{P::fp32, P::nw, P::rw, P::lw, P::cs, P::ex, P::sn, P::eu, reg_fn<P>()};
}

#else

template <int NT, bool FP32, bool GT>
static const void *opt_fn_nt(int S) {
#define MPQP_OPT_FN(s)                                                       \
    (FP32 ? reinterpret_cast<const void *>(&opt_kernel32<NT, s, GT>)         \
          : reinterpret_cast<const void *>(&opt_kernel64<NT, s, GT>))
    switch (S) {
    case 1: return MPQP_OPT_FN(1);
    case 2: return MPQP_OPT_FN(2);
    case 3: return MPQP_OPT_FN(3);
    case 4: return MPQP_OPT_FN(4);
    case 6: return MPQP_OPT_FN(6);
    default: return MPQP_OPT_FN(8);
    }
#undef MPQP_OPT_FN
}

template <int P>
struct Part;
#define MPQP_PICK(part, nt, fp32, gt)                     \
    template <>                                           \
    struct Part<part> {                                   \
        static constexpr int threads = nt;                \
        static constexpr bool single = fp32, split = gt;  \
    };
MPQP_OPT_PARTS(MPQP_PICK)

const void *MPQP_CAT(opt_fn_part, MPQP_PART)(int S) {
    typedef Part<MPQP_PART> P;
    return opt_fn_nt<P::threads, P::single, P::split>(S);
}

#endif
