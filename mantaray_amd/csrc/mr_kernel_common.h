// mr_kernel_common.h -- pieces shared by the kernel translation units
// (mr_kernels.hip, mr_adjoint.hip): the per-lane view loader and the
// constants of the fast dispersion evaluation.  Include from .hip files only.
#pragma once

#include <type_traits>

#include "mr_device.h"

namespace mr {

// Word 3 of a raw buffer descriptor on the gfx9 family (gfx950 among them):
// DATA_FORMAT (bits 18:15) = 4, 32-bit, a valid format for untyped
// accesses; every other field zero.
constexpr int MR_BUFFER_DWORD3 = 0x00020000;
// cache-policy operand of the buffer intrinsics: bit 1 is the nontemporal
// (streaming) hint on gfx950
constexpr int MR_CPOL_NT = 2;

// s_waitcnt on the vector memory count alone: wait until at most N vector
// memory operations are outstanding (gfx9 encoding: vmcnt in bits 3:0,
// expcnt 6:4 and lgkmcnt 11:8 at their no-wait maxima, vmcnt bits 15:14
// zero).
template <int N>
__device__ __forceinline__ void vm_wait()
{
    static_assert(N >= 0 && N < 16, "vmcnt below 16");
    __builtin_amdgcn_s_waitcnt(0x0F70 | N);
}

// Have a loaded view in registers at this point: each word is an input of
// an empty asm statement, so the compiler waits for the view's loads here
// and knows them complete in the code that follows (a loop after this does
// not wait for them again, nor for whatever else is in flight then).
template <class View>
__device__ __forceinline__ void settle(const View &v)
{
    int buf[sizeof(View) / 4];
    __builtin_memcpy(buf, &v, sizeof(View));
#pragma unroll
    for (int i = 0; i < (int)(sizeof(View) / 4); ++i) __asm__ volatile("" ::"v"(buf[i]));
}

static __device__ double mr_fast_consts[sizeof(FastConsts) / sizeof(double)] = {
    -2.0 * 1.4426950408889634,             // -2/ln 2
    0x1.8p52,
    0.5 * 6.93147180369123816490e-01,      // (ln 2)/2 split, upper part
    0.5 * 1.90821492927058770002e-10,      // (ln 2)/2 - upper part
    700.0,
    // expm1(F)/F interpolated at the 10 Chebyshev nodes of [-ln2/2, ln2/2]
    // (computed in 50-digit arithmetic and rounded), c_9 .. c_0, each times
    // 2^(j+1) (exact) for the argument f = F/2
    2.7620075879983367e-07 * 0x1p10,
    2.7632640675430236e-06 * 0x1p9,
    2.4801521322368692e-05 * 0x1p8,
    0.0001984119064754424 * 0x1p7,
    0.0013888888917196719 * 0x1p6,
    0.008333333367311603 * 0x1p5,
    0.041666666666624164 * 0x1p4,
    0.16666666666615648 * 0x1p3,
    0.5000000000000001 * 0x1p2,
    1.0000000000000013 * 0x1p1,
    // (expm1(F) - F)/F^2, interpolated likewise
    2.5100375832561234e-08 * 0x1p10,
    2.7620075879983367e-07 * 0x1p9,
    2.7557268480310024e-06 * 0x1p8,
    2.4801521322368692e-05 * 0x1p7,
    0.00019841269863040545 * 0x1p6,
    0.0013888888917196719 * 0x1p5,
    0.008333333333330065 * 0x1p4,
    0.041666666666624164 * 0x1p3,
    0.16666666666666669 * 0x1p2,
    0.5000000000000001 * 0x1p1,
    G,
    0.5 * G,
    0.25 * G,
};

// The constants in per-lane registers, in place before the code that
// follows.  The clamp goes through an addition, whose result is known to be no
// signalling NaN: the compiler would quiet a loaded value again in every step.
__device__ __forceinline__ FastConsts load_consts()
{
    FastConsts K = load_view<FastConsts>(mr_fast_consts);
    settle(K);
    K.clamp = K.clamp + 0.0;
    return K;
}

// t[0] = t0, t[s] = t[s-1] + dt for s <= n
__device__ __forceinline__ void time_column(double t0, double dt, int64_t n, double *t)
{
    double v = t0;
    t[0] = v;
    for (int64_t s = 1; s <= n; ++s) {
        v = v + dt;
        t[s] = v;
    }
}

// Field kinds and math mode as compile-time parameters.
template <int BK, int CK, int MATH>
struct Kinds {
    static constexpr int bk = BK, ck = CK, math = MATH;
};

// Call f(Kinds<BK, CK, MATH>{}) for the run-time field kinds and math mode.
template <class F>
void dispatch_kinds(int bk, int ck, int math, F &&f)
{
    auto by_math = [&](auto b, auto c) {
        constexpr int BK = decltype(b)::value, CK = decltype(c)::value;
        if (math == MATH_FAST) f(Kinds<BK, CK, MATH_FAST>{});
        else f(Kinds<BK, CK, MATH_LITERAL>{});
    };
    auto by_current = [&](auto b) {
        if (ck == CK_CONSTANT) by_math(b, std::integral_constant<int, CK_CONSTANT>{});
        else by_math(b, std::integral_constant<int, CK_GRID>{});
    };
    switch (bk) {
    case BK_CONSTANT: by_current(std::integral_constant<int, BK_CONSTANT>{}); break;
    case BK_SLOPE: by_current(std::integral_constant<int, BK_SLOPE>{}); break;
    case BK_ARRAY: by_current(std::integral_constant<int, BK_ARRAY>{}); break;
    default: by_current(std::integral_constant<int, BK_GRID>{}); break;
    }
}

}  // namespace mr
