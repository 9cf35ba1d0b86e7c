// The Fock kernels of one (digest mode, precision), behind one launch function: included by a
// source file each, so that they compile side by side.
#pragma once
#include "fock_core.hpp"

namespace uno {

template <int LA, int LB, int LC, int LD, int MODE, typename T, int ROWS, bool TL>
static hipError_t fock_launch_v(const FockArgs& a, int nblocks, size_t dyn, hipStream_t st) {
    static size_t attr = 0;   // dynamic LDS limit set for this instantiation
    if (dyn > attr) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_fock<LA, LB, LC, LD, MODE, T, ROWS, TL>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)dyn);
        if (e != hipSuccess) return e;
        attr = dyn;
    }
    hipLaunchKernelGGL((k_fock<LA, LB, LC, LD, MODE, T, ROWS, TL>), dim3((unsigned)nblocks), dim3((row_threads<LA, LB, LC, LD>())), dyn, st,
                       a);
    return hipGetLastError();
}

// variant 0: outputs straight to W; 1: every bra row and the Rys table in LDS; 2: every bra row;
// 3: the first bra shell's rows
template <int LA, int LB, int LC, int LD, int MODE, typename T>
static hipError_t fock_launch_cls(const FockArgs& a, int nblocks, int variant, size_t dyn, hipStream_t st) {
    using CI = ClassInfo<LA, LB, LC, LD>;
    if constexpr (CI::NCOMP <= kLaneMaxComp) {
        switch (variant) {
            case 0: return fock_launch_v<LA, LB, LC, LD, MODE, T, kRowsNone, (CI::NR <= kLdsTabMaxRoots)>(a, nblocks, dyn, st);
            case 1: return fock_launch_v<LA, LB, LC, LD, MODE, T, kRowsAll, true>(a, nblocks, dyn, st);
            case 2: return fock_launch_v<LA, LB, LC, LD, MODE, T, kRowsAll, false>(a, nblocks, dyn, st);
            case 3: return fock_launch_v<LA, LB, LC, LD, MODE, T, kRowsFirst, false>(a, nblocks, dyn, st);
        }
        return hipErrorInvalidValue;
    } else {
        hipLaunchKernelGGL((k_fock_wave<LA, LB, LC, LD, MODE, T>), dim3((unsigned)nblocks), dim3(64), 0, st, a);
        return hipGetLastError();
    }
}

template <int MODE, typename T>
static hipError_t fock_launch_mode(int cb, int ck, const FockArgs& a, int nblocks, int variant, size_t dyn,
                                   hipStream_t st) {
#define UNO_Q(X, Y, LA, LB, LC, LD) \
    if (cb == X && ck == Y) return fock_launch_cls<LA, LB, LC, LD, MODE, T>(a, nblocks, variant, dyn, st);
    UNO_QUARTET_CLASSES(UNO_Q)
#undef UNO_Q
    return hipErrorInvalidValue;
}

}  // namespace uno
