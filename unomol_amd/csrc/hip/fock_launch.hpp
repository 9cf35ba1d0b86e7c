// The Fock kernels of one (digest mode, precision), behind one launch function: included by a
// source file each, so that they compile side by side.
#pragma once
#include <algorithm>
#include "fock_core.hpp"

namespace uno {

// Blocks of a launch, which take tasks until none is left: what the chip holds at a time.  (More
// only queue up behind them, stage their Rys table and find nothing to do.)
template <class K>
static hipError_t fock_grid(K kernel, int threads, size_t dyn, int ncand, unsigned& grid) {
    int per_cu = 0, dev = 0, cus = 0;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, dyn);
    if (e == hipSuccess) e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return e;
    grid = (unsigned)std::max(1, std::min(ncand, std::max(1, per_cu) * cus));
    return hipSuccess;
}

template <int LA, int LB, int LC, int LD, int MODE, typename T, int ROWS, bool TL>
static hipError_t fock_launch_v(const FockArgs& a, size_t dyn, hipStream_t st) {
    static size_t attr = 0;   // dynamic LDS limit set for this instantiation
    constexpr auto kernel = &k_fock<LA, LB, LC, LD, MODE, T, ROWS, TL>;
    if (dyn > attr) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)dyn);
        if (e != hipSuccess) return e;
        attr = dyn;
    }
    unsigned grid = 1;
    if (hipError_t e = fock_grid(kernel, kRowThreads, dyn, a.ncand, grid)) return e;
    hipLaunchKernelGGL((k_fock<LA, LB, LC, LD, MODE, T, ROWS, TL>), dim3(grid), dim3(kRowThreads), dyn, st,
                       a);
    return hipGetLastError();
}

// variant 0: outputs straight to W; 1: every bra row and the Rys table in LDS; 2: every bra row;
// 3: the first bra shell's rows
template <int LA, int LB, int LC, int LD, int MODE, typename T>
static hipError_t fock_launch_cls(const FockArgs& a, int variant, size_t dyn, hipStream_t st) {
    using CI = ClassInfo<LA, LB, LC, LD>;
    if constexpr (CI::NCOMP <= kLaneMaxComp) {
        switch (variant) {
            case 0: return fock_launch_v<LA, LB, LC, LD, MODE, T, kRowsNone, (CI::NR <= kLdsTabMaxRoots)>(a, dyn, st);
            case 1: return fock_launch_v<LA, LB, LC, LD, MODE, T, kRowsAll, true>(a, dyn, st);
            case 2: return fock_launch_v<LA, LB, LC, LD, MODE, T, kRowsAll, false>(a, dyn, st);
            case 3: return fock_launch_v<LA, LB, LC, LD, MODE, T, kRowsFirst, false>(a, dyn, st);
        }
        return hipErrorInvalidValue;
    } else {
        unsigned grid = 1;
        if (hipError_t e = fock_grid(&k_fock_wave<LA, LB, LC, LD, MODE, T>, 64, 0, a.ncand, grid)) return e;
        hipLaunchKernelGGL((k_fock_wave<LA, LB, LC, LD, MODE, T>), dim3(grid), dim3(64), 0, st, a);
        return hipGetLastError();
    }
}

template <int MODE, typename T>
static hipError_t fock_launch_mode(int cb, int ck, const FockArgs& a, int variant, size_t dyn,
                                   hipStream_t st) {
#define UNO_Q(X, Y, LA, LB, LC, LD) \
    if (cb == X && ck == Y) return fock_launch_cls<LA, LB, LC, LD, MODE, T>(a, variant, dyn, st);
    UNO_QUARTET_CLASSES(UNO_Q)
#undef UNO_Q
    return hipErrorInvalidValue;
}

}  // namespace uno
