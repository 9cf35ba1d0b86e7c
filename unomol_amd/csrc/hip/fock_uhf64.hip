// Fock kernels: open shell, FP64 quartets.
#include "fock_launch.hpp"

namespace uno {

hipError_t fock_launch_uhf64(int cb, int ck, const FockArgs& a, int variant, size_t dyn, hipStream_t st) {
    return fock_launch_mode<kDigestUHF, double>(cb, ck, a, variant, dyn, st);
}

}  // namespace uno
