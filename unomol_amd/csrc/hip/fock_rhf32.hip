// Fock kernels: closed shell, FP32 quartets.
#include "fock_launch.hpp"

namespace uno {

hipError_t fock_launch_rhf32(int cb, int ck, const FockArgs& a, int variant, size_t dyn, hipStream_t st) {
    return fock_launch_mode<kDigestRHF, float>(cb, ck, a, variant, dyn, st);
}

}  // namespace uno
