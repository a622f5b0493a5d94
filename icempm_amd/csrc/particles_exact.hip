// particles_exact.hip -- the particle pass without FMA contraction (the
// build's -ffp-contract=off): used by ORDERED mode, where the results must
// equal a sequential restatement of the reference bit for bit.
#include <climits>

#include "internal.h"
#include "ordered_device.h"

#define ICEMPM_PASS_NS exact
#include "particles.inc"

namespace icempm {
namespace exact {

hipError_t launch_g2p_records(const KParams &k, const double *gridV, const int *chunkStart, int nChunks,
                              int recordPQ, hipStream_t s, int kind, const PassExtra &extra) {
    if (k.nbins + 1 > kFoldBinsMax) return hipErrorInvalidValue;
    // one workgroup more folds the force
    const dim3 grid((unsigned)(((nChunks + 7) / 8) * 8 + 1));
    if (kind != 1 && k.grainVar == 0)
        hipLaunchKernelGGL((k_particles_wave<true, false, false, true>), grid, dim3(kChunk), 0, s, k, gridV, nullptr,
                           chunkStart, nChunks, recordPQ, 1, extra);
    else
        hipLaunchKernelGGL((k_particles_wave<true, false, false>), grid, dim3(kChunk), 0, s, k, gridV, nullptr, chunkStart,
                           nChunks, recordPQ, 1, extra);
    return hipGetLastError();
}

}  // namespace exact
}  // namespace icempm
