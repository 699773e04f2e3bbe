// pa_gen_mfma_q8.hip - the Q8_0-K kernels of pa_gen_mfma.h.
#include "pa_gen_mfma.h"

namespace iian_pa {

hipError_t launch_gen_mfma_q8(const GenMfmaParams &p, int type_v, unsigned wgs, hipStream_t stream) {
    return launch_gen_mfma_k<8>(p, type_v, wgs, stream);
}

}  // namespace iian_pa
