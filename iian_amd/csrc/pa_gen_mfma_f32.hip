// pa_gen_mfma_f32.hip - the F32-K kernels of pa_gen_mfma.h.
#include "pa_gen_mfma.h"

namespace iian_pa {

hipError_t launch_gen_mfma_f32(const GenMfmaParams &p, int type_v, unsigned wgs, hipStream_t stream) {
    return launch_gen_mfma_k<0>(p, type_v, wgs, stream);
}

}  // namespace iian_pa
