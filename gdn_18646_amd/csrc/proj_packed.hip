// The MFMA projection kernel over packed sequences (proj_mfma.hpp), in a
// translation unit of its own for the build's sake.
#include "proj_mfma.hpp"

namespace gdn_proj {

int launch_mfma_packed(int tile, const ProjParams& p, int F3, hipStream_t stream) {
    return launch_mfma_tile<kPacked>(tile, p, F3, stream);
}

}  // namespace gdn_proj
