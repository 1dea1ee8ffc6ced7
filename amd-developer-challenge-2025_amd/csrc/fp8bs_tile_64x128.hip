// The tiled MFMA kernel of fp8bs_tiled.h for the two tiles of 64 rows and at most 128 columns (all modes, both tail
// instantiations).  Both are bound by what one K block costs a workgroup from barrier to barrier, not by the matrix
// cores; measured per block on one CU: 64 x 128 in eight waves of 32 x 32 with three stages 0.34 us against 0.45 in
// four waves of 32 x 64 with two (more waves to hide the transposing reads behind, one block more to land in), 64 x 64
// in four waves with four stages 0.29.  Two workgroups fit a CU either way.
#include "fp8bs_tiled.h"

namespace fp8bs {
hipError_t launch_tile_64x128(const GemmArgs& a, int mode, hipStream_t stream) { return launch_shape<64, 128, 32, 32, true, 3>(a, mode, stream); }
hipError_t launch_tile_64x64(const GemmArgs& a, int mode, hipStream_t stream) { return launch_shape<64, 64, 32, 32, true, 4, true>(a, mode, stream); }
}  // namespace fp8bs
