// The tiled MFMA kernel of fp8bs_tiled.h in the eight waves of 64 x 64 and the three stages of the 256 x 128 tile, columns and rows exchanged:
// for grouped calls of some tens of rows an expert whose weights come from memory.  Bound: HBM.  A round of tiles reads whole 256-byte row
// segments of b, as 64 x 256 does, and holds twice the rows, so that an expert of 65 to 128 rows has its weights read once: 240 tokens to 8 of 32
// experts of unequal shares, 4864 x 3840, 64x256 or 256x256 153.0 us, this 128.7 (4.6 TB/s); 959 to 2 of 32, 5376 x 2944, 136.7 and 111.9.
#include "fp8bs_tiled.h"

namespace fp8bs {
hipError_t launch_tile_128x256s3(const GemmArgs& a, int mode, hipStream_t stream) { return launch_grouped_shape<128, 256, 64, 64, 3>(a, mode, stream); }
}  // namespace fp8bs
