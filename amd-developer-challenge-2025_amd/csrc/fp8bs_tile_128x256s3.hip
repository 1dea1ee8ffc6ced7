// The tiled MFMA kernel of fp8bs_tiled.h in the eight waves of 64 x 64 and the three stages of the 256 x 128 tile, columns and rows exchanged:
// for grouped calls of some tens of rows an expert.  Bound: HBM.  A round of tiles reads whole 256-byte row segments of b, as 64 x 256 does, and holds
// twice the rows, so that an expert of 65 to 128 rows is one row of tiles and has its weights read once: 240 tokens to 8 of 32 experts of unequal shares,
// 4864 x 3840, 64x256 134.9 us, 256x256 139.2, the model's pick without this one 152.4, this 125.4 (4.8 TB/s); 959 to 2 of 32, 5376 x 2944, 136.3, 133.2, 136.4 and 108.6.
#include "fp8bs_tiled.h"

namespace fp8bs {
hipError_t launch_tile_128x256s3(const GemmArgs& a, int mode, hipStream_t stream) { return launch_grouped_shape<128, 256, 64, 64, 3>(a, mode, stream); }
}  // namespace fp8bs
