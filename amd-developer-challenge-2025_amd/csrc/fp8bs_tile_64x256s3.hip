// The tiled MFMA kernel of fp8bs_tiled.h for eight waves of 32 x 64 with a deep copy ring, arranged in two ways (all
// modes, both tail instantiations): two by four, 64 x 256 with three stages - whole 256-byte row segments of b, for calls
// that stream b - and four by two, 128 x 128 with four stages, which moves a fifth less per product and has three blocks
// on their way: what tiles that run alone on a CU finish soonest on.  Per K block on one CU 0.49 and 0.44 us, of
// which 192 transposing reads and 40 or 32 KiB of copies, at 128 bytes a clock, occupy the LDS for 0.45 and 0.43: over the
// whole kernel, first copies and output included, 74 and 77 % of its cycles (matrix cores 35 and 39 %, a wave waits for 30 %;
// profiles/gemm_tr_mid_tiles_counters.txt).  4096 x 1024 x 4096, one tile per CU: 22.9 and 20.5 us, against 28.5 for
// 256 x 128 and 28.8 for 128 x 128 in four waves with two stages, which reads a third less from the LDS and waits more.
#include "fp8bs_tiled.h"

namespace fp8bs {
hipError_t launch_tile_64x256s3(const GemmArgs& a, int mode, hipStream_t stream) { return launch_shape<64, 256, 32, 64, true, 3, true>(a, mode, stream); }
hipError_t launch_tile_128x128s4(const GemmArgs& a, int mode, hipStream_t stream) { return launch_shape<128, 128, 32, 64, true, 4, true>(a, mode, stream); }
}  // namespace fp8bs
