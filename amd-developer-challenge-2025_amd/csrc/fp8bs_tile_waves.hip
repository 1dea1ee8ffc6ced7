// The small tiles of fp8bs_waves.h, eight waves each.  16 x 64 has the shortest block (10 KB of copies, four MFMAs); 32 x 64 makes half
// as many requests for b where there are more rows: 256 x 512 x 1024 3.8 and 3.9 us, 250 x 7168 x 2048 46 and 36.  (Four waves
// of 32 x 64 are 2 % faster than eight and take K splits up to four only; 64 x 64 and 16 x 128 are the fastest on 2 % of 264 shapes.)
#include "fp8bs_waves.h"

namespace fp8bs {
hipError_t launch_waves_16x64(const GemmArgs& a, hipStream_t stream) { return a.epi == 1 ? launch_waves<16, 64, 8, 1>(a, stream) : launch_waves<16, 64, 8, 0>(a, stream); }
hipError_t launch_waves_32x64(const GemmArgs& a, hipStream_t stream) { return a.epi == 1 ? launch_waves<32, 64, 8, 1>(a, stream) : launch_waves<32, 64, 8, 0>(a, stream); }
int waves_lds_bytes(int tile_m) { return tile_m == 16 ? WavesCfg<16, 64, 8>::LDS_BYTES : WavesCfg<32, 64, 8>::LDS_BYTES; }
}  // namespace fp8bs
