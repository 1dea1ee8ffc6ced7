// Internal interface between the C-ABI layer (fp8bs_api.hip) and the device code (fp8bs_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace fp8bs {

// Kernel arguments. Layouts as in include/fp8bs.h. In grouped mode `m` and `lda` are the total row
// count and `b`/`bs` carry a leading expert dimension.
struct GemmArgs {
    const uint8_t* a;
    const uint8_t* b;
    const float* as;
    const float* bs;
    uint16_t* c;            // bf16 bits
    float* ws;              // split-K partial planes [split_k][m][n]
    const int32_t* row_offsets;
    int m, n, k;
    int lda;                // bytes per k row of a (the row count of the whole matrix)
    int nb;                 // ceil(n / 128)
    int split_k, kb_per_split;
    int band_h;             // tile rows per band of the tile walk
    int num_experts;
    int epi;                // 0: bf16 of the product; 1: silu(column 2i) * column 2i+1, n/2 output columns
    int c_whole_lines;      // set by the launcher: rows of c start and end on 128-byte lines
    int order;              // grouped: order of the tiles, ORDER_.. (see the tile walk)
    // K blocks dealt to the workgroups (MODE 3 of the tiled kernel): `ws` then holds a header (a status word, one
    // 8-byte flag per workgroup) and one fp32 partial tile per workgroup, see StreamK below
    unsigned long long sk_nonce;   // value a flag takes when its workgroup's partial tile is complete: differs from call to call
    int sk_grid;            // workgroups of such a call: at most the places on the chip and the number of (tile, K block) pairs
    int sk_spin;            // polls of a flag before the wait gives up (< 0: give up at once - tests of the error path); with a shared-out sum: before a part is left to another workgroup
};
// (A kernel's arguments are read cold at its start: with eight bytes more an unsplit grouped product of 64 tokens to 8 of 16 experts,
// 960 x 768, took 8.27 us instead of 8.18, means of three processes each in turn.)
static_assert(sizeof(GemmArgs) <= 120);

// The weights of a grouped call's experts, as many as can have rows, are as large as the 256 MB cache, and rows of them whole 128-byte lines.
inline bool weights_past_caches(int experts, int rows, int n, int k) {
    return (size_t)(rows < experts ? rows : experts) * (size_t)n * (size_t)k >= ((size_t)256 << 20) && n % 128 == 0;
}

// Whether the weights of an expert of so many tile rows are read past the caches, beside so many experts that have rows (see `b_read_once`).
constexpr unsigned long long ALL_CACHES = 288ull << 20;          // 256 MB and the L2s of the eight XCDs
__host__ __device__ constexpr bool expert_read_once(int experts_with_rows, int tile_rows, int n, int k) {
    return tile_rows == 1 && (unsigned long long)experts_with_rows * ((unsigned long long)n * (unsigned long long)k) >= ALL_CACHES;
}

// Orders of a grouped call's tiles: across the experts, a workgroup's columns of b other ones in each round; expert by expert; across the experts.
enum { ORDER_TURNED, ORDER_BY_EXPERT, ORDER_ACROSS };
// Whether a call across the experts turns its rounds (see `place` in fp8bs_tiled.h).
__host__ __device__ constexpr bool turns_rounds(int n) { return n % 512 == 0; }

// Or'ed into a mode: raise the LDS limit of the kernel that the arguments take and launch nothing (tiles of gemm_tr_kernel).
constexpr int READY_ONLY = 256;

// Workspace of a call that deals K blocks (all offsets from the 16-byte aligned workspace base):
//   [0, 4)                          status word: set to FP8BS_ERR_TIMEOUT by a workgroup whose bounded wait gave up
//   [SK_FLAGS_OFF, + 8 * grid)      one flag per workgroup
//   [SK_SLOTS_OFF, + grid * slot)   one partial tile per workgroup, slot = tile_m * tile_n * 4 bytes, in lane order
struct StreamK {
    static constexpr size_t FLAGS_OFF = 256, SLOTS_OFF = 16384;
    static constexpr int MAX_GRID = (int)((SLOTS_OFF - FLAGS_OFF) / 8);
    static constexpr unsigned STATUS_TIMEOUT = 9;        // FP8BS_ERR_TIMEOUT
    static size_t bytes(int grid, int tile_m, int tile_n) { return SLOTS_OFF + (size_t)grid * (size_t)tile_m * (size_t)tile_n * 4u; }
};

// Per-device bookkeeping of the launchers.  A kernel's dynamic-LDS limit is a property of the kernel
// on one device, so "already raised" is remembered per device; devices beyond the table just set the
// attribute on every launch.  Races between threads are harmless (the call is idempotent).
static constexpr int MAX_DEVICES = 64;
inline int device_slot() {
    int d = 0;
    return (hipGetDevice(&d) == hipSuccess && d >= 0 && d < MAX_DEVICES) ? d : -1;
}
// `raised[slot]` holds the largest limit set so far for this kernel on that device.
inline hipError_t raise_lds_limit(const void* kernel, int bytes, int* raised) {
    const int slot = device_slot();
    if (slot >= 0 && raised[slot] >= bytes) return hipSuccess;
    hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess && slot >= 0) raised[slot] = bytes;
    return e;
}

// CUs of the current device, asked once per device (256, MI355X's count, if the runtime does not say)
inline int device_cus() {
    static int cus[MAX_DEVICES];
    const int slot = device_slot();
    if (slot >= 0 && cus[slot] > 0) return cus[slot];
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    if (slot >= 0) cus[slot] = n;
    return n;
}

// Upper bound on the m-tile slots of a grouped call of `rows` rows: an expert of r rows starts up to 15 rows into its first
// tile and has ceil((r + 15) / bm) <= 1 + r / (bm - 14) of them, and no more experts have rows than there are rows.
// (For row_offsets that do not descend; the kernel cuts the slots of any others here where it sums K partitions, whose
// counters and partial tiles are laid out for this many.)
__host__ __device__ inline long grouped_slots_bound(long rows, long experts, int bm) { return (rows < experts ? rows : experts) + rows / (bm - 14); }

// Can the workgroups of a K split summed in the kernel share out the sums?  One workgroup per (tile, partition), all on the chip
// together, a flag for each in the workspace's header, a partition count the kernel is instantiated for, and a launch that is not
// captured: the flags carry a tag that is new with every call, and a replay would meet its own.  (Up to eight tiles one
// workgroup's sum is as fast: 1 x 512 x 7168 in two to four partitions of 64 x 64, 14.1 / 11.5 / 10.3 us either way.)
inline bool is_capturing(hipStream_t stream) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &cap) != hipSuccess) { (void)hipGetLastError(); return true; }    // (cannot be told: what a captured launch takes is always right)
    return cap != hipStreamCaptureStatusNone;
}
inline bool can_share_sum(long workgroups, long resident, int split_k, hipStream_t stream) {
    return workgroups > 8L * split_k && workgroups <= resident && workgroups <= StreamK::MAX_GRID && (split_k == 2 || split_k == 3 || split_k == 4 || split_k == 6 || split_k == 8) && !is_capturing(stream);
}

// mode: 0 dense bf16, 1 dense split-K partials, 2 grouped, 3 K blocks dealt, 4 dense split-K summed in the kernel, 5 grouped likewise.  tile: FP8BS_VARIANT_* (not AUTO) + 256 * form.
hipError_t launch_gemm(int tile, int mode, const GemmArgs& args, hipStream_t stream);
// one per tile shape of the tiled kernel, each in a translation unit of its own
hipError_t launch_tile_256x256(const GemmArgs& args, int mode, hipStream_t stream);
hipError_t launch_tile_256x192(const GemmArgs& args, int mode, hipStream_t stream);
hipError_t launch_tile_256x128(const GemmArgs& args, int mode, hipStream_t stream);
hipError_t launch_tile_256x128s3(const GemmArgs& args, int mode, hipStream_t stream);
hipError_t launch_tile_128x256s3(const GemmArgs& args, int mode, hipStream_t stream);
hipError_t launch_tile_128x128(const GemmArgs& args, int mode, hipStream_t stream);
hipError_t launch_tile_128x128s4(const GemmArgs& args, int mode, hipStream_t stream);
hipError_t launch_tile_64x128(const GemmArgs& args, int mode, hipStream_t stream);
hipError_t launch_tile_64x64(const GemmArgs& args, int mode, hipStream_t stream);
hipError_t launch_tile_192x192s3(const GemmArgs& args, int mode, hipStream_t stream);
hipError_t launch_tile_64x256s3(const GemmArgs& args, int mode, hipStream_t stream);
// the small tiles whose workgroups hold all K partitions (fp8bs_waves.h): split_k up to eight
hipError_t launch_waves_16x64(const GemmArgs& args, hipStream_t stream);
hipError_t launch_waves_32x64(const GemmArgs& args, hipStream_t stream);
int waves_lds_bytes(int tile_m);
hipError_t launch_splitk_reduce(const float* ws, uint16_t* c, size_t mn, int split_k, int epi, hipStream_t stream);
int variant_lds_bytes(int tile);

}  // namespace fp8bs
