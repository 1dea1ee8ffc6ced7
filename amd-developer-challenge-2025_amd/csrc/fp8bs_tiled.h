// FP8 (OCP e4m3fn) block-scaled GEMM kernels for gfx950 (CDNA4, MI355X).
//
// Computes, per 128-wide K block kb,   P_kb[m][n] = sum_{kk in kb} A[m][kk] * B[n][kk]   on the FP8
// matrix cores (v_mfma_f32_16x16x128_f8f6f4, one instruction = one whole scale block of one 16x16
// tile), then folds   C[m][n] += P_kb[m][n] * (a_scale[m][kb] * b_scale[n/128][kb])   into fp32
// accumulators on the vector ALU, and finally rounds to bf16.  Semantics follow the reference's
// dequantise-then-multiply statement (1-amd-fp8-mm/0-amd-fp8-mm-new-begins.py:17-49, 85-89) and the
// per-block fold of its shipped kernel (1-amd-fp8-mm/amd-fp8-mm-submission.py:333, 350-352).
//
// Memory layouts are the reference's (amd-fp8-mm-submission.py:66-75, 307-316): both operands arrive
// with K as the strided dimension, a[kk*M + i], b[kk*N + j].  The K<->M/N transpose the matrix cores
// need is fused into the LDS read: tiles are copied to LDS untransposed ([k][m] rows, 16-byte chunks,
// asynchronous global->LDS loads that bypass registers) and the operands are fetched with the CDNA4
// transposing read ds_read_b64_tr_b8, which hands every lane 8 consecutive-k bytes of one row.
//
// Layout facts used below were measured on the chip with one-hot operands:
//  * ds_read_b64_tr_b8: inside each group of 16 lanes, source lanes 2r and 2r+1 address the low and
//    high 8 bytes of "k row" r (r = 0..7); result lane i receives, as byte r, column i of row r.
//  * v_mfma_f32_16x16x128_f8f6f4: lane l supplies 32 bytes of row l%16 for k group l/16; operand A
//    and operand B use the same (group, byte) -> k map, so any k order inside the block is valid as
//    long as both operands use the same one.  D[i][j] (i from src0 rows, j from src1 rows) lives in
//    lane 16*(i/4) + j, register i%4.
// The kernel feeds B rows (n) as src0 and A rows (m) as src1, so a lane owns four consecutive n of
// one output row m: one a_scale value per lane per 16x16 tile and 8-byte contiguous bf16 stores.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>
#include <type_traits>
#include <utility>

#include "fp8bs_kernels.h"

namespace fp8bs {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef unsigned int v2u __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef unsigned short v4us __attribute__((ext_vector_type(4)));

#define LDS_V2I(p) ((__attribute__((address_space(3))) v2i*)(p))
#define LDS_VOID(p) ((__attribute__((address_space(3))) void*)(p))

static constexpr int KBLK = 128;  // scale block along K == K extent of one MFMA
static constexpr int GROUP_TABLE_MAX = 264;   // grouped walk: up to 263 experts have their row ranges kept in LDS (4.1 KiB)

__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
    v2f f = {lo, hi};
    v2bf h = __builtin_convertvector(f, v2bf);   // v_cvt_pk_bf16_f32: round to nearest even
    return __builtin_bit_cast(uint32_t, h);
}

// 16 bytes per lane, global -> LDS without passing through registers (buffer_load_dwordx4 ... lds):
// lane l's bytes land at lds_base + 16*l; lds_base and wave_offset must be wave-uniform (SGPRs), the
// address is buffer base + lane_offset + wave_offset.
// M0 (the LDS base of such a load) is written inside the statement.  The compiler reserves M0 and warns
// when it sees it among the clobbers; nothing it generates for these kernels reads M0 (LDS instructions
// need no M0 on gfx9, and there are no indirect register moves, GWS or message instructions here).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void copy16_global_to_lds(__amdgpu_buffer_rsrc_t rsrc, uint32_t lds_base, uint32_t lane_offset, uint32_t wave_offset) {
    asm volatile("s_mov_b32 m0, %2\n\tbuffer_load_dwordx4 %0, %1, %3 offen lds"
                 :: "v"(lane_offset), "s"(rsrc), "s"(lds_base), "s"(wave_offset) : "memory", "m0");
}
// same, with the nontemporal hint where `once` is not zero.  (The hint is a bit of the instruction.  The branch stands inside the assembly: the
// K loop stays one straight-line block to the compiler.  It costs nothing that shows: 256 rows to 32 experts, 4096 x 7168, 152.7 and 152.3.)
__device__ __forceinline__ void copy16_global_to_lds_once(__amdgpu_buffer_rsrc_t rsrc, uint32_t lds_base, uint32_t lane_offset, uint32_t wave_offset, uint32_t once) {
    asm volatile("s_mov_b32 m0, %2\n\ts_cmp_eq_u32 %4, 0\n\ts_cbranch_scc1 0f\n\tbuffer_load_dwordx4 %0, %1, %3 offen nt lds\n\ts_branch 1f\n"
                 "0:\tbuffer_load_dwordx4 %0, %1, %3 offen lds\n1:"
                 :: "v"(lane_offset), "s"(rsrc), "s"(lds_base), "s"(wave_offset), "s"(once) : "memory", "m0", "scc");
}
// same with 4 bytes per lane: lane l's dword lands at lds_base + 4*l
__device__ __forceinline__ void copy4_global_to_lds(__amdgpu_buffer_rsrc_t rsrc, uint32_t lds_base, uint32_t lane_offset, uint32_t wave_offset) {
    asm volatile("s_mov_b32 m0, %2\n\tbuffer_load_dword %0, %1, %3 offen lds"
                 :: "v"(lane_offset), "s"(rsrc), "s"(lds_base), "s"(wave_offset) : "memory", "m0");
}
#pragma clang diagnostic pop

// ---------------------------------------------------------------------------------------------------
// Tile -> workgroup mapping.  Workgroups are dealt round-robin to the 8 XCDs (each with its own L2),
// so workgroup w lives on XCD w%8.  Give every XCD a contiguous run of "virtual" ids, and lay the
// virtual ids over the tile grid in bands of GH tile rows walked column by column, so the tiles that
// share an L2 form a compact block and re-use each other's A and B panels.
// ---------------------------------------------------------------------------------------------------
__device__ __forceinline__ int xcd_virtual_id(int wg, int total) {
    const int NX = 8;
    int x = wg % NX, idx = wg / NX;
    int q = total / NX, r = total % NX;
    return x * q + (x < r ? x : r) + idx;
}

__device__ __forceinline__ void band_tile(int v, int tiles_m, int tiles_n, int gh, int& tm, int& tn) {
    // (divisions only where they are needed: each is some 25 dependent instructions ahead of a kernel's first copies; 27 x 1408 x 1280 3.85
    // -> 3.73 us, 128 x 6080 x 896 5.10 -> 4.90, 64 x 6614 x 1152 6.26 -> 6.09, 111 dense products 0.988 in the geometric mean)
    int band = 0, rem = v;
    if (tiles_m > gh) {
        const int per_band = gh * tiles_n;
        band = v / per_band;
        rem = v - band * per_band;
    }
    int rows = tiles_m - band * gh;           // rows in this band (last band may be short)
    rows = rows < gh ? rows : gh;
    if ((rows & (rows - 1)) == 0) tn = rem >> __builtin_ctz(rows);
    else tn = rem / rows;
    tm = band * gh + (rem - tn * rows);
}

// ---------------------------------------------------------------------------------------------------
// Main kernel.
//   BM x BN : workgroup tile (rows of A x rows of B), WM x WN : wave tile, 64*(BM/WM)*(BN/WN) threads.
//   MODE 0  : dense, bf16 output
//   MODE 1  : dense split-K, fp32 partial planes to the workspace
//   MODE 2  : grouped (row_offsets), bf16 output
//   MODE 3  : dense, K blocks instead of tiles dealt to the workgroups, partial tiles through the workspace, bf16 output
//   MODE 4  : dense split-K, partial tiles to the workspace, the sum of a tile shared out among its workgroups or done by the last of them, bf16 output
//   MODE 5  : grouped like MODE 2 with a K split summed like MODE 4's
//   MODE 6  : MODE 2 with b read past the caches for the experts of one tile row, see the rule at `b_read_once`
// LDS: NSTAGE stages, each [128 k][BM] bytes of A then [128 k][BN] bytes of B, 16-byte chunks XOR-swizzled
// so that the 16 k rows touched by half a wave in one transposing read fall on 16 different 16-byte
// bank groups, then the k block's a_scale row and b_scale values.
// ---------------------------------------------------------------------------------------------------
template <int BM, int BN, int WM, int WN, int MODE, int NSTAGE_ = 2>
struct TileCfg {
    static constexpr int NSTAGE = NSTAGE_;                           // LDS stages of one K block each
    static constexpr int WAVES_M = BM / WM, WAVES_N = BN / WN;
    static constexpr int NWAVES = WAVES_M * WAVES_N;
    static constexpr int NTHREADS = NWAVES * 64;
    static constexpr int MT = WM / 16, NT = WN / 16;
    static constexpr int CPR_A = BM / 16, CPR_B = BN / 16;          // 16-byte chunks per k row
    static constexpr int A_BYTES = KBLK * BM, B_BYTES = KBLK * BN;
    static constexpr int AS_BYTES = BM * 4;                          // the k block's a_scale row
    static constexpr int AS_AREA = AS_BYTES < 1024 ? 1024 : AS_BYTES;
    static constexpr int BS_AREA = 256;                              // the k block's b_scale values of the tile's n blocks
    static constexpr int STAGE_BYTES = A_BYTES + B_BYTES + AS_AREA + BS_AREA;
    static constexpr int LDS_BYTES = NSTAGE * STAGE_BYTES;
    static_assert(NSTAGE >= 2, "at least two stages");
    static_assert(LDS_BYTES <= 160 * 1024, "LDS");
    static constexpr int A_LOADS = A_BYTES / 16 / NTHREADS;         // 16-byte loads per thread per block
    static constexpr int B_LOADS = B_BYTES / 16 / NTHREADS;
    static_assert(A_BYTES % (16 * NTHREADS) == 0 && B_BYTES % (16 * NTHREADS) == 0, "tile/threads");
    // A wave's n range lies inside one b_scale block when the wave width divides 128 and tiles start on a block
    // boundary or, narrower than a block, divide it.  Otherwise (BN = 192, WN = 96) it may cross one boundary, at an n tile that
    // depends on the tile and the wave: the K loop is instantiated per boundary position.
    static constexpr bool SPLIT_SCALES = !(128 % WN == 0 && (BN % 128 == 0 || 128 % BN == 0));
    static_assert(WN <= 128, "a wave's n range crosses at most one b_scale block boundary");
    static_assert(!SPLIT_SCALES || (BN == 192 && WN == 96), "boundary positions are enumerated for the 192-wide tile only");
    static_assert(CPR_A <= 16 && CPR_B <= 16, "swizzle assumes a k row spans at most 256 bytes");
};

template <int N> __device__ __forceinline__ void wait_vmcnt() {
    // s_waitcnt with only vmcnt constrained: vmcnt is split over bits [3:0] and [15:14]
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// same, and all LDS and scalar-memory results back (lgkmcnt(0))
template <int N> __device__ __forceinline__ void wait_vmcnt_lgkm0() {
    __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | ((N >> 4) << 14));
}

template <int CPR>
__device__ __forceinline__ int swz_of_krow(int krow) {
    if constexpr (CPR != 12) {
        // rows per 256-byte bank sweep = 16/CPR; consecutive sweeps get consecutive XOR masks
        constexpr int ROWS_PER_SWEEP = CPR <= 16 ? 16 / CPR : 1;      // (wider rows are never swizzled)
        return (krow / ROWS_PER_SWEEP) % CPR;
    } else {
        // 12 chunks per k row (192 bytes): four consecutive rows start on the four different quarters of
        // a 256-byte bank sweep, the next four repeat them; rotating the chunks of each group of four
        // rows by one more position puts any 16 consecutive rows of one chunk column on 16 different
        // 16-byte bank groups.
        return (krow >> 2) & 3;
    }
}
// position of logical chunk `ch` inside its k row, and back
template <int CPR>
__device__ __forceinline__ int chunk_to_stored(int ch, int swz) {
    if constexpr ((CPR & (CPR - 1)) == 0) return ch ^ swz;
    else { int x = ch + swz; return x >= CPR ? x - CPR : x; }
}
template <int CPR>
__device__ __forceinline__ int stored_to_chunk(int st, int swz) {
    if constexpr ((CPR & (CPR - 1)) == 0) return st ^ swz;
    else { int x = st - swz; return x < 0 ? x + CPR : x; }
}

// The four bytes before `end`, which may be any address (the same in all lanes), from the one or two dwords that hold them.  Scalar
// loads: nothing waits for them but what uses them, where a vector load would be waited for together with the copies.
__device__ __forceinline__ uint32_t load_last_dword(const uint8_t* end) {
    typedef const __attribute__((address_space(4))) uint32_t* dword;
    const uintptr_t at = (uintptr_t)end - 4;
    const uint32_t lo = *(dword)(at & ~(uintptr_t)3), hi = *(dword)((at + 3) & ~(uintptr_t)3);
    return (uint32_t)((((uint64_t)hi << 32) | lo) >> (8 * (at & 3)));
}
// The byte `back` = 1, 2 or 3 before the end of an operand of k rows of ld bytes: bit 31 = the range check cuts it off, bits 29-30 = its k row
// minus k - 3, bits 0-28 = its row (of a) or column (of b).
__device__ __forceinline__ uint32_t tail_candidate(uint32_t back, uint32_t ld, uint32_t k) {
    const uint32_t rows = ld > 2 ? 0 : ld == 2 ? (back - 1) >> 1 : back - 1;       // whole k rows behind its own
    const uint32_t krow = k - 1 - rows, x = (rows + 1) * ld - back, end = k * ld;
    const bool lost = krow * ld + (x & ~3u) + 4u > end;                   // its dword crosses the end
    return lost ? (0x80000000u | ((krow - (k - 3u)) << 29) | x) : 0u;
}

// EPI 0: plain bf16 output.  EPI 1: gate/up pairs - column 2i is gate_i, column 2i+1 is up_i - are
// combined to silu(gate_i) * up_i in fp32 and the output has n/2 columns (role of the fp16 layer's
// re_silu_mul_kernel, 2-amd-moe/amd-moe-submission.py:366-407, fused into the GEMM as in
// 2-amd-moe/5-amd-fp8-moe-hip-fuse.py:366-408).
__device__ __forceinline__ float silu_mul(float gate, float up) {
    // gate / (1 + exp(-gate)) * up; exp2 and rcp are the hardware approximations (~1 ulp)
    return gate * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.44269504088896341f * gate)) * up;
}

// TAILS: lda is not a multiple of four or n not a multiple of eight; the kernel then repairs the last
// bytes of a and b in LDS and stores a row's last, partial 16-byte chunk of c
// in pieces, see below.
// Waves per SIMD when as many workgroups as LDS and thread count allow share a CU.  The modes that exchange partial
// tiles must keep their registers within that (their sums would otherwise take registers the K loop does not need
// and halve the number of workgroups per CU); the other modes fit without being told.
template <int BM, int BN, int WM, int WN, int MODE, int NSTAGE>
constexpr int waves_per_simd() {
    using C = TileCfg<BM, BN, WM, WN, MODE, NSTAGE>;
    const int by_lds = 163840 / C::LDS_BYTES, by_threads = 2048 / C::NTHREADS;
    const int w = C::NWAVES * (by_lds < by_threads ? by_lds : by_threads) / 4;
    return MODE >= 3 && MODE <= 5 && w > 1 ? w : 1;
}

// Tiles whose K partitions can share out the sum of a tile (see there).  Not 64x128: its two workgroups per CU leave 128
// registers a wave, and the sums spill (128 x 7168 x 7168 in three 26.9 us against 24.9 with one workgroup summing); not
// the tiles with more than eight accumulators a wave, which the planner splits in two or three only where the chip is full.
template <int BM, int BN, int WM, int WN> constexpr bool shares_sum() { return (BM == 64 && BN == 64) || (WM == 32 && WN == 64); }
// The fewest partitions it is shared out in.  64x64 has four accumulators a wave: in two parts nothing is gained, in three, of which
// one is twice the others, 1.8 % lost over 210 shapes, 5.5 % where all rows start on 16 bytes (192 x 1280 x 3072: one workgroup summing
// 8.8 us, shared 9.5).  The other tiles gain 2.4 % in three and up to 1 % in two (280 and 310 shapes).
template <int BM, int BN> constexpr int shares_from() { return BM == 64 && BN == 64 ? 4 : 2; }

// SHARED_SUM: the sum of a tile is shared out among its workgroups; without, the last of them does it.  An instantiation each, chosen
// by the launcher: with both forms in one kernel the sum by one workgroup - all that a captured launch can have - was 2 to 5 % slower
// (us, replayed: 448 x 924 x 4480 12.9 and 12.3, 22 x 4544 x 3200 9.8 and 9.3, 1876 x 571 x 4608 20.8 and 20.0).
template <int BM, int BN, int WM, int WN, int MODE, int EPI = 0, int NSTAGE = 2, bool TAILS = false, bool SHARED_SUM = false>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64) __attribute__((amdgpu_waves_per_eu(waves_per_simd<BM, BN, WM, WN, MODE, NSTAGE>())))
void gemm_tr_kernel(const GemmArgs p) {
    using C = TileCfg<BM, BN, WM, WN, MODE, NSTAGE>;
    constexpr bool GROUPED = MODE == 2 || MODE == 5 || MODE == 6, SUMMED = MODE == 4 || MODE == 5, B_ONCE = MODE == 6;
    static_assert(!SHARED_SUM || (SUMMED && shares_sum<BM, BN, WM, WN>()));
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];

    // global store instructions per wave and tile in the bf16 epilogue (always this many: lanes without
    // a valid element are switched off by an out-of-range buffer offset, not by a branch)
    constexpr int EPI_WNO = EPI == 1 ? WN / 2 : WN;
    constexpr int EPI_ROW_CHUNKS = EPI_WNO * 2 / 16;
    constexpr int EPI_ROWS_PER_PASS = (EPI_ROW_CHUNKS & (EPI_ROW_CHUNKS - 1)) == 0 ? 64 / EPI_ROW_CHUNKS : 4;
    // the wave tile is staged in parts of whole m tiles, in one part where a pass of stores covers more rows than half of it
    constexpr int EPI_PARTS = WM / 2 < EPI_ROWS_PER_PASS ? 1 : (WM / 16) % 2 == 0 ? 2 : WM / 16;
    constexpr int EPI_STORES = MODE == 1 ? 0 : EPI_PARTS * ((WM / EPI_PARTS) / EPI_ROWS_PER_PASS);

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, i16 = lane & 15;
    // Waves w and w+4 share a SIMD.  With 4 x 2 waves they get m positions two apart, so that in a tile
    // whose valid rows end at half height (the last tile of an expert, of M) every SIMD keeps one wave
    // with work instead of two SIMDs keeping both.
    const int wave_n = wave / C::WAVES_M;
    const int wave_m = (C::WAVES_M == 4 && C::NWAVES == 8) ? ((wave + 2 * wave_n) & 3) : wave % C::WAVES_M;

    // ---- tiles ---------------------------------------------------------------------------------
    // The workgroup is persistent: it walks the tiles  blockIdx.x, blockIdx.x + gridDim.x, ...  and
    // issues the first K block of the next tile before it converts and stores the current one, so a
    // tile's output and the next tile's first loads overlap (with K = 2048 the per-tile prologue and
    // epilogue are a third of a tile's time otherwise).
    // (No member for one mode only: with one more the compiler keeps parts of a tile in scratch memory, also in modes that do not use it, and 2197 rows to 64
    // experts, 1920 x 1408 in 256x256, takes 50.0 us instead of 47.3.)
    struct Tile {
        int valid, m0, n0, n_hi, kb_begin, kb_end, split_z, row_lo, row_hi;
        int sk_contrib, sk_first;             // MODE 3: the segment ends before the tile's last K block; first workgroup of the tile's earlier segments (-1: none)
                                              // MODE 6: sk_contrib: b is read past the caches
        const uint8_t* bptr;
        const float* bsptr;
    };
    int total_slots = 0;                      // grouped: m-tile slots that exist (from row_offsets)
    [[maybe_unused]] int active = 0;          // MODE 6: experts that have rows
    [[maybe_unused]] int once_rows = 0;       // the tile rows of an expert whose weights are read past the caches, 0: none
    // Grouped, fewer than GROUP_TABLE_MAX experts: a table in LDS, one entry per expert - first row of its first
    // tile (row_offsets[e] rounded down to 16), its row range, and the number of slots before it - built once
    // by wave 0.  Finding a tile's expert is then one LDS read per lane and a count of the lanes whose experts
    // start at or before the tile's slot; as a loop over row_offsets in scalar code it took 1.5-2 us per tile,
    // between the last K block of one tile and the first copies of the next.  More experts: that loop.
    // Up to 64 experts: the table stands in registers, an expert a lane, in every wave - no LDS, no barrier and no shuffles ahead of the
    // first copies: 7 tokens to 8 of 8 experts, 1415 x 768, 6.18 -> 5.82 us; 67 to 4 of 8, 1792 x 768, 6.20 -> 5.88; 46 to 8 of 16, 766 x 1536, 9.40 -> 9.04; 90
    // products 0.973 of the time in the geometric mean.
    [[maybe_unused]] v4i* gtable = nullptr;
    bool use_table = false;
    [[maybe_unused]] v4i lane_entry = {0, 0, 0, 0x7FFFFFFF};   // the entry of expert `lane`
    if constexpr (GROUPED) {
        __shared__ v4i gtable_store[GROUP_TABLE_MAX];        // entry [num_experts]: the slots before the end = all of them
        gtable = gtable_store;
        use_table = p.num_experts < GROUP_TABLE_MAX;
        if (p.num_experts <= 64) {
            int lo = 0, hi = 0;
            if (lane < p.num_experts) { lo = p.row_offsets[lane]; hi = p.row_offsets[lane + 1]; }
            lo = lo < 0 ? 0 : lo; hi = hi > p.m ? p.m : hi;               // a malformed table must not reach beyond the matrix
            const int s = lo & ~15;
            const int nt = (hi > lo) ? (hi - s + BM - 1) / BM : 0;
            int incl = nt;                                                // inclusive prefix sum over the 64 lanes: in rows of 16, then across them
            incl += __builtin_amdgcn_update_dpp(0, incl, 0x111, 0xF, 0xF, false);      // row_shr:1
            incl += __builtin_amdgcn_update_dpp(0, incl, 0x112, 0xF, 0xF, false);
            incl += __builtin_amdgcn_update_dpp(0, incl, 0x114, 0xF, 0xF, false);
            incl += __builtin_amdgcn_update_dpp(0, incl, 0x118, 0xF, 0xF, false);
            incl += __builtin_amdgcn_update_dpp(0, incl, 0x142, 0xA, 0xF, false);      // row_bcast:15, into rows 1 and 3
            incl += __builtin_amdgcn_update_dpp(0, incl, 0x143, 0xC, 0xF, false);      // row_bcast:31, into rows 2 and 3
            if (lane < p.num_experts) lane_entry = (v4i){s, lo, hi, incl - nt};
            total_slots = __builtin_amdgcn_readlane(incl, 63);
            if constexpr (B_ONCE) active = __popcll(__ballot(nt > 0));
        } else if (use_table) {
            if (wave == 0) {
                int carry = 0;
                for (int base = 0; base < p.num_experts; base += 64) {
                    const int x = base + lane;
                    int lo = 0, hi = 0;
                    if (x < p.num_experts) { lo = p.row_offsets[x]; hi = p.row_offsets[x + 1]; }
                    lo = lo < 0 ? 0 : lo; hi = hi > p.m ? p.m : hi;       // a malformed table must not reach beyond the matrix
                    const int s = lo & ~15;
                    const int nt = (hi > lo) ? (hi - s + BM - 1) / BM : 0;
                    int incl = nt;                                        // inclusive prefix sum over the 64 lanes
#pragma unroll
                    for (int d = 1; d < 64; d <<= 1) {
                        const int y = __shfl_up(incl, d, 64);
                        if (lane >= d) incl += y;
                    }
                    if (x < p.num_experts) gtable_store[x] = (v4i){s, lo, hi, carry + incl - nt};
                    carry += __shfl(incl, 63, 64);
                    if constexpr (B_ONCE) active += __popcll(__ballot(nt > 0));
                }
                if (lane == 0) gtable_store[p.num_experts] = (v4i){active, 0, 0, carry};
            }
            __syncthreads();
            total_slots = __builtin_amdgcn_readfirstlane(gtable_store[p.num_experts][3]);
            if constexpr (B_ONCE) active = __builtin_amdgcn_readfirstlane(gtable_store[p.num_experts][0]);
        } else {
            for (int x = 0; x < p.num_experts; x++) {
                int lo = p.row_offsets[x], hi = p.row_offsets[x + 1];
                lo = lo < 0 ? 0 : lo; hi = hi > p.m ? p.m : hi;
                total_slots += (hi > lo) ? (hi - (lo & ~15) + BM - 1) / BM : 0;
                if constexpr (B_ONCE) active += hi > lo ? 1 : 0;
            }
        }
        if constexpr (B_ONCE) once_rows = expert_read_once(active, 1, p.n, p.k) ? 1 : 0;
        if constexpr (MODE == 5) {             // a malformed table must not reach beyond the workspace either
            const int bound = (int)grouped_slots_bound(p.m, p.num_experts, BM);
            total_slots = total_slots < bound ? total_slots : bound;
        }
    }
    // The tile that this workgroup takes in round `it`, -1: none.  The gridDim.x tiles in flight together are dealt to the XCDs in
    // contiguous runs, those of a last round that is not full as well: in runs of a full round's length they kept some XCDs busy and
    // left the others, and their share of the memory's rate, idle.  Where they leave half of the chip, or three quarters, they are cut in
    // two or four by columns (1 << cut parts, the most: one wave's columns each): waves without columns only copy and
    // columns of other parts are not fetched, so a part costs little more than what its columns do.
    // us, before and now: 46 tokens to 8 of 16 experts, 766 x 1536, 15.6 and 9.4; 46 to 4 of 32, 2485 x 2432, 64.1 and 50.4; 900 to 8 of 16,
    // 3072 x 1536, 48.0 and 41.8; 64 to 8 of 32, 7168 x 2048 (3.5 rounds), 101.2 and 97.4; dense 6144 x 4608 x 7168 195 and 177. 90 grouped
    // products (1 .. 4096 tokens) 0.93 of the time in the geometric mean, at worst 1.04 (1920 tokens to 4 of
    // 32 experts, 832 x 4992, where it is a matter of which experts the rows fall on: over four draws 0.93 to 0.97 with even experts, 0.97 to 1.02 with skewed ones).
    // Unsplit tiles of 256 columns: behind twelve full rounds the last one is dealt in runs of a full round's length, and not cut.  By then the workgroups have
    // drifted apart by more than a part saves, and parts for nearly all of them lengthen the longest: 4096 tokens to 8 of 32 experts, 7168 x
    // 2048 (16.2 rounds), over four draws of the experts, us, in runs 506.6-508.3, spread and cut 512.0-515.7; 2200 to 8 of 32, 7168 x 2048 in 64x256 (33 rounds)
    // 487.7-493.4 and 493.3-502.0; at 11.5 rounds 379.5-387.4 and 382.8-387.4, at 9.2 909.6-914.7 and 904.3-916.6, at 4.4 262.8-264.0 and 252.6-255.7.
    [[maybe_unused]] constexpr int SPREAD_ROUNDS = 12;
    constexpr int MOST_CUT = (MODE == 0 || MODE == 2 || MODE == 6) && BN == 256 ? (BN / WN >= 4 ? 2 : 1) : 0;
    // Across the experts, where a call is a stream of their weights, an XCD's workgroups change places from round to round, by a band's
    // rows - one n tile - each time, if rows of b are a multiple of 512 bytes apart.  A column of b then has the same address bits 7 and 8 in each row, and
    // the memory serves one eighth of the bits 7 to 9, 384 to 511, at 0.8 of the others' rate (64x256 tiles of 64 x 18432 x 7168: the fourth that holds
    // those bytes ends its K blocks at 26.5 us, the others at 20.3; with b 256 bytes further on it is the tiles beside them; rows 4352
    // apart: none).  A round being a multiple of the period, a workgroup had such a tile in every round or in none.  us, before and
    // now: 32 tokens to 8 of 32 experts, 4096 x 7168, 177.1 and 170.2; 64 to 8 of 32, 7168 x 2048, 102.7 and 97.1; 8 to 4 of 32, 4096 x 7168, 127.8
    // and 120.9; 8 rows to each of 32, 3584 x 1536, 38.8 and 37.6, 4608 x 1536 49.8 and 48.9; 3072 x 7168 142.4 and 142.8.  Elsewhere columns drift
    // through all of the bits, and turning only takes tiles from the panels that their neighbours read: 110 such calls (1 .. 37 rows an expert, 512 .. 7168 columns) 0.25 %
    // slower in the geometric mean, at worst 1.7 % (64 experts, 3328 x 2816, 118.8 and 120.8), so there it is left.  Not in a round that is cut, whose
    // places are other ones (3072 x 7168, 1.5 rounds: 145.7), and not expert by expert, where the weights are read once for many rows (4096 tokens, 4096 x
    // 7168: 921 as it is, 929 turned).
    [[maybe_unused]] int turn = 0;
    auto place = [&](int it, int total, int& part, int& cut) -> int {
        const int G = gridDim.x, first = it * G, here = total - first;
        int wg = blockIdx.x;
        if (here <= 0) return -1;
        if constexpr (GROUPED)
            if (it > 0 && p.order == ORDER_TURNED && (G >> 3) >= p.band_h) {
                const int x = blockIdx.x & 7, run = (G >> 3) + (x < (G & 7) ? 1 : 0), at = (int)(blockIdx.x >> 3);      // workgroups of this XCD, this one's place among them
                turn += p.band_h;
                if (turn >= run) turn -= run;
                wg = x + 8 * (at + turn >= run ? at + turn - run : at + turn);
            }
        if (here >= G) return first + xcd_virtual_id(wg, G);
        if constexpr (MOST_CUT > 0)
            if (it >= SPREAD_ROUNDS) {
                const int v = xcd_virtual_id(wg, G);
                return v < here ? first + v : -1;
            }
        if constexpr (MOST_CUT > 0)
            if (it > 0 || GROUPED) cut = MOST_CUT > 1 && here * 4 <= G ? 2 : here * 2 <= G ? 1 : 0;
        if (cut > 0) wg = blockIdx.x;
        const int pieces = here << cut;
        if (wg >= pieces) return -1;
        const int v = xcd_virtual_id(wg, pieces);
        part = v - (v >> cut << cut);
        return first + (v >> cut);
    };
    auto take_part = [&](Tile& t, int part, int cut) -> bool {       // false: no columns in it
        if constexpr (MOST_CUT > 0) {
            if (cut > 0) {
                t.n0 += part * (BN >> cut);
                if (t.n0 >= p.n) { t.valid = 0; return false; }
                if (t.n0 + (BN >> cut) < p.n) t.n_hi = t.n0 + (BN >> cut);
            }
        }
        return true;
    };
    [[maybe_unused]] const int sk_self = xcd_virtual_id(blockIdx.x, gridDim.x);
    auto pick_tile = [&](int it) -> Tile {
        Tile t;
        t.valid = 0; t.m0 = 0; t.n0 = 0; t.n_hi = p.n; t.kb_begin = 0; t.kb_end = 0; t.split_z = 0; t.row_lo = 0; t.row_hi = p.m;
        t.sk_contrib = 0; t.sk_first = -1;
        t.bptr = p.b; t.bsptr = p.bs;
        const int G = gridDim.x;
        if (MODE == 3) {
            // K blocks, not tiles, are dealt to the workgroups: the (tile, K block) pairs of the whole product
            // form one sequence - tiles in the band order of the dense walk, K ascending inside a tile - and
            // workgroup v takes a run of total/G pairs (the first total%G runs hold one more), G <= total.  A run
            // covers the end of one tile, whole tiles, and the beginning of another; the workgroup walks its tiles
            // from the last to the first.  A segment that ends before its tile's last K block is stored as an fp32 partial tile in
            // the workgroup's slot of the workspace (only the first segment a workgroup works on can be one);
            // the segment that holds the tile's last K block belongs to the tile's owner, who adds the
            // partial tiles of the workgroups before it in ascending order of K, then its own accumulators,
            // and writes the output.  The owner works on that segment last and every workgroup it waits for
            // has a lower index, started no later and worked on its partial tile first.
            const int tiles_m = (p.m + BM - 1) / BM, tiles_n = (p.n + BN - 1) / BN;
            const uint32_t kbt = (uint32_t)(p.k / KBLK);
            const uint32_t total = (uint32_t)tiles_m * (uint32_t)tiles_n * kbt;           // < 2^31 (checked by the launcher)
            // runs of q or q+1 pairs, the longer ones first
            const uint32_t q = total / (uint32_t)G, r = total - q * (uint32_t)G;
            auto run_start = [&](uint32_t w) -> uint32_t { return w * q + (w < r ? w : r); };
            const uint32_t v = (uint32_t)sk_self;
            const uint32_t s = run_start(v), e = run_start(v + 1);
            if (e <= s) return t;
            const int t_first = (int)(s / kbt), t_last = (int)((e - 1) / kbt);
            const int tile = t_last - it;
            if (tile < t_first) return t;
            t.valid = 1;
            int tm, tn;
            band_tile(tile, tiles_m, tiles_n, p.band_h, tm, tn);
            const uint32_t x0 = (uint32_t)tile * kbt;                                      // the tile's first pair
            int kb0 = tile == t_first ? (int)(s - x0) : 0;
            int kb1 = tile == t_last ? (int)(e - x0) : (int)kbt;
            int first = -1;
            if (kb1 == (int)kbt && kb0 > 0)                                               // the workgroup whose run holds x0
                first = (int)(x0 < r * (q + 1) ? x0 / (q + 1) : r + (x0 - r * (q + 1)) / q);
            // (uniform values that went through the vector ALU's division sequences: back to scalar registers)
            t.m0 = __builtin_amdgcn_readfirstlane(tm * BM); t.n0 = __builtin_amdgcn_readfirstlane(tn * BN);
            t.kb_begin = __builtin_amdgcn_readfirstlane(kb0);
            t.kb_end = __builtin_amdgcn_readfirstlane(kb1);
            t.sk_contrib = t.kb_end < (int)kbt;
            t.sk_first = __builtin_amdgcn_readfirstlane(first);
        } else if (GROUPED) {
            // grouped: m-tile slots are laid over the experts in order; expert e's tiles start at
            // row_offsets[e] rounded down to 16 so that global 16-byte loads stay aligned; rows outside
            // [row_offsets[e], row_offsets[e+1]) are computed but never stored.  The gridDim.x tiles in
            // flight together are dealt to the XCDs in contiguous runs.  Two orders of the tiles.  Across
            // the experts: the (slot, n tile) grid of all slots in bands of band_h slots, as in the dense case.
            // Expert by expert: inside an expert's own grid in bands, an expert of up to eight
            // slots being one band, so that the tiles sharing an L2 form a compact block of few A panels and
            // few B panels of one expert and the tile that holds an expert's last rows runs beside the full
            // tiles that read the same panel of the expert's weights.
            const int tiles_n = (p.n + BN - 1) / BN;
            const int total = total_slots * tiles_n;
            int part = 0, cut = 0;
            int v = place(it, total * (MODE == 5 ? p.split_k : 1), part, cut);
            if (v < 0) return t;
            if (MODE == 5) {                           // partition by partition; the tile's number: its counter and its slots
                t.split_z = __builtin_amdgcn_readfirstlane(v / total);
                v -= t.split_z * total;
                t.sk_first = v;
            }
            const bool by_expert = p.order == ORDER_BY_EXPERT;
            int slot_all = 0, tn = 0;
            if (!by_expert) band_tile(v, total_slots, tiles_n, p.band_h, slot_all, tn);
            int e = 0, found = 0, start = 0, cnt_lo = 0, cnt_hi = 0;
            if (use_table) {
                // the expert whose slots hold slot `key`: the last one that starts at or before it (experts
                // without rows start where the next one starts, and are never the last such)
                const int key = by_expert ? v / tiles_n : slot_all;
                const bool in_lanes = p.num_experts <= 64;
                int cnt = 0;
                if (in_lanes) {
                    cnt = __popcll(__ballot(lane_entry[3] <= key));
                } else {
                    for (int base = 0; base < p.num_experts; base += 64) {
                        const int x = base + lane;
                        const int before = x < p.num_experts ? gtable[x][3] : 0x7FFFFFFF;
                        cnt += __popcll(__ballot(before <= key));
                    }
                }
                cnt = __builtin_amdgcn_readfirstlane(cnt);
                if (cnt > 0) {
                    e = cnt - 1;
                    v4i row;
                    if (in_lanes) {
#pragma unroll
                        for (int i = 0; i < 4; i++) row[i] = __builtin_amdgcn_readlane(lane_entry[i], e);
                    } else {
                        row = gtable[e];
                    }
                    const int s = __builtin_amdgcn_readfirstlane(row[0]), before = __builtin_amdgcn_readfirstlane(row[3]);
                    cnt_lo = __builtin_amdgcn_readfirstlane(row[1]); cnt_hi = __builtin_amdgcn_readfirstlane(row[2]);
                    const int nt = (cnt_hi > cnt_lo) ? (cnt_hi - s + BM - 1) / BM : 0;
                    int slot = slot_all - before;
                    if (by_expert) band_tile(v - before * tiles_n, nt, tiles_n, nt <= 8 ? nt : p.band_h, slot, tn);
                    found = slot < nt;
                    start = s + slot * BM;
                    if constexpr (B_ONCE) t.sk_contrib = nt == once_rows;
                }
            } else {
                int acc_slots = 0;
                for (int x = 0; x < p.num_experts; x++) {
                    int lo = p.row_offsets[x], hi = p.row_offsets[x + 1];
                    lo = lo < 0 ? 0 : lo; hi = hi > p.m ? p.m : hi;
                    int s = lo & ~15;
                    int nt = (hi > lo) ? (hi - s + BM - 1) / BM : 0;
                    if (!found && (by_expert ? v < (acc_slots + nt) * tiles_n : slot_all < acc_slots + nt)) {
                        int slot = slot_all - acc_slots;
                        if (by_expert) band_tile(v - acc_slots * tiles_n, nt, tiles_n, nt <= 8 ? nt : p.band_h, slot, tn);
                        found = 1; e = x; start = s + slot * BM; cnt_lo = lo; cnt_hi = hi;
                        if constexpr (B_ONCE) t.sk_contrib = nt == once_rows;
                    }
                    acc_slots += nt;
                }
            }
            if (!found) return t;                      // uniform for the whole workgroup
            t.valid = 1;
            t.m0 = start; t.n0 = tn * BN;
            if (!take_part(t, part, cut)) return t;
            t.row_lo = cnt_lo; t.row_hi = cnt_hi;
            t.bptr = p.b + (size_t)e * (size_t)p.k * (size_t)p.n;
            t.bsptr = p.bs + (size_t)e * (size_t)(p.k / KBLK) * (size_t)p.nb;
            const int kbt = p.k / KBLK;
            t.kb_begin = MODE == 5 ? t.split_z * p.kb_per_split : 0;
            t.kb_end = MODE == 5 && t.kb_begin + p.kb_per_split < kbt ? t.kb_begin + p.kb_per_split : kbt;
        } else {
            const int tiles_m = (p.m + BM - 1) / BM, tiles_n = (p.n + BN - 1) / BN;
            const int per_split = tiles_m * tiles_n, total = per_split * p.split_k;
            int part = 0, cut = 0;
            const int v = place(it, total, part, cut);
            if (v < 0) return t;
            t.valid = 1;
            if (MODE != 0) t.split_z = v / per_split;
            int tm, tn;
            band_tile(v - t.split_z * per_split, tiles_m, tiles_n, p.band_h, tm, tn);
            if (MODE == 4) t.sk_first = v - t.split_z * per_split;        // the tile's number: its counter and its slots
            t.m0 = tm * BM; t.n0 = tn * BN;
            if (!take_part(t, part, cut)) return t;
            const int kbt = p.k / KBLK;
            t.kb_begin = t.split_z * p.kb_per_split;
            t.kb_end = t.kb_begin + p.kb_per_split;
            t.kb_end = t.kb_end < kbt ? t.kb_end : kbt;
        }
        return t;
    };

    // ---- buffer resources: out-of-range lanes read zeros instead of faulting -------------------
    const uint32_t a_bytes = (uint32_t)p.k * (uint32_t)p.lda;
    const uint32_t b_bytes = (uint32_t)p.k * (uint32_t)p.n;
    __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)p.a, 0, a_bytes, 0x00020000);

    // ---- global -> LDS copy plan of a tile -------------------------------------------------------
    // Wave w, copy q fills the 1 KiB of LDS that starts at chunk slot (q*NWAVES + w)*64; lane l fills
    // slot P = that + l, which holds k row P/CPR, stored chunk P%CPR = logical chunk (P%CPR) ^ swz(k row).
    // The XOR mask of a lane does not depend on q, so a lane's global offset is one constant (k row of
    // copy 0, chunk column) plus a wave-uniform term (k block and q), which travels in an SGPR.
    // A chunk that starts beyond the matrix is pointed at the tile's first chunk (its rows are never
    // stored).  A chunk that starts inside and ends beyond it (m a multiple of 4 but not of 16) runs on
    // into the next k row, or, in the last k row, past the end of the buffer, where the per-dword range
    // check of the buffer load returns zeros: the rows that exist are always read from where they are.
    // Scales of a k block ride along in the tail of the stage: the a_scale row (BM floats, 64 per wave,
    // waves 0 .. BM/64-1) and the b_scale values of the tile's n blocks (the remaining waves, all the same
    // copy to the same place).  Every wave issues exactly one such 4-byte-per-lane copy, with its source
    // and destination in scalar registers: a branch here would split the K loop's straight-line block and
    // the compiler would sink the folds of the first MFMAs below it, away from the MFMAs they are meant
    // to overlap.  With the scales in LDS the K loop has no loads of its own that the compiler would have
    // to order against the output stores of the previous tile.
    constexpr int ROWS_PER_COPY_A = C::NWAVES * 64 / C::CPR_A, ROWS_PER_COPY_B = C::NWAVES * 64 / C::CPR_B;
    // With 12 chunks per k row of B one copy of the workgroup (NWAVES*64 chunks) does not end on a row
    // boundary: a lane's (k row, chunk) then differs from copy to copy and it keeps one offset per copy.
    constexpr bool B_ROWS_WHOLE = (C::NWAVES * 64) % C::CPR_B == 0;
    static_assert(!B_ONCE || B_ROWS_WHOLE);
    constexpr bool A_ROWS_WHOLE = (C::NWAVES * 64) % C::CPR_A == 0;
    constexpr int AS_COPIES = BM / 64;
    static_assert(C::NWAVES > AS_COPIES, "some wave must be left to copy the b_scale values");
    const bool sc_is_b = wave >= AS_COPIES;                       // this wave's scale copy is the b_scale one
    const uint32_t sc_dst = C::A_BYTES + C::B_BYTES + (sc_is_b ? C::AS_AREA : wave * 256);
    const uint32_t sc_kstep = (sc_is_b ? (uint32_t)p.nb : (uint32_t)p.lda) * 4u;
    struct CopyPlan {
        uint32_t a_voff, b_voff, sc_voff;
        uint32_t b_voffq[C::B_LOADS];           // only without B_ROWS_WHOLE
        uint32_t a_voffq[C::A_LOADS];           // only without A_ROWS_WHOLE
        int kb_begin;                           // with B_ONCE, whose tiles begin at block 0: whether b is read past the caches
        __amdgpu_buffer_rsrc_t b_rsrc, sc_rsrc;
    };
    auto copy_plan = [&](const Tile& t) -> CopyPlan {
        CopyPlan c;
        int P = wave * 64 + lane;
        int krow = P / C::CPR_A, ch = stored_to_chunk<C::CPR_A>(P % C::CPR_A, swz_of_krow<C::CPR_A>(krow));
        int col = t.m0 + 16 * ch;
        // A chunk of rows that all lie beyond the matrix, or that all belong to a later expert, is not fetched at
        // all.  Its lanes get an offset at the end of the buffer, for which the range check of the load returns
        // zeros without a memory access: one token row against a 64-row tile then moves one chunk of a per k row
        // instead of four, a tile that holds an expert's last few rows a few instead of sixteen.
        const bool skip = col >= t.row_hi && a_bytes < 0x80000000u;
        col = col < p.lda ? col : t.m0;
        c.a_voff = skip ? a_bytes : (uint32_t)krow * (uint32_t)p.lda + (uint32_t)col;
#pragma unroll
        for (int q = 0; q < C::A_LOADS; q++) {
            c.a_voffq[q] = 0;
            if constexpr (!A_ROWS_WHOLE) {
                const int Pq = q * C::NWAVES * 64 + P;
                const int kr = Pq / C::CPR_A;
                int cl = t.m0 + 16 * stored_to_chunk<C::CPR_A>(Pq % C::CPR_A, swz_of_krow<C::CPR_A>(kr));
                const bool skipq = cl >= t.row_hi && a_bytes < 0x80000000u;
                cl = cl < p.lda ? cl : t.m0;
                c.a_voffq[q] = skipq ? a_bytes : (uint32_t)kr * (uint32_t)p.lda + (uint32_t)cl;
            }
        }
        krow = P / C::CPR_B; ch = stored_to_chunk<C::CPR_B>(P % C::CPR_B, swz_of_krow<C::CPR_B>(krow));
        col = t.n0 + 16 * ch;
        const bool skip_b = col >= t.n_hi && b_bytes < 0x80000000u;   // columns beyond the matrix, or of another part of the tile: not fetched either
        col = col < p.n ? col : t.n0;
        c.b_voff = skip_b ? b_bytes : (uint32_t)krow * (uint32_t)p.n + (uint32_t)col;
#pragma unroll
        for (int q = 0; q < C::B_LOADS; q++) {
            c.b_voffq[q] = 0;
            if constexpr (!B_ROWS_WHOLE) {
                const int Pq = q * C::NWAVES * 64 + P;
                const int kr = Pq / C::CPR_B;
                int cl = t.n0 + 16 * stored_to_chunk<C::CPR_B>(Pq % C::CPR_B, swz_of_krow<C::CPR_B>(kr));
                const bool skipq = cl >= p.n && b_bytes < 0x80000000u;
                cl = cl < p.n ? cl : t.n0;
                c.b_voffq[q] = skipq ? b_bytes : (uint32_t)kr * (uint32_t)p.n + (uint32_t)cl;
            }
        }
        int r = sc_is_b ? t.n0 / 128 + lane : t.m0 + wave * 64 + lane;      // n block or row of a
        const int last = (sc_is_b ? p.nb : p.lda) - 1;
        r = r < last ? r : last;
        c.sc_voff = (uint32_t)r * 4u;
        c.kb_begin = B_ONCE ? __builtin_amdgcn_readfirstlane(t.sk_contrib) : t.kb_begin;
        c.b_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)t.bptr, 0, b_bytes, 0x00020000);
        c.sc_rsrc = __builtin_amdgcn_make_buffer_rsrc(sc_is_b ? (void*)t.bsptr : (void*)p.as, 0,
                                                      sc_is_b ? (uint32_t)(p.k / KBLK) * (uint32_t)p.nb * 4u
                                                              : (uint32_t)(p.k / KBLK) * (uint32_t)p.lda * 4u, 0x00020000);
        return c;
    };
    const uint32_t a_kstep = (uint32_t)KBLK * (uint32_t)p.lda, b_kstep = (uint32_t)KBLK * (uint32_t)p.n;

    // The copies are issued from inline assembly so that the compiler's hazard tracking does not see
    // them: it cannot tell that a copy into one stage never aliases the transposing reads of the other
    // stage and would otherwise make every LDS read wait for all outstanding copies.  Completion is
    // enforced by hand: s_waitcnt vmcnt(0) + workgroup barrier before the first read of a stage.
    const uint32_t lds_base = (uint32_t)(size_t)(__attribute__((address_space(3))) unsigned char*)lds;
    constexpr int NLOADS = C::A_LOADS + C::B_LOADS + 1;     // + the scales
    // the counted waits below name the copies of the blocks that may stay in flight and a tile's output stores; the
    // counter has six bits
    static_assert((NSTAGE - 2) * NLOADS + EPI_STORES <= 63, "vmcnt wait thresholds must fit the counter");
    // copy q (compile-time) of k block `blk` (relative to the tile's first) into `stage`
    auto issue_one = [&](const CopyPlan& cp, int stage, int blk, auto q_tag) {
        constexpr int q = decltype(q_tag)::value;
        const uint32_t sa = lds_base + stage * C::STAGE_BYTES + wave * 1024;
        const uint32_t kb = (uint32_t)((B_ONCE ? 0 : cp.kb_begin) + blk);
        if constexpr (q < C::A_LOADS) {
            if constexpr (A_ROWS_WHOLE)
                copy16_global_to_lds(a_rsrc, sa + q * C::NWAVES * 1024, cp.a_voff, kb * a_kstep + (uint32_t)(q * ROWS_PER_COPY_A) * (uint32_t)p.lda);
            else
                copy16_global_to_lds(a_rsrc, sa + q * C::NWAVES * 1024, cp.a_voffq[q], kb * a_kstep);
        } else if constexpr (q < C::A_LOADS + C::B_LOADS) {
            constexpr int qb = q - C::A_LOADS;
            if constexpr (B_ONCE)
                copy16_global_to_lds_once(cp.b_rsrc, sa + C::A_BYTES + qb * C::NWAVES * 1024, cp.b_voff, kb * b_kstep + (uint32_t)(qb * ROWS_PER_COPY_B) * (uint32_t)p.n, (uint32_t)cp.kb_begin);
            else if constexpr (B_ROWS_WHOLE)
                copy16_global_to_lds(cp.b_rsrc, sa + C::A_BYTES + qb * C::NWAVES * 1024, cp.b_voff, kb * b_kstep + (uint32_t)(qb * ROWS_PER_COPY_B) * (uint32_t)p.n);
            else
                copy16_global_to_lds(cp.b_rsrc, sa + C::A_BYTES + qb * C::NWAVES * 1024, cp.b_voffq[qb], kb * b_kstep);
        } else {
            copy4_global_to_lds(cp.sc_rsrc, lds_base + stage * C::STAGE_BYTES + sc_dst, cp.sc_voff, kb * sc_kstep);
        }
    };
    auto issue_all = [&](const CopyPlan& cp, int stage, int blk) {
        [&]<int... Q>(std::integer_sequence<int, Q...>) {
            (issue_one(cp, stage, blk, std::integral_constant<int, Q>{}), ...);
        }(std::make_integer_sequence<int, NLOADS>{});
    };

    // blocks 0 .. NSTAGE-2 of a tile, as many as it has
    auto issue_first = [&](const CopyPlan& cp, int blocks) {
        issue_all(cp, 0, 0);
#pragma unroll
        for (int s = 1; s < NSTAGE - 1; s++) if (blocks > s) issue_all(cp, s, s);
    };

    // ---- per-lane LDS read addresses -----------------------------------------------------------
    // transposing read j of a 16-row tile: k rows 32j + 8g + (i16>>1), byte half (i16&1)
    const int krow_lane = 8 * g + (i16 >> 1);
    const int swz_a = swz_of_krow<C::CPR_A>(krow_lane);     // independent of j (32j is a multiple of 16)
    const int swz_b = swz_of_krow<C::CPR_B>(krow_lane);
    const int a_lane_off = krow_lane * BM + (i16 & 1) * 8;
    const int b_lane_off = C::A_BYTES + krow_lane * BN + (i16 & 1) * 8;
    const int a_chunk0 = wave_m * (WM / 16), b_chunk0 = wave_n * (WN / 16);

    auto read_a = [&](v8i& dst, int t, const unsigned char* sbase) {
        const unsigned char* q = sbase + a_lane_off + (chunk_to_stored<C::CPR_A>(a_chunk0 + t, swz_a) << 4);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            v2i x = __builtin_amdgcn_ds_read_tr8_b64_v2i32(LDS_V2I(q + j * 32 * BM));
            dst[2 * j] = x[0]; dst[2 * j + 1] = x[1];
        }
    };
    auto read_b = [&](v8i& dst, int u, const unsigned char* sbase) {
        const unsigned char* q = sbase + b_lane_off + (chunk_to_stored<C::CPR_B>(b_chunk0 + u, swz_b) << 4);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            v2i x = __builtin_amdgcn_ds_read_tr8_b64_v2i32(LDS_V2I(q + j * 32 * BN));
            dst[2 * j] = x[0]; dst[2 * j + 1] = x[1];
        }
    };

    const int as_lane_off = C::A_BYTES + C::B_BYTES + (wave_m * WM + i16) * 4;
    const int bs_base = C::A_BYTES + C::B_BYTES + C::AS_AREA;     // slot i: b_scale of n block n0/128 + i

    Tile cur = pick_tile(0);
    if (!cur.valid) return;
    CopyPlan cp = copy_plan(cur);
    bool prefetched = false;                // the first blocks of `cur` are already on their way
    if (TAILS && cur.kb_end > cur.kb_begin) {
        issue_first(cp, cur.kb_end - cur.kb_begin);
        prefetched = true;
    }

    // ---- rows of a that are not a multiple of four, columns of b that are not ------------------------
    // The buffer of a ends on a dword boundary (K is a multiple of 128), but with lda % 4 != 0 the copies
    // fetch its last one to three bytes in dwords that start inside and end beyond it; the range check
    // of a buffer load works on whole dwords and hands back zeros for those.  Every other byte of a
    // arrives intact (a dword that crosses the end of a k row just runs on into the next one).  The
    // workgroup whose tile holds those bytes writes them into LDS itself once the last K block has
    // landed: they are among the last four bytes of a.  The same holds for b with n % 4 != 0.
    // Each is written by the wave whose copy brought the bytes around it, between its wait for the copy and the barrier that
    // publishes the block: lane l < 6 of every wave has one candidate, a's for l < 3, in patch_at, worked out at a tile's
    // start while the first copies are on their way; a lane whose candidate is not lost, not in the tile or another
    // wave's writes to a byte of the stage that nobody reads.  So the store has no condition: a branch at this place, in the middle of
    // a K block's step sequence, makes the compiler move the folds of the MFMAs before it below it, which costs some thirty registers.
    // (Worked out ahead of the first copies, from vector loads, six bytes one after the other behind the barrier and with a second
    // barrier, the repair was 0.4 to 0.9 us of every call that takes this instantiation, and the pieces of c below, stored by all
    // waves, 0.1 to 1.1: 1023 x 3141 x 2048 in 128x128 19.2 -> 18.1 us, 250 x 4096 x 1792 12.5 -> 11.5, 130 x 1000 x 128 5.6 -> 4.4, in
    // 64x64 4.2 -> 3.5; 45 products on five tiles 0.88 of the time in the geometric mean.)
    const bool a_tail = TAILS && (p.lda & 3) != 0 && p.k > 0;
    const bool b_tail = TAILS && (p.n & 3) != 0 && p.k > 0;
    [[maybe_unused]] uint32_t patch_at = 0;                       // bits 0-23: the place in the stage, bits 24-31: the byte
    static_assert(C::STAGE_BYTES <= 1 << 24);
    [[maybe_unused]] auto plan_patch = [&](const Tile& t) {
        const bool of_b = lane >= 3;
        const uint32_t back = 3u - (uint32_t)(of_b ? lane - 3 : lane) % 3u;
        const uint32_t cand = tail_candidate(back, (uint32_t)(of_b ? p.n : p.lda), (uint32_t)p.k);
        const int xt = (int)(cand & 0x1FFFFFFFu) - (of_b ? t.n0 : t.m0);                // row / column inside the tile
        const int kl = KBLK - 3 + (int)((cand >> 29) & 3u);                             // k row inside the last block
        const int cpr = of_b ? C::CPR_B : C::CPR_A;
        const int stored = of_b ? chunk_to_stored<C::CPR_B>((xt >> 4) & 15, swz_of_krow<C::CPR_B>(kl)) : chunk_to_stored<C::CPR_A>((xt >> 4) & 15, swz_of_krow<C::CPR_A>(kl));
        const int slot = kl * cpr + stored;                                             // of 16 bytes; 64 of them are a wave's copy
        const bool mine = lane < 6 && (of_b ? b_tail : a_tail) && (cand >> 31) != 0 && t.kb_end * KBLK == p.k
                          && xt >= 0 && xt < (of_b ? BN : BM) && (slot >> 6) % C::NWAVES == wave;
        uint32_t a_last = 0, b_last = 0;
        if (a_tail) a_last = load_last_dword(p.a + a_bytes);
        if (b_tail) b_last = load_last_dword(t.bptr + b_bytes);                         // grouped: every expert's matrix has last bytes of its own
        const uint32_t byte = (of_b ? b_last : a_last) >> (8u * (4u - back));
        patch_at = (uint32_t)(mine ? (of_b ? C::A_BYTES : 0) + slot * 16 + (xt & 15) : C::STAGE_BYTES - 1) | byte << 24;
    };
    // stage: the tile's last K block, which this wave's copies have just reached
    [[maybe_unused]] auto patch = [&](int stage) { *(volatile unsigned char*)(lds + stage * C::STAGE_BYTES + (patch_at & 0xFFFFFFu)) = (unsigned char)(patch_at >> 24); };

    bool stores_behind = false;             // ... and this wave's output stores of the previous tile were issued after it
    for (int it = 0;; it++) {
    const int m0 = cur.m0, n0 = cur.n0, kb_begin = cur.kb_begin, kb_end = cur.kb_end, split_z = cur.split_z;
    const int row_lo = cur.row_lo, row_hi = cur.row_hi;
    [[maybe_unused]] const int sk_contrib = cur.sk_contrib, sk_first = cur.sk_first;
    if constexpr (TAILS) plan_patch(cur);
    // a_scale: lane's output row of m-tile t is tile row wave_m*WM + 16t + i16, read from the stage's
    // copy of the a_scale row.
    // does any element of this wave's tile get stored?  (rows of the expert / matrix, columns of the matrix)
    const bool wave_active = __builtin_amdgcn_readfirstlane((m0 + wave_m * WM < row_hi && m0 + wave_m * WM + WM > row_lo &&
                                                             n0 + wave_n * WN < cur.n_hi) ? 1 : 0) != 0;
    // b_scale of the wave's n tiles: slot bs_off for n tiles [0, ub), the next slot for [ub, NT)
    const int wave_col = (BN % 128 != 0 ? (n0 & 127) : 0) + wave_n * WN;               // from the start of the tile's first n block
    const int bs_off = bs_base + (wave_col >> 7) * 4;
    const int ub = C::SPLIT_SCALES ? (128 - (wave_col & 127)) >> 4 : C::NT;

    v4f acc[C::MT][C::NT];
#pragma unroll
    for (int t = 0; t < C::MT; t++)
#pragma unroll
        for (int u = 0; u < C::NT; u++) acc[t][u] = (v4f){0.f, 0.f, 0.f, 0.f};

    const int nkb = kb_end - kb_begin;
    if (nkb > 0) {
        constexpr int STEPS = C::MT * C::NT;
        constexpr int LAG = 3, RING = 4;      // fold the result of step s-LAG while step s runs
        // Copies of block j+2 start right behind the barrier of block j (NL_LATE of them, one per
        // trailing step) and continue one every DMA_EVERY steps of block j+1: a burst would block this
        // wave's instruction issue until the texture unit has taken it, and the MFMAs queued behind.
        constexpr int NL_LATE = C::MT < 2 ? C::MT : 2;
        constexpr int NL_EARLY = NLOADS - NL_LATE;
        // (the 192-wide tile is the exception, measured: one copy per step gives it 0.92 us per K block on
        // one CU against 1.02, while the 256-wide tile loses 4 % that way)
        constexpr int DMA_EVERY = BN == 192 ? 1 : ((STEPS - C::MT) / NL_EARLY >= 2 ? 2 : 1), DMA_FIRST = DMA_EVERY - 1;
        // (a small wave tile has fewer steps before the barrier than copies: several go into one step)
        constexpr int DMA_PER_STEP = NL_EARLY * DMA_EVERY <= STEPS - C::MT ? 1 : (NL_EARLY + STEPS - C::MT - 1) / (STEPS - C::MT);

        // ---- prologue: blocks 0 .. NSTAGE-2 -> stages 0 .. NSTAGE-2 (unless the previous tile already
        //      sent them), wait for block 0; first copies of block NSTAGE-1 -> the last stage.  The
        //      barrier also ends the previous tile's use of the last stage as the staging area of its
        //      output ----
        // The vector memory counter retires loads and stores in the order they were issued.  If block 0
        // was sent ahead of the previous tile's NSTORES output stores, "at most NSTORES outstanding" means
        // the block has landed, and the stores are left to finish under the first K block.  With more than
        // two stages the next blocks (NLOADS copies each) sit between block 0 and the stores.
        if (!prefetched) issue_first(cp, nkb);
        {
            const bool sb = prefetched && stores_behind;
            const int behind = (nkb < NSTAGE - 1 ? nkb : NSTAGE - 1) - 1;       // blocks sent after block 0
            [&]<int... I>(std::integer_sequence<int, I...>) {
                ((behind == I ? (sb ? wait_vmcnt<I * NLOADS + EPI_STORES>() : wait_vmcnt<I * NLOADS>()) : (void)0), ...);
            }(std::make_integer_sequence<int, NSTAGE - 1>{});
        }
        if (TAILS && nkb == 1) patch(0);
        __syncthreads();
        if (nkb > NSTAGE - 1) {
            [&]<int... Q>(std::integer_sequence<int, Q...>) {
                (issue_one(cp, NSTAGE - 1, NSTAGE - 1, std::integral_constant<int, Q>{}), ...);
            }(std::make_integer_sequence<int, NL_LATE>{});
        }

        // A block's scales are read ahead of its first operands, behind the barrier that publishes it, and the operands in the
        // order in which they are multiplied, here as in the loop: an LDS wait names how many younger reads may still be out, and
        // where two ways lead into the loop the compiler takes the lower number.  (Read at the block's start, the scales are
        // the youngest, and the first MFMA waits for every read there is.  us, at the start and ahead: 1024 x 1536 x 7168 in 128x128 of eight
        // waves 29.2 and 29.0, of four 46.0 and 45.0, in 64x128 24.1 and 23.2; 512 x 1024 x 2048 in 64x128 8.76 and 8.40, in 64x64 7.80 and 7.33; in
        // 64x256 128 x 8192 x 4096 20.75 and 20.41, but 1024 x 1536 x 7168 32.8 and 33.3; in 256x128 with three stages 1024 x 1536 x 7168 44.8 and 45.8,
        // but 4847 x 480 x 7936 in three partitions 45.1 and 38.0.)
        // Not with waves of 24 tiles and more, whose registers are full: 1000 tokens to 4 of 32 experts, 4096 x 2048, 70.0 us as it is, 73.5
        // ahead in 256x256; 1024 x 1536 x 7168 59.6 and 60.1 in 256x192.  Nor in the summed K split of 192x192 on aligned rows, where the two
        // registers that it spills are reloaded ahead of the loop and waited for inside it, with counts that know nothing of the copies and
        // wait for those as well: 4096 x 2112 x 7168 in two partitions 79.3 at the start, 95.2 ahead.  (With TAILS it spills either way:
        // 4523 x 952 x 6016 53.5 and 51.5.)
        constexpr bool SCALES_AHEAD = STEPS < 24 && !(STEPS >= 18 && SUMMED && !TAILS);
        v8i areg[C::MT], breg[2];
        float asv[C::MT], bsv, bsv1;
        auto read_scales = [&](const unsigned char* sb) {
#pragma unroll
            for (int t = 0; t < C::MT; t++) asv[t] = *(const float*)(sb + as_lane_off + t * 64);
            bsv = *(const float*)(sb + bs_off);
            bsv1 = C::SPLIT_SCALES ? *(const float*)(sb + bs_off + 4) : 0.f;
            __builtin_amdgcn_sched_barrier(0);
        };
        if (wave_active) {
            if (SCALES_AHEAD) read_scales(lds);
            read_a(areg[0], 0, lds);
            __builtin_amdgcn_sched_barrier(0);
            read_b(breg[0], 0, lds);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 1; t < C::MT; t++) { read_a(areg[t], t, lds); __builtin_amdgcn_sched_barrier(0); }
        }

        // All K blocks of the tile.  UB: the wave's n tiles [UB, NT) belong to the next b_scale block
        // (UB = NT: none does).
        auto run_blocks = [&](auto ub_tag) {
        constexpr int UB = decltype(ub_tag)::value;
        // One K block (index j, in stage j&1).  The flags are compile-time so that the step sequence
        // is one straight-line block for the instruction scheduler.
        // Block j lives in stage j % NSTAGE.  While it is multiplied, the rest of block j+NSTAGE-1 is
        // copied into the stage that the barrier of block j-1 freed; behind the barrier of block j the
        // first copies of block j+NSTAGE go into the stage just read.  With two stages a copy has one
        // block's time to land, with three stages two, with four three.
        auto k_block = [&](int j, auto rem_tag) {
            constexpr int REM = decltype(rem_tag)::value;                      // blocks behind block j; NSTAGE stands for that many or more
            constexpr bool HAS_NEXT = REM >= 1;                                // block j+1 exists
            constexpr bool HAS_EARLY = REM >= NSTAGE - 1;                      // block j+NSTAGE-1 exists
            constexpr bool HAS_LATE = REM >= NSTAGE;                           // block j+NSTAGE exists
            constexpr bool LANDS_LAST = REM == 1;                              // block j+1 is the tile's last
            const int cur_stage = NSTAGE == 2 ? (j & 1) : j % NSTAGE;
            const int next_stage = cur_stage + 1 == NSTAGE ? 0 : cur_stage + 1;
            const int early_stage = NSTAGE == 2 ? next_stage : (cur_stage == 0 ? NSTAGE - 1 : cur_stage - 1);
            // what must have landed at the barrier is block j+1; the copies of the blocks behind it (j+2 up to
            // j+NSTAGE-1, as far as they exist) were all issued after it and may stay in flight
            auto wait_next_block = [&]() {
                constexpr int BEHIND = (REM < NSTAGE - 1 ? REM : NSTAGE - 1) - 1;
                wait_vmcnt_lgkm0<(BEHIND > 0 ? BEHIND : 0) * NLOADS>();
            };
            if (!wave_active) {
                // none of this wave's rows is stored: it only does its share of the copies, in the
                // same order and around the same single barrier as the waves that compute
                if constexpr (HAS_EARLY) {
                    [&]<int... Q>(std::integer_sequence<int, Q...>) {
                        (issue_one(cp, early_stage, j + NSTAGE - 1, std::integral_constant<int, NL_LATE + Q>{}), ...);
                    }(std::make_integer_sequence<int, NL_EARLY>{});
                }
                wait_next_block();
                if constexpr (TAILS && LANDS_LAST) patch(next_stage);
                __syncthreads();
                if constexpr (HAS_LATE) {
                    [&]<int... Q>(std::integer_sequence<int, Q...>) {
                        (issue_one(cp, cur_stage, j + NSTAGE, std::integral_constant<int, Q>{}), ...);
                    }(std::make_integer_sequence<int, NL_LATE>{});
                }
                return;
            }
            const unsigned char* sbase = lds + cur_stage * C::STAGE_BYTES;
            const unsigned char* snext = lds + next_stage * C::STAGE_BYTES;
            float sc[C::MT], sc1[C::MT];
            // the step that works out the block's scales: the one that folds first, but before the next block's are read
            constexpr int BARRIER_STEP = STEPS - C::MT, SCALE_STEP = LAG < BARRIER_STEP ? LAG : BARRIER_STEP - 1;
            if constexpr (!SCALES_AHEAD) read_scales(sbase);
            v4f ring[RING];
            auto step = [&](auto s_tag) {
                constexpr int s = decltype(s_tag)::value;
                if constexpr (s < STEPS) {
                    constexpr int u = s / C::MT, t = s % C::MT;
                    if constexpr (HAS_EARLY && DMA_PER_STEP == 1) {
                        if constexpr (s % DMA_EVERY == DMA_FIRST && s / DMA_EVERY < NL_EARLY)
                            issue_one(cp, early_stage, j + NSTAGE - 1, std::integral_constant<int, NL_LATE + s / DMA_EVERY>{});
                    } else if constexpr (HAS_EARLY && s * DMA_PER_STEP < NL_EARLY) {
                        constexpr int FIRST = s * DMA_PER_STEP, COUNT = NL_EARLY - FIRST < DMA_PER_STEP ? NL_EARLY - FIRST : DMA_PER_STEP;
                        [&]<int... Q>(std::integer_sequence<int, Q...>) {
                            (issue_one(cp, early_stage, j + NSTAGE - 1, std::integral_constant<int, NL_LATE + FIRST + Q>{}), ...);
                        }(std::make_integer_sequence<int, COUNT>{});
                    }
                    if constexpr (t == 0 && u + 1 < C::NT) read_b(breg[(u + 1) & 1], u + 1, sbase);
                    if constexpr (t == 0 && u == C::NT - 1) {
                        // All reads of this stage are issued.  Wait for them and for this wave's part
                        // of the next block, then meet the other waves: after the barrier the next
                        // block is complete in the other stage and this stage may be overwritten.
                        wait_next_block();
                        if constexpr (TAILS && LANDS_LAST) patch(next_stage);
                        __syncthreads();
                        if constexpr (HAS_NEXT && SCALES_AHEAD) read_scales(snext);
                    }
                    const v4f z = {0.f, 0.f, 0.f, 0.f};
                    ring[s % RING] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(breg[u & 1], areg[t], z, 0, 0, 0, 0, 0, 0);
                    if constexpr (u == C::NT - 1 && HAS_NEXT) {
                        // operands of the next block, fetched while the last MFMAs of this one run
                        read_a(areg[t], t, snext);
                        if constexpr (t == 0) read_b(breg[0], 0, snext);
                    }
                    if constexpr (u == C::NT - 1 && HAS_LATE && t < NL_LATE)
                        issue_one(cp, cur_stage, j + NSTAGE, std::integral_constant<int, t>{});
                }
                if constexpr (s == SCALE_STEP) {
#pragma unroll
                    for (int t = 0; t < C::MT; t++) {
                        sc[t] = asv[t] * bsv;
                        sc1[t] = UB < C::NT ? asv[t] * bsv1 : 0.f;
                    }
                }
                if constexpr (s >= LAG) {
                    constexpr int sp = s - LAG, u = sp / C::MT, t = sp % C::MT;
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[t][u][r] = __builtin_fmaf(ring[sp % RING][r], u < UB ? sc[t] : sc1[t], acc[t][u][r]);
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            [&]<int... S>(std::integer_sequence<int, S...>) {
                (step(std::integral_constant<int, S>{}), ...);
            }(std::make_integer_sequence<int, STEPS + LAG>{});
        };

        int j = 0;
        for (; j + NSTAGE < nkb; j++) k_block(j, std::integral_constant<int, NSTAGE>{});
        [&]<int... R>(std::integer_sequence<int, R...>) {
            ((j + (NSTAGE - 1 - R) < nkb ? (k_block(j, std::integral_constant<int, NSTAGE - 1 - R>{}), (void)j++) : (void)0), ...);
        }(std::make_integer_sequence<int, NSTAGE - 1>{});
        k_block(j, std::integral_constant<int, 0>{});
        };   // run_blocks
        if constexpr (C::SPLIT_SCALES) {
            // 96-column wave tiles of a 192-column tile start 0, 96, 64 or 160 columns into a block
            if (ub == 2) run_blocks(std::integral_constant<int, 2>{});
            else if (ub == 4) run_blocks(std::integral_constant<int, 4>{});
            else run_blocks(std::integral_constant<int, C::NT>{});
        } else {
            run_blocks(std::integral_constant<int, C::NT>{});
        }
    }

    else if (it > 0) {
        __syncthreads();                    // nothing to multiply: still let the previous tile's staging reads finish
    }

    // ---- the next tile's first K blocks (all stages but the last) start now: after the last barrier
    //      above no wave reads a stage any more, and the output below is staged in the last stage only ----
    Tile nxt = pick_tile(it + 1);
    CopyPlan ncp = cp;
    prefetched = false;
    if (nxt.valid) {
        ncp = copy_plan(nxt);
        if (nxt.kb_end > nxt.kb_begin) {
            issue_first(ncp, nxt.kb_end - nxt.kb_begin);
            prefetched = true;
        }
    }

    // ---- K blocks dealt to the workgroups: partial tiles travel through the workspace ---------------
    // Partial tiles are written and read with agent-scope accesses (sc1: written through to, and read from,
    // the memory side of the eight L2s), in the order of the lanes: the two sides run the same tile shape, so
    // accumulator (t, u) of wave w is the 1 KiB piece number w*MT*NT + t*NT + u of the slot.
    bool store_output = true;
    [[maybe_unused]] uint32_t out_parts = 1;                 // SHARED_SUM: the parts of the tile that this workgroup writes
    if constexpr (MODE == 3) {
        constexpr uint32_t SLOT_BYTES = (uint32_t)BM * (uint32_t)BN * 4u;
        constexpr int NG = C::MT * C::NT;
        constexpr int AUX_AGENT = 16;                                           // sc1
        unsigned char* const ws_base = (unsigned char*)p.ws;
        unsigned long long* const flags = (unsigned long long*)(ws_base + StreamK::FLAGS_OFF);
        unsigned char* const slots = ws_base + StreamK::SLOTS_OFF;
        if (sk_contrib) {
            store_output = false;
            if (wave_active) {
                // (the accumulators are next written after the wait below: nothing follows these stores closely)
                __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)(slots + (size_t)sk_self * SLOT_BYTES), 0, SLOT_BYTES, 0x00020000);
                const uint32_t voff = (uint32_t)(wave * NG) * 1024u + (uint32_t)lane * 16u;
#pragma unroll
                for (int t = 0; t < C::MT; t++)
#pragma unroll
                    for (int u = 0; u < C::NT; u++)
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, acc[t][u]), rs, voff + (uint32_t)(t * C::NT + u) * 1024u, 0, AUX_AGENT);
            }
            // A store with sc1 is written through to the agent's point of coherence and is counted by vmcnt
            // until it is acknowledged from there, so after this wait every wave's part of the tile can be
            // seen by any CU that reads it with sc1; the barrier then lets one lane raise the flag for all.
            // (An agent-scope release fence in its place writes the whole L2 back once per wave: 4096 x 2112
            // x 7168 took 131 us with it against 81 us, 64 x 18432 x 7168 76 us against 30 us.)
            wait_vmcnt<0>();
            __syncthreads();
            if (tid == 0) __hip_atomic_store(&flags[sk_self], p.sk_nonce, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else if (sk_first >= 0) {
            // The tile's owner: wait, a bounded number of polls, for the flags of the workgroups that hold the
            // tile's earlier K blocks (one lane per flag, all polled together), take the flags down again (so
            // that a replay of the same launch starts clean), then add the partial tiles to the accumulators in
            // ascending order of K: ((own + P_first) + P_next) + ...  A wait that gives up leaves the status
            // word set and the kernel runs on to its end with whatever the slots hold.
            if (wave == 0) {
                bool ok = p.sk_spin >= 0;
                for (int base = sk_first; ok && base < sk_self; base += 64) {
                    const int u = base + lane;
                    const bool mine = u < sk_self;
                    int spins = p.sk_spin;
                    for (;;) {
                        const unsigned long long f = mine ? __hip_atomic_load(&flags[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : p.sk_nonce;
                        if (__ballot(f != p.sk_nonce) == 0) break;
                        if (--spins < 0) { ok = false; break; }
                        __builtin_amdgcn_s_sleep(2);
                    }
                    if (ok && mine) __hip_atomic_store(&flags[u], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                if (!ok && lane == 0) __hip_atomic_store((unsigned int*)ws_base, StreamK::STATUS_TIMEOUT, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            __syncthreads();
            if (wave_active) {
                // loads in flight at a time: what the registers beside the accumulators hold
                constexpr int BATCH = NG <= 8 ? NG : (NG % 4 == 0 ? 4 : (NG % 3 == 0 ? 3 : 1));
                __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)slots, 0, (uint32_t)gridDim.x * SLOT_BYTES, 0x00020000);
                const uint32_t voff = (uint32_t)(wave * NG) * 1024u + (uint32_t)lane * 16u;
#pragma unroll
                for (int base = 0; base < NG; base += BATCH) {
#pragma unroll 2
                    for (int u = sk_first; u < sk_self; u++) {
                        const uint32_t soff = (uint32_t)u * SLOT_BYTES + (uint32_t)base * 1024u;
                        v4f part[BATCH];
#pragma unroll
                        for (int i = 0; i < BATCH; i++)
                            part[i] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rs, voff, soff + i * 1024u, AUX_AGENT));
#pragma unroll
                        for (int i = 0; i < BATCH; i++)
                            acc[(base + i) / C::NT][(base + i) % C::NT] += part[i];
                    }
                    __builtin_amdgcn_sched_barrier(0);      // the registers hold the whole tile already: one batch at a time
                }
            }
        }
    } else if constexpr (SUMMED) {
        // K split in one launch, nobody waits: every workgroup leaves its partial tile in the slot
        // (tile, K partition) and then counts itself in at the tile's counter; the one that finds all others
        // counted in before it adds the partial tiles in ascending order of K - ((P0 + P1) + P2) + ..., its own
        // from the registers, the order of the separate reduce kernel - and writes the bf16 tile.  The counter
        // carries the call's tag in its upper 48 bits, so whatever an earlier use of the workspace left there
        // counts as zero; the last workgroup puts it back to zero for a replay of the same launch.
        constexpr uint32_t SLOT_BYTES = (uint32_t)BM * (uint32_t)BN * 4u;
        constexpr int NG = C::MT * C::NT;
        constexpr int AUX_AGENT = 16;                                           // sc1
        __shared__ int last_in, all_in;
        unsigned char* const ws_base = (unsigned char*)p.ws;
        unsigned long long* const counters = (unsigned long long*)(ws_base + StreamK::FLAGS_OFF);
        unsigned char* const tile_slots = ws_base + StreamK::SLOTS_OFF + (size_t)sk_first * (size_t)p.split_k * SLOT_BYTES;
        const uint32_t voff = (uint32_t)(wave * NG) * 1024u + (uint32_t)lane * 16u;
        // Lanes whose row or columns lie outside the matrix neither store nor load their piece (an offset beyond the
        // slot drops a store and makes a load return zeros): one row against 18432 columns leaves 1 KB per workgroup
        // in the workspace instead of 32 KB (31.6 us with every lane storing, against 29.1 as two launches).
        uint32_t rows_in = 0, cols_in = 0;                 // bit t: the lane's row of m tile t exists; bit u: its columns of n tile u
#pragma unroll
        for (int t = 0; t < C::MT; t++) rows_in |= (m0 + wave_m * WM + 16 * t + i16 < row_hi ? 1u : 0u) << t;
#pragma unroll
        for (int u = 0; u < C::NT; u++) cols_in |= (n0 + wave_n * WN + 16 * u + 4 * g < p.n ? 1u : 0u) << u;
        auto piece = [&](int x) -> uint32_t {               // x = t * NT + u, a compile-time number at every use
            return ((rows_in >> (x / C::NT)) & (cols_in >> (x % C::NT)) & 1u) ? voff + (uint32_t)x * 1024u : 0xFFFFFFFFu;
        };
        // (keeps the offsets of all pieces from being worked out ahead of the branches and held in registers)
        [[maybe_unused]] auto here = [](uint32_t& rows, uint32_t& cols) { asm volatile("" : "+v"(rows), "+v"(cols)); };
        auto slot_of = [&](int z) { return __builtin_amdgcn_make_buffer_rsrc((void*)(tile_slots + (size_t)z * SLOT_BYTES), 0, SLOT_BYTES, 0x00020000); };
        if constexpr (SHARED_SUM) {
            // The sum is shared out: of every wave's accumulators partition z adds the z-th S-th part and writes that part of c,
            // so a workgroup stores and loads (S-1)/S of a tile, all of a tile's workgroups at once, where below every one
            // stores a tile and then one loads S-1.  Each raises a flag of its own - one store, no exchange that S workgroups
            // queue for - and polls all S of them with one load.  What is left is a chain of round trips to the point of
            // coherence: stores acknowledged, flag and poll, loads.  Measured against the sum by one workgroup (us): 1024 x 1536 x
            // 7168 in two 21.0 / 21.4, 64 x 18432 x 7168 in three 33.0 / 33.7, 128 x 7168 x 7168 in four 16.3 / 18.4, 64 x 4096 x 7168 in
            // eight 12.4 / 19.2 (128x128 tile, two launches 13.4).  With the partitions of a tile on one XCD, so that the parts travel
            // through its L2, the chain is shorter and the K loops read more: 21.7 and 18.2 on the first and the third.
            // Nobody depends on another workgroup being on the chip: one that has not seen all flags within a bounded number
            // of polls stores its own part too, marks it as left and moves on.  Whoever sees all flags up, with its own known
            // to be visible, claims and adds the parts that are marked by then; one that marks its part looks at the flags
            // again afterwards, so the part of a workgroup that leaves as the last one arrives is claimed by one of the two.
            // Flags: the call's tag and 1 = stored, 2 = its own part left, 3 = that part claimed.  They are not taken down, so
            // the launcher does this only where the tag is new on every run (not in a captured launch) and every pair of tile
            // and partition has a workgroup of its own.
            constexpr auto owner = [](int x, int S) constexpr { return x * S / NG; };
            const unsigned long long tag = (p.sk_nonce | 0x10000ull) & ~0xFFFFull;           // never zero
            auto shared = [&]<int S>() {
                constexpr uint32_t ALL = (1u << S) - 1u;
                unsigned long long* const flags = counters + sk_first * S;
                const uint32_t mine = 1u << split_z;
                auto store_parts = [&](uint32_t parts) {
                    const __amdgpu_buffer_rsrc_t rs = slot_of(split_z);
                    here(rows_in, cols_in);
#pragma unroll
                    for (int x = 0; x < NG; x++)
                        if ((parts >> owner(x, S)) & 1u) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, acc[x / C::NT][x % C::NT]), rs, piece(x), 0, AUX_AGENT);
                };
                auto sum_part = [&]<int Z>() {
                    constexpr int X0 = (Z * NG + S - 1) / S, X1 = ((Z + 1) * NG + S - 1) / S, N = X1 - X0;      // owner(x) == Z for x in [X0, X1)
                    if constexpr (N > 0) {
                        here(rows_in, cols_in);
                        v4f part[S - 1][N];                                          // the other partitions, ascending
#pragma unroll
                        for (int j = 0; j < S - 1; j++) {
                            const __amdgpu_buffer_rsrc_t rs = slot_of(j + (j >= split_z ? 1 : 0));
#pragma unroll
                            for (int i = 0; i < N; i++) part[j][i] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rs, piece(X0 + i), 0, AUX_AGENT));
                        }
#pragma unroll
                        for (int i = 0; i < N; i++) {
                            v4f& own = acc[(X0 + i) / C::NT][(X0 + i) % C::NT];
                            v4f sum = part[0][i];
                            if (split_z == 0) sum = own + sum;                        // (the same bits as sum + own)
#pragma unroll
                            for (int j = 1; j < S - 1; j++) {
                                if (j == split_z) sum += own;
                                sum += part[j][i];
                            }
                            if (split_z == S - 1) sum += own;
                            own = sum;
                        }
                    }
                };
                auto sum_parts = [&](uint32_t parts) {
                    if (wave_active)
                        [&]<int... Z>(std::integer_sequence<int, Z...>) {
                            (((parts >> Z) & 1u ? sum_part.template operator()<Z>() : (void)0), ...);
                        }(std::make_integer_sequence<int, S>{});
                };
                auto read_flags = [&]() -> unsigned long long { return lane < S ? __hip_atomic_load(&flags[lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : tag | 1ull; };
                auto claim = [&](unsigned long long f) -> uint32_t {                  // the marked parts that this workgroup takes
                    unsigned long long left = tag | 2ull;
                    const bool got = lane < S && f == left && __hip_atomic_compare_exchange_strong(&flags[lane], &left, tag | 3ull, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    return (uint32_t)__ballot(got);
                };
                if (wave_active) store_parts(ALL & ~mine);
                wait_vmcnt<0>();                                                      // acknowledged from the agent's point of coherence
                __syncthreads();
                if (wave == 0) {
                    if (lane == 0) __hip_atomic_store(&flags[split_z], tag | 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    bool all = false;
                    for (int polls = p.sk_spin;; polls--) {
                        all = __ballot((read_flags() & ~0xFFFFull) != tag) == 0;
                        if (all || polls <= 0) break;
                        __builtin_amdgcn_s_sleep(1);
                    }
                    if (lane == 0) all_in = all ? 1 : 0;
                }
                __syncthreads();
                const bool all = __builtin_amdgcn_readfirstlane(all_in) != 0;
                if (!all) {
                    if (wave_active) store_parts(mine);
                    wait_vmcnt<0>();
                    __syncthreads();
                    if (wave == 0 && lane == 0) __hip_atomic_store(&flags[split_z], tag | 2ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                unsigned long long f = 0;
                if (wave == 0) {
                    wait_vmcnt<0>();                                                  // this workgroup's flag or mark is visible
                    f = read_flags();
                }
                if (all) sum_parts(mine);
                if (wave == 0) {
                    const uint32_t got = __ballot((f & ~0xFFFFull) != tag) == 0 ? claim(f) : 0u;
                    if (lane == 0) last_in = (int)got;
                }
                __syncthreads();
                const uint32_t taken = (uint32_t)__builtin_amdgcn_readfirstlane(last_in);
                if (taken) sum_parts(taken);
                out_parts = (all ? mine : 0u) | taken;
            };
            switch (p.split_k) {
                case 2: if constexpr (shares_from<BM, BN>() <= 2) shared.template operator()<2>(); break;
                case 3: if constexpr (shares_from<BM, BN>() <= 3) shared.template operator()<3>(); break;
                case 4: shared.template operator()<4>(); break;
                case 6: shared.template operator()<6>(); break;
                default: shared.template operator()<8>(); break;
            }
            store_output = out_parts != 0;
        } else {
        // (the counter is read ahead of the stores: the value only seeds the exchange below, which finds out if it is stale)
        unsigned long long seen = 0;
        if (tid == 0) seen = __hip_atomic_load(&counters[sk_first], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (wave_active) {
            __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)(tile_slots + (size_t)split_z * SLOT_BYTES), 0, SLOT_BYTES, 0x00020000);
#pragma unroll
            for (int t = 0; t < C::MT; t++)
#pragma unroll
                for (int u = 0; u < C::NT; u++)
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, acc[t][u]), rs, piece(t * C::NT + u), 0, AUX_AGENT);
        }
        wait_vmcnt<0>();                                    // acknowledged from the agent's point of coherence
        __syncthreads();
        if (tid == 0) {
            const unsigned long long tag = (p.sk_nonce | 0x10000ull) & ~0xFFFFull;       // never zero
            unsigned long long count;
            for (;;) {
                count = (seen & ~0xFFFFull) == tag ? (seen & 0xFFFFull) : 0ull;
                if (__hip_atomic_compare_exchange_strong(&counters[sk_first], &seen, tag | (count + 1), __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
            }
            const int last = (int)(count + 1) == p.split_k;
            if (last) __hip_atomic_store(&counters[sk_first], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            last_in = last;
        }
        __syncthreads();
        store_output = __builtin_amdgcn_readfirstlane(last_in) != 0;
        if (store_output && wave_active) {
            // S partitions known at compile time: the loads of all other partitions' pieces of a batch are in flight
            // together (up to 16 of 16 bytes per lane); S = 0: any number, one partition at a time
            [[maybe_unused]] auto sum_planes = [&]<int S>() {
                constexpr int WANT = S > 1 ? (16 / (S - 1) > 0 ? 16 / (S - 1) : 1) : 4;
                constexpr int BATCH = WANT >= NG ? NG : (WANT >= 4 && NG % 4 == 0 ? 4 : (WANT >= 3 && NG % 3 == 0 ? 3 : (WANT >= 2 && NG % 2 == 0 ? 2 : 1)));
                const int nz = S > 0 ? S : p.split_k;
                here(rows_in, cols_in);
#pragma unroll
                for (int base = 0; base < NG; base += BATCH) {
                    if constexpr (S > 0) {
                        v4f part[S - 1][BATCH];                              // the other partitions, ascending
#pragma unroll
                        for (int j = 0; j < S - 1; j++) {
                            __amdgpu_buffer_rsrc_t rs = slot_of(j + (j >= split_z ? 1 : 0));
#pragma unroll
                            for (int i = 0; i < BATCH; i++)
                                part[j][i] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rs, piece(base + i), 0, AUX_AGENT));
                        }
#pragma unroll
                        for (int i = 0; i < BATCH; i++) {
                            v4f& own = acc[(base + i) / C::NT][(base + i) % C::NT];
                            v4f sum = part[0][i];
                            if (split_z == 0) sum = own + sum;                  // (the same bits as sum + own)
#pragma unroll
                            for (int j = 1; j < S - 1; j++) {
                                if (j == split_z) sum += own;
                                sum += part[j][i];
                            }
                            if (split_z == S - 1) sum += own;
                            own = sum;
                        }
                    } else {
                        v4f sum[BATCH];
                        for (int z = 0; z < nz; z++) {
                            v4f part[BATCH];
                            if (z == split_z) {
#pragma unroll
                                for (int i = 0; i < BATCH; i++) part[i] = acc[(base + i) / C::NT][(base + i) % C::NT];
                            } else {
                                __amdgpu_buffer_rsrc_t rs = slot_of(z);
#pragma unroll
                                for (int i = 0; i < BATCH; i++)
                                    part[i] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rs, piece(base + i), 0, AUX_AGENT));
                            }
#pragma unroll
                            for (int i = 0; i < BATCH; i++) sum[i] = z == 0 ? part[i] : sum[i] + part[i];
                        }
#pragma unroll
                        for (int i = 0; i < BATCH; i++) acc[(base + i) / C::NT][(base + i) % C::NT] = sum[i];
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            };
            if constexpr (NG > 16) {
                // 72 to 128 accumulator registers leave room for one partition's batch of three or four (the loop of
                // the S = 0 case above, written out: called through the lambda it cost the 256x256 tile ~40 spilled registers)
                constexpr int GB = NG % 4 == 0 ? 4 : (NG % 3 == 0 ? 3 : (NG % 2 == 0 ? 2 : 1));
#pragma unroll
                for (int base = 0; base < NG; base += GB) {
                    v4f sum[GB];
                    for (int z = 0; z < p.split_k; z++) {
                        v4f part[GB];
                        if (z == split_z) {
#pragma unroll
                            for (int i = 0; i < GB; i++) part[i] = acc[(base + i) / C::NT][(base + i) % C::NT];
                        } else {
                            __amdgpu_buffer_rsrc_t rs = slot_of(z);
#pragma unroll
                            for (int i = 0; i < GB; i++)
                                part[i] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rs, piece(base + i), 0, AUX_AGENT));
                        }
#pragma unroll
                        for (int i = 0; i < GB; i++) sum[i] = z == 0 ? part[i] : sum[i] + part[i];
                    }
#pragma unroll
                    for (int i = 0; i < GB; i++) acc[(base + i) / C::NT][(base + i) % C::NT] = sum[i];
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
                switch (p.split_k) {
                    case 2: sum_planes.template operator()<2>(); break;
                    case 3: sum_planes.template operator()<3>(); break;
                    case 4: sum_planes.template operator()<4>(); break;
                    case 5: sum_planes.template operator()<5>(); break;
                    case 6: sum_planes.template operator()<6>(); break;
                    default: sum_planes.template operator()<0>(); break;
                }
            }
        }
        }
    }

    // ---- epilogue (a wave without valid rows has nothing to store; no barrier in here) -----------
    if (!wave_active || !store_output) {
    } else if (MODE == 1) {
        // split-K: fp32 partial tile, 16 bytes per lane
#pragma unroll
        for (int t = 0; t < C::MT; t++) {
            const int row = m0 + wave_m * WM + 16 * t + i16;
            if (row >= row_hi) continue;
#pragma unroll
            for (int u = 0; u < C::NT; u++) {
                const int col = n0 + wave_n * WN + 16 * u + 4 * g;
                if (col >= p.n) continue;
                float* dst = p.ws + ((size_t)split_z * p.m + row) * (size_t)p.n + col;
                if constexpr (!TAILS) {
                    *(v4f*)dst = acc[t][u];
                } else {
                    // rows of the plane start on any 4-byte boundary, which a 16-byte store takes, and may end inside the
                    // lane's four columns
                    typedef v4f v4f_any __attribute__((aligned(4)));
                    if (col + 3 < p.n) {
                        *(v4f_any*)dst = acc[t][u];
                    } else {
#pragma unroll
                        for (int r = 0; r < 3; r++)
                            if (col + r < p.n) dst[r] = acc[t][u][r];
                    }
                }
            }
        }
    } else {
        // bf16 through LDS so that the global stores are 16 bytes per lane and every store
        // instruction writes whole rows of the wave tile (WNO*2 contiguous bytes each).  (Measured against the
        // route through the registers alone - v_permlane16_swap pairing the 8-byte pieces of neighbouring lane
        // groups into 16-byte ones, a rotation by 8 lanes so that an instruction writes 128-byte lines, no LDS:
        // 4096^3 59.9-60.1 us against 60.2-60.5 with this staging on the same box, but 6144 x 7168 x 256 29.5
        // against 27.5, 1024 x 7168 x 2048 19.4 against 18.9, the grouped configuration 915 against 901; with
        // 64-byte pieces per row, no rotation, 58.1 against 56.1 on 4096^3.  Rows of 256 bytes per instruction
        // are what the write path takes best, and the staging costs less than the narrower stores.)  The last
        // stage is free (after the barrier of the last K block no wave reads it and no copy into it is in
        // flight); the stages before it already receive the next tile.  Each wave stages its tile in two halves of
        // WM/2 rows in its own region; 16-byte chunks are XOR-swizzled by row so that neither the
        // writes (16 rows per instruction) nor the 16-byte reads conflict.
        constexpr int WNO = EPI == 1 ? WN / 2 : WN;                   // output columns of the wave tile
        constexpr int ROW_CHUNKS = WNO * 2 / 16;                      // 16-byte chunks per tile row
        constexpr int ROWS_PER_SWEEP = 16 / ROW_CHUNKS > 0 ? 16 / ROW_CHUNKS : 1;
        constexpr int HALF_ROWS = WM / EPI_PARTS, HALF_MT = C::MT / EPI_PARTS;    // a "half" is one of EPI_PARTS parts: two, or one per m tile if their number is odd
        // A row of 12 chunks is staged with one chunk of padding instead of the XOR swizzle: with 13
        // chunks from row to row, 16 consecutive rows of one chunk column fall on 16 different bank groups.
        constexpr bool ROW_POW2 = (ROW_CHUNKS & (ROW_CHUNKS - 1)) == 0;
        constexpr int RSTRIDE = ROW_POW2 ? WNO * 2 : WNO * 2 + 16;    // bytes from row to row in the staging area
        static_assert(C::MT % EPI_PARTS == 0 && C::NWAVES * HALF_ROWS * RSTRIDE <= C::STAGE_BYTES, "output staging must fit one stage");
        unsigned char* region = lds + (NSTAGE - 1) * C::STAGE_BYTES + wave * (HALF_ROWS * RSTRIDE);
        const int ldc = EPI == 1 ? p.n / 2 : p.n, col_hi = EPI == 1 ? cur.n_hi / 2 : cur.n_hi;
        // Stores go through buffer descriptors: an offset of 0xFFFFFFFF drops the lane's store, so the
        // instruction count does not depend on the data.  Each store gets a descriptor based at the first
        // element of its group of rows (scalar arithmetic only); the scalar-offset operand is not used:
        // with it, the vector ALU instruction that follows a 16-byte store was seen to overwrite the
        // store's data register before the store had read it (the compiler pads that case only for
        // stores without a scalar offset).
        const int col0 = EPI == 1 ? n0 / 2 : n0;
        uint16_t* const c_tile = p.c + (size_t)m0 * ldc + col0;
        const bool c_lines = p.c_whole_lines != 0;          // uniform: a kernel argument
#pragma unroll
        for (int half = 0; half < EPI_PARTS; half++) {
#pragma unroll
            for (int th = 0; th < HALF_MT; th++) {
                const int t = half * HALF_MT + th;
                const int r = 16 * th + i16;
                const int sw = ROW_POW2 ? (r / ROWS_PER_SWEEP) % ROW_CHUNKS : 0;
                if constexpr (EPI == 0 && C::NT % 2 == 0) {
                    // The lane's 8 bytes of n tile u and of n tile u+1 become 16 consecutive bytes of one of them:
                    // v_permlane16_swap exchanges lanes 16-31 / 48-63 of its first operand with lanes 0-15 / 32-47 of
                    // its second, so after swapping the low and the high dwords lane group g holds columns
                    // 16*(u + g%2) + 8*(g/2) .. +7 - one whole 16-byte chunk, written to LDS in one instruction
                    // instead of two (half the LDS cycles of the staging: 4096^3 59.3 against 59.6 us, 8192 x 8192 x 2048
                    // 124.7 against 126.3, 4096 x 4096 x 16384 213.0 against 214.9; 6144 x 7168 x 256 28.1 against 27.8).
#pragma unroll
                    for (int u = 0; u < C::NT; u += 2) {
                        const uint32_t lo0 = pack_bf16x2(acc[t][u][0], acc[t][u][1]), hi0 = pack_bf16x2(acc[t][u][2], acc[t][u][3]);
                        const uint32_t lo1 = pack_bf16x2(acc[t][u + 1][0], acc[t][u + 1][1]), hi1 = pack_bf16x2(acc[t][u + 1][2], acc[t][u + 1][3]);
                        const auto sl = __builtin_amdgcn_permlane16_swap(lo0, lo1, false, false);
                        const auto sh = __builtin_amdgcn_permlane16_swap(hi0, hi1, false, false);
                        const v4i o = {(int)sl[0], (int)sh[0], (int)sl[1], (int)sh[1]};
                        const int chunk = 2 * (u + (g & 1)) + (g >> 1);
                        *(v4i*)(region + r * RSTRIDE + ((chunk ^ sw) << 4)) = o;
                    }
                } else {
#pragma unroll
                for (int u = 0; u < C::NT; u++) {
                    if (EPI == 1) {
                        // the lane's four columns are two (gate, up) pairs -> two outputs, 4 bytes
                        const uint32_t o = pack_bf16x2(silu_mul(acc[t][u][0], acc[t][u][1]), silu_mul(acc[t][u][2], acc[t][u][3]));
                        *(uint32_t*)(region + r * RSTRIDE + ((u ^ sw) << 4) + g * 4) = o;
                    } else {
                        v2i o;
                        o[0] = (int)pack_bf16x2(acc[t][u][0], acc[t][u][1]);
                        o[1] = (int)pack_bf16x2(acc[t][u][2], acc[t][u][3]);
                        const int chunk = 2 * u + (g >> 1);
                        *(v2i*)(region + r * RSTRIDE + ((chunk ^ sw) << 4) + (g & 1) * 8) = o;
                    }
                }
                }
            }
            // A pass = one 16-byte store per lane.  With 12 chunks per row a pass covers 4 rows with 48 lanes
            // (the other 16 are switched off like out-of-range ones), so that, as in the power-of-two
            // case, a lane keeps its row-in-pass and chunk over all passes.
            constexpr int ROWS_PER_PASS = ROW_POW2 ? 64 / ROW_CHUNKS : 4, PASSES = HALF_ROWS / ROWS_PER_PASS;
            static_assert(HALF_ROWS % ROWS_PER_PASS == 0 && ROWS_PER_PASS * ROW_CHUNKS <= 64, "a half tile is a whole number of passes");
            static_assert(MODE == 1 || EPI_STORES == EPI_PARTS * PASSES, "store count used by the next tile's wait");
            // lane -> (row inside the pass, chunk); everything else about a store's address is uniform
            // and sits in the descriptor, so the 16 stores need one address register, not 16
            const int lane_r = lane / ROW_CHUNKS, lane_chunk = lane % ROW_CHUNKS;
            const bool lane_live = ROW_POW2 || lane_r < ROWS_PER_PASS;
            const int wave_row0 = wave_m * WM, wave_col0 = wave_n * WNO;              // inside the tile, output columns
            const bool col_ok = lane_live && col0 + wave_col0 + lane_chunk * 8 < col_hi;
            [[maybe_unused]] const bool row_ends = (ldc & 7) != 0 && col0 + wave_col0 + WNO > ldc;      // the wave's tile holds rows' last, partial chunks
            const uint32_t lane_off = ((uint32_t)(wave_row0 + lane_r) * (uint32_t)ldc + (uint32_t)(wave_col0 + lane_chunk * 8)) * 2u;
#pragma unroll
            for (int q = 0; q < PASSES; q++) {
                const int r = q * ROWS_PER_PASS + (lane_live ? lane_r : 0);
                const int sw = ROW_POW2 ? (r / ROWS_PER_SWEEP) % ROW_CHUNKS : 0;
                const v4i val = *(const v4i*)(region + r * RSTRIDE + ((lane_chunk ^ sw) << 4));
                const int pass_row0 = half * HALF_ROWS + q * ROWS_PER_PASS;            // compile-time
                const int row = m0 + wave_row0 + pass_row0 + lane_r;
                bool ok = col_ok && row >= row_lo && row < row_hi;
                if constexpr (SHARED_SUM) {
                    const int x = ((pass_row0 + lane_r) >> 4) * C::NT + (EPI == 1 ? lane_chunk : lane_chunk >> 1);
                    ok = ok && ((out_parts >> (x * p.split_k / (C::MT * C::NT))) & 1u);
                }
                __amdgpu_buffer_rsrc_t c_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(c_tile + (size_t)pass_row0 * ldc), 0, 0xFFFFFFF0u, 0x00020000);
                if constexpr (!TAILS) {
                    // Written once and not read again here: nontemporal where rows of c are whole 128-byte lines.
                    // Where they are not, a tile's row segment begins and ends inside lines that it shares with
                    // the neighbouring tiles; plain stores let the L2 put those lines together before they leave
                    // (4096 x 4088 x 4096: 61 us against 65 us with the hint; with whole lines the hint gains 1 us).
                    if (c_lines) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, val), c_rsrc, ok ? lane_off : 0xFFFFFFFFu, 0, 2);
                    else __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, val), c_rsrc, ok ? lane_off : 0xFFFFFFFFu, 0, 0);
                } else {
                    // n not a multiple of eight: the chunk that holds a row's last columns is stored in
                    // pieces of 4, 2 and 1 elements (the bits of the number of columns left), every piece
                    // its own instruction that the other lanes sit out, by the waves whose tile holds such a chunk; rows then start on 2-, 4- or
                    // 8-byte boundaries only, which the stores take in their stride (plain stores: the lines a
                    // row segment shares with the neighbouring tiles are put together in the L2)
                    int left = ldc - (col0 + wave_col0 + lane_chunk * 8);                  // columns from this chunk's first to the row's end
                    left = left < 0 ? 0 : (left > 8 ? 8 : left);
                    const bool part = ok && left < 8;
                    const v4u v = __builtin_bit_cast(v4u, val);
                    __builtin_amdgcn_raw_buffer_store_b128(v, c_rsrc, ok && left == 8 ? lane_off : 0xFFFFFFFFu, 0, 0);
                    if (row_ends) {
                    const v2i lo = {val[0], val[1]};
                    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, lo), c_rsrc, part && (left & 4) ? lane_off : 0xFFFFFFFFu, 0, 0);
                    const uint32_t d2 = (left & 4) ? v[2] : v[0];                          // elements (left & 4), +1
                    __builtin_amdgcn_raw_buffer_store_b32(d2, c_rsrc, part && (left & 2) ? lane_off + (uint32_t)(left & 4) * 2u : 0xFFFFFFFFu, 0, 0);
                    const int e1 = left & 6;                                               // element (left & 6)
                    const uint32_t d1 = e1 == 0 ? v[0] : e1 == 2 ? v[1] : e1 == 4 ? v[2] : v[3];
                    __builtin_amdgcn_raw_buffer_store_b16((unsigned short)(d1 & 0xFFFFu), c_rsrc, part && (left & 1) ? lane_off + (uint32_t)e1 * 2u : 0xFFFFFFFFu, 0, 0);
                    }
                }
            }
        }
    }
    if (!nxt.valid) break;
    stores_behind = prefetched && wave_active && MODE != 1 && !TAILS && store_output;   // (with TAILS the store count differs from wave to wave, EPI_STORES or four times that where the wave holds rows' ends: only a plain wait is right)
    cur = nxt; cp = ncp;
    }   // tiles
}

// ---------------------------------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------------------------------
// Rows of a that are not a multiple of four, columns that are not a multiple of eight, operands that start off the 16-byte
// grid: the instantiation that repairs the last bytes of a and b and stores c without assuming any alignment of its rows.
// (with the fused epilogue the rows of the output have n/2 columns: 16-byte stores need n/2 on the 8-column grid; MODE 1 writes
// planes of n columns, not c)
template <int EPI>
static inline bool needs_tails(const GemmArgs& a) {
    const int out_cols = EPI == 1 ? a.n / 2 : a.n;
    return (a.lda & 3) != 0 || (a.n & 7) != 0 || (out_cols & 7) != 0 || (((uintptr_t)a.a | (uintptr_t)a.b | (uintptr_t)a.c) & 15) != 0;
}

// The instantiation of a call, its LDS limit raised.
template <int BM, int BN, int WM, int WN, int MODE, int EPI, int NSTAGE, bool SHARED_SUM>
static inline hipError_t ready_tr(const GemmArgs& a, void (**kern)(const GemmArgs)) {
    const bool tails = needs_tails<EPI>(a);
    *kern = tails ? gemm_tr_kernel<BM, BN, WM, WN, MODE, EPI, NSTAGE, true, SHARED_SUM> : gemm_tr_kernel<BM, BN, WM, WN, MODE, EPI, NSTAGE, false, SHARED_SUM>;
    static int raised[2][MAX_DEVICES];
    return raise_lds_limit((const void*)*kern, TileCfg<BM, BN, WM, WN, MODE, NSTAGE>::LDS_BYTES, raised[tails ? 1 : 0]);
}

template <int BM, int BN, int WM, int WN, int MODE, int EPI = 0, int NSTAGE = 2, bool SHARED_SUM = false>
static inline hipError_t launch_tr(const GemmArgs& a, dim3 grid, hipStream_t stream) {
    using C = TileCfg<BM, BN, WM, WN, MODE, NSTAGE>;
    void (*kern)(const GemmArgs);
    hipError_t e = ready_tr<BM, BN, WM, WN, MODE, EPI, NSTAGE, SHARED_SUM>(a, &kern);
    if (e != hipSuccess || grid.x == 0) return e;                       // no workgroups: the kernel was to be readied only
    GemmArgs args = a;
    args.c_whole_lines = ((size_t)(EPI == 1 ? a.n / 2 : a.n) * 2u) % 128u == 0 && ((uintptr_t)a.c & 127) == 0;
    hipLaunchKernelGGL(kern, grid, dim3(C::NTHREADS), C::LDS_BYTES, stream, args);
    return hipGetLastError();
}

// The experts' weights are read past the caches where nothing of them is found there again: those that the call reads are as large as the caches together,
// and one row of tiles, so one workgroup for a column of them, holds the expert.  The instantiation is chosen here, by what the host knows; how many
// experts have rows, and how many tile rows this one has, the kernel sees (`expert_read_once`).  Bound: HBM.  With the hint a read of memory is under way for 6 to 9 %
// less time, and 0.4 to 2.5 % of the reads are saved, lines of a that b no longer pushes out of the L2 (counters of three products).  us, MODE 2 and so
// (32 experts, rows by chance, 4096 x 7168 but where said): 256 rows 166.5 and 152.4, 7168 x 2048 90.5 and 84.0; 1024
// rows in 128x256 177.9 and 164.1; 6144 in 256x256, 4096 x 4096, 153.2 and 144.3; one expert with half of 1024 rows 202.7 and 197.2; of 1024 to 64
// experts, 2048 x 7168, 194.0 and 196.2, the largest loss of 48 (hint for all tiles: 199.4); 2048 rows in 128x256, 4096 x 4096, shares up to 303: 120.3 and 113.3 (126.1).
// The line on the average: beyond it few experts have one row of tiles, and the gain goes: 64x256 at 32, 64 and 80 rows an expert 1.00-1.10, 1.01-1.04,
// 1.00-1.04 times as fast, 128x256 at 96, 112 and 128 rows 1.04-1.10, 0.98-1.08, 0.99-1.05, 256x256 at 192 and 250 rows 1.03-1.16, 1.02-1.06 (three shapes, three draws).
// Bytes: streamed, weights between products of others, the hint gains at any size (20 experts of 8 MB 39.0 and 35.8), but read again with nothing in between
// smaller ones are found in the cache: the same 30.2 and 33.8, 28 experts 35.7 and 40.0, 32 of 8 MB 41.1 and 45.7, 28 of 10 MB 47.5 and 48.8, 21 of 14 MB 54.0 and
// 54.1, 30 of 10 MB 54.0 and 52.8, 32 of 10 MB 63.9 and 56.1: the line is where neither loses.
// Rows of b are whole 128-byte lines: a line that two columns of tiles share would come from memory twice (100 tokens to 4 of 32, 3072 x 4096
// 86.8 and 81.3, 2944 78.7 and 73.8; 3008 78.6 and 79.8, 3064 88.0 and 93.8, 3001 94.0 and 101.1).
template <int BM> static inline bool b_read_once(const GemmArgs& a) {
    return expert_read_once(a.m < a.num_experts ? a.m : a.num_experts, 1, a.n, a.k) && a.n % 128 == 0 && ((uintptr_t)a.b & 127) == 0 && (long)a.m * 4 <= (long)a.num_experts * (BM * 3);
}

// Persistent workgroups: as many as fit the chip at once (LDS and thread limits), each walks tiles  blockIdx.x, blockIdx.x + grid, ...
template <class C>
static inline long resident_workgroups(bool grouped) {
    const int by_lds = 163840 / (C::LDS_BYTES + (grouped ? GROUP_TABLE_MAX * 16 : 0)), by_threads = 2048 / C::NTHREADS;   // (grouped: + the table of the experts)
    return (long)device_cus() * (by_lds < by_threads ? by_lds : by_threads);
}

// A grouped call whose K is not split.
template <int BM, int BN, int WM, int WN, bool WITH_EPI, int NSTAGE>
static inline hipError_t launch_grouped(const GemmArgs& a, dim3 grid, hipStream_t stream) {
    if constexpr (WITH_EPI) {
        if (a.epi != 0 && a.epi != 1) return hipErrorInvalidValue;
        // the tiles that the planner gives calls of few rows an expert
        if constexpr (BN == 256)
            if (b_read_once<BM>(a)) return a.epi == 1 ? launch_tr<BM, BN, WM, WN, 6, 1, NSTAGE>(a, grid, stream) : launch_tr<BM, BN, WM, WN, 6, 0, NSTAGE>(a, grid, stream);
        if (a.epi == 1) return launch_tr<BM, BN, WM, WN, 2, 1, NSTAGE>(a, grid, stream);
    }
    return a.epi == 0 ? launch_tr<BM, BN, WM, WN, 2, 0, NSTAGE>(a, grid, stream) : hipErrorInvalidValue;
}

// A tile for such calls only.
template <int BM, int BN, int WM, int WN, int NSTAGE>
static inline hipError_t launch_grouped_shape(const GemmArgs& a, int mode, hipStream_t stream) {
    if (mode != 2) return hipErrorInvalidValue;
    const long total = grouped_slots_bound(a.m, a.num_experts, BM) * ((a.n + BN - 1) / BN), resident = resident_workgroups<TileCfg<BM, BN, WM, WN, 0, NSTAGE>>(true);
    return launch_grouped<BM, BN, WM, WN, true, NSTAGE>(a, dim3((unsigned)(total < resident ? total : resident)), stream);
}

// WITH_EPI: the fused silu-mul epilogue is instantiated for this tile; GROUPED_SPLIT: the grouped walk with a K split is
template <int BM, int BN, int WM, int WN, bool WITH_EPI = false, int NSTAGE = 2, bool GROUPED_SPLIT = false>
static inline hipError_t launch_shape(const GemmArgs& a, int mode, hipStream_t stream) {
    const bool ready_only = (mode & READY_ONLY) != 0;
    mode &= ~READY_ONLY;
    using C = TileCfg<BM, BN, WM, WN, 0, NSTAGE>;
    const long resident = resident_workgroups<C>(mode == 2 || mode == 5);
    const int tiles_n = (a.n + BN - 1) / BN;
    long total;
    if (mode == 2 || mode == 5) {
        // upper bound on m-tile slots; workgroups beyond the real count find no tile and leave
        total = grouped_slots_bound(a.m, a.num_experts, BM) * tiles_n * (mode == 5 ? a.split_k : 1);
    } else {
        total = (long)((a.m + BM - 1) / BM) * tiles_n * a.split_k;
    }
    if (mode == 3) {
        // K blocks dealt to the workgroups: one workgroup per place on the chip, never more than there are
        // (tile, K block) pairs, so that every workgroup's run holds at least one
        if (a.epi != 0 || a.k < KBLK) return hipErrorInvalidValue;
        const long pairs = (long)((a.m + BM - 1) / BM) * tiles_n * (a.k / KBLK);
        if (a.sk_grid < 1 || a.sk_grid > resident || a.sk_grid > pairs || a.sk_grid > StreamK::MAX_GRID) return hipErrorInvalidValue;
        return launch_tr<BM, BN, WM, WN, 3, 0, NSTAGE>(a, dim3((unsigned)a.sk_grid), stream);
    }
    const dim3 grid(ready_only ? 0u : (unsigned)(total < resident ? total : resident));
    // K partitions summed in the kernel, the sum shared out or not.  A call that shares it readies the kernel that a capture of the
    // same call will launch too: the LDS limit is not a thing to be raised there.
    auto launch_summed = [&](auto mode_tag, auto epi_tag) {
        constexpr int M = decltype(mode_tag)::value, E = decltype(epi_tag)::value;
        if constexpr (shares_sum<BM, BN, WM, WN>())
            if (a.split_k >= shares_from<BM, BN>() && can_share_sum(total, resident, a.split_k, stream)) {
                void (*captured)(const GemmArgs);
                hipError_t e = ready_tr<BM, BN, WM, WN, M, E, NSTAGE, false>(a, &captured);
                if (e != hipSuccess) return e;
                return launch_tr<BM, BN, WM, WN, M, E, NSTAGE, true>(a, grid, stream);
            }
        return launch_tr<BM, BN, WM, WN, M, E, NSTAGE>(a, grid, stream);
    };
    using std::integral_constant;
    if (mode == 5) {
        if constexpr (GROUPED_SPLIT) {
            const long tiles = total / a.split_k;
            if (a.split_k < 2 || a.split_k > 0xFFFF || tiles > StreamK::MAX_GRID || (long)a.split_k * BM * BN * 4 >= (1L << 32)) return hipErrorInvalidValue;
            if constexpr (WITH_EPI) { if (a.epi == 1) return launch_summed(integral_constant<int, 5>{}, integral_constant<int, 1>{}); }
            return a.epi == 0 ? launch_summed(integral_constant<int, 5>{}, integral_constant<int, 0>{}) : hipErrorInvalidValue;
        } else {
            return hipErrorInvalidValue;
        }
    }
    if (mode == 4) {
        // K split summed in the kernel: one counter per tile, or one flag per workgroup, in the workspace's head
        const long tiles = total / a.split_k;
        if (a.split_k < 2 || a.split_k > 0xFFFF || tiles > StreamK::MAX_GRID || (long)a.split_k * BM * BN * 4 >= (1L << 32)) return hipErrorInvalidValue;
        if constexpr (WITH_EPI) { if (a.epi == 1) return launch_summed(integral_constant<int, 4>{}, integral_constant<int, 1>{}); }
        return a.epi == 0 ? launch_summed(integral_constant<int, 4>{}, integral_constant<int, 0>{}) : hipErrorInvalidValue;
    }
    if (mode == 2) return launch_grouped<BM, BN, WM, WN, WITH_EPI, NSTAGE>(a, grid, stream);
    if (a.epi != 0) {
        // (with the reduce launch of a K split the planes are plain sums and the reduce kernel applies the epilogue)
        if constexpr (WITH_EPI) {
            if (a.epi != 1) return hipErrorInvalidValue;
            if (mode == 1) return launch_tr<BM, BN, WM, WN, 1, 0, NSTAGE>(a, grid, stream);
            return launch_tr<BM, BN, WM, WN, 0, 1, NSTAGE>(a, grid, stream);
        } else {
            return hipErrorInvalidValue;
        }
    }
    if (mode == 1) return launch_tr<BM, BN, WM, WN, 1, 0, NSTAGE>(a, grid, stream);
    return launch_tr<BM, BN, WM, WN, 0, 0, NSTAGE>(a, grid, stream);
}

}  // namespace fp8bs
