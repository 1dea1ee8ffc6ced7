// C ABI of libfp8bs.so (declared in include/fp8bs.h): argument checking, the shape-family planner
// and kernel launches.  Host code only; the device code is in fp8bs_kernels.hip.
//
// This layer stands where the reference has its launcher `fp8_mm(...)`
// (1-amd-fp8-mm/amd-fp8-mm-submission.py:514-579).  Differences by design: it is stream-aware,
// returns a status instead of void, never writes the inputs, and picks kernels by shape family
// instead of an exact-shape table.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>
#include <stdlib.h>
#include <unistd.h>
#include <algorithm>
#include <atomic>
#include <chrono>

#include "fp8bs.h"
#include "fp8bs_kernels.h"

namespace {

constexpr int KBLK = 128;

// A kernel is named by its variant (FP8BS_VARIANT_*) and, for the variants that have two, its form: tile = variant + 256 * form.
struct VariantInfo { int bm, bn, threads; };
constexpr int FORM1 = 256;
constexpr int variant_of(int tile) { return tile & 255; }
constexpr int form_of(int tile) { return tile >> 8; }

bool variant_info(int tile, VariantInfo* out) {
    switch (tile) {
        case FP8BS_VARIANT_GENERIC:  *out = {16, 16, 256}; return true;
        case FP8BS_VARIANT_T256x256: *out = {256, 256, 512}; return true;
        case FP8BS_VARIANT_T128x128: *out = {128, 128, 256}; return true;
        case FP8BS_VARIANT_T64x256S3 | FORM1: *out = {128, 128, 512}; return true;
        case FP8BS_VARIANT_T64x128:  *out = {64, 128, 512}; return true;
        case FP8BS_VARIANT_T64x128 | FORM1: *out = {64, 64, 256}; return true;
        case FP8BS_VARIANT_T256x128: *out = {256, 128, 512}; return true;
        case FP8BS_VARIANT_SKINNY64x144: *out = {64, 144, 256}; return true;
        case FP8BS_VARIANT_SKINNY64x256: *out = {64, 256, 256}; return true;
        case FP8BS_VARIANT_SKINNY64x288: *out = {64, 288, 256}; return true;
        case FP8BS_VARIANT_T256x192: *out = {256, 192, 512}; return true;
        case FP8BS_VARIANT_T256x128S3: *out = {256, 128, 512}; return true;
        case FP8BS_VARIANT_T256x128S3 | FORM1: *out = {128, 256, 512}; return true;
        case FP8BS_VARIANT_T192x192S3: *out = {192, 192, 512}; return true;
        case FP8BS_VARIANT_T64x256S3: *out = {64, 256, 512}; return true;
        case FP8BS_VARIANT_T64x256S3 | 2 * FORM1: *out = {16, 64, 512}; return true;
        case FP8BS_VARIANT_T64x256S3 | 3 * FORM1: *out = {32, 64, 512}; return true;
        default: return false;
    }
}

inline long cdiv(long a, long b) { return (a + b - 1) / b; }

// Workgroups of a call that deals K blocks instead of tiles: one per place on the chip (what the tile's LDS
// and thread count let a CU hold), never more than there are (tile, K block) pairs.
int streamk_grid(int tile, int m, int n, int k, int num_cus) {
    VariantInfo vi{};
    if (!variant_info(tile, &vi) || tile == FP8BS_VARIANT_GENERIC || form_of(tile) != 0 || k < KBLK) return 0;
    const int lds = fp8bs::variant_lds_bytes(tile);
    if (lds <= 0 || lds > 163840) return 0;
    if (num_cus <= 0) num_cus = 256;
    const long by_lds = 163840 / lds, by_threads = 2048 / vi.threads;
    long g = (long)num_cus * (by_lds < by_threads ? by_lds : by_threads);
    const long pairs = cdiv(m, vi.bm) * cdiv(n, vi.bn) * (k / KBLK);
    if (pairs >= (1L << 31)) return 0;                  // the kernel counts the pairs in 32 bits
    g = g < pairs ? g : pairs;
    return (int)(g < fp8bs::StreamK::MAX_GRID ? g : fp8bs::StreamK::MAX_GRID);
}

// The tile of a forced variant argument: FP8BS_VARIANT_FORM(variant, form) names a form, a plain variant its first.
int forced_tile(int variant) { return variant < 256 ? variant : variant_of(variant) | ((variant >> 8) - 1) * FORM1; }

// The small tiles whose workgroups hold all partitions of K (fp8bs_waves.h): up to eight, one launch, no workspace.
constexpr int WAVES_MAX = 8;
bool is_waves_tile(int tile) { return tile == (FP8BS_VARIANT_T64x256S3 | 2 * FORM1) || tile == (FP8BS_VARIANT_T64x256S3 | 3 * FORM1); }

// The tile that only grouped calls take (fp8bs_tile_128x256s3.hip).
bool is_grouped_tile(int tile) { return tile == (FP8BS_VARIANT_T256x128S3 | FORM1); }

bool is_streaming_variant(int v) { return v == FP8BS_VARIANT_SKINNY64x144 || v == FP8BS_VARIANT_SKINNY64x256 || v == FP8BS_VARIANT_SKINNY64x288; }

// The fp32 partial planes of a K split followed by the reduce kernel.
uint64_t planes_bytes(int m, int n, int split_k) { return split_k > 1 ? (uint64_t)split_k * (uint64_t)m * (uint64_t)n * 4u : 0u; }

// A plan and what the caller's structure has no field for: whether the sums of the K partitions are better shared out in the kernel
// where the call's workspace holds the flags and partial tiles and the launch is not captured.  The plan itself says what every
// caller with workspace_bytes gets, also under capture: partial planes and the reduce kernel, or the sum by one workgroup.  Tile
// and split are the same for all callers, so that a replayed call returns the bits of an eager one.
struct Planned { fp8bs_plan_t plan; bool share; };

// The choice among (tile, split) in microseconds, each at the price of both forms: the soonest to finish where its sum can be
// shared out, among those that finish within 6 % of the soonest where it cannot.  Of 267 shapes (see choose_tiled), times against the planner before there were
// shared sums, operands from the caches / from HBM: eager 0.988 / 0.975, worst 1.09, replayed 0.996 / 0.979, worst 1.08 (of 270 others, 0.963 /
// 0.970 and 0.997 / 0.997, 1.10 and 1.07).  At the price of the shared form alone 0.994 / 0.970, worst 1.37, and 1.009 / 0.977, worst 1.38
// (896 x 1344 x 2944 in three, 16 us, 12 unsplit); within 4 % instead 250 x 4096 x 7168 would lose its four partitions, 19.3 us eager
// and 21.4 replayed against 21.3 and 21.6 in three.
struct Choice {
    struct Option { int tile, split; double shared, plain, gpu; bool share, fused; } options[80];
    int count = 0;
    // gpu: time on the GPU, which decides among calls that the host's launches make equal.  shared, plain: of the call, the sum shared
    // out where share says so; fused: without sharing, summed in the kernel.
    void add(int tile, int split, double shared, double plain, double gpu, bool share, bool fused) { options[count++] = {tile, split, shared, plain, gpu, share, fused}; }
    const Option& pick() const {
        double soonest = options[0].plain;
        for (int i = 1; i < count; i++) if (options[i].plain < soonest) soonest = options[i].plain;
        const Option* best = nullptr;
        for (int i = 0; i < count; i++) {
            const Option& o = options[i];
            if (o.plain > 1.06 * soonest) continue;
            if (!best || o.shared < best->shared || (o.shared == best->shared && o.gpu < best->gpu)) best = &o;
        }
        return *best;
    }
};

// Can the partial tiles of a K split of this tile shape be summed in the kernel that writes them (one counter per
// tile in the head of the workspace, the partition count in the counter's low 16 bits)?
bool can_sum_in_kernel(int m, int n, int tile, int split_k) {
    VariantInfo vi{};
    if (tile == FP8BS_VARIANT_GENERIC || is_streaming_variant(tile) || !variant_info(tile, &vi)) return false;
    return split_k >= 2 && split_k <= 255 && cdiv(m, vi.bm) * cdiv(n, vi.bn) <= fp8bs::StreamK::MAX_GRID;
}

// Tiles with the fused silu-mul epilogue.
bool has_epilogue(int tile) {
    switch (tile) {
        case FP8BS_VARIANT_T256x256: case FP8BS_VARIANT_T256x128S3: case FP8BS_VARIANT_T256x128S3 | FORM1:
        case FP8BS_VARIANT_T64x128: case FP8BS_VARIANT_T64x128 | FORM1: case FP8BS_VARIANT_T64x256S3: case FP8BS_VARIANT_T64x256S3 | FORM1: return true;
        default: return is_waves_tile(tile);
    }
}

// Tiles with the grouped walk in K partitions.
bool has_grouped_split(int tile) {
    return tile == (FP8BS_VARIANT_T64x128 | FORM1) || tile == FP8BS_VARIANT_T64x256S3 || tile == (FP8BS_VARIANT_T64x256S3 | FORM1);
}

// Fill a plan for a given tile and split count.  in_kernel: the split's partial tiles are summed by the last
// workgroup to finish each tile (where the shape allows it, see above; else the reduce kernel follows).
void fill_plan(int m, int n, int k, int tile, int split_k, fp8bs_plan_t* out, int stream_k = 0, bool in_kernel = false) {
    VariantInfo vi{};
    variant_info(tile, &vi);
    int kbt = k / KBLK;
    if (tile == FP8BS_VARIANT_GENERIC) { split_k = 1; stream_k = 0; }
    if (stream_k > 0) split_k = 1;
    if (split_k < 1) split_k = 1;
    if (split_k > kbt) split_k = kbt > 0 ? kbt : 1;
    const bool waves = is_waves_tile(tile);                                          // (all partitions in a workgroup: one launch, no workspace)
    out->variant = variant_of(tile);
    out->form = form_of(tile);
    out->tile_m = vi.bm;
    out->tile_n = vi.bn;
    out->split_k = split_k;
    out->block_threads = vi.threads;
    out->lds_bytes = fp8bs::variant_lds_bytes(tile);
    out->stream_k = stream_k > 0 ? stream_k : 0;
    out->sum_in_kernel = waves ? split_k > 1 : in_kernel && stream_k <= 0 && can_sum_in_kernel(m, n, tile, split_k) ? 1 : 0;
    if (tile == FP8BS_VARIANT_GENERIC) {
        out->grid_x = (int)cdiv(n, 16); out->grid_y = (int)cdiv(m, 16); out->grid_z = 1;
    } else {
        out->grid_x = stream_k > 0 ? stream_k : (int)(cdiv(m, vi.bm) * cdiv(n, vi.bn) * (waves ? 1 : split_k)); out->grid_y = 1; out->grid_z = 1;
    }
    if (waves) out->workspace_bytes = 0;
    else if (stream_k > 0) out->workspace_bytes = (uint64_t)fp8bs::StreamK::bytes(stream_k, vi.bm, vi.bn);
    else if (out->sum_in_kernel)   // the counters, then one fp32 tile per (tile, K partition)
        out->workspace_bytes = (uint64_t)fp8bs::StreamK::SLOTS_OFF + (uint64_t)(cdiv(m, vi.bm) * cdiv(n, vi.bn)) * (uint64_t)split_k * (uint64_t)vi.bm * (uint64_t)vi.bn * 4u;
    else out->workspace_bytes = planes_bytes(m, n, split_k);
}

// Rows of c (n bf16) that keep 16-byte stores aligned: what the streaming kernels need (forced variants only;
// the tiled kernels take any m and n in every mode: they repair the last bytes of a and b themselves, store a
// row's last chunk of c in pieces and write the partial planes of a K split with stores that need no more than a float's
// alignment, element by element only in a row's last group of four where the row ends inside it).
bool vector_shape(int n) { return (n % 8) == 0; }

// At most 64 rows against a b of 24 MB or more: the call streams b from HBM once and everything else is small.
bool skinny_shape(int m, int n, int k) { return m <= 64 && (double)n * (double)k >= 24.0e6; }

// The tile shape and K split of the tiled MFMA kernel that finish soonest (any m, any n).
void choose_tiled(int m, int n, int k, int num_cus, Planned* out, bool may_split, bool epi) {
    if (num_cus <= 0) num_cus = 256;
    int kbt = k / KBLK;
    // One K block is all first copies and output, which the constants below, fits to two blocks and more, take for too little
    // with large tiles.  us, 64x64 / 128x128 in four waves / 256x128 / 256x256: 1803 x 576 6.0 / 6.1 / 7.4 / 9.9; 2944 x 171 6.4 /
    // 6.2 / 7.9 / 10.8; 9106 x 256 7.8 / 6.5 / 7.9 / 10.1; 10880 x 1484 22.7 / 13.5 / 17.2 / 18.0; 8192 x 8192 48.7 / 26.8 / 26.0 / 28.0.
    // (With the silu-mul epilogue the output is half as large, and 256x128 and 256x256, which the model picks, are the fastest.)
    if (kbt == 1 && !epi) {
        fill_plan(m, n, k, cdiv(m, 64) * cdiv(n, 64) <= 2L * num_cus ? FP8BS_VARIANT_T64x128 | FORM1 : FP8BS_VARIANT_T128x128, 1, &out->plan);
        return;
    }
    // The tile and K split that finish soonest under a cost model in microseconds.  A workgroup advances one K block in
    // max(t_alone x shared, t_power x w / CUs): t_alone is the tile's time per block with one workgroup on a CU, shared
    // the factor with two, t_power what the board's power limit allows when every CU runs one such workgroup - with w
    // workgroups running together the limit is shared by w, so fewer busy CUs clock higher until the full clock is
    // reached.  A round of workgroups (CUs x the most that fit a CU; a last partial round with fewer) costs a fixed time
    // for the launch, the first copies' latency, the output and the drain.  A K split adds the fp32 partial planes
    // (written and read back, mostly through the 256 MB cache) and the reduce launch.  The constants are fits (of
    // logarithms) to measured times on MI355X: those of the four largest tiles to 38 shapes, M 96 .. 16384, N 1024 ..
    // 28672, K 1024 .. 14336; those of the other tiles and of the splits, with the former held fixed, to every (tile,
    // split, form) of 93 shapes - the 18 of the upstream benchmark, 60 log-uniform draws of M 1 .. 8192, N 512 .. 18432,
    // K 256 .. 7168, and 15 others.  Picking by the model costs 0.7 % against the measured best of each of the 93 shapes
    // in the geometric mean, worst 14 % (measured with the line at 80 K blocks, below, at 48).
    struct Cand { int tile; int rmax; double t_alone, t_power, t_fixed, shared; int kb_min; double t_sum = 0, t_part = 0; int shares_from = 0; };
    // kb_min: the fewest K blocks a workgroup of a split keeps.  4; 8 with the 64x256 tile, whose short blocks leave a
    // workgroup's first copies and its partial plane as most of its time (1024 x 512 x 7168: split 8 20.9 us, split 4
    // 18.6); 2 with the small tiles, where the splits are what fills the chip (1 x 2048 x 2048: split 8 6.5 us, 4 6.9).
    const Cand cands[9] = {
        {FP8BS_VARIANT_T256x256, 1, 1.181, 1.462, 6.75, 1.0, 4},
        {FP8BS_VARIANT_T256x192, 1, 1.011, 1.163, 5.51, 1.0, 4},
        {FP8BS_VARIANT_T192x192S3, 1, 0.881, 1.059, 4.11, 1.0, 4},
        {FP8BS_VARIANT_T256x128S3, 1, 0.783, 0.906, 3.70, 1.0, 4},
        {FP8BS_VARIANT_T128x128, 2, 0.765, 0.511, 4.86, 1.38, 4},
        // few output tiles or few K blocks: the call is a chain of K blocks and barriers, so the tile with the shortest
        // block wins (512 x 2048 x 1024: 64x64 5.8 us, 64x128 6.3, 128x128 in eight waves 7.5, 64x256 7.7)
        {FP8BS_VARIANT_T64x128, 2, 0.398, 0.093, 4.76, 1.90, 2},
        {FP8BS_VARIANT_T64x128 | FORM1, 2, 0.323, 0.108, 4.00, 1.76, 2, 2.17, 20.0, 4},
        {FP8BS_VARIANT_T64x256S3, 1, 0.552, 0.540, 5.00, 1.0, 8, 2.90, 9.0, 2},
        // 128x128 in eight waves: see fp8bs_tile_64x256s3.hip (2048^3 12.6 us against 14.2 with 64x256, the best of the others)
        {FP8BS_VARIANT_T64x256S3 | FORM1, 1, 0.467, 0.531, 4.57, 1.0, 4, 2.50, 9.0, 2},
    };
    const int splits[6] = {1, 2, 3, 4, 6, 8};
    Choice choice;                                         // 9 tiles in up to 6 splits and two more
    for (const Cand& c : cands) {
        if (epi && !has_epilogue(c.tile)) continue;
        VariantInfo vi{};
        variant_info(c.tile, &vi);
        const long tiles = cdiv(m, vi.bm) * cdiv(n, vi.bn);
        auto t_block = [&](long w) {          // w workgroups running together
            const long r = cdiv(w, num_cus) < c.rmax ? cdiv(w, num_cus) : c.rmax;
            const double alone = r > 1 ? c.t_alone * c.shared : c.t_alone, power = c.t_power * (double)w / (double)num_cus;
            return alone > power ? alone : power;
        };
        for (int s : splits) {
            if (s > 1 && (kbt / s < c.kb_min || !may_split)) continue;
            // The model is too fast for this tile on chains beyond 80 K blocks.  Unsplit against the best of the other tiles,
            // us, median of five, operands rotated through more than the 256 MB cache: 56 blocks 4096 x 1024 35.5 / 39.3, 2048 x
            // 1536 31.6 / 35.6; 65 640 x 6144 47.7 / 61.7; 80 2048 x 2048 53.5 / 56.5; 88 3072 x 1280 62.7 / 62.6; 112 2048 x 2048
            // 77.1 / 71.4; 128 4096 x 1024 90.3 / 82.9.  Over 86 shapes of 49 .. 128 blocks (half of them with m or n off the
            // 16-byte grid) the picks with the line at 80 are 6 % faster than at 48, 0.7 % than at 72, 0.2 % than at 88.
            if (c.tile == (FP8BS_VARIANT_T64x256S3 | FORM1) && cdiv(kbt, s) > 80) continue;
            const long wgs = tiles * s, per_round = (long)num_cus * c.rmax;
            const long full = wgs / per_round, rem = wgs % per_round;
            const double kb = (double)cdiv(kbt, s);
            double cost = (double)full * (c.t_fixed + kb * t_block(per_round));
            if (rem) cost += c.t_fixed + kb * t_block(rem);
            // the planes and the reduce launch; or, with two or three partitions, the sum in the kernel: no second
            // launch and no pass over whole planes, but the last workgroup of a tile reads s - 1 partial tiles alone
            // (measured on the same 38 shapes: two partitions 1-50 us faster than with the reduce launch, median 4.7;
            // three: median 2.3 faster; four and more: the serial sums cost more than the launch)
            // (Few rows, and n off the 8-column grid: the planes take 0.2 us each more than the constants have, 14 x 3373 x 6144 in eight of
            // 64x64 14.1 us, the sum shared out 11.2.  The picks for 150 shapes of up to 80 rows are 2 and 3 % behind the best, 4 and 4 without.)
            const double planes = 2.66 + 1.656e-6 * s * (double)m * (double)n + ((n & 7) != 0 && m <= 64 ? 0.2 * s : 0.0);
            const double in_kernel = 2.34 + 0.891e-6 * s * (double)m * (double)n
                                     + 13.2 * (s - 1) * (vi.bm * vi.bn * 4e-6) * (double)cdiv(wgs, num_cus);
            // calls issued one after another are never faster than the host launches them: 5.2 to 6.2 us with the checks in Python, or 7.7
            // to 10.2 with the reduce launch of a split, by the machine.  The latter stands as 8.5 here: the constants are 0.5 to 1.2 us over
            // what such small calls take, and at 8.5 neither side loses much on a fast or a slow host (12 x 512 x 1536 unsplit 5.4,
            // in four partitions and two launches 8.1 and 9.1; 1 x 512 x 3456 in three, one launch, 8.8, in eight 7.7 and 9.1).
            // custom_kernel's native call issues one launch in 3 to 4 us.  Calls below 5.3 us are equals here, and the time on the GPU
            // decides among them; so all that the floors do for such a caller is to ask 3.2 us on the GPU of a second launch.
            auto issued = [](double gpu, double host) { return gpu > host ? gpu : host; };
            // Where every (tile, partition) has a workgroup of its own the sums can be shared out (see the kernel): a base that is
            // the tile's, the S - 1 of S parts of a tile that a workgroup stores and loads, and, with S, ever smaller parts: pieces
            // of lines of c, written from as many XCDs.  The constants are fits, with all others held, to every (tile, split, form) of 267
            // shapes (M 1 .. 8000, N 190 .. 18100, K 1024 .. 7168, operands from HBM and from the caches), 200 of them with another plan than
            // without shared sums: the picks are 1.8 and 4.5 % behind the best of each shape, 6.1 and 4.9 % without the last term,
            // which priced eight partitions of full tiles like four (1024 x 512 x 7168 in eight of 128x128 20.4 us, 64x128 in four and a
            // reduce launch 15.1; 619 x 768 x 6272 21.3 in eight, 15.9 in two of 64x64).  250 x 4096 x 7168 in four 128x128 tiles' partitions
            // 19.0 us (three, one workgroup summing: 20.9), 300 x 2112 x 7168 16.6 (19.0), 1 x 1230 x 4864 8.5 (10.8).  Eight tiles and fewer stay
            // with the reduce launch, which is as fast there (1 x 512 x 7168 in eight 7.7 us, shared 8.7) and which the tests run at
            // those sizes.
            // (Four and more partitions from 16 K blocks on: below, the small tiles that hold all partitions are ahead.)
            const bool share = c.t_sum > 0 && s >= c.shares_from && tiles > 8 && wgs <= per_round && wgs <= fp8bs::StreamK::MAX_GRID && (s <= 3 || kbt >= 16);
            const double rows = m < vi.bm ? m : vi.bm, cols = n < vi.bn ? n : vi.bn;
            const double shared_sum = c.t_sum * (1.0 + 0.027 * s) + (20.0 * (s - 1) / s + c.t_part * s) * rows * cols * 4e-6 * (double)cdiv(wgs, num_cus);
            if (s == 1) { choice.add(c.tile, 1, issued(cost, 5.3), issued(cost, 5.3), cost, false, false); continue; }
            // 64x64 always shares where it can: its planes are as fast on the GPU (0.95 to 1.22 of the shared time in the geometric mean, by rows
            // and n on the 8-column grid, 300 shapes), and a second launch costs a caller's host 2 us (quantise, gate/up, quantise and
            // down of 41 x 1280 x 3456, bound by the host, 25.1 us and 27.0).
            const bool level = c.tile == (FP8BS_VARIANT_T64x128 | FORM1);
            const double two = cost + planes, last = cost + in_kernel, parts = cost + (level && planes < shared_sum ? planes : shared_sum);
            const bool can = can_sum_in_kernel(m, n, c.tile, s), shared = can && share && (level || issued(parts, 5.3) < issued(two, 8.5));
            // (where a sum in the kernel can be shared out it is: one that is not better than two launches then is none)
            const bool fused = can && (s == 2 || s == 3) && shared == share && issued(last, 5.3) < issued(two, 8.5);
            const double plain = fused ? issued(last, 5.3) : issued(two, 8.5);
            choice.add(c.tile, s, shared ? issued(parts, 5.3) : plain, plain, shared ? parts : fused ? last : two, shared, fused);
        }
    }
    // The small tiles that hold all K partitions in a workgroup: a launch, first copies and output, a chain of kbt / 8 blocks, and
    // the requests that all workgroups make of the L2 (in units of K blocks per CU).  Fits to 264 shapes (M 1 .. 1024, N 512 ..
    // 12288, K 384 .. 4096, operands from HBM and from the caches): where they are taken for any of these shapes, the calls take 0.81 of
    // the time of the other tiles in the geometric mean, within 1.6 % of the best; at most 1.19 of it where the two are
    // modelled level.  Only where all workgroups are on the chip at once - one or two fit a CU -, the model has no second round: of 34
    // shapes with more, M 17 .. 4203, N 126 .. 18300, all but one were slower than with the other tiles, 14 % in the geometric mean, 36 at
    // worst (320 x 1664 x 384 5.2 us, 64 x 64 3.9); of 90 with fewer, outside the fitted sizes too, none (0.74).  Not beyond 24 K
    // blocks, where the others' splits over workgroups are ahead.  Up to eight blocks the sum is the
    // unsplit one; beyond, eight partitions, summed in the kernel without a workspace.
    if (kbt >= 2 && (kbt <= WAVES_MAX || (may_split && kbt <= 24))) {
        struct Waves { int tile, bm; double fixed, block, load; };
        const Waves waves[2] = {{FP8BS_VARIANT_T64x256S3 | 2 * FORM1, 16, 2.12, 1.223, 0.312}, {FP8BS_VARIANT_T64x256S3 | 3 * FORM1, 32, 2.31, 1.485, 0.385}};
        for (const Waves& w : waves) {
            const int s = kbt <= WAVES_MAX ? 1 : WAVES_MAX;
            if (cdiv(m, w.bm) * cdiv(n, 64) > (long)num_cus * (163840 / fp8bs::waves_lds_bytes(w.bm))) continue;
            const double gpu = w.fixed + w.block * (double)cdiv(kbt, WAVES_MAX) + w.load * (double)(cdiv(m, w.bm) * cdiv(n, 64)) * kbt / 256.0;
            const double cost = gpu > 5.3 ? gpu : 5.3;
            choice.add(w.tile, s, cost, cost, gpu, false, false);
        }
    }
    const Choice::Option& o = choice.pick();
    fill_plan(m, n, k, o.tile, o.split, &out->plan, 0, o.fused);
    out->share = o.share;
}

// Skinny shapes: one of the two tiles of eight 32 x 64 waves - 64 x 256 with three LDS stages, two K blocks of b, 64 KB, in
// flight per workgroup, or 128 x 128 with four stages, three blocks, 48 KB - and the K split that finishes soonest under a
// model in microseconds: a workgroup advances one K block in the time the workgroups running together need to pull
// their 32 or 16 KB of b each (and of a, at a quarter of the price) from HBM at 5.5 or 5.3 TB/s, and never faster than a
// block's copies take to arrive; a time for the first block and the output; the partial planes and the reduce launch, or a sum
// in the kernel, shared out or, in two or three partitions, by one workgroup.  The constants of the 64 x 256 tile's planes and its sums by one
// workgroup are as measured before there was the other tile; its shared sums and the K blocks and shared sums of the other are
// fits to every split of both tiles on 79 shapes (M 1 .. 64, N 3000 .. 28672, K 1024 .. 8192, b streamed from HBM), the planes and the sums by one
// workgroup of the 128 x 128 tile to 94 shapes (N 4300 .. 18400, b from HBM and from the caches).  On these 94 the picks are 9 % (caches) and 7 %
// (HBM) faster than those of the 64 x 256 tile alone, eager as well as replayed, 4 % slower at worst (with its planes left out,
// 12 %: 11 x 6464 x 4096).  us: 64 x 18432 x 7168 33.0 (33.7), 64 x 16384 x 4096 20.5 (22.0), 64 x 12288 x 2048 12.7 (16.4), 64 x 4096 x 7168
// 14.2 (16.3), 64 x 7168 x 7168 18.2 (19.4).  With few rows the planes are small and two launches are ahead, in either tile:
// 1 x 18432 x 7168 28.8, one launch 30.8.
void choose_skinny(int m, int n, int k, int num_cus, Planned* out, bool may_split) {
    if (num_cus <= 0) num_cus = 256;
    const int kbt = k / KBLK;
    const double mn = (double)m * (double)n;
    Choice choice;
    for (int s = 1; s <= 8 && s <= kbt; s++) {
        if (s > 1 && !may_split) break;
        const long wgs = cdiv(n, 256) * s;
        const double together = (double)(wgs < num_cus ? wgs : num_cus);
        double t_block = together * 32768.0 / 5.5e6;
        if (t_block < 1.05) t_block = 1.05;
        double cost = (double)cdiv(wgs, num_cus) * (2.0 + (double)cdiv(kbt, s) * t_block);
        if (s > 1) cost += 4.0 + 0.24 * s + 1.19e-6 * s * mn;
        // In one round of workgroups the sum is done in the kernel where the planes are large enough for the reduce launch to cost
        // more than the chain of round trips that replaces it (acknowledged stores, flags or a count, reads).  One workgroup's sum, b
        // from HBM, three partitions of 18432 x 7168: 64 rows 33.7 us against 34.4 with the reduce launch, 16 rows 30.3 against 29.3.
        const double by_one = 2.05 - 0.78e-6 * s * mn, by_all = 1.13 - 0.37e-6 * s * mn;
        const bool fused = (s == 2 || s == 3) && wgs <= num_cus && by_one < 0;
        const bool shared = s > 1 && s != 5 && s != 7 && wgs <= num_cus && by_all < 0;
        const double plain = fused ? cost + by_one : cost, eager = shared ? cost + by_all : plain;
        choice.add(FP8BS_VARIANT_T64x256S3, s, eager, plain, eager, shared, fused);
    }
    for (int s = 1; s <= 8 && s <= kbt; s++) {
        const long wgs = cdiv(n, 128) * s;
        if ((s > 1 && !may_split) || wgs > num_cus) break;
        // (chains of more than 26 blocks take longer than the model has it: 1 x 28672 x 4096 28.5 us, 26.1 with 64 x 256)
        if (s == 5 || s == 7 || (s > 1 && kbt / s < 2) || cdiv(kbt, s) > 26) continue;
        double t_block = (double)wgs * 128.0 * (128.0 + 0.26 * m) / 5.33e6;
        if (t_block < 0.64) t_block = 0.64;
        const double cost = 5.06 + (double)cdiv(kbt, s) * t_block;
        const double planes = s > 1 ? 2.41 + 0.755e-6 * s * mn : 0.0;
        const double by_one = 2.53 + 0.605e-6 * s * mn, by_all = 2.92 + 19.5 * (s - 1) / s * (double)m * 128.0 * 4e-6;
        const bool fused = (s == 2 || s == 3) && by_one < planes, shared = s > 1 && by_all < planes;
        const double plain = cost + (fused ? by_one : planes), eager = shared ? cost + by_all : plain;
        choice.add(FP8BS_VARIANT_T64x256S3 | FORM1, s, eager, plain, eager, shared, fused);
    }
    const Choice::Option& o = choice.pick();
    fill_plan(m, n, k, o.tile, o.split, &out->plan, 0, o.fused);
    out->share = o.share;
}

// What the planners below return for a shape is kept, 64 shapes a thread: the cost models take 0.4-0.8 us of host time
// (all tiles and splits), in a call whose launch takes 3.  Every argument is in the key, so an entry never goes stale.
template <typename P>
struct PlanMemo {
    struct Entry { int key[6]; P plan; };
    Entry entries[64] = {};                   // no key is all zeros: experts or CUs are at least 1
    template <typename F>
    const P& get(const int (&key)[6], F&& make) {
        uint32_t h = 0;
        for (int v : key) h = (h ^ (uint32_t)v) * 0x9E3779B1u;
        Entry& e = entries[h >> 26];
        bool same = true;
        for (int i = 0; i < 6; i++) same &= e.key[i] == key[i];
        if (!same) {
            make(&e.plan);
            for (int i = 0; i < 6; i++) e.key[i] = key[i];
        }
        return e.plan;
    }
};

// Shape-family rule.  A few rows against a large b -> one of two tiles that stream b.  Everything else -> the
// tile and K split that the cost model of the tiled kernel picks.
const Planned& choose(int m, int n, int k, int num_cus, bool may_split = true, bool epi = false) {
    static thread_local PlanMemo<Planned> memo;
    if (num_cus <= 0) num_cus = 256;
    return memo.get({m, n, k, num_cus, may_split, epi}, [&](Planned* out) {
        *out = {};
        if (skinny_shape(m, n, k)) choose_skinny(m, n, k, num_cus, out, may_split);
        else choose_tiled(m, n, k, num_cus, out, may_split, epi);
    });
}

// The same split with its sums in the kernel.
fp8bs_plan_t summed_in_kernel(int m, int n, int k, const fp8bs_plan_t& plan) {
    fp8bs_plan_t p{};
    fill_plan(m, n, k, plan.variant | plan.form * FORM1, plan.split_k, &p, 0, true);
    return p;
}

// The workspace that every form of a planned call finds room in: the flags and partial tiles of a sum shared out are no less than planes.
uint64_t useful_bytes(int m, int n, int k, const Planned& p) { return (p.share ? summed_in_kernel(m, n, k, p.plan) : p.plan).workspace_bytes; }

// Order of the tiles of a grouped call (the row counts themselves are on the device).  With a tile or more of
// rows per expert on average the tiles go expert by expert: the tile that holds an expert's last rows then runs
// beside the full tiles that read the same weights (32 experts of 1040 rows x 4096 x 7168: 956 us against 1014;
// configuration 5: 2-3 % faster).  With fewer rows every expert is one tile row and the call streams the weights;
// the order across the experts is then 0.7-1.2 % ahead (8 or 100 rows per expert), so it is kept there.
int group_order(int total_rows, int num_experts, int n) {
    return (long)total_rows >= 256L * num_experts ? fp8bs::ORDER_BY_EXPERT : fp8bs::turns_rounds(n) ? fp8bs::ORDER_TURNED : fp8bs::ORDER_ACROSS;
}

struct GroupedPlan { int tile, split; };

// The counters and partial tiles of a grouped K split, for as many tiles as the routing can give.
uint64_t grouped_bytes(const GroupedPlan& p, int experts, int rows, int n) {
    if (p.split <= 1) return 0;
    VariantInfo vi{};
    variant_info(p.tile, &vi);
    return (uint64_t)fp8bs::StreamK::SLOTS_OFF + (uint64_t)(fp8bs::grouped_slots_bound(rows, experts, vi.bm) * cdiv(n, vi.bn)) * (uint64_t)p.split * (uint64_t)vi.bm * (uint64_t)vi.bn * 4u;
}

bool can_split_grouped(const GroupedPlan& p, int experts, int rows, int n, int k) {
    VariantInfo vi{};
    if (!has_grouped_split(p.tile) || !variant_info(p.tile, &vi)) return false;
    return p.split >= 2 && p.split <= 255 && p.split <= k / KBLK && fp8bs::grouped_slots_bound(rows, experts, vi.bm) * cdiv(n, vi.bn) <= fp8bs::StreamK::MAX_GRID;
}

// The tile and K split of a grouped call.  The row counts themselves are on the device, so the model below works with
// averages: experts that get rows, tiles per such expert (its rows plus, on average, half of the 16 it may start late, and
// the last, partial tile), and the share of a tile's rows that exist - waves without rows only copy, so a tile with few
// rows takes its shorter time per K block, t_few.  Terms as in choose_tiled; bw is the rate in TB/s at which tiles of this
// width stream the experts' weights from HBM together (row segments of 256 bytes are taken best), shared by the tiles that
// read the same panel.  The constants are fits to the measured times of every (tile, split) on 210 shapes on MI355X (8, 16
// or 32 experts, 1 .. 4096 tokens to 2, 4 or 8 of them, N 512 .. 7168, K 512 .. 7168, log-uniform): picking by the model
// costs 2.2 % against the best of each shape in the geometric mean and takes 17 % off the rule it replaced (the 256x256
// tile above 32 rows per expert on average, 64x256 below): 194 tokens to 4 of 16 experts, 1299 x 5760: 90.8 -> 49.2 us;
// 801 to 4 of 8, 840 x 1664: 23.2 -> 15.0; 35 to 4 of 8, 1375 x 5504: 43.6 -> 22.8.
// split 0: as many partitions as finish soonest; else that many, {.., 1} if no tile can.
GroupedPlan make_grouped_plan(int experts, int rows, int n, int k, int num_cus, int split) {
    struct Cand { int tile; int rmax; double t_full, t_few, t_power, t_fixed, shared, bw; };
    const Cand cands[5] = {
        {FP8BS_VARIANT_T256x256, 1, 2.010, 1.259, 1.681, 6.01, 1.0, 5.18},
        {FP8BS_VARIANT_T256x128S3, 1, 1.122, 0.618, 0.605, 5.58, 1.0, 5.06},
        {FP8BS_VARIANT_T64x256S3, 1, 0.794, 0.578, 0.500, 5.09, 1.0, 5.32},
        {FP8BS_VARIANT_T64x256S3 | FORM1, 1, 0.728, 0.497, 0.661, 4.34, 1.0, 5.27},
        {FP8BS_VARIANT_T64x128 | FORM1, 2, 0.570, 0.313, 0.100, 3.59, 1.65, 4.02},
    };
    double unused = 1.0;                                           // (1 - 1/E)^rows: an expert's chance to get none
    for (int r = 0; r < rows && unused > 1e-3; r++) unused *= 1.0 - 1.0 / experts;
    const double active = experts * (1.0 - unused), average = rows / active;
    const int kbt = k / KBLK;
    // 128x256 tiles (fp8bs_tile_128x256s3.hip) by the two rules below, never where 64x256 tiles, second rows of them too, are all on the chip at once (300
    // tokens to 4 of 32, 1280 x 7168, 74.2 us, 128x256 77.6; 105 to 8 of 16, 2176 x 3584, 38.1 and 39.8).
    const long tall_tiles = (long)experts * cdiv(n, 256), cus = num_cus;
    const double share = (double)rows / experts;
    const double seconds = 1.0 + share * share / 6400.0;           // tile rows of 64 an expert: 1.06 at 20 rows, 1.64 at 64
    const bool tall_may = split <= 1 && tall_tiles * seconds > cus;
    GroupedPlan best{FP8BS_VARIANT_T256x256, 1};
    double best_cost = 0;
    // more: as many tiles as expected, times this
    auto model = [&](const Cand& c, int s, double more) {
        VariantInfo vi{};
        variant_info(c.tile, &vi);
        double slots = (average + 8.0) / vi.bm + 0.4;
        if (slots < 1.0) slots = 1.0;
        double fill = (average / slots + 24.0) / vi.bm;
        if (fill > 1.0) fill = 1.0;
        const double t_alone = c.t_few + (c.t_full - c.t_few) * fill;
        const double wgs = active * slots * more * (double)cdiv(n, vi.bn) * s, per_round = (double)num_cus * c.rmax, kb = (double)cdiv(kbt, s);
        auto t_block = [&](double w) {
            double t = t_alone * (w > num_cus && c.rmax > 1 ? c.shared : 1.0);
            const double power = c.t_power * fill * w / num_cus, stream = w * 128.0 * vi.bn / slots / (c.bw * 1e6);
            t = power > t ? power : t;
            return stream > t ? stream : t;
        };
        const double full = (double)(long)(wgs / per_round), rem = wgs - full * per_round;
        double cost = full * (c.t_fixed + kb * t_block(per_round));
        if (rem > 0.5) cost += c.t_fixed + kb * t_block(rem);
        if (s > 1) cost += 3.56 + 0.757e-6 * s * (double)rows * (double)n;
        return cost;
    };
    for (const Cand& c : cands) {
        for (int s = split ? split : 1; s <= (split ? split : 4); s++) {
            const GroupedPlan p{c.tile, s};
            if (s > 1 && !can_split_grouped(p, experts, rows, n, k)) break;
            // (partial tiles of 64 MB at most: beyond that a call has tiles enough without a split)
            if (s > 1 && !split && (kbt / s < 2 || grouped_bytes(p, experts, rows, n) > (64u << 20))) break;
            double cost = model(c, s, 1.0);
            // With more than 32 rows per expert the model flatters the smaller tiles against this one: 640 tokens to 4 of 32 experts,
            // 3664 x 5376, 128x128 in eight waves 217 us, this 169; 704 to 8 of 32, 2176 x 1280, 39.2 and 35.2; 931 to 8 of 16, 3806 x
            // 5888, 256x128 278, this 260.  Over 480 further shapes of the same ranges and wider ones any factor from 0.85 to 0.95 brings
            // the picks from 3.6 to 3.2 % behind the best, and from 37 to 19-25 those more than 5 % behind the rule before the model.
            if (c.tile == FP8BS_VARIANT_T256x256 && (long)rows > 32L * experts) cost *= 0.92;
            if (best_cost == 0 || cost < best_cost) { best = p; best_cost = cost; }
        }
    }
    // Some tens of rows an expert and weights that come from memory: one row of these tiles holds an expert where other tiles take two, or leave workgroups
    // without work. Up to 44 rows 64x256 is ahead by 1 to 4 % where no expert has more than 64, and as fast or faster by its second rows, whose weights an L2
    // holds, where these fit the last round; where they start one more it is far behind. 200 such calls, experts by chance and of shares that differ (a deviation
    // of scores of 0.5), tile rows that start no round: 0.98 and 0.99 of 64x256's speed, and left; that do: 0.98 and 1.09 (at most 1.44: 23 rows to each of 32 experts,
    // 4096 x 3712, shares up to 67, 106.8 and 88.1 us; 0.93 at worst), and taken. Against every other pick 1.14 to 1.17 times as fast (28 calls, at worst 0.88; 42
    // rows to each of 64, 4608 x 1024, 84.9 and 71.5), splits among them (10 shapes 1.01 to 1.10, one draw 0.98; the sum without a split is no further from 64 bits).
    // Above 44 rows some expert has more than 128 itself: only where an eighth more tiles takes no further round (512 tokens to 4 of 32, shares that differ, 3072 x 4096,
    // 112.9 and 92.4; where the rounds were full, 256 to 8 of 32, 4096 x 7168, 197.9, this 208.2).
    auto rounds = [&](double tiles) { return (long)__builtin_ceil(tiles / cus); };
    const bool streams = best.tile == FP8BS_VARIANT_T64x256S3 && best.split == 1;
    if (tall_may && fp8bs::weights_past_caches(experts, rows, n, k) && share > 16.0 && share <= 64.0
        && (share <= 44.0 ? !streams || rounds(tall_tiles * seconds) > rounds(tall_tiles) : rounds(tall_tiles + tall_tiles / 8) == rounds(tall_tiles))) return {FP8BS_VARIANT_T256x128S3 | FORM1, 1};
    // From 44 to 128 rows an expert one row of 128x256 tiles holds an expert of the average size. The constants are a fit (12 % off in the mean) to 420 drawn
    // calls (8 to 128 experts, 10 to 420 rows each, 512 .. 7168 x 512 .. 7168). It is taken where it is ahead by 4 % with a twentieth more tiles than
    // expected: the unequal shares that the averages hide cost it a round where the last is full. Of 833 further drawn calls of 16 to 132 rows 247 take it by one
    // of the rules, 214 of them by this one: 1.16 times as fast in the geometric mean of both (experts by chance 1.17, of shares that differ 1.15), 0.83 to 1.44. The worst
    // are unequal shares whose tiles start a round that the average does not (3216 rows to 32, 1344 x 640, 15.0 and 18.1 us). Splits that it takes the place of: 24 shapes,
    // 1.12 to 1.46 (1696 rows to 16, 2176 x 6656, 102.2 and 70.2). Beyond 128 rows the model errs too often: of the drawn calls it gains 2 %, and loses 12 to 21 % on some.
    const Cand tall{FP8BS_VARIANT_T256x128S3 | FORM1, 1, 0.960, 0.628, 0.637, 5.33, 1.0, 5.98};
    if (tall_may && share > 44.0 && share <= 128.0 && best_cost > 1.04 * std::max(model(tall, 1, 1.0), model(tall, 1, 1.05))) best = {tall.tile, 1};
    return best;
}
GroupedPlan choose_grouped(int experts, int rows, int n, int k, int num_cus, int split) {
    static thread_local PlanMemo<GroupedPlan> memo;
    if (num_cus <= 0) num_cus = 256;
    return memo.get({experts, rows, n, k, num_cus, split}, [&](GroupedPlan* plan) { *plan = make_grouped_plan(experts, rows, n, k, num_cus, split); });
}

// The value a flag takes in one call that deals K blocks: never zero, different from call to call (and, through
// the clock and the process id, from run to run), so that whatever an earlier call or an uninitialised workspace
// left in a flag is not mistaken for this call's.
unsigned long long next_nonce() {
    static std::atomic<unsigned long long> counter{0};
    static const unsigned long long seed = ((unsigned long long)std::chrono::steady_clock::now().time_since_epoch().count() * 0x9E3779B97F4A7C15ull)
                                           ^ ((unsigned long long)getpid() << 32);
    unsigned long long x = seed + (counter.fetch_add(1, std::memory_order_relaxed) + 1) * 0xD1342543DE82EF95ull;
    return x ? x : 1ull;
}

// Polls of one flag before a workgroup's wait gives up (each poll is a round trip to memory plus a short sleep,
// about a microsecond: the default is a quarter of a second or so).  FP8BS_STREAMK_SPIN overrides it; a negative
// value makes every such wait give up at once, which exercises the error path without a kernel that hangs.
int streamk_spin_limit() {
    static const int limit = [] {
        const char* e = getenv("FP8BS_STREAMK_SPIN");
        return e && *e ? atoi(e) : (1 << 18);
    }();
    return limit;
}

// Polls after which a workgroup of a K split summed in the kernel leaves its part of the sum to another: some tens of
// microseconds, where workgroups that started together arrive within a few.  (A negative FP8BS_STREAMK_SPIN: one look only.)
int sum_polls() { return streamk_spin_limit() < 0 ? 0 : 32; }

int check_common(const void* a, const void* b, const float* as, const float* bs, void* c, int m, int n, int k) {
    if (m < 0 || n < 0 || k < 0 || (k % KBLK) != 0) return FP8BS_ERR_BAD_SHAPE;
    if (m == 0 || n == 0) return FP8BS_OK;   // nothing to write
    if (!a || !b || !as || !bs || !c) {
        if (k == 0 && c) return FP8BS_OK;
        return FP8BS_ERR_NULL_POINTER;
    }
    if ((uint64_t)m * (uint64_t)k >= (1ull << 32) || (uint64_t)n * (uint64_t)k >= (1ull << 32)) return FP8BS_ERR_TOO_LARGE;
    if ((((uintptr_t)as | (uintptr_t)bs) & 3) != 0 || ((uintptr_t)c & 1) != 0) return FP8BS_ERR_BAD_SHAPE;   // element alignment
    return FP8BS_OK;
}

// Operands and output on 16-byte boundaries: what the streaming kernels need (aligned 8- and 16-byte stores
// of c, aligned copies).
bool vector_aligned(const void* a, const void* b, const void* c) {
    return ((((uintptr_t)a | (uintptr_t)b | (uintptr_t)c) & 15) == 0);
}

}  // namespace

// ---- built-in K-split scratch of fp8bs_gemm_noalloc ---------------------------------------------------
// Device memory that belongs to the library's code object: every GPU the library runs on holds its own
// copy, at its own address, until the process ends.  In host code the array's name is only a handle for
// hipGetSymbolAddress; the address it yields (looked up once per device, with that device current) is what
// kernels, copies and fills are given.
static __device__ __align__(256) unsigned char scratch[FP8BS_NOALLOC_SCRATCH_BYTES];
static void* scratch_ptr[fp8bs::MAX_DEVICES];

static int scratch_address(void** out, hipStream_t stream) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= fp8bs::MAX_DEVICES) return FP8BS_ERR_LAUNCH;
    void* p = __atomic_load_n(&scratch_ptr[dev], __ATOMIC_ACQUIRE);
    if (!p) {
        // the lookup is no stream operation: it must not fall into a capture (the caller makes one eager call first)
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(stream, &cap) != hipSuccess) { (void)hipGetLastError(); cap = hipStreamCaptureStatusNone; }
        if (cap != hipStreamCaptureStatusNone) return FP8BS_ERR_CAPTURE;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return FP8BS_ERR_LAUNCH;
        __atomic_store_n(&scratch_ptr[dev], p, __ATOMIC_RELEASE);     // the same value from every thread
    }
    *out = p;
    return FP8BS_OK;
}

extern "C" {

// 0.4.1: grouped calls take FP8BS_VARIANT_FORM(FP8BS_VARIANT_T256x128S3, 1).  0.4.0: a plan is (variant, form): fp8bs_plan_t::form in the place of a reserved word.
int fp8bs_version(void) { return 401; }

const char* fp8bs_strerror(int status) {
    switch (status) {
        case FP8BS_OK: return "success";
        case FP8BS_ERR_NULL_POINTER: return "a required pointer is NULL";
        case FP8BS_ERR_BAD_SHAPE: return "bad shape: m, n, k must be non-negative and k a multiple of 128 (or a pointer is not aligned to its element type)";
        case FP8BS_ERR_WORKSPACE: return "workspace missing or smaller than fp8bs_workspace_bytes()";
        case FP8BS_ERR_TOO_LARGE: return "operand exceeds the 4 GiB buffer-addressing limit (m*k or n*k >= 2^32)";
        case FP8BS_ERR_LAUNCH: return "kernel launch failed";
        case FP8BS_ERR_BAD_OFFSETS: return "grouped: num_experts must be positive";
        case FP8BS_ERR_BAD_VARIANT: return "unknown or inapplicable kernel variant";
        case FP8BS_ERR_CAPTURE: return "fp8bs_gemm_noalloc: the first call on a device looks up the built-in scratch and must be made outside stream capture";
        case FP8BS_ERR_TIMEOUT: return "a workgroup gave up waiting for another workgroup's partial tile (status word of the workspace); the output of that call is not valid";
        case FP8BS_ERR_SCRATCH_LIMIT: return "fp8bs_gemm_noalloc: the K split planned for this shape needs more than the built-in scratch (FP8BS_NOALLOC_SCRATCH_BYTES); use fp8bs_gemm with a caller workspace";
        default: return "unknown fp8bs status";
    }
}

int fp8bs_plan(int m, int n, int k, int num_cus, fp8bs_plan_t* out) {
    if (!out) return FP8BS_ERR_NULL_POINTER;
    if (m <= 0 || n <= 0 || k <= 0 || (k % KBLK) != 0) return FP8BS_ERR_BAD_SHAPE;
    if (num_cus <= 0) num_cus = fp8bs::device_cus();     // the current device's, 256 where there is none
    *out = choose(m, n, k, num_cus).plan;
    return FP8BS_OK;
}

size_t fp8bs_workspace_bytes(int m, int n, int k) {
    if (m <= 0 || n <= 0 || k <= 0 || (k % KBLK) != 0) return 0;
    return (size_t)useful_bytes(m, n, k, choose(m, n, k, fp8bs::device_cus()));
}

// A dense call, plain or with the silu-mul epilogue (epi 1: c has n/2 columns).
static int dense_call(const void* a, const void* b, const float* a_scale, const float* b_scale, void* c, void* ws, size_t ws_bytes,
                      int m, int n, int k, int variant, int split_k, int epi, void* stream) {
    int st = check_common(a, b, a_scale, b_scale, c, m, n, k);
    if (st != FP8BS_OK) return st;
    if (m == 0 || n == 0) return FP8BS_OK;
    hipStream_t s = (hipStream_t)stream;
    fp8bs_plan_t plan{};
    if (k == 0) variant = FP8BS_VARIANT_GENERIC;   // empty sum: the generic kernel writes zeros
    // Operands off the 16-byte grid and n off the 8-column grid: the tiled kernels take them in every mode
    // (the same instantiation as for rows of a, b and c that start anywhere); only the streaming kernels are
    // left out.  A workspace that starts off the 16-byte grid is used from its first 16-byte boundary on.
    const bool aligned = vector_aligned(a, b, c);
    if (ws && ((uintptr_t)ws & 15) != 0) {
        const size_t skip = 16 - ((uintptr_t)ws & 15);
        if (ws_bytes > skip) { ws = (char*)ws + skip; ws_bytes -= skip; }
        else { ws = nullptr; ws_bytes = 0; }
    }
    const bool simple = aligned && vector_shape(n);      // streaming kernels possible
    const int cus = fp8bs::device_cus();
    bool ready_planes = false;
    if (variant == FP8BS_VARIANT_AUTO) {
        const Planned planned = choose(m, n, k, cus, true, epi != 0);
        plan = planned.plan;
        const int tile = plan.variant | plan.form * FORM1;
        // (a forced split may be any: the small tiles of up to eight partitions give way to 64 x 64)
        if (split_k > 0) fill_plan(m, n, k, is_waves_tile(tile) ? FP8BS_VARIANT_T64x128 | FORM1 : tile, split_k & ~FP8BS_SPLIT_SUM_IN_KERNEL, &plan, 0, (split_k & FP8BS_SPLIT_SUM_IN_KERNEL) != 0);
        else if (split_k < 0) fill_plan(m, n, k, plan.variant, 1, &plan, streamk_grid(plan.variant, m, n, k, cus));   // (the first form only)
        // A captured launch cannot share out its sums: its flags' tag would not change from replay to replay.
        else if (fp8bs_plan_t p{}; planned.share && !plan.sum_in_kernel && ws && ws_bytes >= (p = summed_in_kernel(m, n, k, plan)).workspace_bytes && !fp8bs::is_capturing(s)) {
            plan = p;
            ready_planes = true;                 // a capture of this call takes the two launches
        }
        // the plan needs a workspace the caller did not bring: the best plan that needs none
        else if (plan.workspace_bytes > 0 && (!ws || ws_bytes < plan.workspace_bytes)) {
            // too small for the partial tiles of a sum in the kernel but not for the planes (tiles that overhang
            // the matrix): the same split with the reduce kernel
            if (plan.sum_in_kernel && ws && ws_bytes >= planes_bytes(m, n, plan.split_k)) fill_plan(m, n, k, tile, plan.split_k, &plan);
            else plan = choose(m, n, k, cus, false, epi != 0).plan;
        }
    } else {
        VariantInfo vi{};
        const int tile = forced_tile(variant);
        variant = variant_of(variant);
        if (!variant_info(tile, &vi) || is_grouped_tile(tile)) return FP8BS_ERR_BAD_VARIANT;
        if (is_streaming_variant(variant) && !simple) return FP8BS_ERR_BAD_VARIANT;
        if (is_streaming_variant(variant) && variant != FP8BS_VARIANT_SKINNY64x144 && (m % 4) != 0) return FP8BS_ERR_BAD_VARIANT;   // only the planner's width repairs a
        if (split_k < 0) {
            if (is_streaming_variant(variant) || variant == FP8BS_VARIANT_GENERIC || form_of(tile) != 0) return FP8BS_ERR_BAD_VARIANT;   // K blocks are dealt by the tiled kernel's first forms only
            fill_plan(m, n, k, variant, 1, &plan, streamk_grid(variant, m, n, k, cus));
        } else {
            const bool in_kernel = split_k > 0 && (split_k & FP8BS_SPLIT_SUM_IN_KERNEL) != 0;
            if (in_kernel && (is_streaming_variant(variant) || variant == FP8BS_VARIANT_GENERIC)) return FP8BS_ERR_BAD_VARIANT;   // the tiled kernel only
            fill_plan(m, n, k, tile, split_k > 0 ? (split_k & ~FP8BS_SPLIT_SUM_IN_KERNEL) : 1, &plan, 0, in_kernel);
            if (is_waves_tile(tile) && plan.split_k > WAVES_MAX) return FP8BS_ERR_BAD_VARIANT;
        }
    }
    const bool waves = is_waves_tile(plan.variant | plan.form * FORM1);
    if (plan.workspace_bytes > 0 && (!ws || ws_bytes < plan.workspace_bytes)) return FP8BS_ERR_WORKSPACE;
    if (epi && plan.variant != FP8BS_VARIANT_GENERIC && (!has_epilogue(plan.variant | plan.form * FORM1) || plan.stream_k > 0)) return FP8BS_ERR_BAD_VARIANT;

    fp8bs::GemmArgs g{};
    g.a = (const uint8_t*)a; g.b = (const uint8_t*)b; g.as = a_scale; g.bs = b_scale;
    g.c = (uint16_t*)c; g.ws = (float*)ws; g.row_offsets = nullptr;
    g.m = m; g.n = n; g.k = k; g.lda = m; g.nb = (n + 127) / 128;
    g.split_k = plan.split_k;
    g.kb_per_split = (int)cdiv(k / KBLK, plan.split_k);
    g.band_h = 4;
    g.num_experts = 0;
    g.epi = epi;
    if (ready_planes && fp8bs::launch_gemm(plan.variant | plan.form * FORM1, 1 | fp8bs::READY_ONLY, g, s) != hipSuccess) return FP8BS_ERR_LAUNCH;
    int mode = plan.split_k > 1 && !waves ? 1 : 0;
    if (plan.sum_in_kernel && plan.split_k > 1 && !waves) {
        mode = 4;
        g.sk_nonce = next_nonce();
        g.sk_spin = sum_polls();
    } else if (plan.stream_k > 0) {
        mode = 3;
        g.sk_grid = plan.stream_k;
        g.sk_nonce = next_nonce();
        g.sk_spin = streamk_spin_limit();
    }
    if (fp8bs::launch_gemm(plan.variant | plan.form * FORM1, mode, g, s) != hipSuccess) return FP8BS_ERR_LAUNCH;
    if (mode == 1) {
        if (fp8bs::launch_splitk_reduce(g.ws, g.c, (size_t)m * n, plan.split_k, epi, s) != hipSuccess) return FP8BS_ERR_LAUNCH;
    }
    return FP8BS_OK;
}

int fp8bs_gemm_ex(const void* a, const void* b, const float* a_scale, const float* b_scale,
                  void* c, void* ws, size_t ws_bytes, int m, int n, int k,
                  int variant, int split_k, void* stream) {
    return dense_call(a, b, a_scale, b_scale, c, ws, ws_bytes, m, n, k, variant, split_k, 0, stream);
}

int fp8bs_gemm(const void* a, const void* b, const float* a_scale, const float* b_scale,
               void* c, void* ws, size_t ws_bytes, int m, int n, int k, void* stream) {
    return fp8bs_gemm_ex(a, b, a_scale, b_scale, c, ws, ws_bytes, m, n, k, FP8BS_VARIANT_AUTO, 0, stream);
}

int fp8bs_gemm_noalloc(const void* a, const void* b, const float* a_scale, const float* b_scale,
                       void* c, int m, int n, int k, void* stream) {
    int st = check_common(a, b, a_scale, b_scale, c, m, n, k);
    if (st != FP8BS_OK) return st;
    if (m == 0 || n == 0) return FP8BS_OK;
    // the plan fp8bs_gemm would follow; its partial planes must fit the built-in array
    fp8bs_plan_t plan{};
    if (k > 0) {
        plan = choose(m, n, k, fp8bs::device_cus()).plan;
        uint64_t need = plan.workspace_bytes;
        if (plan.sum_in_kernel && planes_bytes(m, n, plan.split_k) < need) need = planes_bytes(m, n, plan.split_k);   // fp8bs_gemm_ex falls back to the planes
        if (need > (uint64_t)FP8BS_NOALLOC_SCRATCH_BYTES) return FP8BS_ERR_SCRATCH_LIMIT;
    }
    void* ws = nullptr;
    st = scratch_address(&ws, (hipStream_t)stream);
    if (st != FP8BS_OK) return st;
    // Every partial element that the sum reads is written by this call first, and a tile's counter in the head
    // of the array counts only arrivals that carry this call's tag, so nothing in the array has to start at zero.
    return fp8bs_gemm_ex(a, b, a_scale, b_scale, c, ws, (size_t)FP8BS_NOALLOC_SCRATCH_BYTES, m, n, k, FP8BS_VARIANT_AUTO, 0, stream);
}

// A grouped call, plain or with the silu-mul epilogue.
static int grouped_call(const void* a, const void* b, const float* a_scale, const float* b_scale, void* c, const int32_t* row_offsets,
                        int num_experts, int rows, int n, int k, int variant, int split_k, int epi, void* ws, size_t ws_bytes, void* stream) {
    if (num_experts <= 0) return FP8BS_ERR_BAD_OFFSETS;
    if (!row_offsets) return FP8BS_ERR_NULL_POINTER;
    if (split_k < 0) return FP8BS_ERR_BAD_VARIANT;               // K blocks are dealt in dense calls only
    split_k &= ~FP8BS_SPLIT_SUM_IN_KERNEL;                       // the only form a grouped split has
    int st = check_common(a, b, a_scale, b_scale, c, rows, n, k);
    if (st != FP8BS_OK) return st;
    if (rows == 0 || n == 0) return FP8BS_OK;
    if (ws && ((uintptr_t)ws & 15) != 0) {
        const size_t skip = 16 - ((uintptr_t)ws & 15);
        if (ws_bytes > skip) { ws = (char*)ws + skip; ws_bytes -= skip; }
        else { ws = nullptr; ws_bytes = 0; }
    }
    fp8bs::GemmArgs g{};
    g.a = (const uint8_t*)a; g.b = (const uint8_t*)b; g.as = a_scale; g.bs = b_scale;
    g.c = (uint16_t*)c; g.ws = (float*)ws; g.row_offsets = row_offsets;
    g.m = rows; g.n = n; g.k = k; g.lda = rows; g.nb = (n + 127) / 128;
    g.band_h = 4; g.num_experts = num_experts;
    g.order = group_order(rows, num_experts, n);
    g.epi = epi;
    GroupedPlan plan{forced_tile(variant), split_k > 1 ? split_k : 1};
    if (k == 0 && variant == FP8BS_VARIANT_AUTO) plan = {FP8BS_VARIANT_GENERIC, 1};
    else if (variant == FP8BS_VARIANT_AUTO) {
        plan = choose_grouped(num_experts, rows, n, k, fp8bs::device_cus(), split_k);
        if (split_k > 1 && plan.split != split_k) return FP8BS_ERR_BAD_VARIANT;      // no tile takes this split of this call
        if (plan.split > 1 && (!ws || ws_bytes < grouped_bytes(plan, num_experts, rows, n))) {
            if (split_k > 1) return FP8BS_ERR_WORKSPACE;
            plan = choose_grouped(num_experts, rows, n, k, fp8bs::device_cus(), 1);
        }
    } else {
        VariantInfo vi{};
        if (!variant_info(plan.tile, &vi) || is_streaming_variant(plan.tile) || is_waves_tile(plan.tile)) return FP8BS_ERR_BAD_VARIANT;   // no grouped mode in these kernels
        if (plan.tile != FP8BS_VARIANT_GENERIC && k == 0) return FP8BS_ERR_BAD_VARIANT;
        if (epi && plan.tile != FP8BS_VARIANT_GENERIC && !has_epilogue(plan.tile)) return FP8BS_ERR_BAD_VARIANT;
        if (plan.split > 1 && !can_split_grouped(plan, num_experts, rows, n, k)) return FP8BS_ERR_BAD_VARIANT;
        if (plan.split > 1 && (!ws || ws_bytes < grouped_bytes(plan, num_experts, rows, n))) return FP8BS_ERR_WORKSPACE;
    }
    g.split_k = plan.split;
    g.kb_per_split = (int)cdiv(k / KBLK, plan.split);
    if (plan.split > 1) { g.sk_nonce = next_nonce(); g.sk_spin = sum_polls(); }
    if (fp8bs::launch_gemm(plan.tile, plan.split > 1 ? 5 : 2, g, (hipStream_t)stream) != hipSuccess) return FP8BS_ERR_LAUNCH;
    return FP8BS_OK;
}

size_t fp8bs_grouped_workspace_bytes(int num_experts, int total_rows, int n, int k) {
    if (num_experts <= 0 || total_rows <= 0 || n <= 0 || k <= 0 || (k % KBLK) != 0) return 0;
    return (size_t)grouped_bytes(choose_grouped(num_experts, total_rows, n, k, fp8bs::device_cus(), 0), num_experts, total_rows, n);
}

size_t fp8bs_silu_mul_workspace_bytes(int rows, int n, int k) {
    if (rows <= 0 || n <= 0 || k <= 0 || (k % KBLK) != 0) return 0;
    return (size_t)useful_bytes(rows, n, k, choose(rows, n, k, fp8bs::device_cus(), true, true));
}

int fp8bs_gemm_grouped_ex(const void* a, const void* b, const float* a_scale, const float* b_scale,
                          void* c, const int32_t* row_offsets, int num_experts, int total_rows,
                          int n, int k, int variant, void* stream) {
    return grouped_call(a, b, a_scale, b_scale, c, row_offsets, num_experts, total_rows, n, k, variant, 1, 0, nullptr, 0, stream);
}

int fp8bs_gemm_grouped_ws(const void* a, const void* b, const float* a_scale, const float* b_scale,
                          void* c, const int32_t* row_offsets, int num_experts, int total_rows,
                          int n, int k, int variant, int split_k, void* ws, size_t ws_bytes, void* stream) {
    return grouped_call(a, b, a_scale, b_scale, c, row_offsets, num_experts, total_rows, n, k, variant, split_k, 0, ws, ws_bytes, stream);
}

int fp8bs_gemm_grouped(const void* a, const void* b, const float* a_scale, const float* b_scale,
                       void* c, const int32_t* row_offsets, int num_experts, int total_rows,
                       int n, int k, void* stream) {
    return fp8bs_gemm_grouped_ex(a, b, a_scale, b_scale, c, row_offsets, num_experts, total_rows, n, k, FP8BS_VARIANT_AUTO, stream);
}

int fp8bs_gemm_silu_mul_ws(const void* a, const void* b, const float* a_scale, const float* b_scale, void* h,
                           const int32_t* row_offsets, int num_experts, int rows, int n, int k,
                           int variant, int split_k, void* ws, size_t ws_bytes, void* stream) {
    if ((n & 1) != 0) return FP8BS_ERR_BAD_SHAPE;
    if (split_k < 0) return FP8BS_ERR_BAD_VARIANT;               // K blocks are dealt without an epilogue only
    // any even n and any operand alignment: rows of h that do not keep 16-byte stores aligned are stored in pieces
    if (row_offsets)
        return grouped_call(a, b, a_scale, b_scale, h, row_offsets, num_experts, rows, n, k, variant, split_k, 1, ws, ws_bytes, stream);
    return dense_call(a, b, a_scale, b_scale, h, ws, ws_bytes, rows, n, k, variant, split_k, 1, stream);
}

int fp8bs_gemm_silu_mul(const void* a, const void* b, const float* a_scale, const float* b_scale, void* h,
                        const int32_t* row_offsets, int num_experts, int rows, int n, int k, void* stream) {
    return fp8bs_gemm_silu_mul_ws(a, b, a_scale, b_scale, h, row_offsets, num_experts, rows, n, k, FP8BS_VARIANT_AUTO, 0, nullptr, 0, stream);
}

}  // extern "C"
