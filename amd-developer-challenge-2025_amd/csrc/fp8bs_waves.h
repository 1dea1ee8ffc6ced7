// Block-scaled FP8 product for small outputs: every wave of a workgroup multiplies the workgroup's whole tile, over a
// partition of K of its own, with no barrier until the partitions meet.
//
// A small product is a chain - first copies, K blocks, output - on a chip that is nearly empty, and gemm_tr_kernel's K loop
// adds a barrier and a shared wait to every link: 49 x 1280 x 1024, 6.8 us of which an empty launch is 2.5.  Here a wave copies
// its K block into LDS of its own, waits for its own copies only (vmcnt), reads the operands, and sends for its next block
// while it multiplies; the eight waves' chains run side by side and drift apart, so one's waits are covered by the others.
// K blocks of a tile are taken eight at a time, and the code is short (the instruction cache is cold at every
// launch's start).  The partitions are the K split's: partition z holds kb_per_split blocks from z * kb_per_split on, and
// the sums meet in LDS in ascending order of K, so c has the bits of the same split on any other tile.
// IN_ORDER, up to one K block a wave: the waves leave the matrix cores' results and the scales, and the fold - the same fused
// multiply-adds, in ascending K - is done where they meet, so c has the bits of the unsplit sum.
// What bounds it with many tiles: requests at the L2, of which its small tiles make more per product than the others (about
// half a request per clock and CU whatever its length): 1024 x 1536 x 7168 in 32 x 64 tiles 61 us against 26.
// Measured (us, operands from the caches; before, in gemm_tr_kernel): 256 x 512 x 1024 3.8 (5.2), 49 x 1280 x 1024 3.7 (6.8), 1 x 1088 x
// 1664 4.1 (7.9), 18 x 1408 x 1920 5.3 (8.0), 311 x 640 x 512 3.7 (5.5).
#pragma once
#include "fp8bs_tiled.h"

namespace fp8bs {

template <int WM, int WN, int NW>
struct WavesCfg {
    static constexpr int MT = WM / 16, NT = WN / 16, CPR_A = WM / 16, CPR_B = WN / 16;
    static constexpr int A_BYTES = KBLK * WM, B_BYTES = KBLK * WN, REGION = A_BYTES + B_BYTES;
    static constexpr int LDS_BYTES = NW * REGION, NTHREADS = NW * 64;
    static constexpr int A_COPIES = A_BYTES / 1024, B_COPIES = B_BYTES / 1024, NCOPIES = A_COPIES + B_COPIES;
    static_assert(LDS_BYTES <= 160 * 1024, "LDS");
    static_assert(WM % 16 == 0 && 128 % WN == 0, "whole MFMA tiles; one b_scale value a block");
    static_assert(MT * NT * 1024 + WM * 4 <= REGION, "a wave's sums and its block's scales fit its region");
    static_assert((CPR_A & (CPR_A - 1)) == 0 && (CPR_B & (CPR_B - 1)) == 0 && CPR_A <= 4 && CPR_B <= 4, "a copy of 64 chunks is whole swizzle periods of 16 k rows");
};

template <int WM, int WN, int NW, int EPI, bool TAILS, bool IN_ORDER>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(2)))
void gemm_waves_kernel(const GemmArgs p) {
    using C = WavesCfg<WM, WN, NW>;
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, i16 = lane & 15;

    const int tiles_m = (p.m + WM - 1) / WM, tiles_n = (p.n + WN - 1) / WN;
    int tm, tn;
    band_tile(xcd_virtual_id(blockIdx.x, gridDim.x), tiles_m, tiles_n, p.band_h, tm, tn);
    const int m0 = __builtin_amdgcn_readfirstlane(tm * WM), n0 = __builtin_amdgcn_readfirstlane(tn * WN);
    const int kbt = p.k / KBLK;
    const int kb_begin = wave < p.split_k ? wave * p.kb_per_split : kbt;
    const int kb_end = kb_begin + p.kb_per_split < kbt ? kb_begin + p.kb_per_split : kbt;

    const uint32_t a_bytes = (uint32_t)p.k * (uint32_t)p.lda, b_bytes = (uint32_t)p.k * (uint32_t)p.n;
    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)p.a, 0, a_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t b_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)p.b, 0, b_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t as_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)p.as, 0, (uint32_t)kbt * (uint32_t)p.lda * 4u, 0x00020000);
    const __amdgpu_buffer_rsrc_t bs_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)p.bs, 0, (uint32_t)kbt * (uint32_t)p.nb * 4u, 0x00020000);

    // ---- copies: lane l of copy q fills chunk slot 64 q + l of the wave's region; the lanes' (k row, chunk) pattern is the same in
    //      all, the rest of the address uniform.  Chunks beyond the matrix: as in gemm_tr_kernel's copy plan ----
    const int kr_a = lane / C::CPR_A, kr_b = lane / C::CPR_B;
    const int col_a = m0 + 16 * stored_to_chunk<C::CPR_A>(lane % C::CPR_A, swz_of_krow<C::CPR_A>(kr_a));
    const int col_b = n0 + 16 * stored_to_chunk<C::CPR_B>(lane % C::CPR_B, swz_of_krow<C::CPR_B>(kr_b));
    const uint32_t a_voff = col_a >= p.m && a_bytes < 0x80000000u ? a_bytes : (uint32_t)kr_a * (uint32_t)p.lda + (uint32_t)(col_a < p.lda ? col_a : m0);
    const uint32_t b_voff = col_b >= p.n && b_bytes < 0x80000000u ? b_bytes : (uint32_t)kr_b * (uint32_t)p.n + (uint32_t)(col_b < p.n ? col_b : n0);
    const uint32_t a_kstep = (uint32_t)KBLK * (uint32_t)p.lda, b_kstep = (uint32_t)KBLK * (uint32_t)p.n;
    unsigned char* const region = lds + wave * C::REGION;
    const uint32_t region_base = (uint32_t)(size_t)(__attribute__((address_space(3))) unsigned char*)lds + wave * C::REGION;
    auto issue_one = [&](int kb, auto q_tag) {
        constexpr int q = decltype(q_tag)::value;
        if constexpr (q < C::A_COPIES)
            copy16_global_to_lds(a_rsrc, region_base + q * 1024, a_voff, (uint32_t)kb * a_kstep + (uint32_t)(q * (64 / C::CPR_A)) * (uint32_t)p.lda);
        else if constexpr (q < C::NCOPIES) {
            constexpr int qb = q - C::A_COPIES;
            copy16_global_to_lds(b_rsrc, region_base + q * 1024, b_voff, (uint32_t)kb * b_kstep + (uint32_t)(qb * (64 / C::CPR_B)) * (uint32_t)p.n);
        }
    };
    // ---- scales, to registers (lane: its row of every m tile), sent ahead of their block's copies ----
    const uint32_t as_voff = (uint32_t)(m0 + i16) * 4u;
    float as_next[C::MT], bs_next;
    auto load_scales = [&](int kb) {
#pragma unroll
        for (int t = 0; t < C::MT; t++)
            as_next[t] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(as_rsrc, as_voff + t * 64u, (uint32_t)kb * (uint32_t)p.lda * 4u, 0));
        bs_next = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(bs_rsrc, (uint32_t)(n0 / 128) * 4u, (uint32_t)kb * (uint32_t)p.nb * 4u, 0));
    };

    // ---- operand reads: as in gemm_tr_kernel ----
    const int krow_lane = 8 * g + (i16 >> 1);
    const int swz_a = swz_of_krow<C::CPR_A>(krow_lane), swz_b = swz_of_krow<C::CPR_B>(krow_lane);
    const unsigned char* const a_lane = region + krow_lane * WM + (i16 & 1) * 8;
    const unsigned char* const b_lane = region + C::A_BYTES + krow_lane * WN + (i16 & 1) * 8;
    auto read_a = [&](v8i& dst, int t) {
        const unsigned char* q = a_lane + (chunk_to_stored<C::CPR_A>(t, swz_a) << 4);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            v2i x = __builtin_amdgcn_ds_read_tr8_b64_v2i32(LDS_V2I(q + j * 32 * WM));
            dst[2 * j] = x[0]; dst[2 * j + 1] = x[1];
        }
    };
    auto read_b = [&](v8i& dst, int u) {
        const unsigned char* q = b_lane + (chunk_to_stored<C::CPR_B>(u, swz_b) << 4);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            v2i x = __builtin_amdgcn_ds_read_tr8_b64_v2i32(LDS_V2I(q + j * 32 * WN));
            dst[2 * j] = x[0]; dst[2 * j + 1] = x[1];
        }
    };

    v4f acc[C::MT][C::NT];
#pragma unroll
    for (int t = 0; t < C::MT; t++)
#pragma unroll
        for (int u = 0; u < C::NT; u++) acc[t][u] = (v4f){0.f, 0.f, 0.f, 0.f};

    [[maybe_unused]] float sc[C::MT];                      // IN_ORDER: the scales of the wave's block
    auto k_block = [&](int kb, auto next_tag) {
        constexpr bool NEXT = decltype(next_tag)::value;
        constexpr int STEPS = C::MT * C::NT, LAG = 3, RING = 4;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");              // this wave's copies of the block have landed
        if constexpr (TAILS && !NEXT) {
            if (kb == kbt - 1) {
                // the last one to three bytes of a and b, which the copies' dword range check cuts off (see gemm_tr_kernel)
                auto patch = [&](unsigned char* tile, auto cpr_tag, const uint8_t* src, uint32_t ld, int x0) {
                    constexpr int CPR = decltype(cpr_tag)::value;
                    const uint32_t end = (uint32_t)p.k * ld;
                    if (lane < 3) {
                        const uint32_t cand = tail_candidate(3u - lane, ld, (uint32_t)p.k);
                        const int x = (int)(cand & 0x1FFFFFFFu) - x0, kl = KBLK - 3 + (int)((cand >> 29) & 3u);
                        if ((cand >> 31) != 0 && x >= 0 && x < CPR * 16)
                            tile[kl * CPR * 16 + (chunk_to_stored<CPR>(x >> 4, swz_of_krow<CPR>(kl)) << 4) + (x & 15)] = src[end - 3u + lane];
                    }
                };
                if ((p.lda & 3) != 0) patch(region, std::integral_constant<int, C::CPR_A>{}, p.a, (uint32_t)p.lda, m0);
                if ((p.n & 3) != 0) patch(region + C::A_BYTES, std::integral_constant<int, C::CPR_B>{}, p.b, (uint32_t)p.n, n0);
            }
        }
        v8i areg[C::MT], breg[C::NT];
#pragma unroll
        for (int t = 0; t < C::MT; t++) read_a(areg[t], t);
#pragma unroll
        for (int u = 0; u < C::NT; u++) read_b(breg[u], u);
        float scale[C::MT];
#pragma unroll
        for (int t = 0; t < C::MT; t++) { scale[t] = as_next[t] * bs_next; if constexpr (IN_ORDER) sc[t] = scale[t]; }
        __builtin_amdgcn_sched_barrier(0);
        v4f ring[RING];
        constexpr int FROM = C::MT < STEPS ? C::MT : STEPS - 1;           // the step before which the reads are awaited and the copies begin
        constexpr int PER_STEP = (C::NCOPIES + STEPS - FROM - 1) / (STEPS - FROM) < 2 ? 2 : (C::NCOPIES + STEPS - FROM - 1) / (STEPS - FROM);
        auto step = [&](auto s_tag) {
            constexpr int s = decltype(s_tag)::value;
            if constexpr (s < STEPS) {
                constexpr int u = s / C::MT, t = s % C::MT;
                if constexpr (NEXT && s == FROM) {
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");    // the block is in registers: its place is free for the next
                    load_scales(kb + 1);
                }
                if constexpr (NEXT && s >= FROM) {
                    [&]<int... Q>(std::integer_sequence<int, Q...>) {
                        (issue_one(kb + 1, std::integral_constant<int, (s - FROM) * PER_STEP + Q>{}), ...);
                    }(std::make_integer_sequence<int, PER_STEP>{});
                }
                const v4f z = {0.f, 0.f, 0.f, 0.f};
                ring[s % RING] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(breg[u], areg[t], z, 0, 0, 0, 0, 0, 0);
            }
            if constexpr (s >= LAG) {
                constexpr int sp = s - LAG, u = sp / C::MT, t = sp % C::MT;
#pragma unroll
                for (int r = 0; r < 4; r++) acc[t][u][r] = IN_ORDER ? ring[sp % RING][r] : __builtin_fmaf(ring[sp % RING][r], scale[t], acc[t][u][r]);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        [&]<int... S>(std::integer_sequence<int, S...>) {
            (step(std::integral_constant<int, S>{}), ...);
        }(std::make_integer_sequence<int, STEPS + LAG>{});
    };

    if (kb_begin < kb_end) {
        load_scales(kb_begin);
        [&]<int... Q>(std::integer_sequence<int, Q...>) {
            (issue_one(kb_begin, std::integral_constant<int, Q>{}), ...);
        }(std::make_integer_sequence<int, C::NCOPIES>{});
        int kb = kb_begin;
        for (; kb + 1 < kb_end; kb++) k_block(kb, std::true_type{});
        k_block(kb, std::false_type{});
    }

    // ---- the partitions meet, ascending in K: every wave leaves its sums in its region; a thread then adds eight
    //      columns of a row.  Slots of a 16 x 16 piece are permuted so that neither side conflicts ----
    const int ldc = EPI == 1 ? p.n / 2 : p.n;
    const int S = p.split_k;
    if (wave < S) {
#pragma unroll
        for (int t = 0; t < C::MT; t++)
#pragma unroll
            for (int u = 0; u < C::NT; u++) *(v4f*)(region + (t * C::NT + u) * 1024 + (16 * g + (i16 ^ ((4 * u + g) & 15))) * 16) = acc[t][u];
        if constexpr (IN_ORDER)
            if (lane < 16)
#pragma unroll
                for (int t = 0; t < C::MT; t++) *(float*)(region + C::MT * C::NT * 1024 + (16 * t + i16) * 4) = sc[t];
    }
    __syncthreads();
    constexpr int PER_ROW = 2 * C::NT, UNITS = WM * PER_ROW;               // groups of eight columns
#pragma unroll
    for (int base = 0; base < UNITS; base += NW * 64) {
        const int id = base + tid;
        if (id < UNITS) {
            const int r = id / PER_ROW, cu = id % PER_ROW, i = r & 15, u = cu >> 1, g0 = 2 * (cu & 1);
            const unsigned char* const piece = lds + ((r >> 4) * C::NT + u) * 1024;
            const unsigned char* const src0 = piece + (16 * g0 + (i ^ ((4 * u + g0) & 15))) * 16;
            const unsigned char* const src1 = piece + (16 * (g0 + 1) + (i ^ ((4 * u + g0 + 1) & 15))) * 16;
            v4f s0 = *(const v4f*)src0, s1 = *(const v4f*)src1;
            if constexpr (IN_ORDER) {
                const unsigned char* const scales = lds + C::MT * C::NT * 1024 + r * 4;
                auto fold = [&](int z, v4f p0, v4f p1) {
                    const float f = *(const float*)(scales + z * C::REGION);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        s0[e] = __builtin_fmaf(p0[e], f, z == 0 ? 0.f : s0[e]);
                        s1[e] = __builtin_fmaf(p1[e], f, z == 0 ? 0.f : s1[e]);
                    }
                };
                fold(0, s0, s1);
                if (S == NW) {
#pragma unroll
                    for (int z = 1; z < NW; z++) fold(z, *(const v4f*)(src0 + z * C::REGION), *(const v4f*)(src1 + z * C::REGION));
                } else {
                    for (int z = 1; z < S; z++) fold(z, *(const v4f*)(src0 + z * C::REGION), *(const v4f*)(src1 + z * C::REGION));
                }
            } else if (S == NW) {
#pragma unroll
                for (int z = 1; z < NW; z++) { s0 += *(const v4f*)(src0 + z * C::REGION); s1 += *(const v4f*)(src1 + z * C::REGION); }
            } else {
                for (int z = 1; z < S; z++) { s0 += *(const v4f*)(src0 + z * C::REGION); s1 += *(const v4f*)(src1 + z * C::REGION); }
            }
            const int row = m0 + r;
            if (row < p.m) {
                if constexpr (EPI == 1) {
                    const int col = n0 / 2 + u * 8 + (cu & 1) * 4;
                    uint16_t* dst = p.c + (size_t)row * ldc + col;
                    const v2u o = {pack_bf16x2(silu_mul(s0[0], s0[1]), silu_mul(s0[2], s0[3])), pack_bf16x2(silu_mul(s1[0], s1[1]), silu_mul(s1[2], s1[3]))};
                    if (!TAILS) { if (col < ldc) *(v2u*)dst = o; }
                    else
#pragma unroll
                        for (int e = 0; e < 4; e++) if (col + e < ldc) dst[e] = (uint16_t)(o[e >> 1] >> (16 * (e & 1)));
                } else {
                    const int col = n0 + u * 16 + (cu & 1) * 8;
                    uint16_t* dst = p.c + (size_t)row * ldc + col;
                    const v4u o = {pack_bf16x2(s0[0], s0[1]), pack_bf16x2(s0[2], s0[3]), pack_bf16x2(s1[0], s1[1]), pack_bf16x2(s1[2], s1[3])};
                    if (!TAILS) { if (col < ldc) *(v4u*)dst = o; }
                    else {
                        typedef v4u v4u_any __attribute__((aligned(2)));
                        if (col + 8 <= ldc) *(v4u_any*)dst = o;
                        else
#pragma unroll
                            for (int e = 0; e < 8; e++) if (col + e < ldc) dst[e] = (uint16_t)(o[e >> 1] >> (16 * (e & 1)));
                    }
                }
            }
        }
    }
}

template <int WM, int WN, int NW, int EPI>
static inline hipError_t launch_waves(const GemmArgs& a, hipStream_t stream) {
    using C = WavesCfg<WM, WN, NW>;
    const int out_cols = EPI == 1 ? a.n / 2 : a.n;
    const bool tails = (a.lda & 3) != 0 || (a.n & 7) != 0 || (out_cols & 7) != 0 || (((uintptr_t)a.a | (uintptr_t)a.b | (uintptr_t)a.c) & 15) != 0;
    // an unsplit sum of as many K blocks as waves or fewer: one block a wave, folded in order where they meet
    const int kbt = a.k / KBLK;
    const bool in_order = a.split_k == 1 && kbt > 1 && kbt <= NW;
    GemmArgs args = a;
    if (in_order) { args.split_k = kbt; args.kb_per_split = 1; }
    void (*kern)(const GemmArgs) = in_order ? (tails ? gemm_waves_kernel<WM, WN, NW, EPI, true, true> : gemm_waves_kernel<WM, WN, NW, EPI, false, true>)
                                            : (tails ? gemm_waves_kernel<WM, WN, NW, EPI, true, false> : gemm_waves_kernel<WM, WN, NW, EPI, false, false>);
    static int raised[4][MAX_DEVICES];
    hipError_t e = raise_lds_limit((const void*)kern, C::LDS_BYTES, raised[(tails ? 1 : 0) + (in_order ? 2 : 0)]);
    if (e != hipSuccess) return e;
    const long tiles = (long)((a.m + WM - 1) / WM) * ((a.n + WN - 1) / WN);
    hipLaunchKernelGGL(kern, dim3((unsigned)tiles), dim3(C::NTHREADS), C::LDS_BYTES, stream, args);
    return hipGetLastError();
}

}  // namespace fp8bs
