// Block quantisers that produce the operands of the FP8 block-scaled GEMM directly in its storage
// layout, for gfx950 (MI355X).
//
// The reference has no quantiser: its operands arrive quantised from the harness
// (1-amd-fp8-mm/0-amd-fp8-mm-new-begins.py:66-77 describes what arrives).  These kernels are the step
// in front of the GEMM, turning a row-major [rows][K] fp32 or bf16 matrix into
//   q      : e4m3fn, K rows of `rows` bytes      q[kk * rows + i]          (the layout of a and b,
//   scale  : fp32                                                           amd-fp8-mm-submission.py:66-75)
//     per row and 128-wide K block (activations, a_scale[(kk/128) * rows + i]), or
//     per 128x128 block           (weights,     b_scale[(kk/128) * NB + i/128], NB = ceil(rows/128)).
// Rule, bit for bit: scale = max(max|x| / 448, 1e-12) in fp32, q = round-to-nearest-even e4m3fn of
// clamp(x / scale, -448, 448) with a correctly rounded fp32 division.
//
// One workgroup = 32, 64 or 128 rows x 128 k (one K block).  Every lane loads four k of four rows (8- or 16-byte
// loads along k, 32 lanes cover a row's block), the per-row maxima are reduced across those 32 lanes with each lane of a
// quad ending up with one of the four rows, whose scale and reciprocal it works out for the other three; the four rows'
// bytes are transposed 4x4 in registers (v_perm_b32) so that a dword holds four consecutive rows of one k, and the tile is
// staged in LDS ([128 k][rows], padded by 4 bytes) so that the global stores are 16 bytes per lane, on any byte.
// Bound by HBM where the matrix is large (4096 x 7168 bf16: 19.9 us, 88 MB, 4.4 TB/s; a 1 GiB copy runs at 5.1), by the
// vector ALU where the rows are gathered: about 9 instructions per value.  With the scale worked out by all 32 lanes of
// a row, two remainder corrections for bf16, a clamp and a sign repair it took 18 (4096 -> 32768 x 7168: 116 us, now 88).
// An optional row map gathers input rows (out row i = in row row_map[i]): the expert-contiguous
// permutation of MoE tokens (2-amd-moe/3-amd-fp8-moe-hip-myhgemm.py:174-191 does it as a copy of its
// own) then costs nothing extra.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>

#include "fp8bs.h"
#include "fp8bs_kernels.h"

namespace fp8bs {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));

struct QuantArgs {
    const void* x;
    const int32_t* row_map;   // may be null
    uint8_t* q;
    float* scale;
    int64_t ldx;              // elements between input rows
    int rows, k, src_rows;    // output rows, K, rows of the input matrix (row_map targets)
    int nb;                   // per-block mode: ceil(rows/128)
    int row0;                 // first row of this launch
};

static constexpr int TK = 128;

// accesses on any byte
typedef v4i v4i_any __attribute__((aligned(1)));
typedef v2i v2i_any __attribute__((aligned(1)));
typedef uint32_t u32_any __attribute__((aligned(1)));
typedef uint16_t u16_any __attribute__((aligned(1)));

__device__ __forceinline__ v4f cvt4(v4i r, const float*) { return __builtin_bit_cast(v4f, r); }
__device__ __forceinline__ v4f cvt4(v2i r, const uint16_t*) {      // four bf16
    v4f o;
    o[0] = __builtin_bit_cast(float, (uint32_t)r[0] << 16);
    o[1] = __builtin_bit_cast(float, (uint32_t)r[0] & 0xFFFF0000u);
    o[2] = __builtin_bit_cast(float, (uint32_t)r[1] << 16);
    o[3] = __builtin_bit_cast(float, (uint32_t)r[1] & 0xFFFF0000u);
    return o;
}
// four k of one row; an offset of 0xFFFFFFFF is out of range for the buffer and reads zeros
__device__ __forceinline__ v4f load4(__amdgpu_buffer_rsrc_t rsrc, uint32_t byte_off, const float* tag) {
    return cvt4(__builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rsrc, byte_off, 0, 0)), tag);
}
__device__ __forceinline__ v4f load4(__amdgpu_buffer_rsrc_t rsrc, uint32_t byte_off, const uint16_t* tag) {
    return cvt4(__builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(rsrc, byte_off, 0, 0)), tag);
}

__device__ __forceinline__ uint32_t umax(uint32_t a, uint32_t b) { return a > b ? a : b; }
template <int CTRL> __device__ __forceinline__ uint32_t dpp(uint32_t v) { return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, true); }
// Max over the 32 lanes that share four rows, m[r] being the lane's own of row r; every lane gets the one of row (lane & 3).
// Steps 1 and 2 over a quad on all four rows, then 4, 8 (rotations by 4 and by 8, which keep lane & 3) and 16 on one.  On the bit
// patterns of |x|: for non-negative floats the integer order is the float order, and every NaN pattern is above every number,
// so a NaN in the row comes out as the maximum (torch.amax propagates NaN the same way).
__device__ __forceinline__ uint32_t rowmax32(const uint32_t m[4], int lane) {
    uint32_t q[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        q[r] = umax(m[r], dpp<0xB1>(m[r]));               // quad_perm [1,0,3,2]
        q[r] = umax(q[r], dpp<0x4E>(q[r]));               // quad_perm [2,3,0,1]
    }
    const uint32_t lo = (lane & 1) ? q[1] : q[0], hi = (lane & 1) ? q[3] : q[2];
    uint32_t v = (lane & 2) ? hi : lo;
    v = umax(v, dpp<0x124>(v));                           // row_ror:4
    v = umax(v, dpp<0x128>(v));                           // row_ror:8
    return umax(v, (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, 0x401F));               // lane ^ 16
}

// Correctly rounded x / s for finite s >= 1e-12 and |x / s| < 2^96: the arithmetic of the IEEE
// division sequence (reciprocal refined once, quotient corrected by its remainder, all by fused multiply-add)
// without its range scaling, which only acts on quotients or operands at the ends of the exponent
// range; there the result is a zero after conversion to e4m3fn either way.  `y` is refine_rcp(s).
// STEPS corrections: two in general; one where x and the block's maximum are bf16 - 8-bit significands, for all
// 128 x 128 of which it was checked to give the correctly rounded quotient, for the reciprocal rounded correctly and for its
// neighbours on both sides (tests/test_quant_division.py).  The remainder is taken as s*q - x, so that -0 stays -0.
__device__ __forceinline__ float refine_rcp(float s) {
    float y = __builtin_amdgcn_rcpf(s);
    float e = __builtin_fmaf(-s, y, 1.0f);
    return __builtin_fmaf(e, y, y);
}
template <int STEPS> __device__ __forceinline__ float div_by(float x, float s, float y) {
    float q = x * y;
#pragma unroll
    for (int i = 0; i < STEPS; i++) q = __builtin_fmaf(-__builtin_fmaf(s, q, -x), y, q);
    return q;
}
// scale of a block from the bit pattern of its max |x|
__device__ __forceinline__ float scale_of(uint32_t amax_bits) {
    const float amax = __builtin_bit_cast(float, amax_bits);
    float s = div_by<2>(amax, 448.f, refine_rcp(448.f));
    s = s < 1e-12f ? 1e-12f : s;
    return amax_bits >= 0x7F800000u ? amax : s;            // inf stays inf, NaN stays NaN
}

__device__ __forceinline__ float clamp448(float v) {
    // NaN stays NaN (becomes the e4m3fn NaN code), like clamp_ followed by the cast in torch
    return v != v ? v : __builtin_fminf(__builtin_fmaxf(v, -448.f), 448.f);
}

// four fp32 -> four e4m3fn codes in one dword (byte j = value j), round to nearest even
__device__ __forceinline__ uint32_t cvt4_e4m3fn(v4f v) {
    int w = __builtin_amdgcn_cvt_pk_fp8_f32(v[0], v[1], 0, false);
    w = __builtin_amdgcn_cvt_pk_fp8_f32(v[2], v[3], w, true);
    return (uint32_t)w;
}

// bits of the largest |x| of the lane's four values, and those values widened
__device__ __forceinline__ uint32_t absmax4(v4f x) {
    const v4i b = __builtin_bit_cast(v4i, x) & 0x7FFFFFFF;
    return umax(umax((uint32_t)b[0], (uint32_t)b[1]), umax((uint32_t)b[2], (uint32_t)b[3]));
}

// PER_BLOCK false: one scale per row and K block (activations); true: one per 128x128 block (weights)
// ROWS: rows of a workgroup, a multiple of 32 (PER_BLOCK: 128)
template <typename T, bool PER_BLOCK, bool HAS_MAP, int ROWS>
__global__ __launch_bounds__(256)
void quantize_kernel(const QuantArgs p) {
    constexpr int ITERS = ROWS / 32, LD = ROWS + 4;      // LDS row pitch in bytes (an odd number of dwords: spreads banks)
    static_assert(!PER_BLOCK || ROWS == 128, "a block's maximum is taken over one workgroup");
    __shared__ __attribute__((aligned(16))) unsigned char tile[TK * LD];
    __shared__ float row_scale[ROWS];
    __shared__ uint32_t wave_max[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 5, l = lane & 31;
    const int kb = blockIdx.x, m0 = p.row0 + blockIdx.y * ROWS;
    __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)p.x, 0, (uint32_t)((size_t)p.src_rows * (size_t)p.ldx * sizeof(T)), 0x00020000);

    // ---- load: iteration it, row group rg = it*8 + wave*2 + g holds rows 4rg .. 4rg+3 ----
    v4f v[ITERS][4];
    uint32_t rmax[ITERS];                     // of row 4rg + (lane & 3)
    const uint32_t col_off = (uint32_t)((kb * TK + 4 * l) * sizeof(T));
    const uint32_t row_pitch = (uint32_t)(p.ldx * sizeof(T));
    int src[ITERS][4];
    // all row-map entries first, then all data loads: neither waits for the other one by one
#pragma unroll
    for (int it = 0; it < ITERS; it++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = m0 + 4 * (it * 8 + wave * 2 + g) + r;
            if (HAS_MAP) src[it][r] = p.row_map[row < p.rows ? row : p.rows - 1];
            else src[it][r] = row;
        }
#pragma unroll
    for (int it = 0; it < ITERS; it++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = m0 + 4 * (it * 8 + wave * 2 + g) + r;
            const bool ok = row < p.rows && (uint32_t)src[it][r] < (uint32_t)p.src_rows;
            const uint32_t off = ok ? (uint32_t)src[it][r] * row_pitch + col_off : 0xFFFFFFFFu;
            v[it][r] = load4(rsrc, off, (const T*)nullptr);
        }
    // ---- per-row max |x| ----
#pragma unroll
    for (int it = 0; it < ITERS; it++) {
        const uint32_t m[4] = {absmax4(v[it][0]), absmax4(v[it][1]), absmax4(v[it][2]), absmax4(v[it][3])};
        rmax[it] = rowmax32(m, lane);
    }
    float bscale = 0.f;
    if (PER_BLOCK) {
        uint32_t mx = rmax[0];
#pragma unroll
        for (int it = 1; it < ITERS; it++) mx = umax(mx, rmax[it]);
        mx = umax(mx, dpp<0xB1>(mx));
        mx = umax(mx, dpp<0x4E>(mx));
        mx = umax(mx, (uint32_t)__shfl_xor((int)mx, 32, 64));
        if (lane == 0) wave_max[wave] = mx;
        __syncthreads();
        bscale = scale_of(umax(umax(wave_max[0], wave_max[1]), umax(wave_max[2], wave_max[3])));
        if (tid == 0) p.scale[(size_t)kb * p.nb + m0 / ROWS] = bscale;
    }
    // ---- quantise, transpose 4x4 bytes, stage in LDS ----
    const float bscale_rcp = refine_rcp(bscale);
#pragma unroll
    for (int it = 0; it < ITERS; it++) {
        const int rg = it * 8 + wave * 2 + g;
        uint32_t rw[4];
        // the lane's own row (lane & 3): its scale and reciprocal are worked out once and passed around the quad
        const float own = PER_BLOCK ? bscale : scale_of(rmax[it]);
        const float own_rcp = PER_BLOCK ? bscale_rcp : refine_rcp(own);
        if (!PER_BLOCK && l < 4) row_scale[4 * rg + l] = own;
        const bool special = __builtin_amdgcn_ballot_w64(__builtin_bit_cast(uint32_t, own) >= 0x7F800000u) != 0;
        auto row_of = [&](float x, int r) -> float {
            const uint32_t u = __builtin_bit_cast(uint32_t, x);
            return __builtin_bit_cast(float, PER_BLOCK ? u : r == 0 ? dpp<0x00>(u) : r == 1 ? dpp<0x55>(u) : r == 2 ? dpp<0xAA>(u) : dpp<0xFF>(u));
        };
        if (__builtin_expect(special, 0)) {
            // an inf or NaN in some row: the plain division has the IEEE special cases
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float s = row_of(own, r);
                v4f qf;
#pragma unroll
                for (int j = 0; j < 4; j++) qf[j] = clamp448(v[it][r][j] / s);
                rw[r] = cvt4_e4m3fn(qf);
            }
        } else {
            // no clamp: |x| <= max |x| <= 448 s (1 + 2^-24), and the quotient one step above 448 that this allows rounds to 448
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float s = row_of(own, r), y = row_of(own_rcp, r);
                v4f qf;
#pragma unroll
                for (int j = 0; j < 4; j++) qf[j] = div_by<sizeof(T) == 2 ? 1 : 2>(v[it][r][j], s, y);
                rw[r] = cvt4_e4m3fn(qf);
            }
        }
        // rw[r] = bytes (k0..k3) of row r  ->  c[j] = bytes (row0..row3) of k j
        const uint32_t lo01 = __builtin_amdgcn_perm(rw[1], rw[0], 0x05010400u), hi01 = __builtin_amdgcn_perm(rw[1], rw[0], 0x07030602u);
        const uint32_t lo23 = __builtin_amdgcn_perm(rw[3], rw[2], 0x05010400u), hi23 = __builtin_amdgcn_perm(rw[3], rw[2], 0x07030602u);
        const uint32_t c0 = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u), c1 = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
        const uint32_t c2 = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u), c3 = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
        unsigned char* t = tile + (4 * l) * LD + 4 * rg;
        *(uint32_t*)(t) = c0;
        *(uint32_t*)(t + LD) = c1;
        *(uint32_t*)(t + 2 * LD) = c2;
        *(uint32_t*)(t + 3 * LD) = c3;
    }
    __syncthreads();
    // ---- scales of the rows, contiguous ----
    if (!PER_BLOCK && tid < ROWS && m0 + tid < p.rows) p.scale[(size_t)kb * p.rows + m0 + tid] = row_scale[tid];
    // ---- store: chunks of 16 rows x 1 k; ROWS/16 consecutive lanes write one k row ----
    // k rows start on any byte where rows is not a multiple of 16: 16-byte stores take that, and the chunk that holds
    // the last rows leaves in pieces of 8, 4, 2 and 1 bytes (4095 x 7168 bf16: 21.5 us, byte by byte 63.9; 4096 rows 19.9).
    constexpr int CHUNKS = ROWS / 16;
#pragma unroll
    for (int i = 0; i < TK * CHUNKS / 256; i++) {
        const int id = i * 256 + tid;
        const int krow = id / CHUNKS, c = id % CHUNKS;
        const unsigned char* s = tile + krow * LD + 16 * c;
        const int row = m0 + 16 * c;
        if (row >= p.rows) continue;
        uint8_t* dst = p.q + ((size_t)kb * TK + krow) * (size_t)p.rows + row;
        const uint32_t w[4] = {*(const uint32_t*)s, *(const uint32_t*)(s + 4), *(const uint32_t*)(s + 8), *(const uint32_t*)(s + 12)};
        const int left = p.rows - row;
        if (left >= 16) {
            *(v4i_any*)dst = (v4i){(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
        } else {
            if (left & 8) *(v2i_any*)dst = (v2i){(int)w[0], (int)w[1]};
            const uint32_t w4 = (left & 8) ? w[2] : w[0], w2 = (left & 4) ? ((left & 8) ? w[3] : w[1]) : w4;
            if (left & 4) *(u32_any*)(dst + (left & 8)) = w4;
            if (left & 2) *(u16_any*)(dst + (left & 12)) = (uint16_t)w2;
            if (left & 1) dst[left & 14] = (uint8_t)((left & 2) ? w2 >> 16 : w2);
        }
    }
}

template <typename T, bool PER_BLOCK, int ROWS>
static hipError_t launch_quant_rows(QuantArgs a, hipStream_t stream) {
    // a grid has 65535 places in y: one launch per that many workgroups of rows (rows * k < 2^32 keeps rows below 2^25)
    constexpr int MAX_Y = 65535;
    for (a.row0 = 0; a.row0 < a.rows; a.row0 += MAX_Y * ROWS) {
        const int groups = (a.rows - a.row0 + ROWS - 1) / ROWS;
        dim3 grid((unsigned)(a.k / TK), (unsigned)(groups < MAX_Y ? groups : MAX_Y));
        if (a.row_map) hipLaunchKernelGGL((quantize_kernel<T, PER_BLOCK, true, ROWS>), grid, dim3(256), 0, stream, a);
        else hipLaunchKernelGGL((quantize_kernel<T, PER_BLOCK, false, ROWS>), grid, dim3(256), 0, stream, a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// Rows of a workgroup, us measured with 128 / 64 / 32 of them (bf16, inputs from HBM): few values finish soonest in small
// workgroups, many of them short chains (64 x 7168 5.2 / 2.8 / 2.4, 4004 x 1024 5.2 / 5.0 / 4.5, 16384 x 512 7.3 / 6.7 / 8.1);
// large matrices want 128 bytes per k row in one store (4096 x 7168 19.9 / 20.6 / 22.5, 32768 x 2048 41.9 / 43.5 / 44.3; fp32,
// whose loads weigh more, 32.5 / 32.0 / 33.4 and 66.0 / 64.0 / 61.4).  Gathered rows come from the caches and are bound by the
// vector ALU: 2000 -> 4000 x 7168 14.0 / 13.5 / 13.2, 4096 -> 32768 x 7168 88 / 99 / 132, and with rows of the output that do not
// start on 16 bytes, 4095 -> 32760, 116 / 115 / 100.
template <typename T, bool PER_BLOCK>
static hipError_t launch_quant(const QuantArgs& a, hipStream_t stream) {
    if constexpr (PER_BLOCK) {
        return launch_quant_rows<T, true, 128>(a, stream);
    } else {
        const size_t values = (size_t)a.rows * (size_t)a.k;
        const bool large = values >= (24u << 20);
        if (a.row_map) return large && (a.rows & 15) == 0 ? launch_quant_rows<T, false, 128>(a, stream) : launch_quant_rows<T, false, 32>(a, stream);
        if (large && sizeof(T) == 2) return launch_quant_rows<T, false, 128>(a, stream);
        return values >= (6u << 20) ? launch_quant_rows<T, false, 64>(a, stream) : launch_quant_rows<T, false, 32>(a, stream);
    }
}

// e4m3fnuz (gfx942: bias 8, max 240, NaN = 0x80, no -0) -> e4m3fn (bias 7) with the same value.
// Normal fnuz codes with exponent field >= 2 are the fn code with the exponent field one lower, exactly.
// The 16 smallest magnitudes (fnuz subnormals and exponent field 1, steps of 2^-10) fall on fn's
// subnormal grid of 2^-9: magnitude code x becomes x/2 rounded to nearest even.  16 bytes per thread.
__device__ __forceinline__ uint32_t fnuz_to_fn_byte(uint32_t b) {
    const uint32_t mag = b & 0x7Fu;
    const uint32_t out = mag >= 16u ? mag - 8u : (mag + ((mag >> 1) & 1u)) >> 1;
    return b == 0x80u ? 0x7Fu : ((b & 0x80u) | out);
}
__global__ __launch_bounds__(256)
void fnuz_to_fn_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, size_t n) {
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 16;
    if (i + 16 <= n) {
        const v4i v = *(const v4i*)(src + i);
        v4i o;
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const uint32_t x = (uint32_t)v[w];
            o[w] = (int)(fnuz_to_fn_byte(x & 0xFFu) | (fnuz_to_fn_byte((x >> 8) & 0xFFu) << 8) |
                         (fnuz_to_fn_byte((x >> 16) & 0xFFu) << 16) | (fnuz_to_fn_byte(x >> 24) << 24));
        }
        *(v4i*)(dst + i) = o;
    } else {
        for (size_t j = i; j < n; j++) dst[j] = (uint8_t)fnuz_to_fn_byte(src[j]);
    }
}


// ---------------------------------------------------------------------------------------------------
// Row gather of an already quantised activation matrix: out row i = source row row_map[i], bytes and
// scales, in the K-major storage layout (a[kk * rows + i]).  With top-k routing every token appears
// top-k times in the expert-contiguous order (2-amd-moe/3-amd-fp8-moe-hip-myhgemm.py:174-191 copies
// rows the same way); quantising the tokens once and gathering bytes costs an eighth of the arithmetic
// of quantising every copy.
//
// In this layout the gather runs along the contiguous dimension (one byte per row), so it goes through
// LDS: a workgroup takes KC consecutive k rows of the source (KC * src_rows bytes), transposes them in
// registers (v_perm_b32, 4x4 bytes) to token-major order - LDS slot of token t holds its KC bytes - and
// then every lane produces four consecutive output rows: one LDS read of KC bytes per row, the
// transpose back, and KC dword stores (a wave writes 256 contiguous bytes of one k row per store).
// Slot of token t is (t % 4) * ceil(src_rows / 4) + t / 4, which makes the LDS writes of phase 1
// contiguous across lanes.
// ---------------------------------------------------------------------------------------------------
struct GatherArgs {
    const uint8_t* src;       // [k][src_rows]
    const float* src_scale;   // [k/128][src_rows]
    const int32_t* row_map;   // [rows]
    uint8_t* dst;             // [k][rows]
    float* dst_scale;         // [k/128][rows]
    int rows, k, src_rows;
    int rows_per_wg;          // multiple of 4
};

// rw[r] = bytes (c0..c3) of line r  ->  out[j] = bytes (line0..line3) of column j
__device__ __forceinline__ void transpose4x4(const uint32_t rw[4], uint32_t out[4]) {
    const uint32_t lo01 = __builtin_amdgcn_perm(rw[1], rw[0], 0x05010400u), hi01 = __builtin_amdgcn_perm(rw[1], rw[0], 0x07030602u);
    const uint32_t lo23 = __builtin_amdgcn_perm(rw[3], rw[2], 0x05010400u), hi23 = __builtin_amdgcn_perm(rw[3], rw[2], 0x07030602u);
    out[0] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u); out[1] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
    out[2] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u); out[3] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
}

template <int KC>
__global__ __launch_bounds__(256)
void gather_a_kernel(const GatherArgs p) {
    extern __shared__ __attribute__((aligned(16))) unsigned char slots[];     // [4 * quarter][KC]
    constexpr int KG = KC / 4;
    const int tid = threadIdx.x;
    const int k0 = blockIdx.x * KC;
    const int quarter = (p.src_rows + 3) / 4;
    // ---- phase 1: KC source rows -> token-major slots ----
    __amdgpu_buffer_rsrc_t src_rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)p.src, 0, (uint32_t)p.k * (uint32_t)p.src_rows, 0x00020000);
    for (int task = tid; task < quarter; task += 256) {
        uint32_t tok[4][KG];                       // tok[j][kg]: bytes (k rows 4kg..4kg+3) of token 4*task + j
#pragma unroll
        for (int kg = 0; kg < KG; kg++) {
            uint32_t rw[4], c[4];
#pragma unroll
            for (int r = 0; r < 4; r++)
                rw[r] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(src_rsrc, (uint32_t)(k0 + 4 * kg + r) * (uint32_t)p.src_rows + 4u * (uint32_t)task, 0, 0);
            transpose4x4(rw, c);
#pragma unroll
            for (int j = 0; j < 4; j++) tok[j][kg] = c[j];
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            unsigned char* d = slots + (size_t)(j * quarter + task) * KC;
#pragma unroll
            for (int kg = 0; kg < KG; kg++) *(uint32_t*)(d + 4 * kg) = tok[j][kg];
        }
    }
    __syncthreads();
    // ---- phase 2: four consecutive output rows per lane ----
    const int row_begin = blockIdx.y * p.rows_per_wg;
    int row_end = row_begin + p.rows_per_wg;
    row_end = row_end < p.rows ? row_end : p.rows;
    for (int i0 = row_begin + 4 * tid; i0 < row_end; i0 += 1024) {
        const v4i map = *(const v4i*)(p.row_map + i0);
        uint32_t tok[4][KG];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint32_t t = (uint32_t)map[j];
            const bool ok = t < (uint32_t)p.src_rows;
            const unsigned char* sp = slots + (size_t)((t & 3u) * (uint32_t)quarter + (t >> 2)) * KC;
#pragma unroll
            for (int kg = 0; kg < KG; kg++) tok[j][kg] = ok ? *(const uint32_t*)(sp + 4 * kg) : 0u;
        }
#pragma unroll
        for (int kg = 0; kg < KG; kg++) {
            uint32_t rw[4], c[4];
#pragma unroll
            for (int j = 0; j < 4; j++) rw[j] = tok[j][kg];
            transpose4x4(rw, c);                   // c[r] = bytes (rows i0..i0+3) of k row 4kg + r
#pragma unroll
            for (int r = 0; r < 4; r++)
                __builtin_nontemporal_store(c[r], (uint32_t*)(p.dst + (size_t)(k0 + 4 * kg + r) * (size_t)p.rows + i0));
        }
        // the scales of a K block travel with its first k rows
        if ((k0 & 127) == 0) {
            v4f sc;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t t = (uint32_t)map[j];
                sc[j] = t < (uint32_t)p.src_rows ? p.src_scale[(size_t)(k0 >> 7) * p.src_rows + t] : 1e-12f;
            }
            *(v4f*)(p.dst_scale + (size_t)(k0 >> 7) * p.rows + i0) = sc;
        }
    }
}

// any alignment, any size: one output byte per thread
__global__ __launch_bounds__(256)
void gather_a_bytes_kernel(const GatherArgs p) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= p.rows) return;
    const uint32_t t = (uint32_t)p.row_map[i];
    const bool ok = t < (uint32_t)p.src_rows;
    for (int kk = blockIdx.y; kk < p.k; kk += gridDim.y) {
        p.dst[(size_t)kk * p.rows + i] = ok ? p.src[(size_t)kk * p.src_rows + t] : (uint8_t)0;
        if ((kk & 127) == 0) p.dst_scale[(size_t)(kk >> 7) * p.rows + i] = ok ? p.src_scale[(size_t)(kk >> 7) * p.src_rows + t] : 1e-12f;
    }
}

template <int KC>
static hipError_t launch_gather(const GatherArgs& a, hipStream_t stream) {
    const int quarter = (a.src_rows + 3) / 4;
    const int lds = 4 * quarter * KC;
    auto kern = gather_a_kernel<KC>;
    static int raised[MAX_DEVICES];
    if (lds > 65536) {
        hipError_t e = raise_lds_limit((const void*)kern, lds, raised);
        if (e != hipSuccess) return e;
    }
    dim3 grid((unsigned)(a.k / KC), (unsigned)((a.rows + a.rows_per_wg - 1) / a.rows_per_wg));
    hipLaunchKernelGGL(kern, grid, dim3(256), lds, stream, a);
    return hipGetLastError();
}

}  // namespace fp8bs

extern "C" int fp8bs_convert_fnuz_to_fn(const void* src, void* dst, size_t nbytes, void* stream) {
    if (nbytes == 0) return FP8BS_OK;
    if (!src || !dst) return FP8BS_ERR_NULL_POINTER;
    if ((((uintptr_t)src | (uintptr_t)dst) & 15) != 0) return FP8BS_ERR_BAD_SHAPE;
    const size_t threads = (nbytes + 15) / 16;
    hipLaunchKernelGGL(fp8bs::fnuz_to_fn_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       (const uint8_t*)src, (uint8_t*)dst, nbytes);
    return hipGetLastError() == hipSuccess ? FP8BS_OK : FP8BS_ERR_LAUNCH;
}

namespace {
int quantize_common(const void* x, int dtype, int64_t ldx, const int32_t* row_map, int src_rows, void* q, float* scale,
                    int rows, int k, bool per_block, void* stream) {
    if (rows < 0 || k < 0 || (k % 128) != 0) return FP8BS_ERR_BAD_SHAPE;
    if (dtype != FP8BS_DTYPE_F32 && dtype != FP8BS_DTYPE_BF16) return FP8BS_ERR_BAD_SHAPE;
    if (rows == 0 || k == 0) return FP8BS_OK;
    if (!x || !q || !scale) return FP8BS_ERR_NULL_POINTER;
    if (ldx < k) return FP8BS_ERR_BAD_SHAPE;
    // 16-byte loads along k: rows must start on a 16-byte boundary
    const int64_t esz = dtype == FP8BS_DTYPE_F32 ? 4 : 2;
    if (((uintptr_t)x & 15) != 0 || ((ldx * esz) & (dtype == FP8BS_DTYPE_F32 ? 15 : 7)) != 0) return FP8BS_ERR_BAD_SHAPE;
    if ((size_t)rows * (size_t)k > 0xFFFFFFFFull) return FP8BS_ERR_TOO_LARGE;
    if ((size_t)(row_map ? src_rows : rows) * (size_t)ldx * (size_t)esz > 0xFFFFFFFFull) return FP8BS_ERR_TOO_LARGE;   // buffer addressing
    fp8bs::QuantArgs a{x, row_map, (uint8_t*)q, scale, ldx, rows, k, row_map ? src_rows : rows, (rows + 127) / 128, 0};
    hipStream_t s = (hipStream_t)stream;
    hipError_t e;
    if (dtype == FP8BS_DTYPE_F32) e = per_block ? fp8bs::launch_quant<float, true>(a, s) : fp8bs::launch_quant<float, false>(a, s);
    else e = per_block ? fp8bs::launch_quant<uint16_t, true>(a, s) : fp8bs::launch_quant<uint16_t, false>(a, s);
    return e == hipSuccess ? FP8BS_OK : FP8BS_ERR_LAUNCH;
}
}  // namespace

extern "C" int fp8bs_quantize_a(const void* x, int x_dtype, int64_t ldx, const int32_t* row_map, int src_rows,
                                void* a, float* a_scale, int m, int k, void* stream) {
    return quantize_common(x, x_dtype, ldx, row_map, src_rows, a, a_scale, m, k, false, stream);
}

extern "C" int fp8bs_quantize_b(const void* w, int w_dtype, int64_t ldw, void* b, float* b_scale, int n, int k, void* stream) {
    return quantize_common(w, w_dtype, ldw, nullptr, 0, b, b_scale, n, k, true, stream);
}

extern "C" int fp8bs_gather_a(const void* a_src, const float* a_scale_src, int src_rows, const int32_t* row_map,
                              void* a, float* a_scale, int m, int k, void* stream) {
    if (m < 0 || k < 0 || src_rows < 0 || (k % 128) != 0) return FP8BS_ERR_BAD_SHAPE;
    if (m == 0 || k == 0) return FP8BS_OK;
    if (!row_map || !a || !a_scale || (src_rows > 0 && (!a_src || !a_scale_src))) return FP8BS_ERR_NULL_POINTER;
    if ((size_t)src_rows * (size_t)k > 0xFFFFFFFFull) return FP8BS_ERR_TOO_LARGE;       // buffer addressing
    fp8bs::GatherArgs g{(const uint8_t*)a_src, a_scale_src, row_map, (uint8_t*)a, a_scale, m, k, src_rows, 8192};
    hipStream_t s = (hipStream_t)stream;
    // dword loads of source rows, dword stores of output rows, 16-byte loads of the map and stores of
    // the scales: everything must sit on those boundaries, and the KC source rows must fit the LDS
    const bool aligned = (src_rows % 4) == 0 && (m % 4) == 0 && src_rows > 0 &&
                         ((((uintptr_t)a_src | (uintptr_t)a) & 3) == 0) && ((((uintptr_t)row_map | (uintptr_t)a_scale) & 15) == 0);
    hipError_t e;
    if (aligned && src_rows <= 4096) e = fp8bs::launch_gather<16>(g, s);
    else if (aligned && src_rows <= 8192) e = fp8bs::launch_gather<8>(g, s);
    else if (aligned && src_rows <= 40960) e = fp8bs::launch_gather<4>(g, s);
    else {
        hipLaunchKernelGGL(fp8bs::gather_a_bytes_kernel, dim3((unsigned)((m + 255) / 256), (unsigned)(k < 4096 ? k : 4096)), dim3(256), 0, s, g);
        e = hipGetLastError();
    }
    return e == hipSuccess ? FP8BS_OK : FP8BS_ERR_LAUNCH;
}
