// What the prefill GEMM kernels share (gemm.hip, gemm_dma.hip): parameters, the
// epilogue, the dequantization of tiled weight words, the K-slice reduction.
#pragma once

#include "qe_common.hpp"

namespace qe {

struct GemmParams {
    const uint32_t* qw[3];
    const uint16_t* sc[3];
    uint16_t* out[3];
    int col_begin[3];  // first virtual column of each matrix (QKV)
    int out_stride[3]; // row stride of each output
    const uint16_t* A;
    const uint16_t* residual;
    const int8_t* A8;         // W4A8 variant: Q8_1 rows of the activation
    const float* A8_scale;
    float* ws;         // split-K partials (slices > 1 only)
    int M, N, K;       // N = virtual columns (SwiGLU: 2*I)
};

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kPlain = 0;
constexpr int kQKV = 1;
constexpr int kSwiglu = 2;
constexpr int BK = 64;

// silu(g) * u = g * u / (1 + e^-g) with the hardware exp2 and reciprocal
// (about 1 ulp each in fp32; the result is rounded to fp16)
__device__ __forceinline__ float silu_mul(float g, float u) {
    return g * u * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.44269504088896341f * g));
}

// Split-K partials: fp32 tiles of the K slices, reduced by a second kernel
// on the same stream (deterministic order, no atomics or fences).  They live
// in a workspace of at most kWsFloats floats that belongs to the launching
// stream (WorkspaceLease), so GEMMs in flight on different streams never share
// partials.
constexpr size_t kWsFloats = size_t(8) << 20;  // 32 MiB

using Workspace = StreamWorkspace;

// One 32x32 accumulator fragment whose rows start at r0 and whose lane
// column is col.  D[i][j] of a 32x32 MFMA tile: j = lane%32,
// i = 8*(v/4) + 4*(lane/32) + v%4
// Value of the neighbouring lane (lane ^ 1), by DPP within the quad.
__device__ __forceinline__ float swap_adjacent(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0xB1, 0xF, 0xF, false));
}

template <int MODE>
__device__ __forceinline__ void epilogue_frag(const GemmParams& p, const f32x16& acc, int r0, int col, int lane) {
    const int fr = lane & 31;
    // rows of element v: r0 + 8 * (v / 4) + 4 * (lane / 32) + v % 4 (static
    // offsets from the lane's first row; every index into acc is static)
    const int lrow = r0 + 4 * (lane >> 5);
    const bool cols_ok = col < p.N;
    const bool rows_ok = r0 + 32 <= p.M;  // the whole fragment: no per-row checks
    if constexpr (MODE == kSwiglu) {
        // lane pair (gate column, up column): the gate lane finishes rows
        // v < 8 and the up lane rows v >= 8 (16 further down), so every lane
        // evaluates 8 silu; the partner's values arrive by DPP swaps
        const bool gate = (fr & 1) == 0;
        const int row0 = lrow + (gate ? 0 : 16);
        const int stride = p.out_stride[0];
        uint16_t* out = p.out[0] + (col >> 1);
#pragma unroll
        for (int v = 0; v < 8; ++v) {
            const float lo = acc[v], hi = acc[v + 8];
            const float lo_x = swap_adjacent(lo), hi_x = swap_adjacent(hi);
            const float g = gate ? lo : hi_x;
            const float u = gate ? lo_x : hi;
            const int row = row0 + 8 * (v >> 2) + (v & 3);
            if (cols_ok && (rows_ok || row < p.M)) out[static_cast<size_t>(row) * stride] = f2h(silu_mul(g, u));
        }
        return;
    }
    int m = 0, local = col;
    if constexpr (MODE == kQKV) {
        m = (col >= p.col_begin[1]) + (col >= p.col_begin[2]);
        local = col - p.col_begin[m];
    }
    const int stride = MODE == kQKV ? (m == 0 ? p.out_stride[0] : m == 1 ? p.out_stride[1] : p.out_stride[2])
                                    : p.out_stride[0];
    uint16_t* out = (MODE == kQKV ? (m == 0 ? p.out[0] : m == 1 ? p.out[1] : p.out[2]) : p.out[0]) + local;
    const uint16_t* res = (MODE == kPlain && p.residual != nullptr) ? p.residual + local : nullptr;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int row = lrow + 8 * (v >> 2) + (v & 3);
        if (cols_ok && (rows_ok || row < p.M)) {
            const size_t off = static_cast<size_t>(row) * stride;
            _Float16 h = static_cast<_Float16>(acc[v]);
            if (MODE == kPlain && res != nullptr) h = h + __builtin_bit_cast(_Float16, res[off]);  // fp16 add, RNE
            out[off] = __builtin_bit_cast(uint16_t, h);
        }
    }
}

template <int BM, int BN, int WGM, int MODE>
__device__ __forceinline__ void epilogue(const GemmParams& p, const f32x16 (&acc)[BM / WGM / 32][BN / (4 / WGM) / 32],
                                         int m0, int n0, int wm, int wn, int lane) {
    constexpr int WM = BM / WGM, WN = BN / (4 / WGM), MI = WM / 32, NI = WN / 32;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
            epilogue_frag<MODE>(p, acc[i][j], m0 + wm * WM + i * 32, n0 + wn * WN + j * 32 + (lane & 31), lane);
}

// Nibble order of a word of the tiled copy: k0 at bits 0-3, k1 at 16-19, k2 at
// 4-7, k3 at 20-23, k4 at 8-11, k5 at 24-27, k6 at 12-15, k7 at 28-31.  A
// nibble in bits 0-3 of a 16-bit half under the exponent of 1024.0 (0x6400)
// reads as 1024 + q; in bits 4-7 under the exponent of 64.0 (0x5400) as
// 64 + q.  So the 8 values in K order cost five bit operations (two masked
// ORs, a shift, two masked ORs), then the exact subtraction of 1032 or 72 and
// the one fp16 RNE multiply by the scale of unpack_w4_to_half8 - the same
// values as unpack_w4_to_half8 on the original word.
// The four masks live in VGPRs (TiledMasks, set up once per kernel): gfx9
// VOP3 instructions take no literal constants, so with literal masks the
// compiler emits separate AND and OR instructions instead of V_AND_OR_B32.
struct TiledMasks {
    uint32_t lo, hi, bias_lo, bias_hi;
};
__device__ __forceinline__ TiledMasks tiled_masks() {
    TiledMasks m{0x000F000Fu, 0x00F000F0u, 0x64006400u, 0x54005400u};
    asm volatile("" : "+v"(m.lo), "+v"(m.hi), "+v"(m.bias_lo), "+v"(m.bias_hi));
    return m;
}
// elements 0..3 of a word (4..7 of it shifted right by 8)
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f16x4 unpack_w4t_to_half4(uint32_t w, _Float16 scale, const TiledMasks& m) {
    const uint32_t u01 = (w & m.lo) | m.bias_lo;
    const uint32_t u23 = (w & m.hi) | m.bias_hi;
    const qwen::qe_half2_t b1 = {(_Float16)1032.0f, (_Float16)1032.0f};
    const qwen::qe_half2_t b2 = {(_Float16)72.0f, (_Float16)72.0f};
    const qwen::qe_half2_t sc = {scale, scale};
    const qwen::qe_half2_t h01 = (__builtin_bit_cast(qwen::qe_half2_t, u01) - b1) * sc;
    const qwen::qe_half2_t h23 = (__builtin_bit_cast(qwen::qe_half2_t, u23) - b2) * sc;
    return f16x4{h01[0], h01[1], h23[0], h23[1]};
}
__device__ __forceinline__ qwen::qe_half8_t unpack_w4t_to_half8(uint32_t w, _Float16 scale, const TiledMasks& m) {
    return __builtin_shufflevector(unpack_w4t_to_half4(w, scale, m), unpack_w4t_to_half4(w >> 8, scale, m), 0, 1, 2, 3, 4,
                                   5, 6, 7);
}

// Four accumulator elements of a fragment: elements 4 part .. 4 part + 3, with
// SwiGLU the two element pairs (2 part + e, 2 part + e + 8) whose gate and up
// values two neighbouring lanes exchange.  Arithmetic of epilogue_frag.
template <int MODE>
__device__ __forceinline__ int part_element(int part, int e) {
    return MODE == kSwiglu ? 2 * part + (e & 1) + 8 * (e >> 1) : 4 * part + e;
}

template <int MODE>
__device__ __forceinline__ void epilogue_part(const GemmParams& p, const float (&x)[4], int part, int r0, int col,
                                              int lane) {
    const int lrow = r0 + 4 * (lane >> 5);
    if constexpr (MODE == kSwiglu) {
        const bool gate = (lane & 1) == 0;
        const int row0 = lrow + (gate ? 0 : 16);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float lo = x[e], hi = x[e + 2];
            const float lo_x = swap_adjacent(lo), hi_x = swap_adjacent(hi);
            const int v = 2 * part + e, row = row0 + 8 * (v >> 2) + (v & 3);
            if (col < p.N && row < p.M)
                p.out[0][static_cast<size_t>(row) * p.out_stride[0] + (col >> 1)] =
                    f2h(silu_mul(gate ? lo : hi_x, gate ? lo_x : hi));
        }
        return;
    }
    if (col >= p.N) return;
    int m = 0, local = col;
    if constexpr (MODE == kQKV) {
        m = (col >= p.col_begin[1]) + (col >= p.col_begin[2]);
        local = col - p.col_begin[m];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int row = lrow + 8 * part + e;
        if (row >= p.M) continue;
        const size_t off = static_cast<size_t>(row) * p.out_stride[m] + local;
        _Float16 h = static_cast<_Float16>(x[e]);
        if (MODE == kPlain && p.residual != nullptr) h = h + __builtin_bit_cast(_Float16, p.residual[off]);
        p.out[m][off] = __builtin_bit_cast(uint16_t, h);
    }
}

// Sums the K-slice partials in slice order and applies the epilogue.  grid
// (N tiles, M tiles, 4 * fragments): block z takes a quarter of the elements of
// the 32x32 fragment z / 4 of its tile, 256 threads in the MFMA lane layout of
// the 4 waves.  Bound by what a CU takes from L2, so the blocks are small: with
// whole fragments the down projection at M = 128 (6 slices, 4.7 MB) had 48 of
// them and took 7.5 us, now 3.1.  S slices are requested before the first add (one
// memory latency, not S); S = 0: any number, eight at a time.
template <int BM, int BN, int WGM, int MODE, int S>
__global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(GemmParams p, int slices) {
    constexpr int WGN = 4 / WGM;
    constexpr int WM = BM / WGM, WN = BN / WGN, NI = WN / 32;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int tile = blockIdx.y * gridDim.x + blockIdx.x;
    const int n_tiles = gridDim.x * gridDim.y;
    const int f = blockIdx.z >> 2, part = blockIdx.z & 3, i = f / NI, j = f % NI;
    const size_t slice_stride = static_cast<size_t>(n_tiles) * (BM * BN);
    const float* src = p.ws + static_cast<size_t>(tile) * (BM * BN) + f * 16 * 256 + tid;
    constexpr int B = S > 0 ? S : 8;
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int z0 = 0; z0 < (S > 0 ? 1 : slices); z0 += B) {
        float x[B][4];
#pragma unroll
        for (int z = 0; z < B; ++z)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                x[z][e] = src[(S > 0 ? z : min(z0 + z, slices - 1)) * slice_stride + part_element<MODE>(part, e) * 256];
#pragma unroll
        for (int z = 0; z < B; ++z)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (S > 0 || z0 + z < slices) acc[e] += x[z][e];
    }
    const int wm = wave / WGN, wn = wave % WGN;
    epilogue_part<MODE>(p, acc, part, blockIdx.y * BM + wm * WM + i * 32,
                        blockIdx.x * BN + wn * WN + j * 32 + (lane & 31), lane);
}

template <int BM, int BN, int WGM, int MODE>
void launch_reduce(const GemmParams& p, dim3 tiles, int slices, hipStream_t s) {
    constexpr int FR = (BM / WGM / 32) * (BN / (4 / WGM) / 32);  // fragments per wave
    const dim3 grid(tiles.x, tiles.y, 4 * FR);
    switch (slices) {
        case 2: gemm_splitk_reduce_kernel<BM, BN, WGM, MODE, 2><<<grid, 256, 0, s>>>(p, slices); break;
        case 3: gemm_splitk_reduce_kernel<BM, BN, WGM, MODE, 3><<<grid, 256, 0, s>>>(p, slices); break;
        case 4: gemm_splitk_reduce_kernel<BM, BN, WGM, MODE, 4><<<grid, 256, 0, s>>>(p, slices); break;
        case 6: gemm_splitk_reduce_kernel<BM, BN, WGM, MODE, 6><<<grid, 256, 0, s>>>(p, slices); break;
        case 8: gemm_splitk_reduce_kernel<BM, BN, WGM, MODE, 8><<<grid, 256, 0, s>>>(p, slices); break;
        default: gemm_splitk_reduce_kernel<BM, BN, WGM, MODE, 0><<<grid, 256, 0, s>>>(p, slices); break;
    }
}

}  // namespace

// The tiled-weight kernels with both operands through LDS (gemm_dma.hip).
// mode: kPlain, kQKV, kSwiglu; tile: 0 128x256, 1 128x256 and 2 128x128 with two
// k groups a block; p.ws holds the partials when slices > 1.
void launch_gemm_dma(int mode, int tile, const GemmParams& p, int slices, hipStream_t stream);

// W4A8 (gemm_w4a8.hip): bm 64 or 128 rows a block; p.ws holds the partials when slices > 1.
void launch_gemm_w4a8(int mode, int bm, const GemmParams& p, int slices, hipStream_t stream);

// The kernel for up to kSkinnyRows rows (gemm_skinny.hip).
constexpr int kSkinnyRows = 32;
inline int skinny_columns(int M, int N) { return M <= 16 && N >= 16 * 512 ? 32 : 16; }  // of a block
void launch_gemm_skinny(int mode, const GemmParams& p, bool tiled, hipStream_t stream);

}  // namespace qe
