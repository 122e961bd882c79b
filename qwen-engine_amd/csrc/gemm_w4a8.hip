// Prefill W4A8 GEMM: Q8_1 activation rows times packed int4 weights on the int8
// matrix cores (gfx950).
//
// Arithmetic: per 128-group an exact int32 dot, then fp32
// f += float(dot) * (w_scale * x_scale), the GEMV's per-chunk step with the four
// chunk dots summed first (integer addition).  A weight enters as the signed
// byte 16 (q - 8): the nibble with its top bit flipped, in the high half of a
// byte (one xor per word, an and, a shift and an and), so the zero point needs
// no correction term; the factor 16 comes off the scale (a power of two, exact;
// |16 dot| <= 2^21 is exact in fp32).
//
// Layout.  v_mfma_i32_32x32x32_i8 with the weights as the rows and the activation
// rows as the columns: lane (h, r) of a result holds activation row r and the
// weight columns 8 (v / 4) + 4 h + v % 4, so an x_scale is one value per lane, the
// w_scales of a wave's 32 columns serve all its row fragments, SwiGLU pairs sit
// in one lane and four outputs are stored together.  A lane half takes k in
// [64 h, 64 h + 64) of the group, 16 per MFMA.
// A block covers BM rows and 128 columns, a wave all the rows and 32 columns.  One
// 128-group is one stage of a ring of D in LDS, filled by DMA (global_load_lds):
// A rows of 128 bytes, 16-byte chunk ch stored at ch ^ (row / 2 % 8); weight
// columns of 64 bytes, chunk c stored at c ^ (column / 4 % 4); the scales, a dword
// a lane.  The operand reads then touch every bank once; at 64 rows the x_scales of
// rows 16 apart lie 256 bytes apart, in one bank, and a fragment's read of them takes
// twice (0.5 conflict cycles an MFMA counted in all).
//
// What bounds it: the scaling, three vector instructions per result and group
// against a quarter of an MFMA; and latency where a launch has few steps.  The
// kernel before it staged A through registers two steps ahead and kept the zero
// point as a correction per row and group: gate/up (1536 -> 17920) at 8 / 300 / 1024
// rows 14.8 / 34.2 / 80.1 -> 11.1 / 28.9 / 71.2 us; down (8960 -> 1536) with its
// slice sum 15.8 / 35.6 / 81.3 -> 11.6 / 20.6 / 37.5.  Two k groups in a block of eight
// waves were within 5 % either way on small grids and up to 40 % slower on full ones.
#include <algorithm>

#include "gemm_common.hpp"
#include "lds_dma.hpp"

namespace qe {
namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));

constexpr int BN = 128;

// Four results of activation row `row`: weight columns col .. col + 3 (col % 4 == 0).
template <int MODE>
__device__ __forceinline__ void store4(const GemmParams& p, const float (&x)[4], int row, int col) {
    if (row >= p.M || col >= p.N) return;
    if constexpr (MODE == kSwiglu) {  // N is even: columns come as gate, up pairs
        uint16_t* o = p.out[0] + static_cast<size_t>(row) * p.out_stride[0] + (col >> 1);
        o[0] = f2h(silu_mul(x[0], x[1]));
        if (col + 2 < p.N) o[1] = f2h(silu_mul(x[2], x[3]));
        return;
    }
    const bool whole = col + 4 <= p.N;
    if constexpr (MODE == kPlain) {
        const size_t off = static_cast<size_t>(row) * p.out_stride[0] + col;
        if (whole && p.out_stride[0] % 4 == 0 && (reinterpret_cast<uintptr_t>(p.out[0]) & 7) == 0 &&
            (reinterpret_cast<uintptr_t>(p.residual) & 7) == 0) {
            f16x4 v = {static_cast<_Float16>(x[0]), static_cast<_Float16>(x[1]), static_cast<_Float16>(x[2]),
                       static_cast<_Float16>(x[3])};
            if (p.residual != nullptr) v = v + *reinterpret_cast<const f16x4*>(p.residual + off);  // fp16 add, RNE
            *reinterpret_cast<f16x4*>(p.out[0] + off) = v;
            return;
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int c = col + q;
        if (c >= p.N) return;
        int m = 0, local = c;
        if constexpr (MODE == kQKV) {
            m = (c >= p.col_begin[1]) + (c >= p.col_begin[2]);
            local = c - p.col_begin[m];
        }
        const size_t off = static_cast<size_t>(row) * p.out_stride[m] + local;
        _Float16 v = static_cast<_Float16>(x[q]);
        if (MODE == kPlain && p.residual != nullptr) v = v + __builtin_bit_cast(_Float16, p.residual[off]);
        p.out[m][off] = __builtin_bit_cast(uint16_t, v);
    }
}

template <int BM, int MODE>
__global__ __launch_bounds__(256, 2) void gemm_w4a8_kernel(GemmParams p) {
    constexpr int MI = BM / 32;
    constexpr int A_BYTES = BM * 128, B_BYTES = BN * 64, S_BYTES = 4 * 256;  // scales: 64 dwords a wave
    constexpr int STAGE = A_BYTES + B_BYTES + 2 * S_BYTES;
    constexpr int D = 78 * 1024 / STAGE;  // two blocks per CU
    static_assert(D >= 3 && D <= 6, "ring");
    constexpr int LA = BM / 32;   // A loads per wave and stage (8 rows each)
    constexpr int L = LA + 4;     // loads per wave and stage: A, two of weights, the scales
    constexpr int XS = BM > 64 ? BM / 4 : 16;  // rows whose x_scale a wave requests (lane % 32 or % 16)
    __shared__ __align__(16) char smem[D * STAGE];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tid = threadIdx.x;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    const int K = p.K, G = K >> 7;
    const int slices = gridDim.z;
    const int g_begin = static_cast<int>((static_cast<long long>(blockIdx.z) * G) / slices);
    const int KT = static_cast<int>((static_cast<long long>(blockIdx.z + 1) * G) / slices) - g_begin;  // >= 1
    const int fr = lane & 31, h = lane >> 5;
    const uint32_t lds0 =
        static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void*)smem));

    // A load i of a wave: rows 8 (4 i + wave) + lane / 8, stored chunk lane % 8;
    // rows past M read row M - 1 and are never stored
    const char* a_src[LA];
#pragma unroll
    for (int i = 0; i < LA; ++i) {
        const int row = 8 * (4 * i + wave) + (lane >> 3);
        const int ch = (lane & 7) ^ ((row >> 1) & 7);
        a_src[i] = reinterpret_cast<const char*>(p.A8) + static_cast<size_t>(min(m0 + row, p.M - 1)) * K +
                   128 * g_begin + 16 * ch;
    }
    // weight load b: columns 16 b + lane / 4 of the wave, stored chunk lane % 4; columns past N read column N - 1
    auto column = [&](int c, int& m, int& local) __attribute__((always_inline)) {
        const int col = min(n0 + 32 * wave + c, p.N - 1);
        m = 0;
        local = col;
        if constexpr (MODE == kQKV) {
            m = (col >= p.col_begin[1]) + (col >= p.col_begin[2]);
            local = col - p.col_begin[m];
        }
    };
    const char* b_src[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const int c = 16 * b + (lane >> 2);
        int m, local;
        column(c, m, local);
        b_src[b] = reinterpret_cast<const char*>(p.qw[m] + static_cast<size_t>(local) * (K >> 3)) + 64 * g_begin +
                   16 * ((lane & 3) ^ ((c >> 2) & 3));
    }
    const char* ws_src;
    {
        int m, local;
        column(fr, m, local);
        ws_src = reinterpret_cast<const char*>(p.sc[m] + static_cast<size_t>(local) * G + g_begin);
    }
    const char* xs_src = reinterpret_cast<const char*>(
        p.A8_scale + static_cast<size_t>(min(m0 + XS * wave + (lane & (XS - 1)), p.M - 1)) * G + g_begin);

    auto load_stage = [&](int kt, int slot) __attribute__((always_inline)) {
        const uint32_t st = lds0 + slot * STAGE;
#pragma unroll
        for (int i = 0; i < LA; ++i)
            lds_load_x4(st + (4 * i + wave) * 1024, a_src[i] + 128 * kt);
#pragma unroll
        for (int b = 0; b < 2; ++b)
            lds_load_x4(st + A_BYTES + wave * 2048 + b * 1024, b_src[b] + 64 * kt);
        lds_load_dword(st + A_BYTES + B_BYTES + wave * 256, xs_src + 4 * kt);
        lds_load_ushort(st + A_BYTES + B_BYTES + S_BYTES + wave * 256, ws_src + 2 * kt);
    };
    typedef const __attribute__((address_space(3))) i32x4* l_i32x4;
    typedef const __attribute__((address_space(3))) u32x4* l_u32x4;
    typedef const __attribute__((address_space(3))) float* l_f32;

    float f[MI][16];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) f[i][v] = 0.0f;

    // operand addresses within a stage: chunk 4 h + j of row fr (+ 32 i); chunks 2 h, 2 h + 1 of column fr
    const uint32_t a_rd = fr * 128 + 16 * ((4 * h) ^ ((fr >> 1) & 7));
    const uint32_t b_rd = A_BYTES + wave * 2048 + fr * 64 + 16 * ((2 * h) ^ ((fr >> 2) & 3));
    const uint32_t ws_rd = A_BYTES + B_BYTES + S_BYTES + wave * 256 + 16 * h;
    const uint32_t xs_rd = A_BYTES + B_BYTES;
#pragma unroll
    for (int d = 0; d < D - 1; ++d) load_stage(min(d, KT - 1), d);
    int slot = 0;
    for (int kt = 0; kt < KT; ++kt) {
        // this stage has arrived for every wave, and every wave has read the one before it
        constexpr int N = (D - 2) * L;
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | ((N >> 4) << 14));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        load_stage(min(kt + D - 1, KT - 1), slot == 0 ? D - 1 : slot - 1);
        const uint32_t st = lds0 + slot * STAGE;
        slot = slot + 1 == D ? 0 : slot + 1;
        i32x4 wop[4];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const u32x4 raw = *reinterpret_cast<l_u32x4>(st + (b_rd ^ (16 * c)));
#pragma unroll
            for (int e = 0; e < 4; ++e) {  // word e: its low nibbles are k 0..3 of 8, its high nibbles k 4..7
                const uint32_t s = raw[e] ^ 0x88888888u;
                wop[2 * c + (e >> 1)][2 * (e & 1)] = static_cast<int>((s << 4) & 0xF0F0F0F0u);
                wop[2 * c + (e >> 1)][2 * (e & 1) + 1] = static_cast<int>(s & 0xF0F0F0F0u);
            }
        }
        float ws[16];
#pragma unroll
        for (int v4 = 0; v4 < 4; ++v4) {
            const u32x4 raw = *reinterpret_cast<l_u32x4>(st + ws_rd + 32 * v4);
#pragma unroll
            for (int q = 0; q < 4; ++q) ws[4 * v4 + q] = h2f(static_cast<uint16_t>(raw[q])) * 0.0625f;
        }
        float xs[MI];
#pragma unroll
        for (int i = 0; i < MI; ++i)
            xs[i] = *reinterpret_cast<l_f32>(st + xs_rd + ((32 * i + fr) / XS) * 256 + ((32 * i + fr) % XS) * 4);
        // fragment i multiplies while fragment i - 1 is scaled
        i32x16 acc[2];
#pragma unroll
        for (int i = 0; i <= MI; ++i) {
            if (i < MI) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const i32x4 aop = *reinterpret_cast<l_i32x4>(st + (a_rd ^ (16 * j)) + i * 32 * 128);
                    acc[i & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wop[j], aop, j == 0 ? i32x16{} : acc[i & 1], 0, 0, 0);
                }
            }
            if (i > 0) {
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    f[i - 1][v] = __builtin_fmaf(static_cast<float>(acc[(i - 1) & 1][v]), ws[v] * xs[i - 1], f[i - 1][v]);
            }
        }
    }
    __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));  // no request into LDS outlives the block

    const int tile = blockIdx.y * gridDim.x + blockIdx.x;
    f32x4* mine = reinterpret_cast<f32x4*>(p.ws) +
                  (static_cast<size_t>(blockIdx.z) * gridDim.x * gridDim.y + tile) * (BM * BN / 4);
#pragma unroll
    for (int i = 0; i < MI; ++i) {
#pragma unroll
        for (int v4 = 0; v4 < 4; ++v4) {
            const float x[4] = {f[i][4 * v4], f[i][4 * v4 + 1], f[i][4 * v4 + 2], f[i][4 * v4 + 3]};
            if (slices == 1) store4<MODE>(p, x, m0 + 32 * i + fr, n0 + 32 * wave + 8 * v4 + 4 * h);
            else mine[(4 * i + v4) * 256 + tid] = f32x4{x[0], x[1], x[2], x[3]};
        }
    }
}

// Sums the K-slice partials in slice order, eight requested at a time.  grid (N
// tiles, M tiles, BM / 8): block z takes four results a lane, quarter z % 4 of
// fragment z / 4.
template <int BM, int MODE>
__global__ __launch_bounds__(256) void gemm_w4a8_reduce_kernel(GemmParams p, int slices) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int tile = blockIdx.y * gridDim.x + blockIdx.x;
    const size_t stride = static_cast<size_t>(gridDim.x) * gridDim.y * (BM * BN / 4);
    const f32x4* src = reinterpret_cast<const f32x4*>(p.ws) + static_cast<size_t>(tile) * (BM * BN / 4) + blockIdx.z * 256 + tid;
    constexpr int B = 8;
    f32x4 acc = f32x4{};
    for (int z0 = 0; z0 < slices; z0 += B) {
        f32x4 x[B];
#pragma unroll
        for (int z = 0; z < B; ++z) x[z] = src[min(z0 + z, slices - 1) * stride];
#pragma unroll
        for (int z = 0; z < B; ++z)
            if (z0 + z < slices) acc += x[z];
    }
    const float x[4] = {acc[0], acc[1], acc[2], acc[3]};
    const int i = blockIdx.z >> 2, v4 = blockIdx.z & 3;
    store4<MODE>(p, x, blockIdx.y * BM + 32 * i + (lane & 31),
                 blockIdx.x * BN + 32 * wave + 8 * v4 + 4 * (lane >> 5));
}

template <int BM, int MODE>
void launch(const GemmParams& p, int slices, hipStream_t s) {
    const dim3 tiles((p.N + BN - 1) / BN, (p.M + BM - 1) / BM);
    gemm_w4a8_kernel<BM, MODE><<<dim3(tiles.x, tiles.y, slices), 256, 0, s>>>(p);
    if (slices > 1) gemm_w4a8_reduce_kernel<BM, MODE><<<dim3(tiles.x, tiles.y, BM / 8), 256, 0, s>>>(p, slices);
}

template <int MODE>
void launch_bm(const GemmParams& p, int bm, int slices, hipStream_t s) {
    bm == 128 ? launch<128, MODE>(p, slices, s) : launch<64, MODE>(p, slices, s);
}

}  // namespace

void launch_gemm_w4a8(int mode, int bm, const GemmParams& p, int slices, hipStream_t s) {
    switch (mode) {
        case kPlain: launch_bm<kPlain>(p, bm, slices, s); break;
        case kQKV: launch_bm<kQKV>(p, bm, slices, s); break;
        default: launch_bm<kSwiglu>(p, bm, slices, s); break;
    }
}

}  // namespace qe
