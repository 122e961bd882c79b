// Prefill W4A16 dequant-GEMM for a few rows (gfx950): short prompts, where the
// weights are read for a handful of rows.  Math and epilogues as in gemm.hip.
//
// A block owns 16 CT columns and all of K: its waves take contiguous runs of
// 128-k groups, each reading packed words and activations straight into the
// operands of v_mfma_f32_16x16x32_f16 (one word is the 8 k of one lane: lane l
// holds column or row l % 16, k 32 (l / 16) + 8 s of the group in MFMA s), and the
// partial tiles meet in LDS, summed in wave order.  No staging and no barrier
// before that, and every load of a wave's GM groups is requested before the
// first is used: what bounds these launches is the latency of that one round
// of loads and the bytes a CU takes from L2 (45 GB/s of weights and activations
// measured).  Tiled weights, 9 rows, against the 64-row tiles: QKV 7.0 -> 4.1
// us, O 6.8 -> 4.1, gate/up 9.8 -> 8.3, down 11.8 -> 9.2; .qwenbin layout 7.4 ->
// 4.5, 7.0 -> 4.4, 11.4 -> 10.6, 14.0 -> 12.1.
#include <algorithm>

#include "gemm_common.hpp"

namespace qe {
namespace {

// GM: groups requested together; LB: most threads of a block
template <int MT, int CT, int GM, int LB, int MODE, bool TILED>
__global__ __launch_bounds__(LB) void gemm_w4a16_skinny_kernel(GemmParams p) {
    extern __shared__ __align__(16) float s_part[];    // [wave][ct][mt][v][lane]
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int waves = blockDim.x >> 6;
    const int c16 = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * 16 * CT;
    const int K = p.K, G = K >> 7;
    // runs of whole 128-byte weight lines (two groups) where K has them
    const int unit = 2 - (G & 1), units = G / unit;
    const int gr0 = unit * (wave * units / waves), gr1 = unit * ((wave + 1) * units / waves);
    const TiledMasks tmask = tiled_masks();

    // columns past N read column N - 1, rows past M row M - 1; neither is stored
    const u32x4* wp[CT];
    const uint16_t* sp[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const int col = min(n0 + 16 * ct + c16, p.N - 1);
        int m = 0, local = col;
        if constexpr (MODE == kQKV) {
            m = (col >= p.col_begin[1]) + (col >= p.col_begin[2]);
            local = col - p.col_begin[m];
        }
        if constexpr (TILED) {
            const size_t tq = static_cast<size_t>(local >> 5) * (K >> 8);
            wp[ct] = reinterpret_cast<const u32x4*>(p.qw[m]) + tq * 256 + 64 * g + (local & 31);
            sp[ct] = p.sc[m] + tq * 64 + (local & 31);
        } else {
            wp[ct] = reinterpret_cast<const u32x4*>(p.qw[m]) + static_cast<size_t>(local) * (K >> 5) + g;
            sp[ct] = p.sc[m] + static_cast<size_t>(local) * G;
        }
    }
    const uint16_t* ap[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) ap[mt] = p.A + static_cast<size_t>(min(16 * mt + c16, p.M - 1)) * K + 32 * g;

    f32x4 acc[CT][MT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[ct][mt] = f32x4{};
    for (int gr = gr0; gr < gr1; gr += GM) {
        u32x4 w[GM][CT], a[GM][MT][4];
        uint16_t sc[GM][CT];
#pragma unroll
        for (int i = 0; i < GM; ++i) {
            const int x = gr + i;
            if (i > 0 && x >= gr1) continue;  // wave-uniform
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                w[i][ct] = __builtin_nontemporal_load(wp[ct] + (TILED ? (x >> 1) * 256 + (x & 1) * 32 : 4 * x));
                sc[i][ct] = sp[ct][TILED ? (x >> 1) * 64 + (x & 1) * 32 : x];
            }
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                for (int s = 0; s < 4; ++s) a[i][mt][s] = *reinterpret_cast<const u32x4*>(ap[mt] + 128 * x + 8 * s);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < GM; ++i) {
            if (i > 0 && gr + i >= gr1) continue;  // wave-uniform
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                const _Float16 scale = __builtin_bit_cast(_Float16, sc[i][ct]);
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const uint32_t word = w[i][ct][s];
                    const f16x8 b = __builtin_bit_cast(f16x8, TILED ? unpack_w4t_to_half8(word, scale, tmask)
                                                                    : qwen::unpack_w4_to_half8(word, scale));
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt)
                        acc[ct][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a[i][mt][s]), b,
                                                                             acc[ct][mt], 0, 0, 0);
                }
            }
        }
    }
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int v = 0; v < 4; ++v) s_part[((wave * CT + ct) * MT + mt) * 256 + v * 64 + lane] = acc[ct][mt][v];
    __syncthreads();
    // element e = (ct, mt, v, lane l): column 16 ct + l % 16, row 16 mt + 4 (l / 16) + v
    constexpr int E = CT * MT * 256;
    auto total = [&](int e) __attribute__((always_inline)) {
        float x = s_part[e];
        for (int z = 1; z < waves; ++z) x += s_part[z * E + e];
        return x;
    };
    for (int e0 = threadIdx.x; e0 < (MODE == kSwiglu ? E / 2 : E); e0 += blockDim.x) {
        const int e = MODE == kSwiglu ? 2 * e0 : e0;  // gate columns are even, up columns one past
        const int l = e & 63, v = (e >> 6) & 3, mt = (e >> 8) % MT, ct = (e >> 8) / MT;
        const int row = 16 * mt + 4 * (l >> 4) + v, col = n0 + 16 * ct + (l & 15);
        if (row >= p.M || col >= p.N) continue;
        if constexpr (MODE == kSwiglu) {
            p.out[0][static_cast<size_t>(row) * p.out_stride[0] + (col >> 1)] = f2h(silu_mul(total(e), total(e + 1)));
        } else {
            int m = 0, local = col;
            if constexpr (MODE == kQKV) {
                m = (col >= p.col_begin[1]) + (col >= p.col_begin[2]);
                local = col - p.col_begin[m];
            }
            const size_t off = static_cast<size_t>(row) * p.out_stride[m] + local;
            _Float16 h = static_cast<_Float16>(total(e));
            if (MODE == kPlain && p.residual != nullptr) h = h + __builtin_bit_cast(_Float16, p.residual[off]);
            p.out[m][off] = __builtin_bit_cast(uint16_t, h);
        }
    }
}

template <int MT, int CT, int GM, int MAXW, int MODE, bool TILED>
void launch(const GemmParams& p, int max_waves, hipStream_t s) {
    const int G = p.K >> 7, units = G / (2 - (G & 1));
    max_waves = std::max(1, std::min(max_waves, MAXW));
    const int per = (units + max_waves - 1) / max_waves;  // units of the busiest wave ...
    const int waves = (units + per - 1) / per;            // ... and the fewest waves that keep it so
    gemm_w4a16_skinny_kernel<MT, CT, GM, 64 * MAXW, MODE, TILED>
        <<<(p.N + 16 * CT - 1) / (16 * CT), 64 * waves, static_cast<size_t>(waves) * CT * MT * 1024, s>>>(p);
}

// 32 columns a block where that leaves two blocks per CU (half the activation
// reads; at least two units a wave: gate/up on 9 rows 8.3 us, with one 10.2), else
// 16 columns and up to 12 waves.
template <int MODE, bool TILED>
void launch_rows(const GemmParams& p, hipStream_t s) {
    const int units = (p.K >> 7) / (2 - ((p.K >> 7) & 1));
    if (p.M > 16) launch<2, 1, 4, 8, MODE, TILED>(p, 8, s);
    else if (skinny_columns(p.M, p.N) == 32) launch<1, 2, 4, 8, MODE, TILED>(p, (units + 1) / 2, s);
    else launch<1, 1, 6, 12, MODE, TILED>(p, 12, s);
}

template <int MODE>
void launch_layout(const GemmParams& p, bool tiled, hipStream_t s) {
    tiled ? launch_rows<MODE, true>(p, s) : launch_rows<MODE, false>(p, s);
}

}  // namespace

void launch_gemm_skinny(int mode, const GemmParams& p, bool tiled, hipStream_t s) {
    switch (mode) {
        case kPlain: launch_layout<kPlain>(p, tiled, s); break;
        case kQKV: launch_layout<kQKV>(p, tiled, s); break;
        default: launch_layout<kSwiglu>(p, tiled, s); break;
    }
}

}  // namespace qe
