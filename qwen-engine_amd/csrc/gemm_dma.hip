// Prefill W4A16 dequant-GEMM on tiled weights, both operands through LDS by DMA
// (gfx950).  Math and epilogues as in gemm.hip.
#include "gemm_common.hpp"
#include "lds_dma.hpp"

namespace qe {
namespace {

// Both operands reach LDS by DMA (global_load_lds), nothing is staged in
// registers, and a wave covers 128 rows x 32 or 64 columns.
//
// A 64-k step is one stage of a ring of D in LDS: the A tile (BM rows of 128
// bytes) and the packed words of the block's columns.  A row's 16-byte chunk ch
// is stored at ch ^ (row / 2 % 8), so the 16-byte operand reads of 16 rows touch
// every bank once.  Step t of a 256-k quad takes k 128 h + 32 t + 8 s for lane half
// h in sub-step s (chunk ch = 4 h + s), the order of the register-staged kernels:
// with KG = 1 a slice has the bits of their kernel with one k group.  Words and
// scales of a wave's columns are requested and read by that wave alone (WGM = 1);
// only A is shared.
// KG = 2: two groups of four waves, each with a ring of its own, take half of
// the block's k each and add their accumulators through LDS at the end, which is
// another order of the sum (one block per CU; half the split-K partials for the
// same parallelism).
//
// What bounds it.  The 128 x 32 wave tile of the register-staged kernels reads 1
// KB of A per 32-cycle MFMA and wave, 128 bytes a clock per CU at the full
// matrix rate, which is all LDS delivers; 64 columns a wave halve that, and the
// registers for it are the ones the staging held.  Gate/up (1536 -> 17920) at
// M = 4096 265 -> 215 us (1.05 PFLOP/s): MFMAs busy 61 % of the time on a SIMD of a
// busy CU (staged kernels at M = 1024 44 %), 0.64 LDS instructions an MFMA (1.26), 5.7
// vector ones, no bank conflicts counted.  Dequantization is 3.25 vector
// instructions per MFMA at 128 rows a wave; 256 rows would halve it but leave one
// wave per SIMD.
template <int BM, int BN, int WGM, int MODE, int KG>
__global__ __launch_bounds__(256 * KG, 2) void gemm_w4a16_dma_kernel(GemmParams p) {
    constexpr int WGN = 4 / WGM;
    constexpr int WM = BM / WGM, WN = BN / WGN;
    constexpr int MI = WM / 32, NI = WN / 32;
    static_assert(MI >= 1 && (NI == 1 || NI == 2), "wave tile");
    constexpr int A_BYTES = BM * 128, B_BYTES = BN * 32, STAGE = A_BYTES + B_BYTES;
    constexpr int SC_BYTES = 4 * 4 * 256;  // per wave four quads of scales
    constexpr int D = (78 * 1024 - SC_BYTES) / STAGE > 8 ? 8 : (78 * 1024 - SC_BYTES) / STAGE;
    static_assert(D >= 3, "ring");
    constexpr int LA = BM / 32;    // A loads per wave and stage (8 rows each)
    constexpr int L = LA + NI;     // loads per wave and stage
    constexpr int GROUP = D * STAGE + SC_BYTES;  // LDS of one k group
    __shared__ __align__(16) char smem[KG * GROUP];

    const int lane = threadIdx.x & 63;
    const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wave = wave_all & 3, kg = wave_all >> 2;
    const int tid = threadIdx.x & 255;
    const int wm = wave / WGN, wn = wave % WGN;
    // Block b runs on XCD b % 8 (workgroups are dealt out round robin).  Every
    // XCD takes a contiguous run of the tiles in an order that goes down 8 row
    // tiles before the next column tile, so that its ~64 resident blocks share
    // about 8 row tiles of A and 8 column tiles of weights in its L2.
    const int TN = (p.N + BN - 1) / BN, TM = (p.M + BM - 1) / BM, T = TN * TM;
    int tm, tn;
    {
        const int x = blockIdx.x & 7, per = T >> 3, extra = T & 7;
        const int l = x * per + min(x, extra) + static_cast<int>(blockIdx.x >> 3);
        const int g = l / (8 * TN), rem = l - g * 8 * TN, gm = min(8, TM - 8 * g);
        tn = rem / gm;
        tm = 8 * g + rem - tn * gm;
    }
    const int m0 = tm * BM;
    const int n0 = tn * BN;
    const int K = p.K;
    const int slices = gridDim.y;
    const int Q_all = K >> 8;
    const int q_first = static_cast<int>((static_cast<long long>(blockIdx.y) * Q_all) / slices);
    const int q_last = static_cast<int>((static_cast<long long>(blockIdx.y + 1) * Q_all) / slices);
    // group kg takes the kg-th run of the slice's quads; the groups step together
    // (one barrier), the last one may hold fewer quads and then only waits
    const int q_per = (q_last - q_first + KG - 1) / KG;
    const int q_begin = q_first + kg * q_per;
    const int q_mine = max(0, min(q_per, q_last - q_begin));
    const int KT = 4 * q_per, KT_mine = 4 * q_mine;
    const int q_safe = min(q_begin, q_last - 1);  // quads requested are always inside the slice
    const int kt_safe = max(KT_mine, 4) - 1;
    const int fr = lane & 31;
    const int h = lane >> 5;
    const TiledMasks tmask = tiled_masks();
    const uint32_t lds0 =
        static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void*)smem)) + kg * GROUP;

    // A load i of a wave: rows 8 (4 i + wave) + lane / 8, stored chunk lane % 8;
    // rows past M read row M - 1 (valid) and are never stored
    uint32_t a_off[LA];
#pragma unroll
    for (int i = 0; i < LA; ++i) {
        const int row = 8 * (4 * i + wave) + (lane >> 3);
        const int ch = (lane & 7) ^ ((row >> 1) & 7);
        a_off[i] = static_cast<uint32_t>(min(m0 + row, p.M - 1) - m0) * (2 * K) + 16 * (ch & 3) + 256 * (ch >> 2);
    }
    const char* a_base = reinterpret_cast<const char*>(p.A + static_cast<size_t>(m0) * K + 256 * q_safe);
    // words: 1 KB of a 32-column tile per step; columns past N read the last tile
    const uint32_t b_off = 16 * lane;
    const char* b_base[NI];
    const char* s_ptr = nullptr;  // this lane's 4 bytes of scales: lanes 0..31 tile 0, 32..63 tile 1
#pragma unroll
    for (int j = 0; j < NI; ++j) {
        const int col = min(n0 + wn * WN + j * 32, (p.N - 1) & ~31);
        int m = 0, local = col;
        if constexpr (MODE == kQKV) {
            m = (col >= p.col_begin[1]) + (col >= p.col_begin[2]);
            local = col - p.col_begin[m];
        }
        const size_t tq = static_cast<size_t>(local >> 5) * Q_all + q_safe;
        b_base[j] = reinterpret_cast<const char*>(p.qw[m]) + tq * 4096;
        const char* sj = reinterpret_cast<const char*>(p.sc[m]) + tq * 128 + 4 * fr;
        if (j == 0 || h == 1) s_ptr = sj;
    }
    const uint32_t sc_lds = lds0 + D * STAGE + wave * 1024;

    auto load_stage = [&](int kt, int slot) __attribute__((always_inline)) {
        const uint32_t st = lds0 + slot * STAGE;
        const char* ab = a_base + static_cast<size_t>(kt >> 2) * 512 + 64 * (kt & 3);
#pragma unroll
        for (int i = 0; i < LA; ++i)
            lds_load_x4(st + (4 * i + wave) * 1024, ab, a_off[i]);
        const size_t bk = static_cast<size_t>(kt >> 2) * 4096 + 1024 * (kt & 3);
#pragma unroll
        for (int j = 0; j < NI; ++j)
            lds_load_x4(st + A_BYTES + (wn * NI + j) * 1024, b_base[j] + bk, b_off);
    };
    auto load_scales = [&](int q) __attribute__((always_inline)) {
        lds_load_dword(sc_lds + (q & 3) * 256, s_ptr + static_cast<size_t>(q) * 128);
    };
    typedef const __attribute__((address_space(3))) f16x8* l_f16x8;
    typedef const __attribute__((address_space(3))) u32x4* l_u32x4;
    typedef const __attribute__((address_space(3))) uint16_t* l_u16;
    // operand addresses within a stage: A chunk 4 h + s of row fr (+ 32 i rows)
    const uint32_t a_rd = (wm * WM + fr) * 128 + 16 * ((4 * h) ^ ((fr >> 1) & 7));

    f32x16 acc[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = f32x16{};

    // A step: sub-step s multiplies while the operands of sub-step s + 1 are
    // read and dequantized beside it.  Before the last sub-step every wave has
    // read all of the stage and has waited for the next one, so the last
    // sub-step already prepares the next step's operands and requests the
    // stage D ahead into the buffer just read: no wave starts a step by waiting.
    u32x4 w[NI];
    _Float16 sc[NI];
    f16x8 af[2][MI], bf[2][NI];
    auto read_words = [&](int kt, uint32_t st) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            w[j] = *reinterpret_cast<l_u32x4>(st + A_BYTES + (wn * NI + j) * 1024 + 16 * lane);
            sc[j] = __builtin_bit_cast(_Float16, *reinterpret_cast<l_u16>(sc_lds + ((kt >> 2) & 3) * 256 + j * 128 +
                                                                         64 * h + 2 * fr));
        }
    };
    auto read_a = [&](uint32_t st, int s, int i) __attribute__((always_inline)) {
        af[s & 1][i] = *reinterpret_cast<l_f16x8>(st + (a_rd ^ (16 * s)) + i * 32 * 128);
    };
    auto dequant = [&](int s, int t) __attribute__((always_inline)) {  // half t % 2 of column fragment t / 2
        const int j = t >> 1;
        const f16x4 v = unpack_w4t_to_half4(t & 1 ? w[j][s] >> 8 : w[j][s], sc[j], tmask);
#pragma unroll
        for (int e = 0; e < 4; ++e) bf[s & 1][j][4 * (t & 1) + e] = v[e];
    };
    constexpr int NM = MI * NI, NH = 2 * NI;  // MFMAs and dequantization halves of a sub-step
    // MFMAs of sub-step s; beside them the operands of sub-step nx of the stage at st
    auto substep = [&](int s, uint32_t st, int nx) __attribute__((always_inline)) {
#pragma unroll
        for (int x = 0; x < NM; ++x) {
            const int i = x / NI, j = x % NI;
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[s & 1][i], bf[s & 1][j], acc[i][j], 0, 0, 0);
            if (x % NI == 0) read_a(st, nx, i);
#pragma unroll
            for (int t = 0; t < NH; ++t)
                if (x == (NM >= NH ? NM - NH + t : t * NM / NH)) dequant(nx, t);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto wait_stage = [&]() __attribute__((always_inline)) {
        constexpr int N = (D - 2) * L;  // the stages after the next one stay in flight
        __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | ((N >> 4) << 14));  // and every read of this stage is done
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    load_scales(0);
    load_scales(min(1, kt_safe >> 2));
#pragma unroll
    for (int d = 0; d < D - 1; ++d) load_stage(min(d, kt_safe), d);
    wait_stage();
    load_stage(min(D - 1, kt_safe), D - 1);
    read_words(0, lds0);
#pragma unroll
    for (int i = 0; i < MI; ++i) read_a(lds0, 0, i);
#pragma unroll
    for (int t = 0; t < NH; ++t) dequant(0, t);
    int slot = 0;
    for (int kt = 0; kt < KT; ++kt) {
        const uint32_t st = lds0 + slot * STAGE;
        const int done = slot;
        slot = slot + 1 == D ? 0 : slot + 1;
        const uint32_t st_next = lds0 + slot * STAGE;
        const bool live = KG == 1 || kt < KT_mine;  // wave-uniform
        if (live) {
            substep(0, st, 1);
            substep(1, st, 2);
            substep(2, st, 3);
        }
        wait_stage();
        if ((kt & 3) == 0) load_scales(min((kt >> 2) + 2, kt_safe >> 2));
        load_stage(min(kt + D, kt_safe), done);
        if (live) {
            read_words(kt + 1, st_next);
            substep(3, st_next, 0);
        }
    }
    __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));  // no request into LDS outlives the block

    if constexpr (KG == 2) {
        // the groups add their accumulators: group 0 keeps the first half of the
        // fragments, group 1 the rest; each hands the other half over through LDS
        constexpr int NF = MI * NI, KEEP0 = (NF + 1) / 2;
        static_assert(sizeof(smem) >= sizeof(float) * NF * 16 * 256, "the exchange reuses the stages");
        float* xch = reinterpret_cast<float*>(smem);
        __syncthreads();
#pragma unroll
        for (int f = 0; f < NF; ++f)
            if ((f < KEEP0) != (kg == 0))
#pragma unroll
                for (int v = 0; v < 16; ++v) xch[(f * 16 + v) * 256 + tid] = acc[f / NI][f % NI][v];
        __syncthreads();
#pragma unroll
        for (int f = 0; f < NF; ++f)
            if ((f < KEEP0) == (kg == 0))
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[f / NI][f % NI][v] += xch[(f * 16 + v) * 256 + tid];
    }
    float* mine = p.ws + (static_cast<size_t>(blockIdx.y) * T + tm * TN + tn) * (BM * BN);
#pragma unroll
    for (int f = 0; f < MI * NI; ++f) {
        if (KG == 2 && (f < (MI * NI + 1) / 2) != (kg == 0)) continue;
        const int i = f / NI, j = f % NI;
        if (slices == 1) {
            epilogue_frag<MODE>(p, acc[i][j], m0 + wm * WM + i * 32, n0 + wn * WN + j * 32 + fr, lane);
        } else {
#pragma unroll
            for (int v = 0; v < 16; ++v) mine[(f * 16 + v) * 256 + tid] = acc[i][j][v];
        }
    }
}

template <int BM, int BN, int WGM, int MODE, int KG>
void launch_tile(const GemmParams& p, int slices, hipStream_t s) {
    const dim3 tiles((p.N + BN - 1) / BN, (p.M + BM - 1) / BM);
    gemm_w4a16_dma_kernel<BM, BN, WGM, MODE, KG><<<dim3(tiles.x * tiles.y, slices), 256 * KG, 0, s>>>(p);
    if (slices > 1) launch_reduce<BM, BN, WGM, MODE>(p, tiles, slices, s);
}

template <int MODE>
void launch_mode(int tile, const GemmParams& p, int slices, hipStream_t s) {
    switch (tile) {
        case 0: launch_tile<128, 256, 1, MODE, 1>(p, slices, s); break;
        case 1: launch_tile<128, 256, 1, MODE, 2>(p, slices, s); break;
        default: launch_tile<128, 128, 1, MODE, 2>(p, slices, s); break;
    }
}

}  // namespace

void launch_gemm_dma(int mode, int tile, const GemmParams& p, int slices, hipStream_t s) {
    switch (mode) {
        case kPlain: launch_mode<kPlain>(tile, p, slices, s); break;
        case kQKV: launch_mode<kQKV>(tile, p, slices, s); break;
        default: launch_mode<kSwiglu>(tile, p, slices, s); break;
    }
}

}  // namespace qe
