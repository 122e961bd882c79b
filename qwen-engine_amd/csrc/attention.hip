// Decode-loop kernels around the matrix path (gfx950): W4 embedding lookup,
// QKV bias + NeoX RoPE + KV-cache append, split-K flash-decode attention with
// the fused Q8_1 epilogue that feeds the O projection, and causal prefill
// attention.
//
// Reference behaviour: src/kernels/rmsnorm_rope.cu:15-51 (embedding),
// :320-423 (bias/RoPE/KV), src/kernels/attention_gqa.cu:20-311 (flash decode,
// stage-2 Q8_1 epilogue :263-310), :322-462 (prefill).  Layouts: KV cache
// [kv_head][max_seq][head_dim] fp16 per layer; q [T][q_dim], k/v [T][kv_dim].
// Head dim 128: one wave64 covers a head with 2 elements per lane, dot
// products reduce with DPP/swizzle (seg_sum<64>).
#include <algorithm>
#include <type_traits>

#include "attn_common.hpp"
#include "lds_dma.hpp"
#include "rope_common.hpp"

namespace qe {
namespace {

constexpr int kSplits = kFlashSplits;
constexpr int kHeadDim = 128;
constexpr int kVocab = 151936;  // VOCAB_SIZE: out-of-range token ids map to 0


// ---- embedding ---------------------------------------------------------------
__global__ __launch_bounds__(256) void embed_lookup_w4a16_kernel(const uint32_t* __restrict__ qw,
                                                                 const uint16_t* __restrict__ sc,
                                                                 const int32_t* __restrict__ ids,
                                                                 uint16_t* __restrict__ out,
                                                                 const qe_device_control_block* ctl, int H) {
    const int t = blockIdx.x;
    int32_t tok = 0;
    if (ids != nullptr) tok = ids[t];
    else if (ctl != nullptr) tok = ctl->token_id;
    if (tok < 0 || tok >= kVocab) tok = 0;
    const uint32_t* row = qw + static_cast<size_t>(tok) * (H / 8);
    const uint16_t* srow = sc + static_cast<size_t>(tok) * (H / 128);
    for (int i = threadIdx.x; i < H / 8; i += blockDim.x) {
        const qwen::qe_half8_t h = qwen::unpack_w4_to_half8(row[i], __builtin_bit_cast(_Float16, srow[i >> 4]));
        *reinterpret_cast<qwen::qe_half8_t*>(out + static_cast<size_t>(t) * H + i * 8) = h;
    }
}

// ---- QKV bias + NeoX RoPE + KV append ------------------------------------------
// grid (tokens, ceil((nq + nkv) / 2)), 256 threads: thread (hl, e) owns
// element e of head 2*blockIdx.y + hl of the combined [q heads, k heads]
// list; threads of a k head also own element e of the matching v head.
// Every operand is loaded once up front, one barrier separates the reads
// of the rotation partner from the in-place writes.
__global__ __launch_bounds__(256) void qkv_bias_rope_kv_append_kernel(
    uint16_t* __restrict__ q, uint16_t* __restrict__ k, uint16_t* __restrict__ v, const uint16_t* __restrict__ qb,
    const uint16_t* __restrict__ kb, const uint16_t* __restrict__ vb, uint16_t* __restrict__ kc,
    uint16_t* __restrict__ vc, const qe_device_control_block* ctl, int nq, int nkv, int hd, int max_seq,
    int rotary_dim, float rope_theta) {
    const int m = blockIdx.x;
    int pos = ctl != nullptr ? ctl->seq_pos + m : 0;
    if (pos >= max_seq) pos = max_seq - 1;
    const int per_block = blockDim.x / hd;  // heads per block (hd <= 256)
    const int hl = threadIdx.x / hd, e = threadIdx.x % hd;
    const int head = blockIdx.y * per_block + hl;
    const bool live = hl < per_block && head < nq + nkv;
    const bool is_k = head >= nq;
    const int q_dim = nq * hd, kv_dim = nkv * hd;
    const int rot = (rotary_dim > 0 && rotary_dim <= hd) ? rotary_dim : hd;
    const int half_rot = rot / 2;
    const int pe = e < rot ? (e < half_rot ? e + half_rot : e - half_rot) : e;  // rotation partner
    _Float16* hp = nullptr;
    const uint16_t* bp = nullptr;
    if (live) {
        hp = is_k ? reinterpret_cast<_Float16*>(k + static_cast<size_t>(m) * kv_dim + (head - nq) * hd)
                  : reinterpret_cast<_Float16*>(q + static_cast<size_t>(m) * q_dim + head * hd);
        bp = is_k ? (kb ? kb + (head - nq) * hd : nullptr) : (qb ? qb + head * hd : nullptr);
    }
    _Float16 xe = 0, xp = 0, ve = 0;
    if (live) {
        xe = hp[e];
        xp = hp[pe];
        if (bp) {  // bias added in fp16 (rounded) before the rotation
            xe = xe + __builtin_bit_cast(_Float16, bp[e]);
            xp = xp + __builtin_bit_cast(_Float16, bp[pe]);
        }
        if (is_k) {
            const size_t vo = static_cast<size_t>(m) * kv_dim + (head - nq) * hd + e;
            ve = __builtin_bit_cast(_Float16, v[vo]);
            if (vb) ve = ve + __builtin_bit_cast(_Float16, vb[(head - nq) * hd + e]);
        }
    }
    float outv = static_cast<float>(xe);
    if (e < rot) {
        float sn, cs;
        rope_sincos(pos, e < half_rot ? e : e - half_rot, rot, rope_theta, sn, cs);
        outv = rope_rotate(static_cast<float>(xe), static_cast<float>(xp), e < half_rot, sn, cs);
    }
    __syncthreads();  // partners read before anyone writes
    if (!live) return;
    const _Float16 o = static_cast<_Float16>(outv);
    hp[e] = o;
    if (is_k) {
        const size_t co = (static_cast<size_t>(head - nq) * max_seq + pos) * hd + e;
        kc[co] = __builtin_bit_cast(uint16_t, o);
        v[static_cast<size_t>(m) * kv_dim + (head - nq) * hd + e] = __builtin_bit_cast(uint16_t, ve);
        vc[co] = __builtin_bit_cast(uint16_t, ve);
    }
}

// ---- flash decode, stage 1 -----------------------------------------------------
// grid num_q_heads * kSplits, NT = 512 threads, one q head per block (GH = 1:
// the group's blocks each re-read the kv head's K and V rows, from L2 after
// the first, and every block merges one head's lane-group states; half a GQA
// group per block measured slower, the same bits per head).  A split is a contiguous run of
// flash_split_len(seq_len) positions (the reference's ceil(seq_len / 16), at
// least kFlashMinSplit).  The NT/16 lane groups of the block (16 lanes each)
// each take one position per step; lane j of a group holds dims 8j..8j+7 (one
// 16-byte K and V load per position), so a score is a v_dot2 chain plus a
// 16-lane DPP sum.  A round is 64 positions whose K and V rows are requested
// together; with more than one round the next round's rows are requested
// before the current one is used.  Softmax state per lane group in the exp2
// domain, rescaled once per round.  The lane-group states are merged through
// LDS (max, weights, weighted sum).
// Output per (q head, split): unnormalized o relative to the split max m, and
// (m, denominator) with m in natural-log units, as attention_gqa.cu's stage 1
// writes them.

constexpr int kFlashThreads = 512;  // stage-1 block: one q head, 32 lane groups

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

template <int GH>
struct FlashState {
    float m[GH], l[GH], o[GH][8];
};

// One round: step st < kSteps at positions r0 + NG*st + gid (NG lane groups).
template <int GH, int NG>
__device__ __forceinline__ void flash_round(FlashState<GH>& S, const u32x4 (&qraw)[GH], const u32x4 (&kr)[64 / NG],
                                            const u32x4 (&vr)[64 / NG], int r0, int t1, int gid) {
    constexpr int kSteps = 64 / NG;
    constexpr float kScale = 1.4426950408889634f * 0.08838834764831845f;  // log2(e) / sqrt(128)
    const int steps = min(kSteps, (t1 - r0 + NG - 1) / NG);
    float sc[GH][kSteps];
#pragma unroll
    for (int st = 0; st < kSteps; ++st) {
        const bool valid = st < steps && r0 + st * NG + gid < t1;
#pragma unroll
        for (int h = 0; h < GH; ++h) {
            float d = 0.0f;
            if (st < steps) {  // block-uniform
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    // copy the vector element first: a bit_cast straight from an
                    // element of an ext_vector always read element 0 (clang 22)
                    const uint32_t qw = qraw[h][i], kw = kr[st][i];
                    d = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, qw), __builtin_bit_cast(f16x2, kw), d, false);
                }
                d = qwen::seg_sum<16>(d) * kScale;
            }
            sc[h][st] = valid ? d : -INFINITY;
        }
    }
#pragma unroll
    for (int h = 0; h < GH; ++h) {
        float mn = S.m[h];
#pragma unroll
        for (int st = 0; st < kSteps; ++st) mn = fmaxf(mn, sc[h][st]);
        // no valid position yet: keep everything at zero
        const float alpha = mn == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(S.m[h] - mn);
        float l = S.l[h] * alpha;
        float o[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) o[i] = S.o[h][i] * alpha;
#pragma unroll
        for (int st = 0; st < kSteps; ++st) {
            if (st < steps) {
                const float p = sc[h][st] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(sc[h][st] - mn);
                l += p;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    // rows past the context may hold anything: never multiplied in
                    const uint32_t vw = sc[h][st] == -INFINITY ? 0u : static_cast<uint32_t>(vr[st][i]);
                    const f16x2 v2 = __builtin_bit_cast(f16x2, vw);
                    o[2 * i] += p * static_cast<float>(v2.x);
                    o[2 * i + 1] += p * static_cast<float>(v2.y);
                }
            }
        }
        S.m[h] = mn;
        S.l[h] = l;
#pragma unroll
        for (int i = 0; i < 8; ++i) S.o[h][i] = o[i];
    }
}

// 16 bytes of a cache row that other blocks on the XCD read too (SHARED), or that nobody reads again.
template <bool SHARED>
__device__ __forceinline__ u32x4 load_row(const uint16_t* p) {
    if constexpr (SHARED) return *reinterpret_cast<const u32x4*>(p);
    return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
}

// One block: GH q heads (qh0..qh0+GH-1) of kv head kvh over positions [t0, t1)
// with NT threads (NT/16 lane groups).
template <int GH, int NT, bool SHARED>
__device__ __forceinline__ void flash_decode_split(const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc,
                                                   float* __restrict__ part_o, float* __restrict__ part_lse,
                                                   const u32x4 (&qraw)[GH], u32x4 (&ka)[64 / (NT / 16)],
                                                   u32x4 (&va)[64 / (NT / 16)], int kvh, int qh0, int split, int t0,
                                                   int t1, int max_seq) {
    constexpr int NG = NT / 16, kSteps = 64 / NG;
    const int gid = threadIdx.x >> 4, j = threadIdx.x & 15;  // lane group of the block, lane in the group
    const size_t base = static_cast<size_t>(kvh) * max_seq * kHeadDim + 8 * j;
    FlashState<GH> S;
#pragma unroll
    for (int h = 0; h < GH; ++h) {
        S.m[h] = -INFINITY;
        S.l[h] = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i) S.o[h][i] = 0.0f;
    }
    if (t0 == split * kFlashMinSplit && t1 - t0 <= 64) {  // the rows requested ahead (contexts up to 16 * 64 positions)
        flash_round<GH, NG>(S, qraw, ka, va, t0, t1, gid);
    } else {
        // rounds of 64 positions in two register slots: the next round's rows
        // are in flight while this one is used (rounds of 128 and 256 positions
        // measure the same or slower).  Every load is unconditional (positions
        // clamped to the split); cached when other q heads of the group read
        // the same rows through the same L2, else not kept.
        auto load_round = [&](int r0, u32x4 (&kr)[kSteps], u32x4 (&vr)[kSteps]) __attribute__((always_inline)) {
#pragma unroll
            for (int st = 0; st < kSteps; ++st) {
                const size_t off = base + static_cast<size_t>(min(r0 + st * NG + gid, t1 - 1)) * kHeadDim;
                kr[st] = load_row<SHARED>(kc + off);
                vr[st] = load_row<SHARED>(vc + off);
            }
        };
        u32x4 kb[kSteps], vb[kSteps];
        load_round(t0, ka, va);
        for (int r0 = t0;;) {
            load_round(min(r0 + 64, t1 - 1), kb, vb);
            __builtin_amdgcn_sched_barrier(0);
            flash_round<GH, NG>(S, qraw, ka, va, r0, t1, gid);
            r0 += 64;
            if (r0 >= t1) break;
            load_round(min(r0 + 64, t1 - 1), ka, va);
            __builtin_amdgcn_sched_barrier(0);
            flash_round<GH, NG>(S, qraw, kb, vb, r0, t1, gid);
            r0 += 64;
            if (r0 >= t1) break;
        }
    }
    // merge the NG lane-group states through LDS, HP heads per pass (48 KB):
    // M = max_g m_g, w_g = exp2(m_g - M), L = sum_g l_g w_g, o = sum_g w_g o_g
    constexpr int HP = (GH * NG <= 96) ? GH : 96 / NG;
    __shared__ __align__(16) float s_o[NG][HP][kHeadDim];
    __shared__ float s_m[NG][HP], s_l[NG][HP], s_w[HP][NG];
    constexpr float kLn2 = 0.6931471805599453f;
#pragma unroll
    for (int h0 = 0; h0 < GH; h0 += HP) {
        if (h0 > 0) __syncthreads();  // the previous pass has read s_o
#pragma unroll
        for (int hh = 0; hh < HP; ++hh) {
            if (h0 + hh < GH) {
                float4* dst = reinterpret_cast<float4*>(&s_o[gid][hh][8 * j]);
                dst[0] = make_float4(S.o[h0 + hh][0], S.o[h0 + hh][1], S.o[h0 + hh][2], S.o[h0 + hh][3]);
                dst[1] = make_float4(S.o[h0 + hh][4], S.o[h0 + hh][5], S.o[h0 + hh][6], S.o[h0 + hh][7]);
                if (j == 0) {
                    s_m[gid][hh] = S.m[h0 + hh];
                    s_l[gid][hh] = S.l[h0 + hh];
                }
            }
        }
        __syncthreads();
        const int t = threadIdx.x;
        const int nh = min(HP, GH - h0);
        if (t < nh * NG) {  // thread (head t/NG, lane group t%NG): NG consecutive lanes per head
            const int hh = t / NG, g = t % NG;
            const float m = s_m[g][hh];
            const float mx = qwen::seg_max<NG>(m);
            const float w = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - mx);
            const float lt = qwen::seg_sum<NG>(s_l[g][hh] * w);
            s_w[hh][g] = w;
            if (g == 0) {
                const size_t row = static_cast<size_t>(qh0 + h0 + hh) * kSplits + split;
                part_lse[row * 2] = mx * kLn2;  // natural-log units (-inf with no positions; lt is 0 then)
                part_lse[row * 2 + 1] = lt;
            }
        }
        __syncthreads();
        // thread (head t/(32Q), dims 4*((t/Q)%32)..+3, quarter t%Q of the lane groups); the Q
        // partial sums of an output meet through a DPP quad reduction
        constexpr int Q = NT >= 128 * HP ? 4 : 1;
        if (t < nh * 32 * Q) {
            const int hh = t / (32 * Q), d = 4 * ((t / Q) & 31), qg = t % Q;
            float4 o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
            for (int gi = 0; gi < NG / Q; ++gi) {
                const int g = qg * (NG / Q) + gi;
                const float w = s_w[hh][g];
                const float4 v = *reinterpret_cast<const float4*>(&s_o[g][hh][d]);
                o.x += w * v.x;
                o.y += w * v.y;
                o.z += w * v.z;
                o.w += w * v.w;
            }
            if constexpr (Q == 4) {
                o.x = qwen::seg_sum<4>(o.x);
                o.y = qwen::seg_sum<4>(o.y);
                o.z = qwen::seg_sum<4>(o.z);
                o.w = qwen::seg_sum<4>(o.w);
            }
            if (qg == 0) {
                const size_t row = static_cast<size_t>(qh0 + h0 + hh) * kSplits + split;
                *reinterpret_cast<float4*>(part_o + row * kHeadDim + d) = o;
            }
        }
    }
}

// grid num_kv_heads * group / GH * kSplits: a block covers GH q heads of one kv head and split.
template <int GH, int NT, bool SHARED>
__global__ __launch_bounds__(NT) void flash_decode_stage1_kernel(const uint16_t* __restrict__ q,
                                                                 const uint16_t* __restrict__ kc,
                                                                 const uint16_t* __restrict__ vc,
                                                                 float* __restrict__ part_o,
                                                                 float* __restrict__ part_lse,
                                                                 const qe_device_control_block* ctl, int group,
                                                                 int max_seq) {
    constexpr int NG = NT / 16, kSteps = 64 / NG;
    // The blocks of a kv head's split (its group's q heads) share an L2: block b
    // runs on XCD b % 8 (workgroups are dealt out round robin), so unit u =
    // (split, kv head) takes blocks with b % 8 = u % 8.  With heads in launch
    // order every XCD fetched every row: 3.43 -> 2.69 us at 128 positions, 7.1
    // -> 4.4 at 3000, 19.4 -> 10.4 at 16000 (12 q heads, 2 kv heads).
    // With one q head per kv head there is nothing to share, and heads in launch
    // order are the faster ones (28 caches in turn): 16 heads 7.35 -> 6.40 us at 2000
    // positions, 4.25 -> 4.04 at 300; 8 heads 5.26 -> 4.94 and 3.38 -> 3.23.
    static_assert(kSplits % 8 == 0, "units fill the XCDs evenly");
    const int heads = group / GH;  // blocks per unit
    int split, kvh, qh0;
    if constexpr (SHARED) {
        const int x = blockIdx.x & 7, sl = blockIdx.x >> 3;
        const int unit = x + 8 * (sl / heads);
        split = unit % kSplits;
        kvh = unit / kSplits;
        qh0 = kvh * group + (sl % heads) * GH;
    } else {  // nothing to share: heads in launch order
        const int nkv = gridDim.x / kSplits;
        kvh = blockIdx.x % nkv;
        split = blockIdx.x / nkv;
        qh0 = kvh;
    }
    const int gid = threadIdx.x >> 4, j = threadIdx.x & 15;
    // q and the split's first 64 rows are requested before the position is
    // known: with splits of 64 positions (contexts up to 16 * 64) the rows are
    // those of split * 64 onwards; rows past the context are masked later
    u32x4 qraw[GH];
#pragma unroll
    for (int h = 0; h < GH; ++h) qraw[h] = *reinterpret_cast<const u32x4*>(q + (qh0 + h) * kHeadDim + 8 * j);
    u32x4 ka[kSteps], va[kSteps];
    {
        const size_t base = static_cast<size_t>(kvh) * max_seq * kHeadDim + 8 * j;
#pragma unroll
        for (int st = 0; st < kSteps; ++st) {
            const size_t off = base + static_cast<size_t>(min(split * kFlashMinSplit + st * NG + gid, max_seq - 1)) * kHeadDim;
            ka[st] = load_row<SHARED>(kc + off);
            va[st] = load_row<SHARED>(vc + off);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    const int seq_pos = ctl != nullptr ? ctl->seq_pos : 0;
    const int seq_len = min(seq_pos + 1, max_seq);
    const int per = flash_split_len(seq_len);
    const int t0 = split * per;
    const int t1 = min(t0 + per, seq_len);
    if (t0 >= t1) {
        if (threadIdx.x < GH) {
            const size_t li = (static_cast<size_t>(qh0 + threadIdx.x) * kSplits + split) * 2;
            part_lse[li] = -INFINITY;
            part_lse[li + 1] = 0.0f;
        }
        return;
    }
    flash_decode_split<GH, NT, SHARED>(kc, vc, part_o, part_lse, qraw, ka, va, kvh, qh0, split, t0, t1, max_seq);
}

// ---- flash decode, stage 2 + Q8_1 epilogue ---------------------------------------
// grid num_q_heads, 128 threads (one per element of the head).  Every
// thread loads the 16 (m, d) pairs and its 16 partials up front.
// acc = sum_s exp(m_s - m) / d * o_s; attn_out = fp16(acc).  Epilogue
// (attention_gqa.cu:263-310): d = max(max|acc|/127, 1e-8) per head (= one
// 128-group), q = clamp(rint(acc / d)), sum8 over 8 adjacent elements.
__global__ __launch_bounds__(128) void flash_decode_stage2_kernel(const float* __restrict__ part_o,
                                                                  const float* __restrict__ part_lse,
                                                                  uint16_t* __restrict__ attn_out,
                                                                  int8_t* __restrict__ q8, float* __restrict__ q_scale,
                                                                  int32_t* __restrict__ q_sum8) {
    const int qh = blockIdx.x, tid = threadIdx.x;
    float ms[kSplits], ds[kSplits], os[kSplits];
#pragma unroll
    for (int s = 0; s < kSplits; ++s) {
        const size_t row = static_cast<size_t>(qh) * kSplits + s;
        const float2 ml = *reinterpret_cast<const float2*>(part_lse + row * 2);
        ms[s] = ml.x;
        ds[s] = ml.y;
        os[s] = part_o[row * kHeadDim + tid];
    }
    float wt[kSplits];
    flash_split_weights(ms, ds, wt);
    const float acc = flash_combine(ds, wt, os);
    attn_out[static_cast<size_t>(qh) * kHeadDim + tid] = f2h(acc);
    if (q8 == nullptr) return;  // uniform across the block
    __shared__ float s_wmax[2];
    float mx = qwen::seg_max<64>(fabsf(acc));
    if ((tid & 63) == 0) s_wmax[tid >> 6] = mx;
    __syncthreads();
    const float d = flash_q8_scale(fmaxf(s_wmax[0], s_wmax[1]));
    if (tid == 0 && q_scale != nullptr) q_scale[qh] = d;
    const int v = flash_q8_value(acc, d);
    q8[static_cast<size_t>(qh) * kHeadDim + tid] = static_cast<int8_t>(v);
    int s8 = -8 * v;
    s8 += qwen::dpp_i32<0xB1>(s8);
    s8 += qwen::dpp_i32<0x4E>(s8);
    s8 += qwen::dpp_i32<0x141>(s8);  // row_half_mirror: sum over 8 lanes
    if ((tid & 7) == 0 && q_sum8 != nullptr) q_sum8[qh * (kHeadDim / 8) + (tid >> 3)] = s8;
}

// ---- causal prefill attention (matrix cores) ---------------------------------------
// The query heads of a kv head and the queries form one list of rows, row
// r = query r / group, head kvh * group + r % group: a block takes 128
// consecutive rows (32 per wave) of one kv head, whatever the group size, and
// its waves share the K and V tiles (64 keys) in LDS.  grid.x = (split, kv
// head, row block); a split is a run of whole key tiles.  KG = 2: two groups
// of four waves take alternate tiles of the run and merge through LDS at the end.
// v_mfma_f32_32x32x16_f16 with the rows as the columns:
//   S^T (32 keys x 32 rows) = K (keys x 128 dims) . Q^T - lane l holds key
//   l%32 / row l%32, dims 8*(l/32) + 16*kk; Q stays in registers; the result
//   has lane l = row l%32 holding 16 keys (8*(v/4) + 4*(l/32) + v%4), so a
//   row's max and sum are in-lane values plus one lane^32 swap;
//   O^T (128 dims x 32 rows) += V^T . P^T - P^T is the lane's own
//   probabilities (fp16, k order = the keys it holds; the k order inside an
//   MFMA is free when both operands agree), V^T comes out of the row-major V
//   tile through ds_read_b64_tr_b16 (lane i of 16 receives dim i of 4 keys).
// K and V go from memory straight into LDS (global_load_lds, 16 bytes a lane)
// a step ahead of their use.  A tile row is 256 bytes, its 16-byte chunk c
// stored at c ^ swz(key): the 16-byte reads of K (16 keys, one chunk) and the
// transposing reads of V (4 keys x 4 chunks a half wave) then touch every
// bank once (0 conflicts counted).
// Bound by the matrix cores and, beside them, the exponentials: 1024 rows on
// 15000 positions (12 q heads, 2 kv heads) take 113 us, and the merge of the
// splits 7.5 (traced; together 0.81 PFLOP/s), with the MFMAs busy 54 % of the time
// on a SIMD of a busy CU and 4.6 vector instructions an MFMA.  Before, every
// wave read K for itself from L2 and no keys were split: 450 us.  509 rows from
// position 0 23.2 -> 15.0 us, 4096 rows 211 -> 74 us.
// Online softmax in the exp2 domain (1/sqrt(d) folded into the exponent's fused
// multiply-add), fp32 accumulation.  The reference value a row subtracts is
// its running max, renewed only when the max has grown by more than
// kPrefillLag (the probabilities then reach at most 2^kPrefillLag, and their
// relative precision in fp16 does not change).  Each row decides for itself:
// unsplit and with one key group its bits do not depend on the rows beside it.
// The key splits and the two key groups, which follow from the whole launch
// (rows, context, workspace), change the order of its sums.
constexpr int kPaRows = 128;     // rows per block
constexpr int kPaKeys = 64;      // keys per tile
constexpr int kPaTileBytes = kPaKeys * kHeadDim * 2;
constexpr float kPrefillLag = 8.0f;
// A split holds at least this many tiles: with 4 instead of 8, 509 rows at
// position 1000 take 23.0 instead of 23.5 us and 17 rows 13.9 instead of 16.2,
// 1024 rows from position 0 22.4 instead of 24.3; 2 and 12 are slower (27.8, 23.9).
constexpr int kPaMinTiles = 4;
constexpr int kPaMaxSplits = 16;
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

// splits of a row block with `tiles` key tiles, at most `splits`
__device__ __forceinline__ int prefill_live_splits(int tiles, int splits) {
    return max(1, min(splits, tiles / kPaMinTiles));
}
// key tiles of row block rb (the keys its last row sees)
__device__ __forceinline__ int prefill_tiles(int rb, int rows, int group, int base, int max_seq) {
    const int last = min((rb + 1) * kPaRows, rows) - 1;
    const int len = min(base + last / group + 1, max_seq);
    return max(0, (len + kPaKeys - 1) / kPaKeys);
}

struct PrefillAttnParams {
    const uint16_t* q;
    const uint16_t* kc;
    const uint16_t* vc;
    uint16_t* out;
    const qe_device_control_block* ctl;
    float* part_o;   // [split][kv head][row][128] unnormalized
    float* part_ml;  // [split][kv head][row][2] (reference value, sum)
    int T, nq, nkv, group, max_seq, out_stride, splits, row_blocks;
};

__device__ __forceinline__ float xor32_max(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x),
                                                    false, false);
    const uint32_t a = r[0], b = r[1];
    return fmaxf(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
}

// DMA: the caches are 16-byte aligned (else tiles are copied element by element).
template <int KG, bool DMA>
__global__ __launch_bounds__(256 * KG, 2) void prefill_attention_kernel(PrefillAttnParams p) {
    // per key group: K buffers 0 and 1, V buffers 0 and 1
    __shared__ __align__(16) char smem[KG * 4 * kPaTileBytes];
    const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int wave = wave_all & 3, kg = wave_all >> 2;
    const int fr = lane & 31, h = lane >> 5;
    const int rb = p.row_blocks - 1 - static_cast<int>(blockIdx.x) % p.row_blocks;  // longest rows first
    const int cb = static_cast<int>(blockIdx.x) / p.row_blocks;
    const int kvh = cb % p.nkv, split = cb / p.nkv;
    const int rows = p.T * p.group;
    const int base = p.ctl != nullptr ? p.ctl->seq_pos : 0;
    const int nt_all = prefill_tiles(rb, rows, p.group, base, p.max_seq);
    const int live = KG == 2 ? 1 : prefill_live_splits(nt_all, p.splits);  // two groups: never split (the launcher)
    if (split >= live) return;
    const int it0 = static_cast<int>((static_cast<long long>(split) * nt_all) / live);
    const int it1 = static_cast<int>((static_cast<long long>(split + 1) * nt_all) / live);
    const int r = rb * kPaRows + wave * 32 + fr;
    const int rc = min(r, rows - 1);
    const int qi = rc / p.group, qh = kvh * p.group + rc % p.group;
    const int run_end = it1 * kPaKeys - 1;  // last key of the run
    const int lim = min(min(base + qi, p.max_seq - 1), run_end);  // last key this row takes here
    // keys every row of the wave takes: tiles that end at or before it skip the mask
    const int wave_lim = __builtin_amdgcn_readlane(lim, 0);
    // the last key that any row of the wave takes here
    const int wave_last = __builtin_amdgcn_readlane(lim, 31);
    const int key_max = max(0, min(base + p.T, p.max_seq) - 1);  // the last key that holds anything
    constexpr float kScale = 1.4426950408889634f * 0.08838834764831845f;  // log2(e) / sqrt(128)

    u32x4 qf[8];
    {
        const uint16_t* qr = p.q + (static_cast<size_t>(qi) * p.nq + qh) * kHeadDim + 8 * h;
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) qf[kk] = *reinterpret_cast<const u32x4*>(qr + 16 * kk);
    }
    // tile load i of a wave: tile rows 16 i + 4 wave + lane / 16, stored chunk
    // lane % 16, i.e. chunk (lane % 16) ^ swz(row) of memory
    const int lrow = 4 * wave + (lane >> 4);
    const int lcol = 8 * ((lane & 15) ^ (((lane >> 4) << 2) | wave));
    const uint32_t loff = static_cast<uint32_t>(2 * (lrow * kHeadDim + lcol));  // bytes
    const size_t hb = static_cast<size_t>(kvh) * p.max_seq * kHeadDim;
    const uint16_t* khead = p.kc + hb;
    const uint16_t* vhead = p.vc + hb;
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
                              (__attribute__((address_space(3))) void*)smem)) + kg * 4 * kPaTileBytes;
    // Tile t into buffer `buf` (0, 1: K; 2, 3: V); tile_barrier holds the waits.
    auto load_tile = [&](const uint16_t* head, int t, int buf) __attribute__((always_inline)) {
        const uint32_t dst = lds0 + buf * kPaTileBytes + wave * 1024;
        if constexpr (!DMA) {
            for (int i = 0; i < 4; ++i) {
                const uint16_t* src = head + static_cast<size_t>(min(t * kPaKeys + 16 * i + lrow, key_max)) * kHeadDim + lcol;
                uint16_t* to = reinterpret_cast<uint16_t*>(smem + (kg * 4 + buf) * kPaTileBytes + wave * 1024 + 4096 * i + 16 * lane);
                for (int e = 0; e < 8; ++e) to[e] = src[e];
            }
        } else if ((t + 1) * kPaKeys - 1 <= key_max) {  // uniform: one scalar address, one lane offset
#pragma unroll
            for (int i = 0; i < 4; ++i)
                lds_load_x4(dst + 4096 * i, head + (static_cast<size_t>(t) * kPaKeys + 16 * i) * kHeadDim, loff);
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int key = min(t * kPaKeys + 16 * i + lrow, key_max);
                lds_load_x4(dst + 4096 * i, head + static_cast<size_t>(key) * kHeadDim + lcol);
            }
        }
    };
    // every tile requested so far is in LDS, for every wave, and what was read before is read
    auto tile_barrier = [&]() __attribute__((always_inline)) {
        if constexpr (!DMA) __syncthreads();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    // LDS addresses: K chunk 2 kk + h of key fr; V^T reads (dt: 32 dims, u: keys + 8)
    uint32_t ka[8], va[4][2];
    {
        const int swz_k = ((fr & 3) << 2) | ((fr >> 2) & 3);
        const uint32_t k0 = lds0 + fr * 256 + 16 * (h ^ swz_k);
        const int s16 = lane & 15, b16 = (lane >> 4) & 1;
        const uint32_t v0 = lds0 + 2 * kPaTileBytes + (4 * h + (s16 >> 2)) * 256 +
                            16 * ((2 * b16 + ((s16 & 3) >> 1)) ^ (((s16 >> 2) << 2) | h)) + 8 * (s16 & 1);
#pragma unroll
        for (int kk = 0; kk < 8; ++kk) ka[kk] = k0 ^ (32 * kk);
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) {
            va[dt][0] = v0 ^ (64 * dt);
            va[dt][1] = (v0 ^ (64 * dt) ^ 32) + 8 * 256;
        }
    }
    // K operand of MFMA i of a tile: 32-key half i % 2, dims 16 (i / 2); V^T
    // operand: 16-key quarter i / 4, dims 32 (i % 4)
    auto read_k = [&](int buf, int i) __attribute__((always_inline)) {
        typedef const __attribute__((address_space(3))) f16x8* lptr;
        return *reinterpret_cast<lptr>(ka[i >> 1] + buf * kPaTileBytes + (i & 1) * 32 * 256);
    };
    auto read_v = [&](int buf, int i) __attribute__((always_inline)) {
        typedef __attribute__((address_space(3))) s16x4* lptr;
        const uint32_t off = (buf - 2) * kPaTileBytes + (i >> 2) * 16 * 256;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lptr>(va[i & 3][0] + off));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(reinterpret_cast<lptr>(va[i & 3][1] + off));
        return __builtin_bit_cast(f16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };

    f32x16 acc[4];
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) acc[dt] = f32x16{};
    float mref = -INFINITY, lsum = 0.0f;
    auto mask = [&](int t, f32x16 (&sc)[2]) __attribute__((always_inline)) {
        if ((t + 1) * kPaKeys - 1 > wave_lim) {  // wave-uniform
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int key = t * kPaKeys + 32 * j + 8 * (v >> 2) + 4 * h + (v & 3);
                    sc[j][v] = key <= lim ? sc[j][v] : -INFINITY;
                }
        }
    };
    auto renew_ref = [&](float mx) __attribute__((always_inline)) {
        const bool grow = mx > mref + kPrefillLag;
        if (__builtin_amdgcn_ballot_w64(grow) != 0) {
            const float alpha = grow ? __builtin_amdgcn_exp2f(mref - mx) : 1.0f;
            mref = grow ? mx : mref;
            lsum *= alpha;
#pragma unroll
            for (int dt = 0; dt < 4; ++dt)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[dt][v] *= alpha;
        }
    };
    auto row_max = [&](const f32x16 (&sc)[2]) __attribute__((always_inline)) {
        float mx = -INFINITY;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) mx = fmaxf(mx, sc[j][v]);
        return xor32_max(mx) * kScale;  // scaling is monotonic
    };
    // probabilities 2 i and 2 i + 1 of a tile's scores (32-key half i / 8), packed
    auto probs = [&](const f32x16 (&sc)[2], int i, float neg, float (&ps)[2]) __attribute__((always_inline)) {
        const int j = i >> 3, v = 2 * (i & 7);
        const f32x2 e = {__builtin_amdgcn_exp2f(__builtin_fmaf(sc[j][v], kScale, neg)),
                         __builtin_amdgcn_exp2f(__builtin_fmaf(sc[j][v + 1], kScale, neg))};
        ps[0] += e.x;
        ps[1] += e.y;
        uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(e, f16x2));
        asm volatile("" : "+v"(w), "+v"(ps[0]), "+v"(ps[1]));  // here, not past the mask's branch
        return w;
    };
    constexpr int AHEAD = 4;  // operand reads in flight before their MFMA
    // Scores of the K tile in `buf`; beside them, when EXP, the probabilities of
    // the scores `cur`.  Each MFMA is fenced together with its share of the
    // vector work: left alone, the scheduler puts all of the one before all
    // of the other.
    auto scores = [&](auto exp_too, int buf, f32x16 (&sc)[2], const f32x16 (&cur)[2],
                      uint32_t (&pw)[2][8]) __attribute__((always_inline)) {
        const float neg = mref == -INFINITY ? 0.0f : -mref;  // masked scores give exp2(-inf) = 0
        float ps[2] = {0.0f, 0.0f};
        f16x8 kf[AHEAD];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) kf[i] = read_k(buf, i);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            sc[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[i % AHEAD], __builtin_bit_cast(f16x8, qf[i >> 1]),
                                                               i < 2 ? f32x16{} : sc[i & 1], 0, 0, 0);
            if (i + AHEAD < 16) kf[i % AHEAD] = read_k(buf, i + AHEAD);
            if constexpr (decltype(exp_too)::value) pw[i >> 3][i & 7] = probs(cur, i, neg, ps);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (decltype(exp_too)::value) lsum += ps[0] + ps[1];
    };
    // O^T += V^T . P^T; beside it, when MAX, the (scaled) row maximum of nxt
    auto add_pv = [&](auto max_too, const uint32_t (&pw)[2][8], int buf, const f32x16 (&nxt)[2]) __attribute__((always_inline)) {
        f16x8 vf[AHEAD];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) vf[i] = read_v(buf, i);
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int j = i >> 3, ks = (i >> 2) & 1, dt = i & 3;
            const u32x4 pf = {pw[j][4 * ks], pw[j][4 * ks + 1], pw[j][4 * ks + 2], pw[j][4 * ks + 3]};
            acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[i % AHEAD], __builtin_bit_cast(f16x8, pf), acc[dt], 0, 0, 0);
            if (i + AHEAD < 16) vf[i % AHEAD] = read_v(buf, i + AHEAD);
            if constexpr (decltype(max_too)::value)
                mx = fmaxf(fmaxf(mx, nxt[j][2 * (i & 7)]), nxt[j][2 * (i & 7) + 1]);
            __builtin_amdgcn_sched_barrier(0);
        }
        return decltype(max_too)::value ? xor32_max(mx) * kScale : 0.0f;
    };
    typedef std::true_type yes;
    typedef std::false_type no;
    // Tile t of the run's scores are in cur: the scores of the group's next tile
    // beside the probabilities of t, then V of t beside the next tile's maximum.
    // b: parity of the tile; K of the tile after next and V of the next are requested.
    auto step = [&](int t, int b, f32x16 (&cur)[2], f32x16 (&nxt)[2]) __attribute__((always_inline)) {
        uint32_t pw[2][8];
        load_tile(vhead, t + KG, 2 + (b ^ 1));
        load_tile(khead, t + 2 * KG, b);
        scores(yes{}, b ^ 1, nxt, cur, pw);
        mask(t + KG, nxt);
        const float mx = add_pv(yes{}, pw, 2 + b, nxt);
        renew_ref(mx);
        tile_barrier();
    };
    auto finish = [&](int b, f32x16 (&cur)[2]) __attribute__((always_inline)) {
        uint32_t pw[2][8];
        const float neg = mref == -INFINITY ? 0.0f : -mref;
        float ps[2] = {0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < 16; ++i) pw[i >> 3][i & 7] = probs(cur, i, neg, ps);
        lsum += ps[0] + ps[1];
        add_pv(no{}, pw, 2 + b, cur);
    };
    if (it0 < it1) {
        const int n = (it1 - it0 + KG - 1) / KG;  // tiles of each group; past the run's end every key is masked
        int t = it0 + kg;
        load_tile(khead, t, 0);
        load_tile(vhead, t, 2);
        load_tile(khead, t + KG, 1);
        tile_barrier();
        f32x16 s0[2], s1[2];
        {
            uint32_t pw[2][8];
            scores(no{}, 0, s0, s1, pw);
        }
        mask(t, s0);
        renew_ref(row_max(s0));
        tile_barrier();  // K buffer 0 is read
        // Tiles past the wave's last key are not multiplied: they would add nothing but 0 * V, which is NaN where
        // a later position holds an infinity or NaN.
        const int mine = wave_last < t * kPaKeys ? 0 : min(n, (wave_last / kPaKeys - t) / KG + 1);
        int left = mine;
        for (; left > 2; left -= 2) {
            step(t, 0, s0, s1);
            step(t + KG, 1, s1, s0);
            t += 2 * KG;
        }
        if (left == 2) {
            step(t, 0, s0, s1);
            finish(1, s1);
        } else if (left == 1) {
            finish(0, s0);
        }
        for (int i = max(mine - 1, 0); i < n - 1; ++i) {  // the tiles of the other waves
            load_tile(vhead, it0 + kg + (i + 1) * KG, 2 + ((i & 1) ^ 1));
            load_tile(khead, it0 + kg + (i + 2) * KG, i & 1);
            tile_barrier();
        }
    }
    lsum += __shfl_xor(lsum, 32);
    if constexpr (KG == 2) {
        // The groups merge: each rescales to the common reference value, hands
        // over half of its accumulators through the (now idle) tile buffers
        // and finishes the other half: group 0 dims 0..63, group 1 dims 64..127.
        float* xch = reinterpret_cast<float*>(smem);  // [group][value][256 threads]
        float* xml = xch + 2 * 32 * 256;              // [group][2][256 threads]
        const int gt = wave * 64 + lane;
        __syncthreads();
        xml[(kg * 2 + 0) * 256 + gt] = mref;
        xml[(kg * 2 + 1) * 256 + gt] = lsum;
#pragma unroll
        for (int d = 0; d < 2; ++d)
#pragma unroll
            for (int v = 0; v < 16; ++v) xch[(kg * 32 + d * 16 + v) * 256 + gt] = kg == 0 ? acc[2 + d][v] : acc[d][v];
        __syncthreads();
        const float mo = xml[((kg ^ 1) * 2 + 0) * 256 + gt], lo = xml[((kg ^ 1) * 2 + 1) * 256 + gt];
        const float m = fmaxf(mref, mo);
        const float wm = mref == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mref - m);
        const float wo = mo == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mo - m);
        // one order for both groups, so that both hold the same sum
        const float l0 = kg == 0 ? lsum * wm : lo * wo, l1 = kg == 0 ? lo * wo : lsum * wm;
        lsum = l0 + l1;
#pragma unroll
        for (int d = 0; d < 2; ++d)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const float mine = kg == 0 ? acc[d][v] : acc[2 + d][v];
                acc[d][v] = mine * wm + xch[((kg ^ 1) * 32 + d * 16 + v) * 256 + gt] * wo;
            }
    }
    if (r >= rows) return;
    constexpr int ND = KG == 2 ? 2 : 4;  // 32-dim tiles this wave writes, from dim 64 kg
    if (KG == 2 || live == 1) {
        const float inv = lsum > 0.0f ? 1.0f / lsum : 0.0f;
        uint16_t* o = p.out + static_cast<size_t>(qi) * p.out_stride + qh * kHeadDim + 64 * kg;
#pragma unroll
        for (int dt = 0; dt < ND; ++dt)
#pragma unroll
            for (int g = 0; g < 4; ++g) {  // dims 32dt + 8g + 4h .. +3
                const uint32_t w0 = static_cast<uint32_t>(f2h(acc[dt][4 * g] * inv)) |
                                    (static_cast<uint32_t>(f2h(acc[dt][4 * g + 1] * inv)) << 16);
                const uint32_t w1 = static_cast<uint32_t>(f2h(acc[dt][4 * g + 2] * inv)) |
                                    (static_cast<uint32_t>(f2h(acc[dt][4 * g + 3] * inv)) << 16);
                *reinterpret_cast<uint2*>(o + 32 * dt + 8 * g + 4 * h) = make_uint2(w0, w1);
            }
        return;
    }
    const size_t prow = (static_cast<size_t>(split) * p.nkv + kvh) * rows + r;
    if (h == 0) *reinterpret_cast<float2*>(p.part_ml + 2 * prow) = make_float2(mref, lsum);
    float* po = p.part_o + prow * kHeadDim;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *reinterpret_cast<float4*>(po + 32 * dt + 8 * g + 4 * h) =
                make_float4(acc[dt][4 * g], acc[dt][4 * g + 1], acc[dt][4 * g + 2], acc[dt][4 * g + 3]);
}

// Merges the splits of every row: 32 lanes a row (4 dims each), 8 rows a
// block.  Rows whose block of 128 had one split are already written.  Lane s of
// a row reads the (max, sum) of split s, and the partial outputs are requested
// eight splits at a time, so a row waits for two rounds of loads: 1024 rows on
// 15000 positions (5 splits, 31 MB) 9.4 us with a loop over the splits, now 7.0.
__global__ __launch_bounds__(256) void prefill_attention_combine_kernel(PrefillAttnParams p) {
    static_assert(kPaMaxSplits <= 32, "a lane per split");
    const int rows = p.T * p.group;
    const int s_lane = threadIdx.x & 31, d = 4 * s_lane;
    const int base = p.ctl != nullptr ? p.ctl->seq_pos : 0;
    const int all = rows * p.nkv;
    const int i = blockIdx.x * 8 + (threadIdx.x >> 5);
    if (i >= all) return;
    const int kvh = i / rows, r = i - kvh * rows;
    const int live = prefill_live_splits(prefill_tiles(r / kPaRows, rows, p.group, base, p.max_seq), p.splits);
    if (live == 1) return;
    constexpr int B = 8;
    float2 ml = make_float2(-INFINITY, 0.0f);
    if (s_lane < live)
        ml = *reinterpret_cast<const float2*>(p.part_ml + 2 * (static_cast<size_t>(s_lane) * all + i));
    float4 v[B];
    auto request = [&](int s0) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < B; ++b)
            v[b] = *reinterpret_cast<const float4*>(
                p.part_o + (static_cast<size_t>(min(s0 + b, live - 1)) * all + i) * kHeadDim + d);
    };
    request(0);
    const float m = qwen::seg_max<32>(ml.x);
    const float w_lane = ml.x == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ml.x - m);
    float l = 0.0f;
    float4 o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int s0 = 0; s0 < live; s0 += B) {
        if (s0 > 0) request(s0);
#pragma unroll
        for (int b = 0; b < B; ++b) {
            if (s0 + b >= live) break;
            const float w = __shfl(w_lane, s0 + b, 32);
            l += w * __shfl(ml.y, s0 + b, 32);
            o.x += w * v[b].x;
            o.y += w * v[b].y;
            o.z += w * v[b].z;
            o.w += w * v[b].w;
        }
    }
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    uint16_t* dst =
        p.out + static_cast<size_t>(r / p.group) * p.out_stride + (kvh * p.group + r % p.group) * kHeadDim + d;
    *reinterpret_cast<uint2*>(dst) =
        make_uint2(static_cast<uint32_t>(f2h(o.x * inv)) | (static_cast<uint32_t>(f2h(o.y * inv)) << 16),
                   static_cast<uint32_t>(f2h(o.z * inv)) | (static_cast<uint32_t>(f2h(o.w * inv)) << 16));
}

}  // namespace
}  // namespace qe

using namespace qe;

extern "C" int qe_launch_embed_lookup_w4a16(const uint32_t* embed_qweight, const uint16_t* embed_scales,
                                            const int32_t* d_token_ids, uint16_t* out_hidden,
                                            const qe_device_control_block* d_control, int num_tokens,
                                            hipStream_t stream, int hidden_size) {
    QE_REQUIRE(embed_qweight && embed_scales && out_hidden, "embed_lookup_w4a16: NULL pointer");
    QE_REQUIRE(hidden_size > 0 && hidden_size % 128 == 0, "embed_lookup_w4a16: hidden_size=%d", hidden_size);
    QE_REQUIRE(aligned(out_hidden, 16), "embed_lookup_w4a16: out_hidden must be 16-byte aligned");
    if (num_tokens <= 0) return QE_OK;
    embed_lookup_w4a16_kernel<<<num_tokens, 256, 0, stream>>>(embed_qweight, embed_scales, d_token_ids, out_hidden,
                                                              d_control, hidden_size);
    return check_launch("embed_lookup_w4a16");
}

extern "C" int qe_launch_qkv_bias_rope_kv_append(uint16_t* q, uint16_t* k, uint16_t* v, const uint16_t* q_bias,
                                                 const uint16_t* k_bias, const uint16_t* v_bias,
                                                 uint16_t* layer_k_cache, uint16_t* layer_v_cache,
                                                 const qe_device_control_block* d_control, int num_tokens,
                                                 hipStream_t stream, int num_q_heads, int num_kv_heads, int head_dim,
                                                 int max_seq_len, int rotary_dim, float rope_theta) {
    QE_REQUIRE(q && k && v && layer_k_cache && layer_v_cache, "qkv_bias_rope_kv_append: NULL pointer");
    QE_REQUIRE(num_q_heads > 0 && num_kv_heads > 0 && head_dim > 0 && head_dim % 2 == 0 && max_seq_len > 0,
               "qkv_bias_rope_kv_append: bad head shape");
    if (num_tokens <= 0) return QE_OK;
    QE_REQUIRE(head_dim <= 256, "qkv_bias_rope_kv_append: head_dim=%d > 256", head_dim);
    const int heads_per_block = 256 / head_dim;
    const dim3 grid(num_tokens, (num_q_heads + num_kv_heads + heads_per_block - 1) / heads_per_block);
    qkv_bias_rope_kv_append_kernel<<<grid, 256, 0, stream>>>(q, k, v, q_bias, k_bias, v_bias, layer_k_cache,
                                                                   layer_v_cache, d_control, num_q_heads,
                                                                   num_kv_heads, head_dim, max_seq_len,
                                                                   rotary_dim, rope_theta);
    return check_launch("qkv_bias_rope_kv_append");
}

namespace qe {
namespace {
int launch_flash_stage1(const uint16_t* q, const uint16_t* kc, const uint16_t* vc, float* part_o, float* part_lse,
                        const qe_device_control_block* ctl, hipStream_t stream, int num_q_heads, int num_kv_heads,
                        int head_dim, int max_seq_len, const char* what) {
    QE_REQUIRE(q && kc && vc && part_o && part_lse, "%s: NULL pointer", what);
    QE_REQUIRE(head_dim == kHeadDim, "%s: head_dim=%d (only 128 is built)", what, head_dim);
    QE_REQUIRE(num_kv_heads > 0 && num_q_heads % num_kv_heads == 0, "%s: %d q heads over %d kv heads", what,
               num_q_heads, num_kv_heads);
    const int group = num_q_heads / num_kv_heads;
    QE_REQUIRE(max_seq_len > 0, "%s: max_seq_len=%d", what, max_seq_len);
    static_assert(kSplits % 8 == 0, "units fill the XCDs evenly");
    if (group > 1)
        flash_decode_stage1_kernel<1, kFlashThreads, true><<<num_q_heads * kSplits, kFlashThreads, 0, stream>>>(
            q, kc, vc, part_o, part_lse, ctl, group, max_seq_len);
    else
        flash_decode_stage1_kernel<1, kFlashThreads, false><<<num_q_heads * kSplits, kFlashThreads, 0, stream>>>(
            q, kc, vc, part_o, part_lse, ctl, group, max_seq_len);
    return QE_OK;
}
}  // namespace
}  // namespace qe

extern "C" int qe_launch_attention_gqa_flash_decode(const uint16_t* q, const uint16_t* layer_k_cache,
                                                    const uint16_t* layer_v_cache, float* splitk_partial_out,
                                                    float* splitk_partial_lse, uint16_t* attn_out,
                                                    const qe_device_control_block* d_control, hipStream_t stream,
                                                    int num_q_heads, int num_kv_heads, int head_dim,
                                                    int max_seq_len, int8_t* out_q8, float* out_scale,
                                                    int32_t* out_sum8) {
    QE_REQUIRE(attn_out, "attention_gqa_flash_decode: NULL pointer");
    QE_TRY(launch_flash_stage1(q, layer_k_cache, layer_v_cache, splitk_partial_out, splitk_partial_lse, d_control,
                               stream, num_q_heads, num_kv_heads, head_dim, max_seq_len,
                               "attention_gqa_flash_decode"));
    flash_decode_stage2_kernel<<<num_q_heads, 128, 0, stream>>>(splitk_partial_out, splitk_partial_lse, attn_out,
                                                                 out_q8, out_scale, out_sum8);
    return check_launch("attention_gqa_flash_decode");
}


extern "C" int qe_launch_attention_gqa_flash_decode_partials(const uint16_t* q, const uint16_t* layer_k_cache,
                                                             const uint16_t* layer_v_cache, float* splitk_partial_out,
                                                             float* splitk_partial_lse,
                                                             const qe_device_control_block* d_control,
                                                             hipStream_t stream, int num_q_heads, int num_kv_heads,
                                                             int head_dim, int max_seq_len) {
    QE_TRY(launch_flash_stage1(q, layer_k_cache, layer_v_cache, splitk_partial_out, splitk_partial_lse, d_control,
                               stream, num_q_heads, num_kv_heads, head_dim, max_seq_len,
                               "attention_gqa_flash_decode_partials"));
    return check_launch("attention_gqa_flash_decode_partials");
}

extern "C" int qe_launch_attention_gqa_flash_decode_combine(const float* splitk_partial_out,
                                                            const float* splitk_partial_lse, uint16_t* attn_out,
                                                            hipStream_t stream, int num_q_heads, int8_t* out_q8,
                                                            float* out_scale, int32_t* out_sum8) {
    QE_REQUIRE(splitk_partial_out && splitk_partial_lse && attn_out, "flash_decode_combine: NULL pointer");
    QE_REQUIRE(num_q_heads > 0, "flash_decode_combine: num_q_heads=%d", num_q_heads);
    flash_decode_stage2_kernel<<<num_q_heads, 128, 0, stream>>>(splitk_partial_out, splitk_partial_lse, attn_out,
                                                                 out_q8, out_scale, out_sum8);
    return check_launch("flash_decode_combine");
}

namespace qe {

// Whether launches on the stream are being recorded into a graph (or the runtime will not say).
static bool capturing(hipStream_t stream) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &st) == hipSuccess) return st != hipStreamCaptureStatusNone;
    (void)hipGetLastError();
    return true;
}

// Prefill attention; max_context bounds the positions the rows see (the
// engine knows it on the host, the public entry point only max_seq_len).
int launch_prefill_attention(const uint16_t* q, const uint16_t* layer_k_cache, const uint16_t* layer_v_cache,
                             uint16_t* attn_out, const qe_device_control_block* d_control, int num_tokens,
                             hipStream_t stream, int num_q_heads, int num_kv_heads, int head_dim, int max_seq_len,
                             int hidden_size, int max_context) {
    QE_REQUIRE(q && layer_k_cache && layer_v_cache && attn_out, "attention_gqa_prefill: NULL pointer");
    QE_REQUIRE(head_dim == kHeadDim, "attention_gqa_prefill: head_dim=%d (only 128 is built)", head_dim);
    QE_REQUIRE(num_kv_heads > 0 && num_q_heads % num_kv_heads == 0, "attention_gqa_prefill: bad head counts");
    QE_REQUIRE(hidden_size >= num_q_heads * head_dim, "attention_gqa_prefill: hidden_size=%d", hidden_size);
    if (num_tokens <= 0) return QE_OK;
    QE_REQUIRE(aligned(q, 16) && aligned(attn_out, 8) && hidden_size % 4 == 0,
               "attention_gqa_prefill: q must be 16-byte and attn_out 8-byte aligned");
    PrefillAttnParams p{};
    p.q = q;
    p.kc = layer_k_cache;
    p.vc = layer_v_cache;
    p.out = attn_out;
    p.ctl = d_control;
    p.T = num_tokens;
    p.nq = num_q_heads;
    p.nkv = num_kv_heads;
    p.group = num_q_heads / num_kv_heads;
    p.max_seq = max_seq_len;
    p.out_stride = hidden_size;
    const long long rows = static_cast<long long>(num_tokens) * p.group;
    const long long row_blocks = (rows + kPaRows - 1) / kPaRows;
    const long long blocks = row_blocks * num_kv_heads;
    QE_REQUIRE(rows <= INT32_MAX - kPaRows && blocks <= INT32_MAX, "attention_gqa_prefill: num_tokens=%d", num_tokens);
    if (blocks == 0) return QE_OK;  // no q heads
    p.row_blocks = static_cast<int>(row_blocks);
    // Key splits as far as the chip has room for their blocks (two per CU),
    // the stream's workspace for their partials, and the context has tiles;
    // a row block then takes as many of them as its own tiles are worth.
    const int cus = cu_count();
    const WorkspaceLease lease(stream);  // until both kernels are enqueued
    const StreamWorkspace ws = lease.ws;
    const long long part = rows * num_kv_heads * (kHeadDim + 2);  // floats of one split
    p.splits = 1;
    // (contexts below 16 tiles: the second launch costs what the splits save)
    if (ws.ptr != nullptr && max_context >= 16 * kPaKeys)
        p.splits = static_cast<int>(std::max(1LL, std::min({static_cast<long long>(kPaMaxSplits), 2 * cus / blocks,
                                                            static_cast<long long>(ws.floats) / part,
                                                            static_cast<long long>(max_context) / (kPaKeys * kPaMinTiles)})));
    // A graph may be replayed on any stream and after the workspace is gone: a recorded launch touches none.
    if (p.splits > 1 && capturing(stream)) p.splits = 1;
    p.part_o = ws.ptr;
    p.part_ml = ws.ptr + p.splits * rows * num_kv_heads * kHeadDim;
    // Two key groups per block (one block per CU) once there is more than one
    // block per CU: blocks half as long leave a smaller last round (4096 rows
    // from position 0, 384 blocks: 75 against 88 us).  With fewer blocks a
    // wave that has its SIMD to itself finishes its tiles sooner (509 rows: 13.7
    // against 16.3 us).  More blocks than CUs also leave no room for splits (above).
    if (!aligned(layer_k_cache, 16) || !aligned(layer_v_cache, 16))
        prefill_attention_kernel<1, false><<<static_cast<unsigned>(blocks * p.splits), 256, 0, stream>>>(p);
    else if (blocks > cus)
        prefill_attention_kernel<2, true><<<static_cast<unsigned>(blocks), 512, 0, stream>>>(p);
    else
        prefill_attention_kernel<1, true><<<static_cast<unsigned>(blocks * p.splits), 256, 0, stream>>>(p);
    if (p.splits > 1)
        prefill_attention_combine_kernel<<<static_cast<unsigned>((rows * num_kv_heads + 7) / 8), 256, 0, stream>>>(p);
    return check_launch("attention_gqa_prefill");
}

}  // namespace qe

extern "C" int qe_launch_attention_gqa_prefill(const uint16_t* q, const uint16_t* layer_k_cache,
                                               const uint16_t* layer_v_cache, uint16_t* attn_out,
                                               const qe_device_control_block* d_control, int num_tokens,
                                               hipStream_t stream, int num_q_heads, int num_kv_heads, int head_dim,
                                               int max_seq_len, int hidden_size) {
    return qe::launch_prefill_attention(q, layer_k_cache, layer_v_cache, attn_out, d_control, num_tokens, stream,
                                        num_q_heads, num_kv_heads, head_dim, max_seq_len, hidden_size, max_seq_len);
}
