// A decode step in two launches: every wave takes a segment of the context through forward_qk, the softmax
// and forward_ov, with the softmax taken over the segment alone; a second launch puts the segments
// together.  Included by adkv_kernels.hip after the shared device helpers.
//
// Launches of short segments spend much of their time around the loops: table, first loads and the uneven
// end of forward_qk and again of forward_ov, a pass over the logits between them and one over the
// partial outputs behind them.  Here a wave that has finished its keys goes on with its values at
// once.  Its weights are exp(x - m) with m the segment's own maximum, rounded to fp16 like the
// final weights (relative to the segment's largest, so none is rounded more coarsely than before),
// and live in the wave's LDS; their sum is kept in fp32 twice, before and after that rounding.
// step_combine_kernel has the maxima and sums of all segments in hand, writes the weights from the logits
// in the steps of the softmax kernels, and adds the partial outputs, each scaled by exp(m - M) and the
// whole divided by the sum of the rounded weights, so that what they were rounded by cancels in part.  Against 64
// bits the rms error of the outputs, relative to their own rms, two launches / three: 5.86e-4 / 6.04e-4 at
// 64 x 32 heads x 663 tokens masked, 4.80 / 4.90 at 8 x 8 x 16 001 with four query heads, 4.66 / 4.62 at 4 x 8 x
// 8190 of 256 channels; 0.96 to 1.01 times over thirteen such sizes and logit spreads, 0.76 and 0.88 at
// 60 000 tokens, where weights of the whole row are subnormal.
#pragma once

namespace adkv {

// Longest segment, appended token included, whose weights fit a wave's LDS: 512 tokens (256 with eight
// query heads) and one, in whole 16-byte vectors.
template <int GQ> constexpr int step_cap() { return GQ == 8 ? 264 : 520; }

// max or sum over the LPH lanes of a head, in registers: four rotations within the row of 16 lanes, then
// the row and half swaps.  (Through the LDS, as __shfl_xor goes, the dozen trips per head took 4 of the 55
// us of a step of 256-token segments with four query heads.)
template <bool MAX>
__device__ __forceinline__ float fold(float a, float b) { return MAX ? fmaxf(a, b) : a + b; }
template <int CTRL, bool MAX>
__device__ __forceinline__ float fold_row(float v)
{
    const int o = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false);
    return fold<MAX>(v, __builtin_bit_cast(float, o));
}
template <int LPH, bool MAX>
__device__ __forceinline__ float head_reduce(float v)
{
    v = fold_row<0x128, MAX>(v); // row_ror:8
    v = fold_row<0x124, MAX>(v);
    v = fold_row<0x122, MAX>(v);
    v = fold_row<0x121, MAX>(v);
    unsigned a = __builtin_bit_cast(unsigned, v), b; // see xor16_add
    asm volatile("v_mov_b32 %0, %1" : "=v"(b) : "v"(a));
    const u2v r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    unsigned x = r.x, y = r.y;
    asm volatile("" : "+v"(x), "+v"(y));
    v = fold<MAX>(__builtin_bit_cast(float, x), __builtin_bit_cast(float, y));
    if (LPH == 64) {
        a = __builtin_bit_cast(unsigned, v);
        asm volatile("v_mov_b32 %0, %1" : "=v"(b) : "v"(a));
        const u2v h = __builtin_amdgcn_permlane32_swap(a, b, false, false);
        x = h.x;
        y = h.y;
        asm volatile("" : "+v"(x), "+v"(y));
        v = fold<MAX>(__builtin_bit_cast(float, x), __builtin_bit_cast(float, y));
    }
    return v;
}

// The segment's weights of GQ heads: p[g * step_cap + t] = fp16(exp(x - m)) for t < ntok, zeros up to the
// next multiple of 256 or the cap (a vector of eight reads no further than its supergroup); m and the sums over the segment, before and after
// rounding, go to ml[g * nseg].  logits: the first head's row at
// the segment's first token, 16-byte aligned, its pitch a multiple of 8.
template <int LPH, int GQ>
__device__ __forceinline__ void segment_weights(const h1 *logits, long pitch, const Mask &mk, long row0, int n, int t0,
                                                int ntok, float scaling, h1 *p, float4 *ml, int nseg, int lh, bool active)
{
    constexpr int V = 256 / LPH, CAP = step_cap<GQ>(), NC = (CAP + 255) / 256; // values per lane, chunks of 256 tokens
    using Raw = typename std::conditional<V == 4, uint2, uint4>::type;
    Raw raw[GQ][NC];
#pragma unroll
    for (int g = 0; g < GQ; g++)
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const int t = c * 256 + lh * V;
            raw[g][c] = vec_zero<Raw>();
            if (t < ntok) // reads at most to the next multiple of V, inside the row's pitch
                raw[g][c] = *reinterpret_cast<const Raw *>(logits + g * pitch + t);
        }
#pragma unroll
    for (int g = 0; g < GQ; g++) {
        const MaskRow<true> mrow = mk.of<true>((unsigned)row0 + g, n, t0);
        float x[NC][V], mx = -INFINITY;
#pragma unroll
        for (int c = 0; c < NC; c++) {
            if (c * 256 >= ntok)
                break;
            uint32_t w[V / 2];
            vec_words(raw[g][c], w);
            const int t = c * 256 + lh * V;
            float add[V];
            if (mrow) {
                if (t + V <= ntok) {
                    mrow.load<V>(t, add);
                } else {
#pragma unroll
                    for (int k = 0; k < V; k++)
                        add[k] = t + k < ntok ? mrow.at(t + k) : 0.0f;
                }
            }
#pragma unroll
            for (int k = 0; k < V; k++) {
                const h2 pair = as_h2(w[k / 2]);
                float v = (float)(k & 1 ? pair.y : pair.x) * scaling;
                if (mrow)
                    v += add[k];
                x[c][k] = t + k < ntok ? v : -INFINITY;
                mx = fmaxf(mx, x[c][k]);
            }
        }
        mx = head_reduce<LPH, true>(mx);
        const float ref = mx == -INFINITY ? 0.0f : mx; // nothing but -inf: all weights are zero
        float sum = 0.0f, rounded = 0.0f;
#pragma unroll
        for (int c = 0; c < NC; c++) {
            if (c * 256 >= ntok)
                break;
            uint32_t w[V / 2];
#pragma unroll
            for (int k = 0; k < V; k += 2) {
                const float a = __expf(x[c][k] - ref), b = __expf(x[c][k + 1] - ref);
                const h2 ab = (h2){(h1)a, (h1)b};
                sum += a + b;
                rounded += (float)ab.x + (float)ab.y;
                w[k / 2] = as_u32(ab);
            }
            Raw r;
            words_vec(w, r);
            if (c * 256 + lh * V < CAP)
                *reinterpret_cast<Raw *>(p + g * CAP + c * 256 + lh * V) = r;
        }
        sum = head_reduce<LPH, false>(sum);
        rounded = head_reduce<LPH, false>(rounded);
        if (active && lh == 0)
            ml[g * nseg] = make_float4(mx, sum, rounded, 0.0f);
    }
}

template <int D, int CPL, int BITS, int GQ>
struct StepShape {
    static constexpr int LPH = D / CPL, HEADS = 64 / LPH; // lanes per head, heads per wave
    // a wave's LDS: with two channels per lane the key tile, then the weights in the same place
    static constexpr int WEIGHTS = HEADS * GQ * step_cap<GQ>() * 2;
    static constexpr int SLOT = CPL == 2 && WEIGHTS < PAIR_TILE ? PAIR_TILE : (WEIGHTS + 15) / 16 * 16;
};

template <int D, int CPL, int BITS, int GQ, int BLK>
__global__ __launch_bounds__(BLK) void step_segments_kernel(
    const h1 *q, uint4 *__restrict__ k_cache, const h1 *k_new, uint4 *__restrict__ v_cache, const h1 *v_new, Mask mk,
    h1 *logits, float *__restrict__ partial, float4 *__restrict__ ml, FtParams kp, FtParams vp, int BH, int H, int T,
    int n_super_cap, float scaling, Seg ka, Seg va)
{
    using G = Geo<D, CPL>;
    using Shape = StepShape<D, CPL, BITS, GQ>;
    constexpr bool PAIR = CPL == 2, GROUPED = GQ > 1 || BITS != 4;
    constexpr int CAP = step_cap<GQ>();
    static_assert(PAIR || !GROUPED, "grouped queries and 2-bit codes: a KV head per wave");
    __shared__ uint4 smem[(LUT_WORDS64 * 8 + BLK / 64 * Shape::SLOT) / 16];
    ka.groups = va.groups = 0; // only even plans come here
    uint2 *lut = reinterpret_cast<uint2 *>(smem);
    char *slot = reinterpret_cast<char *>(smem) + LUT_WORDS64 * 8 + (threadIdx.x >> 6) * Shape::SLOT;
    const int lane = threadIdx.x & 63;
    const uint32_t lane_copy = table_lane_offset<BITS>(lane);
    const Unit<D, CPL, BLK> un(BH, ka.nseg); // a padding wave's is valid too: it loads and leaves
    const int bx = un.bx, lh = un.lh, c0 = un.c0, h = bx % H;
    const bool active = un.active;

    uint32_t qw[G::NP];
    __builtin_memcpy(qw, q + (size_t)bx * GQ * D + c0, 2 * CPL);
    using Scores = PairScores<BITS, GQ, BLK == 256>;
    Scores scores(slot, lane, q + (size_t)bx * GQ * D); // two channels per lane only
    SegLoads<D, CPL, BITS, PAIR ? Scores::AHEAD : PF> s;
    s.start(k_cache, kp.zp, kp.sc, kp.al, kp.be, kp.tg, h, bx, lh, un.seg, T, n_super_cap, ka);
    fill_table<BITS, BLK>(lut, threadIdx.x);
    __syncthreads();
    if (!un.wave_active)
        return;
    const int t0 = s.t0, ntok = s.t1 - s.t0 + (s.last ? 1 : 0); // the appended token is the last segment's
    if constexpr (PAIR)
        qk_gqa_pair_segment<BITS, GQ>(lut, lane, bx, scores, s, k_new, logits, T, nullptr, ka);
    else
        qk_segment<D, CPL>(lut, lane_copy, lane, bx, lh, c0, active, scores, s, qw, k_new, logits, T, nullptr, ka);

    // the values' state and codes travel while the weights are made
    constexpr int AHEAD = GROUPED ? gqa_ahead<BITS, GQ, CPL>() : PAIR ? PF_PAIR : PF;
    SegLoads<D, CPL, BITS, AHEAD> sv;
    sv.start(v_cache, vp.zp, vp.sc, vp.al, vp.be, vp.tg, h, bx, lh, un.seg, T, n_super_cap, va);
    // this wave's logits were written by other lanes of it
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    h1 *p = reinterpret_cast<h1 *>(slot) + lane / Shape::LPH * CAP; // one head per wave where there are several query heads
    const long row0 = (long)bx * GQ, rows = (long)BH * GQ;
    segment_weights<Shape::LPH, GQ>(logits + row0 * ka.row_pitch + t0, ka.row_pitch, mk, row0, T + 1, t0, ntok, scaling, p,
                                    ml + row0 * ka.nseg + un.seg, ka.nseg, lh, active);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");

    float *part = partial + (un.seg * rows + row0) * D + c0;
    if constexpr (GROUPED) {
        constexpr int NB = (GQ + 3) / 4, UPS = 4 / BITS;
        static_assert(UPS == Code<BITS>::TPW / 8, "units of eight tokens per supergroup");
        const int nunits = sv.nfull * UPS, r = lane & 3;
        auto w8 = [&](int n, int unit) __attribute__((always_inline)) {
            return *reinterpret_cast<const uint4 *>(p + min(4 * n + r, GQ - 1) * CAP + unit * 8);
        };
        uint4 wbuf[GQA_WPF][NB];
#pragma unroll
        for (int i = 0; i < GQA_WPF; i++)
#pragma unroll
            for (int n = 0; n < NB; n++)
                wbuf[i][n] = w8(n, min(i, max(nunits - 1, 0)));
        f4v acc[NB][CPL];
        ov_gqa_segment<BITS, GQ, CPL>(lut, lane_copy, bx, c0, active, sv, wbuf, w8, [&](int g, int t) { return p[g * CAP + t]; },
                                      v_new, T, nullptr, va, acc);
#pragma unroll
        for (int g = 0; g < GQ; g++)
            *reinterpret_cast<float2 *>(part + g * D) = make_float2(acc[g >> 2][0][g & 3], acc[g >> 2][1][g & 3]);
    } else {
        constexpr int WR = 2;
        auto w8 = [&](int sg) __attribute__((always_inline)) { return *reinterpret_cast<const uint4 *>(p + sg * 8); };
        uint4 wbuf[WR];
#pragma unroll
        for (int i = 0; i < WR; i++)
            wbuf[i] = w8(min(i, max(sv.nfull - 1, 0)));
        float acc[CPL];
        ov_segment<D, CPL, WR>(lut, lane_copy, bx, c0, active, sv, wbuf, w8, [&](int t) { return p[t]; }, v_new, T, nullptr, va, acc);
        if (active)
#pragma unroll
            for (int c = 0; c < CPL; c += 2)
                *reinterpret_cast<float2 *>(part + c) = make_float2(acc[c], acc[c + 1]);
    }
}

// The weights of one head of a unit of step_lone_kernel (see segment_weights): a token's logit is the sum of its shares in HW
// rows, `stride` apart; four tokens per lane, and the one behind 256.  writes: this wave leaves the logits, m and the sums too.
template <int HW>
__device__ __forceinline__ void lone_weights(const float *share, int stride, h1 *logits, const MaskRow<true> &mrow, int ntok,
                                             float scaling, h1 *p, float4 *ml, int lane, bool writes)
{
    const int t = lane * 4;
    float4 a = *reinterpret_cast<const float4 *>(share + t);
    float extra = share[256];
#pragma unroll
    for (int i = 1; i < HW; i++) {
        const float4 b = *reinterpret_cast<const float4 *>(share + i * stride + t);
        a = make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
        extra += share[i * stride + 256];
    }
    // Eight shares are added here: the compiler puts the additions behind the mask's loads and keeps all 40 registers until then, beside
    // the units that the values' waves hold (18 spilled; 2 x 8 heads x 2000 of 512 channels 16.9 us, 16.6 like this, 1 x 8 x 8000 19.0 / 18.7).
    if constexpr (HW == 8)
        asm volatile("" : "+v"(a.x), "+v"(a.y), "+v"(a.z), "+v"(a.w), "+v"(extra));
    const h1 l[5] = {(h1)a.x, (h1)a.y, (h1)a.z, (h1)a.w, (h1)extra};
    if (writes) {
        if (t + 4 <= ntok) { // t0 and the pitch are multiples of 8
            *reinterpret_cast<uint2 *>(logits + t) = make_uint2(as_u32((h2){l[0], l[1]}), as_u32((h2){l[2], l[3]}));
        } else {
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (t + k < ntok)
                    logits[t + k] = l[k];
        }
        if (lane == 0 && ntok > 256)
            logits[256] = l[4];
    }
    float add[5] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f}, x[5], mx = -INFINITY;
    if (mrow) {
        if (t + 4 <= ntok) {
            mrow.load<4>(t, add);
        } else {
#pragma unroll
            for (int k = 0; k < 4; k++)
                add[k] = t + k < ntok ? mrow.at(t + k) : 0.0f;
        }
        if (ntok > 256)
            add[4] = mrow.at(256);
    }
#pragma unroll
    for (int k = 0; k < 5; k++) {
        const float v = (float)l[k] * scaling + add[k];
        x[k] = (k < 4 ? t + k : 256) < ntok ? v : -INFINITY;
        mx = fmaxf(mx, x[k]);
    }
    mx = head_reduce<64, true>(mx);
    const float ref = mx == -INFINITY ? 0.0f : mx; // nothing but -inf: all weights are zero
    float e[5];
    h1 w[5];
#pragma unroll
    for (int k = 0; k < 5; k++) {
        e[k] = __expf(x[k] - ref);
        w[k] = (h1)e[k];
    }
    const float sum = head_reduce<64, false>((e[0] + e[1]) + (e[2] + e[3])) + e[4];
    const float rounded = head_reduce<64, false>(((float)w[0] + (float)w[1]) + ((float)w[2] + (float)w[3])) + (float)w[4];
    *reinterpret_cast<uint2 *>(p + t) = make_uint2(as_u32((h2){w[0], w[1]}), as_u32((h2){w[2], w[3]}));
    if (lane == 0)
        *reinterpret_cast<uint4 *>(p + 256) = make_uint4(as_u32((h2){w[4], (h1)0.0f}), 0, 0, 0);
    if (writes && lane == 0)
        *ml = make_float4(mx, sum, rounded, 0.0f);
}

// A wave's channels of a segment's values by its weights p (a row of LONE_SEG per query head), to o.  ahead: the first `done` units
// of the AHEAD that lone_values_ahead was to hold.
template <int D, int BITS, int GQ, int AHEAD>
__device__ __forceinline__ void lone_step_values(const uint2 *lut, uint32_t lane_copy, LoneLoads<D, BITS> &s, Lone &st, const uint32_t *ahead, int done,
                                                 const h1 *p, int bx, int c, int T, int lane, const Seg &va, float *o)
{
    if constexpr (GQ == 1 && D != 512) {
        // measured, adding on the vector pipe / on the matrix cores: 4 x 8 x 8190 of 256 channels 30.4 / 31.3, 8 x 32 x 2000
        // 28.0 / 29.2, 4 x 32 x 2000 19.6 / 19.3; 8 x 8 x 2000 of 512 30.5 / 28.9
        float acc = 0.0f;
        if constexpr (AHEAD > 0)
            lone_weigh<AHEAD>(ahead, done, p, acc);
        lone_values(lut, lane_copy, s, st, s.nfull * s.UPS - done, p + done * 8, acc);
        lone_values_end(s, st, [&](int t) { return p[t]; }, bx, c, T, nullptr, va, true, acc);
        *o = acc;
        return;
    }
    constexpr int NB = (GQ + 3) / 4;
    f4v acc[NB];
#pragma unroll
    for (int n = 0; n < NB; n++)
        acc[n] = (f4v){0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (AHEAD > 0)
        lone_weigh_grouped<GQ, AHEAD>(ahead, done, p, lane, acc);
    lone_values_grouped<GQ>(lut, lane_copy, s, st, s.nfull * s.UPS - done, p + done * 8, lane, acc);
    if (s.last) {
        auto token = [&](int t, float v) __attribute__((always_inline)) {
#pragma unroll
            for (int g = 0; g < GQ; g++)
                acc[g >> 2][g & 3] = __builtin_fmaf((float)p[g * LONE_SEG + t], v, acc[g >> 2][g & 3]);
        };
#pragma unroll
        for (int t = 0; t < s.TPW - 1; t++)
            if (t < s.ntail)
                token(s.TPW * s.nfull + t, (float)lone_token(st, s.code(t)));
        token(T - s.t0, (float)lone_append(s, st, bx, c, T, nullptr, va, true));
    }
#pragma unroll
    for (int g = 0; g < GQ; g++)
        o[g * D] = acc[g >> 2][g & 3];
}

// The same launch with one channel per lane, a KV head over D / 64 waves (adkv_lone.h): segments of at most 256 tokens.
// With few waves per SIMD a step takes as long as one wave's instructions per token, and a lane with four or eight
// channels has two and four times as many of them; the waves of a head meet once, behind the keys, where each has left
// its share of the logits (fp32) in the LDS, and with several query heads again behind the weights.
// Of the 256 + 256 tokens of a full segment a lone wave takes some 9 us (19 ns per token, step_segments_kernel 27 with two
// channels per lane, 50 with four and 90 with eight); from four waves per SIMD on vector issue holds it, 23 cycles per
// wave and token.  us per step: 2 x 8 heads x 1000 of 512 channels 47.7 / 18.7, 2 x 16 x 5021 of 256 31.7 / 23.2, 3 x 8 x 4799 with
// eight query heads 29.4 / 19.8; step_lone_threads has the rest.
template <int D, int BITS, int GQ, int BLK>
__global__ __launch_bounds__(BLK) void step_lone_kernel(
    const h1 *q, uint4 *k_cache, const h1 *k_new, uint4 *v_cache, const h1 *v_new, Mask mk, h1 *logits, float *__restrict__ partial,
    float4 *__restrict__ ml, FtParams kp, FtParams vp, int BH, int H, int T, int n_super_cap, float scaling, Seg ka, Seg va)
{
    constexpr int WAVES = BLK / 64, HW = D / 64, UNITS = WAVES / HW;
    static_assert(WAVES % HW == 0, "whole heads");
    // a wave's key tile; then its copy of the weights, or its share of those that the waves of a unit write together
    constexpr int WEIGHTS = GQ == 1 ? 0 : GQ * LONE_SEG * 2 / HW, SLOT = WEIGHTS > LONE_TILE ? WEIGHTS : LONE_TILE;
    static_assert(SLOT % 16 == 0, "vectors");
    __shared__ uint4 smem[(LUT_WORDS64 * 8 + WAVES * (SLOT + GQ * LONE_SEG * 4)) / 16];
    ka.groups = va.groups = 0; // only even plans come here
    uint2 *lut = reinterpret_cast<uint2 *>(smem);
    char *lds = reinterpret_cast<char *>(smem) + LUT_WORDS64 * 8;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int u = wave / HW, part = wave % HW, c = part * 64 + lane;
    const uint32_t lane_copy = table_lane_offset<BITS>(lane);
    int seg, wis;
    interleave_segment((int)blockIdx.x * UNITS + u, ka.nseg, seg, wis);
    const bool active = wis < BH;
    const int bx = min(wis, BH - 1), h = bx % H;
    float *shares = reinterpret_cast<float *>(lds + WAVES * SLOT) + u * HW * GQ * LONE_SEG;
    LoneScores<false, GQ, D, BITS> scores(lds + wave * SLOT, lane, q + (size_t)bx * GQ * D + part * 64);
    LoneLoads<D, BITS> s;
    s.start(k_cache, kp, k_new, h, bx, c, seg, T, n_super_cap, ka);
    if constexpr (BITS == 4)
        lone_fill<BLK>(lut, threadIdx.x);
    else
        lone_fill2<BLK>(lut, threadIdx.x);
    __syncthreads();

    const int t0 = s.t0, ntok = s.t1 - s.t0 + (s.last ? 1 : 0); // the appended token is the last segment's
    if (active) {
        Lone st = s.state();
        float *mine = shares + part * GQ * LONE_SEG;
        scores.ready(ka.act_bf16);
        scores.run(lut, lane_copy, st, s, s.nfull * s.UPS, mine);
        if (s.last)
            scores.finish(s, st, bx, c, T, nullptr, ka, true, mine + s.nfull * s.TPW);
        // the values' state and codes travel while the weights are made
        s.start(v_cache, vp, v_new, h, bx, c, seg, T, n_super_cap, va);
    }
    __syncthreads();

    const long row0 = (long)bx * GQ, rows = (long)BH * GQ;
    h1 *p = reinterpret_cast<h1 *>(lds + (GQ == 1 ? wave : u * HW) * SLOT);
    if (active) {
        // one query head: every wave of the unit by itself, no wave waits for another
        constexpr int EACH = GQ == 1 ? 1 : GQ / HW;
#pragma unroll
        for (int i = 0; i < EACH; i++) {
            const int g = GQ == 1 ? 0 : part * EACH + i;
            lone_weights<HW>(shares + g * LONE_SEG, GQ * LONE_SEG, logits + (row0 + g) * ka.row_pitch + t0,
                             mk.of<true>((unsigned)row0 + g, T + 1, t0), ntok, scaling, p + g * LONE_SEG, ml + (row0 + g) * ka.nseg + seg,
                             lane, GQ > 1 || part == 0);
        }
    }
    if constexpr (GQ > 1)
        __syncthreads();
    else
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); // the wave's own weights, read by its other lanes
    if (!active)
        return;

    Lone st = s.state();
    lone_step_values<D, BITS, GQ, 0>(lut, lane_copy, s, st, nullptr, 0, p, bx, c, T, lane, va, partial + (seg * rows + row0) * D + c);
}

// The same for launches of at most eight waves per CU: the values have waves of their own, which hold the first AHEAD units of a
// segment's in their registers (see small_step_kernel) while the keys' waves, the older ones, are at work, and
// multiply them by the weights when those are there.  A workgroup is WAVES waves of keys and as many of values; the SIMD has two of
// them with AHEAD = 24 and four with 16.  (Registers for all of a segment, 32 units, keep the softmax waiting for the last of
// them: 1 to 2 % slower than 24.)
template <int D, int BITS, int GQ, int WAVES, int AHEAD>
__global__ __launch_bounds__(WAVES * 128, AHEAD > 16 ? 2 : 4) void step_beside_lone_kernel(
    const h1 *q, uint4 *k_cache, const h1 *k_new, uint4 *v_cache, const h1 *v_new, Mask mk, h1 *logits, float *__restrict__ partial,
    float4 *__restrict__ ml, FtParams kp, FtParams vp, int BH, int H, int T, int n_super_cap, float scaling, Seg ka, Seg va)
{
    constexpr int HW = D / 64, UNITS = WAVES / HW;
    static_assert(WAVES % HW == 0, "whole heads");
    // key tiles, the weights, the shares.  Weights: a copy per values' wave, or, where the tiles were, those that a unit's waves write together
    constexpr int TILES = WAVES * LONE_TILE, WEIGHTS = (GQ == 1 ? WAVES : UNITS * GQ) * LONE_SEG * 2, AT = GQ == 1 ? TILES : 0;
    constexpr int SHARES = AT + WEIGHTS > TILES ? AT + WEIGHTS : TILES;
    __shared__ uint4 smem[(LUT_WORDS64 * 8 + SHARES + WAVES * GQ * LONE_SEG * 4) / 16];
    static_assert(LONE_SEG * 2 % 16 == 0, "vectors");
    ka.groups = va.groups = 0; // only even plans come here
    uint2 *lut = reinterpret_cast<uint2 *>(smem);
    char *lds = reinterpret_cast<char *>(smem) + LUT_WORDS64 * 8;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const bool values = wave >= WAVES;
    const int w = values ? wave - WAVES : wave, u = w / HW, part = w % HW, c = part * 64 + lane;
    const uint32_t lane_copy = table_lane_offset<BITS>(lane);
    int seg, wis;
    interleave_segment((int)blockIdx.x * UNITS + u, ka.nseg, seg, wis);
    const bool active = wis < BH;
    const int bx = min(wis, BH - 1), h = bx % H;
    float *shares = reinterpret_cast<float *>(lds + SHARES) + u * HW * GQ * LONE_SEG;
    h1 *rows_of_weights = reinterpret_cast<h1 *>(lds + AT);
    LoneLoads<D, BITS> s;
    s.start(values ? v_cache : k_cache, values ? vp : kp, values ? v_new : k_new, h, bx, c, seg, T, n_super_cap, values ? va : ka);
    if constexpr (BITS == 4)
        lone_fill<WAVES * 128>(lut, threadIdx.x);
    else
        lone_fill2<WAVES * 128>(lut, threadIdx.x);
    __syncthreads();

    const int t0 = s.t0, ntok = s.t1 - s.t0 + (s.last ? 1 : 0); // the appended token is the last segment's
    const long row0 = (long)bx * GQ, rows = (long)BH * GQ;
    auto weigh = [&](int g, h1 *p, bool writes) __attribute__((always_inline)) {
        lone_weights<HW>(shares + g * LONE_SEG, GQ * LONE_SEG, logits + (row0 + g) * ka.row_pitch + t0,
                         mk.of<true>((unsigned)row0 + g, T + 1, t0), ntok, scaling, p, ml + (row0 + g) * ka.nseg + seg, lane, writes);
    };
    // several query heads: a unit's waves, of both kinds, share them out
    auto weigh_mine = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < (GQ + 2 * HW - 1) / (2 * HW); i++) {
            const int g = i * 2 * HW + (values ? HW : 0) + part;
            if (active && g < GQ)
                weigh(g, rows_of_weights + (u * GQ + g) * LONE_SEG, true);
        }
    };
    Lone st = s.state();
    if (values) {
        uint32_t ahead[AHEAD * 4];
        const int done = active ? lone_values_ahead<AHEAD>(lut, lane_copy, s, st, s.nfull * s.UPS, ahead) : 0;
        __syncthreads();
        const h1 *p;
        if constexpr (GQ == 1) { // every wave by itself, no wave waits for another
            h1 *mine = rows_of_weights + w * LONE_SEG;
            if (active)
                weigh(0, mine, false);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); // the wave's own weights, read by its other lanes
            p = mine;
        } else {
            weigh_mine();
            __syncthreads();
            p = rows_of_weights + u * GQ * LONE_SEG;
        }
        if (active)
            lone_step_values<D, BITS, GQ, AHEAD>(lut, lane_copy, s, st, ahead, done, p, bx, c, T, lane, va, partial + (seg * rows + row0) * D + c);
    } else {
        if (active) {
            LoneScores<(AHEAD > 16), GQ, D, BITS> scores(lds + w * LONE_TILE, lane, q + (size_t)bx * GQ * D + part * 64);
            float *mine = shares + part * GQ * LONE_SEG;
            scores.ready(ka.act_bf16);
            scores.run(lut, lane_copy, st, s, s.nfull * s.UPS, mine);
            if (s.last)
                scores.finish(s, st, bx, c, T, nullptr, ka, true, mine + s.nfull * s.TPW);
        }
        __syncthreads();
        if constexpr (GQ == 1) {
            if (active && part == 0)
                weigh(0, reinterpret_cast<h1 *>(lds + w * LONE_TILE), true);
        } else {
            weigh_mine();
            __syncthreads();
        }
    }
}

// The segments of a row put together, by waves of two kinds: VECS x 512 of its weights each, or a share of its
// outputs: all 128 channels in two groups of segments, or, with many segments, 16 channels in 16 groups.
// Sums are taken in a fixed order.  A wave's chain of loads holds it, then the bytes.  us of this kernel, other form / this:
// a row's maxima and sums side by side (a segment's beside each other, a wave of 64 segments touches 64 lines for them):
// 1 x 8 heads x 60 000 with four query heads 8.8 / 7.4, 8 x 8 x 16 001 equal; long rows with two vectors of weights per
// lane, so that all waves are resident: 8 x 8 x 16 001 8.0 / 7.5; masks read as vectors: 64 x 32 x 663 5.5 / 5.1.
template <int VECS>
__global__ __launch_bounds__(256) void step_combine_kernel(
    const h1 *__restrict__ logits, h1 *__restrict__ weights, h1 *__restrict__ out, Mask mk,
    const float *__restrict__ partial, const float4 *__restrict__ ml, long rows, int n, long pitch, int D, int nseg,
    float scaling, int out_waves, int act_bf16)
{
    constexpr int SHARE = VECS * 512;
    const int lane = threadIdx.x & 63, weight_waves = weights ? (n + SHARE - 1) / SHARE : 0, per_row = weight_waves + out_waves;
    const long wave = (long)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const long row = wave / per_row;
    const int job = (int)(wave - row * per_row);
    if (row >= rows)
        return;
    const int t0 = job * SHARE + lane * 8;
    // the first 64 segments' maxima and sums in registers, the others read twice; a wave needs one of the sums
    const bool writes_weights = job < weight_waves;
    ml += row * nseg;
    const float4 first = lane < nseg ? ml[lane] : make_float4(-INFINITY, 0.0f, 0.0f, 0.0f);
    uint4 raw[VECS];
#pragma unroll
    for (int i = 0; i < VECS; i++) {
        raw[i] = make_uint4(0, 0, 0, 0);
        if (writes_weights && t0 + i * 512 < n) // the pitch is a multiple of 8
            raw[i] = *reinterpret_cast<const uint4 *>(logits + row * pitch + t0 + i * 512);
    }
    // What else a wave reads travels meanwhile: the mask, or its share of the first AHEAD segments' partial outputs.  (Behind the
    // reductions it was a second trip to memory: steps of 1 x 8 KV heads x 16000 tokens with four query heads 15.4 us instead of 14.4, 6 x 8 x
    // 9000 33.7 instead of 33.1; 10 x 8 x 9000 with eight (55 to 58) and 4 x 8 x 8190 of 256 channels (29.5) are the same either way.  Only
    // what is there is read: rows of three segments read four, and tokens behind the row's end, 0.4 us more for 64 x 32 x 663 with a mask.)
    constexpr int AHEAD = 4;
    const MaskRow<true> mrow = mk.of<true>((unsigned)row, n);
    float add[VECS][8] = {};
    if (mrow && writes_weights) {
#pragma unroll
        for (int i = 0; i < VECS; i++) {
            const int t = t0 + i * 512;
            if (t + 8 <= n) {
                mrow.load<8>(t, add[i]);
            } else if (t < n) {
#pragma unroll
                for (int k = 0; k < 8; k++)
                    add[i][k] = mrow.at(min(t + k, n - 1));
            }
        }
    }
    // outputs, a lane: four channels, every `groups`-th segment
    const int lanes = D / 4 / out_waves, groups = 64 / lanes;
    const int c = ((job - weight_waves) * lanes + lane % lanes) * 4;
    auto part = [&](int k) __attribute__((always_inline)) { return *reinterpret_cast<const float4 *>(partial + (k * rows + row) * D + c); };
    float4 ahead[AHEAD];
    float max_ahead[AHEAD];
    if (!writes_weights) {
#pragma unroll
        for (int i = 0; i < AHEAD; i++) {
            const int k = lane / lanes + i * groups;
            if (k < nseg) {
                ahead[i] = part(k);
                max_ahead[i] = ml[k].x;
            }
        }
    }
    float M = first.x;
    for (int k = lane + 64; k < nseg; k += 64)
        M = fmaxf(M, ml[k].x);
    M = head_reduce<64, true>(M);
    float L = lane < nseg ? (writes_weights ? first.y : first.z) * __expf(first.x - M) : 0.0f;
    for (int k = lane + 64; k < nseg; k += 64) {
        const float4 a = ml[k];
        L += (writes_weights ? a.y : a.z) * __expf(a.x - M);
    }
    const float inv = 1.0f / head_reduce<64, false>(L);
    if (writes_weights) {
#pragma unroll
        for (int i = 0; i < VECS; i++) {
            const int t = t0 + i * 512;
            if (t >= n)
                return;
            const uint32_t w[4] = {raw[i].x, raw[i].y, raw[i].z, raw[i].w};
            uint32_t o[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const h2 l = as_h2(w[k]);
                float a = (float)l.x * scaling, b = (float)l.y * scaling;
                if (mrow) {
                    a += add[i][2 * k];
                    b += add[i][2 * k + 1];
                }
                o[k] = as_u32((h2){(h1)(__expf(a - M) * inv), (h1)(__expf(b - M) * inv)});
            }
            h1 *dst = weights + row * pitch + t;
            if (t + 8 <= n) {
                *reinterpret_cast<uint4 *>(dst) = make_uint4(o[0], o[1], o[2], o[3]);
            } else {
#pragma unroll
                for (int k = 0; k < 8; k++)
                    if (t + k < n)
                        dst[k] = k & 1 ? as_h2(o[k / 2]).y : as_h2(o[k / 2]).x;
            }
        }
        return;
    }
    float4 a = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    auto add_part = [&](const float4 &p, float m) __attribute__((always_inline)) {
        const float e = __expf(m - M);
        a.x = __builtin_fmaf(p.x, e, a.x);
        a.y = __builtin_fmaf(p.y, e, a.y);
        a.z = __builtin_fmaf(p.z, e, a.z);
        a.w = __builtin_fmaf(p.w, e, a.w);
    };
#pragma unroll
    for (int i = 0; i < AHEAD; i++)
        if (lane / lanes + i * groups < nseg)
            add_part(ahead[i], max_ahead[i]);
#pragma unroll 4
    for (int k = lane / lanes + AHEAD * groups; k < nseg; k += groups)
        add_part(part(k), ml[k].x);
    for (int m = lanes; m < 64; m <<= 1) {
        a.x += __shfl_xor(a.x, m, 64);
        a.y += __shfl_xor(a.y, m, 64);
        a.z += __shfl_xor(a.z, m, 64);
        a.w += __shfl_xor(a.w, m, 64);
    }
    if (lane < lanes) {
        store_act2(out + row * D + c, a.x * inv, a.y * inv, act_bf16);
        store_act2(out + row * D + c + 2, a.z * inv, a.w * inv, act_bf16);
    }
}

} // namespace adkv
