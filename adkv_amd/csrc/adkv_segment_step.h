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
// rounding, go to ml[g].  logits: the first head's row at
// the segment's first token, 16-byte aligned, its pitch a multiple of 8.
template <int LPH, int GQ>
__device__ __forceinline__ void segment_weights(const h1 *logits, long pitch, const Mask &mk, long row0, int n, int t0,
                                                int ntok, float scaling, h1 *p, float4 *ml, int lh, bool active)
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
            ml[g] = make_float4(mx, sum, rounded, 0.0f);
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
                                    ml + un.seg * rows + row0, lh, active);
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

// The segments of a row put together, by waves of two kinds: 512 of its weights each, or a share of its
// outputs: all 128 channels in two groups of segments, or, with many segments, 16 channels in 16 groups.
// Sums are taken in a fixed order.
__global__ __launch_bounds__(256) void step_combine_kernel(
    const h1 *__restrict__ logits, h1 *__restrict__ weights, h1 *__restrict__ out, Mask mk,
    const float *__restrict__ partial, const float4 *__restrict__ ml, long rows, int n, long pitch, int D, int nseg,
    float scaling, int out_waves, int act_bf16)
{
    const int lane = threadIdx.x & 63, weight_waves = weights ? (n + 511) / 512 : 0, per_row = weight_waves + out_waves;
    const long wave = (long)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const long row = wave / per_row;
    const int job = (int)(wave - row * per_row);
    if (row >= rows)
        return;
    uint4 raw = make_uint4(0, 0, 0, 0);
    const int t = job * 512 + lane * 8;
    if (job < weight_waves && t < n) // the pitch is a multiple of 8
        raw = *reinterpret_cast<const uint4 *>(logits + row * pitch + t);
    // the first 64 segments' maxima and sums in registers, the others read twice; a wave needs one of the sums
    const bool writes_weights = job < weight_waves;
    const float4 first = lane < nseg ? ml[lane * rows + row] : make_float4(-INFINITY, 0.0f, 0.0f, 0.0f);
    float M = first.x;
    for (int k = lane + 64; k < nseg; k += 64)
        M = fmaxf(M, ml[k * rows + row].x);
    M = head_reduce<64, true>(M);
    float L = lane < nseg ? (writes_weights ? first.y : first.z) * __expf(first.x - M) : 0.0f;
    for (int k = lane + 64; k < nseg; k += 64) {
        const float4 a = ml[k * rows + row];
        L += (writes_weights ? a.y : a.z) * __expf(a.x - M);
    }
    const float inv = 1.0f / head_reduce<64, false>(L);
    if (writes_weights) {
        if (t >= n)
            return;
        const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
        const MaskRow<true> mrow = mk.of<true>((unsigned)row, n);
        uint32_t o[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const h2 l = as_h2(w[k]);
            float a = (float)l.x * scaling, b = (float)l.y * scaling;
            if (mrow) {
                a += mrow.at(min(t + 2 * k, n - 1));
                b += mrow.at(min(t + 2 * k + 1, n - 1));
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
        return;
    }
    // a lane: four channels, every `groups`-th segment
    const int lanes = D / 4 / out_waves, groups = 64 / lanes;
    const int c = ((job - weight_waves) * lanes + lane % lanes) * 4;
    float4 a = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (int k = lane / lanes; k < nseg; k += groups) {
        const float4 p = *reinterpret_cast<const float4 *>(partial + (k * rows + row) * D + c);
        const float e = __expf(ml[k * rows + row].x - M);
        a.x = __builtin_fmaf(p.x, e, a.x);
        a.y = __builtin_fmaf(p.y, e, a.y);
        a.z = __builtin_fmaf(p.z, e, a.z);
        a.w = __builtin_fmaf(p.w, e, a.w);
    }
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
