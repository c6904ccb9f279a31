// A whole decode step of a few short sequences in one launch (head dim 128, 4-bit codes, one query head
// per KV head).  Included by adkv_kernels.hip after the shared device helpers.
//
// At this size a step is the launches: forward_qk, the softmax, forward_ov and the sum of its segments
// cost the host 15 us and the device four set-ups and three gaps around two chains of at most 256
// tokens.  A workgroup takes one (sequence, head), four waves per segment: two (adkv_lone.h) for its keys and two for its
// values.  The logits, the weights and the partial outputs never leave the LDS, the code table is built once, and a
// few barriers stand where the launches were.
// The two chains need nothing of each other but the weights.  The values' waves replay their segment's first tokens, as many
// as their registers hold, while the keys' waves are at theirs, whose issue slots they do not miss: a wave alone on its SIMD
// uses half of them, and the older one goes first.  Behind the softmax those tokens cost one multiply-add each.  us per step,
// a wave's keys and values one behind the other / side by side / with the softmax straight from the shares and its reductions in
// registers, sequences x heads x tokens: 1 x 32 x 603 13.5 / 11.9 / 11.0, 4 x 32 x 200 13.2 / 11.0, 1 x 32 x 200 12.9 / 10.7 / 9.5,
// 1 x 32 x 500 14.4 / 12.8 / 11.4, 5 x 40 x 700 17.5 / 14.5, 8 x 32 x 1000 18.9 / 17.3 / 16.3.  More than four
// segments or more heads than CUs would put more waves on a SIMD and leave others idle: those take the separate launches,
// which spread better.
#pragma once

namespace adkv {

constexpr int SMALL_ROW = 3 * 64 * SM_VEC; // longest row of logits: three vectors per lane

// Units of eight tokens that a values' wave holds: four registers each, of 256 / 168 / 128 with two / three / four waves per SIMD.
// (With three segments 24 units fit as well, and keep the keys waiting where the last segment is a part of one: 1 x 32 x 603 11.0 us, with 16
// 10.7, 4 x 32 x 650 11.7 / 11.5.  Three whole ones gain from them, 2 x 8 x 768 12.7 / 13.6; 8 x 32 x 700 13.5 / 13.6, 5 x 40 x 700 12.8 / 13.0,
// 1 x 32 x 520 10.5 / 10.7.)
template <int SEGS> constexpr int small_ahead() { return SEGS == 1 ? 32 : SEGS == 2 ? 24 : SEGS == 3 ? 16 : 8; }

template <int SEGS>
__global__ __launch_bounds__(SEGS * 256) void small_step_kernel(
    const h1 *q, uint4 *k_cache, const h1 *k_new, uint4 *v_cache, const h1 *v_new, Mask mask, h1 *__restrict__ weights,
    h1 *__restrict__ out, FtParams kp, FtParams vp, int H, int T, int n_super_cap, float scaling, Seg ka, Seg va)
{
    constexpr int D = 128, HALF = 2 * SEGS, AHEAD = small_ahead<SEGS>();
    // the table at LDS offset 0; a key tile per keys' wave; both halves' shares of the logits; the weights (and what is read
    // behind them, never used); the partial outputs
    __shared__ uint4 smem[(LUT_WORDS64 * 8 + HALF * LONE_TILE + 2 * SMALL_ROW * 4 + SMALL_ROW * 2 + SEGS * D * 4) / 16];
    char *lds = reinterpret_cast<char *>(smem);
    uint2 *lut = reinterpret_cast<uint2 *>(smem);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const bool values = wave >= HALF;
    const int w2 = values ? wave - HALF : wave, seg = w2 >> 1, half = w2 & 1, c = half * 64 + lane;
    float *share = reinterpret_cast<float *>(lds + LUT_WORDS64 * 8 + HALF * LONE_TILE);
    h1 *w = reinterpret_cast<h1 *>(share + 2 * SMALL_ROW);
    float *partial = reinterpret_cast<float *>(w + SMALL_ROW);
    ka.groups = va.groups = 0;
    const int bx = blockIdx.x, h = bx % H, n = T + 1;
    const uint32_t lane_copy = (uint32_t)(lane & (LUT_COPIES - 1)) * 8u;
    LoneLoads<> s;
    s.start(values ? v_cache : k_cache, values ? vp : kp, values ? v_new : k_new, h, bx, c, seg, T, n_super_cap, values ? va : ka);
    lone_fill<SEGS * 256>(lut, threadIdx.x);
    __syncthreads();

    Lone st = s.state();
    if (values) { // the two kinds of waves meet at the same barriers, and share no registers across them
        uint32_t ahead[AHEAD * 4];
        const int done = lone_values_ahead<AHEAD>(lut, lane_copy, s, st, s.nfull, ahead);
        __syncthreads();
        __syncthreads();
        const h1 *wb = w + s.t0;
        float acc = 0.0f;
        lone_weigh<AHEAD>(ahead, done, wb, acc);
        lone_values(lut, lane_copy, s, st, s.nfull - done, wb + done * 8, acc);
        lone_values_end(s, st, [&](int t) { return wb[t]; }, bx, c, T, nullptr, va, true, acc);
        partial[seg * D + c] = acc;
    } else {
        LoneScores<(SEGS <= 2)> scores(lds + LUT_WORDS64 * 8 + w2 * LONE_TILE, lane, q + (size_t)bx * D + half * 64);
        float *part = share + half * SMALL_ROW + s.t0;
        scores.ready(ka.act_bf16);
        scores.run(lut, lane_copy, st, s, s.nfull, part);
        if (s.last)
            scores.finish(s, st, bx, c, T, nullptr, ka, true, part + s.nfull * 8);
        __syncthreads();
        if (wave == 0) { // the row's logits into weights, in the steps of softmax_wave_kernel
            constexpr int V = SMALL_ROW / 512;
            const MaskRow<true> mrow = mask.of<true>(bx, n);
            float x[V * SM_VEC], mx = -INFINITY;
#pragma unroll
            for (int v = 0; v < V; v++) {
                const int i0 = (v * 64 + lane) * SM_VEC;
                float add[SM_VEC] = {};
                if (mrow && i0 < n) {
                    if (i0 + SM_VEC <= n)
                        mrow.load<SM_VEC>(i0, add);
                    else
#pragma unroll
                        for (int k = 0; k < SM_VEC; k++)
                            add[k] = mrow.at(min(i0 + k, n - 1));
                }
#pragma unroll
                for (int k = 0; k < SM_VEC; k += 4) {
                    const float4 a = *reinterpret_cast<const float4 *>(share + i0 + k), b = *reinterpret_cast<const float4 *>(share + SMALL_ROW + i0 + k);
                    const float l[4] = {a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w};
#pragma unroll
                    for (int m = 0; m < 4; m++) {
                        float &e = x[v * SM_VEC + k + m];
                        e = (float)(h1)l[m] * scaling;
                        if (mrow)
                            e += add[k + m];
                        e = i0 + k + m < n ? e : -INFINITY;
                        mx = fmaxf(mx, e);
                    }
                }
            }
            mx = wave_reduce<true>(mx);
            float sum = 0.0f;
#pragma unroll
            for (int i = 0; i < SMALL_ROW / 64; i++) {
                x[i] = __expf(x[i] - mx);
                sum += x[i];
            }
            sum = wave_reduce<false>(sum);
            softmax_store_chunk<SMALL_ROW / 512, 64>(w, n, 0, x, 1.0f / sum, lane);
            softmax_store_chunk<SMALL_ROW / 512, 64>(weights + (size_t)bx * ka.row_pitch, n, 0, x, 1.0f / sum, lane);
        }
        __syncthreads();
    }
    __syncthreads();
    if (threadIdx.x < 64) { // in segment order, as ov_finalize_kernel adds them
        float2 s = make_float2(0.0f, 0.0f);
        for (int i = 0; i < SEGS; i++) {
            const float2 a = reinterpret_cast<const float2 *>(partial)[i * 64 + lane];
            s.x += a.x;
            s.y += a.y;
        }
        store_act2(out + (size_t)bx * D + lane * 2, s.x, s.y, va.act_bf16);
    }
}

} // namespace adkv
