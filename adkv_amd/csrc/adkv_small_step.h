// A whole decode step of a few short sequences in one launch (head dim 128, 4-bit codes, one query head
// per KV head).  Included by adkv_kernels.hip after the shared device helpers.
//
// At this size a step is the launches: forward_qk, the softmax, forward_ov and the sum of its segments
// cost the host 15 us and the device four set-ups and three gaps around two chains of at most 256
// tokens.  A workgroup of eight waves takes one (sequence, head), two waves per segment (adkv_lone.h): the logits, the
// weights and the partial outputs never leave the LDS, the code table is built once, and a few barriers
// stand where the launches were (a wave per segment and two channels per lane: 1 x 32 heads x 603 tokens 18.9 us, two
// waves 13.2; 4 x 32 x 200 16.9 / 12.8, 8 x 32 x 1000, with four full segments, 21.0 / 20.0).  More than four segments or more heads than CUs would put more
// waves on a SIMD and leave others idle: those take the separate launches, which spread better.
#pragma once

namespace adkv {

constexpr int SMALL_ROW = 3 * 64 * SM_VEC; // longest row of logits: three vectors per lane

__global__ __launch_bounds__(512) void small_step_kernel(
    const h1 *q, uint4 *k_cache, const h1 *k_new, uint4 *v_cache, const h1 *v_new, Mask mask, h1 *__restrict__ weights,
    h1 *__restrict__ out, FtParams kp, FtParams vp, int H, int T, int n_super_cap, float scaling, Seg ka, Seg va)
{
    constexpr int D = 128, WAVE = SMALL_ROW * 2;
    static_assert(LONE_TILE <= WAVE, "a key tile fits where the weights will be");
    // the table at LDS offset 0; per wave a key tile, then its copy of the weights; both halves' shares of the
    // logits; the logits; the partial outputs
    __shared__ uint4 smem[(LUT_WORDS64 * 8 + 8 * WAVE + 2 * SMALL_ROW * 4 + SMALL_ROW * 2 + 4 * D * 4) / 16];
    char *lds = reinterpret_cast<char *>(smem);
    uint2 *lut = reinterpret_cast<uint2 *>(smem);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int seg = wave >> 1, half = wave & 1, c = half * 64 + lane;
    char *mine = lds + LUT_WORDS64 * 8 + wave * WAVE;
    float *share = reinterpret_cast<float *>(lds + LUT_WORDS64 * 8 + 8 * WAVE);
    h1 *logits = reinterpret_cast<h1 *>(share + 2 * SMALL_ROW);
    float *partial = reinterpret_cast<float *>(logits + SMALL_ROW);
    ka.groups = va.groups = 0;
    const int bx = blockIdx.x, h = bx % H, n = T + 1;
    const bool works = seg < ka.nseg;
    const uint32_t lane_copy = (uint32_t)(lane & (LUT_COPIES - 1)) * 8u;
    LoneScores<true> scores(mine, lane, q + (size_t)bx * D + half * 64);
    LoneLoads<> s;
    s.start(k_cache, kp, k_new, h, bx, c, works ? seg : 0, T, n_super_cap, ka);
    lone_fill<512>(lut, threadIdx.x);
    __syncthreads();

    if (works) {
        Lone st = s.state();
        float *part = share + half * SMALL_ROW + s.t0;
        scores.ready(ka.act_bf16);
        scores.run(lut, lane_copy, st, s, s.nfull, part);
        if (s.last)
            scores.finish(s, st, bx, c, T, nullptr, ka, true, part + s.nfull * 8);
        // the V segment's state and codes are on their way while the other waves finish
        s.start(v_cache, vp, v_new, h, bx, c, seg, T, n_super_cap, va);
    }
    __syncthreads();
    for (int t = threadIdx.x; t < n; t += 512)
        logits[t] = (h1)(share[t] + share[SMALL_ROW + t]);
    __syncthreads();

    if (works) {
        // Every wave turns the whole row into weights, in the steps of softmax_wave_kernel: no wave waits
        // for another, and the copy it reads from is its own.
        h1 *w = reinterpret_cast<h1 *>(mine);
        float x[SMALL_ROW / 64], mx;
        softmax_load_chunk<SMALL_ROW / 512, 64>(logits, mask.of<true>(bx, n), n, 0,
                                                scaling, x, mx, lane);
#pragma unroll
        for (int m = 1; m < 64; m <<= 1)
            mx = fmaxf(mx, __shfl_xor(mx, m, 64));
        float sum = 0.0f;
#pragma unroll
        for (int i = 0; i < SMALL_ROW / 64; i++) {
            x[i] = __expf(x[i] - mx);
            sum += x[i];
        }
#pragma unroll
        for (int m = 1; m < 64; m <<= 1)
            sum += __shfl_xor(sum, m, 64);
        softmax_store_chunk<SMALL_ROW / 512, 64>(w, n, 0, x, 1.0f / sum, lane);
        if (wave == 0)
            softmax_store_chunk<SMALL_ROW / 512, 64>(weights + (size_t)bx * ka.row_pitch, n, 0, x, 1.0f / sum, lane);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); // w is read by the wave's other lanes

        const h1 *wb = w + s.t0;
        Lone st = s.state();
        float acc = 0.0f;
        lone_values(lut, lane_copy, s, st, s.nfull, wb, acc);
        lone_values_end(s, st, [&](int t) { return wb[t]; }, bx, c, T, nullptr, va, true, acc);
        partial[seg * D + c] = acc;
    }
    __syncthreads();
    if (threadIdx.x < 64) { // in segment order, as ov_finalize_kernel adds them
        float2 s = make_float2(0.0f, 0.0f);
        for (int i = 0; i < va.nseg; i++) {
            const float2 a = reinterpret_cast<const float2 *>(partial)[i * 64 + lane];
            s.x += a.x;
            s.y += a.y;
        }
        store_act2(out + (size_t)bx * D + lane * 2, s.x, s.y, va.act_bf16);
    }
}

} // namespace adkv
