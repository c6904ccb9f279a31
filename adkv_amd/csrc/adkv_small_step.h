// A whole decode step of a few short sequences in one launch (head dim 128, 4-bit codes, one query head
// per KV head).  Included by adkv_kernels.hip after the shared device helpers.
//
// At this size a step is the launches: forward_qk, the softmax, forward_ov and the sum of its segments
// cost the host 15 us and the device four set-ups and three gaps around two chains of at most 256
// tokens.  A workgroup of four waves takes one (sequence, head), a wave per segment: the logits, the
// weights and the partial outputs never leave the LDS, the code table is built once, and three barriers
// stand where the launches were.  More than four segments or more heads than CUs would put several
// waves on a SIMD and leave others idle: those take the separate launches, which spread better.
#pragma once

namespace adkv {

constexpr int SMALL_ROW = 3 * 64 * SM_VEC; // longest row of logits: three vectors per lane

__global__ __launch_bounds__(256) void small_step_kernel(
    const h1 *q, uint4 *__restrict__ k_cache, const h1 *k_new, uint4 *__restrict__ v_cache,
    const h1 *v_new, Mask mask, h1 *__restrict__ weights,
    h1 *__restrict__ out, FtParams kp, FtParams vp, int H, int T, int n_super_cap, float scaling, Seg ka, Seg va)
{
    constexpr int D = 128, CPL = 2;
    using G = Geo<D, CPL>;
    // the table at LDS offset 0; a tile per wave, which later holds the wave's copy of the weights; the
    // logits; the partial outputs
    __shared__ uint4 smem[(LUT_WORDS64 * 8 + 4 * PAIR_TILE + SMALL_ROW * 2 + 4 * D * 4) / 16];
    static_assert(SMALL_ROW * 2 <= PAIR_TILE, "a row of weights fits a tile");
    char *lds = reinterpret_cast<char *>(smem);
    uint2 *lut = reinterpret_cast<uint2 *>(smem);
    const int lane = threadIdx.x & 63, seg = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    char *tile = lds + LUT_WORDS64 * 8 + seg * PAIR_TILE;
    h1 *logits = reinterpret_cast<h1 *>(lds + LUT_WORDS64 * 8 + 4 * PAIR_TILE);
    float *partial = reinterpret_cast<float *>(lds + LUT_WORDS64 * 8 + 4 * PAIR_TILE + SMALL_ROW * 2);
    ka.groups = va.groups = 0;
    const int bx = blockIdx.x, h = bx % H, c0 = lane * 2, n = T + 1;
    const bool works = seg < ka.nseg;
    const uint32_t lane_copy = (uint32_t)(lane & (LUT_COPIES - 1)) * 8u;
    PairScores<4, 1, true> scores(tile, lane, q + (size_t)bx * D);
    SegLoads<D, CPL, 4, PF_PAIR> s;
    s.start(k_cache, kp.zp, kp.sc, kp.al, kp.be, kp.tg, h, bx, lane, works ? seg : 0, T, n_super_cap, ka);
    const bool last = works && s.last;
    const int t0 = s.t0, nfull = s.nfull, ntail = (s.t1 - s.t0) & 7; // only the last segment has a tail
    lut_fill<256>(lut, threadIdx.x);
    __syncthreads();

    Pair st[1];
    if (works) {
        const uint2 *cb = s.cb;
        s.state(st);
        scores.ready(ka.act_bf16);
        scores.run(lut, lane_copy, st[0], s, [&](int t, int, h1 v) __attribute__((always_inline)) { logits[t0 + t] = v; });
        if (last) {
            const h2 qv = load_act2(q + (size_t)bx * D + c0, ka.act_bf16);
            if (ntail) {
                float part[8] = {0, 0, 0, 0, 0, 0, 0, 0};
                const uint2 w = cb[(size_t)nfull * G::VPS];
                for (int tt = 0; tt < ntail; tt++) {
                    const h2 qc = extract_pair<4>(w.x, w.y, tt);
                    const h2 qs = qc * st[0].sc;
                    const float d = __builtin_amdgcn_fdot2(qv, qs + st[0].zp, 0.0f, false);
#pragma unroll
                    for (int i = 0; i < 8; i++)
                        part[i] += (i == tt) ? d : 0.0f;
                    update_pair(st[0], qc, qs);
                }
                const float s = reduce8_head<64>(part);
                const int tk = token_of_lane(lane);
                if ((lane & 3) == 0 && lane < 32 && tk < ntail)
                    logits[t0 + nfull * 8 + tk] = (h1)s;
            }
            publish_state<D, CPL>(st, nullptr, ka, bx, c0, T);
            h2 deq[1];
            append_new_token<D, CPL>(s.cbh, T, k_new + (size_t)bx * D + c0, st, deq, true, ka.act_bf16);
            const float self = head_allreduce<64>(__builtin_amdgcn_fdot2(qv, deq[0], 0.0f, false));
            if (lane == 0)
                logits[T] = (h1)self;
        }
        // the V segment's state and codes are on their way while the other waves finish
        s.start(v_cache, vp.zp, vp.sc, vp.al, vp.be, vp.tg, h, bx, lane, seg, T, n_super_cap, va);
    }
    __syncthreads();

    if (works) {
        // Every wave turns the whole row into weights, in the steps of softmax_wave_kernel: no wave waits
        // for another, and the copy it reads from is its own.
        h1 *w = reinterpret_cast<h1 *>(tile);
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
        if (seg == 0)
            softmax_store_chunk<SMALL_ROW / 512, 64>(weights + (size_t)bx * ka.row_pitch, n, 0, x, 1.0f / sum, lane);

        const uint2 *cb = s.cb;
        s.state(st);
        float acc[2] = {0.0f, 0.0f};
        if (nfull > 0) {
            auto weights_of = [&](int sg) { return *reinterpret_cast<const uint4 *>(w + t0 + sg * 8); };
            auto &buf = s.buf;
            uint2 e[2][8];
            uint4 wv[2];
            uint32_t nb[1][2];
            auto lookup = [&](uint2 *d, const uint2 *u) __attribute__((always_inline)) {
                pair_bytes_of<D, CPL>(u, nb);
#pragma unroll
                for (int t = 0; t < 8; t++)
                    d[t] = lut_get(lut, nb[0][t & 1], lane_copy, t >> 1);
            };
            lookup(e[0], buf[0]);
            wv[0] = weights_of(0);
            wait_lgkm();
            rotate_over<PF_PAIR>(nfull, [&](int sg, auto ic) __attribute__((always_inline)) {
                constexpr int i = decltype(ic)::value, half = i & 1;
                lookup(e[half ^ 1], buf[(i + 1) % PF_PAIR]); // stale past the end: looked up, never used
                wv[half ^ 1] = weights_of(min(sg + 1, nfull - 1));
                buf[i][0] = load_codes(cb + (size_t)min(sg + PF_PAIR, nfull - 1) * G::VPS);
                __builtin_amdgcn_sched_barrier(0);
                replay_eight_weighted(st[0], e[half], wv[half], acc);
                __builtin_amdgcn_sched_barrier(0);
            });
        }
        if (last) {
            auto add = [&](float wt, h2 v) {
                acc[0] = __builtin_fmaf(wt, (float)v.x, acc[0]);
                acc[1] = __builtin_fmaf(wt, (float)v.y, acc[1]);
            };
            if (ntail) {
                const uint2 u = cb[(size_t)nfull * G::VPS];
                for (int tt = 0; tt < ntail; tt++) {
                    const h2 qc = extract_pair<4>(u.x, u.y, tt);
                    const h2 qs = qc * st[0].sc;
                    add((float)w[t0 + nfull * 8 + tt], qs + st[0].zp);
                    update_pair(st[0], qc, qs);
                }
            }
            publish_state<D, CPL>(st, nullptr, va, bx, c0, T);
            h2 deq[1];
            append_new_token<D, CPL>(s.cbh, T, v_new + (size_t)bx * D + c0, st, deq, true, va.act_bf16);
            add((float)w[T], deq[0]);
        }
        reinterpret_cast<float2 *>(partial)[seg * 64 + lane] = make_float2(acc[0], acc[1]);
    }
    __syncthreads();
    if (threadIdx.x < 64) { // in segment order, as ov_finalize_kernel adds them
        float2 s = make_float2(0.0f, 0.0f);
        for (int i = 0; i < va.nseg; i++) {
            const float2 a = reinterpret_cast<const float2 *>(partial)[i * 64 + lane];
            s.x += a.x;
            s.y += a.y;
        }
        store_act2(out + (size_t)bx * D + c0, s.x, s.y, va.act_bf16);
    }
}

} // namespace adkv
