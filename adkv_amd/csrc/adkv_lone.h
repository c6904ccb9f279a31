// forward_qk and forward_ov of launches that leave SIMDs empty: head dim 128, 4-bit codes, one query head per KV
// head, one channel per lane, a head over two waves; and their parts for steps of any head dim D, a head over D / 64
// waves, with GQ query heads (adkv_segment_step.h).  Included by adkv_kernels.hip after the shared device helpers.
//
// Such a launch takes as long as one wave's instructions per token: a wave alone on its SIMD issues one every four
// or five cycles, LDS reads twelve, whatever the other lanes do.  With two channels per lane that is a lookup and
// five packed instructions per token, nine with the outputs'; with one (lone_eight) half a lookup and three,
// four with them, and twice the waves.
#pragma once

namespace adkv {

constexpr int LONE_PF = 8;          // units of eight tokens whose codes are in flight
constexpr int LONE_TILE = 64 * 32;  // bytes of a wave's key tile: 64 channels x 16 tokens
constexpr int LONE_SEG = 264;       // tokens of a segment of a step, and one vector behind them
constexpr int LONE_CHUNK = 512;     // tokens between two exchanges of partial logits

// Wave w of the launch is half w % 2 of unit w / 2; units are ordered like the waves of a head per wave.
struct LoneUnit {
    int bx, seg, half, c;
    bool active;
    __device__ __forceinline__ LoneUnit(int BH, int nseg, int wave)
    {
        int wis;
        interleave_segment(wave >> 1, nseg, seg, wis);
        half = wave & 1;
        c = half * 64 + (int)(threadIdx.x & 63);
        active = wis < BH;
        bx = min(wis, BH - 1);
    }
};

// See SegLoads; also the word that the appended token goes to and the token itself.
template <int D = 128, int BITS = 4>
struct LoneLoads {
    static constexpr int TPW = Code<BITS>::TPW, UPS = TPW / 8, PF = LONE_PF / UPS; // units, words of codes in flight
    static constexpr int SHIFT = BITS == 4 ? 3 : 4;                                // of tokens to words
    uint32_t *cbh;      // this head, this channel
    // this segment's whole supergroups.  Reads past them are dropped: a load's whole position is in its vector offset, which
    // is what the range check looks at (of the scalar offset the check is not documented to take account).  The offset
    // moves on once for PF loads, whose places behind it are in the instructions (with an addition per load a step of
    // 1 x 32 heads x 603 tokens took 15.8 us instead of 15.4; with a clamped index it was five instructions a load)
    __amdgpu_buffer_rsrc_t codes;
    int next; // where in it this lane's next PF words are
    int t0, t1, nfull, ntail;
    bool last, from_ckpt;
    h1 zp, sc, al, be, tg;
    uint32_t ck, tail, buf[PF];
    uint16_t fresh;

    __device__ __forceinline__ void start(void *cache, const FtParams &p, const h1 *x_new, int h, int bx, int c, int seg, int T,
                                          int n_super_cap, const Seg &sa)
    {
        const int iv = seg_first_interval(sa, seg), pi = h * D + c;
        last = seg_is_last(sa, seg);
        t0 = iv * sa.ckpt_interval;
        t1 = last ? T : seg_end(sa, seg);
        nfull = (t1 - t0) >> SHIFT;
        ntail = (t1 - t0) & (TPW - 1); // of the last segment only: the others are whole intervals
        cbh = reinterpret_cast<uint32_t *>(cache) + (size_t)bx * n_super_cap * D + c;
        codes = __builtin_amdgcn_make_buffer_rsrc(cbh - c + (size_t)(t0 >> SHIFT) * D, 0, nfull * D * 4, 0x00027000);
        next = c * 4;
        from_ckpt = iv > 0;
        ck = 0;
        if (from_ckpt)
            ck = *reinterpret_cast<const uint32_t *>(sa.ckpt + (((size_t)bx * sa.n_ckpt_cap + iv - 1) * D + c) * 2);
        zp = p.zp[pi];
        sc = p.sc[pi];
        al = p.al[pi];
        be = p.be[pi];
        tg = p.tg[pi];
#pragma unroll
        for (int i = 0; i < PF; i++)
            buf[i] = load(i);
        move_on();
        tail = cbh[(size_t)(last ? T >> SHIFT : 0) * D];
        fresh = reinterpret_cast<const uint16_t *>(x_new)[(size_t)bx * D + c];
    }
    // the i-th of the next PF words; read once: not kept in the caches
    __device__ __forceinline__ uint32_t load(int i) const
    {
        return __builtin_amdgcn_raw_buffer_load_b32(codes, next + i * D * 4, 0, 2);
    }
    // behind unit i of LONE_PF: the word that it was the last of, PF words further
    __device__ __forceinline__ void refill(int i)
    {
        if (i % UPS == UPS - 1)
            buf[i / UPS] = load(i / UPS);
        if (i == LONE_PF - 1)
            move_on();
    }
    // hidden from the loop's optimiser, which would count from the last of the places, and add for each of the others
    __device__ __forceinline__ void move_on()
    {
        next += PF * D * 4;
        asm("" : "+v"(next));
    }
    __device__ __forceinline__ int code(int t) const { return (int)(tail >> (BITS * t) & Code<BITS>::FIELD) + Code<BITS>::QLO; }
    __device__ __forceinline__ Lone state() const
    {
        const h2 s = from_ckpt ? as_h2(ck) : (h2){zp, sc};
        const h1 one = (h1)1.0f, bt = be * tg; // omt = 1 - beta*target, both steps rounded (gemv.cu:220-221)
        Lone r;
        r.z = as_u32((h2){s.x, (h1)0.0f});
        r.r = as_u32((h2){(h1)0.0f, s.y});
        r.ca = as_u32((h2){al, one});
        r.cf = as_u32((h2){one, be});
        r.c0 = as_u32((h2){(h1)0.0f, one - bt});
        return r;
    }
};

// The entries of unit i of the words in flight, two tokens each; with 2-bit codes a byte of a word is four tokens and
// an LDS read returns two entries.
template <int BITS>
__device__ __forceinline__ void lone_lookup(uint2 *e, const uint2 *lut, const uint32_t *buf, int i, uint32_t lane_copy)
{
    if constexpr (BITS == 4) {
#pragma unroll
        for (int k = 0; k < 4; k++)
            e[k] = lut_get(lut, buf[i], lane_copy, k);
    } else {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const uint4 v = lut2_get(lut, buf[i / 2], lane_copy, i % 2 * 2 + k);
            e[2 * k] = make_uint2(v.x, v.y);
            e[2 * k + 1] = make_uint2(v.z, v.w);
        }
    }
}
// The table for them (see lone_fill for 4 bits): 16 copies of 16-byte entries.
template <int NT>
__device__ __forceinline__ void lone_fill2(uint2 *lut, int tid)
{
    uint4 *l4 = reinterpret_cast<uint4 *>(lut);
#pragma unroll
    for (int i = 0; i < LUT_ENTRIES * LUT2_COPIES; i += NT) {
        if (LUT_ENTRIES * LUT2_COPIES % NT != 0 && i + tid >= LUT_ENTRIES * LUT2_COPIES)
            break;
        const int b = (i + tid) / LUT2_COPIES;
        const auto entry = [](int code) { return as_u32(splat((h1)(code - 2))) & 0x7FFFFFFFu; };
        l4[i + tid] = make_uint4(entry(b & 3), entry(b >> 2 & 3), entry(b >> 4 & 3), entry(b >> 6));
    }
}

// The last segment's end: hands out the state after token T - 1, records it where token T opens an interval,
// quantises token T into its word (gemv.cu:744-798, 1105-1157) and returns its value r16(q*sc + zp).
template <int D, int BITS>
__device__ __forceinline__ h1 lone_append(const LoneLoads<D, BITS> &s, const Lone &st, int bx, int c, int T, h1 *state_out, const Seg &sa,
                                          bool active)
{
    const uint32_t zs = as_u32((h2){lone_zp(st), lone_sc(st)});
    if (active && state_out != nullptr)
        *reinterpret_cast<uint32_t *>(state_out + ((size_t)bx * D + c) * 2) = zs;
    if (active && sa.ckpt != nullptr && T > 0 && T % sa.ckpt_interval == 0) {
        const int j = T / sa.ckpt_interval - 1;
        if (j < sa.n_ckpt_cap)
            *reinterpret_cast<uint32_t *>(sa.ckpt + (((size_t)bx * sa.n_ckpt_cap + j) * D + c) * 2) = zs;
    }
    const h1 x = act2(s.fresh, sa.act_bf16).x;
    const int q = quantize<BITS>(x, lone_zp(st), lone_sc(st));
    const int sh = BITS * s.ntail;
    if (active)
        s.cbh[(size_t)(T >> s.SHIFT) * D] = (s.tail & ~(Code<BITS>::FIELD << sh)) | ((uint32_t)(q - Code<BITS>::QLO) << sh);
    return __builtin_fmaf16((h1)q, lone_sc(st), lone_zp(st));
}

// forward_qk of a wave's 64 channels.  The values of 16 tokens go to an LDS tile, 32 bytes per channel, from
// which transposing reads hand every lane eight channels of its token as a column for the matrix cores; all rows are
// the query.  Columns of four tiles are put side by side, a lane per token, and written as the half's share of
// the logits (fp32); the two halves of a head are added by who reads them.
// ACC: at most eight waves to a workgroup; the compiler then keeps products in accumulation registers.
// GQ: query heads per KV head.  Row r of the product is head r * GQ / 16, so that a lane has the share of its token and of the
// head of its quarter (of two heads with eight): a store per tile where a single head's columns are collected first.
// The tile's 16-byte pieces change places with every fourth channel, so that eight lanes' writes spread over the banks.
template <bool ACC, int GQ = 1, int D = 128, int BITS = 4>
struct LoneScores {
    char *tile;
    int lane, wr[2], rd[2];
    h8v qa[2], kv[2];
    f4v d;
    float hold;

    // loads the queries (rows are 8-byte aligned); ready() once the rest of the workgroup's loads are out
    __device__ __forceinline__ LoneScores(char *tile_, int lane_, const h1 *q) : tile(tile_), lane(lane_)
    {
#pragma unroll
        for (int m = 0; m < 2; m++) {
            const uint2 *src = reinterpret_cast<const uint2 *>(q + ((lane & 15) * GQ >> 4) * D + m * 32 + (lane >> 4) * 8);
            const uint2 a = src[0], b = src[1];
            qa[m] = __builtin_bit_cast(h8v, make_uint4(a.x, a.y, b.x, b.y));
        }
    }
    __device__ __forceinline__ void ready(int act_bf16)
    {
#pragma unroll
        for (int m = 0; m < 2; m++) {
            if (act_bf16) {
                const uint4 u = __builtin_bit_cast(uint4, qa[m]);
                qa[m] = __builtin_bit_cast(h8v, make_uint4(as_u32(act2(u.x, 1)), as_u32(act2(u.y, 1)),
                                                           as_u32(act2(u.z, 1)), as_u32(act2(u.w, 1))));
            }
            kv[m] = (h8v){};
            wr[m] = lane * 32 + ((m ^ (lane >> 2 & 1)) << 4);
            // rows 4 * m.. of a quarter's eight channels; lane i of 16 reads row i / 4, tokens 4 * (i % 4)..
            rd[m] = ((lane >> 4) * 8 + m * 4 + (lane >> 2 & 3)) * 32 + (((lane >> 1 & 1) ^ m) << 4) + (lane & 1) * 8;
        }
        d = (f4v){0.0f, 0.0f, 0.0f, 0.0f};
        hold = 0.0f;
    }
    __device__ __forceinline__ void write(int half, const uint32_t *x)
    {
        *reinterpret_cast<uint4 *>(tile + wr[half]) = make_uint4(x[0], x[1], x[2], x[3]);
    }
    __device__ __forceinline__ void fetch()
    {
        typedef short s4v __attribute__((ext_vector_type(4)));
        typedef __attribute__((address_space(3))) s4v *Lds;
        const auto base = (__attribute__((address_space(3))) char *)tile;
#pragma unroll
        for (int m = 0; m < 2; m++) {
            const s4v a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((Lds)(base + m * 1024 + rd[0]));
            const s4v b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((Lds)(base + m * 1024 + rd[1]));
            const uint2 x = __builtin_bit_cast(uint2, a), y = __builtin_bit_cast(uint2, b);
            kv[m] = __builtin_bit_cast(h8v, make_uint4(x.x, x.y, y.x, y.y));
        }
    }
    __device__ __forceinline__ void multiply()
    {
        d = (f4v){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int m = 0; m < 2; m++)
            d = __builtin_amdgcn_mfma_f32_16x16x32_f16(qa[m], kv[m], d, 0, 0, 0);
    }
    // the column of the u-th tile of four goes to the lanes of quarter u
    __device__ __forceinline__ void keep(int u)
    {
        if constexpr (ACC) // all of d is held up to here: see PairScores::emit
            asm volatile("" ::"a"(d));
        else
            asm volatile("" ::"v"(d));
        hold = (lane >> 4) == u ? d.x : hold;
    }

    // several query heads: the first ntok tokens of a tile, a row of LONE_SEG per head
    __device__ __forceinline__ void put(float *part, int ntok)
    {
        if constexpr (ACC)
            asm volatile("" ::"a"(d));
        else
            asm volatile("" ::"v"(d));
        const int t = lane & 15, quarter = lane >> 4;
        if (t < ntok) {
            part[(GQ == 8 ? 2 * quarter : quarter * GQ >> 2) * LONE_SEG + t] = d.x;
            if constexpr (GQ == 8)
                part[(2 * quarter + 1) * LONE_SEG + t] = d.z;
        }
    }

    // the segment's next n units, of all calls but the last a multiple of LONE_PF; the shares of their logits to part[0..8n)
    __device__ __forceinline__ void run(const uint2 *lut, uint32_t lane_copy, Lone &st, LoneLoads<D, BITS> &s, int n, float *part)
    {
        if (n <= 0)
            return;
        uint2 e[2][4];
        lone_lookup<BITS>(e[0], lut, s.buf, 0, lane_copy);
        wait_lgkm();
        // tile i / 2 of a group of eight supergroups is written after its two, fetched with the second, multiplied
        // half a tile later and kept another half later
        auto body = [&](int sg, auto ic, auto &&group_done) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value;
            lone_lookup<BITS>(e[(i & 1) ^ 1], lut, s.buf, (i + 1) % LONE_PF, lane_copy); // stale past the end: looked up, never used
            s.refill(i);
            __builtin_amdgcn_sched_barrier(0);
            uint32_t x[4];
            lone_eight(st, e[i & 1], x);
            write(i & 1, x);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (i & 1) {
                if constexpr (GQ > 1) {
                    put(part + max(sg - 3, 0) * 8, 16); // at the first what is stored is overwritten
                } else {
                    keep((i / 2 + 3) & 3);
                    if constexpr (i == 1)
                        group_done();
                }
                fetch();
            } else {
                multiply();
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        int g0 = 0;
        for (; g0 + LONE_PF <= n; g0 += LONE_PF)
            static_for<LONE_PF>([&](auto ic) __attribute__((always_inline)) {
                // the group before this one; at the first what is stored is overwritten by the second's or the end's
                body(g0 + decltype(ic)::value, ic, [&]() __attribute__((always_inline)) { part[max(g0 - LONE_PF, 0) * 8 + lane] = hold; });
            });
        static_for<LONE_PF - 1>([&](auto ic) __attribute__((always_inline)) {
            if (g0 + decltype(ic)::value < n)
                body(g0 + decltype(ic)::value, ic, [&]() __attribute__((always_inline)) {
                    if (g0 > 0)
                        part[(g0 - LONE_PF) * 8 + lane] = hold;
                });
        });
        const int end = n - 1, base = (end & ~7) * 8;
        if constexpr (GQ > 1) {
            if (!(end & 1)) {
                if (end > 0)
                    put(part + (end - 2) * 8, 16);
                fetch();
            }
            multiply();
            put(part + (end & ~1) * 8, end & 1 ? 16 : 8);
            return;
        }
        if (end & 1) {
            multiply();
        } else { // half a tile, and the one before it is still to be kept
            keep((end / 2 + 3) & 3);
            if ((end & 7) == 0 && end > 0)
                part[base - 64 + lane] = hold;
            fetch();
            multiply();
        }
        keep((end / 2) & 3);
        if (lane < 8 * n - base)
            part[base + lane] = hold;
    }
    // up to eight tokens by themselves, sixteen with 2-bit codes
    __device__ __forceinline__ void few(const uint32_t *x, int ntok, float *part)
    {
        write(0, x);
        if constexpr (BITS == 2)
            write(1, x + 4);
        fetch();
        multiply();
        if constexpr (GQ > 1) {
            put(part, ntok);
            return;
        }
        keep(0);
        if (lane < ntok)
            part[lane] = hold;
    }
    // the last segment's ragged tail and the appended token; their shares of the logits to part[0..ntail]
    __device__ __forceinline__ void finish(const LoneLoads<D, BITS> &s, Lone &st, int bx, int c, int T, h1 *state_out, const Seg &sa, bool active,
                                           float *part)
    {
        constexpr int TPW = Code<BITS>::TPW;
        uint32_t v[TPW] = {}, x[TPW / 2];
#pragma unroll
        for (int t = 0; t < TPW - 1; t++)
            if (t < s.ntail)
                v[t] = __builtin_bit_cast(uint16_t, lone_token(st, s.code(t)));
        const uint32_t self = __builtin_bit_cast(uint16_t, lone_append(s, st, bx, c, T, state_out, sa, active));
#pragma unroll
        for (int t = 0; t < TPW; t++)
            v[t] = t == s.ntail ? self : v[t];
#pragma unroll
        for (int k = 0; k < TPW / 2; k++)
            x[k] = v[2 * k] | v[2 * k + 1] << 16;
        few(x, s.ntail + 1, part);
    }
};

// forward_ov of a wave's 64 channels: adds the segment's next n units to acc, of all calls but the last a multiple of
// LONE_PF.  w: their weights, in LDS.
template <int D, int BITS>
__device__ __forceinline__ void lone_values(const uint2 *lut, uint32_t lane_copy, LoneLoads<D, BITS> &s, Lone &st, int n, const h1 *w,
                                            float &acc)
{
    if (n <= 0)
        return;
    const uint4 *w4 = reinterpret_cast<const uint4 *>(w);
    uint2 e[2][4];
    uint4 wv[2];
    lone_lookup<BITS>(e[0], lut, s.buf, 0, lane_copy);
    wv[0] = w4[0];
    wait_lgkm();
    rotate_over<LONE_PF>(n, [&](int sg, auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value, half = i & 1;
        lone_lookup<BITS>(e[half ^ 1], lut, s.buf, (i + 1) % LONE_PF, lane_copy); // stale past the end: looked up, never used
        wv[half ^ 1] = w4[sg + 1]; // so are these: the caller's LDS goes on behind them
        s.refill(i);
        __builtin_amdgcn_sched_barrier(0);
        lone_eight_weighted(st, e[half], wv[half], acc);
        __builtin_amdgcn_sched_barrier(0);
    });
}
// The values of a segment's first tokens before their weights are there: whole groups of LONE_PF units, at most UNITS; x[4u..]
// are unit u's.  Returns the units done, with which lone_values goes on.
template <int UNITS, int D, int BITS>
__device__ __forceinline__ int lone_values_ahead(const uint2 *lut, uint32_t lane_copy, LoneLoads<D, BITS> &s, Lone &st, int n, uint32_t *x)
{
    static_assert(UNITS % LONE_PF == 0, "whole groups");
    uint2 e[2][4];
    lone_lookup<BITS>(e[0], lut, s.buf, 0, lane_copy);
    wait_lgkm();
#pragma unroll
    for (int g = 0; g < UNITS; g += LONE_PF)
        if (g + LONE_PF <= n)
            static_for<LONE_PF>([&](auto ic) __attribute__((always_inline)) {
                constexpr int i = decltype(ic)::value, half = i & 1;
                lone_lookup<BITS>(e[half ^ 1], lut, s.buf, (i + 1) % LONE_PF, lane_copy); // stale past the end: looked up, never used
                s.refill(i);
                __builtin_amdgcn_sched_barrier(0);
                lone_eight(st, e[half], x + (g + i) * 4);
                __builtin_amdgcn_sched_barrier(0);
            });
    return min(UNITS, n & ~(LONE_PF - 1));
}
// Those values by their weights, in the order of lone_values.  done: what lone_values_ahead returned.
template <int UNITS>
__device__ __forceinline__ void lone_weigh(const uint32_t *x, int done, const h1 *w, float &acc)
{
    const uint4 *w4 = reinterpret_cast<const uint4 *>(w);
#pragma unroll
    for (int g = 0; g < UNITS; g += LONE_PF)
        if (g < done) {
#pragma unroll
            for (int u = g; u < g + LONE_PF; u++) {
                const uint4 wv = w4[u];
                const uint32_t ww[4] = {wv.x, wv.y, wv.z, wv.w};
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    acc = __builtin_fmaf((float)as_h2(ww[k]).x, (float)as_h2(x[u * 4 + k]).x, acc);
                    acc = __builtin_fmaf((float)as_h2(ww[k]).y, (float)as_h2(x[u * 4 + k]).y, acc);
                }
            }
        }
}
// The last segment's ragged tail and the appended token.  w1(t): the weight of the segment's token t.
template <int D, int BITS, typename W1>
__device__ __forceinline__ void lone_values_end(const LoneLoads<D, BITS> &s, Lone &st, W1 &&w1, int bx, int c, int T, h1 *state_out, const Seg &sa,
                                                bool active, float &acc)
{
    if (!s.last)
        return;
#pragma unroll
    for (int t = 0; t < s.TPW - 1; t++)
        if (t < s.ntail)
            acc = __builtin_fmaf((float)w1(s.TPW * s.nfull + t), (float)lone_token(st, s.code(t)), acc);
    acc = __builtin_fmaf((float)w1(T - s.t0), (float)lone_append(s, st, bx, c, T, state_out, sa, active), acc);
}

// The same for GQ query heads: the values of four tokens of a lane's channel are a column for the matrix cores as
// they are, the weights of the query heads the rows (see ov_gqa_segment); element i of acc[n] is head 4n + i.
// w: a row of LONE_SEG weights per head, from the first of the n units on.
template <int GQ, int D, int BITS>
__device__ __forceinline__ void lone_values_grouped(const uint2 *lut, uint32_t lane_copy, LoneLoads<D, BITS> &s, Lone &st, int n_units, const h1 *w,
                                                    int lane, f4v *acc)
{
    constexpr int NB = (GQ + 3) / 4;
    if (n_units <= 0)
        return;
    const uint4 *w4[NB];
    uint2 e[2][4];
    uint4 wv[2][NB];
    lone_lookup<BITS>(e[0], lut, s.buf, 0, lane_copy);
#pragma unroll
    for (int n = 0; n < NB; n++) {
        w4[n] = reinterpret_cast<const uint4 *>(w + min(4 * n + (lane & 3), GQ - 1) * LONE_SEG);
        wv[0][n] = w4[n][0];
    }
    wait_lgkm();
    rotate_over<LONE_PF>(n_units, [&](int sg, auto ic) __attribute__((always_inline)) {
        constexpr int i = decltype(ic)::value, half = i & 1;
        lone_lookup<BITS>(e[half ^ 1], lut, s.buf, (i + 1) % LONE_PF, lane_copy); // stale past the end: looked up, never used
#pragma unroll
        for (int n = 0; n < NB; n++)
            wv[half ^ 1][n] = w4[n][sg + 1]; // so are these: a row goes on for a vector
        s.refill(i);
        __builtin_amdgcn_sched_barrier(0);
        uint32_t x[4];
        lone_eight<true>(st, e[half], x);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int n = 0; n < NB; n++) {
            acc[n] = __builtin_amdgcn_mfma_f32_4x4x4f16(as_h4(wv[half][n].x, wv[half][n].y), as_h4(x[0], x[1]), acc[n], 0, 0, 0);
            acc[n] = __builtin_amdgcn_mfma_f32_4x4x4f16(as_h4(wv[half][n].z, wv[half][n].w), as_h4(x[2], x[3]), acc[n], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    });
}

// What lone_values_ahead has left, by the weights of GQ query heads (see lone_weigh).
template <int GQ, int UNITS>
__device__ __forceinline__ void lone_weigh_grouped(const uint32_t *x, int done, const h1 *w, int lane, f4v *acc)
{
#pragma unroll
    for (int n = 0; n < (GQ + 3) / 4; n++) {
        const uint4 *w4 = reinterpret_cast<const uint4 *>(w + min(4 * n + (lane & 3), GQ - 1) * LONE_SEG);
#pragma unroll
        for (int g = 0; g < UNITS; g += LONE_PF)
            if (g < done) {
#pragma unroll
                for (int u = g; u < g + LONE_PF; u++) {
                    const uint4 wv = w4[u];
                    acc[n] = __builtin_amdgcn_mfma_f32_4x4x4f16(as_h4(wv.x, wv.y), as_h4(x[4 * u], x[4 * u + 1]), acc[n], 0, 0, 0);
                    acc[n] = __builtin_amdgcn_mfma_f32_4x4x4f16(as_h4(wv.z, wv.w), as_h4(x[4 * u + 2], x[4 * u + 3]), acc[n], 0, 0, 0);
                }
            }
    }
}

template <int BLK>
__global__ __launch_bounds__(BLK) void qk_lone_kernel(const h1 *q, uint4 *cache, const h1 *k_new, h1 *__restrict__ out, FtParams p, int BH,
                                                      int H, int T, int n_super_cap, h1 *__restrict__ state_out, Seg sa)
{
    constexpr int WAVES = BLK / 64;
    sa.groups = 0; // only even plans come here
    // the table at LDS offset 0, a tile per wave, a chunk of partial logits per wave: half of a CU's LDS
    __shared__ uint4 smem[(LUT_WORDS64 * 8 + WAVES * LONE_TILE + WAVES * LONE_CHUNK * 4) / 16];
    uint2 *lut = reinterpret_cast<uint2 *>(smem);
    char *lds = reinterpret_cast<char *>(smem) + LUT_WORDS64 * 8;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t lane_copy = (uint32_t)(lane & (LUT_COPIES - 1)) * 8u;
    const LoneUnit un(BH, sa.nseg, (int)blockIdx.x * WAVES + wave);
    LoneScores<BLK <= 512> scores(lds + wave * LONE_TILE, lane, q + (size_t)un.bx * 128 + un.half * 64);
    LoneLoads<> s;
    s.start(cache, p, k_new, un.bx % H, un.bx, un.c, un.seg, T, n_super_cap, sa);
    lone_fill<BLK>(lut, threadIdx.x);
    __syncthreads();

    float *unit_part = reinterpret_cast<float *>(lds + WAVES * LONE_TILE) + (wave >> 1) * 2 * LONE_CHUNK;
    float *part = unit_part + un.half * LONE_CHUNK;
    h1 *ob = out + (size_t)un.bx * sa.row_pitch + s.t0;
    // the unit's logits from t on, n of them: the shares of its two waves added
    auto flush = [&](int t, int n) __attribute__((always_inline)) {
        __syncthreads();
        if (un.active)
            for (int i = un.c; i < n; i += 128)
                ob[t + i] = (h1)(unit_part[i] + unit_part[LONE_CHUNK + i]);
        __syncthreads();
    };
    Lone st = s.state();
    scores.ready(sa.act_bf16);
    const int longest = sa.nseg > 1 ? sa.seg_tokens : T; // every wave of the workgroup takes part in every exchange
    for (int t = 0; t < longest; t += LONE_CHUNK) {
        const int n = max(0, min(LONE_CHUNK / 8, s.nfull - t / 8));
        scores.run(lut, lane_copy, st, s, n, part);
        flush(t, 8 * n);
    }
    if (s.last)
        scores.finish(s, st, un.bx, un.c, T, state_out, sa, un.active, part);
    flush(s.nfull * 8, s.last ? s.ntail + 1 : 0);
}

template <int BLK>
__global__ __launch_bounds__(BLK) void ov_lone_kernel(const h1 *attn, uint4 *cache, const h1 *v_new, h1 *__restrict__ out,
                                                      float *__restrict__ partial, FtParams p, int BH, int H, int T, int n_super_cap,
                                                      h1 *__restrict__ state_out, Seg sa)
{
    constexpr int WAVES = BLK / 64;
    sa.groups = 0;
    // the table at LDS offset 0; per wave the weights of a chunk (and a vector that is read behind them, never used)
    __shared__ uint4 smem[LUT_WORDS64 / 2 + WAVES * (LONE_CHUNK / 8 + 1)];
    const uint2 *lut = reinterpret_cast<const uint2 *>(smem);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    uint4 *weights = smem + LUT_WORDS64 / 2 + wave * (LONE_CHUNK / 8 + 1);
    const uint32_t lane_copy = (uint32_t)(lane & (LUT_COPIES - 1)) * 8u;
    const LoneUnit un(BH, sa.nseg, (int)blockIdx.x * WAVES + wave);
    LoneLoads<> s;
    s.start(cache, p, v_new, un.bx % H, un.bx, un.c, un.seg, T, n_super_cap, sa);
    const h1 *wb = attn + (size_t)un.bx * sa.row_pitch + s.t0;
    // a chunk's weights, eight tokens per lane, a chunk ahead: as a load of eight for all lanes alike, one per supergroup,
    // they were a tenth of a lone wave's time (more where rows are only 2-byte aligned).  As built the wave waits at each
    // chunk for its code loads too; with whole chunks in a loop of their own, which waits for the weights alone, it
    // was slower: 1 x 32 heads x 1024 tokens 14.8 / 15.7 us, 2 x 8 x 700 12.0 / 13.1, 3 x 40 x 5000 61.8 / 66.0.
    uint4 ahead = make_uint4(0, 0, 0, 0);
    auto load_chunk = [&](int sg) __attribute__((always_inline)) {
        if (s.nfull > 0)
            __builtin_memcpy(&ahead, wb + (size_t)min(sg + lane, s.nfull - 1) * 8, 16);
    };
    load_chunk(0);
    lone_fill<BLK>(reinterpret_cast<uint2 *>(smem), threadIdx.x);
    __syncthreads();
    if (!un.active)
        return;
    Lone st = s.state();
    float acc = 0.0f;
    for (int sg = 0; sg < s.nfull; sg += LONE_CHUNK / 8) {
        weights[lane] = ahead;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); // read by the wave's other lanes
        load_chunk(sg + LONE_CHUNK / 8);
        lone_values(lut, lane_copy, s, st, min(LONE_CHUNK / 8, s.nfull - sg), reinterpret_cast<const h1 *>(weights), acc);
    }
    lone_values_end(s, st, [&](int t) { return wb[t]; }, un.bx, un.c, T, state_out, sa, true, acc);
    if (sa.nseg == 1) {
        h1 *o = out + (size_t)un.bx * 128 + un.c;
        if (sa.act_bf16)
            *reinterpret_cast<uint16_t *>(o) = (uint16_t)bf16_bits((h1)acc);
        else
            *o = (h1)acc;
    } else {
        partial[((size_t)un.seg * BH + un.bx) * 128 + un.c] = acc;
    }
}

} // namespace adkv
