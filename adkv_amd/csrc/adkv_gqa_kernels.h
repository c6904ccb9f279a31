// Decode kernels for head dim 128 that put the contraction on the matrix cores, for GQ >= 1 query
// heads per KV head and for 4-bit or 2-bit codes.  Included by adkv_kernels.hip after
// the shared device helpers.
//
// The fp16 replay of the filter state (the dominant cost) is the same per-lane arithmetic as in
// qk_kernel / ov_kernel and runs once per KV head; only what happens to the dequantised value
// differs.
//
//   QK:  D[head][token] += A[head][32 channels] * B[32 channels][token], v_mfma_f32_16x16x32_f16
//        The dequantised keys of 8 tokens x 2 heads x 128 channels go through a wave-private LDS
//        tile, whose (head, token) are the 16 columns of four instructions; the rows are the query heads,
//        laid out so that every lane receives the one logit that it stores.
//   The values' product is in blocks: v_mfma_f32_4x4x4_16B_f16 multiplies sixteen independent 4x4 blocks per instruction,
//   lane 4b+r supplies row r of A and column r of B of block b (four fp16 each) and receives column
//   r of D (four fp32, one per row).
//   OV:  D[head][channel] += A[head][4 tokens] * B[4 tokens][channel]
//        B is the lane's own channel over four consecutive tokens (two v_perm_b32 per channel pair
//        repack token-major pairs), A the attention weights of the block's heads: every lane gets
//        the outputs of all GQ heads for its own channels, with no data leaving the lane.
//
// The time axis is walked in units of 8 tokens: one unit per supergroup with 4-bit codes, two with
// 2-bit codes (16 tokens per channel word).  Table lookups for the next unit are issued between
// the tokens of the current one, into the register slots they vacate.
#pragma once

namespace adkv {


constexpr int GQA_D = 128;
// The key tile of a wave: 8 token rows of a lane's two channel pairs (8 bytes) per lane, the wave's two KV heads one
// behind the other.  The LDS takes 16 lanes of an access per clock: of 8-byte writes 16 consecutive ones, over 32
// four-byte banks, which write 128 consecutive bytes here; of 16-byte reads lanes 0-3, 12-15 and 20-27, then the others of
// each 32, over 64 banks (with rows and heads spread for 16 consecutive lanes half of the reads met another:
// SQ_LDS_BANK_CONFLICT).  A matrix operand's lanes are 8 tokens of the first head, 8 of the second, then the same for the next
// 16 bytes: with rows 32 and heads 0 modulo 256 bytes apart the eight reads of either piece meet none of the other's.
// (Read as pairs of 8 bytes, at half the rate, the operand kept the LDS busy for a sixth more.)
constexpr int TILE_HEAD = 256;       // bytes between the heads of a row
constexpr int TILE_ROW = 544;        // bytes per token
constexpr int TILE_WORDS64 = TILE_ROW; // 8-byte words per wave: 8 rows

// The code words of one supergroup -> the per-pair byte streams the table is indexed with.
template <int BITS, typename V>
__device__ __forceinline__ void code_bytes(const V &u, uint32_t (*nb)[2])
{
    uint32_t w[sizeof(V) / 4];
    vec_words(u, w);
#pragma unroll
    for (int p = 0; p < (int)sizeof(V) / 8; p++) {
        if (BITS == 4)
            pair_bytes(w[2 * p], w[2 * p + 1], nb[p][0], nb[p][1]);
        else
            pair_bytes2(w[2 * p], w[2 * p + 1], nb[p][0], nb[p][1]);
    }
}

// Table entries of one 8-token unit held in registers, and how a token finds its (q, |q|):
//   4-bit: slot t, 8 bytes.   2-bit: slot 2*(t/4) + (t&1), 16 bytes, second half for t&2.
template <int BITS, int NP>
struct Lookups {
    static constexpr int SLOTS = BITS == 4 ? 8 : 4;
    using Entry = typename std::conditional<BITS == 4, uint2, uint4>::type;
    Entry e[NP][SLOTS];

    // all lookups of unit `half` (0 or 1 within the supergroup) of the words `nb`
    __device__ __forceinline__ void fill(const uint2 *lut, const uint32_t (*nb)[2], uint32_t lane_copy, int half)
    {
#pragma unroll
        for (int p = 0; p < NP; p++) {
            if constexpr (BITS == 4) {
#pragma unroll
                for (int t = 0; t < 8; t++)
                    e[p][t] = lut_get(lut, nb[p][t & 1], lane_copy, t >> 1);
            } else {
#pragma unroll
                for (int s = 0; s < 4; s++)
                    e[p][s] = lut2_get(lut, nb[p][s & 1], lane_copy, 2 * half + (s >> 1));
            }
        }
    }
    __device__ __forceinline__ void get(int p, int t, h2 &q, h2 &qabs) const
    {
        if constexpr (BITS == 4) {
            q = as_h2(e[p][t].x);
            qabs = as_h2(e[p][t].y);
        } else {
            const uint4 v = e[p][2 * (t >> 2) + (t & 1)];
            q = as_h2((t & 2) ? v.z : v.x);
            qabs = as_h2((t & 2) ? v.w : v.y);
        }
    }
    // after token t: refill the slot it has just finished with, for the unit `next_half` of `nb`
    __device__ __forceinline__ void refill(const uint2 *lut, const uint32_t (*nb)[2], uint32_t lane_copy,
                                           int t, int next_half)
    {
        if constexpr (BITS == 4) {
#pragma unroll
            for (int p = 0; p < NP; p++)
                e[p][t] = lut_get(lut, nb[p][t & 1], lane_copy, t >> 1);
        } else {
            if (t & 2) {
#pragma unroll
                for (int p = 0; p < NP; p++)
                    e[p][2 * (t >> 2) + (t & 1)] = lut2_get(lut, nb[p][t & 1], lane_copy, 2 * next_half + (t >> 2));
            }
        }
    }
};

template <int BITS, int NT>
__device__ __forceinline__ void fill_table(uint2 *lut, int tid)
{
    if (BITS == 4)
        lut_fill<NT>(lut, tid);
    else
        lut2_fill(lut, tid, NT);
}

template <int BITS>
__device__ __forceinline__ uint32_t table_lane_offset(int lane)
{
    return BITS == 4 ? (uint32_t)(lane & (LUT_COPIES - 1)) * 8u : (uint32_t)(lane & (LUT2_COPIES - 1)) * 16u;
}

// forward_qk of one segment, two channels per lane: a KV head fills the wave (see PairScores).
template <int BITS, int GQ, bool LONE>
__device__ __forceinline__ void qk_gqa_pair_segment(const uint2 *lut, int lane, int bx, PairScores<BITS, GQ, LONE> &scores,
                                                    SegLoads<GQA_D, 2, BITS, PairScores<BITS, GQ, LONE>::AHEAD> &s,
                                                    const h1 *k_new, h1 *out, int T, h1 *state_out, const Seg &sa)
{
    constexpr int D = GQA_D, CPL = 2, TPW = Code<BITS>::TPW;
    using G = Geo<D, CPL>;
    const int c0 = lane * CPL;
    Pair st[1];
    s.state(st);
    scores.ready(sa.act_bf16);
    const bool last = s.last;
    const int t0 = s.t0, t1 = s.t1, nfull = s.nfull;
    uint2 *cbh = s.cbh;
    const uint2 *cb = s.cb;
    h1 *ob = out + (size_t)bx * GQ * sa.row_pitch + t0;
    auto put = [&](int t, int g, h1 v) __attribute__((always_inline)) { ob[(size_t)g * sa.row_pitch + t] = v; };
    scores.run(lut, table_lane_offset<BITS>(lane), st[0], s, put);
    if (!last)
        return;
    // ragged tail and the appended token: at most a tile
    const int ntail = (t1 - t0) % TPW;
    if (ntail) {
        const uint2 w = cb[(size_t)nfull * G::VPS];
        for (int tt = 0; tt < ntail; tt++) {
            const h2 qc = extract_pair<BITS>(w.x, w.y, tt);
            const h2 qs = qc * st[0].sc;
            scores.write(tt, as_u32(qs + st[0].zp));
            update_pair(st[0], qc, qs);
        }
    }
    publish_state<D, CPL>(st, state_out, sa, bx, c0, T);
    h2 deq[1];
    append_new_token<D, CPL, BITS>(cbh, T, k_new + (size_t)bx * D + c0, st, deq, true, sa.act_bf16);
    scores.write(ntail, as_u32(deq[0]));
    scores.fetch();
    scores.multiply();
    scores.emit(nfull * TPW, ntail + 1, put);
}

// ---------------------------------------------------------------------------------------------
// forward_qk with GQ query heads per KV head
// ---------------------------------------------------------------------------------------------
template <int BITS, int GQ, int BLK, int CPL>
__global__ __launch_bounds__(BLK) void qk_gqa_kernel(
    const h1 *q, uint4 *__restrict__ cache, const h1 *k_new,
    h1 *__restrict__ out,
    const h1 *zp, const h1 *sc, const h1 *al,
    const h1 *be, const h1 *tg,
    int BH, int H, int T, int n_super_cap, h1 *__restrict__ state_out, Seg sa)
{
    if constexpr (CPL == 2) {
        sa.groups = 0; // only even plans come here
        __shared__ uint2 smem[LUT_WORDS64 + (BLK / 64) * PAIR_TILE / 8];
        const Unit<GQA_D, 2, BLK> un(BH, sa.nseg);
        using Scores = PairScores<BITS, GQ, BLK == 256>;
        Scores scores(reinterpret_cast<char *>(smem + LUT_WORDS64) + (threadIdx.x >> 6) * PAIR_TILE, un.lh,
                      q + (size_t)un.bx * GQ * GQA_D);
        SegLoads<GQA_D, 2, BITS, Scores::AHEAD> s;
        s.start(cache, zp, sc, al, be, tg, un.bx % H, un.bx, un.lh, un.seg, T, n_super_cap, sa);
        fill_table<BITS, BLK>(smem, threadIdx.x);
        __syncthreads();
        if (un.wave_active)
            qk_gqa_pair_segment<BITS, GQ>(smem, un.lh, un.bx, scores, s, k_new, out, T, state_out, sa);
    } else {
    constexpr int D = GQA_D;
    constexpr int NB = (GQ + 3) / 4; // column sets of four heads
    constexpr int TPW = Code<BITS>::TPW, UPS = TPW / 8;
    // supergroups in flight per lane: fewer where a supergroup is 16 tokens or registers are short
    constexpr int GPF = (BITS == 2 || NB > 1) ? 2 : PF;
    using G = Geo<D, CPL>;
    __shared__ __align__(16) uint2 smem[LUT_WORDS64 + (BLK / 64) * TILE_WORDS64];
    const uint2 *lut = smem;
    const int lane = threadIdx.x & 63;
    const uint32_t lane_copy = table_lane_offset<BITS>(lane);
    char *tile = reinterpret_cast<char *>(smem + LUT_WORDS64 + (threadIdx.x >> 6) * TILE_WORDS64);

    const Unit<D, CPL, BLK> un(BH, sa.nseg); // a padding wave's is valid too: it loads and leaves
    const int bx = un.bx, lh = un.lh, c0 = un.c0;
    const bool active = un.active;
    SegLoads<D, CPL, BITS, GPF> s;
    s.start(cache, zp, sc, al, be, tg, bx % H, bx, lh, un.seg, T, n_super_cap, sa);
    fill_table<BITS, BLK>(smem, threadIdx.x);
    __syncthreads();
    if (!un.wave_active)
        return; // padding waves
    const bool last = s.last;

    Pair st[G::NP];
    s.state(st);

    // Matrix-core roles of this lane.  Column lane % 16 of B is a token of one of the wave's two KV heads, and a quarter
    // of the wave has 32 of its channels' 128 (eight per instruction).  Row 4g + r of A is query head g of KV head r % 2 (head
    // 4 + g for r = 2, 3), so that element r of quarter g's result is head g's logit: a lane keeps the one of its
    // column's KV head, and nothing is summed across lanes.  (In sixteen blocks of 4 x 4, each a quarter of the channels, it
    // was twice the instructions for up to four query heads, four times for eight, and six DPP adds for every four heads:
    // 16 x 8 KV heads x 131072 tokens of 2-bit codes, four query heads, 546 k cycles and 282 us, 498 k and 260 in this form.)
    const int quarter = lane >> 4, kv = lane >> 3 & 1, tok = lane & 7;
    const int bx0 = __builtin_amdgcn_readlane(bx, 0), bx1 = __builtin_amdgcn_readlane(bx, 32);
    h8v qa[4];
    {
        const int head = (lane >> 2 & 3) + (lane & 2) * 2;
        const h1 *src = q + ((size_t)(lane & 1 ? bx1 : bx0) * GQ + min(head, GQ - 1)) * D + quarter * 8;
#pragma unroll
        for (int m = 0; m < 4; m++) {
            uint32_t w[4];
#pragma unroll
            for (int i = 0; i < 4; i++)
                w[i] = as_u32(load_act2(src + 32 * m + 2 * i, sa.act_bf16));
            qa[m] = __builtin_bit_cast(h8v, make_uint4(w[0], w[1], w[2], w[3]));
        }
    }
    const char *brow = tile + tok * TILE_ROW + kv * TILE_HEAD + quarter * 16;
    char *wcol = tile + (lane >> 5) * TILE_HEAD + (lane & 31) * 8; // where this lane's values go in the first row
    const uint32_t other = kv ? ~0u : 0u;
    const bool storer = un.wave_active && (kv ? __builtin_amdgcn_readlane(active, 32) : __builtin_amdgcn_readlane(active, 0));
    h1 *orow = out + ((size_t)(kv ? bx1 : bx0) * GQ + min(quarter, GQ - 1)) * sa.row_pitch + s.t0 + tok;

    const int t0 = s.t0, t1 = s.t1, nfull = s.nfull;
    uint4 *cbh = s.cbh;
    const uint4 *cb = s.cb;
    auto &buf = s.buf;

    // logits of the tile's tokens: read the keys, run the instructions, store.  `unit` counts 8-token units from t0.
    h8v keys[4] = {}; // multiplied (and discarded) once before the first unit has filled the tile
    f4v d;
    auto fetch = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < 4; m++)
            keys[m] = *reinterpret_cast<const h8v *>(brow + m * 64);
    };
    auto multiply = [&]() __attribute__((always_inline)) {
        d = (f4v){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int m = 0; m < 4; m++)
            d = __builtin_amdgcn_mfma_f32_16x16x32_f16(qa[m], keys[m], d, 0, 0, 0);
    };
    auto emit = [&](int unit, int ntok) __attribute__((always_inline)) {
        const auto mine = [&](float a, float b) { // a select by lanes as a masked merge
            return __uint_as_float((__float_as_uint(b) & other) | (__float_as_uint(a) & ~other));
        };
        const bool here = storer && tok < ntok;
        if (here && quarter < GQ)
            orow[unit * 8] = (h1)mine(d.x, d.y);
        if constexpr (GQ == 8)
            if (here)
                orow[4 * sa.row_pitch + unit * 8] = (h1)mine(d.z, d.w);
    };

    Lookups<BITS, G::NP> lk;
    // token t of the current unit; then the lookups that reuse its slot for the unit after it
    auto token = [&](int t, const uint32_t (*nbnext)[2], int next_half) {
        uint32_t kh[G::NP];
#pragma unroll
        for (int p = 0; p < G::NP; p++) {
            Pair &s = st[p];
            h2 qc, qa;
            lk.get(p, t, qc, qa);
            const h2 qs = qc * s.sc;
            kh[p] = as_u32(qs + s.zp);
            update_pair_abs(s, qa, qs);
        }
        *reinterpret_cast<uint2 *>(wcol + t * TILE_ROW) = make_uint2(kh[0], kh[1]);
        lk.refill(lut, nbnext, lane_copy, t, next_half);
        __builtin_amdgcn_sched_barrier(0);
    };

    uint32_t nbc[G::NP][2], nbn[G::NP][2]; // byte streams of the current / the next supergroup
    if (nfull > 0) {
        code_bytes<BITS>(buf[0][0], nbc);
        lk.fill(lut, nbc, lane_copy, 0);
    }
    // one supergroup, nothing conditional in it; i = its buffer in the rotation
    auto body = [&](int sg, auto ic) {
        constexpr int i = decltype(ic)::value;
        // bytes of supergroup sg+1 (stale data past the end: looked up, never used)
        code_bytes<BITS>(buf[(i + 1) % GPF][0], nbn);
        // unconditional, clamped to the segment's last supergroup: a load inside a branch makes
        // the next wait cover every load in flight, this one included
        buf[i][0] = load_codes(cb + (size_t)min(sg + GPF, nfull - 1) * G::VPS);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int hf = 0; hf < UPS; hf++) {
            const int unit = sg * UPS + hf;
            const bool into_next_sg = hf == UPS - 1;
#pragma unroll
            for (int t = 0; t < 3; t++)
                token(t, into_next_sg ? nbn : nbc, into_next_sg ? 0 : hf + 1);
            // the tile reads of the previous unit were issued before these three tokens overwrote
            // its first rows (LDS operations of a wave execute in order); nothing is stored for
            // the unit before the first
            multiply();
#pragma unroll
            for (int t = 3; t < 5; t++)
                token(t, into_next_sg ? nbn : nbc, into_next_sg ? 0 : hf + 1);
            emit(unit - 1, unit > 0 ? 8 : 0);
#pragma unroll
            for (int t = 5; t < 8; t++)
                token(t, into_next_sg ? nbn : nbc, into_next_sg ? 0 : hf + 1);
            fetch();
        }
#pragma unroll
        for (int p = 0; p < G::NP; p++) {
            nbc[p][0] = nbn[p][0];
            nbc[p][1] = nbn[p][1];
        }
    };
    rotate_over<GPF>(nfull, body);
    if (nfull > 0) {
        multiply();
        emit(nfull * UPS - 1, 8);
    }
    if (!last)
        return;

    // ragged tail (fewer than a supergroup of tokens, gemv.cu:648-654) and the appended token
    const int ntail = (t1 - t0) % TPW;
    int unit = nfull * UPS, row = 0;
    if (ntail) {
        const uint4 u = cb[(size_t)nfull * G::VPS];
        const uint32_t w[4] = {u.x, u.y, u.z, u.w};
        for (int tt = 0; tt < ntail; tt++) {
            uint32_t kh[2];
#pragma unroll
            for (int pp = 0; pp < 2; pp++) {
                Pair &s = st[pp];
                const h2 qc = extract_pair<BITS>(w[2 * pp], w[2 * pp + 1], tt);
                const h2 qs = qc * s.sc;
                kh[pp] = as_u32(qs + s.zp);
                update_pair(s, qc, qs);
            }
            *reinterpret_cast<uint2 *>(wcol + row * TILE_ROW) = make_uint2(kh[0], kh[1]);
            if (++row == 8) {
                fetch();
                multiply();
                emit(unit, 8);
                unit++;
                row = 0;
            }
        }
    }
    if (active)
        publish_state<D, CPL>(st, state_out, sa, bx, c0, T);
    h2 deq[G::NP];
    append_new_token<D, CPL, BITS>(cbh, T, k_new + (size_t)bx * D + c0, st, deq, active, sa.act_bf16);
    *reinterpret_cast<uint2 *>(wcol + row * TILE_ROW) = make_uint2(as_u32(deq[0]), as_u32(deq[1]));
    fetch();
    multiply();
    emit(unit, row + 1);
    }
}

// ---------------------------------------------------------------------------------------------
// forward_ov with GQ query heads per KV head
// ---------------------------------------------------------------------------------------------
// forward_ov of one segment for GQ query heads: acc[column set][channel of this lane], element i = head
// 4n + i.  w8(n, unit): the weights of the unit's eight tokens for this lane's row of column set n, the
// first two units' in wbuf; w1(head, t): the weight of the segment's token t.
constexpr int GQA_WPF = 2; // weight vectors (8 tokens each) in flight
template <int BITS, int GQ, int CPL>
constexpr int gqa_ahead() { return (BITS == 2 || GQ > 4) ? 2 : PF; } // supergroups in flight per lane
template <int BITS, int GQ, int CPL, typename W8, typename W1>
__device__ __forceinline__ void ov_gqa_segment(const uint2 *lut, uint32_t lane_copy, int bx, int c0, bool active,
                                               SegLoads<GQA_D, CPL, BITS, gqa_ahead<BITS, GQ, CPL>()> &s,
                                               uint4 (*wbuf)[(GQ + 3) / 4], W8 &&w8, W1 &&w1, const h1 *v_new, int T,
                                               h1 *state_out, const Seg &sa, f4v (*acc)[CPL])
{
    constexpr int D = GQA_D, NB = (GQ + 3) / 4, TPW = Code<BITS>::TPW, UPS = TPW / 8;
    constexpr int GPF = gqa_ahead<BITS, GQ, CPL>(), WPF = GQA_WPF;
    static_assert((GPF * UPS) % WPF == 0, "weight ring must line up with the unrolled loop");
    using G = Geo<D, CPL>;
    using Vec = typename G::Vec;
    const bool last = s.last;
    const int t0 = s.t0, t1 = s.t1, nfull = s.nfull, nunits = nfull * UPS;
    Vec *cbh = s.cbh;
    const Vec *cb = s.cb;
    auto &buf = s.buf;
    Pair st[G::NP];
    s.state(st);
#pragma unroll
    for (int n = 0; n < NB; n++)
#pragma unroll
        for (int c = 0; c < CPL; c++)
            acc[n][c] = (f4v){0.0f, 0.0f, 0.0f, 0.0f};

    // four tokens of dequantised values, token-major pairs -> per-channel h4 -> four instructions
    auto contract = [&](const uint32_t (*kh)[4], const uint4 *wv, int half) {
        uint32_t b[CPL][2];
#pragma unroll
        for (int p = 0; p < G::NP; p++) {
            b[2 * p][0] = __builtin_amdgcn_perm(kh[p][1], kh[p][0], 0x05040100u);
            b[2 * p][1] = __builtin_amdgcn_perm(kh[p][3], kh[p][2], 0x05040100u);
            b[2 * p + 1][0] = __builtin_amdgcn_perm(kh[p][1], kh[p][0], 0x07060302u);
            b[2 * p + 1][1] = __builtin_amdgcn_perm(kh[p][3], kh[p][2], 0x07060302u);
        }
#pragma unroll
        for (int n = 0; n < NB; n++) {
            const h4v a = half ? as_h4(wv[n].z, wv[n].w) : as_h4(wv[n].x, wv[n].y);
#pragma unroll
            for (int c = 0; c < CPL; c++)
                acc[n][c] = __builtin_amdgcn_mfma_f32_4x4x4f16(a, as_h4(b[c][0], b[c][1]), acc[n][c], 0, 0, 0);
        }
    };
    if constexpr (CPL == 2 && GQ <= 4) {
        // One pair per lane: eight tokens laid out by hand (replay_eight), whose lookups are out a unit ahead.  Token by token
        // every packed result was read by the next instruction or the one behind it, 51 wait states per 32 tokens: steps of 6 x 8
        // KV heads x 9000 tokens 34.3 us instead of 33.5, 8 x 8 x 16001 58.9 instead of 58.4, 16 x 8 x 6000 45.6 instead of 45.0.  (With eight
        // query heads the registers are short: 10 x 8 x 9000 55.1 us token by token, 55.6 like this.)
        uint2 e[2][8];
        uint32_t nb[2];
        auto bytes = [&](const Vec &u) __attribute__((always_inline)) {
            if constexpr (BITS == 4)
                pair_bytes(u.x, u.y, nb[0], nb[1]);
            else
                pair_bytes2(u.x, u.y, nb[0], nb[1]);
        };
        if (nfull > 0) {
            bytes(buf[0][0]);
            pair_lookup<BITS>(e[0], lut, nb, lane_copy, 0);
            wait_lgkm();
        }
        rotate_over<GPF>(nfull, [&](int sg, auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value;
            static_for<UPS>([&](auto hc) __attribute__((always_inline)) {
                constexpr int hf = decltype(hc)::value, half = (i * UPS + hf) & 1, ws = (i * UPS + hf) % WPF;
                if constexpr (hf == UPS - 1) {
                    bytes(buf[(i + 1) % GPF][0]); // stale past the end: looked up, never used
                    pair_lookup<BITS>(e[half ^ 1], lut, nb, lane_copy, 0);
                    buf[i][0] = load_codes(cb + (size_t)min(sg + GPF, nfull - 1) * G::VPS);
                } else {
                    pair_lookup<BITS>(e[half ^ 1], lut, nb, lane_copy, hf + 1);
                }
                __builtin_amdgcn_sched_barrier(0);
                uint32_t x[8];
                replay_eight(st[0], e[half], x);
                contract(reinterpret_cast<uint32_t (*)[4]>(x), wbuf[ws], 0);
                contract(reinterpret_cast<uint32_t (*)[4]>(x + 4), wbuf[ws], 1);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int n = 0; n < NB; n++)
                    wbuf[ws][n] = w8(n, min(sg * UPS + hf + WPF, nunits - 1)); // reloaded once used: see below
            });
        });
    } else {
        uint32_t kh[G::NP][4];
        Lookups<BITS, G::NP> lk;
        auto token = [&](int t, const uint32_t (*nbnext)[2], int next_half) {
    #pragma unroll
            for (int p = 0; p < G::NP; p++) {
                Pair &s = st[p];
                h2 qc, qa;
                lk.get(p, t, qc, qa);
                const h2 qs = qc * s.sc;
                kh[p][t & 3] = as_u32(qs + s.zp);
                update_pair_abs(s, qa, qs);
            }
            lk.refill(lut, nbnext, lane_copy, t, next_half);
            __builtin_amdgcn_sched_barrier(0);
        };

        uint32_t nbc[G::NP][2], nbn[G::NP][2];
        if (nfull > 0) {
            code_bytes<BITS>(buf[0][0], nbc);
            lk.fill(lut, nbc, lane_copy, 0);
        }
        // one supergroup, nothing conditional in it; i = its buffer in the rotation
        auto body = [&](int sg, auto ic) {
            constexpr int i = decltype(ic)::value;
            code_bytes<BITS>(buf[(i + 1) % GPF][0], nbn);
            buf[i][0] = load_codes(cb + (size_t)min(sg + GPF, nfull - 1) * G::VPS); // unconditional: see qk_gqa_kernel
    #pragma unroll
            for (int hf = 0; hf < UPS; hf++) {
                const int unit = sg * UPS + hf;
                const int ws = (i * UPS + hf) % WPF; // compile-time after unrolling
                __builtin_amdgcn_sched_barrier(0);
                const bool into_next_sg = hf == UPS - 1;
    #pragma unroll
                for (int t = 0; t < 4; t++)
                    token(t, into_next_sg ? nbn : nbc, into_next_sg ? 0 : hf + 1);
                contract(kh, wbuf[ws], 0);
    #pragma unroll
                for (int t = 4; t < 8; t++)
                    token(t, into_next_sg ? nbn : nbc, into_next_sg ? 0 : hf + 1);
                contract(kh, wbuf[ws], 1);
                // reloaded once used: an earlier load into a second register set costs copies at the
                // loop edge, which wait for the load they move
    #pragma unroll
                for (int n = 0; n < NB; n++)
                    wbuf[ws][n] = w8(n, min(unit + WPF, nunits - 1));
            }
    #pragma unroll
            for (int p = 0; p < G::NP; p++) {
                nbc[p][0] = nbn[p][0];
                nbc[p][1] = nbn[p][1];
            }
        };
        rotate_over<GPF>(nfull, body);
    }

    if (last) {
        // ragged tail, then the appended token: a handful of tokens, plain fp32 multiply-adds
        h1 wT[GQ]; // before the stores: they may not be loaded ahead of them afterwards, and cost 0.5 us
#pragma unroll
        for (int g = 0; g < GQ; g++)
            wT[g] = w1(g, T - t0);
        auto add_token = [&](const h2 *vd, auto &&weight) {
#pragma unroll
            for (int g = 0; g < GQ; g++) {
                const float wt = (float)weight(g);
#pragma unroll
                for (int p = 0; p < G::NP; p++) {
                    acc[g >> 2][2 * p][g & 3] = __builtin_fmaf(wt, (float)vd[p].x, acc[g >> 2][2 * p][g & 3]);
                    acc[g >> 2][2 * p + 1][g & 3] =
                        __builtin_fmaf(wt, (float)vd[p].y, acc[g >> 2][2 * p + 1][g & 3]);
                }
            }
        };
        const int ntail = (t1 - t0) % TPW;
        if (ntail) {
            uint32_t w[CPL];
            vec_words(cb[(size_t)nfull * G::VPS], w);
            for (int tt = 0; tt < ntail; tt++) {
                h2 vd[G::NP];
#pragma unroll
                for (int pp = 0; pp < G::NP; pp++) {
                    Pair &s = st[pp];
                    const h2 qc = extract_pair<BITS>(w[2 * pp], w[2 * pp + 1], tt);
                    const h2 qs = qc * s.sc;
                    vd[pp] = qs + s.zp;
                    update_pair(s, qc, qs);
                }
                add_token(vd, [&](int g) { return w1(g, nfull * TPW + tt); });
            }
        }
        if (active)
            publish_state<D, CPL>(st, state_out, sa, bx, c0, T);
        h2 deq[G::NP];
        append_new_token<D, CPL, BITS>(cbh, T, v_new + (size_t)bx * D + c0, st, deq, active, sa.act_bf16);
        add_token(deq, [&](int g) { return wT[g]; });
    }
}

template <int BITS, int GQ, int BLK, int CPL>
__global__ __launch_bounds__(BLK) void ov_gqa_kernel(
    const h1 *attn, uint4 *__restrict__ cache, const h1 *v_new,
    h1 *__restrict__ out, float *__restrict__ partial,
    const h1 *zp, const h1 *sc, const h1 *al,
    const h1 *be, const h1 *tg,
    int BH, int H, int T, int n_super_cap, h1 *__restrict__ state_out, Seg sa)
{
    constexpr int D = GQA_D;
    if (CPL == 2)
        sa.groups = 0; // only even plans come here
    constexpr int NB = (GQ + 3) / 4;
    constexpr int TPW = Code<BITS>::TPW, UPS = TPW / 8;
    constexpr int GPF = gqa_ahead<BITS, GQ, CPL>(), WPF = GQA_WPF;
    __shared__ uint2 lut[LUT_WORDS64];
    const int lane = threadIdx.x & 63;
    const uint32_t lane_copy = table_lane_offset<BITS>(lane);

    const Unit<D, CPL, BLK> un(BH, sa.nseg);
    const int bx = un.bx, lh = un.lh, c0 = un.c0;
    const bool active = un.active;
    const int r = lane & 3;
    SegLoads<D, CPL, BITS, GPF> s;
    s.start(cache, zp, sc, al, be, tg, bx % H, bx, lh, un.seg, T, n_super_cap, sa);
    const int nunits = s.nfull * UPS;
    // A operand rows: the weights of head r (+4 per column set) of this lane's KV head; lanes of no head
    // repeat one, into rows of the product that nobody reads
    const h1 *wb[NB];
#pragma unroll
    for (int n = 0; n < NB; n++)
        wb[n] = attn + ((size_t)bx * GQ + min(4 * n + r, GQ - 1)) * sa.row_pitch + s.t0;
    auto load_w = [&](int n, int unit) {
        uint4 v;
        __builtin_memcpy(&v, wb[n] + (size_t)unit * 8, 16); // rows are only 2-byte aligned
        return v;
    };
    uint4 wbuf[WPF][NB];
    if (nunits > 0)
#pragma unroll
        for (int i = 0; i < WPF; i++)
#pragma unroll
            for (int n = 0; n < NB; n++)
                wbuf[i][n] = load_w(n, min(i, nunits - 1));
    fill_table<BITS, BLK>(lut, threadIdx.x);
    __syncthreads();
    if (!un.wave_active)
        return; // padding waves

    f4v acc[NB][CPL];
    ov_gqa_segment<BITS, GQ, CPL>(lut, lane_copy, bx, c0, active, s, wbuf, load_w,
                                  [&](int g, int t) { return attn[((size_t)bx * GQ + g) * sa.row_pitch + s.t0 + t]; }, v_new, T,
                                  state_out, sa, acc);
    if (!active)
        return;
#pragma unroll
    for (int g = 0; g < GQ; g++) {
        const size_t row = (size_t)bx * GQ + g;
        float o[CPL];
#pragma unroll
        for (int c = 0; c < CPL; c++)
            o[c] = acc[g >> 2][c][g & 3];
#pragma unroll
        for (int c = 0; c < CPL; c += 2) {
            if (sa.nseg == 1)
                store_act2(out + row * D + c0 + c, o[c], o[c + 1], sa.act_bf16);
            else if (CPL == 2)
                *reinterpret_cast<float2 *>(partial + ((size_t)un.seg * BH * GQ + row) * D + c0) = make_float2(o[0], o[1]);
            else if (c == 0)
                *reinterpret_cast<float4 *>(partial + ((size_t)un.seg * BH * GQ + row) * D + c0) =
                    make_float4(o[0], o[1], o[CPL - 2], o[CPL - 1]);
        }
    }
}

} // namespace adkv
