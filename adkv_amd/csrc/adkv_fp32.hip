// fp32 ("train/eval") form of the ADKV recurrence for gfx950.
//
// Restates, per (batch, channel), the step of src/adkv/train/train_model.py:8-22,61-81 and of its
// Triton twin src/adkv/hf/llama_adkv_eval.py:86-97: every operation is a separately rounded fp32
// operation (this file is compiled with contraction off and IEEE division), so results are
// bit-identical to an unfused CPU evaluation.
//
//   s  = max(sc, 1e-8);  q = clamp(rint((x - zp) / s), QL, QU);  r = q*s;  xhat = r + zp
//   zp = zp + alpha*r;   sc = clamp(sc + (sc*beta)*(|q| - tgt), sc_min, sc_max)
//
// The recurrence is serial in t and only channels are parallel (64 to 1024 waves in the sizes this
// form is used at, at most one per SIMD).  A wave alone on its SIMD issues one instruction every 4
// cycles whether or not it depends on the one before (more for some, see recurrence), so the time per
// token is the sum over the instructions of the wave that carries the chain.  quant_kernel therefore
// gives a workgroup two waves: one does nothing but the recurrence, out of LDS and into LDS (four tokens
// per LDS instruction); the other moves rows between memory and LDS, 16 bytes per access, and converts
// types.  4096 channels x 1024 tokens of fp32 take 42 us, 36 ns per token and 5 us for the launch and its
// first rows; with everything in one wave it was 65 us, the rest being loads, stores, their addresses and
// the guards of the rounding.
#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <stdint.h>

#include "../../include/adkv_hip.h"
#include "adkv_device.h"

#pragma clang fp contract(off)

namespace adkv_fp32 {

template <typename T> struct IO;
template <> struct IO<float> {
    typedef float Bits;
    static __device__ __forceinline__ float up(float v) { return v; }
    static __device__ __forceinline__ float down(float v) { return v; }
};
template <> struct IO<_Float16> {
    typedef uint16_t Bits;
    static __device__ __forceinline__ float up(uint16_t v) { return (float)__builtin_bit_cast(_Float16, v); }
    static __device__ __forceinline__ uint16_t down(float v) { return __builtin_bit_cast(uint16_t, (_Float16)v); }
};
template <> struct IO<__hip_bfloat16> {
    typedef uint16_t Bits;
    static __device__ __forceinline__ float up(uint16_t v) { return __uint_as_float((uint32_t)v << 16); }
    static __device__ __forceinline__ uint16_t down(float v)
    {
        // round to nearest even; NaN stays NaN
        const uint32_t u = __float_as_uint(v);
        return (v != v) ? (uint16_t)((u >> 16) | 0x40) : (uint16_t)((u + 0x7FFF + ((u >> 16) & 1)) >> 16);
    }
};

// One tensor of a launch.  Either starting state may be absent: zp0 / sc0 are [C], zp_io / sc_io [B, C].
struct Tensor {
    const void *x;
    void *xhat;
    int8_t *codes;
    float *zp_io, *sc_io;
    const float *zp0, *sc0, *alpha, *beta, *tgt;
    float *zp_seq, *sc_seq;
    long xs_b, xs_t, os_b, os_t; // element strides of x and xhat; channels are contiguous
    bool free; // alpha, beta and sc0 are what training moves: sigmoid, 0.1*sigmoid and exp of them are meant
};

// torch.sigmoid and torch.exp of fp32 (all 2^32 inputs compared)
__device__ __forceinline__ float sigmoid(float v) { return 1.0f / (1.0f + expf(-v)); }

struct Limits {
    float ql, qu, sc_min, sc_max;
    float sure; // see Chan::step_spec
};

// torch.clamp semantics: NaN passes through
__device__ __forceinline__ float clamp_keep_nan(float x, float lo, float hi)
{
    if (x != x)
        return x;
    return x < lo ? lo : (x > hi ? hi : x);
}

// NaN once an operand is one
__device__ __forceinline__ float collect_abs(float acc, float a, float b)
{
    float r;
    asm("v_maximum3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(acc), "v"(a), "v"(b));
    return r;
}

constexpr int GRP = 8; // tokens per speculative group

struct Chan {
    float zp, sc, s, rs; // s = max(sc, 1e-8) (NaN kept), rs ~ 1/s
    float al, be, tg;
    float sure; // no |off| reaches it: what step_spec returned is the reference's (below)
    __device__ __forceinline__ void init(const Tensor &a, int b, int c, int C, const Limits &l)
    {
        zp = a.zp0 ? a.zp0[c] : a.zp_io[(long)b * C + c];
        float s0 = a.sc0 ? a.sc0[c] : a.sc_io[(long)b * C + c];
        al = a.alpha[c];
        be = a.beta[c];
        tg = a.tgt[c];
        if (a.free) { // four elementwise launches otherwise: 8 of the 50 us of a forward of 1024 tokens x 4096 channels
            al = sigmoid(al);
            be = sigmoid(be) * 0.1f;
            s0 = expf(s0);
        }
        set_scale(s0);
        // |sc*be| < 2^60 and |e| < 2^61: no scale of this channel can become a NaN before it is clamped.  A channel
        // that is not known to be so has its groups repeated, every one (a NaN here as well).
        const float most = fmaxf(fmaxf(l.sc_max, -l.sc_min), __builtin_fabsf(sc));
        sure = most <= 0x1p100f && __builtin_fabsf(be) * most < 0x1p60f && __builtin_fabsf(tg) < 0x1p60f ? l.sure : -1.0f;
    }
    __device__ __forceinline__ void set_scale(float v)
    {
        sc = v;
        s = (v != v) ? v : (v < 1e-8f ? 1e-8f : v);
        // a scale whose reciprocal could be subnormal is left to the division
        rs = s <= 0x1p100f ? __builtin_amdgcn_rcpf(s) : __builtin_nanf("");
    }
    // One token with the reference's operations and nothing else.
    __device__ __forceinline__ float step(float xv, const Limits &l, float &q)
    {
        const float d = xv - zp;
        q = clamp_keep_nan(__builtin_rintf(d / s), l.ql, l.qu);
        const float xr = q * s;
        const float xh = xr + zp;
        const float ax = al * xr;
        const float e = __builtin_fabsf(q) - tg;
        const float sb = sc * be;
        const float sbe = sb * e;
        zp = zp + ax;
        set_scale(clamp_keep_nan(sc + sbe, l.sc_min, l.sc_max));
        return xh;
    }
    // The same token for a group that is checked afterwards: 15 instructions (rcp takes two slots).
    //
    // The quotient is r = d*rs with the reciprocal kept from the token before.  |r - u| <= |u|*2^-22
    // for the IEEE quotient u (reciprocal 2^-23, two roundings 2^-24 each).  With L the largest code
    // magnitude, |u| > L + 1 is clamped either way, and below that rint(r) == rint(u) unless r lies
    // closer than (L + 1)*2^-22 to k + 1/2, that is unless |r - rint(r)| >= sure = 1/2 - (L + 1)*2^-21
    // (twice the bound).  `off` returns r - rint(r), a NaN when r is infinite or one.  The caller repeats the
    // group with step() if any |off| is not below `sure`: about one group of 8 tokens x 64 channels in 120 with
    // 4-bit codes.  The clamp here drops a NaN that the reference's keeps: see init.
    // FLOOR: sc_min is below 1e-8 (otherwise s and sc are the same number).
    template <bool FLOOR>
    __device__ __forceinline__ float step_spec(float xv, const Limits &l, float &q, float &off)
    {
        const float d = xv - zp;
        const float r = d * rs;
        const float n = __builtin_rintf(r);
        off = r - n;
        q = __builtin_amdgcn_fmed3f(n, l.ql, l.qu);
        const float xr = q * s;
        const float xh = xr + zp;
        const float ax = al * xr;
        const float e = __builtin_fabsf(q) - tg;
        const float sb = sc * be;
        const float sbe = sb * e;
        zp = zp + ax;
        sc = __builtin_amdgcn_fmed3f(sc + sbe, l.sc_min, l.sc_max);
        s = FLOOR ? __builtin_amdgcn_fmed3f(sc, 1e-8f, __builtin_inff()) : sc;
        rs = __builtin_amdgcn_rcpf(s);
        return xh;
    }
    // GRP tokens; zs, ss: the state before each.
    template <bool FLOOR>
    __device__ __forceinline__ void steps(const float *x, const Limits &l, float *xh, float *q, float *zs, float *ss)
    {
        const Chan saved = *this;
        float off[GRP], worst = 0.0f;
#pragma unroll
        for (int k = 0; k < GRP; k++) {
            zs[k] = zp;
            ss[k] = sc;
            xh[k] = step_spec<FLOOR>(x[k], l, q[k], off[k]);
            if (k & 1)
                worst = collect_abs(worst, off[k - 1], off[k]);
        }
        if (__builtin_expect(__any(!(worst < sure)), 0)) {
            *this = saved;
#pragma unroll
            for (int k = 0; k < GRP; k++) {
                zs[k] = zp;
                ss[k] = sc;
                xh[k] = step(x[k], l, q[k]);
            }
        }
    }
};

constexpr int CH = 32; // tokens per chunk, the unit in which the two waves of a workgroup hand rows over
constexpr int NIN = 3, NOUT = 2;
typedef float Quad __attribute__((ext_vector_type(4))); // four tokens of a channel

// One array of rows a workgroup reads or writes: 64 channels from c0, rows `stride` elements apart.  A lane has four
// channels of rows 4*r0 .. 4*r0+3 of every 16.
// WIDE: whole 4-channel vectors; the array has to be `aligned` and all 64 channels inside the row.
template <typename T, bool WIDE>
struct Rows {
    typedef typename IO<T>::Bits Bits;
    struct alignas(4 * sizeof(Bits)) Vec {
        Bits v[4];
    };
    Bits *base;
    long stride;
    int c, C; // this lane's first channel (of 4)
    uint32_t lane; // bytes from row t of the array to this lane's first in row t + 4*r0 (WIDE)
    __device__ __forceinline__ Rows(void *p, long offset, long stride_, int c0, int C_)
        : stride(stride_), c(c0 + (threadIdx.x & 15) * 4), C(C_)
    {
        base = (Bits *)p + offset;
        lane = ((uint32_t)stride * (((threadIdx.x & 63) >> 4) * 4) + (uint32_t)c) * (uint32_t)sizeof(Bits);
    }
    static __device__ __forceinline__ bool aligned(const void *p, long offset, long stride)
    {
        return ((uintptr_t)p & (sizeof(Vec) - 1)) == 0 && offset % 4 == 0 && stride % 4 == 0 && stride <= 1L << 24;
    }
    // The lane's row k + 4*r0 of a chunk whose first row is at `rows`.
    __device__ __forceinline__ Vec *quad(Bits *rows, int k) const
    {
        return reinterpret_cast<Vec *>(reinterpret_cast<char *>(rows + k * stride) + lane);
    }
    __device__ __forceinline__ void load(long row, Vec &d) const
    {
        const Bits *p = base + row * stride + c;
        if (WIDE) {
            d = *reinterpret_cast<const Vec *>(p);
        } else {
#pragma unroll
            for (int k = 0; k < 4; k++)
                d.v[k] = c + k < C ? p[k] : (Bits)0;
        }
    }
    static __device__ __forceinline__ Vec down(const float4 &f)
    {
        return {{IO<T>::down(f.x), IO<T>::down(f.y), IO<T>::down(f.z), IO<T>::down(f.w)}};
    }
    __device__ __forceinline__ void store(long row, const float4 &f) const
    {
        Bits *p = base + row * stride + c;
        const Vec d = down(f);
        if (WIDE) {
            *reinterpret_cast<Vec *>(p) = d;
        } else {
#pragma unroll
            for (int k = 0; k < 4; k++)
                if (c + k < C)
                    p[k] = d.v[k];
        }
    }
};

// orders LDS accesses across the workgroup's barrier; global accesses in flight are not waited for
__device__ __forceinline__ void hand_over()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Four tokens of a channel lie together: the recurrence reads and writes them in one instruction (an LDS read of
// any width costs a wave that is alone 12 cycles, writes 16, 22 and 34 for one, two and four words).  Position
// p of a row of 64 is channel p%16*4 + p/16, so that the mover, whose lane holds four neighbouring channels,
// reads and writes without bank conflicts as well.
// 40 KB without the optional outputs: four workgroups on a CU
template <bool SEQ, bool CODES>
struct Shared {
    static constexpr int Q = 1, ZP = CODES ? 2 : 1, SC = ZP + 1; // out[0] is xhat
    Quad in[NIN][CH / 4][64];
    Quad out[1 + CODES + 2 * SEQ][NOUT][CH / 4][64];
};

// Chunk i is in `in[i % 3]` from the barrier before phase i-1 on (so the recurrence computes its first
// group before the barrier that ends phase i-1, and writes those results after it); its results are in slot
// i % 2 of the output buffers from the barrier after phase i on.  In phase i the mover
//   writes chunk i+2 (loaded during phase i-1) to the slot chunk i-1 has left,
//   issues the loads of chunk i+3, which have until phase i+2 (a phase is about 1 us) to arrive, and
//   stores the results of chunk i-1.
// Both waves pass nch + 1 barriers.
template <typename T, bool SEQ, bool CODES, bool WIDE>
__device__ __forceinline__ void move_rows(Shared<SEQ, CODES> &sm, const Tensor &a, int b, int c0, int Tn, int C, int nch)
{
    const Rows<T, WIDE> x(const_cast<void *>(a.x), b * a.xs_b, a.xs_t, c0, C);
    const Rows<T, WIDE> xo(a.xhat, b * a.os_b, a.os_t, c0, C);
    const long dense = (long)b * Tn * C; // codes and state sequences are [B, T, C]
    const Rows<float, WIDE> zo(a.zp_seq, dense, C, c0, C), so(a.sc_seq, dense, C, c0, C);
    const int r0 = (threadIdx.x & 63) >> 4, col = (threadIdx.x & 15) * 4; // rows 4*r0.. of every 16, channels col..

    typedef typename Rows<T, WIDE>::Vec Vec;
    typedef uint32_t Raw __attribute__((ext_vector_type(sizeof(Vec) / 4)));
    Vec v[CH / 4];
    // Chunk i, past the end the last row again.
    auto load = [&](int i) __attribute__((always_inline)) {
        if (WIDE && (i + 1) * CH <= Tn) {
#pragma unroll
            for (int j = 0; j < CH / 4; j++)
                v[j] = *x.quad(x.base + i * CH * x.stride, j / 4 * 16 + j % 4);
        } else {
#pragma unroll
            for (int j = 0; j < CH / 4; j++)
                x.load(min(i * CH + j / 4 * 16 + r0 * 4 + j % 4, Tn - 1), v[j]);
        }
    };
    auto fill = [&](int slot) __attribute__((always_inline)) {
        // the rows are waited for here: without this they are put in order, and waited for, as soon as asked for
#pragma unroll
        for (int j = 0; j < CH / 4; j++) {
            Raw raw = __builtin_bit_cast(Raw, v[j]);
            asm volatile("" : "+v"(raw));
            v[j] = __builtin_bit_cast(Vec, raw);
        }
#pragma unroll
        for (int j = 0; j < CH / 4; j += 4)
#pragma unroll
            for (int k = 0; k < 4; k++)
                sm.in[slot][j + r0][k * 16 + (threadIdx.x & 15)] =
                    (Quad){IO<T>::up(v[j].v[k]), IO<T>::up(v[j + 1].v[k]), IO<T>::up(v[j + 2].v[k]), IO<T>::up(v[j + 3].v[k])};
        __builtin_amdgcn_sched_barrier(0);
    };
    // XHAT: a.xhat is there.  FULL: all of the chunk's tokens are.
    auto drain = [&](int i, auto xhat, auto full) __attribute__((always_inline)) {
        constexpr bool FULL = decltype(full)::value;
        const int slot = i & 1;
#pragma unroll
        for (int j = 0; j < CH / 4; j += 4) {
            // rows of four channels from four tokens of each
            auto each_row = [&](int which, auto &&store) __attribute__((always_inline)) {
                Quad f[4];
#pragma unroll
                for (int k = 0; k < 4; k++)
                    f[k] = sm.out[which][slot][j + r0][k * 16 + (threadIdx.x & 15)];
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (FULL || i * CH + (j + r0) * 4 + e < Tn)
                        store(j * 4 + e, make_float4(f[0][e], f[1][e], f[2][e], f[3][e]));
            };
            // into row k + 4*r0 of the chunk
            auto put = [&](auto &rows) {
                return [&](int k, const float4 &f) __attribute__((always_inline)) {
                    if (WIDE)
                        *rows.quad(rows.base + i * CH * rows.stride, k) = rows.down(f);
                    else
                        rows.store(i * CH + k + r0 * 4, f);
                };
            };
            if constexpr (decltype(xhat)::value)
                each_row(0, put(xo));
            if constexpr (SEQ) {
                each_row(sm.ZP, put(zo));
                each_row(sm.SC, put(so));
            }
            if constexpr (CODES)
                each_row(sm.Q, [&](int k, const float4 &f) __attribute__((always_inline)) {
                    auto code = [](float q) { return (q != q) ? (int8_t)0 : (int8_t)q; };
                    const char4 q = make_char4(code(f.x), code(f.y), code(f.z), code(f.w));
                    int8_t *p = a.codes + dense + (long)(i * CH + k + r0 * 4) * C + c0 + col;
                    if (WIDE) {
                        *reinterpret_cast<char4 *>(p) = q;
                    } else {
                        const int8_t kk[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
                        for (int n = 0; n < 4; n++)
                            if (c0 + col + n < C)
                                p[n] = kk[n];
                    }
                });
        }
    };
    // Every phase that repeats has the same loads and stores, a chunk that is not there is loaded as well: where
    // paths with and without them met, more would be waited for than the loads.
    auto phases = [&](auto xhat) __attribute__((always_inline)) {
        load(0);
        fill(0);
        load(1);
        fill(1);
        load(2);
        hand_over();
        fill(2);
        load(3);
        hand_over();
        int slot = 0; // (i + 2) % 3
        auto phase = [&](int i) __attribute__((always_inline)) {
            fill(slot);
            load(i + 3);
            drain(i - 1, xhat, std::true_type());
            slot = slot == 2 ? 0 : slot + 1;
            hand_over();
        };
        if (nch > 1) {
            phase(1);
            for (int i = 2; i < nch; i++)
                phase(i);
        }
        drain(nch - 1, xhat, std::false_type());
    };
    if (a.xhat)
        phases(std::true_type());
    else
        phases(std::false_type());
}

// ~16 instructions per token: 15 of step_spec, a quarter of an LDS read and of an LDS write, half of the check.  The
// chain is the launch: a wave that is alone on its SIMD issues one of them in 4 cycles (the clamps 5, rcp 8, the
// LDS read of four tokens 12, the write 34), 86 cycles or 36 ns per token; with rows read and written two
// tokens at a time, NaNs of the scale looked for in every group and the mover waiting for its loads as it asked
// for them 39.5.  64 blocks x 1024 tokens 45.3 -> 41.9 us, 1024 x 256 in bfloat16 25.4 -> 22.2.
template <bool SEQ, bool CODES, bool FLOOR>
__device__ __forceinline__ void recurrence(Shared<SEQ, CODES> &sm, const Tensor &a, int b, int c0, int Tn, int C, int nch,
                                           Limits l)
{
    const int lane = threadIdx.x & 63;
    const int c = c0 + (lane & 15) * 4 + (lane >> 4);
    Chan ch;
    ch.init(a, b, min(c, C - 1), C, l);
    // med3 takes one scalar operand: the other bound of each pair lives in a vector register
    asm volatile("" : "+v"(l.qu), "+v"(l.sc_max));

    // tokens `row`.. of a chunk: results of GRP tokens into slot `o`
    auto group = [&](const float *x, int row, int o, auto &&before_results) __attribute__((always_inline)) {
        float xh[GRP], q[GRP], zs[GRP], ss[GRP];
        ch.template steps<FLOOR>(x, l, xh, q, zs, ss);
        before_results();
        auto put = [&](int which, const float *f) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < GRP; k += 4)
                sm.out[which][o][(row + k) / 4][lane] = (Quad){f[k], f[k + 1], f[k + 2], f[k + 3]};
        };
        put(0, xh);
        if constexpr (CODES)
            put(sm.Q, q);
        if constexpr (SEQ) {
            put(sm.ZP, zs);
            put(sm.SC, ss);
        }
    };
    auto read = [&](float *x, int slot, int row) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < GRP; k += 4) {
            const Quad f = sm.in[slot][(row + k) / 4][lane];
            x[k] = f.x;
            x[k + 1] = f.y;
            x[k + 2] = f.z;
            x[k + 3] = f.w;
        }
    };

    hand_over();
    const int nfull = Tn / CH;
    float x[2][GRP];
    read(x[0], 0, 0);
    int slot = 0;
    for (int i = 0; i < nfull; i++) {
        const int next = slot == 2 ? 0 : slot + 1;
#pragma unroll
        for (int g = 0; g < CH / GRP; g++) {
            // the next group's rows (past the last chunk: whatever the slot holds, never used)
            read(x[(g + 1) & 1], g + 1 < CH / GRP ? slot : next, (g + 1) * GRP % CH);
            __builtin_amdgcn_sched_barrier(0); // the reads first: they have a group's time
            group(x[g & 1], g * GRP, i & 1, [&]() __attribute__((always_inline)) {
                if (g == 0 && i > 0)
                    hand_over(); // chunk i - 1: its last results are long written by now
            });
        }
        slot = next;
    }
    if (nfull > 0)
        hand_over();
    if (nfull < nch) {
        const int o = nfull & 1, n = Tn - nfull * CH;
        int row = 0;
        for (; row + GRP <= n; row += GRP) {
            read(x[0], slot, row);
            group(x[0], row, o, []() {});
        }
        auto word = [&](Quad (&rows)[CH / 4][64]) -> float & { return reinterpret_cast<float *>(&rows[row / 4][lane])[row % 4]; };
        for (; row < n; row++) {
            if constexpr (SEQ) {
                word(sm.out[sm.ZP][o]) = ch.zp;
                word(sm.out[sm.SC][o]) = ch.sc;
            }
            float q;
            word(sm.out[0][o]) = ch.step(word(sm.in[slot]), l, q);
            if constexpr (CODES)
                word(sm.out[sm.Q][o]) = q;
        }
        hand_over();
    }
    if (a.zp_io && c < C) {
        a.zp_io[(long)b * C + c] = ch.zp;
        a.sc_io[(long)b * C + c] = ch.sc;
    }
}

// grid: (64-channel blocks, batch, tensors)
template <typename T, bool SEQ, bool CODES, bool FLOOR>
__global__ __launch_bounds__(128) void quant_kernel(Tensor a0, Tensor a1, int Tn, int C, Limits l)
{
    __shared__ Shared<SEQ, CODES> sm;
    const Tensor a = blockIdx.z ? a1 : a0;
    const int c0 = blockIdx.x * 64, b = blockIdx.y, nch = (Tn + CH - 1) / CH;
    if (threadIdx.x < 64)
        recurrence<SEQ, CODES, FLOOR>(sm, a, b, c0, Tn, C, nch, l);
    else {
        using R = Rows<T, true>;
        const bool dense_ok = C % 4 == 0 && (((uintptr_t)a.zp_seq | (uintptr_t)a.sc_seq) & 15) == 0 && ((uintptr_t)a.codes & 3) == 0;
        if (c0 + 64 <= C && R::aligned(a.x, b * a.xs_b, a.xs_t) && (!a.xhat || R::aligned(a.xhat, b * a.os_b, a.os_t)) &&
            ((!SEQ && !CODES) || dense_ok))
            move_rows<T, SEQ, CODES, true>(sm, a, b, c0, Tn, C, nch);
        else
            move_rows<T, SEQ, CODES, false>(sm, a, b, c0, Tn, C, nch);
    }
}

constexpr int NBUF = 2; // groups of rows in rotation (3 and 4 were measured: fewer waves fit, 2-10 % slower)

// A lane per channel straight from memory, in groups of GRP tokens.
// SPEC = false: limits that step_spec does not cover, the reference's operations only.
// EXTRA: codes or states are wanted.
template <typename T, bool SPEC, bool EXTRA>
__global__ __launch_bounds__(64) void quant_direct_kernel(Tensor a0, Tensor a1, int Tn, int C, Limits l)
{
    typedef typename IO<T>::Bits Bits;
    const Tensor a = blockIdx.z ? a1 : a0;
    const int c = blockIdx.x * 64 + threadIdx.x, b = blockIdx.y;
    if (c >= C)
        return;
    Chan ch;
    ch.init(a, b, c, C, l);
    const Bits *xp = (const Bits *)a.x + b * a.xs_b + c;
    Bits *op = a.xhat ? (Bits *)a.xhat + b * a.os_b + c : nullptr;
    const long dense = (long)b * Tn * C + c;
    int8_t *cp = a.codes ? a.codes + dense : nullptr;
    float *zq = a.zp_seq ? a.zp_seq + dense : nullptr, *sq = a.zp_seq ? a.sc_seq + dense : nullptr;
    // the next token's results
    auto emit = [&](float xh, float q, float zp, float sc) __attribute__((always_inline)) {
        if (op) {
            *op = IO<T>::down(xh);
            op += a.os_t;
        }
        if (EXTRA && cp) {
            *cp = (q != q) ? (int8_t)0 : (int8_t)q;
            cp += C;
        }
        if (EXTRA && zq) {
            *zq = zp;
            *sq = sc;
            zq += C;
            sq += C;
        }
    };
    const int ng = SPEC ? Tn / GRP : 0;
    Bits buf[NBUF][GRP];
    auto load = [&](int g, Bits *dst) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < GRP; k++)
            dst[k] = xp[(long)(g * GRP + k) * a.xs_t];
    };
    if (ng > 0) {
        adkv::static_for<NBUF - 1>([&](auto ic) { load(min(decltype(ic)::value, ng - 1), buf[decltype(ic)::value]); });
        adkv::rotate_over<NBUF>(ng, [&](int g, auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value;
            // past the last group the same rows again: a condition would make the next wait cover every load
            load(min(g + NBUF - 1, ng - 1), buf[(i + NBUF - 1) % NBUF]);
            float x[GRP], xh[GRP], q[GRP], zs[GRP], ss[GRP];
#pragma unroll
            for (int k = 0; k < GRP; k++)
                x[k] = IO<T>::up(buf[i][k]);
            ch.template steps<true>(x, l, xh, q, zs, ss);
#pragma unroll
            for (int k = 0; k < GRP; k++)
                emit(xh[k], q[k], zs[k], ss[k]);
        });
    }
    for (int t = ng * GRP; t < Tn; t++) {
        const float zp = ch.zp, sc = ch.sc;
        float q;
        const float xh = ch.step(IO<T>::up(xp[t * a.xs_t]), l, q);
        emit(xh, q, zp, sc);
    }
    if (a.zp_io) {
        a.zp_io[(long)b * C + c] = ch.zp;
        a.sc_io[(long)b * C + c] = ch.sc;
    }
}

// Which kernel: quant_kernel while all its workgroups are resident at once (its LDS allows four on a
// CU, two with codes or states, one with both), quant_direct_kernel beyond, where many waves hide what
// quant_kernel moves out of the chain.  us, both kernels, one tensor of
// fp32, 64-channel blocks x tokens, quant_kernel / quant_direct_kernel: 64 x 1024 42 / 121, 512 x 512
// 28 / 66, 1024 x 64 9.5 / 12.1, 1024 x 256 21 / 37; 2048 x 64 20 / 13.0, 8192 x 32 36 / 22.
static int launch(const Tensor *a, int n, int B, int T, int C, int x_dtype, int lower_limit, int upper_limit,
                  float sc_min, float sc_max, hipStream_t st)
{
    for (int i = 0; i < n; i++) {
        if (!a[i].x || !a[i].alpha || !a[i].beta || !a[i].tgt)
            return ADKV_E_NULL;
        if ((a[i].zp_io == nullptr) != (a[i].sc_io == nullptr) || (a[i].zp0 == nullptr) != (a[i].sc0 == nullptr))
            return ADKV_E_NULL;
        if (!a[i].zp_io && !a[i].zp0)
            return ADKV_E_NULL; // no starting state at all
        if ((a[i].zp_seq == nullptr) != (a[i].sc_seq == nullptr))
            return ADKV_E_NULL;
    }
    if (B <= 0 || C <= 0 || T < 0 || B > 65535)
        return ADKV_E_SHAPE;
    for (int i = 0; i < n; i++)
        if (a[i].xs_t < C || a[i].xs_b < 0 || a[i].os_t < C || a[i].os_b < 0)
            return ADKV_E_SHAPE;
    if (lower_limit > 0 || upper_limit < 0 || lower_limit < -128 || upper_limit > 127)
        return ADKV_E_UNSUPPORTED;
    if (x_dtype != ADKV_DT_F32 && x_dtype != ADKV_DT_F16 && x_dtype != ADKV_DT_BF16)
        return ADKV_E_UNSUPPORTED;
    if (T == 0 && !(a[0].zp0 && a[0].zp_io))
        return ADKV_OK;
    const int largest = -lower_limit > upper_limit ? -lower_limit : upper_limit;
    const Limits l = {(float)lower_limit, (float)upper_limit, sc_min, sc_max, 0.5f - (float)(largest + 1) * 0x1p-21f};
    const Tensor &a1 = a[n - 1];
    const dim3 grid((unsigned)((C + 63) / 64), (unsigned)B, (unsigned)n);
    const bool spec = sc_min <= sc_max && sc_max >= 1e-8f && sc_max <= 0x1p100f; // what step_spec relies on
    const bool seq = a[0].zp_seq != nullptr, codes = a[0].codes != nullptr, floored = sc_min < 1e-8f;
    const long resident = adkv::cu_count() * (seq && codes ? 1L : seq || codes ? 2L : 4L);
    const bool direct = (long)grid.x * grid.y * grid.z > resident;
#define ADKV_Q32_K(TYPE, SEQ, CODES, FLOOR)                                                                \
    hipLaunchKernelGGL((quant_kernel<TYPE, SEQ, CODES, FLOOR>), grid, dim3(128), 0, st, a[0], a1, T, C, l)
#define ADKV_Q32_F(TYPE, SEQ, CODES)                                                                       \
    do {                                                                                                   \
        if (floored)                                                                                       \
            ADKV_Q32_K(TYPE, SEQ, CODES, true);                                                            \
        else                                                                                               \
            ADKV_Q32_K(TYPE, SEQ, CODES, false);                                                           \
    } while (0)
#define ADKV_Q32(TYPE)                                                                                     \
    do {                                                                                                   \
        if (T < 2 || !spec)                                                                                \
            hipLaunchKernelGGL((quant_direct_kernel<TYPE, false, true>), grid, dim3(64), 0, st, a[0], a1, T, C, l); \
        else if (direct && (seq || codes))                                                                 \
            hipLaunchKernelGGL((quant_direct_kernel<TYPE, true, true>), grid, dim3(64), 0, st, a[0], a1, T, C, l); \
        else if (direct)                                                                                   \
            hipLaunchKernelGGL((quant_direct_kernel<TYPE, true, false>), grid, dim3(64), 0, st, a[0], a1, T, C, l); \
        else if (seq && codes)                                                                             \
            ADKV_Q32_F(TYPE, true, true);                                                                  \
        else if (seq)                                                                                      \
            ADKV_Q32_F(TYPE, true, false);                                                                 \
        else if (codes)                                                                                    \
            ADKV_Q32_F(TYPE, false, true);                                                                 \
        else                                                                                               \
            ADKV_Q32_F(TYPE, false, false);                                                                \
    } while (0)
    if (x_dtype == ADKV_DT_F32)
        ADKV_Q32(float);
    else if (x_dtype == ADKV_DT_F16)
        ADKV_Q32(_Float16);
    else
        ADKV_Q32(__hip_bfloat16);
#undef ADKV_Q32
#undef ADKV_Q32_F
#undef ADKV_Q32_K
    return adkv::check_launch();
}

} // namespace adkv_fp32

extern "C" int adkv_quant_f32(const void *x, void *xhat, void *codes, void *zp_state, void *sc_state,
                              const void *zp_init, const void *sc_init, const void *alpha,
                              const void *beta, const void *tgt, void *zp_seq, void *sc_seq,
                              int B, int T, int C, int64_t stride_b, int64_t stride_t, int x_dtype,
                              int lower_limit, int upper_limit, float sc_min, float sc_max,
                              void *stream)
{
    const bool free = (x_dtype & ADKV_PARAMS_FREE) != 0;
    if (free && (!zp_init || !sc_init))
        return ADKV_E_NULL;
    const adkv_fp32::Tensor a = {x, xhat, (int8_t *)codes, (float *)zp_state, (float *)sc_state, (const float *)zp_init,
                                 (const float *)sc_init, (const float *)alpha, (const float *)beta, (const float *)tgt,
                                 (float *)zp_seq, (float *)sc_seq, (long)stride_b, (long)stride_t, (long)stride_b,
                                 (long)stride_t, free};
    return adkv_fp32::launch(&a, 1, B, T, C, x_dtype & ~ADKV_PARAMS_FREE, lower_limit, upper_limit, sc_min, sc_max, (hipStream_t)stream);
}

extern "C" int adkv_quant_f32_pair(const void *const *x, const int64_t *x_strides, void *const *xhat,
                                   const int64_t *xhat_strides, void *const *state, const void *const *init,
                                   const void *const *params, int B, int T, int C, int x_dtype, int lower_limit,
                                   int upper_limit, float sc_min, float sc_max, void *stream)
{
    if (!x || !x_strides || !xhat || !xhat_strides || !state || !params)
        return ADKV_E_NULL;
    adkv_fp32::Tensor a[2];
    for (int i = 0; i < 2; i++)
        a[i] = {x[i], xhat[i], nullptr, (float *)state[2 * i], (float *)state[2 * i + 1],
                init ? (const float *)init[2 * i] : nullptr, init ? (const float *)init[2 * i + 1] : nullptr,
                (const float *)params[3 * i], (const float *)params[3 * i + 1], (const float *)params[3 * i + 2],
                nullptr, nullptr, (long)x_strides[2 * i], (long)x_strides[2 * i + 1], (long)xhat_strides[2 * i],
                (long)xhat_strides[2 * i + 1], false};
    return adkv_fp32::launch(a, 2, B, T, C, x_dtype, lower_limit, upper_limit, sc_min, sc_max, (hipStream_t)stream);
}
