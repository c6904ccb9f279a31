// Device-side building blocks of the ADKV kernels (gfx950, wave64).
//
// Arithmetic contract (reference: src/adkv/kernel/gemv.cu:79-88,150-164,220-221): the per-channel
// state (zp, sc) is fp16 and every step below is ONE IEEE round-to-nearest-even fp16 operation, so
// the state trajectory is bit-identical to the reference's half2 code.  This file must be compiled
// with -ffp-contract=off: "q*sc + zp" has to stay two roundings where the reference has two.
#pragma once

#include <hip/hip_runtime.h>
#include <type_traits>
#include <utility>
#include <stdint.h>

#pragma clang fp contract(off)

namespace adkv {

// ADKV_OK, or ADKV_E_LAUNCH with the HIP code kept for adkv_last_hip_error() (host; adkv_kernels.hip)
int check_launch();
int cu_count(); // of the current device (host; adkv_kernels.hip)

typedef _Float16 h1;
typedef _Float16 h2 __attribute__((ext_vector_type(2)));

// operand types of v_mfma_f32_4x4x4_16B_f16: four fp16 (two registers), four fp32
typedef float f4v __attribute__((ext_vector_type(4)));
typedef _Float16 h4v __attribute__((ext_vector_type(4)));
__device__ __forceinline__ h4v as_h4(uint32_t lo, uint32_t hi)
{
    return __builtin_bit_cast(h4v, make_uint2(lo, hi));
}
__device__ __forceinline__ h2 as_h2(uint32_t u) { return __builtin_bit_cast(h2, u); }
__device__ __forceinline__ uint32_t as_u32(h2 h) { return __builtin_bit_cast(uint32_t, h); }
__device__ __forceinline__ h2 pk_fma(h2 a, h2 b, h2 c) { return __builtin_elementwise_fma(a, b, c); }
__device__ __forceinline__ h2 pk_abs(h2 a) { return as_h2(as_u32(a) & 0x7FFF7FFFu); }
__device__ __forceinline__ h2 splat(h1 x) { return (h2){x, x}; }

// f(integral_constant<int, 0>), ..., f(integral_constant<int, N-1>): a loop whose index is a
// compile-time constant inside the body (register arrays indexed by it stay in registers).
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f)
{
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// A decode loop over n items whose buffers rotate with period P: whole rotations without a
// single condition in them (conditions around loads or stores make the compiler wait for every
// load in flight), then the up to P-1 items left.  body(item, integral_constant slot).
template <int P, typename F>
__device__ __forceinline__ void rotate_over(int n, F &&body)
{
    int i0 = 0;
    for (; i0 + P <= n; i0 += P)
        static_for<P>([&](auto ic) { body(i0 + decltype(ic)::value, ic); });
    static_for<P - 1>([&](auto ic) {
        if (i0 + decltype(ic)::value < n)
            body(i0 + decltype(ic)::value, ic);
    });
}

// Activations (q, the new K / V token, the attention output) may be stored as bfloat16 instead of
// fp16: they are rounded to fp16 as they are read (bf16 -> fp32 is exact, fp32 -> fp16 rounds to
// nearest even: torch's .to(float16)) and the fp16 result is rounded to bf16 as it is written
// (torch's .to(bfloat16)), so values are those of the reference's conversions around its kernels
// (src/adkv/hf/llama_adkv.py:248-250, 274).  `bf16` is uniform over the launch.
__device__ __forceinline__ h2 act2(uint32_t w, int bf16)
{
    if (bf16)
        return (h2){(h1)__uint_as_float(w << 16), (h1)__uint_as_float(w & 0xFFFF0000u)};
    return as_h2(w);
}
__device__ __forceinline__ h2 load_act2(const h1 *p, int bf16) { return act2(*reinterpret_cast<const uint32_t *>(p), bf16); }

__device__ __forceinline__ uint32_t bf16_bits(h1 v)
{
    const uint32_t u = __float_as_uint((float)v);
    if ((u & 0x7FFFFFFFu) > 0x7F800000u)
        return (u >> 16) | 0x40u; // NaN stays NaN
    return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
}

__device__ __forceinline__ void store_act2(h1 *p, float a, float b, int bf16)
{
    const h2 v = {(h1)a, (h1)b};
    if (bf16)
        *reinterpret_cast<uint32_t *>(p) = bf16_bits(v.x) | (bf16_bits(v.y) << 16);
    else
        *reinterpret_cast<h2 *>(p) = v;
}

// One channel pair's filter state and fixed parameters (two channels packed per register).
struct Pair {
    h2 zp, sc, al, be, omt;
};

// Loads the pair starting at parameter index pi (even).  omt = 1 - beta*target with both steps
// rounded to fp16 (gemv.cu:220-221).
__device__ __forceinline__ void load_pair(Pair &p, const h1 *zp, const h1 *sc, const h1 *al,
                                          const h1 *be, const h1 *tg, int pi)
{
    p.zp = *reinterpret_cast<const h2 *>(zp + pi);
    p.sc = *reinterpret_cast<const h2 *>(sc + pi);
    p.al = *reinterpret_cast<const h2 *>(al + pi);
    p.be = *reinterpret_cast<const h2 *>(be + pi);
    const h2 t = *reinterpret_cast<const h2 *>(tg + pi);
    const h2 bt = p.be * t;
    p.omt = splat((h1)1.0f) - bt;
}

// EMA update with an already computed qs = r16(q*sc) (gemv.cu:158-164):
//   zp <- r16(alpha*qs + zp)   sc <- r16(sc * r16(beta*|q| + omt))
__device__ __forceinline__ void update_pair(Pair &p, h2 q, h2 qs)
{
    p.zp = pk_fma(p.al, qs, p.zp);
    const h2 f = pk_fma(p.be, pk_abs(q), p.omt);
    p.sc = p.sc * f;
}

// ---------------------------------------------------------------------------------------------
// Code-pair lookup table in LDS.
//
// Decoding a nibble pair in registers costs ~4.5 VALU ops per channel-pair-token (byte permute,
// mask, or, bias subtract, abs) and the scan is VALU-issue-bound, so the conversion is moved to
// the otherwise idle LDS pipe: the byte b = code_A | code_B << 4 of one token indexes a table whose
// entry holds the fp16 pair (q_A, q_B) and its absolute value.  Entry stride is 256 B = 32 copies of
// the 8-byte entry; lane l reads copy l % 32, so the 16 lanes a ds_read_b64 serves per clock always
// hit 16 distinct bank pairs, whatever their codes are.  Address = (b << 8) | (copy << 3) is built
// by ONE v_perm_b32 from the packed code word and a per-lane constant.
// ---------------------------------------------------------------------------------------------
constexpr int LUT_ENTRIES = 256;
constexpr int LUT_COPIES = 32;
constexpr int LUT_WORDS64 = LUT_ENTRIES * LUT_COPIES; // uint2 elements = 64 KB

// nthreads: a multiple of 256.  16 lanes write a row, two copies each; the low nibble of a lane's
// entries never changes and the high one is known once the loop is unrolled.  (An entry per lane and
// iteration, computed from its index, took a 4-wave workgroup 544 instructions per wave, about 1 us.)
template <int NT>
__device__ __forceinline__ void lut_fill(uint2 *lut, int tid)
{
    static_assert(NT % 256 == 0, "whole groups of 256 entries' 16 lanes");
    uint4 *l4 = reinterpret_cast<uint4 *>(lut);
    const uint32_t lo = as_u32((h2){(h1)(((tid >> 4) & 15) - 8), (h1)0.0f});
#pragma unroll
    for (int i = 0; i < LUT_WORDS64 / 2; i += NT) {
        if (LUT_WORDS64 / 2 % NT != 0 && i + tid >= LUT_WORDS64 / 2)
            break;
        const uint32_t hi = as_u32((h2){(h1)0.0f, (h1)(((i + tid) >> 8) - 8)});
        const uint32_t q = lo | hi, a = q & 0x7FFF7FFFu;
        l4[i + tid] = make_uint4(q, a, q, a);
    }
}

// Channel words A, B (8 codes each, token i at bits 4i..4i+3) -> per-token code bytes:
// even.byte[k] = token 2k, odd.byte[k] = token 2k+1, each byte = code_A | code_B << 4.
__device__ __forceinline__ void pair_bytes(uint32_t wa, uint32_t wb, uint32_t &even, uint32_t &odd)
{
    constexpr uint32_t m = 0x0F0F0F0Fu;
    even = (wa & m) | ((wb << 4) & ~m);
    odd = ((wa >> 4) & m) | (wb & ~m);
}

// lane_copy = (lane % 32) * 8.  Returns (q pair, |q| pair) of byte k (0..3) of `bytes`.  k must be
// a compile-time constant after unrolling (the selector becomes a literal).
__device__ __forceinline__ uint2 lut_get(const uint2 *lut, uint32_t bytes, uint32_t lane_copy, int k)
{
    const uint32_t sel = 0x0C0C0000u | ((4u + (uint32_t)k) << 8); // [0, 0, bytes.byte[k], lane_copy.byte[0]]
    const uint32_t addr = __builtin_amdgcn_perm(bytes, lane_copy, sel);
    return *reinterpret_cast<const uint2 *>(reinterpret_cast<const char *>(lut) + addr);
}

// EMA update given qs = r16(q*sc) and |q| (gemv.cu:158-164).
__device__ __forceinline__ void update_pair_abs(Pair &p, h2 qabs, h2 qs)
{
    p.zp = pk_fma(p.al, qs, p.zp);
    const h2 f = pk_fma(p.be, qabs, p.omt);
    p.sc = p.sc * f;
}

// Eight tokens of one channel pair per lane, laid out by hand for a wave that has its SIMD to itself
// (one instruction every 4 cycles, whatever it is, wait states included): q*sc, the next scale, the
// value, the next zero-point and the next token's f, in an order in which no packed result is read by
// the very next instruction, so that no wait state is needed.  x[t] = value of token t.
#define ADKV_REPLAY_TOKEN(Q, VAL)                       \
    "v_pk_mul_f16 %[qs], " Q ", %[sc]\n\t"              \
    "v_pk_mul_f16 %[sc], %[sc], %[f]\n\t"               \
    "v_pk_add_f16 " VAL ", %[qs], %[zp]\n\t"            \
    "v_pk_fma_f16 %[zp], %[al], %[qs], %[zp]\n\t"
#define ADKV_REPLAY_F(A) "v_pk_fma_f16 %[f], %[be], " A ", %[omt]\n\t"
__device__ __forceinline__ void replay_eight(Pair &p, const uint2 *e, uint32_t *x)
{
    uint32_t zp = as_u32(p.zp), sc = as_u32(p.sc), qs, f;
    asm(ADKV_REPLAY_F("%[a0]") ADKV_REPLAY_TOKEN("%[q0]", "%[x0]") ADKV_REPLAY_F("%[a1]") ADKV_REPLAY_TOKEN("%[q1]", "%[x1]")
        ADKV_REPLAY_F("%[a2]") ADKV_REPLAY_TOKEN("%[q2]", "%[x2]") ADKV_REPLAY_F("%[a3]") ADKV_REPLAY_TOKEN("%[q3]", "%[x3]")
        ADKV_REPLAY_F("%[a4]") ADKV_REPLAY_TOKEN("%[q4]", "%[x4]") ADKV_REPLAY_F("%[a5]") ADKV_REPLAY_TOKEN("%[q5]", "%[x5]")
        ADKV_REPLAY_F("%[a6]") ADKV_REPLAY_TOKEN("%[q6]", "%[x6]") ADKV_REPLAY_F("%[a7]") ADKV_REPLAY_TOKEN("%[q7]", "%[x7]")
        "s_nop 0"
        : [zp] "+v"(zp), [sc] "+v"(sc), [qs] "=&v"(qs), [f] "=&v"(f), [x0] "=&v"(x[0]), [x1] "=&v"(x[1]), [x2] "=&v"(x[2]),
          [x3] "=&v"(x[3]), [x4] "=&v"(x[4]), [x5] "=&v"(x[5]), [x6] "=&v"(x[6]), [x7] "=&v"(x[7])
        : [q0] "v"(e[0].x), [q1] "v"(e[1].x), [q2] "v"(e[2].x), [q3] "v"(e[3].x), [q4] "v"(e[4].x), [q5] "v"(e[5].x),
          [q6] "v"(e[6].x), [q7] "v"(e[7].x), [a0] "v"(e[0].y), [a1] "v"(e[1].y), [a2] "v"(e[2].y), [a3] "v"(e[3].y),
          [a4] "v"(e[4].y), [a5] "v"(e[5].y), [a6] "v"(e[6].y), [a7] "v"(e[7].y), [al] "v"(as_u32(p.al)),
          [be] "v"(as_u32(p.be)), [omt] "v"(as_u32(p.omt)));
    p.zp = as_h2(zp);
    p.sc = as_h2(sc);
}
// The same, each value multiplied by its token's weight (two per word of w) and added to acc in fp32.
#define ADKV_REPLAY_ADD(W, HI)                                                            \
    "v_fma_mix_f32 %[c0], " W ", %[x], %[c0] op_sel:[" HI ",0,0] op_sel_hi:[1,1,0]\n\t"   \
    "v_fma_mix_f32 %[c1], " W ", %[x], %[c1] op_sel:[" HI ",1,0] op_sel_hi:[1,1,0]\n\t"
#define ADKV_REPLAY_TWO(Q0, Q1, A1, A2, W)                                                            \
    ADKV_REPLAY_TOKEN(Q0, "%[x]") ADKV_REPLAY_F(A1) ADKV_REPLAY_ADD(W, "0")                           \
    ADKV_REPLAY_TOKEN(Q1, "%[x]") ADKV_REPLAY_F(A2) ADKV_REPLAY_ADD(W, "1")
__device__ __forceinline__ void replay_eight_weighted(Pair &p, const uint2 *e, const uint4 &w, float *acc)
{
    uint32_t zp = as_u32(p.zp), sc = as_u32(p.sc), qs, f, x;
    asm(ADKV_REPLAY_F("%[a0]") ADKV_REPLAY_TWO("%[q0]", "%[q1]", "%[a1]", "%[a2]", "%[w0]")
        ADKV_REPLAY_TWO("%[q2]", "%[q3]", "%[a3]", "%[a4]", "%[w1]") ADKV_REPLAY_TWO("%[q4]", "%[q5]", "%[a5]", "%[a6]", "%[w2]")
        ADKV_REPLAY_TOKEN("%[q6]", "%[x]") ADKV_REPLAY_F("%[a7]") ADKV_REPLAY_ADD("%[w3]", "0")
        ADKV_REPLAY_TOKEN("%[q7]", "%[x]") ADKV_REPLAY_ADD("%[w3]", "1")
        : [zp] "+v"(zp), [sc] "+v"(sc), [qs] "=&v"(qs), [f] "=&v"(f), [x] "=&v"(x), [c0] "+v"(acc[0]), [c1] "+v"(acc[1])
        : [q0] "v"(e[0].x), [q1] "v"(e[1].x), [q2] "v"(e[2].x), [q3] "v"(e[3].x), [q4] "v"(e[4].x), [q5] "v"(e[5].x),
          [q6] "v"(e[6].x), [q7] "v"(e[7].x), [a0] "v"(e[0].y), [a1] "v"(e[1].y), [a2] "v"(e[2].y), [a3] "v"(e[3].y),
          [a4] "v"(e[4].y), [a5] "v"(e[5].y), [a6] "v"(e[6].y), [a7] "v"(e[7].y), [w0] "v"(w.x), [w1] "v"(w.y),
          [w2] "v"(w.z), [w3] "v"(w.w), [al] "v"(as_u32(p.al)), [be] "v"(as_u32(p.be)), [omt] "v"(as_u32(p.omt)));
    p.zp = as_h2(zp);
    p.sc = as_h2(sc);
}
#undef ADKV_REPLAY_TWO
#undef ADKV_REPLAY_ADD
#undef ADKV_REPLAY_F
#undef ADKV_REPLAY_TOKEN

// ---------------------------------------------------------------------------------------------
// One channel per lane: both halves of the packed instructions work for the same channel.  The table is indexed by a
// byte of the channel's word as it is (two tokens, the earlier one in the low nibble) and returns (q, |q|) of each, so
// no bytes are merged and one LDS read serves two tokens.  With f = be*|q| + omt beside q, one packed multiply gives the
// code's value q*sc and the next scale sc*f, and one packed fma by (al, 1) the next zero-point and the token's
// value: three packed instructions per token and channel, the arithmetic of update_pair bit for bit (a product by one
// and a sum with zero are exact).
// ---------------------------------------------------------------------------------------------
struct Lone {
    uint32_t z;  // low half: the zero-point; high half: the last token's value
    uint32_t r;  // high half: the scale; low half: the last token's q*sc
    uint32_t ca; // (al, 1)
    uint32_t cf; // (1, be)
    uint32_t c0; // (0, omt)
};
__device__ __forceinline__ h1 lone_zp(const Lone &s) { return as_h2(s.z).x; }
__device__ __forceinline__ h1 lone_sc(const Lone &s) { return as_h2(s.r).y; }

template <int NT>
__device__ __forceinline__ void lone_fill(uint2 *lut, int tid)
{
    static_assert(NT % 256 == 0, "whole groups of 256 entries' 16 lanes");
    uint4 *l4 = reinterpret_cast<uint4 *>(lut);
    const h1 lo = (h1)(((tid >> 4) & 15) - 8);
    const uint32_t x = as_u32(splat(lo)) & 0x7FFFFFFFu;
#pragma unroll
    for (int i = 0; i < LUT_WORDS64 / 2; i += NT) {
        if (LUT_WORDS64 / 2 % NT != 0 && i + tid >= LUT_WORDS64 / 2)
            break;
        const uint32_t y = as_u32(splat((h1)(((i + tid) >> 8) - 8))) & 0x7FFFFFFFu;
        l4[i + tid] = make_uint4(x, y, x, y);
    }
}

// Eight tokens, entries e[0..3] of two tokens each; x[k] = the values of tokens 2k and 2k + 1.  As in replay_eight no
// packed result is read by the very next instruction.  TO_MATRIX: the next one may be a matrix instruction that reads x,
// two states later; the wait is the block's own (as a statement behind the block the compiler put it in front of it).
#define ADKV_LONE_F(E) "v_pk_fma_f16 %[f], " E ", %[cf], %[c0]\n\t"
#define ADKV_LONE_R "v_pk_mul_f16 %[r], %[f], %[r] op_sel:[0,1] op_sel_hi:[1,1]\n\t"
#define ADKV_LONE_Z(TO, FROM) "v_pk_fma_f16 " TO ", %[r], %[ca], " FROM " op_sel_hi:[0,1,0]\n\t"
#define ADKV_LONE_P(X) "v_perm_b32 " X ", %[z], " X ", %[hi]\n\t"
#define ADKV_LONE_EIGHT(END)                                                                                                \
    asm(ADKV_LONE_F("%[a0]") "s_nop 0\n\t"                                                                                  \
        ADKV_LONE_R ADKV_LONE_F("%[b0]") ADKV_LONE_Z("%[x0]", "%[z]")                                                       \
        ADKV_LONE_R ADKV_LONE_F("%[a1]") ADKV_LONE_Z("%[z]", "%[x0]")                                                       \
        ADKV_LONE_R ADKV_LONE_F("%[b1]") ADKV_LONE_Z("%[x1]", "%[z]")                                                       \
        ADKV_LONE_R ADKV_LONE_F("%[a2]") ADKV_LONE_P("%[x0]") ADKV_LONE_Z("%[z]", "%[x1]")                                  \
        ADKV_LONE_R ADKV_LONE_F("%[b2]") ADKV_LONE_Z("%[x2]", "%[z]")                                                       \
        ADKV_LONE_R ADKV_LONE_F("%[a3]") ADKV_LONE_P("%[x1]") ADKV_LONE_Z("%[z]", "%[x2]")                                  \
        ADKV_LONE_R ADKV_LONE_F("%[b3]") ADKV_LONE_Z("%[x3]", "%[z]")                                                       \
        ADKV_LONE_R ADKV_LONE_P("%[x2]") ADKV_LONE_Z("%[z]", "%[x3]")                                                       \
        "s_nop 0\n\t" ADKV_LONE_P("%[x3]") END                                                                              \
        : [z] "+v"(s.z), [r] "+v"(s.r), [f] "=&v"(f), [x0] "=&v"(x[0]), [x1] "=&v"(x[1]), [x2] "=&v"(x[2]), [x3] "=&v"(x[3])\
        : [a0] "v"(e[0].x), [b0] "v"(e[0].y), [a1] "v"(e[1].x), [b1] "v"(e[1].y), [a2] "v"(e[2].x), [b2] "v"(e[2].y),       \
          [a3] "v"(e[3].x), [b3] "v"(e[3].y), [ca] "v"(s.ca), [cf] "v"(s.cf), [c0] "v"(s.c0), [hi] "s"(0x07060302u))
template <bool TO_MATRIX = false>
__device__ __forceinline__ void lone_eight(Lone &s, const uint2 *e, uint32_t *x)
{
    uint32_t f;
    if constexpr (TO_MATRIX)
        ADKV_LONE_EIGHT("s_nop 1");
    else
        ADKV_LONE_EIGHT("");
}
// The same, each value multiplied by its token's weight (two per word of w) and added to acc in fp32.
#define ADKV_LONE_M(W, HI) "v_fma_mix_f32 %[c], " W ", %[z], %[c] op_sel:[" HI ",1,0] op_sel_hi:[1,1,0]\n\t"
#define ADKV_LONE_TOKEN(NEXT, ADD) ADKV_LONE_R NEXT ADD ADKV_LONE_Z("%[z]", "%[z]")
__device__ __forceinline__ void lone_eight_weighted(Lone &s, const uint2 *e, const uint4 &w, float &acc)
{
    uint32_t f;
    asm(ADKV_LONE_F("%[a0]") "s_nop 0\n\t"
        ADKV_LONE_TOKEN(ADKV_LONE_F("%[b0]"), "")
        ADKV_LONE_TOKEN(ADKV_LONE_F("%[a1]"), ADKV_LONE_M("%[w0]", "0"))
        ADKV_LONE_TOKEN(ADKV_LONE_F("%[b1]"), ADKV_LONE_M("%[w0]", "1"))
        ADKV_LONE_TOKEN(ADKV_LONE_F("%[a2]"), ADKV_LONE_M("%[w1]", "0"))
        ADKV_LONE_TOKEN(ADKV_LONE_F("%[b2]"), ADKV_LONE_M("%[w1]", "1"))
        ADKV_LONE_TOKEN(ADKV_LONE_F("%[a3]"), ADKV_LONE_M("%[w2]", "0"))
        ADKV_LONE_TOKEN(ADKV_LONE_F("%[b3]"), ADKV_LONE_M("%[w2]", "1"))
        ADKV_LONE_TOKEN("", ADKV_LONE_M("%[w3]", "0"))
        "s_nop 0\n\t" ADKV_LONE_M("%[w3]", "1")
        : [z] "+v"(s.z), [r] "+v"(s.r), [f] "=&v"(f), [c] "+v"(acc)
        : [a0] "v"(e[0].x), [b0] "v"(e[0].y), [a1] "v"(e[1].x), [b1] "v"(e[1].y), [a2] "v"(e[2].x), [b2] "v"(e[2].y),
          [a3] "v"(e[3].x), [b3] "v"(e[3].y), [w0] "v"(w.x), [w1] "v"(w.y), [w2] "v"(w.z), [w3] "v"(w.w), [ca] "v"(s.ca),
          [cf] "v"(s.cf), [c0] "v"(s.c0));
}
#undef ADKV_LONE_TOKEN
#undef ADKV_LONE_M
#undef ADKV_LONE_EIGHT
#undef ADKV_LONE_P
#undef ADKV_LONE_Z
#undef ADKV_LONE_R
#undef ADKV_LONE_F

// One token with code q (ragged tails): returns its value.
__device__ __forceinline__ h1 lone_token(Lone &s, int q)
{
    const h1 qh = (h1)q, qs = qh * lone_sc(s), v = qs + lone_zp(s);
    const h1 f = __builtin_fmaf16(as_h2(s.cf).y, (h1)(q < 0 ? -q : q), as_h2(s.c0).y);
    const h1 zp = __builtin_fmaf16(as_h2(s.ca).x, qs, lone_zp(s)), sc = lone_sc(s) * f;
    s.z = as_u32((h2){zp, v});
    s.r = as_u32((h2){qs, sc});
    return v;
}

// Code width.  4 bits is the reference's format (8 tokens per 32-bit channel word, codes in
// [-8, 7], stored as q + 8).  2 bits is the same recurrence over codes in [-2, 1] (the range the
// reference's train model uses for bits = 2, train_model.py:96-97), stored as q + 2, 16 tokens per
// word; the reference has no kernel for it.
template <int BITS>
struct Code {
    static_assert(BITS == 2 || BITS == 4, "code width");
    static constexpr int TPW = 32 / BITS;                 // tokens per channel word = per supergroup
    static constexpr int QLO = -(1 << (BITS - 1));
    static constexpr int QHI = (1 << (BITS - 1)) - 1;
    static constexpr uint32_t FIELD = (1u << BITS) - 1u;
    static constexpr uint32_t BIAS = BITS == 4 ? 0x88888888u : 0xAAAAAAAAu; // -QLO in every field
};

// gemv.cu:150-154: fp32 subtract, IEEE fp32 divide, round-half-even, NaN -> 0, clamp to [-8,7].
template <int BITS = 4>
__device__ __forceinline__ int quantize(h1 x, h1 zp, h1 sc)
{
    const float d = (float)x - (float)zp;
    const float u = d / (float)sc;
    float r = __builtin_rintf(u);
    r = (u != u) ? 0.0f : r;
    r = __builtin_fminf(__builtin_fmaxf(r, (float)Code<BITS>::QLO), (float)Code<BITS>::QHI);
    return (int)r;
}

// The encoder's fast form of quantize(): x - zp is one mixed-precision fma on the fp16 halves in
// place (f32(x)*1 - f32(zp), rounded once: exactly the reference's fp32 difference) instead of two
// conversions and a subtract.
template <bool HI>
__device__ __forceinline__ float enc_diff(uint32_t xw, uint32_t zpw)
{
    float d;
    if (HI)
        asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[1,0,1] op_sel_hi:[1,0,1]" : "=v"(d) : "v"(xw), "v"(zpw));
    else
        asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel_hi:[1,0,1]" : "=v"(d) : "v"(xw), "v"(zpw));
    return d;
}
// The IEEE fp32 quotient d / s for d a difference of two fp16 numbers and s an fp16 number, from
// rs = v_rcp_f32(s) (1 ulp).  q = d*rs is within an ulp or so of the quotient, rem = d - q*s is then
// exact, and q + rem*rs = (d/s)(1 + 2^-46) before its one rounding.  That rounds like d/s itself:
// s has 11 significant bits, so a d/s that is not the midpoint of two fp32 neighbours differs from
// every midpoint (25 bits) by at least 2^-37 of itself, and it cannot be a midpoint, whose product
// with s needs 25 bits or more where d has 24.  Neither overflow nor underflow can occur (|d| from
// 2^-24 to 2^17, |s| from 2^-24 to 2^16).  For s = 0 or a non-finite operand the result is a NaN.
__device__ __forceinline__ float enc_quotient(float d, float s, float rs)
{
    const float q = d * rs;
    const float rem = __builtin_fmaf(-q, s, d);
    return __builtin_fmaf(rem, rs, q);
}
// NaN once any of its operands is (the others only have to be there)
__device__ __forceinline__ float enc_collect_nan(float acc, float a, float b)
{
    float r;
    asm("v_maximum3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(acc), "v"(a), "v"(b));
    return r;
}

// Eight tokens of one channel per lane, 14 instructions each (16 issue slots: v_fma_f16 and v_rcp_f32
// take two) and laid out by hand.  The state keeps the scale in the HIGH half of qs_sc, so that one
// packed multiply by (code, f) gives both the code's value q*sc (low) and the next scale sc*f
// (high); f = be*|q| + omt is written by v_fma_f16 into the high half of the register that holds q.
// Waits the hardware does not make by itself, filled with useful instructions where there is one:
// a packed or half-register result is not read by the next instruction, nor is v_rcp_f32's.  The block
// cannot see what follows it, so a token begins with the reciprocal of the scale and ends with the
// conversion of the next one, whose result needs no wait (with the reciprocal last and an s_nop behind it,
// 32768 tokens of 8 x 32 heads took 1281 us instead of 1267).
struct Chan1 {
    uint32_t zp;    // low half; the high half is never read
    uint32_t qs_sc; // high half: the scale
    float s;        // the scale in fp32
};
template <int BITS>
__device__ __forceinline__ void enc_eight_tokens(Chan1 &c, const uint16_t *x, uint32_t al, uint32_t be, uint32_t omt,
                                                 float lo, float hi, uint32_t &word, float &nan)
{
    float d, r0, r1, t, rs;
    uint32_t u, q;
#define ADKV_ENC_TOKEN(X, R, FILL)                                                                       \
    "v_rcp_f32 %[rs], %[s]\n\t"                                                                          \
    "v_fma_mix_f32 %[d], " X ", 1.0, -%[zp] op_sel_hi:[1,0,1]\n\t"                                       \
    "v_mul_f32 " R ", %[d], %[rs]\n\t"                                                                  \
    "v_fma_mix_f32 %[t], -" R ", %[ss], %[d] op_sel:[0,1,0] op_sel_hi:[0,1,0]\n\t"                      \
    "v_fmac_f32 " R ", %[t], %[rs]\n\t"                                                                 \
    "v_add_f32 %[u], 0x4b400000, " R "\n\t"                                                             \
    "v_med3_f32 %[u], %[u], %[lo], %[hi]\n\t"                                                           \
    "v_cvt_f16_i16 %[q], %[u]\n\t"                                                                      \
    "v_fma_f16 %[q], %[be], |%[q]|, %[omt] op_sel:[0,0,0,1]\n\t"                                        \
    "v_alignbit_b32 %[w], %[u], %[w], %[bits]\n\t"                                                      \
    "v_pk_mul_f16 %[ss], %[ss], %[q] op_sel:[1,0] op_sel_hi:[1,1]\n\t"                                  \
    FILL "\n\t"                                                                                         \
    "v_pk_fma_f16 %[zp], %[al], %[ss], %[zp]\n\t"                                                       \
    "v_cvt_f32_f16_sdwa %[s], %[ss] dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:WORD_1\n\t"
#define ADKV_ENC_PAIR(X0, X1)                       \
    ADKV_ENC_TOKEN(X0, "%[r0]", "s_nop 0")         \
    ADKV_ENC_TOKEN(X1, "%[r1]", "v_maximum3_f32 %[nan], %[nan], %[r0], %[r1]")
    asm(ADKV_ENC_PAIR("%[x0]", "%[x1]") ADKV_ENC_PAIR("%[x2]", "%[x3]") ADKV_ENC_PAIR("%[x4]", "%[x5]") ADKV_ENC_PAIR("%[x6]", "%[x7]")
        : [zp] "+v"(c.zp), [ss] "+v"(c.qs_sc), [s] "+v"(c.s), [w] "+v"(word), [nan] "+v"(nan), [d] "=&v"(d), [t] "=&v"(t),
          [rs] "=&v"(rs), [u] "=&v"(u), [q] "=&v"(q), [r0] "=&v"(r0), [r1] "=&v"(r1)
        : [x0] "v"(x[0]), [x1] "v"(x[1]), [x2] "v"(x[2]), [x3] "v"(x[3]), [x4] "v"(x[4]), [x5] "v"(x[5]), [x6] "v"(x[6]),
          [x7] "v"(x[7]), [al] "v"(al), [be] "v"(be), [omt] "v"(omt), [lo] "s"(lo), [hi] "v"(hi), [bits] "n"(BITS));
#undef ADKV_ENC_PAIR
#undef ADKV_ENC_TOKEN
}

// Sixty-four tokens of one channel per lane, their rows in LDS: eight groups of eight rows of 64 channels,
// 1 KB each from `addr` on.  ds_read_b64_tr_b16 hands every lane four tokens of its own channel (16 lanes read
// four rows of 16 channels), two of them instead of eight narrow loads per group: a wave alone on its SIMD pays 12
// cycles for any LDS read and 16 to 18 for any load from memory, against 4 or 5 for an arithmetic
// instruction.  The reads of a group go out before the arithmetic of the one before it and are waited for
// behind it, all inside one block, so that no register is handed over before its data is there.
// The token is that of enc_eight_tokens with the scale kept NEGATED, in the low half of ss and in fp32
// (nsc), and alpha negated with it: the remainder is then a plain multiply-add into d, and the conversion
// of the next scale needs no half selected.  Negation is exact and products of two negated factors are the
// same, NaNs aside; a run in which a quotient or the state it ends in is a NaN is done again (collect nsc and
// zp behind the block).
struct Chan1Neg {
    uint32_t zp;  // low half; the high half is never read
    uint32_t ss;  // low half: minus the scale
    float nsc;    // minus the scale in fp32
};
#define ADKV_RUN_TOKEN(X, SEL, R, FILL, W)                                                               \
    "v_rcp_f32_e64 %[rs], -%[ns]\n\t"                                                                    \
    "v_fma_mix_f32 %[d], " X ", 1.0, -%[zp] op_sel:[" SEL ",0,0] op_sel_hi:[1,0,1]\n\t"                  \
    "v_mul_f32 " R ", %[d], %[rs]\n\t"                                                                   \
    "v_fmac_f32 %[d], " R ", %[ns]\n\t"                                                                  \
    "v_fmac_f32 " R ", %[d], %[rs]\n\t"                                                                  \
    "v_add_f32 %[u], %[magic], " R "\n\t"                                                                \
    "v_med3_f32 %[u], %[u], %[lo], %[hi]\n\t"                                                            \
    "v_cvt_f16_i16 %[q], %[u]\n\t"                                                                       \
    "v_fma_f16 %[q], %[be], |%[q]|, %[omt] op_sel:[0,0,0,1]\n\t"                                         \
    "v_alignbit_b32 " W ", %[u], " W ", %[bits]\n\t"                                                     \
    "v_pk_mul_f16 %[ss], %[ss], %[q] op_sel:[0,1] op_sel_hi:[0,0]\n\t"                                   \
    FILL "\n\t"                                                                                          \
    "v_pk_fma_f16 %[zp], %[nal], %[ss], %[zp] op_sel:[0,1,0]\n\t"                                        \
    "v_cvt_f32_f16 %[ns], %[ss]\n\t"
#define ADKV_RUN_PAIR(X, W)                                                                              \
    ADKV_RUN_TOKEN(X, "0", "%[r0]", "s_nop 0", W)                                                        \
    ADKV_RUN_TOKEN(X, "1", "%[r1]", "v_maximum3_f32 %[nan], %[nan], %[r0], %[r1]", W)
// bfloat16 pairs become fp16 pairs (nearest even) where they are
#define ADKV_RUN_BF16(X)                                                                                 \
    "v_lshlrev_b32 %[r0], 16, " X "\n\t"                                                                 \
    "v_and_b32 %[r1], %[mask], " X "\n\t"                                                                \
    "v_cvt_pk_f16_f32 " X ", %[r0], %[r1]\n\t"
#define ADKV_RUN_F16(X) ""
#define ADKV_RUN_READ(A, B, OFF0, OFF1)                                                                  \
    "ds_read_b64_tr_b16 " A ", %[addr] offset:" OFF0 "\n\t"                                              \
    "ds_read_b64_tr_b16 " B ", %[addr] offset:" OFF1 "\n\t"
// (the pairs of the next two tokens are converted a pair ahead: a packed result is not read by the next instruction)
#define ADKV_RUN_GROUP(C, X0, X1, X2, X3, NEXT, W)                                                       \
    "s_waitcnt lgkmcnt(0)\n\t" NEXT C(X0) C(X1) ADKV_RUN_PAIR(X0, W) C(X2) ADKV_RUN_PAIR(X1, W)          \
    C(X3) ADKV_RUN_PAIR(X2, W) ADKV_RUN_PAIR(X3, W)
#define ADKV_RUN_A(C, NEXT, W) ADKV_RUN_GROUP(C, "v48", "v49", "v50", "v51", NEXT, W)
#define ADKV_RUN_B(C, NEXT, W) ADKV_RUN_GROUP(C, "v52", "v53", "v54", "v55", NEXT, W)
#define ADKV_RUN_INTO_A(OFF0, OFF1) ADKV_RUN_READ("v[48:49]", "v[50:51]", OFF0, OFF1)
#define ADKV_RUN_INTO_B(OFF0, OFF1) ADKV_RUN_READ("v[52:53]", "v[54:55]", OFF0, OFF1)
#define ADKV_RUN_ALL(C, W0, W1, W2, W3, W4, W5, W6, W7)                                                  \
    ADKV_RUN_INTO_A("0", "512")                                                                          \
    ADKV_RUN_A(C, ADKV_RUN_INTO_B("1024", "1536"), W0) ADKV_RUN_B(C, ADKV_RUN_INTO_A("2048", "2560"), W1) \
    ADKV_RUN_A(C, ADKV_RUN_INTO_B("3072", "3584"), W2) ADKV_RUN_B(C, ADKV_RUN_INTO_A("4096", "4608"), W3) \
    ADKV_RUN_A(C, ADKV_RUN_INTO_B("5120", "5632"), W4) ADKV_RUN_B(C, ADKV_RUN_INTO_A("6144", "6656"), W5) \
    ADKV_RUN_A(C, ADKV_RUN_INTO_B("7168", "7680"), W6) ADKV_RUN_B(C, "", W7)
#define ADKV_RUN_OPERANDS                                                                                \
        : [zp] "+v"(c.zp), [ss] "+v"(c.ss), [ns] "+v"(c.nsc), [nan] "+v"(nan), [d] "=&v"(d), [rs] "=&v"(rs), [u] "=&v"(u), \
          [q] "=&v"(q), [r0] "=&v"(r0), [r1] "=&v"(r1), [w0] "=&v"(w[0]), [w1] "=&v"(w[1]), [w2] "=&v"(w[2]), [w3] "=&v"(w[3])
#define ADKV_RUN_INPUTS                                                                                  \
        : [addr] "v"(addr), [nal] "v"(nal), [be] "v"(be), [omt] "v"(omt), [lo] "s"(lo), [hi] "v"(hi), [magic] "s"(magic), \
          [mask] "s"(0xFFFF0000u), [bits] "n"(BITS)                                                      \
        : "v48", "v49", "v50", "v51", "v52", "v53", "v54", "v55", "memory"
#define ADKV_RUN_EIGHT_WORDS , [w4] "=&v"(w[4]), [w5] "=&v"(w[5]), [w6] "=&v"(w[6]), [w7] "=&v"(w[7])
#define ADKV_RUN_4BIT(C) ADKV_RUN_ALL(C, "%[w0]", "%[w1]", "%[w2]", "%[w3]", "%[w4]", "%[w5]", "%[w6]", "%[w7]")
#define ADKV_RUN_2BIT(C) ADKV_RUN_ALL(C, "%[w0]", "%[w0]", "%[w1]", "%[w1]", "%[w2]", "%[w2]", "%[w3]", "%[w3]")
template <int BITS, bool BF16>
__device__ __forceinline__ void enc_run64(Chan1Neg &c, uint32_t addr, uint32_t nal, uint32_t be, uint32_t omt, float magic,
                                          float lo, float hi, uint32_t *w, float &nan)
{
    float d, r0, r1, rs;
    uint32_t u, q;
    if constexpr (BITS == 4 && BF16)
        asm volatile(ADKV_RUN_4BIT(ADKV_RUN_BF16) ADKV_RUN_OPERANDS ADKV_RUN_EIGHT_WORDS ADKV_RUN_INPUTS);
    else if constexpr (BITS == 4)
        asm volatile(ADKV_RUN_4BIT(ADKV_RUN_F16) ADKV_RUN_OPERANDS ADKV_RUN_EIGHT_WORDS ADKV_RUN_INPUTS);
    else if constexpr (BF16)
        asm volatile(ADKV_RUN_2BIT(ADKV_RUN_BF16) ADKV_RUN_OPERANDS ADKV_RUN_INPUTS);
    else
        asm volatile(ADKV_RUN_2BIT(ADKV_RUN_F16) ADKV_RUN_OPERANDS ADKV_RUN_INPUTS);
}
#undef ADKV_RUN_2BIT
#undef ADKV_RUN_4BIT
#undef ADKV_RUN_EIGHT_WORDS
#undef ADKV_RUN_INPUTS
#undef ADKV_RUN_OPERANDS
#undef ADKV_RUN_ALL
#undef ADKV_RUN_INTO_B
#undef ADKV_RUN_INTO_A
#undef ADKV_RUN_B
#undef ADKV_RUN_A
#undef ADKV_RUN_GROUP
#undef ADKV_RUN_READ
#undef ADKV_RUN_F16
#undef ADKV_RUN_BF16
#undef ADKV_RUN_PAIR
#undef ADKV_RUN_TOKEN

// 64 lanes x 16 bytes from memory into 1 KB of LDS at `lds` (wave-uniform), without a register in between.
// Counted by vmcnt like any load; the compiler does not know what it writes.
typedef uint32_t rsrc4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void load_to_lds(uint32_t lds, uint32_t offset, rsrc4 buffer)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds), "v"(offset), "s"(buffer)
                 : "memory"); // m0 is set before every use, by the compiler too
}

__device__ __forceinline__ h2 codes_to_h2(int q0, int q1) { return (h2){(h1)q0, (h1)q1}; }

// Quantise one new token's channel pair with the current state and patch its two codes into the
// channel words at token slot tt of the supergroup (gemv.cu:91-146).  Returns the code pair.
template <int BITS = 4>
__device__ __forceinline__ h2 append_pair(uint32_t &wa, uint32_t &wb, int tt, h2 x, const Pair &p)
{
    const int q0 = quantize<BITS>(x.x, p.zp.x, p.sc.x);
    const int q1 = quantize<BITS>(x.y, p.zp.y, p.sc.y);
    const uint32_t sh = (uint32_t)BITS * (uint32_t)tt;
    const uint32_t m = ~(Code<BITS>::FIELD << sh);
    wa = (wa & m) | (((uint32_t)(q0 - Code<BITS>::QLO) & Code<BITS>::FIELD) << sh);
    wb = (wb & m) | (((uint32_t)(q1 - Code<BITS>::QLO) & Code<BITS>::FIELD) << sh);
    return codes_to_h2(q0, q1);
}

// Code pair of token slot tt straight from the channel words (ragged tails only).
template <int BITS>
__device__ __forceinline__ h2 extract_pair(uint32_t wa, uint32_t wb, int tt)
{
    const uint32_t sh = (uint32_t)BITS * (uint32_t)tt;
    return codes_to_h2((int)((wa >> sh) & Code<BITS>::FIELD) + Code<BITS>::QLO,
                       (int)((wb >> sh) & Code<BITS>::FIELD) + Code<BITS>::QLO);
}

// ---------------------------------------------------------------------------------------------
// 2-bit codes: the table is indexed by a byte that holds TWO tokens of a channel pair and returns
// 16 bytes, (q, |q|) for the low nibble's token then for the high nibble's.  16 copies per entry
// (256-byte stride again, same 64 KB): a ds_read_b128 serves 16 lanes per clock.
//   even.byte[j] = tokens 4j (low nibble) and 4j+2;  odd.byte[j] = tokens 4j+1 and 4j+3;
//   nibble = code_A | code_B << 2.
// ---------------------------------------------------------------------------------------------
constexpr int LUT2_COPIES = 16;

__device__ __forceinline__ void lut2_fill(uint2 *lut, int tid, int nthreads)
{
    uint4 *l4 = reinterpret_cast<uint4 *>(lut);
    for (int i = tid; i < LUT_ENTRIES * LUT2_COPIES; i += nthreads) {
        const int b = i / LUT2_COPIES;
        const h2 lo = (h2){(h1)((b & 3) - 2), (h1)(((b >> 2) & 3) - 2)};
        const h2 hi = (h2){(h1)(((b >> 4) & 3) - 2), (h1)((b >> 6) - 2)};
        l4[i] = make_uint4(as_u32(lo), as_u32(lo) & 0x7FFF7FFFu, as_u32(hi), as_u32(hi) & 0x7FFF7FFFu);
    }
}

__device__ __forceinline__ void pair_bytes2(uint32_t wa, uint32_t wb, uint32_t &even, uint32_t &odd)
{
    constexpr uint32_t m = 0x33333333u;
    even = (wa & m) | ((wb & m) << 2);
    odd = ((wa >> 2) & m) | (wb & ~m);
}

// lane_copy = (lane % 16) * 16.  k: byte of `bytes`, a compile-time constant after unrolling.
__device__ __forceinline__ uint4 lut2_get(const uint2 *lut, uint32_t bytes, uint32_t lane_copy, int k)
{
    const uint32_t sel = 0x0C0C0000u | ((4u + (uint32_t)k) << 8);
    const uint32_t addr = __builtin_amdgcn_perm(bytes, lane_copy, sel);
    return *reinterpret_cast<const uint4 *>(reinterpret_cast<const char *>(lut) + addr);
}

} // namespace adkv
