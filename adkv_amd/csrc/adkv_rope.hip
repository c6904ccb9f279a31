// Rotary position embedding of q and k in one launch   (llama_adkv.py:336-337 calls transformers'
// apply_rotary_pos_emb: x * cos + rotate_half(x) * sin, ten elementwise launches)
//
// Every operation is rounded to the activations' type the way torch's elementwise kernels round
// it (operands widened to fp32, one fp32 operation, result rounded to nearest even), so the
// output equals that of the torch expression bit for bit.  A row is one (batch, token, head)
// vector of D values.
#include <hip/hip_runtime.h>

#include "adkv_device.h"

#include "../../include/adkv_hip.h"

#pragma clang fp contract(off)

namespace adkv_rope {
using adkv::as_h2;
using adkv::as_u32;
using adkv::h1;
using adkv::h2;

template <bool BF16>
__device__ __forceinline__ float act_to_f32(uint32_t bits16)
{
    if (BF16)
        return __uint_as_float(bits16 << 16);
    return (float)__builtin_bit_cast(h1, (uint16_t)bits16);
}
template <bool BF16>
__device__ __forceinline__ uint32_t f32_to_act(float f)
{
    if (BF16) {
        const uint32_t u = __float_as_uint(f);
        if ((u & 0x7FFFFFFFu) > 0x7F800000u)
            return 0x7FC0u; // torch's bfloat16 NaN
        return (u + 0x7FFFu + ((u >> 16) & 1u)) >> 16;
    }
    return (uint32_t)__builtin_bit_cast(uint16_t, (h1)f);
}
// r(r(x*c) + r(y*s)) with y already negated where rotate_half negates
template <bool BF16>
__device__ __forceinline__ uint32_t rope_one(uint32_t x, uint32_t c, uint32_t y, bool neg_y, uint32_t s)
{
    const float a = act_to_f32<BF16>(f32_to_act<BF16>(act_to_f32<BF16>(x) * act_to_f32<BF16>(c)));
    const float yy = neg_y ? -act_to_f32<BF16>(y) : act_to_f32<BF16>(y);
    const float b = act_to_f32<BF16>(f32_to_act<BF16>(yy * act_to_f32<BF16>(s)));
    return f32_to_act<BF16>(a + b);
}

// two adjacent values of the first half and their partners in the second, as words
// first half: x1*cos + (-x2)*sin; second half: x2*cos + x1*sin
template <bool BF16>
__device__ __forceinline__ void rope_two(uint32_t x1, uint32_t x2, uint32_t c1, uint32_t c2, uint32_t s1, uint32_t s2,
                                         uint32_t &lo, uint32_t &hi)
{
    lo = rope_one<BF16>(x1 & 0xFFFFu, c1 & 0xFFFFu, x2 & 0xFFFFu, true, s1 & 0xFFFFu) |
         rope_one<BF16>(x1 >> 16, c1 >> 16, x2 >> 16, true, s1 >> 16) << 16;
    hi = rope_one<BF16>(x2 & 0xFFFFu, c2 & 0xFFFFu, x1 & 0xFFFFu, false, s2 & 0xFFFFu) |
         rope_one<BF16>(x2 >> 16, c2 >> 16, x1 >> 16, false, s2 >> 16) << 16;
}

struct RopeSide {
    const uint16_t *x;
    uint16_t *out;
    long sb, sh, st; // element strides of x over batch, head, token (channels contiguous)
    int heads;
};

// Rows of any even alignment, in 4-byte pieces.
// grid: (lanes of one token's Hq + H rows in workgroups of 256, token, batch)
template <bool BF16>
__global__ __launch_bounds__(256) void rope_kernel(RopeSide q, RopeSide k, const uint16_t *__restrict__ cos,
                                                   const uint16_t *__restrict__ sin, long cb, long ct,
                                                   int T, int D, int t0, int b0)
{
    const unsigned lpr = (unsigned)D >> 2;                   // lanes per row
    const unsigned idx = blockIdx.x * 256u + threadIdx.x;
    const unsigned hh = idx / lpr;
    if (hh >= (unsigned)(q.heads + k.heads))
        return;
    const int i = (int)(idx - hh * lpr) * 2;                 // first of this lane's two channels
    const int t = t0 + (int)blockIdx.y;
    const long b = (long)b0 + (long)blockIdx.z;
    const RopeSide &sd = hh < (unsigned)q.heads ? q : k;
    const int h = hh < (unsigned)q.heads ? (int)hh : (int)hh - q.heads;
    const uint16_t *x = sd.x + b * sd.sb + h * sd.sh + t * sd.st;
    uint16_t *o = sd.out + ((b * sd.heads + h) * T + t) * D;
    const uint16_t *c = cos + b * cb + t * ct, *s = sin + b * cb + t * ct;
    const int half = D >> 1;
    const uint32_t x1 = *reinterpret_cast<const uint32_t *>(x + i);
    const uint32_t x2 = *reinterpret_cast<const uint32_t *>(x + half + i);
    const uint32_t c1 = *reinterpret_cast<const uint32_t *>(c + i);
    const uint32_t c2 = *reinterpret_cast<const uint32_t *>(c + half + i);
    const uint32_t s1 = *reinterpret_cast<const uint32_t *>(s + i);
    const uint32_t s2 = *reinterpret_cast<const uint32_t *>(s + half + i);
    uint32_t lo, hi;
    rope_two<BF16>(x1, x2, c1, c2, s1, s2, lo, hi);
    *reinterpret_cast<uint32_t *>(o + i) = lo;
    *reinterpret_cast<uint32_t *>(o + half + i) = hi;
}

// ---- rows in 16-byte pieces ------------------------------------------------------------------
// A lane takes eight values of the first half and their partners in the second, for HPT heads of one
// token: cos and sin are loaded once for all of them, and every load is issued before the first
// value is needed.  Consecutive lanes take a row's pieces, consecutive rows the tokens of one head, so
// a workgroup's stores are whole runs of the contiguous [B, H, T, D] result.
// Bound by HBM: q and k of 128 prompts of 512 tokens, 32 + 32 heads of 128 values in bf16, are 2.15 GB
// in 351 us (6.1 TB/s); a lane of two values per half that rounded bf16 with integer instructions took
// 735 us (2.9 TB/s).  Where fp32 is rounded to bf16 the hardware conversion is used; it agrees with
// round-to-nearest-even on every number (all 2^32 patterns compared) but keeps the payload of a
// NaN where torch writes 0x7FC0: a lane that meets a NaN computes its rows again the other way.
template <bool BF16>
__device__ __forceinline__ void rope_piece(const uint4 &x1, const uint4 &x2, const uint4 &c1, const uint4 &c2,
                                           const uint4 &s1, const uint4 &s2, uint4 &lo, uint4 &hi, float &nan)
{
    const uint32_t a[4] = {x1.x, x1.y, x1.z, x1.w}, b[4] = {x2.x, x2.y, x2.z, x2.w};
    const uint32_t ca[4] = {c1.x, c1.y, c1.z, c1.w}, cb[4] = {c2.x, c2.y, c2.z, c2.w};
    const uint32_t sa[4] = {s1.x, s1.y, s1.z, s1.w}, sb[4] = {s2.x, s2.y, s2.z, s2.w};
    uint32_t l[4], h[4];
#pragma unroll
    for (int p = 0; p < 4; p++) {
        if constexpr (BF16) {
            auto f0 = [](uint32_t w) { return __uint_as_float(w << 16); };
            auto f1 = [](uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); };
            auto round2 = [](float x, float y) {
                uint32_t r;
                asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
                return r;
            };
            const uint32_t ac = round2(f0(a[p]) * f0(ca[p]), f1(a[p]) * f1(ca[p]));
            const uint32_t bs = round2(-f0(b[p]) * f0(sa[p]), -f1(b[p]) * f1(sa[p]));
            const uint32_t bc = round2(f0(b[p]) * f0(cb[p]), f1(b[p]) * f1(cb[p]));
            const uint32_t as = round2(f0(a[p]) * f0(sb[p]), f1(a[p]) * f1(sb[p]));
            const float l0 = f0(ac) + f0(bs), l1 = f1(ac) + f1(bs), h0 = f0(bc) + f0(as), h1v = f1(bc) + f1(as);
            l[p] = round2(l0, l1);
            h[p] = round2(h0, h1v);
            asm("v_maximum3_f32 %0, %0, %1, %2" : "+v"(nan) : "v"(l0), "v"(l1));
            asm("v_maximum3_f32 %0, %0, %1, %2" : "+v"(nan) : "v"(h0), "v"(h1v));
        } else {
            // one packed fp16 operation rounds the exact product, and the exact sum, once: the same
            // as fp32 and then fp16 (the fp32 product is exact; 24 bits are enough for the sum)
            l[p] = as_u32(as_h2(a[p]) * as_h2(ca[p]) + (-as_h2(b[p])) * as_h2(sa[p]));
            h[p] = as_u32(as_h2(b[p]) * as_h2(cb[p]) + as_h2(a[p]) * as_h2(sb[p]));
        }
    }
    lo = make_uint4(l[0], l[1], l[2], l[3]);
    hi = make_uint4(h[0], h[1], h[2], h[3]);
}

// grid: (token blocks of tb, head blocks of hb * HPT, batch); lpr = D / 16 lanes per row
template <bool BF16, int HPT>
__global__ __launch_bounds__(256) void rope_vec_kernel(RopeSide q, RopeSide k, const uint16_t *__restrict__ cos,
                                                       const uint16_t *__restrict__ sin, long cb, long ct,
                                                       int T, int D, int lpr, int tb, int hb, int b0)
{
    const int r = (int)threadIdx.x / lpr, i = ((int)threadIdx.x - r * lpr) * 8;
    const int slot = r / tb, t = (int)blockIdx.x * tb + (r - slot * tb);
    if (slot >= hb || t >= T)
        return;
    const int total = q.heads + k.heads, half = D >> 1;
    const long b = (long)b0 + blockIdx.z;
    const int hh0 = (int)blockIdx.y * hb * HPT + slot;
    const uint16_t *c = cos + b * cb + t * ct + i, *s = sin + b * cb + t * ct + i;
    uint4 x1[HPT], x2[HPT];
#pragma unroll
    for (int j = 0; j < HPT; j++) {
        const int hh = min(hh0 + j * hb, total - 1);
        const bool is_q = hh < q.heads;
        const uint16_t *x = is_q ? q.x + b * q.sb + hh * q.sh + t * q.st : k.x + b * k.sb + (hh - q.heads) * k.sh + t * k.st;
        x1[j] = *reinterpret_cast<const uint4 *>(x + i);
        x2[j] = *reinterpret_cast<const uint4 *>(x + half + i);
    }
    const uint4 c1 = *reinterpret_cast<const uint4 *>(c), c2 = *reinterpret_cast<const uint4 *>(c + half);
    const uint4 s1 = *reinterpret_cast<const uint4 *>(s), s2 = *reinterpret_cast<const uint4 *>(s + half);
#pragma unroll
    for (int j = 0; j < HPT; j++) {
        const int hh = hh0 + j * hb;
        if (hh >= total)
            return;
        uint4 lo, hi;
        float nan = 0.0f;
        rope_piece<BF16>(x1[j], x2[j], c1, c2, s1, s2, lo, hi, nan);
        if (BF16 && __builtin_expect(nan != nan, 0)) {
            auto word = [](const uint4 &v, int p) { return p == 0 ? v.x : p == 1 ? v.y : p == 2 ? v.z : v.w; };
            uint32_t l[4], h[4];
#pragma unroll
            for (int p = 0; p < 4; p++)
                rope_two<BF16>(word(x1[j], p), word(x2[j], p), word(c1, p), word(c2, p), word(s1, p), word(s2, p), l[p], h[p]);
            lo = make_uint4(l[0], l[1], l[2], l[3]);
            hi = make_uint4(h[0], h[1], h[2], h[3]);
        }
        uint16_t *o = (hh < q.heads ? q.out + ((b * q.heads + hh) * T + t) * D
                                    : k.out + ((b * k.heads + (hh - q.heads)) * T + t) * D) + i;
        *reinterpret_cast<uint4 *>(o) = lo;
        *reinterpret_cast<uint4 *>(o + half) = hi;
    }
}

} // namespace adkv_rope

extern "C" int adkv_rope_qk(const void *q, const void *k, const void *cos, const void *sin, void *q_out, void *k_out,
                 int B, int Hq, int H, int T, int D,
                 int64_t q_sb, int64_t q_sh, int64_t q_st, int64_t k_sb, int64_t k_sh, int64_t k_st,
                 int64_t cs_sb, int64_t cs_st, int bf16, void *stream)
{
    using namespace adkv_rope;
    if (!q || !k || !cos || !sin || !q_out || !k_out)
        return ADKV_E_NULL;
    if (B <= 0 || Hq <= 0 || H <= 0 || T <= 0 || D <= 0 || (D & 3))
        return ADKV_E_SHAPE;
    // 4-byte accesses: every base and every stride a multiple of two elements
    if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)cos | (uintptr_t)sin | (uintptr_t)q_out | (uintptr_t)k_out) & 3)
        return ADKV_E_ALIGN;
    if ((q_sb | q_sh | q_st | k_sb | k_sh | k_st | cs_sb | cs_st) & 1)
        return ADKV_E_ALIGN;
    if ((long)(Hq + H) * (D >> 2) > (long)INT32_MAX)
        return ADKV_E_SHAPE;
    const RopeSide qs = {(const uint16_t *)q, (uint16_t *)q_out, (long)q_sb, (long)q_sh, (long)q_st, Hq};
    const RopeSide ks = {(const uint16_t *)k, (uint16_t *)k_out, (long)k_sb, (long)k_sh, (long)k_st, H};
    constexpr int GMAX = 65535; // grid limit of the token and batch axes: longer ones take several launches
    // 16-byte pieces wherever every row is made of them and there are enough rows: below some 5000 the
    // 4-byte form, with four times the lanes, is done sooner (us, 4-byte / 16-byte, bf16 rows of 128:
    // 320 rows 2.17 / 2.52, 4096 2.49 / 2.77, 6144 2.87 / 2.82, 8192 3.16 / 2.92)
    const bool wide = (long)B * (Hq + H) * T >= 5120 && D % 16 == 0 && D <= 16 * 256 &&
                      (((uintptr_t)q | (uintptr_t)k | (uintptr_t)cos | (uintptr_t)sin | (uintptr_t)q_out | (uintptr_t)k_out) & 15) == 0 &&
                      ((q_sb | q_sh | q_st | k_sb | k_sh | k_st | cs_sb | cs_st) & 7) == 0;
    if (wide) {
        // a workgroup's rows: as many tokens of a head as it holds, several heads when tokens are few.
        // Four heads per lane share cos and sin; launches too small to fill the CUs that way
        // take one (a token of a batch: latency is all that counts).
        const int lpr = D >> 4, rows = 256 / lpr, tb = min(rows, T), hb = rows / tb;
        const long tblocks = ((long)T + tb - 1) / tb;
        const long full = tblocks * B * ((Hq + H + 4 * hb - 1) / (4 * hb));
        const int hpt = full >= 1024 ? 4 : 1;
        const unsigned gy = (unsigned)((Hq + H + hb * hpt - 1) / (hb * hpt));
        if (gy <= (unsigned)GMAX) {
            for (int b0 = 0; b0 < B; b0 += GMAX) {
                const dim3 grid((unsigned)tblocks, gy, (unsigned)min(B - b0, GMAX));
                const auto kernel = bf16 ? (hpt == 4 ? rope_vec_kernel<true, 4> : rope_vec_kernel<true, 1>)
                                         : (hpt == 4 ? rope_vec_kernel<false, 4> : rope_vec_kernel<false, 1>);
                hipLaunchKernelGGL(kernel, grid, dim3(256), 0, (hipStream_t)stream, qs, ks, (const uint16_t *)cos,
                                   (const uint16_t *)sin, (long)cs_sb, (long)cs_st, T, D, lpr, tb, hb, b0);
            }
            return adkv::check_launch();
        }
    }
    const unsigned gx = (unsigned)(((long)(Hq + H) * (D >> 2) + 255) / 256);
    for (int b0 = 0; b0 < B; b0 += GMAX)
        for (int t0 = 0; t0 < T; t0 += GMAX) {
            const dim3 grid(gx, (unsigned)min(T - t0, GMAX), (unsigned)min(B - b0, GMAX));
            if (bf16)
                hipLaunchKernelGGL(rope_kernel<true>, grid, dim3(256), 0, (hipStream_t)stream, qs, ks,
                                   (const uint16_t *)cos, (const uint16_t *)sin, (long)cs_sb, (long)cs_st, T, D,
                                   t0, b0);
            else
                hipLaunchKernelGGL(rope_kernel<false>, grid, dim3(256), 0, (hipStream_t)stream, qs, ks,
                                   (const uint16_t *)cos, (const uint16_t *)sin, (long)cs_sb, (long)cs_st, T, D,
                                   t0, b0);
        }
    return adkv::check_launch();
}
