// ADKV hot-path kernels for MI355X (gfx950, wave64) and their C ABI (include/adkv_hip.h).
//
// Work decomposition.  Every (batch, head, channel) is an independent fp16 recurrence over the
// time axis (reference: src/adkv/kernel/gemv.cu:187-191).  A LANE owns CPL consecutive channels of
// one head; D/CPL lanes make a head; a wave64 carries 64*CPL/D heads.  One supergroup (8 tokens) of
// a head is D*4 contiguous bytes, which the head's lanes fetch as one run of 16-byte loads; loads
// for the next PF supergroups are in flight while the current one is decoded.
//
// The recurrence rounds to fp16 at every step, so it cannot be re-associated: a sequence can only be
// split where the exact state is known.  The encoder therefore can record the state every
// `ckpt_interval` tokens ("checkpoints", 4 bytes per channel each); given those, the decode kernels
// cut the time axis into segments that replay independently and bit-exactly.  Without checkpoints
// they replay from token 0 exactly like the reference.  More waves matter on this machine: a SIMD
// needs about four resident waves to issue packed-f16 instructions at full rate.
//
// The kernels keep the reference's call structure (encode / QK+append / OV+append) so that they are
// drop-ins for src/adkv/kernel/gemv.cu:368-414, 883-939, 1233-1288.
#include "adkv_device.h"

#include "../../include/adkv_hip.h"

#include <stdlib.h>

#include <atomic>
#include <initializer_list>
#include <mutex>
#include <type_traits>

#pragma clang fp contract(off)

namespace adkv {

constexpr int PF = 4; // supergroups in flight per lane (2, 6 and 8 were measured: no difference)
// two channels per lane: 64 tokens ahead of a loop that takes 29 ns per token (with 32 it ran into the
// memory's latency: forward_ov of 32 x 32 heads x 1024 tokens 38 us, with 64 32)
constexpr int PF_PAIR = 8;

template <int D, int CPL>
struct Geo {
    static constexpr int LPH = D / CPL;       // lanes per head
    static constexpr int NP = CPL / 2;        // channel pairs per lane
    // a lane's CPL code words of one supergroup, loaded as 16-byte vectors (8 bytes when the lane
    // owns only two channels)
    using Vec = typename std::conditional<CPL >= 4, uint4, uint2>::type;
    static constexpr int WPV = sizeof(Vec) / 4; // 32-bit channel words per vector
    static constexpr int NV = CPL / WPV;        // vectors per lane per supergroup
    static constexpr int VPS = D / WPV;         // vectors per supergroup of one head
    static_assert(LPH == 32 || LPH == 64, "a head must fit in one wave");
    static_assert(CPL == 2 || CPL % 4 == 0, "two channels per lane, or a multiple of four");
};

__device__ __forceinline__ void vec_words(const uint4 &u, uint32_t *w)
{
    w[0] = u.x; w[1] = u.y; w[2] = u.z; w[3] = u.w;
}
__device__ __forceinline__ void vec_words(const uint2 &u, uint32_t *w)
{
    w[0] = u.x; w[1] = u.y;
}
__device__ __forceinline__ void words_vec(const uint32_t *w, uint4 &u) { u = make_uint4(w[0], w[1], w[2], w[3]); }
__device__ __forceinline__ void words_vec(const uint32_t *w, uint2 &u) { u = make_uint2(w[0], w[1]); }
template <typename V> __device__ __forceinline__ V vec_zero();
template <> __device__ __forceinline__ uint4 vec_zero<uint4>() { return make_uint4(0, 0, 0, 0); }
template <> __device__ __forceinline__ uint2 vec_zero<uint2>() { return make_uint2(0, 0); }

// The code stream is read exactly once: a non-temporal load keeps it from displacing the logits
// and weights (which the softmax and the next kernel read back) in the caches.  Measured on the
// headline shape: forward_qk -1 %, forward_ov -3 %, the softmax between them -12 %.
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
typedef uint32_t u2v32 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint4 load_codes(const uint4 *p)
{
    const u4v v = __builtin_nontemporal_load(reinterpret_cast<const u4v *>(p));
    return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint2 load_codes(const uint2 *p)
{
    const u2v32 v = __builtin_nontemporal_load(reinterpret_cast<const u2v32 *>(p));
    return make_uint2(v.x, v.y);
}

// How the time axis is cut.  seg_tokens is a multiple of ckpt_interval (itself a multiple of 8);
// segment s covers tokens [s*seg_tokens, min((s+1)*seg_tokens, T)) and starts from checkpoint
// s*seg_tokens/ckpt_interval - 1 (segment 0 starts from the initial parameters).
struct Seg {
    h1 *ckpt;           // [B*H, n_ckpt_cap, D, 2] (zp, sc) before token (j+1)*ckpt_interval; may be null
    int n_ckpt_cap;
    int ckpt_interval;  // 0 when ckpt is null
    int seg_tokens;     // >= T when there is one segment
    int seg_intervals;  // checkpoint intervals of an even segment (0 when there is one segment)
    int nseg;
    long row_pitch;     // elements between rows of the logits / attention-weight matrix (>= T + 1)
    int act_bf16;       // q, the new token and the output are bfloat16 (see load_act2 / store_act2)
    int combine;        // ov_ft_kernel: the segments' partial outputs are added inside the workgroup
    // groups > 0 (per-head-table and matrix-core kernels): the context's `intervals` checkpoint intervals are
    // cut into `groups` groups of four segments of unequal length (uneven_cut).  groups < 0 (matrix-core and shared-table
    // ones of head dim 128): into nseg segments that differ by one interval at most.  phys_per_head (per-head table):
    // workgroups launched per KV head; each walks through the head's virtual workgroups pw,
    // pw + phys_per_head, ... one after the other (same table, no barrier between them).
    int groups;
    int intervals;
    int phys_per_head;
    unsigned skew;      // shares of the four wave slots, oldest first, one byte each, in sixteenths
    int fresh;          // encoder: the cache and checkpoint memory is uninitialised, write what is past the tokens too
};

__host__ __device__ inline int ft_skew(unsigned skew, int k) { return (int)((skew >> (8 * k)) & 0xFFu); }
constexpr unsigned pack_skew(unsigned a, unsigned b, unsigned c, unsigned d) { return a | (b << 8) | (c << 16) | (d << 24); }

// First checkpoint interval of the seg-th segment IN TIME ORDER (seg == 4*groups: one past the
// last) when `intervals` intervals are cut into `groups` groups of four uneven segments.  Group g
// covers [intervals*g/groups, intervals*(g+1)/groups); inside it the shares are rounded down, every
// segment gets at least one interval, and what is left goes to the oldest slots first.  The
// shares are listed oldest wave slot first and laid out LATEST segment first: the oldest slot
// takes the group's last segment (the longest), the youngest its first (see segment_of_slot).
// Needs at least four intervals per group.  The same function plans on the host and indexes on
// the device.
__host__ __device__ inline void uneven_parts(int n, unsigned skew, int *part) // of a group of n intervals, by wave slot, oldest first
{
    int left = n;
    for (int i = 0; i < 4; i++) {
        part[i] = n * ft_skew(skew, i) / 16;
        if (part[i] < 1)
            part[i] = 1;
        left -= part[i];
    }
    for (int i = 0; left > 0; i = (i + 1) & 3, left--)
        part[i]++;
    for (int i = 0; left < 0; i = (i + 1) & 3) // only when n is tiny: take from the longest
        if (part[i] > 1) {
            part[i]--;
            left++;
        }
}
__host__ __device__ inline int uneven_cut(int seg, int groups, int intervals, unsigned skew)
{
    const int g = seg >> 2, k = seg & 3;
    const int lo = (int)((long)intervals * g / groups);
    if (k == 0)
        return lo;
    int part[4];
    uneven_parts((int)((long)intervals * (g + 1) / groups) - lo, skew, part);
    int c = lo;
    for (int i = 0; i < k; i++)
        c += part[3 - i];
    return c;
}

// Which segment (in time order) the waves of slot index `seg` work on.  interleave_segment gives
// quad k of a workgroup slot index k of a group of four, and quad k is wave slot k of its SIMDs
// (oldest first).  In an uneven plan the oldest slot takes the group's LAST segment: that is where
// the work after the loop is (ragged tail, appended token, published state: a chain of dependent
// memory operations), and the oldest slot's waves are the first to finish their loop, so that
// work runs while the other slots are still in theirs instead of at the very end of the launch.
__host__ __device__ inline int segment_of_slot(const Seg &sa, int seg) { return sa.groups > 0 ? seg ^ 3 : seg; }

// first interval of the seg-th of nseg segments as equal as they can be
__host__ __device__ inline int balanced_cut(const Seg &sa, int seg) { return (int)((long)sa.intervals * seg / sa.nseg); }
// first token of the segment of slot index `seg` / of the one after it in time, in checkpoint intervals (0 when there is one segment)
__host__ __device__ inline int seg_first_interval(const Seg &sa, int seg)
{
    return sa.groups > 0   ? uneven_cut(seg ^ 3, sa.groups, sa.intervals, sa.skew)
           : sa.groups < 0 ? balanced_cut(sa, seg)
                           : seg * sa.seg_intervals;
}
// the same in tokens; whether it is the last of the context
__host__ __device__ inline int seg_begin(const Seg &sa, int seg)
{
    return sa.groups ? seg_first_interval(sa, seg) * sa.ckpt_interval : seg * sa.seg_tokens;
}
__host__ __device__ inline int seg_end(const Seg &sa, int seg)
{
    return sa.groups > 0   ? uneven_cut((seg ^ 3) + 1, sa.groups, sa.intervals, sa.skew) * sa.ckpt_interval
           : sa.groups < 0 ? balanced_cut(sa, seg + 1) * sa.ckpt_interval
                           : (seg + 1) * sa.seg_tokens;
}
__host__ __device__ inline bool seg_is_last(const Seg &sa, int seg) { return segment_of_slot(sa, seg) == sa.nseg - 1; }

// waits for every LDS and scalar access in flight, as an instruction that the compiler counts with
__device__ __forceinline__ void wait_lgkm() { __builtin_amdgcn_s_waitcnt(0xC07F); }

__device__ __forceinline__ float wave_xor_add(float v, int mask)
{
    return v + __shfl_xor(v, mask, 64);
}

// s + s[lane ^ 8]: DPP rotate by 8 within each row of 16 lanes (no LDS round trip).
__device__ __forceinline__ float xor8_add(float s)
{
    const int r = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, s), 0x128 /*row_ror:8*/,
                                              0xF, 0xF, false);
    return s + __builtin_bit_cast(float, r);
}

typedef unsigned u2v __attribute__((ext_vector_type(2)));

// s + s[lane ^ 16] / s + s[lane ^ 32] through the gfx950 row/half swap instructions.  Both the copy
// and the results go through opaque asm statements: handed two identical values, or asked for the
// float sum of the two results directly, this compiler folds the pair into one register.
__device__ __forceinline__ float xor16_add(float s)
{
    unsigned a = __builtin_bit_cast(unsigned, s), b;
    asm volatile("v_mov_b32 %0, %1" : "=v"(b) : "v"(a));
    const u2v r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    unsigned x = r.x, y = r.y;
    asm volatile("" : "+v"(x), "+v"(y));
    return __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
}

__device__ __forceinline__ float xor32_add(float s)
{
    unsigned a = __builtin_bit_cast(unsigned, s), b;
    asm volatile("v_mov_b32 %0, %1" : "=v"(b) : "v"(a));
    const u2v r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    unsigned x = r.x, y = r.y;
    asm volatile("" : "+v"(x), "+v"(y));
    return __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
}

// v + v[lane ^ 1], + that of lane ^ 2, ^ 4 .. ^ 32 of the sums (or the largest of them), in registers: inside 4, 8 and 16 lanes that
// agree a mirrored lane has what the exchanged one has.  The sums of a butterfly through __shfl_xor bit for bit, without its six trips
// through the LDS.
template <int CTRL, bool MAX>
__device__ __forceinline__ float mirror_fold(float v)
{
    const float o = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
    return MAX ? fmaxf(v, o) : v + o;
}
template <bool MAX>
__device__ __forceinline__ float wave_reduce(float v)
{
    v = mirror_fold<0xB1, MAX>(v);  // quad_perm [1, 0, 3, 2]
    v = mirror_fold<0x4E, MAX>(v);  // quad_perm [2, 3, 0, 1]
    v = mirror_fold<0x141, MAX>(v); // row_half_mirror
    v = mirror_fold<0x140, MAX>(v); // row_mirror
    unsigned a = __builtin_bit_cast(unsigned, v), b; // see xor16_add
    asm volatile("v_mov_b32 %0, %1" : "=v"(b) : "v"(a));
    const u2v r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    unsigned x = r.x, y = r.y;
    asm volatile("" : "+v"(x), "+v"(y));
    v = MAX ? fmaxf(__builtin_bit_cast(float, x), __builtin_bit_cast(float, y)) : __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
    a = __builtin_bit_cast(unsigned, v);
    asm volatile("v_mov_b32 %0, %1" : "=v"(b) : "v"(a));
    const u2v h = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    x = h.x;
    y = h.y;
    asm volatile("" : "+v"(x), "+v"(y));
    return MAX ? fmaxf(__builtin_bit_cast(float, x), __builtin_bit_cast(float, y)) : __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
}

// Sum over the LPH lanes of a head; every lane of the head gets the total.
template <int LPH>
__device__ __forceinline__ float head_allreduce(float v)
{
#pragma unroll
    for (int m = 1; m < LPH; m <<= 1)
        v = wave_xor_add(v, m);
    return v;
}

// a.x*b.x + a.y*b.y in fp32, as the three-operand form with a literal zero accumulator: the
// accumulating two-operand form the compiler picks needs its destination cleared first, one more
// vector instruction per token.  The leading wait state covers an operand that the instruction
// just before wrote as a packed 16-bit result (on this chip such a result cannot be forwarded to
// the very next instruction; the compiler pads its own code the same way).
__device__ __forceinline__ float dot2_from_zero(h2 a, h2 b)
{
    float d;
    asm("s_nop 0\n\tv_dot2_f32_f16 %0, %1, %2, 0" : "=v"(d) : "v"(a), "v"(b));
    return d;
}

// Sum of 8 per-lane partials over the 32 lanes of a head, scattered: afterwards every lane holds
// the total of ONE token, token_of_lane(lane), the same in the four lanes of a quad.
//   bit 3 of the lane (banks 0,1 | 2,3): keep tokens 0-3 | 4-7, add the partner's    8 instructions
//   bit 2 (banks 0,2 | 1,3):             keep tokens +0,+1 | +2,+3                      4
//   bit 4 (row 0 | 1 of the head):       v_permlane16_swap + add, keep token +0 | +1    2
//   bits 0,1: all-reduce inside the quad                                                2
// A masked DPP add writes only the banks of its mask and keeps the other lanes' destination; a
// DPP operand must not have been written by the two preceding instructions, which the order
// below guarantees inside the block and the leading s_nop for whatever precedes it.
__device__ __forceinline__ float reduce8_head32(const float *p)
{
    float r0, r1, r2, r3, s0, s1;
    asm volatile(
        "s_nop 1\n\t"
        "v_add_f32_dpp %0, %6, %6 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
        "v_add_f32_dpp %1, %7, %7 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
        "v_add_f32_dpp %2, %8, %8 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
        "v_add_f32_dpp %3, %9, %9 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
        "v_add_f32_dpp %0, %10, %10 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %1, %11, %11 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %2, %12, %12 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %3, %13, %13 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        // banks 0,2 take lane+4 (rotate right by 12), banks 1,3 take lane-4 (rotate right by 4)
        "v_add_f32_dpp %4, %0, %0 row_ror:12 row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %5, %1, %1 row_ror:12 row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %4, %2, %2 row_ror:4 row_mask:0xf bank_mask:0xa\n\t"
        "v_add_f32_dpp %5, %3, %3 row_ror:4 row_mask:0xf bank_mask:0xa\n\t"
        "s_nop 1\n\t"
        "v_permlane16_swap_b32 %4, %5\n\t"
        "s_nop 1\n\t"
        "v_add_f32 %4, %4, %5\n\t"
        "s_nop 1\n\t"
        "v_add_f32_dpp %4, %4, %4 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_add_f32_dpp %4, %4, %4 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 0"
        : "=&v"(r0), "=&v"(r1), "=&v"(r2), "=&v"(r3), "=&v"(s0), "=&v"(s1)
        : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]), "v"(p[6]), "v"(p[7]));
    return s0;
}

__device__ __forceinline__ int token_of_lane(int lane)
{
    const int bank = (lane >> 2) & 3, row = (lane >> 4) & 1;
    return 4 * (bank >> 1) + 2 * (bank & 1) + row;
}

// The same for a head of 16 lanes (one row): after the two masked steps a lane holds two tokens'
// sums over the four lanes that differ from it in bits 2 and 3; lanes with bit 1 clear keep the
// first and take the partner's (lane ^ 2) first, the others the second, and bit 0 is an all-reduce.
// Every PAIR of lanes ends with one token's total, token_of_lane16(lane).
__device__ __forceinline__ float reduce8_head16(const float *p)
{
    float r0, r1, r2, r3, s0, s1, keep, give;
    const unsigned long long odd_pairs = 0xCCCCCCCCCCCCCCCCull; // lanes with bit 1 set
    asm volatile(
        "s_nop 1\n\t"
        "v_add_f32_dpp %0, %8, %8 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
        "v_add_f32_dpp %1, %9, %9 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
        "v_add_f32_dpp %2, %10, %10 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
        "v_add_f32_dpp %3, %11, %11 row_ror:8 row_mask:0xf bank_mask:0x3\n\t"
        "v_add_f32_dpp %0, %12, %12 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %1, %13, %13 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %2, %14, %14 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %3, %15, %15 row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
        "v_add_f32_dpp %4, %0, %0 row_ror:12 row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %5, %1, %1 row_ror:12 row_mask:0xf bank_mask:0x5\n\t"
        "v_add_f32_dpp %4, %2, %2 row_ror:4 row_mask:0xf bank_mask:0xa\n\t"
        "v_add_f32_dpp %5, %3, %3 row_ror:4 row_mask:0xf bank_mask:0xa\n\t"
        "v_cndmask_b32_e64 %6, %4, %5, %16\n\t"
        "v_cndmask_b32_e64 %7, %5, %4, %16\n\t"
        "s_nop 1\n\t"
        "v_add_f32_dpp %6, %7, %6 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 1\n\t"
        "v_add_f32_dpp %6, %6, %6 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
        "s_nop 0"
        : "=&v"(r0), "=&v"(r1), "=&v"(r2), "=&v"(r3), "=&v"(s0), "=&v"(s1), "=&v"(keep), "=&v"(give)
        : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]), "v"(p[4]), "v"(p[5]), "v"(p[6]), "v"(p[7]), "s"(odd_pairs));
    return keep;
}

__device__ __forceinline__ int token_of_lane16(int lane)
{
    const int bank = (lane >> 2) & 3;
    return 4 * (bank >> 1) + 2 * (bank & 1) + ((lane >> 1) & 1);
}

// The same sum over a head of LPH lanes: a 64-lane head adds its two halves at the end (both then
// hold every token's total).
template <int LPH>
__device__ __forceinline__ float reduce8_head(const float *p)
{
    const float s = reduce8_head32(p);
    return LPH == 64 ? xor32_add(s) : s;
}

// (zp, sc) of CPL consecutive channels <-> the interleaved [channel][2] fp16 layout used for
// state_out and checkpoints.
template <int CPL>
__device__ __forceinline__ void store_state(h1 *dst, const Pair *st)
{
    h2 *so = reinterpret_cast<h2 *>(dst);
#pragma unroll
    for (int p = 0; p < CPL / 2; p++) {
        so[2 * p] = (h2){st[p].zp.x, st[p].sc.x};
        so[2 * p + 1] = (h2){st[p].zp.y, st[p].sc.y};
    }
}

template <int CPL>
__device__ __forceinline__ void load_state(const h1 *src, Pair *st)
{
    const h2 *so = reinterpret_cast<const h2 *>(src);
#pragma unroll
    for (int p = 0; p < CPL / 2; p++) {
        const h2 a = so[2 * p], b = so[2 * p + 1];
        st[p].zp = (h2){a.x, b.x};
        st[p].sc = (h2){a.y, b.y};
    }
}

// store_state for any channel count, including a single channel held in both halves of a pair
template <int CPL>
__device__ __forceinline__ void store_state_n(h1 *dst, const Pair *st)
{
    if (CPL >= 2)
        store_state<CPL>(dst, st);
    else
        *reinterpret_cast<h2 *>(dst) = (h2){st[0].zp.x, st[0].sc.x};
}

// Which (head, segment) this lane works on.  Every segment's run of units is padded to whole
// waves, so all lanes of a wave work on the same segment and everything derived from it (token
// range, trip counts) is wave-uniform: the decode loops then branch on scalars instead of masking
// lanes.  Units past the end are clamped to a valid one and flagged inactive: they compute but
// never store.
//
// Consecutive waves take DIFFERENT segments of the same sequences (interleave_segment): the last
// segment of a context is shorter than the others whenever the length is not a multiple of the
// segment size (a 640-token context cut at 512 is a 512-token and a 128-token segment), and with
// all short waves in one workgroup and all long ones in another, half the CUs went idle after a
// quarter of the launch (B=128: 640 tokens took as long as 1024).  Mixed, every SIMD holds long
// and short waves and the long ones speed up when the short ones leave (two waves issue nearly as
// fast as four).
//
// wave index -> (segment, wave within the segment).  A wave's SIMD is its index modulo 4 (a
// workgroup's waves go round the SIMDs), so the mapping works on quads of waves: quad q takes
// segment q mod nseg, and its four waves are four consecutive waves' worth of units of that
// segment; every SIMD then walks through the segments in turn.  Each segment's waves are padded
// to a multiple of four (pad4); padding waves leave right after the table is built.
__host__ __device__ inline int pad4(int n) { return (n + 3) & ~3; }
__host__ __device__ inline void interleave_segment(int wave, int nseg, int &seg, int &wave_in_seg)
{
    const int q = wave >> 2, g = q / nseg;
    seg = q - g * nseg;
    wave_in_seg = g * 4 + (wave & 3);
}

template <int LPH>
static inline long padded_units(int BH, int nseg)
{
    constexpr int UPW = 64 / LPH; // units per wave
    return (long)nseg * pad4((BH + UPW - 1) / UPW) * UPW;
}

template <int D, int CPL, int BLK>
struct Unit {
    int bx, seg, lh, c0;
    bool active, wave_active;
    __device__ __forceinline__ Unit(int BH, int nseg)
    {
        using G = Geo<D, CPL>;
        constexpr int UPW = 64 / G::LPH;
        const int waves_per_seg = (BH + UPW - 1) / UPW;
        const long gl = (long)blockIdx.x * BLK + threadIdx.x;
        lh = (int)(gl % G::LPH);
        const int wave = __builtin_amdgcn_readfirstlane((int)(gl >> 6));
        int sg, wis;
        interleave_segment(wave, nseg, sg, wis);
        const int b = wis * UPW + (int)((gl & 63) / G::LPH);
        wave_active = wis < waves_per_seg;
        active = wave_active && b < BH;
        seg = sg;
        bx = b < BH ? b : BH - 1;
        c0 = lh * CPL;
    }
};

// Parameters plus the state this segment starts from.
template <int D, int CPL>
__device__ __forceinline__ void init_pairs(Pair *st, const h1 *zp, const h1 *sc, const h1 *al,
                                           const h1 *be, const h1 *tg, int h, int bx, int c0, int seg,
                                           const Seg &sa)
{
#pragma unroll
    for (int p = 0; p < CPL / 2; p++)
        load_pair(st[p], zp, sc, al, be, tg, h * D + c0 + 2 * p);
    if (seg_begin(sa, seg) > 0) {
        const int j = seg_begin(sa, seg) / sa.ckpt_interval - 1;
        load_state<CPL>(sa.ckpt + (((size_t)bx * sa.n_ckpt_cap + j) * D + c0) * 2, st);
    }
}

// What a unit reads before it can decode: parameters, the state its segment starts from, the first
// supergroups of codes.  start() issues the loads and waits for none of them, so they travel while
// the workgroup writes its table; state() is for after it.  One after the other behind the table (parameters, the
// checkpoint, then codes) these trips to memory took 5 of the 28 us of a segment of 256 tokens at
// four waves per SIMD.  (Kernels take what is read here without __restrict__: the compiler moves loads
// of memory that it knows to be constant past the barrier to their first use.)
template <int D, int CPL, int BITS, int AHEAD>
struct SegLoads {
    using G = Geo<D, CPL>;
    using Vec = typename G::Vec;
    static constexpr int TPW = Code<BITS>::TPW;
    Vec *cbh;       // this head, this lane
    const Vec *cb;  // this segment
    int t0, t1, nfull; // tokens [t0, t1), whole supergroups
    bool last;
    bool from_ckpt;
    uint32_t zp[CPL / 2], sc[CPL / 2], al[CPL / 2], be[CPL / 2], tg[CPL / 2], ck[CPL];
    Vec buf[AHEAD][G::NV];

    __device__ __forceinline__ void start(uint4 *cache, const h1 *zp_, const h1 *sc_, const h1 *al_, const h1 *be_, const h1 *tg_,
                                          int h, int bx, int lh, int seg, int T, int n_super_cap, const Seg &sa)
    {
        const int c0 = lh * CPL, pi = h * D + c0;
        const int iv = seg_first_interval(sa, seg);
        last = seg_is_last(sa, seg);
        t0 = iv * sa.ckpt_interval;
        t1 = last ? T : seg_end(sa, seg);
        nfull = (t1 - t0) / TPW;
        cbh = reinterpret_cast<Vec *>(cache) + (size_t)bx * n_super_cap * G::VPS + lh * G::NV;
        cb = cbh + (size_t)(t0 / TPW) * G::VPS;
        from_ckpt = iv > 0;
        if (from_ckpt)
            __builtin_memcpy(ck, sa.ckpt + (((size_t)bx * sa.n_ckpt_cap + iv - 1) * D + c0) * 2, 4 * CPL);
        // parameters and checkpoints are 4-byte aligned at least
        __builtin_memcpy(zp, zp_ + pi, 2 * CPL);
        __builtin_memcpy(sc, sc_ + pi, 2 * CPL);
        __builtin_memcpy(al, al_ + pi, 2 * CPL);
        __builtin_memcpy(be, be_ + pi, 2 * CPL);
        __builtin_memcpy(tg, tg_ + pi, 2 * CPL);
        // unconditional (a segment without a whole supergroup reads its partial one): with a condition
        // the waits inside the loop have to cover what this entry leaves open
#pragma unroll
        for (int i = 0; i < AHEAD; i++) {
#pragma unroll
            for (int v = 0; v < G::NV; v++)
                buf[i][v] = load_codes(cb + (size_t)min(i, max(nfull - 1, 0)) * G::VPS + v);
        }
    }
    __device__ __forceinline__ void state(Pair *st) const
    {
#pragma unroll
        for (int p = 0; p < CPL / 2; p++) {
            const h2 a = as_h2(ck[2 * p]), b = as_h2(ck[2 * p + 1]);
            st[p].zp = from_ckpt ? (h2){a.x, b.x} : as_h2(zp[p]);
            st[p].sc = from_ckpt ? (h2){a.y, b.y} : as_h2(sc[p]);
            st[p].al = as_h2(al[p]);
            st[p].be = as_h2(be[p]);
            // omt = 1 - beta*target with both steps rounded to fp16 (gemv.cu:220-221)
            st[p].omt = splat((h1)1.0f) - st[p].be * as_h2(tg[p]);
        }
    }
};

// ---------------------------------------------------------------------------------------------
// encode_kv  (gemv.cu:168-308)
// ---------------------------------------------------------------------------------------------
// The state at token t depends on every code before it, so the encoder is one serial chain per
// channel and nothing but B*H*D is parallel.  A lane owns CPL consecutive channels (1 or 2, the
// launcher's choice).  With few channels a wave has its SIMD to itself, and a wave alone issues one
// instruction every 4 cycles whether or not it depends on the one before (5 for 8-byte encodings, 8 for
// v_rcp_f32 and v_fma_f16, 16 and more for a load, 24 and more for a store): the time per token is the
// sum over its instructions, and the loops below are written for that sum.
//  * one channel per lane, rows 16-byte aligned: 8 rows come into the LDS with one buffer load, a run of
//    64 tokens ahead, and a lane reads four tokens of its channel with one transposing LDS read (a load
//    per token was 4 of 39 ns);
//  * otherwise rows come through buffer loads into registers (16 bits per lane with one channel, 32 with
//    two): one instruction per token and nothing else, because the row offsets within a group of 8 tokens
//    sit in scalar registers.  Loads past the end of the stream are dropped by the bounds check instead of
//    being guarded;
//  * the quotient takes three instructions on top of the reciprocal and is the IEEE one
//    (enc_quotient), so nothing has to be checked or repeated for finite values: a form that takes
//    the reciprocal product alone and repeats the groups of 8 tokens in which it comes near a
//    rounding boundary repeats one group in seven, because exact ties are common (both sides of the
//    division have few significant bits);
//  * adding 1.5 * 2^23 + bias rounds the quotient to the nearest integer and leaves the code in the
//    low bits, clamped by one med3; v_alignbit shifts it into the code word (one instruction per
//    code), v_cvt_f16_i16 (one channel) or a byte permute and one packed fma (two) turn it into the
//    fp16 operand of the update.
// Only a quotient that is not a number (a non-finite input or state, a zero scale) sends its run
// of tokens (64 with one channel per lane, 32 with two) through the plain division; half an instruction
// per token looks for one.
constexpr int ENC_PF1 = 8;    // buffers of 8 rows in rotation, one channel per lane (one wave per SIMD: nothing else hides HBM)
constexpr int ENC_AHEAD1 = 6; // groups loaded ahead: 56 loads and their groups' stores fit the 63 the counter holds
constexpr int ENC_PF2 = 4; // two channels per lane (many waves)
constexpr int ENC_RING = 16 * 1024; // a wave's LDS, one channel per lane: two runs of 64 rows of 64 channels
template <int CPL>
__device__ __forceinline__ char *enc_ring(uint4 *ring)
{
    return CPL == 1 ? reinterpret_cast<char *>(ring) + (threadIdx.x >> 6) * ENC_RING : nullptr;
}

// Where the new rows are: element strides between batches, heads and tokens (channels are
// contiguous).  The encoder reads each row once, 256 bytes per head, so a [B, T, H, D] projection
// output viewed as [B, H, T, D] can be quantised in place without a packed copy.
struct RowStrides {
    long b, h, t;
};

__device__ __forceinline__ uint64_t wave_uniform(uint64_t v)
{
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return ((uint64_t)hi << 32) | lo;
}

template <int BITS, int CPL, int BLK, bool BF16 = false>
__device__ __forceinline__ void encode_body(
    uint32_t *__restrict__ cache, const h1 *__restrict__ kv_new, RowStrides xs,
    const h1 *__restrict__ zp, const h1 *__restrict__ sc, const h1 *__restrict__ al,
    const h1 *__restrict__ be, const h1 *__restrict__ tg,
    int BH, int H, int T0, int T, int D, int n_super_cap, const h1 *__restrict__ state_in,
    h1 *__restrict__ state_out, const Seg &sa, char *ring)
{
    // Quantises tokens [T0, T) of a stream whose first T0 tokens are already in the cache; kv_new
    // holds the T - T0 new rows; state_in is the state after token T0-1 (ignored when T0 == 0).
    static_assert(CPL == 1 || CPL == 2, "one channel per lane, or one packed pair");
    constexpr int TPW = Code<BITS>::TPW; // tokens per channel word
    constexpr int G8 = TPW / 8;          // 8-token input groups per word
    constexpr int PF = CPL == 1 ? ENC_PF1 : ENC_PF2;
    constexpr int AHEAD = CPL == 1 ? ENC_AHEAD1 : PF - 1;
    // a wave's 64 * CPL channels lie inside one head (D is a multiple of 128), so everything but
    // the channel itself is uniform over the wave and a wave past the end has no work at all
    const int lane = threadIdx.x & 63;
    const long ci = ((long)blockIdx.x * BLK + (threadIdx.x & ~63)) * CPL; // the wave's first channel
    if (ci >= (long)BH * D)
        return;
    const int bx = __builtin_amdgcn_readfirstlane((int)(ci / D));
    const int cw0 = __builtin_amdgcn_readfirstlane((int)(ci % D));
    const int c0 = cw0 + lane * CPL;
    const int h = bx % H;

    Pair st;
    if (CPL == 2) {
        load_pair(st, zp, sc, al, be, tg, h * D + c0);
    } else {
        const int pi = h * D + c0;
        st.zp = splat(zp[pi]);
        st.sc = splat(sc[pi]);
        st.al = splat(al[pi]);
        st.be = splat(be[pi]);
        st.omt = splat((h1)1.0f) - st.be * splat(tg[pi]);
    }
    if (T0 > 0) {
        const h1 *si = state_in + ((size_t)bx * D + c0) * 2;
        if (CPL == 2) {
            load_state<2>(si, &st);
        } else {
            st.zp = splat(si[0]);
            st.sc = splat(si[1]);
        }
    }

    uint32_t *cw = cache + (size_t)bx * n_super_cap * D + cw0;                                 // the wave's code words
    const h1 *xb = kv_new + (long)(bx / H) * xs.b + (long)h * xs.h + cw0 - (long)T0 * xs.t;    // its row of token 0

    // one token's input: a word with an fp16 (or bf16) pair, or one 16-bit value
    using XW = typename std::conditional<CPL == 2, uint32_t, uint16_t>::type;
    auto as_f16 = [](XW w) -> XW {
        if (!BF16)
            return w;
        // bf16 -> fp32 is exact, fp32 -> fp16 rounds to nearest even: torch's .to(float16)
        const h1 lo = (h1)__uint_as_float((uint32_t)w << 16);
        if constexpr (CPL == 1)
            return __builtin_bit_cast(uint16_t, lo);
        else
            return as_u32((h2){lo, (h1)__uint_as_float(w & 0xFFFF0000u)});
    };
    // exact step with the IEEE divide: partial words and runs that met a NaN
    auto step = [&](XW xw, int *qi) {
        const h2 x = as_h2((uint32_t)as_f16(xw));
        qi[0] = quantize<BITS>(x.x, st.zp.x, st.sc.x);
        if (CPL == 2)
            qi[1] = quantize<BITS>(x.y, st.zp.y, st.sc.y);
        const h2 q = codes_to_h2(qi[0], qi[CPL - 1]);
        update_pair(st, q, q * st.sc);
    };
    auto load_tok = [&](int t) { return *reinterpret_cast<const XW *>(xb + (long)t * xs.t + lane * CPL); };
    // Checkpoints: entry j is the state before token (j+1)*interval.  Words are stored in order,
    // so the next boundary is tracked by comparison instead of a division per word.
    int ck_next = -1, ck_j = 0;
    if (sa.ckpt != nullptr) {
        const int first_end = (T0 / TPW) * TPW + TPW;
        ck_j = (first_end + sa.ckpt_interval - 1) / sa.ckpt_interval - 1;
        ck_next = (ck_j + 1) * sa.ckpt_interval;
    }
    auto checkpoint = [&](int tend) {
        if (__builtin_expect(tend != ck_next, 1))
            return;
        if (tend <= T && ck_j < sa.n_ckpt_cap)
            store_state_n<CPL>(sa.ckpt + (((size_t)bx * sa.n_ckpt_cap + ck_j) * D + c0) * 2, &st);
        ck_next += sa.ckpt_interval;
        ck_j++;
    };
    // a word of which only the codes of tokens [lo, hi) are new (codes below lo are kept, the fields
    // from hi on are zero)
    auto partial_word = [&](int sg, int lo, int hi) {
        uint32_t *dst = cw + (size_t)sg * D + lane * CPL;
        const uint32_t keep = lo ? (1u << (BITS * lo)) - 1u : 0u;
        uint32_t w[CPL];
#pragma unroll
        for (int c = 0; c < CPL; c++)
            w[c] = keep ? dst[c] & keep : 0u;
        for (int tt = lo; tt < hi; tt++) {
            int qi[CPL];
            step(load_tok(sg * TPW + tt), qi);
#pragma unroll
            for (int c = 0; c < CPL; c++)
                w[c] |= (uint32_t)(qi[c] - Code<BITS>::QLO) << (BITS * tt);
        }
#pragma unroll
        for (int c = 0; c < CPL; c++)
            dst[c] = w[c];
        checkpoint(sg * TPW + TPW);
    };

    // a stream that resumes inside a word first completes it
    int sg = T0 / TPW;
    if (T0 % TPW && T0 < T) {
        partial_word(sg, T0 % TPW, T / TPW == sg ? T % TPW : TPW);
        sg++;
    }

    // Full words.  MAGIC + n is exact for the integers that matter, and its low bits are those of n.
    // With two channels n is biased by -QLO, so that they are the stored code (the byte permute
    // needs it non-negative); with one they are n's two's complement, as v_cvt_f16_i16 takes it, and
    // the finished word is biased (an exclusive or with the sign bits).
    constexpr float BIASF = CPL == 2 ? (float)-Code<BITS>::QLO : 0.0f;
    constexpr uint32_t WORD_BIAS = CPL == 2 ? 0u : Code<BITS>::BIAS;
    constexpr float MAGIC = 12582912.0f + BIASF; // 1.5 * 2^23
    constexpr float ULO = MAGIC + (float)Code<BITS>::QLO, UHI = MAGIC + (float)Code<BITS>::QHI;
    float uhi = UHI; // med3 takes one scalar operand
    asm volatile("" : "+v"(uhi));
    uint32_t w[CPL];
    float nan = 0.0f; // becomes a NaN when a quotient was one
    // two channels: the scale in fp32 and its reciprocal
    float scf[2], rs[2];
    // one channel: see enc_eight_tokens
    Chan1 ch;
    auto enter = [&]() {
        if (CPL == 1) {
            ch.zp = as_u32(st.zp);
            ch.qs_sc = as_u32((h2){(h1)0.0f, st.sc.x});
            ch.s = (float)st.sc.x;
        } else {
            scf[0] = (float)st.sc.x;
            scf[1] = (float)st.sc.y;
            rs[0] = __builtin_amdgcn_rcpf(scf[0]);
            rs[1] = __builtin_amdgcn_rcpf(scf[1]);
        }
        nan = 0.0f;
    };
    auto leave = [&]() {
        if (CPL == 1) {
            st.zp = splat(as_h2(ch.zp).x);
            st.sc = splat(as_h2(ch.qs_sc).y);
        }
    };
    auto tokens8 = [&](const XW *x) {
        if constexpr (CPL == 1) {
            uint16_t y[8];
#pragma unroll
            for (int k = 0; k < 8; k++)
                y[k] = as_f16(x[k]);
            enc_eight_tokens<BITS>(ch, y, as_u32(st.al), as_u32(st.be), as_u32(st.omt), ULO, uhi, w[0], nan);
        } else {
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const uint32_t xw = as_f16(x[k]), zw = as_u32(st.zp);
                const float r0 = enc_quotient(enc_diff<false>(xw, zw), scf[0], rs[0]);
                const float r1 = enc_quotient(enc_diff<true>(xw, zw), scf[1], rs[1]);
                const uint32_t u0 = __float_as_uint(__builtin_amdgcn_fmed3f(r0 + MAGIC, ULO, uhi));
                const uint32_t u1 = __float_as_uint(__builtin_amdgcn_fmed3f(r1 + MAGIC, ULO, uhi));
                w[0] = __builtin_amdgcn_alignbit(u0, w[0], BITS);
                w[CPL - 1] = __builtin_amdgcn_alignbit(u1, w[CPL - 1], BITS);
                nan = enc_collect_nan(nan, r0, r1);
                // bytes 3 and 0 of each: 0x4B, code = the fp16 number 14 + code/128
                const h2 b = as_h2(__builtin_amdgcn_perm(u1, u0, 0x07040300u));
                const h2 q = pk_fma(b, splat((h1)128.0f), splat((h1)(-1792.0f - BIASF)));
                update_pair(st, q, q * st.sc);
                scf[0] = (float)st.sc.x;
                scf[1] = (float)st.sc.y;
                rs[0] = __builtin_amdgcn_rcpf(scf[0]);
                rs[1] = __builtin_amdgcn_rcpf(scf[1]);
            }
        }
    };
    // Streams longer than what a buffer descriptor can span are taken in pieces (and rows too far
    // apart for one word's worth in a descriptor the slow way).
    if (xs.t > (1L << 24))
        for (; (sg + 1) * TPW <= T; sg++)
            partial_word(sg, 0, TPW);
    const int sg_end = T / TPW;
    const long span_words = (1L << 30) / (xs.t * 2 * TPW);
    int redo = PF / G8, resumed = -1; // words done with the plain division after a NaN; where the last such stretch ended
    bool through_lds = CPL == 1 && ring != nullptr && ((uintptr_t)(xb + (long)sg * TPW * xs.t) & 15) == 0 && xs.t % 8 == 0 &&
                       (sa.ckpt == nullptr || (sa.ckpt_interval % 64 == 0 && sg * TPW % 64 == 0));
    const int piece = (int)(span_words >= PF ? span_words / PF * PF : max(span_words, 1L)); // whole runs where it can
    while (sg < sg_end) {
        const int sg_piece = sg, nw = min(piece, sg_end - sg), ng = nw * G8; // words, 8-token groups of this piece
        const uint32_t xbytes = (uint32_t)(((long)ng * 8 - 1) * xs.t * 2 + 128 * CPL);
        if constexpr (CPL == 1) {
            // Whole runs of 64 tokens whose rows come through the LDS (enc_run64), a run ahead: 64 tokens or 2 us.  Rows have
            // to be 16-byte aligned; a run that meets a NaN, and all after it, go through the loop below.
            if (through_lds && ng >= 8 && (sa.ckpt == nullptr || sg * TPW % 64 == 0)) {
                constexpr int WORDS = 8 / G8;
                const uint64_t base = wave_uniform((uint64_t)(xb + (long)sg * TPW * xs.t));
                const rsrc4 rows = {(uint32_t)base, (uint32_t)(base >> 32), xbytes, 0x00027000u};
                const uint32_t row = (uint32_t)(xs.t * 2), lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(
                    __attribute__((address_space(3))) char *)ring);
                uint32_t off = (uint32_t)(lane >> 3) * row + (uint32_t)(lane & 7) * 16u, half = 0;
                // lane i of 16 reads token i / 4, channels 4 * (i % 4).. of its 16-channel group
                const uint32_t addr = lds + (uint32_t)((lane & 15) >> 2) * 128u + (uint32_t)(lane >> 4) * 32u + (uint32_t)(lane & 3) * 8u;
                auto load_run = [&](uint32_t to) __attribute__((always_inline)) { // past the end: dropped by the bounds check
#pragma unroll
                    for (int k = 0; k < 8; k++) {
                        load_to_lds(to + (uint32_t)k * 1024u, off, rows);
                        off += row * 8u;
                    }
                };
                uint32_t *dst = cw + (size_t)sg * D + lane;
                const uint32_t nal = as_u32(st.al) ^ 0x80008000u;
                load_run(lds);
                for (int g = 0; g + 8 <= ng; g += 8) {
                    load_run(lds + (half ^ 8192u));
                    // everything but the next run's eight loads and, from the second run on, the codes just
                    // stored (all of them complete in order)
                    if (g == 0)
                        asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
                    else if (WORDS == 8)
                        asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
                    else
                        asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
                    Chan1Neg ch = {as_u32(st.zp), as_u32((h2){-st.sc.x, (h1)0.0f}), -(float)st.sc.x};
                    uint32_t w[WORDS];
                    float nan = 0.0f;
                    enc_run64<BITS, BF16>(ch, addr + half, nal, as_u32(st.be), as_u32(st.omt), MAGIC, ULO, uhi, w, nan);
                    nan = enc_collect_nan(nan, ch.nsc, (float)as_h2(ch.zp).x);
                    if (__builtin_expect(__any(nan != nan), 0)) {
                        through_lds = false;
                        break;
                    }
                    st.zp = splat(as_h2(ch.zp).x);
                    st.sc = splat(-as_h2(ch.ss).x);
#pragma unroll
                    for (int k = 0; k < WORDS; k++)
                        dst[(size_t)k * D] = w[k] ^ WORD_BIAS;
                    dst += (size_t)WORDS * D;
                    sg += WORDS;
                    checkpoint(sg * TPW);
                    half ^= 8192u;
                }
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // nothing is on its way into the LDS any more
                // The words behind the last whole run: their rows are in the LDS already, and no checkpoint lies
                // inside them.  (Loaded again for the loop below they cost a short stream 1 of its 13 to 25 us.)
                const int words = (sg_piece + nw) - sg;
                if (through_lds && words > 0) {
                    typedef const volatile __attribute__((address_space(3))) uint16_t *LdsRows;
                    const LdsRows tail = (LdsRows)(lds + half) + lane;
                    const Pair saved = st;
                    enter();
                    for (int k = 0; k < words * G8; k++) {
                        XW x[8];
#pragma unroll
                        for (int tt = 0; tt < 8; tt++)
                            x[tt] = (XW)tail[(k * 8 + tt) * 64];
                        tokens8(x);
                        if (k % G8 == G8 - 1) {
                            *dst = w[0] ^ WORD_BIAS;
                            dst += D;
                        }
                    }
                    leave();
                    if (__builtin_expect(__any(nan != nan), 0)) {
                        st = saved;
                        through_lds = false;
                    } else {
                        sg += words;
                    }
                }
                continue;
            }
        }
        const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
            (void *)wave_uniform((uint64_t)(xb + (long)sg * TPW * xs.t)), 0, (int)xbytes, 0x00027000);
        uint32_t xoff = (uint32_t)lane * 2u * CPL;
        const uint32_t row = (uint32_t)(xs.t * 2);
        XW xbuf[PF][8];
        auto load_next = [&](XW *xg) {
#pragma unroll
            for (int tt = 0; tt < 8; tt++)
                xg[tt] = CPL == 2 ? (XW)__builtin_amdgcn_raw_buffer_load_b32(xr, (int)xoff, (int)(row * tt), 0)
                                  : (XW)__builtin_amdgcn_raw_buffer_load_b16(xr, (int)xoff, (int)(row * tt), 0);
            xoff += row * 8;
        };
        uint32_t *dst = cw + (size_t)sg * D + lane * CPL;
        // group k of a run that starts at word sg; a word is stored when its last group is done
        auto do_group = [&](auto kc, XW *xg, auto may_checkpoint) {
            constexpr int k = decltype(kc)::value;
            // one wait for the group's rows instead of one per token
            asm volatile("" ::"v"(xg[0]), "v"(xg[1]), "v"(xg[2]), "v"(xg[3]), "v"(xg[4]), "v"(xg[5]), "v"(xg[6]), "v"(xg[7]));
            tokens8(xg);
            if constexpr (k % G8 == G8 - 1) {
                if (CPL == 2)
                    *reinterpret_cast<uint2 *>(dst) = make_uint2(w[0], w[CPL - 1]);
                else
                    *dst = w[0] ^ WORD_BIAS;
                dst += D;
                if constexpr (decltype(may_checkpoint)::value) {
                    leave();
                    checkpoint((sg + k / G8 + 1) * TPW);
                }
            }
        };
        // Quotients are looked at once per run of groups.  False: one of them was a NaN, and everything
        // but the code words is as it was before the run.
        auto run = [&](int words, auto &&groups) -> bool {
            const Pair saved = st;
            const int saved_next = ck_next, saved_j = ck_j;
            groups();
            leave();
            if (__builtin_expect(__any(nan != nan), 0)) {
                st = saved;
                ck_next = saved_next;
                ck_j = saved_j;
                return false;
            }
            sg += words;
            return true;
        };
        enter();
#pragma unroll
        for (int i = 0; i < AHEAD; i++)
            load_next(xbuf[i]);
        int g = 0;
        bool clean = true;
        // Two copies of the loop rather than a test in it: where the paths met again, the buffers
        // in flight would be copied, and waited for.
        auto runs = [&](auto inner_checkpoints) __attribute__((always_inline)) {
            for (; g + PF <= ng; g += PF) {
                clean = run(PF / G8, [&]() __attribute__((always_inline)) {
                    static_for<PF>([&](auto ic) __attribute__((always_inline)) {
                        // loads moved up over the last use of their buffer would be copied into it
                        __builtin_amdgcn_sched_barrier(0);
                        load_next(xbuf[(decltype(ic)::value + AHEAD) % PF]);
                        __builtin_amdgcn_sched_barrier(0);
                        do_group(ic, xbuf[decltype(ic)::value], inner_checkpoints);
                    });
                });
                if (!clean)
                    return;
                if constexpr (!decltype(inner_checkpoints)::value)
                    checkpoint(sg * TPW);
            }
        };
        // Checkpoint boundaries fall between runs (every 64 tokens with one channel per lane) for any
        // usual interval and a stream that starts at one; only other plans look after every word.
        if (sa.ckpt == nullptr || (sa.ckpt_interval % (8 * PF) == 0 && sg * TPW % (8 * PF) == 0))
            runs(std::integral_constant<bool, false>{});
        else
            runs(std::integral_constant<bool, true>{});
        if (clean && g < ng) // at most PF-1 groups, whole words; the first AHEAD of their inputs are in xbuf already
            clean = run((ng - g) / G8, [&]() __attribute__((always_inline)) {
                static_for<PF - 1 - AHEAD>([&](auto ic) __attribute__((always_inline)) { load_next(xbuf[AHEAD + decltype(ic)::value]); });
                static_for<PF - 1>([&](auto ic) __attribute__((always_inline)) {
                    if (g + decltype(ic)::value < ng)
                        do_group(ic, xbuf[decltype(ic)::value], std::integral_constant<bool, true>{});
                });
            });
        if (clean)
            continue;
        // The run that met a NaN again with the plain division, the rows of the next group on their way
        // during this one's steps; then the loop above starts anew behind it.  A channel whose scale is
        // zero, or whose state is a NaN, meets one in every run: as long as no run is clean, twice as many
        // words are taken here each time (up to 16 runs), so that such a wave hardly tries the fast form:
        // 83 ns per token of one channel against 34 of whole runs (145 with a load per token).
        redo = sg == resumed ? min(redo * 2, 16 * (PF / G8)) : PF / G8;
        dst = cw + (size_t)sg * D + lane * CPL;
        xoff = (uint32_t)lane * 2u * CPL + row * 8u * (uint32_t)g;
        load_next(xbuf[0]);
        for (int left = min(redo * G8, ng - g); left > 0; left--) {
            XW x[8];
#pragma unroll
            for (int tt = 0; tt < 8; tt++)
                x[tt] = xbuf[0][tt];
            load_next(xbuf[0]);
#pragma unroll
            for (int tt = 0; tt < 8; tt++) {
                int qi[CPL];
                step(x[tt], qi);
#pragma unroll
                for (int c = 0; c < CPL; c++)
                    w[c] = __builtin_amdgcn_alignbit((uint32_t)(qi[c] - Code<BITS>::QLO), w[c], BITS);
            }
            if (G8 == 1 || (left & 1)) { // whole words: an odd number of groups is left at a word's last
#pragma unroll
                for (int c = 0; c < CPL; c++)
                    dst[c] = w[c];
                dst += D;
                checkpoint(++sg * TPW);
            }
        }
        resumed = sg;
    }
    // ragged last word: codes of the tokens present, zero fields after them
    if (T0 < T && sg * TPW < T)
        partial_word(sg, 0, T - sg * TPW);
    if (sa.fresh) { // free slots are zero, as the appending kernels expect
        for (int i = (T + TPW - 1) / TPW; i < n_super_cap; i++)
#pragma unroll
            for (int c = 0; c < CPL; c++)
                cw[(size_t)i * D + lane * CPL + c] = 0u;
        if (sa.ckpt != nullptr)
            for (int j = T / sa.ckpt_interval; j < sa.n_ckpt_cap; j++)
#pragma unroll
                for (int c = 0; c < CPL; c++)
                    reinterpret_cast<uint32_t *>(sa.ckpt)[((size_t)bx * sa.n_ckpt_cap + j) * D + c0 + c] = 0u;
    }
    if (state_out != nullptr)
        store_state_n<CPL>(state_out + ((size_t)bx * D + c0) * 2, &st);
}

// five waves per SIMD with two channels per lane (many waves): 96 registers
template <int BITS, int CPL, int BLK>
__global__ __launch_bounds__(BLK, CPL == 2 ? 5 : 1) void encode_kernel(
    uint32_t *__restrict__ cache, const h1 *__restrict__ kv_new,
    const h1 *__restrict__ zp, const h1 *__restrict__ sc, const h1 *__restrict__ al,
    const h1 *__restrict__ be, const h1 *__restrict__ tg,
    int BH, int H, int T0, int T, int D, int n_super_cap, const h1 *__restrict__ state_in,
    h1 *__restrict__ state_out, Seg sa)
{
    const RowStrides packed = {(long)H * (T - T0) * D, (long)(T - T0) * D, (long)D};
    __shared__ uint4 ring[CPL == 1 ? BLK / 64 * ENC_RING / 16 : 1];
    encode_body<BITS, CPL, BLK>(cache, kv_new, packed, zp, sc, al, be, tg, BH, H, T0, T, D, n_super_cap,
                                state_in, state_out, sa, enc_ring<CPL>(ring));
}

// Two tensors of one shape (the K and V rows of the same tokens) in one launch: blockIdx.y picks
// the tensor.  A prompt with few channels (small batch) leaves SIMDs idle when the tensors are
// encoded one after the other; together they run in the time of one.
struct EncTensor {
    uint32_t *cache;
    const h1 *kv_new, *zp, *sc, *al, *be, *tg, *state_in;
    h1 *state_out, *ckpt;
    RowStrides xs;
};

// BF16: the new rows are bfloat16 (same strides, in elements) and are rounded to fp16 on the fly.
template <int BITS, int CPL, int BLK, bool BF16>
__global__ __launch_bounds__(BLK, CPL == 2 ? 5 : 1) void encode_pair_kernel(EncTensor k, EncTensor v, int BH, int H,
                                                          int T0, int T, int D, int n_super_cap,
                                                          Seg sa)
{
    const EncTensor e = blockIdx.y ? v : k;
    sa.ckpt = e.ckpt;
    __shared__ uint4 ring[CPL == 1 ? BLK / 64 * ENC_RING / 16 : 1];
    encode_body<BITS, CPL, BLK, BF16>(e.cache, e.kv_new, e.xs, e.zp, e.sc, e.al, e.be, e.tg, BH, H, T0,
                                      T, D, n_super_cap, e.state_in, e.state_out, sa, enc_ring<CPL>(ring));
}

// Shared tail of the two decode kernels: quantise the new token with the state after token T-1,
// patch it into slot T, return the fused dequant r16(q*sc + zp) per pair (gemv.cu:744-798,
// 1105-1157).  The state is NOT advanced.
template <int D, int CPL, int BITS = 4>
__device__ __forceinline__ void append_new_token(typename Geo<D, CPL>::Vec *cb, int T, const h1 *xnew, const Pair *st,
                                                 h2 *deq, bool active, int act_bf16 = 0)
{
    using G = Geo<D, CPL>;
    const int sg = T / Code<BITS>::TPW, tt = T % Code<BITS>::TPW;
#pragma unroll
    for (int v = 0; v < G::NV; v++) {
        typename G::Vec *slot = cb + (size_t)sg * G::VPS + v;
        typename G::Vec u = *slot;
        uint32_t w[G::WPV];
        vec_words(u, w);
#pragma unroll
        for (int pp = 0; pp < G::WPV / 2; pp++) {
            const int p = (G::WPV / 2) * v + pp;
            const h2 x = load_act2(xnew + 2 * p, act_bf16);
            const h2 q = append_pair<BITS>(w[2 * pp], w[2 * pp + 1], tt, x, st[p]);
            deq[p] = pk_fma(q, st[p].sc, st[p].zp);
        }
        if (active) {
            words_vec(w, u);
            *slot = u;
        }
    }
}

// What the last segment does once it holds the state after token T-1: hand it out, and record it
// as a checkpoint when token T opens a new checkpoint interval.
template <int D, int CPL>
__device__ __forceinline__ void publish_state(const Pair *st, h1 *state_out, const Seg &sa, int bx,
                                              int c0, int T)
{
    if (state_out != nullptr)
        store_state<CPL>(state_out + ((size_t)bx * D + c0) * 2, st);
    if (sa.ckpt != nullptr && T > 0 && T % sa.ckpt_interval == 0) {
        const int j = T / sa.ckpt_interval - 1;
        if (j < sa.n_ckpt_cap)
            store_state<CPL>(sa.ckpt + (((size_t)bx * sa.n_ckpt_cap + j) * D + c0) * 2, st);
    }
}

template <int D, int CPL>
__device__ __forceinline__ void pair_bytes_of(const typename Geo<D, CPL>::Vec *u, uint32_t (*nb)[2])
{
    using G = Geo<D, CPL>;
#pragma unroll
    for (int v = 0; v < G::NV; v++) {
        uint32_t w[G::WPV];
        vec_words(u[v], w);
#pragma unroll
        for (int pp = 0; pp < G::WPV / 2; pp++)
            pair_bytes(w[2 * pp], w[2 * pp + 1], nb[(G::WPV / 2) * v + pp][0], nb[(G::WPV / 2) * v + pp][1]);
    }
}

// ---------------------------------------------------------------------------------------------
// forward_qk  (gemv.cu:435-815)
// ---------------------------------------------------------------------------------------------
// Per lane and supergroup: 8 fp32 partial logits (v_dot2_f32_f16 over the lane's channel pairs).
// They are summed across the head's lanes and scattered by reduce8_head (masked DPP adds and row
// swaps, no LDS): afterwards every quad of lanes holds the total of one token.
typedef _Float16 h8v __attribute__((ext_vector_type(8))); // operand of v_mfma_f32_16x16x32_f16
constexpr int PAIR_TILE = 16 * 256; // bytes of a wave's key tile

// Entries of one unit of eight tokens of a lane's channel pair: e[t] for token t.
template <int BITS>
__device__ __forceinline__ void pair_lookup(uint2 *e, const uint2 *lut, const uint32_t *nb, uint32_t lane_copy, int unit)
{
    if constexpr (BITS == 4) {
#pragma unroll
        for (int t = 0; t < 8; t++)
            e[t] = lut_get(lut, nb[t & 1], lane_copy, t >> 1);
    } else { // an entry is tokens s and s + 2
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const int t = 4 * (s >> 1) + (s & 1);
            const uint4 v = lut2_get(lut, nb[s & 1], lane_copy, 2 * unit + (s >> 1));
            e[t] = make_uint2(v.x, v.y);
            e[t + 2] = make_uint2(v.z, v.w);
        }
    }
}

// forward_qk of a segment with the head over a whole wave, two channels per lane, for GQ query heads.
// A wave has its SIMD (nearly) to itself and pays for every instruction, so what is left per
// token is the lookup, the replay (replay_eight) and half a write: the values of 16 tokens go
// to an LDS tile, from which the matrix cores take them as columns against the queries as
// rows.  Row r is head r * GQ / 16, so that lane (token, quarter of the rows) receives its head's
// logit of its token as it is, and nothing is summed across lanes.  ~10 issue slots per token
// where the dot product, its reduction over the lanes and the wait states made it 19
// (32 x 32 heads x 1024 tokens, one segment: 49 -> 34 us).
// The tile: row t = token t, 256 bytes; its 16-byte pieces are permuted by (t / 2) % 8 so that
// both halves of an access to 16 rows at once spread over the banks.
// LONE: workgroups of 256 threads, a wave with a SIMD's registers to itself; the compiler keeps products in
// accumulation registers there and in vector registers elsewhere.
template <int BITS, int GQ, bool LONE>
struct PairScores {
    using G = Geo<128, 2>;
    using Vec = G::Vec;
    static constexpr int TPW = Code<BITS>::TPW, UPS = TPW / 8; // tokens, units of eight tokens per supergroup
    static constexpr int AHEAD = PF_PAIR / UPS;                // supergroups in flight
    char *tile;
    int lane;
    h8v qa[4], kv[4];
    f4v d;
    int rd[4], wr[8];

    // loads the queries (rows are 8-byte aligned); ready() once the rest of the workgroup's loads are out
    __device__ __forceinline__ PairScores(char *tile_, int lane_, const h1 *q) : tile(tile_), lane(lane_)
    {
        const int row = lane & 15, kb = lane >> 4;
#pragma unroll
        for (int m = 0; m < 4; m++) {
            const uint2 *src = reinterpret_cast<const uint2 *>(q + (row * GQ >> 4) * 128 + m * 32 + kb * 8);
            const uint2 a = src[0], b = src[1];
            qa[m] = __builtin_bit_cast(h8v, make_uint4(a.x, a.y, b.x, b.y));
        }
    }
    __device__ __forceinline__ void ready(int act_bf16)
    {
        const int row = lane & 15, kb = lane >> 4;
#pragma unroll
        for (int m = 0; m < 4; m++) {
            if (act_bf16) {
                const uint4 u = __builtin_bit_cast(uint4, qa[m]);
                qa[m] = __builtin_bit_cast(h8v, make_uint4(as_u32(act2(u.x, 1)), as_u32(act2(u.y, 1)),
                                                           as_u32(act2(u.z, 1)), as_u32(act2(u.w, 1))));
            }
            kv[m] = (h8v){};
            rd[m] = row * 256 + (((m * 4 + kb) ^ (row >> 1)) << 4);
        }
#pragma unroll
        for (int j = 0; j < 8; j++)
            wr[j] = (lane * 4) ^ (j << 4);
    }
    // this lane's channel pair of the token in `row` of the tile
    __device__ __forceinline__ void write(int row, uint32_t x)
    {
        *reinterpret_cast<uint32_t *>(tile + row * 256 + ((lane * 4) ^ (row >> 1 << 4))) = x;
    }
    __device__ __forceinline__ void fetch()
    {
#pragma unroll
        for (int m = 0; m < 4; m++)
            kv[m] = *reinterpret_cast<const h8v *>(tile + rd[m]);
    }
    __device__ __forceinline__ void multiply()
    {
        d = (f4v){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int m = 0; m < 4; m++)
            d = __builtin_amdgcn_mfma_f32_16x16x32_f16(qa[m], kv[m], d, 0, 0, 0);
    }
    // put(token, head, logit) for the first ntok tokens of the tile that starts at `token`
    template <typename PUT>
    __device__ __forceinline__ void emit(int token, int ntok, PUT &&put)
    {
        // All of d is held up to here: registers of it that nobody reads would go to the hand-laid block behind
        // multiply() while the matrix cores have yet to write them, and the compiler waits for no block.  (With 2-bit
        // codes the block wrote one of them an instruction later; at two waves per SIMD its value was lost.)  In the
        // registers where it is: moved into the others, it took a lone wave 12 instructions per 64 tokens (1 x 32 heads x
        // 603 tokens with the rotary embedding 21.19 us, 21.08 where they are).
        if constexpr (LONE)
            asm volatile("" ::"a"(d));
        else
            asm volatile("" ::"v"(d));
        const int t = lane & 15, quarter = lane >> 4;
        if (t >= ntok || (GQ == 1 && quarter) || (GQ == 2 && (quarter & 1)))
            return;
        if constexpr (GQ == 8) {
            put(token + t, 2 * quarter, (h1)d.x);
            put(token + t, 2 * quarter + 1, (h1)d.z);
        } else {
            put(token + t, quarter * GQ >> 2, (h1)d.x);
        }
    }

    // all whole supergroups of a segment; put is given tokens from 0
    template <typename PUT>
    __device__ __forceinline__ void run(const uint2 *lut, uint32_t lane_copy, Pair &st, SegLoads<128, 2, BITS, AHEAD> &s, PUT &&put)
    {
        const int nfull = s.nfull;
        if (nfull <= 0)
            return;
        const Vec *cb = s.cb;
        auto &buf = s.buf;
        uint2 e[2][8];
        uint32_t nb[2];
        auto bytes = [&](const Vec &u) __attribute__((always_inline)) {
            if constexpr (BITS == 4)
                pair_bytes(u.x, u.y, nb[0], nb[1]);
            else
                pair_bytes2(u.x, u.y, nb[0], nb[1]);
        };
        auto lookup = [&](uint2 *l, int unit) __attribute__((always_inline)) { pair_lookup<BITS>(l, lut, nb, lane_copy, unit); };
        // no scalar load in flight when the loop starts: its waits would have to cover it
        bytes(buf[0][0]);
        lookup(e[0], 0);
        wait_lgkm();
        rotate_over<AHEAD>(nfull, [&](int sg, auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value;
            static_for<UPS>([&](auto hc) __attribute__((always_inline)) {
                constexpr int hf = decltype(hc)::value, half = (i * UPS + hf) & 1;
                const int unit = sg * UPS + hf;
                if constexpr (hf == UPS - 1) {
                    bytes(buf[(i + 1) % AHEAD][0]); // stale past the end: looked up, never used
                    lookup(e[half ^ 1], 0);
                    buf[i][0] = load_codes(cb + (size_t)min(sg + AHEAD, nfull - 1) * G::VPS);
                } else {
                    lookup(e[half ^ 1], hf + 1);
                }
                __builtin_amdgcn_sched_barrier(0);
                uint32_t kh[8];
                replay_eight(st, e[half], kh);
#pragma unroll
                for (int t = 0; t < 8; t++)
                    *reinterpret_cast<uint32_t *>(tile + (half * 8 + t) * 256 + wr[half * 4 + t / 2]) = kh[t];
                __builtin_amdgcn_sched_barrier(0);
                // the tile before this one: fetched when it was complete, multiplied half a tile later,
                // stored another half later
                if constexpr (half == 0) {
                    multiply();
                } else {
                    emit((unit - 3) * 8, unit > 1 ? 16 : 0, put);
                    fetch();
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        });
        const int last = nfull * UPS - 1;
        if (last & 1) {
            multiply();
            emit((last - 1) * 8, 16, put);
        } else { // half a tile, and the one before it is not stored yet
            emit((last - 2) * 8, last > 0 ? 16 : 0, put);
            fetch();
            multiply();
            emit(last * 8, 8, put);
        }
    }
};


// forward_qk of one (head, segment), from the loads that s.start() and the caller have sent off.
// Writes the segment's logits to out + bx * row_pitch and, with the context's last segment, appends.
template <int D, int CPL, bool LONE>
__device__ __forceinline__ void qk_segment(const uint2 *lut, uint32_t lane_copy, int lane, int bx, int lh, int c0, bool active,
                                           PairScores<4, 1, LONE> &scores, SegLoads<D, CPL, 4, CPL == 2 ? PF_PAIR : PF> &s,
                                           const uint32_t *qw, const h1 *k_new, h1 *out, int T, h1 *state_out, const Seg &sa)
{
    using G = Geo<D, CPL>;
    using Vec = typename G::Vec;
    constexpr bool PAIR = CPL == 2; // the head fills the wave: see PairScores
    Pair st[G::NP];
    h2 qv[G::NP];
    s.state(st);
#pragma unroll
    for (int p = 0; p < G::NP; p++)
        qv[p] = act2(qw[p], sa.act_bf16);

    const bool last = s.last;
    const int t0 = s.t0, t1 = s.t1, nfull = s.nfull;
    Vec *cbh = s.cbh;
    const Vec *cb = s.cb;
    h1 *ob = out + (size_t)bx * sa.row_pitch + t0;
    // the token whose total this lane's quad ends up with, and the one lane per token that stores
    // it (a 64-lane head holds every total twice, once per half)
    const int tk = token_of_lane(lane);
    const bool storer = active && (lane & 3) == 0 && (G::LPH == 32 || lane < 32);
    auto finish = [&](const float *part, int sg, int ntok) {
        const float s = reduce8_head<G::LPH>(part);
        if (storer && tk < ntok)
            ob[sg * 8 + tk] = (h1)s;
    };

    if constexpr (PAIR) {
        scores.ready(sa.act_bf16);
        scores.run(lut, lane_copy, st[0], s, [&](int t, int, h1 v) __attribute__((always_inline)) {
            if (active)
                ob[t] = v;
        });
    } else {
        // ---- software pipeline over the full supergroups.  Global loads run PF supergroups ahead.
        // Table lookups run one supergroup ahead and are issued token by token between the arithmetic
        // of the current supergroup (the LDS counter holds only 15 outstanding operations, so issuing a
        // whole supergroup's lookups at once would stall on them).  The logits of supergroup sg-1 are
        // reduced and stored at the start of iteration sg, while the first lookups are in flight.
        // The lookup for the next supergroup goes into the slot the current token has just vacated, so
        // one supergroup's worth of registers holds both.
        auto token = [&](int t, uint2 (*e)[8], const uint32_t (*nb)[2], float &out_t) {
            float acc;
#pragma unroll
            for (int p = 0; p < G::NP; p++) {
                Pair &s = st[p];
                const h2 qs = as_h2(e[p][t].x) * s.sc;
                const h2 kh = qs + s.zp;
                if (p == 0)
                    acc = dot2_from_zero(qv[p], kh);
                else
                    acc = __builtin_amdgcn_fdot2(qv[p], kh, acc, false);
                update_pair_abs(s, as_h2(e[p][t].y), qs);
            }
            out_t = acc;
#pragma unroll
            for (int p = 0; p < G::NP; p++)
                e[p][t] = lut_get(lut, nb[p][t & 1], lane_copy, t >> 1);
            __builtin_amdgcn_sched_barrier(0);
        };

        auto &buf = s.buf;
        uint2 lk[G::NP][8];
        uint32_t nb[G::NP][2];
        float part[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        if (nfull > 0) {
            pair_bytes_of<D, CPL>(buf[0], nb);
#pragma unroll
            for (int t = 0; t < 8; t++)
#pragma unroll
                for (int p = 0; p < G::NP; p++)
                    lk[p][t] = lut_get(lut, nb[p][t & 1], lane_copy, t >> 1);
        }
        // One supergroup; i = its buffer in the rotation (compile-time).  Nothing in here is
        // conditional: the trip count is wave-uniform, the prefetch index is clamped, and the
        // reduction of the previous supergroup stores nothing when there is none (sg == 0).
        auto body = [&](int sg, auto ic) {
            constexpr int i = decltype(ic)::value;
            // bytes of supergroup sg+1 (stale data past the end: looked up, never used)
            pair_bytes_of<D, CPL>(buf[(i + 1) % PF], nb);
            {
                // unconditional, clamped to the segment's last supergroup: a load inside a branch
                // makes the next wait cover every load in flight, this one included
                const int sgp = min(sg + PF, nfull - 1);
#pragma unroll
                for (int v = 0; v < G::NV; v++)
                    buf[i][v] = load_codes(cb + (size_t)sgp * G::VPS + v);
            }
            __builtin_amdgcn_sched_barrier(0);
            finish(part, sg - 1, sg > 0 ? 8 : 0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < 8; t++)
                token(t, lk, nb, part[t]);
        };
        rotate_over<PF>(nfull, body);
        if (nfull > 0)
            finish(part, nfull - 1, 8);
    }
    if (!last)
        return;

    // ragged tail: T % 8 tokens of the last supergroup, state advances only for t < T
    // (gemv.cu:648-654)
    const int ntail = (t1 - t0) & 7;
    if (ntail) {
        float part[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int v = 0; v < G::NV; v++) {
            uint32_t w[G::WPV];
            vec_words(cb[(size_t)nfull * G::VPS + v], w);
#pragma unroll
            for (int pp = 0; pp < G::WPV / 2; pp++) {
                Pair &s = st[(G::WPV / 2) * v + pp];
                for (int tt = 0; tt < ntail; tt++) {
                    const uint32_t na = (w[2 * pp] >> (4 * tt)) & 0xFu;
                    const uint32_t nbb = (w[2 * pp + 1] >> (4 * tt)) & 0xFu;
                    const h2 qc = codes_to_h2((int)na - 8, (int)nbb - 8);
                    const h2 qs = qc * s.sc;
                    const float d = __builtin_amdgcn_fdot2(qv[(G::WPV / 2) * v + pp], qs + s.zp, 0.0f, false);
#pragma unroll
                    for (int k = 0; k < 8; k++)
                        part[k] += (k == tt) ? d : 0.0f;
                    update_pair(s, qc, qs);
                }
            }
        }
        finish(part, nfull, ntail);
    }

    if (active)
        publish_state<D, CPL>(st, state_out, sa, bx, c0, T);

    h2 deq[G::NP];
    append_new_token<D, CPL>(cbh, T, k_new + (size_t)bx * D + c0, st, deq, active, sa.act_bf16);
    float self = 0.0f;
#pragma unroll
    for (int p = 0; p < G::NP; p++)
        self = __builtin_amdgcn_fdot2(qv[p], deq[p], self, false);
    self = head_allreduce<G::LPH>(self);
    if (active && lh == 0)
        out[(size_t)bx * sa.row_pitch + T] = (h1)self;
}

template <int D, int CPL, int BLK>
__global__ __launch_bounds__(BLK) void qk_kernel(
    const h1 *q, uint4 *__restrict__ cache, const h1 *k_new,
    h1 *__restrict__ out,
    const h1 *zp, const h1 *sc, const h1 *al,
    const h1 *be, const h1 *tg,
    int BH, int H, int T, int n_super_cap, h1 *__restrict__ state_out, Seg sa)
{
    using G = Geo<D, CPL>;
    sa.groups = sa.groups < 0 ? -1 : 0; // no uneven plans come here (a fifth of the code was their cuts)
    constexpr bool PAIR = CPL == 2;
    // the only LDS object: the table sits at LDS offset 0 (its byte address is used as is)
    __shared__ uint2 smem[LUT_WORDS64 + (PAIR ? (BLK / 64) * PAIR_TILE / 8 : 0)];
    const uint2 *lut = smem;
    const int lane = threadIdx.x & 63;
    const uint32_t lane_copy = (uint32_t)(lane & (LUT_COPIES - 1)) * 8u;

    const Unit<D, CPL, BLK> un(BH, sa.nseg); // a padding wave's is valid too: it loads and leaves
    const int bx = un.bx, lh = un.lh, c0 = un.c0;
    const bool active = un.active;
    uint32_t qw[G::NP];
    __builtin_memcpy(qw, q + (size_t)bx * D + c0, 2 * CPL);
    PairScores<4, 1, BLK == 256> scores(reinterpret_cast<char *>(smem + LUT_WORDS64) + (threadIdx.x >> 6) * PAIR_TILE, lane,
                            q + (size_t)bx * D); // two channels per lane only
    SegLoads<D, CPL, 4, PAIR ? PF_PAIR : PF> s;
    s.start(cache, zp, sc, al, be, tg, bx % H, bx, lh, un.seg, T, n_super_cap, sa);
    lut_fill<BLK>(smem, threadIdx.x);
    __syncthreads();
    if (!un.wave_active)
        return; // padding waves

    qk_segment<D, CPL>(lut, lane_copy, lane, bx, lh, c0, active, scores, s, qw, k_new, out, T, state_out, sa);
}

// ---------------------------------------------------------------------------------------------
// forward_ov  (gemv.cu:946-1178)
// ---------------------------------------------------------------------------------------------
// acc[c] accumulates w_t * v_hat[t,c] in fp32 (fp16 operands, exact products: v_fma_mix_f32); the
// reference accumulates in fp16 for the whole sequence (gemv.cu:1087,1096).  With one segment the
// result is rounded to fp16 and stored; with several, each segment stores its fp32 partial into
// `partial` [nseg, B*H, D] and ov_finalize_kernel adds them up.
// forward_ov of one (head, segment): acc = this lane's channels.  w8(sg): the weights of the eight tokens of
// the segment's supergroup sg, of which the first WR are in wbuf; w1(t): the weight of its token t.
template <int D, int CPL, int WR, typename W8, typename W1>
__device__ __forceinline__ void ov_segment(const uint2 *lut, uint32_t lane_copy, int bx, int c0, bool active,
                                           SegLoads<D, CPL, 4, CPL == 2 ? PF_PAIR : PF> &s, uint4 *wbuf, W8 &&w8, W1 &&w1,
                                           const h1 *v_new, int T, h1 *state_out, const Seg &sa, float *acc)
{
    using G = Geo<D, CPL>;
    using Vec = typename G::Vec;
    constexpr int AHEAD = CPL == 2 ? PF_PAIR : PF;
    const bool last = s.last;
    const int t0 = s.t0, t1 = s.t1, nfull = s.nfull;
    Vec *cbh = s.cbh;
    const Vec *cb = s.cb;
    auto &buf = s.buf;
    Pair st[G::NP];
    s.state(st);
#pragma unroll
    for (int c = 0; c < CPL; c++)
        acc[c] = 0.0f;
    // Four-channel (and wider) lanes contract on the matrix cores, as ov_ft_kernel does and for the
    // reason given there: B = the lane's dequantised pair at two tokens, A = (w[t], 0, w[t+1], 0)
    // from lane 0 of each group of four, (0, w[t], 0, w[t+1]) from lane 1, zeros from lanes 2, 3.
    constexpr bool MM = CPL >= 4;
    f4v acc4[G::NP];
#pragma unroll
    for (int p = 0; p < G::NP; p++)
        acc4[p] = (f4v){0.0f, 0.0f, 0.0f, 0.0f};
    const int role = threadIdx.x & 3;
    const uint32_t sel_a0 = role == 0 ? 0x0C0C0100u : role == 1 ? 0x01000C0Cu : 0x0C0C0C0Cu;
    const uint32_t sel_a1 = role == 0 ? 0x0C0C0302u : role == 1 ? 0x03020C0Cu : 0x0C0C0C0Cu;

    // two tokens of the current supergroup on the matrix cores, then the lookups of the same two
    // slots of the next one
    auto token2 = [&](int t, uint2 (*e)[8], const uint32_t (*nb)[2], const uint4 wv) {
        const uint32_t ww[4] = {wv.x, wv.y, wv.z, wv.w};
        const uint32_t w2 = ww[t >> 1];
        const h4v a = as_h4(__builtin_amdgcn_perm(w2, w2, sel_a0), __builtin_amdgcn_perm(w2, w2, sel_a1));
        uint32_t vd[G::NP][2];
#pragma unroll
        for (int k = 0; k < 2; k++)
#pragma unroll
            for (int p = 0; p < G::NP; p++) {
                Pair &s = st[p];
                const h2 qs = as_h2(e[p][t + k].x) * s.sc;
                vd[p][k] = as_u32(qs + s.zp);
                update_pair_abs(s, as_h2(e[p][t + k].y), qs);
            }
#pragma unroll
        for (int p = 0; p < G::NP; p++)
            acc4[p] = __builtin_amdgcn_mfma_f32_4x4x4f16(a, as_h4(vd[p][0], vd[p][1]), acc4[p], 0, 0, 0);
#pragma unroll
        for (int k = 0; k < 2; k++)
#pragma unroll
            for (int p = 0; p < G::NP; p++)
                e[p][t + k] = lut_get(lut, nb[p][(t + k) & 1], lane_copy, (t + k) >> 1);
        __builtin_amdgcn_sched_barrier(0);
    };

    uint2 lk[MM ? G::NP : 2][8]; // two channels per lane: this supergroup's lookups and the next one's
    uint32_t nb[G::NP][2];
    if (nfull > 0) {
        pair_bytes_of<D, CPL>(buf[0], nb);
#pragma unroll
        for (int t = 0; t < 8; t++)
#pragma unroll
            for (int p = 0; p < G::NP; p++)
                lk[p][t] = lut_get(lut, nb[p][t & 1], lane_copy, t >> 1);
        wait_lgkm();
    }
    // one supergroup, nothing conditional in it (see qk_kernel); i = its buffer in the rotation
    auto body = [&](int sg, auto ic) {
        constexpr int i = decltype(ic)::value;
        pair_bytes_of<D, CPL>(buf[(i + 1) % AHEAD], nb);
        const int sgp = min(sg + AHEAD, nfull - 1);
#pragma unroll
        for (int v = 0; v < G::NV; v++)
            buf[i][v] = load_codes(cb + (size_t)sgp * G::VPS + v);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (MM) {
#pragma unroll
            for (int t = 0; t < 8; t += 2)
                token2(t, lk, nb, wbuf[i % WR]);
        } else {
            // a wave (nearly) alone on its SIMD: see replay_eight
#pragma unroll
            for (int t = 0; t < 8; t++)
                lk[(i & 1) ^ 1][t] = lut_get(lut, nb[0][t & 1], lane_copy, t >> 1);
            replay_eight_weighted(st[0], lk[i & 1], wbuf[i % WR], acc);
            __builtin_amdgcn_sched_barrier(0);
        }
        // the weights are reloaded once their last token is done: loading them earlier into a
        // second register set costs copies at the loop edge, which wait for the load they move
        wbuf[i % WR] = w8(min(sg + WR, nfull - 1));
    };
    rotate_over<AHEAD>(nfull, body);
    if (MM) {
#pragma unroll
        for (int p = 0; p < G::NP; p++) {
            acc[2 * p] = acc4[p].x;
            acc[2 * p + 1] = acc4[p].y;
        }
    }

    if (last) {
        const int ntail = (t1 - t0) & 7;
        if (ntail) {
#pragma unroll
            for (int v = 0; v < G::NV; v++) {
                uint32_t w[G::WPV];
                vec_words(cb[(size_t)nfull * G::VPS + v], w);
#pragma unroll
                for (int pp = 0; pp < G::WPV / 2; pp++) {
                    Pair &s = st[(G::WPV / 2) * v + pp];
                    for (int tt = 0; tt < ntail; tt++) {
                        const uint32_t na = (w[2 * pp] >> (4 * tt)) & 0xFu;
                        const uint32_t nbb = (w[2 * pp + 1] >> (4 * tt)) & 0xFu;
                        const h2 qc = codes_to_h2((int)na - 8, (int)nbb - 8);
                        const h2 qs = qc * s.sc;
                        const h2 vd = qs + s.zp;
                        const float wt = (float)w1(nfull * 8 + tt);
                        const int c = G::WPV * v + 2 * pp;
                        acc[c] = __builtin_fmaf(wt, (float)vd.x, acc[c]);
                        acc[c + 1] = __builtin_fmaf(wt, (float)vd.y, acc[c + 1]);
                        update_pair(s, qc, qs);
                    }
                }
            }
        }
        if (active)
            publish_state<D, CPL>(st, state_out, sa, bx, c0, T);

        h2 deq[G::NP];
        append_new_token<D, CPL>(cbh, T, v_new + (size_t)bx * D + c0, st, deq, active, sa.act_bf16);
        const float wT = (float)w1(T - t0);
#pragma unroll
        for (int p = 0; p < G::NP; p++) {
            acc[2 * p] = __builtin_fmaf(wT, (float)deq[p].x, acc[2 * p]);
            acc[2 * p + 1] = __builtin_fmaf(wT, (float)deq[p].y, acc[2 * p + 1]);
        }
    }
}

// forward_ov by itself keeps its loads behind the table and the loop to itself: built from ov_segment with the loads
// on their way meanwhile it was 3 to 8 % longer in long launches of wide heads (4 x 8 heads of 256 channels x 5000 tokens,
// no checkpoints, 188 / 202 us): the compiler orders and waits otherwise.
template <int D, int CPL, int BLK>
__global__ __launch_bounds__(BLK) void ov_kernel(
    const h1 *__restrict__ attn, uint4 *__restrict__ cache, const h1 *__restrict__ v_new,
    h1 *__restrict__ out, float *__restrict__ partial,
    const h1 *__restrict__ zp, const h1 *__restrict__ sc, const h1 *__restrict__ al,
    const h1 *__restrict__ be, const h1 *__restrict__ tg,
    int BH, int H, int T, int n_super_cap, h1 *__restrict__ state_out, Seg sa)
{
    using G = Geo<D, CPL>;
    static_assert(CPL >= 4, "fewer channels per lane: ov_lone_kernel");
    sa.groups = sa.groups < 0 ? -1 : 0; // no uneven plans come here
    __shared__ uint2 lut[LUT_WORDS64];
    lut_fill<BLK>(lut, threadIdx.x);
    __syncthreads();
    const uint32_t lane_copy = (uint32_t)(threadIdx.x & (LUT_COPIES - 1)) * 8u;

    const Unit<D, CPL, BLK> un(BH, sa.nseg);
    if (!un.wave_active)
        return; // padding waves
    const int bx = un.bx, lh = un.lh, c0 = un.c0;
    const bool active = un.active;
    const bool last = seg_is_last(sa, un.seg);
    const int h = bx % H;

    Pair st[G::NP];
    float acc[CPL];
    init_pairs<D, CPL>(st, zp, sc, al, be, tg, h, bx, c0, un.seg, sa);
    // The contraction is the matrix cores', as in ov_ft_kernel and for the reason given there: B = the lane's dequantised pair at two tokens, A = (w[t], 0, w[t+1], 0)
    // from lane 0 of each group of four, (0, w[t], 0, w[t+1]) from lane 1, zeros from lanes 2, 3.
    f4v acc4[G::NP];
#pragma unroll
    for (int p = 0; p < G::NP; p++)
        acc4[p] = (f4v){0.0f, 0.0f, 0.0f, 0.0f};
    const int role = threadIdx.x & 3;
    const uint32_t sel_a0 = role == 0 ? 0x0C0C0100u : role == 1 ? 0x01000C0Cu : 0x0C0C0C0Cu;
    const uint32_t sel_a1 = role == 0 ? 0x0C0C0302u : role == 1 ? 0x03020C0Cu : 0x0C0C0C0Cu;

    const int t0 = seg_begin(sa, un.seg);
    const int t1 = last ? T : seg_end(sa, un.seg);
    using Vec = typename G::Vec;
    Vec *cbh = reinterpret_cast<Vec *>(cache) + (size_t)bx * n_super_cap * G::VPS + lh * G::NV;
    const Vec *cb = cbh + (size_t)(t0 >> 3) * G::VPS;
    const h1 *wrow = attn + (size_t)bx * sa.row_pitch;
    const h1 *wb = wrow + t0;
    const int nfull = (t1 - t0) >> 3;

    auto load_w = [&](int sg) {
        uint4 r;
        __builtin_memcpy(&r, wb + (size_t)sg * 8, 16); // row base is only 2-byte aligned
        return r;
    };
    // two tokens of the current supergroup on the matrix cores, then the lookups of the same two
    // slots of the next one
    auto token2 = [&](int t, uint2 (*e)[8], const uint32_t (*nb)[2], const uint4 wv) {
        const uint32_t ww[4] = {wv.x, wv.y, wv.z, wv.w};
        const uint32_t w2 = ww[t >> 1];
        const h4v a = as_h4(__builtin_amdgcn_perm(w2, w2, sel_a0), __builtin_amdgcn_perm(w2, w2, sel_a1));
        uint32_t vd[G::NP][2];
#pragma unroll
        for (int k = 0; k < 2; k++)
#pragma unroll
            for (int p = 0; p < G::NP; p++) {
                Pair &s = st[p];
                const h2 qs = as_h2(e[p][t + k].x) * s.sc;
                vd[p][k] = as_u32(qs + s.zp);
                update_pair_abs(s, as_h2(e[p][t + k].y), qs);
            }
#pragma unroll
        for (int p = 0; p < G::NP; p++)
            acc4[p] = __builtin_amdgcn_mfma_f32_4x4x4f16(a, as_h4(vd[p][0], vd[p][1]), acc4[p], 0, 0, 0);
#pragma unroll
        for (int k = 0; k < 2; k++)
#pragma unroll
            for (int p = 0; p < G::NP; p++)
                e[p][t + k] = lut_get(lut, nb[p][(t + k) & 1], lane_copy, (t + k) >> 1);
        __builtin_amdgcn_sched_barrier(0);
    };

    Vec buf[PF][G::NV];
    uint4 wbuf[PF];
    uint2 lk[G::NP][8];
    uint32_t nb[G::NP][2];
    if (nfull > 0) {
        // unconditional, in the loop's order: see qk_kernel
#pragma unroll
        for (int i = 0; i < PF; i++) {
            const int sg = min(i, nfull - 1);
#pragma unroll
            for (int v = 0; v < G::NV; v++)
                buf[i][v] = load_codes(cb + (size_t)sg * G::VPS + v);
            wbuf[i] = load_w(sg);
            __builtin_amdgcn_sched_barrier(0);
        }
        pair_bytes_of<D, CPL>(buf[0], nb);
#pragma unroll
        for (int t = 0; t < 8; t++)
#pragma unroll
            for (int p = 0; p < G::NP; p++)
                lk[p][t] = lut_get(lut, nb[p][t & 1], lane_copy, t >> 1);
        wait_lgkm();
    }
    // one supergroup, nothing conditional in it (see qk_kernel); i = its buffer in the rotation
    auto body = [&](int sg, auto ic) {
        constexpr int i = decltype(ic)::value;
        pair_bytes_of<D, CPL>(buf[(i + 1) % PF], nb);
        const int sgp = min(sg + PF, nfull - 1);
#pragma unroll
        for (int v = 0; v < G::NV; v++)
            buf[i][v] = load_codes(cb + (size_t)sgp * G::VPS + v);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < 8; t += 2)
            token2(t, lk, nb, wbuf[i]);
        // the weights are reloaded once their last token is done: loading them earlier into a
        // second register set costs copies at the loop edge, which wait for the load they move
        wbuf[i] = load_w(sgp);
    };
    rotate_over<PF>(nfull, body);
#pragma unroll
    for (int p = 0; p < G::NP; p++) {
        acc[2 * p] = acc4[p].x;
        acc[2 * p + 1] = acc4[p].y;
    }

    if (last) {
        const int ntail = (t1 - t0) & 7;
        if (ntail) {
#pragma unroll
            for (int v = 0; v < G::NV; v++) {
                uint32_t w[G::WPV];
                vec_words(cb[(size_t)nfull * G::VPS + v], w);
#pragma unroll
                for (int pp = 0; pp < G::WPV / 2; pp++) {
                    Pair &s = st[(G::WPV / 2) * v + pp];
                    for (int tt = 0; tt < ntail; tt++) {
                        const uint32_t na = (w[2 * pp] >> (4 * tt)) & 0xFu;
                        const uint32_t nbb = (w[2 * pp + 1] >> (4 * tt)) & 0xFu;
                        const h2 qc = codes_to_h2((int)na - 8, (int)nbb - 8);
                        const h2 qs = qc * s.sc;
                        const h2 vd = qs + s.zp;
                        const float wt = (float)wb[nfull * 8 + tt];
                        const int c = G::WPV * v + 2 * pp;
                        acc[c] = __builtin_fmaf(wt, (float)vd.x, acc[c]);
                        acc[c + 1] = __builtin_fmaf(wt, (float)vd.y, acc[c + 1]);
                        update_pair(s, qc, qs);
                    }
                }
            }
        }
        if (active)
            publish_state<D, CPL>(st, state_out, sa, bx, c0, T);

        h2 deq[G::NP];
        append_new_token<D, CPL>(cbh, T, v_new + (size_t)bx * D + c0, st, deq, active, sa.act_bf16);
        const float wT = (float)wrow[T];
#pragma unroll
        for (int p = 0; p < G::NP; p++) {
            acc[2 * p] = __builtin_fmaf(wT, (float)deq[p].x, acc[2 * p]);
            acc[2 * p + 1] = __builtin_fmaf(wT, (float)deq[p].y, acc[2 * p + 1]);
        }
    }
    if (!active)
        return;
    if (sa.nseg == 1) {
        h1 *o = out + (size_t)bx * D + c0;
#pragma unroll
        for (int p = 0; p < G::NP; p++)
            store_act2(o + 2 * p, acc[2 * p], acc[2 * p + 1], sa.act_bf16);
    } else {
        float2 *o = reinterpret_cast<float2 *>(partial + ((size_t)un.seg * BH + bx) * D + c0);
#pragma unroll
        for (int p = 0; p < G::NP; p++)
            o[p] = make_float2(acc[2 * p], acc[2 * p + 1]);
    }
}

// out[i] = fp16(sum over segments, in segment order, of partial[s][i])
__global__ __launch_bounds__(256) void ov_finalize_kernel(const float *__restrict__ partial,
                                                           h1 *__restrict__ out, long n, int nseg,
                                                           int act_bf16)
{
    const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 2; // n is even (whole heads)
    if (i >= n)
        return;
    float2 s = make_float2(0.0f, 0.0f);
    for (int k = 0; k < nseg; k++) {
        const float2 p = *reinterpret_cast<const float2 *>(partial + (size_t)k * n + i);
        s.x += p.x;
        s.y += p.y;
    }
    store_act2(out + i, s.x, s.y, act_bf16);
}

// The same sum for many segments (long contexts at small batch: 128 segments of a 32 768-token
// context leave the kernel above with 128 dependent additions per thread and few threads).  A
// workgroup owns 64 consecutive outputs: thread (r, j) adds the segments r, r+16, ... of outputs
// 4j..4j+3 in ascending order, then thread (0, j) adds the 16 subtotals in ascending r.  The order
// is fixed, so results are reproducible from run to run.
__global__ __launch_bounds__(256) void ov_finalize_wide_kernel(const float *__restrict__ partial,
                                                                h1 *__restrict__ out, long n, int nseg,
                                                                int act_bf16)
{
    __shared__ float4 sub[16][16];
    const int j = threadIdx.x & 15, r = threadIdx.x >> 4;
    const long i = ((long)blockIdx.x * 16 + j) * 4; // n is a multiple of 4 (whole heads)
    float4 a = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (i < n) {
        for (int k = r; k < nseg; k += 16) {
            const float4 p = *reinterpret_cast<const float4 *>(partial + (size_t)k * n + i);
            a.x += p.x;
            a.y += p.y;
            a.z += p.z;
            a.w += p.w;
        }
    }
    sub[r][j] = a;
    __syncthreads();
    if (r == 0 && i < n) {
#pragma unroll
        for (int k = 1; k < 16; k++) {
            const float4 p = sub[k][j];
            a.x += p.x;
            a.y += p.y;
            a.z += p.z;
            a.w += p.w;
        }
        store_act2(out + i, a.x, a.y, act_bf16);
        store_act2(out + i + 2, a.z, a.w, act_bf16);
    }
}

// ---------------------------------------------------------------------------------------------
// softmax(float(logits)*scaling + mask) -> fp16   (llama_adkv.py:266-271)
// ---------------------------------------------------------------------------------------------
constexpr int SM_BLOCK = 256;
constexpr int SM_VEC = 8;                             // fp16 values per 16-byte access
constexpr int SM_NV = 3;                              // such accesses per thread and chunk
constexpr int SM_KEEP = SM_VEC * SM_NV;               // row elements a thread keeps in registers
constexpr int SM_CHUNK = SM_BLOCK * SM_KEEP;          // row elements a 256-thread workgroup holds
constexpr int SM_ROW_MAX = 24576;                     // longest row a single workgroup keeps in registers

// Rows [.., n] of an additive mask: fp32, fp16 or bfloat16, each widened as it is read (a conversion beforehand is
// a launch, 3 us of a step that takes 25 to 65).  Rows are as aligned as their elements.  HALF: whether the
// 16-bit types may come.  The kernels that keep a row in registers are there with and without: both ways of reading in
// one kernel took 138 registers instead of 109, three waves to a SIMD instead of four (16 384 rows of 1025 with an
// fp32 mask or none 22.5 / 19.0 us, in one kernel 28.5 / 22.8).  The chunked pair takes 2 registers less with both
// (512 rows of 131 073 with an fp32 mask 99 us, 105 without the 16-bit types).
template <bool HALF>
struct MaskRow {
    const char *p; // null: no mask
    int dt;        // ADKV_DT_*
    __device__ __forceinline__ explicit operator bool() const { return p != nullptr; }
    __device__ __forceinline__ float widen(uint16_t v) const
    {
        return dt == ADKV_DT_F16 ? (float)__builtin_bit_cast(h1, v) : __uint_as_float((uint32_t)v << 16);
    }
    __device__ __forceinline__ float at(int i) const
    {
        if (!HALF || dt == ADKV_DT_F32)
            return reinterpret_cast<const float *>(p)[i];
        return widen(reinterpret_cast<const uint16_t *>(p)[i]);
    }
    template <int V> __device__ __forceinline__ void load(int i, float *m) const
    {
        if (!HALF || dt == ADKV_DT_F32) {
            __builtin_memcpy(m, p + (size_t)i * 4, 4 * V);
        } else {
            uint16_t raw[V];
            __builtin_memcpy(raw, p + (size_t)i * 2, 2 * V);
#pragma unroll
            for (int k = 0; k < V; k++)
                m[k] = widen(raw[k]);
        }
    }
};

struct Mask {
    const void *p; // [rows / rows_per_mask_row, n], or null
    int rows_per_mask_row, dt;
    // elements t0.. of the row of logits row `row`
    template <bool HALF> __device__ __forceinline__ MaskRow<HALF> of(unsigned row, int n, int t0 = 0) const
    {
        if (p == nullptr)
            return {nullptr, dt};
        return {(const char *)p + ((size_t)(row / (unsigned)rows_per_mask_row) * n + t0) * (!HALF || dt == ADKV_DT_F32 ? 4 : 2), dt};
    }
};

template <int NT = SM_BLOCK>
__device__ __forceinline__ float block_reduce(float v, float *sm, bool is_max)
{
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
        const float o = __shfl_xor(v, m, 64);
        v = is_max ? fmaxf(v, o) : v + o;
    }
    const int w = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0)
        sm[w] = v;
    __syncthreads();
    float r = sm[0];
#pragma unroll
    for (int i = 1; i < NT / 64; i++)
        r = is_max ? fmaxf(r, sm[i]) : r + sm[i];
    return r;
}

// x[k] = logits*scaling + mask for the SM_KEEP elements of this thread in the chunk that starts at
// `base` (-inf past the end of the row); 16-byte accesses wherever a whole vector lies inside the
// row (rows are only 2-byte aligned: the hardware takes unaligned vector accesses).
template <int NV = SM_NV, int NT = SM_BLOCK, bool HALF>
__device__ __forceinline__ void softmax_load_chunk(const h1 *l, const MaskRow<HALF> &mk, int n, int base,
                                                   float scaling, float *x, float &mx,
                                                   int tid = (int)threadIdx.x)
{
    mx = -INFINITY;
#pragma unroll
    for (int v = 0; v < NV; v++) {
        const int i0 = base + (v * NT + tid) * SM_VEC;
        float *xv = x + v * SM_VEC;
        if (i0 + SM_VEC <= n) {
            uint4 raw;
            __builtin_memcpy(&raw, l + i0, 16);
            const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const h2 p = as_h2(w[k]);
                xv[2 * k] = (float)p.x * scaling;
                xv[2 * k + 1] = (float)p.y * scaling;
            }
            if (mk) {
                float m8[SM_VEC];
                mk.template load<SM_VEC>(i0, m8);
#pragma unroll
                for (int k = 0; k < SM_VEC; k++)
                    xv[k] += m8[k];
            }
        } else {
#pragma unroll
            for (int k = 0; k < SM_VEC; k++) {
                const int i = i0 + k;
                xv[k] = -INFINITY;
                if (i < n) {
                    xv[k] = (float)l[i] * scaling;
                    if (mk)
                        xv[k] += mk.at(i);
                }
            }
        }
#pragma unroll
        for (int k = 0; k < SM_VEC; k++)
            mx = fmaxf(mx, xv[k]);
    }
}

// w[i] = fp16(x[k] * inv) for the same elements
template <int NV = SM_NV, int NT = SM_BLOCK>
__device__ __forceinline__ void softmax_store_chunk(h1 *w, int n, int base, const float *x, float inv,
                                                    int tid = (int)threadIdx.x)
{
#pragma unroll
    for (int v = 0; v < NV; v++) {
        const int i0 = base + (v * NT + tid) * SM_VEC;
        const float *xv = x + v * SM_VEC;
        if (i0 + SM_VEC <= n) {
            uint32_t o[4];
#pragma unroll
            for (int k = 0; k < 4; k++)
                o[k] = as_u32((h2){(h1)(xv[2 * k] * inv), (h1)(xv[2 * k + 1] * inv)});
            const uint4 raw = make_uint4(o[0], o[1], o[2], o[3]);
            __builtin_memcpy(w + i0, &raw, 16);
        } else {
#pragma unroll
            for (int k = 0; k < SM_VEC; k++)
                if (i0 + k < n)
                    w[i0 + k] = (h1)(xv[k] * inv);
        }
    }
}

// Short rows: one wave per row (four rows per workgroup), the row in registers, reductions across
// the wave only.  A workgroup per row would spend most of its time on two barriers for a handful of
// elements per thread; rows of a few hundred tokens are the common decode case.
template <int NV, bool HALF>
__global__ __launch_bounds__(SM_BLOCK) void softmax_wave_kernel(
    const h1 *__restrict__ logits, h1 *__restrict__ weights, Mask mask, int rows, int n,
    long ld, float scaling)
{
    const int row = blockIdx.x * (SM_BLOCK / 64) + (threadIdx.x >> 6);
    if (row >= rows)
        return;
    const int lane = threadIdx.x & 63;
    const h1 *l = logits + (size_t)row * ld;
    h1 *w = weights + (size_t)row * ld;
    const MaskRow<HALF> mk = mask.of<HALF>(row, n);
    float x[NV * SM_VEC], mx;
    softmax_load_chunk<NV, 64>(l, mk, n, 0, scaling, x, mx, lane);
    mx = wave_reduce<true>(mx);
    float sum = 0.0f;
#pragma unroll
    for (int k = 0; k < NV * SM_VEC; k++) {
        x[k] = __expf(x[k] - mx);
        sum += x[k];
    }
    sum = wave_reduce<false>(sum);
    softmax_store_chunk<NV, 64>(w, n, 0, x, 1.0f / sum, lane);
}

// One workgroup of NT threads per row.  A row of up to NT * NV * 8 elements is read once and kept
// in registers (the launcher picks NT and NV by the row length, up to 24576 elements); longer rows
// are walked three times (the chunked kernels below avoid that when the caller gives a workspace).
template <int NT, int NV, bool HALF>
__global__ __launch_bounds__(NT) void softmax_kernel(
    const h1 *__restrict__ logits, h1 *__restrict__ weights, Mask mask, int n, long ld, float scaling)
{
    __shared__ float sm[NT / 64];
    const int row = blockIdx.x;
    const h1 *l = logits + (size_t)row * ld;
    h1 *w = weights + (size_t)row * ld;
    const MaskRow<HALF> mk = mask.of<HALF>(row, n);

    if (n <= NT * NV * SM_VEC) {
        float x[NV * SM_VEC], mx;
        softmax_load_chunk<NV, NT>(l, mk, n, 0, scaling, x, mx);
        mx = block_reduce<NT>(mx, sm, true);
        float sum = 0.0f;
#pragma unroll
        for (int k = 0; k < NV * SM_VEC; k++) {
            x[k] = __expf(x[k] - mx);
            sum += x[k];
        }
        sum = block_reduce<NT>(sum, sm, false);
        softmax_store_chunk<NV, NT>(w, n, 0, x, 1.0f / sum);
        return;
    }
    auto at = [&](int i) {
        float v = (float)l[i] * scaling;
        if (mk)
            v += mk.at(i);
        return v;
    };
    float mx = -INFINITY;
    for (int i = threadIdx.x; i < n; i += NT)
        mx = fmaxf(mx, at(i));
    mx = block_reduce<NT>(mx, sm, true);
    float sum = 0.0f;
    for (int i = threadIdx.x; i < n; i += NT)
        sum += __expf(at(i) - mx);
    sum = block_reduce<NT>(sum, sm, false);
    const float inv = 1.0f / sum;
    for (int i = threadIdx.x; i < n; i += NT)
        w[i] = (h1)(__expf(at(i) - mx) * inv);
}

// Unmasked rows of up to 1024 * NV * 8 elements (139 264 with NV = 17), one 1024-thread workgroup
// per row: the row stays in registers AS FP16 (NV 16-byte vectors per thread), so it is read once
// and written once; maximum, sum and weights are three walks over registers.  Up to 9 vectors
// per thread two such workgroups fit a CU (64 registers per lane), beyond that one (104 registers
// with 17 vectors); few and very long rows are better cut into chunks.
// scaling must be non-zero: elements past the end of the row are held as the infinity that
// scaling turns into -inf.
constexpr int SM_REG_NV = 17;
constexpr int SM_REG_MAX = 1024 * SM_REG_NV * SM_VEC;
#ifndef ADKV_SM_REG_MIN_ROWS
#define ADKV_SM_REG_MIN_ROWS 128
#endif
constexpr int SM_REG_MIN_ROWS = ADKV_SM_REG_MIN_ROWS;

template <int NV>
__global__ __launch_bounds__(1024) void softmax_regrow_kernel(
    const h1 *__restrict__ logits, h1 *__restrict__ weights, int n, long ld, float scaling)
{
    constexpr int NT = 1024;
    __shared__ float sm[NT / 64];
    const h1 *l = logits + (size_t)blockIdx.x * ld;
    h1 *w = weights + (size_t)blockIdx.x * ld;
    const int tid = threadIdx.x;
    const uint32_t pad = scaling > 0.0f ? 0xFC00FC00u : 0x7C007C00u; // scaling * pad = -inf

    uint4 raw[NV];
#pragma unroll
    for (int v = 0; v < NV; v++) {
        const int i0 = (v * NT + tid) * SM_VEC;
        if (i0 + SM_VEC <= n) {
            __builtin_memcpy(&raw[v], l + i0, 16); // rows are only 2-byte aligned
        } else {
            uint32_t u[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint32_t lo = i0 + 2 * k < n ? __builtin_bit_cast(uint16_t, l[i0 + 2 * k]) : (pad & 0xFFFFu);
                const uint32_t hi = i0 + 2 * k + 1 < n ? __builtin_bit_cast(uint16_t, l[i0 + 2 * k + 1]) : (pad & 0xFFFFu);
                u[k] = lo | (hi << 16);
            }
            raw[v] = make_uint4(u[0], u[1], u[2], u[3]);
        }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int v = 0; v < NV; v++) {
        const uint32_t u[4] = {raw[v].x, raw[v].y, raw[v].z, raw[v].w};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const h2 p = as_h2(u[k]);
            mx = fmaxf(mx, fmaxf((float)p.x * scaling, (float)p.y * scaling));
        }
    }
    mx = block_reduce<NT>(mx, sm, true);
    // each walk converts the row again: values carried over from the walk before (which the
    // compiler would otherwise keep, 136 more registers per lane) are cut off here
    auto forget = [&]() {
#pragma unroll
        for (int v = 0; v < NV; v++)
            asm volatile("" : "+v"(raw[v].x), "+v"(raw[v].y), "+v"(raw[v].z), "+v"(raw[v].w));
    };
    forget();
    // exp(x * scaling - mx) = exp2(x * s2 + c2)
    const float s2 = scaling * 1.44269504088896340736f;
    const float c2 = mx == -INFINITY ? 0.0f : -mx * 1.44269504088896340736f;
    float sum = 0.0f;
#pragma unroll
    for (int v = 0; v < NV; v++) {
        const uint32_t u[4] = {raw[v].x, raw[v].y, raw[v].z, raw[v].w};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const h2 p = as_h2(u[k]);
            sum += __builtin_amdgcn_exp2f(__builtin_fmaf((float)p.x, s2, c2));
            sum += __builtin_amdgcn_exp2f(__builtin_fmaf((float)p.y, s2, c2));
        }
    }
    sum = block_reduce<NT>(sum, sm, false);
    const float inv = 1.0f / sum;
    forget();
#pragma unroll
    for (int v = 0; v < NV; v++) {
        const int i0 = (v * NT + tid) * SM_VEC;
        const uint32_t u[4] = {raw[v].x, raw[v].y, raw[v].z, raw[v].w};
        uint32_t o[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const h2 p = as_h2(u[k]);
            o[k] = as_u32((h2){(h1)(__builtin_amdgcn_exp2f(__builtin_fmaf((float)p.x, s2, c2)) * inv),
                               (h1)(__builtin_amdgcn_exp2f(__builtin_fmaf((float)p.y, s2, c2)) * inv)});
        }
        if (i0 + SM_VEC <= n) {
            const uint4 ov = make_uint4(o[0], o[1], o[2], o[3]);
            __builtin_memcpy(w + i0, &ov, 16);
        } else {
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const h2 p = as_h2(o[k]);
                if (i0 + 2 * k < n)
                    w[i0 + 2 * k] = p.x;
                if (i0 + 2 * k + 1 < n)
                    w[i0 + 2 * k + 1] = p.y;
            }
        }
    }
}

// Rows longer than one workgroup can hold in registers are cut into chunks of SM_CHUNK elements,
// one workgroup each: the first pass leaves (max, sum of exp(x - max)) per chunk, the second
// combines a row's chunks and normalises.  Each logit is read twice and nothing depends on the
// order in which workgroups run.

// (m, s) with s = sum of exp(x - m) over a set of elements; the pair of the union of two sets.
__device__ __forceinline__ float2 softmax_merge(float2 a, float2 b)
{
    const float m = fmaxf(a.x, b.x);
    if (m == -INFINITY)
        return make_float2(-INFINITY, 0.0f); // both sets empty or fully masked
    return make_float2(m, a.y * __expf(a.x - m) + b.y * __expf(b.x - m));
}

__device__ __forceinline__ float2 softmax_wave_merge(float2 v)
{
#pragma unroll
    for (int k = 1; k < 64; k <<= 1)
        v = softmax_merge(v, make_float2(__shfl_xor(v.x, k, 64), __shfl_xor(v.y, k, 64)));
    return v;
}

// SUB chunks per workgroup.  With SUB > 1 and every chunk inside the row, all of the workgroup's
// loads are issued before anything waits for one (a 256-thread workgroup that fetches 12 KB and
// leaves is mostly launch and latency: 3.0 TB/s over the 512 rows of 131 073 logits of the
// long-context shape; 48 KB per workgroup: see the kernel trace of that shape); the merged pair
// goes to the first chunk's slot and the other slots get the neutral element.
template <int SUB>
__global__ __launch_bounds__(SM_BLOCK) void softmax_part_kernel(
    const h1 *__restrict__ logits, Mask mask, float2 *__restrict__ part, int n, long ld, int nchunk, float scaling)
{
    __shared__ float2 sm[SM_BLOCK / 64];
    const int row = blockIdx.y, ck0 = blockIdx.x * SUB;
    const h1 *l = logits + (size_t)row * ld;
    const MaskRow<true> mk = mask.of<true>(row, n);
    float mx = -INFINITY, sum = 0.0f;
    if (SUB > 1 && !mk && (ck0 + SUB) * SM_CHUNK <= n) {
        uint4 raw[SUB][SM_NV];
#pragma unroll
        for (int s = 0; s < SUB; s++)
#pragma unroll
            for (int v = 0; v < SM_NV; v++)
                __builtin_memcpy(&raw[s][v], l + (size_t)(ck0 + s) * SM_CHUNK + (v * SM_BLOCK + threadIdx.x) * SM_VEC, 16);
        float x[SUB][SM_KEEP];
#pragma unroll
        for (int s = 0; s < SUB; s++)
#pragma unroll
            for (int v = 0; v < SM_NV; v++) {
                const uint32_t w[4] = {raw[s][v].x, raw[s][v].y, raw[s][v].z, raw[s][v].w};
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const h2 p = as_h2(w[k]);
                    x[s][v * SM_VEC + 2 * k] = (float)p.x * scaling;
                    x[s][v * SM_VEC + 2 * k + 1] = (float)p.y * scaling;
                    mx = fmaxf(mx, fmaxf(x[s][v * SM_VEC + 2 * k], x[s][v * SM_VEC + 2 * k + 1]));
                }
            }
        if (mx > -INFINITY) {
#pragma unroll
            for (int s = 0; s < SUB; s++)
#pragma unroll
                for (int k = 0; k < SM_KEEP; k++)
                    sum += __expf(x[s][k] - mx);
        }
    } else {
        // the generic way, a chunk at a time (chunks past the end of the row are all -inf)
        for (int s = 0; s < SUB; s++) {
            float x[SM_KEEP], m1;
            softmax_load_chunk(l, mk, n, (ck0 + s) * SM_CHUNK, scaling, x, m1);
            float s1 = 0.0f;
            if (m1 > -INFINITY) {
#pragma unroll
                for (int k = 0; k < SM_KEEP; k++)
                    s1 += __expf(x[k] - m1);
            }
            const float2 r = softmax_merge(make_float2(mx, sum), make_float2(m1, s1));
            mx = r.x;
            sum = r.y;
        }
    }
    // the thread's own (max, sum), then ONE reduction of pairs over the workgroup
    const float2 w = softmax_wave_merge(make_float2(mx, sum));
    if ((threadIdx.x & 63) == 0)
        sm[threadIdx.x >> 6] = w;
    __syncthreads();
    if (threadIdx.x == 0) {
        float2 r = sm[0];
#pragma unroll
        for (int i = 1; i < SM_BLOCK / 64; i++)
            r = softmax_merge(r, sm[i]);
        part[(size_t)row * nchunk + ck0] = r;
    }
    if (threadIdx.x > 0 && threadIdx.x < SUB && ck0 + (int)threadIdx.x < nchunk)
        part[(size_t)row * nchunk + ck0 + threadIdx.x] = make_float2(-INFINITY, 0.0f);
}

__global__ __launch_bounds__(SM_BLOCK) void softmax_norm_kernel(
    const h1 *__restrict__ logits, h1 *__restrict__ weights, Mask mask, const float2 *__restrict__ part,
    int n, long ld, int nchunk, float scaling)
{
    __shared__ float2 row_stats;
    const int row = blockIdx.y, ck = blockIdx.x;
    const h1 *l = logits + (size_t)row * ld;
    h1 *w = weights + (size_t)row * ld;
    const MaskRow<true> mk = mask.of<true>(row, n);
    float x[SM_KEEP], mx;
    softmax_load_chunk(l, mk, n, ck * SM_CHUNK, scaling, x, mx);   // issued first: in flight meanwhile
    if (threadIdx.x < 64) {
        // the row's (max, sum) from its chunks: one wave, a chunk per lane and round
        const float2 *pr = part + (size_t)row * nchunk;
        float2 v = make_float2(-INFINITY, 0.0f);
        for (int k = threadIdx.x; k < nchunk; k += 64)
            v = softmax_merge(v, pr[k]);
        v = softmax_wave_merge(v);
        if (threadIdx.x == 0)
            row_stats = v;
    }
    __syncthreads();
    const float M = row_stats.x, inv = 1.0f / row_stats.y;
#pragma unroll
    for (int k = 0; k < SM_KEEP; k++)
        x[k] = __expf(x[k] - M);
    softmax_store_chunk(w, n, ck * SM_CHUNK, x, inv);
}

} // namespace adkv

// ---------------------------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------------------------
using namespace adkv;

static thread_local int g_last_hip_error = 0;

int adkv::check_launch()
{
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        g_last_hip_error = (int)e;
        return ADKV_E_LAUNCH;
    }
    return ADKV_OK;
}

static int check_common(int B, int H, int T, int D, int n_super_cap)
{
    if (B <= 0 || H <= 0 || T < 0 || n_super_cap <= 0)
        return ADKV_E_SHAPE;
    if (D != 128 && D != 256 && D != 512)
        return ADKV_E_DIM;
    if ((int64_t)B * H > (int64_t)INT32_MAX / 64)
        return ADKV_E_SHAPE;
    return ADKV_OK;
}

static inline int lanes_per_head(int D) { return D == 128 ? 32 : 64; }

#include "adkv_gqa_kernels.h"
#include "adkv_ft_kernels.h"
#include "adkv_lone.h"
#include "adkv_small_step.h"
#include "adkv_segment_step.h"

// Waves a SIMD should hold for packed-f16 issue to run near full rate, and SIMDs on the device.
constexpr int WAVES_PER_SIMD_TARGET = 4;
// Compute units of the device the calling thread is on, asked once per device (256 on an MI355X,
// and that is what every measurement behind the plans below was taken on).  Without a device (the
// planning entry points can be called on a host that has none) the MI355X's count is assumed.
static int cus()
{
    constexpr int MAX_DEV = 64, MI355X_CUS = 256;
    static std::atomic<int> cached[MAX_DEV];
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEV) {
        (void)hipGetLastError(); // not this call's error to report
        return MI355X_CUS;
    }
    int n = cached[dev].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) {
            (void)hipGetLastError();
            n = MI355X_CUS;
        }
        cached[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}
static int n_simd() { return 4 * cus(); }
int adkv::cu_count() { return cus(); }

// Segment plan for a decode launch.  Starting from the fewest segments that give every SIMD its
// target of waves, finer splits are taken when they shorten the launch: 16-wave workgroups run one
// per CU, so a launch is ceil(workgroups / 256) rounds of one segment's length each, and a batch
// whose workgroup count falls just past a multiple of 256 (B = 352: 352 workgroups = 2 rounds for
// 1.4 rounds of work) wastes most of a round unless it is cut finer.
static Seg plan_segments(void *ckpt, int n_ckpt_cap, int ckpt_interval, int BH, int T, int D, int lanes = 0)
{
    Seg s;
    s.ckpt = (h1 *)ckpt;
    s.n_ckpt_cap = n_ckpt_cap;
    s.ckpt_interval = ckpt ? ckpt_interval : 0;
    s.seg_tokens = T > 0 ? T : 1;
    s.seg_intervals = 0;
    s.nseg = 1;
    s.row_pitch = T + 1;
    s.act_bf16 = 0;
    s.combine = 0;
    s.groups = 0;
    s.intervals = 0;
    s.phys_per_head = 0;
    s.skew = 0;
    s.fresh = 0;
    if (!ckpt || ckpt_interval <= 0 || T <= ckpt_interval)
        return s;
    const int avail = (T + ckpt_interval - 1) / ckpt_interval;               // finest split
    const int n_cus = cus(); // asks the runtime for the device: once per plan
    const int lph = lanes ? lanes : lanes_per_head(D); // lanes: 16 for the two-pass per-head-table kernels
    const long units_target = 4L * n_cus * WAVES_PER_SIMD_TARGET * (64 / lph);
    long want = (units_target + BH - 1) / BH;
    if (want < 1)
        want = 1;
    if (want > avail)
        want = avail;
    const int m0 = (int)((avail + want - 1) / want);                          // intervals per segment
    // every segment start s*m*interval needs checkpoint s*m-1 < n_ckpt_cap
    auto valid = [&](int m) { return m >= avail || ((avail - 1) / m) * m - 1 < n_ckpt_cap; };
    // launch length in units of one checkpoint interval
    auto cost = [&](int m) {
        const int nseg = (avail + m - 1) / m;
        const long threads = (lph == 16 ? padded_units<16>(BH, nseg) : lph == 32 ? padded_units<32>(BH, nseg) : padded_units<64>(BH, nseg)) * lph;
        if (D == 512 || threads < 1024L * n_cus)
            return (double)m;                        // small workgroups: no round structure to model
        const long wgs = (threads + 1023) / 1024;
        return (double)((wgs + n_cus - 1) / n_cus) * m;
    };
    int best = -1;
    double best_cost = 0.0;
    for (int m = avail; m >= 1; m--) {
        if (m > m0 && m < avail)
            continue;                                // between "one segment" and the occupancy target: skip
        if (!valid(m))
            continue;
        const double c = cost(m);
        if (best < 0 || c < 0.97 * best_cost) {      // a finer split has to pay for its overheads
            best = m;
            best_cost = c;
        }
    }
    // the occupancy target comes first: one segment is only kept when no split is possible
    if (best >= avail && m0 < avail && valid(m0))
        best = m0;
    if (best < 0 || best >= avail)
        return s;
    s.seg_tokens = best * ckpt_interval;
    s.seg_intervals = best;
    s.nseg = (T + s.seg_tokens - 1) / s.seg_tokens;
    return s;
}

// Threads per workgroup of a shared-table launch.  The table takes 64 KB of a CU's 160 KB of LDS, so a
// CU holds two workgroups: 4-wave ones (which spread over the CUs best) put at most two waves on a
// SIMD, and a launch with more than that ran in two rounds although registers allow four.  Launches
// of 9-12 waves per CU therefore take 12-wave workgroups and larger ones 16-wave ones, one table for
// all of them.  us per step, 4-wave workgroups (matrix-core kernels: 8-wave) before /
// now, batch x KV heads x tokens: 64 x 32 x 663 86 / 73, 90 x 32 x 300 77 / 58, 12 x 8 x 8190 of 256
// channels 88 / 78; grouped queries 25 x 8 x 9000 110 / 102, 2-bit 40 x 8 x 4096 99 / 75.
static int threads_per_workgroup(long threads)
{
    const long per_cu = (threads / 64 + cus() - 1) / cus();
    return per_cu <= 8 ? 256 : per_cu <= 12 ? 768 : 1024;
}

#define ADKV_LAUNCH_(KERNEL, DD, CC, BLK, ...)                                                      \
    hipLaunchKernelGGL((KERNEL<DD, CC, BLK>), dim3((unsigned)((threads + (BLK)-1) / (BLK))), dim3(BLK), 0, st, __VA_ARGS__)
#define ADKV_LAUNCH(KERNEL, DD, CC, ...)                                                            \
    do {                                                                                            \
        const long threads = padded_units<DD / CC>(BH, seg.nseg) * (DD / CC);                       \
        const int blk = threads_per_workgroup(threads);                                       \
        if (blk == 1024)                                                                            \
            ADKV_LAUNCH_(KERNEL, DD, CC, 1024, __VA_ARGS__);                                        \
        else if (blk == 768)                                                                        \
            ADKV_LAUNCH_(KERNEL, DD, CC, 768, __VA_ARGS__);                                         \
        else                                                                                        \
            ADKV_LAUNCH_(KERNEL, DD, CC, 256, __VA_ARGS__);                                         \
    } while (0)

#define ADKV_DISPATCH_D(KERNEL, ...)                  \
    switch (D) {                                      \
    case 128:                                         \
        ADKV_LAUNCH(KERNEL, 128, 4, __VA_ARGS__);     \
        break;                                        \
    case 256:                                         \
        ADKV_LAUNCH(KERNEL, 256, 4, __VA_ARGS__);     \
        break;                                        \
    default: {                                        \
        const long threads = padded_units<64>(BH, seg.nseg) * 64; \
        ADKV_LAUNCH_(KERNEL, 512, 8, 256, __VA_ARGS__); \
        break;                                        \
    }                                                 \
    }

// Head dim 128 in launches that leave SIMDs empty: one channel per lane, a head over two waves (adkv_lone.h), as long as
// two channels per lane would leave at most two waves on a SIMD (forward_ov: four of these) or one and a half
// (forward_qk, whose keys take more of the LDS: with four waves it is the two-channel form's equal).  us, two channels per
// lane / one, 32 heads, no checkpoints: 1 x 1024 tokens qk 29.5 / 19.3, ov 28.8 / 14.9, 16 x 1024 30.2 / 20.9 and 28.0 / 16.6,
// 32 x 1024 30.7 / 29.0 and 28.3 / 24.7, 48 x 1024 45.2 / 37.7 and 44.3 / 33.5, 48 x 200 12.3 / 10.6 and 12.5 / 9.0, 64 x 1024
// 48.9 / 48.6 and 47.5 / 43.0, 64 x 200 12.7 / 12.9 and 12.7 / 10.9; every 256: 1 x 4096 10.4 / 8.1 and 12.4 / 8.3, 2 x 8192
// 15.3 / 15.0 and 17.8 / 15.1.
// A buffer descriptor holds a segment's codes: rows of 2^24 tokens and more stay with the other kernels.
// forward_qk's launches of more waves than that, up to two per SIMD, take two channels per lane (a head per wave, see
// PairScores): twice the waves of four channels, each with half the instruction stream per token; with more waves per SIMD
// the four-channel lanes do less work in total.
static bool qk_lone(int BH, int nseg, int T) { return 2 * padded_units<64>(BH, nseg) <= 3L * n_simd() && T < 1 << 24; }
static bool qk_pair(int BH, int nseg) { return padded_units<32>(BH, nseg) <= 2L * n_simd(); }
static bool ov_lone(int BH, int nseg, int T) { return padded_units<64>(BH, nseg) <= 2L * n_simd() && T < 1 << 24; }
#define ADKV_LAUNCH_LONE_(KERNEL, BLK, ...) \
    hipLaunchKernelGGL(KERNEL<BLK>, dim3((unsigned)((threads + (BLK)-1) / (BLK))), dim3(BLK), 0, st, __VA_ARGS__)
// MOST: the largest workgroup that the rule above asks for
#define ADKV_LAUNCH_LONE(KERNEL, MOST, ...)                            \
    do {                                                               \
        const long threads = padded_units<64>(BH, seg.nseg) * 128;     \
        const int blk = threads_per_workgroup(threads);                \
        if (blk == 256)                                                \
            ADKV_LAUNCH_LONE_(KERNEL, 256, __VA_ARGS__);               \
        else if (blk == 768)                                           \
            ADKV_LAUNCH_LONE_(KERNEL, 768, __VA_ARGS__);               \
        else                                                           \
            ADKV_LAUNCH_LONE_(KERNEL, MOST, __VA_ARGS__);              \
    } while (0)

// Matrix-core kernels (head dim 128), four channels per lane: 12- or 16-wave workgroups by the same
// rule.  With eight query heads per KV head ov_gqa_kernel needs 142 registers per lane, more than the 128 a 16-wave
// workgroup leaves: there it spills accumulators and loses (16 x 8 KV heads x 131072 tokens, 64 query heads: 421 -> 533 us
// with 4-bit codes, 346 -> 747 us with 2-bit ones), and takes 8-wave workgroups.  qk_gqa_kernel fits into 118, and gained from
// four waves per SIMD when it still needed 138 and spilled a dozen (563 -> 530 us, 518 -> 425 us).  BIG8 says which of the two
// this is.
// A launch that would leave at most two waves on a SIMD takes two channels per lane instead (a KV head
// per wave): twice the waves, forward_qk without the reduction over the quarters of a head.  With more waves than
// that the four-channel lanes have enough of them and spend fewer instructions on what a wave does once per token.
// forward_ov has nothing to reduce and pays for its weights once per wave: 16 bytes per lane and eight tokens, as often
// with half of the channels, and several times that from rows that are not 16-byte aligned.  So it takes two
// channels up to this many waves of them per SIMD: four with one query head, and with two where rows are aligned,
// three with four heads, two with eight; from other rows two with two heads, less than two with more.  us, four channels
// per lane / two, 16 x 8 KV heads: aligned, four heads x 4000 tokens (two waves) 25.0 / 18.6, 5000 (2.5) 26.1 / 23.0,
// 8000 (four) 29.0 / 29.3, eight heads 30.9 / 27.5, 32.5 / 35.5, 34.2 / 45.4; other rows, two heads 25.1 / 19.1,
// 25.8 / 26.1, 27.5 / 41.0, four 29.7 / 29.5, 30.9 / 41.3, 38.4 / 63.7; 128 x 8 x 300, four heads 19.7 / 25.4.
static bool gqa_pair(long BH, int nseg) { return padded_units<64>((int)BH, nseg) <= 4L * n_simd(); }
static bool ov_gqa_pair(long BH, int nseg, int GQ, bool aligned)
{
    const long waves = padded_units<64>((int)BH, nseg);
    if (GQ == 1 || (GQ == 2 && aligned))
        return waves <= 4L * n_simd();
    if (aligned)
        return waves <= (GQ == 4 ? 3L : 2L) * n_simd();
    return GQ == 2 ? waves <= 2L * n_simd() : waves < 2L * n_simd();
}
#define ADKV_LAUNCH_GQA_(KERNEL, BB, GQV, BLK, CPLV, ...)                                          \
    hipLaunchKernelGGL((KERNEL<BB, GQV, BLK, CPLV>), dim3((unsigned)((threads + (BLK)-1) / (BLK))), dim3(BLK), 0, st, __VA_ARGS__)
#define ADKV_LAUNCH_GQA(KERNEL, BIG8, BB, GQV, ...)                                                \
    do {                                                                                            \
        const long threads = pair ? padded_units<64>(BH, seg.nseg) * 64 : padded_units<32>(BH, seg.nseg) * 32; \
        const int blk = threads_per_workgroup(threads);                                             \
        constexpr bool BIG = GQV <= 4 || BIG8;                                                      \
        if (pair && blk == 1024)                                                                    \
            ADKV_LAUNCH_GQA_(KERNEL, BB, GQV, 1024, 2, __VA_ARGS__);                                \
        else if (pair && blk == 768)                                                                \
            ADKV_LAUNCH_GQA_(KERNEL, BB, GQV, 768, 2, __VA_ARGS__);                                 \
        else if (pair)                                                                              \
            ADKV_LAUNCH_GQA_(KERNEL, BB, GQV, 256, 2, __VA_ARGS__);                                 \
        else if (blk == 1024 || !BIG)                                                               \
            ADKV_LAUNCH_GQA_(KERNEL, BB, GQV, (BIG ? 1024 : 512), 4, __VA_ARGS__);                  \
        else if (blk == 768 || BIG8) /* forward_qk: more than eight waves per CU, never 256 */      \
            ADKV_LAUNCH_GQA_(KERNEL, BB, GQV, (BIG ? 768 : 512), 4, __VA_ARGS__);                   \
        else                                                                                        \
            ADKV_LAUNCH_GQA_(KERNEL, BB, GQV, (BIG8 ? 768 : 512), 4, __VA_ARGS__);                  \
    } while (0)

#define ADKV_DISPATCH_GQ_BITS(KERNEL, BIG8, BB, ...)                                               \
    switch (GQ) {                                                                                   \
    case 1: ADKV_LAUNCH_GQA(KERNEL, BIG8, BB, 1, __VA_ARGS__); break;                               \
    case 2: ADKV_LAUNCH_GQA(KERNEL, BIG8, BB, 2, __VA_ARGS__); break;                               \
    case 4: ADKV_LAUNCH_GQA(KERNEL, BIG8, BB, 4, __VA_ARGS__); break;                               \
    case 8: ADKV_LAUNCH_GQA(KERNEL, BIG8, BB, 8, __VA_ARGS__); break;                               \
    default: return ADKV_E_UNSUPPORTED;                                                             \
    }

#define ADKV_DISPATCH_GQ(KERNEL, BIG8, ...)                                                        \
    if (bits == 4) {                                                                                \
        ADKV_DISPATCH_GQ_BITS(KERNEL, BIG8, 4, __VA_ARGS__)                                         \
    } else {                                                                                        \
        ADKV_DISPATCH_GQ_BITS(KERNEL, BIG8, 2, __VA_ARGS__)                                         \
    }

// Whether single-query-head launches (GQ == 1, head dim 128) also take the matrix-core kernels:
// the built-in choice, overridden by ADKV_MFMA=0/1 in the environment, overridden by
// adkv_set_mha_kernel().
// The environment is read once, when the first launch asks; the override is an atomic so that
// launches from several host threads never see a torn value.
static std::atomic<int> g_mha_kernel{-1};
static int mha_kernel_default()
{
    static const int from_env = [] {
        const char *e = getenv("ADKV_MFMA");
        return (e ? atoi(e) : 0) != 0 ? 1 : 0;
    }();
    return from_env;
}
static bool mfma_for_mha()
{
    const int v = g_mha_kernel.load(std::memory_order_relaxed);
    return (v < 0 ? mha_kernel_default() : v) == 1;
}

// Whether a launch with one query head per KV head takes the kernels with a per-head table
// (adkv_ft_kernels.h).  They need head dim 128 and 4-bit codes.  By default the choice follows a
// model of the two launches, both bound by vector issue: the per-head-table kernels run 16-wave
// workgroups, one per CU, in ceil(workgroups / 256) rounds of one segment each (every head's
// waves padded to whole workgroups), at 0.93 of the shared-table kernels' time per wave; the
// shared-table kernels run the same rounds when the launch is big enough for 16-wave workgroups,
// and otherwise spread 4-wave workgroups over the SIMDs, where the fullest SIMD sets the time
// (its waves / 4 rounds).  Measured (B x 32 heads, ctx; per-head table against shared table):
// 128 x 4096: 587 / 624 us per layer-step, 34 x 3000: 155 / 181, 40 x 1500: 89 / 107, 24 x 3000:
// 141 / 141, 20 x 8192 (288 workgroups, two rounds): 369 / 255.  adkv_set_mha_kernel(2) takes them whenever they can run (3: with 16 lanes per head, 4: with 32), (0) never.
static bool use_head_table(int B, int H, int GQ, int bits, int D, const Seg &seg)
{
    if (D != 128 || bits != 4 || GQ != 1)
        return false;
    const int v = g_mha_kernel.load(std::memory_order_relaxed);
    if (v >= 2)
        return true;
    if (v >= 0 || mha_kernel_default() == 1)
        return false;
    const long BH = (long)B * H;
    const long padded = padded_units<32>((int)BH, seg.nseg);
    const long waves_shared = padded / 2;
    if (waves_shared <= n_simd())
        return false;                                 // every wave a SIMD to itself: two-channel lanes
    const long wgs_ft = (long)H * ft_wgs_per_head(B, seg.nseg, 2);
    const double t_ft = 0.93 * (double)((wgs_ft + cus() - 1) / cus());
    double t_shared;
    if (padded * 32 >= (long)FT_BLK * cus())
        t_shared = (double)(((padded * 32 + FT_BLK - 1) / FT_BLK + cus() - 1) / cus());
    else
        t_shared = (double)((waves_shared + n_simd() - 1) / n_simd()) / WAVES_PER_SIMD_TARGET;
    return t_ft <= t_shared;
}

// The plan of a launch that takes the per-head-table kernels.
//
// A SIMD issues from its OLDEST resident wave whenever that wave has an instruction ready (wave
// priorities set by the program do not change that on this chip), and one wave alone keeps the
// vector pipe only about half busy.  Four waves with equal shares of work therefore finish one
// after the other (measured at B=128, 32 heads, 4096 tokens in two even segments: the four waves of
// a SIMD are done after 131, 188, 261 and 327 us) and the pipe idles more and more towards the end.
// So the shares are made UNEVEN, in the proportions in which the four slots of a SIMD actually
// progress while all are resident (FT_SKEW, oldest first): a workgroup's waves 4k..4k+3 are slot k
// of its four SIMDs, interleave_segment gives quad k of a workgroup segment k of a group of four,
// and the context of every sequence is cut into groups of four such segments, at checkpoints.
//
// That needs four segments where the even plan has one or two, hence more workgroups than CUs;
// a second round of workgroups costs a table build, a launch gap and a second ragged end (12 % at
// the shape above).  Instead each launched workgroup walks through several VIRTUAL workgroups of
// its head one after the other (phys_per_head apart) with no barrier between them.
//
// Measured at B=128, 32 heads, 4096 tokens, checkpoints every 256 (medians of interleaved runs on
// one device, us): forward_qk 300-303 with two even segments, 297 with four even ones walked as
// two virtual workgroups, 280-285 with shares 7:5:2:2 (8:4:2:2 and 6:6:3:1 within 3 us of that,
// 9:4:2:1 302); forward_ov 261 with two even segments added inside the workgroup, 262-266 with the
// best uneven shares (6:5:3:2, 7:5:2:2) plus the 4 us kernel that then adds the partial sums: no
// gain, so forward_ov takes uneven shares only where one group of four segments fills the device and
// the four are added inside the workgroup (plan_ft_ov): with 16 lanes per head at that shape, 259
// even, 250 with 6:5:3:2 (8:4:2:2 251, 7:5:2:2 252, 6:4:3:3 and 5:5:3:3 257).
// Shares of a SIMD's work given to its four wave slots, oldest first, in sixteenths of a group's
// checkpoint intervals: measured on the headline shape, one setting per kernel.
constexpr unsigned FT_SKEW_QK = pack_skew(7, 5, 2, 2);
constexpr unsigned FT_SKEW_OV = pack_skew(6, 5, 3, 2);
// matrix-core kernels in 16-wave workgroups, measured on B=16, 32 query heads over 8 KV heads, 131072
// tokens of 2-bit codes (64 segments, us): forward_qk 320 even, 299 with 6:5:3:2 (305 with 7:5:2:2,
// 318 with 6:6:3:1, 330 with 8:4:2:2); forward_ov 265 even, 252 with 6:5:3:2 / 6:6:3:1 / 8:5:2:1
constexpr unsigned GQA_SKEW_QK = pack_skew(6, 5, 3, 2);
constexpr unsigned GQA_SKEW_OV = pack_skew(6, 5, 3, 2);
constexpr bool FT16_QK = true, FT16_OV = true; // whether forward_qk / forward_ov may take 16 lanes per head
constexpr int FT_MIN_GROUP = 8;  // checkpoint intervals a group needs for its shares to differ
constexpr int FT_MAX_GROUPS = 16;

// Longest segment of an uneven cut, in checkpoint intervals (the oldest wave slot's of the group
// that got the most intervals).
// The groups have intervals / groups intervals, rounded down or up, so two are looked at.
static int uneven_longest(int groups, int intervals, unsigned skew)
{
    int part[4], longest;
    uneven_parts(intervals / groups, skew, part);
    longest = part[0];
    if (intervals % groups) {
        uneven_parts(intervals / groups + 1, skew, part);
        longest = std::max(longest, part[0]);
    }
    return longest;
}

// What a unit (one wave's segment) costs besides its tokens, in tokens: parameters, checkpoint,
// the first loads' latency, the first lookups, the last reduction.
constexpr int FT_UNIT_OVERHEAD_TOKENS = 32;

// Groups and workgroups per head are chosen together, for the shortest launch by the model
//   rounds of workgroups on the CUs x virtual workgroups walked through by each x longest segment.
// (Groups by occupancy alone, then workgroups, left awkward batches on two thirds of the CUs:
// 40 sequences x 32 heads x 8192 tokens took two groups and 160 workgroups of two virtual ones
// where three groups fill 256.)  Ties go to fewer groups, then fewer workgroups.  virtual_ok =
// false (forward_ov, whose kernel runs one virtual workgroup per workgroup) only considers plans
// with as many workgroups as virtual ones.
static void plan_head_table(Seg &seg, int B, int H, int T, unsigned skew, int upw, bool virtual_ok = true)
{
    seg.groups = 0;
    const int n_cus = cus(); // asks the runtime for the device: once per plan
    seg.skew = skew;
    seg.phys_per_head = ft_wgs_per_head(B, seg.nseg, upw);
    if (!seg.ckpt || seg.ckpt_interval <= 0 || skew == 0)
        return;
    const int iv = seg.ckpt_interval;
    const int avail = (T + iv - 1) / iv;
    int gmax = avail / FT_MIN_GROUP; // FT_MIN_GROUP intervals or more per group
    if (gmax > FT_MAX_GROUPS)
        gmax = FT_MAX_GROUPS;
    int best_g = 0, best_p = 0;
    double best_cost = -1.0;
    for (int G = 1; G <= gmax; G++) {
        // segment s > 0 starts from checkpoint cut(s) - 1
        if (uneven_cut(4 * G - 1, G, avail, skew) - 1 >= seg.n_ckpt_cap)
            continue;
        const int W = ft_wgs_per_head(B, 4 * G, upw);
        const double unit = (double)uneven_longest(G, avail, skew) * iv + FT_UNIT_OVERHEAD_TOKENS;
        for (int P = virtual_ok ? 1 : W; P <= W; P++) {
            const double cost = (double)(((long)H * P + n_cus - 1) / n_cus) * ((W + P - 1) / P) * unit;
            if (best_cost < 0.0 || cost < 0.999 * best_cost) {
                best_g = G;
                best_p = P;
                best_cost = cost;
            }
        }
    }
    if (best_g == 0)
        return;
    seg.groups = best_g;
    seg.intervals = avail;
    seg.nseg = 4 * best_g;
    seg.seg_tokens = iv; // not read by the kernels of an uneven plan
    seg.phys_per_head = best_p;
}

// Length of a launch under a per-head-table plan, in tokens of a 32-lane wave's work: rounds of
// workgroups on the CUs x virtual workgroups walked through by each x the longest segment (the
// oldest wave slot's), x 1.86 for a head over 16 lanes (eight channels per lane at 0.93 of the
// instructions per channel).
static double ft_plan_cost(const Seg &s, int B, int H, int T, int upw)
{
    const int W = ft_wgs_per_head(B, s.nseg, upw);
    const int P = s.phys_per_head > 0 ? s.phys_per_head : W;
    const long rounds = ((long)H * P + cus() - 1) / cus();
    const int virt = (W + P - 1) / P;
    const int longest = s.groups ? uneven_longest(s.groups, s.intervals, s.skew) * s.ckpt_interval
                                 : (s.seg_tokens < T ? s.seg_tokens : T);
    return (double)rounds * virt * (longest + FT_UNIT_OVERHEAD_TOKENS) * (upw == 4 ? 1.86 : 1.0);
}

// Lanes per head of the per-head-table kernels for a launch, and its plan (`seg` comes in as the
// launch's even plan for 32 lanes and goes out as the plan to run).  Sixteen lanes per head (four
// sequences per wave, two passes over every supergroup) spend 5-7 % fewer instructions per channel
// but need twice the segments for the same number of waves.  They are taken when their plan is
// uneven with groups of at least FT16_MIN_GROUP checkpoint intervals (so that the four shares keep
// their proportions and the shortest segment its length) and shorter than the 32-lane plan by
// ft_plan_cost; 32 lanes otherwise.  Measured, 32 heads, checkpoints every 256 tokens, layer-step
// with 32 / 16 lanes in us (each with the plan the model picks for it): B x ctx 128 x 4096
// 581 / 552, 100 x 4096 528 / 475, 200 x 4096 1014 / 948, 352 x 4096 1667 / 1563, 16 x 32768
// 570 / 537 (16 lanes shorter by the model); 24 x 16384 463 / 495, 40 x 8192 406 / 473, 96 x 4096
// 466 / 481, 8 x 65536 569 / 714 (32 lanes shorter: the 16-lane plans leave padding waves or CUs
// idle); 64 x 4096 303 / 304, 128 x 2048 290 / 304 (groups of 8); 128 x 640 106 / 131 (even plans).
constexpr int FT16_MIN_GROUP = 16;
static int plan_ft(Seg &seg, int B, int H, int T, unsigned skew, bool sixteen_ok, bool virtual_ok = true)
{
    const int forced = g_mha_kernel.load(std::memory_order_relaxed); // 3: sixteen lanes, 4: thirty-two
    Seg s32 = seg;
    plan_head_table(s32, B, H, T, skew, 2, virtual_ok);
    if (sixteen_ok && forced != 4) {
        Seg s16 = plan_segments(seg.ckpt, seg.n_ckpt_cap, seg.ckpt_interval, B * H, T, 128, 16);
        s16.row_pitch = seg.row_pitch;
        s16.act_bf16 = seg.act_bf16;
        plan_head_table(s16, B, H, T, skew, 4, virtual_ok);
        const bool long_groups = s16.groups > 0 && s16.intervals / s16.groups >= FT16_MIN_GROUP;
        if (forced == 3 ||
            (long_groups && ft_plan_cost(s16, B, H, T, 4) < 0.97 * ft_plan_cost(s32, B, H, T, 2))) {
            seg = s16;
            return 16;
        }
    }
    seg = s32;
    return 32;
}

// forward_ov's plan: ov_ft_kernel runs one virtual workgroup per workgroup and adds two or four
// segments of a sequence inside the workgroup; whatever else it leaves in the workspace costs a
// second kernel of some 5 us.  Uneven shares pay with a head over 16 lanes (measured at 16-lane
// shapes: 128 x 4096 266 -> 249 us added in the workgroup; 16 x 32768, 64 x 8192, 32 x 16384
// 262 -> 242 us through the workspace) and not with a head over 32 (64 x 4096: 127.5 either way;
// 8 x 65536: 250 even, 258 uneven): they are taken when the uneven plan has 16 lanes per head and
// needs no virtual workgroups, the even plan for 32 lanes otherwise.
static int plan_ft_ov(Seg &seg, int B, int H, int T)
{
    Seg un = seg;
    const int lanes_un = plan_ft(un, B, H, T, FT_SKEW_OV, FT16_OV, false);
    if (lanes_un == 16 && un.groups >= 1 && un.phys_per_head == ft_wgs_per_head(B, un.nseg, 4)) {
        seg = un;
        return 16;
    }
    return plan_ft(seg, B, H, T, 0, FT16_OV);
}
static bool ft_ov_combines(const Seg &seg, int B, int lanes)
{
    return (seg.nseg == 2 || seg.nseg == 4) && seg.phys_per_head == ft_wgs_per_head(B, seg.nseg, 64 / lanes);
}

// The same uneven shares for the kernels without virtual workgroups (matrix-core and shared-table
// kernels in 16-wave workgroups, where a workgroup's quads of waves are the four slots of its
// SIMDs as well): the even plan's segments, when their number is a multiple of four, are re-cut
// in groups of four.  The segment count, and with it the workgroup count, stays what it was.
static void plan_uneven(Seg &seg, int T, long threads, unsigned skew)
{
    seg.groups = 0;
    seg.skew = skew;
    if (skew == 0 || !seg.ckpt || seg.ckpt_interval <= 0 || threads < 1024L * cus() || seg.nseg < 4 || (seg.nseg & 3))
        return;
    const int avail = (T + seg.ckpt_interval - 1) / seg.ckpt_interval;
    const int G = seg.nseg / 4;
    if (G > FT_MAX_GROUPS || avail / G < FT_MIN_GROUP)
        return;
    if (uneven_cut(4 * G - 1, G, avail, skew) - 1 >= seg.n_ckpt_cap)
        return;
    seg.groups = G;
    seg.intervals = avail;
}

// The plan of a launch of four channels per lane, of matrix-core ones up to four query heads (`seg` comes in as the even plan).  The even
// plan's segments are whole multiples of an interval, all the same, and leave what they leave: 17 x 8 KV heads x 15467 tokens are 61
// segments of one interval in 260 workgroups, two rounds for four of them, and 128 x 2 x 20219 27 segments of three in 216 of 256
// CUs.  So the number of segments is chosen for the workgroups that it makes: as groups of four uneven ones where an interval more or
// less is little of a group, else nearly equal ones of as many intervals as it takes.  The length of a launch is modelled as rounds of
// workgroups x the intervals of a SIMD's three or four waves, over the part of the time that its vector pipe is busy then: 0.80
// with three waves, 0.83 with four alike, 0.89 with four uneven ones (SQ_ACTIVE_INST_VALU).  Another plan has to be 5 % shorter.
// us per step, the even plan (uneven where its segments are a multiple of four) / this: 17 x 8 x 15467 175 / 116, 128 x 2 x 20219 240 / 226, 69 x 2 x
// 46577 307 / 282 (four query heads), 24 x 32 x 12000 2-bit 331 / 318, 48 x 8 x 9000 (two) 159 / 155; the others of eleven such sizes
// keep theirs.  Of 82 sizes drawn at random among those that take another plan than the even one: 29 of one query head in 2 bits 0.90 of
// the even plan's time, 27 of four 0.94, in 2 bits (26) 0.90; the worst 1.010 (20 x 2 x 58865, 136.8 / 138.2, runs 1.8 apart), the others below 1.
// Eight query heads are not planned like this: forward_ov's workgroups have eight waves then, which is not what the model counts.  For
// forward_qk alone it would hold: 17 x 8 x 15467 193 / 161, 24 x 8 x 12000 187 / 185, 16 x 8 x 131072 2-bit 732 / 726, five others the same.
static void plan_rounds(Seg &seg, int per_seg, int T, unsigned skew) // per_seg: waves per segment; skew: 0, no uneven groups
{
    const int n_cus = cus();
    if (!seg.ckpt || seg.ckpt_interval <= 0 || seg.nseg < 2 || (long)per_seg * seg.nseg <= 8L * n_cus)
        return;
    const int avail = (T + seg.ckpt_interval - 1) / seg.ckpt_interval;
    auto rounds = [&](long waves, int &slots) { // of workgroups; the waves of one on a SIMD, as threads_per_workgroup has them
        slots = (waves + n_cus - 1) / n_cus <= 12 ? 3 : 4;
        return (double)(((waves + slots * 4 - 1) / (slots * 4) + n_cus - 1) / n_cus);
    };
    auto cost = [&](const Seg &s) {
        int slots;
        const double r = rounds((long)per_seg * s.nseg, slots);
        if (s.groups > 0)
            return r * ((avail + s.groups - 1) / s.groups) / 0.89;
        const long sum = s.groups < 0 ? ((long)slots * avail + s.nseg - 1) / s.nseg : (long)slots * s.seg_intervals;
        return r * sum / (slots == 4 ? 0.83 : 0.80);
    };
    double best = 0.95 * cost(seg);
    const Seg even = seg;
    auto consider = [&](int groups, int nseg) {
        Seg s = even;
        s.groups = groups;
        s.nseg = nseg;
        s.intervals = avail;
        s.seg_tokens = s.ckpt_interval; // not read
        // the last segment starts from a checkpoint
        const int last = groups > 0 ? uneven_cut(nseg - 1, groups, avail, skew) : balanced_cut(s, nseg - 1);
        if (last - 1 >= s.n_ckpt_cap)
            return;
        const double c = cost(s);
        if (c < best) {
            best = c;
            seg = s;
        }
    };
    for (int round = 1; round <= 2; round++)
        for (int slots = 4; slots >= 3; slots--) {
            const long most = (long)round * n_cus * slots * 4 / per_seg; // segments in that many rounds
            const int groups = (int)std::min(most / 4, (long)avail / FT_MIN_GROUP);
            if (skew && slots == 4 && groups >= 1 && (long)per_seg * 4 * groups > 12L * n_cus)
                consider(groups, 4 * groups);
            const int n = (int)std::min(most, (long)avail);
            if (n >= 2 && (long)per_seg * n > 8L * n_cus)
                consider(-1, n);
        }
}
static void plan_gqa(Seg &seg, int BH, int T, unsigned skew)
{
    plan_uneven(seg, T, padded_units<32>(BH, seg.nseg) * 32, skew);
    plan_rounds(seg, pad4((BH + 1) / 2), T, skew);
}
// Shared-table launches of head dim 128: nearly equal segments only.  us per step, 32 heads, the even plan / this: 10 x 20000 284 / 260, 6 x
// 68692 518 / 505; 26 sizes drawn at random 0.82 to 0.995 of the even plan's time, 0.95 in the mean.  (256 channels, 3 x 16 x 93341, 73 segments / 85: 367 / 362, where two runs of one side differ by as much.)
static void plan_shared(Seg &seg, int BH, int T, int D)
{
    if (D == 128)
        plan_rounds(seg, pad4((BH + 1) / 2), T, 0);
}

// How many segments the forward_ov partial sums of a launch can have under either plan (what a
// workspace must be sized for: the kernel family can be switched between sizing and launch).
static int max_plan_segments(void *ckpt, int n_ckpt_cap, int ckpt_interval, int B, int H, int T, int D)
{
    Seg seg = plan_segments(ckpt, n_ckpt_cap, ckpt_interval, B * H, T, D);
    int n = seg.nseg;
    if (D == 128) {
        Seg a = seg, b = seg, c = seg;
        plan_head_table(a, B, H, T, FT_SKEW_QK, 2);
        plan_ft(b, B, H, T, FT_SKEW_QK, true);
        plan_ft_ov(c, B, H, T);
        n = std::max(std::max(n, a.nseg), std::max(b.nseg, c.nseg));
        Seg d = seg;
        plan_gqa(d, B * H, T, GQA_SKEW_OV);
        n = std::max(n, d.nseg);
    }
    plan_shared(seg, B * H, T, D);
    return std::max(n, seg.nseg);
}

// Whether adkv_decode_step may run its three stages as ONE launch (decode_ft_kernel): off unless
// adkv_set_fused_step(1) asks for it.  Measured at B=128, 32 heads, 4096 tokens (builds alternating
// in one process): 545 us per layer-step in one launch against 543 us in three.  The launch gaps
// and the softmax kernel that the fused launch saves (some 40 us of device idle time per step) buy
// nothing: the device then runs the same instructions at a lower clock.
static std::atomic<int> g_fused_step{0};

// The plans of a fused step, or 0: per-head-table kernels, forward_qk and forward_ov both on four
// segments per sequence with the same lane width and as many workgroups as virtual ones (then the
// four quads of a workgroup hold the four segments of the same sequences).  Returns the lanes
// per head.
static int fused_step_plan(Seg &ka, Seg &va, int B, int Hq, int H, int T, int D, int bits, void *k_ckpt,
                           void *v_ckpt, int n_ckpt_cap, int ckpt_interval)
{
    if (g_fused_step.load(std::memory_order_relaxed) == 0 || Hq != H || D != 128 || bits != 4 || T < 1 ||
        T + 1 > FT_SOFTMAX_MAX_ROW || !k_ckpt || !v_ckpt)
        return 0;
    ka = plan_segments(k_ckpt, n_ckpt_cap, ckpt_interval, B * H, T, D);
    if (mfma_for_mha() || !use_head_table(B, H, 1, bits, D, ka))
        return 0;
    va = plan_segments(v_ckpt, n_ckpt_cap, ckpt_interval, B * H, T, D);
    const int lanes = plan_ft(ka, B, H, T, FT_SKEW_QK, FT16_QK);
    const int lanes_v = plan_ft_ov(va, B, H, T);
    const int W = ft_wgs_per_head(B, 4, 64 / lanes);
    if (lanes != lanes_v || ka.nseg != 4 || va.nseg != 4 || ka.phys_per_head != W || va.phys_per_head != W)
        return 0;
    return lanes;
}

// Whether a step runs as small_step_kernel, and its plan: a workgroup per (sequence, head), one per CU, four
// waves per segment.  us per step on the device, one launch / the two that it would be otherwise (step_beside_lone_kernel), sequences x
// heads x tokens: 1 x 32 x 603 10.7 / 12.2, 4 x 32 x 200 9.4 / 11.0, 8 x 32 x 500 11.9 / 13.5, 8 x 32 x 1000 16.0 / 18.6, 5 x 40 x 700
// 13.2 / 17.3, 2 x 8 x 64 6.3 / 7.8; the second launch costs the host 3 us more.  Four segments of few heads are the other way round,
// 1 x 32 x 1000 14.6 / 12.7, 4 x 32 x 1000 15.3 / 13.2, 1 x 8 x 1024 14.9 / 12.3 (with the rotary embedding and the host's part 17.5 / 16.4,
// 17.3 / 16.4, 17.4 / 15.9): the line does not lie there yet.
// With five to eight segments four waves share a SIMD while other CUs idle, and beyond one workgroup per CU (its LDS
// allows no second) a launch takes two rounds: those stay with the separate launches.
static bool small_step_plan(Seg &seg, int B, int Hq, int H, int T, int D, int bits, void *k_ckpt, void *v_ckpt,
                            int n_ckpt_cap, int ckpt_interval)
{
    if (D != 128 || bits != 4 || Hq != H || T < 0 || T + 1 > SMALL_ROW || (long)B * H > cus() || !k_ckpt != !v_ckpt ||
        g_mha_kernel.load(std::memory_order_relaxed) >= 0 || mha_kernel_default())
        return false;
    seg = plan_segments(k_ckpt, n_ckpt_cap, ckpt_interval, B * H, T, D);
    return seg.nseg <= 4;
}

static int longest_segment(const Seg &seg, int T) { return seg.nseg > 1 ? seg.seg_tokens : T; } // of an even plan

// Whether a step runs as step_segments_kernel + step_combine_kernel, its plan and its channels per lane.
// Every segment has to fit the LDS of its wave and all waves have to be resident: at most four per SIMD
// (two with 184 registers at head dim 512).  us per step on the device, three to four launches / two,
// sequences x query heads x KV heads x tokens (4-bit, head dim 128, checkpoints every 256 unless said):
// 1 x 32 x 8 x 603 50.8 / 21.9, 4 x 32 x 8 x 3000 51.3 / 24.2, 8 x 32 x 8 x 16001 (bf16, with the rotary embedding)
// 65.6 / 58.0, 2 x 64 x 8 x 4000 2-bit 54.8 / 25.1, 1 x 32 x 32 x 2000 28.1 / 20.7, 16 x 32 x 32 x 1500 55.3 /
// 40.4, 64 x 32 x 32 x 663 masked (bf16, with the rotary embedding) 74.3 / 66.0; head dim 256, 16 x 16 heads x
// 4000 93.6 / 90.0, 1 x 8 x 1000 34.5 / 30.6; head dim 512, 8 x 8 x 2000 57.3 / 50.1.
// With one query head two channels per lane are taken as long as four waves per SIMD hold them (12 x 32 heads x
// 2000 tokens: 48.4 with four channels, 40.6 with two), four beyond.
// Of the launches that a table per head pays for (use_head_table) two kinds stay with the three kernels, where
// forward_qk's workgroups are more than half of the CUs and segments longer than 128 tokens: those whose forward_ov
// adds its segments inside the workgroup, and segments beyond 256 tokens.  Three launches / two, 32 heads, every
// 256: 128 x 300 60.0 / 60.7, 128 x 511 89.8 / 93.0, 64 x 1024 90.4 / 93.8; every 512: 100 x 1000 135.4 / 145.1; every
// 128: 16 x 8000 152.7 / 161.2.  The others: 40 x 1100 80.3 / 78.6, 32 x 2048 (half the CUs) 114.4 / 91.3, every
// 128: 128 x 150 36.6 / 35.3, 32 x 2000 85.2 / 83.7, every 512: 32 x 4000 (half) 195.4 / 161.9.
// Segments cut finer than 128 tokens (by checkpoints closer than that) with one query head per KV head stay
// with the separate launches: such a step is the three calls bit for bit, where here a weight is rounded
// before it is divided by its row's sum, at 15.0 us instead of 11.0 (2 x 3 heads x 530, every 64).
static bool segment_step_plan(Seg &seg, int &cpl, int B, int Hq, int H, int T, int D, int bits, void *k_ckpt, void *v_ckpt,
                              int n_ckpt_cap, int ckpt_interval)
{
    const int GQ = Hq / H;
    if ((GQ != 1 && GQ != 2 && GQ != 4 && GQ != 8) || (bits != 4 && bits != 2) || !k_ckpt != !v_ckpt ||
        g_mha_kernel.load(std::memory_order_relaxed) >= 0 || mha_kernel_default())
        return false;
    const int BH = B * H;
    seg = plan_segments(k_ckpt, n_ckpt_cap, ckpt_interval, BH, T, D);
    const int longest = longest_segment(seg, T);
    if (longest + 1 > (GQ == 8 ? step_cap<8>() : step_cap<1>()) || (GQ == 1 && bits == 4 && seg.nseg > 1 && longest < 128))
        return false;
    const long room = (D == 512 ? 2L : 4L) * n_simd();
    cpl = D == 512 ? 8 : D == 256 ? 4 : 2;
    long waves = padded_units<64>(BH, seg.nseg);
    if (waves > room && GQ == 1 && bits == 4 && D == 128) {
        cpl = 4;
        waves = padded_units<32>(BH, seg.nseg) / 2;
        if (waves <= room && longest > 128 && use_head_table(B, H, 1, bits, D, seg)) {
            Seg k = seg, v = seg;
            plan_ft(k, B, H, T, FT_SKEW_QK, FT16_QK);
            const int lanes = plan_ft_ov(v, B, H, T);
            if (2L * H * k.phys_per_head > cus() && (longest > 256 || ft_ov_combines(v, B, lanes)))
                return false;
        }
    }
    return waves <= room;
}

template <int D, int CPL, int BITS, int GQ, typename... Args>
static int launch_step_shape(long waves, hipStream_t st, Args... args)
{
    const long per_cu = (waves + cus() - 1) / cus();
#define ADKV_STEP(BLK)                                                                              \
    hipLaunchKernelGGL((step_segments_kernel<D, CPL, BITS, GQ, BLK>), dim3((unsigned)((waves * 64 + BLK - 1) / BLK)), dim3(BLK), 0, st, args...)
    if (per_cu <= 4) {
        ADKV_STEP(256);
    } else if (D == 512 || per_cu <= 8) {
        ADKV_STEP(512);
    } else if constexpr (D != 512) { // 184 registers: at most two waves per SIMD
        if (per_cu <= 12)
            ADKV_STEP(768);
        else
            ADKV_STEP(1024);
    }
#undef ADKV_STEP
    return check_launch();
}

template <int BITS, typename... Args>
static int launch_step_grouped(int GQ, long waves, hipStream_t st, Args... args)
{
    switch (GQ) {
    case 1: return launch_step_shape<128, 2, BITS, 1>(waves, st, args...);
    case 2: return launch_step_shape<128, 2, BITS, 2>(waves, st, args...);
    case 4: return launch_step_shape<128, 2, BITS, 4>(waves, st, args...);
    default: return launch_step_shape<128, 2, BITS, 8>(waves, st, args...);
    }
}

// Whether a step of the two launches is of one channel per lane, and how many waves of keys a workgroup has: a wave's 64 channels bring
// twice the waves of two channels per lane and four or eight times those of wide heads, and pay as long as a CU holds
// them at once: 16 waves, and 12 / 8 with four / eight query heads, whose logits take more of the LDS; with one or two
// query heads of 128 channels, whose other form has its waves' LDS reads covered by then, 12.  us per step on the
// device, step_segments_kernel / this, waves per CU in brackets (up to eight: with the values beside the keys, see launch_step_lone):
//   512 channels: 9 x 8 heads x 80 (3) 21.5 / 10.3, 2 x 8 x 1000 (2) 47.0 / 16.3, 8 x 8 x 2000 (16) 48.0 / 29.6
//   256: 1 x 8 x 300 30.1 / 11.6, 2 x 16 x 5021 (10) 31.2 / 23.7, 4 x 8 x 8190 (16) 32.8 / 29.2
//   128: 1 x 32 x 2000 (2) 19.5 / 12.4, 4 x 32 x 2000 (8) 20.5 / 18.3, 6 x 32 x 2000 (12) 26.0 / 23.1, 8 x 32 x 2000 (16)
//     27.4 / 28.0
//   two query heads: 4 x 16 x 2000 (4) 20.2 / 12.8, 8 x 16 x 2000 (8) 21.1 / 17.8, 12 x 16 x 2000 (12) 28.8 / 25.6,
//     16 x 16 x 2000 (16) 31.1 / 30.7
//   four: 1 x 8 x 603 21.4 / 12.1, 28 x 8 x 936 (7) 23.6 / 19.0, 8 x 8 x 6000 (12) 32.3 / 28.1, 8 x 8 x 7000 (14) 34.1 / 46
//   eight: 3 x 8 x 113 18.6 / 11.2, 3 x 8 x 4799 (4) 29.0 / 17.0, 8 x 8 x 4000 (8) 33.3 / 24.9, 8 x 8 x 8000 (16) 45.4 / 46.1
//   2-bit codes: 1 x 32 x 2000 17.8 / 11.6, 6 x 32 x 2000 24.7 / 21.9, 12 x 16 x 2000 26.6 / 23.2, 2 x 8 x 8664 21.2 / 17.3,
//     8 x 8 x 6000 30.6 / 26.6, 8 x 8 x 4000 with eight query heads 29.0 / 23.9
// (The sizes beyond the line, of 14 and 16 waves with 128 channels, and the two paragraphs below: before the second launch read ahead, and with
// the values behind the keys.)
// Beyond 16 waves of wide heads the launch takes two rounds or more, and the line is a cautious one: up to 24 workgroups
// smaller than the CU are still the faster ones, by 32 they are not.  step_segments_kernel / this in workgroups of 4,
// 12 and 16 waves (512 channels: 8 and 16): 256 channels, 5 x 8 x 8000 (20) 47.0 / 43.2, 44.3, 51.5, 6 x 8 x 8000 (24) 47.5
// / 47.4, 44.9, 51.8, 8 x 8 x 8000 (32) 49.2 / 60.2, 62.7, 56.7; 512, 10 x 8 x 2000 (20) 50.7 / 48.5, 51.8, 12 x 8 x 2000 (24)
// 51.1 / 49.8, 51.9, 16 x 8 x 2000 (32) 51.8 / 64.2, 56.7 (these with the rotary embedding's launch, some 2 us).
// Small workgroups spread best; what they leave free of a CU's LDS (the table takes 64 KB) holds a second one only with
// one query head.  A workgroup of as many waves as the CU is to hold otherwise: 2 x 16 x 5021 of 256 channels with 4, 8, 12
// and 16 waves 26.5, 32.6, 23.3, 27.4; 28 x 8 x 936 with four query heads 28.1, 21.3, 25.4.
static int step_lone_threads(long units, int D, int GQ, int longest)
{
    const long per_cu = (units * (D / 64) + cus() - 1) / cus();
    const int most = GQ == 8 ? 8 : D == 128 ? 12 : 16;
    if (longest > 256 || per_cu > most)
        return 0;
    if (D == 512)
        return per_cu <= 8 ? 512 : 1024;
    if (per_cu <= (GQ == 1 ? 8 : 4))
        return 256;
    return per_cu <= 8 ? 512 : per_cu <= 12 ? 768 : 1024;
}

// Up to eight waves per CU the values of such a step have waves beside the keys' (step_beside_lone_kernel): as many again, up to two
// per SIMD with registers for 24 units of a segment's values, up to four with registers for 16.  With more both kinds together are
// more than a CU holds.  us per step, one behind the other (step_lone_kernel) / beside, sequences x KV heads x tokens (waves of keys
// per CU): one query head, 1 x 32 x 2000 (2) 14.8 / 12.8, 2 x 32 x 2048 (4) 15.9 / 14.1, 4 x 32 x 2048 (8) 19.3 / 18.4; two, 2 x 8 x 3000 16.1 /
// 13.3, 8 x 16 x 2048 (8) 20.6 / 18.7; four, 1 x 8 x 603 15.5 / 12.6, 1 x 8 x 4000 16.2 / 13.2, 1 x 8 x 16000 (4) 18.1 / 15.6, 1 x 2 x 30000 18.6 /
// 15.8, 3 x 8 x 6000 (5) 20.7 / 18.4, 8 x 8 x 4096 (8) 22.7 / 20.5; eight, 1 x 8 x 4000 17.5 / 14.2, 5 x 8 x 5632 (8) 26.4 / 24.1; 2-bit,
// four, 1 x 8 x 4000 15.0 / 12.3, 6 x 8 x 4096 (6) 20.3 / 18.2, one, 4 x 32 x 2048 (8) 18.4 / 17.8; 256 channels, 1 x 8 x 2000 14.4 / 12.2, 4 x 8 x
// 4000 (8) 18.8 / 18.2; 512, 1 x 8 x 1000 18.4 / 16.6, 2 x 8 x 2000 (4) 18.5 / 17.0.
// Returns the units that a values' wave holds; 0: a wave takes keys and values.  blk: of step_lone_threads.
static int step_values_ahead(int blk, long units, int D)
{
    if (blk == 256)
        return units * (D / 64) <= 4L * cus() ? 24 : 16;
    return blk == 512 ? 16 : 0;
}
template <int D, int BITS, int GQ, typename... Args>
static int launch_step_lone(int blk, long units, hipStream_t st, Args... args)
{
    const int per_block = blk / D, ahead = step_values_ahead(blk, units, D); // units: a wave per 64 channels
    const dim3 grid((unsigned)((units + per_block - 1) / per_block));
#define ADKV_STEP(BLK) hipLaunchKernelGGL((step_lone_kernel<D, BITS, GQ, BLK>), grid, dim3(BLK), 0, st, args...)
#define ADKV_BESIDE(BLK, AHEAD) hipLaunchKernelGGL((step_beside_lone_kernel<D, BITS, GQ, (BLK) / 64, AHEAD>), grid, dim3(2 * (BLK)), 0, st, args...)
    if constexpr (D != 512) {
        if (ahead == 24)
            ADKV_BESIDE(256, 24);
        if constexpr (GQ == 1) {
            if (blk == 256 && ahead == 16)
                ADKV_BESIDE(256, 16);
        }
        if constexpr (GQ != 8) {
            if (blk == 768)
                ADKV_STEP(768);
        }
    }
    if constexpr (D == 512 || GQ > 1) {
        if (ahead == 16 && blk == 512)
            ADKV_BESIDE(512, 16);
    }
    if constexpr (D != 128) {
        if (blk == 1024)
            ADKV_STEP(1024);
    }
#undef ADKV_BESIDE
#undef ADKV_STEP
    return check_launch();
}

template <int BITS, typename... Args>
static int launch_step_lone_grouped(int GQ, int blk, long units, hipStream_t st, Args... args)
{
    switch (GQ) {
    case 1: return launch_step_lone<128, BITS, 1>(blk, units, st, args...);
    case 2: return launch_step_lone<128, BITS, 2>(blk, units, st, args...);
    case 4: return launch_step_lone<128, BITS, 4>(blk, units, st, args...);
    default: return launch_step_lone<128, BITS, 8>(blk, units, st, args...);
    }
}

template <typename... Args>
static int launch_step_segments(int cpl, int GQ, int bits, int D, int BH, int nseg, int longest, hipStream_t st, Args... args)
{
    const long units = padded_units<64>(BH, nseg);
    if (const int blk = step_lone_threads(units, D, GQ, longest)) {
        if (D == 512)
            return launch_step_lone<512, 4, 1>(blk, units, st, args...);
        if (D == 256)
            return launch_step_lone<256, 4, 1>(blk, units, st, args...);
        return bits == 4 ? launch_step_lone_grouped<4>(GQ, blk, units, st, args...)
                         : launch_step_lone_grouped<2>(GQ, blk, units, st, args...);
    }
    if (D == 512)
        return launch_step_shape<512, 8, 4, 1>(units, st, args...);
    if (D == 256)
        return launch_step_shape<256, 4, 4, 1>(units, st, args...);
    if (cpl == 4)
        return launch_step_shape<128, 4, 4, 1>(padded_units<32>(BH, nseg) / 2, st, args...);
    return bits == 4 ? launch_step_grouped<4>(GQ, units, st, args...) : launch_step_grouped<2>(GQ, units, st, args...);
}

static int check_ckpt(const void *ckpt, int n_ckpt_cap, int ckpt_interval, int bits = 4)
{
    if (!ckpt)
        return ADKV_OK;
    // a checkpoint sits on a supergroup boundary: 8 tokens with 4-bit codes, 16 with 2-bit ones
    if (n_ckpt_cap <= 0 || ckpt_interval <= 0 || (ckpt_interval % (32 / bits)))
        return ADKV_E_SHAPE;
    if ((uintptr_t)ckpt & 3)
        return ADKV_E_ALIGN;
    return ADKV_OK;
}

extern "C" {

int adkv_abi_version(void) { return 17; }

void adkv_set_fused_step(int mode) { g_fused_step.store(mode > 0 ? 1 : 0, std::memory_order_relaxed); }

int adkv_decode_step_is_fused(int B, int Hq, int H, int T, int D, int bits, int n_ckpt_cap, int ckpt_interval,
                              int masked)
{
    int dummy = 0;
    Seg ka, va;
    void *ck = n_ckpt_cap > 0 && ckpt_interval > 0 ? &dummy : nullptr;
    if (B <= 0 || H <= 0 || Hq <= 0 || T < 0)
        return 0;
    if (!masked && fused_step_plan(ka, va, B, Hq, H, T, D, bits, ck, ck, n_ckpt_cap, ckpt_interval))
        return 1;
    return small_step_plan(ka, B, Hq, H, T, D, bits, ck, ck, n_ckpt_cap, ckpt_interval) ? 1 : 0;
}

void adkv_set_mha_kernel(int use_matrix_cores)
{
    g_mha_kernel.store(use_matrix_cores < 0 ? -1 : (use_matrix_cores > 4 ? 1 : use_matrix_cores),
                       std::memory_order_relaxed);
}

int adkv_last_hip_error(void) { return g_last_hip_error; }

const char *adkv_strerror(int code)
{
    switch (code) {
    case ADKV_OK: return "ok";
    case ADKV_E_NULL: return "required pointer is NULL";
    case ADKV_E_DIM: return "DIM must be 128, 256 or 512";
    case ADKV_E_SHAPE: return "invalid shape";
    case ADKV_E_CAPACITY: return "cache capacity too small";
    case ADKV_E_ALIGN: return "pointer not sufficiently aligned";
    case ADKV_E_UNSUPPORTED: return "unsupported configuration";
    case ADKV_E_WORKSPACE: return "workspace too small";
    case ADKV_E_SCRATCH_LIMIT:
        return "launch needs more scratch than the library's static buffer holds (adkv_static_scratch_bytes)";
    case ADKV_E_DEVICE: return "HIP device query failed";
    case ADKV_E_LAUNCH: return "HIP launch failed";
    default: return "unknown error";
    }
}

// One tensor, or two of the same shape (v_cache != NULL) in one launch.
static int encode_common(void *cache, const void *kv_new,
                         const void *zp, const void *sc, const void *alpha, const void *beta,
                         const void *tgt,
                         int B, int H, int T0, int T, int D, int n_super_cap,
                         const void *state_in, void *state_out, void *ckpt_out, int n_ckpt_cap,
                         int ckpt_interval, void *stream, int bits = 4,
                         const EncTensor *second = nullptr, const RowStrides *first_strides = nullptr,
                         bool bf16 = false, bool fresh = false)
{
    if (!cache || !kv_new || !zp || !sc || !alpha || !beta || !tgt)
        return ADKV_E_NULL;
    if (second && (!second->cache || !second->kv_new || !second->zp || !second->sc || !second->al ||
                   !second->be || !second->tg))
        return ADKV_E_NULL;
    if (bits != 2 && bits != 4)
        return ADKV_E_UNSUPPORTED;
    int rc = check_common(B, H, T, D, n_super_cap);
    if (rc)
        return rc;
    if (T0 < 0 || T0 > T)
        return ADKV_E_SHAPE;
    if (T0 > 0 && (!state_in || (second && !second->state_in)))
        return ADKV_E_NULL;
    const int tpw = 32 / bits;
    if ((T + tpw - 1) / tpw > n_super_cap)
        return ADKV_E_CAPACITY;
    if (((uintptr_t)cache & 15) || ((uintptr_t)kv_new & 3))
        return ADKV_E_ALIGN;
    if (second && (((uintptr_t)second->cache & 15) || ((uintptr_t)second->kv_new & 3)))
        return ADKV_E_ALIGN;
    if (second && (ckpt_out == nullptr) != (second->ckpt == nullptr))
        return ADKV_E_NULL; // both tensors keep checkpoints or neither does
    const RowStrides packed = {(long)H * (T - T0) * D, (long)(T - T0) * D, (long)D};
    const RowStrides xs1 = first_strides ? *first_strides : packed;
    for (const RowStrides *xs : {&xs1, second ? &second->xs : &xs1}) {
        // rows are read as aligned 32-bit words
        if (xs->b < 0 || xs->h < 0 || xs->t < D || (xs->b | xs->h | xs->t) & 1)
            return ADKV_E_SHAPE;
    }
    if ((rc = check_ckpt(ckpt_out, n_ckpt_cap, ckpt_interval, bits)))
        return rc;
    if (T == T0 && !second && (state_out == nullptr || state_out == state_in))
        return ADKV_OK;
    const int BH = B * H;
    hipStream_t st = (hipStream_t)stream;
    Seg seg;
    seg.ckpt = (h1 *)ckpt_out;
    seg.n_ckpt_cap = n_ckpt_cap;
    seg.ckpt_interval = ckpt_out ? ckpt_interval : 0;
    seg.seg_tokens = T > 0 ? T : 1;
    seg.nseg = 1;
    seg.row_pitch = T + 1;
    seg.act_bf16 = 0;
    seg.combine = 0;
    seg.groups = 0;
    seg.intervals = 0;
    seg.phys_per_head = 0;
    seg.skew = 0;
    seg.fresh = fresh ? 1 : 0;
    // Lane width: one channel per lane while every wave then has a SIMD to itself (its time per token is
    // its instruction count, 17 against 30 with two channels), two channels beyond (they share the
    // packed updates and the wave's fixed cost), but for launches of two to three one-channel waves per
    // SIMD: two channels per lane put two waves on some SIMDs and one on others, and take as long as two
    // everywhere; one channel per lane takes a round of two waves (their LDS) and a round of one, which
    // is less from some 300 tokens on, where rows come through the LDS.  us, bf16 rows, 4-bit codes, one
    // channel / two, at 2.12, 2.5 and 3 one-channel waves per SIMD: 128 tokens 18.9 / 19.5, 19.9 / 20.0,
    // 21.3 / 19.8; 500 tokens 57 / 62, 58 / 62, 59 / 62; 2048 tokens 200 / 232, 205 / 234, 214 / 238.  Outside: 1.25
    // 41 / 37 (500 tokens) and 137 / 135 (2048), 2 42 / 38 and 282 / 278 (4096), 3.25 76 / 65 and 267 / 247,
    // 16 290 / 285 (512; 4.5 TB/s and the vector pipe 85 % busy).
    const long channels = (long)BH * D;
    const long tensors = second ? 2 : 1;
    const long one_per_simd = 64L * n_simd(), all = tensors * channels;
    auto lds_rows = [](const void *x, const RowStrides &s) {
        return ((uintptr_t)x & 15) == 0 && s.t % 8 == 0 && s.h % 8 == 0 && s.b % 8 == 0;
    };
    const bool two_and_one = all > 2 * one_per_simd && all <= 3 * one_per_simd && T - T0 >= 384 && lds_rows(kv_new, xs1) &&
                             (!second || lds_rows(second->kv_new, second->xs)) &&
                             (!ckpt_out || (ckpt_interval % 64 == 0 && T0 % 64 == 0));
    int cpl = all > one_per_simd && !two_and_one ? 2 : 1;
    const long lanes = channels / cpl;
    const dim3 grid((unsigned)((lanes + 255) / 256), (unsigned)tensors), block(256);
    EncTensor first;
    first.cache = (uint32_t *)cache;
    first.kv_new = (const h1 *)kv_new;
    first.zp = (const h1 *)zp;
    first.sc = (const h1 *)sc;
    first.al = (const h1 *)alpha;
    first.be = (const h1 *)beta;
    first.tg = (const h1 *)tgt;
    first.state_in = (const h1 *)state_in;
    first.state_out = (h1 *)state_out;
    first.ckpt = (h1 *)ckpt_out;
    first.xs = xs1;
#define ADKV_ENC(BB, C)                                                                          \
    do {                                                                                         \
        if (second && bf16)                                                                      \
            hipLaunchKernelGGL((encode_pair_kernel<BB, C, 256, true>), grid, block, 0, st,       \
                               first, *second, BH, H, T0, T, D, n_super_cap, seg);               \
        else if (second)                                                                         \
            hipLaunchKernelGGL((encode_pair_kernel<BB, C, 256, false>), grid, block, 0, st,      \
                               first, *second, BH, H, T0, T, D, n_super_cap, seg);               \
        else                                                                                     \
            hipLaunchKernelGGL((encode_kernel<BB, C, 256>), grid, block, 0, st, first.cache,     \
                               first.kv_new, first.zp, first.sc, first.al, first.be, first.tg,   \
                               BH, H, T0, T, D, n_super_cap, first.state_in, first.state_out,    \
                               seg);                                                             \
    } while (0)
#define ADKV_ENC_CPL(BB)                                                                         \
    do {                                                                                         \
        if (cpl == 2)                                                                            \
            ADKV_ENC(BB, 2);                                                                     \
        else                                                                                     \
            ADKV_ENC(BB, 1);                                                                     \
    } while (0)
    if (bits == 4)
        ADKV_ENC_CPL(4);
    else
        ADKV_ENC_CPL(2);
#undef ADKV_ENC_CPL
#undef ADKV_ENC
    return check_launch();
}

int adkv_encode_kv_ex(void *cache, const void *kv_new,
                      const void *zp, const void *sc, const void *alpha, const void *beta,
                      const void *tgt,
                      int B, int H, int T, int D, int n_super_cap,
                      void *state_out, void *ckpt_out, int n_ckpt_cap, int ckpt_interval,
                      void *stream)
{
    return encode_common(cache, kv_new, zp, sc, alpha, beta, tgt, B, H, 0, T, D, n_super_cap,
                         nullptr, state_out, ckpt_out, n_ckpt_cap, ckpt_interval, stream);
}

int adkv_append_kv(void *cache, const void *kv_new,
                   const void *zp, const void *sc, const void *alpha, const void *beta,
                   const void *tgt,
                   int B, int H, int T0, int n_new, int D, int n_super_cap, int bits,
                   void *state_io, void *ckpt, int n_ckpt_cap, int ckpt_interval, void *stream)
{
    if (!state_io)
        return ADKV_E_NULL;
    if (n_new < 0)
        return ADKV_E_SHAPE;
    if (n_new == 0)
        return ADKV_OK; // nothing to quantise; state_io already is the answer
    return encode_common(cache, kv_new, zp, sc, alpha, beta, tgt, B, H, T0, T0 + n_new, D,
                         n_super_cap, state_io, state_io, ckpt, n_ckpt_cap, ckpt_interval, stream,
                         bits);
}

static int encode_pair(bool fresh, void *k_cache, void *v_cache, const void *k_new, const void *v_new,
                        int kv_dtype, const int64_t *k_strides, const int64_t *v_strides,
                        const void *const *k_params, const void *const *v_params,
                        int B, int H, int T0, int n_new, int D, int n_super_cap, int bits,
                        void *k_state_io, void *v_state_io, void *k_ckpt, void *v_ckpt,
                        int n_ckpt_cap, int ckpt_interval, void *stream)
{
    if (!k_params || !v_params || !k_state_io || !v_state_io)
        return ADKV_E_NULL;
    if (kv_dtype != ADKV_DT_F16 && kv_dtype != ADKV_DT_BF16)
        return ADKV_E_UNSUPPORTED;
    if (n_new < 0)
        return ADKV_E_SHAPE;
    if (n_new == 0)
        return ADKV_OK;
    const RowStrides packed = {(long)H * n_new * D, (long)n_new * D, (long)D};
    const RowStrides ks = k_strides ? RowStrides{(long)k_strides[0], (long)k_strides[1], (long)k_strides[2]} : packed;
    EncTensor v;
    v.cache = (uint32_t *)v_cache;
    v.kv_new = (const h1 *)v_new;
    v.zp = (const h1 *)v_params[0];
    v.sc = (const h1 *)v_params[1];
    v.al = (const h1 *)v_params[2];
    v.be = (const h1 *)v_params[3];
    v.tg = (const h1 *)v_params[4];
    v.state_in = (const h1 *)v_state_io;
    v.state_out = (h1 *)v_state_io;
    v.ckpt = (h1 *)v_ckpt;
    v.xs = v_strides ? RowStrides{(long)v_strides[0], (long)v_strides[1], (long)v_strides[2]} : packed;
    return encode_common(k_cache, k_new, k_params[0], k_params[1], k_params[2], k_params[3],
                         k_params[4], B, H, T0, T0 + n_new, D, n_super_cap, k_state_io, k_state_io,
                         k_ckpt, n_ckpt_cap, ckpt_interval, stream, bits, &v, &ks,
                         kv_dtype == ADKV_DT_BF16, fresh);
}

int adkv_append_kv_pair(void *k_cache, void *v_cache, const void *k_new, const void *v_new,
                        int kv_dtype, const int64_t *k_strides, const int64_t *v_strides,
                        const void *const *k_params, const void *const *v_params,
                        int B, int H, int T0, int n_new, int D, int n_super_cap, int bits,
                        void *k_state_io, void *v_state_io, void *k_ckpt, void *v_ckpt,
                        int n_ckpt_cap, int ckpt_interval, void *stream)
{
    return encode_pair(false, k_cache, v_cache, k_new, v_new, kv_dtype, k_strides, v_strides, k_params, v_params,
                       B, H, T0, n_new, D, n_super_cap, bits, k_state_io, v_state_io, k_ckpt, v_ckpt, n_ckpt_cap,
                       ckpt_interval, stream);
}

int adkv_prefill_kv_pair(void *k_cache, void *v_cache, const void *k_new, const void *v_new,
                         int kv_dtype, const int64_t *k_strides, const int64_t *v_strides,
                         const void *const *k_params, const void *const *v_params,
                         int B, int H, int n_new, int D, int n_super_cap, int bits,
                         void *k_state_out, void *v_state_out, void *k_ckpt, void *v_ckpt,
                         int n_ckpt_cap, int ckpt_interval, void *stream)
{
    if (n_new <= 0)
        return ADKV_E_SHAPE; // nothing would be written
    return encode_pair(true, k_cache, v_cache, k_new, v_new, kv_dtype, k_strides, v_strides, k_params, v_params,
                       B, H, 0, n_new, D, n_super_cap, bits, k_state_out, v_state_out, k_ckpt, v_ckpt, n_ckpt_cap,
                       ckpt_interval, stream);
}

int adkv_encode_kv(void *cache, const void *kv_new,
                   const void *zp, const void *sc, const void *alpha, const void *beta,
                   const void *tgt,
                   int B, int H, int T, int D, int n_super_cap,
                   float, float, void *state_out, void *stream)
{
    return adkv_encode_kv_ex(cache, kv_new, zp, sc, alpha, beta, tgt, B, H, T, D, n_super_cap,
                             state_out, nullptr, 0, 0, stream);
}

} // extern "C"

template <bool HALF>
static int softmax_launch(const void *logits, void *weights, const Mask &mask, int rows, int n, int64_t ld, float scaling,
                          void *workspace, int64_t workspace_bytes, void *stream)
{
    if (!logits || !weights)
        return ADKV_E_NULL;
    if (rows <= 0 || n <= 0 || (mask.p && mask.rows_per_mask_row <= 0) || (ld != 0 && ld < n))
        return ADKV_E_SHAPE;
    if (ld == 0)
        ld = n;
    if (n <= 64 * SM_VEC * 4) {
        // short rows: a wave per row, the row in 8, 16 or 32 registers per lane (longer rows were
        // measured slower this way: 27 us against 22 us for 4096 rows of 4097 elements)
        const dim3 grid((unsigned)((rows + SM_BLOCK / 64 - 1) / (SM_BLOCK / 64)));
#define ADKV_SM_WAVE(NVW)                                                                           \
    hipLaunchKernelGGL((softmax_wave_kernel<NVW, HALF>), grid, dim3(SM_BLOCK), 0, (hipStream_t)stream,      \
                       (const h1 *)logits, (h1 *)weights, mask, rows, n, (long)ld, scaling)
        if (n <= 64 * SM_VEC)
            ADKV_SM_WAVE(1);
        else if (n <= 64 * SM_VEC * 2)
            ADKV_SM_WAVE(2);
        else
            ADKV_SM_WAVE(4);
#undef ADKV_SM_WAVE
        return check_launch();
    }
    const int reg_nv = (n + 1024 * SM_VEC - 1) / (1024 * SM_VEC); // 16-byte vectors per thread
    if (n > SM_ROW_MAX && !mask.p && n <= SM_REG_MAX && (rows >= SM_REG_MIN_ROWS || reg_nv <= 9) &&
        scaling != 0.0f && scaling == scaling) {
        // long unmasked rows stay in registers, unless they are few and very long (32 rows of
        // 131 073: 14.6 us cut into chunks, 19.8 us this way; 128 rows: 28.1 and 24.8; 512 rows:
        // 74.8 and 56.7; 64 rows of 32 769: 11.4 and 9.4; 4096 rows of 24 577: 148 and 80)
#define ADKV_SM_REG(NV)                                                                             \
    case NV:                                                                                        \
        hipLaunchKernelGGL(softmax_regrow_kernel<NV>, dim3((unsigned)rows), dim3(1024), 0,          \
                           (hipStream_t)stream, (const h1 *)logits, (h1 *)weights, n, (long)ld,     \
                           scaling);                                                                \
        break
        switch (reg_nv) {
            ADKV_SM_REG(4); ADKV_SM_REG(5); ADKV_SM_REG(6); ADKV_SM_REG(7); ADKV_SM_REG(8);
            ADKV_SM_REG(9); ADKV_SM_REG(10); ADKV_SM_REG(11); ADKV_SM_REG(12); ADKV_SM_REG(13);
            ADKV_SM_REG(14); ADKV_SM_REG(15); ADKV_SM_REG(16);
        default:
            ADKV_SM_REG(17);
        }
#undef ADKV_SM_REG
        return check_launch();
    }
    const int64_t need = adkv_softmax_workspace_bytes(rows, n);
    if (need == 0 || !workspace || rows > 65535) {
        // one workgroup per row, sized so that the row stays in its registers (read once, written
        // once); rows beyond 24576 elements without a workspace are read three times
#define ADKV_SM_ROW(NT, NV)                                                                         \
    hipLaunchKernelGGL((softmax_kernel<NT, NV, HALF>), dim3((unsigned)rows), dim3(NT), 0,                 \
                       (hipStream_t)stream, (const h1 *)logits, (h1 *)weights, mask, n, (long)ld, scaling)
        // (threads, 16-byte vectors per thread) per row length, measured on 4096 rows: 4097 elements
        // 18.4 us with 256 x 3 and 16.7 with 320 x 2; 8192: 35.5 with 512 x 3, 24.3 with 512 x 2;
        // 10000: 36.9 with 512 x 3, 33.0 with 256 x 6; 16384: 76.5 with 1024 x 3, 46.9 with 1024 x 2;
        // 2048 rows of 24576: 42.1 with 1024 x 3, 37.4 with 512 x 6
        if (n <= 5120)
            ADKV_SM_ROW(320, 2);
        else if (n <= SM_CHUNK || n > SM_ROW_MAX)
            ADKV_SM_ROW(SM_BLOCK, SM_NV);
        else if (n <= 8192)
            ADKV_SM_ROW(512, 2);
        else if (n <= 12288)
            ADKV_SM_ROW(256, 6);
        else if (n <= 16384)
            ADKV_SM_ROW(1024, 2);
        else
            ADKV_SM_ROW(512, 6);
#undef ADKV_SM_ROW
        return check_launch();
    }
    if (workspace_bytes < need)
        return ADKV_E_WORKSPACE;
    if ((uintptr_t)workspace & 7)
        return ADKV_E_ALIGN;
    const int nchunk = (n + SM_CHUNK - 1) / SM_CHUNK;
    const dim3 grid((unsigned)nchunk, (unsigned)rows);
    if (nchunk >= 8 && !mask.p) {
        // long rows: four chunks per workgroup in the first pass
        const dim3 grid4((unsigned)((nchunk + 3) / 4), (unsigned)rows);
        hipLaunchKernelGGL(softmax_part_kernel<4>, grid4, dim3(SM_BLOCK), 0, (hipStream_t)stream,
                           (const h1 *)logits, mask, (float2 *)workspace, n, (long)ld, nchunk, scaling);
    } else {
        hipLaunchKernelGGL(softmax_part_kernel<1>, grid, dim3(SM_BLOCK), 0, (hipStream_t)stream,
                           (const h1 *)logits, mask, (float2 *)workspace, n, (long)ld, nchunk, scaling);
    }
    hipLaunchKernelGGL(softmax_norm_kernel, grid, dim3(SM_BLOCK), 0, (hipStream_t)stream,
                       (const h1 *)logits, (h1 *)weights, mask, (const float2 *)workspace, n, (long)ld, nchunk, scaling);
    return check_launch();
}

// Which decode kernel family and shape forward_qk (ov: forward_ov, of 16-byte aligned rows) takes for these sizes: the
// dispatch below, as text.
static const char *decode_kernel_name(bool ov, int B, int Hq, int H, int T, int D, int bits, int n_ckpt_cap,
                                      int ckpt_interval)
{
    if (B <= 0 || H <= 0 || Hq <= 0 || Hq % H || T < 0 || (D != 128 && D != 256 && D != 512) ||
        (bits != 2 && bits != 4))
        return "invalid";
    const int GQ = Hq / H, BH = B * H;
    if ((GQ > 1 || bits != 4) && D != 128)
        return "invalid";
    int dummy = 0;
    const Seg seg = plan_segments(n_ckpt_cap > 0 && ckpt_interval > 0 ? &dummy : nullptr, n_ckpt_cap,
                                  ckpt_interval, BH, T, D);
    if (D == 128 && (GQ > 1 || bits != 4 || mfma_for_mha())) {
        if (ov ? ov_gqa_pair(BH, seg.nseg, GQ, true) : gqa_pair(BH, seg.nseg))
            return "gqa_kernel, two channels per lane (matrix cores)";
        Seg s = seg;
        if (GQ <= 4)
            plan_gqa(s, BH, T, ov ? GQA_SKEW_OV : GQA_SKEW_QK);
        const int blk = threads_per_workgroup(padded_units<32>(BH, s.nseg) * 32);
        if (ov && (GQ > 4 || blk == 256))
            return "gqa_kernel, 8-wave workgroups (matrix cores)";
        return blk == 1024 ? "gqa_kernel, 16-wave workgroups (matrix cores)"
                           : "gqa_kernel, 12-wave workgroups (matrix cores)";
    }
    if (use_head_table(B, H, GQ, bits, D, seg)) {
        Seg s2 = seg;
        const int lanes = ov ? plan_ft_ov(s2, B, H, T) : plan_ft(s2, B, H, T, FT_SKEW_QK, FT16_QK);
        if (lanes == 16)
            return s2.groups ? "ft_kernel (per-head table, 16 lanes per head, 16-wave workgroups, uneven segments)"
                             : "ft_kernel (per-head table, 16 lanes per head, 16-wave workgroups)";
        return s2.groups ? "ft_kernel (per-head table, 16-wave workgroups, uneven segments)"
                         : "ft_kernel (per-head table, 16-wave workgroups)";
    }
    if (D == 128) {
        if (ov ? ov_lone(BH, seg.nseg, T) : qk_lone(BH, seg.nseg, T))
            return "lone_kernel (shared table, one channel per lane)";
        if (!ov && qk_pair(BH, seg.nseg))
            return "kernel<128,2,256> (shared table, two channels per lane)";
        Seg s2 = seg;
        plan_shared(s2, BH, T, D);
        const int blk = threads_per_workgroup(padded_units<32>(BH, s2.nseg) * 32);
        return blk == 1024 ? "kernel<128,4,1024> (shared table)"
               : blk == 768 ? "kernel<128,4,768> (shared table)"
                            : "kernel<128,4,256> (shared table)";
    }
    return D == 256 ? "kernel<256,4,*> (shared table)" : "kernel<512,8,256> (shared table)";
}

// act_bf16: q, k_new / v_new and the output are bfloat16 (only adkv_decode_step asks for it)
static int forward_qk_impl(const void *q, void *k_cache, const void *k_new, void *logits,
                           const void *zp, const void *sc, const void *alpha, const void *beta,
                           const void *tgt,
                           int B, int Hq, int H, int T, int D, int n_super_cap, int bits, int64_t ld,
                           void *state_out, void *ckpt, int n_ckpt_cap, int ckpt_interval,
                           void *stream, int act_bf16)
{
    if (ld != 0 && ld < (int64_t)T + 1)
        return ADKV_E_SHAPE;
    if (!q || !k_cache || !k_new || !logits || !zp || !sc || !alpha || !beta || !tgt)
        return ADKV_E_NULL;
    if (bits != 2 && bits != 4)
        return ADKV_E_UNSUPPORTED;
    int rc = check_common(B, H, T, D, n_super_cap);
    if (rc)
        return rc;
    if (Hq <= 0 || Hq % H)
        return ADKV_E_SHAPE;
    const int GQ = Hq / H;
    if ((GQ > 1 || bits != 4) && D != 128)
        return ADKV_E_UNSUPPORTED;
    if (T / (32 / bits) >= n_super_cap)
        return ADKV_E_CAPACITY;
    if (((uintptr_t)k_cache & 15) || ((uintptr_t)q & 7) || ((uintptr_t)k_new & 3))
        return ADKV_E_ALIGN;
    if ((rc = check_ckpt(ckpt, n_ckpt_cap, ckpt_interval, bits)))
        return rc;
    const int BH = B * H;
    hipStream_t st = (hipStream_t)stream;
    Seg seg = plan_segments(ckpt, n_ckpt_cap, ckpt_interval, BH, T, D);
    seg.act_bf16 = act_bf16;
    if (ld)
        seg.row_pitch = ld;
    if (D == 128 && (GQ > 1 || bits != 4 || mfma_for_mha())) {
        const bool pair = gqa_pair(BH, seg.nseg);
        if (GQ <= 4 && !pair)
            plan_gqa(seg, BH, T, GQA_SKEW_QK);
        ADKV_DISPATCH_GQ(qk_gqa_kernel, true, (const h1 *)q, (uint4 *)k_cache, (const h1 *)k_new,
                         (h1 *)logits, (const h1 *)zp, (const h1 *)sc, (const h1 *)alpha,
                         (const h1 *)beta, (const h1 *)tgt, BH, H, T, n_super_cap, (h1 *)state_out,
                         seg);
        return check_launch();
    }
    if (use_head_table(B, H, GQ, bits, D, seg)) {
        const int lanes = plan_ft(seg, B, H, T, FT_SKEW_QK, FT16_QK);
        const auto kernel = lanes == 16 ? qk_ft_kernel<16> : qk_ft_kernel<32>;
        hipLaunchKernelGGL(kernel, dim3((unsigned)(H * seg.phys_per_head)), dim3(FT_BLK), 0, st,
                           (const h1 *)q, (uint4 *)k_cache, (const h1 *)k_new, (h1 *)logits,
                           (const h1 *)zp, (const h1 *)sc, (const h1 *)alpha, (const h1 *)beta,
                           (const h1 *)tgt, B, H, T, n_super_cap, (h1 *)state_out, seg);
        return check_launch();
    }
    if (D == 128 && qk_lone(BH, seg.nseg, T)) {
        const FtParams p = {(const h1 *)zp, (const h1 *)sc, (const h1 *)alpha, (const h1 *)beta, (const h1 *)tgt};
        ADKV_LAUNCH_LONE(qk_lone_kernel, 768, (const h1 *)q,
                           (uint4 *)k_cache, (const h1 *)k_new, (h1 *)logits, p, BH, H, T, n_super_cap, (h1 *)state_out, seg);
        return check_launch();
    }
    if (D == 128 && qk_pair(BH, seg.nseg)) {
        const long threads = padded_units<64>(BH, seg.nseg) * 64;
        ADKV_LAUNCH_(qk_kernel, 128, 2, 256, (const h1 *)q, (uint4 *)k_cache, (const h1 *)k_new, (h1 *)logits, (const h1 *)zp,
                     (const h1 *)sc, (const h1 *)alpha, (const h1 *)beta, (const h1 *)tgt, BH, H, T, n_super_cap, (h1 *)state_out, seg);
        return check_launch();
    }
    plan_shared(seg, BH, T, D);
    ADKV_DISPATCH_D(qk_kernel, (const h1 *)q, (uint4 *)k_cache, (const h1 *)k_new, (h1 *)logits,
                    (const h1 *)zp, (const h1 *)sc, (const h1 *)alpha, (const h1 *)beta,
                    (const h1 *)tgt, BH, H, T, n_super_cap, (h1 *)state_out, seg);
    return check_launch();
}

extern "C" {

const char *adkv_decode_kernel_name(int B, int Hq, int H, int T, int D, int bits, int n_ckpt_cap,
                                    int ckpt_interval)
{
    return decode_kernel_name(false, B, Hq, H, T, D, bits, n_ckpt_cap, ckpt_interval);
}

const char *adkv_decode_ov_kernel_name(int B, int Hq, int H, int T, int D, int bits, int n_ckpt_cap,
                                       int ckpt_interval)
{
    return decode_kernel_name(true, B, Hq, H, T, D, bits, n_ckpt_cap, ckpt_interval);
}

int adkv_decode_step_launches(int B, int Hq, int H, int T, int D, int bits, int n_ckpt_cap, int ckpt_interval,
                              int masked)
{
    if (adkv_decode_step_is_fused(B, Hq, H, T, D, bits, n_ckpt_cap, ckpt_interval, masked))
        return 1;
    if (adkv_decode_segments(B, Hq, H, T, D, bits, n_ckpt_cap, ckpt_interval, nullptr, 0, nullptr) < 0)
        return 3;
    int dummy = 0, cpl;
    Seg seg;
    void *ck = n_ckpt_cap > 0 && ckpt_interval > 0 ? &dummy : nullptr;
    return segment_step_plan(seg, cpl, B, Hq, H, T, D, bits, ck, ck, n_ckpt_cap, ckpt_interval) ? 2 : 3;
}

const char *adkv_decode_step_kernel_name(int B, int Hq, int H, int T, int D, int bits, int n_ckpt_cap, int ckpt_interval,
                                         int masked)
{
    int dummy = 0, cpl;
    Seg seg, vseg;
    void *ck = n_ckpt_cap > 0 && ckpt_interval > 0 ? &dummy : nullptr;
    switch (adkv_decode_step_launches(B, Hq, H, T, D, bits, n_ckpt_cap, ckpt_interval, masked)) {
    case 1:
        return !masked && fused_step_plan(seg, vseg, B, Hq, H, T, D, bits, ck, ck, n_ckpt_cap, ckpt_interval) ? "decode_ft_kernel"
                                                                                                             : "small_step_kernel";
    case 2:
        segment_step_plan(seg, cpl, B, Hq, H, T, D, bits, ck, ck, n_ckpt_cap, ckpt_interval);
        switch (step_lone_threads(padded_units<64>(B * H, seg.nseg), D, Hq / H, longest_segment(seg, T))) {
        case 0: return "step_segments_kernel";
        case 256: return "step_lone_kernel, 4-wave workgroups"; // of keys, see adkv_decode_step_values_ahead
        case 512: return "step_lone_kernel, 8-wave workgroups";
        case 768: return "step_lone_kernel, 12-wave workgroups";
        default: return "step_lone_kernel, 16-wave workgroups";
        }
    default:
        return nullptr;
    }
}

int adkv_decode_step_values_ahead(int B, int Hq, int H, int T, int D, int bits, int n_ckpt_cap, int ckpt_interval)
{
    int dummy = 0, cpl;
    Seg seg;
    void *ck = n_ckpt_cap > 0 && ckpt_interval > 0 ? &dummy : nullptr;
    if (adkv_decode_step_launches(B, Hq, H, T, D, bits, n_ckpt_cap, ckpt_interval, 0) != 2 ||
        !segment_step_plan(seg, cpl, B, Hq, H, T, D, bits, ck, ck, n_ckpt_cap, ckpt_interval))
        return 0;
    const long units = padded_units<64>(B * H, seg.nseg);
    return step_values_ahead(step_lone_threads(units, D, Hq / H, longest_segment(seg, T)), units, D);
}

int adkv_decode_segments(int B, int Hq, int H, int T, int D, int bits, int n_ckpt_cap,
                         int ckpt_interval, int *bounds, int max_bounds, int *info)
{
    if (B <= 0 || H <= 0 || Hq <= 0 || Hq % H || T < 0 || (D != 128 && D != 256 && D != 512) ||
        (bits != 2 && bits != 4))
        return -1;
    const int GQ = Hq / H;
    if ((GQ > 1 || bits != 4) && D != 128)
        return -1;
    int dummy = 0;
    Seg seg = plan_segments(n_ckpt_cap > 0 && ckpt_interval > 0 ? &dummy : nullptr, n_ckpt_cap,
                            ckpt_interval, B * H, T, D);
    const bool matrix_cores = D == 128 && (GQ > 1 || bits != 4 || mfma_for_mha());
    const bool head_table = !matrix_cores && use_head_table(B, H, GQ, bits, D, seg);
    long wgs = 0;
    int virt = 1;
    if (matrix_cores && GQ <= 4 && !gqa_pair((long)B * H, seg.nseg))
        plan_gqa(seg, B * H, T, GQA_SKEW_QK);
    if (head_table) {
        const int lanes = plan_ft(seg, B, H, T, FT_SKEW_QK, FT16_QK);
        const int W = ft_wgs_per_head(B, seg.nseg, 64 / lanes);
        wgs = (long)H * seg.phys_per_head;
        virt = (W + seg.phys_per_head - 1) / seg.phys_per_head;
    } else if (!matrix_cores && !(D == 128 && (qk_lone(B * H, seg.nseg, T) || qk_pair(B * H, seg.nseg)))) {
        plan_shared(seg, B * H, T, D);
    }
    if (bounds != nullptr && max_bounds > seg.nseg) {
        for (int s = 0; s < seg.nseg; s++)
            bounds[s] = seg.groups > 0   ? uneven_cut(s, seg.groups, seg.intervals, seg.skew) * seg.ckpt_interval
                        : seg.groups < 0 ? balanced_cut(seg, s) * seg.ckpt_interval
                                         : s * seg.seg_tokens; // in time order
        bounds[seg.nseg] = T;
    }
    if (info != nullptr) {
        info[0] = (int)wgs; // 0: not a per-head-table launch (workgroup count follows the kernel's shape)
        info[1] = virt;
    }
    return seg.nseg;
}

int adkv_forward_qk_gqa(const void *q, void *k_cache, const void *k_new, void *logits,
                        const void *zp, const void *sc, const void *alpha, const void *beta,
                        const void *tgt,
                        int B, int Hq, int H, int T, int D, int n_super_cap, int bits, int64_t ld,
                        void *state_out, void *ckpt, int n_ckpt_cap, int ckpt_interval,
                        void *stream)
{
    return forward_qk_impl(q, k_cache, k_new, logits, zp, sc, alpha, beta, tgt, B, Hq, H, T, D,
                           n_super_cap, bits, ld, state_out, ckpt, n_ckpt_cap, ckpt_interval, stream, 0);
}

int adkv_forward_qk_ex(const void *q, void *k_cache, const void *k_new, void *logits,
                       const void *zp, const void *sc, const void *alpha, const void *beta,
                       const void *tgt,
                       int B, int H, int T, int D, int n_super_cap,
                       void *state_out, void *ckpt, int n_ckpt_cap, int ckpt_interval,
                       void *stream)
{
    return adkv_forward_qk_gqa(q, k_cache, k_new, logits, zp, sc, alpha, beta, tgt, B, H, H, T, D,
                               n_super_cap, 4, 0, state_out, ckpt, n_ckpt_cap, ckpt_interval, stream);
}

int adkv_forward_qk(const void *q, void *k_cache, const void *k_new, void *logits,
                    const void *zp, const void *sc, const void *alpha, const void *beta,
                    const void *tgt,
                    int B, int H, int T, int D, int n_super_cap,
                    float, float, void *state_out, void *stream)
{
    return adkv_forward_qk_ex(q, k_cache, k_new, logits, zp, sc, alpha, beta, tgt, B, H, T, D,
                              n_super_cap, state_out, nullptr, 0, 0, stream);
}

int64_t adkv_forward_ov_workspace_bytes(int B, int H, int T, int D, int n_ckpt_cap, int ckpt_interval)
{
    if (B <= 0 || H <= 0 || T < 0 || n_ckpt_cap <= 0 || ckpt_interval <= 0)
        return 0;
    int dummy = 0;
    const int nseg = max_plan_segments(&dummy, n_ckpt_cap, ckpt_interval, B, H, T, D);
    return nseg > 1 ? (int64_t)nseg * B * H * D * 4 : 0;
}

} // extern "C"

static int forward_ov_impl(const void *attn, void *v_cache, const void *v_new, void *out,
                           const void *zp, const void *sc, const void *alpha, const void *beta,
                           const void *tgt,
                           int B, int Hq, int H, int T, int D, int n_super_cap, int bits, int64_t ld,
                           void *state_out, void *ckpt, int n_ckpt_cap, int ckpt_interval,
                           void *workspace, int64_t workspace_bytes, void *stream, int act_bf16)
{
    if (ld != 0 && ld < (int64_t)T + 1)
        return ADKV_E_SHAPE;
    if (!attn || !v_cache || !v_new || !out || !zp || !sc || !alpha || !beta || !tgt)
        return ADKV_E_NULL;
    if (bits != 2 && bits != 4)
        return ADKV_E_UNSUPPORTED;
    int rc = check_common(B, H, T, D, n_super_cap);
    if (rc)
        return rc;
    if (Hq <= 0 || Hq % H)
        return ADKV_E_SHAPE;
    const int GQ = Hq / H;
    if ((GQ > 1 || bits != 4) && D != 128)
        return ADKV_E_UNSUPPORTED;
    if (T / (32 / bits) >= n_super_cap)
        return ADKV_E_CAPACITY;
    if (((uintptr_t)v_cache & 15) || ((uintptr_t)out & 3) || ((uintptr_t)v_new & 3))
        return ADKV_E_ALIGN;
    if ((rc = check_ckpt(ckpt, n_ckpt_cap, ckpt_interval, bits)))
        return rc;
    const int BH = B * H;
    hipStream_t st = (hipStream_t)stream;
    Seg seg = plan_segments(ckpt, n_ckpt_cap, ckpt_interval, BH, T, D);
    seg.act_bf16 = act_bf16;
    if (ld)
        seg.row_pitch = ld;
    const bool matrix_cores = D == 128 && (GQ > 1 || bits != 4 || mfma_for_mha());
    const bool head_table = !matrix_cores && use_head_table(B, H, GQ, bits, D, seg);
    const int ft_lanes = head_table ? plan_ft_ov(seg, B, H, T) : 32;
    // per-head table, two or four segments, one virtual workgroup per workgroup: the waves of one
    // sequence pair sit in the same workgroup (interleave_segment) and add their partial outputs
    // there; no second launch and nothing in the workspace
    seg.combine = (head_table && ft_ov_combines(seg, B, ft_lanes)) ? 1 : 0;
    const bool pair = matrix_cores && ov_gqa_pair(BH, seg.nseg, GQ, ((uintptr_t)attn & 15) == 0 && seg.row_pitch % 8 == 0);
    const bool lone = !matrix_cores && !head_table && D == 128 && ov_lone(BH, seg.nseg, T);
    // a workspace has to hold the even plan's sums, whichever plan runs
    if (seg.nseg > 1 && !seg.combine) {
        if (!workspace || workspace_bytes < (int64_t)seg.nseg * BH * GQ * D * 4)
            return ADKV_E_WORKSPACE;
        if ((uintptr_t)workspace & 15)
            return ADKV_E_ALIGN;
    }
    if (matrix_cores ? GQ <= 4 && !pair : !head_table && !lone) {
        Seg s = seg;
        if (matrix_cores)
            plan_gqa(s, BH, T, GQA_SKEW_OV);
        else
            plan_shared(s, BH, T, D);
        if (workspace_bytes >= (int64_t)s.nseg * BH * GQ * D * 4)
            seg = s;
        else if (matrix_cores) // one that holds no more keeps the even plan's number of segments
            plan_uneven(seg, T, padded_units<32>(BH, seg.nseg) * 32, GQA_SKEW_OV);
    }
    if (matrix_cores) {
        ADKV_DISPATCH_GQ(ov_gqa_kernel, false, (const h1 *)attn, (uint4 *)v_cache, (const h1 *)v_new,
                         (h1 *)out, (float *)workspace, (const h1 *)zp, (const h1 *)sc,
                         (const h1 *)alpha, (const h1 *)beta, (const h1 *)tgt, BH, H, T, n_super_cap,
                         (h1 *)state_out, seg);
    } else if (head_table) {
        const auto kernel = ft_lanes == 16 ? ov_ft_kernel<16> : ov_ft_kernel<32>;
        hipLaunchKernelGGL(kernel, dim3((unsigned)(H * ft_wgs_per_head(B, seg.nseg, 64 / ft_lanes))),
                           dim3(FT_BLK), 0, st, (const h1 *)attn, (uint4 *)v_cache, (const h1 *)v_new, (h1 *)out,
                           (float *)workspace, (const h1 *)zp, (const h1 *)sc, (const h1 *)alpha,
                           (const h1 *)beta, (const h1 *)tgt, B, H, T, n_super_cap, (h1 *)state_out, seg);
    } else if (lone) {
        const FtParams p = {(const h1 *)zp, (const h1 *)sc, (const h1 *)alpha, (const h1 *)beta, (const h1 *)tgt};
        ADKV_LAUNCH_LONE(ov_lone_kernel, 1024, (const h1 *)attn,
                           (uint4 *)v_cache, (const h1 *)v_new, (h1 *)out, (float *)workspace, p, BH, H, T, n_super_cap,
                           (h1 *)state_out, seg);
    } else {
        ADKV_DISPATCH_D(ov_kernel, (const h1 *)attn, (uint4 *)v_cache, (const h1 *)v_new, (h1 *)out,
                        (float *)workspace, (const h1 *)zp, (const h1 *)sc, (const h1 *)alpha,
                        (const h1 *)beta, (const h1 *)tgt, BH, H, T, n_super_cap, (h1 *)state_out,
                        seg);
    }
    if ((rc = check_launch()))
        return rc;
    if (seg.nseg > 1 && !seg.combine) {
        const long n = (long)BH * GQ * D;
        if (seg.nseg > 8)
            hipLaunchKernelGGL(ov_finalize_wide_kernel, dim3((unsigned)((n + 63) / 64)), dim3(256), 0, st,
                               (const float *)workspace, (h1 *)out, n, seg.nseg, seg.act_bf16);
        else
            hipLaunchKernelGGL(ov_finalize_kernel, dim3((unsigned)((n + 511) / 512)), dim3(256), 0, st,
                               (const float *)workspace, (h1 *)out, n, seg.nseg, seg.act_bf16);
        rc = check_launch();
    }
    return rc;
}

// ---------------------------------------------------------------------------------------------
// Static scratch for callers that cannot allocate (code under HIP graph capture, serving loops,
// harnesses that forbid hipMalloc): the fp32 partial sums of a segmented forward_ov live in a
// device array that is part of the code object, one copy per GPU, held until the process ends.
// In host code the array's name is only a handle for hipGetSymbolAddress; the device address it
// yields (a different one on every GPU) is what launches are given.
// ---------------------------------------------------------------------------------------------
constexpr int64_t STATIC_SCRATCH_FLOATS = (int64_t)8 << 20; // 32 MiB
static __device__ __align__(256) float scratch[STATIC_SCRATCH_FLOATS];

constexpr int MAX_DEVICES = 64;
static std::atomic<float *> g_scratch_ptr[MAX_DEVICES];
static std::mutex g_scratch_mu;

// Device address of `scratch` on the current device, resolved once per device.
static int static_scratch(float **out)
{
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) {
        g_last_hip_error = (int)e;
        return ADKV_E_DEVICE;
    }
    if (dev < 0 || dev >= MAX_DEVICES)
        return ADKV_E_UNSUPPORTED;
    float *p = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (p == nullptr) {
        std::lock_guard<std::mutex> lock(g_scratch_mu);
        p = g_scratch_ptr[dev].load(std::memory_order_relaxed);
        if (p == nullptr) {
            void *addr = nullptr;
            e = hipGetSymbolAddress(&addr, HIP_SYMBOL(scratch));
            if (e != hipSuccess || addr == nullptr) {
                g_last_hip_error = (int)e;
                return ADKV_E_DEVICE;
            }
            p = (float *)addr;
            g_scratch_ptr[dev].store(p, std::memory_order_release);
        }
    }
    *out = p;
    return ADKV_OK;
}

extern "C" {

int64_t adkv_static_scratch_bytes(void) { return STATIC_SCRATCH_FLOATS * 4; }

int adkv_init(void)
{
    float *p = nullptr;
    return static_scratch(&p);
}

int adkv_forward_ov_noalloc(const void *attn, void *v_cache, const void *v_new, void *out,
                            const void *zp, const void *sc, const void *alpha, const void *beta,
                            const void *tgt,
                            int B, int Hq, int H, int T, int D, int n_super_cap, int bits, int64_t ld,
                            void *state_out, void *ckpt, int n_ckpt_cap, int ckpt_interval,
                            void *stream)
{
    // what the segment plan of this launch needs, priced before anything touches the device
    // (nothing when the kernel adds its two or four segments inside the workgroup)
    int64_t need = 0;
    if (ckpt != nullptr && B > 0 && H > 0 && Hq > 0 && Hq % H == 0 && T >= 0 && n_ckpt_cap > 0 &&
        ckpt_interval > 0 && (D == 128 || D == 256 || D == 512)) {
        int dummy = 0;
        Seg seg = plan_segments(&dummy, n_ckpt_cap, ckpt_interval, B * H, T, D);
        const int GQ = Hq / H;
        const bool matrix_cores = D == 128 && (GQ > 1 || bits != 4 || mfma_for_mha());
        bool in_workgroup = false;
        if (!matrix_cores && use_head_table(B, H, GQ, bits, D, seg)) {
            const int lanes = plan_ft_ov(seg, B, H, T);
            in_workgroup = ft_ov_combines(seg, B, lanes);
        }
        if (seg.nseg > 1 && !in_workgroup)
            need = (int64_t)seg.nseg * B * Hq * D * 4;
    }
    if (need > adkv_static_scratch_bytes())
        return ADKV_E_SCRATCH_LIMIT;
    float *ws = nullptr;
    const int rc = static_scratch(&ws);
    if (rc)
        return rc;
    // Every partial a launch reads was written by the same launch (each segment stores its whole
    // [B*Hq, D] slice before the summing kernel runs), so nothing has to start at zero.
    return forward_ov_impl(attn, v_cache, v_new, out, zp, sc, alpha, beta, tgt, B, Hq, H, T, D,
                           n_super_cap, bits, ld, state_out, ckpt, n_ckpt_cap, ckpt_interval, ws,
                           adkv_static_scratch_bytes(), stream, 0);
}

int adkv_forward_ov_gqa(const void *attn, void *v_cache, const void *v_new, void *out,
                        const void *zp, const void *sc, const void *alpha, const void *beta,
                        const void *tgt,
                        int B, int Hq, int H, int T, int D, int n_super_cap, int bits, int64_t ld,
                        void *state_out, void *ckpt, int n_ckpt_cap, int ckpt_interval,
                        void *workspace, int64_t workspace_bytes, void *stream)
{
    return forward_ov_impl(attn, v_cache, v_new, out, zp, sc, alpha, beta, tgt, B, Hq, H, T, D,
                           n_super_cap, bits, ld, state_out, ckpt, n_ckpt_cap, ckpt_interval, workspace,
                           workspace_bytes, stream, 0);
}

int adkv_forward_ov_ex(const void *attn, void *v_cache, const void *v_new, void *out,
                       const void *zp, const void *sc, const void *alpha, const void *beta,
                       const void *tgt,
                       int B, int H, int T, int D, int n_super_cap,
                       void *state_out, void *ckpt, int n_ckpt_cap, int ckpt_interval,
                       void *workspace, int64_t workspace_bytes, void *stream)
{
    return adkv_forward_ov_gqa(attn, v_cache, v_new, out, zp, sc, alpha, beta, tgt, B, H, H, T, D,
                               n_super_cap, 4, 0, state_out, ckpt, n_ckpt_cap, ckpt_interval, workspace,
                               workspace_bytes, stream);
}

int adkv_forward_ov(const void *attn, void *v_cache, const void *v_new, void *out,
                    const void *zp, const void *sc, const void *alpha, const void *beta,
                    const void *tgt,
                    int B, int H, int T, int D, int n_super_cap,
                    float, float, void *state_out, void *stream)
{
    return adkv_forward_ov_ex(attn, v_cache, v_new, out, zp, sc, alpha, beta, tgt, B, H, T, D,
                              n_super_cap, state_out, nullptr, 0, 0, nullptr, 0, stream);
}

int64_t adkv_softmax_workspace_bytes(int rows, int n)
{
    if (rows <= 0 || n <= SM_ROW_MAX)
        return 0;
    return (int64_t)rows * ((n + SM_CHUNK - 1) / SM_CHUNK) * 8;
}

int64_t adkv_row_pitch(int n)
{
    // smallest odd multiple of 128 elements (256 bytes) that holds n: consecutive rows then start
    // in different memory channels even when n itself is a power of two
    int64_t k = ((int64_t)n + 127) / 128;
    if (!(k & 1))
        k++;
    return k * 128;
}

int adkv_softmax_ex(const void *logits, void *weights, const void *mask,
                    int rows, int n, int64_t ld, int rows_per_mask_row, float scaling,
                    void *workspace, int64_t workspace_bytes, void *stream)
{
    return softmax_launch<false>(logits, weights, {mask, rows_per_mask_row, ADKV_DT_F32}, rows, n, ld, scaling, workspace,
                          workspace_bytes, stream);
}

int adkv_softmax(const void *logits, void *weights, const void *mask,
                 int rows, int n, int rows_per_mask_row, float scaling, void *stream)
{
    return adkv_softmax_ex(logits, weights, mask, rows, n, 0, rows_per_mask_row, scaling, nullptr, 0,
                           stream);
}

static int64_t pad256(int64_t n) { return (n + 255) & ~(int64_t)255; }

// Events adkv_decode_step records around its stages in this thread (a measurement hook: what runs does
// not depend on it).
static thread_local hipEvent_t g_stage_events[4] = {nullptr, nullptr, nullptr, nullptr};

void adkv_set_stage_events(void *const *events)
{
    for (int i = 0; i < 4; i++)
        g_stage_events[i] = events ? (hipEvent_t)events[i] : nullptr;
}

static int stage_mark(int i, void *stream)
{
    if (g_stage_events[i] == nullptr)
        return ADKV_OK;
    const hipError_t e = hipEventRecord(g_stage_events[i], (hipStream_t)stream);
    if (e != hipSuccess) {
        g_last_hip_error = (int)e;
        return ADKV_E_LAUNCH;
    }
    return ADKV_OK;
}

// after a launch that is all three stages
static int mark_one_launch(void *stream)
{
    int rc = ADKV_OK;
    for (int i = 1; i <= 3 && !rc; i++)
        rc = stage_mark(i, stream);
    return rc;
}

int64_t adkv_forward_ov_gqa_workspace_bytes(int B, int Hq, int H, int T, int D, int n_ckpt_cap,
                                            int ckpt_interval)
{
    if (H <= 0 || Hq <= 0 || Hq % H)
        return 0;
    return adkv_forward_ov_workspace_bytes(B, H, T, D, n_ckpt_cap, ckpt_interval) * (Hq / H);
}

int64_t adkv_decode_step_workspace_bytes(int B, int Hq, int H, int T, int D, int n_ckpt_cap,
                                          int ckpt_interval)
{
    if (B <= 0 || H <= 0 || Hq <= 0 || T < 0)
        return 0;
    const int64_t mat = pad256((int64_t)B * Hq * adkv_row_pitch(T + 1) * 2);
    const int64_t ov = adkv_forward_ov_gqa_workspace_bytes(B, Hq, H, T, D, n_ckpt_cap, ckpt_interval);
    // a step in two launches leaves a maximum, two sums and D partial outputs per row and segment
    int dummy = 0;
    const int64_t nseg = H > 0 ? plan_segments(n_ckpt_cap > 0 && ckpt_interval > 0 ? &dummy : nullptr, n_ckpt_cap, ckpt_interval,
                                               B * H, T, D).nseg : 1;
    const int64_t step = pad256(nseg * B * Hq * 16) + nseg * B * Hq * D * 4;
    return 2 * mat + std::max(pad256(adkv_softmax_workspace_bytes(B * Hq, T + 1)) + ov, step);
}

static FtParams ft_params(const void *const *p)
{
    return {(const h1 *)p[0], (const h1 *)p[1], (const h1 *)p[2], (const h1 *)p[3], (const h1 *)p[4]};
}

// What forward_qk and forward_ov would refuse, for the steps that run otherwise.
static int check_step(const void *q, const void *k_cache, const void *v_cache, const void *k_new, const void *v_new,
                      const void *const *k_params, const void *const *v_params, const void *out, const void *weights, int B,
                      int Hq, int H, int T, int D, int n_super_cap, int bits, const void *k_ckpt, const void *v_ckpt,
                      int n_ckpt_cap, int ckpt_interval)
{
    int rc = check_common(B, H, T, D, n_super_cap);
    if (rc)
        return rc;
    if ((Hq > H || bits != 4) && D != 128)
        return ADKV_E_UNSUPPORTED;
    if (T / (32 / bits) >= n_super_cap)
        return ADKV_E_CAPACITY;
    if (!q || !k_cache || !v_cache || !k_new || !v_new || !out)
        return ADKV_E_NULL;
    for (int i = 0; i < 5; i++)
        if (!k_params[i] || !v_params[i])
            return ADKV_E_NULL;
    if (((uintptr_t)k_cache & 15) || ((uintptr_t)v_cache & 15) || ((uintptr_t)q & 7) || ((uintptr_t)k_new & 3) ||
        ((uintptr_t)v_new & 3) || ((uintptr_t)out & 3) || ((uintptr_t)weights & 1))
        return ADKV_E_ALIGN;
    if ((rc = check_ckpt(k_ckpt, n_ckpt_cap, ckpt_interval, bits)))
        return rc;
    return check_ckpt(v_ckpt, n_ckpt_cap, ckpt_interval, bits);
}

int adkv_decode_step(const void *q, void *k_cache, void *v_cache, const void *k_new, const void *v_new,
                      const void *const *k_params, const void *const *v_params,
                      const void *mask, int rows_per_mask_row, float scaling,
                      void *out, void *weights_out, int64_t weights_ld,
                      int B, int Hq, int H, int T, int D, int n_super_cap, int bits, int act_dtype,
                      void *k_ckpt, void *v_ckpt, int n_ckpt_cap, int ckpt_interval,
                      void *workspace, int64_t workspace_bytes, void *stream)
{
    if (!k_params || !v_params || !workspace)
        return workspace ? ADKV_E_NULL : ADKV_E_WORKSPACE;
    const int mask_dtype = act_dtype >> 8;
    act_dtype &= 255;
    if ((act_dtype != ADKV_DT_F16 && act_dtype != ADKV_DT_BF16) ||
        (mask_dtype != ADKV_DT_F32 && mask_dtype != ADKV_DT_F16 && mask_dtype != ADKV_DT_BF16))
        return ADKV_E_UNSUPPORTED;
    const int act_bf16 = act_dtype == ADKV_DT_BF16;
    const Mask mk = {mask, rows_per_mask_row, mask_dtype};
    if (B <= 0 || H <= 0 || Hq <= 0 || Hq % H || T < 0)
        return ADKV_E_SHAPE;
    if (workspace_bytes < adkv_decode_step_workspace_bytes(B, Hq, H, T, D, n_ckpt_cap, ckpt_interval))
        return ADKV_E_WORKSPACE;
    if ((uintptr_t)workspace & 255)
        return ADKV_E_ALIGN;
    // The logits live in the workspace with padded rows.  The weights do too unless the caller
    // wants them; the softmax writes them with the logits' pitch, so a caller-provided matrix
    // must use that pitch as well (weights_ld == adkv_row_pitch(T + 1)) or be avoided.
    const int64_t ld = adkv_row_pitch(T + 1);
    if (weights_out && weights_ld != ld)
        return ADKV_E_SHAPE;
    const int64_t mat = pad256((int64_t)B * Hq * ld * 2);
    char *ws = (char *)workspace;
    void *logits = ws;
    void *weights = weights_out ? weights_out : (void *)(ws + mat);
    int rc = stage_mark(0, stream);
    if (rc)
        return rc;
    {
        // one launch for the whole step where the plans allow it (decode_ft_kernel)
        Seg ka, va;
        const int lanes = mask ? 0 : fused_step_plan(ka, va, B, Hq, H, T, D, bits, k_ckpt, v_ckpt, n_ckpt_cap, ckpt_interval);
        if (lanes) {
            if ((rc = check_step(q, k_cache, v_cache, k_new, v_new, k_params, v_params, out, weights, B, Hq, H, T, D, n_super_cap,
                                 bits, k_ckpt, v_ckpt, n_ckpt_cap, ckpt_interval)))
                return rc;
            ka.row_pitch = va.row_pitch = ld;
            ka.act_bf16 = va.act_bf16 = act_bf16;
            va.combine = 1;
            const FtParams kp = ft_params(k_params), vp = ft_params(v_params);
            const auto kernel = lanes == 16 ? decode_ft_kernel<16> : decode_ft_kernel<32>;
            hipLaunchKernelGGL(kernel, dim3((unsigned)(H * ka.phys_per_head)), dim3(FT_BLK), 0, (hipStream_t)stream,
                               (const h1 *)q, (uint4 *)k_cache, (const h1 *)k_new, (uint4 *)v_cache, (const h1 *)v_new,
                               (h1 *)logits, (h1 *)weights, (h1 *)out, kp, vp, B, H, T, n_super_cap, scaling, ka, va);
            return (rc = check_launch()) ? rc : mark_one_launch(stream);
        }
    }
    {
        Seg ka;
        if (small_step_plan(ka, B, Hq, H, T, D, bits, k_ckpt, v_ckpt, n_ckpt_cap, ckpt_interval)) {
            if ((rc = check_step(q, k_cache, v_cache, k_new, v_new, k_params, v_params, out, weights, B, Hq, H, T, D, n_super_cap,
                                 bits, k_ckpt, v_ckpt, n_ckpt_cap, ckpt_interval)))
                return rc;
            if (mask && rows_per_mask_row <= 0)
                return ADKV_E_SHAPE;
            ka.row_pitch = ld;
            ka.act_bf16 = act_bf16;
            Seg va = ka;
            va.ckpt = (h1 *)v_ckpt;
            const FtParams kp = ft_params(k_params), vp = ft_params(v_params);
            const auto kernel = ka.nseg == 1 ? small_step_kernel<1> : ka.nseg == 2 ? small_step_kernel<2>
                              : ka.nseg == 3 ? small_step_kernel<3> : small_step_kernel<4>;
            hipLaunchKernelGGL(kernel, dim3((unsigned)(B * H)), dim3((unsigned)ka.nseg * 256), 0, (hipStream_t)stream, (const h1 *)q,
                               (uint4 *)k_cache, (const h1 *)k_new, (uint4 *)v_cache, (const h1 *)v_new, mk, (h1 *)weights,
                               (h1 *)out, kp, vp, H, T, n_super_cap, scaling, ka, va);
            return (rc = check_launch()) ? rc : mark_one_launch(stream);
        }
    }
    {
        Seg ka;
        int cpl;
        if (segment_step_plan(ka, cpl, B, Hq, H, T, D, bits, k_ckpt, v_ckpt, n_ckpt_cap, ckpt_interval)) {
            if ((rc = check_step(q, k_cache, v_cache, k_new, v_new, k_params, v_params, out, weights, B, Hq, H, T, D, n_super_cap,
                                 bits, k_ckpt, v_ckpt, n_ckpt_cap, ckpt_interval)))
                return rc;
            if (mask && rows_per_mask_row <= 0)
                return ADKV_E_SHAPE;
            ka.row_pitch = ld;
            ka.act_bf16 = act_bf16;
            Seg va = ka;
            va.ckpt = (h1 *)v_ckpt;
            const long rows = (long)B * Hq;
            float4 *ml = (float4 *)(ws + 2 * mat);
            float *partial = (float *)(ws + 2 * mat + pad256(ka.nseg * rows * 16));
            if ((rc = launch_step_segments(cpl, Hq / H, bits, D, B * H, ka.nseg, longest_segment(ka, T), (hipStream_t)stream,
                                           (const h1 *)q, (uint4 *)k_cache, (const h1 *)k_new, (uint4 *)v_cache, (const h1 *)v_new,
                                           mk, (h1 *)logits, partial, ml, ft_params(k_params), ft_params(v_params), B * H, H, T,
                                           n_super_cap, scaling, ka, va)))
                return rc;
            for (int i = 1; i <= 2; i++)
                if ((rc = stage_mark(i, stream)))
                    return rc;
            const int out_waves = ka.nseg > 16 ? D / 16 : D / 128;
            // two vectors of weights per lane where one would give more waves than the device holds at once
            const int vecs = rows * ((T + 1 + 511) / 512 + out_waves) > 32L * cus() ? 2 : 1;
            const long waves = rows * ((T + 1 + 512 * vecs - 1) / (512 * vecs) + out_waves);
            const auto combine = vecs == 2 ? step_combine_kernel<2> : step_combine_kernel<1>;
            hipLaunchKernelGGL(combine, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, (hipStream_t)stream,
                               (const h1 *)logits, (h1 *)weights, (h1 *)out, mk, partial, ml, rows, T + 1, (long)ld, D, ka.nseg,
                               scaling, out_waves, act_bf16);
            return (rc = check_launch()) ? rc : stage_mark(3, stream);
        }
    }
    rc = forward_qk_impl(q, k_cache, k_new, logits, k_params[0], k_params[1], k_params[2],
                         k_params[3], k_params[4], B, Hq, H, T, D, n_super_cap, bits, ld,
                         nullptr, k_ckpt, n_ckpt_cap, ckpt_interval, stream, act_bf16);
    if (rc || (rc = stage_mark(1, stream)))
        return rc;
    const int64_t smb = pad256(adkv_softmax_workspace_bytes(B * Hq, T + 1));
    rc = (mask && mask_dtype != ADKV_DT_F32 ? softmax_launch<true> : softmax_launch<false>)(
        logits, weights, mk, B * Hq, T + 1, ld, scaling, smb ? ws + 2 * mat : nullptr, smb, stream);
    if (rc || (rc = stage_mark(2, stream)))
        return rc;
    rc = forward_ov_impl(weights, v_cache, v_new, out, v_params[0], v_params[1], v_params[2],
                         v_params[3], v_params[4], B, Hq, H, T, D, n_super_cap, bits, ld,
                         nullptr, v_ckpt, n_ckpt_cap, ckpt_interval, ws + 2 * mat + smb,
                         workspace_bytes - 2 * mat - smb, stream, act_bf16);
    if (rc)
        return rc;
    return stage_mark(3, stream);
}

} // extern "C"
