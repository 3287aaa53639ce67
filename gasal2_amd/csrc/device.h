// device.h -- device helpers shared by the kernels' translation units: packed
// bases, substitution scores and their tables, packed 16-bit arithmetic.
#ifndef GASAL2_DEVICE_H
#define GASAL2_DEVICE_H

#include "engine.h"

namespace {

constexpr int32_t MINUS_INF = -32768;   // SHRT_MIN, src/gasal_kernels.h:35
constexpr int WAVE = 64;

enum { A_GLOBAL = 1, A_SEMI_GLOBAL = 2, A_LOCAL = 3, A_BANDED = 5, A_KSW = 6 };
enum { S_WITHOUT_START = 0, S_WITH_START = 1, S_WITH_TB = 2 };
enum { D_NONE = 0, D_QUERY = 1, D_TARGET = 2, D_BOTH = 3 };

__device__ __forceinline__ int32_t sx16(uint32_t v) { return (int32_t)(int16_t)(uint16_t)(v & 0xFFFFu); }
// (h & 0xFFFF) | (e << 16): one byte select (bytes 0-1 of h, then bytes 0-1 of e)
__device__ __forceinline__ uint32_t pk16(int32_t h, int32_t e) {
    return __builtin_amdgcn_perm((uint32_t)e, (uint32_t)h, 0x05040100u);
}
__device__ __forceinline__ int32_t t16(int32_t v) { return (int32_t)(int16_t)(uint16_t)((uint32_t)v & 0xFFFFu); }
__device__ __forceinline__ int32_t dregs(uint32_t len) { return (int32_t)((len >> 3) + ((len & 7) ? 1 : 0)); }

// DEV_GET_SUB_SCORE_LOCAL (src/gasal_kernels.h:40-42, :49-51)
__device__ __forceinline__ int32_t sub_local(const G2Scores &c, int32_t nval, uint32_t r, uint32_t g) {
    int32_t s = (r == g) ? c.match : -c.mismatch;
    return (r == c.n_value || g == c.n_value) ? nval : s;
}
// DEV_GET_SUB_SCORE_GLOBAL (src/gasal_kernels.h:44-46, :53-54)
__device__ __forceinline__ int32_t sub_global(const G2Scores &c, uint32_t r, uint32_t g) {
    int32_t s = (r == g) ? c.match : -c.mismatch;
    return (c.has_np && (r == c.n_value || g == c.n_value)) ? -c.np : s;
}

__device__ __forceinline__ uint32_t nib_reverse(uint32_t x) {
    x = ((x & 0x0F0F0F0Fu) << 4) | ((x >> 4) & 0x0F0F0F0Fu);
    return __builtin_bswap32(x);
}
__device__ __forceinline__ bool census_fast(uint32_t m) { return ((m & (m >> 8)) & 0xFFu) == 0u; }

// GLOBAL_SEM: DEV_GET_SUB_SCORE_GLOBAL (N is an ordinary base unless N_PENALTY).
template <bool GLOBAL_SEM = false>
__device__ __forceinline__ uint32_t score_lut(const G2Scores &c, int32_t nval, uint32_t census, uint32_t tnib) {
    uint32_t lut = 0;
#pragma unroll
    for (uint32_t cls = 0; cls < 8; cls++) {
        const uint32_t q = ((census >> cls) & 1u) ? cls : cls + 8u;   // the nibble this class stands for
        int32_t s = GLOBAL_SEM ? sub_global(c, q, tnib) : sub_local(c, nval, q, tnib);
        lut |= ((uint32_t)s & 15u) << (4 * cls);
    }
    return lut;
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef short pk16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ pk16x2 as_pk(uint32_t u) { return __builtin_bit_cast(pk16x2, u); }
__device__ __forceinline__ uint32_t as_u32(pk16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ pk16x2 pmax(pk16x2 a, pk16x2 b) { return __builtin_elementwise_max(a, b); }
// a - b per half, clamped at 0 (unsigned saturation; a, b >= 0)
__device__ __forceinline__ pk16x2 psubsat(pk16x2 a, pk16x2 b) {
    typedef unsigned short pu16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(pk16x2, __builtin_elementwise_sub_sat(__builtin_bit_cast(pu16x2, a),
                                                                    __builtin_bit_cast(pu16x2, b)));
}
// {lo16(lo), lo16(hi)} and {hi16(lo), hi16(hi)}
__device__ __forceinline__ uint32_t pack_lo(uint32_t lo, uint32_t hi) { return __builtin_amdgcn_perm(hi, lo, 0x05040100u); }
__device__ __forceinline__ uint32_t pack_hi(uint32_t lo, uint32_t hi) { return __builtin_amdgcn_perm(hi, lo, 0x07060302u); }

// h * 8 + r per half in one packed multiply-add (h >= 0, r < 8 in both halves
// of r2): left to itself the compiler turns the product into a shift and an or
__device__ __forceinline__ pk16x2 prank(pk16x2 h, uint32_t r2) {
    uint32_t v;
    asm("v_pk_mad_u16 %0, %1, 8, %2 op_sel_hi:[1,0,1]" : "=v"(v) : "v"(as_u32(h)), "s"(r2));
    return as_pk(v);
}

// Stands for MINUS_INF in packed 16-bit halves: it never wins a maximum against
// a real value of the pairs those kernels take.
constexpr int32_t NEG16 = -30000;

// Reversed copy word k of a sequence
// (src/kernels/semiglobal_kernel_template.h:244-266): base 8k+b at bits 28-4b is the
// original base len-1-(8k+b); positions past the start are nibble 0.
// It is the nibble-reversed 8-base window of the forward sequence that starts
// at base len-8(k+1): one funnel shift of two forward words, then a nibble
// reverse.
__device__ __forceinline__ uint32_t rev_word(const uint32_t *W, int32_t len, int32_t k) {
    const int32_t st = len - 8 * (k + 1);
    uint32_t win;
    if (st >= 0) {
        const int32_t w0 = st >> 3, off = st & 7;
        win = off == 0 ? W[w0] : __builtin_amdgcn_alignbit(W[w0], W[w0 + 1], 32 - 4 * off);
    } else {
        win = W[0] >> (4 * (-st));   // bases before the start are nibble 0
    }
    return nib_reverse(win);
}

}  // namespace

#endif
