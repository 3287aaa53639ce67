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

// the previous lane's v within the group; the group's first lane: first
template <int GW>
__device__ __forceinline__ uint32_t from_above(uint32_t first, uint32_t v) {
    static_assert(GW == 4 || GW == 16 || GW == 32 || GW == 64, "lanes of a group");
    const uint32_t w = (uint32_t)__builtin_amdgcn_update_dpp((int)first, (int)v, GW >= 32 ? 0x138 : 0x111, 0xF, 0xF, false);
    return (GW == 4 || GW == 32) && (threadIdx.x & (GW - 1u)) == 0 ? first : w;
}
// maximum over the wave of a value that is uniform within groups of GW lanes
template <int GW = 16>
__device__ __forceinline__ int32_t wave_max(int32_t v) {
#pragma unroll
    for (int off = GW; off < WAVE; off <<= 1) v = max(v, __shfl_xor(v, off));
    return __builtin_amdgcn_readfirstlane(v);
}
__device__ __forceinline__ pk16x2 pmaxu(pk16x2 a, pk16x2 b) {
    typedef unsigned short pu16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(pk16x2, __builtin_elementwise_max(__builtin_bit_cast(pu16x2, a), __builtin_bit_cast(pu16x2, b)));
}
// 0xFFFF in each half that is not 0 (written out: the compiler makes compares
// and selects per half of it)
__device__ __forceinline__ uint32_t nonzero_mask(pk16x2 v) {
    uint32_t one, m;
    asm("v_pk_min_u16 %0, %1, 1 op_sel_hi:[1,0]" : "=v"(one) : "v"(as_u32(v)));
    asm("v_pk_sub_i16 %0, 0, %1" : "=v"(m) : "v"(one));
    return m;
}
__device__ __forceinline__ uint32_t bits_of(uint32_t mask, uint32_t a, uint32_t b) { return (a & mask) | (b & ~mask); }
__device__ __forceinline__ pk16x2 set_lo(pk16x2 v, int32_t x) { return as_pk(bits_of(0xFFFFu, (uint32_t)x, as_u32(v))); }
__device__ __forceinline__ pk16x2 set_hi(pk16x2 v, int32_t x) { return as_pk(pack_lo(as_u32(v), (uint32_t)x)); }

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

// Recomputes one 8x8 tile's direction words from the checkpoints that the
// lane kernels (k_local_fast<.., CK>, k_local_pk2) or the packed one-wave path
// stored: the previous strip's bottom row above the tile and the tile's left
// column state.  Same recurrences and score tables (lut: the strip's eight rows).
// top: the row above, entry kk = (H at column kk - 1, E at column kk), so the
// entry left of the tile's first column (the corner) comes with it; zero above
// strip 0.  left: the left column state; lut: the strip's score tables (the
// kernels store checkpoints only when the batch's nibble census allows tables).
// The words hold the reference's nibbles (src/kernels/local_kernel_template.h
// :45-60): [3] F continues (t <= f - extend), [2] E continues, [1:0] source:
// diagonal 0 / 1 by the score's sign, F 3, E 2, ties in that order.
template <bool LOCALT>
__device__ __forceinline__ void ck_tile(const uint32_t *top, const uint32_t *left, uint32_t qword,
                                        const uint32_t *lut, const G2Scores &c, uint32_t *ch) {
    int32_t h[9], f[9];
#pragma unroll
    for (int m = 1; m < 9; m++) { h[m] = sx16(left[m - 1]); f[m] = (int32_t)left[m - 1] >> 16; }
    const int32_t gapoe = c.gapoe, gape = c.gape;
#pragma unroll
    for (int kk = 0; kk < 8; kk++) {
        const uint32_t qsh = kk < 7 ? (qword >> (26 - 4 * kk)) & 0x1Cu : (qword << 2) & 0x1Cu;
        int32_t e = (int32_t)top[kk] >> 16;
        int32_t p = sx16(top[kk]);
        uint32_t dir = 0;
#pragma unroll
        for (int m = 1; m < 9; m++) {
            const int32_t sc = __builtin_amdgcn_sbfe(lut[m - 1], qsh, 4);
            const int32_t tmp = p + sc;
            const int32_t hm = LOCALT ? max(max(max(tmp, f[m]), e), 0) : max(max(tmp, f[m]), e);
            const int32_t t = tmp - gapoe;
            const int32_t fx = f[m] - gape, ex = e - gape;
            const uint32_t na = (uint32_t)(tmp - hm);                       // sign: not from the diagonal
            dir = __builtin_amdgcn_alignbit(dir, (uint32_t)t + ~(uint32_t)fx, 31);   // sign: fx >= t
            dir = __builtin_amdgcn_alignbit(dir, (uint32_t)t + ~(uint32_t)ex, 31);   // sign: ex >= t
            dir = __builtin_amdgcn_alignbit(dir, na, 31);
            // low bit: from F (hm <= f) when not diagonal, else the mismatch flag (score < 0)
            dir = __builtin_amdgcn_alignbit(dir, (na & ((uint32_t)hm + ~(uint32_t)f[m])) | (~na & (uint32_t)sc), 31);
            f[m] = max(t, fx);
            e = max(t, ex);
            p = h[m];
            h[m] = hm;
        }
        ch[kk] = dir;
    }
}

// Checkpoints of the one-wave traceback path (wavetb.hip).  A wave's region
// is a log of its iterations: 8 KiB each, four streams of one 32-byte record a
// lane -- left column state of the low and the high strip, bottom row of the
// low and the high strip -- so that every store of a wave covers whole lines.
// at: the pair's first iteration, first lane | log2(lanes of its group) << 8; for
// a pair on a block's four waves 8 there, | its passes << 12 (dealt to the waves in
// turn; the waves' regions follow each other).
constexpr uint32_t WV_STREAM = WAVE * 8, WV_ITER = 4 * WV_STREAM;   // dwords
enum { WV_LEFT = 0, WV_BOTTOM = 2 };
// Iterations from a wave's pass to its next one: its words, or the lag of the
// lanes.  On four waves (gw 256) each wave runs 65 iterations behind the one
// above, and the first wave's next pass waits for the last wave: with a shorter
// period it would wait before its own lanes have fed the waves between.
constexpr int32_t WV_COOP_PERIOD = 4 * 65;
__device__ __forceinline__ int32_t wv_period(int32_t QW, int32_t gw) { return max(QW, gw == 256 ? WV_COOP_PERIOD : gw + 1); }
// first iteration of wave w's region among those of a pair on four waves
__device__ __forceinline__ uint32_t wv_region(uint32_t passes, int32_t P, uint32_t w) {
    return w * WAVE + (uint32_t)P * (w * (passes >> 2) + min(w, passes & 3u));
}
__device__ __forceinline__ uint32_t *wv_tile(const G2Dev &d, uint2 at, int32_t QW, int32_t strip, int32_t word, int32_t what) {
    const bool coop = (at.y >> 8 & 15u) == 8u;
    const int32_t lg = coop ? 6 : (int32_t)(at.y >> 8 & 15u), gw = 1 << lg, u = strip >> 1, l = u & (gw - 1);
    const int32_t pass = u >> lg, own = coop ? pass >> 2 : pass;
    const int32_t P = wv_period(QW, coop ? 256 : gw);
    const uint32_t it = at.x + (uint32_t)(own * P + word + l) + (coop ? wv_region(at.y >> 12, P, (uint32_t)(pass & 3)) : 0u);
    return d.tb + (size_t)it * WV_ITER + (uint32_t)(what + (strip & 1)) * WV_STREAM + ((at.y & 255u) + (uint32_t)l) * 8u;
}

}  // namespace

#endif
