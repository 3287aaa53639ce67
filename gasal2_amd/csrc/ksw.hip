// ksw.hip -- KSW extension (gasal_ksw_kernel, src/kernels/ksw_kernel_template.h:46-199)
// in packed 16-bit strips.
//
// The reference keeps one row (H, E) per pair and narrows the columns of the
// next row to [first nonzero entry, last nonzero entry + 2).  Row by row that
// is a memory round trip per eight cells and lanes whose ranges differ (k_ksw:
// VALU issue 34%, 26 ms for 500,000 pairs of 100-250 bases).  Here a lane takes
// sixteen rows at a time over all their columns, two 8-row strips in the
// halves of its registers as in lane_local_pk, so the row goes through memory
// once per sixteen rows, and strips are narrowed by words, for the wave.
//
// Why the narrowed rows' values come out.  A cell left of a row's first
// nonzero entry is 0 in the full recurrence too (dead diagonals stay dead, the
// left boundary only falls).  To the right, E(i + 1, j) > 0 needs H(i, j) > 0, so
// with L the last column of row i whose H is not 0, row i + 1 ends before
// column L + 3; the full recurrence differs only if H(i + 1, j) > 0 for a
// j >= L + 3, and then first where H(i, j - 2..j) are all 0 (an F chain that
// outruns the row above by three columns).  That test is made at every cell.
// A row whose maximum is 0 ends the reference's 8-row tile; it changes
// nothing once the left boundary is 0 as well, and is tested for while it is
// not.  A pair that meets either goes on a list that k_ksw runs from the start
// (none of 5,000 simulated pairs of the seed workload; with unrelated sequences
// 0.2% by the first and 21% by the second, all of them short-lived).
//
// The score at the query's end counts only rows whose range reaches it, whose H
// there is 0 otherwise; where the query is whole words the reference also
// takes the last H of rows that end earlier, an F value, at most the maximum
// less one gap open: with an end bonus no larger than that it never decides.
//
// Bound: packed VALU, 19 instructions per row pair and column (the dead diagonals
// take two, the test four, the rank two), at 228 VGPRs and two waves per SIMD
// (held to 168 for three, with 156 bytes spilled, the same 5.4 ms).  DP of 500,000
// pairs of 100-250 bases: 26.5 -> 4.5 ms, 1,000 pairs 3.7 -> 1.2; 200,000
// unrelated pairs, a fifth of them run again by k_ksw, 2.4 -> 1.1 ms.
#include "device.h"

#include <type_traits>

namespace {

typedef unsigned short pu16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ pk16x2 pmin(pk16x2 a, pk16x2 b) { return __builtin_elementwise_min(a, b); }
// 1 in each half that is not 0
__device__ __forceinline__ pk16x2 nonzero_one(pk16x2 v) {
    uint32_t r;
    asm("v_pk_min_u16 %0, %1, 1 op_sel_hi:[1,0]" : "=v"(r) : "v"(as_u32(v)));
    return as_pk(r);
}
__device__ __forceinline__ pk16x2 times8(pk16x2 v) {
    uint32_t r;
    asm("v_pk_lshlrev_b16 %0, 3, %1 op_sel_hi:[0,1]" : "=v"(r) : "v"(as_u32(v)));
    return as_pk(r);
}
__device__ __forceinline__ uint32_t or3(uint32_t a, uint32_t b, uint32_t c) { return a | b | c; }

// One lane per pair, strips 2k and 2k + 1 in the low and high halves, the high
// one a column behind.
__global__ __launch_bounds__(64) void k_ksw_pk(G2Dev d, G2Scores c, int32_t end_bonus) {
    const uint32_t census = d.aux[0];
    if (!census_fast(census)) return;   // k_ksw takes this batch
    __shared__ uint32_t lut16[16];      // score tables of the 16 target nibbles
    if (threadIdx.x < 16) lut16[threadIdx.x] = score_lut(c, c.has_np ? -c.np : 0, census, threadIdx.x);
    __syncthreads();
    const uint32_t lane = threadIdx.x, grp = blockIdx.x, slot = grp * WAVE + lane;
    const bool ok = slot < d.n;
    const uint32_t pr = d.perm[ok ? slot : d.n - 1];
    const int32_t qlen = ok ? (int32_t)d.qlen[pr] : 0, tlen = ok ? (int32_t)d.tlen[pr] : 0;
    const int32_t QW = dregs((uint32_t)qlen), TW = dregs((uint32_t)tlen);
    const uint32_t *Qp = d.pq + (d.qoff[pr] >> 3), *Tp = d.pt + (d.toff[pr] >> 3);
    // a word in eight columns of sixteen rows: transposed panels gain nothing
    // (200,000 pairs 2.37 ms with them, 2.34 without) and take a row of the
    // longest target's words for every pair
    const int32_t q_last = max(QW - 1, 0), t_last = max(TW - 1, 0);   // words the pair holds
    uint32_t *__restrict__ bd = d.bnd + (size_t)grp * d.bnd_cols * WAVE + lane;
    const int32_t h0 = ok ? (int32_t)d.seeds[pr] : 0;
    const int32_t gapo = c.gapo, gape = c.gape, gapoe = c.gapoe;
    const pk16x2 gapoe2 = {(short)gapoe, (short)gapoe}, gape2 = {(short)gape, (short)gape};
    const pk16x2 zero2 = {0, 0};
    auto left = [&](int32_t R) -> int32_t { return max(h0 - (gapo + gape * (R + 1)), 0); };   // H(R, -1), :103-109

    int32_t bv = h0, bi = -1, bj = -1;      // the reference's max, max_i, max_j
    int32_t gs = -1, gi = -1;               // gscore, max_ie
    uint32_t redo = 0;                      // the pair needs the row by row kernel
    const int32_t TWm = wave_max<1>(TW);
    // The wave's words.  Of the first sixteen rows only those that a path can
    // reach: a cell (i, j) lies j - i insertions and more to the right, so H(i, j) <=
    // h0 + best * (i + 1) - open - extend * (j - i), best the best score of a
    // cell; the row above the later ones is 0 from there on.  1000 pairs of 600 x
    // 800 bases, unrelated, with all words 768 us, so 580, row by row 630.
    int32_t ws = 0, we = wave_max<1>(QW);
    {
        const int32_t best = max(max(c.match, -c.mismatch), max(c.has_np ? -c.np : 0, 0));
        const int32_t reach = gape > 0 ? (15 + max(wave_max<1>(h0) + 16 * best - gapo, 0) / gape) / 8 + 2 : we;
        for (int32_t cc = 8 * reach; cc < 8 * we; cc++) bd[(size_t)cc * WAVE] = 0u;
        we = min(we, reach);
    }
    asm volatile("" : "+s"(we));   // with the bound in sight the compiler's sweeps are 4% slower
    // we <= ws: no columns left, from the start where every query is empty (their
    // score is the seed); a sweep stores the column before we
    for (int32_t s0 = 0; s0 < TWm && ws < we; s0 += 2) {
        const bool act = s0 < TW;
        const int32_t RL = 8 * s0, RH = RL + 8;   // first rows of the two strips
        uint32_t lutL[9], lutH[9];
        {
            const uint32_t gL = Tp[min(s0, t_last)], gH = Tp[min(s0 + 1, t_last)];
#pragma unroll
            for (int m = 1; m < 9; m++) {   // rows past the target score -8: they raise no maximum
                lutL[m] = RL + m - 1 < tlen ? lut16[(gL >> (32 - 4 * m)) & 15u] : 0x88888888u;
                lutH[m] = RH + m - 1 < tlen ? lut16[(gH >> (32 - 4 * m)) & 15u] : 0x88888888u;
            }
        }
        // column -1, and the one before it (0), when the strips start at column 0
        pk16x2 h[9], o[9], f[9];
        h[0] = as_pk(ws == 0 ? (uint32_t)(s0 == 0 ? h0 : left(RL - 1)) & 0xFFFFu : 0u);
#pragma unroll
        for (int m = 1; m < 9; m++) h[m] = as_pk(ws == 0 ? (uint32_t)left(RL + m - 1) & 0xFFFFu : 0u);
#pragma unroll
        for (int m = 0; m < 9; m++) { o[m] = zero2; f[m] = zero2; }
        uint32_t carry = 0, qshH = 0;
        uint32_t best2 = 0, bpos2 = 0, viol = 0;
        uint32_t alive[9];   // early strips: OR of each row's H
#pragma unroll
        for (int m = 0; m < 9; m++) alive[m] = 0;
        const uint32_t row0 = s0 == 0 ? 0xFFFFu : 0u;   // row 0 runs over all columns: nothing to test
        int32_t first_w = 0x7FFF, last_w = -1;          // words of the bottom row that are not all 0

        auto strips = [&](auto early) {
            constexpr bool EARLY = decltype(early)::value;
            // the low strip at column t, the high one at t - 1; vm: halves inside
            // the query when `tail`
            auto step = [&](int32_t t, uint32_t qshL, uint32_t top, bool tail, uint32_t vm) -> uint32_t {
                pk16x2 e = as_pk(pack_hi(top, carry));
                pk16x2 up_new = as_pk(pack_lo(top, carry)), up_old = h[0], up_older = o[0];
                o[0] = h[0];
                h[0] = up_new;
                pk16x2 colmax = zero2, v = zero2;
#pragma unroll
                for (int m = 1; m < 9; m++) {
                    const uint32_t sl = (uint32_t)__builtin_amdgcn_sbfe(lutL[m], qshL, 4);
                    const uint32_t sh = (uint32_t)__builtin_amdgcn_sbfe(lutH[m], qshH, 4);
                    // M ? M + s : 0, below 0 where that is (:117; s <= 7, so 8 M >= M + s for M >= 1)
                    const pk16x2 M = pmin(up_old + as_pk(pack_lo(sl, sh)), times8(up_old));
                    const pk16x2 hm = pmax(pmax(M, f[m]), e);
                    const pk16x2 tt = M - gapoe2;
                    f[m] = pmax(tt, psubsat(f[m], gape2));
                    e = pmax(tt, psubsat(e, gape2));
                    uint32_t dead = or3(as_u32(up_new), as_u32(up_old), as_u32(up_older));
                    if (m == 1) dead |= row0;
                    v = as_pk(as_u32(v) | as_u32(psubsat(nonzero_one(hm), as_pk(dead))));
                    colmax = pmaxu(colmax, prank(hm, (uint32_t)(8 - m) * 0x00010001u));
                    if (EARLY) alive[m] |= tail ? as_u32(hm) & vm : as_u32(hm);
                    up_new = hm;
                    up_old = h[m];
                    up_older = o[m];
                    o[m] = h[m];
                    h[m] = hm;
                }
                qshH = qshL;
                const uint32_t h8 = as_u32(h[8]), e8 = as_u32(e), bottom = pack_hi(h8, e8);
                carry = pack_lo(h8, e8);
                // the best moves to a column that ranks as high or higher: more H,
                // then the upper row, then the later column
                uint32_t keep;
                asm("v_pk_sub_i16 %0, 0, %1" : "=v"(keep) : "v"(as_u32(nonzero_one(psubsat(as_pk(best2), colmax)))));
                if (tail) {
                    keep |= ~vm;
                    v = as_pk(as_u32(v) & vm);
                    // the query's last column (:155-158; ties go to the later row)
                    const bool lo = t == qlen - 1, hi = t == qlen;
                    if (lo || hi) {
#pragma unroll
                        for (int m = 1; m < 9; m++) {
                            const int32_t hv = (int32_t)(lo ? as_u32(h[m]) & 0xFFFFu : as_u32(h[m]) >> 16);
                            const int32_t R = (lo ? RL : RH) + m - 1;
                            if (R < tlen && hv >= gs) { gs = hv; gi = R; }
                        }
                    }
                }
                viol |= as_u32(v);
                best2 = bits_of(keep, best2, as_u32(colmax));
                bpos2 = bits_of(keep, bpos2, (uint32_t)t * 0x00010001u);
                // one column at a time: left to itself the compiler ranks and tests
                // several columns later and keeps their values (222 VGPRs)
                asm volatile("" : "+v"(best2), "+v"(bpos2), "+v"(viol));
                __builtin_amdgcn_sched_barrier(0);
                return bottom;
            };
            uint32_t nxt[8];
            uint32_t qn = Qp[min(ws, q_last)];
            auto fetch = [&](int32_t j) {
                const uint32_t *p = bd + (size_t)(8 * j) * WAVE;
#pragma unroll
                for (int kk = 0; kk < 8; kk++) nxt[kk] = p[kk * WAVE];
            };
            fetch(ws);
            for (int32_t j = ws; j < we; j++) {
                uint32_t cur[8];
#pragma unroll
                for (int kk = 0; kk < 8; kk++) cur[kk] = nxt[kk];
                const uint32_t q = qn;
                fetch(min(j + 1, we - 1));
                qn = Qp[min(j + 1, q_last)];
                if (s0 == 0) {   // above row 0 (:78-81)
#pragma unroll
                    for (int kk = 0; kk < 8; kk++) cur[kk] = (uint32_t)max(h0 - gapoe - gape * (8 * j + kk), 0);
                }
                const bool tail = __any(act && 8 * j + 8 >= qlen);
                uint32_t any = 0;
                uint32_t *out = bd + ((int64_t)8 * j - 1) * WAVE;   // the high strip's column of step 8 j
#pragma unroll
                for (int kk = 0; kk < 8; kk++) {
                    const int32_t t = 8 * j + kk;
                    const uint32_t vm = (t < qlen ? 0xFFFFu : 0u) | (t <= qlen ? 0xFFFF0000u : 0u);
                    const uint32_t b = step(t, kk < 7 ? (q >> (26 - 4 * kk)) & 0x1Cu : (q << 2) & 0x1Cu, cur[kk], tail, vm);
                    if (kk > 0 || j > ws) {
                        out[kk * WAVE] = b;
                        any |= b;
                    } else {   // the high strip starts at the next step: its column -1
                        h[0] = as_pk(pack_lo(as_u32(h[0]), ws == 0 ? (uint32_t)left(RH - 1) : 0u));
#pragma unroll
                        for (int m = 1; m < 9; m++)
                            h[m] = as_pk(pack_lo(as_u32(h[m]), ws == 0 ? (uint32_t)left(RH + m - 1) : 0u));
#pragma unroll
                        for (int m = 0; m < 9; m++) {
                            o[m] = as_pk(as_u32(o[m]) & 0xFFFFu);
                            f[m] = as_pk(as_u32(f[m]) & 0xFFFFu);
                            alive[m] &= 0xFFFFu;
                        }
                        best2 &= 0xFFFFu;
                        viol &= 0xFFFFu;
                    }
                }
                if (any) { first_w = min(first_w, j); last_w = j; }
            }
            // the high strip's last column
            const uint32_t b = step(8 * we, 0, 0u, true, 8 * we <= qlen ? 0xFFFF0000u : 0u);
            bd[(size_t)(8 * we - 1) * WAVE] = b;
            if (b) { first_w = min(first_w, we - 1); last_w = we - 1; }
        };
        const bool early = __any(act && left(RL) > 0);
        if (early) strips(std::true_type{});
        else strips(std::false_type{});

        const bool hi_ok = s0 + 1 < TW;
        if (act) {
            redo |= hi_ok ? viol : viol & 0xFFFFu;
            if (early) {
#pragma unroll
                for (int m = 1; m < 9; m++) {
                    if (RL + m - 1 < tlen && left(RL + m - 1) > 0 && !(alive[m] & 0xFFFFu)) redo = 1;
                    if (RH + m - 1 < tlen && left(RH + m - 1) > 0 && !(alive[m] >> 16)) redo = 1;
                }
            }
            const int32_t vL = (int32_t)((best2 & 0xFFFFu) >> 3), vH = (int32_t)(best2 >> 19);
            if (vL > bv) { bv = vL; bi = RL + 7 - (int32_t)(best2 & 7u); bj = (int32_t)(bpos2 & 0xFFFFu); }
            if (hi_ok && vH > bv) { bv = vH; bi = RH + 7 - (int32_t)((best2 >> 16) & 7u); bj = (int32_t)(bpos2 >> 16) - 1; }
        }
        // The next sixteen rows: from the first word the row above is not 0 in
        // (a stored column may belong to the word before; word 0 while the left
        // boundary lives) to two columns a row past its last one, and the column
        // at which the test above would fail.
        const bool more = s0 + 2 < TW, lb = left(RH + 7) > 0;
        const bool dead = !more || (last_w < 0 && !lb);
        const int32_t lo = dead ? 0x7FFF : (lb ? 0 : max(first_w - 1, 0));
        const int32_t hi = dead ? 0 : min(QW, last_w + 6);
        ws = max(ws, -wave_max<1>(-lo));
        we = wave_max<1>(hi);
    }
    if (!ok) return;
    if (redo) {
        d.keys[atomicAdd(&d.aux[3], 1u)] = pr;
        return;
    }
    if (gs <= 0 || gs <= bv - end_bonus) {   // :188-197 (PEN_CLIP5 there)
        d.score[pr] = bv; d.qend[pr] = bj + 1; d.tend[pr] = bi + 1;
    } else {
        d.score[pr] = gs; d.qend[pr] = qlen; d.tend[pr] = gi + 1;
    }
}

}  // namespace

hipError_t g2_ksw_packed(const G2Scores &sc, const G2Opts &op, const G2Dev &d, hipStream_t s) {
    k_ksw_pk<<<(d.n + WAVE - 1) / WAVE, WAVE, 0, s>>>(d, sc, op.ksw_eb);
    return hipGetLastError();
}
