// wave.hip -- the packed one-wave path: a group of 16 or 64 lanes per pair.
//
// The lane-per-pair kernels need tens of thousands of pairs of like size to
// fill the chip, and a long pair takes its whole serial time on one lane.
// Here a group of GW lanes runs one pair as a wavefront: lane l of pass k holds
// target strips 2 (GW k + l) and the one after it (8 rows each) in the low and
// high 16-bit halves of its registers, the low strip at column t = tau - 2l of
// step tau, the high strip at column t - 1, under the low strip's bottom row
// of the step before.  The high strip's bottom row and its query class go to
// the next lane with one DPP move each (row_shr:1 for 16 lanes, four pairs a
// wave; wave_shr:1 for 64).  The bottom row of a pass with strips below it is
// kept in the pair's slice of the boundary rows for the next pass.
//
// The longest pairs of a batch that would otherwise wait for them run on a
// block of four waves, its passes in turn: a pass follows the one above it
// through the boundary row, by the number of columns that one has stored (a
// count in LDS).  A wave issues an instruction every
// four to five cycles at best, so a 5000 x 5500 pair takes 10.5 ms on one wave
// (six passes of 5100 steps at 0.34 us) whatever else the chip does.
//
// Bound: packed-16 VALU issue, 13 instructions per row pair and step plus about
// 25 per step for the hand-over and the end tracking, times the share of lanes
// and steps that hold cells: C / (C + 2 GW) per full pass of C columns.  Hence 16 lanes
// wherever a pair's serial time allows it (a pass of 256 rows fills after 32
// steps), 64 for the longest pairs.
//
// The recurrences and boundary rows are those of the lane kernels, whose
// 16-bit bounds the host checks for the batch's largest shape; every output is the
// reference's choice: ends by the first strict maximum in (strip, column, row)
// order, merged over lanes by that order.
#include "device.h"

#include <type_traits>

namespace {

constexpr int PW_WAVES = 4;   // per block
enum { PW_LOCAL, PW_GLOBAL, PW_SEMI };
enum { PW_FORWARD, PW_LOCAL_REVERSE, PW_SEMI_REVERSE };   // how a run reads its sequences

// One DP over a group's pair (uniform within the group).
struct PwPair {
    const uint32_t *q, *t;   // forward, semi reverse: the first word; LOCAL reverse: the last word
    int32_t qw, nst;         // query words, strips
    int32_t qlen, tlen;
    int32_t i0;              // SEMI reverse: index of the first strip (may be negative)
};
struct PwSemi {
    bool ht, hq, tt, tq;     // heads free on the target / query, tails on the target / query
};
// LOCAL: first maximal cell.  GLOBAL: v = score.  SEMI: v and row = the target
// tail's maximum and its row, bb and bcol = the query tail's (MINUS_INF: none).
struct PwEnd {
    int32_t v, strip, col, row, bb, bcol;
};

template <int REV>
__device__ __forceinline__ uint32_t pw_qword(const PwPair &r, int32_t j) {
    if (REV == PW_FORWARD) return r.q[j];
    if (REV == PW_LOCAL_REVERSE) return nib_reverse(*(r.q - j));
    return rev_word(r.q, r.qlen, j);
}
template <int REV>
__device__ __forceinline__ uint32_t pw_tword(const PwPair &r, int32_t s) {
    if (REV == PW_FORWARD) return r.t[s];
    if (REV == PW_LOCAL_REVERSE) return nib_reverse(*(r.t - s));
    return r.i0 + s >= 0 ? rev_word(r.t, r.tlen, r.i0 + s) : 0u;
}

struct PwShared {
    uint32_t lut16[16];          // score tables of the 16 target nibbles
    int32_t done[PW_WAVES];      // COOP: 8-column blocks of the row each wave has stored
    int32_t end[PW_WAVES][9];    // COOP: each wave's results
};

// COOP: the block's waves share the pair's passes; every wave calls this, with
// sh.done cleared.
// RANK (LOCAL): cells are ranked as h * 8 + (7 - row) (h <= 8191), else by h
// alone, the row taken from the registers of the steps that raise a maximum.
// fwd (SEMI reverse): strips run until one holds a value >= fwd.
template <int MODE, int GW, int REV, bool RANK, bool COOP>
__device__ __forceinline__ void pw_run(const G2Scores &c, const PwSemi &sm, PwShared &sh, const PwPair &r, uint32_t *row,
                                       int32_t fwd, PwEnd &res) {
    const int32_t wv = COOP ? __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE) : 0;
    const int32_t lane = (int32_t)(threadIdx.x & (WAVE - 1)), l = lane & (GW - 1), lane0 = lane - l;
    const int32_t gapo = c.gapo, gape = c.gape, gapoe = c.gapoe;
    const pk16x2 gapoe2 = {(short)gapoe, (short)gapoe}, gape2 = {(short)gape, (short)gape};
    const pk16x2 zero2 = {0, 0};
    const int32_t C = 8 * r.qw, last_word = max(r.qw - 1, 0);
    const bool live = r.nst > 0 && C > 0;
    const int32_t Cmax = wave_max(live ? C : 0), Cmin = -wave_max(live ? -C : -0x7FFFFFFF);
    const int32_t npass = live ? (r.nst + 2 * GW - 1) / (2 * GW) : 0, npass_max = wave_max(npass);
    int32_t nst = live ? r.nst : 0;
    // boundary values left of column 0: GLOBAL's H of row R (1-based; 0 above
    // the first), SEMI's strip initialisation for the row counter u
    // (src/kernels/global.h:67-71, src/kernels/semiglobal_kernel_template.h:114-129)
    auto hl = [&](int32_t R) -> int32_t { return R == 0 ? 0 : -(gapo + gape * R); };
    auto semi_h = [&](int32_t u, int32_t m) -> int32_t { return sm.ht ? 0 : -(gapo + gape * (u + m - 2)); };
    auto semi_p = [&](int32_t u, int32_t m) -> int32_t { return (sm.ht || u + m - 1 == 1) ? 0 : -(gapo + gape * (u + m - 2)); };

    int32_t bv = MODE == PW_SEMI ? MINUS_INF : 0, bs = 0x7FFFFFFF, bc = 0x7FFFFFFF, br = 0, beff = MINUS_INF;
    int32_t pick_strip = 0x7FFFFFFF, bb = MINUS_INF, bcol = 0;   // SEMI: the strip whose bottom row the query tail reads
    for (int32_t k = wv; k < npass_max; k += COOP ? PW_WAVES : 1) {
        // COOP: blocks of the row above this pass, counted in the upper wave's done
        const int32_t *above = &sh.done[(k + PW_WAVES - 1) % PW_WAVES];
        const int32_t above0 = k > 0 ? (k - 1) / PW_WAVES * (r.qw + 1) : 0, mine0 = k / PW_WAVES * (r.qw + 1);
        auto await = [&](int32_t blocks) {
            if (!COOP || k == 0) return;
            while (__hip_atomic_load(above, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) < above0 + blocks)
                __builtin_amdgcn_s_sleep(1);
        };
        auto publish = [&](int32_t blocks) {
            if (COOP) __hip_atomic_store(&sh.done[wv], mine0 + blocks, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
        };
        const int32_t sL = 2 * (GW * k + l), sH = sL + 1;
        const int32_t nact = min(max((nst - 2 * GW * k + 1) / 2, 0), GW), nact_max = wave_max(nact);
        const bool more = nst > 0 && k + 1 < npass;   // strips of the pair below this pass (then nact = GW)
        uint32_t lutL[9], lutH[9];
        {
            const uint32_t gL = sL < nst ? pw_tword<REV>(r, sL) : 0u, gH = sH < nst ? pw_tword<REV>(r, sH) : 0u;
#pragma unroll
            for (int m = 1; m < 9; m++) {
                lutL[m] = sh.lut16[(gL >> (32 - 4 * m)) & 15u];
                lutH[m] = sh.lut16[(gH >> (32 - 4 * m)) & 15u];
            }
        }
        pk16x2 h[9], f[9];
#pragma unroll
        for (int m = 0; m < 9; m++) { h[m] = zero2; f[m] = zero2; }
        uint32_t outb = 0, carry = 0;          // bottom (H | E << 16) of the high / low strip, previous step
        uint32_t qA = 0, qB = 0;               // query classes (times 4) of the low / high strip, previous step
        uint32_t best2 = 0, bpos2 = 0, brow2 = 0;   // LOCAL: per half the pass's best, its step and (no RANK) row
        int32_t bbL = MINUS_INF, bcL = 0, bbH = MINUS_INF, bcH = 0;   // SEMI query tail: bottom row's first maximum
        // one step; q0 and top0: the group's first lane's query class and row
        // above; starts: lanes may start in this step; ends: lanes may be past
        // their columns or at the column they report
        auto step = [&](int32_t tau, uint32_t q0, uint32_t top0, bool starts, bool ends) {
            const uint32_t tin = from_above<GW>(top0, outb);
            const uint32_t qL = from_above<GW>(q0, qB), qH = qA;
            qA = qL;
            qB = qH;
            const int32_t t = tau - 2 * l;
            if (starts && t == 0) {   // the low strip starts: its column -1
#pragma unroll
                for (int m = 0; m < 9; m++) {
                    if (MODE == PW_LOCAL) {
                        h[m] = set_lo(h[m], 0);
                        f[m] = set_lo(f[m], 0);
                    } else if (MODE == PW_GLOBAL) {
                        h[m] = set_lo(h[m], hl(8 * sL + m));
                        f[m] = set_lo(f[m], NEG16);
                    } else {
                        // diagonals of column 0 where the step reads them (H of
                        // the row above one column back), F such that this
                        // step's extension gives the strip's own open from H
                        h[m] = set_lo(h[m], m < 8 ? semi_p(8 * sL + 1, m + 1) : semi_h(8 * sL + 1, 8));
                        f[m] = set_lo(f[m], semi_h(8 * sL + 1, m) - gapoe + gape);
                    }
                }
                if (MODE == PW_LOCAL) best2 &= 0xFFFF0000u;
                if (MODE == PW_SEMI) bbL = MINUS_INF;
            }
            pk16x2 e = as_pk(pack_hi(tin, carry));
            pk16x2 p = h[0];
            h[0] = as_pk(pack_lo(tin, carry));
            pk16x2 colmax = zero2;
            if (MODE == PW_SEMI) {   // E and F open from H (src/kernels/semiglobal_kernel_template.h:17-28)
                pk16x2 open = h[0] - gapoe2;
#pragma unroll
                for (int m = 1; m < 9; m++) {
                    const uint32_t sl = (uint32_t)__builtin_amdgcn_sbfe(lutL[m], qL, 4);
                    const uint32_t sh = (uint32_t)__builtin_amdgcn_sbfe(lutH[m], qH, 4);
                    f[m] = pmax(h[m] - gapoe2, f[m] - gape2);
                    e = pmax(open, e - gape2);
                    const pk16x2 cur = pmax(pmax(p + as_pk(pack_lo(sl, sh)), f[m]), e);
                    p = h[m];
                    h[m] = cur;
                    open = cur - gapoe2;
                }
            } else {
#pragma unroll
                for (int m = 1; m < 9; m++) {
                    const uint32_t sl = (uint32_t)__builtin_amdgcn_sbfe(lutL[m], qL, 4);
                    const uint32_t sh = (uint32_t)__builtin_amdgcn_sbfe(lutH[m], qH, 4);
                    const pk16x2 tmp = p + as_pk(pack_lo(sl, sh));
                    const pk16x2 hm = pmax(pmax(tmp, f[m]), e);
                    const pk16x2 tt = tmp - gapoe2;
                    if (MODE == PW_LOCAL) {   // E and F held as max(E, 0) and max(F, 0): no max of H with 0
                        f[m] = pmax(tt, psubsat(f[m], gape2));
                        e = pmax(tt, psubsat(e, gape2));
                        colmax = RANK ? pmaxu(colmax, prank(hm, (uint32_t)(8 - m) * 0x00010001u)) : pmaxu(colmax, hm);
                    } else {
                        f[m] = pmax(tt, f[m] - gape2);
                        e = pmax(tt, e - gape2);
                    }
                    p = h[m];
                    h[m] = hm;
                }
            }
            const uint32_t h8 = as_u32(h[8]), e8 = as_u32(e);
            outb = pack_hi(h8, e8);
            carry = pack_lo(h8, e8);
            if (more && l == GW - 1 && t >= 1 && t <= C) row[t - 1] = outb;
            if (MODE == PW_LOCAL) {
                // a half's best moves to this column when its h beats the best's h
                const pk16x2 one2 = {1, 1};
                uint32_t up = nonzero_mask(psubsat(colmax, as_pk(RANK ? best2 | 0x00070007u : best2)));
                if (ends) up &= (t < C ? 0xFFFFu : 0u) | (t <= C ? 0xFFFF0000u : 0u);
                if (!RANK && __any(up != 0)) {   // the first row holding the column's maximum
                    pk16x2 r2 = zero2;
#pragma unroll
                    for (int m = 1; m < 8; m++) {
                        const pk16x2 same = psubsat(one2, as_pk(as_u32(h[m]) ^ as_u32(colmax)));
                        r2 = pmaxu(r2, same * (pk16x2){(short)(8 - m), (short)(8 - m)});
                    }
                    brow2 = bits_of(up, as_u32(r2), brow2);
                }
                best2 = bits_of(up, as_u32(colmax), best2);
                bpos2 = bits_of(up, (uint32_t)tau * 0x00010001u, bpos2);
            }
            if (MODE == PW_GLOBAL && ends) {   // the score: row tlen, column qlen (src/kernels/global.h:98-103, 299)
                const bool at_lo = sL == nst - 1 && t == r.qlen - 1, at_hi = sH == nst - 1 && t - 1 == r.qlen - 1;
                if (at_lo || at_hi) {
                    const int32_t rowsel = 8 - (8 * nst - r.tlen);
#pragma unroll
                    for (int m = 1; m < 9; m++) {
                        const uint32_t u = as_u32(h[m]);
                        if (m == rowsel) bv = at_lo ? sx16(u) : sx16(u >> 16);
                    }
                    bs = 0;
                }
            }
            if (MODE == PW_SEMI) {
                if (sm.tt && ends) {   // the query's last column (:160-178, :269-360)
                    const bool at_lo = sL < nst && t == r.qlen - 1, at_hi = sH < nst && t - 1 == r.qlen - 1;
                    if (at_lo || at_hi) {
                        const int32_t s = at_lo ? sL : sH;
                        int32_t cv = MINUS_INF, cy = 0;
#pragma unroll
                        for (int m = 1; m < 9; m++) {
                            const int32_t hv = at_lo ? sx16(as_u32(h[m])) : sx16(as_u32(h[m]) >> 16);
                            const int32_t y = 8 * (r.i0 + s) + m - 1;
                            if (hv > cv && y < r.tlen) { cv = hv; cy = y; }
                        }
                        const int32_t eff = min(cv, fwd);
                        if (eff > beff) { beff = eff; bv = cv; br = cy; bs = s; }
                    }
                }
                if (sm.tq) {   // the strips' bottom rows: first maximum over the query's columns
                    const int32_t vl = sx16(h8), vh = sx16(h8 >> 16);
                    if (t < r.qlen && vl > bbL) { bbL = vl; bcL = t; }
                    if (t - 1 < r.qlen && vh > bbH) { bbH = vh; bcH = t - 1; }
                }
            }
            if (starts && t == 0) {   // the high strip starts at the next step
#pragma unroll
                for (int m = 0; m < 9; m++) {
                    if (MODE == PW_LOCAL) {
                        h[m] = set_hi(h[m], 0);
                        f[m] = set_hi(f[m], 0);
                    } else if (MODE == PW_GLOBAL) {
                        h[m] = set_hi(h[m], hl(8 * sH + m));
                        f[m] = set_hi(f[m], NEG16);
                    } else {
                        h[m] = set_hi(h[m], m < 8 ? semi_p(8 * sH + 1, m + 1) : semi_h(8 * sH + 1, 8));
                        f[m] = set_hi(f[m], semi_h(8 * sH + 1, m) - gapoe + gape);
                    }
                }
                if (MODE == PW_LOCAL) best2 &= 0xFFFFu;
                if (MODE == PW_SEMI) bbH = MINUS_INF;
            }
        };
        // Eight steps, one query word of the first lane, at a time; the next
        // word and the next eight entries of the row above are in flight
        // meanwhile (on the first pass those entries are not used).
        const int32_t steps = nact_max > 0 ? Cmax + 2 * nact_max - 1 : 0;
        const u32x4 *row4 = reinterpret_cast<const u32x4 *>(row);
        uint32_t qn = live ? pw_qword<REV>(r, 0) : 0u;
        await(1);
        u32x4 na = row4[0], nb = row4[1];
        for (int32_t j = 0; 8 * j < steps; j++) {
            const uint32_t qw = qn;
            const u32x4 ra = na, rb = nb;
            const int32_t jn = min(j + 1, last_word);
            qn = live ? pw_qword<REV>(r, jn) : 0u;
            await(jn + 1);
            na = row4[2 * jn];
            nb = row4[2 * jn + 1];
            const bool starts = 8 * j < 2 * nact_max, ends = 8 * j + 7 >= Cmin - 8;
#pragma unroll
            for (int kk = 0; kk < 8; kk++) {
                const int32_t tau = 8 * j + kk;
                uint32_t top0 = kk < 4 ? ra[kk & 3] : rb[kk & 3];
                if (k == 0) top0 = MODE == PW_GLOBAL || (MODE == PW_SEMI && !sm.hq)
                                       ? pk16(tau == 0 ? 0 : -(gapo + gape * tau), NEG16) : 0u;
                step(tau, kk < 7 ? (qw >> (26 - 4 * kk)) & 0x1Cu : (qw << 2) & 0x1Cu, top0, starts, ends);
            }
            // the last lane's high strip is 2 GW - 1 columns behind
            if (j >= 2 * GW / 8) publish(min(j - 2 * GW / 8 + 1, last_word));
        }
        publish(r.qw);

        if (MODE == PW_LOCAL) {
            const uint32_t eL = best2 & 0xFFFFu, eH = best2 >> 16;
            const int32_t vL = (int32_t)(RANK ? eL >> 3 : eL), vH = (int32_t)(RANK ? eH >> 3 : eH);
            if (sL < nst && vL > bv) {
                bv = vL; bs = sL; bc = (int32_t)(bpos2 & 0xFFFFu) - 2 * l;
                br = 7 - (int32_t)(RANK ? eL & 7u : brow2 & 0xFFFFu);
            }
            if (sH < nst && vH > bv) {
                bv = vH; bs = sH; bc = (int32_t)(bpos2 >> 16) - 2 * l - 1;
                br = 7 - (int32_t)(RANK ? eH & 7u : brow2 >> 16);
            }
        }
        if (MODE == PW_SEMI && (sm.tq || (REV == PW_SEMI_REVERSE && sm.tt))) {
            // the strip whose bottom row the query tail reads: the one that
            // ends a reverse run, else the pair's last
            int32_t ge = beff, gs = bs;
#pragma unroll
            for (int off = GW / 2; off > 0; off >>= 1) {
                const int32_t oe = __shfl_xor(ge, off), os = __shfl_xor(gs, off);
                if (oe > ge || (oe == ge && os < gs)) { ge = oe; gs = os; }
            }
            const bool stop = REV == PW_SEMI_REVERSE && sm.tt && ge >= fwd && nst > 0;
            const int32_t pick = stop ? gs : (nst > 0 && k + 1 == npass ? nst - 1 : -1);
            const int32_t from = lane0 + (pick >= 0 ? ((pick >> 1) - GW * k) & (GW - 1) : 0);
            const int32_t xl = __shfl(bbL, from), xcl = __shfl(bcL, from), xh = __shfl(bbH, from), xch = __shfl(bcH, from);
            if (pick >= 0) {
                pick_strip = pick;
                bb = (pick & 1) ? xh : xl;
                bcol = (pick & 1) ? xch : xcl;
            }
            if (stop) nst = 0;   // this pair needs no further pass; other pairs of the wave go on
        }
        // the row stored by this pass is read by the next
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        __builtin_amdgcn_wave_barrier();
    }
    // merge the group's lanes in the reference's order
#pragma unroll
    for (int off = GW / 2; off > 0; off >>= 1) {
        const int32_t ov = __shfl_xor(bv, off), os = __shfl_xor(bs, off), oc = __shfl_xor(bc, off), orow = __shfl_xor(br, off);
        const int32_t oe = __shfl_xor(beff, off);
        bool take;
        if (MODE == PW_LOCAL) take = ov > bv || (ov == bv && (os < bs || (os == bs && oc < bc)));
        else if (MODE == PW_GLOBAL) take = os < bs;   // the one lane that holds the score
        else take = oe > beff || (oe == beff && os < bs);
        if (take) { bv = ov; bs = os; bc = oc; br = orow; beff = oe; }
    }
    if (COOP) {   // and the block's waves in the same way; the first strip picked is the one that ends a reverse run
        if (lane == 0) {
            int32_t *o = sh.end[wv];
            o[0] = bv; o[1] = bs; o[2] = bc; o[3] = br; o[4] = beff; o[5] = pick_strip; o[6] = bb; o[7] = bcol;
        }
        __syncthreads();
        for (int w = 0; w < PW_WAVES; w++) {
            const int32_t *o = sh.end[w];
            bool take;
            if (MODE == PW_LOCAL) take = o[0] > bv || (o[0] == bv && (o[1] < bs || (o[1] == bs && o[2] < bc)));
            else if (MODE == PW_GLOBAL) take = o[1] < bs;
            else take = o[4] > beff || (o[4] == beff && o[1] < bs);
            if (take) { bv = o[0]; bs = o[1]; bc = o[2]; br = o[3]; beff = o[4]; }
            if (o[5] < pick_strip) { pick_strip = o[5]; bb = o[6]; bcol = o[7]; }
        }
        __syncthreads();
    }
    res.bb = bb;
    res.bcol = bcol;
    res.v = bv;
    res.strip = bs;
    res.col = bc;
    res.row = br;
}

template <int MODE, bool START, bool RANK, int GW, bool COOP>
__device__ __forceinline__ void pw_pairs(const G2Dev &d, const G2Scores &c, PwShared &sh, uint32_t slot0, int32_t head,
                                         int32_t tail) {
    auto fresh = [&]() {   // COOP: no column stored yet
        if (!COOP) return;
        if (threadIdx.x < PW_WAVES) sh.done[threadIdx.x] = 0;
        __syncthreads();
    };
    const uint32_t lane = threadIdx.x & (WAVE - 1), slot = slot0 + lane / GW;
    const bool ok = slot < d.n;
    const uint32_t pr = d.perm[ok ? slot : d.n - 1];
    const uint32_t qoff = d.qoff[pr], toff = d.toff[pr];
    const int32_t qlen = ok ? (int32_t)d.qlen[pr] : 0, tlen = ok ? (int32_t)d.tlen[pr] : 0;
    const uint32_t *Q = d.pq + (qoff >> 3), *T = d.pt + (toff >> 3);
    uint32_t *row = d.bnd + (size_t)(ok ? slot : d.n - 1) * d.bnd_cols;   // only pairs of several passes use it
    const int32_t QW = dregs((uint32_t)qlen), TW = dregs((uint32_t)tlen);
    const PwSemi sm = {head == D_TARGET || head == D_BOTH, head == D_QUERY || head == D_BOTH,
                       tail == D_TARGET || tail == D_BOTH, tail == D_QUERY || tail == D_BOTH};
    const bool first = ok && (lane & (GW - 1)) == 0 && (!COOP || threadIdx.x == 0);
    fresh();
    PwEnd e;
    const PwPair fw = {Q, T, QW, TW, qlen, tlen, 0};
    pw_run<MODE, GW, PW_FORWARD, RANK, COOP>(c, sm, sh, fw, row, 0x7FFFFFFF, e);
    if (MODE == PW_GLOBAL) {
        if (first) d.score[pr] = e.v;
        return;
    }
    if (MODE == PW_LOCAL) {
        const int32_t qe = e.v > 0 ? e.col : 0, te = e.v > 0 ? e.strip * 8 + e.row : 0;
        if (first) {
            d.score[pr] = e.v;
            d.qend[pr] = qe;
            d.tend[pr] = te;
        }
        if (START) {   // the DP over the reversed prefix rectangle (src/kernels/local_kernel_template.h:441-511)
            const int32_t rend = min((qe >> 3) + 1, QW), gend = min((te >> 3) + 1, TW);
            const PwPair rv = {Q + max(rend - 1, 0), T + max(gend - 1, 0), rend, e.v > 0 ? gend : 0, qlen, tlen, 0};
            PwEnd s;
            fresh();
            pw_run<MODE, GW, PW_LOCAL_REVERSE, RANK, COOP>(c, sm, sh, rv, row, 0x7FFFFFFF, s);
            if (first) {
                d.qstart[pr] = s.v > 0 ? 8 * rend - 1 - s.col : 0;
                d.tstart[pr] = s.v > 0 ? 8 * (gend - s.strip) - 1 + s.row : 0;
            }
        }
        return;
    }
    // SEMI_GLOBAL: initial values, target tail, query tail (:49-74, :160-214)
    int32_t best = MINUS_INF, x = tlen, y = qlen;
    auto tails = [&](const PwEnd &s, bool run) {
        if (sm.tt && s.v > best) { best = s.v; y = s.row; }
        if (sm.tq) {
            // no strip run: the boundary row itself, whose first entry is its maximum
            const int32_t bb = run ? s.bb : (qlen > 0 ? 0 : MINUS_INF), bcol = run ? s.bcol : 0;
            if (bb > best) { best = bb; x = bcol; }
            if (x != tlen) y = qlen;
        }
    };
    tails(e, TW > 0 && QW > 0);
    if (first) {
        d.score[pr] = best;
        d.tend[pr] = y;
        d.qend[pr] = x;
    }
    if (START) {   // reversed copies, from the strip holding the end (:227-384)
        const int32_t fwd = best, dd = TW - ((y >> 3) + 1), i0 = dd > 0 ? dd - 1 : dd;
        const PwPair rv = {Q, T, QW, fwd > MINUS_INF ? TW - i0 : 0, qlen, tlen, i0};
        PwEnd s;
        fresh();
        pw_run<MODE, GW, PW_SEMI_REVERSE, RANK, COOP>(c, sm, sh, rv, row, fwd, s);
        best = MINUS_INF;
        y = 0;
        tails(s, rv.nst > 0 && QW > 0);
        if (first) {
            d.tstart[pr] = (tlen - 1) - y;
            d.qstart[pr] = (qlen - 1) - x;
        }
    }
}

// Launch: a block for each of the first d.wave_coop sorted slots, then four of
// the next d.wave64 slots a block (one a wave), then sixteen of the others.
// (Two launches, the others in blocks of one wave, ran the same batches no
// faster and kept the long pairs' waves from sharing the chip: 20,000 pairs of
// 50-5000 bases 6.5 against 4.1 ms.)
template <int MODE, bool START, bool RANK>
__global__ __launch_bounds__(PW_WAVES * WAVE) void k_wave(G2Dev d, G2Scores c, int32_t head, int32_t tail) {
    // the SEMI WITH_START run reads reversed copies padded with nibble 0
    const uint32_t census = d.aux[0] | (MODE == PW_SEMI && START ? 1u : 0u);
    if (!census_fast(census)) return;   // the lane kernels take this batch
    __shared__ PwShared sh;
    if (threadIdx.x < 16)
        sh.lut16[threadIdx.x] = MODE == PW_GLOBAL ? score_lut<true>(c, 0, census, threadIdx.x)
                                                  : score_lut(c, c.has_np ? -c.np : 0, census, threadIdx.x);
    __syncthreads();
    const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), b0 = d.wave_coop, b1 = b0 + (d.wave64 + 3) / 4;
    const uint32_t b = blockIdx.x;
    if (b < b0) {
        pw_pairs<MODE, START, RANK, 64, true>(d, c, sh, b, head, tail);
    } else if (b < b1) {
        const uint32_t k = 4 * (b - b0) + wv;
        if (k < d.wave64) pw_pairs<MODE, START, RANK, 64, false>(d, c, sh, b0 + k, head, tail);
    } else {
        const uint32_t slot = b0 + d.wave64 + 16 * (b - b1) + 4 * wv;
        if (slot < d.n) pw_pairs<MODE, START, RANK, 16, false>(d, c, sh, slot, head, tail);
    }
}

template <int MODE, bool START, bool RANK>
void wave_launch(const G2Scores &sc, const G2Opts &op, const G2Dev &d, hipStream_t s) {
    const uint32_t narrow = d.n - d.wave_coop - d.wave64;
    const uint32_t blocks = d.wave_coop + (d.wave64 + 3) / 4 + (narrow + 15) / 16;
    k_wave<MODE, START, RANK><<<blocks, PW_WAVES * WAVE, 0, s>>>(d, sc, op.head, op.tail);
}

}  // namespace

hipError_t g2_wave_run(const G2Scores &sc, const G2Opts &op, const G2Dev &d, hipStream_t s) {
    const bool start = op.start == S_WITH_START;
    if (op.algo == A_LOCAL) {
        if (d.wave == 1) start ? wave_launch<PW_LOCAL, true, true>(sc, op, d, s) : wave_launch<PW_LOCAL, false, true>(sc, op, d, s);
        else start ? wave_launch<PW_LOCAL, true, false>(sc, op, d, s) : wave_launch<PW_LOCAL, false, false>(sc, op, d, s);
    } else if (op.algo == A_GLOBAL) {
        wave_launch<PW_GLOBAL, false, true>(sc, op, d, s);
    } else {
        start ? wave_launch<PW_SEMI, true, true>(sc, op, d, s) : wave_launch<PW_SEMI, false, true>(sc, op, d, s);
    }
    return hipGetLastError();
}
