// wavetb.hip -- LOCAL and GLOBAL WITH_TB on groups of 4, 16, 32 or 64 lanes per
// pair, with the checkpoints the traceback rebuilds its tiles from.
//
// Lane l of pass k holds target strips 2 (GW k + l) and the next one (8 rows
// each) in the low and high 16-bit halves of its registers, the high strip one
// column behind the low one.  A lane works one query word (eight columns) an
// iteration, one word behind the lane above it, so that all lanes of a wave
// begin and end their 8x8 tiles in the same instruction: the tiles' records
// need no per-lane phase.  A lane goes on to its strips of the next pass right
// after its last word, and the first lane's row above comes from the records
// of the pass before: a pair fills its lanes once, whatever its passes.
//
// Bound: the records' writes, 1 B per cell in whole lines (a record a lane, 64
// lanes side by side), 3 TB/s of them: 100,001 pairs GLOBAL take 2.32 ms, 1.86
// with a quarter of the records left out and 1.47 with half, and five in a
// hundred fewer instructions change nothing.  Behind it packed-16 VALU issue, 14
// instructions per row pair and step and about 25 a step for the hand-over, the
// ends and the records (2.6 G wave instructions on 300,000 pairs, 65% of 7.1 ms),
// times the share of lanes and iterations that hold cells: a pair fills its lanes
// in GW iterations, strips are rounded up to 2 GW.  Hence 4 lanes wherever the
// batch has pairs enough, more for few or long ones.
// DP, before and after: 100,001 pairs of 100-300 x 100-400 bases GLOBAL 5.95 ms
// (one lane a pair, direction words) -> 2.3; 50,000 pairs of 50-5000 bases LOCAL 32
// -> 9.2 (13.6 with the longest on one wave); 50,000 pairs with second best (half a
// wave a SIMD on two pairs a lane) 5.5 -> 1.6.
//
// The values are those of the lane kernels (k_local_fast, k_global), whose
// 16-bit bounds the host checks for the batch's largest shape; ends are the
// first strict maximum in (strip, column, row) order.
//
// Second best (LOCAL): the largest h below the running maximum in that order,
// which a wavefront does not have when it meets a cell.  The DP keeps, per
// strip, its maximum and a lower bound of what lies below its own running
// maximum; k_second_scan then knows the running maximum every strip starts
// from and a lower bound of the answer, and k_second_strips recomputes only the
// strips that could beat it -- the last one or two the best path crosses -- from
// the bottom row stored above them.
#include "device.h"

namespace {

enum { TB_LOCAL, TB_GLOBAL };

__device__ __forceinline__ void rec_store(uint32_t *p, const uint32_t *w) {
    reinterpret_cast<u32x4 *>(p)[0] = u32x4{w[0], w[1], w[2], w[3]};
    reinterpret_cast<u32x4 *>(p)[1] = u32x4{w[4], w[5], w[6], w[7]};
}
__device__ __forceinline__ void rec_load(const uint32_t *p, uint32_t *w) {
    const u32x4 a = reinterpret_cast<const u32x4 *>(p)[0], b = reinterpret_cast<const u32x4 *>(p)[1];
    w[0] = a.x; w[1] = a.y; w[2] = a.z; w[3] = a.w;
    w[4] = b.x; w[5] = b.y; w[6] = b.z; w[7] = b.w;
}

constexpr int WV_WAVES = 4;   // per block
struct WvShared {
    uint32_t lut16[16];          // score tables of the 16 target nibbles
    uint32_t it0;                // COOP: the pair's first iteration
    uint32_t strip0;             // and its strips' first record
    int32_t done[WV_WAVES];      // COOP: iterations whose records each wave has stored
    int32_t end[WV_WAVES][4];    // COOP: each wave's best
};

// The pairs of one wave: slots slot0, slot0 + 1, ... below slot_end, GW lanes
// each.  COOP: the block's four waves share one pair, wave w its passes w, w + 4,
// ...; a pass follows the one above it by the iterations that one has stored.
template <int MODE, bool SECOND, int GW, bool COOP>
__device__ __forceinline__ void wv_pairs(const G2Dev &d, const G2Scores &c, WvShared &sh, uint32_t slot0, uint32_t slot_end) {
    const uint32_t *lut16 = sh.lut16;
    constexpr int NW = COOP ? WV_WAVES : 1;
    const int32_t wv = COOP ? (int32_t)__builtin_amdgcn_readfirstlane(threadIdx.x / WAVE) : 0;
    const int32_t lane = (int32_t)(threadIdx.x & (WAVE - 1)), l = lane & (GW - 1);
    const int32_t gapo = c.gapo, gape = c.gape;
    const pk16x2 gapoe2 = {(short)c.gapoe, (short)c.gapoe}, gape2 = {(short)c.gape, (short)c.gape};
    const pk16x2 zero2 = {0, 0};
    const uint32_t slot = slot0 + (uint32_t)(lane / GW);
    const bool ok = slot < slot_end;
    const uint32_t pr = d.perm[ok ? slot : slot_end - 1];
    const int32_t qlen = (int32_t)d.qlen[pr], tlen = (int32_t)d.tlen[pr];
    const int32_t QW = dregs((uint32_t)qlen), TW = dregs((uint32_t)tlen);   // at least one word each (the host checks)
    const uint32_t *Q = d.pq + (d.qoff[pr] >> 3), *T = d.pt + (d.toff[pr] >> 3);
    const int32_t passes = ok ? (TW + 2 * GW - 1) / (2 * GW) : 0;        // of the pair
    const int32_t P = wv_period(QW, COOP ? 256 : GW), npass = (passes - wv + NW - 1) / NW, strips = ok ? TW : 0;   // npass: this wave's
    const int32_t its = wave_max<GW>(npass > 0 ? npass * P + GW : 0);
    const bool slack = !__any(P < GW + 3);
    // The wave's iterations and, for the second best, its pairs' strips, claimed by
    // one atomic (a second one on the word next to it cost 50 us of 440 on 20,000
    // pairs, 1250 waves that all start with it).  The strips' records take a place
    // per strip of the batch (a row of the longest target's strips per pair took n
    // times its length); k_second_scan finds the pair's first one in wv_sec.
    uint32_t it0 = 0, strip0 = 0;
    if (wv == 0) {
        const uint32_t own = SECOND && ok && l == 0 ? (uint32_t)TW : 0u;
        uint32_t upto = own;
        if (SECOND) {
#pragma unroll
            for (uint32_t off = 1; off < WAVE; off <<= 1) {
                const uint32_t o = __shfl_up(upto, off);
                upto += lane >= (int32_t)off ? o : 0u;
            }
        }
        unsigned long long got = 0;
        if (lane == WAVE - 1)
            got = atomicAdd(reinterpret_cast<unsigned long long *>(d.aux + 6),
                            (unsigned long long)upto << 32 |
                                (COOP ? wv_region((uint32_t)passes, P, WV_WAVES) : (uint32_t)its));
        it0 = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)got, WAVE - 1);
        if (SECOND) {
            strip0 = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(got >> 32), WAVE - 1) + __shfl(upto - own, lane - l);
            if (own) d.wv_sec[slot] = strip0;
        }
    }
    if (COOP) {
        if (threadIdx.x == 0) { sh.it0 = it0; sh.strip0 = strip0; }
        if (lane == 0) sh.done[wv] = 0;
        __syncthreads();
        it0 = __builtin_amdgcn_readfirstlane(sh.it0);
        if (SECOND) strip0 = __builtin_amdgcn_readfirstlane(sh.strip0);
    }
    uint32_t *out = d.tb + (size_t)(it0 + (COOP ? wv_region((uint32_t)passes, P, (uint32_t)wv) : 0u)) * WV_ITER + (uint32_t)lane * 8u;   // this iteration's records of the lane
    if (ok && l == 0 && wv == 0)
        d.wv_at[pr] = make_uint2(it0, (uint32_t)lane | (uint32_t)(COOP ? 8 : __builtin_ctz(GW)) << 8 |
                                          (COOP ? (uint32_t)passes << 12 : 0u));
    auto strip_of = [&](int32_t k) -> int32_t { return 2 * (GW * (NW * k + wv) + l); };   // the lane's low strip of pass k
    // COOP: the row above word j of the wave's pass k, from the wave of the pass
    // above; waits until it is stored
    const int32_t up = (wv + NW - 1) % NW;
    auto coop_row = [&](int32_t k, int32_t j) -> const uint32_t * {
        const int32_t it = (wv > 0 ? k : k - 1) * P + j + GW - 1;
        const int32_t need = __builtin_amdgcn_readfirstlane(it + 2);   // the first lane's word; its record is stored an iteration later
        const bool waits = __builtin_amdgcn_readfirstlane(NW * k + wv > 0 && k < npass && j < QW);
        while (waits && __hip_atomic_load(&sh.done[up], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP) < need)
            __builtin_amdgcn_s_sleep(1);
        return d.tb + (size_t)(it0 + wv_region((uint32_t)passes, P, (uint32_t)up) + (uint32_t)it) * WV_ITER + 3 * WV_STREAM + (GW - 1) * 8;
    };
    auto hl = [&](int32_t R) -> int32_t { return R == 0 ? 0 : -(gapo + gape * R); };   // src/kernels/global.h:67-71
    // GLOBAL: H(column - 1) and E of the row above the matrix (src/kernels/global.h:57-60)
    auto top_row = [&](int32_t col) -> uint32_t {
        return MODE == TB_LOCAL ? 0u : pk16(col < 2 ? 0 : -(gapo + gape * (col - 1)), NEG16);
    };

    // the lane's word and pass; before its first word it waits at the end of pass -1
    int32_t j = P - 1 - l, k = -1, sH = 0x7FFFFFFF;
    uint32_t gL = T[min(strip_of(0), TW - 1)], gH = T[min(strip_of(0) + 1, TW - 1)];   // target words of the next strips
    uint32_t qcur = 0, qn = Q[0];                   // query word; the first lane's next one
    uint32_t row[8];                                // first lane: the row above, H one column back | E << 16
#pragma unroll
    for (int kk = 0; kk < 8; kk++) row[kk] = top_row(kk);
    if (COOP && wv > 0 && npass > 0) rec_load(coop_row(0, 0), row);
    uint32_t lutL[9], lutH[9], oH[8], carry = 0, qlast = 0;
    pk16x2 h[9], f[9], hb = zero2;                  // hb: bottom row's H one column back
#pragma unroll
    for (int m = 0; m < 9; m++) { h[m] = zero2; f[m] = zero2; lutL[m] = 0; lutH[m] = 0; }
#pragma unroll
    for (int kk = 0; kk < 8; kk++) oH[kk] = 0;
    uint32_t best2 = 0, bpos2 = 0, col2 = 0, low2 = 0;   // per half: ranked best of the strip, its column; column; best below it
    int32_t bv = 0, bs = 0x7FFFFFFF, bc = 0x7FFFFFFF, br = 0;

    // a finished strip's maximum (e) joins the pair's
    auto strip_done = [&](int32_t s, uint32_t e, int32_t col, uint32_t low) {
        if (MODE != TB_LOCAL) return;
        if (SECOND) d.wv_strip[(size_t)strip0 + (uint32_t)s] = e | low << 16;
        const int32_t v = (int32_t)(e >> 3);
        if (v > bv) { bv = v; bs = s; bc = col; br = 7 - (int32_t)(e & 7u); }
    };

    for (int32_t it = 0; it < its; it++, out += WV_ITER) {
        j++;
        const bool ended = j == QW && k >= 0, wrap = j == P;
        if (ended) {
            const int32_t sL = strip_of(k);
            if (sL < strips) strip_done(sL, best2 & 0xFFFFu, (int32_t)(bpos2 & 0xFFFFu), low2 & 0xFFFFu);
        }
        if (wrap) {   // the low strip of the next pass
            j = 0;
            k++;
            const int32_t sL = strip_of(k);
#pragma unroll
            for (int m = 1; m < 9; m++) {
                lutL[m] = lut16[(gL >> (32 - 4 * m)) & 15u];
                h[m] = set_lo(h[m], MODE == TB_LOCAL ? 0 : hl(8 * sL + m));
                f[m] = set_lo(f[m], MODE == TB_LOCAL ? 0 : NEG16);
            }
            hb = set_lo(hb, MODE == TB_LOCAL ? 0 : hl(8 * sL + 8));
            best2 &= 0xFFFF0000u;
            low2 &= 0xFFFF0000u;
            col2 &= 0xFFFF0000u;
            gL = T[min(sL + 2 * GW * NW, TW - 1)];
        }
        qcur = from_above<GW>(qn, qcur);
        const uint32_t qodd = qcur & 0x07070707u, qeven = qcur & 0x70707070u;   // classes, neighbours cleared
        // the first lane's next word
        const int32_t jn = j + 1 == P ? 0 : j + 1, kn = j + 1 == P ? k + 1 : k;
        const bool next_row = l == 0 && NW * kn + wv > 0 && kn < npass && jn < QW;
        const uint32_t *above = out + (ptrdiff_t)(GW - P) * (ptrdiff_t)WV_ITER + 3 * WV_STREAM + (GW - 1) * 8;   // !COOP
        if (l == 0) qn = Q[min(jn, QW - 1)];
        uint32_t w[8];
#pragma unroll
        for (int m = 1; m < 9; m++) w[m - 1] = pack_lo(as_u32(h[m]), as_u32(f[m]));
        rec_store(out + WV_LEFT * WV_STREAM, w);
#pragma unroll
        for (int kk = 0; kk < 8; kk++) {
            const uint32_t q = kk < 7 ? ((kk & 1) ? qodd : qeven) >> (26 - 4 * kk) : qodd << 2;
            const uint32_t tin = from_above<GW>(row[kk], oH[kk]);
            pk16x2 e = as_pk(pack_hi(tin, carry)), p = as_pk(pack_lo(tin, carry));
            pk16x2 colmax = zero2;
#pragma unroll
            for (int m = 1; m < 9; m++) {
                const uint32_t sl = (uint32_t)__builtin_amdgcn_sbfe(lutL[m], q, 4);
                const uint32_t sh = (uint32_t)__builtin_amdgcn_sbfe(lutH[m], qlast, 4);
                const pk16x2 tmp = p + as_pk(pack_lo(sl, sh));
                pk16x2 hm = pmax(pmax(tmp, f[m]), e);
                if (MODE == TB_LOCAL) hm = pmax(hm, zero2);
                const pk16x2 tt = tmp - gapoe2;
                f[m] = pmax(tt, f[m] - gape2);   // the reference's E and F, negative ones too: a traceback reads them
                e = pmax(tt, e - gape2);
                if (MODE == TB_LOCAL) colmax = pmaxu(colmax, prank(hm, (uint32_t)(8 - m) * 0x00010001u));
                p = h[m];
                h[m] = hm;
            }
            qlast = q;
            carry = pack_lo(as_u32(hb), as_u32(e));
            w[kk] = carry;
            oH[(kk + 7) & 7] = pack_hi(as_u32(hb), as_u32(e));
            hb = h[8];
            if (MODE == TB_LOCAL) {
                // a half's best moves to this column when its h beats the best's h
                if (SECOND)
                    low2 = as_u32(pmaxu(as_pk(low2), as_pk(as_u32(colmax) & nonzero_mask(psubsat(as_pk(best2 & 0xFFF8FFF8u), colmax)))));
                const uint32_t up = nonzero_mask(psubsat(colmax, as_pk(best2 | 0x00070007u)));
                best2 = bits_of(up, as_u32(colmax), best2);
                bpos2 = bits_of(up, col2, bpos2);
                col2 += 0x00010001u;
                if (SECOND) asm volatile("" : "+v"(best2), "+v"(bpos2), "+v"(low2));
                else asm volatile("" : "+v"(best2), "+v"(bpos2));
            }
            __builtin_amdgcn_sched_barrier(0);   // one column at a time (else the compiler holds several)
            if (kk == 0) {
                // the high strip's last column of the word before
                if (it > 0) rec_store(out - WV_ITER + 3 * WV_STREAM, oH);
                if (ended && sH < strips) strip_done(sH, best2 >> 16, (int32_t)(bpos2 >> 16), low2 >> 16);
                if (wrap) {   // and its strip of the next pass, from the next step on
                    sH = strip_of(k) + 1;
#pragma unroll
                    for (int m = 1; m < 9; m++) {
                        lutH[m] = lut16[(gH >> (32 - 4 * m)) & 15u];
                        h[m] = set_hi(h[m], MODE == TB_LOCAL ? 0 : hl(8 * sH + m));
                        f[m] = set_hi(f[m], MODE == TB_LOCAL ? 0 : NEG16);
                    }
                    hb = set_hi(hb, MODE == TB_LOCAL ? 0 : hl(8 * sH + 8));
                    best2 &= 0xFFFFu;
                    low2 &= 0xFFFFu;
                    col2 &= 0xFFFFu;
                    gH = T[min(sH + 2 * GW * NW, TW - 1)];
                }
                uint32_t v[8];
#pragma unroll
                for (int m = 1; m < 9; m++) v[m - 1] = pack_hi(as_u32(h[m]), as_u32(f[m]));
                rec_store(out + (WV_LEFT + 1) * WV_STREAM, v);
            }
            if (kk == 3 || kk == 7) {
                // The first lane's next row above, stored P - GW - 1 iterations
                // ago by the last lane: two and more, and all but the newest
                // eight of the wave's accesses hold it (an iteration issues
                // eight stores and more).
                if (COOP && kk == 3) {
                    __hip_atomic_store(&sh.done[wv], it + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
                    above = coop_row(kn, jn);
                } else if (kk == 3) {
                    if (slack) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
                    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                }
                const int o = kk - 3;
                if (next_row) {
                    const u32x4 a = reinterpret_cast<const u32x4 *>(above)[o / 4];
                    row[o] = a.x; row[o + 1] = a.y; row[o + 2] = a.z; row[o + 3] = a.w;
                } else {
#pragma unroll
                    for (int i = 0; i < 4; i++) row[o + i] = NW * kn + wv == 0 ? top_row(8 * jn + o + i) : 0u;
                }
            }
        }
        rec_store(out + WV_BOTTOM * WV_STREAM, w);
    }

    if (MODE == TB_GLOBAL) {   // the score: row tlen, column qlen of the last tile, rebuilt (src/kernels/global.h:98-103, 299)
        if (COOP) __syncthreads();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        if (!ok || l != 0 || wv != 0) return;
        const uint2 at = d.wv_at[pr];
        uint32_t top[8], left[8];
        rec_load(wv_tile(d, at, QW, TW - 1, QW - 1, WV_LEFT), left);
        if (TW > 1) rec_load(wv_tile(d, at, QW, TW - 2, QW - 1, WV_BOTTOM), top);
        int32_t hh[9], ff[9], score = 0;
        const uint32_t tw = T[TW - 1], qw = Q[QW - 1];
#pragma unroll
        for (int m = 1; m < 9; m++) { hh[m] = sx16(left[m - 1]); ff[m] = (int32_t)left[m - 1] >> 16; }
        const int32_t want = (qlen - 1) & 7, rowsel = 8 - (8 * TW - tlen);
#pragma unroll
        for (int kk = 0; kk < 8; kk++) {
            const uint32_t tin = TW > 1 ? top[kk] : top_row(8 * (QW - 1) + kk);
            int32_t e = (int32_t)tin >> 16, p = sx16(tin);
            const uint32_t q = kk < 7 ? (qw >> (26 - 4 * kk)) & 0x1Cu : (qw << 2) & 0x1Cu;
#pragma unroll
            for (int m = 1; m < 9; m++) {
                const int32_t tmp = p + __builtin_amdgcn_sbfe(lut16[(tw >> (32 - 4 * m)) & 15u], q, 4);
                const int32_t hm = max(max(tmp, ff[m]), e), t = tmp - c.gapoe;
                ff[m] = max(t, ff[m] - gape);
                e = max(t, e - gape);
                p = hh[m];
                hh[m] = hm;
                if (kk == want && m == rowsel) score = hm;
            }
        }
        d.score[pr] = score;
        return;
    }
    // merge the group's lanes in the reference's order
#pragma unroll
    for (int off = GW / 2; off > 0; off >>= 1) {
        const int32_t ov = __shfl_xor(bv, off), os = __shfl_xor(bs, off), oc = __shfl_xor(bc, off), orow = __shfl_xor(br, off);
        if (ov > bv || (ov == bv && (os < bs || (os == bs && oc < bc)))) { bv = ov; bs = os; bc = oc; br = orow; }
    }
    if (COOP) {   // and the block's waves in the same way
        if (lane == 0) { sh.end[wv][0] = bv; sh.end[wv][1] = bs; sh.end[wv][2] = bc; sh.end[wv][3] = br; }
        __syncthreads();
        for (int w = 0; w < NW; w++) {
            const int32_t *o = sh.end[w];
            if (o[0] > bv || (o[0] == bv && (o[1] < bs || (o[1] == bs && o[2] < bc)))) { bv = o[0]; bs = o[1]; bc = o[2]; br = o[3]; }
        }
    }
    if (ok && l == 0 && wv == 0) {
        d.score[pr] = bv;
        d.qend[pr] = bv > 0 ? bc : 0;
        d.tend[pr] = bv > 0 ? bs * 8 + br : 0;
    }
}

// Launch: a block for each of the first d.wave_coop sorted slots, then a wave for
// each of the next d.wave64, for two of the next d.wave32, four of the next
// d.wave16 and sixteen of the others, four waves a block.
template <int MODE, bool SECOND>
__global__ __launch_bounds__(WV_WAVES * WAVE) void k_wave_tb(G2Dev d, G2Scores c) {
    const uint32_t census = d.aux[0];
    if (!census_fast(census)) return;   // the lane kernels take this batch
    __shared__ WvShared sh;
    if (threadIdx.x < 16)
        sh.lut16[threadIdx.x] = MODE == TB_GLOBAL ? score_lut<true>(c, 0, census, threadIdx.x)
                                                  : score_lut(c, c.has_np ? -c.np : 0, census, threadIdx.x);
    __syncthreads();
    const uint32_t b = blockIdx.x, s0 = d.wave_coop, s1 = s0 + d.wave64, s2 = s1 + d.wave32, s3 = s2 + d.wave16;
    if (b < s0) {
        wv_pairs<MODE, SECOND, 64, true>(d, c, sh, b, s0);
        return;
    }
    const uint32_t u = WV_WAVES * (b - s0) + __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const uint32_t u1 = d.wave64, u2 = u1 + (d.wave32 + 1) / 2, u3 = u2 + (d.wave16 + 3) / 4, u4 = u3 + (d.n - s3 + 15) / 16;
    if (u < u1) wv_pairs<MODE, SECOND, 64, false>(d, c, sh, s0 + u, s1);
    else if (u < u2) wv_pairs<MODE, SECOND, 32, false>(d, c, sh, s1 + 2 * (u - u1), s2);
    else if (u < u3) wv_pairs<MODE, SECOND, 16, false>(d, c, sh, s2 + 4 * (u - u2), s3);
    else if (u < u4) wv_pairs<MODE, SECOND, 4, false>(d, c, sh, s3 + 16 * (u - u3), d.n);
}

// Second best from the strips' records (the header's rule).  A strip's record:
// its ranked maximum, and the largest ranked column maximum below the strip's
// maximum so far.  With M the maximum of the strips above: a strip whose
// maximum is below M has that maximum as its candidate; any other has no
// candidate above its maximum less one, and at least its record's lower bound.
// A candidate's key: h, then the earlier strip, then the rank's row.
__device__ __forceinline__ uint64_t second_key(uint32_t rank, int32_t strip) {
    return rank < 8 ? 0 : (uint64_t)(rank >> 3) << 32 | (uint32_t)(0x1FFFFFFF - strip) << 3 | (rank & 7u);
}

// One pair a lane: the candidates that need no cells, and the strips that do
// (all those whose maximum exceeds every known candidate), appended to
// wv_item by wave.
__global__ __launch_bounds__(WAVE) void k_second_scan(G2Dev d) {
    if (!census_fast(d.aux[0])) return;
    const uint32_t slot = blockIdx.x * WAVE + threadIdx.x, lane = threadIdx.x;
    const int32_t TW = slot < d.n ? dregs(d.tlen[d.perm[slot]]) : 0;
    const uint32_t *rec = d.wv_strip + (slot < d.n ? d.wv_sec[slot] : 0);   // the DP left its place there
    int32_t run = 0, bound = 0;
    for (int32_t s = 0; s < TW; s++) {
        const uint32_t r = rec[s];
        const int32_t mx = (int32_t)((r & 0xFFFFu) >> 3);
        bound = max(bound, mx < run ? mx : (int32_t)(r >> 19));
        run = max(run, mx);
    }
    uint64_t key = 0;
    uint32_t items = 0;
    run = 0;
    for (int32_t s = 0; s < TW; s++) {
        const uint32_t r = rec[s];
        const int32_t mx = (int32_t)((r & 0xFFFFu) >> 3);
        if (mx < run) {
            const uint64_t k = second_key(r & 0xFFFFu, s);
            if (k > key) key = k;
        } else if (mx > bound) {
            items++;
        }
        run = max(run, mx);
    }
    if (slot < d.n) d.wv_sec[slot] = key;
    uint32_t at = items;
#pragma unroll
    for (uint32_t off = 1; off < WAVE; off <<= 1) {
        const uint32_t o = __shfl_up(at, off);
        at += lane >= off ? o : 0u;
    }
    uint32_t base = 0;
    if (lane == WAVE - 1 && at) base = atomicAdd(&d.aux[5], at);
    at += __shfl(base, WAVE - 1) - items;
    run = 0;
    for (int32_t s = 0; s < TW && items; s++) {
        const int32_t mx = (int32_t)((rec[s] & 0xFFFFu) >> 3);
        if (mx >= run && mx > bound) {
            d.wv_item[at++] = make_uint2(slot, (uint32_t)s << 13 | (uint32_t)run);   // run <= 8191
            items--;
        }
        run = max(run, mx);
    }
}

// The strips of wv_item, two a lane in 16-bit halves: the ranked h of cells
// below the running maximum, which starts at the strips' above.
__global__ __launch_bounds__(WAVE) void k_second_strips(G2Dev d, G2Scores c) {
    const uint32_t census = d.aux[0];
    if (!census_fast(census)) return;
    __shared__ uint32_t lut16[16];
    if (threadIdx.x < 16) lut16[threadIdx.x] = score_lut(c, c.has_np ? -c.np : 0, census, threadIdx.x);
    __syncthreads();
    const uint32_t count = d.aux[5];
    const pk16x2 gapoe2 = {(short)c.gapoe, (short)c.gapoe}, gape2 = {(short)c.gape, (short)c.gape}, zero2 = {0, 0};
    struct Item {
        const uint32_t *q, *above;   // query words; the strip above's bottom records, a word every WV_ITER dwords (null: none)
        uint32_t t, slot;
        int32_t QW, strip, run;
    };
    for (uint32_t w = blockIdx.x; w * 128 < count; w += gridDim.x) {
        Item it[2];
        bool ok[2];
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const uint32_t i = w * 128 + 64 * k + threadIdx.x;
            ok[k] = i < count;
            const uint2 v = d.wv_item[ok[k] ? i : count - 1];
            const uint32_t pr = d.perm[v.x];
            it[k].slot = v.x;
            it[k].strip = (int32_t)(v.y >> 13);
            it[k].run = (int32_t)(v.y & 0x1FFFu);
            it[k].QW = dregs(d.qlen[pr]);
            it[k].q = d.pq + (d.qoff[pr] >> 3);
            it[k].t = d.pt[(d.toff[pr] >> 3) + it[k].strip];
            it[k].above = it[k].strip > 0 ? wv_tile(d, d.wv_at[pr], it[k].QW, it[k].strip - 1, 0, WV_BOTTOM) : nullptr;
        }
        const int32_t QWm = max(it[0].QW, it[1].QW);
        uint32_t lutA[9], lutB[9];
        pk16x2 h[9], f[9];
#pragma unroll
        for (int m = 1; m < 9; m++) {
            lutA[m] = lut16[(it[0].t >> (32 - 4 * m)) & 15u];
            lutB[m] = lut16[(it[1].t >> (32 - 4 * m)) & 15u];
            h[m] = zero2;
            f[m] = zero2;
        }
        pk16x2 run = as_pk(pack_lo((uint32_t)it[0].run, (uint32_t)it[1].run));
        uint32_t sec2 = 0;
        uint32_t nA[8], nB[8], nqA, nqB;
        auto fetch = [&](int32_t j) {   // past a half's last word: its last (those cells are masked)
            const int32_t ja = min(j, it[0].QW - 1), jb = min(j, it[1].QW - 1);
            nqA = it[0].q[ja];
            nqB = it[1].q[jb];
#pragma unroll
            for (int kk = 0; kk < 8; kk++) { nA[kk] = 0; nB[kk] = 0; }
            if (it[0].above) rec_load(it[0].above + (size_t)ja * WV_ITER, nA);
            if (it[1].above) rec_load(it[1].above + (size_t)jb * WV_ITER, nB);
        };
        fetch(0);
        for (int32_t j = 0; j < QWm; j++) {
            const uint32_t rA = nqA, rB = nqB;
            const uint32_t valid = (j < it[0].QW ? 0xFFFFu : 0u) | (j < it[1].QW ? 0xFFFF0000u : 0u);
            uint32_t pe[8], ph[8];
#pragma unroll
            for (int kk = 0; kk < 8; kk++) { pe[kk] = pack_hi(nA[kk], nB[kk]); ph[kk] = pack_lo(nA[kk], nB[kk]); }
            fetch(j + 1);
#pragma unroll
            for (int kk = 0; kk < 8; kk++) {
                const uint32_t qa = kk < 7 ? (rA >> (26 - 4 * kk)) & 0x1Cu : (rA << 2) & 0x1Cu;
                const uint32_t qb = kk < 7 ? (rB >> (26 - 4 * kk)) & 0x1Cu : (rB << 2) & 0x1Cu;
                pk16x2 e = as_pk(pe[kk]), p = as_pk(ph[kk]), colsec = zero2;
#pragma unroll
                for (int m = 1; m < 9; m++) {
                    const uint32_t sa = (uint32_t)__builtin_amdgcn_sbfe(lutA[m], qa, 4);
                    const uint32_t sb = (uint32_t)__builtin_amdgcn_sbfe(lutB[m], qb, 4);
                    const pk16x2 tmp = p + as_pk(pack_lo(sa, sb));
                    const pk16x2 hm = pmax(pmax(pmax(tmp, f[m]), e), zero2);
                    const pk16x2 tt = tmp - gapoe2;
                    f[m] = pmax(tt, f[m] - gape2);
                    e = pmax(tt, e - gape2);
                    const uint32_t below = __builtin_amdgcn_perm(0u, as_u32(hm - run), 0x09090808u);   // sign masks
                    colsec = pmaxu(colsec, as_pk(as_u32(prank(hm, (uint32_t)(8 - m) * 0x00010001u)) & below));
                    run = pmax(run, hm);
                    p = h[m];
                    h[m] = hm;
                }
                const uint32_t up = nonzero_mask(psubsat(colsec, as_pk(sec2 | 0x00070007u))) & valid;
                sec2 = bits_of(up, as_u32(colsec), sec2);
                asm volatile("" : "+v"(sec2));
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        const uint64_t ka = second_key(sec2 & 0xFFFFu, it[0].strip), kb = second_key(sec2 >> 16, it[1].strip);
        if (ok[0] && ka) atomicMax(reinterpret_cast<unsigned long long *>(&d.wv_sec[it[0].slot]), (unsigned long long)ka);
        if (ok[1] && kb) atomicMax(reinterpret_cast<unsigned long long *>(&d.wv_sec[it[1].slot]), (unsigned long long)kb);
    }
}

__global__ __launch_bounds__(256) void k_second_out(G2Dev d) {
    if (!census_fast(d.aux[0])) return;
    const uint32_t slot = blockIdx.x * blockDim.x + threadIdx.x;
    if (slot >= d.n) return;
    const uint32_t pr = d.perm[slot], low = (uint32_t)d.wv_sec[slot];
    const int32_t sec = (int32_t)(d.wv_sec[slot] >> 32);
    d.s_score[pr] = sec;
    d.s_tend[pr] = sec > 0 ? 8 * (0x1FFFFFFF - (int32_t)(low >> 3)) + 7 - (int32_t)(low & 7u) : 0;
    d.s_qend[pr] = d.score[pr] > 0 ? 8 * dregs(d.qlen[pr]) - 1 : 0;   // compares with the best (src/kernels/local_kernel_template.h:162)
}

// ------------------------------------------------------------ traceback ----
// gasal_get_tb<T> (src/kernels/get_tb.h:4-149), one wave per pair: each lane
// rebuilds one tile of the diagonal the path is about to follow (from the
// current tile (s, w): (s - a, w - b) with |a - b| <= 1, 21 tiles along the
// diagonal), then the wave walks the path through those tiles until it leaves
// them.  The walk's state is wave-uniform, so it runs on the scalar unit, tiles
// read out of their lanes; a stretch of matches inside a tile is one step (the
// first other cell on the diagonal, from the tile's 64-bit mask).  One lane per
// pair (k_get_tb) waits for a tile's records and rebuilds it at every tile it
// enters, 1.4 us per path cell: the walk of 64 pairs of 100-300 bases took 486 us
// so, and takes 53; of 50,000 pairs of 50-5000 bases 8.7 ms, and takes 1.6.
// Bound: of a lone pair the records' latency and a tile's recompute, once per 21
// tiles of the diagonal; of many the two tiles in three rebuilt off the path.
template <bool LOCALT>
__global__ __launch_bounds__(WAVE) void k_wave_walk(G2Dev d, G2Scores c) {
    const uint32_t census = d.aux[0];
    if (!census_fast(census)) return;
    __shared__ uint32_t lut16[16];
    if (threadIdx.x < 16)
        lut16[threadIdx.x] = LOCALT ? score_lut(c, c.has_np ? -c.np : 0, census, threadIdx.x)
                                    : score_lut<true>(c, 0, census, threadIdx.x);
    __syncthreads();
    auto uniform = [](uint32_t v) -> uint32_t { return __builtin_amdgcn_readfirstlane(v); };
    const int32_t lane = (int32_t)threadIdx.x;
    const uint32_t pr = uniform(d.perm[blockIdx.x]);
    const int32_t qlen = (int32_t)uniform(d.qlen[pr]), tlen = (int32_t)uniform(d.tlen[pr]);
    const int32_t QW = dregs((uint32_t)qlen), TW = dregs((uint32_t)tlen), cols = 8 * QW;
    const uint32_t *Qw = d.pq + (uniform(d.qoff[pr]) >> 3), *Tw = d.pt + (uniform(d.toff[pr]) >> 3);
    const uint2 at = make_uint2(uniform(d.wv_at[pr].x), uniform(d.wv_at[pr].y));
    uint8_t *__restrict__ cg = d.cigar + (size_t)pr * d.cigar_cap;
    int32_t i = tlen, j = qlen, total = 0, score = 0;
    if (LOCALT) {
        i = (int32_t)uniform((uint32_t)d.tend[pr]);
        j = (int32_t)uniform((uint32_t)d.qend[pr]);
        total = (int32_t)uniform((uint32_t)d.score[pr]);
    }
    int32_t n_ops = 0, op_select = 3, op_shift = 0, count = 0;
    uint32_t prev_op = 0;
    auto put = [&]() {
        if (lane == 0) cg[n_ops] = (uint8_t)(prev_op | (uint32_t)(count << 2));
        n_ops++;
    };
    int32_t s0 = -1, w0 = -1;   // the tiles' first strip and word
    // this lane's tile: diagonal step lane / 3, on, below or right of the diagonal
    const int32_t my_a = lane / 3 + (lane % 3 == 1), my_b = lane / 3 + (lane % 3 == 2);
    uint32_t words[8];          // its columns' nibbles, and a bit per cell that is no match: column * 8 + 7 - row
    uint32_t other_lo = 0, other_hi = 0;
#pragma unroll
    for (int k = 0; k < 8; k++) words[k] = 0;
    bool done = !(i >= 0 && j >= 0);
    while (!done) {
        // a column index of 8 QW (GLOBAL start at Lq == 8 QW) is column 0 of
        // the next strip (src/kernels/get_tb.h:50); cells past the strips read as 0
        const bool wrapped = !LOCALT && j >= cols;
        const int32_t strip = (i >> 3) + (wrapped ? 1 : 0), word = (wrapped ? j - cols : j) >> 3;
        const bool in = LOCALT || strip < TW;
        uint32_t ch[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        uint64_t other = 0;
        if (in) {
            const int32_t a = s0 - strip, b = w0 - word;
            int32_t idx = 3 * min(a, b) + (a > b ? 1 : (a < b ? 2 : 0));
            if (s0 < 0 || min(a, b) < 0 || abs(a - b) > 1 || idx >= WAVE) {
                s0 = strip;
                w0 = word;
                idx = 0;
                const int32_t s = s0 - my_a, w = w0 - my_b;
                if (s >= 0 && w >= 0) {
                    uint32_t top[8], left[8], lut[8];
                    if (s > 0) rec_load(wv_tile(d, at, QW, s - 1, w, WV_BOTTOM), top);
                    rec_load(wv_tile(d, at, QW, s, w, WV_LEFT), left);
                    const uint32_t qword = Qw[w], tword = Tw[s];
                    if (s == 0) {
#pragma unroll
                        for (int k = 0; k < 8; k++)
                            top[k] = LOCALT ? 0u : pk16(8 * w + k < 2 ? 0 : -(c.gapo + c.gape * (8 * w + k - 1)), NEG16);
                    }
#pragma unroll
                    for (int m = 0; m < 8; m++) lut[m] = lut16[(tword >> (28 - 4 * m)) & 15u];
                    ck_tile<LOCALT>(top, left, qword, lut, c, words);
                    other_lo = 0;
                    other_hi = 0;
#pragma unroll
                    for (int k = 0; k < 8; k++) {
                        uint32_t z = (words[k] | words[k] >> 1) & 0x11111111u;   // source not 0
                        z = (z | z >> 3) & 0x03030303u;
                        z = (z | z >> 6) & 0x000F000Fu;
                        z = (z | z >> 12) & 0xFFu;
                        if (k < 4) other_lo |= z << (8 * k);
                        else other_hi |= z << (8 * (k - 4));
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < 8; k++) ch[k] = (uint32_t)__builtin_amdgcn_readlane((int)words[k], idx);
            other = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)other_hi, idx) << 32 |
                    (uint32_t)__builtin_amdgcn_readlane((int)other_lo, idx);
        }
        while (true) {
            const int32_t c7 = (wrapped ? j - cols : j) & 7, r7 = i & 7;
            const int32_t i0 = i, j0 = j;
            if (in && !wrapped && op_select == 3) {   // matches ahead in this tile
                const int32_t bit = 8 * c7 + 7 - r7, most = min(c7, r7) + 1;
                const uint64_t x = other & (0x8102040810204081ull >> (63 - bit)) & (~0ull << (bit - 7 * (most - 1)));
                const int32_t n = x ? ((bit - (63 - (int32_t)__builtin_clzll(x))) * 37) >> 8 : most;   // cells before x's top bit
                // LOCAL ends where the score reaches the total: not inside these
                // when they raise it and do not pass it
                const int32_t left = total - score;
                if (n > 0 && (!LOCALT || (c.match > 0 && (left <= 0 || left > n * c.match)))) {
                    if (prev_op == 0) {
                        count += n;
                        if (count > 63) {
                            const int32_t rest = count - 63;
                            count = 63;
                            put();
                            count = rest;
                        }
                    } else {
                        put();
                        prev_op = 0;
                        count = n;
                    }
                    if (LOCALT) score += n * c.match;
                    i -= n;
                    j -= n;
                    if (!(i >= 0 && j >= 0)) { done = true; break; }
                    if (((i0 ^ i) | (j0 ^ j)) & ~7) break;
                    continue;
                }
            }
            const uint32_t wcol = c7 < 4 ? (c7 < 2 ? (c7 == 0 ? ch[0] : ch[1]) : (c7 == 2 ? ch[2] : ch[3]))
                                         : (c7 < 6 ? (c7 == 4 ? ch[4] : ch[5]) : (c7 == 6 ? ch[6] : ch[7]));
            const uint32_t cell_op = (wcol >> (28 - 4 * r7)) & 15u;
            const uint32_t op = (cell_op >> op_shift) & (uint32_t)op_select;
            const uint32_t fill = op == 0 || op_select == 3 ? op : (uint32_t)op_shift;
            op_select = op == 0 || (op == 1 && op_select == 3) ? 3 : 1;
            op_shift = op_select == 3 ? 0 : ((op == 2 || op == 3) ? (int32_t)op : op_shift);
            const bool opens = prev_op != fill;
            if (count < 63 && !opens) {
                count++;
            } else {
                if (count > 0) put();
                count = 1;
            }
            if (LOCALT) {
                score += fill >= 2 ? (opens ? -c.gapoe : -c.gape) : (fill == 1 ? -c.mismatch : c.match);
                if (score == total) { done = true; break; }   // the last run keeps the op before it (get_tb.h)
            }
            prev_op = fill;
            i = fill != 3 ? i - 1 : i;   // ops 0, 1, 2 move up
            j = fill != 2 ? j - 1 : j;   // ops 0, 1, 3 move left
            if (!(i >= 0 && j >= 0)) { done = true; break; }
            if (!in || wrapped || (((i0 ^ i) | (j0 ^ j)) & ~7)) break;
        }
    }
    put();
    if (!LOCALT) {
        for (prev_op = 2; i >= 0; i -= 63) { count = min(i + 1, 63); put(); }
        for (prev_op = 3; j >= 0; j -= 63) { count = min(j + 1, 63); put(); }
    }
    if (lane == 0) {
        if (LOCALT) { d.tstart[pr] = i; d.qstart[pr] = j; }
        d.n_ops[pr] = (uint32_t)n_ops;
    }
}

}  // namespace

hipError_t g2_wave_tb_run(const G2Scores &sc, const G2Opts &op, const G2Dev &d, hipStream_t s) {
    const uint32_t narrow = d.n - d.wave_coop - d.wave64 - d.wave32 - d.wave16;
    const uint32_t waves = d.wave64 + (d.wave32 + 1) / 2 + (d.wave16 + 3) / 4 + (narrow + 15) / 16;
    const uint32_t blocks = d.wave_coop + (waves + WV_WAVES - 1) / WV_WAVES;
    if (op.algo == A_GLOBAL) {
        k_wave_tb<TB_GLOBAL, false><<<blocks, WV_WAVES * WAVE, 0, s>>>(d, sc);
    } else if (op.second) {
        k_wave_tb<TB_LOCAL, true><<<blocks, WV_WAVES * WAVE, 0, s>>>(d, sc);
        const uint32_t groups = (d.n + WAVE - 1) / WAVE;
        k_second_scan<<<groups, WAVE, 0, s>>>(d);
        k_second_strips<<<groups < 4096 ? groups : 4096, WAVE, 0, s>>>(d, sc);
        k_second_out<<<(d.n + 255) / 256, 256, 0, s>>>(d);
    } else {
        k_wave_tb<TB_LOCAL, false><<<blocks, WV_WAVES * WAVE, 0, s>>>(d, sc);
    }
    return hipGetLastError();
}

hipError_t g2_wave_walk(const G2Scores &sc, const G2Opts &op, const G2Dev &d, hipStream_t s) {
    if (op.algo == A_LOCAL) k_wave_walk<true><<<d.n, WAVE, 0, s>>>(d, sc);
    else k_wave_walk<false><<<d.n, WAVE, 0, s>>>(d, sc);
    return hipGetLastError();
}
