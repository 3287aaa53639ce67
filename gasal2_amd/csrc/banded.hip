// banded.hip -- BANDED in packed 16-bit halves, two strips a sweep.
//
// gasal_banded_tiled_kernel (src/kernels/banded.h:10-139): per 8-row strip the
// 8x8 tiles of a word range that moves one word a strip.  One lane per pair runs
// strips 2k and 2k + 1 in the low and high halves of its registers, the high
// strip one column behind the low one, under the low strip's bottom row of the
// step before.  Where a strip's range has no word of the other's, the boundary
// row passes through it unchanged; the ranges begin and end at words, so that is
// one mask per half and word.  The end is the reference's first strict maximum in
// (strip, column, row) order: cells ranked h * 8 + (7 - row), a half's best
// kept per strip.
//
// Bound: the boundary row through memory, 8 bytes read and written per column
// and sweep (500,000 rows of 270 columns outgrow the caches) -- half the bytes
// per cell of a sweep of one strip -- then packed VALU issue, 13 instructions per
// pair of cells.  Two pairs a lane in the halves, one strip a sweep, has the same
// instructions and twice the bytes: 500,000 pairs of 100-250 bases, band 32,
// 2.03 ms one pair a lane in 32 bits, 1.74 two pairs, 1.32 two strips.
#include "device.h"

namespace {

__global__ __launch_bounds__(WAVE) void k_banded_pk(G2Dev d, G2Scores c, int32_t k_band_width) {
    const uint32_t census = d.aux[0];
    if (!census_fast(census)) return;   // k_banded takes this batch
    __shared__ uint32_t lut16[16];
    if (threadIdx.x < 16) lut16[threadIdx.x] = score_lut(c, c.has_np ? -c.np : 0, census, threadIdx.x);
    __syncthreads();
    const uint32_t lane = threadIdx.x, slot = blockIdx.x * WAVE + lane;
    if (slot >= d.n) return;
    const uint32_t pr = d.perm[slot];
    const int32_t QW = dregs(d.qlen[pr]), TW = dregs(d.tlen[pr]);
    const uint32_t *Q = d.pq + (d.qoff[pr] >> 3), *T = d.pt + (d.toff[pr] >> 3);
    const int32_t q1 = max(QW - 1, 0), t1 = max(TW - 1, 0);
    const int32_t other = TW - (QW - k_band_width);                                        // :35
    uint32_t *__restrict__ bd = d.bnd + (size_t)blockIdx.x * d.bnd_cols * WAVE + lane;
    for (int32_t cc = 0; cc < 8 * QW; cc++) bd[cc * WAVE] = 0u;
    const pk16x2 gapoe2 = {(short)c.gapoe, (short)c.gapoe}, gape2 = {(short)c.gape, (short)c.gape}, zero2 = {0, 0};
    int32_t best = 0, bcol = 0, brow = 0;
    uint32_t gL = T[0], gH = T[min(1, t1)];   // target words of the next two strips
    for (int32_t s0 = 0; s0 < TW; s0 += 2) {
        // word ranges of the two strips (:83-85); empty past the target
        const int32_t a0 = max(0, s0 - other + 1), a1 = min(k_band_width + s0, QW);
        const int32_t b0 = max(0, s0 - other + 2), b1 = s0 + 1 < TW ? min(k_band_width + s0 + 1, QW) : 0;
        const int32_t first = a0 < a1 ? a0 : b0, last = max(a0 < a1 ? a1 : 0, b0 < b1 ? b1 : 0);
        uint32_t lutL[9], lutH[9];
        pk16x2 h[9], f[9], diag = zero2;   // diag: H of the row above, one column back (0 at a range's start)
#pragma unroll
        for (int m = 1; m < 9; m++) {
            lutL[m] = lut16[(gL >> (32 - 4 * m)) & 15u];
            lutH[m] = lut16[(gH >> (32 - 4 * m)) & 15u];
            h[m] = zero2;
            f[m] = zero2;
        }
        gL = T[min(s0 + 2, t1)];
        gH = T[min(s0 + 3, t1)];
        if (first >= last) continue;
        uint32_t carry = 0, qlast = 0;               // low strip's bottom (H | E << 16), its query class, previous step
        uint32_t best2 = 0, bcol2 = 0;               // per half: ranked best of the strip, its step
        uint32_t next[8], nq;
        auto fetch = [&](int32_t j) {                // the row above and the query word, one word ahead
            nq = Q[min(j, q1)];
#pragma unroll
            for (int kk = 0; kk < 8; kk++) next[kk] = bd[(8 * j + kk) * WAVE];   // the slice has a spare word
        };
        fetch(first);
        uint32_t high_before = 0;
        for (int32_t j = first;; j++) {
            const uint32_t q8 = nq;
            uint32_t top[8];
#pragma unroll
            for (int kk = 0; kk < 8; kk++) top[kk] = next[kk];
            if (j < last) fetch(j + 1);
            const uint32_t low = j >= a0 && j < a1 ? 0xFFFFu : 0u, high = j >= b0 && j < b1 ? 0xFFFF0000u : 0u;
            const uint32_t low_all = low | low << 16, high_all = high | high >> 16;
            auto step = [&](int kk, uint32_t q, uint32_t high_now, uint32_t high_row) {
                pk16x2 e = as_pk(pack_hi(top[kk], carry)), p = diag;
                diag = as_pk(pack_lo(top[kk], carry));
                pk16x2 open = diag - gapoe2, colmax = zero2;
#pragma unroll
                for (int m = 1; m < 9; m++) {                                              // :100-115
                    // E and F open from H and are held as max(E, 0) and max(F, 0)
                    // (saturating extensions): H needs no max with 0
                    const uint32_t sl = (uint32_t)__builtin_amdgcn_sbfe(lutL[m], q, 4);
                    const uint32_t sh = (uint32_t)__builtin_amdgcn_sbfe(lutH[m], qlast, 4);
                    const pk16x2 tmp = p + as_pk(pack_lo(sl, sh));
                    f[m] = pmax(h[m] - gapoe2, psubsat(f[m], gape2));
                    e = pmax(open, psubsat(e, gape2));
                    const pk16x2 hm = pmax(pmax(tmp, f[m]), e);
                    colmax = pmaxu(colmax, prank(hm, (uint32_t)(8 - m) * 0x00010001u));
                    open = hm - gapoe2;
                    p = h[m];
                    h[m] = hm;
                }
                qlast = q;
                const uint32_t outH = pack_hi(as_u32(h[8]), as_u32(e)), outL = pack_lo(as_u32(h[8]), as_u32(e));
                if (kk > 0 || j > first) bd[(8 * j + kk - 1) * WAVE] = bits_of(high_row, outH, carry);
                carry = bits_of(low_all, outL, top[kk]);
                const uint32_t up = nonzero_mask(psubsat(colmax, as_pk(best2 | 0x00070007u))) & (low | high_now);
                best2 = bits_of(up, as_u32(colmax), best2);
                bcol2 = bits_of(up, (uint32_t)(8 * j + kk) * 0x00010001u, bcol2);
                asm volatile("" : "+v"(best2), "+v"(bcol2));
                __builtin_amdgcn_sched_barrier(0);   // one column at a time
            };
            step(0, (q8 >> 26) & 0x1Cu, high_before, high_before | high_before >> 16);
            if (j == last) break;
            // the high strip starts at the next step: its column -1
            const uint32_t keep = j > b0 ? 0xFFFFFFFFu : 0xFFFFu;
            diag = as_pk(as_u32(diag) & keep);
#pragma unroll
            for (int m = 1; m < 9; m++) { h[m] = as_pk(as_u32(h[m]) & keep); f[m] = as_pk(as_u32(f[m]) & keep); }
#pragma unroll
            for (int kk = 1; kk < 8; kk++)
                step(kk, kk < 7 ? (q8 >> (26 - 4 * kk)) & 0x1Cu : (q8 << 2) & 0x1Cu, high, high_all);
            high_before = high;
        }
        const int32_t vL = (int32_t)((best2 & 0xFFFFu) >> 3), vH = (int32_t)(best2 >> 19);
        if (vL > best) { best = vL; bcol = (int32_t)(bcol2 & 0xFFFFu); brow = 8 * s0 + 7 - (int32_t)(best2 & 7u); }
        if (vH > best) { best = vH; bcol = (int32_t)(bcol2 >> 16) - 1; brow = 8 * s0 + 15 - (int32_t)((best2 >> 16) & 7u); }
    }
    d.score[pr] = best;
    d.qend[pr] = bcol;
    d.tend[pr] = brow;
}

}  // namespace

hipError_t g2_banded_packed(const G2Scores &sc, const G2Opts &op, const G2Dev &d, hipStream_t s) {
    k_banded_pk<<<(d.n + WAVE - 1) / WAVE, WAVE, 0, s>>>(d, sc, op.k_band >> 3);   // src/gasal_align.h:80
    return hipGetLastError();
}
