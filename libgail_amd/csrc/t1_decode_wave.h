// EBCOT Tier-1 decoding of one code-block by a whole wave (ISO/IEC 15444-1 Annexes C.3 and D,
// no mode switches).
//
// Everything that is not the arithmetic decoder's serial chain is done for all columns at once:
// lane x (and x + 32, the same values) holds column x as 32-bit row masks (t1_cm_masks.h). For a
// stripe this side forms which samples the pass codes and their contexts as they are now, one
// word per column.
//
// In significance propagation and cleanup the chain walks the columns on scalar registers and
// decodes until a sample becomes significant: only then do contexts change, and the stripe's
// words are formed again for the samples the scan has not reached. In magnitude refinement
// nothing changes on the way: the stripe's decisions are listed in scan order and made four at
// a time in vector registers (the same values in every lane), where independent operations
// follow each other in 4 cycles and a decision takes no branch.
//
// Decoded bits are kept as one row mask per bit-plane (LDS); the reconstruction words
// (t1_dec.cpp:85-97, 117-127: twice the magnitude so far plus the mid-point of the planes not
// decoded, sign in bit 31) are formed from them at the end and stored once.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "t1_cm_masks.h"
#include "t1_wave_mq.h"

namespace gail_amd {

constexpr uint32_t kDecRun = (17u + 1u) << 2;  // a column in run-length mode

// Inclusive prefix sum over each half-wave.
__device__ __forceinline__ uint32_t dw_scan(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, false);  // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, false);  // row_shr:2
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, false);  // row_shr:4
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, false);  // row_shr:8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false);  // row_bcast:15, rows 1, 3
    return v;
}

// Decodes the first `passes` coding passes of a w x h block (1..32 each) of orientation
// `orient` with nbps magnitude bit-planes (1..30) and stores its words (row pitch `stride`).
// pack: in LDS, for each set of rows of a stripe the rows in order, a byte each, 0x0C (zero, as a
// byte selector) past the last. sign_lut: in LDS, by the left, right, upper and lower neighbour's
// two bits (significant, negative) the sign context + 1 << 1 | flip (build_sign_table).
__device__ __forceinline__ void t1_decode_wave(WaveMq& mq, uint32_t w, uint32_t h, uint32_t orient, uint32_t nbps,
                                               uint32_t passes, uint32_t* words, uint32_t stride, const uint32_t* pack,
                                               const uint8_t* sign_lut) {
    const uint32_t lane = threadIdx.x & 63u, x = lane & 31u;
    const bool hl = orient == 1u, hh = orient == 3u;
    const uint32_t valid = x < w ? (h == 32u ? 0xFFFFFFFFu : (1u << h) - 1u) : 0u;
    auto left = [&](uint32_t v) {  // the column to the left / right; zero at the block's edges
        const uint32_t r = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x138, 0xF, 0xF, true);
        return x == 0u ? 0u : r;
    };
    auto right = [&](uint32_t v) {
        const uint32_t r = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x130, 0xF, 0xF, true);
        return x == 31u ? 0u : r;
    };
    // rows r0..r0+3 of a mask as bit 0 of four bytes
    auto bytes = [](uint32_t m, uint32_t r0) {
        uint32_t t = __umul24((m >> r0) & 0xFu, 0x204081u) & 0x01010101u;
        asm("" : "+v"(t));  // the product stays a 24-bit one
        return t;
    };
    mq.init();
    uint32_t S = 0, G = 0, V = 0, R = 0;  // significant, negative, coded in this plane's first pass, refined before
    uint32_t B = 0, Q = 0;                // this plane's bits, samples it has coded a bit of
    uint32_t plane = 0, type = 2;         // 0 significance propagation, 1 magnitude refinement, 2 cleanup
    if (passes > 3u * nbps - 2u) passes = 3u * nbps - 2u;
    for (uint32_t pass = 0; pass < passes; ++pass) {
        for (uint32_t r0 = 0; r0 < h; r0 += 4u) {
            uint32_t rest = 15u;  // rows the scan has not passed
            for (;;) {
                // What the pass codes of the stripe and in which contexts: a byte per coded row
                // ((context + 1) << 2 | row), lowest row first, no gaps; context 17 alone:
                // run-length mode.
                const uint32_t SL = left(S), SR = right(S);
                const uint32_t any = neighbour_any(S, SL, SR);
                if (type == 1u) {
                    // D.3.3: samples significant before this plane's first pass; context 16 if
                    // refined before, else 15 if a neighbour is significant, else 14
                    const uint32_t todo = ((S & ~V) >> r0) & 15u;
                    uint32_t word = (bytes(R, r0) * 17u) | (bytes(~R, r0) * 15u);
                    word += bytes(any & ~R, r0);
                    word = __builtin_amdgcn_perm(0u, (word << 2) | 0x03020100u, pack[todo]);
                    // the decisions in scan order, then neutral ones
                    const uint32_t have = (uint32_t)__popc(todo);
                    const uint32_t upto = dw_scan(have), from = upto - have;
                    const uint32_t total = dw_lane(upto, 31u);
                    if (total == 0u) break;
                    uint8_t* const list = (uint8_t*)mq.ws->list;
#pragma unroll
                    for (uint32_t j = 0; j < 4u; ++j)
                        *(j < have ? list + from + j : mq.ws->junk + lane) = (uint8_t)(word >> (8u * j));
                    if (x < 8u) list[total + x] = 0u;
                    mq.refine(total);
                    // the lane's bits from the list's, then to their rows
                    const uint8_t* const bits = mq.ws->bits + (from >> 2);
                    const uint32_t mine = ((uint32_t)bits[0] | ((uint32_t)bits[1] << 4)) >> (from & 3u);
                    uint32_t rows = 0;
#pragma unroll
                    for (uint32_t k = 0; k < 4u; ++k)
                        rows |= ((mine >> __popc(todo & ((1u << k) - 1u))) & 1u) << k;
                    B |= (rows & todo) << r0;
                    Q |= todo << r0;
                    R |= todo << r0;
                    break;
                }
                // D.3.1: insignificant samples with a significant neighbour; D.3.4: every sample
                // neither significant nor coded in this plane
                const Seen seen{SL, SR, S << 1, S >> 1, SL << 1, SL >> 1, SR << 1, SR >> 1};
                const ZcCtx z = zc_context(seen, hl, hh);
                const uint32_t open = type == 0u ? any : ~V;
                const uint32_t todo = ((valid & ~S & open) >> r0) & rest;
                const bool run = type == 2u && todo == 15u && ((any >> r0) & 15u) == 0u;
                uint32_t word = bytes(z.c0, r0) | (bytes(z.c1, r0) << 1) | (bytes(z.c2, r0) << 2) | (bytes(z.c3, r0) << 3);
                word = __builtin_amdgcn_perm(0u, ((word + 0x01010101u) << 2) | 0x03020100u, pack[todo]);
                word = run ? kDecRun : word;
                uint32_t cols = (uint32_t)__builtin_amdgcn_ballot_w64(todo != 0u);
                // Both loops end on a value that the decision's bit 31 is part of: with a flag and
                // jumps out of them the compiler keeps conditions in register pairs, a third more
                // scalar instructions.
                uint32_t c = 0, pk = 0, was = 0, d = 0;
                if (cols) do {
                    c = (uint32_t)__builtin_ctz(cols);
                    pk = dw_lane(word, c);
                    do {
                        was = pk;
                        d = mq.decode(pk >> 2);
                        pk = (pk >> 8) | (d & 0x80000000u);  // a sample turned significant: the loops end
                        asm("" : "+s"(pk));
                    } while ((int32_t)pk > 0);
                    cols &= (cols - 1u) & ~(uint32_t)((int32_t)d >> 31);
                    asm("" : "+s"(cols));
                } while (cols);
                if ((int32_t)d >= 0) {
                    if (type == 0u) V |= todo << r0;
                    break;
                }
                // Sample (r0 + k, c) is significant from this plane on: in run-length mode two
                // bits give its row; then its sign (D.3.2), by the signs of the significant
                // neighbours on its four sides, two bits each.
                uint32_t k = was & 3u;
                uint32_t i = (was & 0x7Cu) == kDecRun ? 0u : 2u;
                if (i == 0u) k = 0u;
                uint32_t flip = 0, neg;
                for (;;) {
                    uint32_t cx = 18u + 1u;
                    if (i == 2u) {
                        auto side = [](uint32_t s, uint32_t g, uint32_t row) {
                            return ((s >> row) & 1u) | (((g >> row) & 1u) << 1);
                        };
                        const uint32_t row = r0 + k;
                        const uint32_t around = side(SL, left(G), row) | (side(SR, right(G), row) << 2) |
                                                (side(S << 1, G << 1, row) << 4) | (side(S >> 1, G >> 1, row) << 6);
                        const uint32_t sc = dw_lane(sign_lut[around], c);
                        flip = sc & 1u;
                        cx = sc >> 1;
                    }
                    const uint32_t d = mq.decode(cx) >> 31;
                    neg = d ^ flip;
                    if (i == 2u) break;
                    k = (k << 1) | d;
                    ++i;
                }
                const uint32_t at = r0 + k;
                const uint32_t r = at;
                const uint32_t down = (2u << k) - 1u;  // the scan has passed these rows of column c
                const uint32_t passed = x < c ? 15u : (x == c ? down : 0u);
                if (type == 0u) V |= (todo & passed) << r0;
                rest &= ~passed;
                const uint32_t bit = x == c ? 1u << r : 0u;
                S |= bit;
                B |= bit;
                Q |= bit;
                G |= neg ? bit : 0u;
            }
        }
        if (type == 2u) {
            mq.ws->planes[plane][x] = B;
            if (pass + 1u < passes) {
                ++plane;
                B = Q = V = 0;
            }
            type = 0u;
        } else {
            ++type;
            if (pass + 1u == passes) mq.ws->planes[plane][x] = B;
        }
    }
    // The words: lanes 0-31 the rows 0-15 of their columns, lanes 32-63 the rows 16-31.
    const uint32_t row0 = (lane >> 5) * 16u;
    uint32_t m[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) m[i] = 0u;
    for (uint32_t j = 0; j <= plane; ++j) {
        const uint32_t b = mq.ws->planes[j][x] >> row0;
#pragma unroll
        for (int i = 0; i < 16; ++i) m[i] = (m[i] << 1) | ((b >> i) & 1u);
    }
    const uint32_t p = nbps - 1u - plane;  // the last plane
    uint32_t* const dst = words + x;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const uint32_t r = row0 + (uint32_t)i;
        const uint32_t half = (Q >> r) & 1u ? 1u << p : 2u << p;
        const uint32_t v = ((S >> r) & 1u) ? (((m[i] << 1) << p) + half) | (((G >> r) & 1u) << 31) : 0u;
        if (x < w && r < h) dst[(size_t)r * stride] = v;
    }
}

}  // namespace gail_amd
