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

namespace gail_amd {

constexpr int kDecMaxPlanes = 30;
constexpr uint32_t kDecRun = 18u << 2;  // a column in run-length mode

__device__ __forceinline__ uint32_t dw_lane(uint32_t v, uint32_t lane) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)lane);
}

// Inclusive prefix sum over each half-wave.
__device__ __forceinline__ uint32_t dw_scan(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, false);  // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, false);  // row_shr:2
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, false);  // row_shr:4
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, false);  // row_shr:8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false);  // row_bcast:15, rows 1, 3
    return v;
}

// What a wave keeps in LDS.
struct DecWave {
    uint32_t ctx[32];      // entry 0: a neutral context (Qe = 0, always the MPS); k + 1: context k
    uint32_t bytes[64];    // codeword bytes 4 i .. 4 i + 3 of a 256-byte window, the first highest
    uint32_t special[64];  // the dword has a byte that is 0xFF or follows one
    uint32_t rel;          // next byte of the codeword, in the window
    uint32_t base;         // the window's first byte (a multiple of 4)
    uint32_t list[36];     // the stripe's decisions in scan order, a byte each
    uint8_t bits[40];      // a refinement stripe's decisions, four to a byte
    uint8_t junk[64];      // where lanes write the decisions they do not have
    uint32_t pad[2];
    uint32_t planes[kDecMaxPlanes][32];
};

// MQ decoder (C.3). C holds the code register with the codeword bits that follow it: bits 62-47
// are its upper half, `extra` bits below them are valid. A state is MPS << 31 | Qe << 15 | 8 x its
// index in the successor table (2 x the row of Table C.2 + MPS). Bytes are appended when bits
// run out, two at a time unless one is special (0xFF or after it, or past the end, where the
// codeword continues with ones). A byte of 0x80-0x8F after 0xFF overlaps the bit before it: it
// is added exactly when the standard's BYTEIN would, with no bit left.
struct WaveMq {
    uint32_t hi, lo;  // C
    uint32_t A;       // interval << 15
    int32_t extra;
    uint32_t ctx;     // lane k: state of context k
    uint32_t next_m, next_l;  // lane i: the successors of row i with MPS 0
    const uint2* next;        // successors of a state, after an MPS and after an LPS (LDS)
    DecWave* ws;
    const uint8_t* src;
    uint32_t len;
    uint32_t zero;  // 0 in a vector register: what is read through it stays in vector registers

    static __device__ __forceinline__ uint32_t uniform(uint32_t v) {
        return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
    }
    __device__ __forceinline__ void load_window(uint32_t at) {
        const uint32_t lane = threadIdx.x & 63u, i = at + 4u * lane;
        uint32_t w;
        __builtin_memcpy(&w, src + (i < len ? i : 0u), 4);  // the buffer is readable past the codeword
        const uint32_t have = i < len ? len - i : 0u;
        if (have < 4u) w |= have ? 0xFFFFFFFFu << (8u * have) : 0xFFFFFFFFu;
        w = __builtin_bswap32(w);
        const uint32_t before = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, 0x138, 0xF, 0xF, true) & 0xFFu;
        const bool ff = ((~w - 0x01010101u) & w & 0x80808080u) != 0u;
        ws->bytes[lane] = w;
        ws->special[lane] = ff || before == 0xFFu ? 1u : 0u;
        ws->base = at;
    }
    __device__ __forceinline__ uint32_t byte_at(uint32_t a) const {
        return (uniform(ws->bytes[a >> 2]) >> (24u - 8u * (a & 3u))) & 0xFFu;
    }
    // INITDEC (C.3.5)
    __device__ __forceinline__ void init() {
        asm("v_mov_b32 %0, 0" : "=v"(zero));
        load_window(0u);
        const uint32_t b0 = byte_at(0u), b1 = byte_at(1u);
        uint64_t C = (uint64_t)b0 << 54;
        uint32_t rel = 2u;
        if (b0 != 0xFFu) {
            C += (uint64_t)b1 << 46;
            extra = 1;
        } else if (b1 <= 0x8Fu) {
            C += (uint64_t)b1 << 47;
            extra = 0;
        } else {
            C += 0xFFull << 46;
            extra = 1;
            rel = 1u;
        }
        ws->rel = rel;
        hi = (uint32_t)(C >> 32);
        lo = (uint32_t)C;
        A = 0x40000000u;
    }
    // Appends bytes until `want` (at most 32) bits are there, or as many as may be.
    __device__ __forceinline__ void refill(int32_t want) {
        asm volatile("" ::: "memory");  // the window stays in LDS
        uint32_t rel = uniform(ws->rel);
        int32_t e = extra;
        uint64_t C = ((uint64_t)hi << 32) | lo;
        while (e < want) {
            if (rel >= 256u) {  // the byte before the next stays in the window
                load_window(uniform(ws->base) + 252u);
                rel -= 252u;
            }
            const uint32_t w = uniform(ws->bytes[rel >> 2]);
            if (!uniform(ws->special[rel >> 2]) && (rel & 1u) == 0u) {
                const uint32_t h = (rel & 2u) ? w & 0xFFFFu : w >> 16;
                C += (uint64_t)h << (31 - e);
                e += 16;
                rel += 2u;
                continue;
            }
            const uint32_t b = (w >> (24u - 8u * (rel & 3u))) & 0xFFu;
            const bool after_ff = byte_at(rel - 1u) == 0xFFu;
            if (!after_ff) {
                C += (uint64_t)b << (39 - e);
                e += 8;
                ++rel;
            } else if (b > 0x8Fu) {  // a marker, which stays unread: ones
                C += 0xFFull << (39 - e);
                e += 8;
            } else if (b > 0x7Fu && e > 0) {
                break;  // not before the bits left are used
            } else {
                C += (uint64_t)b << (40 - e);
                e += 7;
                ++rel;
            }
        }
        ws->rel = rel;
        extra = e;
        hi = (uint32_t)(C >> 32);
        lo = (uint32_t)C;
        asm volatile("" ::: "memory");
    }
    __device__ __forceinline__ void shift(uint32_t n) {
        const uint64_t v = (((uint64_t)hi << 32) | lo) << n;
        hi = (uint32_t)(v >> 32) & 0x7FFFFFFFu;
        lo = (uint32_t)v;
        extra -= (int32_t)n;
    }
    // All ones where x < y: each choice below is then one or two operations on the mask.
    static __device__ __forceinline__ uint32_t below(uint32_t x, uint32_t y) {
        uint32_t m;
        asm("s_sub_u32 %0, %1, %2\n\ts_subb_u32 %0, 0, 0" : "=&s"(m) : "s"(x), "s"(y) : "scc");
        return m;
    }
    // DECODE (C.3.2) in scalar registers
    __device__ __forceinline__ uint32_t decode(uint32_t cx) {
        const uint32_t st = dw_lane(ctx, cx);
        const uint32_t qe = st & 0x3FFF8000u;
        const uint32_t a = A - qe;
        const uint32_t lower = below(hi, qe);
        hi -= qe & ~lower;
        A = a ^ ((a ^ qe) & lower);
        uint32_t d = st >> 31;
        if (A < 0x40000000u) {  // else the MPS without renormalisation
            // upper sub-interval: the MPS unless a < Qe; lower: the LPS unless a < Qe
            const uint32_t lps = below(a, qe) ^ lower;
            const uint32_t row = (st >> 4) & 63u;
            const uint32_t m = dw_lane(next_m, row), l = dw_lane(next_l, row);
            const uint32_t to = m ^ ((m ^ l) & lps) ^ (st & 0x80000008u);
            ctx = (threadIdx.x & 63u) == cx ? to : ctx;
            d ^= lps & 1u;
            uint32_t n = (uint32_t)__builtin_clz(A) - 1u;
            A <<= n;
            while (extra < (int32_t)n) {
                refill((int32_t)n);
                if (extra >= (int32_t)n) break;
                n -= (uint32_t)extra;
                shift((uint32_t)extra);
            }
            shift(n);
        }
        return d;
    }

    // ---- four decisions at a time in vector registers
    __device__ __forceinline__ void vector() {
        asm("" : "+v"(hi));
        asm("" : "+v"(lo));
        asm("" : "+v"(extra));
        asm("" : "+v"(A));
    }
    __device__ __forceinline__ void to_vector() {
        const uint32_t lane = threadIdx.x & 63u;
        if (lane < 19u) ws->ctx[lane + 1u] = ctx;
        vector();
    }
    __device__ __forceinline__ void refill_vector() {
        scalar();
        refill(32);
        vector();
    }
    __device__ __forceinline__ void to_scalar() {
        const uint32_t lane = threadIdx.x & 63u;
        ctx = ws->ctx[lane < 19u ? lane + 1u : 0u];
        scalar();
    }
    __device__ __forceinline__ void scalar() {
        hi = uniform(hi);
        lo = uniform(lo);
        A = uniform(A);
        extra = (int32_t)uniform((uint32_t)extra);
    }
    // the state of the context of a list byte
    __device__ __forceinline__ uint32_t* slot(uint32_t byte) const {
        return (uint32_t*)((char*)ws->ctx + ((byte & 0x7Cu) | zero));
    }
    // Decisions are made without asking whether their bits are there; extra < 0 afterwards says
    // that they were not, and the decisions are taken back and made again.
    struct Saved {
        uint32_t hi, lo, A;
        int32_t extra;
    };
    struct Four {
        uint32_t w;      // the decisions' list bytes
        uint32_t state;  // of the first one's context, up to date
        uint32_t st[4];  // the states that they found
        Saved was;
    };
    __device__ __forceinline__ void start(Four& f, uint32_t i) {
        f.w = ws->list[(i >> 2) | zero];
        f.state = *slot(f.w);
    }
    // The next four decisions, one to a bit: straight code, each context's state read one decision
    // ahead, before the decision that may change it.
    __device__ __forceinline__ uint32_t four(Four& f, uint32_t w1) {
        uint32_t* at = slot(f.w);
        uint32_t got = 0u;
        f.was = Saved{hi, lo, A, extra};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint32_t* const nat = slot(j < 3 ? f.w >> (8 * (j + 1)) : w1);
            const uint32_t ahead = *nat, st = f.state;
            f.st[j] = st;
            const uint2 succ = *(const uint2*)((const char*)next + (st & 0x3F8u));
            const uint32_t qe = st & 0x3FFF8000u;
            const uint32_t a = A - qe, t = hi - qe;
            const uint32_t x = t ^ (a - qe);  // < 0: the LPS
            const bool lower = (int32_t)t < 0;
            hi = lower ? hi : t;
            const uint32_t a2 = lower ? qe : a;
            const uint32_t n = (uint32_t)__builtin_clz(a2) - 1u;
            A = a2 << n;
            const uint32_t to = (int32_t)x < 0 ? succ.y : succ.x;
            const uint32_t st_new = a2 & 0x40000000u ? st : to;
            *at = st_new;
            shift(n);
            got |= ((st ^ x) >> 31) << j;
            f.state = nat == at ? st_new : ahead;
            at = nat;
        }
        return got;
    }
    __device__ __forceinline__ void undo(const Four& f) {
        *slot(f.w >> 24) = f.st[3];
        *slot(f.w >> 16) = f.st[2];
        *slot(f.w >> 8) = f.st[1];
        *slot(f.w) = f.st[0];
        hi = f.was.hi;
        lo = f.was.lo;
        A = f.was.A;
        extra = f.was.extra;
    }
    // The decisions of the stripe's list (refinement contexts), to ws->bits.
    __device__ __forceinline__ void refine(uint32_t total) {
        to_vector();
        Four f;
        bool fresh = false;  // bits were just appended
        start(f, 0u);
        for (uint32_t i = 0;;) {
            const uint32_t w1 = ws->list[((i >> 2) + 1u) | zero];
            uint32_t got = four(f, w1);
            if (__builtin_amdgcn_ballot_w64((int32_t)((uint32_t)(extra - 20) | (total - 5u - i)) < 0)) {
                asm volatile("" ::: "memory");
                if (__builtin_amdgcn_ballot_w64(extra < 0)) {
                    undo(f);
                    if (!fresh) {
                        refill_vector();
                        fresh = true;
                        start(f, i);
                        continue;
                    }
                    // bits that must be used before more come: one by one
                    to_scalar();
                    const uint32_t w = uniform(f.w);
                    got = 0u;
                    for (uint32_t j = 0; j < 4u; ++j) {
                        const uint32_t s = (w >> (8u * j + 2u)) & 31u;
                        if (s) got |= decode(s - 1u) << j;
                    }
                    to_vector();
                    f.state = *slot(w1);
                }
                ws->bits[i >> 2] = (uint8_t)got;
                if (i + 4u >= total) break;
                refill_vector();
            } else {
                ws->bits[i >> 2] = (uint8_t)got;
            }
            fresh = false;
            i += 4u;
            f.w = w1;
        }
        to_scalar();
    }
};

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
                uint32_t c = 0, pk = 0, was = 0, one = 0;
                if (cols) do {
                    c = (uint32_t)__builtin_ctz(cols);
                    pk = dw_lane(word, c);
                    do {
                        was = pk;
                        one = mq.decode(((pk >> 2) & 31u) - 1u);
                        pk = (pk >> 8) | (one << 31);  // a sample turned significant: the loops end
                        asm("" : "+s"(pk));
                    } while ((int32_t)pk > 0);
                    cols = one ? 0u : cols & (cols - 1u);
                    asm("" : "+s"(cols));
                } while (cols);
                if (!one) {
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
                    uint32_t cx = 18u;
                    if (i == 2u) {
                        auto side = [](uint32_t s, uint32_t g, uint32_t row) {
                            return ((s >> row) & 1u) | (((g >> row) & 1u) << 1);
                        };
                        const uint32_t row = r0 + k;
                        const uint32_t around = side(SL, left(G), row) | (side(SR, right(G), row) << 2) |
                                                (side(S << 1, G << 1, row) << 4) | (side(S >> 1, G >> 1, row) << 6);
                        const uint32_t sc = dw_lane(sign_lut[around], c);
                        flip = sc & 1u;
                        cx = (sc >> 1) - 1u;
                    }
                    const uint32_t d = mq.decode(cx);
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
