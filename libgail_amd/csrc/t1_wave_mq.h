// The arithmetic decoder of the wave Tier-1 decoder (t1_decode_wave.h), written once for the GPU
// and for a host build that checks it against the sequential decoder. On the GPU a whole wave runs
// it with the same values in every lane; only the context states and the successor table's rows
// (DwLanes) differ from lane to lane, and each lane loads a dword of a window.
#pragma once
#include <cstdint>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define DW_FN __device__ __forceinline__
#define DW_UNROLL _Pragma("unroll")
#define DW_IN_VECTOR_REG(x) asm("" : "+v"(x))
#else
#define DW_FN inline
#define DW_UNROLL
#define DW_IN_VECTOR_REG(x)
#endif

namespace gail_amd {

constexpr int kDecMaxPlanes = 30;

#if defined(__HIPCC__)
using DwLanes = uint32_t;  // a value per lane
using DwPair = uint2;
DW_FN uint32_t dw_lane(DwLanes v, uint32_t lane) { return (uint32_t)__builtin_amdgcn_readlane((int)v, (int)lane); }
// lane's value of a ^ (b & mask)
DW_FN uint32_t dw_lane_masked(DwLanes a, DwLanes b, uint32_t lane, uint32_t mask) {
    return dw_lane(a ^ (b & mask), lane);
}
DW_FN uint32_t dw_uniform(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
DW_FN bool dw_any(bool c) { return __builtin_amdgcn_ballot_w64(c) != 0; }
DW_FN void dw_set_lane(DwLanes& v, uint32_t lane, uint32_t x) { v = (threadIdx.x & 63u) == lane ? x : v; }
// f(lane, the lane's value of v) in every lane
template <class F> DW_FN void dw_each(DwLanes& v, const F& f) { f(threadIdx.x & 63u, v); }
#else
struct DwLanes {
    uint32_t v[64];
};
struct DwPair {
    uint32_t x, y;
};
DW_FN uint32_t dw_lane(const DwLanes& v, uint32_t lane) { return v.v[lane]; }
DW_FN uint32_t dw_lane_masked(const DwLanes& a, const DwLanes& b, uint32_t lane, uint32_t mask) {
    return a.v[lane] ^ (b.v[lane] & mask);
}
DW_FN uint32_t dw_uniform(uint32_t v) { return v; }
DW_FN bool dw_any(bool c) { return c; }
DW_FN void dw_set_lane(DwLanes& v, uint32_t lane, uint32_t x) { v.v[lane] = x; }
template <class F> DW_FN void dw_each(DwLanes& v, const F& f) {
    for (uint32_t lane = 0; lane < 64u; ++lane) f(lane, v.v[lane]);
}
#endif

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
// is added exactly when the standard's BYTEIN would: by a shift that finds no bit left.
struct WaveMq {
    uint32_t hi, lo;  // C
    uint32_t A;       // interval << 15
    int32_t extra;
    DwLanes ctx;      // lane k + 1: state of context k
    DwLanes next_m, next_x;  // lane i: row i's successor after an MPS, and what differs after an LPS (MPS 0)
    const DwPair* next;       // successors of a state, after an MPS and after an LPS (LDS)
    DecWave* ws;
    const uint8_t* src;
    uint32_t len;
    uint32_t zero;  // 0 in a vector register: what is read through it stays in vector registers

    // Codeword bytes i .. i + 3, the first highest; ones past the end.
    DW_FN uint32_t dword_at(uint32_t i) const {
        uint32_t w;
        __builtin_memcpy(&w, src + (i < len ? i : 0u), 4);  // the buffer is readable past the codeword
        const uint32_t have = i < len ? len - i : 0u;
        if (have < 4u) w |= have ? 0xFFFFFFFFu << (8u * have) : 0xFFFFFFFFu;
        return __builtin_bswap32(w);
    }
    // A lane's dword of the window, and the byte before it.
    DW_FN void put_window(uint32_t lane, uint32_t w, uint32_t before) {
        const bool ff = ((~w - 0x01010101u) & w & 0x80808080u) != 0u;
        ws->bytes[lane] = w;
        ws->special[lane] = ff || before == 0xFFu ? 1u : 0u;
    }
    DW_FN void load_window(uint32_t at) {
#if defined(__HIPCC__)
        const uint32_t lane = threadIdx.x & 63u, w = dword_at(at + 4u * lane);
        put_window(lane, w, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, 0x138, 0xF, 0xF, true) & 0xFFu);
#else
        for (uint32_t lane = 0; lane < 64u; ++lane)
            put_window(lane, dword_at(at + 4u * lane), lane ? dword_at(at + 4u * lane - 4u) & 0xFFu : 0u);
#endif
        ws->base = at;
    }
    DW_FN uint32_t byte_at(uint32_t a) const {
        return (dw_uniform(ws->bytes[a >> 2]) >> (24u - 8u * (a & 3u))) & 0xFFu;
    }
    // INITDEC (C.3.5)
    DW_FN void init() {
#if defined(__HIPCC__)
        asm("v_mov_b32 %0, 0" : "=v"(zero));
#else
        zero = 0u;
#endif
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
    // Appends bytes until `want` (at most 32) bits are there, or as many as may be. due: a shift
    // waits for them, the only time when a byte that overlaps the bit before it may be added
    // (with none left). Added earlier, its carry into the upper half would take part in the
    // decisions before that shift.
    DW_FN void refill(int32_t want, bool due) {
        asm volatile("" ::: "memory");  // the window stays in LDS
        uint32_t rel = dw_uniform(ws->rel);
        int32_t e = extra;
        uint64_t C = ((uint64_t)hi << 32) | lo;
        while (e < want) {
            if (rel >= 256u) {  // the byte before the next stays in the window
                load_window(dw_uniform(ws->base) + 252u);
                rel -= 252u;
            }
            const uint32_t w = dw_uniform(ws->bytes[rel >> 2]);
            if (!dw_uniform(ws->special[rel >> 2]) && (rel & 1u) == 0u) {
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
            } else if (b > 0x7Fu && !(due && e == 0)) {
                break;  // not before the bits left are used and the next is wanted
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
    DW_FN void shift(uint32_t n) {
        const uint64_t v = (((uint64_t)hi << 32) | lo) << n;
        hi = (uint32_t)(v >> 32) & 0x7FFFFFFFu;
        lo = (uint32_t)v;
        extra -= (int32_t)n;
    }
    // All ones where x < y: each choice below is then one or two operations on the mask.
    static DW_FN uint32_t below(uint32_t x, uint32_t y) {
#if defined(__HIPCC__)
        uint32_t m;
        asm("s_sub_u32 %0, %1, %2\n\ts_subb_u32 %0, 0, 0" : "=&s"(m) : "s"(x), "s"(y) : "scc");
        return m;
#else
        return x < y ? 0xFFFFFFFFu : 0u;
#endif
    }
    // DECODE (C.3.2) in scalar registers; at: the lane of the context's state (modulo 64). The
    // decision is bit 31 of the result. Few scalar instructions are what counts here, 8 without
    // and 25 with renormalisation: C is the smaller of hi and hi - Qe (which wraps around where
    // hi < Qe); the comparison is one select where it is used at once and masks made again for
    // the renormalisation; the choice of the successor is a vector operation.
    DW_FN uint32_t decode(uint32_t at) {
        const uint32_t st = dw_lane(ctx, at & 63u);
        const uint32_t qe = st & 0x3FFF8000u;
        const uint32_t a = A - qe, was = hi;
        const bool lower = hi < qe;
        hi = lower ? hi : hi - qe;
        A = lower ? qe : a;
        uint32_t d = st;
        if (A < 0x40000000u) {  // else the MPS without renormalisation
            // upper sub-interval: the MPS unless a < Qe; lower: the LPS unless a < Qe
            const uint32_t lps = below(a, qe) ^ below(was, qe);
            const uint32_t row = (st >> 4) & 63u;
            dw_set_lane(ctx, at & 63u, dw_lane_masked(next_m, next_x, row, lps) ^ (st & 0x80000008u));
            d ^= lps;
            uint32_t n = (uint32_t)__builtin_clz(A) - 1u;
            A <<= n;
            while (extra < (int32_t)n) {
                refill((int32_t)n, true);
                if (extra >= (int32_t)n) break;
                n -= (uint32_t)extra;
                shift((uint32_t)extra);
            }
            shift(n);
        }
        return d;
    }

    // ---- four decisions at a time in vector registers
    DW_FN void vector() {
        DW_IN_VECTOR_REG(hi);
        DW_IN_VECTOR_REG(lo);
        DW_IN_VECTOR_REG(extra);
        DW_IN_VECTOR_REG(A);
    }
    DW_FN void to_vector() {
        dw_each(ctx, [&](uint32_t lane, uint32_t state) {
            if (lane < 20u) ws->ctx[lane] = state;
        });
        vector();
    }
    DW_FN void refill_vector() {
        scalar();
        refill(32, false);  // ahead of need
        vector();
    }
    DW_FN void to_scalar() {
        dw_each(ctx, [&](uint32_t lane, uint32_t& state) { state = ws->ctx[lane < 20u ? lane : 0u]; });
        scalar();
    }
    DW_FN void scalar() {
        hi = dw_uniform(hi);
        lo = dw_uniform(lo);
        A = dw_uniform(A);
        extra = (int32_t)dw_uniform((uint32_t)extra);
    }
    // the state of the context of a list byte
    DW_FN uint32_t* slot(uint32_t byte) const {
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
    DW_FN void start(Four& f, uint32_t i) {
        f.w = ws->list[(i >> 2) | zero];
        f.state = *slot(f.w);
    }
    // The next four decisions, one to a bit: straight code, each context's state read one decision
    // ahead, before the decision that may change it.
    DW_FN uint32_t four(Four& f, uint32_t w1) {
        uint32_t* at = slot(f.w);
        uint32_t got = 0u;
        f.was = Saved{hi, lo, A, extra};
DW_UNROLL
        for (int j = 0; j < 4; ++j) {
            uint32_t* const nat = slot(j < 3 ? f.w >> (8 * (j + 1)) : w1);
            const uint32_t ahead = *nat, st = f.state;
            f.st[j] = st;
            const DwPair succ = *(const DwPair*)((const char*)next + (st & 0x3F8u));
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
    DW_FN void undo(const Four& f) {
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
    DW_FN void refine(uint32_t total) {
        to_vector();
        Four f;
        bool fresh = false;  // bits were just appended
        start(f, 0u);
        for (uint32_t i = 0;;) {
            const uint32_t w1 = ws->list[((i >> 2) + 1u) | zero];
            uint32_t got = four(f, w1);
            if (dw_any((int32_t)((uint32_t)(extra - 20) | (total - 5u - i)) < 0)) {
                asm volatile("" ::: "memory");
                if (dw_any(extra < 0)) {
                    undo(f);
                    if (!fresh) {
                        refill_vector();
                        fresh = true;
                        start(f, i);
                        continue;
                    }
                    // bits that must be used before more come: one by one
                    to_scalar();
                    const uint32_t w = dw_uniform(f.w);
                    got = 0u;
                    for (uint32_t j = 0; j < 4u; ++j) {
                        const uint32_t s = (w >> (8u * j + 2u)) & 31u;
                        if (s) got |= (decode(s) >> 31) << j;
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

}  // namespace gail_amd
