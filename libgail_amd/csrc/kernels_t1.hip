// EBCOT Tier-1 for CDNA4 (gfx950, wave64): fused dead-zone quantisation + context
// modelling, block ordering, MQ coding with exact truncation lengths, and compaction.
//
// Context modelling: one wave codes two 32x32 code-blocks, lanes 0-31 and 32-63; lane x
// owns column x and keeps its column's state as 32-bit row masks (significant, refined,
// visited, current magnitude bit) plus its 32 quantised magnitudes in registers. Left and
// right neighbours come from lane shuffles, above and below are bit shifts. Per 4-row
// stripe the significance-propagation pass is solved as a monotone fixpoint over the
// half-wave (no change anywhere => the sequential scan's result), cleanup needs no
// fixpoint because every remaining sample is coded. Each lane holds its column's symbols of
// a stripe (at most 10) as bytes of registers; a scan over the half-wave gives the exclusive
// prefix over the columns, so symbols land in scan order in a per-block LDS staging buffer,
// copied to an HBM pool once per bit-plane.
//
// MQ coding: one lane per code-block, blocks ordered largest first so a wave's lanes
// finish together. The coder keeps A, C, CT and the pending byte in registers, with several
// bytes' room in C so that bytes are taken rarely and for all lanes at once, and the context
// states in LDS; at each pass end it snapshots its state, and after the final flush it derives
// every pass's truncation length from the snapshots.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "device_types.h"
#include "kernels.h"
#include "t1_cm_masks.h"
#include "t1_tables.h"

namespace gail_amd {

namespace {

// ---------------------------------------------------------------- helpers
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Value of the lane one column to the left / right within the same half-wave; zero at
// the block's edges.
// DPP wave_shr:1 / wave_shl:1 move a register one lane up / down across the whole wave in
// one VALU operation; the lanes at a block's edge (x = 0 / 31) see zero.
__device__ __forceinline__ uint32_t from_left(uint32_t v, int x) {
    const uint32_t r = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x138, 0xF, 0xF, true);
    return x == 0 ? 0u : r;
}
__device__ __forceinline__ uint32_t from_right(uint32_t v, int x) {
    const uint32_t r = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x130, 0xF, 0xF, true);
    return x == 31 ? 0u : r;
}

__device__ __forceinline__ double half_sum_d(double v) {
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) v += __shfl_xor(v, o, 32);
    return v;
}
__device__ __forceinline__ uint32_t half_max_u(uint32_t v) {
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) {
        const uint32_t t = (uint32_t)__shfl_xor((int)v, o, 32);
        v = t > v ? t : v;
    }
    return v;
}

// Inclusive prefix sum over the lanes of each half-wave (lanes 0-31 and 32-63 separately):
// four row shifts within each 16-lane row, then row 0's (row 2's) last lane added to row 1
// (row 3). Lanes without a source add zero.
__device__ __forceinline__ uint32_t half_scan(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, false);  // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, false);  // row_shr:2
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, false);  // row_shr:4
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, false);  // row_shr:8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false);  // row_bcast:15, rows 1, 3
    return v;
}

// Sum over the lane's half-wave, in every lane of that half (the scan's last lanes hold the
// two sums).
__device__ __forceinline__ int half_total(int v) {
    const int inc = (int)half_scan((uint32_t)v);
    const int lo = __builtin_amdgcn_readlane(inc, 31), hi = __builtin_amdgcn_readlane(inc, 63);
    return (threadIdx.x & 32) ? hi : lo;
}

// Rows r0..r0+3 of mask m as bit 0 of bytes 0..3. The product is kept opaque so that a shift
// applied afterwards is not folded into the multiplier (a 24-bit multiply stays one).
__device__ __forceinline__ uint32_t stripe_bytes(uint32_t m, int r0) {
    uint32_t t = __umul24((m >> r0) & 0xFu, 0x204081u) & 0x01010101u;
    asm("" : "+v"(t));
    return t;
}

// The same at bit J of each byte (J <= 2, so that the multiplier keeps its 24 bits), into w.
__device__ __forceinline__ uint32_t stripe_bits(uint32_t w, uint32_t m, int r0, int j) {
    uint32_t t = __umul24((m >> r0) & 0xFu, 0x204081u << j);
    asm("" : "+v"(t));
    const uint32_t at = 0x01010101u << j;
    return (t & at) | (w & ~at);
}

// The first n (at most 4) bytes of w to out; every lane stores all four, those it does not have
// to junk, so that no lane diverges.
__device__ __forceinline__ void put_bytes(uint32_t w, uint32_t n, uint8_t* out, uint8_t* junk) {
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) (j < n ? out : junk)[j] = (uint8_t)(w >> (8 * j));
}

constexpr int kChunkBytes = 65536;  // symbol pool grabbed per wave at a time

}  // namespace

// ---------------------------------------------------------------- counters
__global__ void clear_counters_kernel(JobCounters* c, uint32_t* work, int nwork, uint32_t* order) {
    const int t = threadIdx.x;
    if (t < (int)(sizeof(JobCounters) / 4)) ((uint32_t*)c)[t] = 0;
    if (t < nwork) work[t] = 0;
    order[t] = 0;
}

hipError_t launch_clear_counters(JobCounters* c, uint32_t* work, int nwork, uint32_t* order, hipStream_t s) {
    static_assert(sizeof(JobCounters) / 4 <= kOrderWords);
    hipLaunchKernelGGL(clear_counters_kernel, dim3(1), dim3(kOrderWords), 0, s, c, work, nwork, order);
    return hipGetLastError();
}

// ---------------------------------------------------------------- debug quantiser
// The coefficient words the context-modelling kernel quantises for itself, materialised
// (1,024 per block, row-major, zero-padded) for the debug taps.
__global__ void __launch_bounds__(256) quant_debug_kernel(const T1Block* blocks, const T1Band* bands,
                                                          const T1FrameRef* frames, uint32_t n, uint32_t* out) {
    const size_t gid = (size_t)blockIdx.x * 256 + threadIdx.x;
    const uint32_t cb = (uint32_t)(gid >> 10);
    if (cb >= n) return;
    const int k = (int)(gid & 1023), r = k >> 5, x = k & 31;
    const T1Block b = blocks[cb];
    uint32_t word = 0;
    if (x < b.w && r < b.h) {
        const T1Band band = bands[b.band];
        const T1FrameRef fr = frames[b.frame];
        const float v = fr.coef[b.coef_off + (size_t)r * fr.stride + x];
        const float a = (v < 0.f ? -v : v) * band.inv_delta * 64.0f;
        const uint32_t q = a >= (float)band.max_mag ? band.max_mag : (uint32_t)a;
        word = q | ((v < 0.f && q >= 64u) ? 0x80000000u : 0u);
    }
    out[gid] = word;
}

hipError_t launch_quant_debug(const T1Block* blocks, const T1Band* bands, const T1FrameRef* frames, uint32_t n,
                              uint32_t* out, hipStream_t s) {
    hipLaunchKernelGGL(quant_debug_kernel, dim3((unsigned)(((size_t)n * 1024 + 255) / 256)), dim3(256), 0, s, blocks,
                       bands, frames, n, out);
    return hipGetLastError();
}

// ---------------------------------------------------------------- context modelling
// Bound by vector issue: 0.86-0.89 vector instructions a cycle and CU at 16 4K frames, three waves
// a SIMD (the magnitudes and planes of a column need 168 registers), LDS busy 40 % of the time
// with the symbols' byte stores. So instructions are what is saved: the quantiser and the
// stores have no branches (a lane without a symbol stores to a junk byte), a symbol's bits are
// set for four rows by one multiplication each, and a stripe's bytes are put in order by
// v_perm with selectors from a table of all 256 cases. With divergent stores, selectors
// built per stripe and a masked quantiser the same 16 frames took 5.42 ms (20 % more vector and
// 57 % more scalar instructions), now 4.80; one 2K frame 0.232 and 0.213, 512x256 0.097 and 0.081.
template <int WAVES>
__global__ void __launch_bounds__(WAVES * 64, 3) t1_cm_kernel(CmParams P) {
    // a plane's symbols per block, then 128 bytes where each lane writes the symbols its rows
    // do not have (so that every lane stores on every step)
    __shared__ __attribute__((aligned(16))) uint8_t s_sym[WAVES][2][kPlaneStage + 144];
    // For the sets of a stripe's rows that have a zero-coding (low nibble) and a sign symbol (high
    // nibble), the order of their bytes as selectors: the rows in turn, each one's zero-coding
    // byte (0-3) before its sign byte (4-7).
    __shared__ uint2 s_order[256];
    for (uint32_t i = threadIdx.x; i < 256u; i += WAVES * 64) {
        unsigned long long v = 0x0C0C0C0C0C0C0C0Cull;
        uint32_t j = 0;
        for (uint32_t k = 0; k < 8; ++k)
            if ((i >> (k >> 1 | (k & 1u) << 2)) & 1u) {
                const uint32_t sel = k >> 1 | (k & 1u) << 2;
                v = (v & ~(0xFFull << (8 * j))) | ((unsigned long long)sel << (8 * j));
                ++j;
            }
        s_order[i] = make_uint2((uint32_t)v, (uint32_t)(v >> 32));
    }
    __syncthreads();
    // Early-termination counts per context of the current plane (d = 0 low half, d = 1 high
    // half) and the contexts' entropy terms.
    __shared__ uint32_t s_hist[WAVES][2][32];
    __shared__ __attribute__((aligned(16))) float s_term[WAVES][2][20];

    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, half = lane >> 5, x = lane & 31;
    uint8_t* const sym = s_sym[wv][half];
    uint8_t* const junk = sym + kPlaneStage + 4 * x;
    uint32_t* const hist = s_hist[wv][half];
    float* const terms = s_term[wv][half];
    unsigned long long chunk_cur = 0, chunk_end = 0;  // wave-uniform sub-allocator

    for (;;) {
        uint32_t pair = 0;
        if (lane == 0) pair = atomicAdd(P.work_next, 1u);
        pair = __shfl((int)pair, 0);
        if (2 * pair >= P.nblocks) break;
        const uint32_t cb = 2 * pair + half;
        const bool has = cb < P.nblocks;
        T1Block blk{};
        if (has) blk = P.blocks[cb];
        const int w = has ? blk.w : 0, h = has ? blk.h : 0;
        const T1Band band = P.bands[has ? blk.band : 0];
        const T1FrameRef fr = P.frames[has ? blk.frame : 0];
        const bool hl = has && blk.orient == 1, hh = has && blk.orient == 3;

        // Fused dead-zone quantisation of the block's column (quant.h:20-25).
        uint32_t m[32];
        uint32_t sgn = 0, colmax = 0;
        {
            // all 32 loads in flight at once: rows and columns outside the block read the
            // block's first sample (a valid address). What they quantise to is a value of the
            // block, so it changes no maximum, and the passes mask it out; so do they the signs
            // of samples that quantise to 0.
            const float* src = fr.coef + blk.coef_off + (x < w ? x : 0);
            const float scale = band.inv_delta * 64.0f;  // a power of two apart: the same rounding
            float v[32];
#pragma unroll
            for (int r = 0; r < 32; ++r) v[r] = src[(size_t)(r < h ? r : 0) * fr.stride];
#pragma unroll
            for (int r = 31; r >= 0; --r) {
                uint32_t q;  // saturating, unlike the language's conversion
                asm("v_cvt_u32_f32 %0, %1" : "=v"(q) : "v"(__builtin_fabsf(v[r]) * scale));
                q = q < band.max_mag ? q : band.max_mag;
                sgn = __builtin_amdgcn_alignbit(sgn, __float_as_uint(v[r]), 31);
                m[r] = q;
                colmax = q > colmax ? q : colmax;
            }
        }
        const uint32_t bmax = half_max_u(colmax) >> 6;
        const int nbps = has && bmax ? 32 - __clz((int)bmax) : 0;
        // the pair's plane count, in a scalar register (a wave-uniform loop bound)
        const int nbps_lo = __builtin_amdgcn_readlane(nbps, 0), nbps_hi = __builtin_amdgcn_readlane(nbps, 32);
        const int jmax = nbps_lo > nbps_hi ? nbps_lo : nbps_hi;
        const uint32_t sgnL = from_left(sgn, x), sgnR = from_right(sgn, x);
        const uint32_t sgnU = sgn << 1, sgnD = sgn >> 1;
        const uint32_t rowsValid = h >= 32 ? 0xFFFFFFFFu : ((1u << h) - 1u);
        const float thr = fr.slope_thresh;
        const bool track = thr > 0.f;
        if (x < 20) hist[x] = 0;

        // Bit-plane masks of the column: pl[k] holds bit (p + k) of every row's magnitude
        // (bits p..p+6: the current magnitude bit is pl[6], the six below it feed the
        // distortion estimates). Moving to the next plane shifts the register down by one
        // and extracts a single new mask.
        uint32_t pl[7];
        {
            const int p0 = nbps > 0 ? nbps - 1 : 0;
#pragma unroll
            for (int k = 0; k < 7; ++k) {
                uint32_t mk = 0;
#pragma unroll
                for (int r = 0; r < 32; ++r) mk |= __builtin_amdgcn_ubfe(m[r], (uint32_t)(p0 + k), 1u) << r;
                pl[k] = mk;
            }
        }
        // Sum of the 7-bit windows (bits p..p+6) of the rows in mask s.
        auto window_sum = [&](uint32_t s) {
            int t = 0;
#pragma unroll
            for (int k = 6; k >= 0; --k) t = 2 * t + __popc(pl[k] & s);
            return t;
        };

        uint32_t S = 0, R = 0;  // significant, refined before
        uint32_t np = 0, sym_total = 0, planes = 0;
        bool done = !has || nbps == 0 || nbps > kMaxPlanes;
        for (int j = 0; j < jmax; ++j) {
            const bool act = !done && j < nbps;
            const int p = nbps - 1 - j;  // current bit-plane (valid when act)
            if (j > 0) {
#pragma unroll
                for (int k = 6; k > 0; --k) pl[k] = pl[k - 1];
                const int sh = p > 0 ? p : 0;
                uint32_t mk = 0;
#pragma unroll
                for (int r = 0; r < 32; ++r) mk |= __builtin_amdgcn_ubfe(m[r], (uint32_t)sh, 1u) << r;
                pl[0] = act ? mk : 0u;
            }
            const uint32_t Bp = pl[6];
            const uint32_t sig0 = S;
            uint32_t V = 0, plane_count = 0;
            int plane_dist = 0;
            for (int type = (j == 0 ? 2 : 0); type < 3; ++type) {
                const bool pact = act && np < P.max_passes;
                const uint32_t pass_start = plane_count;
                const uint32_t colMask = (pact && x < w) ? rowsValid : 0u;
                const uint32_t SL = from_left(S, x), SR = from_right(S, x);
                // The pass over the whole column: keep0 the rows whose zero-coding (or
                // refinement) symbol is written, keep1 those whose sign symbol is written,
                // rl the run-length symbols of each stripe (a nibble per stripe); m0 / m1 the
                // bits of those symbol bytes, one mask per bit.
                uint32_t keep0 = 0, keep1 = 0, runs = 0, rl = 0;
                uint32_t m0[5] = {Bp, 0, 0, 0, 0}, m1[4] = {0, 0, 0, 0};
                int dist = 0;
                if (type == 1) {
                    // ---- magnitude refinement (D.3.3): samples significant before this plane;
                    // symbol 28 + (bit | (context - 14) << 1), context 16 if refined before,
                    // else 15 if a neighbour is significant, else 14
                    keep0 = sig0 & colMask;
                    m0[1] = neighbour_any(S, SL, SR) & ~R;
                    m0[2] = R;
                    // t1_dist_ref summed: 64 w - 5120 where bit p+6 is set, 3072 - 64 w elsewhere.
                    // A window bit counts for the first rows and against the others: the rows
                    // where it equals bit p+6, less the others' number.
                    const int ones = __popc(keep0 & Bp), zeros = __popc(keep0) - ones;
                    int t = 0;
#pragma unroll
                    for (int k = 6; k >= 0; --k) t = 2 * t + __popc(keep0 & ~(pl[k] ^ Bp));
                    dist = 64 * (t - 127 * zeros) - 5120 * ones + 3072 * zeros;
                    R |= keep0;
                } else {
                    uint32_t N = 0;  // samples the pass turns significant
                    if (type == 0) {
                        // ---- significance propagation (D.3.1): the least fixed point of "an
                        // insignificant row is coded when a neighbour is significant as the scan
                        // sees it"; each round every lane fills its column given the other
                        // columns' current new significance, until no lane's set changes
                        const uint32_t open = ~S & colMask;
                        const uint32_t around = neighbour_any(S, SL, SR);
                        uint32_t E = 0;
                        if (__any((open & around) != 0)) {
                            for (;;) {
                                const uint32_t seen = around | new_seen(from_left(N, x), from_right(N, x));
                                E = column_fill(open & seen, open, Bp);
                                const uint32_t turned = E & Bp;
                                if (!__any(turned != N)) break;
                                N = turned;
                            }
                        }
                        keep0 = E;
                        V |= E;
                    } else {
                        // ---- cleanup with run-length mode (D.3.4): every remaining sample
                        const uint32_t Cc = colMask & ~S & ~V;
                        N = Cc & Bp;
                        runs = run_stripes(Cc, S, SL, SR, N, from_left(N, x), from_right(N, x));
                        cleanup_run_symbols(Cc, N, runs, keep0, rl);
                    }
                    keep1 = N;
                    if (__any((keep0 | keep1 | rl) != 0)) {
                        const Seen v = seen_at_coding(S, SL, SR, N, from_left(N, x), from_right(N, x));
                        const ZcCtx z = zc_context(v, hl, hh);
                        const ScCtx g = sign_context(v, sgnL, sgnR, sgn, sgnU, sgnD);
                        m0[1] = z.c0;
                        m0[2] = z.c1;
                        m0[3] = z.c2;
                        m0[4] = z.c3;
                        m1[0] = g.d;
                        m1[1] = g.c0;
                        m1[2] = g.c1;
                        m1[3] = g.c2;
                    }
                    S |= N;
                    // t1_dist_sig summed over the new significances: 192 w - 9216 each
                    dist = 192 * window_sum(N) - 9216 * __popc(N);
                }
                if (__any((keep0 | keep1 | rl) != 0)) {
                    // symbols per stripe (a nibble each), placed stripe after stripe and, within
                    // a stripe, column after column by an exclusive prefix over the half-wave;
                    // stripes k and k + 4 share a register, 16 bits each
                    const uint32_t cnt = nibble_counts(keep0) + nibble_counts(keep1) + rl;
                    uint32_t e0, e1, e2, e3, t0, t1, t2, t3, u0, u1, u2, u3;
                    {
                        uint32_t f = cnt & 0x000F000Fu, inc = half_scan(f);
                        e0 = inc - f;
                        t0 = (uint32_t)__builtin_amdgcn_readlane((int)inc, 31);
                        u0 = (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
                        f = (cnt >> 4) & 0x000F000Fu;
                        inc = half_scan(f);
                        e1 = inc - f;
                        t1 = (uint32_t)__builtin_amdgcn_readlane((int)inc, 31);
                        u1 = (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
                        f = (cnt >> 8) & 0x000F000Fu;
                        inc = half_scan(f);
                        e2 = inc - f;
                        t2 = (uint32_t)__builtin_amdgcn_readlane((int)inc, 31);
                        u2 = (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
                        f = (cnt >> 12) & 0x000F000Fu;
                        inc = half_scan(f);
                        e3 = inc - f;
                        t3 = (uint32_t)__builtin_amdgcn_readlane((int)inc, 31);
                        u3 = (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
                    }
                    uint32_t base = plane_count;
                    const uint32_t pre[4] = {e0, e1, e2, e3}, lo[4] = {t0, t1, t2, t3}, hi[4] = {u0, u1, u2, u3};
#pragma unroll
                    for (int s = 0; s < 8; ++s) {
                        // this stripe's prefix and half-wave totals
                        const uint32_t ex = s < 4 ? pre[s & 3] & 0xFFFFu : pre[s & 3] >> 16;
                        const uint32_t tlo = s < 4 ? lo[s & 3] & 0xFFFFu : lo[s & 3] >> 16;
                        const uint32_t thi = s < 4 ? hi[s & 3] & 0xFFFFu : hi[s & 3] >> 16;
                        if (tlo + thi == 0) continue;
                        uint8_t* out = sym + base + ex;
                        base += half ? thi : tlo;
                        const int r0 = 4 * s;
                        const uint32_t z = (keep0 >> r0) & 0xFu;
                        if (type == 1) {
                            const uint32_t w0 = 0x1C1C1C1Cu + stripe_bits(stripe_bits(stripe_bytes(m0[0], r0), m0[1], r0, 1),
                                                                          m0[2], r0, 2);
                            put_bytes(__builtin_amdgcn_perm(0u, w0, s_order[z].x), (uint32_t)__popc(z), out, junk);
                        } else {
                            const uint32_t gn = (keep1 >> r0) & 0xFu;
                            if (type == 2 && __any(((runs >> r0) & 1u) != 0)) {
                                // run-length symbols: context 17 with whether a row turns
                                // significant, then that row's position in two context-18 bits
                                const bool run = (runs >> r0) & 1u, hit = run && gn != 0;
                                const uint32_t first = gn ? (uint32_t)__builtin_ctz(gn) : 0u;
                                *(run ? out : junk) = (uint8_t)(34u | (gn != 0));
                                uint8_t* const more = hit ? out : junk;
                                more[1] = (uint8_t)(36u | (first >> 1));
                                more[2] = (uint8_t)(36u | (first & 1u));
                                out += run ? (hit ? 3u : 1u) : 0u;
                            }
                            uint32_t w0 = stripe_bits(stripe_bytes(m0[3], r0), m0[4], r0, 1) << 3;
                            w0 |= stripe_bits(stripe_bits(stripe_bytes(m0[0], r0), m0[1], r0, 1), m0[2], r0, 2);
                            const uint32_t w1 =
                                0x12121212u + (stripe_bits(stripe_bits(stripe_bytes(m1[0], r0), m1[1], r0, 1), m1[2], r0, 2) |
                                               stripe_bytes(m1[3], r0) << 3);
                            // the stripe's symbols in order, without gaps
                            const uint2 order = s_order[z | gn << 4];
                            const uint32_t n = (uint32_t)(__popc(z) + __popc(gn));
                            put_bytes(__builtin_amdgcn_perm(w1, w0, order.x), n, out, junk);
                            if (__any(n > 4u)) put_bytes(__builtin_amdgcn_perm(w1, w0, order.y), n > 4u ? n - 4u : 0u, out + 4, junk);
                        }
                    }
                    sym_total += base - plane_count;
                    plane_count = base;
                }
                const int total = half_total(dist);
                if (pact) {
                    // the pass ends a 4-byte word of the MQ coder's input, the word's top bit set
                    const uint32_t pad = plane_count == pass_start ? 4u : (0u - plane_count) & 3u;
                    if ((uint32_t)x < pad) sym[plane_count + x] = (uint8_t)kSymPad;
                    plane_count += pad;
                    if (x == 0) {
                        sym[plane_count - 1] |= (uint8_t)kSymPassEnd;
                        P.pass_dist[(size_t)cb * kMaxPasses + np] = total;
                    }
                    ++np;
                    plane_dist += total;
                }
            }
            // ---- the plane's symbols to the pool (wave-uniform sub-allocation), filled up to
            // whole 16-byte groups with neutral symbols
            {
                const uint32_t fill = (16u - (plane_count & 15u)) & 15u;
                if ((uint32_t)x < fill) sym[plane_count + x] = (uint8_t)kSymPad;
                plane_count += fill;
            }
            wave_sync();
            // early-termination counts of the plane's symbols, 32 lanes per block at a time (not
            // one lane per column inside the emission loops): per context the symbols, and the
            // ones among them << 16. The plane is a multiple of 16 symbols long.
            if (track && act)
                for (uint32_t i = 4u * (uint32_t)x; i < plane_count; i += 128u) {
                    const uint32_t w4 = *(const uint32_t*)(sym + i);  // within the staging area
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j) {
                        const uint32_t at = (j ? w4 >> (8 * j - 1) : w4 << 1) & 0x7Cu;
                        atomicAdd((uint32_t*)((char*)hist + at), ((w4 >> (8 * j)) & 1u) << 16 | 1u);
                    }
                }
            const uint32_t cnt_lo = __shfl((int)plane_count, 0), cnt_hi = __shfl((int)plane_count, 32);
            // 64-byte aligned: the MQ coder reads a plane in 64-byte groups
            const uint32_t al_lo = (cnt_lo + 63u) & ~63u, al_hi = (cnt_hi + 63u) & ~63u;
            if (chunk_cur + al_lo + al_hi > chunk_end) {
                const unsigned long long want = kChunkBytes > al_lo + al_hi ? kChunkBytes : al_lo + al_hi;
                unsigned long long got = 0;
                if (lane == 0) got = atomicAdd(&P.counters->sym_next, want);
                got = __shfl((long long)got, 0);
                chunk_cur = got;
                chunk_end = got + want;
                if (chunk_end > P.pool_cap && lane == 0) atomicOr(&P.counters->flags, 1u);
            }
            const unsigned long long off = chunk_cur + (half ? al_lo : 0u);
            chunk_cur += al_lo + al_hi;
            const bool fits = chunk_end <= P.pool_cap;
            if (act && fits) {
                for (uint32_t i = (uint32_t)x * 16u; i < plane_count; i += 512u)
                    *(uint4*)(P.pool + off + i) = *(const uint4*)(sym + i);
                if (x == 0) P.chunks[(size_t)cb * kMaxPlanes + j] = make_uint2((uint32_t)(off >> 4), plane_count);
            }
            if (act) ++planes;
            wave_sync();
            // ---- early termination after plane p > 0 (t1_ref.cpp:128-162)
            bool stop_now = false;
            if (__any(track)) {
                float term = 0.f;
                if (track && x < 19) {
                    const uint32_t hv = hist[x];
                    const uint32_t n = hv & 0xFFFFu, n1 = hv >> 16, n0 = n - n1;
                    if (n > 0 && n <= kLog2Max) {
                        const float* row = P.log2tab + (size_t)n * (n + 1) / 2;
                        const float a = (float)n0 * row[n0];
                        const float b = (float)n1 * row[n1];
                        term = -(a + b) + 2.f;
                    }
                }
                if (x < 20) terms[x] = term;
                wave_sync();
                if (track && x < 20) hist[x] = 0;
                float bits = 0.f;  // the contexts' terms summed in context order
                {
                    float4 tv[5];
#pragma unroll
                    for (int k = 0; k < 5; ++k) tv[k] = ((const float4*)terms)[k];
#pragma unroll
                    for (int k = 0; k < 5; ++k) {
                        bits += tv[k].x;
                        bits += tv[k].y;
                        bits += tv[k].z;
                        if (k < 4) bits += tv[k].w;
                    }
                }
                const float bytes = bits * 0.125f + 1.f;
                bool cand = track && act && p > 0;
                float dabs = 0.f;
                if (cand) dabs = (float)plane_dist * ldexpf(1.0f, 2 * p) * (1.f / 4096.f) * band.dist_scale;
                cand = cand && dabs < thr * bytes;
                if (__any(cand)) {
                    // Remaining squared error (t1_ref.cpp:142-154): the CPU sums the samples'
                    // float terms in row-major order. That float sum of at most 1,024
                    // non-negative terms is within 1023 * 2^-24 (< 6.2e-5, relative) of their
                    // exact sum; the half-wave's sum (float column sums, within 31 * 2^-24,
                    // then a double shuffle tree) is within 2e-6 of it. Unless that sum lies
                    // within 1e-4 of the threshold it decides the comparison the same way;
                    // only then is the row-major float sum formed.
                    const int pp = act ? p : 0;
                    const float step = ldexpf(1.0f, pp);
                    auto term = [&](uint32_t mm) {
                        const float v = (float)mm * (1.f / 64.f);
                        const uint32_t q = mm >> (pp + 6);
                        const float rec = q == 0 ? 0.f : ((float)q + 0.5f) * step;
                        const float dd = v - rec;
                        return dd * dd;
                    };
                    float col = 0.f;
#pragma unroll
                    for (int r = 0; r < 32; ++r)
                        if (x < w && r < h) col += term(m[r]);
                    const double lhs = half_sum_d((double)col) * (double)band.dist_scale;
                    const double T = (double)(thr * bytes);
                    const bool low = lhs * (1.0 + 1e-4) < T, high = lhs * (1.0 - 1e-4) >= T;
                    const bool unsure = cand && !low && !high;
                    bool stop = cand && low;
                    if (__any(unsure)) {
                        float e = 0.f;
                        float* scratch = (float*)sym;
#pragma unroll
                        for (int part = 0; part < 2; ++part) {
#pragma unroll
                            for (int rr = 0; rr < 16; ++rr) {
                                uint32_t mm = m[part * 16 + rr];
                                asm volatile("" : "+v"(mm));  // recomputed here, not kept from the fast path
                                scratch[rr * 32 + x] = term(mm);
                            }
                            wave_sync();
                            if (x == 0 && unsure) {
                                const int r1 = h < part * 16 + 16 ? h : part * 16 + 16;
                                for (int r = part * 16; r < r1; ++r)
                                    for (int c = 0; c < w; ++c) e += scratch[(r - part * 16) * 32 + c];
                            }
                            wave_sync();
                        }
                        e = __shfl(e, half << 5);
                        if (unsure) stop = e * band.dist_scale < thr * bytes;
                    }
                    stop_now = stop;
                }
            }
            if (act && (stop_now || np >= P.max_passes)) done = true;
            if (!act) done = true;
        }
        if (has && x == 0) {
            T1Info inf;
            inf.nbps = (uint32_t)(nbps <= kMaxPlanes ? nbps : 0);
            inf.passes = np;
            inf.planes = planes;
            inf.symbols = sym_total;
            P.info[cb] = inf;
            if (nbps > kMaxPlanes) atomicOr(&P.counters->flags, 4u);
        }
    }
}

hipError_t launch_t1_cm(const CmParams& p, int waves, int groups, hipStream_t s) {
    switch (waves) {
    case 1: hipLaunchKernelGGL(t1_cm_kernel<1>, dim3(groups), dim3(64), 0, s, p); break;
    case 2: hipLaunchKernelGGL(t1_cm_kernel<2>, dim3(groups), dim3(128), 0, s, p); break;
    case 8: hipLaunchKernelGGL(t1_cm_kernel<8>, dim3(groups), dim3(512), 0, s, p); break;
    default: hipLaunchKernelGGL(t1_cm_kernel<4>, dim3(groups), dim3(256), 0, s, p); break;
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------- ordering and offsets
// Before MQ coding: a counting sort of the blocks by symbol count, largest first (128 buckets,
// four per octave), and the exclusive sum of their codewords' capacities; before compaction: the
// exclusive sum of what is kept. Each takes two launches over groups of kPlanSpan blocks: the
// first counts and sums per group, and in the second every group adds up the counts and sums
// of those before it for itself. These kernels do next to nothing and cost their launch, 4 us and
// more each, so there are few: with the clearing, the scans of the counts and of the sums and the
// capacities' own two passes as separate launches, ten in all, these kernels took 59 us of one 4K
// frame, now 20; of 16 frames 102, now 49.
namespace {
constexpr int kBuckets = 128;
constexpr int kPlanSpan = kPlanGroupBlocks;  // blocks per workgroup
constexpr int kPlanPer = kPlanSpan / 256;
static_assert(kOrderWords == 2 * kBuckets);

__device__ __forceinline__ uint32_t bucket_of(uint32_t s) {
    if (s < 4) return kBuckets - 1;
    const int l = 31 - __clz((int)s);
    const uint32_t sub = (s >> (l - 2)) & 3u;
    const uint32_t b = (uint32_t)l * 4 + sub;
    return kBuckets - 1 - (b < kBuckets - 1 ? b : kBuckets - 1);
}

__device__ __forceinline__ uint32_t out_capacity(const T1Info& f) {
    // A block's codeword never needs more than half a byte per symbol plus the flush; a
    // block that still overflows is reported and the job re-run with more room.
    return f.passes ? ((f.symbols / 2u + 64u + 63u) & ~63u) : 0u;
}

// The sum of v over the 256 threads, in every thread; s holds 4 values.
__device__ __forceinline__ unsigned long long group_sum(unsigned long long v, unsigned long long* s) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
    __syncthreads();
    v = s[0] + s[1] + s[2] + s[3];
    __syncthreads();
    return v;
}

// The sum of v over the threads before this one.
__device__ __forceinline__ unsigned long long group_before(unsigned long long v, unsigned long long* s) {
    unsigned long long inc = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned long long u = __shfl_up(inc, o);
        if ((threadIdx.x & 63) >= (unsigned)o) inc += u;
    }
    if ((threadIdx.x & 63) == 63) s[threadIdx.x >> 6] = inc;
    __syncthreads();
    unsigned long long base = 0;
    for (unsigned k = 0; k < (threadIdx.x >> 6); ++k) base += s[k];
    __syncthreads();
    return base + inc - v;
}

// The sum of the groups' values before group g.
__device__ __forceinline__ unsigned long long groups_before(const unsigned long long* partial, uint32_t g,
                                                            unsigned long long* s) {
    unsigned long long v = 0;
    for (uint32_t i = threadIdx.x; i < g; i += 256) v += partial[i];
    return group_sum(v, s);
}
}  // namespace

__global__ void __launch_bounds__(256) plan_count_kernel(const T1Info* info, uint32_t n, uint32_t* order,
                                                         unsigned long long* partial, JobCounters* counters) {
    __shared__ uint32_t h[kBuckets];
    __shared__ unsigned long long s[4];
    if (threadIdx.x < kBuckets) h[threadIdx.x] = 0;
    __syncthreads();
    unsigned long long symbols = 0, bytes = 0;
    for (uint32_t j = 0; j < kPlanPer; ++j) {
        const uint32_t i = blockIdx.x * kPlanSpan + 256 * j + threadIdx.x;
        if (i >= n) break;
        const T1Info f = info[i];
        symbols += f.symbols;
        bytes += out_capacity(f);
        atomicAdd(&h[bucket_of(f.symbols)], 1u);
    }
    symbols = group_sum(symbols, s);  // its barriers also end the counting
    bytes = group_sum(bytes, s);
    if (threadIdx.x < kBuckets && h[threadIdx.x]) atomicAdd(&order[threadIdx.x], h[threadIdx.x]);
    if (threadIdx.x == 0) {
        partial[blockIdx.x] = bytes;
        atomicAdd(&counters->symbols, symbols);
    }
}

__global__ void __launch_bounds__(256) plan_place_kernel(const T1Info* info, uint32_t n, uint32_t* order,
                                                         const unsigned long long* partial, uint32_t* perm,
                                                         unsigned long long* out_off) {
    __shared__ uint32_t h[kBuckets], base[kBuckets];
    __shared__ unsigned long long s[4];
    if (threadIdx.x < kBuckets) h[threadIdx.x] = 0;
    const unsigned long long start = group_before(threadIdx.x < kBuckets ? order[threadIdx.x] : 0u, s);
    unsigned long long run = groups_before(partial, blockIdx.x, s);
    const uint32_t i0 = blockIdx.x * kPlanSpan + kPlanPer * threadIdx.x;
    T1Info f[kPlanPer];
    unsigned long long bytes = 0;
#pragma unroll
    for (uint32_t j = 0; j < kPlanPer; ++j) {
        f[j] = i0 + j < n ? info[i0 + j] : T1Info{};
        bytes += out_capacity(f[j]);
        if (i0 + j < n) atomicAdd(&h[bucket_of(f[j].symbols)], 1u);
    }
    run += group_before(bytes, s);
#pragma unroll
    for (uint32_t j = 0; j < kPlanPer; ++j) {
        if (i0 + j < n) out_off[i0 + j] = run;
        run += out_capacity(f[j]);
    }
    // one reservation per bucket and group, in the bucket's cursor
    if (threadIdx.x < kBuckets) {
        base[threadIdx.x] =
            (uint32_t)start + (h[threadIdx.x] ? atomicAdd(&order[kBuckets + threadIdx.x], h[threadIdx.x]) : 0u);
        h[threadIdx.x] = 0;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kPlanPer; ++j)
        if (i0 + j < n) {
            const uint32_t b = bucket_of(f[j].symbols);
            perm[base[b] + atomicAdd(&h[b], 1u)] = i0 + j;
        }
}

hipError_t launch_plan(const T1Info* info, uint32_t n, uint32_t* order, uint32_t* perm, unsigned long long* out_off,
                       unsigned long long* partial, JobCounters* counters, hipStream_t s) {
    const uint32_t groups = (n + kPlanSpan - 1) / kPlanSpan;
    hipLaunchKernelGGL(plan_count_kernel, dim3(groups), dim3(256), 0, s, info, n, order, partial, counters);
    hipLaunchKernelGGL(plan_place_kernel, dim3(groups), dim3(256), 0, s, info, n, order, partial, perm, out_off);
    return hipGetLastError();
}

// What a block keeps: its codeword's bytes in whole words, and its passes << 36.
__device__ __forceinline__ unsigned long long kept_size(const T1Info* info, const uint32_t* len, uint32_t i) {
    return (unsigned long long)((len[i] + 3u) & ~3u) | ((unsigned long long)info[i].passes << 36);
}

__global__ void __launch_bounds__(256) data_sizes_kernel(const T1Info* info, const uint32_t* len, uint32_t n,
                                                         unsigned long long* partial) {
    __shared__ unsigned long long s[4];
    unsigned long long v = 0;
    for (uint32_t j = 0; j < kPlanPer; ++j) {
        const uint32_t i = blockIdx.x * kPlanSpan + 256 * j + threadIdx.x;
        if (i < n) v += kept_size(info, len, i);
    }
    v = group_sum(v, s);
    if (threadIdx.x == 0) partial[blockIdx.x] = v;
}

__global__ void __launch_bounds__(256) data_offsets_kernel(const T1Info* info, const uint32_t* len, uint32_t n,
                                                           const unsigned long long* partial,
                                                           unsigned long long* data_off, JobCounters* counters) {
    __shared__ unsigned long long s[4];
    unsigned long long run = groups_before(partial, blockIdx.x, s);
    const uint32_t i0 = blockIdx.x * kPlanSpan + kPlanPer * threadIdx.x;
    unsigned long long v[kPlanPer], sum = 0;
#pragma unroll
    for (uint32_t j = 0; j < kPlanPer; ++j) {
        v[j] = i0 + j < n ? kept_size(info, len, i0 + j) : 0ull;
        sum += v[j];
    }
    run += group_before(sum, s);
#pragma unroll
    for (uint32_t j = 0; j < kPlanPer; ++j) {
        if (i0 + j < n) data_off[i0 + j] = run;
        run += v[j];
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 255) counters->kept = run;
}

hipError_t launch_compact_offsets(const T1Info* info, const uint32_t* code_len, uint32_t n,
                                  unsigned long long* data_off, unsigned long long* partial, JobCounters* counters,
                                  hipStream_t s) {
    const uint32_t groups = (n + kPlanSpan - 1) / kPlanSpan;
    hipLaunchKernelGGL(data_sizes_kernel, dim3(groups), dim3(256), 0, s, info, code_len, n, partial);
    hipLaunchKernelGGL(data_offsets_kernel, dim3(groups), dim3(256), 0, s, info, code_len, n, partial, data_off, counters);
    return hipGetLastError();
}

// ---------------------------------------------------------------- MQ coding
namespace {
// The coder's states (t1_tables.h: build_mq_coder_table).
__constant__ uint32_t kMqTable[2 * kMqCoderStates];
__constant__ uint32_t kMqInitial[4];  // contexts start in states 0, 4 (zero coding 0), 3 (run length), 46 (uniform)

}  // namespace

// The MQ encoder (C.2) with its byte-outs put off. The code register L holds C << 5 in 64
// bits: bits 5-31 are the 27 bits below the carry, bit 32 is the carry into the pending byte B,
// and whatever has been shifted past it are bytes that BYTEOUT (C.2.7) has not taken yet. D is
// CT + 16, so BYTEOUT is due when D <= 16 and must run before D would fall below -15.
//
// Taking bytes late gives the same bytes as taking them at once, except where an addition
// carries into a byte of 0xFF that is due but not taken: a byte of 0xFF takes no carry, which
// goes to the bit stuffed after it. Such a carry passes bit 31 on its way up, so the caller
// takes every byte that is due before it makes an addition that carries out of bit 31.
struct MqCode {
    uint64_t L;
    int32_t D;
    uint32_t B;
    int32_t bp;  // index of the pending byte

    // BYTEOUT, due (D <= 16): returns the byte at bp, final, and the next one becomes pending;
    // the caller counts bp on.
    __device__ __forceinline__ uint32_t byteout() {
        const int sh = 40 - D;
        const uint32_t X = (uint32_t)(L >> sh);  // carry and the 8 bits of the byte due
        const uint32_t carry = B != 0xFFu ? X >> 8 : 0u;
        const uint32_t byte = B + carry;
        const uint32_t stuff = byte == 0xFFu ? 1u : 0u;
        L -= (uint64_t)(X & ~stuff) << sh;
        B = (X - (carry << 8)) >> stuff;
        D += 8 - (int)stuff;
        return byte;
    }
};

// Truncation length of every pass but the last (mq_encoder.h:146-169): the shortest prefix,
// never ending in 0xFF, that with the decoder's 1-fill stays inside the interval the coder had
// at the pass end. out holds the block's len codeword bytes, readable to cap (a multiple of 64).
// At most 6 bytes decide a pass: they are read at once, the next snapshot one pass ahead.
__device__ __forceinline__ void mq_pass_lengths(const uint8_t* out, uint32_t len, uint32_t cap, const MqSnapshot* snaps,
                                                uint32_t np, uint32_t* plen) {
    uint32_t prev = 1;
    MqSnapshot next = snaps[0];
    for (uint32_t q = 0; q + 1 < np; ++q) {
        const MqSnapshot sn = next;
        next = snaps[q + 1];
        MqCode m{((uint64_t)sn.c_hi << 32) | sn.c_lo, (int32_t)(sn.bp_b_d & 0xFFu), (sn.bp_b_d >> 8) & 0xFFu,
                 (int32_t)(sn.bp_b_d >> 16) - 1};
        for (; m.D <= 16; ++m.bp) m.byteout();
        const uint32_t at = m.bp < 0 ? 0u : (uint32_t)m.bp, g = at & ~7u, r = 8u * (at & 7u);
        const uint64_t g0 = g < cap ? *(const uint64_t*)(out + g) : 0ull;
        const uint64_t g1 = g + 8u < cap ? *(const uint64_t*)(out + g + 8u) : 0ull;
        uint64_t bytes = (g0 >> r) | ((g1 << 1) << (63u - r));
        if (m.bp < 0) bytes <<= 8;  // the dummy byte
        const int base_sh = 43 - (m.D - 16);
        const unsigned long long low = ((unsigned long long)m.B << base_sh) + (m.L << 11);
        const unsigned long long high = low + sn.a;
        unsigned long long prefix = 0;
        int sh = base_sh;
        uint32_t L = len;
        for (int i = m.bp; i < (int)len && sh >= 0; ++i) {
            const uint32_t byte = (uint32_t)bytes & 0xFFu;
            bytes >>= 8;
            prefix += (unsigned long long)byte << sh;
            const unsigned long long tail = prefix + (1ull << sh);
            if ((uint32_t)(i + 1) >= prev && byte != 0xFFu && tail <= high && tail > low) {
                L = (uint32_t)(i + 1);
                break;
            }
            sh -= byte == 0xFFu ? 7 : 8;
        }
        plen[q] = L;
        prev = L > prev ? L : prev;
    }
    plen[np - 1] = len;
}

// One lane per code-block, P.lanes blocks per wave. GROUP lanes per workgroup; NQ: 16-byte
// groups of symbols read per lane at a time (1 or 4), the following ones in flight while these
// are coded. A lane goes on to its next plane by itself; the lanes of a wave only share the
// steps within NQ groups.
//
// Large launches are bound by VALU issue: 40 wave-instructions per 64 symbols (35 in the four
// unrolled steps of a word, the rest bytes taken, pass ends and the cursor), 2.12 ms for 16 4K
// frames (1,650 M symbols) where a coder that took each byte when it was due spent 94 and
// 6.1 ms: some lane of 64 had a byte on nearly every step. Small launches are bound by the
// longest block's chain: about 155 cycles a symbol in the steps (state -> successors from LDS ->
// state, the interval beside it) and 60-130 in the rest; one 4K frame 1.63 ms (3.0 before), one
// 512x256 frame 1.23 ms (2.1). What shapes the steps is latency: a dependent VALU operation
// takes 9 cycles, LDS 50, but a mask that goes through a scalar instruction 20 more and a
// branch on a vector comparison 28, so there are no scalar mask operations in the steps and
// one branch per four symbols.
template <int GROUP, int NQ>
__global__ void __launch_bounds__(GROUP) t1_mq_kernel(MqParams P) {
    __shared__ uint32_t s_ctx[kMqContexts][GROUP];
    __shared__ uint2 s_next[kMqCoderStates];
    for (int i = threadIdx.x; i < kMqCoderStates; i += GROUP)
        s_next[i] = make_uint2(kMqTable[2 * i], kMqTable[2 * i + 1]);
    __syncthreads();
    // A full symbol pool left some chunk tables unwritten: nothing to code, the host
    // re-runs Tier-1 with a larger pool.
    if (P.counters->flags & 1u) return;
    const int t = threadIdx.x;
    const uint32_t lane = (uint32_t)t & 63u;
    // Lanes beyond P.lanes code the same blocks again, to the same bytes: a wave of a few active
    // lanes runs slower than a full one (a dependent VALU operation takes 17-23 cycles instead
    // of 9 in waves of one active lane, four to a CU).
    const uint32_t mine = lane % P.lanes;
    // the lane's context states, GROUP words apart
    char* const slots = (char*)&s_ctx[0][t];
    constexpr int kSlotShift = GROUP == 64 ? 8 : (GROUP == 128 ? 9 : 10);
    for (;;) {
        // P.lanes blocks at a time, in largest-first order
        uint32_t base = 0;
        if (lane == 0) base = atomicAdd(P.work_next, P.lanes);
        base = (uint32_t)__builtin_amdgcn_readfirstlane(__shfl((int)base, 0));
        if (base >= P.nblocks) break;
        const uint32_t cb = P.perm[min(base + mine, P.nblocks - 1u)];
        const T1Info inf = P.info[cb];
        const uint32_t np = inf.passes;
        if (np == 0) {
            P.code_len[cb] = 0;
            continue;
        }
        const unsigned long long obase = P.out_off[cb];
        uint8_t* out = P.out + obase;
        uint32_t cap = out_capacity(inf);  // a multiple of 64, as every block's offset
        if (obase + cap > P.out_cap) cap = 0;
        for (int i = 0; i < 19; ++i) s_ctx[i][t] = kMqInitial[0];
        s_ctx[0][t] = kMqInitial[1];
        s_ctx[17][t] = kMqInitial[2];
        s_ctx[18][t] = kMqInitial[3];
        s_ctx[19][t] = 0;          // neutral symbols: Qe = 0, always the MPS
        uint32_t A = 0x80000000u;  // A << 16
        MqCode m{0ull, 12 + 16, 0u, -1};
        // The bp & 7 finished bytes of the current aligned 8-byte group, the last one lowest. The
        // byte at bp = -1 is the coder's initial dummy: it is 0 and takes no carry (C + A stays
        // within 2^27 until the first byte-out), and ends a group that is not written.
        uint64_t acc = 0ull;
        // count (1..4) finished bytes, the last one lowest
        auto put = [&](uint32_t bytes, uint32_t count) {
            const uint32_t have = ((uint32_t)m.bp & 7u) + count;
            if (have < 8u) {
                acc = (acc << (8u * count)) | bytes;
            } else {
                const uint32_t over = have - 8u;
                const uint64_t group = (acc << (8u * (count - over))) | (bytes >> (8u * over));
                const uint32_t at = (uint32_t)m.bp & ~7u;
                if (at < cap) *(uint64_t*)(out + at) = __builtin_bswap64(group);  // cap: a multiple of 64
                acc = bytes & ((1u << (8u * over)) - 1u);
            }
            m.bp += (int)count;
        };
        // BYTEOUT for every byte that is due
        auto take_bytes = [&]() {
            if (m.D <= 16) {
                // all of them at once unless one is 0xFF: the pending byte with its carry and
                // the due ones but the last, which becomes the pending one
                const uint32_t k = 16u - (uint32_t)m.D, count = (k >> 3) + 1u, sh = 24u + (k & 7u);
                const uint64_t V = m.L >> sh;
                const uint32_t bytes = (m.B << (8u * (count - 1u))) + (uint32_t)(V >> 8);
                if (m.B != 0xFFu && !((~bytes - 0x01010101u) & bytes & 0x80808080u)) {
                    put(bytes, count);
                    m.L -= V << sh;
                    m.B = (uint32_t)V & 0xFFu;
                    m.D += (int)(8u * count);
                } else {
                    do put(m.byteout(), 1u);
                    while (m.D <= 16);
                }
            }
        };
        MqSnapshot* snap = P.snaps + (size_t)cb * kMaxPasses;
        const uint2* chunk = P.chunks + (size_t)cb * kMaxPlanes;
        const uint32_t planes = inf.planes;
        // The groups are read two steps ahead: q is being coded, n has arrived (the last symbol
        // of q looks up the first context of n), the next are in flight. A plane's symbols start
        // 64-byte aligned and take a multiple of 64 bytes of the pool, so NQ groups can be read
        // from any multiple of NQ.
        // No load depends on a condition and what is loaded is next touched a step later, so that
        // no step waits for memory.
        const uint2 ch = chunk[0];
        const uint8_t* src = P.pool + ((unsigned long long)ch.x << 4);
        uint32_t left = ch.y >> 4;  // 16-byte groups from src to the end of the plane; 0: no more
        uint32_t j = planes > 1 ? 1u : 0u;
        uint2 chn = chunk[j];       // the next plane's, if j is one
        // the groups at src (the pool's first when there are no more), how many of them are the
        // plane's, and on to the next
        auto read = [&](uint4(&g)[NQ]) {
#pragma unroll
            for (int e = 0; e < NQ; ++e) g[e] = *(const uint4*)(src + 16 * e);
            const uint32_t count = left < (uint32_t)NQ ? left : (uint32_t)NQ;
            const bool more = left > (uint32_t)NQ;
            const uint8_t* const next = P.pool + ((unsigned long long)chn.x << 4);
            src = more ? src + 16 * NQ : next;
            left = more ? left - NQ : (j ? chn.y >> 4 : 0u);
            j = more ? j : (j && j + 1 < planes ? j + 1 : 0u);
            chn = chunk[j];
            return count;
        };
        uint4 q[NQ], n[NQ];
        uint32_t nq = read(q), nn = read(n);
        // the state of the next symbol's context and that context's slot
        uint32_t* cslot = (uint32_t*)(slots + (((q[0].x & 0xFFu) >> 1) << kSlotShift));
        uint32_t t_cur = *cslot;
        for (;;) {
            uint4 f[NQ];
            const uint32_t nf = read(f);
#pragma unroll 1
            for (uint32_t sub = 0; sub < (uint32_t)NQ; ++sub) {
                if (sub < nq) {
                    uint32_t w = q[0].x, w1 = q[0].y, w2 = q[0].z, w3 = q[0].w;
                    const uint32_t w4 = NQ > 1 && sub + 1 < nq ? q[NQ > 1 ? 1 : 0].x : (nn ? n[0].x : 0u);
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        // Four symbols with the code register assumed to hold them: no byte is
                        // taken, and what would have needed it is looked at after them.
                        const uint64_t L0 = m.L;
                        const int32_t D0 = m.D;
                        uint32_t adds[4], shifts[4], carries = 0;
#pragma unroll
                        for (int b = 0; b < 4; ++b) {
                            // the next symbol's context state, read before this symbol may change it
                            const uint32_t nctx = b < 3 ? (w >> (8 * b + 9)) & 31u : (w1 >> 1) & 31u;
                            uint32_t* const nslot = (uint32_t*)(slots + (nctx << kSlotShift));
                            const uint32_t t_next = *nslot;
                            const uint32_t st = t_cur;
                            const uint2 succ = *(const uint2*)((const char*)s_next + (st & 0x3F8u));
                            const bool lps = (int)(st ^ (w << (31 - 8 * b))) < 0;
                            // C.2.5 / C.2.6 with the conditional exchange: the MPS takes the
                            // larger of a and Qe, the LPS the smaller; C grows by Qe where a,
                            // the upper part, is taken (on a tie: by the MPS)
                            const uint32_t qe = st & 0x7FFF0000u;
                            const uint32_t a = A - qe;
                            const uint32_t hi = a > qe ? a : qe, lo = a < qe ? a : qe;
                            const uint32_t below = a < qe ? qe : 0u;
                            const uint32_t add = (lps ? below : qe - below) >> 11;
                            A = lps ? lo : hi;
                            // The state changes and A, C renormalise unless the symbol is the
                            // MPS with A still >= 0x8000; then the shift count is 0 and the
                            // state written back is the old one, so every lane runs the same
                            // instructions.
                            const uint32_t t_new = lps ? succ.y : succ.x;
                            const uint32_t st_new = (int)A < 0 ? st : t_new;
                            *cslot = st_new;
                            const uint32_t nsh = (uint32_t)__builtin_clz(A);  // A is never 0
                            A <<= nsh;
                            uint32_t low;
                            carries += __builtin_add_overflow((uint32_t)m.L, add, &low) ? 1u : 0u;
                            m.L = ((m.L & 0xFFFFFFFF00000000ull) | low) << nsh;
                            m.D -= (int)nsh;
                            adds[b] = add;
                            shifts[b] = nsh;
                            t_cur = nslot == cslot ? st_new : t_next;
                            cslot = nslot;
                        }
                        // a pass ends with the word (its top bit), or the register wants looking at
                        if (__builtin_amdgcn_ballot_w64((m.D | (int32_t)w | (int32_t)(0u - carries)) < 0)) {
                            asm volatile("");
                            if (__builtin_amdgcn_ballot_w64((m.D | (int32_t)(0u - carries)) < 0)) {
                                // The bytes due, of all lanes, so that they are due at the same
                                // time again. After a carry out of bit 31 (about 1 addition in
                                // 4,000) or more shifts than the register holds, the symbols'
                                // additions and shifts once more with the bytes taken in between.
                                int r = 4;
                                if (__builtin_amdgcn_ballot_w64(carries != 0u || m.D < -15)) {
                                    m.L = L0;
                                    m.D = D0;
                                    r = 0;
                                }
                                for (;; ++r) {
                                    take_bytes();
                                    if (r == 4) break;
                                    m.L = (m.L + adds[0]) << shifts[0];
                                    m.D -= (int)shifts[0];
                                    adds[0] = adds[1], adds[1] = adds[2], adds[2] = adds[3];
                                    shifts[0] = shifts[1], shifts[1] = shifts[2], shifts[2] = shifts[3];
                                }
                            }
                            if ((int32_t)w < 0)  // the coder state is the truncation reference of the pass
                                *snap++ = MqSnapshot{((uint32_t)(m.bp + 1) << 16) | (m.B << 8) | (uint32_t)m.D,
                                                     (uint32_t)m.L, (uint32_t)(m.L >> 32), A};
                        }
                        w = w1;
                        w1 = w2;
                        w2 = w3;
                        w3 = w4;
                    }
                }
#pragma unroll
                for (int e = 0; e + 1 < NQ; ++e) q[e] = q[e + 1];
            }
            if (!nn) break;
#pragma unroll
            for (int e = 0; e < NQ; ++e) q[e] = n[e], n[e] = f[e];
            nq = nn;
            nn = nf;
        }
        // FLUSH (C.2.9)
        take_bytes();
        {
            uint32_t C = (uint32_t)(m.L >> 5);
            const uint32_t tempc = C + (A >> 16);
            C |= 0xFFFFu;
            if (C >= tempc) C -= 0x8000u;
            m.L = (uint64_t)C << 5;
        }
#pragma unroll 1
        for (int k = 0; k < 2; ++k) {
            m.L <<= m.D - 16;
            m.D = 16;
            take_bytes();
        }
        const uint32_t flushed = (uint32_t)m.bp & ~7u;  // codeword bytes already written out
        uint32_t len = (uint32_t)m.bp, have = len & 7u;
        if (m.B != 0xFFu) {
            acc = (acc << 8) | m.B;
            ++len;
            ++have;
        }
        acc = have ? __builtin_bswap64(acc << (8u * (8u - have))) : 0ull;
        if (len > cap) {
            atomicOr(&P.counters->flags, 2u);
            P.code_len[cb] = 0;
            continue;
        }
        // the bytes after the last full group, as whole words
        const uint32_t nw = (len + 3u) >> 2;
        for (uint32_t wi = flushed >> 2; wi < nw; ++wi)
            *(uint32_t*)(out + 4u * wi) = (uint32_t)(acc >> (32u * (wi & 1u)));
        mq_pass_lengths(out, len, cap, P.snaps + (size_t)cb * kMaxPasses, np, P.pass_len + (size_t)cb * kMaxPasses);
        P.code_len[cb] = len;
    }
}

static hipError_t upload_mq_table() {
    uint32_t tab[2 * kMqCoderStates], initial[4];
    build_mq_coder_table(tab, initial, 16);
    const hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(kMqTable), tab, sizeof tab);
    return e != hipSuccess ? e : hipMemcpyToSymbol(HIP_SYMBOL(kMqInitial), initial, sizeof initial);
}

hipError_t t1_tables_init() { return upload_mq_table(); }

hipError_t launch_t1_mq(const MqParams& p, int group, int read_bytes, int groups, hipStream_t s) {
    const bool wide = read_bytes >= 64;
    switch (group) {
    case 64:
        if (wide) hipLaunchKernelGGL((t1_mq_kernel<64, 4>), dim3(groups), dim3(64), 0, s, p);
        else hipLaunchKernelGGL((t1_mq_kernel<64, 1>), dim3(groups), dim3(64), 0, s, p);
        break;
    case 128:
        if (wide) hipLaunchKernelGGL((t1_mq_kernel<128, 4>), dim3(groups), dim3(128), 0, s, p);
        else hipLaunchKernelGGL((t1_mq_kernel<128, 1>), dim3(groups), dim3(128), 0, s, p);
        break;
    default:
        if (wide) hipLaunchKernelGGL((t1_mq_kernel<256, 4>), dim3(groups), dim3(256), 0, s, p);
        else hipLaunchKernelGGL((t1_mq_kernel<256, 1>), dim3(groups), dim3(256), 0, s, p);
        break;
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------- compaction
// One wave per block: info record, pass tables and the codeword into dense arrays.
__global__ void __launch_bounds__(256) compact_kernel(CompactParams P) {
    if (P.counters->flags & 3u) return;  // the run is repeated with larger buffers
    const uint32_t cb = blockIdx.x * 4 + (threadIdx.x >> 6);
    const uint32_t l = threadIdx.x & 63;
    if (cb >= P.nblocks) return;
    const T1Info inf = P.info[cb];
    const uint32_t len = P.code_len[cb];
    const unsigned long long packed = P.data_off[cb];
    const unsigned long long doff = packed & ((1ull << 36) - 1);
    const uint32_t poff = (uint32_t)(packed >> 36);
    if (l == 0) {
        uint32_t* di = P.dense_info + 5 * (size_t)cb;
        di[0] = inf.nbps;
        di[1] = inf.passes;
        di[2] = (uint32_t)doff;
        di[3] = len;
        di[4] = poff;
    }
    if (l < inf.passes) {
        P.dense_pass_len[poff + l] = P.pass_len[(size_t)cb * kMaxPasses + l];
        P.dense_pass_dist[poff + l] = P.pass_dist[(size_t)cb * kMaxPasses + l];
    }
    const uint32_t words = (len + 3) >> 2;
    const uint32_t* s = (const uint32_t*)(P.out + P.out_off[cb]);
    uint32_t* d = (uint32_t*)(P.dense_data + doff);
    for (uint32_t i = l; i < words; i += 64) d[i] = s[i];
}

hipError_t launch_compact(const CompactParams& p, hipStream_t s) {
    hipLaunchKernelGGL(compact_kernel, dim3((p.nblocks + 3) / 4), dim3(256), 0, s, p);
    return hipGetLastError();
}

}  // namespace gail_amd
