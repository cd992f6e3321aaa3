// PCRD-opt rate control on the GPU (rate_control.cpp:11-279 with the Tier-2 sizes of
// t2.cpp:31-254), between MQ coding and compaction, so the rate-control state stays in HBM
// and only the kept bytes of each code-block leave the GPU. The launches, in order:
//
//   rc_hull_kernel   one thread per code-block of every frame: the block's hull
//                    (rc_block_hull_to), stored point-major ([point][block]) so that the
//                    lanes of a wave read neighbouring blocks' points together, each point's
//                    slope bin floor(1024 log2 s), and per workgroup the smallest and largest
//                    finite slope;
//   rc_range_kernel  one workgroup per frame: the frame's slope range and histogram bins;
//   rc_fill_kernel   one thread per code-block: the slope histogram (bytes and included
//                    blocks per component, 32-bit integer atomics);
//   rc_scan_kernel   two passes over 1,024-bin segments: suffix sums of the histogram;
//   rc_measure_kernel  a few times: a size measurement of every frame, one wave per packet
//                    (its blocks' choices, then its exact size), the tile-part sums in global
//                    memory; the workgroup that is last to finish a frame runs one step of the
//                    search of rc_shared.h. A frame whose search is over does nothing.
//   rc_finish_kernel one workgroup per frame: any further steps of the search, and the result;
//   rc_dist_kernel   the distortion left, and the histogram bins the run used cleared, so that
//                    every run finds them zero.
//
// The host library runs the same shared code, so both choose the same passes.
#include <hip/hip_runtime.h>

#include "device_types.h"
#include "kernels.h"
#include "rc_shared.h"

namespace gail_amd {

// A frame's search between the launches of a run.
struct RcRun {
    RcSearch search;
    unsigned long long tp[6];  // tile-part bytes of the measurement under way
    uint32_t arrived;          // its workgroups that are through
    uint32_t done;
    uint32_t summed;           // workgroups of rc_dist_kernel that are through
};

namespace {

// LDS written by other lanes of the wave is read after this.
__device__ __forceinline__ void lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int kHullGroup = kRcPartBlocks;  // blocks per hull workgroup (one partial slope range each)
constexpr int kHullThreads = 256;          // blocks per fill workgroup
constexpr int kScanThreads = 256;
constexpr int kScanBins = 4 * kScanThreads;  // bins per scan workgroup
constexpr int kScanSegs = (kRcMaxBins + 1 + kScanBins - 1) / kScanBins;
constexpr int kMeasureWaves = 4;   // packets per workgroup of a measurement
constexpr int kFinishWaves = 16;
constexpr int kMeasureLaunches = 6;
constexpr int32_t kBinAbove = 0x7FFFFFFF;      // slope bin of an infinite slope
constexpr int32_t kBinBelow = -0x7FFFFFFF - 1;  // of a slope <= 0

__device__ __forceinline__ uint32_t* hist_of(const RcParams& P, uint32_t f, int a) {
    return P.hist + ((size_t)f * 6 + (size_t)a) * (kRcMaxBins + 1);
}

// Partial slope range of hull workgroup x of frame f: frames never share an entry.
__device__ __forceinline__ uint32_t part_index(const RcFrame& F, uint32_t f, uint32_t x) {
    return F.first_block / kHullGroup + f + x;
}

// RcSearch's view of the histogram sums, for a whole wave that runs the search with the same
// values in every lane.
struct DevHistView {
    const uint32_t* rate[3];
    const uint32_t* incl_[3];
    __device__ double data(int c, int b) const { return (double)rate[c][b]; }
    __device__ double incl(int c, int b) const { return (double)incl_[c][b]; }
    // 64 probes at once: 3 rounds of loads for 65,536 bins instead of a chain of 16
    template <class Ok> __device__ int first(int lo, int hi, const Ok& ok) const {
        const int lane = threadIdx.x & 63;
        while (lo < hi) {
            const int step = (hi - lo + 63) / 64;
            const int at = lo + (lane + 1) * step - 1;
            const unsigned long long m = __ballot(at >= hi || ok(at));
            if (!m) return hi;
            const int l = __ffsll(m) - 1;
            hi = min(hi, lo + (l + 1) * step - 1);
            lo += l * step;
        }
        return lo;
    }
};

// Widens a slope range (the bits of positive doubles, ~0 and 0 when empty) by another.
__device__ __forceinline__ void slope_range(unsigned long long& lo, unsigned long long& hi, unsigned long long lo2,
                                            unsigned long long hi2) {
    lo = lo2 < lo ? lo2 : lo;
    hi = hi2 > hi ? hi2 : hi;
}

// Point-major hull store of one block, with the points' slope bins and the slope range.
struct HullSink {
    const RcParams& P;
    uint32_t cb;
    unsigned long long lmin, lmax;  // positive doubles order as their bits
    __device__ void operator()(int j, const RcPoint& q) {
        const size_t at = (size_t)j * P.stride + cb;
        P.h_slope[at] = q.slope;
        P.h_gain[at] = q.gain;
        P.h_sel[at] = q.passes << 24 | q.rate;
        int32_t k;
        if (!rc_finite(q.slope)) k = kBinAbove;
        else if (!(q.slope > 0)) k = kBinBelow;
        else {
            k = (int32_t)rc_slope_bin(q.slope, P.mantissa, P.first);
            const unsigned long long bits = __builtin_bit_cast(unsigned long long, q.slope);
            lmin = bits < lmin ? bits : lmin;
            lmax = bits > lmax ? bits : lmax;
        }
        P.h_kbin[at] = k;
    }
};

// A block's pass tables are rows of kMaxPasses entries: four at a time, the last four again
// beyond the row's end.
struct DevPassRows {
    static constexpr int kGroup = 4;
    const uint4* len;
    const int4* dist;
    __device__ void load(int k, int, uint32_t* l, int32_t* d) const {
        const int q = min(k >> 2, kMaxPasses / 4 - 1);
        const uint4 a = len[q];
        const int4 b = dist[q];
        l[0] = a.x, l[1] = a.y, l[2] = a.z, l[3] = a.w;
        d[0] = b.x, d[1] = b.y, d[2] = b.z, d[3] = b.w;
    }
};

// The hull under construction, a column of LDS per lane.
struct DevHullStack {
    uint32_t (*sel)[64];  // passes << 24 | rate
    double (*D)[64];
    int lane;
    __device__ void put(int m, uint32_t r, uint32_t k, double d) {
        sel[m][lane] = k << 24 | r;
        D[m][lane] = d;
    }
    __device__ uint32_t rate(int m) const { return sel[m][lane] & 0xFFFFFFu; }
    __device__ uint32_t passes(int m) const { return sel[m][lane] >> 24; }
    __device__ double dist(int m) const { return D[m][lane]; }
};

}  // namespace

// Bound by latency (a serial scan of each block's passes with a division or more per pass). The
// stack is in LDS, 50 KB a wave, so one-wave workgroups, three to a CU: with the stack in
// scratch memory and the bins from a second pass over the stored slopes one 4K frame took 118 us
// and 16 frames 404, now 38 and 184.
__global__ void __launch_bounds__(kHullGroup) rc_hull_kernel(RcParams P) {
    __shared__ double s_D[kMaxPasses + 1][64];
    __shared__ uint32_t s_sel[kMaxPasses + 1][64];
    static_assert(kHullGroup == 64);
    const uint32_t f = blockIdx.y;
    const RcFrame& F = P.frames[f];
    if (F.max_total == 0) return;          // no rate control for this frame
    if (P.counters->flags & 3u) return;    // Tier-1 overflowed: the job is re-run
    if (blockIdx.x * kHullGroup >= F.nblocks) return;
    const uint32_t i = blockIdx.x * kHullGroup + threadIdx.x;
    unsigned long long lmin = ~0ull, lmax = 0ull;
    if (i < F.nblocks) {
        const uint32_t cb = F.first_block + i;
        const T1Info inf = P.info[cb];
        const uint32_t band = P.blocks[cb].band;
        DevHullStack stack{s_sel, s_D, (int)threadIdx.x};
        HullSink sink{P, cb, lmin, lmax};
        const DevPassRows rows{(const uint4*)(P.pass_len + (size_t)cb * kMaxPasses),
                               (const int4*)(P.pass_dist + (size_t)cb * kMaxPasses)};
        const int cnt = rc_block_hull_to((int)inf.passes, (int)inf.nbps, P.band_scale[band], rows, stack, sink);
        P.hull_n[cb] = (uint32_t)cnt | (P.bands[band].comp_mb & 3u) << 8;
        lmin = sink.lmin;
        lmax = sink.lmax;
    }
    for (int o = 32; o > 0; o >>= 1) slope_range(lmin, lmax, __shfl_xor(lmin, o), __shfl_xor(lmax, o));
    if (threadIdx.x == 0) {
        unsigned long long* part = P.part + 2 * (size_t)part_index(F, f, blockIdx.x);
        part[0] = lmin;
        part[1] = lmax;
    }
}

__global__ void __launch_bounds__(kHullThreads) rc_range_kernel(RcParams P) {
    __shared__ unsigned long long s_min, s_max;
    const uint32_t f = blockIdx.x;
    RcFrame& F = P.frames[f];
    if (F.max_total == 0) return;
    if (P.counters->flags & 3u) return;
    const int t = threadIdx.x;
    if (t == 0) {
        s_min = ~0ull;
        s_max = 0ull;
    }
    __syncthreads();
    const uint32_t nparts = (F.nblocks + kHullGroup - 1) / kHullGroup;
    unsigned long long lmin = ~0ull, lmax = 0ull;
    for (uint32_t x = t; x < nparts; x += kHullThreads) {
        const unsigned long long* part = P.part + 2 * (size_t)part_index(F, f, x);
        slope_range(lmin, lmax, part[0], part[1]);
    }
    for (int o = 32; o > 0; o >>= 1) slope_range(lmin, lmax, __shfl_xor(lmin, o), __shfl_xor(lmax, o));
    if ((t & 63) == 0) {
        atomicMin(&s_min, lmin);
        atomicMax(&s_max, lmax);
    }
    __syncthreads();
    if (t == 0) {
        double mn = __builtin_bit_cast(double, s_min), mx = __builtin_bit_cast(double, s_max);
        if (s_max == 0) mn = mx = 1.0;
        int64_t kLo;
        int nb;
        rc_bin_range(mn, mx, P.mantissa, P.first, kLo, nb);
        F.k_lo = kLo;
        F.nb = nb;
        F.min_slope = mn;
        F.max_slope = mx;
        RcRun& R = P.runs[f];
        RcSearch S{};
        S.init();
        S.kLo = kLo;
        S.nb = nb;
        S.minSlope = mn;
        S.maxSlope = mx;
        S.maxTotal = F.max_total;
        S.maxComp = F.max_comp;
        S.mantissa = P.mantissa;
        S.first = P.first;
        R.search = S;
        for (int k = 0; k < 6; ++k) R.tp[k] = 0;
        R.arrived = 0;
        R.done = 0;
        R.summed = 0;
    }
}

__global__ void __launch_bounds__(kHullThreads) rc_fill_kernel(RcParams P) {
    const uint32_t f = blockIdx.y;
    const RcFrame& F = P.frames[f];
    if (F.max_total == 0) return;
    if (P.counters->flags & 3u) return;
    const uint32_t i = blockIdx.x * kHullThreads + threadIdx.x;
    if (i >= F.nblocks) return;
    const uint32_t cb = F.first_block + i;
    const int64_t kLo = F.k_lo;
    const int nb = F.nb;
    const uint32_t hn = P.hull_n[cb];
    const uint32_t cnt = hn & 0xFFu, c = hn >> 8;
    uint32_t* rate = hist_of(P, f, (int)c);
    uint32_t* incl = hist_of(P, f, 3 + (int)c);
    uint32_t prev = 0;
    for (uint32_t h = 0; h < cnt; ++h) {
        const size_t at = (size_t)h * P.stride + cb;
        const int64_t r = (int64_t)P.h_kbin[at] - kLo;
        const int b = (int)(r < 0 ? 0 : (r > nb - 1 ? nb - 1 : r));  // rc_bin_of on the stored bin
        const uint32_t rt = P.h_sel[at] & 0xFFFFFFu;
        atomicAdd(rate + b, rt - prev);
        if (h == 0) atomicAdd(incl + b, 1u);
        prev = rt;
    }
}

// Suffix sums of the 6 histogram arrays of each frame (v[b] += v[b + 1] + ... + v[nb]) in
// two passes over segments of kScanBins bins: PASS 0 stores each segment's total, PASS 1
// adds the totals of the segments above and scans its own segment in LDS.
template <int PASS>
__global__ void __launch_bounds__(kScanThreads) rc_scan_kernel(RcParams P) {
    __shared__ uint32_t s_v[kScanThreads];
    const uint32_t f = blockIdx.z;
    const int a = (int)blockIdx.y, seg = (int)blockIdx.x;
    const RcFrame& F = P.frames[f];
    if (F.max_total == 0) return;
    if (P.counters->flags & 3u) return;
    const int n1 = F.nb + 1;
    if (seg * kScanBins >= n1) return;
    const int t = threadIdx.x;
    uint32_t* v = hist_of(P, f, a);
    uint32_t* segsum = P.segsum + ((size_t)f * 6 + (size_t)a) * kScanSegs;
    const int b0 = seg * kScanBins + 4 * t;
    uint32_t x[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = b0 + j < n1 ? v[b0 + j] : 0u;
    if (PASS == 0) {
        s_v[t] = x[0] + x[1] + x[2] + x[3];
        __syncthreads();
        for (int w = kScanThreads / 2; w > 0; w >>= 1) {
            if (t < w) s_v[t] += s_v[t + w];
            __syncthreads();
        }
        if (t == 0) segsum[seg] = s_v[0];
        return;
    }
    // totals of the segments above this one
    const int nseg = (n1 + kScanBins - 1) / kScanBins;
    uint32_t above = 0;
    if (t < 64)
        for (int s = seg + 1 + t; s < nseg; s += 64) above += segsum[s];
    // suffix sums inside the thread's four bins, then across the threads (Hillis-Steele)
    x[2] += x[3];
    x[1] += x[2];
    x[0] += x[1];
    s_v[t] = x[0];
    __syncthreads();
    for (int d = 1; d < kScanThreads; d <<= 1) {
        const uint32_t add = t + d < kScanThreads ? s_v[t + d] : 0u;
        __syncthreads();
        s_v[t] += add;
        __syncthreads();
    }
    __shared__ uint32_t s_above[64];
    if (t < 64) s_above[t] = above;
    __syncthreads();
    if (t == 0) {
        uint32_t sum = 0;
        for (int k = 0; k < 64; ++k) sum += s_above[k];
        s_above[0] = sum;
    }
    __syncthreads();
    const uint32_t carry = s_above[0] + (t + 1 < kScanThreads ? s_v[t + 1] : 0u);
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (b0 + j < n1) v[b0 + j] = x[j] + carry;
}

namespace {

// Waits for an atomic that returned v, so that a ticket taken afterwards (RcRun::arrived, summed)
// tells the last workgroup that the value is in place. There is no release and no acquire: a
// device-scope fence writes back the whole L2 (a measurement of 16 4K frames 285 us with fences,
// 50 without). So only what is written by device-scope atomics and read by them, past the L2s
// that the XCDs have of their own, may cross to the last workgroup of the same launch. A plain
// store (a block's choice, its length) is seen by the next launch, not by that workgroup.
__device__ __forceinline__ void atomic_done(unsigned long long v) {
    asm volatile("" ::"v"((uint32_t)v), "v"((uint32_t)(v >> 32)) : "memory");
}

// Bits of the longest packet header: 48 blocks of at most 3 inclusion bits, 258 for the zero
// bit-planes (Mb fits in 8 bits), 16 for the passes, 22 for Lblock and 29 for the length.
constexpr int kHeaderWords = 512;

// The bits v (below 1 << n, n <= 32) at bit `at` of a string whose bit 0 is word 0's highest.
__device__ __forceinline__ void put_bits(uint32_t* words, uint32_t at, uint32_t v, uint32_t n) {
    if (!v) return;  // the string is zero before
    const unsigned long long w = (unsigned long long)v << (64u - n - (at & 31u));
    const uint32_t hi = (uint32_t)(w >> 32), lo = (uint32_t)w;
    if (hi) atomicOr(words + (at >> 5), hi);
    if (lo) atomicOr(words + (at >> 5) + 1, lo);
}

// One packet at thresholds lambda, by a whole wave: lane q of each group of 16 chooses the
// passes of leaf q of one precinct-band and writes its part of the header; returns the
// packet's bytes (rc_packet_bytes of the same choices) in every lane.
//
// A hull's slopes fall strictly, so its points of slope >= lambda are a prefix: their number
// is counted, eight at a time. The choice and its length replace the block's pass
// count and codeword length at once (the last measurement's stay).
__device__ unsigned long long measure_packet(const RcParams& P, const RcFrame& F, uint32_t k, const double lambda[3],
                                             uint32_t* words) {
    const int lane = threadIdx.x & 63, q = lane & 15, group = lane >> 4;
    const RcPacket pk = F.packets[k];
    const bool band = group < pk.nband;
    const RcPBand pb = F.pbands[pk.first + (band ? group : 0)];
    const int w = band ? pb.ncbx : 0, h = band ? pb.ncby : 0;
    const bool leaf = (q & 3) < w && (q >> 2) < h;
    uint32_t np = 0, len = 0;
    int zv = 255;
    if (leaf) {
        const uint32_t cb = F.first_block + pb.block0 + (uint32_t)(q >> 2) * pb.stride + (uint32_t)(q & 3);
        const uint32_t hn = P.hull_n[cb], nbps = P.info[cb].nbps;
        const uint32_t cnt = hn & 0xFFu, c = hn >> 8;
        const double lam = c == 0 ? lambda[0] : c == 1 ? lambda[1] : lambda[2];
        uint32_t kept = 0;
        for (uint32_t i = 0; i < cnt; i += 8) {  // eight points' loads in flight at once
            double s[8];
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j) s[j] = P.h_slope[(size_t)(i + j < cnt ? i + j : i) * P.stride + cb];
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j) kept += i + j < cnt && s[j] >= lam;
            if (kept < i + 8) break;
        }
        const uint32_t sel = kept ? P.h_sel[(size_t)(kept - 1) * P.stride + cb] : 0u;
        np = sel >> 24;
        len = sel & 0xFFFFFFu;
        zv = (int)pb.mb - (int)nbps;
        P.sel[cb] = kept;
        P.info[cb].passes = np;
        P.code_len[cb] = len;
    }
    const unsigned long long included = __ballot(np != 0);
    if (!included) return 1;  // an empty packet is one zero byte

    // The band's tag trees (rc_packet_code): which lane meets each node first, in leaf order.
    const uint32_t incl = (uint32_t)(included >> (lane & 48)) & 0xFFFFu;
    const int levels = (w == 1 && h == 1) ? 1 : ((w <= 2 && h <= 2) ? 2 : 3);
    const int qm = (q >> 3) * 8 + ((q >> 1) & 1) * 2;  // the quad's first leaf
    const uint32_t quad = incl & (0x33u << qm);
    int zq = min(zv, __shfl_xor(zv, 1));
    zq = min(zq, __shfl_xor(zq, 4));
    int zroot = min(zq, __shfl_xor(zq, 2));
    zroot = min(zroot, __shfl_xor(zroot, 8));
    uint32_t ibits = 0, icount = 0;  // inclusion
    if (leaf) {
        bool go = true;
        if (levels >= 2) {
            go = incl != 0;
            if (q == 0) {
                ibits = go;
                icount = 1;
            }
        }
        if (go && levels == 3) {
            go = quad != 0;
            if (q == qm) {
                ibits = ibits << 1 | (go ? 1u : 0u);
                ++icount;
            }
        }
        if (go) {
            ibits = ibits << 1 | (np ? 1u : 0u);
            ++icount;
        }
    }
    // zero bit-planes: at each node met first, (value - parent's value) zeros and a one
    uint32_t zr = 0, zn = 0, zl = 0, pbits = 0, pcount = 0, lcount = 0, incr = 0;
    if (np) {
        const uint32_t before = incl & ((1u << q) - 1u);
        int prev = 0;
        if (levels >= 2) {
            if (!before) zr = (uint32_t)max(zroot - prev + 1, 0);
            prev = zroot;
        }
        if (levels == 3) {
            if (!(before & quad)) zn = (uint32_t)max(zq - prev + 1, 0);
            prev = zq;
        }
        zl = (uint32_t)max(zv - prev + 1, 0);
        // Table B.4: codewords for the number of coding passes
        pbits = np == 1 ? 0u : np == 2 ? 2u : np <= 5 ? 0xCu | (np - 3) : np <= 36 ? 0x1E0u | (np - 6) : 0xFF80u | (np - 37);
        pcount = np == 1 ? 1u : np == 2 ? 2u : np <= 5 ? 4u : np <= 36 ? 9u : 16u;
        const uint32_t extra = (uint32_t)rc_floor_log2(np), need = len ? (uint32_t)rc_floor_log2(len) + 1 : 1u;
        incr = need > 3 + extra ? need - (3 + extra) : 0u;
        lcount = 3 + incr + extra;
    }
    const uint32_t bits = icount + zr + zn + zl + pcount + (np ? incr + 1 : 0u) + lcount;
    uint32_t end = bits, body = len;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t e = (uint32_t)__shfl_up((int)end, o), b = (uint32_t)__shfl_up((int)body, o);
        if (lane >= o) {
            end += e;
            body += b;
        }
    }
    const uint32_t total = 1u + (uint32_t)__shfl((int)end, 63);  // the leading 1: not empty
    const unsigned long long bytes = (uint32_t)__shfl((int)body, 63);

    // the header as one bit string, without the bits that marker stuffing adds
    for (uint32_t i = lane; i <= (total + 63) / 32; i += 64) words[i] = 0;
    lds_sync();
    uint32_t at = 1u + end - bits;
    if (lane == 0) put_bits(words, 0, 1, 1);
    put_bits(words, at, ibits, icount);
    at += icount;
    if (np) {
        if (zr) put_bits(words, at += zr - 1, 1, 1), ++at;
        if (zn) put_bits(words, at += zn - 1, 1, 1), ++at;
        if (zl) put_bits(words, at += zl - 1, 1, 1), ++at;
        put_bits(words, at, pbits, pcount);
        at += pcount;
        put_bits(words, at, ((1u << incr) - 1u) << 1, incr + 1);
        at += incr + 1;
        put_bits(words, at, len, lcount);
    }
    lds_sync();
    // A byte after 0xFF holds 7 bits: from each start, 64 bytes at a time, to the next 0xFF.
    uint32_t pos = 0, count = 0;
    for (;;) {
        const uint32_t p = pos + 8u * (uint32_t)lane;
        uint32_t byte = 0;
        if (p + 8 <= total) {
            const unsigned long long v = (unsigned long long)words[p >> 5] << 32 | words[(p >> 5) + 1];
            byte = (uint32_t)(v >> (56u - (p & 31u))) & 0xFFu;
        }
        const unsigned long long ff = __ballot(byte == 0xFFu);
        if (ff) {
            const uint32_t n = (uint32_t)__ffsll(ff);
            pos += 8 * n + 7;
            count += n + 1;  // with the 7-bit byte that follows, full or padded or empty
        } else {
            const uint32_t left = pos < total ? (total - pos + 7) / 8 : 0u;
            const uint32_t n = left < 64 ? left : 64;
            pos += 8 * n;
            count += n;
        }
        if (pos >= total) break;
    }
    return bytes + count;
}

// One step of a frame's search by a whole wave, after a measurement whose tile-part sums are
// tp; returns whether another is wanted and leaves the state for it.
__device__ bool search_step(const RcParams& P, uint32_t f, RcFrame& F, const unsigned long long tp[6]) {
    RcRun& R = P.runs[f];
    RcSearch S = R.search;
    DevHistView H;
    for (int c = 0; c < 3; ++c) {
        H.rate[c] = hist_of(P, f, c);
        H.incl_[c] = hist_of(P, f, 3 + c);
    }
    RcSizes sz;
    sz.total = F.fixed_bytes;
    sz.comp[0] = sz.comp[1] = sz.comp[2] = 0;
    for (uint32_t k = 0; k < F.ntp; ++k) {
        const unsigned long long b = tp[k] + 14;  // SOT + SOD of each tile-part
        const int c = F.tp_comp[k];
        sz.comp[0] += c == 0 ? b : 0;
        sz.comp[1] += c == 1 ? b : 0;
        sz.comp[2] += c == 2 ? b : 0;
        sz.total += b;
    }
    const bool more = S.next(H, sz);
    if ((threadIdx.x & 63) == 0) {
        R.search = S;
        R.done = more ? 0u : 1u;
        R.arrived = 0;
        for (int k = 0; k < 6; ++k) R.tp[k] = 0;
        if (!more) {
            for (int c = 0; c < 3; ++c) F.lambda[c] = S.lambda[c];
            F.total = sz.total;
            for (int c = 0; c < 3; ++c) F.comp[c] = sz.comp[c];
            for (uint32_t k = 0; k < 6; ++k) F.tile_part[k] = k < F.ntp ? tp[k] + 14 : 0ull;
            F.iterations = S.iterations;
            F.status = 0;
        }
    }
    return more;
}

}  // namespace

// Bound by latency: the loads of a block's hull, the scan of its packet's header bits and the
// search's probes, one after the other. One 4K frame has some 600 packets, a wave each. With
// one workgroup per frame for the whole search (a thread per packet's header, 26 blocks a
// thread, a thread's chain of 16 probes) a search of three measurements took 615 us for one 4K
// frame and 660 for 16; these launches with the finish and distortion kernels take 109 and 197.
// Frames with one budget take 3 or 4 measurements, those held by a component's cap 5 and more:
// six launches, each 4 us when there is nothing left to do (24 us otherwise); further steps run
// in rc_finish_kernel at 180 us each.
__global__ void __launch_bounds__(kMeasureWaves * 64) rc_measure_kernel(RcParams P) {
    __shared__ uint32_t s_words[kMeasureWaves][kHeaderWords];
    __shared__ uint32_t s_last;
    const uint32_t f = blockIdx.y;
    RcFrame& F = P.frames[f];
    if (F.max_total == 0) return;
    if (P.counters->flags & 3u) return;
    RcRun& R = P.runs[f];
    const uint32_t groups = (F.npackets + kMeasureWaves - 1) / kMeasureWaves;
    if (R.done || blockIdx.x >= groups) return;
    const uint32_t wv = threadIdx.x >> 6, k = blockIdx.x * kMeasureWaves + wv;
    const double lambda[3] = {R.search.lambda[0], R.search.lambda[1], R.search.lambda[2]};
    if (k < F.npackets) {
        const unsigned long long b = measure_packet(P, F, k, lambda, s_words[wv]);
        if ((threadIdx.x & 63) == 0) atomic_done(atomicAdd(&R.tp[F.packets[k].tp], b));
    }
    // The state is read above by every wave before the last workgroup to arrive replaces it; of
    // the other workgroups' results that one reads R.tp alone, by atomics (atomic_done).
    __syncthreads();
    if (threadIdx.x == 0) s_last = atomicAdd(&R.arrived, 1u) == groups - 1;
    __syncthreads();
    if (!s_last || wv != 0) return;
    unsigned long long tp[6];
    for (int i = 0; i < 6; ++i) tp[i] = __hip_atomic_load(&R.tp[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    search_step(P, f, F, tp);
}

__global__ void __launch_bounds__(kFinishWaves * 64) rc_finish_kernel(RcParams P) {
    __shared__ uint32_t s_words[kFinishWaves][kHeaderWords];
    __shared__ unsigned long long s_tp[6];
    __shared__ uint32_t s_more;
    const uint32_t f = blockIdx.x;
    RcFrame& F = P.frames[f];
    if (F.max_total == 0) return;
    if (P.counters->flags & 3u) return;
    RcRun& R = P.runs[f];
    if (R.done) return;
    const uint32_t wv = threadIdx.x >> 6;
    for (;;) {
        const double lambda[3] = {R.search.lambda[0], R.search.lambda[1], R.search.lambda[2]};
        if (threadIdx.x < 6) s_tp[threadIdx.x] = 0;
        __syncthreads();
        for (uint32_t k = wv; k < F.npackets; k += kFinishWaves) {
            const unsigned long long b = measure_packet(P, F, k, lambda, s_words[wv]);
            if ((threadIdx.x & 63) == 0) atomicAdd(&s_tp[F.packets[k].tp], b);
        }
        __syncthreads();
        if (wv == 0) {
            unsigned long long tp[6];
            for (int i = 0; i < 6; ++i) tp[i] = s_tp[i];
            const bool more = search_step(P, f, F, tp);
            if (threadIdx.x == 0) s_more = more;
        }
        __threadfence_block();
        __syncthreads();
        if (!s_more) break;
    }
}

// The distortion left: the gains of the points left out, summed by 1,024 threads over blocks
// t, t + 1024, ... in turn and then as a tree, an order that does not depend on the launch.
__global__ void __launch_bounds__(kHullThreads) rc_dist_kernel(RcParams P) {
    const uint32_t f = blockIdx.y;
    RcFrame& F = P.frames[f];
    if (F.max_total == 0) return;
    if (P.counters->flags & 3u) return;
    constexpr uint32_t groups = kRcDistSums / 64;
    if (threadIdx.x >= 64) {  // the other waves clear the histogram
        const uint32_t i0 = blockIdx.x * (kHullThreads - 64) + threadIdx.x - 64, step = groups * (kHullThreads - 64);
        for (int a = 0; a < 6; ++a) {
            uint32_t* v = hist_of(P, f, a);
            for (uint32_t b = i0; b <= (uint32_t)F.nb; b += step) v[b] = 0u;
        }
        return;
    }
    const uint32_t t = blockIdx.x * 64 + threadIdx.x, n = F.nblocks;
    double dist = 0;
    for (uint32_t i = t; i < n; i += 4 * kRcDistSums) {
        uint32_t from[4], to[4];
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
            const uint32_t at = i + j * kRcDistSums, cb = F.first_block + (at < n ? at : i);
            from[j] = P.sel[cb];
            to[j] = at < n ? P.hull_n[cb] & 0xFFu : 0u;
        }
        double g[4][4];
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j)
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k)
                g[j][k] = from[j] + k < to[j]
                              ? P.h_gain[(size_t)(from[j] + k) * P.stride + F.first_block + i + j * kRcDistSums]
                              : 0.0;
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) dist += g[j][k];
            const size_t cb = (size_t)F.first_block + i + j * kRcDistSums;
            for (uint32_t h = from[j] + 4; h < to[j]; h += 4) {
                double r[4];
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) r[k] = h + k < to[j] ? P.h_gain[(size_t)(h + k) * P.stride + cb] : 0.0;
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) dist += r[k];
            }
        }
    }
    unsigned long long* sums = P.dist + (size_t)f * kRcDistSums;
    atomic_done(atomicExch(&sums[t], __builtin_bit_cast(unsigned long long, dist)));
    uint32_t last = 0;  // reads the other workgroups' sums by atomics only (atomic_done)
    if (threadIdx.x == 0) last = atomicAdd(&P.runs[f].summed, 1u) == groups - 1;
    if (!__shfl((int)last, 0)) return;
    double s[groups];
#pragma unroll
    for (uint32_t k = 0; k < groups; ++k)
        s[k] = __builtin_bit_cast(double, __hip_atomic_load(&sums[64 * k + threadIdx.x], __ATOMIC_RELAXED,
                                                            __HIP_MEMORY_SCOPE_AGENT));
#pragma unroll
    for (uint32_t w = groups / 2; w > 0; w >>= 1)
#pragma unroll
        for (uint32_t k = 0; k < w; ++k) s[k] += s[k + w];
    for (int w = 32; w > 0; w >>= 1) s[0] += __shfl_down(s[0], w);
    if (threadIdx.x == 0) F.distortion = s[0];
}

hipError_t launch_rc(const RcParams& p, int frames, uint32_t max_frame_blocks, uint32_t max_frame_packets,
                     hipStream_t s) {
    const uint32_t gx = (max_frame_blocks + kHullThreads - 1) / kHullThreads;
    if (!gx || !frames) return hipSuccess;
    const uint32_t hx = (max_frame_blocks + kHullGroup - 1) / kHullGroup;
    hipLaunchKernelGGL(rc_hull_kernel, dim3(hx, frames), dim3(kHullGroup), 0, s, p);
    hipLaunchKernelGGL(rc_range_kernel, dim3(frames), dim3(kHullThreads), 0, s, p);
    hipLaunchKernelGGL(rc_fill_kernel, dim3(gx, frames), dim3(kHullThreads), 0, s, p);
    hipLaunchKernelGGL(rc_scan_kernel<0>, dim3(kScanSegs, 6, frames), dim3(kScanThreads), 0, s, p);
    hipLaunchKernelGGL(rc_scan_kernel<1>, dim3(kScanSegs, 6, frames), dim3(kScanThreads), 0, s, p);
    const uint32_t px = (max_frame_packets + kMeasureWaves - 1) / kMeasureWaves;
    for (int i = 0; px && i < kMeasureLaunches; ++i)
        hipLaunchKernelGGL(rc_measure_kernel, dim3(px, frames), dim3(kMeasureWaves * 64), 0, s, p);
    hipLaunchKernelGGL(rc_finish_kernel, dim3(frames), dim3(kFinishWaves * 64), 0, s, p);
    hipLaunchKernelGGL(rc_dist_kernel, dim3(kRcDistSums / 64, frames), dim3(kHullThreads), 0, s, p);
    return hipGetLastError();
}

size_t rc_run_bytes(size_t frames) { return frames * sizeof(RcRun); }

size_t rc_segsum_entries(size_t frames) { return frames * 6 * kScanSegs; }

}  // namespace gail_amd
