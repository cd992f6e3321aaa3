// Tier-2, rate control and the DCI structural check (see codestream.h).
#include "codestream.h"
#include "host_pool.h"
#include "rc_shared.h"

#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <thread>
#include <utility>

namespace gail_amd {

namespace {

// ---------------------------------------------------------------- packets
// Resolutions a tile-part carries: the 2K frame puts all of a component in one tile-part;
// the 4K frame's POC sends the 2K resolutions of every component first, then the top
// resolution of every component (SMPTE 429-4 / progression.h:20-26), six tile-parts.
void tilePartResolutions(const Layout& L, int part, int& r0, int& r1) {
    r0 = (L.fourk && part == 1) ? L.levels : 0;
    r1 = (L.fourk && part == 0) ? L.levels : L.levels + 1;
}

// log2 of the precinct size of resolution r (COD: 2^7 at r = 0, 2^8 above).
int precinctLog2(int r) { return r == 0 ? 7 : 8; }

// The packet table of a layout: every packet in codestream order with its precinct-bands.
// Within a tile-part (one component, a range of resolutions) the order is CPRL with the tile
// at the origin (B.12.1.5): a precinct of resolution r covers 2^(PP_r + NL - r) image samples
// each way, and the packets come in raster order of their precincts' image-domain origins,
// lower resolutions first at a shared origin. A band-domain precinct of resolution r > 0 is
// half the resolution's (B.6), so every precinct-band spans 4 x 4 code-blocks at most.
RcTables buildPacketTables(const Layout& L) {
    RcTables T;
    const int ntp = L.fourk ? 6 : 3;
    T.ntp = (uint32_t)ntp;
    struct Entry {
        int y, x, r, px, py;
    };
    std::vector<Entry> order;
    for (int part = 0; part < (L.fourk ? 2 : 1); ++part) {
        int r0, r1;
        tilePartResolutions(L, part, r0, r1);
        order.clear();
        for (int r = r0; r < r1; ++r) {
            const int pp = precinctLog2(r), shift = pp + L.levels - r;
            const int wr = (L.width + (1 << (L.levels - r)) - 1) >> (L.levels - r);
            const int hr = (L.height + (1 << (L.levels - r)) - 1) >> (L.levels - r);
            const int npx = (wr + (1 << pp) - 1) >> pp, npy = (hr + (1 << pp) - 1) >> pp;
            for (int py = 0; py < npy; ++py)
                for (int px = 0; px < npx; ++px) order.push_back(Entry{py << shift, px << shift, r, px, py});
        }
        std::sort(order.begin(), order.end(), [](const Entry& a, const Entry& b) {
            return a.y != b.y ? a.y < b.y : a.x != b.x ? a.x < b.x : a.r < b.r;
        });
        for (int c = 0; c < kComps; ++c) {
            const int tp = part * kComps + c;
            T.tpComp[tp] = c;
            for (const Entry& e : order) {
                const int nbands = e.r == 0 ? 1 : 3;
                const int span = 1 << ((e.r == 0 ? precinctLog2(e.r) : precinctLog2(e.r) - 1) - kCblkLog2);
                RcPacket pk{(uint32_t)T.pbands.size(), (uint16_t)nbands, (uint16_t)tp};
                for (int k = 0; k < nbands; ++k) {
                    const Subband& b = L.bands[L.bandIndex(c, e.r, e.r == 0 ? 0 : k + 1)];
                    if (b.Mb > 31) throw std::logic_error("subband with more than 31 magnitude bit-planes");
                    const int cx = e.px * span, cy = e.py * span;
                    const int w = std::max(0, std::min(span, b.ncbx - cx)), h = std::max(0, std::min(span, b.ncby - cy));
                    RcPBand q{};
                    q.block0 = (uint32_t)(b.cblkBase + cy * b.ncbx + cx);
                    q.stride = (uint16_t)b.ncbx;
                    q.ncbx = (uint8_t)(w && h ? w : 0);
                    q.ncby = (uint8_t)(w && h ? h : 0);
                    q.mb = (uint8_t)b.Mb;
                    T.pbands.push_back(q);
                }
                T.packets.push_back(pk);
            }
        }
    }
    return T;
}

// A frame's blocks as the packet coder reads them: passes[i] of block i kept.
struct KeptBlocks {
    const Tier1Ref* t1;
    const uint8_t* p;
    uint32_t passes(uint32_t i) const { return p[i]; }
    uint32_t nbps(uint32_t i) const { return t1->nbps((int)i); }
    uint32_t len(uint32_t i) const { return p[i] ? t1->len((int)i, p[i] - 1) : 0u; }
};

struct AppendByte {
    std::vector<uint8_t>* v;
    void operator()(uint32_t b) const { v->push_back((uint8_t)b); }
};

void put16(std::vector<uint8_t>& v, uint32_t x) {
    v.push_back((uint8_t)(x >> 8));
    v.push_back((uint8_t)x);
}
void put32(std::vector<uint8_t>& v, uint32_t x) {
    put16(v, x >> 16);
    put16(v, x & 0xFFFFu);
}

enum : uint16_t {
    SOC = 0xFF4F, SIZ = 0xFF51, COD = 0xFF52, TLM = 0xFF55, QCD = 0xFF5C, POC = 0xFF5F, COM = 0xFF64,
    SOT = 0xFF90, SOD = 0xFF93, EOC = 0xFFD9
};

// Main header of a DCI frame (t2.cpp:126-183): SIZ (Rsiz 3 / 4), COD (CPRL, one layer,
// ICT, 32x32 blocks, 9/7, precincts 128 / 256), QCD (scalar expounded), the 4K POC, COM,
// and a TLM patched once the tile-parts are known (kept last).
void mainHeader(const Layout& L, std::vector<uint8_t>& v, int ntp, const std::string& comment) {
    const int nres = L.numRes();
    put16(v, SOC);
    put16(v, SIZ);
    put16(v, 38 + 3 * kComps);
    put16(v, L.fourk ? 4 : 3);
    put32(v, L.width);
    put32(v, L.height);
    put32(v, 0);
    put32(v, 0);
    put32(v, L.width);
    put32(v, L.height);
    put32(v, 0);
    put32(v, 0);
    put16(v, kComps);
    for (int c = 0; c < kComps; ++c) {
        v.push_back(kBitDepth - 1);
        v.push_back(1);
        v.push_back(1);
    }
    put16(v, COD);
    put16(v, 12 + nres);
    v.push_back(0x01);
    v.push_back(4);
    put16(v, 1);
    v.push_back(1);
    v.push_back((uint8_t)L.levels);
    v.push_back(kCblkLog2 - 2);
    v.push_back(kCblkLog2 - 2);
    v.push_back(0);
    v.push_back(0);
    for (int r = 0; r < nres; ++r) v.push_back(r == 0 ? 0x77 : 0x88);
    put16(v, QCD);
    const int nb = L.bandsPerComp();
    put16(v, 3 + 2 * nb);
    v.push_back((uint8_t)((L.guardBits << 5) | 2));
    for (int i = 0; i < nb; ++i) put16(v, (uint32_t)((L.bands[i].eps << 11) | L.bands[i].mu));
    if (L.fourk) {
        put16(v, POC);
        put16(v, 2 + 7 * 2);
        const int NL = L.levels;
        const uint8_t e[2][7] = {{0, 0, 0, 1, (uint8_t)NL, 3, 4}, {(uint8_t)NL, 0, 0, 1, (uint8_t)(NL + 1), 3, 4}};
        for (auto& p : e) v.insert(v.end(), p, p + 7);
    }
    put16(v, COM);
    put16(v, (uint32_t)(4 + comment.size()));
    put16(v, 1);
    v.insert(v.end(), comment.begin(), comment.end());
    put16(v, TLM);
    put16(v, 4 + 5 * ntp);
    v.push_back(0);
    v.push_back(0x50);
    for (int i = 0; i < ntp; ++i) {
        v.push_back(0);
        put32(v, 0);
    }
}

}  // namespace

const char* codestreamLabel() { return "GAIL 1.1.0"; }

static const RcTables& packetTables(const Layout& L) {
    // one table per frame geometry (the six DCI containers, and any other size asked for)
    static std::mutex m;
    static std::vector<std::pair<std::array<int, 3>, std::unique_ptr<RcTables>>> cache;
    const std::array<int, 3> key{L.width, L.height, L.fourk ? 1 : 0};
    std::lock_guard<std::mutex> lock(m);
    for (auto& e : cache)
        if (e.first == key) return *e.second;
    auto t = std::make_unique<RcTables>(makeRcTables(L));
    cache.emplace_back(key, std::move(t));
    return *cache.back().second;
}

namespace {

// Helper threads shared by every rate-control and Tier-2 call in the process that asks for
// them. The calling thread takes chunks of its own work as well, so a call completes even
// while the helpers serve another.
Pool& rcHelpers() {
    static Pool* const p = new Pool(std::clamp((int)std::thread::hardware_concurrency() - 1, 1, 4));
    return *p;
}

int rcSlots() { return rcHelpers().size() + 1; }

constexpr int kChunks = 32;

std::pair<int, int> chunkRange(int n, int chunk) {
    return {(int)((int64_t)n * chunk / kChunks), (int)((int64_t)n * (chunk + 1) / kChunks)};
}

// fn(chunk, slot) for every chunk in [0, kChunks) on the caller and the helpers. Partial sums
// kept per slot are integers or minima/maxima, so their totals do not depend on the split.
template <class F>
void rcParallel(const F& fn) {
    parallelChunks(rcHelpers(), kChunks, fn);
}

CodestreamSizes measureParallel(const RcTables& T, const Tier1Ref& t1, const uint8_t* passes);

}  // namespace

void buildCodestream(const Layout& L, const Tier1Ref& t1, const uint8_t* passes, std::vector<uint8_t>* out,
                     CodestreamSizes* sizes, const std::string& tag, bool parallel) {
    if (tag.size() > kMaxDeviceTagBytes) throw std::logic_error("device tag too long");
    const RcTables& T = packetTables(L);
    const CodestreamSizes sz = parallel ? measureParallel(T, t1, passes) : rcMeasure(L, T, t1, passes);
    if (sizes) *sizes = sz;
    if (!out) return;
    const std::string comment = tag.empty() ? std::string(codestreamLabel()) : std::string(codestreamLabel()) + " " + tag;
    const size_t slack = std::strlen(codestreamLabel()) + 1 + kMaxDeviceTagBytes - comment.size();
    std::vector<uint8_t>& v = *out;
    v.clear();
    v.reserve(sz.total);
    mainHeader(L, v, (int)T.ntp, comment);
    const size_t tlmPos = v.size() - 5 * T.ntp;
    const KeptBlocks view{&t1, passes};
    // every packet coded into its chunk's bytes (chunks of consecutive packets, coded in
    // parallel or in turn), then copied out in codestream order
    const int npk = (int)T.packets.size();
    std::vector<std::vector<uint8_t>> chunkBytes(kChunks);
    std::vector<uint32_t> pkBegin(npk), pkEnd(npk);
    std::vector<uint8_t> pkChunk(npk);
    auto code = [&](int chunk, int) {
        const auto [k0, k1] = chunkRange(npk, chunk);
        std::vector<uint8_t>& o = chunkBytes[chunk];
        std::vector<uint8_t> header;
        std::vector<std::pair<uint32_t, uint32_t>> bodies;
        for (int k = k0; k < k1; ++k) {
            pkChunk[k] = (uint8_t)chunk;
            pkBegin[k] = (uint32_t)o.size();
            header.clear();
            bodies.clear();
            RcBitsT<AppendByte> bw{AppendByte{&header}};
            bw.init();
            const bool any = rc_packet_code(T.packets[k], T.pbands.data(), view, bw,
                                            [&](uint32_t i, uint32_t len) { bodies.emplace_back(i, len); });
            if (!any) {
                o.push_back(0);
            } else {
                bw.finish();
                o.insert(o.end(), header.begin(), header.end());
                for (const auto& [i, len] : bodies) o.insert(o.end(), t1.code((int)i), t1.code((int)i) + len);
            }
            pkEnd[k] = (uint32_t)o.size();
        }
    };
    if (parallel) parallelChunks(rcHelpers(), kChunks, code);
    else
        for (int c = 0; c < kChunks; ++c) code(c, 0);
    size_t next = 0;
    for (uint32_t tp = 0; tp < T.ntp; ++tp) {
        const size_t sot = v.size();
        put16(v, SOT);
        put16(v, 10);
        put16(v, 0);  // tile index
        put32(v, 0);  // Psot, patched below
        v.push_back((uint8_t)tp);
        v.push_back((uint8_t)T.ntp);
        put16(v, SOD);
        for (; next < T.packets.size() && T.packets[next].tp == tp; ++next) {
            const uint8_t* o = chunkBytes[pkChunk[next]].data();
            v.insert(v.end(), o + pkBegin[next], o + pkEnd[next]);
        }
        const uint32_t psot = (uint32_t)(v.size() - sot);
        if (psot != sz.tilePart[tp]) throw std::logic_error("tile-part size differs from its measurement");
        for (int b = 0; b < 4; ++b) {
            v[sot + 6 + b] = (uint8_t)(psot >> (24 - 8 * b));
            v[tlmPos + 5 * tp + 1 + b] = (uint8_t)(psot >> (24 - 8 * b));
        }
    }
    put16(v, EOC);
    if (v.size() + slack != sz.total) throw std::logic_error("codestream size differs from its measurement");
}

RcTables makeRcTables(const Layout& L) {
    RcTables T = buildPacketTables(L);
    std::vector<uint8_t> hdr;
    mainHeader(L, hdr, (int)T.ntp, codestreamLabel());
    const size_t slack = 1 + kMaxDeviceTagBytes;  // the COM text at its longest
    T.fixedBytes = hdr.size() + slack + 2;
    return T;
}

namespace {

// Sizes from the packet bytes of each tile-part (its 14 header bytes added here).
CodestreamSizes sizesOf(const RcTables& T, unsigned long long tp[6]) {
    CodestreamSizes sz;
    sz.numTileParts = (int)T.ntp;
    for (uint32_t k = 0; k < T.ntp; ++k) tp[k] += 14;
    sz.total = T.fixedBytes;
    for (uint32_t k = 0; k < T.ntp; ++k) {
        sz.tilePart[k] = tp[k];
        sz.comp[T.tpComp[k]] += tp[k];
        sz.total += tp[k];
    }
    return sz;
}

}  // namespace

CodestreamSizes rcMeasure(const Layout& L, const RcTables& T, const Tier1Ref& t1, const uint8_t* passes) {
    const KeptBlocks view{&t1, passes};
    (void)L;
    unsigned long long tp[6] = {};
    for (const RcPacket& pk : T.packets) tp[pk.tp] += rc_packet_bytes(pk, T.pbands.data(), view);
    return sizesOf(T, tp);
}

size_t emptyCodestreamBytes(const Layout& L) {
    std::vector<uint32_t> info((size_t)L.numCblks() * 5, 0);
    const Tier1Ref t1{info.data(), nullptr, nullptr, nullptr, (size_t)L.numCblks()};
    const std::vector<uint8_t> passes((size_t)L.numCblks(), 0);
    CodestreamSizes sz;
    buildCodestream(L, t1, passes.data(), nullptr, &sz);
    return sz.total;
}

RateLimits dciLimits(double fps, double maxMbps, double compMbps) {
    auto budget = [fps](double mbps) {
        const double b = std::floor(mbps * 1e6 / (8.0 * fps)) - 16;
        return std::isfinite(b) && b > 0 ? (size_t)b : (size_t)0;
    };
    return RateLimits{budget(maxMbps), budget(compMbps)};
}

// ---------------------------------------------------------------- rate control
namespace {

// Lower convex hull of each block's (rate, distortion) points (rate_control.cpp:38-86). Block
// i's count[i] points start at pts[start[i]]; start[] leaves room for one point per coding
// pass, so the blocks are hulled independently.
struct Hull {
    std::vector<uint32_t> start, count;
    std::vector<RcPoint> pts;
    double minSlope = 0, maxSlope = 0;  // over the finite positive slopes; 0 if there are none
    const RcPoint* at(int i) const { return pts.data() + start[i]; }
};

// Fills H (its buffers are reused from call to call, so a worker thread that codes many
// frames does not fault fresh pages in for every one).
void buildHull(const Layout& L, const Tier1Ref& t1, Hull& H) {
    const int n = L.numCblks();
    H.start.resize(n + 1);
    H.count.resize(n);
    uint32_t total = 0;
    for (int i = 0; i < n; ++i) {
        const uint32_t np = t1.passes(i);
        if (np > (uint32_t)kMaxPasses) throw std::runtime_error("code-block with more than 64 coding passes");
        H.start[i] = total;
        total += np;
    }
    H.start[n] = total;
    H.pts.resize(total);
    struct alignas(64) Range {
        double lo = INFINITY, hi = 0;
    };
    std::vector<Range> range(rcSlots());
    rcParallel([&](int chunk, int s) {
        const auto [i0, i1] = chunkRange(n, chunk);
        Range& r = range[s];
        for (int i = i0; i < i1; ++i) {
            const int np = (int)t1.passes(i);
            H.count[i] = 0;
            if (!np) continue;
            const Subband& b = L.bands[L.cblks[i].band];
            const double scale = (double)b.delta * b.delta * b.weight;
            RcPoint* q = H.pts.data() + H.start[i];
            const int m = rc_block_hull(np, (int)t1.nbps(i), scale, &t1.passLen[t1.info5[5 * i + 4]],
                                        &t1.passDist[t1.info5[5 * i + 4]], q);
            H.count[i] = (uint32_t)m;
            for (int h = 0; h < m; ++h)
                if (std::isfinite(q[h].slope) && q[h].slope > 0) {
                    r.hi = std::max(r.hi, q[h].slope);
                    r.lo = std::min(r.lo, q[h].slope);
                }
        }
    });
    H.minSlope = INFINITY;
    H.maxSlope = 0;
    for (const Range& r : range) {
        H.maxSlope = std::max(H.maxSlope, r.hi);
        H.minSlope = std::min(H.minSlope, r.lo);
    }
}

void select(const Layout& L, const Hull& H, const double lambda[3], std::vector<uint8_t>& passes) {
    const int n = L.numCblks();
    rcParallel([&](int chunk, int) {
        const auto [i0, i1] = chunkRange(n, chunk);
        for (int i = i0; i < i1; ++i)
            passes[i] = (uint8_t)rc_select(H.at(i), (int)H.count[i], lambda[L.bands[L.cblks[i].band].comp]);
    });
}

// rcMeasure over packet ranges on the helpers: the same integer sums.
CodestreamSizes measureParallel(const RcTables& T, const Tier1Ref& t1, const uint8_t* passes) {
    const KeptBlocks view{&t1, passes};
    struct alignas(64) Part {
        unsigned long long tp[6] = {};
    };
    std::vector<Part> part(rcSlots());
    const int np = (int)T.packets.size();
    rcParallel([&](int chunk, int s) {
        const auto [k0, k1] = chunkRange(np, chunk);
        for (int k = k0; k < k1; ++k)
            part[s].tp[T.packets[k].tp] += rc_packet_bytes(T.packets[k], T.pbands.data(), view);
    });
    unsigned long long tp[6] = {};
    for (const Part& p : part)
        for (int k = 0; k < 6; ++k) tp[k] += p.tp[k];
    return sizesOf(T, tp);
}

}  // namespace

// Slopes on the absolute 1/1024-octave grid: bin k holds the slopes s with
// floor(1024 log2 s) = k. The bin of a double comes from its binary exponent and a table of
// the 1,024 steps of one octave (integer arithmetic only), and a bin's lower edge is a
// double read from the same table, so any implementation that shares the table makes the
// same choices.
const OctaveSteps& octaveSteps() {
    static const OctaveSteps t = [] {
        OctaveSteps o{};
        for (int j = 0; j < 1024; ++j) {
            const double v = std::exp2(j / 1024.0);  // in [1, 2)
            uint64_t bits;
            std::memcpy(&bits, &v, 8);
            o.mantissa[j] = bits & ((1ull << 52) - 1);
        }
        o.mantissa[1024] = 1ull << 52;
        // the first step at or above each of 1,024 equal mantissa ranges
        for (int r = 0, j = 0; r < 1024; ++r) {
            const uint64_t start = (uint64_t)r << 42;
            while (j < 1023 && o.mantissa[j + 1] <= start) ++j;
            o.first[r] = (uint16_t)j;
        }
        return o;
    }();
    return t;
}

int64_t slopeBin(double s) {  // s finite and > 0
    const OctaveSteps& t = octaveSteps();
    return rc_slope_bin(s, t.mantissa, t.first);
}

double binEdge(int64_t k) { return rc_bin_edge(k, octaveSteps().mantissa); }

namespace {

// Hull points binned by slope with suffix sums over the bins: data bytes and included-block
// counts for any bin threshold in O(1) (rate_control.cpp:117-162). Integer sums.
class SlopeHistogram {
public:
    // Buffers are reused across frames by the thread that owns the histogram. Each helper
    // slot counts its blocks into counts of its own, summed per bin afterwards.
    void build(const Layout& L, const Hull& H, int64_t kLo, int nb) {
        const OctaveSteps& t = octaveSteps();
        nb_ = nb;
        const size_t bins = 3 * (size_t)(nb + 1);
        part_.resize(rcSlots());
        for (Part& p : part_) p.used = false;
        const int n = L.numCblks();
        rcParallel([&](int chunk, int s) {
            Part& p = part_[s];
            if (!p.used) {  // a slot clears its counts when it first takes a chunk
                p.used = true;
                p.rate.assign(bins, 0ull);
                p.incl.assign(bins, 0ull);
            }
            const auto [i0, i1] = chunkRange(n, chunk);
            for (int i = i0; i < i1; ++i) {
                const size_t c = (size_t)L.bands[L.cblks[i].band].comp * (nb + 1);
                const RcPoint* q = H.at(i);
                uint32_t prev = 0;
                for (uint32_t h = 0; h < H.count[i]; ++h) {
                    const int b = rc_bin_of(q[h].slope, kLo, nb, t.mantissa, t.first);
                    p.rate[c + b] += q[h].rate - prev;
                    if (h == 0) p.incl[c + b] += 1;
                    prev = q[h].rate;
                }
            }
        });
        rate_.assign(bins, 0ull);
        incl_.assign(bins, 0ull);
        rcParallel([&](int chunk, int) {
            const auto [b0, b1] = chunkRange((int)bins, chunk);
            for (const Part& p : part_)
                if (p.used)
                    for (int b = b0; b < b1; ++b) {
                        rate_[b] += p.rate[b];
                        incl_[b] += p.incl[b];
                    }
        });
        for (int c = 0; c < 3; ++c) {
            unsigned long long* r = &rate_[(size_t)c * (nb + 1)];
            unsigned long long* k = &incl_[(size_t)c * (nb + 1)];
            for (int b = nb - 1; b >= 0; --b) {
                r[b] += r[b + 1];
                k[b] += k[b + 1];
            }
        }
    }
    double data(int c, int b) const { return (double)rate_[(size_t)c * (nb_ + 1) + b]; }
    double incl(int c, int b) const { return (double)incl_[(size_t)c * (nb_ + 1) + b]; }
    template <class Ok> int first(int lo, int hi, const Ok& ok) const {
        while (lo < hi) {
            const int mid = lo + (hi - lo) / 2;
            if (ok(mid)) hi = mid;
            else lo = mid + 1;
        }
        return lo;
    }

private:
    struct Part {
        bool used = false;
        std::vector<unsigned long long> rate, incl;
    };
    int nb_ = 0;
    std::vector<unsigned long long> rate_, incl_;  // [component][bin], nb + 1 bins each
    std::vector<Part> part_;
};

struct RateScratch {
    Hull hull;
    SlopeHistogram hist;
};

}  // namespace

RateResult allocateRate(const Layout& L, const Tier1Ref& t1, const RateLimits& lim) {
    thread_local RateScratch scratch;
    const Hull& H = scratch.hull;
    buildHull(L, t1, scratch.hull);
    RateResult res;
    res.passes.assign(L.numCblks(), 0);
    const OctaveSteps& t = octaveSteps();
    double maxSlope = H.maxSlope, minSlope = H.minSlope;
    if (maxSlope == 0) maxSlope = minSlope = 1;
    RcSearch S;
    S.init();
    rc_bin_range(minSlope, maxSlope, t.mantissa, t.first, S.kLo, S.nb);
    S.minSlope = minSlope;
    S.maxSlope = maxSlope;
    S.maxTotal = lim.maxTotal;
    S.maxComp = lim.maxComp;
    S.mantissa = t.mantissa;
    S.first = t.first;
    SlopeHistogram& hist = scratch.hist;
    hist.build(L, H, S.kLo, S.nb);
    const RcTables& T = packetTables(L);
    auto measure = [&](const double l[3]) {
        select(L, H, l, res.passes);
        res.sizes = measureParallel(T, t1, res.passes.data());
        return RcSizes{res.sizes.total, {res.sizes.comp[0], res.sizes.comp[1], res.sizes.comp[2]}};
    };
    RcSizes sz = measure(S.lambda);
    while (S.next(hist, sz)) sz = measure(S.lambda);
    res.iterations = (int)S.iterations;
    res.lambda = std::max({S.lambda[0], S.lambda[1], S.lambda[2]});
    for (int c = 0; c < 3; ++c) res.lambdaComp[c] = S.lambda[c];
    double dist = 0;  // one running sum in block order
    for (int i = 0; i < L.numCblks(); ++i) {
        const RcPoint* q = H.at(i);
        for (uint32_t h = 0; h < H.count[i]; ++h)
            if (q[h].passes > res.passes[i]) dist += q[h].gain;
    }
    res.distortion = dist;
    return res;
}

// ---------------------------------------------------------------- DCI check
std::string checkDciCodestream(const uint8_t* d, size_t n, double fps, bool fourk) {
    auto u16 = [&](size_t i) { return i + 1 < n ? (uint32_t)d[i] << 8 | d[i + 1] : 0u; };
    auto u32 = [&](size_t i) { return u16(i) << 16 | u16(i + 2); };
    if (n < 4 || u16(0) != SOC) return "no SOC";
    if (u16(n - 2) != EOC) return "no EOC";
    const double limit = std::rint(250e6 / (8.0 * fps));
    if ((double)n > limit) return "frame larger than the DCI limit";
    size_t p = 2;
    bool siz = false, cod = false, qcd = false, tlm = false, poc = false;
    std::vector<uint32_t> tlmLen;
    while (p + 4 <= n && u16(p) != SOT) {
        const uint32_t m = u16(p), len = u16(p + 2);
        if (len < 2 || p + 2 + len > n) return "truncated marker segment";
        if (m == SIZ) {
            siz = true;
            if (u16(p + 4) != (fourk ? 4u : 3u)) return "Rsiz is not the DCI profile";
            const uint32_t W = u32(p + 6), H = u32(p + 10);
            if (fourk ? (W > 4096 || H > 2160) : (W > 2048 || H > 1080)) return "picture exceeds the container";
            if (u16(p + 38) != 3) return "not three components";
            for (int c = 0; c < 3; ++c)
                if (d[p + 40 + 3 * c] != 11) return "component is not 12-bit";
        } else if (m == COD) {
            cod = true;
            if (d[p + 5] != 4) return "progression is not CPRL";
            if (u16(p + 6) != 1) return "more than one layer";
            if (d[p + 10] != 3 || d[p + 11] != 3) return "code-blocks are not 32x32";
            if (d[p + 12] != 0) return "code-block style is not 0";
            if (d[p + 13] != 0) return "transform is not 9/7";
            const int nl = d[p + 9];
            if (nl != (fourk ? 6 : 5)) return "unexpected decomposition levels";
        } else if (m == QCD) {
            qcd = true;
            if ((d[p + 4] & 0x1F) != 2) return "quantisation is not scalar expounded";
        } else if (m == POC) {
            poc = true;
        } else if (m == TLM) {
            tlm = true;
            if (d[p + 5] != 0x50) return "TLM is not 8/32-bit";
            for (size_t q = p + 6; q + 5 <= p + 2 + len; q += 5) tlmLen.push_back(u32(q + 1));
        }
        p += 2 + len;
    }
    if (!siz || !cod || !qcd || !tlm) return "missing main-header marker";
    if (fourk && !poc) return "4K frame without POC";
    const size_t ntp = fourk ? 6 : 3;
    if (tlmLen.size() != ntp) return "TLM does not list every tile-part";
    const double compLimit = 200e6 / (8.0 * fps);
    size_t comp[3] = {0, 0, 0};
    for (size_t t = 0; t < ntp; ++t) {
        if (u16(p) != SOT) return "tile-part without SOT";
        const uint32_t psot = u32(p + 6);
        if (psot != tlmLen[t]) return "Psot does not match TLM";
        if (d[p + 10] != t || d[p + 11] != ntp) return "tile-part numbering";
        if (u16(p + 12) != SOD) return "no SOD";
        comp[t % 3] += psot;
        p += psot;
        if (p > n - 2) return "tile-part runs past the end";
    }
    if (p != n - 2) return "bytes after the last tile-part";
    for (size_t c : comp)
        if ((double)c > compLimit) return "component exceeds 200 Mbit/s";
    return "";
}

}  // namespace gail_amd
