// Host build of the wave decoder's arithmetic decoder (libgail_amd/csrc/t1_wave_mq.h) for the CPU
// tests: the source the GPU runs, one lane's values in place of a wave's. Test infrastructure.
//   host_wave_t1_words    a code-block through it, in the order t1_decode_wave.h makes the
//                         decisions: refinement a stripe at a time as a list, the rest one by one
//   host_wave_mq_fuzz     decisions against the sequential decoder (MqDec, t1_decode_block.h)
// With WAVEMQ_MAIN a program that runs both under the sanitizers.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <random>
#include <vector>

#include "t1_decode_block.h"
#include "t1_tables.h"
#include "t1_wave_mq.h"

using namespace gail_amd;

namespace {

struct Tables {
    DwPair next[kMqCoderStates];
    uint32_t initial[4], mq[47];
    uint8_t sign[256], zc[4 * 128];
    Tables() {
        uint32_t tab[2 * kMqCoderStates];
        build_mq_coder_table(tab, initial, 15);
        for (int i = 0; i < kMqCoderStates; ++i) next[i] = DwPair{tab[2 * i], tab[2 * i + 1]};
        build_mq_table(mq);
        build_sign_table(sign);
        build_zc_table(zc);
    }
};
const Tables g_tab;

// The codeword in memory as the device buffer holds it: readable 64 bytes past its end.
std::vector<uint8_t> padded(const uint8_t* data, uint32_t len) {
    std::vector<uint8_t> buf((size_t)len + 64, 0xA5);
    if (len) std::memcpy(buf.data(), data, len);
    return buf;
}

struct Wave {
    std::unique_ptr<DecWave> ws{new DecWave()};
    WaveMq mq{};
    Wave(const uint8_t* src, uint32_t len) {
        for (uint32_t lane = 0; lane < 64; ++lane) {
            const uint32_t row = lane < 46 ? lane : 46;
            mq.next_m.v[lane] = g_tab.next[2 * row].x;
            mq.next_x.v[lane] = g_tab.next[2 * row].x ^ g_tab.next[2 * row].y;
            mq.ctx.v[lane] = lane ? g_tab.initial[lane == 1 ? 1 : (lane == 18 ? 2 : (lane == 19 ? 3 : 0))] : 0u;
        }
        mq.next = g_tab.next;
        mq.ws = ws.get();
        mq.src = src;
        mq.len = len;
        mq.init();
    }
    uint32_t decide(uint32_t cx) { return mq.decode(cx + 1) >> 31; }
    // Decisions in the given contexts through a stripe's list.
    std::vector<uint32_t> list(const std::vector<uint32_t>& cx) {
        uint8_t* const l = (uint8_t*)ws->list;
        for (size_t i = 0; i < cx.size(); ++i) l[i] = (uint8_t)((cx[i] + 1) << 2 | (i & 3));
        for (size_t i = 0; i < 8; ++i) l[cx.size() + i] = 0;
        mq.refine((uint32_t)cx.size());
        std::vector<uint32_t> out(cx.size());
        for (size_t i = 0; i < cx.size(); ++i) out[i] = (ws->bits[i >> 2] >> (i & 3)) & 1u;
        return out;
    }
};

struct SeqState {
    uint32_t c[19];
    SeqState() {
        for (uint32_t i = 0; i < 19; ++i) c[i] = g_tab.mq[t1d_initial_state(i)];
    }
    uint32_t ctx(uint32_t i) const { return c[i]; }
    void set_ctx(uint32_t i, uint32_t v) { c[i] = v; }
    uint32_t tab(uint32_t i) const { return g_tab.mq[i]; }
};

}  // namespace

extern "C" {

int host_wave_t1_words(const uint8_t* data, uint32_t len, int w, int h, int orient, int nbps, int passes,
                       uint32_t* words) {
    const std::vector<uint8_t> buf = padded(data, len);
    Wave wave(buf.data(), len);
    // a border of insignificant samples around the block
    static thread_local uint8_t sig[34][34], neg[34][34], seen[34][34], refined[34][34];
    for (auto* a : {&sig, &neg, &seen, &refined}) std::memset(*a, 0, sizeof *a);
    std::memset(words, 0, sizeof(uint32_t) * w * h);
    const uint8_t* zc = g_tab.zc + 128 * (orient & 3);
    auto code = [&](int y, int x) {
        auto s = [&](int dy, int dx) { return (int)sig[y + 1 + dy][x + 1 + dx]; };
        return (s(0, -1) + s(0, 1)) | (s(-1, 0) + s(1, 0)) << 2 |
               (s(-1, -1) + s(-1, 1) + s(1, -1) + s(1, 1)) << 4;
    };
    int p = nbps - 1, type = 2;
    auto significant = [&](int y, int x) {
        auto side = [&](int dy, int dx) { return sig[y + 1 + dy][x + 1 + dx] | neg[y + 1 + dy][x + 1 + dx] << 1; };
        const int e = g_tab.sign[side(0, -1) | side(0, 1) << 2 | side(-1, 0) << 4 | side(1, 0) << 6];
        const uint32_t s = wave.decide((uint32_t)(e >> 1) - 1u) ^ (uint32_t)(e & 1);
        sig[y + 1][x + 1] = 1;
        neg[y + 1][x + 1] = (uint8_t)s;
        words[y * w + x] = (s << 31) | (3u << p);
    };
    passes = passes < 3 * nbps - 2 ? passes : 3 * nbps - 2;
    for (int pass = 0; pass < passes; ++pass) {
        for (int y0 = 0; y0 < h; y0 += 4) {
            const int y1 = y0 + 4 < h ? y0 + 4 : h;
            if (type == 1) {
                std::vector<uint32_t> cx;
                std::vector<int> at;
                for (int x = 0; x < w; ++x)
                    for (int y = y0; y < y1; ++y)
                        if (sig[y + 1][x + 1] && !seen[y + 1][x + 1]) {
                            cx.push_back(refined[y + 1][x + 1] ? 16u : (code(y, x) ? 15u : 14u));
                            at.push_back(y * w + x);
                            refined[y + 1][x + 1] = 1;
                        }
                if (cx.empty()) continue;
                const std::vector<uint32_t> bit = wave.list(cx);
                for (size_t i = 0; i < at.size(); ++i) words[at[i]] += bit[i] ? 1u << p : 0u - (1u << p);
                continue;
            }
            for (int x = 0; x < w; ++x) {
                int y = y0;
                if (type == 2 && y1 - y0 == 4) {
                    bool run = true;
                    for (int k = y0; k < y1; ++k) run = run && !sig[k + 1][x + 1] && !seen[k + 1][x + 1] && !code(k, x);
                    if (run) {
                        if (!wave.decide(17u)) continue;
                        y = (int)(wave.decide(18u) << 1);
                        y = y0 + (y | (int)wave.decide(18u));
                        significant(y++, x);
                    }
                }
                for (; y < y1; ++y) {
                    if (sig[y + 1][x + 1] || (type == 2 && seen[y + 1][x + 1])) continue;
                    const int c = code(y, x);
                    if (type == 0 && !c) continue;
                    if (type == 0) seen[y + 1][x + 1] = 1;
                    if (wave.decide(zc[c])) significant(y, x);
                }
            }
        }
        if (type == 2) {
            std::memset(seen, 0, sizeof seen);
            type = 0;
            --p;
        } else {
            ++type;
        }
    }
    return 0;
}

// Codewords that differ: random bytes, 0xFF followed by what may follow it (0x80-0x8F among it),
// markers; each decoded by runs of single decisions and of lists in random contexts.
int host_wave_mq_fuzz(uint32_t seed, int codewords) {
    std::mt19937 rng(seed);
    auto below = [&](uint32_t n) { return (uint32_t)(rng() % n); };
    int bad = 0;
    for (int k = 0; k < codewords; ++k) {
        const uint32_t len = below(8) ? below(64) : below(700), kind = below(4);
        std::vector<uint8_t> data(len);
        static const uint8_t after[5] = {0x00, 0x7F, 0x80, 0x85, 0x8F}, marks[6] = {0xFF, 0xFF, 0x80, 0x8F, 0x90, 0x00};
        for (uint32_t i = 0; i < len; ++i) {
            data[i] = kind == 3 ? marks[below(6)] : (uint8_t)rng();
            if (kind < 2 && i + 1 < len && !below(4)) {
                data[i] = 0xFF;
                data[++i] = after[below(5)];
            }
        }
        const std::vector<uint8_t> buf = padded(data.data(), len);
        std::vector<uint8_t> seq_buf((size_t)len + 64, 0xA5);  // MqDec reads whole 8-byte words
        if (len) std::memcpy(seq_buf.data(), data.data(), len);
        Wave wave(buf.data(), len);
        SeqState st;
        MqDec seq;
        seq.init(seq_buf.data(), 0, len);
        const uint32_t total = 8 * len + 40;
        bool same = true;
        for (uint32_t done = 0; done < total && same;) {
            const uint32_t n = 1 + below(below(3) ? 12 : 128);
            const bool lists = below(3) != 0;
            std::vector<uint32_t> cx(n), got(n);
            for (uint32_t i = 0; i < n; ++i) cx[i] = lists && below(8) ? 14 + below(3) : below(19);
            if (lists) got = wave.list(cx);
            else
                for (uint32_t i = 0; i < n; ++i) got[i] = wave.decide(cx[i]);
            for (uint32_t i = 0; i < n; ++i) same = seq.decode(st, cx[i]) == got[i] && same;
            done += n;
        }
        bad += !same;
    }
    return bad;
}

}  // extern "C"

#ifdef WAVEMQ_MAIN
int main(int argc, char** argv) {
    const int n = argc > 1 ? std::atoi(argv[1]) : 20000;
    const int bad = host_wave_mq_fuzz(1u, n);
    std::mt19937 rng(2);
    for (int k = 0; k < n / 10; ++k) {
        std::vector<uint8_t> data(rng() % 300);
        for (uint8_t& b : data) b = rng() % 3 ? (uint8_t)rng() : 0xFF;
        uint32_t words[32 * 32];
        const int nbps = 1 + (int)(rng() % 30);
        host_wave_t1_words(data.data(), (uint32_t)data.size(), 1 + (int)(rng() % 32), 1 + (int)(rng() % 32), k & 3, nbps,
                           1 + (int)(rng() % (3 * nbps)), words);
    }
    std::printf("%d of %d codewords differ\n", bad, n);
    return bad != 0;
}
#endif
