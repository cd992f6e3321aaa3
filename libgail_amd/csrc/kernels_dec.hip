// Decoder kernels for CDNA4 (gfx950, wave64).
//
// Tier-1: a wave per code-block, longest first (t1_decode_wave.h), which stores a block's
// reconstruction words once, or under load a lane per block (t1_decode_block.h), which adds to
// them. The planes are cleared beforehand, for the blocks without data too.
//
// Inverse DWT: one launch per level; a workgroup owns a TX x TY tile of the level's output
// and all three components. It gathers the tile plus a 4-sample mirrored halo from the four
// quadrants (dequantising the high bands, and the top level's LL, from their words on load),
// lifts the rows, then the columns, in registers, and writes the interleaved tile with
// coalesced row stores. Every sample sees the CPU reference's operations in its order
// (rows, then columns; scaling, then lifting steps -delta, -gamma, -beta, -alpha), and the
// kernels are built with -ffp-contract=off, so results are bit-identical to it.
//
// Inverse ICT: one thread per pixel, level shift, rounding, clamping to 12 bits, packing.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "kernels_dec.h"
#include "t1_decode_block.h"
#include "t1_decode_wave.h"
#include "t1_tables.h"

namespace gail_amd {

namespace {

__constant__ uint32_t kDecNext[2 * kMqCoderStates];
__constant__ uint32_t kDecInitial[4];
__constant__ uint8_t kDecSign[256];
__constant__ uint32_t kDecMq[47];
__constant__ uint8_t kDecZc[4 * 128];

// ISO/IEC 15444-1 Table F.4, rounded to float as the CPU reference rounds them.
constexpr float kK = (float)1.230174104914001;
constexpr float kInvK = (float)(1.0 / 1.230174104914001);
constexpr float kNegAlpha = (float)1.586134342059924;
constexpr float kNegBeta = (float)0.052980118572961;
constexpr float kNegGamma = (float)-0.882911075530934;
constexpr float kNegDelta = (float)-0.443506852043971;
// Inverse ICT (G.3).
constexpr float kR2 = (float)1.402, kG1 = (float)-0.34413, kG2 = (float)-0.71414, kB1 = (float)1.772;

// ---------------------------------------------------------------- Tier-1
__device__ __forceinline__ bool block_fields(const T1DecodeParams& P, const DecBlock& d, uint32_t& w, uint32_t& h,
                                             uint32_t& orient, uint32_t& nbps, uint32_t& passes) {
    w = (d.geom & 31u) + 1u;
    h = ((d.geom >> 5) & 31u) + 1u;
    orient = (d.geom >> 10) & 3u;
    nbps = (d.geom >> 12) & 63u;
    passes = (d.geom >> 18) & 255u;
    // the host builds the table from the layout; a wrong one still writes nothing outside
    return d.dst < P.nwords && P.nwords - d.dst >= (h - 1u) * P.stride + w;
}

// One frame at a time is bound by latency: it takes as long as its longest block, whose decisions
// are one serial chain. 4K at 250 Mbit/s: 2.00 ms, its longest block (1,477 bytes) alone 1.92. One
// lane per block, or a wave on the same sequential code with its state in scalar registers for
// the longest blocks, took 3.83 ms. With every decision in vector registers it is 2.6 ms (a
// decision that may end the walk pays 28 cycles and more to get from a vector comparison to a
// branch).
//
// Several decoders at once are bound by scalar issue, one instruction a cycle and CU: 5.3e8 of
// them in a 4K frame (19 million decisions), 0.87 ms, and 4.4e8 vector instructions beside them.
// So decode() and the column walk are written for few scalar instructions (t1_wave_mq.h). Eight
// decoders with everything in HBM run 765-775 frames/s; with 6.5e8 it was 675-690, and with a lane
// per block 735-750.
__global__ void __launch_bounds__(64 * kDecWaves) t1_decode_kernel(T1DecodeParams P) {
    __shared__ DecWave s_wave[kDecWaves];
    __shared__ uint2 s_next[kMqCoderStates];
    __shared__ uint32_t s_pack[16];
    __shared__ uint8_t s_sign[256];
    const int t = threadIdx.x;
    if (t < 16) {
        uint32_t v = 0x0C0C0C0Cu, j = 0;
        for (uint32_t k = 0; k < 4; ++k)
            if ((t >> k) & 1) {
                v = (v & ~(0xFFu << (8 * j))) | (k << (8 * j));
                ++j;
            }
        s_pack[t] = v;
    }
    for (int i = t; i < kMqCoderStates; i += 64 * kDecWaves) s_next[i] = make_uint2(kDecNext[2 * i], kDecNext[2 * i + 1]);
    for (int i = t; i < 256; i += 64 * kDecWaves) s_sign[i] = kDecSign[i];
    const uint32_t lane = (uint32_t)t & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
    __syncthreads();
    const uint32_t gw = blockIdx.x * kDecWaves + wave;
    if (gw >= P.nblocks) return;
    uint32_t w, h, orient, nbps, passes;
    const DecBlock d = P.blocks[gw];
    if (!block_fields(P, d, w, h, orient, nbps, passes)) return;
    WaveMq mq;
    const uint32_t row = min(lane, 46u);
    mq.next_m = s_next[2u * row].x;
    mq.next_x = s_next[2u * row].x ^ s_next[2u * row].y;
    mq.next = s_next;
    // contexts start in their Table D.7 states
    mq.ctx = kDecInitial[lane == 1u ? 1u : (lane == 18u ? 2u : (lane == 19u ? 3u : 0u))];
    mq.ctx = lane == 0u ? 0u : mq.ctx;
    mq.ws = &s_wave[wave];
    mq.src = P.bytes + d.off;
    mq.len = d.len;
    t1_decode_wave(mq, w, h, orient, nbps, passes, P.words + d.dst, P.stride, s_pack, s_sign);
}

// What a wave with a block in each of its first lanes keeps in LDS, at [entry][lane]: a bank per
// lane, whatever row each lane is on.
struct DecLanes {
    uint32_t rows[4][32][kDecWaveLanes];
    uint32_t ctx[19][kDecWaveLanes];
};

struct LaneState {
    DecLanes* s;
    const uint32_t* mq;   // Table C.2
    const uint8_t* zct;   // Table D.1 of the block's orientation
    uint32_t lane;
    __device__ __forceinline__ void reset() {
        for (uint32_t r = 0; r < 32u; ++r)
#pragma unroll
            for (int t = 0; t < 4; ++t) s->rows[t][r][lane] = 0u;
        for (uint32_t c = 0; c < 19u; ++c) s->ctx[c][lane] = mq[t1d_initial_state(c)];
    }
    __device__ __forceinline__ uint32_t rows(int t, uint32_t r) const { return s->rows[t][r][lane]; }
    __device__ __forceinline__ void set_rows(int t, uint32_t r, uint32_t v) { s->rows[t][r][lane] = v; }
    __device__ __forceinline__ uint32_t ctx(uint32_t c) const { return s->ctx[c][lane]; }
    __device__ __forceinline__ void set_ctx(uint32_t c, uint32_t v) { s->ctx[c][lane] = v; }
    __device__ __forceinline__ uint32_t tab(uint32_t i) const { return mq[i]; }
    __device__ __forceinline__ uint32_t zc(uint32_t code) const { return zct[code]; }
};

// A lane's words, added to as its samples are decoded: no lane waits for a read of its output.
struct AtomicSink {
    uint32_t* base;
    uint32_t stride;
    __device__ __forceinline__ void add(uint32_t i, uint32_t v) {
        __hip_atomic_fetch_add(base + i, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
};

// For devices that several decoders keep busy with long codewords (DescPlan::plan): the sequential
// decoder (t1_decode_block.h), a block in each of a wave's first 16 lanes. Lanes that are at the
// same kind of decision share its instructions, which a wave per block cannot; each one's chain
// takes three times as long. 22 MB 4K frames, eight decoders: 189 frames/s, 88 with a wave per
// block. The states of 16 lanes take 9.4 KB, so 16 waves a CU fit (more lanes, fewer waves).
__global__ void __launch_bounds__(64 * kDecWaves) t1_decode_lanes_kernel(T1DecodeParams P) {
    __shared__ DecLanes s_lanes[kDecWaves];
    __shared__ uint32_t s_mq[47];
    __shared__ uint8_t s_zc[4 * 128];
    const int t = threadIdx.x;
    if (t < 47) s_mq[t] = kDecMq[t];
    for (int i = t; i < 4 * 128; i += 64 * kDecWaves) s_zc[i] = kDecZc[i];
    __syncthreads();
    const uint32_t lane = (uint32_t)t & 63u, wave = (uint32_t)t >> 6;
    const uint32_t at = (blockIdx.x * kDecWaves + wave) * kDecWaveLanes + lane;
    if (lane >= kDecWaveLanes || at >= P.nblocks) return;
    uint32_t w, h, orient, nbps, passes;
    const DecBlock d = P.blocks[at];
    if (d.dst == kDecEmpty || !block_fields(P, d, w, h, orient, nbps, passes)) return;
    LaneState st{&s_lanes[wave], s_mq, s_zc + 128u * orient, lane};
    AtomicSink out{P.words + d.dst, P.stride};
    t1d_decode_block(st, P.bytes, d.off, d.len, w, h, nbps, passes, out);
}

// ---------------------------------------------------------------- inverse DWT
// Whole-sample symmetric extension of index i into [0, n).
__device__ __forceinline__ int mirror(int i, int n) {
    if ((unsigned)i < (unsigned)n) return i;
    if (n == 1) return 0;
    const int period = 2 * (n - 1);
    i %= period;
    if (i < 0) i += period;
    return i < n ? i : period - i;
}

__device__ __forceinline__ float dequant(uint32_t wd, float half) {
    const float a = (float)(wd & 0x7FFFFFFFu) * half;
    return (wd & 0x80000000u) ? -a : a;
}

// Inverse lifting of N samples in registers, sample k at parity k & 1 (the tile origin is
// even). The end samples lack a neighbour and are left alone; the halo absorbs the damage.
template <int N> __device__ __forceinline__ void unlift97(float (&v)[N]) {
#pragma unroll
    for (int k = 2; k + 1 < N; k += 2) v[k] += kNegDelta * (v[k - 1] + v[k + 1]);
#pragma unroll
    for (int k = 1; k + 1 < N; k += 2) v[k] += kNegGamma * (v[k - 1] + v[k + 1]);
#pragma unroll
    for (int k = 2; k + 1 < N; k += 2) v[k] += kNegBeta * (v[k - 1] + v[k + 1]);
#pragma unroll
    for (int k = 1; k + 1 < N; k += 2) v[k] += kNegAlpha * (v[k - 1] + v[k + 1]);
}

constexpr int kIdwtTX = 64, kIdwtTY = 32;

template <int TX, int TY> __global__ void __launch_bounds__(256) idwt_level_kernel(IdwtLevel P) {
    constexpr int RX = TX + 8, RY = TY + 8, PITCH = RX + 1;
    constexpr int NPOS = RX * RY;
    constexpr int PER = (NPOS + 255) / 256;
    __shared__ float tile[3][RY][PITCH];
    // Workgroup b runs on XCD b % 8; each XCD takes a contiguous range of tiles, so tiles
    // that share halo rows meet in the same L2.
    const int nb = (int)gridDim.x, q = nb >> 3, rem = nb & 7;
    const int xcd = (int)blockIdx.x & 7, jb = (int)blockIdx.x >> 3;
    const int t = xcd * q + min(xcd, rem) + jb;
    const int x0 = (t % P.tiles_x) * TX, y0 = (t / P.tiles_x) * TY;
    const int w = P.w, h = P.h, sw = (w + 1) >> 1, sh = (h + 1) >> 1;
    const bool rows_on = w >= 2, cols_on = h >= 2;
    const int tid = threadIdx.x;

    // Gather: the interleaved sample (gx, gy) is column gx / 2 of the low or high half and
    // row gy / 2 of the low or high half, by parity.
    uint32_t at[PER];
    int orient[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int i = tid + 256 * j;
        const int ry = i / RX, rx = i - ry * RX;
        const int gy = mirror(y0 - 4 + ry, h), gx = mirror(x0 - 4 + rx, w);
        const int r = (gy & 1) ? sh + (gy >> 1) : (gy >> 1);
        const int c = (gx & 1) ? sw + (gx >> 1) : (gx >> 1);
        at[j] = (uint32_t)r * P.stride + (uint32_t)c;
        orient[j] = (gx & 1) | ((gy & 1) << 1);
    }
#pragma unroll
    for (int comp = 0; comp < 3; ++comp) {
        const uint32_t* wsrc = P.words + (size_t)comp * P.plane;
        const float* lsrc = P.ll ? P.ll + (size_t)comp * P.plane : nullptr;
        const float h0 = P.half[comp][0], h1 = P.half[comp][1], h2 = P.half[comp][2], h3 = P.half[comp][3];
        float v[PER];
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            if (NPOS % 256 != 0 && tid + 256 * j >= NPOS) continue;
            const int o = orient[j];
            if (o == 0 && lsrc) {
                v[j] = lsrc[at[j]];
            } else {
                v[j] = dequant(wsrc[at[j]], o == 0 ? h0 : (o == 1 ? h1 : (o == 2 ? h2 : h3)));
            }
        }
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const int i = tid + 256 * j;
            if (NPOS % 256 != 0 && i >= NPOS) continue;
            const int ry = i / RX, rx = i - ry * RX;
            // the row transform starts by scaling: low half times K, high half times 1/K
            tile[comp][ry][rx] = rows_on ? v[j] * ((rx & 1) ? kInvK : kK) : v[j];
        }
    }
    __syncthreads();
    // Rows: one thread per staged row of each component.
    if (rows_on) {
        for (int i = tid; i < 3 * RY; i += 256) {
            const int c = i / RY, ry = i - c * RY;
            float v[RX];
#pragma unroll
            for (int k = 0; k < RX; ++k) v[k] = tile[c][ry][k];
            unlift97(v);
#pragma unroll
            for (int k = 4; k < TX + 4; ++k) tile[c][ry][k] = v[k];
        }
        __syncthreads();
    }
    // Columns: one thread per output column of each component.
    if (cols_on) {
        for (int i = tid; i < 3 * TX; i += 256) {
            const int c = i / TX, rx = 4 + (i - c * TX);
            float v[RY];
#pragma unroll
            for (int k = 0; k < RY; ++k) v[k] = tile[c][k][rx] * ((k & 1) ? kInvK : kK);
            unlift97(v);
#pragma unroll
            for (int k = 4; k < TY + 4; ++k) tile[c][k][rx] = v[k];
        }
        __syncthreads();
    }
    // Coalesced row stores of the interleaved tile.
    constexpr int ROWS = 256 / TX;
    const int k = tid % TX, r0 = tid / TX, gx = x0 + k;
    if (gx >= w) return;
#pragma unroll 4
    for (int j = 0; j < 3 * TY / ROWS; ++j) {
        const int c = j / (TY / ROWS), r = r0 + ROWS * (j % (TY / ROWS)), gy = y0 + r;
        if (gy < h) P.dst[(size_t)c * P.plane + (size_t)gy * P.stride + gx] = tile[c][4 + r][4 + k];
    }
}

// Dequantised words of a whole frame (the wavelet planes before the inverse DWT).
__global__ void __launch_bounds__(256) dequant_frame_kernel(DequantFrame P) {
    __shared__ float s_half[9 * 4];
    const uint32_t x = blockIdx.x * 256 + threadIdx.x, y = blockIdx.y, c = blockIdx.z;
    if (threadIdx.x < 36) s_half[threadIdx.x] = P.half[c][threadIdx.x >> 2][threadIdx.x & 3];
    __syncthreads();
    if (x >= P.width) return;
    // the band holding (x, y) in the Mallat layout
    uint32_t ww = P.width, hh = P.height, level = P.levels, orient = 0;
    for (uint32_t l = 1; l <= P.levels; ++l) {
        const uint32_t nw = (ww + 1) >> 1, nh = (hh + 1) >> 1;
        if (x >= nw || y >= nh) {
            level = l;
            orient = (x >= nw ? 1u : 0u) | (y >= nh ? 2u : 0u);
            break;
        }
        ww = nw;
        hh = nh;
    }
    const size_t i = (size_t)c * P.width * P.height + (size_t)y * P.width + x;
    P.dst[i] = dequant(P.words[i], s_half[level * 4 + orient]);
}

// ---------------------------------------------------------------- inverse ICT and packing
__global__ void __launch_bounds__(256) ict_pack_kernel(IctPack P) {
    const int x = blockIdx.x * 256 + threadIdx.x, y = blockIdx.y;
    if (x >= P.w) return;
    const size_t i = (size_t)y * P.stride + x;
    const float y0 = P.planes[i], y1 = P.planes[P.plane + i], y2 = P.planes[2 * (size_t)P.plane + i];
    float v[3];
    v[0] = y0 + kR2 * y2;
    v[1] = y0 + kG1 * y1 + kG2 * y2;
    v[2] = y0 + kB1 * y1;
    uint16_t* o = reinterpret_cast<uint16_t*>(P.out + (int64_t)y * P.pitch) + 3 * (size_t)x;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        int code = (int)floorf(v[k] + 2048.5f);
        code = code < 0 ? 0 : (code > 4095 ? 4095 : code);
        o[k] = (uint16_t)(code << P.shift);
    }
}

}  // namespace

hipError_t dec_tables_init() {
    uint32_t tab[2 * kMqCoderStates], initial[4];
    build_mq_coder_table(tab, initial, 15);
    uint8_t sign[256];
    build_sign_table(sign);
    uint32_t mq[47];
    build_mq_table(mq);
    uint8_t zc[4 * 128];
    build_zc_table(zc);
    hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(kDecMq), mq, sizeof mq);
    if (e == hipSuccess) e = hipMemcpyToSymbol(HIP_SYMBOL(kDecZc), zc, sizeof zc);
    if (e == hipSuccess) e = hipMemcpyToSymbol(HIP_SYMBOL(kDecNext), tab, sizeof tab);
    if (e == hipSuccess) e = hipMemcpyToSymbol(HIP_SYMBOL(kDecInitial), initial, sizeof initial);
    return e != hipSuccess ? e : hipMemcpyToSymbol(HIP_SYMBOL(kDecSign), sign, sizeof sign);
}

// Zeroes n words at p (16-byte aligned): four words per store, a grid-stride loop.
__global__ void __launch_bounds__(256) zero_words_kernel(uint32_t* p, uint64_t n) {
    const uint64_t quads = n / 4, step = (uint64_t)gridDim.x * blockDim.x;
    uint4* q = reinterpret_cast<uint4*>(p);
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < quads; i += step) q[i] = make_uint4(0, 0, 0, 0);
    const uint64_t t = quads * 4 + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (blockIdx.x == 0 && t < n) p[t] = 0u;
}

hipError_t launch_zero_words(uint32_t* p, size_t n, hipStream_t s) {
    if (!n) return hipSuccess;
    if ((uintptr_t)p % 16) return hipErrorInvalidValue;
    const uint64_t quads = n / 4;
    const unsigned groups = (unsigned)std::min<uint64_t>(4096, (quads + 255) / 256 + 1);
    hipLaunchKernelGGL(zero_words_kernel, dim3(groups), dim3(256), 0, s, p, (uint64_t)n);
    return hipGetLastError();
}

hipError_t launch_t1_decode(const T1DecodeParams& p, hipStream_t s) {
    if (!p.nblocks) return hipSuccess;
    const uint32_t per = (uint32_t)kDecWaves * p.lanes, groups = (p.nblocks + per - 1) / per;
    if (p.lanes == 1)
        hipLaunchKernelGGL(t1_decode_kernel, dim3(groups), dim3(64 * kDecWaves), 0, s, p);
    else
        hipLaunchKernelGGL(t1_decode_lanes_kernel, dim3(groups), dim3(64 * kDecWaves), 0, s, p);
    return hipGetLastError();
}

void idwt_tile_size(int& tx, int& ty) {
    tx = kIdwtTX;
    ty = kIdwtTY;
}

hipError_t launch_idwt_level(const IdwtLevel& p, hipStream_t s) {
    hipLaunchKernelGGL((idwt_level_kernel<kIdwtTX, kIdwtTY>), dim3(p.tiles), dim3(256), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_dequant_frame(const DequantFrame& p, hipStream_t s) {
    hipLaunchKernelGGL(dequant_frame_kernel, dim3((p.width + 255) / 256, p.height, 3), dim3(256), 0, s, p);
    return hipGetLastError();
}

hipError_t launch_ict_pack(const IctPack& p, hipStream_t s) {
    hipLaunchKernelGGL(ict_pack_kernel, dim3((p.w + 255) / 256, p.h), dim3(256), 0, s, p);
    return hipGetLastError();
}

}  // namespace gail_amd
