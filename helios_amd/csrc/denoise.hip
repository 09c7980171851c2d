// denoise.hip — the learned denoiser: a U-Net (levels of 32/48/64/96
// channels, 3x3 convolutions, ReLU, 2x2 average pooling, nearest upsampling
// with skip concatenation, 1x1 head adding the input's log radiance) trained
// and run with hand-written BF16 MFMA kernels that accumulate in FP32.
//
// The reference has no denoiser; this network is the build's own. Its
// restatement in numpy (oracle/unet.py) is the checker of these kernels.
//
// Layout: activations are NHWC BF16 with the channel count a multiple of 8,
// so a lane's 8-channel group is one 16-byte load. The network image is the
// input padded with zeros to multiples of 8 (three pooling levels).
//
// Convolution = implicit GEMM on v_mfma_f32_16x16x32_bf16 with output
// channels as the M dimension, pixels as N and K = 9 taps x input channels:
//   A (16 x 32)  weights  [Cout][Kpad], k = tap * Cin + c  (lane: row l%16,
//                k = 8 (l/16) .. +7)
//   B (32 x 16)  inputs   pixel (l%16) of the tile, channels of k's tap
//   D (16 x 16)  lane holds pixel l%16, rows 4 (l/16) .. +3 of A
// The decoder's "upsample, then concatenate with the skip tensor" is not
// materialized: the B loader reads channels [0, C0) from the low-resolution
// tensor at (y/2, x/2) and [C0, C0+C1) from the skip tensor.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "internal.hpp"

namespace hh {
namespace dn {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));

// What a convolution does with its sums: bias + ReLU -> BF16 (also 2x2 averaged
// into `pool`, or through the 1x1 head instead of being stored), times a ReLU
// mask -> BF16, or FP32. EPI_SPLIT is EPI_BIAS_RELU with another order of the
// sums (see k_conv3x3).
enum Epi { EPI_BIAS_RELU = 0, EPI_MASK = 1, EPI_F32 = 2, EPI_POOL = 3, EPI_HEAD = 4, EPI_SPLIT = 5 };
struct ConvExtra {
    __bf16* pool;              // EPI_POOL: half-resolution average
    const __bf16* wh;          // EPI_HEAD: head weights (3, 32) and bias,
    const float* bh;
    const float4* resid;       // the input's log radiance,
    float4* out;               // the network output in log space (when set)
    float4* surface;           // and the h x w surface (when set)
    uint32_t h, w;
};

__device__ inline bf16x8 zero8() {
    bf16x8 z;
#pragma unroll
    for (int i = 0; i < 8; i++) z[i] = (__bf16)0.0f;
    return z;
}

// ---------------------------------------------------------------------------
// 3x3 convolution (forward, and the input gradient with flipped weights).
// A workgroup of four waves computes tiles of output rows x pixels of CB output
// channels (gridDim.y slices of them). Input channels are taken 32 at a time:
// the halo tile of those channels and their weights are staged in LDS (16-byte
// loads, zero outside the image and beyond CT; the upsample + concat of the
// decoder is resolved here), then all 9 taps read their operands from LDS. The
// K order is (channel group, tap, channel), whatever the tile.
//
// A wave holds R rows x 16 NT pixels x CB channels of accumulators and keeps
// the weights of a tap row in registers: per 9 R NT MT MFMAs of a group it
// reads 9 (MT + R NT) fragments from LDS.
//
// EPI_SPLIT (the 48^ + 32 -> 32 decoder layer in inference): groups of one
// source each, and the order (group, horizontal tap, vertical tap, channel),
// which reads an input row once for up to three output rows, 9 MT +
// 3 (R + 2) NT fragments: 156 -> 128 us at 1920 x 1080. The other layers gain
// nothing from it (632 us in all with it everywhere, 641 here); training
// keeps one order of the sums throughout.
//
// What bounds it is the vector instructions around the MFMAs: with the places
// of a tile's chunks divided out of the thread number and checked per lane, a
// tile of the 32 -> 32 layer took 650 of them per wave beside 72 MFMAs, and
// prefetching or fusing gained nothing. So a pass of the staging takes a fixed
// column per thread and a row per pass, whose address and range check are the
// wave's (a buffer descriptor, of length zero for a row outside); workgroups
// are persistent and keep the weights of a single-group layer, and load the
// next group or tile during the MFMAs. 2x2 pooling and the 1x1 head are done
// on the accumulators: their activations need not be read again (nor, for the
// head in inference, written). 1920 x 1080, one state kept: 867 -> 641 us for
// the network (32 -> 32 at full resolution 77 -> 64 us with pooling, its
// activations' copy time 58; the 48^ + 32 -> 32 decoder layer 180 -> 128).
// Two workgroups per resident slot instead of one: 689 against 668; a tile per
// workgroup: 718.
//
// Large images: tiles 64 pixels wide, whose halo is 1.5 (1.25) times the tile.
// Eight rows (R = 4) only for 32 channels of several groups, where the staged
// weights and the fragment reads of LDS weigh most: 174 -> 128 us; with 48
// channels they spill (69 -> 100 us), and single-group layers are bound by
// memory and want the third workgroup per CU.
// Images with too few such tiles to fill the chip: 4 rows x 16 pixels and
// slices of 32 or 48 channels, a shorter chain for more workgroups. 417 x 233:
// 173 -> 98 us (large tiles there: 204); eight 128 x 128 images of a training
// step: 1143 -> 990.
struct ConvLarge {
    static constexpr int R(int cout, int ng) { return cout <= 32 && ng > 1 ? 4 : 2; }
    static constexpr int NT = 2, WR = 2, WC = 2;
    static constexpr int CB(int cout) { return cout > 112 ? cout / 2 : cout; }
};
struct ConvSmall {
    static constexpr int R(int, int) { return 1; }
    static constexpr int NT = 1, WR = 4, WC = 1;
    static constexpr int CB(int cout) { return cout % 48 == 0 ? 48 : (cout % 32 == 0 ? 32 : cout); }
};
struct ConvSmallPool : ConvSmall {   // a wave needs both rows of a 2 x 2 average
    static constexpr int R(int, int) { return 2; }
};
constexpr int kConvThreads = 256;
// Waves per SIMD that the LDS of one workgroup (halo tile + staged weights)
// allows on a 160 KB CU, one wave per SIMD per workgroup, and that the
// accumulators and the chunks in flight leave registers for: the register
// budget is held to it.
constexpr int conv_waves(int lds, int acc) {
    const int w = 163840 / lds, v = acc <= 32 ? 3 : (acc <= 64 ? 2 : 1);
    return w < 1 ? 1 : (w < v ? w : v);
}
template <typename CFG, int C0, int C1, int COUT>
struct ConvShape {
    static constexpr int NG = (C0 + C1 + 31) / 32;           // groups of 32 channels
    static constexpr int R = CFG::R(COUT, NG), NT = CFG::NT, WR = CFG::WR, WC = CFG::WC, CB = CFG::CB(COUT);
    static constexpr int MT = CB / 16, ROWS = R * WR, COLS = 16 * NT * WC;
    static constexpr int TR = ROWS + 2, TC = COLS + 2;       // halo tile
    static constexpr int LDS = (TR * TC + 9 * CB) * 64, ACC = 4 * R * MT * NT;
    static_assert(WR * WC * 64 == kConvThreads && COUT % CB == 0 && CB % 16 == 0, "workgroup shape");
};
// LC consecutive BF16 channels (LC a multiple of 4) as the widest aligned stores.
template <int LC>
__device__ inline void store_channels(__bf16* p, const __bf16* v) {
    if constexpr (LC % 8 == 0) {
#pragma unroll
        for (int j = 0; j < LC; j += 8) {
            bf16x8 q;
#pragma unroll
            for (int i = 0; i < 8; i++) q[i] = v[j + i];
            *(bf16x8*)(p + j) = q;
        }
    } else {
#pragma unroll
        for (int j = 0; j < LC; j += 4) {
            bf16x4 q;
#pragma unroll
            for (int i = 0; i < 4; i++) q[i] = v[j + i];
            *(bf16x4*)(p + j) = q;
        }
    }
}
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
// The value of the lane whose number differs in the last bit.
__device__ inline bf16x2 lane_pair(bf16x2 v) {
    return __builtin_bit_cast(bf16x2, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));
}
// a summed over lanes l and l + 32 in lanes 0-31, b likewise in lanes 32-63.
__device__ inline float add_halves(float a, float b) {
    const auto s = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false);
    return __builtin_bit_cast(float, (uint32_t)s[0]) + __builtin_bit_cast(float, (uint32_t)s[1]);
}
// a summed over rows of 16 lanes 2k and 2k + 1 in row 2k, b likewise in row 2k + 1.
__device__ inline float add_rows(float a, float b) {
    const auto s = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false);
    return __builtin_bit_cast(float, (uint32_t)s[0]) + __builtin_bit_cast(float, (uint32_t)s[1]);
}
template <int C0, int UP0, int C1, int COUT, int EPI, typename CFG>
__global__ void __launch_bounds__(kConvThreads)
__attribute__((amdgpu_waves_per_eu(conv_waves(ConvShape<CFG, C0, C1, COUT>::LDS, ConvShape<CFG, C0, C1, COUT>::ACC))))
k_conv3x3(const __bf16* __restrict__ src0, const __bf16* __restrict__ src1, const __bf16* __restrict__ wgt,
          const float* __restrict__ bias, const __bf16* __restrict__ mask, void* __restrict__ out, uint32_t N, uint32_t H,
          uint32_t W, ConvExtra ex) {
    using SH = ConvShape<CFG, C0, C1, COUT>;
    constexpr int CT = C0 + C1;
    constexpr int KPAD = (9 * CT + 31) / 32 * 32;
    constexpr int R = SH::R, NT = SH::NT, MT = SH::MT, CB = SH::CB, TR = SH::TR, TC = SH::TC;
    constexpr bool SPLIT = EPI == EPI_SPLIT;
    constexpr int G0 = (C0 + 31) / 32, NG = SPLIT ? G0 + (C1 + 31) / 32 : SH::NG;
    static_assert(C0 % 8 == 0 && C1 % 8 == 0 && (UP0 == 1 || UP0 == 2), "channel groups");
    // Halo tile: a thread stages one 8-channel chunk of one column in RPP rows
    // at a time; columns past the 64th (of a tile 64 wide) are one more pass.
    constexpr int ROWCH = TC * 4 > kConvThreads ? kConvThreads : TC * 4;
    constexpr int RPP = kConvThreads / ROWCH, PASSES = (TR + RPP - 1) / RPP;
    constexpr int EXTRA = TC * 4 - ROWCH;
    static_assert(EXTRA * TR <= kConvThreads, "one more pass");
    constexpr int SPT = PASSES + (EXTRA > 0 ? 1 : 0);
    // Weights: CB rows of four chunks per tap.
    constexpr int TAPCH = CB * 4, TPP = TAPCH > kConvThreads ? 1 : kConvThreads / TAPCH;
    constexpr int PPT = (TAPCH + kConvThreads - 1) / kConvThreads;
    constexpr int WPT = PPT * ((9 + TPP - 1) / TPP);
    // [row][col][4 chunks of 8 channels], the chunks of pixel (row, col) stored
    // in the order chunk ^ ((row + (col >> 1)) & 3), which spreads the fragment
    // reads of neighbouring pixels over the banks
    __shared__ bf16x8 tile[TR * TC * 4];
    // [tap][row] weights; row m * 16 + 4 g + i holds output channel 4 MT g + 4 m + i,
    // so that a lane's sums are 4 MT consecutive channels of its pixels; a row's
    // four chunks are in the order chunk ^ ((row >> 1) & 3)
    __shared__ bf16x8 wl[9 * CB * 4];
    const int tid = (int)threadIdx.x;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = tid & 15, g = (tid >> 4) & 3;
    const uint32_t segs = (W + SH::COLS - 1) / SH::COLS, rblocks = (H + SH::ROWS - 1) / SH::ROWS;
    const uint32_t tiles = N * rblocks * segs, step = gridDim.x;
    const int cb0 = (int)blockIdx.y * CB;
    const int wr = wv / SH::WC * R, wc = wv % SH::WC * NT * 16;   // the wave's part of the tile
    struct Place { uint32_t n; int y0, x0; };
    auto place = [&](uint32_t tl) {
        const uint32_t rest = __builtin_amdgcn_readfirstlane(tl / segs), n = __builtin_amdgcn_readfirstlane(rest / rblocks);
        return Place{n, (int)((rest - n * rblocks) * SH::ROWS), (int)((tl - rest * segs) * SH::COLS)};
    };

    const int prow = RPP == 1 ? 0 : tid / ROWCH, pcol = (tid - prow * ROWCH) >> 2, pchunk = tid & 3;
    static_assert(ROWCH % 4 == 0, "a thread's chunk is tid & 3");
    const int wtap = TPP == 1 ? 0 : tid / TAPCH, wrow0 = (tid - wtap * TAPCH) >> 2;
    bf16x8 stage[SPT], wstage[WPT];
    // Channel group cg of tile tl: every load of a thread is issued before any
    // is stored. Lanes with nothing to load ask for an offset past the end of
    // the buffer descriptor, which returns zeros.
    constexpr uint32_t kEnd = 0x7FFFFFFFu, kNone = 0x80000000u, kRaw = 0x00020000u;
    // `kc` is the group's first channel in `src` (negative if the other source has it).
    auto load_tile = [&](const Place& p, const __bf16* src, int C, int up, int kc) {
        const uint32_t HS = H >> up, WS = W >> up;
        const bool chunk_ok = kc + pchunk * 8 < C;
        const int sx = p.x0 - 1 + pcol;
        const bool col_ok = chunk_ok && (uint32_t)sx < W;
        if constexpr (RPP == 1) {
            // one row per pass: its address is the wave's
            const uint32_t off = col_ok && pcol * 4 < ROWCH ? (uint32_t)(((pcol + up) >> up) * C + pchunk * 8) * 2u : kNone;
#pragma unroll
            for (int i = 0; i < PASSES; i++) {
                const int sy = p.y0 - 1 + i;
                const __bf16* base = src + (((int64_t)p.n * HS + (sy >> up)) * WS + (p.x0 >> up) - 1) * C + kc;
                const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (uint32_t)sy < H ? kEnd : 0u, kRaw);
                stage[i] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
            }
        } else {
            // offsets within one image, which is small here
            const __bf16* base = src + (int64_t)p.n * HS * WS * C + kc;
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, kEnd, kRaw);
#pragma unroll
            for (int i = 0; i < PASSES; i++) {
                const int ty = i * RPP + prow, sy = p.y0 - 1 + ty;
                const bool ok = col_ok && prow < RPP && ty < TR && (uint32_t)sy < H;
                const uint32_t off = ok ? (uint32_t)(((sy >> up) * (int)WS + (sx >> up)) * C + pchunk * 8) * 2u : kNone;
                stage[i] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
            }
        }
        if constexpr (EXTRA > 0) {
            const int ty = tid / EXTRA, ex_x = p.x0 - 1 + ROWCH / 4 + ((tid % EXTRA) >> 2), sy = p.y0 - 1 + ty;
            bf16x8 v = zero8();
            if (ty < TR && chunk_ok && (uint32_t)sy < H && (uint32_t)ex_x < W)
                v = *(const bf16x8*)(src + (((size_t)p.n * HS + (uint32_t)(sy >> up)) * WS + (uint32_t)(ex_x >> up)) * C + (kc + pchunk * 8));
            stage[PASSES] = v;
        }
    };
    auto load_group = [&](uint32_t tl, int cg, bool weights) {
        if (weights) {
            const int c = SPLIT && cg >= G0 ? C0 + (cg - G0) * 32 : cg * 32, end = SPLIT && cg < G0 ? C0 : CT;
            const __bf16* base = wgt + (size_t)cb0 * KPAD + c;
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, kEnd, kRaw);
#pragma unroll
            for (int i = 0; i < WPT; i++) {
                const int row = wrow0 + (i % PPT) * (kConvThreads / 4), tap0 = i / PPT * TPP;
                const bool ok = c + pchunk * 8 < end && row < CB && wtap < TPP && tap0 + wtap < 9;
                const uint32_t off = ok ? (uint32_t)(row * KPAD + wtap * CT + pchunk * 8) * 2u : kNone;
                wstage[i] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rs, off, tap0 * CT * 2, 0));
            }
        }
        const Place p = place(tl);
        if constexpr (SPLIT) {
            load_tile(p, cg < G0 ? src0 : src1, cg < G0 ? C0 : C1, cg < G0 ? UP0 - 1 : 0, (cg < G0 ? cg : cg - G0) * 32);
        } else if constexpr (C1 != 0 && C0 % 32 != 0) {   // a group may have chunks of both sources
            if (cg * 32 + pchunk * 8 < C0) load_tile(p, src0, C0, UP0 - 1, cg * 32);
            else load_tile(p, src1, C1, 0, cg * 32 - C0);
        } else {
            const bool first = C1 == 0 || cg * 32 < C0;
            load_tile(p, first ? src0 : src1, first ? C0 : C1, first ? UP0 - 1 : 0, first ? cg * 32 : cg * 32 - C0);
        }
    };
    auto slot = [](int ty, int tx, int chunk) { return (ty * TC + tx) * 4 + (chunk ^ ((ty + (tx >> 1)) & 3)); };
    auto store_group = [&](bool weights) {
#pragma unroll
        for (int i = 0; i < PASSES; i++) {
            const int ty = i * RPP + prow;
            if (RPP == 1 ? pcol * 4 < ROWCH : prow < RPP && ty < TR) tile[slot(ty, pcol, pchunk)] = stage[i];
        }
        if constexpr (EXTRA > 0) {
            const int ty = tid / EXTRA;
            if (ty < TR) tile[slot(ty, ROWCH / 4 + ((tid % EXTRA) >> 2), pchunk)] = stage[PASSES];
        }
        if (weights) {
#pragma unroll
            for (int i = 0; i < WPT; i++) {
                const int co = wrow0 + (i % PPT) * (kConvThreads / 4), tap = i / PPT * TPP + wtap;
                const int row = (co % (4 * MT)) / 4 * 16 + co / (4 * MT) * 4 + (co & 3);
                if (co < CB && wtap < TPP && tap < 9)
                    wl[(tap * CB + row) * 4 + (pchunk ^ ((row >> 1) & 3))] = wstage[i];
            }
        }
    };
    // The next group's (or tile's) loads are in flight during a group's MFMAs
    // and a tile's stores; the weights of a single group stay in LDS.
    bool weights = true;
    uint32_t tl = blockIdx.x;
    if (tl < tiles) load_group(tl, 0, true);
    for (; tl < tiles; tl += step) {
        f32x4 acc[R][MT][NT];
#pragma unroll
        for (int o = 0; o < R; o++)
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int t = 0; t < NT; t++) acc[o][m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int cg = 0; cg < NG; cg++) {
            __syncthreads();  // every wave is done reading the previous group
            store_group(weights);
            __syncthreads();
            weights = NG > 1;
            if (cg + 1 < NG) load_group(tl, cg + 1, true);
            else if (tl + step < tiles) load_group(tl + step, 0, weights);
            if constexpr (SPLIT) {
#pragma unroll
                for (int dx = 0; dx < 3; dx++) {
                    bf16x8 a[3][MT];
#pragma unroll
                    for (int dy = 0; dy < 3; dy++)
#pragma unroll
                        for (int m = 0; m < MT; m++)
                            a[dy][m] = wl[((dy * 3 + dx) * CB + m * 16 + r) * 4 + (g ^ ((r >> 1) & 3))];
                    const int col = wc + r + dx;             // tile column (of pixel t = 0)
#pragma unroll
                    for (int ir = 0; ir < R + 2; ir++) {
                        const bf16x8* row = tile + ((wr + ir) * TC + col) * 4 + (g ^ ((wr + ir + (col >> 1)) & 3));
#pragma unroll
                        for (int t = 0; t < NT; t++) {
                            const bf16x8 b = row[t * 64];
#pragma unroll
                            for (int dy = 0; dy < 3; dy++) {
                                const int o = ir - dy;
                                if (o < 0 || o >= R) continue;
#pragma unroll
                                for (int m = 0; m < MT; m++)
                                    acc[o][m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[dy][m], b, acc[o][m][t], 0, 0, 0);
                            }
                        }
                    }
                }
            } else {
#pragma unroll
                for (int dy = 0; dy < 3; dy++) {
                    // 32 channels leave 168 registers to three waves: loads of a
                    // later row moved up here would spill where these epilogues
                    // or two sources add to them
                    if constexpr (CB == 32 && (EPI == EPI_POOL || EPI == EPI_HEAD || C1 != 0))
                        if (dy > 0) __builtin_amdgcn_sched_barrier(0);
                    bf16x8 a[3][MT];
#pragma unroll
                    for (int dx = 0; dx < 3; dx++)
#pragma unroll
                        for (int m = 0; m < MT; m++)
                            a[dx][m] = wl[((dy * 3 + dx) * CB + m * 16 + r) * 4 + (g ^ ((r >> 1) & 3))];
#pragma unroll
                    for (int o = 0; o < R; o++)
#pragma unroll
                        for (int dx = 0; dx < 3; dx++) {
                            const int col = wc + r + dx;     // tile column (of pixel t = 0)
                            const bf16x8* row = tile + ((wr + o + dy) * TC + col) * 4 + (g ^ ((wr + o + dy + (col >> 1)) & 3));
#pragma unroll
                            for (int t = 0; t < NT; t++) {
                                const bf16x8 b = row[t * 64];
#pragma unroll
                                for (int m = 0; m < MT; m++)
                                    acc[o][m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[dx][m], b, acc[o][m][t], 0, 0, 0);
                            }
                        }
                }
            }
        }

        const Place p = place(tl);
        constexpr int LC = 4 * MT;                        // channels of this lane: c0 .. c0 + LC - 1
        const int c0 = cb0 + LC * g;
        // pixel (o, t) of this lane: row y(o), column x(t), at `px` channels of the row's `wide`
        auto y = [&](int o) { return (uint32_t)(p.y0 + wr + o); };
        auto x = [&](int t) { return (uint32_t)(p.x0 + wc + t * 16 + r); };
        auto first_pixel = [&](int o, int t) { return ((size_t)p.n * H + y(o)) * W + (uint32_t)(p.x0 + wc + t * 16); };
        const uint32_t mine = (uint32_t)(r * COUT + c0);
        if constexpr (EPI == EPI_F32 || EPI == EPI_MASK) {
#pragma unroll
            for (int o = 0; o < R; o++)
#pragma unroll
                for (int t = 0; t < NT; t++) {
                    if (y(o) >= H || x(t) >= W) continue;
                    const size_t at = first_pixel(o, t) * COUT;
#pragma unroll
                    for (int m = 0; m < MT; m++) {
                        const f32x4 v = acc[o][m][t];
                        if constexpr (EPI == EPI_F32) {
                            *(f32x4*)((float*)out + at + (mine + 4 * m)) = v;
                        } else {
                            const bf16x4 mk = *(const bf16x4*)(mask + at + (mine + 4 * m));
                            bf16x4 q;
#pragma unroll
                            for (int i = 0; i < 4; i++) q[i] = (__bf16)((float)mk[i] > 0.0f ? v[i] : 0.0f);
                            *(bf16x4*)((__bf16*)out + at + (mine + 4 * m)) = q;
                        }
                    }
                }
        } else {
            f32x4 bv[MT];
#pragma unroll
            for (int m = 0; m < MT; m++) bv[m] = *(const f32x4*)(bias + c0 + 4 * m);
            __bf16 q[R][NT][LC];
#pragma unroll
            for (int o = 0; o < R; o++)
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int j = 0; j < LC; j++) q[o][t][j] = (__bf16)fmaxf(acc[o][j / 4][t][j & 3] + bv[j / 4][j & 3], 0.0f);
            if constexpr (EPI != EPI_HEAD) {
#pragma unroll
                for (int o = 0; o < R; o++)
#pragma unroll
                    for (int t = 0; t < NT; t++) {
                        if (y(o) >= H || x(t) >= W) continue;
                        store_channels<LC>((__bf16*)out + first_pixel(o, t) * COUT + mine, q[o][t]);
                    }
            }
            if constexpr (EPI == EPI_POOL) {
                // 2 x 2 averages of the stored values; the right pixel is the
                // next lane's (x0, wc and 16 t are even, as are H and W)
                static_assert(R % 2 == 0, "a wave holds whole row pairs");
#pragma unroll
                for (int o = 0; o < R; o += 2)
#pragma unroll
                    for (int t = 0; t < NT; t++) {
                        __bf16 a[LC];
#pragma unroll
                        for (int j = 0; j < LC; j += 2) {
                            const bf16x2 u = {q[o][t][j], q[o][t][j + 1]}, l = {q[o + 1][t][j], q[o + 1][t][j + 1]};
                            const bf16x2 u1 = lane_pair(u), l1 = lane_pair(l);
#pragma unroll
                            for (int i = 0; i < 2; i++)
                                a[j + i] = (__bf16)(((((float)u[i] + (float)u1[i]) + (float)l[i]) + (float)l1[i]) * 0.25f);
                        }
                        if (y(o) >= H || x(t) >= W || (r & 1) != 0) continue;
                        const size_t at = ((size_t)p.n * (H / 2) + y(o) / 2) * (W / 2) + (uint32_t)(p.x0 + wc + t * 16) / 2;
                        store_channels<LC>(ex.pool + at * COUT + (uint32_t)(r / 2 * COUT + c0), a);
                    }
            }
            if constexpr (EPI == EPI_HEAD) {
                // out = W_head a + b + residual: partial sums over the lane's
                // channels, added over the four lanes of a pixel such that
                // each of them has the sums of a quarter of the wave's pixels
                constexpr int P = R * NT;
                static_assert(CB == COUT && (P == 1 || P == 4), "every channel of a pixel in one wave");
                float v[3];
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    float s[P];
#pragma unroll
                    for (int q0 = 0; q0 < P; q0++) s[q0] = 0.0f;
#pragma unroll
                    for (int j = 0; j < LC; j += 4) {
                        const bf16x4 wk = *(const bf16x4*)(ex.wh + k * COUT + c0 + j);
#pragma unroll
                        for (int i = 0; i < 4; i++)
#pragma unroll
                            for (int q0 = 0; q0 < P; q0++) s[q0] = fmaf((float)wk[i], (float)q[q0 / NT][q0 % NT][j + i], s[q0]);
                    }
                    if constexpr (P == 4) v[k] = add_rows(add_halves(s[0], s[1]), add_halves(s[2], s[3]));
                    else v[k] = add_rows(add_halves(s[0], s[0]), add_halves(s[0], s[0]));
                }
                // add_halves leaves its first argument's sums in lanes 0-31, its
                // second's in 32-63; add_rows its first's in even rows of 16
                const int q0 = P == 4 ? (g >> 1) + 2 * (g & 1) : 0, o = q0 / NT, t = q0 % NT;
                const uint32_t yy = y(o), xx = x(t);
                if ((P > 1 || g == 0) && yy < H && xx < W) {
                    const size_t pix = ((size_t)p.n * H + yy) * W + xx;
                    const float4 rs = ex.resid[pix];
                    const float4 res = make_float4(v[0] + ex.bh[0] + rs.x, v[1] + ex.bh[1] + rs.y, v[2] + ex.bh[2] + rs.z, 0.0f);
                    if (ex.out) ex.out[pix] = res;
                    if (ex.surface && p.n == 0 && xx < ex.w && yy < ex.h)
                        ex.surface[(size_t)yy * ex.w + xx] = make_float4(fmaxf(expm1f(res.x), 0.0f), fmaxf(expm1f(res.y), 0.0f),
                                                                         fmaxf(expm1f(res.z), 0.0f), 1.0f);
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Weight and bias gradients: dW[co][tap][c] = sum over pixels p of dY[p][co] *
// X[p + offset(tap)][c] and db[co] = sum over p of dY[p][co], on MFMA with the
// pixels as K (32 pixels of one row per instruction).
//
// A workgroup walks 32-pixel-wide strips of `rows` rows. Wave w owns the 16
// input channels [16 w, 16 w + 16) and all 9 taps of MTW x 16 output channels,
// so each row's dY and X are read from HBM once per workgroup. Both operands
// need 8 pixels of one channel per lane while memory holds the channels of a
// pixel together: a thread loads 8 channels of two neighbouring pixels and
// stores 8 dwords (pixel pair, one per channel) into a channel-major LDS row
// of 20 dwords (the stride puts the 16 channels x 16 bytes a wave reads at
// once on distinct banks). The three horizontal taps of a row are one 20-byte
// read: taps -1 and +1 are its dwords 0..3 and 1..4, tap 0 their 16-bit
// funnel shift. X rows y - 1, y, y + 1 stay in a ring of four row slots, so a
// row is staged once; the next rows' global loads are in flight during the
// MFMAs and one barrier per row publishes them.
//
// Every workgroup writes its sums to its own slice of the workspace
// (k_reduce_grads adds the slices): same-address atomics run at about 90 M
// per second on this chip. What bounds it is the latency of one row (barrier,
// LDS, 9 MTW dependent-free MFMAs) at 1 to 2 workgroups per CU.
// Measured on 8 images of 128 x 128, all 14 layers: 960 us for one wave per 16 x 16
// tile gathering single elements and adding with atomics, plus 335 us of bias
// column sums; this form takes 235 us and k_reduce_grads 45 us (3.3 -> 1.19 ms
// for the whole training step, with the head's backward pass below).
constexpr int kGradStride = 20;           // dwords per channel of a staged row
constexpr int kGradTileW = 32;            // pixels per strip (K of one MFMA)
template <int C0, int UP0, int C1, int COUT, int CW, int MTW>
__global__ void __launch_bounds__(64 * CW) k_conv_wgrad(const __bf16* __restrict__ dy, const __bf16* __restrict__ src0,
                                                        const __bf16* __restrict__ src1, float* __restrict__ part,
                                                        uint32_t cin_real, uint32_t H, uint32_t W, uint32_t rows,
                                                        uint32_t rblocks, uint32_t segs, uint32_t strips) {
    constexpr int CT = C0 + C1;
    static_assert(CT % (16 * CW) == 0 && COUT % (16 * MTW) == 0, "channel tiles");
    constexpr int NTHR = 64 * CW;
    constexpr int XI = 17 * 2 * CW, YI = 16 * 2 * MTW;         // staged items (pixel pair x 8 channels) per row
    constexpr int PER = (XI + YI + NTHR - 1) / NTHR;
    __shared__ __align__(16) uint32_t xs[4][16 * CW][kGradStride];
    __shared__ __align__(16) uint32_t ys[2][16 * MTW][kGradStride];
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    const uint32_t r = lane & 15u, g = lane >> 4;
    int x0 = 0, y0 = 0, y1 = 0;               // the strip: columns x0.., rows [y0, y1) of image n
    uint32_t n = 0;
    const int cb = (int)blockIdx.y * 16 * CW, mb = (int)blockIdx.z * 16 * MTW;
    const uint32_t H0 = H / UP0, W0 = W / UP0;

    bf16x8 st0[PER], st1[PER];
    // Items of X row yx (channels cb..) and dY row yy (channels mb..), zero
    // outside the image.
    auto load_rows = [&](int yx, int yy) {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            int e = (int)threadIdx.x + i * NTHR;
            bf16x8 v[2] = {zero8(), zero8()};
            if (e < XI) {
                const int pair = e % 17, c = cb + (e / 17) * 8;
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    const int sx = x0 - 1 + 2 * pair + k;
                    if (yx >= 0 && yx < (int)H && sx >= 0 && sx < (int)W) {
                        const __bf16* p;
                        if (C1 == 0 || c < C0)
                            p = src0 + (((size_t)n * H0 + (uint32_t)yx / UP0) * W0 + (uint32_t)sx / UP0) * C0 + c;
                        else
                            p = src1 + (((size_t)n * H + (uint32_t)yx) * W + (uint32_t)sx) * C1 + (c - C0);
                        v[k] = *(const bf16x8*)p;
                    }
                }
            } else if (e < XI + YI) {
                e -= XI;
                const int pair = e % 16, c = mb + (e / 16) * 8;
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    const int sx = x0 + 2 * pair + k;
                    if (yy < y1 && sx < (int)W)
                        v[k] = *(const bf16x8*)(dy + (((size_t)n * H + (uint32_t)yy) * W + (uint32_t)sx) * COUT + c);
                }
            }
            st0[i] = v[0];
            st1[i] = v[1];
        }
    };
    auto store_rows = [&](int yx, int yy) {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            int e = (int)threadIdx.x + i * NTHR;
            uint32_t* d = nullptr;
            if (e < XI) d = &xs[(yx + 4) & 3][(e / 17) * 8][e % 17];
            else if (e < XI + YI) d = &ys[yy & 1][((e - XI) / 16) * 8][(e - XI) % 16];
            if (d) {
                const u16x8 a = __builtin_bit_cast(u16x8, st0[i]), b = __builtin_bit_cast(u16x8, st1[i]);
#pragma unroll
                for (int k = 0; k < 8; k++) d[k * kGradStride] = (uint32_t)a[k] | ((uint32_t)b[k] << 16);
            }
        }
    };

    f32x4 acc[MTW][9], accb[MTW];
#pragma unroll
    for (int m = 0; m < MTW; m++) {
        accb[m] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 9; t++) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    bf16x8 ones;
#pragma unroll
    for (int k = 0; k < 8; k++) ones[k] = (__bf16)1.0f;
    const bool bias = blockIdx.y == 0 && wv == 0;

    for (uint32_t strip = blockIdx.x; strip < strips; strip += gridDim.x) {
        const uint32_t rest = strip / segs;
        n = rest / rblocks;
        x0 = (int)((strip % segs) * kGradTileW);
        y0 = (int)((rest % rblocks) * rows);
        y1 = min((int)H, y0 + (int)rows);
        // rows y0 - 1, y0, y0 + 1 of X and y0 of dY (y1, past the strip, stores zeros)
        load_rows(y0 - 1, y1);
        store_rows(y0 - 1, y0 + 1);
        load_rows(y0, y1);
        store_rows(y0, y0 + 1);
        load_rows(y0 + 1, y0);
        store_rows(y0 + 1, y0);
        __syncthreads();
        for (int y = y0; y < y1; y++) {
            if (y + 1 < y1) load_rows(y + 2, y + 1);
            bf16x8 a[MTW];
#pragma unroll
            for (int m = 0; m < MTW; m++) a[m] = *(const bf16x8*)&ys[y & 1][m * 16 + r][4 * g];
#pragma unroll
            for (int ky = 0; ky < 3; ky++) {
                const uint32_t* p = &xs[(y + ky + 3) & 3][wv * 16 + r][4 * g];
                const u32x4 q = *(const u32x4*)p;
                const uint32_t q4 = p[4];
                const u32x4 mid = {__builtin_amdgcn_alignbit(q.y, q.x, 16), __builtin_amdgcn_alignbit(q.z, q.y, 16),
                                   __builtin_amdgcn_alignbit(q.w, q.z, 16), __builtin_amdgcn_alignbit(q4, q.w, 16)};
                const u32x4 right = {q.y, q.z, q.w, q4};
                const bf16x8 b[3] = {__builtin_bit_cast(bf16x8, q), __builtin_bit_cast(bf16x8, mid),
                                     __builtin_bit_cast(bf16x8, right)};
#pragma unroll
                for (int kx = 0; kx < 3; kx++)
#pragma unroll
                    for (int m = 0; m < MTW; m++)
                        acc[m][ky * 3 + kx] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], b[kx], acc[m][ky * 3 + kx], 0, 0, 0);
            }
            if (bias) {
#pragma unroll
                for (int m = 0; m < MTW; m++) accb[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], ones, accb[m], 0, 0, 0);
            }
            if (y + 1 < y1) store_rows(y + 2, y + 1);
            __syncthreads();
        }
    }
    // D: lane holds input channel r of its tile, output channels 4 g + i
    float* out = part + (size_t)blockIdx.x * (COUT * 9 * cin_real + COUT);
    const uint32_t c = (uint32_t)cb + wv * 16 + r;
#pragma unroll
    for (int m = 0; m < MTW; m++) {
        const uint32_t co = (uint32_t)(mb + m * 16) + 4 * g;
        if (c < cin_real) {
#pragma unroll
            for (int t = 0; t < 9; t++)
#pragma unroll
                for (int i = 0; i < 4; i++) out[((size_t)(co + i) * 9 + t) * cin_real + c] = acc[m][t][i];
        }
        if (bias && r == 0) {
#pragma unroll
            for (int i = 0; i < 4; i++) out[(size_t)COUT * 9 * cin_real + co + i] = accb[m][i];
        }
    }
}

// Adds the workgroups' partial gradients: element i of slice l is the sum of
// its nblk partials, each `size` elements apart.
struct GradSlices {
    static constexpr int kMax = kDnLayers + 2;   // convolutions, head, loss
    struct S {
        float* dst;
        const float* part;
        uint32_t size, nblk, first;              // first: its first block of the launch
    } s[kMax];
};
__global__ void __launch_bounds__(256) k_reduce_grads(GradSlices t) {
    int l = 0;
#pragma unroll
    for (int k = 1; k < GradSlices::kMax; k++) l = blockIdx.x >= t.s[k].first ? k : l;
    const uint32_t i = (blockIdx.x - t.s[l].first) * 256u + threadIdx.x, size = t.s[l].size, nblk = t.s[l].nblk;
    if (i >= size) return;
    const float* p = t.s[l].part + i;
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    uint32_t b = 0;
    for (; b + 4 <= nblk; b += 4)
#pragma unroll
        for (int k = 0; k < 4; k++) s[k] += p[(size_t)(b + k) * size];
    for (; b < nblk; b++) s[0] += p[(size_t)b * size];
    t.s[l].dst[i] = (s[0] + s[1]) + (s[2] + s[3]);
}

// ---------------------------------------------------------------------------
// Pooling and the gradients of upsampling / pooling
// ---------------------------------------------------------------------------
// Gradient of "upsample then concatenate" for the upsampled part: the sum of
// the four children (channels [0, C0) of the FP32 input gradient, CT wide),
// times the ReLU mask of the low-resolution activation -> BF16.
__global__ void k_upback_mask(const float* __restrict__ gx, uint32_t CT, const __bf16* __restrict__ act,
                              __bf16* __restrict__ gout, uint32_t N, uint32_t Hl, uint32_t Wl, uint32_t C0) {
    const uint32_t G = C0 / 8;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)N * Hl * Wl * G) return;
    const uint32_t gi = (uint32_t)(i % G);
    size_t q = i / G;
    const uint32_t xl = (uint32_t)(q % Wl);
    q /= Wl;
    const uint32_t yl = (uint32_t)(q % Hl), n = (uint32_t)(q / Hl);
    const uint32_t H = 2 * Hl, W = 2 * Wl;
    float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int d = 0; d < 4; d++) {
        const size_t pix = ((size_t)n * H + 2 * yl + (d >> 1)) * W + 2 * xl + (d & 1);
        const float* p = gx + pix * CT + gi * 8;
#pragma unroll
        for (int e = 0; e < 8; e++) s[e] += p[e];
    }
    const size_t lp = ((size_t)n * Hl + yl) * Wl + xl;
    const bf16x8 a = *(const bf16x8*)(act + lp * C0 + gi * 8);
    bf16x8 o;
#pragma unroll
    for (int e = 0; e < 8; e++) o[e] = (__bf16)((float)a[e] > 0.0f ? s[e] : 0.0f);
    *(bf16x8*)(gout + lp * C0 + gi * 8) = o;
}

// Gradient reaching an encoder output that is both pooled and skipped:
// (pooled-path gradient / 4 + skip gradient) times its ReLU mask -> BF16.
// gpool: FP32, half resolution, C channels; gskip: FP32, channels
// [coff, coff + C) of a CT-wide tensor at full resolution.
__global__ void k_poolback_skip_mask(const float* __restrict__ gpool, const float* __restrict__ gskip, uint32_t CT,
                                     uint32_t coff, const __bf16* __restrict__ act, __bf16* __restrict__ gout, uint32_t N,
                                     uint32_t H, uint32_t W, uint32_t C) {
    const uint32_t G = C / 8;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)N * H * W * G) return;
    const uint32_t gi = (uint32_t)(i % G);
    const size_t pix = i / G;
    const uint32_t x = (uint32_t)(pix % W);
    const size_t q = pix / W;
    const uint32_t y = (uint32_t)(q % H), n = (uint32_t)(q / H);
    const size_t pp = ((size_t)n * (H / 2) + y / 2) * (W / 2) + x / 2;
    const float* gp = gpool + pp * C + gi * 8;
    const float* gs = gskip + pix * CT + coff + gi * 8;
    const bf16x8 a = *(const bf16x8*)(act + pix * C + gi * 8);
    bf16x8 o;
#pragma unroll
    for (int e = 0; e < 8; e++) o[e] = (__bf16)((float)a[e] > 0.0f ? gp[e] * 0.25f + gs[e] : 0.0f);
    *(bf16x8*)(gout + pix * C + gi * 8) = o;
}

// ---------------------------------------------------------------------------
// Input packing, head, loss
// ---------------------------------------------------------------------------
__device__ inline void octahedral(float x, float y, float z, float& ox, float& oy) {
    const float l1 = fabsf(x) + fabsf(y) + fabsf(z);
    if (!(l1 > 1e-12f)) {
        ox = oy = 0.0f;
        return;
    }
    x /= l1;
    y /= l1;
    z /= l1;
    if (z < 0.0f) {
        ox = (1.0f - fabsf(y)) * (x >= 0.0f ? 1.0f : -1.0f);
        oy = (1.0f - fabsf(x)) * (y >= 0.0f ? 1.0f : -1.0f);
    } else {
        ox = x;
        oy = y;
    }
}

// Raw features -> network input (BF16, 16 channels, 10 used) and the FP32
// log radiance for the head's residual. Source: either raw records
// (12 floats per pixel: radiance, albedo, depth code, normal, M2, samples)
// or a surface (radiance plane + two feature planes, `held` samples).
// Pixels of the padded network image outside (h, w) are zero. A wave takes 64
// pixels of a row (the row is the wave's, so no lane divides).
__global__ void k_pack(const float* __restrict__ raw, const float4* __restrict__ rad, const float4* __restrict__ aux,
                       uint32_t held, uint32_t N, uint32_t h, uint32_t w, uint32_t Hp, uint32_t Wp,
                       __bf16* __restrict__ xin, float4* __restrict__ resid) {
    const uint32_t segs = (Wp + 63) / 64, rb = blockIdx.x / segs;
    const uint32_t row = __builtin_amdgcn_readfirstlane(rb * 4 + threadIdx.x / 64), n = row / Hp, y = row - n * Hp;
    const uint32_t x = (blockIdx.x - rb * segs) * 64 + threadIdx.x % 64;
    if (n >= N || x >= Wp) return;
    const size_t i = (size_t)row * Wp + x;
    float f[12] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    const bool valid = x < w && y < h;
    if (valid) {
        const size_t src = ((size_t)n * h + y) * w + x;
        if (raw) {
#pragma unroll
            for (int k = 0; k < 12; k++) f[k] = raw[src * 12 + k];
        } else {
            const float4 c = rad[src], a0 = aux[src], a1 = aux[(size_t)w * h + src];
            f[0] = c.x; f[1] = c.y; f[2] = c.z;
            f[3] = a0.x; f[4] = a0.y; f[5] = a0.z; f[6] = a0.w;
            f[7] = a1.x; f[8] = a1.y; f[9] = a1.z; f[10] = a1.w;
            f[11] = (float)held;
        }
    }
    float v[16];
#pragma unroll
    for (int k = 0; k < 16; k++) v[k] = 0.0f;
    if (valid) {
        v[0] = log1pf(fmaxf(f[0], 0.0f));
        v[1] = log1pf(fmaxf(f[1], 0.0f));
        v[2] = log1pf(fmaxf(f[2], 0.0f));
        v[3] = f[3];
        v[4] = f[4];
        v[5] = f[5];
        float nx = f[7], ny = f[8], nz = f[9];
        const float ln = sqrtf(nx * nx + ny * ny + nz * nz);
        if (ln > 1e-12f) {
            nx /= ln;
            ny /= ln;
            nz /= ln;
        } else {
            nx = ny = nz = 0.0f;
        }
        octahedral(nx, ny, nz, v[6], v[7]);
        v[8] = f[6];
        const float nh = f[11];
        v[9] = nh >= 2.0f ? sqrtf(fmaxf(f[10], 0.0f) / fmaxf(nh * (nh - 1.0f), 1.0f)) : 0.0f;
    }
    bf16x8 lo, hi;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        lo[k] = (__bf16)v[k];
        hi[k] = (__bf16)v[8 + k];
    }
    *(bf16x8*)(xin + i * 16) = lo;
    *(bf16x8*)(xin + i * 16 + 8) = hi;
    resid[i] = make_float4(v[0], v[1], v[2], 0.0f);
}

// 1x1 head: out = W_head (3 x 32) . act + b + residual (FP32). Optionally also
// writes the denoised radiance max(expm1(out), 0) into an RGBA32F surface.
__global__ void k_head(const __bf16* __restrict__ act, const __bf16* __restrict__ wh, const float* __restrict__ bh,
                       const float4* __restrict__ resid, float4* __restrict__ out, uint32_t N, uint32_t Hp, uint32_t Wp) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)N * Hp * Wp) return;
    float o[3];
#pragma unroll
    for (int k = 0; k < 3; k++) o[k] = 0.0f;
#pragma unroll
    for (int gi = 0; gi < 4; gi++) {
        const bf16x8 a = *(const bf16x8*)(act + i * 32 + gi * 8);
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const bf16x8 wv = *(const bf16x8*)(wh + k * 32 + gi * 8);
#pragma unroll
            for (int e = 0; e < 8; e++) o[k] += (float)wv[e] * (float)a[e];
        }
    }
    const float4 rs = resid[i];
    out[i] = make_float4(o[0] + bh[0] + rs.x, o[1] + bh[1] + rs.y, o[2] + bh[2] + rs.z, 0.0f);
}

// Loss over the valid pixels (0 gradient on padding); the sum goes to *loss.
//   kind 0: MSE in log1p space, dout = 2 (out - log1p(t)) / count
//   kind 1: relMSE of y = expm1(out) against t, (y - t)^2 / (t^2 + 0.01),
//           dout = 2 (y - t) (y + 1) / ((t^2 + 0.01) count)
__device__ inline float loss_term(float o, float t, uint32_t kind, float inv, float& g) {
    t = fmaxf(t, 0.0f);
    if (kind == 0u) {
        const float d = o - log1pf(t);
        g = d * inv;
        return d * d;
    }
    const float y = expm1f(o), e = y - t, wgt = 1.0f / (t * t + 0.01f);
    g = e * wgt * (y + 1.0f) * inv;
    return e * e * wgt;
}

// Loss, its gradient and the head's backward pass in one walk over the pixels:
// g_act = (W_head^T dout) * mask(act) -> BF16, and per workgroup the partial
// sums of dW_head (3 x 32), db_head (3) and the loss, by wave reductions and
// LDS, into the workgroup's slice of the workspace (head partials `part`, 99
// per workgroup; loss partials `lpart`, one). HBM bound; the sums cost 100
// wave reductions per workgroup, so a launch holds at most kHeadBlocks.
// One atomic per wave and parameter instead took 1,010 us on 131,072 pixels
// (200 K atomics on seven lines) and 29 us for the loss; this form takes 29 us.
constexpr uint32_t kHeadBlocks = 256;
__global__ void __launch_bounds__(256) k_loss_head_backward(const float4* __restrict__ out, const float* __restrict__ target,
                                                            const __bf16* __restrict__ act, const __bf16* __restrict__ wh,
                                                            __bf16* __restrict__ gact, float* __restrict__ part,
                                                            float* __restrict__ lpart, uint32_t N, uint32_t h, uint32_t w,
                                                            uint32_t Hp, uint32_t Wp, uint32_t kind) {
    float sw[3][32];
    float sb[3] = {0.f, 0.f, 0.f}, sl = 0.f;
#pragma unroll
    for (int k = 0; k < 3; k++)
#pragma unroll
        for (int c = 0; c < 32; c++) sw[k][c] = 0.0f;
    const size_t P = (size_t)N * Hp * Wp;
    const float inv = 2.0f / (3.0f * (float)N * (float)h * (float)w);
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < P; i += (size_t)gridDim.x * blockDim.x) {
        const uint32_t x = (uint32_t)(i % Wp);
        const size_t q = i / Wp;
        const uint32_t y = (uint32_t)(q % Hp), n = (uint32_t)(q / Hp);
        float dv[3] = {0.f, 0.f, 0.f};
        if (x < w && y < h) {
            const size_t src = ((size_t)n * h + y) * w + x;
            const float4 o = out[i];
            sl += loss_term(o.x, target[src * 3 + 0], kind, inv, dv[0]) + loss_term(o.y, target[src * 3 + 1], kind, inv, dv[1]) +
                  loss_term(o.z, target[src * 3 + 2], kind, inv, dv[2]);
        }
#pragma unroll
        for (int gi = 0; gi < 4; gi++) {
            const bf16x8 a = *(const bf16x8*)(act + i * 32 + gi * 8);
            bf16x8 o;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int c = gi * 8 + e;
                float s = 0.0f;
#pragma unroll
                for (int k = 0; k < 3; k++) {
                    s += (float)wh[k * 32 + c] * dv[k];
                    sw[k][c] += dv[k] * (float)a[e];
                }
                o[e] = (__bf16)((float)a[e] > 0.0f ? s : 0.0f);
            }
            *(bf16x8*)(gact + i * 32 + gi * 8) = o;
        }
#pragma unroll
        for (int k = 0; k < 3; k++) sb[k] += dv[k];
    }
    __shared__ float red[4][100];
    const uint32_t wv = threadIdx.x >> 6;
    auto wave_sum = [&](float v, int at) {
        for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
        if ((threadIdx.x & 63u) == 0) red[wv][at] = v;
    };
#pragma unroll
    for (int k = 0; k < 3; k++) {
#pragma unroll
        for (int c = 0; c < 32; c++) wave_sum(sw[k][c], k * 32 + c);
        wave_sum(sb[k], 96 + k);
    }
    wave_sum(sl, 99);
    __syncthreads();
    if (threadIdx.x < 100) {
        const float v = (red[0][threadIdx.x] + red[1][threadIdx.x]) + (red[2][threadIdx.x] + red[3][threadIdx.x]);
        if (threadIdx.x < 99) part[blockIdx.x * 99u + threadIdx.x] = v;
        else lpart[blockIdx.x] = v;
    }
}

// ---------------------------------------------------------------------------
// Parameters: Adam on the FP32 master vector, then BF16 copies in the
// forward layout [Cout][Kpad] (k = tap * CT + c) and the input-gradient
// layout [CT][Kpad'] (k' = tap' * Cout + co, holding W[co][8 - tap'][c]).
// ---------------------------------------------------------------------------
__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m1, float* __restrict__ m2,
                       size_t n, float lr, float b1, float b2, float eps, float c1, float c2) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float a = b1 * m1[i] + (1.0f - b1) * gi;
    const float b = b2 * m2[i] + (1.0f - b2) * gi * gi;
    m1[i] = a;
    m2[i] = b;
    p[i] -= lr * (a / c1) / (sqrtf(b / c2) + eps);
}

// Every layer in one launch (14 launches of 2.6 us each before).
struct LayoutTable {
    struct L {
        const float* w;
        __bf16 *fwd, *bwd;
        uint32_t cout, cin, ct, kpad_f, kpad_b, first;   // first: its first block of the launch
    } l[kDnLayers];
    const float* head;
    __bf16* head_out;
};
__global__ void __launch_bounds__(256) k_relayout(LayoutTable t) {
    int li = 0;
#pragma unroll
    for (int k = 1; k < kDnLayers; k++) li = blockIdx.x >= t.l[k].first ? k : li;
    const LayoutTable::L& L = t.l[li];
    if (blockIdx.x == 0 && threadIdx.x < 96) t.head_out[threadIdx.x] = (__bf16)t.head[threadIdx.x];
    const uint32_t cout = L.cout, cin = L.cin, ct = L.ct, kpad_f = L.kpad_f, kpad_b = L.kpad_b;
    const uint32_t i = (blockIdx.x - L.first) * 256u + threadIdx.x;
    const uint32_t nf = cout * kpad_f;
    if (i < nf) {
        const uint32_t co = i / kpad_f, k = i % kpad_f;
        const uint32_t tap = k / ct, c = k % ct;
        const float v = (k < 9 * ct && c < cin) ? L.w[((size_t)co * 9 + tap) * cin + c] : 0.0f;
        L.fwd[i] = (__bf16)v;
        return;
    }
    const uint32_t j = i - nf;
    if (j >= ct * kpad_b) return;
    const uint32_t c = j / kpad_b, k = j % kpad_b;
    const uint32_t tapb = k / cout, co = k % cout;
    const float v = (k < 9 * cout && c < cin) ? L.w[((size_t)co * 9 + (8 - tapb)) * cin + c] : 0.0f;
    L.bwd[j] = (__bf16)v;
}

__global__ void k_zero_f32(float* __restrict__ p, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0f;
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
static inline uint32_t cdiv(size_t a, uint32_t b) { return (uint32_t)((a + b - 1) / b); }

// Large tiles from one workgroup per CU on. The whole network at 417 x 233 and
// 1280 x 720, training step of eight 128 x 128: from 128 workgroups 94, 333 us
// and 1005; from 256 97, 339 and 990; from 512 101, 337 and 990; from 1024 102,
// 361 and 1006 (800 x 600: 222, 215, 214 and 226).
constexpr uint32_t kConvFill = 256;
template <typename SHAPE>
static uint32_t conv_tiles(uint32_t N, uint32_t H, uint32_t W) {
    return N * cdiv(H, SHAPE::ROWS) * cdiv(W, SHAPE::COLS);
}
template <int C0, int UP0, int C1, int COUT, int EPI>
static void conv(hipStream_t st, const __bf16* s0, const __bf16* s1, const __bf16* w, const float* b, const __bf16* mask,
                 void* out, uint32_t N, uint32_t H, uint32_t W, const ConvExtra& ex = ConvExtra{}) {
    using LG = ConvLarge;
    using SM = std::conditional_t<EPI == EPI_POOL, ConvSmallPool, ConvSmall>;
    using LS = ConvShape<LG, C0, C1, COUT>;
    using SS = ConvShape<SM, C0, C1, COUT>;
    constexpr uint32_t ls = COUT / LS::CB, ss = COUT / SS::CB;
    const uint32_t large = conv_tiles<LS>(N, H, W), small = conv_tiles<SS>(N, H, W);
    if (large * ls >= kConvFill) {
        constexpr uint32_t resident = 256 * conv_waves(LS::LDS, LS::ACC);
        k_conv3x3<C0, UP0, C1, COUT, EPI, LG><<<dim3(std::min(large, resident / ls), ls), kConvThreads, 0, st>>>(
            s0, s1, w, b, mask, out, N, H, W, ex);
    } else {
        k_conv3x3<C0, UP0, C1, COUT, EPI, SM><<<dim3(small, ss), kConvThreads, 0, st>>>(s0, s1, w, b, mask, out, N, H, W, ex);
    }
}

// Layer table (matches oracle/unet.py LAYERS): c0, up0, c1, cout, level.
struct LayerDesc {
    int c0, up0, c1, cout, level, cin_real;
};
static const LayerDesc kLayers[kDnLayers] = {
    {16, 1, 0, 32, 0, 10},  {32, 1, 0, 32, 0, 32},  {32, 1, 0, 48, 1, 32},  {48, 1, 0, 48, 1, 48},  {48, 1, 0, 64, 2, 48},
    {64, 1, 0, 64, 2, 64},  {64, 1, 0, 96, 3, 64},  {96, 1, 0, 96, 3, 96},  {96, 2, 64, 64, 2, 160}, {64, 1, 0, 64, 2, 64},
    {64, 2, 48, 48, 1, 112}, {48, 1, 0, 48, 1, 48}, {48, 2, 32, 32, 0, 80}, {32, 1, 0, 32, 0, 32},
};

// Workgroups of a layer's weight gradient: 32-pixel strips of `rows` rows.
// More workgroups fill the chip, but each adds a slice of partial sums to write
// and read back (4 bytes per parameter): up to 256 slices of at most 12 MB in
// all. On 8 images of 128 x 128 that is 128 to 256 strips at full resolution
// and 32 to 64 at the coarsest level.
struct GradPlan {
    uint32_t rows, rblocks, segs, strips, nblk, size;
};
static GradPlan grad_plan(const LayerDesc& L, uint32_t N, uint32_t H, uint32_t W) {
    GradPlan p;
    p.size = (uint32_t)(L.cout * 9 * L.cin_real + L.cout);
    p.segs = (W + kGradTileW - 1) / kGradTileW;
    const uint64_t want = std::max<uint64_t>(16, std::min<uint64_t>(256, (12u << 20) / (p.size * 4ull)));
    // columns of strips split into strips of at least 4 rows (each also stages
    // the row above and below); a workgroup takes several when there are more
    const uint64_t columns = (uint64_t)N * p.segs, per = std::max<uint64_t>(1, want / columns);
    p.rows = std::min(H, std::max<uint32_t>(4, (uint32_t)((H + per - 1) / per)));
    p.rblocks = (H + p.rows - 1) / p.rows;
    p.strips = (uint32_t)(columns * p.rblocks);
    p.nblk = (uint32_t)std::min<uint64_t>(p.strips, want);
    return p;
}

// (channel tiles per workgroup, output tiles per wave): at most 7 waves, and
// accumulators of at most 4 x 9 tiles (144 registers).
template <int C0, int UP0, int C1, int COUT>
static void wgrad(hipStream_t st, const GradPlan& p, float* part, const __bf16* dy, const __bf16* s0, const __bf16* s1,
                  uint32_t cin_real, uint32_t H, uint32_t W) {
    constexpr int NCT = (C0 + C1) / 16, CW = NCT > 7 ? NCT / 2 : NCT;
    constexpr int MT = COUT / 16, MTW = MT > 4 ? MT / 2 : MT;
    k_conv_wgrad<C0, UP0, C1, COUT, CW, MTW><<<dim3(p.nblk, NCT / CW, MT / MTW), 64 * CW, 0, st>>>(
        dy, s0, s1, part, cin_real, H, W, p.rows, p.rblocks, p.segs, p.strips);
}

size_t net_num_params() {
    size_t n = 0;
    for (const LayerDesc& L : kLayers) n += (size_t)L.cout * 9 * L.cin_real + L.cout;
    return n + 3 * 32 + 3;
}

// He-normal weights (standard deviation sqrt(2 / fan_in)), zero biases, and
// a head at a tenth of that scale, so an untrained network returns nearly its
// noisy input (the head adds to the input's log radiance); Box-Muller over a
// 64-bit LCG, so the vector depends only on the seed.
void net_he_init(uint64_t seed, float* p) {
    uint64_t s = seed * 6364136223846793005ull + 1442695040888963407ull;
    auto uni = [&]() {
        s = s * 6364136223846793005ull + 1442695040888963407ull;
        return ((double)(s >> 11) + 0.5) * (1.0 / 9007199254740992.0);
    };
    auto fill = [&](float* w, size_t nw, size_t fan_in, double scale = 1.0) {
        const double sd = scale * std::sqrt(2.0 / (double)fan_in);
        for (size_t i = 0; i < nw; i++) {
            const double u1 = uni(), u2 = uni();
            w[i] = (float)(sd * std::sqrt(-2.0 * std::log(u1)) * std::cos(6.283185307179586 * u2));
        }
    };
    size_t off = 0;
    for (const LayerDesc& L : kLayers) {
        const size_t nw = (size_t)L.cout * 9 * L.cin_real;
        fill(p + off, nw, 9 * (size_t)L.cin_real);
        for (int i = 0; i < L.cout; i++) p[off + nw + i] = 0.0f;
        off += nw + L.cout;
    }
    fill(p + off, 96, 32, 0.1);
    for (int i = 0; i < 3; i++) p[off + 96 + i] = 0.0f;
}

static inline int kpad(int k) { return (k + 31) / 32 * 32; }

hipError_t Net::init() {
    if (master) return hipSuccess;
    nparams = net_num_params();
    HH_TRY(hipMalloc(&master, nparams * 4));
    HH_TRY(hipMalloc(&grad, nparams * 4));
    HH_TRY(hipMalloc(&adam_m, nparams * 4));
    HH_TRY(hipMalloc(&adam_v, nparams * 4));
    size_t off = 0;
    for (int l = 0; l < kDnLayers; l++) {
        const LayerDesc& L = kLayers[l];
        const int ct = L.c0 + L.c1;
        w_off[l] = off;
        off += (size_t)L.cout * 9 * L.cin_real + L.cout;
        HH_TRY(hipMalloc(&wf[l], (size_t)L.cout * kpad(9 * ct) * 2));
        HH_TRY(hipMalloc(&wb[l], (size_t)ct * kpad(9 * L.cout) * 2));
    }
    w_off[kDnLayers] = off;
    HH_TRY(hipMalloc(&whead, 96 * 2));
    return hipSuccess;
}

hipError_t Net::zero_state(hipStream_t st) {
    k_zero_f32<<<cdiv(nparams, 256), 256, 0, st>>>(adam_m, nparams);
    k_zero_f32<<<cdiv(nparams, 256), 256, 0, st>>>(adam_v, nparams);
    k_zero_f32<<<cdiv(nparams, 256), 256, 0, st>>>(grad, nparams);
    steps = 0;
    return hipGetLastError();
}

hipError_t Net::refresh_weights(hipStream_t st) {
    LayoutTable t;
    uint32_t blocks = 0;
    for (int l = 0; l < kDnLayers; l++) {
        const LayerDesc& L = kLayers[l];
        const int ct = L.c0 + L.c1;
        const size_t n = (size_t)L.cout * kpad(9 * ct) + (size_t)ct * kpad(9 * L.cout);
        t.l[l] = {master + w_off[l], wf[l], wb[l], (uint32_t)L.cout, (uint32_t)L.cin_real, (uint32_t)ct,
                  (uint32_t)kpad(9 * ct), (uint32_t)kpad(9 * L.cout), blocks};
        blocks += cdiv(n, 256);
    }
    t.head = master + w_off[kDnLayers];
    t.head_out = whead;
    k_relayout<<<blocks, 256, 0, st>>>(t);
    return hipGetLastError();
}

static hipError_t alloc_bf16(__bf16** p, size_t n) { return hipMalloc(p, n * 2); }

hipError_t Net::ensure(uint32_t N, uint32_t Hp, uint32_t Wp, bool training) {
    const size_t P = (size_t)N * Hp * Wp;
    if (P <= cap_px && (!training || cap_train)) {
        n = N;
        H = Hp;
        W = Wp;
        return hipSuccess;
    }
    release_acts();
    HH_TRY(alloc_bf16(&xin, P * 16));
    HH_TRY(hipMalloc(&resid, P * 16));
    HH_TRY(hipMalloc(&out, P * 16));
    for (int l = 0; l < kDnLayers; l++) {
        const size_t Pl = P >> (2 * kLayers[l].level);
        HH_TRY(alloc_bf16(&act[l], Pl * kLayers[l].cout));
    }
    for (int k = 0; k < 3; k++) HH_TRY(alloc_bf16(&pool[k], (P >> (2 * (k + 1))) * kLayers[2 * k + 1].cout));
    if (training) {
        size_t gmax = 0;
        for (int l = 0; l < kDnLayers; l++) gmax = std::max(gmax, (P >> (2 * kLayers[l].level)) * kLayers[l].cout);
        HH_TRY(alloc_bf16(&gy[0], gmax));
        HH_TRY(alloc_bf16(&gy[1], gmax));
        for (int k = 0; k < 3; k++) {
            HH_TRY(hipMalloc(&gskip[k], (P >> (2 * k)) * (kLayers[12 - 2 * k].c0 + kLayers[12 - 2 * k].c1) * 4));
            HH_TRY(hipMalloc(&gpool[k], (P >> (2 * (k + 1))) * kLayers[2 * k + 1].cout * 4));
        }
        HH_TRY(hipMalloc(&loss, 64));
        cap_train = true;
    }
    cap_px = P;
    n = N;
    H = Hp;
    W = Wp;
    return hipSuccess;
}

void Net::release_acts() {
    void* ps[] = {xin, resid, out, gy[0], gy[1], loss};
    for (void* p : ps)
        if (p) (void)hipFree(p);
    xin = nullptr;
    resid = nullptr;
    out = nullptr;
    gy[0] = gy[1] = nullptr;
    loss = nullptr;
    for (int l = 0; l < kDnLayers; l++) {
        if (act[l]) (void)hipFree(act[l]);
        act[l] = nullptr;
    }
    for (int k = 0; k < 3; k++) {
        if (pool[k]) (void)hipFree(pool[k]);
        if (gskip[k]) (void)hipFree(gskip[k]);
        if (gpool[k]) (void)hipFree(gpool[k]);
        pool[k] = nullptr;
        gskip[k] = nullptr;
        gpool[k] = nullptr;
    }
    cap_px = 0;
    cap_train = false;
}

void Net::release() {
    release_acts();
    void* ps[] = {master, grad, adam_m, adam_v, whead, gpart};
    for (void* p : ps)
        if (p) (void)hipFree(p);
    master = grad = adam_m = adam_v = gpart = nullptr;
    gpart_cap = 0;
    whead = nullptr;
    for (int l = 0; l < kDnLayers; l++) {
        if (wf[l]) (void)hipFree(wf[l]);
        if (wb[l]) (void)hipFree(wb[l]);
        wf[l] = wb[l] = nullptr;
    }
}

hipError_t Net::pack(hipStream_t st, const float* raw, const float4* rad, const float4* aux, uint32_t held, uint32_t h,
                     uint32_t w) {
    k_pack<<<cdiv(W, 64) * cdiv((size_t)n * H, 4), 256, 0, st>>>(raw, rad, aux, held, n, h, w, H, W, xin, (float4*)resid);
    return hipGetLastError();
}

// `training` keeps the last activation (the backward pass reads it); else the
// head is part of the last convolution, which writes the surface when there is
// one and the network output when there is not.
hipError_t Net::forward(hipStream_t st, float4* surface, uint32_t h, uint32_t w, bool training) {
    const float* b[kDnLayers];
    for (int l = 0; l < kDnLayers; l++) b[l] = master + w_off[l] + (size_t)kLayers[l].cout * 9 * kLayers[l].cin_real;
    const uint32_t N = n;
    auto Hl = [&](int lv) { return H >> lv; };
    auto Wl = [&](int lv) { return W >> lv; };
    auto pooled = [&](int k) {
        ConvExtra ex{};
        ex.pool = pool[k];
        return ex;
    };
    conv<16, 1, 0, 32, EPI_BIAS_RELU>(st, xin, nullptr, wf[0], b[0], nullptr, act[0], N, Hl(0), Wl(0));
    conv<32, 1, 0, 32, EPI_POOL>(st, act[0], nullptr, wf[1], b[1], nullptr, act[1], N, Hl(0), Wl(0), pooled(0));
    conv<32, 1, 0, 48, EPI_BIAS_RELU>(st, pool[0], nullptr, wf[2], b[2], nullptr, act[2], N, Hl(1), Wl(1));
    conv<48, 1, 0, 48, EPI_POOL>(st, act[2], nullptr, wf[3], b[3], nullptr, act[3], N, Hl(1), Wl(1), pooled(1));
    conv<48, 1, 0, 64, EPI_BIAS_RELU>(st, pool[1], nullptr, wf[4], b[4], nullptr, act[4], N, Hl(2), Wl(2));
    conv<64, 1, 0, 64, EPI_POOL>(st, act[4], nullptr, wf[5], b[5], nullptr, act[5], N, Hl(2), Wl(2), pooled(2));
    conv<64, 1, 0, 96, EPI_BIAS_RELU>(st, pool[2], nullptr, wf[6], b[6], nullptr, act[6], N, Hl(3), Wl(3));
    conv<96, 1, 0, 96, EPI_BIAS_RELU>(st, act[6], nullptr, wf[7], b[7], nullptr, act[7], N, Hl(3), Wl(3));
    conv<96, 2, 64, 64, EPI_BIAS_RELU>(st, act[7], act[5], wf[8], b[8], nullptr, act[8], N, Hl(2), Wl(2));
    conv<64, 1, 0, 64, EPI_BIAS_RELU>(st, act[8], nullptr, wf[9], b[9], nullptr, act[9], N, Hl(2), Wl(2));
    conv<64, 2, 48, 48, EPI_BIAS_RELU>(st, act[9], act[3], wf[10], b[10], nullptr, act[10], N, Hl(1), Wl(1));
    conv<48, 1, 0, 48, EPI_BIAS_RELU>(st, act[10], nullptr, wf[11], b[11], nullptr, act[11], N, Hl(1), Wl(1));
    if (training) conv<48, 2, 32, 32, EPI_BIAS_RELU>(st, act[11], act[1], wf[12], b[12], nullptr, act[12], N, Hl(0), Wl(0));
    else conv<48, 2, 32, 32, EPI_SPLIT>(st, act[11], act[1], wf[12], b[12], nullptr, act[12], N, Hl(0), Wl(0));
    const float* bh = master + w_off[kDnLayers] + 96;
    if (training) {
        conv<32, 1, 0, 32, EPI_BIAS_RELU>(st, act[12], nullptr, wf[13], b[13], nullptr, act[13], N, Hl(0), Wl(0));
        k_head<<<cdiv((size_t)N * H * W, 256), 256, 0, st>>>(act[13], whead, bh, (const float4*)resid, (float4*)out, N, H, W);
        return hipGetLastError();
    }
    ConvExtra ex{};
    ex.wh = whead;
    ex.bh = bh;
    ex.resid = (const float4*)resid;
    ex.out = surface ? nullptr : (float4*)out;
    ex.surface = surface;
    ex.h = h;
    ex.w = w;
    conv<32, 1, 0, 32, EPI_HEAD>(st, act[12], nullptr, wf[13], b[13], nullptr, nullptr, N, Hl(0), Wl(0), ex);
    return hipGetLastError();
}

hipError_t Net::loss_and_backward(hipStream_t st, const float* target, uint32_t h, uint32_t w, uint32_t kind) {
    const uint32_t N = n;
    const size_t P = (size_t)N * H * W;
    auto Hl = [&](int lv) { return H >> lv; };
    auto Wl = [&](int lv) { return W >> lv; };
    // workspace of partial gradients: every layer's slices, then the head's and the loss's
    GradPlan plan[kDnLayers];
    GradSlices gs;
    size_t total = 0;
    uint32_t blocks = 0;
    size_t at[GradSlices::kMax];
    auto slice = [&](int k, float* dst, uint32_t size, uint32_t nblk) {
        gs.s[k] = {dst, nullptr, size, nblk, blocks};
        at[k] = total;
        total += (size_t)size * nblk;
        blocks += cdiv(size, 256);
    };
    for (int l = 0; l < kDnLayers; l++) {
        plan[l] = grad_plan(kLayers[l], N, Hl(kLayers[l].level), Wl(kLayers[l].level));
        slice(l, grad + w_off[l], plan[l].size, plan[l].nblk);
    }
    const uint32_t hblocks = std::min<uint32_t>(cdiv(P, 256), kHeadBlocks);
    slice(kDnLayers, grad + w_off[kDnLayers], 99, hblocks);
    slice(kDnLayers + 1, loss, 1, hblocks);
    if (total > gpart_cap) {
        if (gpart) HH_TRY(hipFree(gpart));
        gpart = nullptr;
        gpart_cap = 0;
        HH_TRY(hipMalloc(&gpart, total * 4));
        gpart_cap = total;
    }
    for (int k = 0; k < GradSlices::kMax; k++) gs.s[k].part = gpart + at[k];
    auto part = [&](int k) { return gpart + at[k]; };
    __bf16* g = gy[0];
    __bf16* g2 = gy[1];
    k_loss_head_backward<<<hblocks, 256, 0, st>>>((const float4*)out, target, act[13], whead, g, part(kDnLayers),
                                                  part(kDnLayers + 1), N, h, w, H, W, kind);
    // dec0b (13): input act[12]
    wgrad<32, 1, 0, 32>(st, plan[13], part(13), g, act[12], nullptr, 32, Hl(0), Wl(0));
    conv<32, 1, 0, 32, EPI_MASK>(st, g, nullptr, wb[13], nullptr, act[12], g2, N, Hl(0), Wl(0));
    std::swap(g, g2);
    // dec0a (12): input [up(act[11]), act[1]] -> gx (80 ch, FP32)
    wgrad<48, 2, 32, 32>(st, plan[12], part(12), g, act[11], act[1], 80, Hl(0), Wl(0));
    conv<32, 1, 0, 80, EPI_F32>(st, g, nullptr, wb[12], nullptr, nullptr, gskip[0], N, Hl(0), Wl(0));
    k_upback_mask<<<cdiv((size_t)N * Hl(1) * Wl(1) * 6, 256), 256, 0, st>>>(gskip[0], 80, act[11], g2, N, Hl(1), Wl(1), 48);
    std::swap(g, g2);
    // dec1b (11): input act[10]
    wgrad<48, 1, 0, 48>(st, plan[11], part(11), g, act[10], nullptr, 48, Hl(1), Wl(1));
    conv<48, 1, 0, 48, EPI_MASK>(st, g, nullptr, wb[11], nullptr, act[10], g2, N, Hl(1), Wl(1));
    std::swap(g, g2);
    // dec1a (10): input [up(act[9]), act[3]] -> gskip[1] (112 ch)
    wgrad<64, 2, 48, 48>(st, plan[10], part(10), g, act[9], act[3], 112, Hl(1), Wl(1));
    conv<48, 1, 0, 112, EPI_F32>(st, g, nullptr, wb[10], nullptr, nullptr, gskip[1], N, Hl(1), Wl(1));
    k_upback_mask<<<cdiv((size_t)N * Hl(2) * Wl(2) * 8, 256), 256, 0, st>>>(gskip[1], 112, act[9], g2, N, Hl(2), Wl(2), 64);
    std::swap(g, g2);
    // dec2b (9): input act[8]
    wgrad<64, 1, 0, 64>(st, plan[9], part(9), g, act[8], nullptr, 64, Hl(2), Wl(2));
    conv<64, 1, 0, 64, EPI_MASK>(st, g, nullptr, wb[9], nullptr, act[8], g2, N, Hl(2), Wl(2));
    std::swap(g, g2);
    // dec2a (8): input [up(act[7]), act[5]] -> gskip[2] (160 ch)
    wgrad<96, 2, 64, 64>(st, plan[8], part(8), g, act[7], act[5], 160, Hl(2), Wl(2));
    conv<64, 1, 0, 160, EPI_F32>(st, g, nullptr, wb[8], nullptr, nullptr, gskip[2], N, Hl(2), Wl(2));
    k_upback_mask<<<cdiv((size_t)N * Hl(3) * Wl(3) * 12, 256), 256, 0, st>>>(gskip[2], 160, act[7], g2, N, Hl(3), Wl(3), 96);
    std::swap(g, g2);
    // midb (7): input act[6]
    wgrad<96, 1, 0, 96>(st, plan[7], part(7), g, act[6], nullptr, 96, Hl(3), Wl(3));
    conv<96, 1, 0, 96, EPI_MASK>(st, g, nullptr, wb[7], nullptr, act[6], g2, N, Hl(3), Wl(3));
    std::swap(g, g2);
    // mida (6): input pool[2] -> gpool[2] (FP32)
    wgrad<64, 1, 0, 96>(st, plan[6], part(6), g, pool[2], nullptr, 64, Hl(3), Wl(3));
    conv<96, 1, 0, 64, EPI_F32>(st, g, nullptr, wb[6], nullptr, nullptr, gpool[2], N, Hl(3), Wl(3));
    // enc2b (5): gradient = pooled path + skip of dec2a (channels 96..159)
    k_poolback_skip_mask<<<cdiv((size_t)N * Hl(2) * Wl(2) * 8, 256), 256, 0, st>>>(gpool[2], gskip[2], 160, 96, act[5], g, N,
                                                                                  Hl(2), Wl(2), 64);
    wgrad<64, 1, 0, 64>(st, plan[5], part(5), g, act[4], nullptr, 64, Hl(2), Wl(2));
    conv<64, 1, 0, 64, EPI_MASK>(st, g, nullptr, wb[5], nullptr, act[4], g2, N, Hl(2), Wl(2));
    std::swap(g, g2);
    // enc2a (4): input pool[1] -> gpool[1]
    wgrad<48, 1, 0, 64>(st, plan[4], part(4), g, pool[1], nullptr, 48, Hl(2), Wl(2));
    conv<64, 1, 0, 48, EPI_F32>(st, g, nullptr, wb[4], nullptr, nullptr, gpool[1], N, Hl(2), Wl(2));
    // enc1b (3): pooled path + skip of dec1a (channels 64..111)
    k_poolback_skip_mask<<<cdiv((size_t)N * Hl(1) * Wl(1) * 6, 256), 256, 0, st>>>(gpool[1], gskip[1], 112, 64, act[3], g, N,
                                                                                  Hl(1), Wl(1), 48);
    wgrad<48, 1, 0, 48>(st, plan[3], part(3), g, act[2], nullptr, 48, Hl(1), Wl(1));
    conv<48, 1, 0, 48, EPI_MASK>(st, g, nullptr, wb[3], nullptr, act[2], g2, N, Hl(1), Wl(1));
    std::swap(g, g2);
    // enc1a (2): input pool[0] -> gpool[0]
    wgrad<32, 1, 0, 48>(st, plan[2], part(2), g, pool[0], nullptr, 32, Hl(1), Wl(1));
    conv<48, 1, 0, 32, EPI_F32>(st, g, nullptr, wb[2], nullptr, nullptr, gpool[0], N, Hl(1), Wl(1));
    // enc0b (1): pooled path + skip of dec0a (channels 48..79)
    k_poolback_skip_mask<<<cdiv((size_t)N * Hl(0) * Wl(0) * 4, 256), 256, 0, st>>>(gpool[0], gskip[0], 80, 48, act[1], g, N,
                                                                                  Hl(0), Wl(0), 32);
    wgrad<32, 1, 0, 32>(st, plan[1], part(1), g, act[0], nullptr, 32, Hl(0), Wl(0));
    conv<32, 1, 0, 32, EPI_MASK>(st, g, nullptr, wb[1], nullptr, act[0], g2, N, Hl(0), Wl(0));
    std::swap(g, g2);
    // enc0a (0): weights only
    wgrad<16, 1, 0, 32>(st, plan[0], part(0), g, xin, nullptr, 10, Hl(0), Wl(0));
    k_reduce_grads<<<blocks, 256, 0, st>>>(gs);
    return hipGetLastError();
}

hipError_t Net::adam(hipStream_t st, float lr) {
    steps++;
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.0f - powf(b1, (float)steps), c2 = 1.0f - powf(b2, (float)steps);
    k_adam<<<cdiv(nparams, 256), 256, 0, st>>>(master, grad, adam_m, adam_v, nparams, lr, b1, b2, 1e-8f, c1, c2);
    HH_TRY(hipGetLastError());
    return refresh_weights(st);
}

}  // namespace dn
}  // namespace hh
