// Codec operators of the resident NanoCodec decode (decode_codec_resident, src/graph.c:2504-2638; res_layer_device
// :2423-2498): causal dilated conv1d, grouped causal transposed conv and the half-snake activation, on device rows of
// layout [channels, length].  Weights, biases and snake alphas arrive as HOST pointers and are cached on the device at
// first sight like every other weight (the seam's contract).  None of the three synchronises.
//
//   conv1d          out[o][t] = bias[o] + sum_i sum_k w[(o*in + i)*K + k] * in[i][t - (K-1-k)*dilation]   (conv1d_causal,
//                   src/graph.c:2010-2160).  The reference builds an im2col matrix and calls sgemm; here the same GEMM
//                   (M = out channels, N = length, inner = in channels x taps) runs on the bf16 matrix cores in three-piece
//                   form (split_product.h: f32 operands, f32 accumulation, the accuracy of an f32 product) with the im2col
//                   done by addressing: a workgroup stages the input rows of sixteen channels once, with a halo of
//                   (K-1)*dilation positions, and every tap reads the same rows at its own offset.
//   conv_transpose  grouped, trimmed to output_length (conv_transpose_causal / convt_channel, src/graph.c:2179-2231):
//                   one thread per output element, contributions added in the reference's order (input channel, then
//                   input position), so the result is bit-identical to the scalar CPU loop.
//   snake           x + sin(a x)^2 * (1 / (a + 1e-9)) on the first snake_channels rows, leaky ReLU (0.01) on the rest
//                   (snake_row, src/backend.c:643-658).
#include <limits.h>
#include <stddef.h>

#include <type_traits>
#include <utility>

#include "split_product.h"

using namespace mynah;

namespace {

typedef f32x16 floatx16;
typedef unsigned short ushort8 __attribute__((ext_vector_type(8)));

// A value at `bytes` behind an address that is the same for every lane: one instruction with the address in scalar registers, where
// pointer arithmetic by lanes takes 64-bit addresses in vector registers.
// (opaque: what stays the same from request to request is otherwise added up ahead of all loops, 64 bits a lane and request)
template <class T>
__device__ __forceinline__ T load_behind(const T *base, unsigned bytes) { return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + bytes); }
__device__ __forceinline__ unsigned opaque(unsigned v) {
    asm volatile("" : "+v"(v));
    return v;
}
__device__ __forceinline__ int opaque_scalar(int v) {
    asm volatile("" : "+s"(v));
    return v;
}

constexpr int kConvMaxKernel = 16;
constexpr int kConvMaxHalo = 128;     // (kernel - 1) * dilation
constexpr int kTileStride = 65;       // floats per row of a wavefront's 32 x 64 tile in LDS (fused epilogue)

struct ConvArgs {
    const float *in;     // [in_ch, length]
    float *out;          // [out_ch, length]
    const float *bias;   // [out_ch] or null
    int in_ch, out_ch, length, kernel, dilation;
    // what mynah_hip_conv1d_fused adds after conv + bias, in this order (each step is the arithmetic of the seam operator it replaces)
    const float *residual = nullptr;    // [out_ch, length] added (residual_inplace); may be `out` itself
    const float *residual2 = nullptr;   // then this one
    float scale = 1.0f;                 // then multiplied (scale_dev) when `scaled`
    int scaled = 0;
    int activate = 0;                   // then the half-snake of the value's output channel (snake_dev)
    const float *alpha = nullptr;       // [snake_channels]
    int snake_channels = 0;
    float *act_out = nullptr;           // null: `out` gets the activated value; else `out` keeps the value before it and this gets the activated one
    // channel-split tiles only: workgroups that share a tile's channels, and where each leaves its sums ([splits][out_ch][length])
    int splits = 1;
    float *parts = nullptr;
    const uint4 *weights = nullptr;   // ConvBlocks data
};

// sin(x) in some twenty instructions for |x| < kShortSineLimit (the library routine, which also serves arguments of any
// size, is about 150, and inside a convolution's epilogue nothing hides them): x = k * pi/2 + r with pi/2 in three pieces
// and fused multiply-adds, then the sine or cosine polynomial of r on [-pi/4, pi/4] (Cephes' single-precision
// coefficients).  Largest difference from the double-precision sine over every 7th float of (-8192, 8192): 9.3e-8, against
// 6e-8 for a correctly rounded result near 1.
constexpr float kShortSineLimit = 8192.0f;
__device__ __forceinline__ float short_sine(float x) {
    const float k = __builtin_rintf(x * 0.636619772367581343f);
    float r = __builtin_fmaf(k, -1.57079637050628662109375f, x);
    r = __builtin_fmaf(k, 4.37113882867379289e-8f, r);
    r = __builtin_fmaf(k, 1.71512460692744033e-15f, r);
    const float z = r * r;
    const float s = __builtin_fmaf(r * z, __builtin_fmaf(z, __builtin_fmaf(z, -1.9515295891e-4f, 8.3321608736e-3f), -1.6666654611e-1f), r);
    const float c = __builtin_fmaf(z * z, __builtin_fmaf(z, __builtin_fmaf(z, 2.443315711809948e-5f, -1.388731625493765e-3f), 4.166664568298827e-2f),
                                   __builtin_fmaf(z, -0.5f, 1.0f));
    const int q = (int)k;
    const float v = (q & 1) ? c : s;
    return (q & 2) ? -v : v;
}
// The codec's sine: the short routine where it holds, the library's beyond.
__device__ __forceinline__ float snake_sine(float x) { return fabsf(x) < kShortSineLimit ? short_sine(x) : sinf(x); }

// snake_row, src/backend.c:643-658.  inv_a = 1 / (alpha + 1e-9) for a snake row; a row past snake_channels is a leaky ReLU.
__device__ __forceinline__ float half_snake(float v, bool snake_row, float al, float inv_a) {
    if (snake_row) {
        const float sn = snake_sine(al * v);
        return v + sn * sn * inv_a;
    }
    return v < 0.0f ? v * 0.01f : v;
}

// One finished output value (conv + bias) on its way to memory, in two steps so that a kernel can run the first (two
// requests and three operations) for all of a thread's values at once, requests side by side, and the second (some
// hundred instructions when there is an activation) in a rolled loop.
__device__ __forceinline__ float conv_combine(const ConvArgs &a, size_t index, float v) {
    if (a.residual != nullptr) v = a.residual[index] + v;
    if (a.residual2 != nullptr) v = a.residual2[index] + v;
    return v * a.scale;   // 1.0f when there is no scaling: the value's own bits
}
// al, inv_a: the output channel's alpha and 1 / (alpha + 1e-9), which the kernels keep in LDS: read from global memory value
// by value inside the rolled loops, that request was most of what an activation cost.
__device__ __forceinline__ void conv_emit(const ConvArgs &a, int m, size_t index, float v, float al, float inv_a) {
    if (a.activate) {
        const float act = half_snake(v, m < a.snake_channels, al, inv_a);
        if (a.act_out != nullptr) {
            a.out[index] = v;
            a.act_out[index] = act;
        } else {
            a.out[index] = act;
        }
    } else {
        a.out[index] = v;
    }
}

// The convolution's inner dimension goes in steps of one tap of sixteen input channels: one 16-deep matrix instruction per pair of
// pieces.  Weights: taken apart once, when they are cached, in the order of the steps (ConvBlocks), so that a wavefront's three
// pieces of a step are three requests of 1 KiB straight to its registers.  Inputs: a staged (position, eight channels) is 16 bytes
// of LDS per piece, so a tap's operand is 512 consecutive bytes for 32 positions, whatever the tap's offset.
struct ConvWeights {   // the weight pieces of one row tile, requested kAhead steps before they are multiplied
    static constexpr int kAhead = kConvStepsAhead;
    const uint4 *next;   // the same for every lane, like the inputs' rows below: an address is then a pair of scalar registers and the lane's offset, where
                         // one of 64 bits per lane and request had taken the products' registers (and spilled)
    unsigned bytes;   // a lane's 16
    size_t skip;       // from the end of a block to the next one this wavefront multiplies
    int blocks;        // it multiplies
    int tap = 0;       // of the next request (a constant wherever the tap count is one)
    uint4 ring[kAhead][3];
    __device__ __forceinline__ void request(int slot, int taps) {
        bytes = opaque(bytes);
#pragma unroll
        for (int q = 0; q < 3; ++q) ring[slot][q] = load_behind(next + 64 * q, bytes);
        next += 192;
        if (++tap == taps) {
            tap = 0;
            if (--blocks > 0) next += skip;
        }
    }
    // The request that is multiplied next, in slot BY, to slot 0 (and so on).
    template <int BY>
    __device__ __forceinline__ void turn() {
        if constexpr (BY != 0) {
            uint4 was[kAhead][3];
#pragma unroll
            for (int i = 0; i < kAhead; ++i)
#pragma unroll
                for (int q = 0; q < 3; ++q) was[i][q] = ring[i][q];
#pragma unroll
            for (int i = 0; i < kAhead; ++i)
#pragma unroll
                for (int q = 0; q < 3; ++q) ring[i][q] = was[(i + BY) % kAhead][q];
        }
    }
    // (what runs past the last step is requested and not used: it is what follows the last block, and the cache pads its copies)
    __device__ __forceinline__ ConvWeights(const uint4 *first, unsigned lane, size_t skip_arg, int blocks_arg, int taps)
        : next(first), bytes(lane * 16), skip(skip_arg), blocks(blocks_arg) {
#pragma unroll
        for (int i = 0; i < kAhead; ++i) request(i, taps);
    }
};

// The products of the blocks of sixteen channels a wavefront multiplies, for its 32 rows x (32 * NT) positions.
// stage(block): makes the block's inputs readable and returns where this lane's first operand lies: element [piece * PIECE + position]
// (a constant: one address register serves a tap's reads), lanes 32.. eight channels on.  With the tap count known (KF) the loop over a block's steps is unrolled, and three blocks at
// a time, after which the weights' registers repeat.  (A step's fragments are read right before it: two or three wavefronts share a
// SIMD, and a second set of fragment registers, read a step ahead, spilled: 1884 against 1754 us for a 64-frame decode.)
template <int KF, int NT, int PIECE, bool AHEAD = false, class Stage>
__device__ __forceinline__ void conv_products(ConvWeights &w, const int taps, const int dilation, const int blocks, const Stage stage,
                                              floatx16 (&acc)[NT]) {
    bf16x8 x[AHEAD ? 2 : 1][NT][3];
    const auto read = [&](int set, const uint4 *at) {
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int q = 0; q < 3; ++q) x[set][n][q] = __builtin_bit_cast(bf16x8, at[q * PIECE + 32 * n]);
    };
    const auto multiply = [&](int set, int slot) {
        bf16x8 fw[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) fw[q] = __builtin_bit_cast(bf16x8, w.ring[slot][q]);
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n] = split_multiply(fw, x[set][n], acc[n]);
    };
    if constexpr (KF != 0 && AHEAD) {
        // (the one-launch block: its few blocks run once, and code that is run once is waited for, instruction by instruction; so one copy of a
        // block's steps, the weights' registers turned back in place at its end: as fast as three copies (54 channels x 13824 112.5 us a layer, 111.3 with one) in less code)
        for (int block = 0; block < blocks; ++block) {
            const uint4 *at = stage(block);
            read(0, at);
#pragma unroll
            for (int tap = 0; tap < KF; ++tap) {
                if (tap + 1 < KF) read((tap + 1) & 1, at + (tap + 1) * dilation);
                multiply(tap & 1, tap % ConvWeights::kAhead);
                w.request(tap % ConvWeights::kAhead, KF);
                __builtin_amdgcn_sched_barrier(0);
            }
            w.template turn<KF % ConvWeights::kAhead>();
        }
    } else if constexpr (KF != 0) {
        for (int block = 0;;) {
#pragma unroll
            for (int u = 0; u < ConvWeights::kAhead; ++u) {
                const uint4 *at = stage(block);
#pragma unroll
                for (int tap = 0; tap < KF; ++tap) {
                    const int s = u * KF + tap;
                    read(0, at + tap * dilation);
                    multiply(0, s % ConvWeights::kAhead);
                    w.request(s % ConvWeights::kAhead, KF);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (++block == blocks) return;
            }
        }
    } else {
        for (int block = 0; block < blocks; ++block) {
            const uint4 *at = stage(block);
            for (int tap = 0; tap < taps; ++tap) {
                read(0, at + tap * dilation);
                multiply(0, 0);
#pragma unroll
                for (int i = 0; i + 1 < ConvWeights::kAhead; ++i)
#pragma unroll
                    for (int q = 0; q < 3; ++q) w.ring[i][q] = w.ring[i + 1][q];
                w.request(ConvWeights::kAhead - 1, taps);
            }
        }
    }
}

// What a sum of pieces that is no finite number stands for (split_product.h): the chain of f32 multiply-adds, from `s`, over the channels
// (eight, then the taps, then the next eight) of every block that mine(block) names.  w: the output row's first piece of the first block and
// tap; inside(tap): whether the tap's position lies in the row; fetch(channel, tap, x): its eight inputs from that channel on.
template <class Mine, class Inside, class Fetch>
__device__ __forceinline__ float conv_chain(const uint4 *const w, const int channels, const int taps, const Mine mine, const Inside inside, const Fetch fetch, float s) {
#pragma unroll 1
    for (int c = 0; c < channels && s == s; c += 8) {
        if (!mine(c >> 4)) continue;
#pragma unroll 1
        for (int tap = 0; tap < taps; ++tap) {
            if (!inside(tap)) continue;
            const uint4 *const at = w + (size_t)((c >> 4) * taps + tap) * 192 + ((c >> 3) & 1) * 32;
            const ushort8 h = __builtin_bit_cast(ushort8, at[0]), m = __builtin_bit_cast(ushort8, at[64]), l = __builtin_bit_cast(ushort8, at[128]);
            float x[8];
            fetch(c, tap, x);
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (c + e < channels) s = __builtin_fmaf(split_value(h[e], m[e], l[e]), x[e], s);
        }
    }
    return s;
}
// An output row's first piece of the first block and tap.
__device__ __forceinline__ const uint4 *conv_row(const uint4 *data, const int blocks, const int taps, const int row) {
    return data + (size_t)(row >> 5) * blocks * taps * 192 + (row & 31);
}
// ... of a convolution's own input rows, at output position t of row m.
template <class Mine>
__device__ __forceinline__ float conv_chain_rows(const ConvArgs &a, const int m, const int t, const Mine mine, const float s) {
    const int back = (a.kernel - 1) * a.dilation;
    return conv_chain(conv_row(a.weights, (a.in_ch + 15) / 16, a.kernel, m), a.in_ch, a.kernel, mine, [&](int tap) { return t - back + tap * a.dilation >= 0; },
                      [&](int c, int tap, float (&x)[8]) {
#pragma unroll
                          for (int e = 0; e < 8; ++e) x[e] = a.in[(size_t)min(c + e, a.in_ch - 1) * a.length + t - back + tap * a.dilation];
                      }, s);
}

// Eight rows' values at one position: row channel + e, the last one for what there is not.
__device__ __forceinline__ void request_rows(float (&v)[8], const float *first, int channel, int channels, int length, unsigned bytes) {
    const float *row = first + (size_t)min(channel, channels - 1) * length;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        v[e] = load_behind(row, bytes);
        row += channel + e + 1 < channels ? length : 0;
    }
}
__device__ __forceinline__ void store_pieces(const float (&v)[8], uint4 *at, int piece_stride) {
    bf16x8 p[3];
    split_eight(make_float4(v[0], v[1], v[2], v[3]), make_float4(v[4], v[5], v[6], v[7]), p);
#pragma unroll
    for (int q = 0; q < 3; ++q) at[q * piece_stride] = __builtin_bit_cast(uint4, p[q]);
}
// One (position, eight channels) on its way to LDS: eight requests, then the pieces of the eight values.
struct ConvColumn {
    float v[8];
    // rows channel .. channel + 7 of the input, `bytes` behind `origin` of the first row (channel and origin are the same for
    // every lane); a channel the input does not have repeats its last one -- its weights are zeros
    __device__ __forceinline__ void request(const float *origin, int channel, int channels, int length, unsigned &bytes) {
        bytes = opaque(bytes);
        channel = opaque_scalar(channel);
        request_rows(v, origin, channel, channels, length, bytes);
    }
    __device__ __forceinline__ void store(uint4 *at, int piece_stride, bool inside) const {
        float u[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) u[e] = inside ? v[e] : 0.0f;   // (in front of the row)
        store_pieces(u, at, piece_stride);
    }
};

// What is hardly ever run of the tiles below, with the arguments read from memory once more, behind an empty asm statement that keeps the
// reads there (at the kernel's start they were 0.6 us of every call).
__device__ __forceinline__ ConvArgs conv_again(const ConvArgs *args) {
    asm volatile("" : "+s"(args));
    return *args;
}
// conv_tile's values of one position through the loop over its rows: conv_chain for a sum that is no finite number, and the library's sine.
// A call of its own for the fused builds: inline its registers came on top of the products' (11 taps: 4 to 11 % of a call, some of it
// spilled).  The other builds have room for it.
__device__ __forceinline__ void conv_tile_rest(const ConvArgs &a, const float *s_tile, const float *const s_alpha, const int m_first, const int rows, const int t) {
#pragma unroll 1
    for (int row = 0; row < rows; ++row, s_tile += kTileStride) {
        const int m = m_first + row;
        const size_t index = (size_t)m * a.length + t;
        float v = *s_tile;
        if (!split_finite(v))
            v = conv_combine(a, index, conv_chain_rows(a, m, t, [](int) { return true; }, a.bias != nullptr ? a.bias[m] : 0.0f));
        conv_emit(a, m, index, v, s_alpha[row], s_alpha[32 + row]);
    }
}
__device__ __noinline__ void conv_tile_rest_call(const ConvArgs *const args, const float *const s_tile, const float *const s_alpha, const int m_first, const int rows, const int t) {
    conv_tile_rest(*args, s_tile, s_alpha, m_first, rows, t);
}
// conv_split_tile's partial sums of a thread's eight values (see there), the first taking the whole where it is no finite number.
__device__ __forceinline__ void conv_split_rest(const ConvArgs *const args, float *const s_part, const int split, const int m0, const int t) {
    const ConvArgs a = conv_again(args);
    const int tid = threadIdx.x, pos = tid & 63;
#pragma unroll 1
    for (int j = 0; j < 8; ++j) {
        const int row = (tid >> 6) + 4 * j, m = m0 + row;
        float *const at = s_part + ((((row >> 3) << 2) | (row & 3)) + 16 * (pos >> 5)) * 64 + ((row >> 2) & 1) * 32 + (pos & 31);
        if (m >= a.out_ch || split_finite(((at[0] + at[2048]) + at[4096]) + at[6144])) continue;
        at[0] = conv_chain_rows(a, m, t, [&](int block) { return block % (4 * a.splits) / 4 == split; }, 0.0f);
        at[2048] = at[4096] = at[6144] = 0.0f;
    }
}

constexpr int conv_pitch(int positions) { return positions + kConvMaxHalo; }
// (channel-split tiles: 64 * parts positions hold the window)
constexpr int conv_split_pitch(int nt, int parts) { return 64 * parts < conv_pitch(32 * nt) ? 64 * parts : conv_pitch(32 * nt); }
struct ConvTileRows {   // of a tile's output rows
    alignas(16) float bias[64];
    float alpha[32], inverse_alpha[32];   // (channel-split tiles) of the rows' half-snake, and 1 / (alpha + 1e-9)
};

// Workgroup tile: (32 * WM) output channels x (64 * WN) positions; a wavefront owns 32 x 64 (two 32 x 32 tiles of sums).
// KF: number of taps known at compile time (0 = from the arguments); the codec's 3, 7 and 11 taps get such builds.
// FUSED: the build that mynah_hip_conv1d_fused launches (residuals, scale, activation after the products); the seam's
// conv1d keeps a build without any of it.
// Two stages of one block of channels: a block is stored while the one before it is multiplied (by other wavefronts: three
// to a SIMD), its requests leave a block earlier.
// (the tile's work as a function: the kernel of one convolution and the kernel of several side by side both run it; `again`: the
// arguments as they lie in memory, for conv_tile_rest)
template <int WM, int WN, int KF, bool FUSED>
__device__ __forceinline__ void conv_tile(const ConvArgs &a_arg, const ConvBlocks &w_arg, const ConvArgs *const again, uint4 *const lds, ConvTileRows &s_rows) {
    constexpr int TM = 32 * WM, TN = 64 * WN;
    ConvArgs a = a_arg;
    if constexpr (KF != 0) a.kernel = KF;
    const int halo = (a.kernel - 1) * a.dilation;
    const int win = TN + halo;                 // staged positions
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN;
    const int m0 = blockIdx.y * TM, t0 = blockIdx.x * TN;
    const int half = lane >> 5, col = lane & 31;

    // Staging: a thread takes one position of the first eight channels and one of the second, half a workgroup apart (a window of
    // 128 + halo positions then leaves every wavefront the same work); windows beyond 256 positions a third, the first
    // half of the workgroup for the first eight channels.
    constexpr int kColumns = TN + kConvMaxHalo > 256 ? 3 : 2;
    static_assert(TN + kConvMaxHalo <= 384, "three columns a thread cover the window");
    int place[kColumns];      // window position, or -1
    unsigned from[kColumns];  // bytes from the window's first position (in the row) to this one, clamped into the row
    bool inside[kColumns];
    const int first = max(t0 - halo, 0);
#pragma unroll
    for (int x = 0; x < kColumns; ++x) {
        const int p = x == 0 ? tid : x == 1 ? (tid + 128) & 255 : 256 + (tid & 127);
        const int t = t0 - halo + p;
        place[x] = p < win ? p : -1;
        inside[x] = t >= 0;
        from[x] = (unsigned)(min(max(t, 0), a.length - 1) - first) * 4;
    }
    const auto group_of = [&](int x) { return x < 2 ? x : __builtin_amdgcn_readfirstlane(tid >> 7); };
    ConvColumn column[kColumns];
    const auto fetch = [&](int block) {
#pragma unroll
        for (int x = 0; x < kColumns; ++x) column[x].request(a.in + first, 16 * block + 8 * group_of(x), a.in_ch, a.length, from[x]);
    };
    constexpr int kPitch = conv_pitch(TN);
    uint4 *stage_now = lds, *stage_next = lds + 6 * kPitch;   // [piece][eight channels][position]
    const auto publish = [&](uint4 *stage) {
#pragma unroll
        for (int x = 0; x < kColumns; ++x)
            if (place[x] >= 0) column[x].store(stage + group_of(x) * kPitch + place[x], 2 * kPitch, inside[x]);
    };
    const int tile = min((int)blockIdx.y * WM + wm, w_arg.tiles - 1);
    // (requested here, beside the first block: at the end they would be a round trip in front of the stores)
    if (tid < TM) s_rows.bias[tid] = a.bias != nullptr && m0 + tid < a.out_ch ? a.bias[m0 + tid] : 0.0f;
    const auto stage = [&](int block) {
        __syncthreads();   // this block is stored, and nobody multiplies the one whose place the next one takes
        const uint4 *at = stage_now + half * kPitch + wn * 64 + col;
        if (block + 1 < w_arg.blocks) {
            publish(stage_next);
            fetch(min(block + 2, w_arg.blocks - 1));
        }
        uint4 *t = stage_now;
        stage_now = stage_next;
        stage_next = t;
        return at;
    };
    // The sums start from the rows' biases, so a value is bias + products in the products' order.
    floatx16 sums[2];
    fetch(0);
    ConvWeights w(w_arg.data + (size_t)tile * w_arg.blocks * a.kernel * 192, lane, 0, 1, a.kernel);
    publish(stage_now);
    fetch(min(1, w_arg.blocks - 1));
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r) sums[0][r] = s_rows.bias[wm * 32 + split_acc_row(r, lane)];
    sums[1] = sums[0];
    conv_products<KF, 2, 2 * kPitch>(w, a.kernel, a.dilation, w_arg.blocks, stage, sums);
    __syncthreads();   // the epilogue's pieces of LDS overwrite the stages
    // What follows starts from the thread's number anew: what the compiler may take from above it forms ahead of the products and keeps in
    // scratch memory meanwhile (35 values of a thread, 27 MB a launch written before the first product and read behind the last).
    const int tid_after = (int)opaque(threadIdx.x), lane_after = tid_after & 63, wave_after = __builtin_amdgcn_readfirstlane(tid_after >> 6);
    const auto finish = [&](const int lane, const int wave) {
    const int wm = wave / WN, wn = wave % WN, half = lane >> 5, col = lane & 31;
    floatx16 (&acc)[2] = sums;
    floatx16 &acc0 = acc[0], &acc1 = acc[1];
    // The fused build's residual values, requested side by side; a residual may be the output itself -- every workgroup reads and
    // writes its own tile only.
    float res_first[FUSED ? 32 : 1], res_second[FUSED ? 32 : 1];
    if constexpr (FUSED) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m = m0 + wm * 32 + 8 * (r >> 2) + 4 * half + (r & 3);
            const int t = t0 + wn * 64 + col;
            const bool in0 = m < a.out_ch && t < a.length, in1 = m < a.out_ch && t + 32 < a.length;
            const size_t i0 = in0 ? (size_t)m * a.length + t : 0, i1 = in1 ? (size_t)m * a.length + t + 32 : 0;
            if (a.residual != nullptr) { res_first[r] = a.residual[i0]; res_first[16 + r] = a.residual[i1]; }
            if (a.residual2 != nullptr) { res_second[r] = a.residual2[i0]; res_second[16 + r] = a.residual2[i1]; }
        }
    }
    // accumulator element r of a lane: row 8 * (r / 4) + 4 * (lane / 32) + r % 4, column lane % 32
    // conv + bias, then the residuals (requested to a legal address whatever the value's place)
    // and the scale, in conv_combine's order, without a branch per value: an addition that is not wanted at all is left out
    // by the build of this loop that runs.
    // A finished tile on its way to memory: from the accumulators' layout (a store instruction there covers 32 positions of
    // two rows, and a row's validity differs between the halves of a wavefront: a mask and a branch per store) through the
    // wavefront's own piece of LDS (free after the last products' barrier) to whole rows of 64 consecutive positions, whose
    // validity is the same for every lane -- a loop over the rows that exist, the positions' own check once around it.
    const auto store_tile = [&](float *dst, const floatx16 &first, const floatx16 &second) {
        float *s_tile = reinterpret_cast<float *>(lds) + wave * (32 * kTileStride);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = 8 * (r >> 2) + 4 * half + (r & 3);
            s_tile[row * kTileStride + col] = first[r];
            s_tile[row * kTileStride + col + 32] = second[r];
        }
        const int t = t0 + wn * 64 + lane;
        const int rows = min(32, a.out_ch - (m0 + wm * 32));   // the same for the whole wavefront
        if (t < a.length) {
            float *p = dst + (size_t)(m0 + wm * 32) * a.length + t;
#pragma unroll 8
            for (int row = 0; row < rows; ++row, p += a.length) *p = s_tile[row * kTileStride + lane];
        }
    };
    const auto combine = [&](auto has_first, auto has_second) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float v0 = acc0[r], v1 = acc1[r];
            if constexpr (decltype(has_first)::value) { v0 = res_first[r] + v0; v1 = res_first[16 + r] + v1; }
            if constexpr (decltype(has_second)::value) { v0 = res_second[r] + v0; v1 = res_second[16 + r] + v1; }
            if constexpr (FUSED) {
                v0 = v0 * a.scale;   // 1.0f when there is no scaling: the value's own bits
                v1 = v1 * a.scale;
            }
            acc0[r] = v0;
            acc1[r] = v1;
        }
    };
    const bool finite = FUSED && (a.activate || split_all_finite(acc));   // (here, while the residual's values are on their way)
    if constexpr (FUSED) {
        if (a.residual2 != nullptr) combine(std::true_type{}, std::true_type{});    // the launch refuses a second residual without a first
        else if (a.residual != nullptr) combine(std::true_type{}, std::false_type{});
        else combine(std::false_type{}, std::false_type{});
    }
    if constexpr (!FUSED) {   // the seam's conv1d; what is no finite number is stored once more below
        store_tile(a.out, acc0, acc1);
        if (__builtin_expect(split_all_finite(acc), 1)) return;
    } else if (!a.activate && __builtin_expect(finite, 1)) {
        store_tile(a.out, acc0, acc1);
        return;
    }
    // The rows' alphas and 1 / (alpha + 1e-9) through the wavefront's own piece of LDS (free after the last products' barrier)
    float *s_alpha = reinterpret_cast<float *>(lds) + 4 * (32 * kTileStride) + wave * 64;
    if (FUSED && a.activate) {
        if (lane < 32) {
            const int m = m0 + wm * 32 + lane;
            const float al = m < a.snake_channels ? a.alpha[m] : 0.0f;
            s_alpha[lane] = al;
            s_alpha[32 + lane] = 1.0f / (al + 1e-9f);
        }
        // Common case, every sine argument below the short routine's limit: the activation on the values where they are, in
        // registers, the short sine inlined 32 times and no branch among them.  (A sum that is no finite number is not below it
        // either, whatever the alpha.)
        bool large = false;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float al = s_alpha[8 * (r >> 2) + 4 * half + (r & 3)];
            large = large || !(fabsf(al * acc0[r]) < kShortSineLimit) || !(fabsf(al * acc1[r]) < kShortSineLimit);
        }
        if (__builtin_expect(!__any(large), 1)) {
            floatx16 act0, act1;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = 8 * (r >> 2) + 4 * half + (r & 3), m = m0 + wm * 32 + row;
                const float al = s_alpha[row], inv_a = s_alpha[32 + row];
                const float v0 = acc0[r], v1 = acc1[r];
                act0[r] = v0 < 0.0f ? v0 * 0.01f : v0;
                act1[r] = v1 < 0.0f ? v1 * 0.01f : v1;
                if (m0 + wm * 32 + 8 * (r >> 2) < a.snake_channels) {   // (else no lane's row of these registers is a snake row: half of all)
                    const float s0 = short_sine(al * v0), s1 = short_sine(al * v1);
                    const bool snake_row = m < a.snake_channels;
                    act0[r] = snake_row ? v0 + s0 * s0 * inv_a : act0[r];
                    act1[r] = snake_row ? v1 + s1 * s1 * inv_a : act1[r];
                }
            }
            if (a.act_out != nullptr) {
                store_tile(a.out, acc0, acc1);
                store_tile(a.act_out, act0, act1);
            } else {
                store_tile(a.out, act0, act1);
            }
            return;
        }
    }
    // Some argument needs the library's sine, or some sum is no finite number: the wavefront's 32 x 64 tile goes through LDS and a rolled
    // loop finishes it a row at a time, with one copy of that long routine.  (Nothing of a fused tile has been stored: a residual that is
    // the output is still there to be added again.)
    float *s_tile = reinterpret_cast<float *>(lds) + wave * (32 * kTileStride);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int row = 8 * (r >> 2) + 4 * half + (r & 3);
        s_tile[row * kTileStride + col] = acc0[r];
        s_tile[row * kTileStride + col + 32] = acc1[r];
    }
    const int t = t0 + wn * 64 + lane;
    if (t >= a.length) return;
    const int rows = min(32, a.out_ch - (m0 + wm * 32));   // the same for the whole wavefront
    if constexpr (FUSED) conv_tile_rest_call(again, s_tile + lane, s_alpha, m0 + wm * 32, rows, t);
    else conv_tile_rest(conv_again(again), s_tile + lane, s_alpha, m0 + wm * 32, rows, t);
    };
    finish(lane_after, wave_after);
}

// (the rows, the weights and the shape lead the arguments and repeat fields of a_arg: leading scalar arguments are in registers
// when a wavefront starts, a structure passed by value is fetched from memory where its fields are first used)
struct ConvKernarg {
    const float *in;
    float *out;
    const uint4 *weights;
    const float *bias;
    int in_ch, out_ch, length, kernel, dilation, tiles;
    ConvArgs a;
};
static_assert(offsetof(ConvKernarg, a) == 56 && alignof(ConvArgs) == 8, "the kernels' argument lists");
// A kernel's arguments where they lie (one structure of them, or the arguments of k_conv1d and k_conv1d_split in order).
template <class T>
__device__ __forceinline__ const T *conv_kernarg() { return (const T *)__builtin_amdgcn_kernarg_segment_ptr(); }

template <int WM, int WN, int KF, bool FUSED>
__global__ void __launch_bounds__(256, 3) k_conv1d(const float *const in_arg, float *const out_arg, const uint4 *const weights_arg, const float *const bias_arg, const int in_ch_arg,
                                                   const int out_ch_arg, const int length_arg, const int kernel_arg, const int dilation_arg, const int tiles_arg,
                                                   const ConvArgs a_arg) {
    extern __shared__ __align__(16) uint4 lds[];
    __shared__ ConvTileRows s_rows;
    ConvArgs a = a_arg;
    a.in = in_arg; a.out = out_arg; a.bias = bias_arg; a.in_ch = in_ch_arg; a.out_ch = out_ch_arg; a.length = length_arg;
    a.kernel = kernel_arg; a.dilation = dilation_arg;
    conv_tile<WM, WN, KF, FUSED>(a, ConvBlocks{weights_arg, tiles_arg, (a.in_ch + 15) / 16}, &conv_kernarg<ConvKernarg>()->a, lds, s_rows);
}

// The same product for short rows (few positions, many channels: the codec's first stages), where 64 x 128 tiles would
// leave most of the chip idle: a workgroup owns a 32 x 64 tile and its four wavefronts split the input channels between
// them (wavefront w takes blocks w, w + 4, ... of sixteen channels), each staging its own blocks in its own
// part of LDS; the four partial tiles are added in wavefront order at the end, so the result does not depend on timing.
// NT: 32-position halves per tile (2, or 1 for the very shortest rows: twice the workgroups).
// PARTS: positions of the window a lane stages (2 while the window is no longer than 128: the third costs 16 registers).
// a.splits > 1: that many workgroups share the tile's channels (wavefront w of workgroup s is wavefront 4 s + w of them all), each
// leaves its sum in a.parts, and k_conv_finish adds them in order and does what is left.
template <int KF, int NT, int PARTS>
__device__ __forceinline__ void conv_split_tile(const ConvArgs &a_arg, const ConvBlocks &w_arg, const ConvArgs *const again, uint4 *const lds, ConvTileRows &s_rows) {
    constexpr int TM = 32, TN = 32 * NT;
    ConvArgs a = a_arg;
    if constexpr (KF != 0) a.kernel = KF;
    const int halo = (a.kernel - 1) * a.dilation;
    const int win = TN + halo;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int kPitch = conv_split_pitch(NT, PARTS);
    uint4 *s_in = lds + wave * (6 * kPitch);   // [piece][eight channels][position] of this wavefront
    const int split = (int)blockIdx.x % a.splits, sharing = 4 * a.splits, rank = 4 * split + wave;   // this wavefront among those that share the channels
    const int m0 = blockIdx.y * TM, t0 = (int)blockIdx.x / a.splits * TN;
    const int half = lane >> 5, col = lane & 31;

    floatx16 acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[n] = floatx16{0};
    // what the finished rows need (behind the products each request would be a round trip of its own)
    if (tid < TM) {
        const int m = m0 + tid;
        const float al = a.activate && m < a.snake_channels ? a.alpha[m] : 0.0f;
        s_rows.bias[tid] = a.bias != nullptr && m < a.out_ch ? a.bias[m] : 0.0f;
        s_rows.alpha[tid] = al;
        s_rows.inverse_alpha[tid] = 1.0f / (al + 1e-9f);
    }
    const int mine = (w_arg.blocks - rank + sharing - 1) / sharing;   // this wavefront's blocks
    if (mine > 0) {
        ConvColumn column[2][PARTS];
        const int first = max(t0 - halo, 0);
        unsigned from[PARTS];   // see conv_tile
#pragma unroll
        for (int x = 0; x < PARTS; ++x) from[x] = (unsigned)(min(max(t0 - halo + lane + 64 * x, 0), a.length - 1) - first) * 4;
        const auto fetch = [&](int i) {
#pragma unroll
            for (int x = 0; x < PARTS; ++x)
                if (64 * x < win) {   // (the same for every lane)
#pragma unroll
                    for (int g = 0; g < 2; ++g)
                        column[g][x].request(a.in + first, 16 * (sharing * i + rank) + 8 * g, a.in_ch, a.length, from[x]);
                }
        };
        const size_t per_block = (size_t)a.kernel * 192;
        // (no workgroup barrier in the loop: a wavefront stages into its own part of LDS and reads nothing else, and its own
        // LDS accesses complete in the order it issued them -- the four wavefronts walk their channel blocks independently)
        const auto stage = [&](int i) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
            for (int x = 0; x < PARTS; ++x) {
                const int p = lane + 64 * x;
                if (p < win) {
#pragma unroll
                    for (int g = 0; g < 2; ++g) column[g][x].store(s_in + g * kPitch + p, 2 * kPitch, t0 - halo + p >= 0);
                }
            }
            fetch(min(i + 1, mine - 1));   // in flight during this block's products
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            return const_cast<const uint4 *>(s_in + half * kPitch + col);
        };
        fetch(0);
        ConvWeights w(w_arg.data + ((size_t)blockIdx.y * w_arg.blocks + rank) * per_block, lane, (size_t)(sharing - 1) * per_block, mine, a.kernel);
        conv_products<KF, NT, 2 * kPitch>(w, a.kernel, a.dilation, mine, stage, acc);
    }
    // A thread finishes the tile's values at (row wave + 4 j, position lane): a store instruction then covers one row's 64
    // consecutive positions and whether the row exists is the same for all its lanes (in the accumulators' order an
    // instruction covers halves of two rows, four apart).  e: where that value sits in a partial tile (element r of lane l).
    // Residuals are requested here, side by side, before the wavefronts meet, and the activation is straight-line code for all eight values: in
    // a loop a value at a time, with the requests where they are used, the finish was 7,000 to 9,000 cycles (108 channels x 1280).
    const int pos = lane, t = t0 + pos;
    const bool t_ok = (NT > 1 || pos < 32) && t < a.length;
    float first[8], second[8];
    const auto at = [&](int j) { return (size_t)min(m0 + wave + 4 * j, a.out_ch - 1) * a.length + min(t, a.length - 1); };
    if (a.residual != nullptr && a.splits == 1) {
#pragma unroll
        for (int j = 0; j < 8; ++j) first[j] = a.residual[at(j)];
        if (a.residual2 != nullptr) {
#pragma unroll
            for (int j = 0; j < 8; ++j) second[j] = a.residual2[at(j)];
        }
    }
    __syncthreads();   // the partial tiles below overwrite every wavefront's staging area
    // partial tiles through LDS: [wavefront][element r][lane], then ((p0 + p1) + p2) + p3 + bias
    float *s_part = reinterpret_cast<float *>(lds);
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) s_part[(wave * 32 + 16 * n + r) * 64 + lane] = acc[n][r];
    __syncthreads();
    float sum[8], zero = 0.0f;
    const auto add_parts = [&]() {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int row = wave + 4 * j;
            const int e = ((((row >> 3) << 2) | (row & 3)) + 16 * (pos >> 5)) * 64 + ((row >> 2) & 1) * 32 + (pos & 31);
            sum[j] = ((s_part[e] + s_part[2048 + e]) + s_part[4096 + e]) + s_part[6144 + e];
            zero = __builtin_fmaf(sum[j], 0.0f, zero);
        }
    };
    add_parts();
    if (__builtin_expect(__any(t_ok && zero != 0.0f), 0)) {   // (see split_all_finite)
        if (t_ok) conv_split_rest(again, s_part, split, m0, t);
        add_parts();
    }
    const int rows = min(TM, a.out_ch - m0);   // rows wave + 4 j below it exist
    if (a.splits > 1) {
        if (!t_ok) return;
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (wave + 4 * j < rows) a.parts[((size_t)split * a.out_ch + m0 + wave + 4 * j) * a.length + t] = sum[j];
        return;
    }
    // conv_combine's operations
    float value[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) value[j] = sum[j] + s_rows.bias[wave + 4 * j];
    if (a.residual != nullptr) {
#pragma unroll
        for (int j = 0; j < 8; ++j) value[j] = first[j] + value[j];
        if (a.residual2 != nullptr) {
#pragma unroll
            for (int j = 0; j < 8; ++j) value[j] = second[j] + value[j];
        }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) value[j] = value[j] * a.scale;
    float *const out = a.out + (size_t)(m0 + wave) * a.length + t;
    const size_t step = (size_t)4 * a.length;
    if (!a.activate) {
        if (t_ok) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (wave + 4 * j < rows) out[j * step] = value[j];
        }
        return;
    }
    float al[8], act[8];
    bool large = false;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        al[j] = s_rows.alpha[wave + 4 * j];
        act[j] = value[j] < 0.0f ? value[j] * 0.01f : value[j];
        large = large || !(fabsf(al[j] * value[j]) < kShortSineLimit);
    }
    if (__builtin_expect(!__any(t_ok && large), 1)) {
        if (m0 < a.snake_channels) {   // (else no row of the tile is a snake row)
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float sn = short_sine(al[j] * value[j]), y = value[j] + sn * sn * s_rows.inverse_alpha[wave + 4 * j];
                act[j] = m0 + wave + 4 * j < a.snake_channels ? y : act[j];
            }
        }
        if (t_ok) {
            float *const act_out = a.act_out != nullptr ? a.act_out + (size_t)(m0 + wave) * a.length + t : out;
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (wave + 4 * j < rows) {
                    if (a.act_out != nullptr) out[j * step] = value[j];
                    act_out[j * step] = act[j];
                }
        }
        return;
    }
    // some argument needs the library's sine: the values go through LDS (a thread reads what it wrote, behind the partial tiles, which other
    // wavefronts may still read) so that one copy of that routine serves the eight of them
    s_part += 4 * 2048;
#pragma unroll
    for (int j = 0; j < 8; ++j) s_part[tid + 256 * j] = value[j];
#pragma unroll 1
    for (int j = 0; j < 8; ++j) {
        const int row = wave + 4 * j, m = m0 + row;
        if (t_ok && row < rows) conv_emit(a, m, (size_t)m * a.length + t, s_part[tid + 256 * j], s_rows.alpha[row], s_rows.inverse_alpha[row]);
    }
}

template <int KF, int NT, int PARTS>
__global__ void __launch_bounds__(256, 2) k_conv1d_split(const float *const in_arg, float *const out_arg, const uint4 *const weights_arg, const float *const bias_arg, const int in_ch_arg,
                                                         const int out_ch_arg, const int length_arg, const int kernel_arg, const int dilation_arg, const int tiles_arg,
                                                         const ConvArgs a_arg) {
    extern __shared__ __align__(16) uint4 lds[];
    __shared__ ConvTileRows s_rows;
    // (leading scalar arguments: see k_conv1d)
    ConvArgs a = a_arg;
    a.in = in_arg; a.out = out_arg; a.bias = bias_arg; a.in_ch = in_ch_arg; a.out_ch = out_ch_arg; a.length = length_arg;
    a.kernel = kernel_arg; a.dilation = dilation_arg;
    conv_split_tile<KF, NT, PARTS>(a, ConvBlocks{weights_arg, tiles_arg, (a.in_ch + 15) / 16}, &conv_kernarg<ConvKernarg>()->a, lds, s_rows);
}

// Several convolutions of one shape side by side in one launch (the three branches of a residual layer: same rows in and
// out, own weights, taps, dilation and epilogue): blockIdx.z names the convolution, every workgroup runs the tile's work of
// its own, so the values are those of the single launches.  A launch's fixed cost (dispatch, kernel start, the first
// block's round trip, the stores behind the last product) is paid once for all of them, and a CU holds workgroups of
// different convolutions whose staging and products overlap.  Tap counts 3, 7 and 11 only (the builds with straight-line
// products); always the build with the fused epilogue (with nothing to add it leaves the product's own bits).
constexpr int kConvBatchMax = 4;
constexpr int kConvMaxSplits = 8;
struct ConvBatchArgs {
    ConvArgs item[kConvBatchMax];
    int order[kConvBatchMax];   // blockIdx.z -> member (order_members)
};

__device__ __forceinline__ ConvBlocks conv_blocks(const ConvArgs &a) { return ConvBlocks{a.weights, (a.out_ch + 31) / 32, (a.in_ch + 15) / 16}; }

template <int WM, int WN>
__global__ void __launch_bounds__(256, 3) k_conv1d_batch(const ConvBatchArgs b) {
    extern __shared__ __align__(16) uint4 lds[];
    __shared__ ConvTileRows s_rows;
    const int z = b.order[blockIdx.z];
    switch (b.item[z].kernel) {
        case 3: conv_tile<WM, WN, 3, true>(b.item[z], conv_blocks(b.item[z]), &conv_kernarg<ConvBatchArgs>()->item[z], lds, s_rows); break;
        case 7: conv_tile<WM, WN, 7, true>(b.item[z], conv_blocks(b.item[z]), &conv_kernarg<ConvBatchArgs>()->item[z], lds, s_rows); break;
        default: conv_tile<WM, WN, 11, true>(b.item[z], conv_blocks(b.item[z]), &conv_kernarg<ConvBatchArgs>()->item[z], lds, s_rows); break;
    }
}

template <int NT, int PARTS>
__global__ void __launch_bounds__(256, 2) k_conv1d_split_batch(const ConvBatchArgs b) {
    extern __shared__ __align__(16) uint4 lds[];
    __shared__ ConvTileRows s_rows;
    const int z = b.order[blockIdx.z];
    switch (b.item[z].kernel) {
        case 3: conv_split_tile<3, NT, PARTS>(b.item[z], conv_blocks(b.item[z]), &conv_kernarg<ConvBatchArgs>()->item[z], lds, s_rows); break;
        case 7: conv_split_tile<7, NT, PARTS>(b.item[z], conv_blocks(b.item[z]), &conv_kernarg<ConvBatchArgs>()->item[z], lds, s_rows); break;
        default: conv_split_tile<11, NT, PARTS>(b.item[z], conv_blocks(b.item[z]), &conv_kernarg<ConvBatchArgs>()->item[z], lds, s_rows); break;
    }
}

// What is left of convolutions whose channels several workgroups shared: their sums in order, the bias, and the epilogue.
__global__ void __launch_bounds__(256) k_conv_finish(const ConvBatchArgs b) {
    const ConvArgs &a = b.item[blockIdx.z];
    const int t = (int)blockIdx.x * 256 + (int)threadIdx.x, m = (int)blockIdx.y;
    if (t >= a.length) return;
    const size_t index = (size_t)m * a.length + t, set = (size_t)a.out_ch * a.length;
    float part[kConvMaxSplits];
#pragma unroll
    for (int s = 0; s < kConvMaxSplits; ++s) part[s] = a.parts[index + (size_t)min(s, a.splits - 1) * set];   // (side by side, under no condition)
    const bool snake_row = a.activate && m < a.snake_channels;
    const float al = snake_row ? a.alpha[m] : 0.0f, bias = a.bias != nullptr ? a.bias[m] : 0.0f;
    float sum = part[0];
#pragma unroll
    for (int s = 1; s < kConvMaxSplits; ++s)
        if (s < a.splits) sum += part[s];
    conv_emit(a, m, index, conv_combine(a, index, sum + bias), al, 1.0f / (al + 1e-9f));
}

// ---- a residual block in one launch ---------------------------------------------------------------------------------------
// out = x + conv_skip(snake(conv_in(snake(x)))) for up to four branches of a residual layer side by side, up to 128 channels: what
// would be two launches and, between them and around them, three row sets written and read again.  A workgroup takes all rows of a
// window of 64 * WN positions of the inner rows r = snake(conv_in(snake(x))), (taps - 1) more than the positions it finishes:
// it stages snake(x) (a position and its halo are activated once, since every row is here), multiplies, activates, leaves the
// pieces of r in LDS over the stages, and multiplies again from there.  Every value is the separate calls' arithmetic in their
// order: the same bits.  SPLIT: the order of the channel-split tiles, whose four wavefronts take a block of channels each up to
// 64 channels -- a block's sums from zero, added block after block, then the bias; else that of the large tiles, one chain from the bias.
struct ResMember {
    const float *in;                      // [channels, length]
    float *out;
    const float2 *snake_in, *snake_skip;  // (alpha, 1 / (alpha + 1e-9)) of the first snake_channels rows
    const uint4 *w_in, *w_skip;           // ConvBlocks data
    const float *b_in, *b_skip;           // or null
    int kernel, dilation;
};
constexpr int kResMaxChannels = 128, kResMaxReach = 64;
struct ResArgs {
    ResMember member[kConvBatchMax];
    int order[kConvBatchMax];
    int channels, length, snake_channels, blocks, tiles;
};

// The block's channels: (alpha, 1 / (alpha + 1e-9), a bound, -) of the inner rows' half-snake, and the biases of both convolutions.
struct ResRows {
    float4 pair[kResMaxChannels];
    float in[kResMaxChannels], skip[kResMaxChannels];
};

template <int WM, int WN, int NT, bool SPLIT, int KF>
__device__ __forceinline__ void res_block_tile(const ResArgs &a, const ResMember &m, uint4 *const lds, ResRows &s_rows) {
    constexpr int WP = 32 * NT, RN = WP * WN, T = 64 * WM * WN, TN = RN - (KF - 1), kPitch = RN + kResMaxReach;
    const int t0 = blockIdx.x * TN;
    if (t0 >= a.length) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = lane >> 5, col = lane & 31;
    const int wm = wave / WN, wn = wave % WN;
    const int halo = (KF - 1) * m.dilation, win = RN + halo;
    const int first = t0 - (KF - 1) - halo;   // position of the window's first column

    // staging: columns (a position, eight channels) of a thread; a wavefront's columns are of one half of a block's channels.  Up to
    // T / 2 positions: a thread takes one column, the workgroup's halves the two halves of the channels; else one of each half, the
    // second half a workgroup apart, and (windows of more than T positions) the first 128 threads a third.
    constexpr int kReach = RN + kResMaxReach, kColumns = kReach <= T / 2 ? 1 : kReach <= T ? 2 : 3;
    static_assert(kReach <= T + 64 && (kColumns == 1 || T == 256), "columns cover the window");
    int place[kColumns];
    const auto group_of = [&](int x) { return kColumns == 1 ? wave / (T / 128) : x < 2 ? x : wave & 1; };
#pragma unroll
    for (int x = 0; x < kColumns; ++x) {
        const int p = kColumns == 1 ? tid & (T / 2 - 1) : x == 0 ? tid : x == 1 ? (kColumns == 2 ? (tid + 128) & 255 : tid) : tid < 128 ? 256 + (tid & 63) : win;
        place[x] = p < win ? p : -1;
    }
    float column[kColumns][8];
    const auto fetch = [&](int block) {
#pragma unroll
        for (int x = 0; x < kColumns; ++x) {
            const int channel = opaque_scalar(16 * block + 8 * group_of(x));
            const int origin = max(first, 0);
            const unsigned bytes = opaque((unsigned)(min(max(first + max(place[x], 0), 0), a.length - 1) - origin) * 4);   // (never in front of origin)
            request_rows(column[x], m.in + origin, channel, a.channels, a.length, bytes);
        }
    };
    const auto publish = [&](int block, uint4 *stage) {
#pragma unroll
        for (int x = 0; x < kColumns; ++x) {
            if (place[x] < 0) continue;
            const int channel = 16 * block + 8 * group_of(x);
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = column[x][e];
            // (one branch for the eight channels, which are the same for every lane: their alphas come in one request, their sines side by side)
            if (channel < a.snake_channels) {
                float2 pair[8];
                float argument[8], most = 0.0f;
#pragma unroll
                for (int e = 0; e < 8; ++e) pair[e] = m.snake_in[channel + e < a.snake_channels ? channel + e : channel];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    argument[e] = pair[e].x * v[e];
                    most = fmaxf(most, fabsf(argument[e]));   // (of a row without a sine, too: the long way gives its value as well)
                }
                if (__builtin_expect(!__any(most >= kShortSineLimit), 1)) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float sn = short_sine(argument[e]), y = v[e] + sn * sn * pair[e].y;
                        v[e] = channel + e < a.snake_channels ? y : v[e] < 0.0f ? v[e] * 0.01f : v[e];
                    }
                } else {
#pragma unroll 1
                    for (int e = 0; e < 8; ++e) {
                        const bool snake_row = channel + e < a.snake_channels;
                        const float2 p = snake_row ? m.snake_in[channel + e] : make_float2(0.0f, 0.0f);
                        v[e] = half_snake(v[e], snake_row, p.x, p.y);
                    }
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = v[e] < 0.0f ? v[e] * 0.01f : v[e];
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = first + place[x] < 0 ? 0.0f : v[e];   // in front of the rows
            store_pieces(v, stage + group_of(x) * kPitch + place[x], 2 * kPitch);
        }
    };
    // the inner rows' alphas, 1 / (alpha + 1e-9), and what a value is multiplied by to be told from those that need the long way: the
    // library's sine, or (no finite number, or none that three pieces add up to) more than that; an infinite 1 / (alpha + 1e-9) sends all that way.
    // (Requested here, looked at behind the first block's requests.)
    constexpr int kRowsEach = (kResMaxChannels + T - 1) / T;
    float2 row_pair[kRowsEach];
    float row_in[kRowsEach], row_skip[kRowsEach];
#pragma unroll
    for (int i = 0; i < kRowsEach; ++i) {
        const int c = tid + T * i;
        const bool there = c < a.channels;   // (else zero: a wavefront without a row tile of its own multiplies the last one's weights)
        row_pair[i] = c < a.snake_channels ? m.snake_skip[c] : make_float2(0.0f, 0.0f);
        row_in[i] = there && m.b_in != nullptr ? m.b_in[c] : 0.0f;
        row_skip[i] = there && m.b_skip != nullptr ? m.b_skip[c] : 0.0f;
    }
    const auto keep_rows = [&]() {
#pragma unroll
        for (int i = 0; i < kRowsEach; ++i) {
            const int c = tid + T * i;
            if (c >= kResMaxChannels) break;
            const float2 pair = row_pair[i];
            const float bound = fmaxf(fabsf(pair.x), 1.01f * (kShortSineLimit / kSplitLimit));
            s_rows.pair[c] = make_float4(pair.x, pair.y, split_finite(pair.y) ? bound : __builtin_inff(), 0.0f);
            s_rows.in[c] = row_in[i];
            s_rows.skip[c] = row_skip[i];
        }
    };

    f32x16 acc[NT], sum[SPLIT ? NT : 1];
    const auto start = [&](const float (&bias)[kResMaxChannels]) {
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            if constexpr (SPLIT) {
                acc[n] = f32x16{0};
                sum[n] = f32x16{0};
            } else {
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[n][r] = bias[wm * 32 + split_acc_row(r, lane)];
            }
        }
    };
    // (SPLIT) a block's sums to those of the blocks before it; in the end, the bias
    const auto add_block = [&]() {
        if constexpr (SPLIT) {
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                sum[n] += acc[n];
                acc[n] = f32x16{0};
            }
        }
    };
    const auto finish = [&](const float (&bias)[kResMaxChannels]) {
        add_block();
        if constexpr (SPLIT) {
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[n][r] = sum[n][r] + bias[wm * 32 + split_acc_row(r, lane)];
        }
    };
    const size_t w_at = (size_t)min(wm, a.tiles - 1) * a.blocks * KF * 192;
    uint4 *stage_now = lds, *stage_next = lds + 6 * kPitch;
    fetch(0);
    ConvWeights w(m.w_in + w_at, lane, 0, 1, KF);
    keep_rows();
    publish(0, stage_now);
    fetch(min(1, a.blocks - 1));
    __syncthreads();
    start(s_rows.in);
    conv_products<KF, NT, 2 * kPitch, true>(w, KF, m.dilation, a.blocks, [&](int block) {
        if (block > 0) add_block();
        __syncthreads();
        const uint4 *at = stage_now + half * kPitch + wn * WP + col;
        if (block + 1 < a.blocks) {
            publish(block + 1, stage_next);
            fetch(min(block + 2, a.blocks - 1));
        }
        uint4 *t = stage_now;
        stage_now = stage_next;
        stage_next = t;
        return at;
    }, acc);
    finish(s_rows.in);
    bool large = false, kept = false;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const float bound = s_rows.pair[wm * 32 + split_acc_row(r, lane)].z;
#pragma unroll
        for (int n = 0; n < NT; ++n) large = large || !(fabsf(bound * acc[n][r]) < kShortSineLimit);
    }
    if (__builtin_expect(!__any(large), 1)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = wm * 32 + split_acc_row(r, lane);
            const float4 pair = s_rows.pair[row];
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                const float v = acc[n][r];
                float y = v < 0.0f ? v * 0.01f : v;
                if (wm * 32 + 8 * (r >> 2) < a.snake_channels) {   // (else no lane's row of these registers is a snake row)
                    const float sn = short_sine(pair.x * v);
                    y = row < a.snake_channels ? v + sn * sn * pair.y : y;
                }
                acc[n][r] = y;
            }
        }
    } else {
#pragma unroll 1
        for (int r = 0; r < 16; ++r) {
            const int row = wm * 32 + split_acc_row(r, lane);
            const float4 pair = s_rows.pair[row];
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                const int t = t0 - (KF - 1) + wn * WP + 32 * n + col;
                float v = acc[n][r];
                if (row < a.channels && t >= 0 && t < a.length && !split_finite(SPLIT ? sum[SPLIT ? n : 0][r] : v)) {
                    const float bias = s_rows.in[row];
                    v = conv_chain(conv_row(m.w_in, a.blocks, KF, row), a.channels, KF, [](int) { return true; }, [&](int tap) { return t - halo + tap * m.dilation >= 0; },
                                   [&](int c, int tap, float (&x)[8]) {
#pragma unroll 1
                                       for (int e = 0; e < 8; ++e) {
                                           const int channel = min(c + e, a.channels - 1);
                                           const float2 in_pair = channel < a.snake_channels ? m.snake_in[channel] : make_float2(0.0f, 0.0f);
                                           x[e] = half_snake(m.in[(size_t)channel * a.length + t - halo + tap * m.dilation], channel < a.snake_channels, in_pair.x, in_pair.y);
                                       }
                                   }, SPLIT ? 0.0f : bias);
                    if (SPLIT) v = v + bias;
                }
                v = row < a.channels ? half_snake(v, row < a.snake_channels, pair.x, pair.y) : 0.0f;
                kept = kept || !(fabsf(v) < kSplitLimit);
                acc[n][r] = v;
            }
        }
        kept = __any(kept);
    }
    // the finished rows' residual (x itself), on its way during the rest: whole rows of consecutive positions, as it is stored
    const int rows = min(32, a.channels - wm * 32);
    constexpr int kRowsAtOnce = 64 / WP;                 // rows a wavefront stores with one instruction
    const int row0 = lane / WP, p_out = wn * WP + lane % WP, t_out = t0 + p_out;
    const size_t at_out = (size_t)(rows > 0 ? wm * 32 : 0) * a.length + min(t_out, a.length - 1);
    float x[32 / kRowsAtOnce];
#pragma unroll
    for (int i = 0; i < 32 / kRowsAtOnce; ++i) x[i] = m.in[at_out + (size_t)max(min(row0 + kRowsAtOnce * i, rows - 1), 0) * a.length];
    // the inner rows: activated, zero in front of the first position, in pieces to LDS where the second convolution reads them
    ConvWeights w2(m.w_skip + w_at, lane, 0, 1, KF);
    __syncthreads();   // the stages have been read
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int p = wn * WP + 32 * n + col;
        const bool in_front = t0 - (KF - 1) + p < 0;
#pragma unroll
        for (int g = 0; g < 4; ++g) {   // rows 8 g + 4 half .. + 3 of the tile: half of the eight channels of one place
            const int block = wm * 2 + (g >> 1);
            if (block >= a.blocks) continue;
            const float4 v = make_float4(acc[n][4 * g], acc[n][4 * g + 1], acc[n][4 * g + 2], acc[n][4 * g + 3]);
            SplitFour s(in_front ? make_float4(0.0f, 0.0f, 0.0f, 0.0f) : v);
            if (__builtin_expect(kept, 0) && !in_front) s.keep_bits(v);   // (the rows themselves are nowhere else)
#pragma unroll
            for (int q = 0; q < 3; ++q) reinterpret_cast<uint2 *>(&lds[(block * 6 + q * 2 + (g & 1)) * RN + p])[half] = s.piece[q];
        }
    }
    start(s_rows.skip);
    __syncthreads();
    conv_products<KF, NT, 2 * RN, true>(w2, KF, 1, a.blocks, [&](int block) {
        if (block > 0) add_block();
        return const_cast<const uint4 *>(lds + (block * 6 + half) * RN + wn * WP + col);
    }, acc);
    finish(s_rows.skip);
    bool finite;
    if constexpr (SPLIT) finite = split_all_finite(sum);
    else finite = split_all_finite(acc);
    if (__builtin_expect(!finite, 0)) {
#pragma unroll 1
        for (int r = 0; r < 16; ++r) {
            const int row = wm * 32 + split_acc_row(r, lane);
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                const int p = wn * WP + 32 * n + col, t = t0 + p;
                if (row >= a.channels || p >= TN || t >= a.length || split_finite(SPLIT ? sum[SPLIT ? n : 0][r] : acc[n][r])) continue;
                const float bias = s_rows.skip[row];
                const float v = conv_chain(conv_row(m.w_skip, a.blocks, KF, row), a.channels, KF, [](int) { return true; },
                                           [&](int tap) { return t - (KF - 1) + tap >= 0; },
                                           [&](int c, int tap, float (&x)[8]) {
                                               const uint4 *const at = lds + ((c >> 4) * 6 + ((c >> 3) & 1)) * RN + p + tap;
                                               const ushort8 xh = __builtin_bit_cast(ushort8, at[0]), xm = __builtin_bit_cast(ushort8, at[2 * RN]),
                                                             xl = __builtin_bit_cast(ushort8, at[4 * RN]);
#pragma unroll
                                               for (int e = 0; e < 8; ++e) x[e] = split_value(xh[e], xm[e], xl[e]);
                                           }, SPLIT ? 0.0f : bias);
                acc[n][r] = SPLIT ? v + bias : v;
            }
        }
    }

    // + x, and out, in whole rows (see store_tile of conv_tile)
    __syncthreads();   // the inner rows have been read
    constexpr int kRowPitch = WP + 1;
    float *const s_tile = reinterpret_cast<float *>(lds) + wave * (32 * kRowPitch);
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) s_tile[split_acc_row(r, lane) * kRowPitch + 32 * n + col] = acc[n][r];
    if (rows <= 0 || p_out >= TN || t_out >= a.length) return;
#pragma unroll
    for (int i = 0; i < 32 / kRowsAtOnce; ++i) {
        const int row = row0 + kRowsAtOnce * i;
        if (row < rows) m.out[at_out + (size_t)row * a.length] = x[i] + s_tile[row * kRowPitch + lane % WP];
    }
}

template <int WM, int WN, int NT, bool SPLIT>
__global__ void __launch_bounds__(64 * WM * WN, 2) k_res_block(const ResArgs a) {
    extern __shared__ __align__(16) uint4 lds[];
    __shared__ ResRows s_rows;
    const int z = a.order[blockIdx.y];
    switch (a.member[z].kernel) {
        case 3: res_block_tile<WM, WN, NT, SPLIT, 3>(a, a.member[z], lds, s_rows); break;
        case 7: res_block_tile<WM, WN, NT, SPLIT, 7>(a, a.member[z], lds, s_rows); break;
        default: res_block_tile<WM, WN, NT, SPLIT, 11>(a, a.member[z], lds, s_rows); break;
    }
}

// The order in which a launch's members start, `each` workgroups apiece.  Workgroups are dealt to the CUs in turn, so member p of the order
// covers CUs p * each .. on, round and round: the order whose most loaded CU has the fewest taps, and of equal ones the one that starts the most
// taps first (a long workgroup is not started last).  Taps 3 / 7 / 11, us a layer of three positions, most taps first / this order: 432
// channels x 512 (112 workgroups each) 240 / 225, 216 x 1024 (112) 140 / 129, 108 x 8192 (128) 237 / 216; where nothing is gained it is the same
// order, and another is slower: 108 x 12288 (192) 318 / 325, 432 x 320 (140) 181 / 195.  With one or two workgroups of each member for every CU, and
// more members than two, the second one by its taps goes first: 108 x 4096 (256) 154 / 136, 216 x 2560 (280) 265 / 260, x 4096 (448) 360 / 350.
void order_members(const State *st, const int *taps, int count, long each, int *order) {
    int by_taps[kConvBatchMax], at[kConvBatchMax], best = INT_MAX;
    for (int i = 0; i < count; ++i) {
        int j = i;
        for (; j > 0 && taps[by_taps[j - 1]] < taps[i]; --j) by_taps[j] = by_taps[j - 1];
        by_taps[j] = i;
    }
    const long cus = st->cu_count, rest = each % cus;
    if (each >= cus && each < 2 * cus && count > 2) {
        std::swap(by_taps[0], by_taps[1]);
        for (int i = 0; i < count; ++i) order[i] = by_taps[i];
        return;
    }
    int permutations = 1;
    for (int i = 2; i <= count; ++i) permutations *= i;
    for (int p = 0; p < permutations; ++p) {   // (the first one is by_taps itself)
        bool used[kConvBatchMax] = {};
        for (int i = 0, code = p, base = permutations; i < count; ++i) {
            base /= count - i;
            int skip = code / base, k = 0;
            code %= base;
            for (; used[k] || skip > 0; ++k) skip -= used[k] ? 0 : 1;
            used[k] = true;
            at[i] = by_taps[k];
        }
        int most = 0;   // a CU's taps beyond those that every CU has: highest where some member's last round begins
        for (int i = 0; i < count; ++i) {
            const long cu = i * each % cus;
            int load = 0;
            for (int j = 0; j < count; ++j) load += (cu - j * each % cus + cus) % cus < rest ? taps[at[j]] : 0;
            most = load > most ? load : most;
        }
        if (most < best) {
            best = most;
            for (int i = 0; i < count; ++i) order[i] = at[i];
        }
    }
}
void order_members(const State *st, ConvBatchArgs &b, int count, long each) {
    int taps[kConvBatchMax];
    for (int i = 0; i < count; ++i) taps[i] = b.item[i].kernel;
    order_members(st, taps, count, each, b.order);
}

template <int WM, int WN, int NT, bool SPLIT = false>
int launch_res_block(State *st, ResArgs &a, int count, char *error, size_t capacity) {
    constexpr int RN = 32 * NT * WN;
    int taps = 0;
    for (int i = 0; i < count; ++i) taps = a.member[i].kernel > taps ? a.member[i].kernel : taps;
    size_t lds = (size_t)2 * 6 * (RN + kResMaxReach) * 16;                             // two stages, or
    const size_t inner = ((size_t)a.blocks * 6 * RN + 16) * 16;                        // the inner rows (a tap past the last place is read, not used), or
    const size_t tiles = (size_t)WM * WN * 32 * (32 * NT + 1) * sizeof(float);        // the finished tiles
    lds = inner > lds ? inner : lds;
    lds = tiles > lds ? tiles : lds;
    static std::atomic<bool> raised{false};   // per instantiation; states on separate threads meet here
    if (!raised) {
        MYNAH_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_res_block<WM, WN, NT, SPLIT>), hipFuncAttributeMaxDynamicSharedMemorySize, 112 * 1024));
        raised = true;
    }
    const int finished = RN - (taps - 1), each = (a.length + finished - 1) / finished;
    int kernels[kConvBatchMax];
    for (int i = 0; i < count; ++i) kernels[i] = a.member[i].kernel;
    order_members(st, kernels, count, each, a.order);
    hipLaunchKernelGGL((k_res_block<WM, WN, NT, SPLIT>), dim3((unsigned)each, (unsigned)count), dim3(64 * WM * WN), lds, st->stream, a);
    return hip_check(hipGetLastError(), "residual block launch", error, capacity);
}

__global__ void __launch_bounds__(256) k_conv_pack(const float *src, uint4 *dst, size_t count, int out_ch, int in_ch, int kernel, int blocks) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= count) return;
    const int lane = (int)(i & 63);
    const size_t step = i >> 6, tile = step / ((size_t)blocks * kernel);
    const int tap = (int)(step % (size_t)kernel), block = (int)(step / (size_t)kernel % (size_t)blocks);
    const size_t o = tile * 32 + (lane & 31);
    const int c0 = block * 16 + (lane >> 5) * 8;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = o < (size_t)out_ch && c0 + e < in_ch ? src[(o * in_ch + c0 + e) * kernel + tap] : 0.0f;
    bf16x8 p[3];
    split_eight(make_float4(v[0], v[1], v[2], v[3]), make_float4(v[4], v[5], v[6], v[7]), p);
    ushort8 at[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) at[q] = __builtin_bit_cast(ushort8, p[q]);
#pragma unroll
    for (int e = 0; e < 8; ++e) {   // (the kernels have no other copy of a weight)
        unsigned short h = at[0][e], m = at[1][e], l = at[2][e];
        split_keep_bits(v[e], h, m, l);
        at[0][e] = h;
        at[1][e] = m;
        at[2][e] = l;
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) dst[step * 192 + q * 64 + lane] = __builtin_bit_cast(uint4, at[q]);
}

struct ConvTransposeArgs {
    const float *in;     // [in_ch, length]
    float *out;          // [out_ch, output_length]
    const float *w;      // [in_ch, out_ch / groups, kernel]
    const float *bias;   // [out_ch] or null
    int in_ch, out_ch, length, output_length, kernel, stride, groups;
};

// Grids over rows: 256 threads along a row (no thread divides its index by the length, in 64 bits), at most 65535 channels side by
// side, each workgroup taking every 65535th.
constexpr unsigned kRowsSideBySide = 65535;
inline dim3 row_grid(size_t channels, size_t threads) {
    return dim3((unsigned)((threads + 255) / 256), (unsigned)(channels < kRowsSideBySide ? channels : kRowsSideBySide));
}
// S: the stride where it is 2, 4 or 8 and the kernel between one and two strides (the codec's): a thread finishes the S positions that begin at its
// input position, from that input and the one before it, with weights that are the same for all threads (scalar requests), and stores them
// together where `aligned`.  0: any shape, a thread per position.  us, the one / the other: 27 channels x 65536 7.9 / 11.8, 54 x 32768 7.8 / 11.7,
// 108 x 16384 5.8 / 11.7, 216 x 4096 5.0 / 6.9, 432 x 512 4.7 / 4.7, 27 x 5120 3.5 / 3.8 (requests of one input channel at a time: 3.9 and, with 8
// positions a thread, 5.3).
template <int S>
__global__ void __launch_bounds__(256) k_conv_transpose(const ConvTransposeArgs a, const int aligned) {
    const int ipg = a.in_ch / a.groups, opg = a.out_ch / a.groups;
    const unsigned first = blockIdx.x * 256u + threadIdx.x;
    for (unsigned channel = blockIdx.y; channel < (unsigned)a.out_ch; channel += gridDim.y) {
        const int o = (int)channel, group = o / opg, o_local = o - group * opg;
        const float bias = a.bias != nullptr ? a.bias[o] : 0.0f;
        float *const out = a.out + (size_t)o * a.output_length;
        if constexpr (S != 0) {
            const size_t p = (size_t)first * S;
            if (p >= (size_t)a.output_length) return;
            const bool have_now = first < (unsigned)a.length, have_before = first > 0u;   // (first <= length: the output ends there)
            float value[S];
#pragma unroll
            for (int k = 0; k < S; ++k) value[k] = bias;
            for (int i = group * ipg; i < (group + 1) * ipg; i += 2) {   // two input channels' requests side by side, then their sums
                float now[2], before[2], w_now[2][S], w_before[2][S];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int c = min(i + u, (group + 1) * ipg - 1);
                    const float *const row = a.in + (size_t)c * a.length, *const w = a.w + ((size_t)c * opg + o_local) * a.kernel;
                    now[u] = row[min(first, (unsigned)a.length - 1u)];
                    before[u] = row[have_before ? first - 1u : 0u];
#pragma unroll
                    for (int k = 0; k < S; ++k) {
                        w_now[u][k] = w[k];
                        w_before[u][k] = w[min(k + S, a.kernel - 1)];
                    }
                }
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const bool there = i + u < (group + 1) * ipg;
#pragma unroll
                    for (int k = 0; k < S; ++k) {
                        const float earlier = value[k] + before[u] * w_before[u][k];
                        value[k] = there && have_before && k + S < a.kernel ? earlier : value[k];
                        const float later = value[k] + now[u] * w_now[u][k];
                        value[k] = there && have_now ? later : value[k];
                    }
                }
            }
            if (aligned && p + S <= (size_t)a.output_length) {
                typedef float vector_t __attribute__((ext_vector_type(S)));
                vector_t v;
#pragma unroll
                for (int k = 0; k < S; ++k) v[k] = value[k];
                *reinterpret_cast<vector_t *>(out + p) = v;
            } else {
#pragma unroll
                for (int k = 0; k < S; ++k)
                    if (p + k < (size_t)a.output_length) out[p + k] = value[k];
            }
        } else {
            const unsigned p = first, stride = (unsigned)a.stride;
            if (p >= (unsigned)a.output_length) return;
            // input positions t with 0 <= p - t * stride < kernel
            const int t_hi = (int)min((unsigned)a.length - 1u, p / stride);
            const int t_lo = p < (unsigned)a.kernel ? 0 : (int)((p - (unsigned)a.kernel) / stride + 1u);
            float value = bias;
            for (int i = group * ipg; i < (group + 1) * ipg; ++i) {
                const float *in_row = a.in + (size_t)i * a.length;
                const float *w = a.w + ((size_t)i * opg + o_local) * a.kernel;
                for (int t = t_lo; t <= t_hi; ++t) value += in_row[t] * w[p - (unsigned)t * stride];
            }
            out[p] = value;
        }
    }
}

__global__ void __launch_bounds__(256) k_snake(const float *in, float *out, const float *alpha, size_t count, int length, int snake_channels) {
    const size_t index = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (index >= count) return;
    const int channel = (int)(index / (size_t)length);
    const bool snake_row = channel < snake_channels;
    const float al = snake_row ? alpha[channel] : 0.0f;
    const float v = in[index];
    if (in == out && !snake_row && !(v < 0.0f)) return;   // in place, a leaky row's value that stays as it is: no store
    out[index] = half_snake(v, snake_row, al, 1.0f / (al + 1e-9f));
}

// Row sets added in order, scaled, and written to one or more outputs, each plain or through its own half-snake:
// v = ((in0 + in1) + in2 ...) * scale; out_j = alpha_j ? half_snake(v) : v.  One pass instead of residual_inplace per
// addend, scale_dev and snake_dev (or snake_copy_dev per output), with the same arithmetic in the same order.
constexpr int kRowsMax = 4;
struct RowsCombineArgs {
    const float *in[kRowsMax];
    float *out[kRowsMax];
    const float *alpha[kRowsMax];   // null: the value as it is
    int inputs, outputs;
    float scale;
    int channels, length, snake_channels;
};

// (the grid is k_conv_transpose's)
__global__ void __launch_bounds__(256) k_rows_combine(const RowsCombineArgs a) {
    const unsigned p = blockIdx.x * 256u + threadIdx.x;
    if (p >= (unsigned)a.length) return;
    for (unsigned c = blockIdx.y; c < (unsigned)a.channels; c += gridDim.y) {
        const int channel = (int)c;
        const size_t row = (size_t)channel * a.length;
        const bool snake_row = channel < a.snake_channels;
        float in[kRowsMax], al[kRowsMax];
        // every request ahead of the first sum (an input or alpha there is not repeats the first input's)
#pragma unroll
        for (int j = 0; j < kRowsMax; ++j) in[j] = (j < a.inputs ? a.in[j] : a.in[0])[row + p];
#pragma unroll
        for (int j = 0; j < kRowsMax; ++j) al[j] = j < a.outputs && a.alpha[j] != nullptr && snake_row ? a.alpha[j][channel] : 0.0f;
        float v = in[0];
#pragma unroll
        for (int j = 1; j < kRowsMax; ++j) v = j < a.inputs ? v + in[j] : v;
        v = v * a.scale;   // 1.0f keeps the bits
#pragma unroll
        for (int j = 0; j < kRowsMax; ++j) {
            if (j >= a.outputs) break;
            a.out[j][row + p] = a.alpha[j] != nullptr ? half_snake(v, snake_row, al[j], 1.0f / (al[j] + 1e-9f)) : v;
        }
    }
}

// LDS of a launch: two stages of one block of channels (the channel-split kernel: one per wavefront), or what the epilogue keeps there.
template <int WM, int WN>
constexpr size_t conv_lds() {
    constexpr size_t stages = (size_t)2 * 6 * conv_pitch(64 * WN) * 16, epilogue = (4 * 32 * kTileStride + 4 * 64) * sizeof(float);
    return stages > epilogue ? stages : epilogue;
}
template <int NT, int PARTS>
constexpr size_t conv_split_lds() {
    constexpr size_t stages = (size_t)4 * 6 * conv_split_pitch(NT, PARTS) * 16, epilogue = 5 * 2048 * sizeof(float);
    return stages > epilogue ? stages : epilogue;
}
constexpr int kConvMaxLds = 2 * 6 * (256 + kConvMaxHalo) * 16;   // the largest of them

template <int WM, int WN, int KF, bool FUSED>
int launch_conv_f(State *st, const ConvArgs &a, const ConvBlocks &weights, char *error, size_t capacity) {
    constexpr int TM = 32 * WM, TN = 64 * WN;
    static std::atomic<bool> raised{false};   // per instantiation; states on separate threads meet here
    if (!raised) {
        MYNAH_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_conv1d<WM, WN, KF, FUSED>), hipFuncAttributeMaxDynamicSharedMemorySize, kConvMaxLds));
        raised = true;
    }
    const dim3 grid((unsigned)((a.length + TN - 1) / TN), (unsigned)((a.out_ch + TM - 1) / TM));
    hipLaunchKernelGGL((k_conv1d<WM, WN, KF, FUSED>), grid, dim3(256), (conv_lds<WM, WN>()), st->stream, a.in, a.out, weights.data, a.bias, a.in_ch, a.out_ch, a.length, a.kernel,
                       a.dilation, weights.tiles, a);
    return hip_check(hipGetLastError(), "conv1d launch", error, capacity);
}

template <int WM, int WN, int KF>
int launch_conv_k(State *st, const ConvArgs &a, const ConvBlocks &weights, char *error, size_t capacity) {
    if (a.residual != nullptr || a.residual2 != nullptr || a.scaled || a.activate) return launch_conv_f<WM, WN, KF, true>(st, a, weights, error, capacity);
    return launch_conv_f<WM, WN, KF, false>(st, a, weights, error, capacity);
}

template <int WM, int WN>
int launch_conv(State *st, const ConvArgs &a, const ConvBlocks &weights, char *error, size_t capacity) {
    switch (a.kernel) {
        case 3: return launch_conv_k<WM, WN, 3>(st, a, weights, error, capacity);
        case 7: return launch_conv_k<WM, WN, 7>(st, a, weights, error, capacity);
        case 11: return launch_conv_k<WM, WN, 11>(st, a, weights, error, capacity);
        default: return launch_conv_k<WM, WN, 0>(st, a, weights, error, capacity);
    }
}

inline int conv_split_parts(const ConvArgs &a, int tn) { return tn + (a.kernel - 1) * a.dilation <= 128 ? 2 : 3; }

template <int KF, int NT, int PARTS>
int launch_conv_split_p(State *st, const ConvArgs &a, const ConvBlocks &weights, char *error, size_t capacity) {
    static std::atomic<bool> raised{false};   // per instantiation; states on separate threads meet here
    if (!raised) {
        MYNAH_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_conv1d_split<KF, NT, PARTS>), hipFuncAttributeMaxDynamicSharedMemorySize, kConvMaxLds));
        raised = true;
    }
    const dim3 grid((unsigned)((a.length + 32 * NT - 1) / (32 * NT) * a.splits), (unsigned)((a.out_ch + 31) / 32));
    hipLaunchKernelGGL((k_conv1d_split<KF, NT, PARTS>), grid, dim3(256), (conv_split_lds<NT, PARTS>()), st->stream, a.in, a.out, weights.data, a.bias, a.in_ch, a.out_ch, a.length, a.kernel,
                       a.dilation, weights.tiles, a);
    return hip_check(hipGetLastError(), "conv1d launch", error, capacity);
}

template <int KF, int NT>
int launch_conv_split_k(State *st, const ConvArgs &a, const ConvBlocks &weights, char *error, size_t capacity) {
    return conv_split_parts(a, 32 * NT) == 2 ? launch_conv_split_p<KF, NT, 2>(st, a, weights, error, capacity) : launch_conv_split_p<KF, NT, 3>(st, a, weights, error, capacity);
}

template <int NT>
int launch_conv_split_n(State *st, const ConvArgs &a, const ConvBlocks &weights, char *error, size_t capacity) {
    switch (a.kernel) {
        case 3: return launch_conv_split_k<3, NT>(st, a, weights, error, capacity);
        case 7: return launch_conv_split_k<7, NT>(st, a, weights, error, capacity);
        case 11: return launch_conv_split_k<11, NT>(st, a, weights, error, capacity);
        default: return launch_conv_split_k<0, NT>(st, a, weights, error, capacity);
    }
}

int launch_conv_finish(State *st, const ConvBatchArgs &b, int count, char *error, size_t capacity) {
    const ConvArgs &a = b.item[0];
    hipLaunchKernelGGL(k_conv_finish, dim3((unsigned)((a.length + 255) / 256), (unsigned)a.out_ch, (unsigned)count), dim3(256), 0, st->stream, b);
    return hip_check(hipGetLastError(), "conv1d finish launch", error, capacity);
}

// The channel-split tiles of `count` convolutions side by side: 32 positions wide while 64 would leave CUs without one.  (The width does
// not enter a value's arithmetic -- same channel blocks per wavefront, same order.)
bool conv_split_narrow(const State *st, int out_channels, int length, long count) {
    return (long)((out_channels + 31) / 32) * ((length + 63) / 64) * count < st->cu_count;
}

int launch_conv_split(State *st, const ConvArgs &a, const ConvBlocks &weights, char *error, size_t capacity) {
    if (a.splits > 1) {
        ConvBatchArgs b{};
        b.item[0] = a;
        const int rc = a.length <= 32 ? launch_conv_split_n<1>(st, a, weights, error, capacity) : launch_conv_split_n<2>(st, a, weights, error, capacity);
        return rc != 0 ? rc : launch_conv_finish(st, b, 1, error, capacity);
    }
    if (conv_split_narrow(st, a.out_ch, a.length, 1)) return launch_conv_split_n<1>(st, a, weights, error, capacity);
    return launch_conv_split_n<2>(st, a, weights, error, capacity);
}

template <int WM, int WN>
int launch_conv_batch(State *st, ConvBatchArgs &b, int count, char *error, size_t capacity) {
    constexpr int TM = 32 * WM, TN = 64 * WN;
    constexpr size_t lds = conv_lds<WM, WN>();
    static std::atomic<bool> raised{false};   // per instantiation; states on separate threads meet here
    if (!raised) {
        MYNAH_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_conv1d_batch<WM, WN>), hipFuncAttributeMaxDynamicSharedMemorySize, kConvMaxLds));
        raised = true;
    }
    const ConvArgs &a = b.item[0];
    const dim3 grid((unsigned)((a.length + TN - 1) / TN), (unsigned)((a.out_ch + TM - 1) / TM), (unsigned)count);
    order_members(st, b, count, (long)grid.x * grid.y);
    hipLaunchKernelGGL((k_conv1d_batch<WM, WN>), grid, dim3(256), lds, st->stream, b);
    return hip_check(hipGetLastError(), "conv1d batch launch", error, capacity);
}

template <int NT, int PARTS>
int launch_conv_split_batch_p(State *st, ConvBatchArgs &b, int count, char *error, size_t capacity) {
    constexpr size_t lds = conv_split_lds<NT, PARTS>();
    static std::atomic<bool> raised{false};   // per instantiation; states on separate threads meet here
    if (!raised) {
        MYNAH_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_conv1d_split_batch<NT, PARTS>), hipFuncAttributeMaxDynamicSharedMemorySize, kConvMaxLds));
        raised = true;
    }
    const ConvArgs &a = b.item[0];
    const dim3 grid((unsigned)((a.length + 32 * NT - 1) / (32 * NT) * a.splits), (unsigned)((a.out_ch + 31) / 32), (unsigned)count);
    order_members(st, b, count, (long)grid.x * grid.y);
    hipLaunchKernelGGL((k_conv1d_split_batch<NT, PARTS>), grid, dim3(256), lds, st->stream, b);
    return hip_check(hipGetLastError(), "conv1d batch launch", error, capacity);
}

template <int NT>
int launch_conv_split_batch(State *st, ConvBatchArgs &b, int count, char *error, size_t capacity) {
    bool two = true;
    for (int i = 0; i < count; ++i) two = two && conv_split_parts(b.item[i], 32 * NT) == 2;
    return two ? launch_conv_split_batch_p<NT, 2>(st, b, count, error, capacity) : launch_conv_split_batch_p<NT, 3>(st, b, count, error, capacity);
}

}  // namespace

int mynah::launch_conv_pack(State *st, const float *src, uint4 *dst, size_t out_ch, size_t in_ch, size_t kernel, char *error, size_t capacity) {
    const size_t blocks = (in_ch + 15) / 16, count = (out_ch + 31) / 32 * blocks * kernel * 64;
    hipLaunchKernelGGL(k_conv_pack, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, st->stream, src, dst, count, (int)out_ch, (int)in_ch, (int)kernel, (int)blocks);
    return hip_check(hipGetLastError(), "weight packing launch", error, capacity);
}

// Too few large tiles to fill the chip and more than one block of channels to share out: small tiles with the channels split over the
// wavefronts.  (Few output channels: the large tiles are one row of wavefronts, wider in time.)  The two add in different orders, so
// the choice is the shape's alone, for single, batched and fused launches alike, and the line lies where a residual layer's
// three members meet; one convolution alone would change over later.  us, small tiles / large:
//   three members of taps 3, 7, 11, six launches:  432 channels x 2048 600 / 601, x 2560 754 / 764, x 3072 (168 large tiles) 892 / 832;
//     216 x 3584 340 / 346, x 4608 394 / 450, x 5120 (160) 446 / 458, x 6144 522 / 543;  160 x 4096 209 / 257, x 6144 302 / 343;
//     108 x 5120 161 / 200, x 6144 200 / 202, x 7168 212 / 209, x 8192 231 / 217
//   alone, 3 / 11 taps:  216 x 3072 14.0 27 / 21 44, x 4608 14.7 30 / 21 45;  108 x 5120 9.5 15.5 / 11.6 23;  54 x 12000 6.9 10.4 (8.4 with 7 taps) / 7.8 14;
//     64 -> 864 x 640 6.8 (8.4) / 7.8 11, x 1280 10.5 (12.8) / 8.2 11.3;  32 -> 864 x 5, 7 taps: 5.2 / 6.6, x 128 5.1 / 6.7
// A layer of at most 32 channels has two blocks at most and runs as one launch a block, in the large tiles' order.
static bool conv_takes_split(const State *st, int in_channels, int out_channels, int length) {
    const long tiles = out_channels <= 32 ? (long)((length + 255) / 256) : (long)((out_channels + 63) / 64) * ((length + 127) / 128);
    if (in_channels < 32 || (in_channels == 32 && out_channels <= 32)) return false;
    return in_channels > kResMaxChannels ? tiles <= (long)st->cu_count * 9 / 16 : tiles < (long)st->cu_count * 3 / 8;
}

// How many workgroups share a channel-split tile.  A few short rows leave most of the chip idle while each tile's workgroup pulls the
// weights of all channels through one CU (some 40 GB/s: 0.9 MB with 432 channels and eleven taps); so as many as bring a wavefront's
// blocks of channels down while three members' workgroups are two to a CU at most.  The sums' order follows, so this is the shape's
// alone, too.  k_conv_finish is 3.4 us of a launch, so a wavefront must be spared three blocks at least.  us a layer of three positions, taps 3 / 7 /
// 11, unshared / shared by so many: 432 channels (27 blocks) x 40 131 / 79 by 7, x 128 145 / 102 by 4, x 320 219 / 181 by 2; 216 (14) x 320 101 / 90 by 4,
// x 640 110 / 122 by 2, which spares two; 160 (10) x 160 76 / 73 by 3, x 320 79 / 80, x 640 79 / 95, which spares two as well.
constexpr int kConvSharedTiles = 160;
static int conv_splits(int in_channels, int out_channels, int length) {
    const long tiles = (long)((out_channels + 31) / 32) * ((length + 63) / 64), blocks = (in_channels + 15) / 16;
    if (in_channels <= kResMaxChannels) return 1;
    for (long each = 1; 4 * each < blocks; ++each) {
        const long splits = (blocks + 4 * each - 1) / (4 * each);
        if (splits <= kConvMaxSplits && tiles * splits <= kConvSharedTiles) return (blocks + 3) / 4 - each >= 3 ? (int)splits : 1;
    }
    return 1;
}

// Checks one convolution's arguments, caches its weights and fills the kernels' argument block.
static int conv1d_prepare(State *st, int member, const float *dev_input, float *dev_output, int in_channels, int out_channels, int length,
                          int kernel, int dilation, const float *weight, const float *bias, const mynah_hip_conv1d_extra *extra,
                          ConvArgs *out_args, ConvBlocks *out_weights, char *error, size_t capacity) {
    if (st == nullptr || dev_input == nullptr || dev_output == nullptr || weight == nullptr || in_channels <= 0 || out_channels <= 0 ||
        length <= 0 || kernel <= 0 || dilation <= 0) {
        set_error(error, capacity, "invalid conv1d arguments");   // the checks of metal_ops_conv1d, gpu/metal/backend_metal_ops.m:371-372
        return -1;
    }
    if (kernel > kConvMaxKernel || (kernel - 1) * (long)dilation > kConvMaxHalo || (size_t)in_channels * kernel > (size_t)INT_MAX ||
        (size_t)in_channels * (size_t)length > (size_t)INT_MAX * 4u || (size_t)out_channels * (size_t)length > (size_t)INT_MAX * 4u) {
        set_error(error, capacity, "conv1d: kernel above 16 taps, reach above 128 positions or tensor too large");
        return -1;
    }
    ConvBlocks weights;
    if (cached_conv_blocks(st, weight, (size_t)out_channels, (size_t)in_channels, (size_t)kernel, &weights, error, capacity) != 0) return -1;
    const float *dev_bias = nullptr;
    if (cached_vector(st, bias, (size_t)out_channels, &dev_bias, error, capacity) != 0) return -1;
    ConvArgs a{dev_input, dev_output, dev_bias, in_channels, out_channels, length, kernel, dilation};
    if (extra != nullptr) {
        if (extra->snake_channels > (size_t)out_channels || (extra->snake_channels != 0 && extra->snake_alpha == nullptr) ||
            (extra->dev_activated != nullptr && !extra->activate) || extra->dev_activated == dev_output || dev_input == dev_output ||
            (extra->dev_residual2 != nullptr && extra->dev_residual == nullptr) || !(extra->scale == extra->scale) ||
            extra->dev_activated == dev_input) {
            set_error(error, capacity, "conv1d_fused: invalid activation or residual arguments, or the input is also an output");
            return -1;
        }
        a.residual = extra->dev_residual;
        a.residual2 = extra->dev_residual2;
        a.scaled = extra->scale != 1.0f;
        a.scale = extra->scale;
        a.activate = extra->activate != 0;
        a.snake_channels = (int)extra->snake_channels;
        a.act_out = extra->dev_activated;
        if (a.activate && a.snake_channels != 0 && cached_vector(st, extra->snake_alpha, extra->snake_channels, &a.alpha, error, capacity) != 0) return -1;
    }
    if (in_channels > kResMaxChannels) {   // (whatever the length: a call that is captured then finds the memory that an earlier one with its weights allocated)
        constexpr size_t floats = (size_t)kConvSharedTiles * 32 * 64;   // of one convolution
        if (st->conv_parts == nullptr &&
            hip_check(hipMalloc(reinterpret_cast<void **>(&st->conv_parts), kConvBatchMax * floats * sizeof(float)), "conv1d workspace", error, capacity) != 0)
            return -1;
        if (conv_takes_split(st, in_channels, out_channels, length)) {
            a.splits = conv_splits(in_channels, out_channels, length);
            a.parts = st->conv_parts + (size_t)member * floats;
        }
    }
    a.weights = weights.data;
    *out_args = a;
    *out_weights = weights;
    return 0;
}

static int conv1d_launch(State *st, const ConvArgs &a, const ConvBlocks &weights, char *error, size_t capacity) {
    if (conv_takes_split(st, a.in_ch, a.out_ch, a.length)) return launch_conv_split(st, a, weights, error, capacity);
    if (a.out_ch <= 32) return launch_conv<1, 4>(st, a, weights, error, capacity);
    return launch_conv<2, 2>(st, a, weights, error, capacity);
}

static int conv1d_entry(void *state, const float *dev_input, float *dev_output, int in_channels, int out_channels, int length,
                        int kernel, int dilation, const float *weight, const float *bias, const mynah_hip_conv1d_extra *extra,
                        char *error, size_t capacity) {
    State *st = enter_state(state);
    ConvArgs a;
    ConvBlocks weights;
    if (conv1d_prepare(st, 0, dev_input, dev_output, in_channels, out_channels, length, kernel, dilation, weight, bias, extra, &a, &weights, error, capacity) != 0)
        return -1;
    return conv1d_launch(st, a, weights, error, capacity);
}

extern "C" int mynah_hip_conv1d(void *state, const float *dev_input, float *dev_output, int in_channels, int out_channels, int length,
                                int kernel, int dilation, const float *weight, const float *bias, char *error, size_t capacity) {
    return conv1d_entry(state, dev_input, dev_output, in_channels, out_channels, length, kernel, dilation, weight, bias, nullptr, error, capacity);
}

extern "C" int mynah_hip_conv1d_fused(void *state, const float *dev_input, float *dev_output, int in_channels, int out_channels, int length,
                                      int kernel, int dilation, const float *weight, const float *bias, const mynah_hip_conv1d_extra *extra,
                                      char *error, size_t capacity) {
    if (extra == nullptr) {
        set_error(error, capacity, "conv1d_fused: null extra");
        return -1;
    }
    return conv1d_entry(state, dev_input, dev_output, in_channels, out_channels, length, kernel, dilation, weight, bias, extra, error, capacity);
}

extern "C" int mynah_hip_conv1d_fused_batch(void *state, const mynah_hip_conv1d_item *items, size_t count, int in_channels, int out_channels,
                                            int length, char *error, size_t capacity) {
    State *st = enter_state(state);
    if (st == nullptr || items == nullptr || count == 0 || count > (size_t)kConvBatchMax) {
        set_error(error, capacity, "conv1d_fused_batch: one to four convolutions");
        return -1;
    }
    ConvBatchArgs b{};
    ConvBlocks weights[kConvBatchMax];
    bool side_by_side = true;
    for (size_t i = 0; i < count; ++i) {
        const mynah_hip_conv1d_item &it = items[i];
        if (conv1d_prepare(st, (int)i, it.dev_input, it.dev_output, in_channels, out_channels, length, it.kernel, it.dilation, it.weight, it.bias, &it.extra,
                           &b.item[i], &weights[i], error, capacity) != 0)
            return -1;
        side_by_side = side_by_side && (it.kernel == 3 || it.kernel == 7 || it.kernel == 11);
        // the members run at the same time: what one writes, no other may read or write
        for (size_t j = 0; j < count; ++j) {
            if (j == i) continue;
            const mynah_hip_conv1d_item &o = items[j];
            const float *const written[2] = {it.dev_output, it.extra.dev_activated};
            for (const float *w : written) {
                if (w == nullptr) continue;
                if (w == o.dev_input || w == o.dev_output || w == o.extra.dev_residual || w == o.extra.dev_residual2 || w == o.extra.dev_activated) {
                    set_error(error, capacity, "conv1d_fused_batch: a member writes rows that another member reads or writes");
                    return -1;
                }
            }
        }
    }
    if (!side_by_side || count == 1) {   // other tap counts: one after the other (the same values)
        for (size_t i = 0; i < count; ++i)
            if (conv1d_launch(st, b.item[i], weights[i], error, capacity) != 0) return -1;
        return 0;
    }
    if (conv_takes_split(st, in_channels, out_channels, length)) {
        // (the wider tile, half the weight traffic per product, as soon as all members together fill the chip)
        if (b.item[0].splits > 1) {
            const int rc = length <= 32 ? launch_conv_split_batch<1>(st, b, (int)count, error, capacity) : launch_conv_split_batch<2>(st, b, (int)count, error, capacity);
            return rc != 0 ? rc : launch_conv_finish(st, b, (int)count, error, capacity);
        }
        if (conv_split_narrow(st, out_channels, length, (long)count)) return launch_conv_split_batch<1>(st, b, (int)count, error, capacity);
        return launch_conv_split_batch<2>(st, b, (int)count, error, capacity);
    }
    if (out_channels <= 32) return launch_conv_batch<1, 4>(st, b, (int)count, error, capacity);
    return launch_conv_batch<2, 2>(st, b, (int)count, error, capacity);
}

extern "C" int mynah_hip_conv_transpose_dev(void *state, const float *dev_input, float *dev_output, int in_channels, int out_channels,
                                            int length, int output_length, int kernel, int stride, int groups, const float *weight,
                                            const float *bias, char *error, size_t capacity) {
    State *st = enter_state(state);
    if (st == nullptr || dev_input == nullptr || dev_output == nullptr || weight == nullptr || in_channels <= 0 || out_channels <= 0 ||
        length <= 0 || output_length <= 0 || kernel <= 0 || stride <= 0 || groups <= 0 || in_channels % groups != 0 ||
        out_channels % groups != 0) {
        set_error(error, capacity, "invalid conv_transpose arguments");
        return -1;
    }
    const size_t per_in = (size_t)(out_channels / groups) * kernel;
    const CachedWeight *cw = nullptr;
    if (cached_matrix(st, weight, (size_t)in_channels, per_in, MYNAH_HIP_F32, &cw, error, capacity) != 0) return -1;
    if (cw->qtype != MYNAH_HIP_F32) {
        set_error(error, capacity, "conv_transpose: weight could not be kept as f32");
        return -1;
    }
    const float *dev_bias = nullptr;
    if (cached_vector(st, bias, (size_t)out_channels, &dev_bias, error, capacity) != 0) return -1;
    ConvTransposeArgs a{dev_input, dev_output, static_cast<const float *>(cw->data), dev_bias, in_channels, out_channels, length,
                        output_length, kernel, stride, groups};
    const size_t count = (size_t)out_channels * output_length;
    if (count > (size_t)INT_MAX * 256u) {   // one thread per output value, 256 to a workgroup
        set_error(error, capacity, "conv_transpose: output too large");
        return -1;
    }
    // (further than the last input's reach a position has no inputs: the general form)
    const bool between = kernel >= stride && kernel <= 2 * (long)stride && output_length <= ((long)length + 1) * stride;
    const auto launch = [&](auto form, int each) {
        const bool aligned = reinterpret_cast<uintptr_t>(dev_output) % (4 * (size_t)each) == 0 && output_length % each == 0;
        hipLaunchKernelGGL(form, row_grid((size_t)out_channels, ((size_t)output_length + each - 1) / each), dim3(256), 0, st->stream, a, (int)aligned);
    };
    if (between && stride == 8) launch(k_conv_transpose<8>, 8);
    else if (between && stride == 4) launch(k_conv_transpose<4>, 4);
    else if (between && stride == 2) launch(k_conv_transpose<2>, 2);
    else launch(k_conv_transpose<0>, 1);
    return hip_check(hipGetLastError(), "conv_transpose launch", error, capacity);
}

static int snake_entry(void *state, const float *dev_input, float *dev_output, const float *alpha, size_t channels, size_t length,
                       size_t snake_channels, char *error, size_t capacity) {
    State *st = enter_state(state);
    if (st == nullptr || dev_input == nullptr || dev_output == nullptr || channels > (size_t)INT_MAX || length > (size_t)INT_MAX ||
        snake_channels > channels || (snake_channels != 0 && alpha == nullptr)) {
        set_error(error, capacity, "invalid snake arguments");   // metal_ops_snake, gpu/metal/backend_metal_ops.m:343-346
        return -1;
    }
    const size_t count = channels * length;
    if (count == 0) return 0;
    if (count > (size_t)INT_MAX * 256u) {   // one thread per value, 256 to a workgroup
        set_error(error, capacity, "snake: tensor too large");
        return -1;
    }
    const float *dev_alpha = nullptr;
    if (snake_channels != 0 && cached_vector(st, alpha, snake_channels, &dev_alpha, error, capacity) != 0) return -1;
    hipLaunchKernelGGL(k_snake, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, st->stream, dev_input, dev_output, dev_alpha, count,
                       (int)length, (int)snake_channels);
    return hip_check(hipGetLastError(), "snake launch", error, capacity);
}

extern "C" int mynah_hip_rows_combine_dev(void *state, const float *const *dev_inputs, size_t inputs, float scale, float *const *dev_outputs,
                                          const float *const *alphas, size_t outputs, size_t channels, size_t length, size_t snake_channels,
                                          char *error, size_t capacity) {
    State *st = enter_state(state);
    if (st == nullptr || dev_inputs == nullptr || dev_outputs == nullptr || inputs == 0 || inputs > (size_t)kRowsMax || outputs == 0 ||
        outputs > (size_t)kRowsMax || channels > (size_t)INT_MAX || length > (size_t)INT_MAX || snake_channels > channels || !(scale == scale)) {
        set_error(error, capacity, "invalid rows_combine arguments (one to four inputs and outputs)");
        return -1;
    }
    RowsCombineArgs a{};
    a.inputs = (int)inputs;
    a.outputs = (int)outputs;
    a.scale = scale;
    a.channels = (int)channels;
    a.length = (int)length;
    a.snake_channels = (int)snake_channels;
    if (channels == 0 || length == 0) return 0;
    if (channels * length > (size_t)INT_MAX * 256u) {
        set_error(error, capacity, "rows_combine: tensor too large");
        return -1;
    }
    for (size_t i = 0; i < inputs; ++i) {
        if (dev_inputs[i] == nullptr) { set_error(error, capacity, "rows_combine: null input"); return -1; }
        a.in[i] = dev_inputs[i];
    }
    for (size_t j = 0; j < outputs; ++j) {
        if (dev_outputs[j] == nullptr) { set_error(error, capacity, "rows_combine: null output"); return -1; }
        for (size_t k = 0; k < j; ++k)
            if (dev_outputs[k] == dev_outputs[j]) { set_error(error, capacity, "rows_combine: an output named twice"); return -1; }
        a.out[j] = dev_outputs[j];
        if (alphas != nullptr && alphas[j] != nullptr) {
            if (snake_channels == 0) { a.alpha[j] = reinterpret_cast<const float *>(a.in[0]); continue; }   // only leaky rows: any non-null pointer, never read
            if (cached_vector(st, alphas[j], snake_channels, &a.alpha[j], error, capacity) != 0) return -1;
        }
    }
    hipLaunchKernelGGL(k_rows_combine, row_grid(channels, length), dim3(256), 0, st->stream, a);
    return hip_check(hipGetLastError(), "rows_combine launch", error, capacity);
}

// The one-launch build for a position of a layer, or none.  Which are there follows the order in which the layer's convolutions add
// (conv_takes_split) and how many workgroups find a place at once: three to a CU with 32 positions to a wavefront (narrow), whose chain of
// products is half as long, two with 64 (wide), one of 512 threads.  Narrow while all find a place; else, up to 32 channels, wide while all of those do and
// then narrow again, and up to 64 wide.  Measured per layer of three positions, branches of 3 / 7 / 11 taps (or those named), us:
//   27 channels: x 5120 47 narrow, 70 wide, 101 as two launches a position; x 28672 73, 80, 123; x 32768 (more than three to a CU) 94, 97, 127;
//     11 taps x 98304 120, 112; 3 and 11 x 49152 98, 94; x 43008 (more wide than two to a CU) 106, 128, 156; x 65536 151, 158, 216
//   54, split order: x 1024 69 narrow, 50 as two launches of split tiles; x 2560 73, 63; x 4096 (192 tiles of 64 positions) 73, 68; x 4224 73, 79;
//     x 8192 90, 100; x 10240 102, 113
//   54, large order: x 13824 110 narrow, 111 wide, 154 as two launches; x 16384 142, 143, 157; x 20480 167, 151, 207; x 24576 180, 177, 239; x 28672
//     216, 186, 249; x 32768 247, 234, 259; x 40960 297, 266, 334; 11 taps x 40960 154, 164, 201; 11 taps x 65536 240, 244, 234
//   108, large order: 11 taps x 6144 146, 186 as two launches; x 12288 161, 190; x 16384 (more than one to a CU) 271, 203.  (Where no CU gets the
//     member with the most taps twice, more than one to a CU is faster as well: 3 and 11 x 12288 202, 237; three branches x 6144 160, 203, but x 7168 223, 209.)
enum ResBuild { RES_NONE, RES_32_NARROW, RES_32_WIDE, RES_64_SPLIT, RES_64_NARROW, RES_64_WIDE, RES_128 };
static ResBuild res_build(const State *st, const mynah_hip_res_block *blocks, size_t branches, size_t stride, size_t channels, size_t length) {
    if (channels > (size_t)kResMaxChannels) return RES_NONE;
    for (size_t i = 0; i < branches; ++i) {
        const int k = blocks[i * stride].kernel_in;
        if (k != blocks[i * stride].kernel_skip || (k != 3 && k != 7 && k != 11) || (k - 1) * (long)blocks[i * stride].dilation > kResMaxReach) return RES_NONE;
    }
    const auto fit = [&](long columns, int each) {   // workgroups of that many columns, the taps' reach of them only read
        long n = 0;
        for (size_t i = 0; i < branches; ++i) n += ((long)length + columns - blocks[i * stride].kernel_in) / (columns - (blocks[i * stride].kernel_in - 1));
        return n <= (long)st->cu_count * each;
    };
    if (channels <= 32) return fit(128, 3) || !fit(256, 2) ? RES_32_NARROW : RES_32_WIDE;
    const bool split = conv_takes_split(st, (int)channels, (int)channels, (int)length);
    if (channels > 64) return !split && fit(64, 1) ? RES_128 : RES_NONE;
    if (split) return 4 * (long)((length + 63) / 64) * (long)branches <= 3 * (long)st->cu_count ? RES_NONE : RES_64_SPLIT;
    return fit(64, 3) ? RES_64_NARROW : RES_64_WIDE;
}

// One position (block) of every branch in one launch, where there is a build for it; *done tells.
static int res_position(State *st, const mynah_hip_res_block *blocks, size_t branches, size_t stride, const float *const *in, float *const *out, size_t channels,
                        size_t length, bool *done, char *error, size_t capacity) {
    const ResBuild build = res_build(st, blocks, branches, stride, channels, length);
    *done = build != RES_NONE;
    if (!*done) return 0;
    ResArgs a{};
    a.channels = (int)channels;
    a.length = (int)length;
    a.snake_channels = (int)(channels / 2);
    for (size_t i = 0; i < branches; ++i) {
        const mynah_hip_res_block &b = blocks[i * stride];
        ResMember &m = a.member[i];
        ConvBlocks w_in, w_skip;
        if (cached_conv_blocks(st, b.weight_in, channels, channels, (size_t)b.kernel_in, &w_in, error, capacity) != 0 ||
            cached_conv_blocks(st, b.weight_skip, channels, channels, (size_t)b.kernel_skip, &w_skip, error, capacity) != 0 ||
            cached_vector(st, b.bias_in, channels, &m.b_in, error, capacity) != 0 || cached_vector(st, b.bias_skip, channels, &m.b_skip, error, capacity) != 0)
            return -1;
        if (a.snake_channels > 0) {
            const float *in_pairs = nullptr, *skip_pairs = nullptr;
            if (cached_snake_pairs(st, b.alpha_in, channels / 2, &in_pairs, error, capacity) != 0 ||
                cached_snake_pairs(st, b.alpha_skip, channels / 2, &skip_pairs, error, capacity) != 0)
                return -1;
            m.snake_in = reinterpret_cast<const float2 *>(in_pairs);
            m.snake_skip = reinterpret_cast<const float2 *>(skip_pairs);
        }
        m.in = in[i];
        m.out = out[i];
        m.w_in = w_in.data;
        m.w_skip = w_skip.data;
        m.kernel = b.kernel_in;
        m.dilation = b.dilation;
        a.blocks = w_in.blocks;
        a.tiles = w_in.tiles;
    }
    switch (build) {
        case RES_32_NARROW: return launch_res_block<1, 4, 1>(st, a, (int)branches, error, capacity);
        case RES_32_WIDE: return launch_res_block<1, 4, 2>(st, a, (int)branches, error, capacity);
        case RES_64_SPLIT: return launch_res_block<2, 2, 1, true>(st, a, (int)branches, error, capacity);
        case RES_64_NARROW: return launch_res_block<2, 2, 1>(st, a, (int)branches, error, capacity);
        case RES_64_WIDE: return launch_res_block<2, 2, 2>(st, a, (int)branches, error, capacity);
        default: return launch_res_block<4, 2, 1>(st, a, (int)branches, error, capacity);
    }
}

extern "C" int mynah_hip_res_layer_dev(void *state, const mynah_hip_res_block *blocks, size_t branches, size_t positions, const float *dev_input,
                                       float *dev_output, size_t channels, size_t length, const float *then_alpha, float *const *dev_work, char *error,
                                       size_t capacity) {
    State *st = enter_state(state);
    if (st == nullptr || blocks == nullptr || branches == 0 || branches > (size_t)kConvBatchMax || positions == 0 || dev_input == nullptr || dev_output == nullptr ||
        dev_work == nullptr || channels == 0 || channels > (size_t)INT_MAX || length == 0 || length > (size_t)INT_MAX) {
        set_error(error, capacity, "invalid residual layer arguments (one to four branches)");
        return -1;
    }
    // (the output is written by the last launch alone, value by value from the branches' rows: it may be the input or any of the work rows;
    // a single branch may also grow in its input)
    for (size_t i = 0; i < 3 * branches; ++i) {
        bool distinct = dev_work[i] != nullptr && (dev_work[i] != dev_input || (i == 0 && branches == 1));
        for (size_t j = 0; j < i; ++j) distinct = distinct && dev_work[i] != dev_work[j];
        if (!distinct) {
            set_error(error, capacity, "residual layer: work rows must be buffers of their own");
            return -1;
        }
    }
    for (size_t i = 0; i < branches * positions; ++i) {
        const mynah_hip_res_block &b = blocks[i];
        if (b.weight_in == nullptr || b.weight_skip == nullptr || b.kernel_in <= 0 || b.kernel_skip <= 0 || b.dilation <= 0 ||
            (channels >= 2 && (b.alpha_in == nullptr || b.alpha_skip == nullptr))) {
            set_error(error, capacity, "residual layer: missing weight or alpha");
            return -1;
        }
    }
    const size_t snake = channels / 2;
    float *const *const currents = dev_work, *const *const activated = dev_work + branches, *const *const residuals = dev_work + 2 * branches;
    const float *source[kConvBatchMax];   // each branch's rows so far
    float *target[kConvBatchMax];
    for (size_t i = 0; i < branches; ++i) source[i] = dev_input;
    bool have_activated = false;          // `activated` holds the source rows through the next block's first half-snake
    for (size_t p = 0; p < positions; ++p) {
        bool done = false;
        // (the fused block reads its neighbours' rows: never in place)
        for (size_t i = 0; i < branches; ++i) target[i] = source[i] == currents[i] ? residuals[i] : currents[i];
        if (res_position(st, blocks + p, branches, positions, source, target, channels, length, &done, error, capacity) != 0) return -1;
        if (!done) {
            const float *alphas[kConvBatchMax];
            if (!have_activated)
                for (size_t i = 0; i < branches; ++i) {
                    // (one launch when all branches start from the same rows)
                    if (source[i] == dev_input && i > 0) continue;
                    const size_t outs = source[i] == dev_input ? branches : 1;
                    for (size_t j = 0; j < outs; ++j) alphas[j] = snake != 0 ? blocks[(i + j) * positions + p].alpha_in : dev_input;
                    const float *in[1] = {source[i]};
                    if (mynah_hip_rows_combine_dev(state, in, 1, 1.0f, activated + i, alphas, outs, channels, length, snake, error, capacity) != 0) return -1;
                }
            mynah_hip_conv1d_item items[kConvBatchMax] = {};
            float *const *const inner = target[0] == residuals[0] ? currents : residuals;   // the buffers neither read nor finished by this position
            for (size_t i = 0; i < branches; ++i) {
                const mynah_hip_res_block &b = blocks[i * positions + p];
                items[i] = mynah_hip_conv1d_item{activated[i], inner[i], b.kernel_in, b.dilation, b.weight_in, b.bias_in, {nullptr, nullptr, 1.0f, 1, b.alpha_skip, snake, nullptr}};
            }
            bool in_place = source[0] == inner[0];   // the source rows are still needed: they move on in place below
            if (in_place) {
                for (size_t i = 0; i < branches; ++i) {
                    items[i].dev_output = target[i];
                    target[i] = const_cast<float *>(source[i]);
                }
            }
            if (mynah_hip_conv1d_fused_batch(state, items, branches, (int)channels, (int)channels, (int)length, error, capacity) != 0) return -1;
            const bool more = p + 1 < positions;
            for (size_t i = 0; i < branches; ++i) {
                const mynah_hip_res_block &b = blocks[i * positions + p];
                const float *inner_rows = items[i].dev_output;
                items[i] = mynah_hip_conv1d_item{inner_rows, target[i], b.kernel_skip, 1, b.weight_skip, b.bias_skip,
                                                 {source[i], nullptr, 1.0f, more ? 1 : 0, more ? blocks[i * positions + p + 1].alpha_in : nullptr, more ? snake : 0,
                                                  more ? activated[i] : nullptr}};
            }
            if (mynah_hip_conv1d_fused_batch(state, items, branches, (int)channels, (int)channels, (int)length, error, capacity) != 0) return -1;
            have_activated = more;
        } else {
            have_activated = false;
        }
        for (size_t i = 0; i < branches; ++i) source[i] = target[i];
    }
    float *outs[1] = {dev_output};
    const float *alphas[1] = {then_alpha};
    return mynah_hip_rows_combine_dev(state, source, branches, (float)(1.0 / (double)branches), outs, alphas, 1, channels, length, snake, error, capacity);
}

extern "C" int mynah_hip_snake_dev(void *state, float *dev_data, const float *alpha, size_t channels, size_t length, size_t snake_channels,
                                   char *error, size_t capacity) {
    return snake_entry(state, dev_data, dev_data, alpha, channels, length, snake_channels, error, capacity);
}

extern "C" int mynah_hip_snake_copy_dev(void *state, const float *dev_input, float *dev_output, const float *alpha, size_t channels,
                                        size_t length, size_t snake_channels, char *error, size_t capacity) {
    return snake_entry(state, dev_input, dev_output, alpha, channels, length, snake_channels, error, capacity);
}
