// Products of many f32 rows with a weight, in f32, on the f16 matrix cores (half_product.h): the encoder prefill with f32
// operands and the cross-attention K/V.  out[m][n] = sum over taps j and channels c of in[m - (taps - 1) + j][c] * W[n][c][j]; one tap is
// a plain product, three are the causal convolution of the encoder's FFN (causal_conv_ffn, src/graph.c:302-352).
#include <type_traits>

#include "half_product.h"

namespace mynah {
namespace {

// The weight lies in memory in the order in which the wavefronts take it, taken apart once (four bytes a value, as f32 is): per tile of 32
// outputs, block of 32 channels, half of the block and tap (a step) two runs of 64 uint4s, one per piece, lane l's being output l % 32,
// channels 8 * (l / 32) .. of the half.  A request is then 1 KiB of consecutive bytes and goes straight to the registers of the one
// wavefront that multiplies it.  Behind all steps the values themselves (two float4 runs a step, channels 0 .. 3 and 4 .. 7 of a lane's eight)
// for sums that are no finite number, and behind those the outputs' inverse scales.
struct SplitWeight {
    const uint4 *data;
    size_t steps;
    __host__ __device__ SplitWeight(const uint4 *data_arg, size_t n, size_t channels, size_t taps) : data(data_arg), steps(n / 32 * (channels / 16) * taps) {}
    __device__ __forceinline__ const float4 *values() const { return reinterpret_cast<const float4 *>(data + steps * 128); }
    __device__ __forceinline__ const float *inverses() const { return reinterpret_cast<const float *>(data + steps * 256); }
};

__global__ void __launch_bounds__(256) k_split_pack(const float *src, uint4 *dst, int n_all, int channels, int taps) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const SplitWeight w(dst, (size_t)n_all, (size_t)channels, (size_t)taps);
    if (i >= w.steps * 64) return;
    const int lane = (int)(i & 63);
    const size_t step = i >> 6;
    size_t j = step;
    const int tap = (int)(j % (size_t)taps);
    j /= (size_t)taps;
    const int half = (int)(j & 1);
    j >>= 1;
    const int blocks = channels / 32, block = (int)(j % (size_t)blocks);
    const size_t n = (j / (size_t)blocks) * 32 + (lane & 31);
    const size_t c = (size_t)block * 32 + half * 16 + (lane >> 5) * 8;
    const float *p = src + (n * (size_t)channels + c) * taps + tap;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = p[(size_t)e * taps];
    float largest = 0.0f;
    half_eight(v, 1.0f / w.inverses()[n], largest, dst[step * 128 + lane], dst[step * 128 + 64 + lane]);
    float4 *const values = reinterpret_cast<float4 *>(dst + w.steps * 128) + step * 128 + lane;
    values[0] = make_float4(v[0], v[1], v[2], v[3]);
    values[64] = make_float4(v[4], v[5], v[6], v[7]);
}

// LDS of a tile: three stages of one block of 16 G channels (32 * MT + taps - 1 rows), operand-major per 16-deep part, piece and
// 8-deep half, and afterwards the later groups' sums; and the largest input of each wavefront.  The row pitch puts the two halves of a row 64 bytes
// apart modulo 256; fragment reads are 512 consecutive bytes.  (Bank conflicts are 2 % of a launch's cycles; a pitch of kRows + 2 with the pieces
// innermost has as many.)
template <int MT, int TAPS, int G>
struct SplitTile {
    static constexpr int kRows = 32 * MT + (TAPS - 1), kPitch = (kRows + 11) / 16 * 16 + 4;
    static_assert(kPitch >= kRows && kPitch % 16 == 4 && (G == 2 || G == 4), "bank layout");
    union {
        uint4 a[3][G][2][2][kPitch];
        float sums[8 - 8 / G][MT][16][64];
    };
    float largest[8];
};

constexpr int kBlocksAhead = 2;   // blocks per round of the loop below: a split's block count is a multiple of it

// acc[t] = the tile's sums over `blocks` blocks of 16 G channels, for rows 32 t .. of the tile and the wavefront's 32 columns;
// valid in the first 8 / G of the eight wavefronts.
// Wavefront w multiplies columns 32 * (w % (8 / G)) .. over the 16-deep part w / (8 / G) of every block: two wavefronts to a SIMD, because
// one alone cannot issue its vector instructions beside its own matrix instructions.
// A wavefront's weight pieces come from memory R steps ahead and are multiplied where they arrive; the rows are staged by all eight
// wavefronts, taken apart on the way to LDS, and serve every tap from there.  A block is stored into a stage two blocks after it was last
// read, its requests leave two blocks before that; what runs past the last block is requested (the buffers are padded) and not
// used, so that no request stands under a condition.  One tap: four blocks are unrolled (left after two where there are no more), so
// that four steps of weights are in flight: a step is 192 cycles of matrix instructions, a round trip to L2 some 2,000.
template <int MT, int TAPS, int G>
__device__ __forceinline__ void split_tile(const float *const a, const int lda, const int row0, const int rows, const uint4 *const w, const float inverse,
                                           const int blocks, SplitTile<MT, TAPS, G> &lds, f32x16 (&acc)[MT]) {
    using Tile = SplitTile<MT, TAPS, G>;
    constexpr int UB = TAPS == 1 ? 2 * kBlocksAhead : kBlocksAhead, R = TAPS == 1 ? 4 : 2 * TAPS;   // blocks per round; steps of weights in flight
    static_assert((UB * TAPS) % R == 0 && UB % 2 == 0 && kBlocksAhead == 2, "register stages must repeat with the round");
    const int tid = threadIdx.x, lane = tid & 63, group = tid / (512 / G);
    constexpr int kPass = 512 / (4 * G);   // rows staged at once
    const int srow = tid / (4 * G), sc = tid % (4 * G);
    constexpr int kRows = Tile::kRows, NP = (kRows + kPass - 1) / kPass;
    constexpr int kStage = G * 2 * 2 * Tile::kPitch;
    uint4 *const stages = &lds.a[0][0][0][0][0];
    float scale = 1.0f, unscale = 1.0f, largest = 0.0f;
    HalfSums sums[MT];
    for (bool once_more = false;; once_more = true) {
        const float *ap[NP];
#pragma unroll
        for (int i = 0; i < NP; ++i) ap[i] = a + (ptrdiff_t)min(row0 - (TAPS - 1) + min(srow + kPass * i, kRows - 1), rows - 1) * lda + 4 * sc;
        float4 ra[2][NP];
        const auto request_a = [&](int set, int block) {
#pragma unroll
            for (int i = 0; i < NP; ++i) ra[set][i] = *reinterpret_cast<const float4 *>(ap[i] + block * (16 * G));
        };
        const auto store_a = [&](int set, uint4 *stage, bool counts) {   // (counts: not past the last block, where anything may lie)
#pragma unroll
            for (int i = 0; i < NP; ++i)
                if (kPass * i + kPass <= kRows || srow + kPass * i < kRows) {
                    const float4 v = ra[set][i];
                    uint2 piece[2];
                    float rest[2];
                    half_pieces(v.x, v.y, scale, piece[0].x, piece[1].x, rest);
                    half_pieces(v.z, v.w, scale, piece[0].y, piece[1].y, rest);
                    const float most = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
                    largest = fmaxf(largest, counts ? most : 0.0f);
#pragma unroll
                    for (int q = 0; q < 2; ++q)
                        reinterpret_cast<uint2 *>(&stage[(((sc >> 2) * 2 + q) * 2 + ((sc >> 1) & 1)) * Tile::kPitch + srow + kPass * i])[sc & 1] = piece[q];
                }
        };
        const uint4 *wp = w + (size_t)group * (TAPS * 128) + lane;
        uint4 rw[R][2];
        const auto request_w = [&](int slot, int step) {   // step counted from wp: block step / TAPS, tap step % TAPS
            const uint4 *p = wp + ((step / TAPS) * G * TAPS + step % TAPS) * 128;
            rw[slot][0] = p[0];
            rw[slot][1] = p[64];
        };
        half8_t fa[2][MT][2];
        const auto read_a = [&](int set, const uint4 *stage, int tap) {
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int q = 0; q < 2; ++q)
                    fa[set][t][q] = __builtin_bit_cast(half8_t, stage[((group * 2 + q) * 2 + (lane >> 5)) * Tile::kPitch + (lane & 31) + 32 * t + tap]);
        };
        int now = 0, next = kStage, after = 2 * kStage;
#pragma unroll
        for (int t = 0; t < MT; ++t) sums[t].clear();
        request_a(0, 0);
#pragma unroll
        for (int i = 0; i < R; ++i) request_w(i, i);
        request_a(1, 1);
        store_a(0, stages, true);
        request_a(0, 2);
        __syncthreads();
        read_a(0, stages, 0);
        __builtin_amdgcn_sched_barrier(0);
        for (int block = 0; block < blocks; block += UB) {
#pragma unroll
            for (int u = 0; u < UB; ++u) {
                if (u == kBlocksAhead && block + u >= blocks) break;
#pragma unroll
                for (int tap = 0; tap < TAPS; ++tap) {
                    const int s = u * TAPS + tap;
                    if (tap == 0) {
                        store_a((u + 1) & 1, stages + next, block + u + 1 < blocks);
                        request_a((u + 1) & 1, u + 3);
                    }
                    if (TAPS == 1) __syncthreads();   // (the next step already reads the block stored here)
                    if (tap + 1 < TAPS) read_a((s + 1) & 1, stages + now, tap + 1);
                    else read_a((s + 1) & 1, stages + next, 0);
                    half8_t fw[2];
#pragma unroll
                    for (int q = 0; q < 2; ++q) fw[q] = __builtin_bit_cast(half8_t, rw[s % R][q]);
#pragma unroll
                    for (int t = 0; t < MT; ++t) sums[t].multiply(fa[s & 1][t], fw);
                    request_w(s % R, s + R);   // into the registers multiplied here
                    __builtin_amdgcn_sched_barrier(0);
                    if (TAPS > 1 && tap == 0) {
                        __syncthreads();
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
                const int t = now;
                now = next;
                next = after;
                after = t;
            }
            wp += UB * G * TAPS * 128;
#pragma unroll
            for (int i = 0; i < NP; ++i) ap[i] += UB * 16 * G;
        }
        largest = wave_max(largest);
        if (lane == 0) lds.largest[tid >> 6] = largest;
        __syncthreads();
        float of_all = lds.largest[0];
#pragma unroll
        for (int i = 1; i < 8; ++i) of_all = fmaxf(of_all, lds.largest[i]);
        const int e = once_more ? 0 : __builtin_amdgcn_readfirstlane(half_rescale(of_all));
        if (__builtin_expect(e == 0, 1)) break;
        scale = power_of_two(e);
        unscale = power_of_two(-e);
    }
    if (group > 0) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) lds.sums[(tid >> 6) - 8 / G][t][r][lane] = sums[t].sum(r);
    }
    __syncthreads();
    if (group == 0) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                float sum = sums[t].sum(r) + lds.sums[tid >> 6][t][r][lane];
#pragma unroll
                for (int g = 2; g < G; ++g) sum += lds.sums[(tid >> 6) + (g - 1) * (8 / G)][t][r][lane];
                acc[t][r] = sum * unscale * inverse;
            }
    }
}

// A finished tile to memory, a lane's column at `out`.  A sum that is no finite number is stored again as the chain of f32 multiply-adds
// over the same blocks (half_product.h): looked for behind the stores, where it is cheapest (before them: 0.4 us a launch).
// values: the tile's weights.
template <int MT, int TAPS>
__device__ __forceinline__ void split_store(const float *const a, const int lda, const int row0, const int rows, const float4 *const values, const int blocks, const f32x16 (&acc)[MT], float *const out, const int pitch) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m = row0 + 32 * t + split_acc_row(r, lane);
            if (m < rows) out[(size_t)m * pitch] = acc[t][r];
        }
    if (split_all_finite(acc)) return;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll 1
        for (int r = 0; r < 16; ++r) {
            const int m = row0 + 32 * t + split_acc_row(r, lane);
            if (m >= rows || split_finite(acc[t][r])) continue;
            float s = 0.0f;
#pragma unroll 1
            for (int c = 0; c < 32 * blocks && s == s; c += 8)
#pragma unroll 1
                for (int tap = 0; tap < TAPS; ++tap) {
                    const int row = m - (TAPS - 1) + tap;
                    if (row < 0) continue;
                    const float4 *const x = reinterpret_cast<const float4 *>(a + (size_t)row * lda + c);
                    const float4 *const v = values + ((c >> 4) * TAPS + tap) * 128 + ((c >> 3) & 1) * 32 + (lane & 31);
#pragma unroll
                    for (int part = 0; part < 2; ++part) {
                        const float4 xs = x[part], vs = v[64 * part];
                        s = __builtin_fmaf(xs.x, vs.x, s);
                        s = __builtin_fmaf(xs.y, vs.y, s);
                        s = __builtin_fmaf(xs.z, vs.z, s);
                        s = __builtin_fmaf(xs.w, vs.w, s);
                    }
                }
            out[(size_t)m * pitch] = s;
        }
}

// Workgroup -> (row tile, column tile and split): the row tiles of one piece of the weight run on one XCD (workgroup i runs on
// XCD i % 8), which then fetches that piece once.
struct SplitWork {
    int m, nz;
    __device__ __forceinline__ SplitWork(int id, int mtiles) : m((id >> 3) % mtiles), nz(((id >> 3) / mtiles) * 8 + (id & 7)) {}
};

// part[z][m][n]: the sums over split z's channels (splits == 1: the product).
// A workgroup's columns: 32 for each of its 8 / G wavefronts of a group.
template <int MT, int TAPS, int G>
__global__ void __launch_bounds__(512) k_split_rows(const float *const a, const uint4 *const w, const int M, const int N, const int channels, const int mtiles,
                                                    const int ntiles, const int splits, float *const part) {
    __shared__ SplitTile<MT, TAPS, G> lds;
    constexpr int kWide = 8 / G, kDeep = 16 * G;
    const SplitWork work((int)blockIdx.x, mtiles);
    if (work.nz >= ntiles * splits) return;
    const int lane = threadIdx.x & 63, wave = (threadIdx.x >> 6) % kWide;
    const int z = work.nz / ntiles, share = channels / splits;
    const int col0 = ((work.nz % ntiles) * kWide + wave) * 32, m0 = work.m * 32 * MT;
    f32x16 acc[MT];
    const SplitWeight weight(w, (size_t)N, (size_t)channels, TAPS);
    const size_t step = ((size_t)(min(col0, N - 32) / 32) * (channels / 16) + z * (share / 16)) * TAPS;   // the tile's first
    const uint4 *tile = w + step * 128;
    const float inverse = weight.inverses()[min(col0, N - 32) + (lane & 31)];
    split_tile<MT, TAPS, G>(a + z * share, channels, m0, M, tile, inverse, share / kDeep, lds, acc);
    if (threadIdx.x >= 64 * kWide || col0 >= N) return;
    split_store<MT, TAPS>(a + z * share, channels, m0, M, weight.values() + step * 128, share / 32, acc, part + (size_t)z * M * N + col0 + (lane & 31), N);
}

// The K and V halves of every layer's kv_net on that layer's normalised memory, one launch: blockIdx.y names the layer.
__global__ void __launch_bounds__(512) k_split_cross_kv(const float *const normed, const SplitLayers weights, const int M, const int width, const int xw,
                                                        const int mtiles, float *const k_out, float *const v_out) {
    __shared__ SplitTile<2, 1, 2> lds;
    const int N = 2 * xw, ntiles = (N + 127) / 128;
    const SplitWork work((int)blockIdx.x, mtiles);
    if (work.nz >= ntiles) return;
    const int lane = threadIdx.x & 63, wave = (threadIdx.x >> 6) & 3, layer = (int)blockIdx.y;
    const int col0 = work.nz * 128 + wave * 32, m0 = work.m * 64;
    f32x16 acc[2];
    const SplitWeight weight(weights.w[layer], (size_t)N, (size_t)width, 1);
    const size_t step = (size_t)(min(col0, N - 32) / 32) * (width / 32) * 2;
    const uint4 *tile = weights.w[layer] + step * 128;
    const float inverse = weight.inverses()[min(col0, N - 32) + (lane & 31)];
    split_tile<2, 1, 2>(normed + (size_t)layer * M * width, width, m0, M, tile, inverse, width / 32, lds, acc);
    if (threadIdx.x >= 256 || col0 >= N) return;
    float *const out = (col0 < xw ? k_out + col0 : v_out + col0 - xw) + (size_t)layer * M * xw + (lane & 31);
    split_store<2, 1>(normed + (size_t)layer * M * width, width, m0, M, weight.values() + step * 128, width / 32, acc, out, xw);
}

// The same for more than 64 rows: a workgroup takes 64 * MT rows and 128 columns of a layer, wavefront w rows 32 MT (w / 4) .. and columns
// 32 (w % 4) .. over all channels.  What a CU has to fetch bounds these products -- 64 rows a workgroup are 24 KB for 384 cycles of its matrix cores, 42 us
// at 180 rows x 12 layers, 35 % of what it fetches the weight's third reading -- so the rows go as far as the registers do.  The rows come
// normalised once, without any layer's gain and bias, which are applied as they are staged (the same operations in the same order as a
// LayerNorm of each layer's own, which wrote and read twelve times the rows).
template <int MT>
struct WideTile {
    static constexpr int kRows = 64 * MT, kPitch = kRows + 4;
    uint4 a[2][2][2][2][kPitch];   // [stage][16-deep half][piece][8-deep quarter][row]
    float largest[8];
};
template <int MT, bool BIAS>
__global__ void __launch_bounds__(512) k_wide_cross_kv(const float *const rows_in, const SplitLayers layers, const int M, const int width, const int xw,
                                                       const int mtiles, float *const k_out, float *const v_out) {
    using Tile = WideTile<MT>;
    extern __shared__ __align__(16) unsigned char smem[];
    Tile &lds = *reinterpret_cast<Tile *>(smem);
    const int N = 2 * xw, ntiles = (N + 127) / 128;
    const SplitWork work((int)blockIdx.x, mtiles);
    if (work.nz >= ntiles) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave >> 2, wn = wave & 3, layer = (int)blockIdx.y;
    const int srow = tid >> 3, sc = tid & 7, blocks = width / 32;
    const int col0 = work.nz * 128 + wn * 32, m0 = work.m * Tile::kRows;
    const float *const gain = layers.gain[layer], *const bias = layers.bias[layer];
    const SplitWeight weight(layers.w[layer], (size_t)N, (size_t)width, 1);
    const size_t step0 = (size_t)(min(col0, N - 32) / 32) * blocks * 2;
    const float inverse = weight.inverses()[min(col0, N - 32) + (lane & 31)];
    constexpr int kStage = 2 * 2 * 2 * Tile::kPitch;
    uint4 *const stages = &lds.a[0][0][0][0][0];
    float scale = 1.0f, unscale = 1.0f, largest = 0.0f;
    HalfSums sums[MT];
    for (bool once_more = false;; once_more = true) {
        // (an address the same for every lane and 32 bits of a lane's own: less registers than a pointer a row)
        const float *const rows0 = rows_in + (size_t)m0 * width;
        unsigned at[MT], own = 16u * sc, lane_bytes = 16u * lane;
#pragma unroll
        for (int i = 0; i < MT; ++i) at[i] = ((unsigned)(min(m0 + srow + 64 * i, M - 1) - m0) * (unsigned)width + 4u * sc) * 4u;
        float4 ra[2][MT], rg[2], rb[BIAS ? 2 : 1];
        const auto request_a = [&](int set, int block) {   // (past the last block: the last one again)
            const size_t channel = (size_t)min(block, blocks - 1) * 32;
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                at[i] = opaque(at[i]);
                ra[set][i] = load_behind(reinterpret_cast<const float4 *>(rows0 + channel), at[i]);
            }
            own = opaque(own);
            rg[set] = load_behind(reinterpret_cast<const float4 *>(gain + channel), own);
            if constexpr (BIAS) rb[set] = load_behind(reinterpret_cast<const float4 *>(bias + channel), own);
        };
        const auto store_a = [&](int set, uint4 *stage) {
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                float4 v = ra[set][i];
                v.x *= rg[set].x; v.y *= rg[set].y; v.z *= rg[set].z; v.w *= rg[set].w;
                if constexpr (BIAS) { v.x += rb[set].x; v.y += rb[set].y; v.z += rb[set].z; v.w += rb[set].w; }
                uint2 piece[2];
                float rest[2];
                half_pieces(v.x, v.y, scale, piece[0].x, piece[1].x, rest);
                half_pieces(v.z, v.w, scale, piece[0].y, piece[1].y, rest);
                largest = fmaxf(largest, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
#pragma unroll
                for (int q = 0; q < 2; ++q)
                    reinterpret_cast<uint2 *>(&stage[(((sc >> 2) * 2 + q) * 2 + ((sc >> 1) & 1)) * Tile::kPitch + srow + 64 * i])[sc & 1] = piece[q];
            }
        };
        const uint4 *wp = layers.w[layer] + step0 * 128;
        uint4 rw[4][2];
        const auto request_w = [&](int slot, int step) {
            lane_bytes = opaque(lane_bytes);
            rw[slot][0] = load_behind(wp + step * 128, lane_bytes);
            rw[slot][1] = load_behind(wp + step * 128 + 64, lane_bytes);
        };
#pragma unroll
        for (int t = 0; t < MT; ++t) sums[t].clear();
        request_a(0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) request_w(i, i);
        request_a(1, 1);
        store_a(0, stages);
        request_a(0, 2);
        __syncthreads();
        for (int block = 0; block < blocks; block += 2) {   // (an even number of blocks)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const uint4 *const now = stages + u * kStage;
                store_a((u + 1) & 1, stages + (1 - u) * kStage);
                request_a((u + 1) & 1, block + u + 3);
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    const int s = 2 * u + half;
                    half8_t fw[2], fa[MT][2];
#pragma unroll
                    for (int t = 0; t < MT; ++t)
#pragma unroll
                        for (int q = 0; q < 2; ++q)
                            fa[t][q] = __builtin_bit_cast(half8_t, now[((half * 2 + q) * 2 + (lane >> 5)) * Tile::kPitch + wm * 32 * MT + 32 * t + (lane & 31)]);
#pragma unroll
                    for (int q = 0; q < 2; ++q) fw[q] = __builtin_bit_cast(half8_t, rw[s][q]);
#pragma unroll
                    for (int t = 0; t < MT; ++t) sums[t].multiply(fa[t], fw);
                    request_w(s, s + 4);   // into the registers multiplied here
                }
                __syncthreads();   // the block stored here may be read, and the one read here overwritten
            }
            wp += 4 * 128;
        }
        largest = wave_max(largest);
        if (lane == 0) lds.largest[wave] = largest;
        __syncthreads();
        float of_all = lds.largest[0];
#pragma unroll
        for (int i = 1; i < 8; ++i) of_all = fmaxf(of_all, lds.largest[i]);
        const int e = once_more ? 0 : __builtin_amdgcn_readfirstlane(half_rescale(of_all));
        if (__builtin_expect(e == 0, 1)) break;
        scale = power_of_two(e);
        unscale = power_of_two(-e);
    }
    if (col0 >= N) return;
    f32x16 acc[MT];
    float *const out = (col0 < xw ? k_out + col0 : v_out + col0 - xw) + (size_t)layer * M * xw + (lane & 31);
    const int row0 = m0 + wm * 32 * MT;
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            acc[t][r] = sums[t].sum(r) * unscale * inverse;
            const int m = row0 + 32 * t + split_acc_row(r, lane);
            if (m < M) out[(size_t)m * xw] = acc[t][r];
        }
    if (split_all_finite(acc)) return;
    // (see split_store)
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll 1
        for (int r = 0; r < 16; ++r) {
            const int m = row0 + 32 * t + split_acc_row(r, lane);
            if (m >= M || split_finite(acc[t][r])) continue;
            const float *const x = rows_in + (size_t)m * width;
            const float4 *const values = weight.values() + step0 * 128 + (lane & 31);
            float s = 0.0f;
#pragma unroll 1
            for (int c = 0; c < width && s == s; c += 4) {
                const float4 v = values[(size_t)(c >> 4) * 128 + ((c >> 2) & 1) * 64 + ((c >> 3) & 1) * 32];
                const float w4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float n = x[c + e] * gain[c + e];
                    if constexpr (BIAS) n += bias[c + e];
                    s = __builtin_fmaf(n, w4[e], s);
                }
            }
            out[(size_t)m * xw] = s;
        }
}

// The memory's rows under every layer's LayerNorm (gain, optional bias), one workgroup per row and layer: normed[layer][row].
__global__ void __launch_bounds__(256) k_layernorm_layers(const float *in, float *normed, const SplitLayers layers, int rows, int width) {
    __shared__ float s4[4];
    const int row = (int)blockIdx.x, layer = (int)blockIdx.y;
    layernorm_row(in + (size_t)row * width, normed + ((size_t)layer * rows + row) * width, layers.gain[layer], layers.bias[layer], width, s4);
}

}  // namespace

int launch_split_pack(State *st, const float *src, uint4 *dst, size_t n, size_t channels, size_t taps, char *error, size_t capacity) {
    const SplitWeight w(dst, n, channels, taps);
    if (launch_half_row_scales(st, src, reinterpret_cast<float *>(dst + w.steps * 256), n, n, channels * taps, error, capacity) != 0) return -1;
    hipLaunchKernelGGL(k_split_pack, dim3((unsigned)((w.steps * 64 + 255) / 256)), dim3(256), 0, st->stream, src, dst, (int)n, (int)channels, (int)taps);
    return hip_check(hipGetLastError(), "weight packing launch", error, capacity);
}

// A weight's rows get a scale each: the largest value under it lies in [2^13, 2^14), unless it is 2^20 times the row's usual size and
// more -- then what is 2^20 times that lies there, and what does not fit above it is kept as its bits (half_product.h).  A workgroup a row, four
// requests of a thread side by side (a wavefront a row and one request at a time: 39 us for 768 x 6912); rows past the last one get 1.
__global__ void __launch_bounds__(256) k_half_row_scales(const float *src, float *inverses, int rows, size_t per_row) {
    __shared__ float s4[4];
    const int row = (int)blockIdx.x, tid = (int)threadIdx.x;
    float sum = 0.0f, count = 0.0f, most = -127.0f;
    if (row < rows)
        for (size_t i0 = 0; i0 < per_row; i0 += 1024) {
            float v[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] = src[(size_t)row * per_row + min(i0 + 256 * k + tid, per_row - 1)];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int e = exponent_of(v[k]);
                const bool counts = i0 + 256 * k + tid < per_row && v[k] != 0.0f && e != 128;   // (else nothing, or no finite number)
                sum += counts ? (float)e : 0.0f;
                count += counts ? 1.0f : 0.0f;
                most = counts ? fmaxf(most, (float)e) : most;
            }
        }
    sum = block_sum(sum, s4);
    count = block_sum(count, s4);
    most = block_max(most, s4);
    const int top = count == 0.0f ? 13 : (int)fminf(most, floorf(sum / count) + 20.0f);
    if (tid == 0) inverses[row] = power_of_two(max(top - 13, -126));
}
int launch_half_row_scales(State *st, const float *src, float *inverses, size_t rows, size_t padded_rows, size_t per_row, char *error, size_t capacity) {
    hipLaunchKernelGGL(k_half_row_scales, dim3((unsigned)padded_rows), dim3(256), 0, st->stream, src, inverses, (int)rows, per_row);
    return hip_check(hipGetLastError(), "weight scale launch", error, capacity);
}

// Tiles of 64 rows unless a call has 32 or fewer, or (no split: nothing to fill the chip with) they would leave half of it idle.
static int split_row_tiles(const State *st, size_t rows, size_t n, bool may_split) {
    const size_t columns = (n + 127) / 128;
    return rows <= 32 || (!may_split && (rows + 63) / 64 * columns * 2 <= (size_t)st->cu_count) ? 1 : 2;
}

// The most splits that still give every workgroup a CU of its own: a second one on a CU runs behind the first (192 x 3072,
// three taps of 768: 19.0 us as 216 workgroups, 26.6 as 288).
int split_product_splits(const State *st, size_t rows, size_t channels, size_t n, size_t most) {
    const size_t mt = (size_t)split_row_tiles(st, rows, n, true), tiles = (rows + 32 * mt - 1) / (32 * mt) * ((n + 127) / 128);
    size_t best = 1;
    for (size_t s = 2; s <= most; ++s)
        if (channels % (32 * kBlocksAhead * s) == 0 && tiles * s <= (size_t)st->cu_count) best = s;
    return (int)best;
}

int launch_split_product(State *st, const float *in, const uint4 *w, size_t rows, size_t channels, size_t taps, size_t n, int splits, float *part,
                         char *error, size_t capacity) {
    if (rows == 0 || n == 0 || n % 32 != 0 || channels == 0 || splits < 1 || channels % (32 * kBlocksAhead * (size_t)splits) != 0 || (taps != 1 && taps != 3) ||
        rows > 0x100000 || n > 0x100000 || channels > 0x100000) {
        set_error(error, capacity, "f32 product: shape outside the matrix-core kernel's");
        return -1;
    }
    const int mt = split_row_tiles(st, rows, n, splits > 1), mtiles = (int)((rows + 32 * mt - 1) / (32 * mt));
    // An unsplit product of 32-row tiles, where that still gives every workgroup a CU of its own: 64 columns a workgroup and four groups of
    // wavefronts over the channels, twice the workgroups with half the chain.  us a launch, 768 -> 2304 by 64 / 128 columns: 16 rows 8.8 / 11.7,
    // 96 8.9 / 12.1, 192 10.1 / 13.7.  (Split ones fill the chip by their splits: 16 rows of 3072 -> 768 as twelve, 7.2 / 7.0.)
    const bool deep = mt == 1 && taps == 1 && splits == 1 && channels % 128 == 0 && (n + 63) / 64 * mtiles <= (size_t)st->cu_count;
    const int ntiles = (int)((n + (deep ? 63 : 127)) / (deep ? 64 : 128));
    const dim3 grid((unsigned)((ntiles * splits + 7) / 8 * 8 * mtiles)), block(512);
    const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, block, 0, st->stream, in, w, (int)rows, (int)n, (int)channels, mtiles, ntiles, splits, part);
    };
    if (deep) launch(k_split_rows<1, 1, 4>);
    else if (taps == 1) mt == 1 ? launch(k_split_rows<1, 1, 2>) : launch(k_split_rows<2, 1, 2>);
    else mt == 1 ? launch(k_split_rows<1, 3, 2>) : launch(k_split_rows<2, 3, 2>);
    return hip_check(hipGetLastError(), "f32 product launch", error, capacity);
}

template <int MT, bool BIAS>
static int launch_wide(State *st, size_t rows, size_t width, const SplitLayers &layers, size_t count, size_t xw, const float *normed, float *k_out, float *v_out,
                       char *error, size_t capacity) {
    static bool raised = false;
    if (!raised) {
        MYNAH_TRY(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_wide_cross_kv<MT, BIAS>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(WideTile<MT>)));
        raised = true;
    }
    const size_t mtiles = (rows + 64 * MT - 1) / (64 * MT);
    hipLaunchKernelGGL((k_wide_cross_kv<MT, BIAS>), dim3((unsigned)(((2 * xw + 127) / 128 + 7) / 8 * 8 * mtiles), (unsigned)count), dim3(512), sizeof(WideTile<MT>),
                       st->stream, normed, layers, (int)rows, (int)width, (int)xw, (int)mtiles, k_out, v_out);
    return hip_check(hipGetLastError(), "cross K/V launch", error, capacity);
}

int launch_split_cross_kv(State *st, const float *memory, size_t rows, size_t width, const SplitLayers &layers, size_t count, size_t xw, float *normed,
                          float *k_out, float *v_out, char *error, size_t capacity) {
    bool biased = false, plain = false;
    for (size_t l = 0; l < count; ++l) (layers.bias[l] != nullptr ? biased : plain) = true;
    // Above 64 rows (all layers with a bias or all without: a launch is one build or the other).  us with the LayerNorm, 12 layers of 768,
    // the wide product / 64 rows a workgroup: 48 rows 21.7 / 20.9, 64 22.1 / 22.0, 65 27.6 / 32.6, 128 28.6 / 34.4, 180 38 / 50
    if (rows > 64 && !(biased && plain)) {
        SplitLayers none{};   // (null gain: ones)
        hipLaunchKernelGGL(k_layernorm_layers, dim3((unsigned)rows, 1), dim3(256), 0, st->stream, memory, normed, none, (int)rows, (int)width);
        const size_t tiles = (rows + 255) / 256, mt = ((rows + tiles - 1) / tiles + 63) / 64;   // as few row tiles as there must be, and those small
        const auto launch = [&](auto mt_constant) {
            constexpr int MT = decltype(mt_constant)::value;
            return biased ? launch_wide<MT, true>(st, rows, width, layers, count, xw, normed, k_out, v_out, error, capacity)
                          : launch_wide<MT, false>(st, rows, width, layers, count, xw, normed, k_out, v_out, error, capacity);
        };
        switch (mt) {
            case 1: return launch(std::integral_constant<int, 1>{});
            case 2: return launch(std::integral_constant<int, 2>{});
            case 3: return launch(std::integral_constant<int, 3>{});
            default: return launch(std::integral_constant<int, 4>{});
        }
    }
    hipLaunchKernelGGL(k_layernorm_layers, dim3((unsigned)rows, (unsigned)count), dim3(256), 0, st->stream, memory, normed, layers, (int)rows, (int)width);
    const int mtiles = (int)((rows + 63) / 64), ntiles = (int)((2 * xw + 127) / 128);
    hipLaunchKernelGGL(k_split_cross_kv, dim3((unsigned)((ntiles + 7) / 8 * 8 * mtiles), (unsigned)count), dim3(512), 0, st->stream, normed, layers, (int)rows,
                       (int)width, (int)xw, mtiles, k_out, v_out);
    return hip_check(hipGetLastError(), "cross K/V launch", error, capacity);
}

}  // namespace mynah
