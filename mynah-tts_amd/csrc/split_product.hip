// Products of many f32 rows with a weight, in f32, on the bf16 matrix cores (split_product.h): the encoder prefill with f32
// operands and the cross-attention K/V.  out[m][n] = sum over taps j and channels c of in[m - (taps - 1) + j][c] * W[n][c][j]; one tap is
// a plain product, three are the causal convolution of the encoder's FFN (causal_conv_ffn, src/graph.c:302-352).
#include "split_product.h"

namespace mynah {
namespace {

// The weight lies in memory in the order in which the wavefronts take it: per tile of 32 outputs, block of 32 channels, half of
// the block, tap, and half of a lane's eight values 64 float4s, lane l's being output l % 32, channels 8 * (l / 32) .. of the half.
// A request is then 1 KiB of consecutive bytes, it goes straight to the registers of the one wavefront that multiplies it,
// and it stays four bytes a value (three bf16 pieces would be six, and the weight is read once per 64 rows).
__global__ void __launch_bounds__(256) k_split_pack(const float *src, float4 *dst, size_t pieces, int channels, int taps) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= pieces) return;
    const int lane = (int)(i & 63);
    size_t j = i >> 6;
    const int part = (int)(j & 1);
    j >>= 1;
    const int tap = (int)(j % (size_t)taps);
    j /= (size_t)taps;
    const int half = (int)(j & 1);
    j >>= 1;
    const int blocks = channels / 32, block = (int)(j % (size_t)blocks);
    const size_t n = (j / (size_t)blocks) * 32 + (lane & 31);
    const size_t c = (size_t)block * 32 + half * 16 + (lane >> 5) * 8 + part * 4;
    const float *p = src + (n * (size_t)channels + c) * taps + tap;
    dst[i] = make_float4(p[0], p[taps], p[2 * taps], p[3 * taps]);
}

// LDS of a tile: three stages of one block of 16 G channels (32 * MT + taps - 1 rows), operand-major per 16-deep part, piece and
// 8-deep half, and afterwards the later groups' sums.  The row pitch puts the two halves of a row 64 bytes apart modulo 256; fragment
// reads are 512 consecutive bytes.
template <int MT, int TAPS, int G>
struct SplitTile {
    static constexpr int kRows = 32 * MT + (TAPS - 1), kPitch = (kRows + 11) / 16 * 16 + 4;
    static_assert(kPitch >= kRows && kPitch % 16 == 4 && (G == 2 || G == 4 || G == 8), "bank layout");
    union {
        uint4 a[3][G][3][2][kPitch];
        float sums[8 - 8 / G][MT][16][64];
    };
};

constexpr int kBlocksAhead = 2;   // blocks per round of the loop below: a split's block count is a multiple of it

// acc[t] = the tile's sums over `blocks` blocks of 16 G channels, for rows 32 t .. of the tile and the wavefront's 32 columns;
// valid in the first 8 / G of the eight wavefronts.
// Wavefront w multiplies columns 32 * (w % (8 / G)) .. over the 16-deep part w / (8 / G) of every block: two wavefronts to a SIMD, because
// one alone cannot issue its vector instructions beside its own matrix instructions (a matrix instruction of 16 ns holds its
// wavefront's issue for 10 ns; a step of 12 with its 70 vector instructions took 300 ns alone, 200 ns per wavefront in pairs).
// A wavefront's weight values come from memory three (one tap: two) steps ahead, are taken apart in registers and multiplied;
// the rows are staged by all eight wavefronts, taken apart on the way to LDS, and serve every tap from there.  A block is
// stored into a stage two blocks after it was last read, its requests leave two blocks before that; what runs past the last
// block is requested (the buffers are padded) and not used, so that no request stands under a condition.
template <int MT, int TAPS, int G>
__device__ __forceinline__ void split_tile(const float *const a, const int lda, const int row0, const int rows, const float4 *const w,
                                           const int blocks, SplitTile<MT, TAPS, G> &lds, f32x16 (&acc)[MT]) {
    using Tile = SplitTile<MT, TAPS, G>;
    constexpr int R = TAPS == 1 ? 2 : TAPS, UB = kBlocksAhead;   // steps of weights in flight; blocks per round
    static_assert((UB * TAPS) % R == 0 && UB % 2 == 0, "register stages must repeat with the round");
    const int tid = threadIdx.x, lane = tid & 63, group = tid / (512 / G);
    constexpr int kPass = 512 / (4 * G);   // rows staged at once
    const int srow = tid / (4 * G), sc = tid % (4 * G);
    constexpr int kRows = Tile::kRows, NP = (kRows + kPass - 1) / kPass;
    constexpr int kStage = G * 3 * 2 * Tile::kPitch;
    uint4 *const stages = &lds.a[0][0][0][0][0];
    const float *ap[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) ap[i] = a + (ptrdiff_t)min(row0 - (TAPS - 1) + min(srow + kPass * i, kRows - 1), rows - 1) * lda + 4 * sc;
    float4 ra[2][NP];
    const auto request_a = [&](int set, int block) {
#pragma unroll
        for (int i = 0; i < NP; ++i) ra[set][i] = *reinterpret_cast<const float4 *>(ap[i] + block * (16 * G));
    };
    const auto store_a = [&](int set, uint4 *stage) {
#pragma unroll
        for (int i = 0; i < NP; ++i)
            if (kPass * i + kPass <= kRows || srow + kPass * i < kRows) {
                const SplitFour s(ra[set][i]);
#pragma unroll
                for (int q = 0; q < 3; ++q)
                    reinterpret_cast<uint2 *>(&stage[(((sc >> 2) * 3 + q) * 2 + ((sc >> 1) & 1)) * Tile::kPitch + srow + kPass * i])[sc & 1] = s.piece[q];
            }
    };
    const float4 *wp = w + (size_t)group * (TAPS * 128) + lane;
    float4 rw[R][2];
    const auto request_w = [&](int slot, int step) {   // step counted from wp: block step / TAPS, tap step % TAPS
        const float4 *p = wp + ((step / TAPS) * G * TAPS + step % TAPS) * 128;
        rw[slot][0] = p[0];
        rw[slot][1] = p[64];
    };
    bf16x8 fa[2][MT][3], fw[2][3];
    const auto read_a = [&](int set, const uint4 *stage, int tap) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int q = 0; q < 3; ++q)
                fa[set][t][q] = __builtin_bit_cast(bf16x8, stage[((group * 3 + q) * 2 + (lane >> 5)) * Tile::kPitch + (lane & 31) + 32 * t + tap]);
    };
    int now = 0, next = kStage, after = 2 * kStage;
    request_a(0, 0);
#pragma unroll
    for (int i = 0; i < R; ++i) request_w(i, i);
    request_a(1, 1);
    store_a(0, stages);
    request_a(0, 2);
    __syncthreads();
    read_a(0, stages, 0);
    split_eight(rw[0][0], rw[0][1], fw[0]);
    __builtin_amdgcn_sched_barrier(0);
    for (int block = 0; block < blocks; block += UB) {
#pragma unroll
        for (int u = 0; u < UB; ++u) {
#pragma unroll
            for (int tap = 0; tap < TAPS; ++tap) {
                const int s = u * TAPS + tap;
                request_w(s % R, s + R);   // into the registers taken apart a step ago
                if (tap == 0) {
                    store_a((u + 1) & 1, stages + next);
                    request_a((u + 1) & 1, u + 3);
                }
                if (TAPS == 1) __syncthreads();   // (the next step already reads the block stored here)
                split_eight(rw[(s + 1) % R][0], rw[(s + 1) % R][1], fw[(s + 1) & 1]);
                if (tap + 1 < TAPS) read_a((s + 1) & 1, stages + now, tap + 1);
                else read_a((s + 1) & 1, stages + next, 0);
#pragma unroll
                for (int t = 0; t < MT; ++t) acc[t] = split_multiply(fa[s & 1][t], fw[s & 1], acc[t]);
                // the next step's work between this step's matrix instructions
#pragma unroll
                for (int i = 0; i < 6 * MT; ++i) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);     // a matrix instruction,
                    __builtin_amdgcn_sched_group_barrier(0x2, 5, 0);     // five vector instructions,
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // one LDS read
                }
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
    __syncthreads();
    if (group > 0) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) lds.sums[(tid >> 6) - 8 / G][t][r][lane] = acc[t][r];
    }
    __syncthreads();
    if (group == 0) {
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r)
#pragma unroll
                for (int g = 1; g < G; ++g) acc[t][r] += lds.sums[(tid >> 6) + (g - 1) * (8 / G)][t][r][lane];
    }
}

// A finished tile to memory, a lane's column at `out`.  A sum that is no finite number is stored again as the chain of f32 multiply-adds
// over the same blocks (split_product.h): looked for behind the stores, where it is cheapest (before them: 0.4 us a launch).
template <int MT, int TAPS>
__device__ __forceinline__ void split_store(const float *const a, const int lda, const int row0, const int rows, const float4 *const w, const int blocks,
                                            const f32x16 (&acc)[MT], float *const out, const int pitch) {
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
            for (int c = 0; c < 32 * blocks && s == s; c += 4)
#pragma unroll
                for (int tap = 0; tap < TAPS; ++tap) {
                    const int row = m - (TAPS - 1) + tap;
                    if (row < 0) continue;
                    const float4 x = *reinterpret_cast<const float4 *>(a + (size_t)row * lda + c);
                    const float4 v = w[((c >> 4) * TAPS + tap) * 128 + ((c >> 2) & 1) * 64 + ((c >> 3) & 1) * 32 + (lane & 31)];
                    s = __builtin_fmaf(x.x, v.x, s);
                    s = __builtin_fmaf(x.y, v.y, s);
                    s = __builtin_fmaf(x.z, v.z, s);
                    s = __builtin_fmaf(x.w, v.w, s);
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
__global__ void __launch_bounds__(512) k_split_rows(const float *const a, const float4 *const w, const int M, const int N, const int channels, const int mtiles,
                                                    const int ntiles, const int splits, float *const part) {
    __shared__ SplitTile<MT, TAPS, G> lds;
    constexpr int kWide = 8 / G, kDeep = 16 * G;
    const SplitWork work((int)blockIdx.x, mtiles);
    if (work.nz >= ntiles * splits) return;
    const int lane = threadIdx.x & 63, wave = (threadIdx.x >> 6) % kWide;
    const int z = work.nz / ntiles, share = channels / splits;
    const int col0 = ((work.nz % ntiles) * kWide + wave) * 32, m0 = work.m * 32 * MT;
    f32x16 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = f32x16{0};
    const float4 *tile = w + ((size_t)(min(col0, N - 32) / 32) * (channels / 16) + z * (share / 16)) * (TAPS * 128);
    split_tile<MT, TAPS, G>(a + z * share, channels, m0, M, tile, share / kDeep, lds, acc);
    if (threadIdx.x >= 64 * kWide || col0 >= N) return;
    split_store<MT, TAPS>(a + z * share, channels, m0, M, tile, share / 32, acc, part + (size_t)z * M * N + col0 + (lane & 31), N);
}

// The K and V halves of every layer's kv_net on that layer's normalised memory, one launch.  The column tiles of all layers make one
// list, of which an XCD takes every eighth: layer by layer the twelve of a 768-wide one give XCDs 0 to 3 two each and the others one, and the
// launch waits for the fullest.  `places` of the list are a layer's: its tiles, or (launch_split_cross_kv) the next multiple of eight.
// (Two workgroups to a CU at 180 rows, some 23 ns a matrix instruction with its 6.4 vector instructions; a pass over the weight to have it in L2 first: slower.)
__global__ void __launch_bounds__(512) k_split_cross_kv(const float *const normed, const SplitLayers weights, const int M, const int width, const int xw,
                                                        const int mtiles, const int layers, const int places, float *const k_out, float *const v_out) {
    __shared__ SplitTile<2, 1, 2> lds;
    const int N = 2 * xw, ntiles = (N + 127) / 128;
    const SplitWork work((int)blockIdx.x, mtiles);
    const int layer = work.nz / places, ntile = work.nz - layer * places;
    if (layer >= layers || ntile >= ntiles) return;
    const int lane = threadIdx.x & 63, wave = (threadIdx.x >> 6) & 3;
    const int col0 = ntile * 128 + wave * 32, m0 = work.m * 64;
    f32x16 acc[2] = {f32x16{0}, f32x16{0}};
    const float4 *tile = weights.w[layer] + (size_t)(min(col0, N - 32) / 32) * (width / 32) * 256;
    split_tile<2, 1, 2>(normed + (size_t)layer * M * width, width, m0, M, tile, width / 32, lds, acc);
    if (threadIdx.x >= 256 || col0 >= N) return;
    float *const out = (col0 < xw ? k_out + col0 : v_out + col0 - xw) + (size_t)layer * M * xw + (lane & 31);
    split_store<2, 1>(normed + (size_t)layer * M * width, width, m0, M, tile, width / 32, acc, out, xw);
}

// The memory's rows under every layer's LayerNorm (gain, optional bias), one workgroup per row and layer: normed[layer][row].
__global__ void __launch_bounds__(256) k_layernorm_layers(const float *in, float *normed, const SplitLayers layers, int rows, int width) {
    __shared__ float s4[4];
    const int row = (int)blockIdx.x, layer = (int)blockIdx.y;
    layernorm_row(in + (size_t)row * width, normed + ((size_t)layer * rows + row) * width, layers.gain[layer], layers.bias[layer], width, s4);
}

// The same, and the table of the products that follow, which the first workgroup leaves in device memory: what changes from call to call
// arrives as arguments, and nothing is copied.
__global__ void __launch_bounds__(256) k_layernorm_products(const float *in, float *normed, const SplitLayers layers, int rows, int width,
                                                            LinearProduct *list, const CrossProducts products, int count) {
    __shared__ float s4[4];
    const int row = (int)blockIdx.x, layer = (int)blockIdx.y;
    if (row == 0 && layer == 0 && (int)threadIdx.x < count) list[threadIdx.x] = products.of[threadIdx.x];
    layernorm_row(in + (size_t)row * width, normed + ((size_t)layer * rows + row) * width, layers.gain[layer], layers.bias[layer], width, s4);
}

}  // namespace

int launch_cross_norms(State *st, const float *memory, size_t rows, size_t width, const SplitLayers &layers, size_t count, float *normed,
                       const CrossProducts *products, LinearProduct *list, char *error, size_t capacity) {
    static_assert(2 * kSplitMaxLayers <= 256, "a thread an entry of the table");
    const dim3 grid((unsigned)rows, (unsigned)count);
    if (list != nullptr)
        hipLaunchKernelGGL(k_layernorm_products, grid, dim3(256), 0, st->stream, memory, normed, layers, (int)rows, (int)width, list, *products, (int)(2 * count));
    else
        hipLaunchKernelGGL(k_layernorm_layers, grid, dim3(256), 0, st->stream, memory, normed, layers, (int)rows, (int)width);
    return hip_check(hipGetLastError(), "cross K/V LayerNorm launch", error, capacity);
}

int launch_split_pack(State *st, const float *src, float4 *dst, size_t n, size_t channels, size_t taps, char *error, size_t capacity) {
    const size_t pieces = n * channels * taps / 4;
    hipLaunchKernelGGL(k_split_pack, dim3((unsigned)((pieces + 255) / 256)), dim3(256), 0, st->stream, src, dst, pieces, (int)channels, (int)taps);
    return hip_check(hipGetLastError(), "weight packing launch", error, capacity);
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

// Groups of wavefronts over the channels: the most, and so the narrowest tile (256 / groups columns), that still give every workgroup a CU of
// its own.  What bounds these launches is how fast a CU gets its piece of the weight, and few rows make few workgroups: with four groups a
// workgroup has half the piece, with eight (tiles of 32 rows) a quarter.  us a prefill of six layers with two groups (four in the unsplit
// QKV product) / this, one tap: 20 rows 292 / 274, 60 325 / 308, 96 344 / 332; three taps: 20 350 / 318, 60 386 / 351, 96 410 / 398.  A quarter more
// workgroups than CUs instead: 303, 325, 353 and 341, 380, 448.
// A sum is then more and shorter chains of additions: the prefill's error against double precision (2-norm) 4.5e-7 / 3.7e-7 at 20 rows, 4.5e-7 /
// 3.9e-7 at 50 with one tap, 6.3e-7 / 5.4e-7 and 6.6e-7 / 5.6e-7 with three.
// A group of 32 channels, one round of the loop, pays for one more share of the sums to add where its weights are three taps or the row tiles are two at most:
// four layers of width 256, one tap, us with groups of 64 at least / of 32: 16 rows 149.2 / 147.8, 64 167.7 / 165.7, 129 189.6 / 191.6, 160 189.6 / 191.9, 256 211.2 / 212.9;
// three taps 16 rows 166.0 / 159.8, 256 235.9 / 229.1.
static int split_groups(const State *st, size_t mt, size_t mtiles, size_t channels, size_t taps, size_t n, size_t splits) {
    const size_t least = taps == 3 || mtiles <= 2 ? 32 : 64;
    for (size_t groups = mt == 1 ? 8 : 4; groups > 2; groups /= 2)
        if (channels >= least * groups * splits && channels % (16 * groups * kBlocksAhead * splits) == 0 && (n * groups + 255) / 256 * mtiles * splits <= (size_t)st->cu_count) return (int)groups;
    return 2;
}

int launch_split_product(State *st, const float *in, const float4 *w, size_t rows, size_t channels, size_t taps, size_t n, int splits, float *part,
                         char *error, size_t capacity) {
    if (rows == 0 || n == 0 || n % 32 != 0 || channels == 0 || splits < 1 || channels % (32 * kBlocksAhead * (size_t)splits) != 0 || (taps != 1 && taps != 3) ||
        rows > 0x100000 || n > 0x100000 || channels > 0x100000) {
        set_error(error, capacity, "f32 product: shape outside the matrix-core kernel's");
        return -1;
    }
    const int mt = split_row_tiles(st, rows, n, splits > 1), mtiles = (int)((rows + 32 * mt - 1) / (32 * mt));
    const int groups = split_groups(st, (size_t)mt, (size_t)mtiles, channels, taps, n, (size_t)splits);
    const int wide = 256 / groups, ntiles = (int)((n + wide - 1) / wide);
    const dim3 grid((unsigned)((ntiles * splits + 7) / 8 * 8 * mtiles)), block(512);
    const auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, block, 0, st->stream, in, w, (int)rows, (int)n, (int)channels, mtiles, ntiles, splits, part);
    };
    if (taps == 1) {
        if (mt == 1) groups == 8 ? launch(k_split_rows<1, 1, 8>) : groups == 4 ? launch(k_split_rows<1, 1, 4>) : launch(k_split_rows<1, 1, 2>);
        else groups == 4 ? launch(k_split_rows<2, 1, 4>) : launch(k_split_rows<2, 1, 2>);
    } else {
        if (mt == 1) groups == 8 ? launch(k_split_rows<1, 3, 8>) : groups == 4 ? launch(k_split_rows<1, 3, 4>) : launch(k_split_rows<1, 3, 2>);
        else groups == 4 ? launch(k_split_rows<2, 3, 4>) : launch(k_split_rows<2, 3, 2>);
    }
    return hip_check(hipGetLastError(), "f32 product launch", error, capacity);
}

int launch_split_cross_kv(State *st, const float *memory, size_t rows, size_t width, const SplitLayers &layers, size_t count, size_t xw, float *normed,
                          float *k_out, float *v_out, char *error, size_t capacity) {
    if (launch_cross_norms(st, memory, rows, width, layers, count, normed, nullptr, nullptr, error, capacity) != 0) return -1;
    const int mtiles = (int)((rows + 63) / 64), ntiles = (int)((2 * xw + 127) / 128);
    // Layers one behind the other in the list, or each from a multiple of eight on (its first tile on XCD 0), by what the fullest XCD has to do.  The list is the
    // shorter, but where either way some CUs have two workgroups and the list gives them to only a few of each XCD, layer by layer
    // is faster.  us a call, layers of 768, layer by layer / list (workgroups of the fullest XCD, 32 CUs): twelve layers, 64 rows 23.4 / 23.5 (24 / 18), 100 35.8 /
    // 37.0 (48 / 36), 180 53.9 / 42.8 (72 / 54), 256 61.6 / 59.4 (96 / 72), 320 78.5 / 63.6; 128 rows, nine layers 34.7 / 25.8 (36 / 28), eleven 35.6 / 37.2 (44 / 34),
    // fourteen 39.1 / 39.5 (56 / 42), sixteen 42.6 / 42.2 (64 / 48); 192 rows, ten layers 41.1 / 40.8 (60 / 45); six layers of 256 rows 36.6 / 38.0 (48 / 36).
    const int cus = st->cu_count / 8, apart = (ntiles + 7) / 8 * (int)count * mtiles, together = (ntiles * (int)count + 7) / 8 * mtiles;
    const bool by_layer = together > cus && together <= cus + 3 * cus / 8 && apart <= 2 * cus;
    const int places = by_layer ? (ntiles + 7) / 8 * 8 : ntiles;
    hipLaunchKernelGGL(k_split_cross_kv, dim3((unsigned)((places * (int)count + 7) / 8 * 8 * mtiles)), dim3(512), 0, st->stream, normed, layers,
                       (int)rows, (int)width, (int)xw, mtiles, (int)count, places, k_out, v_out);
    return hip_check(hipGetLastError(), "cross K/V launch", error, capacity);
}

}  // namespace mynah
