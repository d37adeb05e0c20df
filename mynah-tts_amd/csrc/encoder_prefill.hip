// Text-encoder prefill on the matrix cores: the dense, many-rows twin of the decode step.
//
// encode_text / transformer_stack (src/graph.c:713-748, :634-711) run, per layer, LayerNorm -> QKV
// linear -> per-head scaled QK^T -> row softmax -> PV -> O -> residual -> LayerNorm -> FFN -> residual
// through an f32 BLAS.  Here the weights are f16 (converted once at load, IEEE round to nearest even,
// third_party/ingot/src/dtype.c:246-268), the activations entering a product are rounded to f16, and
// every product accumulates in f32 on v_mfma_f32_32x32x16_f16.  The residual stream, the LayerNorm
// statistics, the softmax and the GELU stay f32.  Attention is bidirectional or causal (the mask of
// src/graph.c:446-449: query t sees keys 0 .. t).  The FFN is causal_conv_ffn (src/graph.c:302-352) with kernel 1
// (two plain products) or kernel 3: out[t][o] = sum_{i,j} W[o][i][j] * in[t - 2 + j][i], rows before the first
// being zero.  The conv is an NT product too: its weights are stored tap-major, W'[o][j * in + i], so that the
// A operand of token t is rows t-2, t-1, t of the activation side by side, and a K step of the product reads one
// of those rows -- addressing only, no unfolded copy.  The two rows before row 0 of nrm and hid exist and stay zero.
//
// Layout in device memory (T tokens padded to a multiple of 64 rows; pad rows are kept finite and are
// masked out as attention keys, so they never reach a real row):
//   x    f32 [Tpad, w]       residual stream
//   nrm  f16 [2 + Tpad, w]   LayerNorm output = A operand of the QKV / FFN-up products (after two zero rows)
//   qk   f16 [2, heads, Tpad/32][2048]   q, then k, operand-major: per (head, 32-token tile) the 32 x 64 block in the order in
//                            which a wavefront's four matrix instructions take it -- element (token r of the tile, d) at
//                            ((d / 16) * 64 + ((d % 16) / 8) * 32 + r) * 8 + d % 8 -- so that one operand request of
//                            the attention kernel is 1 KiB of consecutive bytes (read row-major, lane l: 16 bytes of row
//                            l % 32, a request touches 32 cache lines for 32 bytes each)
//   vt   f16 [heads*2, Tpad/16][512]     v, operand-major for PV (rows = 32 output columns, inner index = 16 keys): element
//                            (d, t) at block (d / 32, t / 16), ((t % 16) / 8 * 32 + d % 32) * 8 + t % 8
//   ctx  f16 [Tpad, w]       attention output = A operand of the O product
//   hid  f16 [2 + Tpad, ffn] GELU(up) = A operand of the FFN-down product (after two zero rows)
//   part f32 [4, Tpad, w]    K-split partial sums of the O and FFN-down products; the row pass that follows
//                            adds them to x in a fixed order (no atomics: results do not depend on scheduling)
//
// All products are "NT": C[m][n] = sum_k A[m][k] * W[n][k], both operands K-contiguous, which is how
// the 32x32x16 MFMA wants them: lane l supplies row (l % 32) of A (or of W) and the eight consecutive
// k values 8*(l / 32) .. +7 of the 16-deep step.
#include <algorithm>
#include <new>

#include "device_common.h"

using namespace mynah;

// Per-call values read by the kernels from device memory, so that one captured graph per padded length
// serves every call: the token count and the caller's output pointers.
struct EncParams {
    int tokens;
    int reserved;
    uint16_t *embed_out;
    float *out;
};

struct mynah_hip_encoder {
    size_t layers = 0, width = 0, heads = 0, head_width = 0, ffn = 0, vocab = 0, max_positions = 0, tpad_max = 0;
    size_t taps = 1;           // FFN conv kernel size, 1 or 3
    int causal = 0;
    const CachedWeight *tok = nullptr, *pos = nullptr;
    std::vector<const CachedWeight *> qkv, o, up, down;
    std::vector<_Float16 *> conv_up, conv_down;   // taps == 3: tap-major f16 copies owned by the encoder
    std::vector<const float *> n1g, n1b, n2g, n2b;
    const float *nog = nullptr, *nob = nullptr;
    float *x = nullptr, *part = nullptr;   // part: [splits, Tpad, w] partial products of the O and FFN-down products
    _Float16 *nrm = nullptr, *qk = nullptr, *vt = nullptr, *ctx = nullptr, *hid = nullptr;
    _Float16 *nrm_alloc = nullptr, *hid_alloc = nullptr;   // nrm and hid begin kLeadRows rows into these
    EncParams *params = nullptr;
    std::unordered_map<int, hipGraphExec_t> graphs;   // by padded length
    std::unordered_map<int, int> eager_runs;          // a padded length runs eagerly once before it is captured
    size_t max_lds = 0;
    // f32 operands (the reference's own arithmetic, src/graph.c:634-711: every product an f32 GEMM): f32 tables, weights in the
    // order of split_product.hip, f32 rows padded like the f16 form's
    bool f32 = false;
    const CachedWeight *tok32 = nullptr, *pos32 = nullptr;
    std::vector<const float4 *> qkv32, o32, up32, down32;
    float *f_nrm = nullptr, *f_qkv = nullptr, *f_ctx = nullptr, *f_hid = nullptr;
    float *f_nrm_alloc = nullptr, *f_hid_alloc = nullptr;   // f_nrm and f_hid begin kLeadRows rows into these
};

namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int kTile = 64;            // widths and padded lengths are multiples of this; the products' largest tile is 64 x 64
constexpr int kStep = 64;            // K step of the products
constexpr int kQTile = 32;           // queries per attention workgroup
constexpr int kScorePad = 8;         // floats appended to a score row (bank spread for the row-wise softmax)
constexpr int kLeadRows = 2;         // zero rows in front of the conv FFN's activations (kernel size 3 looks two rows back)

enum { ENC_QKV = 0, ENC_PARTIAL = 1, ENC_GELU = 2 };

struct GemmArgs {
    const _Float16 *a;     // [M, K] row-major, lda = K
    const _Float16 *w;     // [N, K]
    int M, N, K;
    float *part;           // ENC_PARTIAL: part[z][m][n] = this K split's share of the product (summed by the next LayerNorm pass)
    _Float16 *out;         // ENC_QKV: qk [M, 2*width];  ENC_GELU: hid [M, N]
    _Float16 *vt;          // ENC_QKV: v, operand-major (see the layout note)
    int width;
    int taps, cin;         // conv form: K = taps * cin, A is [M, cin] with (taps - 1) zero rows before row 0
};

// tanh-GELU (src/kernels.c:382-389) for a value that is rounded to f16 at once: 0.5 x (1 + tanh c) = x / (1 + e^(-2c)),
// with the hardware exponential and reciprocal (relative error about 1e-6, a five-hundredth of the f16 rounding that
// follows).  c -> -inf gives x * 0, c -> +inf gives x.  The decode step's GELU is gelu_tanh of device_common.h, with tanhf.
__device__ __forceinline__ float gelu_tanh_for_f16(float x) {
    const float cubic = x * x * x;
    const float c = 0.7978845608f * (x + 0.044715f * cubic);
    return x * __builtin_amdgcn_rcpf(1.0f + __expf(-2.0f * c));
}

// Row of C held in accumulator register r of lane l for a 32x32 MFMA tile; the column is l % 32.
__device__ __forceinline__ int acc_row(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

// What becomes of a wavefront's finished 32 x 32 piece (registers as acc_row has them): rows from mbase, this lane's column n.
template <int EPI>
__device__ __forceinline__ void finish_piece(const GemmArgs &g, const floatx16 &acc, int mbase, int n, int lane, int split) {
    if constexpr (EPI == ENC_PARTIAL) {
        float *part = g.part + (size_t)split * g.M * g.N;
#pragma unroll
        for (int r = 0; r < 16; ++r) part[(size_t)(mbase + acc_row(r, lane)) * g.N + n] = acc[r];
    } else if constexpr (EPI == ENC_GELU) {
#pragma unroll
        for (int r = 0; r < 16; ++r) g.out[(size_t)(mbase + acc_row(r, lane)) * g.N + n] = (_Float16)gelu_tanh_for_f16(acc[r]);
    } else {
        // q, k and v leave in the order in which the attention kernel's matrix instructions take them (see the layout
        // note at the top): a wavefront's 32 x 32 piece lies inside one (part, head, 32-token tile) block.
        const int heads = g.width / 64;
        if (n < 2 * g.width) {   // uniform per workgroup: width is a multiple of the tile
            const int part = n >= g.width ? 1 : 0, d = n & 63, head = (n - part * g.width) >> 6;
            _Float16 *block = g.out + ((size_t)(part * heads + head) * (g.M / 32) + mbase / 32) * 2048 + ((d >> 4) * 64 + ((d >> 3) & 1) * 32) * 8 + (d & 7);
#pragma unroll
            for (int r = 0; r < 16; ++r) block[acc_row(r, lane) * 8] = (_Float16)acc[r];
        } else {
            const int d = n - 2 * g.width;   // d / 32: the (head, 32-column half) block row; d % 32 = lane % 32
            _Float16 *block = g.vt + ((size_t)(d >> 5) * (g.M / 16) + mbase / 16) * 512 + (d & 31) * 8 + 4 * (lane >> 5);
#pragma unroll
            for (int q = 0; q < 4; ++q) {   // registers 4q .. 4q+3 are the four consecutive tokens mbase + 8q + 4 (lane / 32) ..
                half4 v = {(_Float16)acc[4 * q], (_Float16)acc[4 * q + 1], (_Float16)acc[4 * q + 2], (_Float16)acc[4 * q + 3]};
                *reinterpret_cast<half4 *>(block + (q >> 1) * 512 + (q & 1) * 256) = v;
            }
        }
    }
}

// 64 lanes' 16 bytes from base + lane_bytes to consecutive LDS bytes from `lds` on (base and lds the same for the whole wavefront).
__device__ __forceinline__ void global_to_lds(const void *base, unsigned lane_bytes, unsigned lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(lane_bytes), "s"(base) : "memory", "m0");
}

// Waits until at most PER requests for each of the `left` steps behind this one (MOST at most) are out and this wavefront's LDS
// reads are done, then (MEET) for the workgroup's other wavefronts.
template <int PER, int MOST, bool MEET>
__device__ __forceinline__ void step_arrived(int left) {
    if (left >= MOST) {
        if constexpr (MEET) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(PER * MOST) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(PER * MOST) : "memory");
    } else if constexpr (MOST > 0) {
        step_arrived<PER, MOST - 1, MEET>(left);
    }
}

// C tile of 32 * WM rows and 32 * WN columns, a wavefront 32 x 32 of it, K in steps of 64 through a ring of D stages in LDS.
// The operands go from global memory straight to LDS, D - 2 steps ahead of their use: no registers, no LDS stores, one wait and one
// barrier (none where a tile is one wavefront's) a step.  What bounds a launch at these sizes is how fast one CU gets its tile's rows
// (some 64 KB in flight, a round trip for each such piece) and the step's own chain; through registers that was store, request,
// barrier, read, multiply, on 64 x 64 tiles always.  us a prefill then / now, tokens: 20 211 / 176, 100 216 / 191, 192 223 / 208, 256 227 / 221,
// 384 276 / 260, 512 315 / 287; three taps: 60 297 / 247, 128 294 / 255, 256 305 / 299, 400 414 / 392.
// Iteration kt: wait for step kt, meet, request step kt + D - 2 (over step kt - 2, whose reads every wavefront has finished), read kt's
// fragments, multiply step kt - 1 meanwhile.  A value's additions run over k in ascending order whatever the tile.
// CONV: the A operand of K step s is the 64 channels (s % (cin / 64)) * 64 .. of row m - (taps - 1) + s / (cin / 64).
// The fields of GemmArgs as scalar arguments, in the order in which the kernel needs them: the first fourteen dwords of
// scalar kernel arguments are in registers when a wavefront starts (the build asks for that), a structure passed by value
// is fetched from memory.
template <int EPI, int WM, int WN, int D, bool CONV>
__global__ void __launch_bounds__(64 * WM * WN)
k_enc_gemm(const _Float16 *const a_arg, const _Float16 *const w_arg, const int M, const int N, const int K, const int steps, const int cin, const int taps,
           float *const part, _Float16 *const out, _Float16 *const vt, const int width) {
    GemmArgs g;
    g.a = a_arg; g.w = w_arg; g.M = M; g.N = N; g.K = K; g.part = part; g.out = out; g.vt = vt; g.width = width;
    g.taps = taps; g.cin = cin;
    constexpr int kWaves = WM * WN, kRowBytes = kStep * 2, kTileA = 32 * WM * kRowBytes, kStage = kTileA + 32 * WN * kRowBytes;
    constexpr int kAskA = 4 * WM / kWaves, kAskW = 4 * WN / kWaves;   // a wavefront's requests a step: eight rows of 128 bytes each
    static_assert(D >= 4 && (kAskA + kAskW) * (D - 3) < 64, "the wait's counter ends at 63");
    __shared__ __align__(16) unsigned char stages[D * kStage];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int wm = wave % WM, wn = wave / WM;
    const int m0 = blockIdx.y * 32 * WM, n0 = blockIdx.x * 32 * WN, first = (int)blockIdx.z * steps;   // (blockIdx.z: the K split)
    const int lda = CONV ? g.cin : g.K;
    // LDS piece s of row r holds the row's 16-byte piece s ^ (r % 8): a request writes consecutive bytes, eight rows without padding,
    // and the fragment reads of eight rows still lie on different banks.
    const unsigned piece = (unsigned)((lane & 7) ^ (lane >> 3)) * 16;
    const unsigned lane_a = (unsigned)(wave * kAskA * 8 + (lane >> 3)) * (unsigned)lda * 2 + piece;
    const unsigned lane_w = (unsigned)(wave * kAskW * 8 + (lane >> 3)) * (unsigned)g.K * 2 + piece;
    const unsigned char *const abase = reinterpret_cast<const unsigned char *>(g.a + (ptrdiff_t)m0 * lda);
    const unsigned char *const wbase = reinterpret_cast<const unsigned char *>(g.w + (size_t)n0 * g.K) + (ptrdiff_t)first * kRowBytes;
    const int steps_per_tap = CONV ? g.cin / kStep : 1;
    const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char *)stages;
    const auto request = [&](int step, int slot) {
        const unsigned char *a;
        if constexpr (!CONV) a = abase + (ptrdiff_t)(first + step) * kRowBytes;
        else {
            const int s = first + step, tap = (s >= steps_per_tap ? 1 : 0) + (s >= 2 * steps_per_tap ? 1 : 0);   // taps <= 3
            a = abase + ((ptrdiff_t)(tap - (g.taps - 1)) * lda + (ptrdiff_t)(s - tap * steps_per_tap) * kStep) * 2;
        }
        const unsigned char *const w = wbase + (ptrdiff_t)step * kRowBytes;
        const unsigned to_a = lds0 + slot * kStage + wave * kAskA * 1024, to_w = lds0 + slot * kStage + kTileA + wave * kAskW * 1024;
#pragma unroll
        for (int i = 0; i < kAskA; ++i) global_to_lds(a, lane_a + (unsigned)(i * 16 * lda), to_a + i * 1024);
#pragma unroll
        for (int i = 0; i < kAskW; ++i) global_to_lds(w, lane_w + (unsigned)(i * 16 * g.K), to_w + i * 1024);
    };
#pragma unroll
    for (int d = 0; d < D - 2; ++d)
        if (d < steps) request(d, d);

    floatx16 acc = {0};
    half8 fa[2][kStep / 16], fw[2][kStep / 16];   // fragments of step kt in set kt % 2
    const int row = lane & 31, high = lane >> 5;
    int slot = 0, next = D - 2;
    const auto iteration = [&](int kt, int set) {
        const int left = steps - 1 - kt;
        step_arrived<kAskA + kAskW, D - 3, (kWaves > 1)>(left);
        if (left >= D - 2) {
            request(kt + D - 2, next);
            next = next + 1 == D ? 0 : next + 1;
        }
        const unsigned char *const sa = stages + slot * kStage + (wm * 32 + row) * kRowBytes, *const sw = stages + slot * kStage + kTileA + (wn * 32 + row) * kRowBytes;
        slot = slot + 1 == D ? 0 : slot + 1;
#pragma unroll
        for (int j = 0; j < kStep / 16; ++j) {
            const int at = ((2 * j + high) ^ (row & 7)) * 16;
            fa[set][j] = *reinterpret_cast<const half8 *>(sa + at);
            fw[set][j] = *reinterpret_cast<const half8 *>(sw + at);
        }
        if (kt > 0) {
#pragma unroll
            for (int j = 0; j < kStep / 16; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[set ^ 1][j], fw[set ^ 1][j], acc, 0, 0, 0);
        }
    };
    const auto last = [&](int set) {
#pragma unroll
        for (int j = 0; j < kStep / 16; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[set][j], fw[set][j], acc, 0, 0, 0);
    };
    int kt = 0;
    for (; kt + 1 < steps; kt += 2) {
        iteration(kt, 0);
        iteration(kt + 1, 1);
    }
    if (kt < steps) {
        iteration(kt, 0);
        last(0);
    } else {
        last(1);
    }
    finish_piece<EPI>(g, acc, m0 + wm * 32, n0 + wn * 32 + (lane & 31), lane, (int)blockIdx.z);
}

// A lane's part of a row pass from here on: the LayerNorm of the row it holds in v (pieces past the row are zero), written as f16
// (operand of the next product) or f32.  Two-pass statistics (src/kernels.c:186-244, eps 1e-5).
enum { ROWS_RESULT = 0, ROWS_F16 = 1, ROWS_F32 = 2 };   // params->out (real rows only), f16 operand rows, f32 operand rows
template <int OUT, int NV>
__device__ __forceinline__ void norm_row(const float4 (&v)[NV], const float4 (&gg)[NV], const float4 (&bb)[NV], int lane, int row, int width, void *out_rows) {
    const int n4 = width / 4;
    float s = 0.0f;
#pragma unroll
    for (int u = 0; u < NV; ++u) s += (v[u].x + v[u].y) + (v[u].z + v[u].w);   // pieces past the row are zero
    const float mean = wave_sum(s) / (float)width;
    float q = 0.0f;
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        if (lane + 64 * u < n4) {
            const float a = v[u].x - mean, b = v[u].y - mean, c = v[u].z - mean, d = v[u].w - mean;
            q += (a * a + b * b) + (c * c + d * d);
        }
    }
    const float rstd = 1.0f / sqrtf(wave_sum(q) / (float)width + 1.0e-5f);
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int i = lane + 64 * u;
        if (i < n4) {
            const float y0 = (v[u].x - mean) * rstd * gg[u].x + bb[u].x, y1 = (v[u].y - mean) * rstd * gg[u].y + bb[u].y;
            const float y2 = (v[u].z - mean) * rstd * gg[u].z + bb[u].z, y3 = (v[u].w - mean) * rstd * gg[u].w + bb[u].w;
            if constexpr (OUT == ROWS_F16) {
                half4 h = {(_Float16)y0, (_Float16)y1, (_Float16)y2, (_Float16)y3};
                reinterpret_cast<half4 *>(static_cast<_Float16 *>(out_rows) + (size_t)row * width)[i] = h;
            } else {
                reinterpret_cast<float4 *>(static_cast<float *>(out_rows) + (size_t)row * width)[i] = make_float4(y0, y1, y2, y3);
            }
        }
    }
}

// Row pass between two products, one wavefront per row: first the residual update
// x += sum over K splits of the previous product's partials (src/graph.c:470, :316), then LayerNorm (norm_row), the
// encoder's output going to params->out, rows below params->tokens only.  gain == nullptr: no
// LayerNorm, the updated row is copied out as f32.  A lane keeps its NV float4 pieces of the row in
// registers (width <= 256 * NV; the widest supported row, 4096, takes NV = 16).
// (Argument order: what the row's first requests are formed from stands among the first fourteen dwords, which are in registers
// at wavefront start; bias and the f16 destination, needed last, come out of memory.)
// RPW: rows (wavefronts) per workgroup.  One: a row's 3 KB and the up to four partial planes that go with it are 15 KB of
// requests, and four rows to a workgroup put 60 KB through one CU's L1 while three quarters of the CUs have nothing to do
// (256 rows: 64 workgroups) -- a row per workgroup spreads them over the chip.
// No request stands under a condition (a place beyond the row, or a partial plane the product did not write, asks for a
// place that exists and is set to zero afterwards): the waits then name exactly the requests they need.
template <int OUT, int NV, int RPW>
__global__ void __launch_bounds__(64 * RPW) k_enc_rows(float *x, const float *part, const EncParams *params, int rows, int width, int splits,
                                                        size_t split_stride, const float *gain, const float *bias, void *out_rows) {
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * RPW + (threadIdx.x >> 6);
    if (row >= rows) return;
    if constexpr (OUT == ROWS_RESULT) {
        if (row >= params->tokens) return;
    }
    float4 *xr = reinterpret_cast<float4 *>(x + (size_t)row * width);
    const int n4 = width / 4;
    const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);
    float4 v[NV], gg[NV], bb[NV];
    const float4 *const gain4 = reinterpret_cast<const float4 *>(gain != nullptr ? gain : x);   // (x: a place that exists)
    const float4 *const bias4 = reinterpret_cast<const float4 *>(bias != nullptr ? bias : x);
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int i = lane + 64 * u, at = i < n4 ? i : n4 - 1;
        v[u] = xr[at];
        gg[u] = gain4[at];
        bb[u] = bias4[at];
    }
    if (part != nullptr) {
        // the splits are requested kSplits at a time and added in split order: the sum does not depend on how the splits were
        // scheduled.  (The f16 products make at most four planes; the f32 form, whose products have more K to split, up to kMaxSplitsF32.)
        constexpr int kSplits = OUT == ROWS_F16 ? 4 : 6;
        float4 t[NV];
#pragma unroll
        for (int u = 0; u < NV; ++u) t[u] = zero4;
        for (int z0 = 0; z0 < (OUT == ROWS_F16 ? 1 : splits); z0 += kSplits) {
            float4 p[kSplits][NV];
#pragma unroll
            for (int z = 0; z < kSplits; ++z) {
                const float4 *const plane = reinterpret_cast<const float4 *>(part + (z0 + z < splits ? z0 + z : splits - 1) * split_stride + (size_t)row * width);
#pragma unroll
                for (int u = 0; u < NV; ++u) {
                    const int i = lane + 64 * u;
                    p[z][u] = plane[i < n4 ? i : n4 - 1];
                }
            }
#pragma unroll
            for (int u = 0; u < NV; ++u) {
#pragma unroll
                for (int z = 0; z < kSplits; ++z)
                    if (z0 + z >= splits || lane + 64 * u >= n4) p[z][u] = zero4;
            }
#pragma unroll
            for (int u = 0; u < NV; ++u) {
#pragma unroll
                for (int z = 0; z < kSplits; ++z) { t[u].x += p[z][u].x; t[u].y += p[z][u].y; t[u].z += p[z][u].z; t[u].w += p[z][u].w; }
            }
        }
#pragma unroll
        for (int u = 0; u < NV; ++u) {
            const int i = lane + 64 * u;
            if (i >= n4) v[u] = zero4;
            v[u].x += t[u].x; v[u].y += t[u].y; v[u].z += t[u].z; v[u].w += t[u].w;
            if (i < n4) xr[i] = v[u];
        }
    }
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const bool in = lane + 64 * u < n4;
        if (!in) v[u] = zero4;
        if (!in || gain == nullptr) gg[u] = zero4;
        if (!in || bias == nullptr) bb[u] = zero4;
    }
    if (gain == nullptr) {
        if constexpr (OUT == ROWS_RESULT) {
#pragma unroll
            for (int u = 0; u < NV; ++u)
                if (lane + 64 * u < n4) reinterpret_cast<float4 *>(params->out + (size_t)row * width)[lane + 64 * u] = v[u];
        }
        return;
    }
    norm_row<OUT, NV>(v, gg, bb, lane, row, width, OUT == ROWS_RESULT ? static_cast<void *>(params->out) : out_rows);
}

template <int OUT>
void launch_rows(State *st, int width, float *x, const float *part, int splits, size_t split_stride, const float *gain, const float *bias, void *out_rows,
                 const EncParams *params, int rows) {
    constexpr int kRowsPerWg = 1;
    const dim3 rows_grid((unsigned)((rows + kRowsPerWg - 1) / kRowsPerWg));
    if (width <= 1024)
        hipLaunchKernelGGL((k_enc_rows<OUT, 4, kRowsPerWg>), rows_grid, dim3(64 * kRowsPerWg), 0, st->stream, x, part, params, rows, width, splits, split_stride,
                           gain, bias, out_rows);
    else
        hipLaunchKernelGGL((k_enc_rows<OUT, 16, kRowsPerWg>), rows_grid, dim3(64 * kRowsPerWg), 0, st->stream, x, part, params, rows, width, splits, split_stride,
                           gain, bias, out_rows);
}

// The pass in front of the first product: token gather + position add (src/graph.c:729-737, :649-651), then the first layer's
// LayerNorm; a wavefront per row, rows [tokens, rows) zero.  All that changes from call to call arrives with this launch: the
// ids are kernel arguments, and the first workgroup leaves the rest (EncParams) in device memory for the graph that follows.
// So a call neither copies nor waits for the previous one's copies, and calls queue up behind each other: with two copies of
// 6 us and a wait in front of them, and the gather and the norm launches of their own, 256 rows took 254 us, 192 rows of the f32
// form 560; now 234 and 532.
constexpr int kIdsPerLaunch = 512;   // kernel arguments end at 4 KiB; longer inputs take a second launch
struct EncFirst {
    const void *tok, *pos;     // f16 or f32, as the operands
    float *x;
    const float *gain, *bias;
    void *out_rows;
    EncParams *params;
    EncParams call;
    int first, rows, width;
    int ids[kIdsPerLaunch];
};
template <int OUT, int NV>
__global__ void __launch_bounds__(64) k_enc_first(const EncFirst a) {
    const int lane = threadIdx.x, at_row = blockIdx.x, row = a.first + at_row, n4 = a.width / 4;
    const bool real = row < a.call.tokens;
    const size_t id = real ? (size_t)a.ids[at_row] : 0, pos = real ? (size_t)row : 0;
    if (row == 0 && lane == 0) *a.params = a.call;
    const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);
    float4 v[NV], gg[NV], bb[NV];
    const float4 *const gain4 = reinterpret_cast<const float4 *>(a.gain), *const bias4 = reinterpret_cast<const float4 *>(a.bias != nullptr ? a.bias : a.gain);
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int i = lane + 64 * u, at = i < n4 ? i : n4 - 1;
        gg[u] = gain4[at];
        bb[u] = bias4[at];
        if constexpr (OUT == ROWS_F16) {
            const half4 t = reinterpret_cast<const half4 *>(static_cast<const _Float16 *>(a.tok) + id * a.width)[at];
            const half4 p = reinterpret_cast<const half4 *>(static_cast<const _Float16 *>(a.pos) + pos * a.width)[at];
            if (a.call.embed_out != nullptr && real && i < n4) reinterpret_cast<half4 *>(a.call.embed_out + (size_t)row * a.width)[i] = t;
            v[u] = make_float4((float)t[0] + (float)p[0], (float)t[1] + (float)p[1], (float)t[2] + (float)p[2], (float)t[3] + (float)p[3]);
        } else {
            const float4 t = reinterpret_cast<const float4 *>(static_cast<const float *>(a.tok) + id * a.width)[at];
            const float4 p = reinterpret_cast<const float4 *>(static_cast<const float *>(a.pos) + pos * a.width)[at];
            v[u] = make_float4(t.x + p.x, t.y + p.y, t.z + p.z, t.w + p.w);
        }
    }
#pragma unroll
    for (int u = 0; u < NV; ++u) {
        const int i = lane + 64 * u;
        if (!real || i >= n4) v[u] = zero4;
        if (a.bias == nullptr) bb[u] = zero4;
        if (i < n4) reinterpret_cast<float4 *>(a.x + (size_t)row * a.width)[i] = v[u];
    }
    norm_row<OUT, NV>(v, gg, bb, lane, row, a.width, a.out_rows);
}

template <int OUT>
int launch_first(State *st, EncFirst &a, const int32_t *ids, char *error, size_t capacity) {
    for (a.first = 0; a.first < a.rows; a.first += kIdsPerLaunch) {
        const int rows = std::min(kIdsPerLaunch, a.rows - a.first), real = std::clamp(a.call.tokens - a.first, 0, kIdsPerLaunch);
        std::copy(ids + a.first, ids + a.first + real, a.ids);
        if (a.width <= 1024) hipLaunchKernelGGL((k_enc_first<OUT, 4>), dim3((unsigned)rows), dim3(64), 0, st->stream, a);
        else hipLaunchKernelGGL((k_enc_first<OUT, 16>), dim3((unsigned)rows), dim3(64), 0, st->stream, a);
    }
    return hip_check(hipGetLastError(), "encoder embedding launch", error, capacity);
}

constexpr int kAttentionThreads = 512;

// One (32-query tile, head): S = scale * Q K^T over all keys (f32, in LDS) -> row softmax numerators
// (f16, written over the row's own storage) and denominators -> O = P V / denom.
// Wavefront w takes key tiles w, w+8, ... for the scores and, for PV, output columns 32*(w & 1) .. +31
// over the key quarter (w >> 1); the quarters meet in LDS.
// Its chain bounds a launch (96 workgroups at 256 tokens x 12 heads): eight wavefronts, so that each has half the requests, tiles and steps of four, and
// sixteen lanes a row with no more pieces than the length has.  us a launch, four wavefronts and 32 pieces a lane / this: 60 tokens 5.5 / 4.6,
// 128 6.7 / 4.7, 192 7.4 / 5.3, 512 11.4 / 8.8; a prefill of 256 tokens 235 / 223.
// kKeyTiles, kValueSteps: score tiles and PV steps of a wavefront whose fragments are requested up front; kPieces: float4 pieces of a
// score row that a softmax lane may hold.  The launch picks the smallest set that covers the padded length (tiles and steps up to 512
// tokens, pieces up to 1024), so that none is requested or stepped over in vain.
template <int kKeyTiles, int kValueSteps, int kPieces>
__global__ void __launch_bounds__(kAttentionThreads) k_enc_attention(const _Float16 *qk, const _Float16 *vt, _Float16 *ctx, const EncParams *params,
                                                            int tpad, int width, float scale, int causal) {
    const int tokens = params->tokens;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ float s_inv[kQTile];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int q0 = blockIdx.x * kQTile, head = blockIdx.y;
    const int sstride = tpad + kScorePad;                    // floats per score row
    float *S = reinterpret_cast<float *>(smem);

    // ---- every global request of this workgroup is independent of the others and is issued here: the query
    // fragments, the key fragments of this wavefront's first kKeyTiles score tiles and the V fragments of its first
    // kValueSteps PV steps (all of them up to 512 tokens); they are consumed in that order while the rest arrives.
    // None of the requests is under a condition -- a tile or step this call does not have repeats the last one it has and
    // is never used -- so that the number of requests behind each one is a constant: loads return in order, a wait names
    // how many may still be out, and behind a conditional request the compiler has to wait for everything.
    const int heads = width / 64;
    const int ntiles = tpad / 32;
    const int wn = wave & 1, quarter = wave >> 1;
    const int kspan = tpad / 4;                              // keys per PV quarter, multiple of 16
    // Every request is one operand of one matrix instruction for the whole wavefront, 1 KiB of consecutive bytes (see the
    // layout note at the top).
    const half8 *qblock = reinterpret_cast<const half8 *>(qk + ((size_t)head * ntiles + q0 / 32) * 2048) + lane;
    const half8 *kblocks = reinterpret_cast<const half8 *>(qk + (size_t)(heads + head) * ntiles * 2048) + lane;
    const half8 *vblocks = reinterpret_cast<const half8 *>(vt + ((size_t)(head * 2 + wn) * (tpad / 16) + quarter * (kspan / 16)) * 512) + lane;
    half8 fq[4], fk[kKeyTiles][4], fv[kValueSteps];
#pragma unroll
    for (int j = 0; j < 4; ++j) fq[j] = qblock[j * 64];
#pragma unroll
    for (int t = 0; t < kKeyTiles; ++t) {
        const int tile = min(wave + 8 * t, ntiles - 1);
#pragma unroll
        for (int j = 0; j < 4; ++j) fk[t][j] = kblocks[(size_t)tile * 256 + j * 64];
    }
#pragma unroll
    for (int st = 0; st < kValueSteps; ++st) fv[st] = vblocks[min(st, kspan / 16 - 1) * 64];

    // ---- scores
    {
        auto score_tile = [&](int tile, const half8 (&k4)[4]) {
            floatx16 acc = {0};
#pragma unroll
            for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(fq[j], k4[j], acc, 0, 0, 0);
            const int key = tile * 32 + (lane & 31);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                // causal: query q0 + row sees keys up to itself (src/graph.c:446-449); its own key is always in range
                const bool seen = key < tokens && (!causal || key <= q0 + acc_row(r, lane));
                S[acc_row(r, lane) * sstride + key] = seen ? acc[r] * scale : -3.0e38f;
            }
        };
#pragma unroll
        for (int t = 0; t < kKeyTiles; ++t)
            if (wave + 8 * t < ntiles) score_tile(wave + 8 * t, fk[t]);
        for (int tile = wave + 8 * kKeyTiles; tile < ntiles; tile += 8) {   // beyond the tiles requested up front (more than 512 tokens)
            half8 k4[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) k4[j] = kblocks[(size_t)tile * 256 + j * 64];
            score_tile(tile, k4);
        }
    }
    __syncthreads();

    // ---- softmax of row tid / 16 by sixteen adjacent lanes (softmax_row_inplace, src/graph.c:245-257).  A lane takes
    // float4 pieces part, part + 16, ... of the row (up to kPieces of them in registers), so the row is
    // read from LDS once.  The numerators go back as f16 over the first half of the row's own bytes: the sixteen lanes
    // of a row belong to one wavefront and all of their reads are done before the first of these writes is issued.
    {
        const int row = tid >> 4, part = tid & 15;
        const float4 *srow = reinterpret_cast<const float4 *>(S + row * sstride);
        half4 *prow = reinterpret_cast<half4 *>(S + row * sstride);
        const int npieces = tpad / 4;
        float4 v[kPieces];
        float m = -3.0e38f;
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            const int c = part + 16 * i;
            if (c < npieces) {
                v[i] = srow[c];
                m = fmaxf(fmaxf(m, fmaxf(v[i].x, v[i].y)), fmaxf(v[i].z, v[i].w));
            }
        }
        m = fmaxf(m, __shfl_xor(m, 1));
        m = fmaxf(m, __shfl_xor(m, 2));
        m = fmaxf(m, __shfl_xor(m, 4));
        m = fmaxf(m, __shfl_xor(m, 8));
        float l = 0.0f;
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            const int c = part + 16 * i;
            if (c < npieces) {
                // hardware exponential: the numerators are rounded to f16 anyway; masked keys hold -3e38 and give 0
                const float e0 = __expf(v[i].x - m), e1 = __expf(v[i].y - m), e2 = __expf(v[i].z - m), e3 = __expf(v[i].w - m);
                l += (e0 + e1) + (e2 + e3);
                const half4 h = {(_Float16)e0, (_Float16)e1, (_Float16)e2, (_Float16)e3};
                prow[c] = h;
            }
        }
        l += __shfl_xor(l, 1);
        l += __shfl_xor(l, 2);
        l += __shfl_xor(l, 4);
        l += __shfl_xor(l, 8);
        if (part == 0) s_inv[row] = 1.0f / l;
    }
    __syncthreads();

    // ---- P V
    {
        const _Float16 *prow = reinterpret_cast<const _Float16 *>(S + (lane & 31) * sstride) + quarter * kspan + 8 * (lane >> 5);
        floatx16 acc = {0};
#pragma unroll
        for (int st = 0; st < kValueSteps; ++st) {
            if (16 * st < kspan) {
                const half8 fp = *reinterpret_cast<const half8 *>(prow + 16 * st);
                acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(fp, fv[st], acc, 0, 0, 0);
            }
        }
        for (int k = 16 * kValueSteps; k < kspan; k += 16) {   // beyond the steps requested up front (more than 512 tokens)
            const half8 fp = *reinterpret_cast<const half8 *>(prow + k);
            const half8 fvk = vblocks[(k / 16) * 64];
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(fp, fvk, acc, 0, 0, 0);
        }
        __syncthreads();   // (S is read: the quarters' sums go over it)
        float *const sums = S + wn * 16 * 64 + lane;
        if (quarter > 0) {
#pragma unroll
            for (int r = 0; r < 16; ++r) sums[((quarter - 1) * 32 + r) * 64] = acc[r];
        }
        __syncthreads();
        if (quarter == 0) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = acc_row(r, lane);
                const float o = (((acc[r] + sums[r * 64]) + sums[(32 + r) * 64]) + sums[(64 + r) * 64]) * s_inv[row];
                ctx[(size_t)(q0 + row) * width + head * 64 + wn * 32 + (lane & 31)] = (_Float16)o;
            }
        }
    }
}

template <int EPI, int WM, int WN, int D, bool CONV>
void launch_gemm_tiles(State *st, const GemmArgs &g, int splits) {
    hipLaunchKernelGGL((k_enc_gemm<EPI, WM, WN, D, CONV>), dim3(g.N / (32 * WN), g.M / (32 * WM), splits), dim3(64 * WM * WN), 0, st->stream, g.a, g.w, g.M, g.N,
                       g.K, g.K / kStep / splits, g.cin, g.taps, g.part, g.out, g.vt, g.width);
}

template <int EPI, bool CONV = false>
int launch_gemm(State *st, const GemmArgs &g, int splits, char *error, size_t capacity) {
    if (g.M % kTile != 0 || g.N % kTile != 0 || g.M <= 0 || g.N <= 0 || g.K <= 0 || splits < 1 || g.K % (kTile * splits) != 0 ||
        (splits > 1 && EPI != ENC_PARTIAL) ||
        (CONV && (g.taps < 1 || g.taps > kLeadRows + 1 || g.cin <= 0 || g.cin % kTile != 0 || g.taps * g.cin != g.K))) {
        set_error(error, capacity, "encoder product: shape is not a multiple of the 64 x 64 x 64 tile");
        return -1;
    }
    // The smallest tile that still puts no more than about a workgroup on a CU: fewer rows to fetch for each (98, 147 or 196 KB at
    // twelve steps), while a second round costs more than that.  us a launch (12 steps, weights no cache holds) with 32 x 32 / 64 x 32 /
    // 64 x 64 tiles, in brackets their workgroups: FFN up, 64 rows 5.1 (192) / 5.5 / 6.6; 128 5.8 (384) / 5.7 (192) / 6.4; 192 10.0
    // / 6.4 (288) / 6.5 (144); 256 - / 6.7 (384) / 6.4 (192).  Deeper rings than these leave a CU one workgroup where two are wanted (64 x 64 with
    // six stages at 512 rows: 11.0 against 8.4), shallower ones wait for weights (FFN up, 64 x 64 with four stages: 7.2 against 6.4).
    const int small = g.M / 32 * (g.N / 32) * splits, middle = g.M / 64 * (g.N / 32) * splits, most = st->cu_count + st->cu_count / 4;
    if (small <= most) launch_gemm_tiles<EPI, 1, 1, 7, CONV>(st, g, splits);
    else if (middle <= most) launch_gemm_tiles<EPI, 2, 1, 6, CONV>(st, g, splits);
    else launch_gemm_tiles<EPI, 2, 2, 5, CONV>(st, g, splits);
    return hip_check(hipGetLastError(), "encoder product launch", error, capacity);
}

int f16_matrix(State *st, const float *host, size_t n, size_t k, const CachedWeight **out, char *error, size_t capacity) {
    if (cached_matrix(st, host, n, k, MYNAH_HIP_F16, out, error, capacity) != 0) return -1;
    if ((*out)->qtype != MYNAH_HIP_F16) {
        set_error(error, capacity, "encoder: weight shape cannot be stored as f16");
        return -1;
    }
    return 0;
}

// Conv weight [n][cin][taps] (the reference's conv1d layout, src/graph.c:318-352) as f16 [n][taps][cin] in device memory:
// the K order in which k_enc_gemm's conv form walks the activation rows.  The caller owns the allocation.
int tap_major_f16(State *st, const float *host, size_t n, size_t cin, size_t taps, _Float16 **out, char *error, size_t capacity) {
    *out = nullptr;
    std::vector<uint16_t> packed;
    try {
        packed.resize(n * cin * taps);
    } catch (...) {
        set_error(error, capacity, "out of memory converting an encoder conv weight");
        return -1;
    }
    for (size_t o = 0; o < n; ++o)
        for (size_t i = 0; i < cin; ++i)
            for (size_t j = 0; j < taps; ++j) packed[(o * taps + j) * cin + i] = f32_to_f16_rne(host[(o * cin + i) * taps + j]);
    void *dev = nullptr;
    if (hip_check(hipMalloc(&dev, packed.size() * sizeof(uint16_t)), "encoder conv weight", error, capacity) != 0) return -1;
    if (hip_check(hipMemcpy(dev, packed.data(), packed.size() * sizeof(uint16_t), hipMemcpyHostToDevice), "encoder conv weight upload", error, capacity) != 0) {
        (void)hipFree(dev);
        return -1;
    }
    *out = static_cast<_Float16 *>(dev);
    return 0;
}

// The scores, and over them what P V's partial sums take.
size_t attention_lds_bytes(size_t tpad) { return std::max((size_t)kQTile * (tpad + kScorePad), (size_t)3 * 32 * 64) * sizeof(float); }

constexpr int kMaxSplits = 4;   // k_enc_rows reads exactly this many partial planes at most
// Most splits that leave each workgroup at least three K steps, preferring a step count that is a multiple of four, else an even one: fewer planes
// for the row pass to add where the steps are few.  The O product (twelve steps) in three splits / in four, us a prefill, tokens: one tap, 64 169.8 / 169.9,
// 192 205.4 / 207.9, 256 212.0 / 215.2, 384 251.2 / 256.4, 512 282.3 / 283.6; three taps, 100 248.6 / 255.3, 512 392.1 / 391.8.
int pick_splits(int k) {
    for (const int multiple : {4, 2, 1})
        for (int s = kMaxSplits; s > 1; --s)
            if (k % (kTile * s) == 0 && k / (kTile * s) >= 3 && (k / (kTile * s)) % multiple == 0) return s;
    return 1;
}

// Every kernel of one prefill over `tpad` padded rows behind k_enc_first, in stream order.  Everything that changes from call to
// call (token count, output pointers) is read from e->params on the device, so the sequence can be captured once.
int enqueue_prefill(State *st, mynah_hip_encoder *e, int tpad, char *error, size_t capacity) {
    const int w = (int)e->width, f = (int)e->ffn;
    const float scale = 1.0f / sqrtf((float)e->head_width);
    const size_t lds = attention_lds_bytes((size_t)tpad);
    const size_t split_stride = (size_t)tpad * w;
    // K splits of the two width-wide products (few output tiles, long K): enough workgroups to occupy the chip
    const int taps = (int)e->taps;
    const int o_splits = pick_splits(w), down_splits = pick_splits(f * taps);
    const float *pending = nullptr;   // partials of the last product, not yet added to x
    int pending_splits = 0;
    for (size_t l = 0; l < e->layers; ++l) {
        if (l > 0) launch_rows<ROWS_F16>(st, w, e->x, pending, pending_splits, split_stride, e->n1g[l], e->n1b[l], e->nrm, e->params, tpad);
        GemmArgs g{};
        g.a = e->nrm; g.w = static_cast<const _Float16 *>(e->qkv[l]->data); g.M = tpad; g.N = 3 * w; g.K = w;
        g.out = e->qk; g.vt = e->vt; g.width = w;
        if (launch_gemm<ENC_QKV>(st, g, 1, error, capacity) != 0) return -1;
        {
            // a wavefront scores every eighth 32-key tile and multiplies a quarter of the keys in steps of 16
            const dim3 agrid(tpad / kQTile, (unsigned)e->heads), ablock(kAttentionThreads);
            if (tpad <= 128) hipLaunchKernelGGL((k_enc_attention<1, 2, 2>), agrid, ablock, lds, st->stream, e->qk, e->vt, e->ctx, e->params, tpad, w, scale, e->causal);
            else if (tpad <= 256) hipLaunchKernelGGL((k_enc_attention<1, 4, 4>), agrid, ablock, lds, st->stream, e->qk, e->vt, e->ctx, e->params, tpad, w, scale, e->causal);
            else hipLaunchKernelGGL((k_enc_attention<2, 8, 16>), agrid, ablock, lds, st->stream, e->qk, e->vt, e->ctx, e->params, tpad, w, scale, e->causal);
        }
        g = GemmArgs{};
        g.a = e->ctx; g.w = static_cast<const _Float16 *>(e->o[l]->data); g.M = tpad; g.N = w; g.K = w; g.part = e->part;
        if (launch_gemm<ENC_PARTIAL>(st, g, o_splits, error, capacity) != 0) return -1;
        launch_rows<ROWS_F16>(st, w, e->x, e->part, o_splits, split_stride, e->n2g[l], e->n2b[l], e->nrm, e->params, tpad);
        g = GemmArgs{};
        g.a = e->nrm; g.M = tpad; g.N = f; g.K = w * taps; g.out = e->hid; g.taps = taps; g.cin = w;
        g.w = taps > 1 ? e->conv_up[l] : static_cast<const _Float16 *>(e->up[l]->data);
        if ((taps > 1 ? launch_gemm<ENC_GELU, true>(st, g, 1, error, capacity) : launch_gemm<ENC_GELU>(st, g, 1, error, capacity)) != 0) return -1;
        g = GemmArgs{};
        g.a = e->hid; g.M = tpad; g.N = w; g.K = f * taps; g.part = e->part; g.taps = taps; g.cin = f;
        g.w = taps > 1 ? e->conv_down[l] : static_cast<const _Float16 *>(e->down[l]->data);
        if ((taps > 1 ? launch_gemm<ENC_PARTIAL, true>(st, g, down_splits, error, capacity)
                      : launch_gemm<ENC_PARTIAL>(st, g, down_splits, error, capacity)) != 0)
            return -1;
        pending = e->part;
        pending_splits = down_splits;
    }
    // last residual update, then the final norm (src/graph.c:696-701) or a plain copy when the stack has none
    launch_rows<ROWS_RESULT>(st, w, e->x, pending, pending_splits, split_stride, e->nog, e->nob, nullptr, e->params, tpad);
    return hip_check(hipGetLastError(), "encoder prefill launch", error, capacity);
}

// ---- f32 operands: the stack as the reference computes it ---------------------------------------------------------------
// transformer_stack (src/graph.c:634-711) is LayerNorm -> QKV linear -> per head scaled Q K^T -> masked row softmax -> P V -> O linear
// -> residual -> LayerNorm -> causal_conv_ffn -> residual, all f32.  This form keeps every value f32 -- only the order of additions
// inside a product differs from the CPU: 1e-5 instead of the 2e-3 of f16 operands.  The products run on the bf16 matrix cores in
// three-piece form (split_product.h: f32 operands, f32 sums), scores and P V on the f32 ones, in eight kernels a layer, captured like
// the f16 form's.  192 tokens, causal, three taps: 3.5 ms as the library's f32 operators one after the other (some forty launches
// a layer, most of them a fraction of the chip).

// One (32-query tile, head), f32 throughout: S = scale * Q K^T (in LDS) -> softmax numerators and 1 / sum -> P V.
// Eight wavefronts:
// the longest workgroup's chain bounds the launch (72 workgroups at 192 tokens x 12 heads, whose matrix instructions are 3 of its 11.5 us), and a second wavefront
// on a SIMD hides a part of the requests.  Wavefront w scores key tiles w, w + 8, ..; for P V it takes columns 32 * (w % 2) .. over the sixteens of keys
// w / 2, w / 2 + 4, ..  Causal, 192 tokens: 12.2 us by four wavefronts, 11.5 by eight; V requested before the scores as well: 12.0.
// A matrix instruction (v_mfma_f32_32x32x2_f32) takes one value per lane and operand, of inner index l / 32: the scores give lanes
// below 32 columns 0..3 of eight and the rest 4..7, P V the same of eight keys, so that both come in 16-byte reads (any pairing of
// inner indices is the same sum).  qkv rows are read as they lie, 32 line visits a request (64 with columns 0..31 and 32..63: 0.3 us
// a launch more).
__global__ void __launch_bounds__(kAttentionThreads) k_enc_attention_f32(const float *qkv, float *ctx, const EncParams *params, int tpad, int width, float scale,
                                                                int causal) {
    const int tokens = params->tokens;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ float s_inv[kQTile];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, hi = lane >> 5;
    const int q0 = blockIdx.x * kQTile, head = blockIdx.y;
    const int keys = causal ? q0 + kQTile : tpad;            // what lies behind is masked for every query here; a multiple of 32
    const int sstride = tpad + kScorePad;
    float *S = reinterpret_cast<float *>(smem);
    const size_t stride = 3 * (size_t)width;
    const float *const base = qkv + head * 64;
    float fq[32], fk[32];
    const auto fetch = [&](float (&f)[32], const float *row) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float4 v = *reinterpret_cast<const float4 *>(row + 8 * i + 4 * hi);
            f[4 * i] = v.x; f[4 * i + 1] = v.y; f[4 * i + 2] = v.z; f[4 * i + 3] = v.w;
        }
    };
    fetch(fq, base + (size_t)(q0 + (lane & 31)) * stride);
    for (int tile = wave; tile < keys / 32; tile += kAttentionThreads / 64) {
        fetch(fk, base + width + (size_t)(tile * 32 + (lane & 31)) * stride);
        floatx16 acc = {0};
#pragma unroll
        for (int i = 0; i < 32; ++i) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fq[i], fk[i], acc, 0, 0, 0);
        const int key = tile * 32 + (lane & 31);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const bool seen = key < tokens && (!causal || key <= q0 + acc_row(r, lane));   // src/graph.c:446-449
            S[acc_row(r, lane) * sstride + key] = seen ? acc[r] * scale : -__builtin_inff();
        }
    }
    __syncthreads();
    {   // softmax_row_inplace (src/graph.c:245-257) of row tid / 16 by sixteen lanes; the division by the sum is left to the end
        const int row = tid >> 4, part = tid & 15;
        float4 *srow = reinterpret_cast<float4 *>(S + row * sstride);
        const int npieces = keys / 4;
        float m = -__builtin_inff();   // (every row sees a key: m is one of its scores in the end)
        for (int c = part; c < npieces; c += 16) {
            const float4 v = srow[c];
            m = fmaxf(fmaxf(m, fmaxf(v.x, v.y)), fmaxf(v.z, v.w));
        }
        m = fmaxf(m, __shfl_xor(m, 1));
        m = fmaxf(m, __shfl_xor(m, 2));
        m = fmaxf(m, __shfl_xor(m, 4));
        m = fmaxf(m, __shfl_xor(m, 8));
        float l = 0.0f;
        for (int c = part; c < npieces; c += 16) {
            float4 v = srow[c];
            v.x = expf(v.x - m); v.y = expf(v.y - m); v.z = expf(v.z - m); v.w = expf(v.w - m);
            l += (v.x + v.y) + (v.z + v.w);
            srow[c] = v;
        }
        l += __shfl_xor(l, 1);
        l += __shfl_xor(l, 2);
        l += __shfl_xor(l, 4);
        l += __shfl_xor(l, 8);
        if (part == 0) s_inv[row] = 1.0f / l;
    }
    __syncthreads();
    {
        const int wn = wave & 1, quarter = wave >> 1, last = keys - 16;
        const float *prow = S + (lane & 31) * sstride + 4 * hi;
        const float *vcol = base + 2 * width + (size_t)(4 * hi) * stride + wn * 32 + (lane & 31);
        floatx16 acc = {0};
        float fv[2][8];   // sixteen keys of this wavefront's columns, requested a step ahead
        const auto request = [&](float (&f)[8], int k) {
#pragma unroll
            for (int i = 0; i < 8; ++i) f[i] = vcol[(size_t)(k + 8 * (i >> 2) + (i & 3)) * stride];
        };
        const auto multiply = [&](const float (&f)[8], int k) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float4 p = *reinterpret_cast<const float4 *>(prow + k + 8 * j);
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(p.x, f[4 * j], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(p.y, f[4 * j + 1], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(p.z, f[4 * j + 2], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(p.w, f[4 * j + 3], acc, 0, 0, 0);
            }
        };
        request(fv[0], min(16 * quarter, last));
        for (int k = 16 * quarter; k < keys; k += 128) {
            request(fv[1], min(k + 64, last));
            multiply(fv[0], k);
            request(fv[0], min(k + 128, last));
            if (k + 64 < keys) multiply(fv[1], k + 64);
        }
        __syncthreads();   // (S is read: the quarters' sums go over it)
        float *const sums = S + (wn * 16) * 64 + lane;
        if (quarter > 0) {
#pragma unroll
            for (int r = 0; r < 16; ++r) sums[((quarter - 1) * 32 + r) * 64] = acc[r];
        }
        __syncthreads();
        if (quarter == 0) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = acc_row(r, lane);
                const float sum = ((acc[r] + sums[r * 64]) + sums[(32 + r) * 64]) + sums[(64 + r) * 64];
                ctx[(size_t)(q0 + row) * width + head * 64 + wn * 32 + (lane & 31)] = sum * s_inv[row];
            }
        }
    }
}

// hid = GELU(sum of the up product's splits, in split order); a float4 per thread.
__global__ void __launch_bounds__(256) k_enc_sum_gelu(const float4 *part, float4 *hid, int pieces, int splits) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= pieces) return;
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int z0 = 0; z0 < splits; z0 += 4) {
        float4 p[4];
#pragma unroll
        for (int z = 0; z < 4; ++z) p[z] = part[(size_t)min(z0 + z, splits - 1) * pieces + i];
#pragma unroll
        for (int z = 0; z < 4; ++z)
            if (z0 + z < splits) { s.x += p[z].x; s.y += p[z].y; s.z += p[z].z; s.w += p[z].w; }
    }
    hid[i] = make_float4(gelu_tanh(s.x), gelu_tanh(s.y), gelu_tanh(s.z), gelu_tanh(s.w));
}

constexpr size_t kMaxSplitsF32 = 12;   // planes of partial sums; the next pass reads them all

// The splits of a padded length's products, and the floats that their partial sums take.
struct SplitsF32 {
    int o, up, down;
    size_t floats;
    SplitsF32(const State *st, const mynah_hip_encoder *e, size_t rows) {
        const size_t w = e->width, f = e->ffn;
        o = split_product_splits(st, rows, w, w, kMaxSplitsF32);
        up = split_product_splits(st, rows, w, f, kMaxSplitsF32);
        down = split_product_splits(st, rows, f, w, kMaxSplitsF32);
        const size_t narrow = (size_t)(o > down ? o : down) * w, wide = (size_t)up * f;
        floats = rows * (narrow > wide ? narrow : wide);
    }
};

int enqueue_prefill_f32(State *st, mynah_hip_encoder *e, int tpad, char *error, size_t capacity) {
    const size_t w = e->width, f = e->ffn, taps = e->taps, rows = (size_t)tpad;
    const float scale = 1.0f / sqrtf((float)e->head_width);
    const SplitsF32 splits(st, e, rows);
    const int o_splits = splits.o, up_splits = splits.up, down_splits = splits.down;
    const float *pending = nullptr;   // partial sums of the last product, not yet added to x
    for (size_t l = 0; l < e->layers; ++l) {
        if (l > 0) launch_rows<ROWS_F32>(st, (int)w, e->x, pending, down_splits, rows * w, e->n1g[l], e->n1b[l], e->f_nrm, e->params, tpad);
        // (not split: the attention kernel reads every row several times and would add the planes up as often)
        if (launch_split_product(st, e->f_nrm, e->qkv32[l], rows, w, 1, 3 * w, 1, e->f_qkv, error, capacity) != 0) return -1;
        hipLaunchKernelGGL(k_enc_attention_f32, dim3(tpad / kQTile, (unsigned)e->heads), dim3(kAttentionThreads), attention_lds_bytes(rows), st->stream, e->f_qkv, e->f_ctx,
                           e->params, tpad, (int)w, scale, e->causal);
        if (launch_split_product(st, e->f_ctx, e->o32[l], rows, w, 1, w, o_splits, e->part, error, capacity) != 0) return -1;
        launch_rows<ROWS_F32>(st, (int)w, e->x, e->part, o_splits, rows * w, e->n2g[l], e->n2b[l], e->f_nrm, e->params, tpad);
        if (launch_split_product(st, e->f_nrm, e->up32[l], rows, w, taps, f, up_splits, e->part, error, capacity) != 0) return -1;
        const int pieces = (int)(rows * f / 4);
        hipLaunchKernelGGL(k_enc_sum_gelu, dim3((unsigned)((pieces + 255) / 256)), dim3(256), 0, st->stream, reinterpret_cast<const float4 *>(e->part),
                           reinterpret_cast<float4 *>(e->f_hid), pieces, up_splits);
        if (launch_split_product(st, e->f_hid, e->down32[l], rows, f, taps, w, down_splits, e->part, error, capacity) != 0) return -1;
        pending = e->part;
    }
    launch_rows<ROWS_RESULT>(st, (int)w, e->x, pending, down_splits, rows * w, e->nog, e->nob, nullptr, e->params, tpad);
    return hip_check(hipGetLastError(), "encoder prefill launch", error, capacity);
}

}  // namespace

extern "C" int mynah_hip_encoder_create(void *state, const mynah_hip_encoder_desc *d, mynah_hip_encoder **out, char *error, size_t capacity) {
    State *st = enter_state(state);
    if (out != nullptr) *out = nullptr;
    if (st == nullptr || d == nullptr || out == nullptr) {
        set_error(error, capacity, "encoder_create: null argument");
        return -1;
    }
    if (d->layers == 0 || d->width == 0 || d->heads == 0 || d->heads * d->head_width != d->width || d->head_width != 64 ||
        d->width % kTile != 0 || d->ffn_width % kTile != 0 || d->ffn_width == 0 || d->vocab == 0 || d->max_positions == 0 ||
        d->width > 4096 || d->ffn_width > 32768 || d->max_positions > 4096 || d->tok_table == nullptr || d->pos_table == nullptr ||
        d->qkv_w == nullptr || d->o_w == nullptr || d->up_w == nullptr || d->down_w == nullptr || d->norm1 == nullptr || d->norm2 == nullptr) {
        set_error(error, capacity, "encoder_create: unsupported shape (needs 64-wide heads, widths that are multiples of 64) or missing weights");
        return -1;
    }
    if (d->ffn_kernel != 0 && d->ffn_kernel != 1 && d->ffn_kernel != 3) {
        set_error(error, capacity, "encoder_create: ffn_kernel must be 1 or 3");
        return -1;
    }
    auto *e = new (std::nothrow) mynah_hip_encoder();
    if (e == nullptr) {
        set_error(error, capacity, "out of memory creating the encoder");
        return -1;
    }
    e->layers = d->layers; e->width = d->width; e->heads = d->heads; e->head_width = d->head_width; e->ffn = d->ffn_width;
    e->vocab = d->vocab; e->max_positions = d->max_positions;
    e->taps = d->ffn_kernel == 3 ? 3 : 1;
    e->causal = d->causal != 0;
    e->tpad_max = (d->max_positions + kTile - 1) / kTile * kTile;
    int lds = 0;
    if (hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, 0) != hipSuccess || lds <= 0) lds = 65536;
    e->max_lds = (size_t)lds;
    auto fail = [&](void) { mynah_hip_encoder_destroy(state, e); return -1; };
    if (e->tpad_max > 1024 || attention_lds_bytes(e->tpad_max) + 10 * 1024 > e->max_lds) {   // 1024: sixteen softmax lanes keep a row, sixteen float4 pieces each
        set_error(error, capacity, "encoder_create: max_positions beyond 1024, or more LDS per workgroup than this device has");
        return fail();
    }
    e->f32 = d->operands_f32 != 0;
    if (e->f32) {
        if (cached_matrix(st, d->tok_table, d->vocab, d->width, MYNAH_HIP_F32, &e->tok32, error, capacity) != 0) return fail();
        if (cached_matrix(st, d->pos_table, d->max_positions, d->width, MYNAH_HIP_F32, &e->pos32, error, capacity) != 0) return fail();
    } else {
        if (f16_matrix(st, d->tok_table, d->vocab, d->width, &e->tok, error, capacity) != 0) return fail();
        if (f16_matrix(st, d->pos_table, d->max_positions, d->width, &e->pos, error, capacity) != 0) return fail();
    }
    for (size_t l = 0; l < d->layers; ++l) {
        const CachedWeight *cw = nullptr;
        const float *v = nullptr;
        if (d->qkv_w[l] == nullptr || d->o_w[l] == nullptr || d->up_w[l] == nullptr || d->down_w[l] == nullptr || d->norm1[l] == nullptr ||
            d->norm2[l] == nullptr) {
            set_error(error, capacity, "encoder_create: missing layer weight");
            return fail();
        }
        if (e->f32) {
            const float4 *packed = nullptr;
            if (cached_split_weight(st, d->qkv_w[l], 3 * d->width, d->width, 1, &packed, error, capacity) != 0) return fail();
            e->qkv32.push_back(packed);
            if (cached_split_weight(st, d->o_w[l], d->width, d->width, 1, &packed, error, capacity) != 0) return fail();
            e->o32.push_back(packed);
            if (cached_split_weight(st, d->up_w[l], d->ffn_width, d->width, e->taps, &packed, error, capacity) != 0) return fail();
            e->up32.push_back(packed);
            if (cached_split_weight(st, d->down_w[l], d->width, d->ffn_width, e->taps, &packed, error, capacity) != 0) return fail();
            e->down32.push_back(packed);
        } else {
        if (f16_matrix(st, d->qkv_w[l], 3 * d->width, d->width, &cw, error, capacity) != 0) return fail();
        e->qkv.push_back(cw);
        if (f16_matrix(st, d->o_w[l], d->width, d->width, &cw, error, capacity) != 0) return fail();
        e->o.push_back(cw);
        if (e->taps == 1) {
            if (f16_matrix(st, d->up_w[l], d->ffn_width, d->width, &cw, error, capacity) != 0) return fail();
            e->up.push_back(cw);
            if (f16_matrix(st, d->down_w[l], d->width, d->ffn_width, &cw, error, capacity) != 0) return fail();
            e->down.push_back(cw);
        } else {
            _Float16 *dev = nullptr;
            if (tap_major_f16(st, d->up_w[l], d->ffn_width, d->width, e->taps, &dev, error, capacity) != 0) return fail();
            e->conv_up.push_back(dev);
            if (tap_major_f16(st, d->down_w[l], d->width, d->ffn_width, e->taps, &dev, error, capacity) != 0) return fail();
            e->conv_down.push_back(dev);
        }
        }
        if (cached_vector(st, d->norm1[l], d->width, &v, error, capacity) != 0) return fail();
        e->n1g.push_back(v);
        v = nullptr;
        if (d->norm1_bias != nullptr && d->norm1_bias[l] != nullptr && cached_vector(st, d->norm1_bias[l], d->width, &v, error, capacity) != 0) return fail();
        e->n1b.push_back(v);
        if (cached_vector(st, d->norm2[l], d->width, &v, error, capacity) != 0) return fail();
        e->n2g.push_back(v);
        v = nullptr;
        if (d->norm2_bias != nullptr && d->norm2_bias[l] != nullptr && cached_vector(st, d->norm2_bias[l], d->width, &v, error, capacity) != 0) return fail();
        e->n2b.push_back(v);
    }
    if (d->norm_out != nullptr && cached_vector(st, d->norm_out, d->width, &e->nog, error, capacity) != 0) return fail();
    if (d->norm_out != nullptr && d->norm_out_bias != nullptr && cached_vector(st, d->norm_out_bias, d->width, &e->nob, error, capacity) != 0) return fail();
    const size_t tp = e->tpad_max, w = e->width, f = e->ffn;
    auto alloc = [&](void **p, size_t bytes) {
        if (hip_check(hipMalloc(p, bytes), "encoder workspace", error, capacity) != 0) return -1;
        return hip_check(hipMemsetAsync(*p, 0, bytes, st->stream), "encoder workspace clear", error, capacity);
    };
    if (e->f32) {
        const size_t pad = kSplitOverrun;
        size_t part = 0;   // (a product is split only as far as its tiles leave CUs idle: the most are not the longest rows')
        for (size_t rows = kQTile; rows <= tp; rows += kQTile) {
            const size_t floats = SplitsF32(st, e, rows).floats;
            part = floats > part ? floats : part;
        }
        if (alloc(reinterpret_cast<void **>(&e->x), tp * w * sizeof(float)) != 0 ||
            alloc(reinterpret_cast<void **>(&e->f_nrm_alloc), ((kLeadRows + tp) * w + pad) * sizeof(float)) != 0 ||
            alloc(reinterpret_cast<void **>(&e->f_qkv), tp * 3 * w * sizeof(float)) != 0 || alloc(reinterpret_cast<void **>(&e->f_ctx), (tp * w + pad) * sizeof(float)) != 0 ||
            alloc(reinterpret_cast<void **>(&e->f_hid_alloc), ((kLeadRows + tp) * f + pad) * sizeof(float)) != 0 ||
            alloc(reinterpret_cast<void **>(&e->part), part * sizeof(float)) != 0 ||
            alloc(reinterpret_cast<void **>(&e->params), sizeof(EncParams)) != 0)
            return fail();
        e->f_nrm = e->f_nrm_alloc + kLeadRows * w;   // rows -2 and -1 stay zero
        e->f_hid = e->f_hid_alloc + kLeadRows * f;
    } else {
        if (alloc(reinterpret_cast<void **>(&e->x), tp * w * sizeof(float)) != 0 || alloc(reinterpret_cast<void **>(&e->nrm_alloc), (kLeadRows + tp) * w * 2) != 0 ||
            alloc(reinterpret_cast<void **>(&e->qk), tp * 2 * w * 2) != 0 || alloc(reinterpret_cast<void **>(&e->vt), w * tp * 2) != 0 ||
            alloc(reinterpret_cast<void **>(&e->ctx), tp * w * 2) != 0 || alloc(reinterpret_cast<void **>(&e->hid_alloc), (kLeadRows + tp) * f * 2) != 0 ||
            alloc(reinterpret_cast<void **>(&e->params), sizeof(EncParams)) != 0 ||
            alloc(reinterpret_cast<void **>(&e->part), kMaxSplits * tp * w * sizeof(float)) != 0)
            return fail();
        e->nrm = e->nrm_alloc + kLeadRows * w;   // rows -2 and -1 stay zero; widths are multiples of 64, so both stay 16-byte aligned
        e->hid = e->hid_alloc + kLeadRows * f;
    }
    if (attention_lds_bytes(e->tpad_max) > 48 * 1024) {
        const int bytes = (int)attention_lds_bytes(e->tpad_max);
        if (hip_check(hipFuncSetAttribute(reinterpret_cast<const void *>(k_enc_attention<1, 2, 2>), hipFuncAttributeMaxDynamicSharedMemorySize, bytes), "encoder attention LDS size", error, capacity) != 0 ||
            hip_check(hipFuncSetAttribute(reinterpret_cast<const void *>(k_enc_attention<1, 4, 4>), hipFuncAttributeMaxDynamicSharedMemorySize, bytes), "encoder attention LDS size", error, capacity) != 0 ||
            hip_check(hipFuncSetAttribute(reinterpret_cast<const void *>(k_enc_attention<2, 8, 16>), hipFuncAttributeMaxDynamicSharedMemorySize, bytes), "encoder attention LDS size", error, capacity) != 0 ||
            hip_check(hipFuncSetAttribute(reinterpret_cast<const void *>(k_enc_attention_f32), hipFuncAttributeMaxDynamicSharedMemorySize, bytes), "encoder attention LDS size", error, capacity) != 0)
            return fail();
    }
    if (hip_check(hipStreamSynchronize(st->stream), "encoder create", error, capacity) != 0) return fail();
    *out = e;
    return 0;
}

extern "C" void mynah_hip_encoder_destroy(void *state, mynah_hip_encoder *e) {
    State *st = enter_state(state);
    if (e == nullptr) return;
    if (st != nullptr) (void)hipStreamSynchronize(st->stream);
    for (auto &g : e->graphs)
        if (g.second != nullptr) (void)hipGraphExecDestroy(g.second);
    for (void *p : {(void *)e->x, (void *)e->nrm_alloc, (void *)e->qk, (void *)e->vt, (void *)e->ctx, (void *)e->hid_alloc, (void *)e->params, (void *)e->part})
        if (p != nullptr) (void)hipFree(p);
    for (_Float16 *p : e->conv_up) (void)hipFree(p);
    for (_Float16 *p : e->conv_down) (void)hipFree(p);
    for (void *p : {(void *)e->f_nrm_alloc, (void *)e->f_qkv, (void *)e->f_ctx, (void *)e->f_hid_alloc})
        if (p != nullptr) (void)hipFree(p);
    delete e;
}

extern "C" int mynah_hip_encoder_prefill(void *state, mynah_hip_encoder *e, const int32_t *ids, size_t tokens, uint16_t *dev_embed_f16,
                                         float *dev_out, char *error, size_t capacity) {
    State *st = enter_state(state);
    if (st == nullptr || e == nullptr || ids == nullptr || dev_out == nullptr) {
        set_error(error, capacity, "encoder_prefill: null argument");
        return -1;
    }
    if (tokens == 0 || tokens > e->max_positions) {
        set_error(error, capacity, "encoder_prefill: token count outside [1, max_positions]");
        return -1;
    }
    for (size_t t = 0; t < tokens; ++t) {
        if (ids[t] < 0 || (size_t)ids[t] >= e->vocab) {   // src/graph.c:730-735
            set_error(error, capacity, "encoder_prefill: token id out of range");
            return -1;
        }
    }
    if (e->f32 && dev_embed_f16 != nullptr) {
        set_error(error, capacity, "encoder_prefill: with f32 operands there are no f16 token rows to return");
        return -1;
    }
    const int granule = e->f32 ? kQTile : kTile, tpad = ((int)tokens + granule - 1) / granule * granule;
    EncFirst first;
    first.tok = e->f32 ? e->tok32->data : e->tok->data;
    first.pos = e->f32 ? e->pos32->data : e->pos->data;
    first.x = e->x;
    first.gain = e->n1g[0];
    first.bias = e->n1b[0];
    first.out_rows = e->f32 ? static_cast<void *>(e->f_nrm) : e->nrm;
    first.params = e->params;
    first.call = EncParams{(int)tokens, 0, dev_embed_f16, dev_out};
    first.rows = tpad;
    first.width = (int)e->width;
    if ((e->f32 ? launch_first<ROWS_F32>(st, first, ids, error, capacity) : launch_first<ROWS_F16>(st, first, ids, error, capacity)) != 0) return -1;
    const auto enqueue = e->f32 ? enqueue_prefill_f32 : enqueue_prefill;
    if (!st->graph_mode || e->eager_runs[tpad] == 0) {
        e->eager_runs[tpad] = 1;
        return enqueue(st, e, tpad, error, capacity);
    }
    hipGraphExec_t &exec = e->graphs[tpad];
    if (exec == nullptr) {
        hipGraph_t graph = nullptr;
        MYNAH_TRY(hipStreamBeginCapture(st->stream, hipStreamCaptureModeThreadLocal));
        const int rc = enqueue(st, e, tpad, error, capacity);
        const hipError_t end = hipStreamEndCapture(st->stream, &graph);
        if (rc != 0 || end != hipSuccess) {
            if (graph != nullptr) (void)hipGraphDestroy(graph);
            if (rc == 0) (void)hip_check(end, "encoder graph capture", error, capacity);
            return -1;
        }
        const hipError_t inst = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
        (void)hipGraphDestroy(graph);
        if (hip_check(inst, "encoder graph instantiate", error, capacity) != 0) {
            exec = nullptr;
            return -1;
        }
    }
    return hip_check(hipGraphLaunch(exec, st->stream), "encoder graph launch", error, capacity);
}
