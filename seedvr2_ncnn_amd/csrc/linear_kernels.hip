// gfx950 kernels of the SharedLinear projection (src/seedvr2/shared_linear.cpp:83-96):
// y = act(x W^T + b) for the video and the text stream in one grouped launch.
//
// x [m][k] and W [n][k] are both k-contiguous, which is the natural operand
// layout of the bf16 MFMAs (each lane supplies 8 consecutive k of one row of A
// and one column of B), so both tiles are staged in LDS unchanged.  fp32 and
// fp16 activations are rounded to bf16 while they are staged.  k that is a
// multiple of 64 takes the 256x256-tile kernel, other k (and rows too long for
// its 32-bit offsets) the 128x128 one.
#include <math.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "awa_index.h"
#include "awa_kernels.h"
#include "s2_device.h"
#include "stream_scratch.h"


namespace s2 {

namespace {

__device__ __forceinline__ uint4 load_chunk(const uint16_t* p) {
    return *reinterpret_cast<const uint4*>(p);
}

__device__ __forceinline__ uint4 load_chunk(const _Float16* p) {
    const uint4 raw = *reinterpret_cast<const uint4*>(p);
    const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
    uint16_t h[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        h[2 * i] = f32_to_bf16((float)__builtin_bit_cast(_Float16, (uint16_t)(w[i] & 0xffffu)));
        h[2 * i + 1] = f32_to_bf16((float)__builtin_bit_cast(_Float16, (uint16_t)(w[i] >> 16)));
    }
    return pack8_bf16(h);
}

// one output element of type YK (0 fp32, 1 bf16, 2 fp16)
template <int YK>
__device__ __forceinline__ void store1(void* y, long idx, float v) {
    if (YK == 1)
        ((uint16_t*)y)[idx] = f32_to_bf16(v);
    else if (YK == 2)
        ((_Float16*)y)[idx] = f32_to_f16(v);
    else
        ((float*)y)[idx] = v;
}

__device__ __forceinline__ uint4 load_chunk(const float* p) {
    float v[8];
    load8(p, v);
    uint16_t h[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) h[i] = f32_to_bf16(v[i]);
    return pack8_bf16(h);
}

// erf-GELU, 0.5 x (1 + erf(x / sqrt 2)) = max(x, 0) - |x| Q(|x|) with
// Q(a) = 0.5 erfc(a / sqrt 2): both signs reduce to one fma, and for x < 0
// the result is the product -|x| Q directly, without cancellation.  erfc is
// Abramowitz & Stegun 7.1.26, erfc(z) = (a1 t + ... + a5 t^5) e^(-z^2),
// t = 1 / (1 + p z), |error| <= 1.5e-7; the factor 0.5 is folded into a1..a5
// and e^(-z^2) = 2^(-w^2) with w = z sqrt(log2 e).  (Q as 2^p(a), p a degree-8
// fit of log2 Q, has one transcendental less and took 1854 us for the 720p
// MLP against 1882, but its rms error over |x| <= 0.1 is 3.5 times this one's,
// 1.8e-8 against 5.3e-9, and its relative error over [-8, -6] 5% against 1%.)
__device__ __forceinline__ float gelu(float x) {
    constexpr float kSqrtLog2e = 1.2011224087864498f;
    const float ax = fabsf(x);
    const float w = ax * (0.70710678118654752f * kSqrtLog2e);
    const float t = __builtin_amdgcn_rcpf(fmaf(w, 0.3275911f / kSqrtLog2e, 1.f));
    const float poly =
        t * (0.5f * 0.254829592f +
             t * (0.5f * -0.284496736f +
                  t * (0.5f * 1.421413741f + t * (0.5f * -1.453152027f + t * (0.5f * 1.061405429f)))));
    const float q = poly * __builtin_amdgcn_exp2f(-w * w);   // Q(|x|)
    return fmaf(-ax, q, fmaxf(x, 0.f));
}

}  // namespace

// Block tile 128x128, k-step 64, four waves in a 2x2 grid of 64x64 wave tiles
// (2x2 MFMA 32x32 accumulators per wave).  LDS double buffered, rows padded
// by 16 bytes against bank conflicts.
template <typename TX, int YK, int ACT>
__global__ __launch_bounds__(256, 2) void shared_linear_kernel(
    const TX* __restrict__ x0, int m0, const TX* __restrict__ x1, int m1,
    const uint16_t* __restrict__ wgt, const float* __restrict__ bias, int n, int k,
    void* __restrict__ y0, void* __restrict__ y1, int mt0, int mtiles, int ntiles) {
    constexpr int BM = 128, BN = 128, BK = 64, P = BK + 8;
    constexpr int A_CHUNKS = BM * BK / 8 / 256;
    constexpr int B_CHUNKS = BN * BK / 8 / 256;
    constexpr int GROUP = 8;
    __shared__ __attribute__((aligned(16))) uint16_t a_lds[2][BM * P];
    __shared__ __attribute__((aligned(16))) uint16_t b_lds[2][BN * P];

    // XCD-aware, grouped rasterisation: consecutive logical tiles share an
    // XCD's L2, and GROUP m-tiles sweep the n-tiles together.
    const int lid = xcd_remap(blockIdx.x, gridDim.x);
    const int group_size = GROUP * ntiles;
    const int first_m = (lid / group_size) * GROUP;
    const int gm = min(mtiles - first_m, GROUP);
    const int mt = first_m + (lid % group_size) % gm;
    const int nt = (lid % group_size) / gm;

    const TX* x;
    int m, row0;
    void* y;
    if (mt < mt0) {
        x = x0; m = m0; y = y0; row0 = mt * BM;
    } else {
        x = x1; m = m1; y = y1; row0 = (mt - mt0) * BM;
    }
    const int col0 = nt * BN;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int l32 = lane & 31;
    const int g = lane >> 5;
    const int wm = wave >> 1;
    const int wn = wave & 1;

    uint4 areg[A_CHUNKS], breg[B_CHUNKS];
    auto load_tile = [&](int kt) {
        const int k0 = kt * BK;
#pragma unroll
        for (int c = 0; c < A_CHUNKS; ++c) {
            const int idx = tid + 256 * c;
            const int r = idx / (BK / 8);
            const int kc = k0 + (idx % (BK / 8)) * 8;
            areg[c] = make_uint4(0, 0, 0, 0);
            if (row0 + r < m && kc < k) areg[c] = load_chunk(x + (long)(row0 + r) * k + kc);
        }
#pragma unroll
        for (int c = 0; c < B_CHUNKS; ++c) {
            const int idx = tid + 256 * c;
            const int r = idx / (BK / 8);
            const int kc = k0 + (idx % (BK / 8)) * 8;
            breg[c] = make_uint4(0, 0, 0, 0);
            if (col0 + r < n && kc < k) breg[c] = load_chunk(wgt + (long)(col0 + r) * k + kc);
        }
    };
    auto store_tile = [&](int buf) {
#pragma unroll
        for (int c = 0; c < A_CHUNKS; ++c) {
            const int idx = tid + 256 * c;
            *reinterpret_cast<uint4*>(&a_lds[buf][(idx / (BK / 8)) * P + (idx % (BK / 8)) * 8]) =
                areg[c];
        }
#pragma unroll
        for (int c = 0; c < B_CHUNKS; ++c) {
            const int idx = tid + 256 * c;
            *reinterpret_cast<uint4*>(&b_lds[buf][(idx / (BK / 8)) * P + (idx % (BK / 8)) * 8]) =
                breg[c];
        }
    };

    f32x16 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    const int nk = (k + BK - 1) / BK;
    load_tile(0);
    store_tile(0);
    __syncthreads();
#pragma unroll 1
    for (int kt = 0; kt < nk; ++kt) {
        const int buf = kt & 1;
        if (kt + 1 < nk) load_tile(kt + 1);
#pragma unroll
        for (int kk = 0; kk < BK / 16; ++kk) {
            bf16x8 a[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; ++i)
                a[i] = as_bf16x8(*reinterpret_cast<const uint4*>(
                    &a_lds[buf][(wm * 64 + 32 * i + l32) * P + 16 * kk + 8 * g]));
#pragma unroll
            for (int j = 0; j < 2; ++j)
                b[j] = as_bf16x8(*reinterpret_cast<const uint4*>(
                    &b_lds[buf][(wn * 64 + 32 * j + l32) * P + 16 * kk + 8 * g]));
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        if (kt + 1 < nk) store_tile(buf ^ 1);
        __syncthreads();
    }

    // Epilogue: register r of a 32x32 accumulator is row 8(r/4) + 4g + r%4,
    // column l32; bias and the activation are applied in fp32.
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int col = col0 + wn * 64 + 32 * j + l32;
        if (col >= n) continue;
        const float b = bias ? bias[col] : 0.f;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = row0 + wm * 64 + 32 * i + 8 * (r >> 2) + 4 * g + (r & 3);
                if (row >= m) continue;
                float v = acc[i][j][r] + b;
                if (ACT == S2_ACT_GELU) v = gelu(v);
                store1<YK>(y, (long)row * n + col, v);
            }
    }
}

// ---------------------------------------------------------------------------
// Large-tile path, k % 64 == 0.
//
// Block tile 256x256 with eight waves, two per SIMD, in a 2 (m) x 4 (n) grid
// of 128x64 wave tiles (8x4 MFMA 16x16x32 accumulators = 128 fp32 per lane).
// 16x16x32 takes the same operand bytes from LDS as 32x32x16 and the same
// matrix cycles, but moves half the accumulator registers per flop; under the
// power limit that clocks higher: MLP up + down of the 720p video 1973 -> 1868
// us, QKV projection + attention 988 -> 953 us.
// The two waves of a SIMD ping-pong: one issues a whole 64-k step of MFMAs
// from fragment registers while the other reads its next step's fragments
// from LDS (the main loop below).  The operands stream through two 64-k LDS
// stages (64 KB each) filled by buffer_load_dwordx4 ... lds (global -> LDS,
// no VGPR staging).  The buffer descriptors bound each tile to its valid
// rows, so ragged m and n read zeros.  LDS rows are 128 bytes; 16-byte chunk
// c of row r is stored at position c ^ (((r >> 1) ^ ((r & 1) << 2)) & 7), so
// the rows one ds_read_b128 phase touches land on distinct banks.  (That is for
// bf16 activations; fp32 and fp16 ones have a main loop of their own, which
// converts A in registers.)  The epilogues add the bias and activation in fp32;
// each wave converts, stages and stores its own 128x64 part, except for SwiGLU
// and the fused QKV projection, which assemble the tile in LDS.
//
// Tail balancing.  When the tile count leaves the last wave of workgroups
// partly idle, the tiles of that wave are not given one workgroup each:
// their 64-k iterations are dealt out evenly to sk_groups workgroups, each
// taking one contiguous range of (tile, k-iteration) pairs (with sk_groups
// a multiple of the tile count, every range lies inside one tile).  A tile
// finished by one workgroup takes the normal epilogue; a tile split between workgroups has every part store its fp32 accumulators to a
// per-workgroup slot and bump the tile's arrival counter, and the last part
// to arrive sums all the slots in workgroup order (so the result does not
// depend on which part arrives last), runs the epilogue and resets the
// counter.  No workgroup waits on another.
namespace {

__device__ __forceinline__ int lds_swizzle(int r) { return ((r >> 1) ^ ((r & 1) << 2)) & 7; }

// Sum over aligned groups of N lanes (N = 8 or 16) by DPP lane moves: quad
// permutations [1,0,3,2] and [2,3,0,1], then the half-row and row mirrors.
// Each step adds the value of a lane of the other half of the group, which
// after the previous steps holds the same partial sum as lane ^ (N/2), so
// the result equals the shuffle-xor reduction over masks 1, 2, 4, 8 bit for
// bit (and needs no LDS round trip).
template <int N>
__device__ __forceinline__ float row_sum(float x) {
    static_assert(N == 8 || N == 16, "row_sum over 8 or 16 lanes");
    x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xB1, 0xF, 0xF, false));
    x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x4E, 0xF, 0xF, false));
    x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x141, 0xF, 0xF, false));
    if (N == 16) x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x140, 0xF, 0xF, false));
    return x;
}

constexpr int kSlotFloats = 128 * 512;   // one workgroup's accumulators
constexpr int kWaveStage = 2 * 32 * 144; // a wave's own LDS in wave_epilogue (bytes)

// Cache policy of the slot stores and loads: sc0 sc1, coherent across the
// XCDs' L2s (stores write through, loads do not hit a stale L2 line), so the
// parts of a tile can meet without cache-wide writeback or invalidation.
constexpr int kCoherent = 1 | 16;
// nt: a streaming store, not kept in the L2
constexpr int kNonTemporal = 2;
// word 3 of a raw (untyped, stride 0) buffer descriptor
constexpr int kRawBufferFormat = 0x00020000;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

}  // namespace

struct SkTail {
    int dp_tiles;      // tiles [0, dp_tiles): one workgroup each
    int sk_tiles;      // tiles [dp_tiles, dp_tiles + sk_tiles): shared out along k
    int sk_groups;     // workgroups sharing them: a multiple of sk_tiles, so that
                       // each workgroup's k range lies inside one tile
    float* slots;      // [sk_groups][kSlotFloats] partial accumulators
    int* counters;     // [sk_tiles] arrivals; zero between launches
};

// The fused QKV projection of the attention layer (AWA = head dim): the
// tile rows are the plan's QKV row space (video tokens in window order, then
// the text tokens), gathered from the source-ordered activations, and the
// epilogue writes the attention workspace directly: RMS-normalised and
// rotated Q and K rows [head][seg_total][D] and V transposed [head][D][seg_total]
// (adaptive_window_attention.cpp:886-927), text tokens to their staging rows.
struct AwaQkvArgs {
    const QkvRow* row_table;  // the plan's rows, [mtiles * 256]
    int inner;                // heads * head_dim
    long seg_total;           // row pitch of Q, K and V^T
    long seg_text;            // first text staging row
    const float* norm;        // [4][D]: video q, video k, text q, text k
    const float2* rope;       // (cos, sin) [position][pairs]
    int pairs;
    float eps;
    int official_bf16;
    uint16_t* q;
    uint16_t* k;
    uint16_t* vt;
};

// four values of one column, rows `pitch` bytes apart, as 16-bit LDS elements:
// two pair conversions (one per value otherwise) and four 2-byte writes
template <int YK>
__device__ __forceinline__ void stage_rows4(uint8_t* p, int pitch, const float (&v)[4]) {
    const uint32_t a = YK == 2 ? pack2_f16_rne(v[0], v[1]) : pack2_bf16_rne(v[0], v[1]);
    const uint32_t b = YK == 2 ? pack2_f16_rne(v[2], v[3]) : pack2_bf16_rne(v[2], v[3]);
    *(uint16_t*)p = (uint16_t)a;
    *(uint16_t*)(p + pitch) = (uint16_t)(a >> 16);
    *(uint16_t*)(p + 2 * pitch) = (uint16_t)b;
    *(uint16_t*)(p + 3 * pitch) = (uint16_t)(b >> 16);
}

// Epilogues of the VAE attention's products (one stream, bf16 output):
//   kActExp       rows are keys, columns queries: y[query][key] = exp(acc -
//                 reference of the query), zeros for keys past m0 up to the
//                 row pitch, and per 128 keys the fp32 sums of a query's values
//                 as stored.
//                 A lane holds four consecutive keys of a query: packed
//                 conversions, 8-byte LDS writes and sums within the lane
//   kActRowScale  y = acc * (scale of the row) + bias
constexpr int kActExp = 100, kActRowScale = 101;

// How the plain epilogues store a wave's staged rows: 16-byte chunks of rows
// whose pitch is a multiple of 64 bytes, non-temporal; of other rows, by way of
// the L2; or single elements, where chunks would not keep to the rows.
enum : int { kWholeSectors, kPieces, kElements };

// XK is the element type of x0 and x1 (0 fp32, 1 bf16, 2 fp16).
template <int YK, int ACT, int AWA = 0, int RES = 0, int XK = 1>
__global__ __launch_bounds__(512, 1) void shared_linear_256_kernel(
    const uint16_t* __restrict__ x0, int m0, const uint16_t* __restrict__ x1, int m1,
    const uint16_t* __restrict__ wgt, const float* __restrict__ bias, int n, int k,
    void* __restrict__ y0, void* __restrict__ y1, int mv, int mtiles, int ntiles, SkTail sk,
    AwaQkvArgs awa, LinearResidual res, LinearRows lr) {
    constexpr int BM = 256, BN = 256, BK = 64;
    constexpr int TB = BM * BK * 2;   // 32 KB per operand per stage
    constexpr int SB = 2 * TB;        // 64 KB per stage
    constexpr int RB = BK * 2;        // LDS row bytes
    constexpr int EP = BN * 2 + 16;   // epilogue LDS row pitch (bytes)
    constexpr int LDS_BYTES = 2 * SB > BM * EP ? 2 * SB : BM * EP;
    // row-tiles per raster group: 4 is 1-3% faster than 8 or 16 on a video's 85
    // row-tiles.  (An image's 5 to 12 row-tiles in groups of about one height:
    // 0.97 to 1.02 of these times over 4 to 20 row-tiles and five weight shapes,
    // which is also how far the unchanged sizes spread.)
    constexpr int GROUP = 4;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[LDS_BYTES];
    __shared__ int arrival;
    __shared__ QkvRow qrows[AWA ? BM : 1];
    // fused QKV: byte offsets of the gathered A rows of every lane of the
    // four A-loading waves, eight per lane (read back at each DMA issue:
    // the main loop has no registers to spare for them)
    __shared__ uint4 goff_lds[AWA ? 4 * 64 * 2 : 1];

    if constexpr (AWA == 0 && RES == 0)
        if (lr.gate && *lr.gate != lr.gate_want) return;   // uniform: no workgroup waits

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform
    const int l16 = lane & 15;
    const int g = lane >> 4;
    const int wm = wave >> 2;
    const int wn = wave & 3;
    const int nk = k / BK;
    const int sw = lds_swizzle(l16);   // fragment rows differ from l16 by multiples of 16
    const uint32_t lds_base = (uint32_t)(uintptr_t)lds;

    // The two token streams share one row space: video row r is row r, text
    // row r is row mv + r (mv = m0 rounded up to a multiple of 8), so the
    // tile holding the video tail also holds the first text rows.  Every
    // 8-row DMA group lies in one stream.
    int row0, col0;   // the current tile
    auto set_tile = [&](int t) {
        // grouped raster: GROUP m-tiles share each sweep over the n-tiles
        const int group_size = GROUP * ntiles;
        const int first_m = (t / group_size) * GROUP;
        const int gm = min(mtiles - first_m, GROUP);
        const int mt = first_m + (t % group_size) % gm;
        const int nt = (t % group_size) / gm;
        row0 = mt * BM;
        col0 = nt * BN;
    };
    // output row of tile row rl, or null past either stream
    // output row pitch: n, or n / 2 for SwiGLU, whose weight has a gate and
    // an up row per output column
    const int ny = ACT == S2_ACT_SWIGLU ? n / 2 : ACT == kActExp ? lr.pitch : n;
    auto out_row = [&](int rl) -> void* {
        const int r = row0 + rl;
        if (r < m0) return (char*)y0 + (long)r * ny * (YK ? 2 : 4);
        if (r >= mv && r < mv + m1) return (char*)y1 + (long)(r - mv) * ny * (YK ? 2 : 4);
        return nullptr;
    };

    // Fused QKV projection: the current tile's rows of the plan's row table
    // (one row per thread of the first four waves).
    auto build_rows = [&]() {
        if constexpr (AWA != 0) {
            if (tid < BM) qrows[tid] = awa.row_table[row0 + tid];
        }
    };

    // register r of accumulator [i][j] is row 16 i + 4 g + r, column 16 j + l16
    // of the wave's 128x64 tile
    f32x4 acc[8][4];

    // Thread coordinates for the epilogues, derived from an opaque copy of
    // the thread index: addresses computed from them are not hoisted above
    // the main loop, where every register is taken and hoisted values would
    // be spilled and reloaded one scratch round trip at a time.
    struct EpiIds {
        int tid, l16, g, wm, wn;
    };
    auto epi_ids = [&]() {
        EpiIds e;
        int t = tid;
        asm volatile("" : "+v"(t));
        const int w = __builtin_amdgcn_readfirstlane(t >> 6);
        e.tid = t;
        e.l16 = t & 15;
        e.g = (t >> 4) & 3;
        e.wm = w >> 2;
        e.wn = w & 3;
        return e;
    };

    // 16-bit outputs without a residual: every wave writes its own 128x64
    // sub-tile, a quarter at a time, through two 4.5 KB LDS buffers of its own,
    // so no wave waits for another.  A quarter's stores drain under the next
    // one's arithmetic, and group 0 is done with its part while group 1 still
    // issues its last MFMAs (no wave reads a stage by then: mainloop).  A store
    // covers 128 bytes of 8 rows (kActExp: 256 bytes of 4 queries).  Assembling
    // 512-byte rows from the four waves of a group instead took two barriers
    // and left the stores to the end: MLP of the 720p video 1842 us, 1824 so;
    // of 1485 rows 223 and 218; the VAE attention 533 and 508.
    //
    // Each stream's rows of the tile go through a buffer descriptor bounded by
    // those rows, so the range check drops a row past its stream, and a chunk
    // past n (an offset with bit 31 set: offsets are below 2^31, the launcher
    // checks 256 rows of output), without a branch per store; the 8 rows of a
    // store lie in one stream.  The output is not read again by this launch:
    // the stores are non-temporal, leaving the L2 to the operand tiles, where
    // row pitches are multiples of 64 bytes.  Elsewhere the pieces of two waves
    // meet inside a 64-byte sector, which the L2 has to put together: 9000 x 64 by
    // 9000 x 64 took 84 us with non-temporal stores, 51 by way of the L2 (62 from
    // 512-byte rows); 21664 x 2560 by 3112 x 2560 287 and 285.  Rows of n % 8 != 0
    // leave as elements, 64 columns of a row a store: 3677 x 2560 by 2561 x 2560
    // 67 us straight from the accumulators (16 columns of a row), 51 so; 4609 x
    // 512 by 4609 x 512 67 and 36.
    auto wave_epilogue = [&]() {
        if constexpr (YK != 0 && AWA == 0 && RES == 0 && ACT != S2_ACT_SWIGLU) {
            const EpiIds ei = epi_ids();
            const int ln = ei.tid & 63;
            const int pitch = ny * 2;
            uint8_t* mine = lds + (ei.wm * 4 + ei.wn) * kWaveStage;
            if constexpr (ACT == kActExp) {
                constexpr float kLog2e = 1.4426950408889634f;
                constexpr int QP = 128 * 2 + 16;   // staged query row (bytes)
                static_assert(2 * 16 * QP <= kWaveStage, "two quarters of 16 queries");
                const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc(
                    (char*)y0 + (long)col0 * pitch, (short)0, min(n - col0, BN) * pitch,
                    kRawBufferFormat);
                const int key = row0 + 128 * ei.wm + (ln & 15) * 8;
                const uint32_t past = key < ny ? 0u : 0x80000000u;
                auto quarters = [&](auto full_tag) {
                    constexpr bool FULL = decltype(full_tag)::value;   // no key past m0
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        uint8_t* buf = mine + (j & 1) * 16 * QP;
                        const int q0 = ei.wn * 64 + 16 * j;   // the quarter's first query
                        const float ref = lr.ref[col0 + q0 + ei.l16];
                        float sum = 0.f;
#pragma unroll
                        for (int i = 0; i < 8; ++i) {
                            const int rl = 16 * i + 4 * ei.g;
                            float v[4];
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                v[r] = __builtin_amdgcn_exp2f(fmaf(acc[i][j][r], kLog2e, -ref));
                                if (!FULL && row0 + 128 * ei.wm + rl + r >= m0) v[r] = 0.f;
                            }
                            // the sums are of the rounded values: the weights
                            // that the product with V uses then add up to one,
                            // and a row with few large ones keeps the precision
                            // that rounding normalised probabilities gives
                            const uint32_t w0 = pack2_bf16_rne(v[0], v[1]);
                            const uint32_t w1 = pack2_bf16_rne(v[2], v[3]);
                            sum += (__uint_as_float(w0 << 16) + __uint_as_float(w0 & 0xffff0000u)) +
                                   (__uint_as_float(w1 << 16) + __uint_as_float(w1 & 0xffff0000u));
                            *(uint2*)(buf + ei.l16 * QP + rl * 2) = make_uint2(w0, w1);
                        }
                        sum += __shfl_xor(sum, 16);
                        sum += __shfl_xor(sum, 32);
                        if (ei.g == 0)
                            lr.sums[(long)(row0 / 128 + ei.wm) * lr.sums_pitch + col0 + q0 + ei.l16] = sum;
                        asm volatile("" ::: "memory");   // a wave's LDS accesses run in order
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const int ql = (ln >> 4) + 4 * r;
                            __builtin_amdgcn_raw_buffer_store_b128(
                                *(const u32x4*)(buf + ql * QP + (ln & 15) * 16), rq,
                                (uint32_t)((q0 + ql) * pitch + key * 2) | past, 0, kNonTemporal);
                        }
                        asm volatile("" ::: "memory");
                    }
                };
                if (row0 + BM <= m0)
                    quarters(std::true_type{});
                else
                    quarters(std::false_type{});
            } else {
                constexpr int RP = 64 * 2 + 16;   // staged row (bytes)
                static_assert(2 * 32 * RP <= kWaveStage, "two quarters of 32 rows");
                const __amdgpu_buffer_rsrc_t rs0 = __builtin_amdgcn_make_buffer_rsrc(
                    (char*)y0 + (long)row0 * pitch, (short)0, max(min(m0 - row0, BM), 0) * pitch,
                    kRawBufferFormat);
                const __amdgpu_buffer_rsrc_t rs1 = __builtin_amdgcn_make_buffer_rsrc(
                    (char*)y1 + (long)(row0 - mv) * pitch, (short)0,
                    row0 + BM > mv ? min(mv + m1 - row0, BM) * pitch : 0, kRawBufferFormat);
                float bv[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int col = col0 + ei.wn * 64 + 16 * j + ei.l16;
                    bv[j] = (bias && col < n) ? bias[col] : 0.f;
                }
                const int cw = col0 + ei.wn * 64;     // the wave's first column
                const int cb = cw + (ln & 7) * 8;     // the lane's 16-byte chunk
                const uint32_t drop = cb < ny ? 0u : 0x80000000u;
                const uint32_t drop1 = cw + ln < ny ? 0u : 0x80000000u;
                auto store = [&](auto mode, const uint8_t* buf, int r0) {
                    constexpr int MODE = decltype(mode)::value;
                    constexpr int POLICY = MODE == kWholeSectors ? kNonTemporal : 0;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {   // eight rows, of one stream
                        const __amdgpu_buffer_rsrc_t rs = row0 + r0 + 8 * r < mv ? rs0 : rs1;
                        if constexpr (MODE == kElements) {
#pragma unroll
                            for (int i = 0; i < 8; ++i)
                                __builtin_amdgcn_raw_buffer_store_b16(
                                    *(const uint16_t*)(buf + (8 * r + i) * RP + ln * 2), rs,
                                    (uint32_t)((r0 + 8 * r + i) * pitch + (cw + ln) * 2) | drop1, 0, POLICY);
                        } else {
                            __builtin_amdgcn_raw_buffer_store_b128(
                                *(const u32x4*)(buf + (8 * r + (ln >> 3)) * RP + (ln & 7) * 16), rs,
                                (uint32_t)((r0 + 8 * r + (ln >> 3)) * pitch + cb * 2) | drop, 0, POLICY);
                        }
                    }
                };
                // (row scales come with whole chunks: linear_rows)
                const int mode = ACT != kActRowScale && (ny & 7) != 0 ? kElements
                                 : pitch % 64 == 0                    ? kWholeSectors
                                                                      : kPieces;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    uint8_t* buf = mine + (c & 1) * 32 * RP;
                    const int r0 = ei.wm * 128 + 32 * c;   // the quarter's first tile row
#pragma unroll
                    for (int ii = 0; ii < 2; ++ii) {
                        const int rl = 16 * ii + 4 * ei.g;
                        f32x4 sc;
                        if constexpr (ACT == kActRowScale)
                            sc = *reinterpret_cast<const f32x4*>(lr.scale + row0 + r0 + rl);
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            float v[4];
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                const float a = acc[2 * c + ii][j][r];
                                v[r] = ACT == kActRowScale ? fmaf(a, sc[r], bv[j]) : a + bv[j];
                                if (ACT == S2_ACT_GELU) v[r] = gelu(v[r]);
                            }
                            stage_rows4<YK>(buf + rl * RP + (16 * j + ei.l16) * 2, RP, v);
                        }
                    }
                    asm volatile("" ::: "memory");   // a wave's LDS accesses run in order
                    if (mode == kWholeSectors)
                        store(std::integral_constant<int, kWholeSectors>{}, buf, r0);
                    else if (mode == kPieces)
                        store(std::integral_constant<int, kPieces>{}, buf, r0);
                    else
                        store(std::integral_constant<int, kElements>{}, buf, r0);
                    asm volatile("" ::: "memory");
                }
            }
        }
    };

    // acc = sum over 64-k iterations [kb, ke) of the current tile.
    //
    // Ping-pong main loop.  The two waves of each SIMD (wave w and w + 4:
    // group 0 owns tile rows 0-127, group 1 rows 128-255) take turns: one
    // issues the 64 MFMAs of a whole 64-k step from fragment registers while
    // the other reads its fragments of the next step from LDS, so the matrix
    // core never waits on an LDS read.  Every phase ends at a workgroup
    // barrier; group 1 runs one phase behind group 0.  The DMA of a step is
    // split between the groups: group 1 loads the B rows into the stage it
    // has just finished reading (it is that stage's last reader), group 0 the
    // A rows one phase later; each waits for its DMA two phases after issuing
    // it, before the barrier that opens the stage to its first reader.
    //
    //   phase     2s                        2s + 1
    //   group 0   DMA A of step s + 1,      MFMAs of step s,
    //             read step s               wait for its DMA
    //   group 1   MFMAs of step s - 1       read step s, wait for its DMA of
    //                                       step s + 1, DMA B of step s + 2
    auto mainloop = [&](int kb, int ke, bool free) {
        const int grp = wave >> 2;
        const int wq = wave & 3;
        const int ld = lr.ld ? lr.ld : k;   // row pitch of x and of the weight
        // plain: the tile's rows of each stream; fused QKV: whole streams,
        // each DMA lane addressing its gathered row
        const i32x4 rav = AWA ? wave_uniform(buffer_rsrc(x0, (uint32_t)((long)m0 * k * 2)))
                              : wave_uniform(buffer_rsrc(
                                    x0 + (long)row0 * ld, (uint32_t)(max(min(m0 - row0, BM), 0) * ld * 2)));
        const i32x4 rat =
            AWA ? wave_uniform(buffer_rsrc(x1, (uint32_t)((long)m1 * k * 2)))
                : wave_uniform(buffer_rsrc(x1 + (long)(row0 - mv) * ld,
                                           (uint32_t)(row0 + BM > mv ? min(mv + m1 - row0, BM) * ld * 2 : 0)));
        const int wrow = __builtin_amdgcn_readfirstlane(row0 + wq * 64);
        const i32x4 rb =
            wave_uniform(buffer_rsrc(wgt + (long)col0 * ld, (uint32_t)(min(n - col0, BN) * ld * 2)));
        // Wave wq of a group fills LDS rows 64 wq .. 64 wq + 63 of its operand
        // (group 0: A, group 1: B) with 8 DMA instructions of 8 rows.  Row
        // r + 8j has the swizzle of row r with bit 2 flipped for odd j, so two
        // offsets serve all eight.
        const int row_a = wq * 64 + (lane >> 3);
        const uint32_t vrow =
            (uint32_t)((ACT == S2_ACT_SWIGLU && grp ? wq * 32 + (lane >> 3) : row_a) * ld * 2);
        const uint32_t voff_even = vrow + (((lane & 7) ^ lds_swizzle(row_a)) * 16);
        const uint32_t voff_odd = vrow + (((lane & 7) ^ lds_swizzle(row_a) ^ 4) * 16);
        // fused QKV: byte offsets of this lane's eight gathered A rows (a gap
        // or padding row points one row past its stream: the DMA reads zeros)
        if constexpr (AWA != 0) {
            if (grp == 0) {
                uint32_t go[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int src = qrows[row_a + 8 * j].src;
                    const int rr = src >= 0 ? src : (wrow + j * 8 < mv ? m0 : m1);
                    go[j] = (uint32_t)rr * (uint32_t)(k * 2) +
                            (uint32_t)((((lane & 7) ^ lds_swizzle(row_a) ^ ((j & 1) << 2))) * 16);
                }
                // lanes 16 bytes apart in each half, so a 16-lane read
                // phase covers all banks once
                goff_lds[wq * 64 + lane] = make_uint4(go[0], go[1], go[2], go[3]);
                goff_lds[256 + wq * 64 + lane] = make_uint4(go[4], go[5], go[6], go[7]);
            }
        }
        auto issue = [&](int stage, int kt, int operand) {
            const uint32_t soff = __builtin_amdgcn_readfirstlane((uint32_t)(kt * BK * 2));
            const uint32_t st = lds_base + stage * SB + operand * TB + wq * 8 * 1024;
            uint32_t go[8];
            if constexpr (AWA != 0) {
                if (!operand) {
                    const uint4 g0 = goff_lds[wq * 64 + lane];
                    const uint4 g1 = goff_lds[256 + wq * 64 + lane];
                    go[0] = g0.x; go[1] = g0.y; go[2] = g0.z; go[3] = g0.w;
                    go[4] = g1.x; go[5] = g1.y; go[6] = g1.z; go[7] = g1.w;
                }
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                uint32_t vo = ((j & 1) ? voff_odd : voff_even) + (uint32_t)(j * 8 * ld * 2);
                uint32_t so = soff;
                if constexpr (ACT == S2_ACT_SWIGLU)
                    if (operand) {
                        // LDS rows 64 wq + 16 q + c of the weight hold gate row
                        // 32 wq + 16 (q / 2) + c for even q and its up row for
                        // odd q; no tile of the weight is ragged
                        const int rj = ((j >> 1) & 1) * 128 + (j >> 2) * 16 + (j & 1) * 8;
                        vo = (j & 1) ? voff_odd : voff_even;
                        so = __builtin_amdgcn_readfirstlane(soff + (uint32_t)(rj * ld * 2));
                    }
                if constexpr (AWA != 0)
                    if (!operand) vo = go[j];
                lds_dma16(operand ? rb : (wrow + j * 8 < mv ? rav : rat),
                          __builtin_amdgcn_readfirstlane(st + j * 1024), vo, so);
            }
        };
        bf16x8 fa[2][8], fb[2][4];
        auto read_step = [&](int stage) {
            const uint8_t* st = lds + stage * SB;
#pragma unroll
            for (int kk = 0; kk < BK / 32; ++kk) {
                const int pc = ((4 * kk + g) ^ sw) * 16;
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    fa[kk][i] = as_bf16x8(*(const uint4*)(st + (wm * 128 + 16 * i + l16) * RB + pc));
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    fb[kk][j] =
                        as_bf16x8(*(const uint4*)(st + TB + (wn * 64 + 16 * j + l16) * RB + pc));
            }
        };
        auto barrier = [] {
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_barrier" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int steps = ke - kb;
        // steps 0 and 1: group 0 loads A, group 1 B
        issue(0, kb, grp);
        if (steps > 1) {
            issue(1, kb + 1, grp);
            asm volatile("s_waitcnt vmcnt(8)" ::: "memory");   // step 0; step 1 as in the loop
        } else {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        barrier();
        if (grp == 1) barrier();
#pragma unroll 1
        for (int s = 0; s < steps; ++s) {
            // memory phase
            if (grp == 0 && s >= 1 && s + 1 < steps) issue((s + 1) & 1, kb + s + 1, 0);
            read_step(s & 1);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (grp == 1) {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // B of step s + 1
                if (s + 2 < steps) issue(s & 1, kb + s + 2, 1);
            }
            barrier();
            // MFMA phase
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int kk = 0; kk < BK / 32; ++kk)
#pragma unroll
                for (int i = 0; i < 8; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[kk][i], fb[kk][j],
                                                                            acc[i][j], 0, 0, 0);
            __builtin_amdgcn_s_setprio(0);
            if (grp == 0) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // A of step s + 1
            if (!(free && grp == 1 && s + 1 == steps)) barrier();
        }
        // group 0's barrier matching group 1's last MFMA phase (free: neither;
        // group 1 read its last fragments before the barrier above)
        if (grp == 0 && !free) barrier();
    };

    // The same sum for fp32 and fp16 activations (XK != 1), which are rounded
    // to bf16 (nearest even) between global memory and LDS.
    //
    // The DMA cannot convert, so A passes through registers: 32-k steps halve
    // the fragments (48 registers) and leave room for two steps of A in flight
    // (2 x 16 registers of fp32).  Lane l of wave w loads four consecutive k
    // (chunk l % 8) of rows 32 w + l / 8 + 8 i, whole 128-byte lines for fp32,
    // and writes them as 8 bytes of LDS; B comes by DMA.  Four 32 KB stages of
    // 64-byte rows, 16-byte chunk c of row r at position c ^ ((r >> 2) & 3):
    // a read phase covers rows that share banks only four apart.  The groups
    // ping-pong as above, a phase being 32 k:
    //
    //   memory phase of step s   read step s; write A of step s + 2 (loaded
    //                            two steps ago) and DMA B of step s + 2 into
    //                            stage (s + 2) % 4, read last in step s - 2;
    //                            load A of step s + 4; wait for B of step s + 1
    //
    // 3677 x 2560 by 2560 x 2560 from fp32: 101 us (150 tiles on 256 CUs), 262 us
    // with the 128 kernel, which staged A through registers one step ahead and
    // rounded it with integer operations; 15064 x 3072 by 9216 x 3072 from fp32
    // 1074 against 2775 us, 1038 us from fp16, 272 x 2560 by 2560 x 2560 50
    // against 131 us.
    auto mainloop_cvt = [&](int kb, int ke) {
        if constexpr (XK != 1) {
        constexpr int ES = XK == 0 ? 4 : 2;      // bytes per activation
        constexpr int SBC = 2 * 256 * 64;        // stage bytes: A, then B
        typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
        typedef typename std::conditional<XK == 0, u32x4, u32x2>::type Raw;   // four k
        const int grp = wave >> 2;
        const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
            (char*)x0 + (long)row0 * k * ES, (short)0, max(min(m0 - row0, BM), 0) * k * ES,
            kRawBufferFormat);
        const __amdgpu_buffer_rsrc_t rt = __builtin_amdgcn_make_buffer_rsrc(
            (char*)x1 + (long)(row0 - mv) * k * ES, (short)0,
            row0 + BM > mv ? min(mv + m1 - row0, BM) * k * ES : 0, kRawBufferFormat);
        const i32x4 rb =
            wave_uniform(buffer_rsrc(wgt + (long)col0 * k, (uint32_t)(min(n - col0, BN) * k * 2)));
        const int wrow = __builtin_amdgcn_readfirstlane(row0 + wave * 32);
        const int arow = wave * 32 + (lane >> 3);
        const uint32_t aoff = (uint32_t)(arow * k * ES + (lane & 7) * 4 * ES);
        // LDS bytes of the lane's chunk in row arow; rows 8 apart differ in
        // bit 1 of the swizzle
        const uint32_t awr = (uint32_t)(arow * 64 + ((((lane & 7) >> 1) ^ ((arow >> 2) & 3)) << 4) +
                                        (lane & 1) * 8);
        const int brow = wave * 32 + (lane >> 2);
        const uint32_t boff = (uint32_t)(brow * k * 2 + (((lane & 3) ^ ((lane >> 4) & 3)) * 16));
        auto load_a = [&](int kt, Raw (&raw)[4]) {
            const int soff = __builtin_amdgcn_readfirstlane(kt * 32 * ES);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int vo = (int)aoff + i * 8 * k * ES;
                if constexpr (XK == 0) {
                    if (wrow + 8 * i < mv)
                        raw[i] = __builtin_amdgcn_raw_buffer_load_b128(rv, vo, soff, 0);
                    else
                        raw[i] = __builtin_amdgcn_raw_buffer_load_b128(rt, vo, soff, 0);
                } else {
                    if (wrow + 8 * i < mv)
                        raw[i] = __builtin_amdgcn_raw_buffer_load_b64(rv, vo, soff, 0);
                    else
                        raw[i] = __builtin_amdgcn_raw_buffer_load_b64(rt, vo, soff, 0);
                }
            }
        };
        auto write_a = [&](int stage, const Raw (&raw)[4]) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float f[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if constexpr (XK == 0)
                        f[e] = __uint_as_float(raw[i][e]);
                    else
                        f[e] = (float)__builtin_bit_cast(_Float16, (uint16_t)(raw[i][e >> 1] >> (16 * (e & 1))));
                }
                *(uint2*)(lds + stage * SBC + i * 512 + (awr ^ ((i & 1) << 5))) =
                    make_uint2(pack2_bf16_rne(f[0], f[1]), pack2_bf16_rne(f[2], f[3]));
            }
        };
        auto dma_b = [&](int stage, int kt) {
            const uint32_t soff = __builtin_amdgcn_readfirstlane((uint32_t)(kt * 64));
            const uint32_t st = lds_base + stage * SBC + SBC / 2 + wave * 32 * 64;
#pragma unroll
            for (int j = 0; j < 2; ++j)
                lds_dma16(rb, __builtin_amdgcn_readfirstlane(st + j * 1024),
                          boff + (uint32_t)(j * 16 * k * 2), soff);
        };
        bf16x8 fa[8], fb[4];
        const int pc = ((g ^ (l16 >> 2)) & 3) * 16;
        auto barrier = [] {
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_barrier" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int steps = 2 * (ke - kb);   // even, at least 2
        const int k0 = 2 * kb;
        Raw ra0[4], ra1[4];   // A of the next even and odd step to write
        {
            Raw p0[4], p1[4];
            load_a(k0, p0);
            load_a(k0 + 1, p1);
            dma_b(0, k0);
            dma_b(1, k0 + 1);
            if (steps > 2) {
                load_a(k0 + 2, ra0);
                load_a(k0 + 3, ra1);
            }
            write_a(0, p0);
            write_a(1, p1);
            if (steps > 2)
                asm volatile("s_waitcnt vmcnt(8)" ::: "memory");   // B of steps 0 and 1
            else
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        barrier();
        if (grp == 1) barrier();
        auto step = [&](int s, Raw (&raw)[4]) {
            const uint8_t* st = lds + (s & 3) * SBC;
#pragma unroll
            for (int i = 0; i < 8; ++i)
                fa[i] = as_bf16x8(*(const uint4*)(st + (wm * 128 + 16 * i + l16) * 64 + pc));
#pragma unroll
            for (int j = 0; j < 4; ++j)
                fb[j] = as_bf16x8(*(const uint4*)(st + SBC / 2 + (wn * 64 + 16 * j + l16) * 64 + pc));
            if (s + 2 < steps) {
                write_a((s + 2) & 3, raw);
                dma_b((s + 2) & 3, k0 + s + 2);
                if (s + 4 < steps) load_a(k0 + s + 4, raw);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            // B of step s + 1: in flight behind it are A of step s + 3, B of
            // step s + 2 and A of step s + 4
            if (s + 4 < steps)
                asm volatile("s_waitcnt vmcnt(10)" ::: "memory");
            else
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            barrier();
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_s_setprio(0);
            barrier();
        };
#pragma unroll 1
        for (int s = 0; s < steps; s += 2) {
            step(s, ra0);
            step(s + 1, ra1);
        }
        if (grp == 0) barrier();
        }
    };

    // Fused QKV epilogue.  The tile's 256 columns lie in one of q, k, v
    // (inner is a multiple of 256) and cover 256 / D heads from hbase.  The
    // tile is first rounded to bf16 (acc + bias, nearest even: the values a
    // bf16 QKV blob would hold) and staged in LDS, so that every value the
    // attention then reads is bit-identical to what the separate projection
    // and the attention prologue (awa_prologue_kernel) produce.
    //   q, k: row-major staging; D/8 threads per (row, head) hold 8
    //     channels each, reduce the sum of squares with DPP lane moves, apply
    //     rms_norm (:510-519) with the video or text weights, then
    //     apply_mm_rope (:521-543) at the row's position, in the prologue's
    //     fp32 operation order, and store 16 bytes of the head's row.
    //   v: transposed staging (channel rows of the 256 tile rows); every
    //     thread then stores 4-byte key pairs of V^T.  Window runs and the
    //     text rows start at even rows of the row space and segments at
    //     even workspace rows, so each pair of tile rows is one aligned pair
    //     of workspace keys.
    auto awa_epilogue = [&]() {
        if constexpr (AWA != 0) {
#pragma clang fp contract(off)
            constexpr int D = AWA;
            constexpr int SP = BN * 2 + 16;   // bytes per staged row
            // transposed (v) staging: 8-byte writes of 16 lanes to 16 rows,
            // of the next 16 lanes beside them; a pitch of 132 dwords puts
            // 32 lanes on distinct bank pairs
            constexpr int SPV = BN * 2 + 16;
            // an opaque copy of the thread index: nothing the epilogue derives
            // from it is hoisted above the main loop, where every register is
            // taken
            const EpiIds ei = epi_ids();
            const int etid = ei.tid;
            // the stores below are plain ones: the attention reads Q, K and V
            // next, from the caches where they fit (4160 rows: 190 us with
            // non-temporal stores, 188 with these; 21,664 rows: the same)
            const int part = col0 / awa.inner;   // 0 q, 1 k, 2 v
            const int hbase = (col0 - part * awa.inner) / D;
            __syncthreads();   // every wave is done reading the last stage
            auto stage = [&](auto v_tag) {
                constexpr bool V = decltype(v_tag)::value;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int cl = ei.wn * 64 + 16 * j + ei.l16;
                    const float bv = bias ? bias[col0 + cl] : 0.f;
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        // the four registers: rows rl .. rl + 3 of column cl
                        const int rl = ei.wm * 128 + 16 * i + 4 * ei.g;
                        float v[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = acc[i][j][e] + bv;
                        if constexpr (V)
                            *(uint2*)(lds + cl * SPV + rl * 2) =
                                make_uint2(pack2_bf16_rne(v[0], v[1]), pack2_bf16_rne(v[2], v[3]));
                        else
                            stage_rows4<1>(lds + rl * SP + cl * 2, SP, v);
                    }
                }
            };
            // one branch for the whole tile: with the choice inside the loop
            // the compiler branched for every fragment
            if (part < 2)
                stage(std::false_type{});
            else
                stage(std::true_type{});
            __syncthreads();
            if (part < 2) {
                constexpr int TPR = D / 8;        // threads per (row, head)
                uint16_t* dst = part == 0 ? awa.q : awa.k;
                const int ch = etid & 31;          // 8-channel chunk of the 256 columns
                const int hl = ch * 8 / D;
                const int d0 = ch * 8 - hl * D;
                float wv[8], wt[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    wv[i] = awa.norm[part * D + d0 + i];
                    wt[i] = awa.norm[(2 + part) * D + d0 + i];
                }
                // RoPE slots of this thread's four channel pairs: pair
                // (2p, 2p+1) of axis a lies in [a*2P, (a+1)*2P); 6P <= D.
                // The four pairs are consecutive, so they lie on axis axA
                // from pair pairA on, then (pairs split.. of a chunk that
                // crosses an axis boundary) on axis axA + 1 from pair 0.  A
                // row's position on axis a is bits [16(a & 1), +16) of
                // position word a / 2.
                const int P = awa.pairs;
                bool rot[4];
#pragma unroll
                for (int pp = 0; pp < 4; ++pp) rot[pp] = d0 + 2 * pp < 6 * P;
                const int axA = P > 0 ? min(d0 / (2 * P), 2) : 0;
                const int pairA = rot[0] ? (d0 - axA * 2 * P) >> 1 : 0;
                const int split = rot[0] ? min(P - pairA, 4) : 4;
                const int axB = min(axA + 1, 2);
                // (cos, sin) of the four pairs at a row's position, without
                // branches (so that the wait for these loads is exact): gap
                // rows hold position 0, and a pair past the rotated width
                // reads an entry at most three past its row's (the table has
                // kRopePad entries of slack) and does not use it.  The loads
                // of pass p + 1 are issued before pass p computes.
                const char* rope_b = reinterpret_cast<const char*>(awa.rope);
                auto rope_load = [&](const QkvRow& ri, float2 (&cs)[4]) {
                    const uint32_t wa = axA == 2 ? ri.pos2 : ri.pos01;
                    const uint32_t wb = axB == 2 ? ri.pos2 : ri.pos01;
                    const uint32_t posA = (wa >> (16 * (axA & 1))) & 0xffff;
                    const uint32_t posB = (wb >> (16 * (axB & 1))) & 0xffff;
                    // byte offsets of pair 0 of the chunk on each axis
                    const uint32_t offA = (__umul24(posA, (uint32_t)P) + pairA) * 8;
                    const uint32_t offB = __umul24(posB, (uint32_t)P) * 8 - split * 8;
#pragma unroll
                    for (int pp = 0; pp < 4; ++pp) {
                        const uint32_t off = (pp < split ? offA : offB) + 8 * pp;
                        cs[pp] = *reinterpret_cast<const float2*>(rope_b + off);
                    }
                };
                // The results of all passes stay in registers (the
                // accumulators are dead by now) and are stored after the
                // loop, so the loop holds loads only and each pass waits for
                // its own loads, not for earlier stores.
                constexpr int PASSES = BM / 16;
                uint4 res[PASSES];
                // Only the tile holding the first text row (the row space is
                // the video rows in window order, then the text rows) selects
                // between the video and text weights per row.
                // (and the rounding mode is one branch around the passes: a
                // branch in each would keep the compiler from overlapping them)
                auto passes = [&](auto text_tag, auto official_tag) {
                constexpr bool TEXT = decltype(text_tag)::value;
                constexpr bool OFFICIAL = decltype(official_tag)::value;
                QkvRow ri_next = qrows[etid >> 5];
                uint4 raw_next = *(const uint4*)(lds + (etid >> 5) * SP + ch * 16);
                float2 cs_next[4];
                rope_load(ri_next, cs_next);
#pragma unroll
                for (int pass = 0; pass < PASSES; ++pass) {
                    const int rl = pass * 16 + (etid >> 5);
                    const QkvRow ri = ri_next;
                    float2 cs[4];
#pragma unroll
                    for (int pp = 0; pp < 4; ++pp) cs[pp] = cs_next[pp];
                    const uint4 raw = raw_next;
                    if (pass + 1 < PASSES) {
                        ri_next = qrows[rl + 16];
                        raw_next = *(const uint4*)(lds + (rl + 16) * SP + ch * 16);
                        rope_load(ri_next, cs_next);
                    }
                    const int kind = ri.pos2 >> 16;
                    const uint32_t wd[4] = {raw.x, raw.y, raw.z, raw.w};
                    float x[8];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        x[2 * i] = __uint_as_float(wd[i] << 16);
                        x[2 * i + 1] = __uint_as_float(wd[i] & 0xffff0000u);
                    }
                    float ss = x[0] * x[0];
#pragma unroll
                    for (int i = 1; i < 8; ++i) ss = fmaf(x[i], x[i], ss);
                    ss = row_sum<TPR>(ss);
                    const float inv = __builtin_amdgcn_rsqf(ss / (float)D + awa.eps);
                    const bool video = !TEXT || kind == 1;
#pragma unroll
                    for (int i = 0; i < 8; ++i) x[i] = x[i] * inv * (video ? wv[i] : wt[i]);
#pragma unroll
                    for (int pp = 0; pp < 4; ++pp) {
                        if (rot[pp]) {
                            const float a0 = x[2 * pp], a1 = x[2 * pp + 1];
                            x[2 * pp] = fmaf(a0, cs[pp].x, -(a1 * cs[pp].y));
                            x[2 * pp + 1] = fmaf(a0, cs[pp].y, a1 * cs[pp].x);
                        }
                    }
                    if constexpr (OFFICIAL) {
                        uint16_t hb[8];
#pragma unroll
                        for (int i = 0; i < 8; ++i) hb[i] = round_bf16_ref_bits(x[i]);
                        res[pass] = pack8_bf16(hb);
                    } else {
                        res[pass] = cvt8_bf16(x);
                    }
                }
                };
                const bool text = row0 + BM > mv;
                if (awa.official_bf16)
                    text ? passes(std::true_type{}, std::true_type{})
                         : passes(std::false_type{}, std::true_type{});
                else
                    text ? passes(std::true_type{}, std::false_type{})
                         : passes(std::false_type{}, std::false_type{});
#pragma unroll
                for (int pass = 0; pass < PASSES; ++pass) {
                    const QkvRow ri = qrows[pass * 16 + (etid >> 5)];
                    if (ri.pos2 >> 16)
                        *(u32x4*)(dst + ((long)(hbase + hl) * awa.seg_total + ri.dest) * D + d0) =
                            __builtin_bit_cast(u32x4, res[pass]);
                }
            } else {
                // thread t stores key pair t % 128 (tile rows 2q, 2q + 1) of
                // channels t / 128 + 4c
                const int qp = etid & 127;
                const QkvRow ri = qrows[2 * qp];
                if (ri.pos2 >> 16) {
                    uint16_t* base = awa.vt + (long)hbase * D * awa.seg_total + ri.dest;
#pragma unroll 8
                    for (int c = 0; c < 64; ++c) {
                        const int cl = (etid >> 7) + 4 * c;
                        const uint32_t v = *(const uint32_t*)(lds + cl * SPV + qp * 4);
                        *(uint32_t*)(base + (long)cl * awa.seg_total) = v;
                    }
                }
            }
        }
    };

    // SwiGLU: the weight's rows come in blocks of 256, the first 128 gate
    // rows and the next 128 up rows of output columns col0/2 .. col0/2 + 127.
    // The DMA puts a column's gate and up rows 16 LDS rows apart (issue), so
    // that a lane's accumulators [i][2q] and [i][2q + 1] are the gate and the
    // up of column 32 wn + 16 q + l16: silu(g) * u is formed in registers and
    // staged once, in the output type.  (2464 rows of the v3 MLP: 147 us, 151
    // with fp32 gates and ups staged in two halves of 128 rows.)
    auto swiglu_epilogue = [&]() {
        if constexpr (ACT == S2_ACT_SWIGLU) {
            const EpiIds ei = epi_ids();
            constexpr int ES = YK ? 2 : 4;
            constexpr int SP = 128 * ES + 16;   // staged row pitch (bytes)
            static_assert(BM * SP <= LDS_BYTES, "staged tile exceeds the LDS");
            __syncthreads();   // every wave is done reading the last stage
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int cl = ei.wn * 32 + 16 * q + ei.l16;
                const bool in = col0 + cl < n;   // n is a multiple of 256
                const float bg = bias && in ? bias[col0 + cl] : 0.f;
                const float bu = bias && in ? bias[col0 + 128 + cl] : 0.f;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int rl = ei.wm * 128 + 16 * i + 4 * ei.g;
                    float o[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        // silu(g) = g / (1 + e^-g), e^-g = 2^(-g log2 e)
                        const float gg = acc[i][2 * q][e] + bg;
                        const float sig = __builtin_amdgcn_rcpf(
                            1.f + __builtin_amdgcn_exp2f(-gg * 1.4426950408889634f));
                        o[e] = gg * sig * (acc[i][2 * q + 1][e] + bu);
                    }
                    if constexpr (YK == 0) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) *(float*)(lds + (rl + e) * SP + cl * 4) = o[e];
                    } else {
                        stage_rows4<YK>(lds + rl * SP + cl * 2, SP, o);
                    }
                }
            }
            __syncthreads();
            constexpr int CPR = 128 * ES / 16;   // 16-byte chunks per row
#pragma unroll 8
            for (int it = 0; it < BM * CPR / 512; ++it) {
                const int idx = it * 512 + ei.tid;
                const int rl = idx / CPR, ch = idx % CPR;
                char* yr = (char*)out_row(rl);
                const int col = col0 / 2 + ch * (16 / ES);
                if (yr && col < ny)
                    __builtin_nontemporal_store(*(const u32x4*)(lds + rl * SP + ch * 16),
                                                (u32x4*)(yr + (long)col * ES));
            }
        }
    };

    // fp32 outputs, as in wave_epilogue: a wave's rows leave 16 at a time, 256
    // bytes of 4 rows a store (in two halves of 128 whole rows before: 3677 x 2560
    // by 2560 x 2560 from fp32 104 us, 101 so), or of one row where n % 4 != 0 (4609
    // x 512 by 4609 x 512 65 us straight from the accumulators, 40 so).
    auto wave_epilogue_f32 = [&]() {
        if constexpr (YK == 0 && AWA == 0 && RES == 0 && ACT != S2_ACT_SWIGLU) {
            const EpiIds ei = epi_ids();
            const int ln = ei.tid & 63;
            constexpr int RP = 64 * 4 + 16;   // staged row (bytes)
            static_assert(2 * 16 * RP <= kWaveStage, "two parts of 16 rows");
            uint8_t* mine = lds + (ei.wm * 4 + ei.wn) * kWaveStage;
            const int pitch = n * 4;
            const __amdgpu_buffer_rsrc_t rs0 = __builtin_amdgcn_make_buffer_rsrc(
                (char*)y0 + (long)row0 * pitch, (short)0, max(min(m0 - row0, BM), 0) * pitch,
                kRawBufferFormat);
            const __amdgpu_buffer_rsrc_t rs1 = __builtin_amdgcn_make_buffer_rsrc(
                (char*)y1 + (long)(row0 - mv) * pitch, (short)0,
                row0 + BM > mv ? min(mv + m1 - row0, BM) * pitch : 0, kRawBufferFormat);
            float bv[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int col = col0 + ei.wn * 64 + 16 * j + ei.l16;
                bv[j] = (bias && col < n) ? bias[col] : 0.f;
            }
            const int cw = col0 + ei.wn * 64;      // the wave's first column
            const int cb = cw + (ln & 15) * 4;     // the lane's 16-byte chunk
            const uint32_t drop = cb < n ? 0u : 0x80000000u;
            const uint32_t drop1 = cw + ln < n ? 0u : 0x80000000u;
            auto store = [&](auto mode, const uint8_t* buf, int r0) {
                constexpr int MODE = decltype(mode)::value;
                constexpr int POLICY = MODE == kWholeSectors ? kNonTemporal : 0;
#pragma unroll
                for (int r = 0; r < 4; ++r) {   // four rows, of one stream
                    const __amdgpu_buffer_rsrc_t rs = row0 + r0 + 4 * r < mv ? rs0 : rs1;
                    if constexpr (MODE == kElements) {
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            __builtin_amdgcn_raw_buffer_store_b32(
                                *(const uint32_t*)(buf + (4 * r + i) * RP + ln * 4), rs,
                                (uint32_t)((r0 + 4 * r + i) * pitch + (cw + ln) * 4) | drop1, 0, POLICY);
                    } else {
                        __builtin_amdgcn_raw_buffer_store_b128(
                            *(const u32x4*)(buf + (4 * r + (ln >> 4)) * RP + (ln & 15) * 16), rs,
                            (uint32_t)((r0 + 4 * r + (ln >> 4)) * pitch + cb * 4) | drop, 0, POLICY);
                    }
                }
            };
            const int mode = (n & 3) != 0 ? kElements : pitch % 64 == 0 ? kWholeSectors : kPieces;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                uint8_t* buf = mine + (i & 1) * 16 * RP;
                const int r0 = ei.wm * 128 + 16 * i;
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        float v = acc[i][j][r] + bv[j];
                        if (ACT == S2_ACT_GELU) v = gelu(v);
                        *(float*)(buf + (4 * ei.g + r) * RP + (16 * j + ei.l16) * 4) = v;
                    }
                asm volatile("" ::: "memory");   // a wave's LDS accesses run in order
                if (mode == kWholeSectors)
                    store(std::integral_constant<int, kWholeSectors>{}, buf, r0);
                else if (mode == kPieces)
                    store(std::integral_constant<int, kPieces>{}, buf, r0);
                else
                    store(std::integral_constant<int, kElements>{}, buf, r0);
                asm volatile("" ::: "memory");
            }
        }
    };

    // Residual epilogue, as in wave_epilogue: a quarter's projection, rounded
    // to bf16, is staged in the wave's own LDS while the residual of the next
    // quarter is on its way; a lane then holds 4 columns of 8 rows.  out may be
    // x: each element is read and written by one lane.  (Assembled over a
    // workgroup and loaded in two halves before: MLP of 1485 rows 216 us, 210
    // so; of the 720p video 1816 and 1803.)
    //
    // A wave goes over its part once for each (stream, sample) that it has rows
    // of, nearly always one, behind descriptors that end with those rows: the
    // gate, the descriptor and the residual's type are then fixed for straight
    // code, where the loads of a quarter are waited for without the stores issued
    // since.  With their branches in every row a launch of few tiles, which
    // nothing else hides, took 14 us longer: 64 rows of 2560 to 2560 50.1 us (40.2
    // assembled over a workgroup), 33.8 so; 1549 rows of 10240 to 2560 109 and 98,
    // 21,664 rows 879 and 854.
    auto wave_residual = [&]() {
        if constexpr (RES != 0) {
#pragma clang fp contract(off)
            const EpiIds ei = epi_ids();
            const int ln = ei.tid & 63;
            constexpr int RP = 64 * 2 + 16;   // staged row (bytes)
            uint8_t* mine = lds + (ei.wm * 4 + ei.wn) * kWaveStage;
            const int wrow = row0 + 128 * ei.wm;   // the wave's first row
            const int sub = ln >> 4;
            const int col = col0 + ei.wn * 64 + (ln & 15) * 4;   // n is a multiple of 8
            const bool in = col < n;
            float bv[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int c = col0 + ei.wn * 64 + 16 * j + ei.l16;
                bv[j] = (bias && c < n) ? bias[c] : 0.f;
            }
            // rows [l, e) of the stream, which lies `at` rows above the wave
            auto segment = [&](auto kind, const void* x, void* out, f32x4 g, int at, int l, int e) {
                constexpr int KIND = decltype(kind)::value;
                constexpr int ES = KIND == 0 ? 4 : 2;
                typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
                typedef typename std::conditional<KIND == 0, u32x4, u32x2>::type Raw;   // four columns
                const int pitch = n * ES;
                const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
                    (char*)const_cast<void*>(x) + (long)l * pitch, (short)0, (e - l) * pitch, kRawBufferFormat);
                const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
                    (char*)out + (long)l * pitch, (short)0, (e - l) * pitch, kRawBufferFormat);
                // (rows above l have negative offsets, which are past the end too;
                // a column past n starts half the range away, so that no row's
                // offset brings it back)
                const uint32_t off = in ? (uint32_t)((at + sub - l) * pitch + col * ES) : 0x80000000u;
                auto load = [&](int c, Raw (&raw)[8]) {
#pragma unroll
                    for (int r = 0; r < 8; ++r) {
                        const int so = (32 * c + 4 * r) * pitch;
                        if constexpr (KIND == 0)
                            raw[r] = __builtin_amdgcn_raw_buffer_load_b128(rx, off + so, 0, kNonTemporal);
                        else
                            raw[r] = __builtin_amdgcn_raw_buffer_load_b64(rx, off + so, 0, kNonTemporal);
                    }
                };
                Raw raw[2][8];
                load(0, raw[0]);
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    if (c < 3) load(c + 1, raw[(c + 1) & 1]);
                    uint8_t* buf = mine + (c & 1) * 32 * RP;
#pragma unroll
                    for (int ii = 0; ii < 2; ++ii)
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            float v[4];
#pragma unroll
                            for (int r = 0; r < 4; ++r) v[r] = acc[2 * c + ii][j][r] + bv[j];
                            stage_rows4<1>(buf + (16 * ii + 4 * ei.g) * RP + (16 * j + ei.l16) * 2, RP, v);
                        }
                    asm volatile("" ::: "memory");   // a wave's LDS accesses run in order
#pragma unroll
                    for (int r = 0; r < 8; ++r) {
                        const Raw xr = raw[c & 1][r];
                        const uint2 yw = *(const uint2*)(buf + (4 * r + sub) * RP + (ln & 15) * 8);
                        float o[4];
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const uint16_t hv = (uint16_t)(xr[i >> 1] >> (16 * (i & 1)));
                            const float xf = KIND == 0   ? __uint_as_float(xr[KIND == 0 ? i : 0])
                                             : KIND == 1 ? bf16_to_f32(hv)
                                                         : (float)__builtin_bit_cast(_Float16, hv);
                            const uint32_t w = i >> 1 ? yw.y : yw.x;
                            const float y = __uint_as_float(i & 1 ? (w & 0xffff0000u) : (w << 16));
                            const float p = y * g[i];
                            o[i] = xf + p;
                        }
                        const int so = (32 * c + 4 * r) * pitch;
                        if constexpr (KIND == 0) {
                            const u32x4 ov = {__float_as_uint(o[0]), __float_as_uint(o[1]),
                                              __float_as_uint(o[2]), __float_as_uint(o[3])};
                            __builtin_amdgcn_raw_buffer_store_b128(ov, ro, off + so, 0, kNonTemporal);
                        } else {
                            const u32x2 ov = KIND == 1
                                                 ? u32x2{pack2_bf16_rne(o[0], o[1]), pack2_bf16_rne(o[2], o[3])}
                                                 : u32x2{pack2_f16_rne(o[0], o[1]), pack2_f16_rne(o[2], o[3])};
                            __builtin_amdgcn_raw_buffer_store_b64(ov, ro, off + so, 0, kNonTemporal);
                        }
                    }
                    asm volatile("" ::: "memory");
                }
            };
#pragma unroll 1
            for (int stream = wrow < mv ? 0 : 1; stream < 2; ++stream) {
                const int* ends = res.rows.end + stream * kAdaMaxBatch;
                const int at = wrow - (stream ? mv : 0);   // the wave's first row, from the stream's
                const int last = min(at + 128, stream ? m1 : m0);
                int l = max(at, 0), b = 0;
#pragma unroll 1
                while (l < last) {
                    while (b + 1 < res.rows.batch && l >= ends[b]) ++b;
                    const int e = b + 1 < res.rows.batch ? min(ends[b], last) : last;
                    const void* x = stream ? res.x[1] : res.x[0];
                    void* out = stream ? res.out[1] : res.out[0];
                    const float* gs = stream ? res.gate_s[1] : res.gate_s[0];
                    f32x4 g = {0.f, 0.f, 0.f, 0.f};
                    if (in) {
                        g = *reinterpret_cast<const f32x4*>(res.gate + (long)b * n + col);
                        if (gs) g += *reinterpret_cast<const f32x4*>(gs + col);
                    }
                    if (res.x_kind == 0)
                        segment(std::integral_constant<int, 0>{}, x, out, g, at, l, e);
                    else if (res.x_kind == 1)
                        segment(std::integral_constant<int, 1>{}, x, out, g, at, l, e);
                    else
                        segment(std::integral_constant<int, 2>{}, x, out, g, at, l, e);
                    l = e;
                }
            }
        }
    };

    // y tile = act(acc + bias)
    auto epilogue = [&]() {
        if constexpr (AWA != 0) {
            awa_epilogue();
            return;
        }
        if constexpr (ACT == S2_ACT_SWIGLU) {
            swiglu_epilogue();
            return;
        }
        if constexpr (RES != 0) {
            wave_residual();
            return;
        }
        if constexpr (YK != 0)
            wave_epilogue();
        else
            wave_epilogue_f32();
    };

    // Work of this workgroup as segments (tile, k-iterations [kb, ke)).  A
    // data-parallel workgroup has one whole tile.  Stream-K workgroup s owns
    // iterations [bound(s), bound(s + 1)) of the split tiles, iteration i
    // being k-step i % nk of split tile i / nk.
    const bool split = (int)blockIdx.x >= sk.dp_tiles;
    // consecutive ranges (neighbouring tiles of the raster) on one XCD, so
    // that they share A and B panels in its L2 (dp_tiles is a multiple of 8)
    const int s = split ? xcd_remap(blockIdx.x - sk.dp_tiles, sk.sk_groups) : 0;
    const long total = (long)sk.sk_tiles * nk;
    auto bound = [&](long q) { return q * total / sk.sk_groups; };
    // the stream-K workgroup whose range holds iteration i
    auto owner = [&](long i) { return (int)(((i + 1) * sk.sk_groups - 1) / total); };
    long i = split ? bound(s) : 0;
    const long iend = split ? bound(s + 1) : nk;
    bool first = true;
#pragma unroll 1
    while (i < iend) {
        int t, kb, ke;
        if (split) {
            t = (int)(i / nk);
            kb = (int)(i - (long)t * nk);
            ke = (int)min((long)nk, kb + (iend - i));
            set_tile(sk.dp_tiles + t);
        } else {
            t = 0;
            kb = 0;
            ke = nk;
            set_tile(xcd_remap(blockIdx.x, sk.dp_tiles));
        }
        if (!first) __syncthreads();   // the previous segment's LDS is no longer read
        if constexpr (AWA != 0) {
            build_rows();
            __syncthreads();
        }
        bool finish = kb == 0 && ke == nk;
        // a whole tile whose waves write their own parts: no wave meets
        // another after the last MFMA phase, so the barrier there is left out
        const bool free = AWA == 0 && XK == 1 && ACT != S2_ACT_SWIGLU && finish;
        if constexpr (XK == 1)
            mainloop(kb, ke, free);
        else
            mainloop_cvt(kb, ke);
        if (!finish) {
            // slot layout: float4 c (4 accumulator registers) of thread tid
            // at byte (c * 512 + tid) * 16; the chunk index goes in soffset
            const __amdgpu_buffer_rsrc_t mine = __builtin_amdgcn_make_buffer_rsrc(
                sk.slots + (long)s * kSlotFloats, (short)0, kSlotFloats * 4, kRawBufferFormat);
#pragma unroll
            for (int ii = 0; ii < 8; ++ii)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    __builtin_amdgcn_raw_buffer_store_b128(
                        __builtin_bit_cast(u32x4, acc[ii][j]), mine, tid * 16,
                        (ii * 4 + j) * 512 * 16, kCoherent);
            // The slot stores write through to memory; every wave waits for
            // its own before the workgroup barrier.  The arrival is an
            // agent-scope acquire-release read-modify-write: it releases this
            // part's slot (ordered after the barrier) and, for the last part,
            // acquires every earlier part's, which the second barrier passes
            // on to the other waves of the workgroup.
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            if (tid == 0)
                arrival = __hip_atomic_fetch_add(&sk.counters[t], 1, __ATOMIC_ACQ_REL,
                                                 __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();
            const int lo = owner((long)t * nk);
            const int hi = owner((long)t * nk + nk - 1);
            if (arrival == hi - lo) {
                // sum every part, this one's included, in workgroup order so
                // that the result does not depend on the order of arrival; of
                // two parts only the other is read (p0 + p1 either way round)
                const bool two = hi == lo + 1;
                if (!two) {
#pragma unroll
                    for (int ii = 0; ii < 8; ++ii)
#pragma unroll
                        for (int j = 0; j < 4; ++j) acc[ii][j] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
#pragma unroll 1
                for (int q = lo; q <= hi; ++q) {
                    if (two && q == s) continue;
                    const __amdgpu_buffer_rsrc_t other = __builtin_amdgcn_make_buffer_rsrc(
                        sk.slots + (long)q * kSlotFloats, (short)0, kSlotFloats * 4, kRawBufferFormat);
                    // sixteen 16-byte loads in flight per batch (sixteen
                    // accumulators; the fragment registers are free here)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        __builtin_amdgcn_sched_barrier(0);
                        f32x4 v[4][4];
#pragma unroll
                        for (int iq = 0; iq < 4; ++iq)
#pragma unroll
                            for (int j = 0; j < 4; ++j)
                                v[iq][j] = __builtin_bit_cast(
                                    f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                               other, tid * 16,
                                               ((4 * h + iq) * 4 + j) * 512 * 16, kCoherent));
#pragma unroll
                        for (int iq = 0; iq < 4; ++iq)
#pragma unroll
                            for (int j = 0; j < 4; ++j)
#pragma unroll
                                for (int r = 0; r < 4; ++r) acc[4 * h + iq][j][r] += v[iq][j][r];
                    }
                }
                if (tid == 0)
                    __hip_atomic_store(&sk.counters[t], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                finish = true;
            }
        }
        if (finish) epilogue();
        // every memory operation of this segment is complete: a real
        // s_waitcnt (not asm) lets the compiler's wait insertion know, so
        // it adds no vmcnt wait of its own inside the next main loop
        __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
        first = false;
        i += ke - kb;
    }
}

__global__ void cast_f32_bf16_kernel(const float* __restrict__ src, uint16_t* __restrict__ dst,
                                     size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = f32_to_bf16(src[i]);
}

__global__ void cast_bf16_f32_kernel(const uint16_t* __restrict__ src, float* __restrict__ dst,
                                     size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = bf16_to_f32(src[i]);
}

// Elementwise erf-GELU (the epilogue's gelu) over fp32, bf16 or fp16 values,
// four per thread.
template <typename T>
__global__ void gelu_kernel(const T* x, T* y, size_t n) {
    const size_t i0 = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const size_t i = i0 + j;
        if (i >= n) return;
        if constexpr (std::is_same<T, float>::value)
            y[i] = gelu(x[i]);
        else if constexpr (std::is_same<T, uint16_t>::value)
            y[i] = __builtin_bit_cast(uint16_t, (__bf16)gelu(bf16_to_f32(x[i])));
        else
            y[i] = f32_to_f16(gelu((float)x[i]));
    }
}

hipError_t launch_gelu(const void* x, void* y, size_t n, int kind, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    const unsigned blocks = (unsigned)((n + 1023) / 1024);
    if (kind == 1)
        gelu_kernel<uint16_t><<<blocks, 256, 0, stream>>>((const uint16_t*)x, (uint16_t*)y, n);
    else if (kind == 2)
        gelu_kernel<_Float16><<<blocks, 256, 0, stream>>>((const _Float16*)x, (_Float16*)y, n);
    else
        gelu_kernel<float><<<blocks, 256, 0, stream>>>((const float*)x, (float*)y, n);
    return hipGetLastError();
}

hipError_t launch_cast_f32_bf16(const float* src, uint16_t* dst, size_t n, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    cast_f32_bf16_kernel<<<(unsigned)((n + 255) / 256), 256, 0, stream>>>(src, dst, n);
    return hipGetLastError();
}

hipError_t launch_cast_bf16_f32(const uint16_t* src, float* dst, size_t n, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    cast_bf16_f32_kernel<<<(unsigned)((n + 255) / 256), 256, 0, stream>>>(src, dst, n);
    return hipGetLastError();
}

// Scratch of the split-k tail: one partial-accumulator slot per workgroup
// that shares a tile (at most one per CU), then one arrival counter per
// shared tile (fewer than the CUs).
namespace {

constexpr int kMaxDevices = 64;

// Compute units of the current device (the workgroups of one wave of tiles).
hipError_t device_cus(int* cus) {
    static int g_cus[kMaxDevices];
    static std::once_flag g_once[kMaxDevices];
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    std::call_once(g_once[dev], [dev] {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            n = 0;
        g_cus[dev] = n > 0 ? n : 256;
    });
    *cus = g_cus[dev];
    return hipSuccess;
}

size_t sk_scratch_bytes(int groups) {
    return (size_t)groups * kSlotFloats * sizeof(float) + (size_t)groups * sizeof(int);
}

}  // namespace

// Split-k scratch of a stream on the current device: a slot per compute unit.
hipError_t splitk_scratch_bytes(size_t* bytes) {
    int G = 0;
    const hipError_t e = device_cus(&G);
    if (e == hipSuccess) *bytes = sk_scratch_bytes(G);
    return e;
}

namespace {

// The no-allocation entry point's scratch: slots and counters for up to
// kNoallocGroups sharing workgroups (the split of a 256-CU device), about
// 64 MB that every GPU the library runs on holds until the process ends.
constexpr int kNoallocGroups = 256;
constexpr size_t kNoallocBytes = (size_t)kNoallocGroups * kSlotFloats * sizeof(float) +
                                 (size_t)kNoallocGroups * sizeof(int);
static __device__ __align__(256) unsigned char scratch[kNoallocBytes];

// Device address of `scratch` on the current device.  The host-side name is
// only a stand-in for the symbol: kernels get this address instead.
hipError_t noalloc_scratch(void** out) {
    static void* g_ptr[kMaxDevices];
    static hipError_t g_err[kMaxDevices];
    static std::once_flag g_once[kMaxDevices];
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    std::call_once(g_once[dev], [dev] {
        void* p = nullptr;
        g_err[dev] = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        g_ptr[dev] = p;
    });
    if (g_err[dev] != hipSuccess) return g_err[dev];
    *out = g_ptr[dev];
    return hipSuccess;
}

__global__ void zero_counters_kernel(int* counters, int n) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) counters[i] = 0;
}

}  // namespace

// Where the split-k tail keeps its partial tiles: the calling stream's own
// allocation (stream_scratch), or, for the no-allocation entry point, the
// static `scratch` array (whose counters are cleared before every launch
// that uses them, since a call keeps whatever the last one left).  kOptional is
// the stream's where there is one or one can be made, else no split: for calls
// that have to work on a capturing stream that nobody owns.
enum class SkSource { kStream, kOptional, kStatic };

// Split-k tail of a launch of `tiles` 256x256 tiles with nk 64-k steps:
// when the last wave of tiles would leave more than 3% of the workgroup
// slots idle, each tile of that wave is split along k into P equal parts on
// P workgroups (P <= 4, at least 8 k-iterations a part): the wave then takes
// about 1/P of a tile's time plus the reduction of P partial tiles.
static hipError_t plan_sk_tail(long tiles, int nk, SkSource source, hipStream_t stream, SkTail* out) {
    int G = 0;
    hipError_t e = device_cus(&G);
    if (e != hipSuccess) return e;
    SkTail sk{(int)tiles, 0, 0, nullptr, nullptr};
    const long waves = (tiles + G - 1) / G;
    const long rem = tiles % G == 0 ? G : tiles % G;
    if ((double)tiles / (double)(waves * G) < 0.97) {
        const long parts = std::min<long>(4, std::min<long>(G / rem, nk / 8));
        if (parts >= 2) {
            sk.dp_tiles = (int)(tiles - rem);
            sk.sk_tiles = (int)rem;
            sk.sk_groups = (int)(rem * parts);
        }
    }
    if (sk.sk_groups > 0) {
        void* base = nullptr;
        if (source == SkSource::kStatic) {
            // (hipErrorNotSupported: the caller reports a size beyond the
            // static scratch)
            if (sk.sk_groups > kNoallocGroups) return hipErrorNotSupported;
            e = noalloc_scratch(&base);
            if (e != hipSuccess) return e;
            sk.slots = (float*)base;
            sk.counters = (int*)((char*)base + (size_t)kNoallocGroups * kSlotFloats * 4);
            zero_counters_kernel<<<1, 256, 0, stream>>>(sk.counters, sk.sk_tiles);
            e = hipGetLastError();
            if (e != hipSuccess) return e;
        } else {
            e = source == SkSource::kOptional
                    ? stream_scratch_optional(kScratchSplitK, stream, sk_scratch_bytes(G), &base)
                    : stream_scratch(kScratchSplitK, stream, sk_scratch_bytes(G), &base);
            if (e != hipSuccess) return e;
            if (!base) {
                *out = SkTail{(int)tiles, 0, 0, nullptr, nullptr};
                return hipSuccess;
            }
            sk.slots = (float*)base;
            sk.counters = (int*)((char*)base + (size_t)G * kSlotFloats * 4);
        }
    }
    *out = sk;
    return hipSuccess;
}

template <typename TX, int YK, int ACT>
static hipError_t linear_impl(const void* x0, int m0, const void* x1, int m1, const uint16_t* w,
                              const float* bias, int n, int k, void* y0, void* y1,
                              hipStream_t stream, SkSource source) {
    // k that is no multiple of the 64-k step, and tiles beyond the buffers'
    // 32-bit offsets, take the 128 kernel
    if (k % 64 == 0 && (long)256 * k * (long)sizeof(TX) <= 0x7fffffffL &&
        (long)256 * n * 4 <= 0x7fffffffL) {
        constexpr int XK = std::is_same<TX, float>::value ? 0 : std::is_same<TX, uint16_t>::value ? 1 : 2;
        const int mv = (m0 + 7) / 8 * 8;   // first text row in the joint row space
        const int ntiles = (n + 255) / 256;
        const int mtiles = (mv + m1 + 255) / 256;
        const long tiles = (long)mtiles * ntiles;
        if (tiles == 0) return hipSuccess;
        SkTail sk;
        hipError_t e = plan_sk_tail(tiles, k / 64, source, stream, &sk);
        if (e != hipSuccess) return e;
        const long blocks = (long)sk.dp_tiles + sk.sk_groups;
        shared_linear_256_kernel<YK, ACT, 0, 0, XK><<<(unsigned)blocks, 512, 0, stream>>>(
            (const uint16_t*)x0, m0, (const uint16_t*)x1, m1, w, bias, n, k, y0, y1, mv, mtiles,
            ntiles, sk, AwaQkvArgs{}, LinearResidual{}, LinearRows{});
        return hipGetLastError();
    }
    if constexpr (ACT == S2_ACT_SWIGLU) {
        return hipErrorInvalidValue;   // the 128 kernel has no gate
    } else {
        const int mt0 = (m0 + 127) / 128;
        const int mt1 = (m1 + 127) / 128;
        const int ntiles = (n + 127) / 128;
        const int mtiles = mt0 + mt1;
        const long blocks = (long)mtiles * ntiles;
        if (blocks == 0) return hipSuccess;
        shared_linear_kernel<TX, YK, ACT><<<(unsigned)blocks, 256, 0, stream>>>(
            (const TX*)x0, m0, (const TX*)x1, m1, w, bias, n, k, y0, y1, mt0, mtiles, ntiles);
        return hipGetLastError();
    }
}

template <typename TX, int YK>
static hipError_t linear_act(int act, const void* x0, int m0, const void* x1, int m1,
                             const uint16_t* w, const float* bias, int n, int k, void* y0,
                             void* y1, hipStream_t stream, SkSource src) {
    if (act == S2_ACT_SWIGLU) {
        // bf16 activations on the 256-tile path only (the caller checks), whose
        // epilogue it is; n is the output width, the weight has 2n interleaved
        // rows
        if constexpr (std::is_same<TX, uint16_t>::value) {
            if (!swiglu_shape_ok(n, k)) return hipErrorInvalidValue;
            return linear_impl<TX, YK, S2_ACT_SWIGLU>(x0, m0, x1, m1, w, bias, 2 * n, k, y0, y1,
                                                      stream, src);
        }
        return hipErrorInvalidValue;
    }
    if (act == S2_ACT_GELU)
        return linear_impl<TX, YK, S2_ACT_GELU>(x0, m0, x1, m1, w, bias, n, k, y0, y1, stream, src);
    return linear_impl<TX, YK, S2_ACT_NONE>(x0, m0, x1, m1, w, bias, n, k, y0, y1, stream, src);
}

template <typename TX>
static hipError_t linear_out(int y_kind, int act, const void* x0, int m0, const void* x1, int m1,
                             const uint16_t* w, const float* bias, int n, int k, void* y0,
                             void* y1, hipStream_t stream, SkSource src) {
    if (y_kind == 1)
        return linear_act<TX, 1>(act, x0, m0, x1, m1, w, bias, n, k, y0, y1, stream, src);
    if (y_kind == 2)
        return linear_act<TX, 2>(act, x0, m0, x1, m1, w, bias, n, k, y0, y1, stream, src);
    return linear_act<TX, 0>(act, x0, m0, x1, m1, w, bias, n, k, y0, y1, stream, src);
}

static hipError_t linear_dispatch(const void* x0, int m0, const void* x1, int m1, int x_kind,
                                  const uint16_t* w, const float* bias, int n, int k, int act,
                                  void* y0, void* y1, int y_kind, hipStream_t stream,
                                  SkSource src) {
    if (x_kind == 1)
        return linear_out<uint16_t>(y_kind, act, x0, m0, x1, m1, w, bias, n, k, y0, y1, stream, src);
    if (x_kind == 2)
        return linear_out<_Float16>(y_kind, act, x0, m0, x1, m1, w, bias, n, k, y0, y1, stream, src);
    return linear_out<float>(y_kind, act, x0, m0, x1, m1, w, bias, n, k, y0, y1, stream, src);
}

hipError_t launch_shared_linear(const void* x0, int m0, const void* x1, int m1, int x_kind,
                                const uint16_t* w, const float* bias, int n, int k, int act,
                                void* y0, void* y1, int y_kind, hipStream_t stream,
                                bool optional_split) {
    // (fp32 and fp16 activations can do without the scratch: they took the
    // 128-tile kernel, which has no split, until the 256-tile one converted them)
    return linear_dispatch(x0, m0, x1, m1, x_kind, w, bias, n, k, act, y0, y1, y_kind, stream,
                           optional_split || x_kind != 1 ? SkSource::kOptional : SkSource::kStream);
}

hipError_t launch_shared_linear_noalloc(const void* x0, int m0, const void* x1, int m1,
                                        int x_kind, const uint16_t* w, const float* bias, int n,
                                        int k, int act, void* y0, void* y1, int y_kind,
                                        hipStream_t stream) {
    return linear_dispatch(x0, m0, x1, m1, x_kind, w, bias, n, k, act, y0, y1, y_kind, stream,
                           SkSource::kStatic);
}

hipError_t launch_shared_linear_residual(const uint16_t* x0, int m0, const uint16_t* x1, int m1,
                                         const uint16_t* w, const float* bias, int n, int k,
                                         const LinearResidual& res, hipStream_t stream) {
    if (k % 64 != 0 || n % 8 != 0 || (long)256 * k * 2 > 0x7fffffffL ||
        (long)256 * n * 4 > 0x7fffffffL)
        return hipErrorInvalidValue;
    const int mv = (m0 + 7) / 8 * 8;
    const int ntiles = (n + 255) / 256;
    const int mtiles = (mv + m1 + 255) / 256;
    const long tiles = (long)mtiles * ntiles;
    if (tiles == 0) return hipSuccess;
    SkTail sk;
    hipError_t e = plan_sk_tail(tiles, k / 64, SkSource::kStream, stream, &sk);
    if (e != hipSuccess) return e;
    const long blocks = (long)sk.dp_tiles + sk.sk_groups;
    shared_linear_256_kernel<1, S2_ACT_NONE, 0, 1><<<(unsigned)blocks, 512, 0, stream>>>(
        x0, m0, x1, m1, w, bias, n, k, nullptr, nullptr, mv, mtiles, ntiles, sk, AwaQkvArgs{},
        res, LinearRows{});
    return hipGetLastError();
}

// One stream of bf16 rows on the 256-tile kernel with the epilogue ACT of
// LinearRows.
template <int YK, int ACT>
static hipError_t linear_rows(const uint16_t* x, int m, const uint16_t* w, const float* bias, int n,
                              int k, void* y, const LinearRows& lr, hipStream_t stream) {
    const long row = ACT == kActExp ? lr.pitch : n;   // output row pitch
    if (m <= 0 || n <= 0 || k % 64 != 0 || (YK && row % 8 != 0) || lr.ld % 8 != 0 ||
        (long)256 * std::max(k, lr.ld) * 2 > 0x7fffffffL ||
        256 * row * 4 > 0x7fffffffL)
        return hipErrorInvalidValue;
    const int mv = (m + 7) / 8 * 8;
    const int ntiles = (n + 255) / 256;
    const int mtiles = (mv + 255) / 256;
    SkTail sk;
    hipError_t e = plan_sk_tail((long)mtiles * ntiles, k / 64, SkSource::kStream, stream, &sk);
    if (e != hipSuccess) return e;
    const long blocks = (long)sk.dp_tiles + sk.sk_groups;
    shared_linear_256_kernel<YK, ACT><<<(unsigned)blocks, 512, 0, stream>>>(
        x, m, nullptr, 0, w, bias, n, k, y, nullptr, mv, mtiles, ntiles, sk, AwaQkvArgs{},
        LinearResidual{}, lr);
    return hipGetLastError();
}

hipError_t launch_linear_exp(const uint16_t* q, int m, const uint16_t* keys, int n, int k,
                             uint16_t* y, const LinearRows& lr, hipStream_t stream) {
    return linear_rows<1, kActExp>(keys, n, q, nullptr, m, k, y, lr, stream);
}

hipError_t launch_linear_row_scale(const uint16_t* x, int m, const uint16_t* w, const float* bias,
                                   int n, int k, uint16_t* y, const LinearRows& lr,
                                   hipStream_t stream) {
    return linear_rows<1, kActRowScale>(x, m, w, bias, n, k, y, lr, stream);
}

hipError_t launch_linear_gated(const uint16_t* x, int m, const uint16_t* w, int n, int k, float* y,
                               const LinearRows& lr, hipStream_t stream) {
    return linear_rows<0, S2_ACT_NONE>(x, m, w, nullptr, n, k, y, lr, stream);
}

hipError_t launch_awa_qkv(const s2_awa_plan& plan, const uint16_t* x_video, const uint16_t* x_text,
                          int k, const uint16_t* w, const float* bias, const float* norm,
                          const float2* rope, uint16_t* q, uint16_t* kk, uint16_t* vt,
                          hipStream_t stream) {
    const int d = plan.config.head_dim;
    const int inner = plan.config.heads * d;
    if ((d != 64 && d != 128) || inner % 256 != 0 || k % 64 != 0 ||
        (long)(plan.video_tokens + 1) * k * 2 > 0x7fffffffL ||
        (long)(plan.text_tokens + 1) * k * 2 > 0x7fffffffL)
        return hipErrorInvalidValue;
    const int n = 3 * inner;
    const int ntiles = n / 256;
    const int mtiles = (plan.qkv_rows + 255) / 256;
    const long tiles = (long)mtiles * ntiles;
    if (tiles == 0) return hipSuccess;
    SkTail sk;
    hipError_t e = plan_sk_tail(tiles, k / 64, SkSource::kStream, stream, &sk);
    if (e != hipSuccess) return e;
    AwaQkvArgs a;
    a.row_table = plan.d_qkv_rows;
    a.inner = inner;
    a.seg_total = plan.seg_total;
    a.seg_text = plan.seg_text;
    a.norm = norm;
    a.rope = rope;
    a.pairs = plan.config.rope_pairs_per_axis;
    a.eps = plan.config.epsilon;
    a.official_bf16 = plan.config.official_bf16_attention;
    a.q = q;
    a.k = kk;
    a.vt = vt;
    const long blocks = (long)sk.dp_tiles + sk.sk_groups;
    if (d == 128)
        shared_linear_256_kernel<1, S2_ACT_NONE, 128><<<(unsigned)blocks, 512, 0, stream>>>(
            x_video, plan.video_tokens, x_text, plan.text_tokens, w, bias, n, k, nullptr, nullptr,
            plan.qkv_text_row, mtiles, ntiles, sk, a, LinearResidual{}, LinearRows{});
    else
        shared_linear_256_kernel<1, S2_ACT_NONE, 64><<<(unsigned)blocks, 512, 0, stream>>>(
            x_video, plan.video_tokens, x_text, plan.text_tokens, w, bias, n, k, nullptr, nullptr,
            plan.qkv_text_row, mtiles, ntiles, sk, a, LinearResidual{}, LinearRows{});
    return hipGetLastError();
}

}  // namespace s2
