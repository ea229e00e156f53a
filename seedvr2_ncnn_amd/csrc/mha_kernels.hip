// gfx950 kernels of the VAE's VAEChunkedMHA (src/seedvr2/vae_chunked_mha.cpp:223-281):
// ncnn MultiHeadAttention over one blob, i.e. self attention of seq tokens of
// width qdim.
//
// The VAE attends with one head of width 512 over every pixel of a latent
// frame (14,400 tokens at 720p).  At that head width a flash kernel holds
// few query rows per wave (a 16-row x 512 fp32 output tile is 128 registers
// per lane) and its K/V fragment reads from LDS outgrow the matrix-core
// time.  With 288 GB of HBM the score matrix fits many times over, so the
// forward runs through the SharedLinear GEMM instead: the projections, P =
// exp(Q K^T - reference) in bf16 with the fp32 row sums from the same epilogue,
// O = P V scaled by them, and the output projection.  Short sequences, and
// heads whose scores no reference covers, take S = Q K^T in fp32 and a row
// softmax into bf16 P instead.  This file holds the kernels between the GEMMs.
#include <math.h>

#include "mha_kernels.h"
#include "s2_device.h"

namespace s2 {
namespace {

// the first `valid` of `total` elements of x (element type KIND), as bf16,
// and zeros for the rest; both are multiples of 8, which a thread moves
// (one element a thread took 19 us for 14400 rows of 512)
template <int KIND>
__global__ __launch_bounds__(256) void mha_stage_kernel(const void* __restrict__ x, long valid,
                                                        long total, uint16_t* __restrict__ xp) {
    const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 8;
    if (i >= total) return;
    uint4 out = make_uint4(0u, 0u, 0u, 0u);
    if (i < valid) {
        if (KIND == 1) {
            out = *reinterpret_cast<const uint4*>((const uint16_t*)x + i);
        } else {
            float v[8];
            if (KIND == 2) {
                const uint4 u = *reinterpret_cast<const uint4*>((const uint16_t*)x + i);
                const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    v[e] = (float)__builtin_bit_cast(_Float16, (uint16_t)(w[e >> 1] >> (16 * (e & 1))));
            } else {
                load8((const float*)x + i, v);
            }
            out = cvt8_bf16(v);
        }
    }
    *reinterpret_cast<uint4*>(xp + i) = out;
}

// ---- the exponentials' reference -------------------------------------------
//
// The scores of row r are bounded by B_r = |q_r| max_j |k_j| (log2 domain,
// with 2^-6 of slack for the products' rounding).  Their exponentials are
// taken relative to c_r = max(0, B_r - 80): no value exceeds 2^80, and a
// row's largest one is at least 2^-70 if its score lies within 150 of B_r,
// with 2^-26 of it still 30 powers of two above the smallest normal number.  A
// row's own key shows that: the reference is good for a head when q_r k_r >=
// B_r - 150 for every row.  The product with V is divided by the row's sum
// afterwards, so V has to leave it room: with every |v| at most 2^24 (and 2^21
// keys) its sums stay below 2^125, and with one of at least 2^-30 in every run
// of d values of V^T (or none but zeros) no channel's sums leave the normal
// numbers.  Otherwise (also for non-finite operands) `general` sends the head
// through fp32 scores and the softmax pass, whose weights are normalised
// before V meets them.  (With no look at V, values of 1e30 came out as
// infinity where every score was near its bound; it costs 1.5 us of 490 for
// 14,400 tokens.)
constexpr float kRefBelow = 80.f, kRefSpan = 150.f;
constexpr uint32_t kValueMax = 0x4b800000u, kValueMin = 0x30800000u;   // 2^24, 2^-30

// |q_r|^2, |k_r|^2 (NaN where V is out of range) and q_r k_r, one wave a row
// (row pitch ld); clears the flag.  The wave also looks at run r of d values of
// V^T [d][lp], and at run rows + r, of the padding, where there is one.
__global__ __launch_bounds__(256) void mha_norms_kernel(const uint16_t* __restrict__ q,
                                                        const uint16_t* __restrict__ k, int ld,
                                                        const uint16_t* __restrict__ vt, int lp,
                                                        int rows, int d, int pitch,
                                                        float* __restrict__ stats,
                                                        int* __restrict__ general) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *general = 0;
    const int r = (int)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (r >= rows) return;
    float qq = 0.f, kk = 0.f, qk = 0.f;
    // magnitudes as fp32 bits: they order like the values, infinity and NaN on top
    uint32_t vm = 0u;
    auto magnitudes = [&](uint4 u) {
        const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int e = 0; e < 4; ++e)
            vm = max(vm, max((w[e] << 16) & 0x7fff0000u, w[e] & 0x7fff0000u));
    };
    for (int c = lane * 8; c < d; c += 512) {
        const uint4 u = *reinterpret_cast<const uint4*>(vt + (long)r * d + c);
        float a[8], b[8];
        load8(q + (long)r * ld + c, a);
        load8(k + (long)r * ld + c, b);
        magnitudes(u);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            qq = fmaf(a[e], a[e], qq);
            kk = fmaf(b[e], b[e], kk);
            qk = fmaf(a[e], b[e], qk);
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        qq += __shfl_xor(qq, off);
        kk += __shfl_xor(kk, off);
        qk += __shfl_xor(qk, off);
        vm = max(vm, (uint32_t)__shfl_xor((int)vm, off));
    }
    bool fits = vm <= kValueMax && (vm == 0u || vm >= kValueMin);
    if (rows + r < lp) {   // lp < rows + 64 <= 2 rows
        vm = 0u;
        for (int c = lane * 8; c < d; c += 512)
            magnitudes(*reinterpret_cast<const uint4*>(vt + (long)(rows + r) * d + c));
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) vm = max(vm, (uint32_t)__shfl_xor((int)vm, off));
        fits = fits && vm <= kValueMax && (vm == 0u || vm >= kValueMin);
    }
    if (lane == 0) {
        stats[r] = qq;
        stats[pitch + r] = fits ? kk : __uint_as_float(0x7fc00000u);
        stats[2 * pitch + r] = qk;
    }
}

// c_r of every row (0 in the padding up to `pitch`) and the head's `general`
// flag: a block takes 256 rows, and finds the largest |k_j| itself (one block
// for all rows took 12-14 us for 14,400 of them)
__global__ __launch_bounds__(256) void mha_reference_kernel(const float* __restrict__ stats,
                                                            int rows, int pitch,
                                                            float* __restrict__ ref,
                                                            int* __restrict__ general) {
    constexpr float kLog2e = 1.4426950408889634f;
    __shared__ float red[4];
    const int t = threadIdx.x;
    const int r = blockIdx.x * 256 + t;
    // (statistics past `rows` are read and not used; pitch % 256 == 0)
    const float qq = stats[r], own = stats[2 * pitch + r] * kLog2e;
    float m = 0.f;
    int bad = 0;
#pragma unroll 8
    for (int i = t * 4; i < rows; i += 1024) {
        const float4 kk = *reinterpret_cast<const float4*>(stats + pitch + i);
        const float v[4] = {kk.x, kk.y, kk.z, kk.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (i + e >= rows) continue;
            bad |= !(v[e] <= 3.0e38f);   // also for NaN (mha_norms_kernel's too)
            m = fmaxf(m, v[e]);
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    if ((t & 63) == 0) red[t >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float b = sqrtf(qq) * sqrtf(m) * (kLog2e * (1.f + 0.015625f));
    const bool in = r < rows;
    bad |= in && !(own >= b - kRefSpan);
    ref[r] = in ? fmaxf(b - kRefBelow, 0.f) : 0.f;
    if (__any(bad) && (t & 63) == 0)
        __hip_atomic_store(general, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// 1 / (sum of a row's exponentials over the column parts), or 1 when the
// probabilities are already normalised; a block takes 64 rows, its waves
// every fourth part
__global__ __launch_bounds__(256) void mha_row_scale_kernel(const float* __restrict__ sums, int parts,
                                                            int pitch, const int* __restrict__ general,
                                                            float* __restrict__ scale, int rows) {
    __shared__ float red[4][64];
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int r = blockIdx.x * 64 + l;   // pitch is a multiple of 64
    float s = 0.f;
    if (!*general) {
#pragma unroll 8
        for (int i = w; i < parts; i += 4) s += sums[(long)i * pitch + r];
    }
    red[w][l] = s;
    __syncthreads();
    if (w == 0) {
        s = (red[0][l] + red[1][l]) + (red[2][l] + red[3][l]);
        scale[r] = r < rows && !*general ? 1.f / s : 1.f;
    }
}

// weights: fp32 -> bf16, times `scale`
__global__ __launch_bounds__(256) void mha_weight_kernel(const float* __restrict__ w, long n,
                                                         float scale, uint16_t* __restrict__ out) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[i] = f32_to_bf16(w[i] * scale);
}

__global__ __launch_bounds__(256) void mha_bias_kernel(const float* __restrict__ b, int n,
                                                       float scale, float* __restrict__ out) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[i] = b[i] * scale;
}

// One block per row of S [rows][ld_s] (fp32, scores already scaled):
// P[r][c] = exp(S - max) / sum for c < cols, 0 for cols <= c < ld_p.  The
// row is read once from HBM for the running (max, sum) and once more, from
// L2, to write P.
__global__ __launch_bounds__(256) void mha_softmax_kernel(const float* __restrict__ s, long ld_s,
                                                          int cols, int ld_p,
                                                          uint16_t* __restrict__ p,
                                                          const int* __restrict__ gate) {
    constexpr float kLog2e = 1.4426950408889634f;
    if (gate && !*gate) return;
    __shared__ float red_m[4], red_s[4];
    const float* row = s + (long)blockIdx.x * ld_s;
    uint16_t* out = p + (long)blockIdx.x * ld_p;
    const int t = threadIdx.x;
    float m = -INFINITY, sum = 0.f;
    for (int c = t; c < cols; c += 256) {
        const float v = row[c];
        if (v > m) {
            sum = sum * __builtin_amdgcn_exp2f((m - v) * kLog2e) + 1.f;
            m = v;
        } else {
            sum += __builtin_amdgcn_exp2f((v - m) * kLog2e);
        }
    }
    // combine (max, sum) over the wave, then over the four waves
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        const float om = __shfl_xor(m, off), os = __shfl_xor(sum, off);
        const float nm = fmaxf(m, om);
        sum = (m == -INFINITY ? 0.f : sum * __builtin_amdgcn_exp2f((m - nm) * kLog2e)) +
              (om == -INFINITY ? 0.f : os * __builtin_amdgcn_exp2f((om - nm) * kLog2e));
        m = nm;
    }
    if ((t & 63) == 0) {
        red_m[t >> 6] = m;
        red_s[t >> 6] = sum;
    }
    __syncthreads();
    m = fmaxf(fmaxf(red_m[0], red_m[1]), fmaxf(red_m[2], red_m[3]));
    sum = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w)
        if (red_m[w] != -INFINITY) sum += red_s[w] * __builtin_amdgcn_exp2f((red_m[w] - m) * kLog2e);
    const float inv = 1.f / sum;
    for (int c = t; c < ld_p; c += 256)
        out[c] = c < cols ? f32_to_bf16(__builtin_amdgcn_exp2f((row[c] - m) * kLog2e) * inv)
                          : (uint16_t)0;
}

// The same softmax with the row held in registers: thread t owns the float4
// groups t, t + 256, ... (NV of them, so rows up to NV * 1024 columns).  All
// loads are issued at once and the row is read from HBM once.  VEC: the row
// stride and the row start allow 16-byte loads.
template <int NV, bool VEC>
__global__ __launch_bounds__(256) void mha_softmax_reg_kernel(const float* __restrict__ s,
                                                              long ld_s, int cols, int ld_p,
                                                              uint16_t* __restrict__ p,
                                                              const int* __restrict__ gate) {
    constexpr float kLog2e = 1.4426950408889634f;
    if (gate && !*gate) return;
    __shared__ float red[4];
    const float* row = s + (long)blockIdx.x * ld_s;
    uint16_t* out = p + (long)blockIdx.x * ld_p;
    const int t = threadIdx.x;
    float v[NV][4];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = (i * 256 + t) * 4;
        if (VEC && c + 3 < cols) {
            const float4 f = *reinterpret_cast<const float4*>(row + c);
            v[i][0] = f.x, v[i][1] = f.y, v[i][2] = f.z, v[i][3] = f.w;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[i][e] = c + e < cols ? row[c + e] : -INFINITY;
        }
    }
    float m = -INFINITY;
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) m = fmaxf(m, v[i][e]);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    if ((t & 63) == 0) red[t >> 6] = m;
    __syncthreads();
    m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    __syncthreads();   // red is reused for the sums
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[i][e] = __builtin_amdgcn_exp2f((v[i][e] - m) * kLog2e);   // -inf -> 0
            sum += v[i][e];
        }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off);
    if ((t & 63) == 0) red[t >> 6] = sum;
    __syncthreads();
    const float inv = 1.f / ((red[0] + red[1]) + (red[2] + red[3]));
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = (i * 256 + t) * 4;
        if (c >= ld_p) continue;
        // columns past `cols` hold exp(-inf) = 0; ld_p is a multiple of 4
        *reinterpret_cast<uint2*>(out + c) =
            make_uint2(pack2_bf16_rne(v[i][0] * inv, v[i][1] * inv),
                       pack2_bf16_rne(v[i][2] * inv, v[i][3] * inv));
    }
}

// head h's output [rows][d] (bf16) into columns [h*d, (h+1)*d) of O [rows][embed]
__global__ __launch_bounds__(256) void mha_interleave_kernel(const uint16_t* __restrict__ oh,
                                                             int rows, int d, int embed, int h,
                                                             uint16_t* __restrict__ o) {
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= (long)rows * d) return;
    const long r = i / d;
    o[r * embed + (long)h * d + (i - r * d)] = oh[i];
}

unsigned blocks(long n) { return (unsigned)((n + 255) / 256); }

}  // namespace

hipError_t launch_mha_stage(const void* x, int kind, int rows, int rows_padded, int qdim,
                            uint16_t* xp, hipStream_t stream) {
    const long valid = (long)rows * qdim, total = (long)rows_padded * qdim;   // qdim % 8 == 0
    if (total <= 0) return hipSuccess;
    if (kind == 1)
        mha_stage_kernel<1><<<blocks(total / 8), 256, 0, stream>>>(x, valid, total, xp);
    else if (kind == 2)
        mha_stage_kernel<2><<<blocks(total / 8), 256, 0, stream>>>(x, valid, total, xp);
    else
        mha_stage_kernel<0><<<blocks(total / 8), 256, 0, stream>>>(x, valid, total, xp);
    return hipGetLastError();
}

hipError_t launch_mha_reference(const uint16_t* q, const uint16_t* k, int ld, const uint16_t* vt,
                                int lp, int rows, int d, int pitch, float* stats, float* ref,
                                int* general, hipStream_t stream) {
    mha_norms_kernel<<<(unsigned)((rows + 3) / 4), 256, 0, stream>>>(q, k, ld, vt, lp, rows, d,
                                                                     pitch, stats, general);
    mha_reference_kernel<<<(unsigned)(pitch / 256), 256, 0, stream>>>(stats, rows, pitch, ref, general);
    return hipGetLastError();
}

hipError_t launch_mha_row_scale(const float* sums, int parts, int pitch, const int* general,
                                float* scale, int rows, hipStream_t stream) {
    mha_row_scale_kernel<<<(unsigned)(pitch / 64), 256, 0, stream>>>(sums, parts, pitch, general,
                                                                     scale, rows);
    return hipGetLastError();
}

hipError_t launch_mha_weight(const float* w, long n, float scale, uint16_t* out,
                             hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    mha_weight_kernel<<<blocks(n), 256, 0, stream>>>(w, n, scale, out);
    return hipGetLastError();
}

hipError_t launch_mha_bias(const float* b, int n, float scale, float* out, hipStream_t stream) {
    if (n <= 0) return hipSuccess;
    mha_bias_kernel<<<blocks(n), 256, 0, stream>>>(b, n, scale, out);
    return hipGetLastError();
}

template <int NV>
static void softmax_reg(const float* s, long ld_s, int rows, int cols, int ld_p, uint16_t* p,
                        const int* gate, hipStream_t stream) {
    if (ld_s % 4 == 0 && ((uintptr_t)s % 16) == 0)
        mha_softmax_reg_kernel<NV, true>
            <<<(unsigned)rows, 256, 0, stream>>>(s, ld_s, cols, ld_p, p, gate);
    else
        mha_softmax_reg_kernel<NV, false>
            <<<(unsigned)rows, 256, 0, stream>>>(s, ld_s, cols, ld_p, p, gate);
}

hipError_t launch_mha_softmax(const float* s, long ld_s, int rows, int cols, int ld_p,
                              uint16_t* p, const int* gate, hipStream_t stream) {
    if (rows <= 0) return hipSuccess;
    // rows of up to 16,384 columns live in registers (up to 64 floats per
    // thread); longer rows take the streaming kernel
    const int groups = (ld_p + 1023) / 1024;   // float4 groups per thread
    if (ld_p % 4 != 0 || groups > 16)
        mha_softmax_kernel<<<(unsigned)rows, 256, 0, stream>>>(s, ld_s, cols, ld_p, p, gate);
    else if (groups <= 2)
        softmax_reg<2>(s, ld_s, rows, cols, ld_p, p, gate, stream);
    else if (groups <= 4)
        softmax_reg<4>(s, ld_s, rows, cols, ld_p, p, gate, stream);
    else if (groups <= 8)
        softmax_reg<8>(s, ld_s, rows, cols, ld_p, p, gate, stream);
    else
        softmax_reg<16>(s, ld_s, rows, cols, ld_p, p, gate, stream);
    return hipGetLastError();
}

hipError_t launch_mha_interleave(const uint16_t* oh, int rows, int d, int embed, int h,
                                 uint16_t* o, hipStream_t stream) {
    const long n = (long)rows * d;
    if (n <= 0) return hipSuccess;
    mha_interleave_kernel<<<blocks(n), 256, 0, stream>>>(oh, rows, d, embed, h, o);
    return hipGetLastError();
}

}  // namespace s2
