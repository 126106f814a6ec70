// Quantizer kernels: the fused Q8_0 activation quantizer (the engine caller's
// quantize_x, board/tp/tp_llama.cpp:330-352, with the contract's rounding,
// src/llm_kv260/q4_0.py:83-97) and a Q4_0 weight quantizer
// (src/llm_kv260/q4_0.py:100-121) for building matrices on the device.
//
// Both are element-wise over 32-element blocks. The activation quantizers
// give each block eight threads (one 16-byte load, four values each) and
// meet for the block's max through DPP: a launch of them is latency, and a
// thread that quantized a whole block alone spent ~250 instructions on it.
// The weight quantizer keeps one thread per block (weights are quantized
// once).
#include "kernels.h"
#include "q4_0_device.h"

namespace w4a8 {

namespace {

__device__ __forceinline__ void load_block(const float *src, float v[32]) {
    const float4 *p = reinterpret_cast<const float4 *>(src);
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        const float4 f = p[m];
        v[4 * m] = f.x; v[4 * m + 1] = f.y; v[4 * m + 2] = f.z; v[4 * m + 3] = f.w;
    }
}

// Q8_0 (q4_0.py:83-97) of values 4g .. 4g + 3 of a 32-element block, thread g
// (0..7) of an aligned group of eight, stored in block b of row `row` of the
// engine layout (int8[k] | float32[k/32]) or of ggml Q8_0 blocks: amax is the group's max (DPP quad_perm [1,0,3,2],
// [2,3,0,1], then row_half_mirror), so every thread computes the same d and
// inv as a thread holding the whole block.
template <int OUT>
__device__ __forceinline__ void quantize_store8(const float4 v, int row, int b, int g, int k, uint8_t *__restrict__ out) {
    const int nb = k >> 5;
    float amax = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
    amax = fmaxf(amax, dpp_mov<0xB1>(amax));
    amax = fmaxf(amax, dpp_mov<0x4E>(amax));
    amax = fmaxf(amax, dpp_mov<0x141>(amax));
    const float d = q8_scale(amax);
    const float inv = safe_recip(d);
    const uint32_t word = (uint32_t)(uint8_t)q8_round(v.x, inv) | ((uint32_t)(uint8_t)q8_round(v.y, inv) << 8) |
                          ((uint32_t)(uint8_t)q8_round(v.z, inv) << 16) | ((uint32_t)(uint8_t)q8_round(v.w, inv) << 24);
    const uint16_t dh = float_to_half_bits(d);
    if constexpr (OUT == X_ENGINE) {
        uint8_t *rowp = out + (size_t)row * (k + 4 * nb);
        reinterpret_cast<uint32_t *>(rowp + 32 * b)[g] = word;
        if (g == 0) reinterpret_cast<float *>(rowp + k)[b] = half_bits_to_float(dh);
    } else {
        uint16_t *dst = reinterpret_cast<uint16_t *>(out + ((size_t)row * nb + b) * Q8_0_BYTES);
        if (g == 0) dst[0] = dh;
        dst[1 + 2 * g] = (uint16_t)(word & 0xFFFFu);
        dst[2 + 2 * g] = (uint16_t)(word >> 16);
    }
}

template <int OUT>
__global__ __launch_bounds__(256) void quantize_q8_0_kernel(const float *__restrict__ x, int k, int m,
                                                            uint8_t *__restrict__ out) {
    const int nb = k >> 5;
    const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= (long)nb * m * 8) return;           // whole groups of eight leave together
    const long blk = gid >> 3;
    const int g = (int)(gid & 7);
    const int row = (int)(blk / nb), b = (int)(blk - (long)row * nb);
    const float4 v = reinterpret_cast<const float4 *>(x + (size_t)row * k + 32 * b)[g];
    quantize_store8<OUT>(v, row, b, g, k, out);
}

// act = silu(gate) * up (tp_llama.cpp:612-619) of m rows gate | up
// (float32[2k] each, the gate|up GEMV's output), quantized to the engine layout.
__global__ __launch_bounds__(256) void silu_mul_q8_0_kernel(const float *__restrict__ gate_up, int k, int m,
                                                            uint8_t *__restrict__ out) {
    const int nb = k >> 5;
    const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= (long)nb * m * 8) return;           // whole groups of eight leave together
    const long blk = gid >> 3;
    const int t = (int)(gid & 7);
    const int row = (int)(blk / nb), b = (int)(blk - (long)row * nb);
    const float *src = gate_up + (size_t)row * 2 * k + 32 * b;
    const float4 g = reinterpret_cast<const float4 *>(src)[t];
    const float4 u = reinterpret_cast<const float4 *>(src + k)[t];
    const float4 v = make_float4(silu_mul(g.x, u.x), silu_mul(g.y, u.y), silu_mul(g.z, u.z), silu_mul(g.w, u.w));
    quantize_store8<X_ENGINE>(v, row, b, t, k, out);
}

// h = rmsnorm(x) * norm_w (tp_llama.cpp:557-569) of m rows of float32[k],
// quantized to the engine layout: one workgroup per row (the sum of squares
// runs over the whole row). Latency: thread t holds the row's float4s t + 256 j
// (x and the norm weight, all NV of each in flight at once), so x is read once,
// and eight consecutive threads hold a block, as quantize_store8 takes it.
template <int NV>
__global__ __launch_bounds__(256) void rmsnorm_q8_0_kernel(const float *__restrict__ x, const float *__restrict__ w,
                                                           float eps, int k, uint8_t *__restrict__ out) {
    __shared__ double part[RMS_PART(4)];
    const int row = blockIdx.x, n4 = k >> 2;
    const float *xr = x + (size_t)row * k;
    float4 xv[NV], wv[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int i = threadIdx.x + 256 * j;       // n4 % 64 == 0: waves are in or out as a whole
        const int c = i < n4 ? i : 0;
        xv[j] = reinterpret_cast<const float4 *>(xr)[c];
        wv[j] = reinterpret_cast<const float4 *>(w)[c];
    }
    double p = 0.0;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        if (threadIdx.x + 256 * j < n4) {
            const double a = xv[j].x, b = xv[j].y, c = xv[j].z, d = xv[j].w;
            p = fma(a, a, p);
            p = fma(b, b, p);
            p = fma(c, c, p);
            p = fma(d, d, p);
        }
    }
    const float sc = rms_scale_block(p, k, eps, 4, part, [&](int i) { return xr[i]; });
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int i = threadIdx.x + 256 * j;
        if (i < n4) {
            const float4 v = make_float4((xv[j].x * sc) * wv[j].x, (xv[j].y * sc) * wv[j].y, (xv[j].z * sc) * wv[j].z,
                                         (xv[j].w * sc) * wv[j].w);
            quantize_store8<X_ENGINE>(v, row, i >> 3, i & 7, k, out);
        }
    }
}

__global__ __launch_bounds__(256) void quantize_q4_0_kernel(const float *__restrict__ w, int rows, int k,
                                                            uint8_t *__restrict__ out) {
    const int nb = k >> 5;
    const long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= (long)nb * rows) return;
    float v[32];
    load_block(w + gid * 32, v);   // rows are contiguous: block gid starts at float 32 * gid
    // The signed element of largest magnitude, first index on ties.
    float extreme = v[0], amax = fabsf(v[0]);
#pragma unroll
    for (int e = 1; e < 32; ++e) {
        const float a = fabsf(v[e]);
        if (a > amax) { amax = a; extreme = v[e]; }
    }
    const float d = extreme / -8.0f;
    const float inv = safe_recip(d);
    uint32_t nib[32];
#pragma unroll
    for (int e = 0; e < 32; ++e) {
        const float s = v[e] * inv;
        const float u = s + 8.5f;
        const int n = (int)truncf(u);   // u >= 0.5 for every finite block; clamp keeps nibbles 4-bit
        nib[e] = (uint32_t)(n > 15 ? 15 : (n < 0 ? 0 : n));
    }
    uint16_t *dst = reinterpret_cast<uint16_t *>(out + gid * Q4_0_BYTES);
    dst[0] = float_to_half_bits(d);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const uint32_t b0 = nib[2 * j] | (nib[2 * j + 16] << 4);
        const uint32_t b1 = nib[2 * j + 1] | (nib[2 * j + 17] << 4);
        dst[1 + j] = (uint16_t)(b0 | (b1 << 8));
    }
}

}  // namespace

hipError_t launch_quantize_q8_0(const float *x, int k, int m, uint8_t *out, XFormat out_fmt, hipStream_t stream) {
    const long blocks = (long)(k / 32) * m;
    if (blocks == 0) return hipSuccess;
    const long grid = (8 * blocks + 255) / 256;
    if (grid > 0x7fffffffL) return hipErrorInvalidValue;
    if (out_fmt == X_ENGINE)
        hipLaunchKernelGGL(quantize_q8_0_kernel<X_ENGINE>, dim3((unsigned)grid), dim3(256), 0, stream, x, k, m, out);
    else if (out_fmt == X_Q8_0)
        hipLaunchKernelGGL(quantize_q8_0_kernel<X_Q8_0>, dim3((unsigned)grid), dim3(256), 0, stream, x, k, m, out);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_silu_mul_q8_0(const float *gate_up, int k, int m, uint8_t *out, hipStream_t stream) {
    const long blocks = (long)(k / 32) * m;
    if (blocks == 0) return hipSuccess;
    const long grid = (8 * blocks + 255) / 256;
    if (grid > 0x7fffffffL) return hipErrorInvalidValue;
    hipLaunchKernelGGL(silu_mul_q8_0_kernel, dim3((unsigned)grid), dim3(256), 0, stream, gate_up, k, m, out);
    return hipGetLastError();
}

hipError_t launch_rmsnorm_q8_0(const float *x, const float *w, float eps, int k, int m, uint8_t *out,
                               hipStream_t stream) {
    if (m <= 0) return hipSuccess;
    // The float4s a thread holds: k / 1024, rounded up to a power of two.
    auto *kernel = k <= 1024   ? &rmsnorm_q8_0_kernel<1>
                   : k <= 2048 ? &rmsnorm_q8_0_kernel<2>
                   : k <= 4096 ? &rmsnorm_q8_0_kernel<4>
                   : k <= 8192 ? &rmsnorm_q8_0_kernel<8>
                               : &rmsnorm_q8_0_kernel<16>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)m), dim3(256), 0, stream, x, w, eps, k, out);
    return hipGetLastError();
}

hipError_t launch_quantize_q4_0(const float *w, int rows, int k, uint8_t *out, hipStream_t stream) {
    const long blocks = (long)(k / 32) * rows;
    if (blocks == 0) return hipSuccess;
    const long grid = (blocks + 255) / 256;
    if (grid > 0x7fffffffL) return hipErrorInvalidValue;
    hipLaunchKernelGGL(quantize_q4_0_kernel, dim3((unsigned)grid), dim3(256), 0, stream, w, rows, k, out);
    return hipGetLastError();
}

}  // namespace w4a8
