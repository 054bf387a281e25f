// silu(gate) * up over the library product of a gate||up weight, and its gradient: the middle of LlamaMLP where
// the product itself is the library's (prompts that vrl_int4_gemm_bf16 is not the faster form for), and in the
// backward of every training replay (policy.py:419-424).  Bound by memory: each value is read once and written once, 16 bytes per lane, where the
// separate tensor operations passed over halves and temporaries (1664 x 5632: 10.6 us, 5.3 TB/s, against
// 14.6 + 11.8; its gradient 15.8 us, 5.9 TB/s, against 15.9 + 17.9 + 9.9 + 11.8).  All arithmetic in fp32, one
// rounding per result.
#include "host_checks.hpp"

namespace {

__device__ __forceinline__ void unpack8(const u32x4_t &v, float f[8]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f[2 * i] = bf16_bits_to_f32(v[i] & 0xFFFFu);
        f[2 * i + 1] = bf16_bits_to_f32(v[i] >> 16);
    }
}

__device__ __forceinline__ u32x4_t pack8(const float f[8]) {
    return u32x4_t{pack_bf16_rne(f[0], f[1]), pack_bf16_rne(f[2], f[3]), pack_bf16_rne(f[4], f[5]),
                   pack_bf16_rne(f[6], f[7])};
}

// one thread: eight neighbouring columns of one row; words: 16-byte words of a row of y
__global__ __launch_bounds__(256) void silu_mul_kernel(const u32x4_t *__restrict__ gate_up, u32x4_t *__restrict__ y,
                                                       uint32_t words, uint32_t total) {
    const uint32_t idx = blockIdx.x * 256u + threadIdx.x;
    if (idx >= total) return;
    const uint32_t row = idx / words;
    const size_t at = (size_t)idx + (size_t)row * words;   // 2 * words per row of gate||up
    float g[8], u[8];
    unpack8(gate_up[at], g);
    unpack8(gate_up[at + words], u);
#pragma unroll
    for (int i = 0; i < 8; ++i) g[i] = g[i] / (1.0f + __expf(-g[i])) * u[i];
    y[idx] = pack8(g);
}

__global__ __launch_bounds__(256) void silu_mul_backward_kernel(const u32x4_t *__restrict__ gate_up,
                                                                const u32x4_t *__restrict__ grad,
                                                                u32x4_t *__restrict__ out, uint32_t words,
                                                                uint32_t total) {
    const uint32_t idx = blockIdx.x * 256u + threadIdx.x;
    if (idx >= total) return;
    const uint32_t row = idx / words;
    const size_t at = (size_t)idx + (size_t)row * words;
    float g[8], u[8], d[8];
    unpack8(gate_up[at], g);
    unpack8(gate_up[at + words], u);
    unpack8(grad[idx], d);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float s = 1.0f / (1.0f + __expf(-g[i]));
        const float du = d[i] * (g[i] * s);
        g[i] = d[i] * u[i] * (s * (1.0f + g[i] * (1.0f - s)));
        u[i] = du;
    }
    out[at] = pack8(g);
    out[at + words] = pack8(u);
}

int silu_mul_check(const void *a, const void *b, const void *c, long M, long inter) {
    if (!a || !b || !c) return VRL_INT4_ENULL;
    if (M < 1 || inter < 8 || inter % 8 != 0 || M * inter >= (1L << 31)) return VRL_INT4_ESHAPE;
    if (!aligned16(a) || !aligned16(b) || !aligned16(c)) return VRL_INT4_EALIGN;
    return VRL_INT4_OK;
}

}  // namespace

extern "C" {

int vrl_silu_mul_bf16(const void *gate_up, void *y, int M, int inter, void *hip_stream) {
    const int rc = silu_mul_check(gate_up, y, y, M, inter);
    if (rc != VRL_INT4_OK) return rc;
    const uint32_t words = inter / 8, total = (uint32_t)M * words;
    return vrl_launch(&silu_mul_kernel, dim3((total + 255) / 256), dim3(256), 0, reinterpret_cast<hipStream_t>(hip_stream),
                      static_cast<const u32x4_t *>(gate_up), static_cast<u32x4_t *>(y), words, total);
}

int vrl_silu_mul_backward_bf16(const void *gate_up, const void *grad_y, void *grad_gate_up, int M, int inter,
                               void *hip_stream) {
    const int rc = silu_mul_check(gate_up, grad_y, grad_gate_up, M, inter);
    if (rc != VRL_INT4_OK) return rc;
    const uint32_t words = inter / 8, total = (uint32_t)M * words;
    return vrl_launch(&silu_mul_backward_kernel, dim3((total + 255) / 256), dim3(256), 0,
                      reinterpret_cast<hipStream_t>(hip_stream), static_cast<const u32x4_t *>(gate_up),
                      static_cast<const u32x4_t *>(grad_y), static_cast<u32x4_t *>(grad_gate_up), words, total);
}

}  // extern "C"
