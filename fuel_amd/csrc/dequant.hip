// Dequantize blocks to f32 (DynQuantizedStorage::dequantize) or f16
// (dequantize_f16), bit-exact with to_float: Q8_0 k_quants.rs:611-627,
// Q4K :1595-1622, Q6K :2158-2189.  Built with -ffp-contract=off so
// d1*q - m1 rounds twice, as in the reference.
#include "common.hpp"
#include "kernels.hpp"

namespace frq {

// f16 bits of f: the hardware conversion rounds to nearest even (the mode
// kernels start in, which nothing here changes); NaN takes the integer form.
__device__ __forceinline__ uint32_t half_bits(float f) {
    return f == f ? (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)f) : (uint32_t)f32_to_f16_rne(f);
}

template <bool F16>
__device__ __forceinline__ void store4(void* y, size_t idx, float a, float b, float c, float d) {
    if constexpr (F16) {
        reinterpret_cast<uint2*>(y)[idx / 4] =
            uint2{half_bits(a) | (half_bits(b) << 16), half_bits(c) | (half_bits(d) << 16)};
    } else {
        reinterpret_cast<float4*>(y)[idx / 4] = make_float4(a, b, c, d);
    }
}

// Eight values: two 8-byte stores of f16, two 16-byte ones of f32.  (The entry
// points ask for 4-byte aligned f32 outputs and any f16 ones: the stores rely on
// the unaligned global access that common.hpp states.)
template <bool F16>
__device__ __forceinline__ void store8(void* y, size_t idx, const float (&v)[8]) {
    if constexpr (F16) {
        uint32_t h[4];
#pragma unroll
        for (int i = 0; i < 4; i++) h[i] = half_bits(v[2 * i]) | (half_bits(v[2 * i + 1]) << 16);
        reinterpret_cast<uint2*>(y)[idx / 4] = uint2{h[0], h[1]};
        reinterpret_cast<uint2*>(y)[idx / 4 + 1] = uint2{h[2], h[3]};
    } else {
        reinterpret_cast<float4*>(y)[idx / 4] = make_float4(v[0], v[1], v[2], v[3]);
        reinterpret_cast<float4*>(y)[idx / 4 + 1] = make_float4(v[4], v[5], v[6], v[7]);
    }
}

// Memory bound: eight elements a lane, eight superblocks a workgroup (one
// superblock per 64-lane workgroup was bound by launching the workgroups:
// 49 us for 11008 x 4096 to f16, 24.7 us now).
constexpr int DQ_WG = 256;

// Lane t of a superblock's 32 writes elements 8t..8t+7.
template <bool F16>
__global__ __launch_bounds__(DQ_WG) void dequant_q4k_kernel(const uint8_t* __restrict__ w, size_t nblocks, void* y) {
    const size_t ib = (size_t)blockIdx.x * (DQ_WG / 32) + (threadIdx.x >> 5);
    if (ib >= nblocks) return;
    const uint8_t* blk = w + ib * Q4K_BYTES;
    const int e = 8 * (threadIdx.x & 31);   // element within the superblock
    const int c = e >> 6, hi = (e >> 5) & 1, l = e & 31;
    const int j = 2 * c + hi;               // sub-block
    const uint8_t* sc = blk + 4;
    int s, m;
    if (j < 4) {
        s = sc[j] & 63;
        m = sc[j + 4] & 63;
    } else {
        s = (sc[j + 4] & 0xF) | ((sc[j - 4] >> 6) << 4);
        m = (sc[j + 4] >> 4) | ((sc[j] >> 6) << 4);
    }
    const float d = f16_to_f32(load_u16(blk)), dmin = f16_to_f32(load_u16(blk + 2));
    const float d1 = d * (float)s, m1 = dmin * (float)m;
    const uint32_t* q = reinterpret_cast<const uint32_t*>(blk + 16 + 32 * c + l);
    const uint32_t n[2] = {(hi ? q[0] >> 4 : q[0]) & 0x0f0f0f0fu, (hi ? q[1] >> 4 : q[1]) & 0x0f0f0f0fu};
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = d1 * (float)((n[i >> 2] >> (8 * (i & 3))) & 0xffu) - m1;
    store8<F16>(y, ib * QK_K + e, v);
}

template <bool F16>
__global__ __launch_bounds__(DQ_WG) void dequant_q6k_kernel(const uint8_t* __restrict__ w, size_t nblocks, void* y) {
    const size_t ib = (size_t)blockIdx.x * (DQ_WG / 32) + (threadIdx.x >> 5);
    if (ib >= nblocks) return;
    const uint8_t* blk = w + ib * Q6K_BYTES;
    const int e = 8 * (threadIdx.x & 31);
    const int hh = e >> 7, r = e & 127, qd = r >> 5, l = r & 31;
    const float d = f16_to_f32(load_u16(blk + 208));
    const int8_t scv = (int8_t)blk[192 + 8 * hh + (l >> 4) + 2 * qd];
    const uint8_t* ql = blk + 64 * hh + 32 * (qd & 1) + l;
    const uint8_t* qh = blk + 128 + 32 * hh + l;
    float v[8];
#pragma unroll
    for (int i = 0; i < 4; i++) {  // (210-byte blocks: 2-byte aligned)
        const uint32_t lo2 = load_u16(ql + 2 * i), hi2 = load_u16(qh + 2 * i);
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int lb = (int)((lo2 >> (8 * t)) & 0xffu), hb = (int)((hi2 >> (8 * t)) & 0xffu);
            const int q = (((qd >> 1) ? lb >> 4 : lb & 0xF) | (((hb >> (2 * qd)) & 3) << 4)) - 32;
            v[2 * i + t] = d * (float)scv * (float)q;
        }
    }
    store8<F16>(y, ib * QK_K + e, v);
}

// Eight 32-element blocks per wavefront.
template <bool F16>
__global__ __launch_bounds__(DQ_WG) void dequant_q8_0_kernel(const uint8_t* __restrict__ w, size_t nblocks,
                                                             void* y) {
    const size_t ib = (size_t)blockIdx.x * (DQ_WG / 8) + (threadIdx.x >> 3);
    if (ib >= nblocks) return;
    const int t = threadIdx.x & 7;
    const uint8_t* blk = w + ib * Q8_0_BYTES;
    const float d = f16_to_f32(load_u16(blk));
    const int8_t* qs = reinterpret_cast<const int8_t*>(blk + 2 + 4 * t);
    store4<F16>(y, ib * QK8_0 + 4 * t, (float)qs[0] * d, (float)qs[1] * d, (float)qs[2] * d,
                (float)qs[3] * d);
}

hipError_t launch_dequantize(int dtype, const uint8_t* w, size_t nblocks, float* y, bool to_f16,
                             hipStream_t s) {
    if (nblocks == 0) return hipSuccess;
    const dim3 grid8((unsigned)((nblocks + DQ_WG / 32 - 1) / (DQ_WG / 32)));
    switch (dtype) {
        case GGML_Q4K:
            if (to_f16) hipLaunchKernelGGL(dequant_q4k_kernel<true>, grid8, dim3(DQ_WG), 0, s, w, nblocks, (void*)y);
            else hipLaunchKernelGGL(dequant_q4k_kernel<false>, grid8, dim3(DQ_WG), 0, s, w, nblocks, (void*)y);
            break;
        case GGML_Q6K:
            if (to_f16) hipLaunchKernelGGL(dequant_q6k_kernel<true>, grid8, dim3(DQ_WG), 0, s, w, nblocks, (void*)y);
            else hipLaunchKernelGGL(dequant_q6k_kernel<false>, grid8, dim3(DQ_WG), 0, s, w, nblocks, (void*)y);
            break;
        case GGML_Q8_0: {
            dim3 grid((unsigned)((nblocks + DQ_WG / 8 - 1) / (DQ_WG / 8)));
            if (to_f16) hipLaunchKernelGGL(dequant_q8_0_kernel<true>, grid, dim3(DQ_WG), 0, s, w, nblocks, (void*)y);
            else hipLaunchKernelGGL(dequant_q8_0_kernel<false>, grid, dim3(DQ_WG), 0, s, w, nblocks, (void*)y);
            break;
        }
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace frq
