// The passes beside the projections: the FP32 -> bf16 convert and its inverse, and
// the attention dots L[i,h] = Z[i,h,:] . aL[h], R[i,h] = Z[i,h,:] . aR[h] of the
// FP32 layers whose projection does not form them.
//
// Reference: the FP32 -> bf16 RNE convert (baseline/src/common.cpp:80-93) and
// lr_from_z (baseline/src/baseline_standard.cpp:7-20).
#include "internal.hpp"

namespace gatgpu {
namespace {

constexpr int kThreads = 256;

// x [n][d] FP32 -> y [n][dp] bf16, columns d..dp-1 zero.  Bound by memory: four
// columns a thread, 16 bytes in and 8 out (one column a thread: 271 us for 300K
// rows of 500, 3.3 TB/s).
__global__ void __launch_bounds__(kThreads)
k_to_bf16_pad(const float* __restrict__ x, uint16_t* __restrict__ y, uint64_t n, uint32_t d, uint32_t dp) {
    const uint32_t per_row = dp / 4;
    const uint64_t count = n * uint64_t(per_row);
    for (uint64_t i = blockIdx.x * uint64_t(kThreads) + threadIdx.x; i < count;
         i += uint64_t(gridDim.x) * kThreads) {
        const uint64_t r = i / per_row;
        const uint32_t c = uint32_t(i - r * per_row) * 4;
        const float* p = x + r * d + c;
        float v[4] = {};
        if (c + 4 <= d) {
            __builtin_memcpy(v, p, 16);  // rows of any width: 4-byte alignment
        } else {
#pragma unroll
            for (int q = 0; q < 3; ++q)
                if (c + q < d) v[q] = p[q];
        }
        *reinterpret_cast<uint2*>(y + r * dp + c) =
            make_uint2(bf16_rne(v[0]) | uint32_t(bf16_rne(v[1])) << 16, bf16_rne(v[2]) | uint32_t(bf16_rne(v[3])) << 16);
    }
}

__global__ void __launch_bounds__(kThreads)
k_widen_bf16(const uint16_t* __restrict__ x, float* __restrict__ y, uint64_t count) {
    for (uint64_t i = blockIdx.x * uint64_t(kThreads) + threadIdx.x; i < count;
         i += uint64_t(gridDim.x) * kThreads)
        y[i] = bf16_widen(x[i]);
}

// G lanes per (row, head): the dots of lr_from_z over the FP32 Z row, VEC
// features a load.  Bound by the reads of Z, so consecutive lanes read
// consecutive features: one lane per dot, reading its head's features one by
// one, took 142 us on 120K rows of 8 x 32 (0.9 TB/s).
template <int VEC, int G>
__global__ void __launch_bounds__(kThreads)
k_lr_from_z(const float* __restrict__ z, uint64_t n, int K, int dim, int zs, const float* __restrict__ al,
            const float* __restrict__ ar, float* __restrict__ left, float* __restrict__ right) {
    const uint64_t q = blockIdx.x * uint64_t(kThreads) + threadIdx.x, t = q / G;
    const int sub = int(q % G);
    if (t >= n * K) return;  // whole groups
    const uint64_t i = t / K;
    const int h = int(t % K);
    const float* zi = z + i * zs + h * dim;
    float l = 0.0f, r = 0.0f;
    for (int f = sub * VEC; f < dim; f += G * VEC) {
        float v[VEC];
        __builtin_memcpy(v, __builtin_assume_aligned(zi + f, 4 * VEC), 4 * VEC);
#pragma unroll
        for (int x = 0; x < VEC; ++x)
            if (f + x < dim) {  // (a one-head row's last vector reaches into its padding)
                l += v[x] * al[h * dim + f + x];
                r += v[x] * ar[h * dim + f + x];
            }
    }
#pragma unroll
    for (int off = 1; off < G; off <<= 1) {
        l += __shfl_xor(l, off);
        r += __shfl_xor(r, off);
    }
    if (sub == 0) {
        left[t] = l;
        right[t] = r;
    }
}

uint32_t grid_for(uint64_t items, uint32_t cap) {
    uint64_t g = (items + kThreads - 1) / kThreads;
    if (g < 1) g = 1;
    return uint32_t(g > cap ? cap : g);
}

}  // namespace

hipError_t launch_to_bf16_pad(const float* x, uint16_t* y, uint64_t n, int d, int dp, hipStream_t s) {
    if (dp % 4 || dp < d) return hipErrorInvalidValue;
    k_to_bf16_pad<<<grid_for(n * uint64_t(dp / 4), 1u << 16), kThreads, 0, s>>>(x, y, n, uint32_t(d), uint32_t(dp));
    return hipGetLastError();
}

hipError_t launch_widen_bf16(const uint16_t* x, float* y, uint64_t count, hipStream_t s) {
    k_widen_bf16<<<grid_for(count, 1u << 16), kThreads, 0, s>>>(x, y, count);
    return hipGetLastError();
}

namespace {
template <int VEC, int G>
hipError_t lr_from_z_lanes(const float* z, uint64_t n, int heads, int dim, int zs, const float* al, const float* ar,
                           float* left, float* right, hipStream_t s) {
    const uint64_t blocks = (n * uint64_t(heads) * G + kThreads - 1) / kThreads;
    if (blocks < 1 || blocks > 0x7fffffffu) return hipErrorInvalidValue;
    k_lr_from_z<VEC, G><<<dim3(uint32_t(blocks)), kThreads, 0, s>>>(z, n, heads, dim, zs, al, ar, left, right);
    return hipGetLastError();
}
}  // namespace

// 16-byte loads where every head starts on 16 bytes (rows do: zs % 4 == 0).
hipError_t launch_lr_from_z(const float* z, uint64_t n, int heads, int dim, int zs, const float* al, const float* ar,
                            float* left, float* right, hipStream_t s) {
    const bool vec = zs % 4 == 0 && (dim % 4 == 0 || heads == 1);
    if (vec)
        return dim <= 8 ? lr_from_z_lanes<4, 2>(z, n, heads, dim, zs, al, ar, left, right, s)
                        : lr_from_z_lanes<4, 8>(z, n, heads, dim, zs, al, ar, left, right, s);
    return dim <= 8 ? lr_from_z_lanes<1, 2>(z, n, heads, dim, zs, al, ar, left, right, s)
                    : lr_from_z_lanes<1, 8>(z, n, heads, dim, zs, al, ar, left, right, s);
}

}  // namespace gatgpu
