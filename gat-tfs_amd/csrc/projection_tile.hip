// bf16 projection for few rows, and for the shapes of no other kernel: one
// output block a wave, the input tile through LDS.
//
// k_proj_fast (projection_mfma.hip) gives each wave a 32-row tile and all output
// blocks, 8 tiles a block with the whole of W in its LDS: below 8 tiles per CU it
// leaves CUs idle and every block still waits for W (1024 rows of 128 -> 8 x 32:
// 10 us on 4 of 256 CUs).  Here a block takes one tile (2 or 4 where the layer has
// few output blocks) and each of its waves one output block, whose W^T fragments
// sit in its registers: the chip fills from 32 rows per CU on, and the wait is one
// round trip for the fragments and the tile.  FP32 input of any width and
// alignment is rounded while it is staged (the convert stage,
// baseline/src/common.cpp:80-93, fused; nothing past a row's `in` values is read).
// Blocks are persistent; the next tile is requested before this one multiplies.
// The MFMA chain of an output block runs its k steps in the order of the other
// paths, so Z, L and R carry the same bits.
#include "internal.hpp"

namespace gatgpu {
namespace {

typedef __bf16 bf16x8 __attribute__((__vector_size__(8 * sizeof(__bf16))));
typedef float f32x16 __attribute__((__vector_size__(16 * sizeof(float))));


// KS: the most k steps (a.ksteps of them used).  tpb: tiles a block takes at once.
// TAIL: R lies in the 16 bytes of the row's last features (one head of 57 to 60):
// the L/R block's wave writes R, in no order with the wave of those features, so
// that one leaves the four bytes out.  (A template parameter: the test of a kernel
// argument in the store cost 1.5 us a launch, in registers spilled.)
template <int KS, bool F32IN, bool TAIL>
__global__ void __launch_bounds__((KS > 16 ? 8 : 9) * kWave) k_proj_tile(ProjArgs a, int tpb) {
    extern __shared__ __attribute__((aligned(16))) uint4 xs[];  // [2][tpb][ksteps][64]
    const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave), l = threadIdx.x % kWave;
    const int half = l / 32, col = l % 32;
    const int nb = a.head_blocks + 1, ks_n = a.ksteps;
    const int tl = w / nb, ob = w % nb;
    const bool lr = ob == a.head_blocks, act = tl < tpb;
    clear_words(a.clear, a.nclear);
    uint4 wf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
        wf[ks] = act && ks < ks_n ? a.wpk[(size_t(ks) * a.nmb + ob) * kWave + l] : make_uint4(0, 0, 0, 0);
    __shared__ __attribute__((aligned(16))) float arl[256];
    if (a.r_from_z)
        for (int q = threadIdx.x; q < 256; q += int(blockDim.x)) arl[q] = a.ar[q];
    // Staging: a unit is one k step of one tile, a wave's in one instruction (bf16:
    // 2 lanes a row) or two (FP32: 4 lanes a row, rows l / 4 and 16 + l / 4).
    constexpr int PER = F32IN ? 4 : 2, RI = F32IN ? 2 : 1;
    constexpr int UN = (KS == 16 ? 4 : 8) / RI;  // 16 k steps: 8 loads ahead no longer fit the registers of 9 waves
    const int units = tpb * ks_n, waves = int(blockDim.x) / kWave;
    const int buf_len = units * kWave;
    const int p = l % PER, r0 = l / PER;
    const uint64_t groups = (a.tiles + tpb - 1) / tpb;
    uint4 pre[UN][RI];
    // Units u0, u0 + waves, ... (UN of them) of tile group g.
    auto request = [&](uint64_t g, int u0) {
#pragma unroll
        for (int y = 0; y < UN; ++y) {
            const int u = u0 + y * waves;
            if (u >= units) continue;
            const int t = u / ks_n, ks = u - t * ks_n;
#pragma unroll
            for (int i = 0; i < RI; ++i) {
                const uint64_t row = (g * tpb + t) * 32 + r0 + 16 * i, rs = row < a.n ? row : a.n - 1;
                if constexpr (F32IN) {
                    const int k = 16 * ks + 4 * p;
                    const float* x = a.x32 + rs * a.in + k;
                    float v[4] = {};
                    if (k + 4 <= a.in) {
                        __builtin_memcpy(v, x, 16);  // rows of any width: 4-byte alignment
                    } else {
#pragma unroll
                        for (int z = 0; z < 3; ++z)
                            if (k + z < a.in) v[z] = x[z];
                    }
                    __builtin_memcpy(&pre[y][i], v, 16);
                } else {
                    pre[y][i] = *reinterpret_cast<const uint4*>(a.x + rs * a.xs + 16 * ks + 8 * p);
                }
            }
        }
    };
    auto store = [&](uint64_t g, int u0, uint4* buf) {
#pragma unroll
        for (int y = 0; y < UN; ++y) {
            const int u = u0 + y * waves;
            if (u >= units) continue;
#pragma unroll
            for (int i = 0; i < RI; ++i) {
                const uint4 v = pre[y][i];
                const int r = r0 + 16 * i;
                if constexpr (F32IN) {
                    const uint2 b = make_uint2(bf16x2(__builtin_bit_cast(float, v.x), __builtin_bit_cast(float, v.y)),
                                               bf16x2(__builtin_bit_cast(float, v.z), __builtin_bit_cast(float, v.w)));
                    reinterpret_cast<uint2*>(buf + u * kWave + (p / 2) * 32 + r)[p % 2] = b;
                    if (a.xout) {  // the rounded rows also leave the kernel
                        const int t = u / ks_n;
                        const uint64_t row = (g * tpb + t) * 32 + r;
                        if (row < a.n)
                            *reinterpret_cast<uint2*>(a.xout + row * a.xouts + 16 * (u - t * ks_n) + 4 * p) = b;
                    }
                } else {
                    buf[u * kWave + p * 32 + r] = v;
                }
            }
        }
    };
    auto rest = [&](uint64_t g, uint4* buf) {  // what pre does not hold
        for (int u0 = w + UN * waves; u0 < units; u0 += UN * waves) {
            request(g, u0);
            store(g, u0, buf);
        }
    };
    uint64_t g = blockIdx.x;
    request(g, w);
    store(g, w, xs);
    rest(g, xs);
    for (int buf = 0; g < groups; g += gridDim.x, buf ^= 1) {
        // LDS only: the stores of the tile before stay in flight.  (Every wave
        // has read the other buffer: it is the next tile's.)
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const uint64_t next = g + gridDim.x;
        if (next < groups) request(next, w);
        if (act) {
            const uint4* xb = xs + buf * buf_len + tl * ks_n * kWave + l;
            f32x16 acc;
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
                if (ks < ks_n)
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, wf[ks]),
                                                                  __builtin_bit_cast(bf16x8, xb[ks * kWave]), acc, 0, 0, 0);
            const uint64_t row = (g * tpb + tl) * 32 + col;
            const bool ok = row < a.n;
            if (!lr) {
                // Permuted packing: features 32 ob + 16 half + {0..15} of row col.
                uint32_t zp[8];
#pragma unroll
                for (int x = 0; x < 8; ++x) zp[x] = bf16x2(acc[2 * x], acc[2 * x + 1]);
#pragma unroll
                for (int q8 = 0; q8 < 2; ++q8) {
                    const int f0 = 32 * ob + 16 * half + 8 * q8;
                    if (!ok || f0 >= a.width) continue;
                    uint16_t* to = a.z + row * a.zs + f0;
                    if (TAIL && f0 + 8 > a.r_off) {
                        *reinterpret_cast<uint2*>(to) = make_uint2(zp[4 * q8], zp[4 * q8 + 1]);
                        *reinterpret_cast<uint32_t*>(to + 4) = zp[4 * q8 + 2];
                        continue;
                    }
                    *reinterpret_cast<uint4*>(to) =
                        make_uint4(zp[4 * q8], zp[4 * q8 + 1], zp[4 * q8 + 2], zp[4 * q8 + 3]);
                }
                if (a.r_from_z) {
                    // R = Z_bf16 . aR in the aggregation's order: an FMA chain over
                    // each 8 features, then (s0 + s1) + (s2 + s3).
                    float s8[2];
#pragma unroll
                    for (int q8 = 0; q8 < 2; ++q8) {
                        float t = 0.0f;
#pragma unroll
                        for (int x = 0; x < 8; ++x) {
                            const uint32_t pr = zp[4 * q8 + x / 2];
                            t = __builtin_fmaf(__builtin_bit_cast(float, (x & 1) ? (pr & 0xffff0000u) : (pr << 16)),
                                               arl[32 * ob + 16 * half + 8 * q8 + x], t);
                        }
                        s8[q8] = t;
                    }
                    const float part = s8[0] + s8[1];
                    const float r = part + __shfl_xor(part, 32);
                    if (ok && half == 0) a.right[row * 8 + ob] = r;
                }
            } else if (ok) {
                // L/R block: lane half h4 holds heads 4 h4 + {0..3} of each quarter
                // (L hi, R hi, L lo, R lo) in registers {0..3}, {4..7}, {8..11}, {12..15}.
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int h = 4 * half + q;
                    if (h < a.heads) {
                        a.left[row * a.heads + h] = acc[q] + acc[8 + q];
                        const float rv = acc[4 + q] + acc[12 + q];
                        if (!a.r_from_z) a.right[row * a.heads + h] = rv;
                        if (a.r_in_z) *reinterpret_cast<float*>(a.z + row * a.zs + a.r_off + 2 * h) = rv;
                    }
                }
            }
        }
        if (next < groups) {
            uint4* nb_ = xs + (buf ^ 1) * buf_len;
            store(next, w, nb_);
            rest(next, nb_);
        }
    }
}

int tiles_per_block(int head_blocks) { return head_blocks == 1 ? 4 : head_blocks <= 3 ? 2 : 1; }

template <int KS, bool F32IN, bool TAIL>
hipError_t launch(const ProjArgs& a, hipStream_t s, int cus) {
    // Few tiles: one a block, so that more CUs share them; and what fits LDS
    // beside the 1 KB of aR.
    int tpb = tiles_per_block(a.head_blocks);
    const auto bytes = [&](int t) { return size_t(2) * t * a.ksteps * kWave * sizeof(uint4); };
    while (tpb > 1 && ((a.tiles + tpb - 1) / tpb < uint64_t(cus) || bytes(tpb) > 128 * 1024)) tpb /= 2;
    const size_t lds = bytes(tpb);
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_proj_tile<KS, F32IN, TAIL>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
        if (e != hipSuccess) return e;
    }
    // At least 8 waves: those without an output block help with the input.
    const int compute = tpb * (a.head_blocks + 1), threads = (compute < 8 ? 8 : compute) * kWave;
    // Resident blocks: as many as the CU's LDS and 16 waves allow.
    uint64_t per_cu = 16 * kWave / threads;
    if (per_cu > 159 * 1024 / (lds + 1024)) per_cu = 159 * 1024 / (lds + 1024);
    if (per_cu < 1) per_cu = 1;
    uint64_t grid = uint64_t(cus) * per_cu;
    const uint64_t groups = (a.tiles + tpb - 1) / tpb;
    if (grid > groups) grid = groups;
    k_proj_tile<KS, F32IN, TAIL><<<dim3(uint32_t(grid)), threads, lds, s>>>(a, tpb);
    return hipGetLastError();
}

template <bool F32IN, bool TAIL>
hipError_t launch_ks(const ProjArgs& a, hipStream_t s, int cus) {
    if (a.ksteps <= 4) return launch<4, F32IN, TAIL>(a, s, cus);
    if (a.ksteps <= 8) return launch<8, F32IN, TAIL>(a, s, cus);
    if (a.ksteps <= 16) return launch<16, F32IN, TAIL>(a, s, cus);
    return launch<32, F32IN, TAIL>(a, s, cus);
}

}  // namespace

bool projection_tile_shape(const ProjArgs& a) {
    return a.n > 0 && a.groups == 1 && a.head_blocks >= 1 && a.head_blocks <= 8 && a.nmb > a.head_blocks &&
           a.ksteps >= 1 && (a.ksteps <= 16 || (a.ksteps <= 32 && a.head_blocks <= 7)) && !(a.r_from_z && a.heads == 1);
}

hipError_t launch_projection_tile(const ProjArgs& a, hipStream_t s, int cus) {
    if (!projection_tile_shape(a) || a.tiles != (a.n + 31) / 32 || (a.r_from_z && (!a.ar || a.heads != 8 || a.width != 256)))
        return hipErrorInvalidValue;
    // R in the row: the last four bytes of its last 16-byte piece.
    if (a.r_in_z && (a.heads != 1 || a.zs % 8 || a.r_off != a.zs - 2 || a.width > a.r_off)) return hipErrorInvalidValue;
    if (a.r_in_z && a.width > a.zs - 8) return a.x32 ? launch_ks<true, true>(a, s, cus) : launch_ks<false, true>(a, s, cus);
    return a.x32 ? launch_ks<true, false>(a, s, cus) : launch_ks<false, false>(a, s, cus);
}

}  // namespace gatgpu
