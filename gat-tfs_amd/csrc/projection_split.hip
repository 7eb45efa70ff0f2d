// FP32 projection Z = X W with the attention dots, on the bf16 matrix units at
// FP32 accuracy.
//
// Reference: projection (baseline/src/baseline_standard.cpp:3-6, cblas_sgemm)
// and lr_from_z (:7-20).
//
// Each FP32 operand, times a power of two, is the sum of three bf16 parts, x = x1 +
// x2 + x3 (x1 the rounding of x, x2 of x - x1, x3 of the rest).  That is exact as
// long as no part is below bf16's normal range: inputs take 2^24, which keeps the
// parts of every FP32 number above it, subnormals included (x3 loses bits from
// 2^-103 down without), and weights 2^-24, which the inputs' factor cancels.  A
// layer with weights below 2^-79 takes 2^24 for them too, and the sums are brought
// back once a tile is done (projection_split_scale).
//
// The product keeps the six terms down to 2^-18 of it: x3 w1, x2 w2, x1 w3,
// x2 w1, x1 w2, x1 w1, the small ones first, in one FP32 accumulator chain; the
// dropped x2 w3 + x3 w2 are below 2^-25 of |x w|.  v_mfma_f32_32x32x16_bf16
// runs 16 times the rate of v_mfma_f32_32x32x2_f32, so six of them cost 0.38 of
// the FP32 instruction's time.  Error of the whole forward against 64 bits (2.5M
// edges): 2.2e-7, 2.5e-7 with the FP32 instruction; over other widths 0.8 to 1.0
// of it.  On 169K rows: 128 -> 8 x 32 in 75 us (141 with the FP32 instruction),
// 256 -> 8 x 32 in 125 (251), 256 -> 40 in 67 (93); 120K rows of 100 inputs,
// which had a VALU product: 55 us (297).  What is left above the 50 to 65 us of
// memory traffic is the matrix units: 53 us at their peak for 256 inputs.
//
// Work split: W-stationary.  A wave keeps one 32-feature output block's three
// parts of W^T in registers (12 KS of them) for the whole launch, and a block of
// 8 waves takes tiles of 32 rows: the output blocks of a layer share a tile, and
// where a layer has at most 2 or 4 of them the block takes TPB = 4 or 2 tiles.
// The input is read from HBM once, split once by the thread that loaded it, and
// handed round through two LDS slots of CK k steps (one LDS-only barrier a
// slot), with the loads PD slots ahead.  Persistent blocks, one per CU.
// A tile's Z leaves as 64-byte row segments after a 4 x 4 transpose of 16-byte
// pieces inside the lane quad.
//
// L and R are dots of the FP32 Z row, as the reference forms them.  Heads of
// whole output blocks (32, 64, or a layer's only head): each wave's share
// through LDS, stored a tile late as whole rows of heads.  Heads of 1 to 16 that
// divide 16: inside the lane.  Other widths: launch_lr_from_z (3 us and a read of
// Z more).
//
// Values that leave the range (NaN, infinities, inputs of 2^103 and more, weights
// of 2^103 beside some below 2^-79) leave an infinity or NaN in the accumulators,
// and so in their dot with aL: the wave that finds one takes its block of the tile
// again in plain FP32.  (Marks set in LDS while the input was split cost 2 to 4 us
// of the times above.)
//
// More than 256 inputs run as several launches, each adding its k range to the
// Z the one before left; the last forms L and R.
#include <cmath>

#include "internal.hpp"

namespace gatgpu {
namespace {

typedef __bf16 bf16x8 __attribute__((__vector_size__(8 * sizeof(__bf16))));
typedef float f32x16 __attribute__((__vector_size__(16 * sizeof(float))));

constexpr int kWaves = 8;
constexpr int kThreads = kWaves * kWave;
constexpr float kScaleX = 0x1p24f;
enum { kLrNone = 0, kLrShare = 1, kLrLane = 2 };  // where a launch forms L and R

// scale x = p[0] + p[1] + p[2], pairs of bf16 (lo = first).
__device__ inline void split2(float a, float b, float scale, uint32_t (&p)[3]) {
    a *= scale;
    b *= scale;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        p[q] = bf16x2(a, b);
        a -= __builtin_bit_cast(float, p[q] << 16);
        b -= __builtin_bit_cast(float, p[q] & 0xffff0000u);
    }
}

// KS: k steps of 16; TPB: tiles a block takes at once; LR: where it forms L and
// R (a runtime choice spilled 50 more scalars: 126 -> 141 us on 169K x 256 -> 8 x 32).
template <int KS, int TPB, int LR>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2))) k_proj_split(ProjF32Args a) {
    constexpr int U = KS > 8 ? 4 : 8;             // (tile, k step) pairs a slot holds
    constexpr int UT = U / 4;                     // of them a thread stages (a float4 each)
    constexpr int CK = U / TPB;                   // k steps per slot
    constexpr int NCH = (KS + CK - 1) / CK;       // slots per tile
    constexpr int PD = NCH % 2 == 0 ? 2 : NCH;    // slots requested ahead (divides NCH)
    __shared__ __attribute__((aligned(16))) uint2 xs[2][U][3][2 * kWave];
    __shared__ float plr[2][kWaves][2][32];       // L and R shares of a wave's rows, two tiles
    __shared__ float alr[2][kWaves][32];          // aL, aR of the group's output blocks
    clear_words(a.clear, a.nclear);
    // Beyond 128 inputs the third parts of W (one of the six terms) stay in LDS:
    // 12 KS registers would not leave room for the rest.
    constexpr int WP = KS > 8 ? 2 : 3;
    __shared__ __attribute__((aligned(16))) uint4 w3[WP == 2 ? kWaves * KS * kWave : 1];
    const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / kWave), l = threadIdx.x % kWave;
    const int half = l / 32, col = l % 32;
    const int g = blockIdx.y;
    const int nb = a.nob - 8 * g < 8 ? a.nob - 8 * g : 8;  // output blocks of this group
    const int tl = w / nb, ob = 8 * g + w % nb;
    const bool act = tl < TPB;
    uint4 wf[KS][WP];
    if (act) {
        const uint4* src = a.wpk + (size_t(ob) * KS * 3) * kWave + l;
#pragma unroll
        for (int q = 0; q < KS * 3; ++q) {
            if (q % 3 < WP) wf[q / 3][q % 3] = src[q * kWave];
            else w3[(w * KS + q / 3) * kWave + l] = src[q * kWave];  // read by this wave only
        }
    }
    if constexpr (LR != kLrNone) {
        for (int q = threadIdx.x; q < 2 * kWaves * 32; q += kThreads) {
            const int f = 256 * g + q % 256;
            (&alr[0][0][0])[q] = f < a.width ? (q < 256 ? a.al : a.ar)[f] : 0.0f;
        }
    }
    __syncthreads();
    // Staging: wave w takes rows 16 (w % 2) .. + 15 of units w / 2 (and w / 2 +
    // 4), four lanes a row (64 bytes); unit u is k step u % CK of tile u / CK.
    const int srow = 16 * (w % 2) + l / 4, sp = l % 4;
    const uint64_t groups = (a.tiles + TPB - 1) / TPB;
    float4 pre[PD][UT];
    auto load = [&](uint64_t tg, int c, float4 (&to)[UT]) {
#pragma unroll
        for (int y = 0; y < UT; ++y) {
            const int su = w / 2 + 4 * y;
            const uint64_t r = (tg * TPB + su / CK) * 32 + srow;
            const int k = (c * CK + su % CK) * 16 + 4 * sp;
            const float* p = a.x + (r < a.n ? r : a.n - 1) * a.xs + a.k0 + k;
            float4 v = make_float4(0, 0, 0, 0);
            if (k + 4 <= a.kn) {
                __builtin_memcpy(&v, p, 16);  // rows of any width: 4-byte alignment
            } else {
                if (k < a.kn) v.x = p[0];
                if (k + 1 < a.kn) v.y = p[1];
                if (k + 2 < a.kn) v.z = p[2];
            }
            to[y] = v;
        }
    };
    // (No constant to the compiler: it would fold the product into both arms of the
    // load, which then waits: 125 -> 141 us on 169K rows of 256 -> 8 x 32.)
    float scale_x = kScaleX;
    asm("" : "+s"(scale_x));
    // The loaded values as three parts into a slot.
    auto stage = [&](const float4 (&from)[UT], int slot) {
#pragma unroll
        for (int y = 0; y < UT; ++y) {
            const float4 v = from[y];
            uint32_t p0[3], p1[3];
            split2(v.x, v.y, scale_x, p0);
            split2(v.z, v.w, scale_x, p1);
#pragma unroll
            for (int q = 0; q < 3; ++q)
                xs[slot][w / 2 + 4 * y][q][((sp / 2) * 32 + srow) * 2 + sp % 2] = make_uint2(p0[q], p1[q]);
        }
    };
    // L and R of the tile group before: shares summed over a head's blocks.
    const int bph = LR == kLrShare ? (a.dim + 31) / 32 : 1, hpg = nb / bph;
    auto store_lr = [&](uint64_t tg, int par) {
        for (int q = threadIdx.x; q < TPB * 64 * hpg; q += kThreads) {
            const int h = q % hpg, r = (q / hpg) % 32, side = (q / hpg / 32) % 2, t = q / hpg / 64;
            float v = 0.0f;
            for (int b = 0; b < bph; ++b) v += plr[par][t * nb + h * bph + b][side][r];
            const uint64_t row = (tg * TPB + t) * 32 + r;
            if (row < a.n) (side ? a.right : a.left)[row * a.heads + (8 * g) / bph + h] = v;
        }
    };
    // Slots run PD + 1 ahead of the loads: slot s + 1 is staged (from the
    // registers) and slot s + 1 + PD requested while slot s multiplies.
    uint64_t tg = blockIdx.x;
    load(tg, 0, pre[0]);
    stage(pre[0], 0);
    if (NCH == 1) load(tg + gridDim.x < groups ? tg + gridDim.x : groups - 1, 0, pre[0]);
#pragma unroll
    for (int c = 1; c < NCH && c < PD + 1; ++c) load(tg, c, pre[c % PD]);
    if (NCH > 1 && NCH < PD + 1) load(tg + gridDim.x < groups ? tg + gridDim.x : groups - 1, 0, pre[0]);
    uint64_t prev = groups;  // the tile group whose L and R wait in plr
    int it = 0;
    for (; tg < groups; prev = tg, tg += gridDim.x, ++it) {
        const uint64_t nx = tg + gridDim.x < groups ? tg + gridDim.x : groups - 1;
        const uint64_t nx2 = tg + 2 * uint64_t(gridDim.x) < groups ? tg + 2 * uint64_t(gridDim.x) : groups - 1;
        const uint64_t tile = tg * TPB + tl;
        const uint64_t row = tile * 32 + col;
        const uint64_t rs = row < a.n ? row : a.n - 1;
        f32x16 acc;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
        if (a.add && act) {  // the k ranges before
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int f = 32 * ob + 16 * half + r;
                if (f < a.width) acc[r] = a.z[rs * a.zs + f] * a.sum_scale;
            }
        }
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const int slot = (it * NCH + c) & 1;
            // The slots are LDS only: the loads and stores in flight stay so.
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            // Every wave has left the tile before: its L and R shares are whole.
            if (c == 0 && LR == kLrShare && prev < groups) store_lr(prev, (it + 1) & 1);
            {
                const int cn = (c + 1) % NCH;  // the next slot's part of its tile
                stage(pre[cn % PD], slot ^ 1);
                const int ahead = c + 1 + PD;
                if (ahead < NCH) load(tg, ahead, pre[cn % PD]);
                else if (ahead < 2 * NCH) load(nx, ahead - NCH, pre[cn % PD]);
                else load(nx2, ahead - 2 * NCH, pre[cn % PD]);
            }
            if (act) {
#pragma unroll
                for (int q = 0; q < CK; ++q) {
                    const int ks = c * CK + q;
                    if (ks >= KS) continue;
                    bf16x8 b[3], m[3];
#pragma unroll
                    for (int p = 0; p < 3; ++p) {
                        b[p] = __builtin_bit_cast(bf16x8, reinterpret_cast<const uint4*>(xs[slot][tl * CK + q][p])[l]);
                        if (p < WP) m[p] = __builtin_bit_cast(bf16x8, wf[ks][p < WP ? p : 0]);
                        else m[p] = __builtin_bit_cast(bf16x8, w3[(w * KS + ks) * kWave + l]);
                    }
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(m[0], b[2], acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(m[1], b[1], acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(m[2], b[0], acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(m[0], b[1], acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(m[1], b[0], acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(m[0], b[0], acc, 0, 0, 0);
                }
            }
        }
        if (!act) continue;
        // NaN or infinite where an accumulator is (a dot of finite values that
        // overflows by itself only costs the plain products).
        float over = 0.0f;
        // kLrLane: feature r of the lane ends its head.
        auto lane_lr = [&](int r, float& lv, float& rv) {
            const int f = 32 * ob + 16 * half + r;
            if ((r & (a.dim - 1)) != a.dim - 1) return;
            if (f < a.width && row < a.n) {
                const uint64_t at = row * a.heads + f / a.dim;
                a.left[at] = lv;
                a.right[at] = rv;
            }
            lv = rv = 0.0f;
        };
        if (a.sum_scale != 1.0f) {
            const float back = 1.0f / a.sum_scale;
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[r] *= back;
        }
        if constexpr (LR != kLrNone) {
            float lv = 0.0f, rv = 0.0f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                lv = __builtin_fmaf(acc[r], alr[0][ob - 8 * g][16 * half + r], lv);
                rv = __builtin_fmaf(acc[r], alr[1][ob - 8 * g][16 * half + r], rv);
                if constexpr (LR == kLrLane) lane_lr(r, lv, rv);
            }
            if constexpr (LR == kLrShare) {
                over = lv;
                lv = xor32_add(lv);
                rv = xor32_add(rv);
                plr[it & 1][w][half][col] = half ? rv : lv;
            }
        }
        if constexpr (LR != kLrShare) {
            float o2 = 0.0f;
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                over = __builtin_fmaf(acc[r], 0.0f, over);
                o2 = __builtin_fmaf(acc[r + 1], 0.0f, o2);
            }
            over += o2;
        }
        // Lane (half, col) holds features 32 ob + 16 half + {0..15} of row
        // col: four 16-byte pieces.  After the transpose lane c of a quad
        // (rows 4a .. 4a + 3) holds piece c of each of its rows.
        const int c = l & 3;
        uint32_t S[4][4], U[4][4];
#pragma unroll
        for (int r = 0; r < 16; ++r) S[r / 4][r % 4] = __builtin_bit_cast(uint32_t, float(acc[r]));
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const uint32_t o = uint32_t(__builtin_amdgcn_mov_dpp(int(S[p ^ 1][v]), 0xB1, 0xF, 0xF, false));
                U[p][v] = (c & 1) == (p & 1) ? S[p][v] : o;  // quad_perm [1, 0, 3, 2]
            }
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const uint32_t o = uint32_t(__builtin_amdgcn_mov_dpp(int(U[p ^ 2][v]), 0x4E, 0xF, 0xF, false));
                S[p][v] = (c & 2) == (p & 2) ? U[p][v] : o;  // quad_perm [2, 3, 0, 1]
            }
        const int f0 = 32 * ob + 16 * half + 4 * c;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint64_t rj = tile * 32 + uint64_t((col & ~3) + j);
            if (rj < a.n && f0 < a.width)
                *reinterpret_cast<uint4*>(a.z + rj * a.zs + f0) = make_uint4(S[j][0], S[j][1], S[j][2], S[j][3]);
        }
        if (__any(!(fabsf(over) < INFINITY))) {
            // Plain FP32 products of the block, one feature at a time, from the
            // first input on (the sums of the launches before are stored over).
            // Last, so that the chain of `over` holds nothing else up; the
            // stores above come from other lanes of the wave and go first.
            __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
            asm volatile("" ::: "memory");
            const float* x = a.x + rs * a.xs;
            float lv = 0.0f, rv = 0.0f;
#pragma unroll 1
            for (int r = 0; r < 16; ++r) {
                const int f = 32 * ob + 16 * half + r;
                if (f >= a.width) break;
                float s = 0.0f;
                for (int k = 0; k < a.k0 + a.kn; ++k) s = __builtin_fmaf(x[k], a.w32[size_t(k) * a.width + f], s);
                if (row < a.n) a.z[row * a.zs + f] = s;
                if constexpr (LR != kLrNone) {
                    lv = __builtin_fmaf(s, alr[0][ob - 8 * g][16 * half + r], lv);
                    rv = __builtin_fmaf(s, alr[1][ob - 8 * g][16 * half + r], rv);
                }
                if constexpr (LR == kLrLane) lane_lr(r, lv, rv);
            }
            if constexpr (LR == kLrShare) {
                lv = xor32_add(lv);
                rv = xor32_add(rv);
                plr[it & 1][w][half][col] = half ? rv : lv;
            }
        }
    }
    if (LR == kLrShare && prev < groups) {
        __syncthreads();
        store_lr(prev, (it + 1) & 1);
    }
}

// Three bf16 parts of W in the fragment order [launch][block][k step][part]
// [lane][8]: lane (half, c) of block b holds W[16 ks + 8 half + j][32 b + phi(c)],
// phi(c) = 16 ((c % 8) / 4) + 4 (c / 8) + c % 4, so that a lane's D rows are 16
// consecutive features; zeros past the inputs and the width.  One wave per
// (launch, block, k step).
__global__ void __launch_bounds__(kWave) k_pack_split(const float* __restrict__ w, int in, int width, int ks,
                                                      float scale, uint4* __restrict__ out) {
    const int l = threadIdx.x, c = l % 32, hb = (width + 31) / 32;
    const int step = blockIdx.x % ks, b = blockIdx.x / ks % hb, pass = blockIdx.x / ks / hb;
    const int f = 32 * b + 16 * ((c % 8) / 4) + 4 * (c / 8) + c % 4;
    uint32_t part[3][4];
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        const int k = 16 * (pass * ks + step) + 8 * (l / 32) + 2 * x;
        uint32_t p[3];
        split2(k < in && f < width ? w[size_t(k) * width + f] : 0.0f,
               k + 1 < in && f < width ? w[size_t(k + 1) * width + f] : 0.0f, scale, p);
#pragma unroll
        for (int q = 0; q < 3; ++q) part[q][x] = p[q];
    }
#pragma unroll
    for (int q = 0; q < 3; ++q)
        out[(size_t(blockIdx.x) * 3 + q) * kWave + l] = make_uint4(part[q][0], part[q][1], part[q][2], part[q][3]);
}

constexpr int kKsOf[] = {2, 4, 6, 7, 8, 12, 16};

// k steps per launch and launches for `in` inputs: the fewest launches of at
// most 256 inputs, their ranges as equal as whole k steps allow.
void split_passes(int in, int& ks, int& passes) {
    passes = (in + 255) / 256;
    const int need = ((in + 15) / 16 + passes - 1) / passes;
    ks = 16;
    for (int q : kKsOf)
        if (q >= need) {
            ks = q;
            break;
        }
    passes = (in + 16 * ks - 1) / (16 * ks);
}

int split_lr_mode(int heads, int dim) {
    if (heads == 1 || dim == 32 || dim == 64) return kLrShare;
    return dim <= 16 && 16 % dim == 0 ? kLrLane : kLrNone;
}

template <int KS, int TPB, int LR>
hipError_t launch_ks(const ProjF32Args& a, hipStream_t s, int cus) {
    const uint64_t groups = (a.tiles + TPB - 1) / TPB;
    const uint32_t gy = uint32_t((a.nob + 7) / 8);
    uint64_t gx = uint64_t(cus) / gy;
    if (gx > groups) gx = groups;
    if (gx < 1) gx = 1;
    k_proj_split<KS, TPB, LR><<<dim3(uint32_t(gx), gy), kThreads, 0, s>>>(a);
    return hipGetLastError();
}

template <int KS, int LR>
hipError_t launch_tpb(const ProjF32Args& a, hipStream_t s, int cus) {
    if (a.nob <= 2) return launch_ks<KS, 4, LR>(a, s, cus);
    if (a.nob <= 4) return launch_ks<KS, 2, LR>(a, s, cus);
    return launch_ks<KS, 1, LR>(a, s, cus);
}

template <int KS>
hipError_t launch_lr(const ProjF32Args& a, int lr, hipStream_t s, int cus) {
    if (lr == kLrShare) return launch_tpb<KS, kLrShare>(a, s, cus);
    if (lr == kLrLane) return launch_tpb<KS, kLrLane>(a, s, cus);
    return launch_tpb<KS, kLrNone>(a, s, cus);
}

}  // namespace

// The weights' factor (see the top).  w is the host copy.
float projection_split_scale(const float* w, int in, int heads, int dim) {
    const size_t count = size_t(in) * heads * dim;
    bool small = false;  // a weight whose last bits would fall below 2^-126
    for (size_t q = 0; q < count; ++q) small |= w[q] != 0.0f && std::fabs(w[q]) < 0x1p-79f;
    return small ? 0x1p24f : 0x1p-24f;
}

size_t projection_split_bytes(int in, int heads, int dim) {
    int ks, passes;
    split_passes(in, ks, passes);
    return size_t(passes) * ((heads * dim + 31) / 32) * ks * 3 * kWave * 16;
}

hipError_t launch_pack_split(const float* w, int in, int heads, int dim, float scale, void* out, hipStream_t s) {
    int ks, passes;
    split_passes(in, ks, passes);
    const int frags = passes * ((heads * dim + 31) / 32) * ks;
    k_pack_split<<<dim3(uint32_t(frags)), kWave, 0, s>>>(w, in, heads * dim, ks, scale, static_cast<uint4*>(out));
    return hipGetLastError();
}

hipError_t launch_projection_split(ProjF32Args a, hipStream_t s, int cus) {
    if (a.n == 0) return hipSuccess;
    if (a.in < 1 || a.heads < 1 || a.heads > 8 || a.dim < 1 || a.dim > 64 || a.width != a.heads * a.dim || a.zs % 4 ||
        a.zs < (a.width + 3) / 4 * 4 || a.tiles != (a.n + 31) / 32 || !a.wpk || !(a.wscale > 0.0f))
        return hipErrorInvalidValue;
    a.sum_scale = a.wscale * kScaleX;
    int ks, passes;
    split_passes(a.in, ks, passes);
    const uint4* wpk = a.wpk;
    const int lr = split_lr_mode(a.heads, a.dim);
    a.nob = (a.width + 31) / 32;
    for (int p = 0; p < passes; ++p) {
        a.k0 = 16 * ks * p;
        a.kn = a.in - a.k0 < 16 * ks ? a.in - a.k0 : 16 * ks;
        a.add = p > 0;
        const int form = p == passes - 1 ? lr : kLrNone;
        a.wpk = wpk + size_t(p) * a.nob * ks * 3 * kWave;
        hipError_t e;
        switch (ks) {
            case 2: e = launch_lr<2>(a, form, s, cus); break;
            case 4: e = launch_lr<4>(a, form, s, cus); break;
            case 6: e = launch_lr<6>(a, form, s, cus); break;
            case 7: e = launch_lr<7>(a, form, s, cus); break;
            case 8: e = launch_lr<8>(a, form, s, cus); break;
            case 12: e = launch_lr<12>(a, form, s, cus); break;
            default: e = launch_lr<16>(a, form, s, cus); break;
        }
        if (e != hipSuccess) return e;
    }
    return lr != kLrNone ? hipSuccess
                         : launch_lr_from_z(a.z, a.n, a.heads, a.dim, a.zs, a.al, a.ar, a.left, a.right, s);
}

}  // namespace gatgpu
