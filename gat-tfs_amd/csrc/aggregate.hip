// Fused exact-max softmax + CSR SpMM aggregation (transform-first GAT layer)
// for every shape but 8 heads of 32 or 64 (aggregate_vec.hip): the one-head
// output layer and hidden layers of other widths.
//
// For destination row i and head h (reference: max_prescan and
// standard_aggregate, baseline/src/baseline_standard.cpp:44-84, and finish,
// :85-97):
//   M[i,h]   = LeakyReLU(L[i,h] + max_{j in N(i)} R[j,h])      (0 for an empty row)
//   p_ij^h   = exp(LeakyReLU(L[i,h] + R[j,h]) - M[i,h])
//   den[i,h] = sum_j p_ij^h
//   out[i,h,:] = ELU?( (sum_j p_ij^h Z[j,h,:]) * (den>0 ? 1/den : 0) )
//
// A Z row is W / VEC vectors (VEC: the widest of 8/4/2/1 features that fits
// 16 bytes and lies inside one head), and a group of G lanes owns them, one
// vector a lane (rows of more than 64 vectors: VPL a lane).  A lane scores its
// own head's edges, so nothing is exchanged but the source ids (lane t of a
// group loads the id of edge t of the batch; a shuffle hands it round).  Edges
// run in batches whose loads are all in flight together, in one pass with the
// softmax online: the running maximum m, the denominator and the accumulators
// are rescaled when a batch raises m (the running-maximum form of
// implementation/src/gat_tfs_online.cpp:86-117); the final m equals
// leaky(L + max R) bit for bit, because leaky and the addition are monotone.
// Scores of -inf weigh 0 as soon as the row has a finite one.
//
// Bound: misses in flight times latency, and for rows of many edges the chain
// of batches.  So rows are split by degree (sorted, heaviest first), all in
// one launch:
//   * rows of the split table: chunks, one wave each, every chunk from its own
//     maximum; the last chunk of a row to arrive scales the partials to the
//     row's maximum and adds them (a fixed order, so results are repeatable);
//   * rows of kWaveDeg edges or more: one wave each, the wave's 64 / G groups
//     taking every (64 / G)-th batch, their partials merged at the end;
//   * lighter rows: one group each, 64 / G rows of (nearly) equal degree a wave.
// Measured against one group per row up to the split degree, and one wave (or
// block) per row with the scores exchanged through LDS for the other widths:
// 169K nodes / 2.5M edges, one head of 40: bf16 155 -> 49 us, FP32 161 -> 87;
// 60K / 1.2M, one head of 47: 95 -> 27 us; 20K / 300K, 4 heads of 16, FP32:
// 247 -> 16 us; 20K / 160K, 8 heads of 8, bf16: 56 -> 11 us; R-MAT 2^20 / 24M,
// one head of 16: 710 -> 355 us.
#include "internal.hpp"

namespace gatgpu {
namespace {

constexpr int kThreads = 256;
constexpr int kWavesPerBlock = kThreads / kWave;
constexpr uint32_t kPartStride = 512 + 16;  // sums, denominators of the heads, maxima of the heads

template <int BYTES>
struct RawOf;
template <>
struct RawOf<16> { using type = uint4; };
template <>
struct RawOf<8> { using type = uint2; };
template <>
struct RawOf<4> { using type = uint32_t; };
template <>
struct RawOf<2> { using type = uint16_t; };

// Source of R: its own array [n][K]; the last four bytes of the (one-head) Z
// row; or recomputed from a one-head row of 64 bf16 features as the projection
// wrote it: lane sub takes the FMA chain of its 8 features with aR, and the
// group adds ((p0 + p1) + (p2 + p3)) + ((p4 + p5) + (p6 + p7)) by xor shuffles.
enum { kRArray = 0, kRInRow = 1, kRFromZ = 2 };

template <class ZT_, int VEC_, int G_, int VPL_, int RM_>
struct Grp {
    using ZT = ZT_;
    static constexpr int VEC = VEC_, G = G_, VPL = VPL_, RM = RM_;
    static constexpr int GPW = kWave / G;                // groups per wave
    static constexpr int B = VPL == 1 ? 8 : 8 / VPL < 2 ? 2 : 8 / VPL;  // edges per batch
    using Raw = typename RawOf<VEC * int(sizeof(ZT))>::type;
    static_assert(RM == kRArray || VPL == 1, "one vector a lane");
    static_assert(B <= G, "a batch's ids come from one group");
};

template <class ZT>
struct GrpArgs {
    const uint64_t* prow;
    const uint32_t* pcol;
    const uint32_t* perm;
    const float* L;
    const float* R;
    const ZT* Z;
    int K, dim, W, zs;
    bool hidden, round_bf16;
    float* mx;
    float* den;
    float* out32;
    uint16_t* outbf;
    uint64_t n, e;
    uint64_t light, rows;   // sorted positions [0, light): a group each; [light, rows): a wave each
    uint64_t chunks;
    const uint32_t* chunk_k;
    const uint32_t* chunk_first;
    uint32_t chunk_edges;
    float* part;
    uint32_t* counter;
    const uint32_t* operm;  // output row of sorted position k: operm[k] (null: the node index)
    const float* ar;        // aR [W] when R is recomputed from the gathered rows
    int os;                 // out32 row stride: W, or G * VEC with operm (whole padded rows)
};

template <class ZT, int VEC, class Raw>
__device__ inline void unpack(const Raw& v, float (&f)[VEC]) {
    constexpr int WORDS = int(sizeof(Raw)) / 4;
    if constexpr (WORDS == 0) {
        f[0] = bf16_widen(v);
    } else {
        uint32_t w[WORDS];
        __builtin_memcpy(w, &v, sizeof(Raw));
        if constexpr (sizeof(ZT) == 4) {
#pragma unroll
            for (int q = 0; q < VEC; ++q) f[q] = __builtin_bit_cast(float, w[q]);
        } else {
#pragma unroll
            for (int q = 0; q < WORDS; ++q) {
                f[2 * q] = __builtin_bit_cast(float, w[q] << 16);
                f[2 * q + 1] = __builtin_bit_cast(float, w[q] & 0xffff0000u);
            }
        }
    }
}

// What a lane holds of its row: its vectors' offsets and heads, and the
// softmax state of each.
template <class C>
struct Lane {
    int sub, gbase;
    int off[C::VPL];    // first feature of the lane's vector v (past W: no features of its own)
    int load[C::VPL];   // the vector it loads (its own, or the row's last)
    int head[C::VPL];
    bool lead[C::VPL];  // the head's first vector: stores the head's max and den
    float Li[C::VPL], m[C::VPL], d[C::VPL];
    float acc[C::VPL][C::VEC];
    float arl[C::VEC];

    __device__ inline void init(const GrpArgs<typename C::ZT>& a, int lane) {
        sub = lane % C::G;
        gbase = lane - sub;
        const int nvec = (a.W + C::VEC - 1) / C::VEC;
#pragma unroll
        for (int v = 0; v < C::VPL; ++v) {
            const int vec = sub + v * C::G;
            const int own = vec < nvec ? vec : nvec - 1;
            off[v] = vec * C::VEC;
            load[v] = (C::RM == kRInRow ? vec : own) * C::VEC;
            head[v] = own * C::VEC / a.dim;
            lead[v] = vec < nvec && head[v] * a.dim == off[v];
        }
        if constexpr (C::RM == kRFromZ) {
#pragma unroll
            for (int x = 0; x < C::VEC; ++x) arl[x] = a.ar[off[0] + x];
        }
    }
    __device__ inline void start(const GrpArgs<typename C::ZT>& a, uint32_t i) {
#pragma unroll
        for (int v = 0; v < C::VPL; ++v) {
            Li[v] = a.L[uint64_t(i) * a.K + head[v]];
            m[v] = kNoMax;
            d[v] = 0.0f;
#pragma unroll
            for (int x = 0; x < C::VEC; ++x) acc[v][x] = 0.0f;
        }
    }
};

// One batch of NB edges: all loads, then scores, the rescale and the sums.  Only
// the first cnt of them (SURE at least) are real.  The others read the row's
// last source again (the batch loads it anyway) and add 0 * 0, whatever it holds:
// a weight of 0 alone would make NaN of an infinity.
template <class C, int NB, int SURE>
__device__ inline void batch(const GrpArgs<typename C::ZT>& a, Lane<C>& s, uint32_t j, int cnt) {
    using ZT = typename C::ZT;
    using Raw = typename C::Raw;
    Raw raw[NB][C::VPL];
    float r[NB][C::VPL];
#pragma unroll
    for (int t = 0; t < NB; ++t) {
        const uint32_t jt = __shfl(j, s.gbase + t);
        const ZT* z = a.Z + uint64_t(jt) * a.zs;
#pragma unroll
        for (int v = 0; v < C::VPL; ++v) {
            raw[t][v] = *reinterpret_cast<const Raw*>(z + s.load[v]);
            if constexpr (C::RM == kRArray) r[t][v] = a.R[uint64_t(jt) * a.K + s.head[v]];
        }
    }
    float mb[C::VPL];
#pragma unroll
    for (int v = 0; v < C::VPL; ++v) mb[v] = -INFINITY;
#pragma unroll
    for (int t = 0; t < NB; ++t) {
        if constexpr (C::RM == kRInRow) {
            uint32_t w[4];
            __builtin_memcpy(w, &raw[t][0], 16);
            r[t][0] = __builtin_bit_cast(float, __shfl(w[3], s.gbase + C::G - 1));
        }
        if constexpr (C::RM == kRFromZ) {
            float f[C::VEC];
            unpack<ZT, C::VEC>(raw[t][0], f);
            float pr = 0.0f;
#pragma unroll
            for (int x = 0; x < C::VEC; ++x) pr = __builtin_fmaf(f[x], s.arl[x], pr);
            pr += __shfl_xor(pr, 1);
            pr += __shfl_xor(pr, 2);
            r[t][0] = pr + __shfl_xor(pr, 4);
        }
#pragma unroll
        for (int v = 0; v < C::VPL; ++v) {
            r[t][v] = t < SURE || t < cnt ? leaky(s.Li[v] + r[t][v]) : -INFINITY;
            mb[v] = fmaxf(mb[v], r[t][v]);
        }
    }
    if constexpr (C::RM == kRFromZ) {
        // Unpack the rows again below rather than keep the unpacked rows live.
#pragma unroll
        for (int t = 0; t < NB; ++t) {
            uint32_t w[4];
            __builtin_memcpy(w, &raw[t][0], 16);
            asm volatile("" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]));
            __builtin_memcpy(&raw[t][0], w, 16);
        }
    }
#pragma unroll
    for (int v = 0; v < C::VPL; ++v) {
        const float mn = fmaxf(s.m[v], mb[v]);
        const float sc = exp_w(s.m[v] - mn);  // 0 on the first batch (m = kNoMax)
        s.m[v] = mn;
        s.d[v] *= sc;
#pragma unroll
        for (int x = 0; x < C::VEC; ++x) s.acc[v][x] *= sc;
    }
#pragma unroll
    for (int t = 0; t < NB; ++t) {
#pragma unroll
        for (int v = 0; v < C::VPL; ++v) {
            const bool real = t < SURE || t < cnt;
            const float p = real ? exp_w(r[t][v] - s.m[v]) : 0.0f;
            s.d[v] += p;
            float f[C::VEC];
            unpack<ZT, C::VEC>(real ? raw[t][v] : Raw{}, f);
#pragma unroll
            for (int x = 0; x < C::VEC; ++x) s.acc[v][x] += p * f[x];
        }
    }
}

// Batches start, start + step, ... of the `total` edges at beg.  Groups of a
// wave may run different trip counts (their shuffles stay inside the group).
// The next batch's ids are requested before this one's rows are used.
template <class C>
__device__ inline void edges(const GrpArgs<typename C::ZT>& a, Lane<C>& s, uint64_t beg, uint32_t total,
                             uint32_t start, uint32_t step) {
    if (start >= total) return;
    const uint32_t* ids = a.pcol + beg;
    const uint32_t lane_t = s.sub < C::B ? uint32_t(s.sub) : 0u;
    auto id_at = [&](uint32_t q) { return ids[q < total ? q : total - 1]; };
    uint32_t next = id_at(start + lane_t);
    for (uint32_t done = start;; done += step) {
        const uint32_t left = total - done;
        const int cnt = left < uint32_t(C::B) ? int(left) : C::B;
        const uint32_t j = next;  // past the end: the last source
        next = id_at(done + step + lane_t);
        // Half a batch's loads where half hold the rest of the row: most rows
        // of a skewed graph have a few edges only.
        if (left > uint32_t(C::B) / 2) batch<C, C::B, C::B / 2 + 1>(a, s, j, cnt);
        else batch<C, C::B / 2, 1>(a, s, j, cnt);
        if (left <= step) return;  // (not done + step < total: that sum may pass 2^32)
    }
}

// Partials of the wave's groups into every group: m to the common maximum, the
// sums scaled to it and added.  Groups without edges (m = kNoMax, sums 0) add 0.
template <class C>
__device__ inline void merge_groups(Lane<C>& s) {
#pragma unroll
    for (int off = C::G; off < kWave; off <<= 1) {
#pragma unroll
        for (int v = 0; v < C::VPL; ++v) {
            const float mo = __shfl_xor(s.m[v], off), dn = __shfl_xor(s.d[v], off);
            const float mn = fmaxf(s.m[v], mo);
            const float sa = s.m[v] == mn ? 1.0f : exp_w(s.m[v] - mn), so = mo == mn ? 1.0f : exp_w(mo - mn);
            s.m[v] = mn;
            s.d[v] = s.d[v] * sa + dn * so;
#pragma unroll
            for (int x = 0; x < C::VEC; ++x) s.acc[v][x] = s.acc[v][x] * sa + __shfl_xor(s.acc[v][x], off) * so;
        }
    }
}

// Normalise, activate and store the row: max and den at node i, features at
// output row o.  any: the row has edges.
template <class C>
__device__ inline void finish(const GrpArgs<typename C::ZT>& a, const Lane<C>& s, uint32_t i, uint32_t o, bool any) {
    constexpr int V = C::VEC;
#pragma unroll
    for (int v = 0; v < C::VPL; ++v) {
        const bool none = any && no_softmax(s.m[v], s.d[v]);
        const float d = none ? NAN : s.d[v];
        if (s.lead[v]) {
            a.mx[uint64_t(i) * a.K + s.head[v]] = none ? -INFINITY : any ? s.m[v] : 0.0f;
            a.den[uint64_t(i) * a.K + s.head[v]] = d;
        }
        const float scale = none ? NAN : d > 0.0f ? 1.0f / d : 0.0f;
        float y[V];
#pragma unroll
        for (int x = 0; x < V; ++x) {
            y[x] = s.acc[v][x] * scale;
            if (a.hidden) y[x] = elu(y[x]);
            if (a.round_bf16) y[x] = bf16_widen(bf16_hw(y[x]));
        }
        const int f = s.off[v];
        if (a.out32 && a.os != a.W) {
            // Padded FP32 rows (the logits in original node order): each lane
            // stores its pieces whole, zeros past W, so the scattered rows are
            // written as whole lines.
            float* dst = a.out32 + uint64_t(o) * a.os + f;
#pragma unroll
            for (int x = 0; x < V; ++x) y[x] = f + x < a.W ? y[x] : 0.0f;
            if constexpr (V % 4 == 0) {
#pragma unroll
                for (int x = 0; x < V; x += 4)
                    *reinterpret_cast<float4*>(dst + x) = make_float4(y[x], y[x + 1], y[x + 2], y[x + 3]);
            }
            continue;
        }
        if (f >= a.W) continue;
        const bool whole = f + V <= a.W && a.W % V == 0;  // then rows start at multiples of V
        if (a.out32) {
            float* dst = a.out32 + uint64_t(o) * a.W + f;
            if (V % 4 == 0 && whole) {
                if constexpr (V % 4 == 0)
#pragma unroll
                    for (int x = 0; x < V; x += 4)
                        *reinterpret_cast<float4*>(dst + x) = make_float4(y[x], y[x + 1], y[x + 2], y[x + 3]);
            } else {
#pragma unroll
                for (int x = 0; x < V; ++x)
                    if (f + x < a.W) dst[x] = y[x];
            }
        }
        if (a.outbf) {
            uint16_t* dst = a.outbf + uint64_t(o) * a.W + f;
            if (V % 4 == 0 && whole) {
                if constexpr (V % 4 == 0)
#pragma unroll
                    for (int x = 0; x < V; x += 4)
                        *reinterpret_cast<uint2*>(dst + x) = make_uint2(bf16x2(y[x], y[x + 1]), bf16x2(y[x + 2], y[x + 3]));
            } else {
#pragma unroll
                for (int x = 0; x < V; ++x)
                    if (f + x < a.W) dst[x] = bf16_hw(y[x]);
            }
        }
    }
}

template <class C>
__global__ void __launch_bounds__(kThreads) k_agg_rows(GrpArgs<typename C::ZT> a) {
    const int w = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const uint64_t wave = uint64_t(blockIdx.x) * kWavesPerBlock + w;
    const int g = lane / C::G;
    Lane<C> s;
    s.init(a, lane);
    const uint64_t heavy = a.rows - a.light;
    if (wave < a.chunks + heavy) {
        // ---------------- one chunk of a split row, or one whole row, per wave
        const bool chunk = wave < a.chunks;
        const uint64_t k = chunk ? a.chunk_k[wave] : a.rows - 1 - (wave - a.chunks);
        const uint64_t rbeg = a.prow[k], rend = a.prow[k + 1];
        const uint32_t i = a.perm[k];
        if (i >= a.n || rbeg > rend || rend > a.e) return;  // schedule invariants
        uint64_t beg = rbeg, end = rend;
        uint32_t first = 0, nch = 1;
        if (chunk) {
            first = a.chunk_first[wave];
            nch = uint32_t((rend - rbeg + a.chunk_edges - 1) / a.chunk_edges);
            beg = rbeg + uint64_t(wave - first) * a.chunk_edges;
            end = beg + a.chunk_edges < rend ? beg + a.chunk_edges : rend;
        }
        s.start(a, i);
        edges(a, s, beg, uint32_t(end - beg), uint32_t(g * C::B), uint32_t(C::GPW * C::B));
        merge_groups(s);
        if (chunk) {
            float* part = a.part + wave * kPartStride;
            if (g == 0) {
#pragma unroll
                for (int v = 0; v < C::VPL; ++v) {
                    if (s.off[v] >= a.W) continue;
#pragma unroll
                    for (int x = 0; x + 1 < C::VEC; x += 2)
                        store_coherent2(part + s.off[v] + x, s.acc[v][x], s.acc[v][x + 1]);
                    if constexpr (C::VEC == 1) store_coherent(part + s.off[v], s.acc[v][0]);
                    if (s.lead[v]) {
                        store_coherent(part + 512 + s.head[v], s.d[v]);
                        store_coherent(part + 520 + s.head[v], s.m[v]);
                    }
                }
            }
            if (arrive(a.counter + first, lane) + 1 != nch) return;
            // The row's maximum, then the groups take every GPW-th chunk each.
            const float* base = a.part + uint64_t(first) * kPartStride;
#pragma unroll
            for (int v = 0; v < C::VPL; ++v) {
                float M = -INFINITY;
#pragma unroll 16
                for (uint32_t q = 0; q < nch; ++q)
                    M = fmaxf(M, load_coherent(base + uint64_t(q) * kPartStride + 520 + s.head[v]));
                s.m[v] = M;
                s.d[v] = 0.0f;
#pragma unroll
                for (int x = 0; x < C::VEC; ++x) s.acc[v][x] = 0.0f;
                const int f = s.off[v] < a.W ? s.off[v] : 0;
#pragma unroll 4
                for (uint32_t q = uint32_t(g); q < nch; q += C::GPW) {
                    const float* p = base + uint64_t(q) * kPartStride;
                    const float mq = load_coherent(p + 520 + s.head[v]);
                    const float sc = mq == M ? 1.0f : exp_w(mq - M);
                    s.d[v] += load_coherent(p + 512 + s.head[v]) * sc;
#pragma unroll
                    for (int x = 0; x + 1 < C::VEC; x += 2) {
                        const float2 t = load_coherent2(p + f + x);
                        s.acc[v][x] += t.x * sc;
                        s.acc[v][x + 1] += t.y * sc;
                    }
                    if constexpr (C::VEC == 1) s.acc[v][0] += load_coherent(p + f) * sc;
                }
            }
            merge_groups(s);
            if (lane == 0) a.counter[first] = 0;
        }
        if (g == 0) finish(a, s, i, a.operm ? a.operm[k] : i, rend > rbeg);
        return;
    }
    // ---------------- 64 / G whole rows per wave, heaviest first
    const uint64_t idx = (wave - a.chunks - heavy) * C::GPW + g;
    if (idx >= a.light) return;  // whole groups exit; no wave-wide exchange follows
    const uint64_t k = a.light - 1 - idx;
    const uint32_t i = a.perm[k];
    const uint64_t beg = a.prow[k], end = a.prow[k + 1];
    if (i >= a.n || beg > end || end > a.e) return;
    s.start(a, i);
    edges(a, s, beg, uint32_t(end - beg), 0u, uint32_t(C::B));
    finish(a, s, i, a.operm ? a.operm[k] : i, end > beg);
}

template <class ZT, int VEC, int G, int VPL, int RM>
hipError_t run(const AggArgs& g, const RowBins& bins, const SplitTable& t, hipStream_t s) {
    using C = Grp<ZT, VEC, G, VPL, RM>;
    const int W = g.heads * g.dim;
    GrpArgs<ZT> a{};
    a.prow = g.prow;
    a.pcol = g.pcol;
    a.perm = g.perm;
    a.L = g.left;
    a.R = g.right;
    a.Z = static_cast<const ZT*>(g.feat);
    a.K = g.heads;
    a.dim = g.dim;
    a.W = W;
    a.zs = g.fstride;
    a.hidden = g.hidden;
    a.round_bf16 = g.round_bf16;
    a.mx = g.mx;
    a.den = g.den;
    a.out32 = g.out32;
    a.outbf = g.outbf;
    a.n = g.n;
    a.e = g.e;
    a.rows = bins.split_begin;
    // One group spans the wave: every row is a wave's.
    a.light = C::GPW == 1 ? 0 : bins.wave_begin < bins.split_begin ? bins.wave_begin : bins.split_begin;
    a.chunks = t.chunks;
    a.chunk_k = t.chunk_k;
    a.chunk_first = t.chunk_first;
    a.chunk_edges = t.chunk_edges;
    a.part = t.part;
    a.counter = t.counter;
    a.operm = g.out_perm;
    a.ar = g.ar;
    a.os = g.out_perm && g.ostride ? g.ostride : W;
    if (a.os != W && (!a.operm || a.outbf || VPL != 1 || VEC % 4 != 0 || a.os != G * VEC)) return hipErrorInvalidValue;
    if (RM == kRInRow && (g.heads != 1 || g.fstride != G * VEC || W > g.fstride - 4 / int(sizeof(ZT)))) return hipErrorInvalidValue;
    if (RM == kRFromZ && (!g.ar || g.heads != 1 || g.dim != 64 || g.fstride != 64)) return hipErrorInvalidValue;
    const uint64_t waves = a.chunks + (a.rows - a.light) + (a.light + C::GPW - 1) / C::GPW;
    if (!waves) return hipSuccess;
    k_agg_rows<C><<<dim3(uint32_t((waves + kWavesPerBlock - 1) / kWavesPerBlock)), kThreads, 0, s>>>(a);
    return hipGetLastError();
}

// Lanes for the row's vectors: a group of 8 to 64, beyond that VPL vectors each.
template <class ZT, int VEC>
hipError_t run_lanes(const AggArgs& g, const RowBins& bins, const SplitTable& t, hipStream_t s) {
    const int nvec = (g.heads * g.dim + VEC - 1) / VEC;
    if (nvec <= 8) return run<ZT, VEC, 8, 1, kRArray>(g, bins, t, s);
    if (nvec <= 16) return run<ZT, VEC, 16, 1, kRArray>(g, bins, t, s);
    if (nvec <= 32) return run<ZT, VEC, 32, 1, kRArray>(g, bins, t, s);
    if (nvec <= 64) return run<ZT, VEC, 64, 1, kRArray>(g, bins, t, s);
    if constexpr (VEC <= 4)
        if (nvec <= 128) return run<ZT, VEC, 64, 2, kRArray>(g, bins, t, s);
    if constexpr (VEC <= 2)
        if (nvec <= 256) return run<ZT, VEC, 64, 4, kRArray>(g, bins, t, s);
    if constexpr (VEC <= 1)
        if (nvec <= 512) return run<ZT, VEC, 64, 8, kRArray>(g, bins, t, s);
    return hipErrorInvalidValue;
}

}  // namespace

int k1_out_stride(bool feat_bf16, int W) { return feat_bf16 || W > 32 ? 64 : 32; }

hipError_t launch_aggregate_tf(const AggArgs& a, const RowBins& bins, const SplitTable& split,
                               hipStream_t s) {
    if (a.heads < 1 || a.heads > 8 || a.dim < 1 || a.dim > 64) return hipErrorInvalidValue;
    if (aggregate_vec_supported(a)) return launch_aggregate_vec(a, bins, split, s);
    // Z rows are 16-byte aligned (their stride is a multiple of 16 bytes), so a
    // vector of VEC features at a multiple of VEC is aligned to its own size.
    if (a.fstride % (a.feat_bf16 ? 8 : 4) || a.fstride < a.heads * a.dim) return hipErrorInvalidValue;
    if (a.heads == 1) {  // a vector may reach past W, into the row's padding
        if (!a.feat_bf16)
            return a.dim <= 32 ? run<float, 4, 8, 1, kRArray>(a, bins, split, s)
                               : run<float, 4, 16, 1, kRArray>(a, bins, split, s);
        if (a.r_in_feat) return run<uint16_t, 8, 8, 1, kRInRow>(a, bins, split, s);
        if (a.r_from_z) return run<uint16_t, 8, 8, 1, kRFromZ>(a, bins, split, s);
        return run<uint16_t, 8, 8, 1, kRArray>(a, bins, split, s);
    }
    if (a.feat_bf16) {
        if (a.dim % 8 == 0) return run_lanes<uint16_t, 8>(a, bins, split, s);
        if (a.dim % 4 == 0) return run_lanes<uint16_t, 4>(a, bins, split, s);
        if (a.dim % 2 == 0) return run_lanes<uint16_t, 2>(a, bins, split, s);
        return run_lanes<uint16_t, 1>(a, bins, split, s);
    }
    if (a.dim % 4 == 0) return run_lanes<float, 4>(a, bins, split, s);
    if (a.dim % 2 == 0) return run_lanes<float, 2>(a, bins, split, s);
    return run_lanes<float, 1>(a, bins, split, s);
}

}  // namespace gatgpu
