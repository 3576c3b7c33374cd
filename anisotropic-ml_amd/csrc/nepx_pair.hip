// Pair kernels: descriptor forward, MFMA energy network, adjoint, and the
// fused step kernel.  See nepx_desc.h and nepx_ffnn.h for the math and layouts.
#include "nepx_pairk.h"

#include <string.h>

namespace nepx {

// Descriptor row of one pair (or cloud), one pass over the sites per l range.
template <class Cfg, class Sites, class Row>
__device__ __forceinline__ void desc_forward_sites(const Sites& sites, Row&& G) {
    float grad[Cfg::NRAD + 1];
    for_passes<Cfg>([&](auto range, auto first) {
        using LR = decltype(range);
        float A[Cfg::NANG + 1][LR::N];
        accumulate_sites<Cfg, LR, decltype(first)::value>(sites, grad, A);
        desc_finish<Cfg, LR>(A, G);
        if constexpr (decltype(first)::value) {
#pragma unroll
            for (int n = 0; n <= Cfg::NRAD; ++n) G[n] = grad[n];
        }
    });
}

template <class Cfg, class Row>
__device__ __forceinline__ void desc_forward(const nepx_pair_model& m, const PairIn& g, Row&& G) {
    desc_forward_sites<Cfg>(PairSites<Cfg>{m, g, 1.f / m.r_nep}, G);
}

// Adjoint over every l range, recomputing each range's forward accumulators.
template <class Cfg>
__device__ __forceinline__ void adjoint_all(const nepx_pair_model& m, const PairIn& g, const float (&dG)[Cfg::D],
                                            AdjAcc& acc) {
    for_passes<Cfg>([&](auto range, auto first) {
        using LR = decltype(range);
        float grad[Cfg::NRAD + 1];
        float A[Cfg::NANG + 1][LR::N];
        desc_accumulate<Cfg, LR, false>(m, g, grad, A);
        desc_adjoint<Cfg, LR, decltype(first)::value>(m, g, dG, A, acc);
    });
}

// ---------------------------------------------------------------------------
template <class Cfg>
__global__ __launch_bounds__(kBlock) void k_desc_fwd(nepx_pair_model m, const float4* __restrict__ qf,
                                                     const int32_t* __restrict__ pi,
                                                     const int32_t* __restrict__ pj,
                                                     const float4* __restrict__ pt,
                                                     const int32_t* __restrict__ np_dev, int64_t maxp,
                                                     float* __restrict__ G) {
    const int P = n_pairs(np_dev, maxp);
    for (int idx = blockIdx.x * kBlock + threadIdx.x; idx < P; idx += gridDim.x * kBlock) {
        float4 qi, qj, t;
        load_pair(qf, pi, pj, pt, idx, qi, qj, t);
        const PairIn g = pair_in<Cfg>(m, qi, qj, t.x, t.y, t.z);
        if constexpr (Cfg::ONE_PASS) {
            float Gr[Cfg::D];
            desc_forward<Cfg>(m, g, Gr);
            store_row<Cfg>(G + (size_t)idx * Cfg::D, Gr);
        } else {  // several passes: each writes its entries (no D-float row held in registers)
            desc_forward<Cfg>(m, g, G + (size_t)idx * Cfg::D);
        }
    }
}

// few: up to this many pairs are left to the four-lane kernel launched with it (0: this one takes them all).
template <class Cfg>
__global__ __launch_bounds__(kBlock) NEPX_ADJ_ATTR void k_adjoint(nepx_pair_model m, const float4* __restrict__ qf,
                                                    const int32_t* __restrict__ pi,
                                                    const int32_t* __restrict__ pj,
                                                    const float4* __restrict__ pt,
                                                    const int32_t* __restrict__ np_dev, int64_t maxp, int few,
                                                    const float* __restrict__ dEdG,
                                                    const float* __restrict__ E, float clip,
                                                    float* __restrict__ out) {
    const int P = n_pairs(np_dev, maxp);
    if (P <= few) return;
    for (int idx = blockIdx.x * kBlock + threadIdx.x; idx < P; idx += gridDim.x * kBlock) {
        float4 qi, qj, t;
        load_pair(qf, pi, pj, pt, idx, qi, qj, t);
        const PairIn g = pair_in<Cfg>(m, qi, qj, t.x, t.y, t.z);
        float dG[Cfg::D];
        load_row<Cfg>(dEdG + (size_t)idx * Cfg::D, dG);
        AdjAcc acc;
        adjoint_all<Cfg>(m, g, dG, acc);
        store_out(out, idx, adj_finish<Cfg>(acc), E ? E[idx] : 0.f, clip);
    }
}

// Multi-pass shapes with few pairs: the l-range passes of a pair run on different waves of a block
// (four waves, one per SIMD, as the register-heavy passes need; 64 pairs per block).  Wave w takes
// passes w and NP - 1 - w (the cheap low-l passes with the dear high-l ones).  The forward writes
// each pass's descriptor entries as k_desc_fwd does; the adjoint leaves each pass's per-body sums
// in LDS and sums them in pass order, so both give k_desc_fwd's and k_adjoint's results bit for
// bit (every pass's sums start from zero, as k_adjoint's running sums do not become -0).
// The forward can also be launched with one pass a block (blockIdx.y, high l first; 64 threads): the
// time of few pairs is the longest wave's, here one pass instead of two.
template <class Cfg>
constexpr int pass_waves() {
    constexpr int np = n_passes(Cfg::NANG, Cfg::LMAX);
    return np < 4 ? np : 4;
}
template <class Cfg>
__device__ __forceinline__ int pass_owner(int p) {
    constexpr int np = n_passes(Cfg::NANG, Cfg::LMAX), w = pass_waves<Cfg>();
    return p < w ? p : (np - 1 - p < w ? np - 1 - p : p % w);
}

template <class Cfg>
__global__ __launch_bounds__(64 * pass_waves<Cfg>()) NEPX_ADJ_ATTR void k_desc_fwd_passes(
    nepx_pair_model m, const float4* __restrict__ qf, const int32_t* __restrict__ pi, const int32_t* __restrict__ pj,
    const float4* __restrict__ pt, const int32_t* __restrict__ np_dev, int64_t maxp, float* __restrict__ G) {
    const int P = n_pairs(np_dev, maxp);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool alone = gridDim.y > 1;  // one pass a block
    const int pass = (int)gridDim.y - 1 - (int)blockIdx.y;
    for (int idx = blockIdx.x * 64 + (threadIdx.x & 63); idx < P; idx += gridDim.x * 64) {
        float4 qi, qj, t;
        load_pair(qf, pi, pj, pt, idx, qi, qj, t);
        const PairIn g = pair_in<Cfg>(m, qi, qj, t.x, t.y, t.z);
        const PairSites<Cfg> sites{m, g, 1.f / m.r_nep};
        float* row = G + (size_t)idx * Cfg::D;
        int k = 0;
        for_passes<Cfg>([&](auto range, auto first) {
            const bool mine = alone ? k == pass : pass_owner<Cfg>(k) == wave;
            ++k;
            if (mine) {
                using LR = decltype(range);
                float grad[Cfg::NRAD + 1];
                float A[Cfg::NANG + 1][LR::N];
                accumulate_sites<Cfg, LR, decltype(first)::value>(sites, grad, A);
                desc_finish<Cfg, LR>(A, row);
                if constexpr (decltype(first)::value) {
#pragma unroll
                    for (int n = 0; n <= Cfg::NRAD; ++n) row[n] = grad[n];
                }
            }
        });
    }
}

template <class Cfg>
__global__ __launch_bounds__(64 * pass_waves<Cfg>()) NEPX_ADJ_ATTR void k_adjoint_passes(
    nepx_pair_model m, const float4* __restrict__ qf, const int32_t* __restrict__ pi, const int32_t* __restrict__ pj,
    const float4* __restrict__ pt, const int32_t* __restrict__ np_dev, int64_t maxp,
    const float* __restrict__ dEdG, const float* __restrict__ E, float clip, float* __restrict__ out) {
    constexpr int NP = n_passes(Cfg::NANG, Cfg::LMAX);
    __shared__ float part[NP][12][64];  // per pass: G0, T0, G1, T1 (xyz) of the block's 64 pairs
    const int P = n_pairs(np_dev, maxp);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int base = blockIdx.x * 64; base < P; base += gridDim.x * 64) {  // uniform over the block
        const int idx = base + lane;
        const bool valid = idx < P;
        AdjAcc arms;  // pass 0 sets the pair's arm sums
        if (valid) {
            float4 qi, qj, t;
            load_pair(qf, pi, pj, pt, idx, qi, qj, t);
            const PairIn g = pair_in<Cfg>(m, qi, qj, t.x, t.y, t.z);
            const float(&dG)[Cfg::D] = *reinterpret_cast<const float(*)[Cfg::D]>(dEdG + (size_t)idx * Cfg::D);
            int k = 0;
            for_passes<Cfg>([&](auto range, auto first) {
                const int p = k++;
                if (pass_owner<Cfg>(p) == wave) {
                    using LR = decltype(range);
                    float grad[Cfg::NRAD + 1];
                    float A[Cfg::NANG + 1][LR::N];
                    AdjAcc a;
                    desc_accumulate<Cfg, LR, false>(m, g, grad, A);
                    desc_adjoint<Cfg, LR, decltype(first)::value>(m, g, dG, A, a);
                    const float v[12] = {a.G0x, a.G0y, a.G0z, a.T0x, a.T0y, a.T0z,
                                         a.G1x, a.G1y, a.G1z, a.T1x, a.T1y, a.T1z};
#pragma unroll
                    for (int c = 0; c < 12; ++c) part[p][c][lane] = v[c];
                    if constexpr (decltype(first)::value) arms = a;
                }
            });
        }
        __syncthreads();
        if (wave == 0 && valid) {  // pass 0 runs on wave 0, so `arms` is set here
            AdjAcc acc;
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                acc.G0x += part[p][0][lane]; acc.G0y += part[p][1][lane]; acc.G0z += part[p][2][lane];
                acc.T0x += part[p][3][lane]; acc.T0y += part[p][4][lane]; acc.T0z += part[p][5][lane];
                acc.G1x += part[p][6][lane]; acc.G1y += part[p][7][lane]; acc.G1z += part[p][8][lane];
                acc.T1x += part[p][9][lane]; acc.T1y += part[p][10][lane]; acc.T1z += part[p][11][lane];
            }
            acc.A0x = arms.A0x; acc.A0y = arms.A0y; acc.A0z = arms.A0z;
            acc.A1x = arms.A1x; acc.A1y = arms.A1y; acc.A1z = arms.A1z;
            store_out(out, idx, adj_finish<Cfg>(acc), E ? E[idx] : 0.f, clip);
        }
        __syncthreads();  // the sums are read before the next pairs' passes write them
    }
}

template <class N, int NT, int PREC, int ACT>
__global__ __launch_bounds__(kBlock) void k_ffnn(const float* __restrict__ Wg, const void* __restrict__ Whg,
                                                 float en_min, float scale, int D, const float* __restrict__ G,
                                                 const int32_t* __restrict__ np_dev, int64_t maxp,
                                                 float* __restrict__ E, float* __restrict__ dEdG) {
    using R = NetRun<N, NT, PREC>;
    __shared__ __attribute__((aligned(16))) float wl[weight_lds_floats<N, PREC>()];
    const float* W;
    const void* WH;
    stage_net<N, PREC>(wl, Wg, Whg, W, WH);
    const int P = n_pairs(np_dev, maxp);
    const int lane = threadIdx.x & 63;
    const int nt = (P + 16 * NT - 1) / (16 * NT);
    const int wave = (blockIdx.x * kBlock + threadIdx.x) >> 6;
    const int nwaves = (gridDim.x * kBlock) >> 6;
    for (int tile = wave; tile < nt; tile += nwaves) {
        v4f gin[NT][R::IC];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int p = (tile * NT + t) * 16 + (lane & 15);
            gather_chunks<R::IC>(G + (size_t)p * D, p < P, D, gin[t]);
        }
        v4f dg[NT][N::MD];
        float y[NT];
        R::run(W, WH, ACT, gin, scale, dg, y);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int p = (tile * NT + t) * 16 + (lane & 15);
            if (p < P && lane < 16) E[p] = en_min + scale * y[t];
            scatter_chunks<N::MD>(dEdG + (size_t)p * D, p < P, D, dg[t]);
        }
    }
}

// FP32 network with the layers' unit blocks spread over a block's waves.  Wave w computes 16-unit
// block w of every hidden layer and of every backward delta for the block's NT tiles of 16 pairs, over
// all k-steps; the layer outputs go through LDS to the next layer's B operands.  The bound is the FP32
// matrix rate once a weight operand read from L2 (256 bytes for the wave) serves several products:
// one wave per tile read the whole network (780 KB for 121 -> 150 x 4) for every 16 pairs.  NT tiles
// share each operand read, and the operands are loaded kDepth chunks ahead, across the layers'
// barriers, so that L2 latency is covered even with one tile per block.  Every accumulator takes the
// same products in the same order as ffnn_tiles, and the output sum is formed the same way, so E and
// dE/dG equal k_ffnn's bit for bit, for any NT.  121 -> 150 x 4: 241 rows 46 -> 18 us, 100,001 rows
// 1,960 -> 355 us, 400,003 rows 6,980 -> 1,295 us (120 TFLOP/s of padded products, 0.81 of the FP32 rate a
// large matrix product reaches).
//
// NT: four tiles for ReLU, which keeps one bit per hidden unit for the backward pass; two for deep tanh
// networks, which keep the activations; one for few pairs.
//
// WV waves per block.  With fewer waves than unit blocks (WV = 8 for the ten of a 160-wide layer) each wave
// takes its block for the NT tiles and one (block, tile) of the EX blocks left over: four tiles make five
// equal units for each of eight waves, two per SIMD, where ten waves fall 3, 3, 2, 2 on the SIMDs and wait
// for the fuller ones at every layer's barrier (100,001 rows of 121 -> 150 x 4: 355 against 406 us).  Few
// tiles take a wave per unit block, the shorter chain, and so do groups of two, which leave four units for
// eight waves.
template <class N, int ACT, int WV, int NT_>
struct SpreadNet {
    static constexpr int MT = N::MT, NL = N::NL, BLOCK = 64 * WV, EX = MT - WV;
    static_assert(EX >= 0 && N::MD <= WV, "one dE/dG block per wave at most");
    static constexpr int NT = NT_;
    static_assert(EX * NT <= WV || EX == 0, "one left-over unit per wave");
    static constexpr int BLOCKS_PER_CU = 2;  // LDS and registers allow two; each hides the other's barriers
    static constexpr int WAVES_PER_SIMD = (BLOCKS_PER_CU * WV + 3) / 4;
    // products in order: forward layers 0..NL-1, backward layers NL-1..0; chunks of four k-steps
    static constexpr int chunks(int q) { return (q == 0 ? N::KD : N::KH) / 4; }
    static constexpr int first(int q) { return q == 0 ? 0 : first(q - 1) + chunks(q - 1); }
    static constexpr int TOTAL = first(2 * NL);
    static constexpr int product_of(int f) {
        int q = 0;
        while (f >= first(q + 1)) ++q;
        return q;
    }
};
// Operand chunks in flight per wave: the fewer products a chunk feeds, the further ahead it is read.
constexpr int spread_depth(int nt) { return nt >= 3 ? 2 : nt == 2 ? 4 : 6; }

template <class S, class N, int ACT, int WV, int NT>
__device__ __forceinline__ void ffnn_spread(const float* __restrict__ W, float en_min, float scale, int D,
                                            const float* __restrict__ G, int P, int tile0, float* __restrict__ E,
                                            float* __restrict__ dEdG,
                                            v4f (&xs)[2][S::NT][N::MT][64]) {
    constexpr NetLayout Lay = N::layout();
    constexpr int MT = N::MT, NL = N::NL, kDepth = spread_depth(NT);
    uint32_t lane = threadIdx.x;
    asm volatile("" : "+v"(lane));  // keeps the operand reads inside the caller's loop
    lane &= 63u;                    // known range: the reads take a scalar base and this offset
    const int g = lane >> 4, pl = lane & 15;
    const int m = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // this wave's 16-unit block
    // and its left-over unit: block m2 of tile t2 (with fewer than WV of them, some are computed twice)
    constexpr bool LEFT = S::EX > 0;
    const int t2 = m % NT, m2 = LEFT ? WV + (m / NT) % S::EX : 0;
    // operands of chunk f of the whole sequence for this wave's block (dE/dG has MD blocks only: the
    // other waves read block 0's there and drop out before using them)
    float ring[kDepth][4], ring2[LEFT ? kDepth : 1][4];
    auto load_chunk = [&](auto fc) {
        constexpr int f = decltype(fc)::value;
        if constexpr (f < S::TOTAL) {
            constexpr int q = S::product_of(f), c = f - S::first(q);
            constexpr int k = q < NL ? q : 2 * NL - 1 - q;
            constexpr int ks = q == 0 ? N::KD : N::KH;
            constexpr int off = (q < NL ? Lay.fwd_off(k) : Lay.bwd_off(k)) + 4 * c * 64;
            const int mm = (q == 2 * NL - 1 && N::MD < WV && m >= N::MD) ? 0 : m;
            const float* src = W + (off + mm * ks * 64);
#pragma unroll
            for (int r = 0; r < 4; ++r) ring[f % kDepth][r] = src[r * 64 + lane];
            if constexpr (LEFT && q != 2 * NL - 1) {
                const float* src2 = W + (off + m2 * ks * 64);
#pragma unroll
                for (int r = 0; r < 4; ++r) ring2[f % kDepth][r] = src2[r * 64 + lane];
            }
        }
    };
    auto load4 = [&](const float* src, int mb) {  // units 16 mb + 4 g + 0..3 of a bias or the output layer
        const float4 v = *reinterpret_cast<const float4*>(src + 16 * mb + 4 * g);
        return v4f{v.x, v.y, v.z, v.w};
    };
    v4f bias = load4(W + Lay.bias_off(0), m), bias2 = bias;  // one layer ahead
    if constexpr (LEFT) bias2 = load4(W + Lay.bias_off(0), m2);
    static_for<kDepth>([&](auto f) { load_chunk(f); });
    // the input rows in the B operand's layout: wave c loads chunk c
    if (m < N::MD) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int p = (tile0 + t) * 16 + pl;
            v4f v;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int e = 16 * m + 4 * g + r;
                v[r] = (p < P && e < D) ? G[(size_t)p * D + e] : 0.f;
            }
            xs[0][t][m][lane] = v;
        }
    }
    __syncthreads();
    // acc += the product q of this wave's block with the vectors in xs[buf]
    auto product = [&](auto qc, v4f (&acc)[NT], v4f& acc2) {
        constexpr int q = decltype(qc)::value, buf = (q < NL ? q : q + 1) & 1;
        constexpr bool two = LEFT && q != 2 * NL - 1;
        v4f x[2][NT];  // one chunk ahead
#pragma unroll
        for (int t = 0; t < NT; ++t) x[0][t] = xs[buf][t][0][lane];
        static_for<S::chunks(q)>([&](auto cc) {
            constexpr int c = decltype(cc)::value, f = S::first(q) + c;
            if constexpr (c + 1 < S::chunks(q)) {
#pragma unroll
                for (int t = 0; t < NT; ++t) x[(c + 1) & 1][t] = xs[buf][t][c + 1][lane];
            }
            v4f x2;  // the left-over unit's products come last in the chunk, after this read
            if constexpr (two) x2 = xs[buf][t2][c][lane];
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(ring[f % kDepth][r], x[c & 1][t][r], acc[t], 0, 0, 0);
            if constexpr (two) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    acc2 = __builtin_amdgcn_mfma_f32_16x16x4f32(ring2[f % kDepth][r], x2[r], acc2, 0, 0, 0);
            }
            load_chunk(std::integral_constant<int, f + kDepth>{});
            // reads stay this far ahead (all at once they would spill; with a left-over unit the compiler
            // keeps them apart by itself and the barrier is what spills)
            if constexpr (!LEFT) __builtin_amdgcn_sched_barrier(0);
        });
    };
    constexpr bool BITS = ACT == NEPX_ACT_RELU;
    v4f h[BITS ? 1 : NL][BITS ? 1 : NT + 1];  // this wave's activations (tanh), the left-over unit's at NT
    uint32_t on[BITS ? NL : 1] = {};          // its active units (ReLU), bit 4 t + r
    auto der = [&](int k, int t, int r) {
        if constexpr (BITS) return (on[k] >> (4 * t + r)) & 1u ? 1.f : 0.f;
        else return act_der(h[k][t][r], ACT);
    };
    static_for<NL>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        v4f acc[NT], acc2 = bias2;
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = bias;
        constexpr int next = k + 1 < NL ? Lay.bias_off(k + 1) : Lay.wout_off();
        bias = load4(W + next, m);
        if constexpr (LEFT) bias2 = load4(W + next, m2);
        product(kc, acc, acc2);
        auto finish = [&](int t, const v4f& a) {
            v4f o;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                o[r] = act_fwd(a[r], ACT);
                if constexpr (BITS) on[k] |= (o[r] > 0.f ? 1u : 0u) << (4 * t + r);
            }
            if constexpr (!BITS) h[k][t] = o;
            return o;
        };
#pragma unroll
        for (int t = 0; t < NT; ++t) xs[(k + 1) & 1][t][m][lane] = finish(t, acc[t]);
        if constexpr (LEFT) xs[(k + 1) & 1][t2][m2][lane] = finish(NT, acc2);
        __syncthreads();
    });
    // the last layer's deltas (`bias` holds the output layer's weights of this wave's units)
    auto last_delta = [&](int t, const v4f& w) {
        v4f d;
#pragma unroll
        for (int r = 0; r < 4; ++r) d[r] = scale * w[r] * der(NL - 1, t, r);
        return d;
    };
#pragma unroll
    for (int t = 0; t < NT; ++t) xs[(NL + 1) & 1][t][m][lane] = last_delta(t, bias);
    if constexpr (LEFT) xs[(NL + 1) & 1][t2][m2][lane] = last_delta(NT, bias2);
    // output layer: wave t forms tile t's sum from the whole last layer, in ffnn_tiles' order
    if (m < NT) {
        const float* wo = W + Lay.wout_off();
        float y = 0.f;
#pragma unroll
        for (int c = 0; c < MT; ++c) {
            const float4 w4 = *reinterpret_cast<const float4*>(wo + 16 * c + 4 * g);
            const float wv[4] = {w4.x, w4.y, w4.z, w4.w};
            const v4f hv = xs[NL & 1][m][c][lane];
#pragma unroll
            for (int r = 0; r < 4; ++r) y += wv[r] * hv[r];
        }
        y += __shfl_xor(y, 16);
        y += __shfl_xor(y, 32);
        y += W[Lay.bout_off()];
        const int p = (tile0 + m) * 16 + pl;
        if (p < P && lane < 16) E[p] = en_min + scale * y;
    }
    __syncthreads();
    static_for<NL - 1>([&](auto jc) {  // the deltas of layer k - 1 from those of layer k
        constexpr int q = NL + decltype(jc)::value, k = 2 * NL - 1 - q;
        v4f acc[NT], acc2 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
        product(std::integral_constant<int, q>{}, acc, acc2);
        auto delta = [&](int t, const v4f& a) {
            v4f d;
#pragma unroll
            for (int r = 0; r < 4; ++r) d[r] = a[r] * der(k - 1, t, r);
            return d;
        };
#pragma unroll
        for (int t = 0; t < NT; ++t) xs[q & 1][t][m][lane] = delta(t, acc[t]);
        if constexpr (LEFT) xs[q & 1][t2][m2][lane] = delta(NT, acc2);
        __syncthreads();
    });
    if (m < N::MD) {  // dE/dG (uniform per wave)
        v4f acc[NT], none;
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
        product(std::integral_constant<int, 2 * NL - 1>{}, acc, none);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int p = (tile0 + t) * 16 + pl;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int e = 16 * m + 4 * g + r;
                if (p < P && e < D) dEdG[(size_t)p * D + e] = acc[t][r];
            }
        }
    }
}

// Each block takes an equal run of tiles, in groups of NT and one of what is left: with many pairs the
// operand reads are shared four ways and the blocks end together, with few every block has one tile.
template <class N, int ACT, int WV, int NT>
__global__ __launch_bounds__((SpreadNet<N, ACT, WV, NT>::BLOCK)) __attribute__((
    amdgpu_waves_per_eu(SpreadNet<N, ACT, WV, NT>::WAVES_PER_SIMD, SpreadNet<N, ACT, WV, NT>::WAVES_PER_SIMD))) void k_ffnn_spread(
    const float* __restrict__ W, float en_min, float scale, int D, const float* __restrict__ G,
    const int32_t* __restrict__ np_dev, int64_t maxp, float* __restrict__ E, float* __restrict__ dEdG) {
    using S = SpreadNet<N, ACT, WV, NT>;
    __shared__ v4f xs[2][S::NT][N::MT][64];  // one layer's outputs: block c of lane l of tile t at [t][c][l]
    const int P = n_pairs(np_dev, maxp);
    const int nt = (P + 15) / 16;
    const int per = (nt + gridDim.x - 1) / gridDim.x;
    int tile = blockIdx.x * per;
    const int end = tile + per < nt ? tile + per : nt;
    while (tile < end) {  // uniform over the block
        const int left = end - tile;
        auto group = [&](auto nt) {
            ffnn_spread<S, N, ACT, WV, decltype(nt)::value>(W, en_min, scale, D, G, P, tile, E, dEdG, xs);
            tile += decltype(nt)::value;
        };
        if constexpr (NT >= 4) {
            if (left >= 4) group(std::integral_constant<int, 4>{});
            else if (left == 3) group(std::integral_constant<int, 3>{});
        }
        if constexpr (NT >= 2) {
            if (left == 2 || (NT < 4 && left > 2)) group(std::integral_constant<int, 2>{});
        }
        if (left == 1 || NT == 1) group(std::integral_constant<int, 1>{});
        __syncthreads();  // the last reads of xs are done before the next tiles write it
    }
}

// Fused: descriptor -> LDS -> MFMA network -> LDS -> adjoint.  Each block
// takes 256 consecutive pairs per iteration (64 per wave), so every wave of a
// block runs the same number of iterations and the barriers are uniform.
// The forward accumulators A of each lane's pair stay in registers through
// the network phase and feed the adjoint directly.
template <class Cfg, class N, int PREC, int ACT>
__global__ __launch_bounds__(kBlock) NEPX_ADJ_ATTR void k_fused(nepx_pair_model m, const float* __restrict__ Wg,
                                                                const void* __restrict__ Whg,
                                                                float en_min, float scale,
                                                                const float4* __restrict__ qf,
                                                                const int32_t* __restrict__ pi,
                                                                const int32_t* __restrict__ pj,
                                                                const float4* __restrict__ pt,
                                                                const int32_t* __restrict__ np_dev, int64_t maxp,
                                                                float clip, float* __restrict__ out, RevOut rv) {
    constexpr int LD = (Cfg::D + 3) / 4 * 4 + 4;  // row stride in LDS (16-byte aligned)
    __shared__ __attribute__((aligned(16))) float tile[kBlock * LD];
    __shared__ float etile[kBlock];
    using R = NetRun<N, kNetTiles, PREC>;
    __shared__ __attribute__((aligned(16))) float wl[weight_lds_floats<N, PREC>()];
    const float* W;
    const void* WH;
    stage_net<N, PREC>(wl, Wg, Whg, W, WH);
    const int P = n_pairs(np_dev, maxp);
    const int tag = rev_tag(rv);
    const int lane = threadIdx.x & 63;
    const int wv = threadIdx.x >> 6;
    float* myrow = tile + threadIdx.x * LD;
    for (int base = blockIdx.x * kBlock; base < P; base += gridDim.x * kBlock) {
        const int idx = base + threadIdx.x;
        const bool valid = idx < P;
        float4 qi = make_float4(1.f, 0.f, 0.f, 0.f), qj = qi, t = make_float4(1.f, 0.f, 0.f, 0.f);
        if (valid) load_pair(qf, pi, pj, pt, idx, qi, qj, t);
        const PairIn g = pair_in<Cfg>(m, qi, qj, t.x, t.y, t.z);
        // one-pass shapes keep the forward accumulators in registers for the adjoint; multi-pass
        // shapes recompute every range there (keeping the last range's through the network phase
        // spills: measured slower on the 262,144-cylinder step, 14.8 vs 12.9 ms)
        using LRL = LastPass<Cfg>;
        constexpr bool KEEP = Cfg::ONE_PASS;
        float A[KEEP ? Cfg::NANG + 1 : 1][KEEP ? LRL::N : 1];
        {
            if constexpr (Cfg::ONE_PASS) {
                float Gr[Cfg::D];
                float grad[Cfg::NRAD + 1];
                desc_accumulate<Cfg, LRL, true>(m, g, grad, A);
                desc_finish<Cfg, LRL>(A, Gr);
#pragma unroll
                for (int n = 0; n <= Cfg::NRAD; ++n) Gr[n] = grad[n];
#pragma unroll
                for (int k = 0; k < Cfg::D; ++k) myrow[k] = valid ? Gr[k] : 0.f;
            } else {  // several passes: each writes its entries straight into the LDS row
                float grad[Cfg::NRAD + 1];
                for_passes<Cfg>([&](auto range, auto first) {
                    using LR = decltype(range);
                    float Ap[Cfg::NANG + 1][LR::N];
                    desc_accumulate<Cfg, LR, decltype(first)::value>(m, g, grad, Ap);
                    desc_finish<Cfg, LR>(Ap, myrow);
                    if constexpr (decltype(first)::value) {
#pragma unroll
                        for (int n = 0; n <= Cfg::NRAD; ++n) myrow[n] = grad[n];
                    }
                });
                if (!valid)
                    for (int k = 0; k < Cfg::D; ++k) myrow[k] = 0.f;
            }
        }
        __syncthreads();
#pragma unroll 1
        for (int sub = 0; sub < 64 / (16 * kNetTiles); ++sub) {
            v4f gin[kNetTiles][R::IC];
#pragma unroll
            for (int tt = 0; tt < kNetTiles; ++tt) {
                const int local = wv * 64 + (sub * kNetTiles + tt) * 16 + (lane & 15);
                gather_chunks<R::IC>(tile + local * LD, true, Cfg::D, gin[tt]);
            }
            v4f dg[kNetTiles][N::MD];
            float y[kNetTiles];
            R::run(W, WH, ACT, gin, scale, dg, y);
#pragma unroll
            for (int tt = 0; tt < kNetTiles; ++tt) {
                const int local = wv * 64 + (sub * kNetTiles + tt) * 16 + (lane & 15);
                if (lane < 16) etile[local] = en_min + scale * y[tt];
                scatter_chunks<N::MD>(tile + local * LD, true, Cfg::D, dg[tt]);
            }
        }
        __syncthreads();
        if (valid) {
            float dG[Cfg::D];
#pragma unroll
            for (int k = 0; k < Cfg::D; ++k) dG[k] = myrow[k];
            AdjAcc acc;
            for_passes<Cfg>([&](auto range, auto first) {
                using LR = decltype(range);
                if constexpr (KEEP) {
                    desc_adjoint<Cfg, LR, decltype(first)::value>(m, g, dG, A, acc);
                } else {
                    float grad[Cfg::NRAD + 1];
                    float Ap[Cfg::NANG + 1][LR::N];
                    desc_accumulate<Cfg, LR, false>(m, g, grad, Ap);
                    desc_adjoint<Cfg, LR, decltype(first)::value>(m, g, dG, Ap, acc);
                }
            });
            store_out(out, idx, adj_finish<Cfg>(acc), etile[threadIdx.x], clip, rv, tag);
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// Reference-compat finite-difference stencil (PosToPtsKernels.py:153-446).
// Translating i's sites by +dx e equals translating j by -dx e (the
// descriptor depends only on the cloud up to translation); rotating i's sites
// about X_i by dteta about e equals q_i -> dq q_i with dq = (cos dteta/2,
// sin dteta/2 e); the rows in the frame of j rotate q_j the same way.
__device__ __forceinline__ float4 qmul4(float4 a, float4 b) {  // (w, x, y, z) in (x, y, z, w) slots
    return make_float4(a.x * b.x - (a.y * b.y + a.z * b.z + a.w * b.w),
                       a.x * b.y + b.x * a.y + (a.z * b.w - a.w * b.z),
                       a.x * b.z + b.x * a.z + (a.w * b.y - a.y * b.w),
                       a.x * b.w + b.x * a.w + (a.y * b.z - a.z * b.y));
}

__global__ __launch_bounds__(kBlock) void k_stencil_rows(const float4* __restrict__ qf, const int32_t* __restrict__ pi,
                                                         const int32_t* __restrict__ pj,
                                                         const float4* __restrict__ pt, int P, float dx,
                                                         float dteta, float4* __restrict__ qrows,
                                                         int32_t* __restrict__ ri, int32_t* __restrict__ rj,
                                                         float4* __restrict__ trows) {
    const int r = blockIdx.x * kBlock + threadIdx.x;
    if (r >= 10 * P) return;
    const int o = r / P, p = r % P;
    float4 qi = qf[pi[p]], qj = qf[pj[p]], t = pt[p];
    const float c = cosf(0.5f * dteta), s = sinf(0.5f * dteta);
    if (o >= 1 && o <= 3) {
        if (o == 1) t.x -= dx;
        if (o == 2) t.y -= dx;
        if (o == 3) t.z -= dx;
    } else if (o >= 4) {
        const int ax = (o - 4) % 3;
        const float4 dq = make_float4(c, ax == 0 ? s : 0.f, ax == 1 ? s : 0.f, ax == 2 ? s : 0.f);
        if (o <= 6) qi = qmul4(dq, qi);
        else qj = qmul4(dq, qj);
    }
    qrows[2 * (size_t)r] = qi;
    qrows[2 * (size_t)r + 1] = qj;
    ri[r] = 2 * r;
    rj[r] = 2 * r + 1;
    trows[r] = t;
}

__global__ __launch_bounds__(kBlock) void k_fd_forces(const float* __restrict__ E, int P, float dx, float dteta,
                                                      float clip, float* __restrict__ out) {
    const int p = blockIdx.x * kBlock + threadIdx.x;
    if (p >= P) return;
    const float e0 = E[p];
    PairOut o;
    o.fx = -(E[1 * (size_t)P + p] - e0) / dx;
    o.fy = -(E[2 * (size_t)P + p] - e0) / dx;
    o.fz = -(E[3 * (size_t)P + p] - e0) / dx;
    o.tix = -(E[4 * (size_t)P + p] - e0) / dteta;
    o.tiy = -(E[5 * (size_t)P + p] - e0) / dteta;
    o.tiz = -(E[6 * (size_t)P + p] - e0) / dteta;
    o.tjx = -(E[7 * (size_t)P + p] - e0) / dteta;
    o.tjy = -(E[8 * (size_t)P + p] - e0) / dteta;
    o.tjz = -(E[9 * (size_t)P + p] - e0) / dteta;
    store_out(out, p, o, e0, clip);
}

// ---------------------------------------------------------------------------
// Dispatch tables.

static int grid_for_cap(int64_t units, int per_block, int64_t cap) {
    int64_t g = (units + per_block - 1) / per_block;
    if (g > cap) g = cap;
    if (g < 1) g = 1;
    return (int)g;
}

static int grid_for(int64_t maxp, int per_block) {
    return grid_for_cap(maxp, per_block, (int64_t)device_cus() * tuning().pair_blocks_per_cu);
}

#define NEPX_DESC_CASES(X)                          \
    X(8, 11, 6, 4, CfgCube8)                        \
    X(10, 11, 6, 4, CfgTet10)                       \
    X(12, 17, 6, 6, CfgCyl12)                       \
    X(6, 10, 8, 4, CfgCubeV2)                       \
    X(4, 10, 8, 4, CfgThV1)                         \
    X(6, 10, 10, 10, CfgCubeV2L10)                  \
    X(4, 10, 10, 10, CfgThV1L10)

// Multi-pass shapes with at most two blocks of 64 pairs per CU run their passes on separate waves
// (k_desc_fwd_passes, k_adjoint_passes; same results): one lane per pair would leave most SIMDs idle.
template <class Cfg>
static bool by_passes(int64_t maxp) {
    return !Cfg::ONE_PASS && (maxp + 63) / 64 <= 2 * (int64_t)device_cus();
}
static int pass_grid(int64_t maxp) { return (int)((maxp + 63) / 64); }
// The forward's passes go one to a block while every one of those waves has a SIMD to itself (4 a CU);
// up to four passes have a wave each already.  hypers 10 10 10, one call, two passes a wave -> one:
//   4 sites: 241 pairs 16.2 -> 13.0 us, 3,000 16.5 -> 13.6, 8,000 17.4 -> 15.7
//   6 sites: 241 pairs 21.5 -> 14.9 us, 3,000 22.1 -> 17.0, 8,000 22.9 -> 19.1
// With more waves than SIMDs it mostly loses: 4 sites, 20,000 pairs 33.7 -> 36.3 us, 100,001 pairs (there
// against one lane per pair) 110 -> 135 us; 6 sites, 20,000 pairs 44.8 -> 42.6 us, 100,001 pairs 143 -> 166 us.
template <class Cfg>
static bool passes_alone(int64_t maxp) {
    constexpr int np = n_passes(Cfg::NANG, Cfg::LMAX);
    return np > pass_waves<Cfg>() && (int64_t)pass_grid(maxp) * np <= 4 * (int64_t)device_cus();
}

template <class T>
static void launch_desc_fwd(const nepx_pair_model& m, const float* qf, const int32_t* pair_i, const int32_t* pair_j,
                            const float* pair_t, const int32_t* np_dev, int64_t maxp, float* G, void* stream) {
    if constexpr (!T::ONE_PASS) {
        if (by_passes<T>(maxp)) {
            const bool alone = passes_alone<T>(maxp);
            const dim3 grid(pass_grid(maxp), alone ? n_passes(T::NANG, T::LMAX) : 1);
            hipLaunchKernelGGL(k_desc_fwd_passes<T>, grid, dim3(alone ? 64 : 64 * pass_waves<T>()), 0,
                               as_stream(stream), m, (const float4*)qf, pair_i, pair_j, (const float4*)pair_t,
                               np_dev, maxp, G);
            return;
        }
    }
    hipLaunchKernelGGL(k_desc_fwd<T>, dim3(grid_for(maxp, kBlock)), dim3(kBlock), 0, as_stream(stream), m,
                       (const float4*)qf, pair_i, pair_j, (const float4*)pair_t, np_dev, maxp, G);
}

// Hypers 10 8 4, four sites: many pairs keep one lane per pair, whose two passes cost less than the four lanes'
// exchange once the chip is full (two rounds of its lanes).  One lane -> four, one call of that many pairs:
//   4 sites: 100,001 pairs 52 -> 45 us, 200,000 100 -> 98, 260,000 106 -> 121, 500,000 198 -> 228, 1,000,000 382 -> 450
//   6 sites: 100,001 pairs 71 -> 54 us, 200,000 139 -> 119, 260,000 143 -> 148, 350,000 207 -> 198, 1,000,000 531 -> 550
// Six sites lie within 4 % either way beyond the line and stay on four lanes, as do hypers 10 10 10 (eight
// passes), which gain at every size.  The count decides, on the device: a capacity past the line launches
// both kernels, and one of them leaves at once (3 us; by the capacity alone, 70,000 pairs in a list of
// 280,000 slots would take 50 us in place of 34).
template <class T>
constexpr bool one_lane_for_many() { return adjoint_on_quads<T>() && T::LMAX <= 4 && T::NS <= 4; }
template <class T>
static int quad_adjoint_pairs() {
    return one_lane_for_many<T>() ? 14 * 64 * device_cus() : INT32_MAX;
}

template <class T>
static int launch_adjoint(const nepx_pair_model& m, const float* qf, const int32_t* pair_i, const int32_t* pair_j,
                          const float* pair_t, const int32_t* np_dev, int64_t maxp, const float* dEdG,
                          const float* E, float clip, float* out, void* stream) {
    int few = 0;
    if constexpr (adjoint_on_quads<T>()) {
        few = quad_adjoint_pairs<T>();
        const int rc = launch_adjoint_quad<T>(m, (int)(device_cus() * (int64_t)tuning().pair_blocks_per_cu), qf, pair_i,
                                              pair_j, pair_t, np_dev, maxp, few, dEdG, E, clip, out, stream);
        if (rc || maxp <= few) return rc;
    } else if constexpr (!T::ONE_PASS) {
        if (by_passes<T>(maxp)) {
            hipLaunchKernelGGL(k_adjoint_passes<T>, dim3(pass_grid(maxp)), dim3(64 * pass_waves<T>()), 0,
                               as_stream(stream), m, (const float4*)qf, pair_i, pair_j, (const float4*)pair_t,
                               np_dev, maxp, dEdG, E, clip, out);
            NEPX_LAUNCH_CHECK();
            return NEPX_OK;
        }
    }
    if constexpr (!adjoint_on_quads<T>() || one_lane_for_many<T>()) {
        hipLaunchKernelGGL(k_adjoint<T>, dim3(grid_for(maxp, kBlock)), dim3(kBlock), 0, as_stream(stream), m,
                           (const float4*)qf, pair_i, pair_j, (const float4*)pair_t, np_dev, maxp, few, dEdG, E, clip,
                           out);
        NEPX_LAUNCH_CHECK();
    }
    return NEPX_OK;
}

static bool desc_supported(const nepx_pair_model* m) {
#define X(ns, a, b, c, T) \
    if (m->n_sites == ns && m->nrad == a && m->nang == b && m->lmax == c) return true;
    NEPX_DESC_CASES(X)
#undef X
    return false;
}

static int check_model(const nepx_pair_model* m) {
    NEPX_REQUIRE(m != nullptr, NEPX_EINVAL, "null pair model");
    NEPX_REQUIRE(m->n_sites > 0 && m->n_sites <= NEPX_MAX_SITES, NEPX_EINVAL, "n_sites %d out of range",
                 m->n_sites);
    NEPX_REQUIRE(m->nang <= m->nrad, NEPX_EINVAL, "nang (%d) must not exceed nrad (%d)", m->nang, m->nrad);
    NEPX_REQUIRE(m->r_nep > 0.f, NEPX_EINVAL, "r_nep must be positive");
    NEPX_REQUIRE(desc_supported(m), NEPX_EUNSUP,
                 "no descriptor kernel for n_sites=%d hypers=(%d,%d,%d)", m->n_sites, m->nrad, m->nang,
                 m->lmax);
    return NEPX_OK;
}

static int check_net(const nepx_net* n, int D) {
    NEPX_REQUIRE(n != nullptr && n->w_packed != nullptr, NEPX_EINVAL, "null network");
    NEPX_REQUIRE(n->d_in == D, NEPX_EINVAL, "network input %d != descriptor size %d", n->d_in, D);
    NEPX_REQUIRE(n->act == NEPX_ACT_TANH || n->act == NEPX_ACT_RELU, NEPX_EINVAL, "bad activation %d",
                 n->act);
    return NEPX_OK;
}

static int model_D(const nepx_pair_model* m) { return (m->nrad + 1) + (m->nang + 1) * m->lmax; }

}  // namespace nepx

using namespace nepx;

extern "C" int64_t nepx_net_packed_floats(int32_t d_in, int32_t width, int32_t n_hidden) {
    if (d_in <= 0 || width <= 0 || n_hidden < 0) return -1;
    NetLayout L{round16(d_in), round16(width), n_hidden + 1};
    return L.total();
}

extern "C" int nepx_net_pack(int32_t d_in, int32_t width, int32_t n_hidden, const float* const* ws,
                             const float* const* bs, float* out) {
    NEPX_REQUIRE(d_in > 0 && width > 0 && n_hidden >= 0, NEPX_EINVAL, "bad network dims");
    NEPX_REQUIRE(ws && bs && out, NEPX_EINVAL, "null pointer");
    const int DP = round16(d_in), HP = round16(width), NL = n_hidden + 1;
    NetLayout L{DP, HP, NL};
    memset(out, 0, sizeof(float) * L.total());
    for (int k = 0; k < NL; ++k) {
        const int kin = k == 0 ? d_in : width, kinp = k == 0 ? DP : HP;
        const float* W = ws[k];  // (width x kin)
        NEPX_REQUIRE(W && bs[k], NEPX_EINVAL, "null layer %d", k);
        // forward operand: [mt][s][lane] = W[16mt + lane%16][16(s/4) + 4(lane/16) + s%4]
        float* F = out + L.fwd_off(k);
        for (int mt = 0; mt < HP / 16; ++mt)
            for (int s = 0; s < kinp / 4; ++s)
                for (int lane = 0; lane < 64; ++lane) {
                    const int row = 16 * mt + lane % 16;
                    const int col = 16 * (s / 4) + 4 * (lane / 16) + s % 4;
                    F[(mt * (kinp / 4) + s) * 64 + lane] = (row < width && col < kin) ? W[row * kin + col] : 0.f;
                }
        // backward operand (W^T): [mt][s][lane] = W[16(s/4) + 4(lane/16) + s%4][16mt + lane%16]
        float* B = out + L.bwd_off(k);
        for (int mt = 0; mt < kinp / 16; ++mt)
            for (int s = 0; s < HP / 4; ++s)
                for (int lane = 0; lane < 64; ++lane) {
                    const int row = 16 * (s / 4) + 4 * (lane / 16) + s % 4;
                    const int col = 16 * mt + lane % 16;
                    B[(mt * (HP / 4) + s) * 64 + lane] = (row < width && col < kin) ? W[row * kin + col] : 0.f;
                }
        for (int u = 0; u < width; ++u) out[L.bias_off(k) + u] = bs[k][u];
    }
    NEPX_REQUIRE(ws[NL] && bs[NL], NEPX_EINVAL, "null output layer");
    for (int u = 0; u < width; ++u) out[L.wout_off() + u] = ws[NL][u];
    out[L.bout_off()] = bs[NL][0];
    return NEPX_OK;
}

static bool lowp_precision(int p) {
    return p == NEPX_NET_F16X3 || p == NEPX_NET_BF16 || p == NEPX_NET_BF16X3;
}

// float -> bf16 bits, round to nearest even (NaN stays NaN).
static uint16_t bf16_bits(float f) {
    uint32_t u;
    memcpy(&u, &f, 4);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
static float bf16_value(uint16_t b) {
    const uint32_t u = (uint32_t)b << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}

extern "C" int64_t nepx_net_packed_lowp(int32_t precision, int32_t d_in, int32_t width, int32_t n_hidden) {
    if (!lowp_precision(precision) || d_in <= 0 || width <= 0 || n_hidden < 0 || round16(width) % 32) return -1;
    NetLayoutH L{round32(round16(d_in)), round16(d_in), round16(width), n_hidden + 1,
                 precision == NEPX_NET_BF16 ? 1 : 2};
    return L.total();
}

extern "C" int nepx_net_pack_lowp(int32_t precision, int32_t d_in, int32_t width, int32_t n_hidden,
                                  const float* const* ws, uint16_t* out) {
    NEPX_REQUIRE(lowp_precision(precision), NEPX_EINVAL, "precision %d has no 16-bit operands", precision);
    NEPX_REQUIRE(d_in > 0 && width > 0 && n_hidden >= 0, NEPX_EINVAL, "bad network dims");
    NEPX_REQUIRE(round16(width) % 32 == 0, NEPX_EUNSUP,
                 "16-bit operand paths need a padded width that is a multiple of 32");
    NEPX_REQUIRE(ws && out, NEPX_EINVAL, "null pointer");
    const int parts = precision == NEPX_NET_BF16 ? 1 : 2;
    const int DP = round16(d_in), DPH = round32(DP), HP = round16(width), NL = n_hidden + 1;
    NetLayoutH L{DPH, DP, HP, NL, parts};
    for (int64_t k = 0; k < L.total(); ++k) out[k] = 0;
    // hi = w rounded to the 16-bit type, lo = the remainder rounded (split forms only)
    auto put = [&](int base, int lo_off, int idx, float w) {
        if (precision == NEPX_NET_F16X3) {
            const _Float16 h = (_Float16)w;
            const _Float16 l = (_Float16)(w - (float)h);
            memcpy(&out[base + idx], &h, 2);
            memcpy(&out[base + lo_off + idx], &l, 2);
        } else {
            const uint16_t h = bf16_bits(w);
            out[base + idx] = h;
            if (parts == 2) out[base + lo_off + idx] = bf16_bits(w - bf16_value(h));
        }
    };
    for (int k = 0; k < NL; ++k) {
        const int kin = k == 0 ? d_in : width;
        const float* W = ws[k];
        NEPX_REQUIRE(W, NEPX_EINVAL, "null layer %d", k);
        const int ksf = (k == 0 ? DPH : HP) / 32;
        const int lof = (HP / 16) * ksf * 512;
        for (int mt = 0; mt < HP / 16; ++mt)
            for (int s = 0; s < ksf; ++s)
                for (int lane = 0; lane < 64; ++lane)
                    for (int j = 0; j < 8; ++j) {
                        const int row = 16 * mt + lane % 16;
                        const int col = 16 * (2 * s + j / 4) + 4 * (lane / 16) + j % 4;
                        const float w = (row < width && col < kin) ? W[row * kin + col] : 0.f;
                        put(L.fwd_off(k), lof, ((mt * ksf + s) * 64 + lane) * 8 + j, w);
                    }
        const int mtb = (k == 0 ? DP : HP) / 16, ksb = HP / 32;
        const int lob = mtb * ksb * 512;
        for (int mt = 0; mt < mtb; ++mt)
            for (int s = 0; s < ksb; ++s)
                for (int lane = 0; lane < 64; ++lane)
                    for (int j = 0; j < 8; ++j) {
                        const int unit = 16 * (2 * s + j / 4) + 4 * (lane / 16) + j % 4;   // output unit of layer k
                        const int col = 16 * mt + lane % 16;                               // input unit of layer k
                        const float w = (unit < width && col < kin) ? W[unit * kin + col] : 0.f;
                        put(L.bwd_off(k), lob, ((mt * ksb + s) * 64 + lane) * 8 + j, w);
                    }
    }
    return NEPX_OK;
}

extern "C" int64_t nepx_net_packed_halves(int32_t d_in, int32_t width, int32_t n_hidden) {
    return nepx_net_packed_lowp(NEPX_NET_F16X3, d_in, width, n_hidden);
}

extern "C" int nepx_net_pack_half(int32_t d_in, int32_t width, int32_t n_hidden, const float* const* ws,
                                  uint16_t* out) {
    return nepx_net_pack_lowp(NEPX_NET_F16X3, d_in, width, n_hidden, ws, out);
}

extern "C" int nepx_descriptor_fwd(const nepx_pair_model* m, const float* qf, const int32_t* pair_i,
                                   const int32_t* pair_j, const float* pair_t, const int32_t* np_dev,
                                   int64_t maxp, float* G, void* stream) {
    int rc = check_model(m);
    if (rc) return rc;
    NEPX_REQUIRE(qf && pair_i && pair_j && pair_t && np_dev && G, NEPX_EINVAL, "null buffer");
    if (maxp <= 0) return NEPX_OK;
#define X(ns, a, b, c, T)                                                                           \
    if (m->n_sites == ns && m->nrad == a && m->nang == b && m->lmax == c) {                        \
        launch_desc_fwd<T>(*m, qf, pair_i, pair_j, pair_t, np_dev, maxp, G, stream);                \
        NEPX_LAUNCH_CHECK();                                                                        \
        return NEPX_OK;                                                                             \
    }
    NEPX_DESC_CASES(X)
#undef X
    return NEPX_EUNSUP;
}

#define NEPX_NET_CASES(X)              \
    X(40, 64, 1, Net40x64, kNetTiles)  \
    X(60, 128, 1, Net60x128, 1)        \
    X(47, 150, 3, Net47x150, 1)        \
    X(121, 150, 3, Net121x150, 1)

static bool net_supported(const nepx_net* n) {
#define X(d, w, h, T, NT) if (n->d_in == d && n->width == w && n->n_hidden == h) return true;
    NEPX_NET_CASES(X)
#undef X
    return false;
}

static int check_precision(const nepx_net* net) {
    const int p = net->precision;
    NEPX_REQUIRE(p == NEPX_NET_F32 || lowp_precision(p), NEPX_EINVAL, "bad network precision %d", p);
    NEPX_REQUIRE(p == NEPX_NET_F32 || net->w_half, NEPX_EINVAL, "precision %d without packed 16-bit operands", p);
    NEPX_REQUIRE(p == NEPX_NET_F32 || round16(net->width) % 32 == 0, NEPX_EUNSUP,
                 "no 16-bit network kernel for width %d", net->width);
    // bf16 rounding moves pre-activations across zero, where ReLU's derivative jumps
    NEPX_REQUIRE((p != NEPX_NET_BF16 && p != NEPX_NET_BF16X3) || net->act == NEPX_ACT_TANH, NEPX_EUNSUP,
                 "the bf16 network forms are for tanh networks only");
    return NEPX_OK;
}

template <class T, int NT, int PREC>
static void launch_ffnn_p(const nepx_net* net, int grid, float scale, int d, const float* G, const int32_t* np_dev,
                          int64_t maxp, float* E, float* dEdG, void* stream) {
#define NEPX_LAUNCH_FFNN(A)                                                                                   \
    hipLaunchKernelGGL((k_ffnn<T, NT, PREC, A>), dim3(grid), dim3(kBlock), 0, as_stream(stream), net->w_packed, \
                       net->w_half, net->en_min, scale, d, G, np_dev, maxp, E, dEdG)
    if (net->act == NEPX_ACT_TANH) NEPX_LAUNCH_FFNN(NEPX_ACT_TANH);
    else if constexpr (PREC == NEPX_NET_F32 || PREC == NEPX_NET_F16X3) NEPX_LAUNCH_FFNN(NEPX_ACT_RELU);
#undef NEPX_LAUNCH_FFNN
}

template <class T, int NT>
static int launch_ffnn(const nepx_net* net, int grid, float scale, int d, const float* G, const int32_t* np_dev,
                       int64_t maxp, float* E, float* dEdG, void* stream) {
    switch (net->precision) {
        case NEPX_NET_F16X3:
            launch_ffnn_p<T, NT, NEPX_NET_F16X3>(net, grid, scale, d, G, np_dev, maxp, E, dEdG, stream);
            break;
        case NEPX_NET_BF16:
            launch_ffnn_p<T, NT, NEPX_NET_BF16>(net, grid, scale, d, G, np_dev, maxp, E, dEdG, stream);
            break;
        case NEPX_NET_BF16X3:
            launch_ffnn_p<T, NT, NEPX_NET_BF16X3>(net, grid, scale, d, G, np_dev, maxp, E, dEdG, stream);
            break;
        default:  // networks too wide for LDS run on k_ffnn_spread
            if constexpr (weights_in_lds<T, NEPX_NET_F32>())
                launch_ffnn_p<T, NT, NEPX_NET_F32>(net, grid, scale, d, G, np_dev, maxp, E, dEdG, stream);
    }
    NEPX_LAUNCH_CHECK();
    return NEPX_OK;
}

// The FP32 network runs on k_ffnn_spread where a block's copy of its operands does not fit in LDS (one
// wave per tile would read them from L2 for every tile: 60 -> 128 x 2 at 20,000 rows 93 us against
// 26, 121 -> 150 x 4 536 against 86), and, for the network that fits, up to four tiles per CU (too few
// for a wave each; beyond, k_ffnn's copy in LDS is as fast); same results.  The grid is capped by
// tuning().net_blocks_per_cu, as k_ffnn's is; by default at the two blocks that a CU holds.
template <class T>
static bool launch_ffnn_spread(const nepx_net* net, float scale, int d, const float* G, const int32_t* np_dev,
                               int64_t maxp, float* E, float* dEdG, void* stream) {
    const int64_t tiles = (maxp + 15) / 16, cus = device_cus(), most = cus * tuning().net_blocks_per_cu;
    if (net->precision != NEPX_NET_F32 || (weights_in_lds<T, NEPX_NET_F32>() && tiles > 4 * cus)) return false;
    constexpr int TANH_NT = T::NL <= 2 ? 4 : 2;
    constexpr int RELU_WV = T::MT > 8 ? 8 : T::MT;
#define NEPX_LAUNCH_SPREAD(A, WV, NT)                                                                              \
    hipLaunchKernelGGL((k_ffnn_spread<T, A, WV, NT>), dim3((unsigned)(few ? tiles : most)),                        \
                       dim3((SpreadNet<T, A, WV, NT>::BLOCK)), 0, as_stream(stream), net->w_packed, net->en_min,   \
                       scale, d, G, np_dev, maxp, E, dEdG)
    const bool few = tiles <= most;  // one tile per block at most
    if (net->act == NEPX_ACT_TANH) {
        if (few) NEPX_LAUNCH_SPREAD(NEPX_ACT_TANH, T::MT, 1);
        else NEPX_LAUNCH_SPREAD(NEPX_ACT_TANH, T::MT, TANH_NT);
    } else {
        if (few) NEPX_LAUNCH_SPREAD(NEPX_ACT_RELU, T::MT, 1);
        else NEPX_LAUNCH_SPREAD(NEPX_ACT_RELU, RELU_WV, 4);
    }
#undef NEPX_LAUNCH_SPREAD
    return true;
}

extern "C" int nepx_ffnn_fwd_bwd(const nepx_net* net, const float* G, const int32_t* np_dev, int64_t maxp,
                                 float* E, float* dEdG, void* stream) {
    NEPX_REQUIRE(net && net->w_packed, NEPX_EINVAL, "null network");
    NEPX_REQUIRE(G && np_dev && E && dEdG, NEPX_EINVAL, "null buffer");
    NEPX_REQUIRE(net_supported(net), NEPX_EUNSUP, "no network kernel for %d -> %d x%d", net->d_in,
                 net->width, net->n_hidden + 1);
    int rc = check_precision(net);
    if (rc) return rc;
    if (maxp <= 0) return NEPX_OK;
    const float scale = net->en_max - net->en_min;
#define X(d, w, h, T, NT)                                                                        \
    if (net->d_in == d && net->width == w && net->n_hidden == h) {                               \
        if (launch_ffnn_spread<T>(net, scale, d, G, np_dev, maxp, E, dEdG, stream)) {              \
            NEPX_LAUNCH_CHECK();                                                                 \
            return NEPX_OK;                                                                      \
        }                                                                                        \
        const int grid = grid_for_cap((maxp + 16 * NT - 1) / (16 * NT), kBlock / 64,            \
                                      (int64_t)device_cus() * tuning().net_blocks_per_cu);       \
        return launch_ffnn<T, NT>(net, grid, scale, d, G, np_dev, maxp, E, dEdG, stream);       \
    }
    NEPX_NET_CASES(X)
#undef X
    return NEPX_EUNSUP;
}

extern "C" int nepx_descriptor_adjoint(const nepx_pair_model* m, const float* qf, const int32_t* pair_i,
                                       const int32_t* pair_j, const float* pair_t, const int32_t* np_dev,
                                       int64_t maxp, const float* dEdG, const float* E, float clip,
                                       float* out, void* stream) {
    int rc = check_model(m);
    if (rc) return rc;
    NEPX_REQUIRE(qf && pair_i && pair_j && pair_t && np_dev && dEdG && out, NEPX_EINVAL, "null buffer");
    if (maxp <= 0) return NEPX_OK;
#define X(ns, a, b, c, T)                                                                            \
    if (m->n_sites == ns && m->nrad == a && m->nang == b && m->lmax == c) {                         \
        return launch_adjoint<T>(*m, qf, pair_i, pair_j, pair_t, np_dev, maxp, dEdG, E, clip, out, stream); \
    }
    NEPX_DESC_CASES(X)
#undef X
    return NEPX_EUNSUP;
}

#define NEPX_FUSED_CASES(X)                      \
    X(8, 11, 6, 4, CfgCube8, 40, 64, 1, Net40x64) \
    X(10, 11, 6, 4, CfgTet10, 40, 64, 1, Net40x64) \
    X(12, 17, 6, 6, CfgCyl12, 60, 128, 1, Net60x128)

// The bf16 forms exist for tanh networks only (check_precision).
static bool fused_precision_ok(const nepx_net* net) {
    return net->precision == NEPX_NET_F32 || net->precision == NEPX_NET_F16X3 || net->act == NEPX_ACT_TANH;
}

extern "C" int nepx_pair_fused_supported(const nepx_pair_model* m, const nepx_net* net) {
    if (!m || !net) return 0;
#define X(ns, a, b, c, T, d, w, h, NT)                                                            \
    if (m->n_sites == ns && m->nrad == a && m->nang == b && m->lmax == c && net->d_in == d &&    \
        net->width == w && net->n_hidden == h && fused_precision_ok(net))                        \
        return QuadCfg<T>::OK && tuning().pair_lanes == 4 ? 4 : 1;
    NEPX_FUSED_CASES(X)
#undef X
    return 0;
}

template <class Cfg, class N, int PREC>
static void launch_fused_p(const nepx_pair_model& m, const nepx_net* net, int grid, float scale, const float* qf,
                           const int32_t* pair_i, const int32_t* pair_j, const float* pair_t,
                           const int32_t* np_dev, int64_t maxp, float clip, float* out, RevOut rv, void* stream) {
#define NEPX_LAUNCH_FUSED(A)                                                                                     \
    hipLaunchKernelGGL((k_fused<Cfg, N, PREC, A>), dim3(grid), dim3(kBlock), 0, as_stream(stream), m,            \
                       net->w_packed, net->w_half, net->en_min, scale, (const float4*)qf, pair_i, pair_j,          \
                       (const float4*)pair_t, np_dev, maxp, clip, out, rv)
    if (net->act == NEPX_ACT_TANH) NEPX_LAUNCH_FUSED(NEPX_ACT_TANH);
    else if constexpr (PREC == NEPX_NET_F32 || PREC == NEPX_NET_F16X3) NEPX_LAUNCH_FUSED(NEPX_ACT_RELU);
#undef NEPX_LAUNCH_FUSED
}

template <class Cfg, class N>
static int launch_fused(const nepx_pair_model& m, const nepx_net* net, float scale,
                        const float* qf, const int32_t* pair_i, const int32_t* pair_j, const float* pair_t,
                        const int32_t* np_dev, int64_t maxp, float clip, float* out, RevOut rv, void* stream) {
    const int64_t cap = (int64_t)device_cus() * tuning().fused_blocks_per_cu;
    // four lanes per pair (site sums on MFMA) where the shape allows it, unless tuned off
    if (tuning().pair_lanes == 4) {
        const int rc = launch_fused_quad<Cfg, N>(m, net, net->precision, (int)cap, scale, qf, pair_i, pair_j,
                                                 pair_t, np_dev, maxp, clip, out, rv, stream);
        if (rc != NEPX_EUNSUP) return rc;
    }
    const int grid = grid_for_cap(maxp, kBlock, cap);
    switch (net->precision) {
        case NEPX_NET_F16X3:
            launch_fused_p<Cfg, N, NEPX_NET_F16X3>(m, net, grid, scale, qf, pair_i, pair_j, pair_t, np_dev, maxp,
                                                    clip, out, rv, stream);
            break;
        case NEPX_NET_BF16:
            launch_fused_p<Cfg, N, NEPX_NET_BF16>(m, net, grid, scale, qf, pair_i, pair_j, pair_t, np_dev, maxp,
                                                   clip, out, rv, stream);
            break;
        case NEPX_NET_BF16X3:
            launch_fused_p<Cfg, N, NEPX_NET_BF16X3>(m, net, grid, scale, qf, pair_i, pair_j, pair_t, np_dev,
                                                     maxp, clip, out, rv, stream);
            break;
        default:
            launch_fused_p<Cfg, N, NEPX_NET_F32>(m, net, grid, scale, qf, pair_i, pair_j, pair_t, np_dev, maxp,
                                                  clip, out, rv, stream);
    }
    NEPX_LAUNCH_CHECK();
    return NEPX_OK;
}

static int pair_fused(const nepx_pair_model* m, const nepx_net* net, const float* qf, const int32_t* pair_i,
                      const int32_t* pair_j, const float* pair_t, const int32_t* np_dev, int64_t maxp, float clip,
                      float* out, RevOut rv, void* stream) {
    int rc = check_model(m);
    if (rc) return rc;
    rc = check_net(net, model_D(m));
    if (rc) return rc;
    rc = check_precision(net);
    if (rc) return rc;
    NEPX_REQUIRE(qf && pair_i && pair_j && pair_t && np_dev && out, NEPX_EINVAL, "null buffer");
    if (maxp <= 0) return NEPX_OK;
    const float scale = net->en_max - net->en_min;
#define X(ns, a, b, c, T, d, w, h, NT)                                                               \
    if (m->n_sites == ns && m->nrad == a && m->nang == b && m->lmax == c && net->d_in == d &&        \
        net->width == w && net->n_hidden == h)                                                       \
        return launch_fused<T, NT>(*m, net, scale, qf, pair_i, pair_j, pair_t, np_dev, maxp, clip, out, rv, stream);
    NEPX_FUSED_CASES(X)
#undef X
    set_error("no fused kernel for n_sites=%d hypers=(%d,%d,%d) net %d->%dx%d", m->n_sites, m->nrad,
              m->nang, m->lmax, net->d_in, net->width, net->n_hidden + 1);
    return NEPX_EUNSUP;
}

extern "C" int nepx_pair_fused(const nepx_pair_model* m, const nepx_net* net, const float* qf,
                               const int32_t* pair_i, const int32_t* pair_j, const float* pair_t,
                               const int32_t* np_dev, int64_t maxp, float clip, float* out, void* stream) {
    return pair_fused(m, net, qf, pair_i, pair_j, pair_t, np_dev, maxp, clip, out, RevOut{}, stream);
}

extern "C" int nepx_pair_fused_list(const nepx_pair_model* m, const nepx_net* net, const nepx_state* st,
                                    nepx_nlist* nl, float clip, float* out, void* stream) {
    NEPX_REQUIRE(st && nl && st->qf && nl->flags, NEPX_EINVAL, "null state or list");
    NEPX_REQUIRE(!(nl->pair_e || nl->rrec) || (nl->rpos && nl->pair_e && nl->rrec), NEPX_EINVAL,
                 "reverse-order records need rpos, pair_e and rrec together");
    RevOut rv;
    if (nl->rrec) {
        rv.pe = nl->pair_e;
        rv.rrec = nl->rrec;
        rv.flags = nl->flags;
    }
    return pair_fused(m, net, st->qf, nl->pair_i, nl->pair_j, nl->pair_t, nl->flags + F_P, nl->cap, clip, out, rv,
                      stream);
}

extern "C" int nepx_stencil_rows(const float* qf, const int32_t* pair_i, const int32_t* pair_j, const float* pair_t,
                                 int64_t P, float dx, float dteta, float* q_rows, int32_t* row_i, int32_t* row_j,
                                 float* t_rows, void* stream) {
    NEPX_REQUIRE(P >= 0 && P <= (int64_t)1 << 27, NEPX_ECAP, "pair count %lld out of range", (long long)P);
    if (P == 0) return NEPX_OK;
    NEPX_REQUIRE(qf && pair_i && pair_j && pair_t && q_rows && row_i && row_j && t_rows, NEPX_EINVAL, "null buffer");
    const int rows = (int)(10 * P);
    hipLaunchKernelGGL(k_stencil_rows, dim3((rows + kBlock - 1) / kBlock), dim3(kBlock), 0, as_stream(stream),
                       (const float4*)qf, pair_i, pair_j, (const float4*)pair_t, (int)P, dx, dteta,
                       (float4*)q_rows, row_i, row_j, (float4*)t_rows);
    NEPX_LAUNCH_CHECK();
    return NEPX_OK;
}

extern "C" int nepx_fd_forces(const float* E_rows, int64_t P, float dx, float dteta, float clip, float* out,
                              void* stream) {
    NEPX_REQUIRE(P >= 0 && P <= (int64_t)1 << 27, NEPX_ECAP, "pair count %lld out of range", (long long)P);
    if (P == 0) return NEPX_OK;
    NEPX_REQUIRE(E_rows && out, NEPX_EINVAL, "null buffer");
    NEPX_REQUIRE(dx != 0.f && dteta != 0.f, NEPX_EINVAL, "zero finite-difference step");
    hipLaunchKernelGGL(k_fd_forces, dim3((P + kBlock - 1) / kBlock), dim3(kBlock), 0, as_stream(stream), E_rows,
                       (int)P, dx, dteta, clip, out);
    NEPX_LAUNCH_CHECK();
    return NEPX_OK;
}

// ---------------------------------------------------------------------------
// Descriptors of site clouds, one cloud per lane (four lanes: nepx_quad_cloud.h): nd points of a cloud (xyz
// interleaved) about their centroid, optional per-point weights.
struct CloudSites {
    const float* __restrict__ pts;
    const float* __restrict__ w;
    int nd;
    float cx, cy, cz, inv_rn;
    __device__ __forceinline__ CloudSites(const float* pts_, const float* w_, int nd_, float inv_rn_)
        : pts(pts_), w(w_), nd(nd_), inv_rn(inv_rn_) {
        float sx = 0.f, sy = 0.f, sz = 0.f;
        for (int a = 0; a < nd; ++a) {
            sx += pts[3 * a];
            sy += pts[3 * a + 1];
            sz += pts[3 * a + 2];
        }
        const float inv = 1.f / (float)nd;
        cx = sx * inv;
        cy = sy * inv;
        cz = sz * inv;
    }
    template <class S, class B>
    __device__ __forceinline__ void visit(S&& site, B&& body_done) const {
#pragma unroll 1
        for (int a = 0; a < nd; ++a) {
            SiteGeo s;
            s.ax = s.ay = s.az = 0.f;
            const float rx = pts[3 * a] - cx, ry = pts[3 * a + 1] - cy, rz = pts[3 * a + 2] - cz;
            const float r2 = rx * rx + ry * ry + rz * rz;
            s.ir = __builtin_amdgcn_rsqf(r2);
            s.r = r2 * s.ir;
            s.ux = rx * s.ir;
            s.uy = ry * s.ir;
            s.uz = rz * s.ir;
            s.rho = s.r * inv_rn;
            site(s, w ? w[a] : 1.f);
        }
        body_done(0);
    }
};

template <class Cfg>
__global__ __launch_bounds__(kBlock) void k_cloud_desc(const float* __restrict__ clouds, int64_t P, int nd,
                                                       const float* __restrict__ w, float r_nep,
                                                       float* __restrict__ G) {
    for (int64_t idx = blockIdx.x * (int64_t)kBlock + threadIdx.x; idx < P; idx += (int64_t)gridDim.x * kBlock) {
        const CloudSites sites(clouds + idx * 3 * (int64_t)nd, w, nd, 1.f / r_nep);
        if constexpr (Cfg::ONE_PASS) {
            float Gr[Cfg::D];
            desc_forward_sites<Cfg>(sites, Gr);
            store_row<Cfg>(G + idx * Cfg::D, Gr);
        } else {
            desc_forward_sites<Cfg>(sites, G + idx * Cfg::D);
        }
    }
}

// Many clouds of 1, 2, 5 or 6 sites take one lane each where the rows are seven n wide: a quad's last trip is
// then half idle, and closing a tile costs more than the sites.  One lane -> four lanes per cloud:
//   hypers 11 6 4, 1,000,000 clouds: 1 site 57 -> 64 us, 2 sites 62 -> 66, 3 sites 67 -> 66, 4 sites 72 -> 66,
//     5 sites 79 -> 92, 6 sites 85 -> 94, 8 sites 99 -> 97; 60,000 clouds: 5 sites 9.4 -> 9.3, 6 sites 10.0 -> 9.4
//   hypers 17 6 6, 1,000,000 clouds: 1 site 94 -> 127 us, 2 sites 107 -> 128, 3 sites 122 -> 126, 4 sites
//     135 -> 127, 5 sites 151 -> 174, 6 sites 162 -> 174, 8 sites 202 -> 176; 100,000 clouds: 5 sites 20.5 -> 22.8;
//     60,000 clouds: 5 sites 15.8 -> 15.1, 6 sites 17.4 -> 15.2
// From seven sites on, and with the other hypers, four lanes gain at every size.
template <class Cfg>
constexpr bool few_sites_on_lanes() { return Cfg::NANG == 6; }
static bool one_lane_clouds(int64_t n_clouds, int n_sites) {
    return n_sites <= 6 && (n_sites - 1) % 4 < 2 && n_clouds >= 320 * (int64_t)device_cus();
}

template <class Cfg>
static int launch_clouds(const float* clouds, int64_t n_clouds, int n_sites, const float* site_w, float r_nep,
                         float* G, void* stream) {
    if constexpr (few_sites_on_lanes<Cfg>()) {
        if (one_lane_clouds(n_clouds, n_sites)) {
            hipLaunchKernelGGL(k_cloud_desc<Cfg>, dim3(grid_for(n_clouds, kBlock)), dim3(kBlock), 0,
                               as_stream(stream), clouds, n_clouds, n_sites, site_w, r_nep, G);
            NEPX_LAUNCH_CHECK();
            return NEPX_OK;
        }
    }
    return launch_cloud_quad<Cfg>(clouds, n_clouds, n_sites, site_w, r_nep, G, stream);
}

extern "C" int nepx_cloud_descriptor(const float* clouds, int64_t n_clouds, int32_t n_sites, const float* site_w,
                                     int32_t nrad, int32_t nang, int32_t lmax, float r_nep, float* G,
                                     void* stream) {
    NEPX_REQUIRE(n_clouds >= 0 && n_sites > 0, NEPX_EINVAL, "bad cloud count %lld or size %d",
                 (long long)n_clouds, n_sites);
    NEPX_REQUIRE(r_nep > 0.f, NEPX_EINVAL, "r_nep must be positive");
    if (n_clouds == 0) return NEPX_OK;
    NEPX_REQUIRE(clouds && G, NEPX_EINVAL, "null buffer");
#define X(a, b, c)                                                                                       \
    if (nrad == a && nang == b && lmax == c)                                                             \
        return launch_clouds<DescCfg<1, a, b, c>>(clouds, n_clouds, (int)n_sites, site_w, r_nep, G, stream);
    NEPX_CLOUD_CASES(X)
#undef X
    set_error("no cloud descriptor kernel for hypers (%d, %d, %d)", nrad, nang, lmax);
    return NEPX_EUNSUP;
}
