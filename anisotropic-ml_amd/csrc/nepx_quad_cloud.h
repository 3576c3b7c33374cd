// Descriptors of site clouds (training-set featurisation, 05/NEP.py:171-219 get_g_fast and
// 04/Processors.py:48-88): four lanes per cloud, 16 clouds per tile, the angular sums
// A_nlm = sum_a w_a f_n(a) Z_lm(a) on v_mfma_f32_4x4x1_16b_f32 as in the fused kernel (nepx_quad.h).
// Each lane evaluates every fourth site; lanes past the last site carry weight zero.  A tile's harmonics
// of hypers 10 10 10 are spread over four waves by sets of m (nepx_msets.h), whose sums of squares meet
// in LDS; the other hypers take one wave.  The descriptor rows of a tile are contiguous, so they are
// assembled in LDS and stored whole.
//
// One lane per cloud held at most 176 accumulators, so hypers 10 8 4 walked the sites twice and
// 10 10 10 eight times, and its loads and stores strode by whole clouds and rows.  The bound is issue:
// VALU work (radial functions, harmonics, sums of squares; 865 instructions per tile of 12 sites, hypers
// 10 8 4) and the products, next to the memory traffic.  12 sites: hypers 10 8 4, 1,000,003 clouds
// 252 -> 156 us (2.1 TB/s), 5,000 clouds 17 -> 11 us; hypers 10 10 10, 1,375 -> 977 us, 5,000 clouds
// 80 -> 11 us.  Many clouds of a few sites stay one to a lane (launch_clouds).
#pragma once
#include "nepx_msets.h"
#include "nepx_quad.h"

namespace nepx {

template <class Cfg>
struct QuadCloud {
    using MG = MGroups<Cfg::LMAX>;
    static constexpr int NA = Cfg::NANG + 1, NC = (NA + 3) / 4, BLOCK = 64 * MG::COUNT;
    static constexpr int TS = (NC + max_chunks<MG>()) * 16 + 4;  // exchange floats per cloud, TS / 4 odd
    static_assert(Cfg::D <= TS, "a descriptor row fits in the exchange area");
    // Clouds of up to this many sites are staged in LDS; larger ones are read from memory where they are
    // needed (a tile's coordinates would take LDS from other waves).
    static constexpr int STAGED = 64;
    // waves per SIMD that the accumulators leave room for, and the blocks of a CU that come of it: the grid
    // is what runs at once, so that every block has the same share of the tiles
    static constexpr int WAVES_PER_SIMD = NC * max_chunks<MG>() <= 18 ? 3 : 2;
    static constexpr int BLOCKS_PER_CU = 4 * WAVES_PER_SIMD / MG::COUNT;
};

// Sums over one cloud's sites for the harmonics of MS: g_ang[n][l] (the set's share) and, with RAD,
// g_rad[n], the same in the cloud's four lanes.  sites_done() is called after the last read of pts.
template <class Cfg, class MS, bool RAD, class Done>
__device__ __forceinline__ void quad_cloud_sums(const float* pts, const float* __restrict__ w, int nd,
                                                float inv_rn, float cx, float cy, float cz, float* xp, int q,
                                                float (&gr)[Cfg::NRAD + 1],
                                                float (&ga)[Cfg::NANG + 1][Cfg::LMAX], Done&& sites_done) {
    using Q = QuadCloud<Cfg>;
    constexpr int NC = Q::NC, NA = Q::NA, LC = (MS::N + 3) / 4, LMAX = Cfg::LMAX;
    // The set's first l, a compile-time constant: found at run time it leaves the sums below in scratch memory,
    // walked by loops (hypers 10 10 10: 50 us a tile, 50,000 clouds of 12 sites 325 us against 55 us).
    constexpr int FIRST = MS::l_of(0);
    v4f Af[NC][LC];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int d = 0; d < LC; ++d) Af[c][d] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int n = 0; n <= Cfg::NRAD; ++n) gr[n] = 0.f;
#pragma unroll 1
    for (int a0 = 0; a0 < nd; a0 += 4) {
        const int a = a0 + q;
        const bool in = a < nd;
        float rx = 1.f, ry = 0.f, rz = 0.f, wa = 0.f;
        if (in) {
            rx = pts[3 * a] - cx;
            ry = pts[3 * a + 1] - cy;
            rz = pts[3 * a + 2] - cz;
            wa = w ? w[a] : 1.f;
        }
        const float r2 = rx * rx + ry * ry + rz * rz;
        const float ir = __builtin_amdgcn_rsqf(r2);
        float fv[4 * NC];
#pragma unroll
        for (int n = NA; n < 4 * NC; ++n) fv[n] = 0.f;
        radial_values<RAD ? Cfg::NRAD : Cfg::NANG>(in ? r2 * ir * inv_rn : 0.f, wa, [&](int n, float f) {
            if constexpr (RAD) gr[n] += f;
            if (n < NA) fv[n] = f;
        });
        HarmM<MS> h;
        h.eval(rx * ir, ry * ir, rz * ir);
        wave_lds_order();  // after the previous trip's reads
#pragma unroll
        for (int n = 0; n < 4 * NC; ++n) xp[16 * (n / 4) + 4 * (n % 4) + q] = fv[n];
#pragma unroll
        for (int mm = 0; mm <= LMAX; ++mm)
#pragma unroll
            for (int part = 0; part < (MS::has(mm) ? (mm ? 2 : 1) : 0); ++part)
#pragma unroll
                for (int l = MS::first_l(mm); l <= LMAX; ++l) {
                    const int o = MS::slot(l, mm, part);
                    xp[16 * (NC + o / 4) + 4 * (o % 4) + q] = h.z(l, mm, part);
                }
#pragma unroll
        for (int o = MS::N; o < 4 * LC; ++o) xp[16 * (NC + o / 4) + 4 * (o % 4) + q] = 0.f;
        wave_lds_order();
        v4f xf[NC], xz[LC];
#pragma unroll
        for (int c = 0; c < NC; ++c) xf[c] = *reinterpret_cast<const v4f*>(xp + 16 * c + 4 * q);
#pragma unroll
        for (int d = 0; d < LC; ++d) xz[d] = *reinterpret_cast<const v4f*>(xp + 16 * (NC + d) + 4 * q);
        // one block of products at the lower wave priority, so that other waves' VALU work issues first
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(0);
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int d = 0; d < LC; ++d)
                    Af[c][d] = __builtin_amdgcn_mfma_f32_4x4x1f32(xf[c][k], xz[d][k], Af[c][d], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
    }
    sites_done();
    if constexpr (RAD) {
#pragma unroll
        for (int n = 0; n <= Cfg::NRAD; ++n) gr[n] = quad_sum(gr[n]);
    }
#pragma unroll
    for (int n = 0; n < NA; ++n)
#pragma unroll
        for (int l = 0; l < LMAX; ++l) ga[n][l] = 0.f;
    // This lane's column of chunk d is slot 4d + q; a chunk spans two l at most.  A lane adds to its slot's own l
    // only: with a zero weight for the other, a square past FP32's range (large site weights) would be NaN there
    // (the selects: 1,000,003 clouds of 12 sites, hypers 10 8 4, 152 -> 154 us).
    static_for<LC>([&](auto dc) {
        constexpr int d = decltype(dc)::value, last = 4 * d + 3 < MS::N ? 4 * d + 3 : MS::N - 1;
        constexpr int lo = MS::l_of(4 * d), hi = MS::l_of(last);
        constexpr float w0 = MS::k2(4 * d), w1 = MS::k2(4 * d + 1), w2 = MS::k2(4 * d + 2), w3 = MS::k2(4 * d + 3);
        constexpr int up = MS::off(hi) - 4 * d;  // first lane of the upper l
        static_assert(hi <= lo + 1, "a chunk spans two l at most");
        const float kk = sel4(q, w0, w1, w2, w3);
        const bool below = lo == hi || q < up;
#pragma unroll
        for (int n = 0; n < NA; ++n) {
            const float v = Af[n / 4][d][n % 4];
            const float v2 = v * v;
            ga[n][lo - 1] += kk * (below ? v2 : 0.f);
            if (lo != hi) ga[n][hi - 1] += kk * (below ? 0.f : v2);
        }
    });
#pragma unroll
    for (int n = 0; n < NA; ++n)
#pragma unroll
        for (int l = FIRST - 1; l < LMAX; ++l) ga[n][l] = quad_sum(ga[n][l]);  // zero below the set's first l
}

// STAGED: the coordinates of the next tile go straight from memory to LDS (no registers) while this tile's
// sums of squares are formed, so a wave does not wait for memory once per trip.
template <class Cfg, bool STAGED>
__global__ __launch_bounds__((QuadCloud<Cfg>::BLOCK)) __attribute__((
    amdgpu_waves_per_eu(QuadCloud<Cfg>::WAVES_PER_SIMD, QuadCloud<Cfg>::WAVES_PER_SIMD))) void k_cloud_quad(
    const float* __restrict__ clouds, int64_t P, int nd, const float* __restrict__ w, float r_nep,
    float* __restrict__ G) {
    using Q = QuadCloud<Cfg>;
    using MG = typename Q::MG;
    constexpr int PW = 16, D = Cfg::D, COUNT = MG::COUNT, GA = Cfg::NRAD + 1, LMAX = Cfg::LMAX;
    __shared__ __attribute__((aligned(16))) float xch[COUNT][PW * Q::TS];
    extern __shared__ float coords[];  // a tile's clouds (STAGED)
    const int lane = threadIdx.x & 63, q = lane & 3, slot = lane >> 2;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float* const xp = xch[wave] + slot * Q::TS;
    float* const row = xch[wave] + slot * D;  // the set's descriptor row (reuses the exchange area)
    const float inv_rn = 1.f / r_nep;
    const bool wide = ((uintptr_t)G & 15) == 0;  // whole tiles are then stored 16 bytes at a time
    auto fetch = [&](int64_t base) {  // a tile's coordinates are contiguous in memory
        if constexpr (STAGED) {
            if (base >= P) return;
            const int have = (int)(P - base < PW ? P - base : PW) * 3 * nd;
            const float* src = clouds + base * 3 * nd;
            for (int e0 = wave * 64; e0 < have; e0 += Q::BLOCK) {
                if (e0 + lane < have)
                    __builtin_amdgcn_global_load_lds(
                        (const __attribute__((address_space(1))) void*)(src + e0 + lane),
                        (__attribute__((address_space(3))) void*)(coords + e0), 4, 0, 0);
            }
        }
    };
    auto arrived = [&]() {
        if constexpr (STAGED) __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wave's copies are in LDS
    };
    fetch((int64_t)blockIdx.x * PW);
    arrived();
    __syncthreads();
    for (int64_t base = (int64_t)blockIdx.x * PW; base < P; base += (int64_t)gridDim.x * PW) {  // uniform per block
        const int last = (int)(P - base < PW ? P - base : PW) - 1;
        const int here = slot < last ? slot : last;  // quads past the end repeat the last cloud
        const float* pts;
        if constexpr (STAGED) pts = coords + here * 3 * nd;
        else pts = clouds + (base + here) * 3 * (int64_t)nd;
        float sx = 0.f, sy = 0.f, sz = 0.f;
        for (int a = q; a < nd; a += 4) {
            sx += pts[3 * a];
            sy += pts[3 * a + 1];
            sz += pts[3 * a + 2];
        }
        const float inv = 1.f / (float)nd;
        const float cx = quad_sum(sx) * inv, cy = quad_sum(sy) * inv, cz = quad_sum(sz) * inv;
        static_for<COUNT>([&](auto gc) {
            constexpr int S = decltype(gc)::value;
            using MS = typename MG::template Set<S>;
            if (COUNT == 1 || wave == S) {  // every wave runs one set: one barrier in sites_done each
                float gr[Cfg::NRAD + 1], ga[Cfg::NANG + 1][LMAX];
                quad_cloud_sums<Cfg, MS, S == MG::RAD>(pts, w, nd, inv_rn, cx, cy, cz, xp, q, gr, ga, [&]() {
                    if constexpr (STAGED) {
                        __syncthreads();  // every wave has read this tile's sites
                        fetch(base + (int64_t)gridDim.x * PW);
                    }
                });
                wave_lds_order();  // the exchange reads are done before the rows overwrite the area
#pragma unroll
                for (int n = 0; n <= Cfg::NRAD; ++n) row[n] = S == MG::RAD ? gr[n] : 0.f;
#pragma unroll
                for (int n = 0; n <= Cfg::NANG; ++n)
#pragma unroll
                    for (int l = 0; l < LMAX; ++l) row[GA + n * LMAX + l] = ga[n][l];
            }
        });
        arrived();  // before the stores below, which it would wait for as well
        __syncthreads();
        if (wide && last == PW - 1) {
            v4f* const dst = reinterpret_cast<v4f*>(G + base * D);
#pragma unroll
            for (int k = 0; k < (PW * D / 4 + Q::BLOCK - 1) / Q::BLOCK; ++k) {
                const int e = k * Q::BLOCK + threadIdx.x;
                if (e < PW * D / 4) {
                    v4f v = *reinterpret_cast<const v4f*>(&xch[0][4 * e]);
#pragma unroll
                    for (int s = 1; s < COUNT; ++s) v += *reinterpret_cast<const v4f*>(&xch[s][4 * e]);
                    dst[e] = v;
                }
            }
        } else {
            for (int k = threadIdx.x; k < (last + 1) * D; k += Q::BLOCK) {
                float v = xch[0][k];
#pragma unroll
                for (int s = 1; s < COUNT; ++s) v += xch[s][k];
                G[base * D + k] = v;
            }
        }
        __syncthreads();  // the rows are read before the next tile's exchange overwrites them
    }
}

}  // namespace nepx
