// Descriptor adjoint from dE/dG in memory with the per-pair contractions on matrix cores: four lanes
// per pair, 16 pairs per tile, as in the fused kernel (nepx_quad.h has the layout of the
// v_mfma_f32_4x4x1_16b_f32 products), for the shapes whose network has no fused kernel.
//
// The one-lane-per-pair adjoint (k_adjoint) cuts the l range into passes that fit one lane's registers
// and evaluates the sites' geometry, radial functions and harmonics again for every pass, forward and
// back: eight passes for hypers 10 10 10.  Here the harmonics are cut by m (nepx_msets.h).  Each
// group of a tile runs on its own wave (hypers 10 10 10: m = {0, 1}, {2, 5}, {3, 4} and {6..10}, 30 of
// the 120 harmonics each, two waves per SIMD; hypers 10 8 4: {0, 1} and {2, 3, 4}), and the groups' per-body
// sums meet in LDS in a fixed order.  Sites' geometry and radial functions are evaluated once per tile, the
// trips dealt to the waves, and read from LDS.  The bound is VALU issue (site geometry, radial functions and the
// per-site gradient sums) and, with two waves per SIMD, the waits of its chains.  8 (12) sites, hypers
// 10 10 10: 241 pairs 45 -> 13 us (61 -> 13), 20,000 pairs 92 -> 46 us (128 -> 57), 100,001 pairs
// 300 -> 190 us (419 -> 230); hypers 10 8 4: 241 pairs 15 -> 13 us (20 -> 13), 100,001 pairs 52 -> 47 us
// (71 -> 59); more than 896 pairs a CU of 8 sites go one to a lane (launch_adjoint).
#pragma once
#include "nepx_msets.h"
#include "nepx_quad.h"

namespace nepx {

// The part of angular_site_grad (nepx_desc.h) that the m of a set contribute.
template <class MS, class CD>
__device__ __forceinline__ void angular_site_grad_m(const HarmM<MS>& h, float ux, float uy, CD&& cd, float& dEdrho,
                                                    float& gx, float& gy, float& gz) {
    float E1 = 0.f, Gz = 0.f, X1 = 0.f, Y1 = 0.f;
#pragma unroll
    for (int mm = 0; mm <= MS::LMAX; ++mm) {
        if (!MS::has(mm)) continue;
        float U[2] = {0.f, 0.f}, V[2] = {0.f, 0.f}, W[2] = {0.f, 0.f}, Dq[2] = {0.f, 0.f};
#pragma unroll
        for (int l = MS::first_l(mm); l <= MS::LMAX; ++l) {
            const float ql = h.q(l, mm);
            const float qa = (mm + 1 <= l - 1) ? h.q(l - 1, mm + 1) : 0.f;
            const float qc = (mm <= l - 1) ? (float)(l + mm) * h.q(l - 1, mm) : 0.f;
#pragma unroll
            for (int part = 0; part < (mm ? 2 : 1); ++part) {
                float c, d;
                cd(MS::slot(l, mm, part), c, d);
                Dq[part] += d * ql;
                if (mm + 1 <= l - 1) U[part] += qa * c;
                if (mm <= l - 1) V[part] += qc * c;
                if (mm >= 1) W[part] += ql * c;
            }
        }
        dEdrho += mm == 0 ? Dq[0] : h.C[mm] * Dq[0] + h.S[mm] * Dq[1];
        if (mm == 0) {
            E1 += U[0];
            Gz += V[0];
        } else {
            E1 += h.C[mm] * U[0] + h.S[mm] * U[1];
            Gz += h.C[mm] * V[0] + h.S[mm] * V[1];
            const float fm = (float)mm;
            X1 += fm * (h.C[mm - 1] * W[0] + h.S[mm - 1] * W[1]);
            Y1 += fm * (h.C[mm - 1] * W[1] - h.S[mm - 1] * W[0]);
        }
    }
    gx = ux * E1 + X1;
    gy = uy * E1 + Y1;
    gz = Gz;
}

// The adjoint's sets: hypers 10 8 4 take two waves of 12 harmonics each, as one wave's sites would fill the
// LDS of a whole SIMD's waves.  (One wave of all 24, each wave evaluating its own sites, took 50 (40) us at
// 100,001 pairs of 12 (8) sites, but its sums lay further from 64 bits: 8.4e-7 against 8.0e-7 at 12 sites.)
template <int LMAX>
struct AdjSets : MGroups<LMAX> {};
template <>
struct AdjSets<4> {
    static constexpr int COUNT = 2, RAD = 1;
    static constexpr unsigned MASK[2] = {0x03, 0x1c};
    template <int G>
    using Set = MSet<4, MASK[G]>;
};

template <class Cfg>
struct QuadAdj {
    using MG = AdjSets<Cfg::LMAX>;
    static constexpr int NA = Cfg::NANG + 1, NC = (NA + 3) / 4, STEPS = Cfg::ND / 4, BLOCK = 64 * MG::COUNT;
    static_assert(MG::COUNT > 1, "the groups' sums meet in LDS");
    static constexpr bool OK = Cfg::ND % 4 == 0;
    // floats per pair of a trip's f and f' and of a wave's harmonics: strides of 4 odd keep the lanes' 64
    // scalar writes on 64 banks
    static constexpr int FS = NC * 16 + 4, TS = max_chunks<MG>() * 16 + 4;
};

// What every wave of a tile needs of its sites, evaluated once: trip s holds the tile's 64 sites 4 s + q.
template <class Cfg>
struct QuadSites {
    using Q = QuadAdj<Cfg>;
    float4 u[Q::STEPS][64];    // unit vector from the centroid, 1 / distance
    float4 arm[Q::STEPS][64];  // lever arm about the body's centre, sum_n dE/dg_rad[n] f_n'
    float f[Q::STEPS][16][Q::FS];   // value 4 ch + i of site 4 s + q at 16 ch + 4 i + q (rows past NANG zero)
    float df[Q::STEPS][16][Q::FS];  // f_n' of site 4 s + q at 4 NC q + n
    float s[6][16];                 // the pairs' arm sums s_i and s_j
};

template <class Cfg>
__device__ __forceinline__ void quad_adjoint_site(const nepx_pair_model& m, const float4* stab, const PairIn& g,
                                                  const float* grow, int s, int lane, QuadSites<Cfg>& st) {
    using Q = QuadAdj<Cfg>;
    constexpr int NC = Q::NC, NA = Q::NA;
    const int q = lane & 3, slot = lane >> 2, a = 4 * s + q;
    const bool bj = a >= Cfg::NS;
    const float4 b = stab[a];
    const Mat3 Rb = quat_matrix(bj ? g.qj.x : g.qi.x, bj ? g.qj.y : g.qi.y, bj ? g.qj.z : g.qi.z,
                                bj ? g.qj.w : g.qi.w);
    const SiteGeo sg = site_geo_b(Rb, b.x, b.y, b.z, (bj ? g.tx : 0.f) - g.cx, (bj ? g.ty : 0.f) - g.cy,
                                  (bj ? g.tz : 0.f) - g.cz, 1.f / m.r_nep);
    float fv[4 * NC], dv[4 * NC];
#pragma unroll
    for (int n = NA; n < 4 * NC; ++n) fv[n] = dv[n] = 0.f;
    float rad = 0.f;
    radial_derivs<Cfg::NRAD>(sg.rho, [&](int n, float f, float df) {
        rad += grow[n] * df;
        if (n < NA) {
            fv[n] = f;
            dv[n] = df;
        }
    });
    st.u[s][lane] = make_float4(sg.ux, sg.uy, sg.uz, sg.ir);
    st.arm[s][lane] = make_float4(sg.ax, sg.ay, sg.az, rad);
    float* const fp = st.f[s][slot];
    float* const dp = st.df[s][slot] + 4 * NC * q;
#pragma unroll
    for (int n = 0; n < 4 * NC; ++n) fp[16 * (n / 4) + 4 * (n % 4) + q] = fv[n];
#pragma unroll
    for (int c = 0; c < NC; ++c)
        *reinterpret_cast<v4f*>(dp + 4 * c) = v4f{dv[4 * c], dv[4 * c + 1], dv[4 * c + 2], dv[4 * c + 3]};
}

// One tile's sums over its sites for the harmonics of MS (and the radial terms with RAD): dE/dr and
// arm x dE/dr per body, the same in all four lanes of a pair.
template <class Cfg, class MS, bool RAD>
__device__ __forceinline__ void quad_adjoint_sums(float inv_rn, const QuadSites<Cfg>& st, const float* grow, float* xp,
                                                  int lane, float (&sum)[12]) {
    using Q = QuadAdj<Cfg>;
    constexpr int NC = Q::NC, NA = Q::NA, LC = (MS::N + 3) / 4, LMAX = Cfg::LMAX;
    constexpr int GA = Cfg::NRAD + 1;
    const int q = lane & 3, slot = lane >> 2;
    // ---- forward: A[n][slot] ----
    v4f Af[NC][LC];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int d = 0; d < LC; ++d) Af[c][d] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int s = 0; s < Q::STEPS; ++s) {
        const float4 u = st.u[s][lane];
        HarmM<MS> h;
        h.eval(u.x, u.y, u.z);
        wave_lds_order();  // after the previous trip's reads
#pragma unroll
        for (int mm = 0; mm <= LMAX; ++mm)
#pragma unroll
            for (int part = 0; part < (MS::has(mm) ? (mm ? 2 : 1) : 0); ++part)
#pragma unroll
                for (int l = MS::first_l(mm); l <= LMAX; ++l) {
                    const int o = MS::slot(l, mm, part);
                    xp[16 * (o / 4) + 4 * (o % 4) + q] = h.z(l, mm, part);
                }
#pragma unroll
        for (int o = MS::N; o < 4 * LC; ++o) xp[16 * (o / 4) + 4 * (o % 4) + q] = 0.f;
        wave_lds_order();
        v4f xf[NC], xz[LC];
#pragma unroll
        for (int c = 0; c < NC; ++c) xf[c] = *reinterpret_cast<const v4f*>(st.f[s][slot] + 16 * c + 4 * q);
#pragma unroll
        for (int d = 0; d < LC; ++d) xz[d] = *reinterpret_cast<const v4f*>(xp + 16 * d + 4 * q);
        // each trip's products are one block at the lower wave priority, so that the other waves' VALU
        // work issues first (as in the fused kernel)
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
    // ---- B = dE/dA = 2 K^2 dE/dg_ang[n][l] A: this lane's column of chunk d is slot 4d + q ----
    static_for<LC>([&](auto dc) {
        constexpr int d = decltype(dc)::value;
        constexpr float w0 = 2.f * MS::k2(4 * d), w1 = 2.f * MS::k2(4 * d + 1), w2 = 2.f * MS::k2(4 * d + 2),
                        w3 = 2.f * MS::k2(4 * d + 3);
        constexpr int a0 = MS::row_of(4 * d), a1 = MS::row_of(4 * d + 1), a2 = MS::row_of(4 * d + 2),
                      a3 = MS::row_of(4 * d + 3);
        const float kw = sel4(q, w0, w1, w2, w3);
        const float* row = grow + GA + (q == 0 ? a0 : q == 1 ? a1 : q == 2 ? a2 : a3);
#pragma unroll
        for (int n = 0; n < NA; ++n) Af[n / 4][d][n % 4] *= kw * row[n * LMAX];
    });
    // ---- adjoint ----
    float ig_x = 0.f, ig_y = 0.f, ig_z = 0.f, it_x = 0.f, it_y = 0.f, it_z = 0.f;
    float jg_x = 0.f, jg_y = 0.f, jg_z = 0.f, jt_x = 0.f, jt_y = 0.f, jt_z = 0.f;
#pragma unroll 1
    for (int s = 0; s < Q::STEPS; ++s) {
        const float4 u = st.u[s][lane], arm = st.arm[s][lane];
        float fa[NA];
        v4f da[NC];
#pragma unroll
        for (int n = 0; n < NA; ++n) fa[n] = st.f[s][slot][16 * (n / 4) + 4 * (n % 4) + q];
#pragma unroll
        for (int c = 0; c < NC; ++c) da[c] = *reinterpret_cast<const v4f*>(st.df[s][slot] + 4 * NC * q + 4 * c);
        v4f cc[LC], dd[LC];
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(0);
#pragma unroll
        for (int n = 0; n < NA; ++n)
#pragma unroll
            for (int d = 0; d < LC; ++d) {
                const float b = Af[n / 4][d][n % 4];
                const v4f z4 = {0.f, 0.f, 0.f, 0.f};
                cc[d] = __builtin_amdgcn_mfma_f32_4x4x1f32(b, fa[n], n == 0 ? z4 : cc[d], 0, 0, 0);
                dd[d] = __builtin_amdgcn_mfma_f32_4x4x1f32(b, da[n / 4][n % 4], n == 0 ? z4 : dd[d], 0, 0, 0);
            }
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
        HarmM<MS> h;
        h.eval(u.x, u.y, u.z);
        float dEdrho = RAD ? arm.w : 0.f, gx, gy, gz;
        angular_site_grad_m<MS>(
            h, u.x, u.y,
            [&](int o, float& c, float& dv) {
                c = cc[o / 4][o % 4];
                dv = dd[o / 4][o % 4];
            },
            dEdrho, gx, gy, gz);
        SiteGeo sg;
        sg.ux = u.x;
        sg.uy = u.y;
        sg.uz = u.z;
        sg.ir = u.w;
        float ex, ey, ez;
        site_dEdr(sg, dEdrho, inv_rn, gx, gy, gz, ex, ey, ez);
        const float tx = arm.y * ez - arm.z * ey, ty = arm.z * ex - arm.x * ez, tz = arm.x * ey - arm.y * ex;
        const float wj = 4 * s + q >= Cfg::NS ? 1.f : 0.f, wi = 1.f - wj;
        ig_x += wi * ex; ig_y += wi * ey; ig_z += wi * ez;
        it_x += wi * tx; it_y += wi * ty; it_z += wi * tz;
        jg_x += wj * ex; jg_y += wj * ey; jg_z += wj * ez;
        jt_x += wj * tx; jt_y += wj * ty; jt_z += wj * tz;
    }
    sum[0] = quad_sum(ig_x); sum[1] = quad_sum(ig_y); sum[2] = quad_sum(ig_z);
    sum[3] = quad_sum(it_x); sum[4] = quad_sum(it_y); sum[5] = quad_sum(it_z);
    sum[6] = quad_sum(jg_x); sum[7] = quad_sum(jg_y); sum[8] = quad_sum(jg_z);
    sum[9] = quad_sum(jt_x); sum[10] = quad_sum(jt_y); sum[11] = quad_sum(jt_z);
}

template <class Cfg>
__global__ __launch_bounds__((QuadAdj<Cfg>::BLOCK)) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_adjoint_quad(
    nepx_pair_model m, const float4* __restrict__ qf, const int32_t* __restrict__ pi, const int32_t* __restrict__ pj,
    const float4* __restrict__ pt, const int32_t* __restrict__ np_dev, int64_t maxp, int most,
    const float* __restrict__ dEdG, const float* __restrict__ E, float clip, float* __restrict__ out) {
    using Q = QuadAdj<Cfg>;
    using MG = typename Q::MG;
    constexpr int PW = 16, D = Cfg::D, COUNT = MG::COUNT;
    __shared__ __attribute__((aligned(16))) QuadSites<Cfg> st;
    __shared__ __attribute__((aligned(16))) float xch[COUNT][PW * Q::TS];
    __shared__ float rows[PW * D];
    __shared__ float part[COUNT][12][PW];
    __shared__ float4 stab[Cfg::ND];
    const int P = n_pairs(np_dev, maxp);
    // the grid is sized by the capacity; more than `most` pairs go one to a lane (k_adjoint)
    if ((int64_t)blockIdx.x * PW >= P || P > most) return;
    if (threadIdx.x < Cfg::ND) {
        const int k = threadIdx.x % Cfg::NS;
        stab[threadIdx.x] = make_float4(m.sites[3 * k], m.sites[3 * k + 1], m.sites[3 * k + 2], 0.f);
    }
    const int lane = threadIdx.x & 63, q = lane & 3, slot = lane >> 2;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    float* const xp = xch[wave] + slot * Q::TS;
    const float* const grow = rows + slot * D;
    const float inv_rn = 1.f / m.r_nep;
    for (int base = blockIdx.x * PW; base < P; base += gridDim.x * PW) {  // uniform over the block
        const int idx = base + slot;
        const bool valid = idx < P;
        // the tile's dE/dG rows are contiguous
        const int have = (P - base < PW ? P - base : PW) * D;
        for (int k = threadIdx.x; k < PW * D; k += Q::BLOCK) rows[k] = k < have ? dEdG[(size_t)base * D + k] : 0.f;
        if (wave < Q::STEPS) {  // the trips' sites, dealt to the waves
            float4 qi = make_float4(1.f, 0.f, 0.f, 0.f), qj = qi, t = make_float4(1.f, 0.f, 0.f, 0.f);
            if (valid) load_pair(qf, pi, pj, pt, idx, qi, qj, t);
            const PairIn g = pair_in<Cfg>(m, qi, qj, t.x, t.y, t.z);
            __syncthreads();  // the rows are there
            for (int s = wave; s < Q::STEPS; s += COUNT) quad_adjoint_site<Cfg>(m, stab, g, grow, s, lane, st);
            if (wave == 0 && q == 0) {
                const float v[6] = {g.six, g.siy, g.siz, g.sjx, g.sjy, g.sjz};
#pragma unroll
                for (int c = 0; c < 6; ++c) st.s[c][slot] = v[c];
            }
        } else {
            __syncthreads();
        }
        __syncthreads();  // the sites are there
        float sum[12];
        static_for<COUNT>([&](auto gc) {
            constexpr int G = decltype(gc)::value;
            if (wave == G)
                quad_adjoint_sums<Cfg, typename MG::template Set<G>, G == MG::RAD>(inv_rn, st, grow, xp, lane, sum);
        });
        if (q == 0) {
#pragma unroll
            for (int c = 0; c < 12; ++c) part[wave][c][slot] = sum[c];
        }
        __syncthreads();  // the groups' sums are there, and the rows and sites are used up
        if (wave == 0 && q == 0 && valid) {
#pragma unroll
            for (int c = 0; c < 12; ++c) {
                sum[c] = part[0][c][slot];
#pragma unroll
                for (int w = 1; w < COUNT; ++w) sum[c] += part[w][c][slot];
            }
            AdjAcc acc;
            acc.G0x = sum[0]; acc.G0y = sum[1]; acc.G0z = sum[2];
            acc.T0x = sum[3]; acc.T0y = sum[4]; acc.T0z = sum[5];
            acc.G1x = sum[6]; acc.G1y = sum[7]; acc.G1z = sum[8];
            acc.T1x = sum[9]; acc.T1y = sum[10]; acc.T1z = sum[11];
            acc.A0x = st.s[0][slot]; acc.A0y = st.s[1][slot]; acc.A0z = st.s[2][slot];
            acc.A1x = st.s[3][slot]; acc.A1y = st.s[4][slot]; acc.A1z = st.s[5][slot];
            store_out(out, idx, adj_finish<Cfg>(acc), E ? E[idx] : 0.f, clip);
        }
        // wave 0 reads `part` and `st.s` here; the next tile's are written after a barrier that it reaches past
        // these reads (st.s by wave 0 itself)
    }
}

}  // namespace nepx
