// Soft bead-bead repulsion between rigid bodies: the label potential of the
// reference's training-data generator (01/SamplerUtils.py:555-631, calc_en_unred):
//   E_ij = sum_{a in i, b in j} eps ((r0 - |p_b - p_a|) / sigma)^2   for |p_b - p_a| < r0
// with body-frame beads b_a (the same table for both bodies), p_a = X_i + R(q_i) b_a and
// p_b = X_i + t + R(q_j) b_b.  Forces and torques are analytic:
//   g = dE/dp_b = -2 eps (r0 - d) / sigma^2 * (p_b - p_a) / d
//   F_i = sum g,  tau_i = sum (R_i b_a) x g,  tau_j = -sum (R_j b_b) x g   (F_j = -F_i).
// Output per pair in the layout of the NEP pair kernels: {F_i, E}{tau_i, 0}{tau_j, 0},
// so the deterministic gather and the integrator take it unchanged.
//
// One wave per pair.  Only beads in reach of the other body's bounding box take part: each lane
// rotates beads of both bodies, tests them against the box of the bead table in the other body's frame
// grown by r0, and the survivors are compacted into LDS; the wave then splits the survivors' distances
// over its lanes (b of body j across lanes, a of body i across the lane groups that are left).  Most
// pairs of a list within the potential's reach do not touch, and touching faces leave a layer or two of
// each body, so of a 152-bead pair's 23,104 distances a few hundred are left: the bound is the VALU work
// of the rotations and tests (12,700 pairs of cubes at 0.004 bodies per unit volume: 97 us with every
// distance, 15 us so; where bodies overlap so deeply that nearly every bead survives, the cull costs 3 to 10 % of
// the distances' time).  FP32 accumulation, fixed-order butterfly reduction over the wave.
#include "nepx_common.h"

namespace nepx {

constexpr int kBeadBlock = 256;                  // 4 waves, one pair each per iteration
constexpr int kBeadWaves = kBeadBlock / 64;

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o, 64));
    return v;
}

// Bounding box of the bead table.
struct Box {
    float lx, ly, lz, hx, hy, hz;
};
__device__ __forceinline__ Box bead_box(const float* __restrict__ beads, int nb, int lane) {
    Box b{INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    for (int a = lane; a < nb; a += 64) {
        const float x = beads[3 * a], y = beads[3 * a + 1], z = beads[3 * a + 2];
        b.lx = fminf(b.lx, x); b.ly = fminf(b.ly, y); b.lz = fminf(b.lz, z);
        b.hx = fmaxf(b.hx, x); b.hy = fmaxf(b.hy, y); b.hz = fmaxf(b.hz, z);
    }
    b.lx = wave_min(b.lx); b.ly = wave_min(b.ly); b.lz = wave_min(b.lz);
    b.hx = -wave_min(-b.hx); b.hy = -wave_min(-b.hy); b.hz = -wave_min(-b.hz);
    return b;
}

// A body's frame as the cull sees it: R is |q|^2 times a rotation (quat_matrix), s = |q|^2, so
// R^T p / s has the lengths of the lab frame and the body fills the box scaled by s.
struct Reach {
    Mat3 R;
    float is, lx, ly, lz, hx, hy, hz;
};
// Below 1e-30 the division overflows or R has lost its bits to the end of FP32's range: NaN, which culls nothing.
__device__ __forceinline__ Reach body_reach(const Mat3& R, const float4& q, const Box& b, float grow) {
    const float s = q.x * q.x + q.y * q.y + q.z * q.z + q.w * q.w;
    return Reach{R, s > 1e-30f ? 1.f / s : NAN, s * b.lx - grow, s * b.ly - grow, s * b.lz - grow,
                 s * b.hx + grow, s * b.hy + grow, s * b.hz + grow};
}
// False only for a point (relative to the body's centre) outside the grown box; a NaN stays in, so
// what the distance test decides is left to it.
__device__ __forceinline__ bool in_reach(const Reach& c, float x, float y, float z) {
    const float u = (c.R.m[0] * x + c.R.m[3] * y + c.R.m[6] * z) * c.is;
    const float v = (c.R.m[1] * x + c.R.m[4] * y + c.R.m[7] * z) * c.is;
    const float w = (c.R.m[2] * x + c.R.m[5] * y + c.R.m[8] * z) * c.is;
    return !(u < c.lx || u > c.hx || v < c.ly || v > c.hy || w < c.lz || w > c.hz);
}

__global__ __launch_bounds__(kBeadBlock) void k_bead_pairs(const float* __restrict__ beads, int nb, float eps,
                                                            float sigma, float r0, const float4* __restrict__ qf,
                                                            const int32_t* __restrict__ pi,
                                                            const int32_t* __restrict__ pj,
                                                            const float4* __restrict__ pt,
                                                            const int32_t* __restrict__ np_dev, int64_t maxp,
                                                            float clip, float* __restrict__ out) {
    __shared__ float4 arm_i[kBeadWaves][NEPX_MAX_BEADS], arm_j[kBeadWaves][NEPX_MAX_BEADS];
    const int64_t P = np_dev ? ((int64_t)*np_dev < maxp ? (int64_t)*np_dev : maxp) : maxp;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    float4* const li = arm_i[wv];
    float4* const lj = arm_j[wv];
    const float r02 = r0 * r0;
    const float c = -2.f * eps / (sigma * sigma);
    // up to 64 distances are one round of the wave: nothing to cull (two beads, 12,700 pairs in reach: 16.5 -> 13.5 us)
    const bool cull = nb * nb > 64;
    Box box{};
    if (cull) box = bead_box(beads, nb, lane);
    const float ext = fmaxf(fmaxf(fabsf(box.lx), fabsf(box.hx)),
                            fmaxf(fmaxf(fabsf(box.ly), fabsf(box.hy)), fmaxf(fabsf(box.lz), fabsf(box.hz))));
    // waves share nothing, so each runs through its own pairs without block barriers
    for (int64_t p = (int64_t)blockIdx.x * kBeadWaves + wv; p < P; p += (int64_t)gridDim.x * kBeadWaves) {
        const float4 qi = qf[pi[p]], qj = qf[pj[p]], t = pt[p];
        const Mat3 Ri = quat_matrix(qi.x, qi.y, qi.z, qi.w), Rj = quat_matrix(qj.x, qj.y, qj.z, qj.w);
        // the box grows by r0 and a margin far above the rounding of the rotations (1e-7 of the lengths)
        const float si = qi.x * qi.x + qi.y * qi.y + qi.z * qi.z + qi.w * qi.w;
        const float sj = qj.x * qj.x + qj.y * qj.y + qj.z * qj.z + qj.w * qj.w;
        const float grow = r0 + 1e-4f * (r0 + (si + sj) * ext + fabsf(t.x) + fabsf(t.y) + fabsf(t.z));
        const Reach ri = body_reach(Ri, qi, box, grow), rj = body_reach(Rj, qj, box, grow);
        int ni = 0, nj = 0;
        for (int base = 0; base < nb; base += 64) {  // uniform over the wave
            const int a = base + lane;
            const bool have = a < nb;
            float bx = 0.f, by = 0.f, bz = 0.f;
            if (have) {
                bx = beads[3 * a];
                by = beads[3 * a + 1];
                bz = beads[3 * a + 2];
            }
            float x, y, z;
            mat_vec(Ri, bx, by, bz, x, y, z);
            const bool ki = have && (!cull || in_reach(rj, x - t.x, y - t.y, z - t.z));
            const uint64_t mi = __ballot(ki);
            if (ki) li[ni + __popcll(mi & ((1ull << lane) - 1ull))] = make_float4(x, y, z, 0.f);
            ni += __popcll(mi);
            mat_vec(Rj, bx, by, bz, x, y, z);
            const bool kj = have && (!cull || in_reach(ri, x + t.x, y + t.y, z + t.z));
            const uint64_t mj = __ballot(kj);
            if (kj) lj[nj + __popcll(mj & ((1ull << lane) - 1ull))] = make_float4(x, y, z, 0.f);
            nj += __popcll(mj);
        }
        float4* o4 = reinterpret_cast<float4*>(out) + 3 * p;
        if (ni == 0 || nj == 0) {  // uniform over the wave: nothing in reach
            if (lane < 3) o4[lane] = make_float4(0.f, 0.f, 0.f, 0.f);
            continue;
        }
        wave_lds_order();
        // lanes across b: the power of two that holds body j's survivors (at most 64); the remaining
        // lane bits across a
        int lw = 64;
        while (lw / 2 >= nj) lw >>= 1;
        const int lb = lane & (lw - 1), la = lane / lw, ga = 64 / lw;
        float e = 0.f, fx = 0.f, fy = 0.f, fz = 0.f, tix = 0.f, tiy = 0.f, tiz = 0.f, tjx = 0.f, tjy = 0.f,
              tjz = 0.f;
        for (int b = lb; b < nj; b += lw) {
            const float4 ab = lj[b];
            const float bx = t.x + ab.x, by = t.y + ab.y, bz = t.z + ab.z;
            float gbx = 0.f, gby = 0.f, gbz = 0.f;  // sum of g over this lane's a for this bead b
            auto bead = [&](int a) {
                const float4 aa = li[a];
                const float dx = bx - aa.x, dy = by - aa.y, dz = bz - aa.z;
                const float d2 = dx * dx + dy * dy + dz * dz;
                if (d2 < r02) {
                    const float d = sqrtf(d2);
                    const float w = r0 - d;
                    e += eps * (w * w) / (sigma * sigma);
                    const float s = c * w / d;  // dE/dd / d
                    const float gx = s * dx, gy = s * dy, gz = s * dz;
                    gbx += gx;
                    gby += gy;
                    gbz += gz;
                    tix += aa.y * gz - aa.z * gy;
                    tiy += aa.z * gx - aa.x * gz;
                    tiz += aa.x * gy - aa.y * gx;
                }
            };
            // deep overlap leaves most of both tables: a uniform walk, read by all lanes at once
            if (lw == 64) {
                for (int a = 0; a < ni; ++a) bead(a);
            } else {
                for (int a = la; a < ni; a += ga) bead(a);
            }
            fx += gbx;
            fy += gby;
            fz += gbz;
            tjx -= ab.y * gbz - ab.z * gby;
            tjy -= ab.z * gbx - ab.x * gbz;
            tjz -= ab.x * gby - ab.y * gbx;
        }
        e = wave_sum(e);
        fx = wave_sum(fx);
        fy = wave_sum(fy);
        fz = wave_sum(fz);
        tix = wave_sum(tix);
        tiy = wave_sum(tiy);
        tiz = wave_sum(tiz);
        tjx = wave_sum(tjx);
        tjy = wave_sum(tjy);
        tjz = wave_sum(tjz);
        if (lane == 0) {
            auto cl = [clip](float v) { return clipf(v, clip); };
            o4[0] = make_float4(cl(fx), cl(fy), cl(fz), e);
            o4[1] = make_float4(cl(tix), cl(tiy), cl(tiz), 0.f);
            o4[2] = make_float4(cl(tjx), cl(tjy), cl(tjz), 0.f);
        }
        wave_lds_order();  // the survivors are read before the next pair's overwrite them
    }
}

}  // namespace nepx

using namespace nepx;

extern "C" int nepx_bead_pair_forces(const float* beads, int32_t n_beads, float eps, float sigma, float r0,
                                     const float* qf, const int32_t* pair_i, const int32_t* pair_j,
                                     const float* pair_t, const int32_t* n_pairs_dev, int64_t max_pairs,
                                     float clip, float* out, void* stream) {
    NEPX_REQUIRE(n_beads > 0 && n_beads <= NEPX_MAX_BEADS, NEPX_EINVAL, "n_beads %d not in 1..%d", n_beads,
                 NEPX_MAX_BEADS);
    NEPX_REQUIRE(sigma > 0.f && r0 > 0.f, NEPX_EINVAL, "sigma and r0 must be positive");
    if (max_pairs <= 0) return NEPX_OK;
    NEPX_REQUIRE(beads && qf && pair_i && pair_j && pair_t && out, NEPX_EINVAL, "null buffer");
    int64_t grid = (max_pairs + kBeadWaves - 1) / kBeadWaves;
    const int64_t cap = (int64_t)device_cus() * 8;
    if (grid > cap) grid = cap;
    hipLaunchKernelGGL(k_bead_pairs, dim3((unsigned)grid), dim3(kBeadBlock), 0, as_stream(stream), beads, n_beads,
                       eps, sigma, r0, (const float4*)qf, pair_i, pair_j, (const float4*)pair_t, n_pairs_dev,
                       max_pairs, clip, out);
    NEPX_LAUNCH_CHECK();
    return NEPX_OK;
}
