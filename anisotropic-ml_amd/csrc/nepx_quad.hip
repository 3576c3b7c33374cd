// Four-lanes-per-pair fused kernel (nepx_quad.h), adjoint (nepx_quad_adjoint.h) and cloud
// descriptor (nepx_quad_cloud.h), and their launchers.  Built in
// its own translation unit so that its matrix-core accumulators can be kept in
// VGPRs (-mllvm -amdgpu-mfma-vgpr-form), next to the VALU code that reads them.
#include "nepx_pairk.h"
#include "nepx_quad.h"
#include "nepx_quad_adjoint.h"
#include "nepx_quad_cloud.h"

namespace nepx {

template <class Cfg, class N, int PREC>
static void launch_quad_p(const nepx_pair_model& m, const nepx_net* net, int grid, int half_pairs, float scale, const float* qf,
                          const int32_t* pair_i, const int32_t* pair_j, const float* pair_t, const int32_t* np_dev,
                          int64_t maxp, float clip, float* out, RevOut rv, void* stream) {
#define NEPX_LAUNCH_QUAD(A)                                                                                      \
    hipLaunchKernelGGL((k_fused_quad<Cfg, N, PREC, A>), dim3(grid), dim3(QuadCfg<Cfg>::BLOCK), 0,                \
                       as_stream(stream), m, net->w_packed, net->w_half, net->en_min, scale, (const float4*)qf,   \
                       pair_i, pair_j, (const float4*)pair_t, np_dev, maxp, half_pairs, clip, out, rv)
    if (net->act == NEPX_ACT_TANH) NEPX_LAUNCH_QUAD(NEPX_ACT_TANH);
    else if constexpr (PREC == NEPX_NET_F32 || PREC == NEPX_NET_F16X3) NEPX_LAUNCH_QUAD(NEPX_ACT_RELU);
#undef NEPX_LAUNCH_QUAD
}

template <class Cfg, class N>
int launch_fused_quad(const nepx_pair_model& m, const nepx_net* net, int prec, int max_blocks, float scale,
                      const float* qf, const int32_t* pair_i, const int32_t* pair_j, const float* pair_t,
                      const int32_t* np_dev, int64_t maxp, float clip, float* out, RevOut rv, void* stream) {
    if constexpr (!QuadCfg<Cfg>::OK) {
        return NEPX_EUNSUP;
    } else {
        using Q = QuadCfg<Cfg>;
        // Few pairs: with two waves per SIMD, half a block's waves take pairs while one round of half blocks, one
        // a CU, holds them all: they spread over twice the CUs and a wave has its SIMD to itself (512 cubes,
        // 4,800 pairs: 19.2 -> 14.7 us).  The kernel decides by the pair count, not the capacity: with half
        // blocks up to some capacity, calls whose capacity is their count took two rounds where whole blocks
        // take one (cube8, 17,000 pairs 24.5 us against 19.8, 50,000 pairs 44.8 against 35.0).
        constexpr int HALF = Q::WAVES_PER_SIMD == 2 ? Q::BLOCK / 8 : 0;
        const int half_pairs = device_cus() * HALF;
        const int64_t least = HALF ? HALF : Q::BLOCK / 4;  // pairs a block takes at least
        const int64_t g = (maxp + least - 1) / least;
        const int grid = (int)(g < 1 ? 1 : g > max_blocks ? max_blocks : g);
        switch (prec) {
            case NEPX_NET_F16X3:
                launch_quad_p<Cfg, N, NEPX_NET_F16X3>(m, net, grid, half_pairs, scale, qf, pair_i, pair_j, pair_t, np_dev, maxp,
                                                       clip, out, rv, stream);
                break;
            case NEPX_NET_BF16:
                launch_quad_p<Cfg, N, NEPX_NET_BF16>(m, net, grid, half_pairs, scale, qf, pair_i, pair_j, pair_t, np_dev, maxp,
                                                      clip, out, rv, stream);
                break;
            case NEPX_NET_BF16X3:
                launch_quad_p<Cfg, N, NEPX_NET_BF16X3>(m, net, grid, half_pairs, scale, qf, pair_i, pair_j, pair_t, np_dev,
                                                        maxp, clip, out, rv, stream);
                break;
            default:
                launch_quad_p<Cfg, N, NEPX_NET_F32>(m, net, grid, half_pairs, scale, qf, pair_i, pair_j, pair_t, np_dev, maxp,
                                                     clip, out, rv, stream);
        }
        NEPX_LAUNCH_CHECK();
        return NEPX_OK;
    }
}

#define NEPX_QUAD_INSTANCE(T, N)                                                                              \
    template int launch_fused_quad<T, N>(const nepx_pair_model&, const nepx_net*, int, int, float, const float*, \
                                         const int32_t*, const int32_t*, const float*, const int32_t*, int64_t,  \
                                         float, float*, RevOut, void*);
NEPX_QUAD_INSTANCE(CfgCube8, Net40x64)
NEPX_QUAD_INSTANCE(CfgTet10, Net40x64)
NEPX_QUAD_INSTANCE(CfgCyl12, Net60x128)
#undef NEPX_QUAD_INSTANCE

template <class Cfg>
int launch_adjoint_quad(const nepx_pair_model& m, int max_blocks, const float* qf, const int32_t* pair_i,
                        const int32_t* pair_j, const float* pair_t, const int32_t* np_dev, int64_t maxp, int most,
                        const float* dEdG, const float* E, float clip, float* out, void* stream) {
    static_assert(QuadAdj<Cfg>::OK, "whole quads of sites");
    const int64_t tiles = (maxp + 15) / 16;
    const int grid = (int)(tiles < max_blocks ? tiles : max_blocks);
    hipLaunchKernelGGL(k_adjoint_quad<Cfg>, dim3(grid), dim3(QuadAdj<Cfg>::BLOCK), 0, as_stream(stream), m,
                       (const float4*)qf, pair_i, pair_j, (const float4*)pair_t, np_dev, maxp, most, dEdG, E, clip,
                       out);
    NEPX_LAUNCH_CHECK();
    return NEPX_OK;
}
#define NEPX_QUAD_ADJOINT(T)                                                                                  \
    template int launch_adjoint_quad<T>(const nepx_pair_model&, int, const float*, const int32_t*,            \
                                        const int32_t*, const float*, const int32_t*, int64_t, int,           \
                                        const float*, const float*, float, float*, void*);
NEPX_QUAD_ADJOINT(CfgCubeV2)
NEPX_QUAD_ADJOINT(CfgThV1)
NEPX_QUAD_ADJOINT(CfgCubeV2L10)
NEPX_QUAD_ADJOINT(CfgThV1L10)
#undef NEPX_QUAD_ADJOINT

template <class Cfg>
int launch_cloud_quad(const float* clouds, int64_t n_clouds, int n_sites, const float* site_w, float r_nep,
                      float* G, void* stream) {
    const int64_t tiles = (n_clouds + 15) / 16;
    const int64_t resident = (int64_t)device_cus() * QuadCloud<Cfg>::BLOCKS_PER_CU;
    const dim3 grid((unsigned)(tiles < resident ? tiles : resident)), block(QuadCloud<Cfg>::BLOCK);
    if (n_sites <= QuadCloud<Cfg>::STAGED)
        hipLaunchKernelGGL((k_cloud_quad<Cfg, true>), grid, block, 16 * 3 * n_sites * sizeof(float),
                           as_stream(stream), clouds, n_clouds, n_sites, site_w, r_nep, G);
    else
        hipLaunchKernelGGL((k_cloud_quad<Cfg, false>), grid, block, 0, as_stream(stream), clouds, n_clouds, n_sites,
                           site_w, r_nep, G);
    NEPX_LAUNCH_CHECK();
    return NEPX_OK;
}
#define NEPX_QUAD_CLOUD(a, b, c)                                                                               \
    template int launch_cloud_quad<DescCfg<1, a, b, c>>(const float*, int64_t, int, const float*, float,      \
                                                        float*, void*);
NEPX_CLOUD_CASES(NEPX_QUAD_CLOUD)
#undef NEPX_QUAD_CLOUD

}  // namespace nepx
