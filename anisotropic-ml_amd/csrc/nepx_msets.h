// Solid harmonics cut into sets of m, for the four-lane kernels that spread one tile's harmonics over
// several waves (nepx_quad_adjoint.h, nepx_quad_cloud.h).  The columns Q_l^m follow from Q_m^m by a
// recurrence in l alone, and the gradient of column m needs only columns m and m + 1, so a set repeats
// next to nothing of another set's harmonics (a cut by l would repeat the whole recurrence).
#pragma once
#include "nepx_desc.h"

namespace nepx {

// Harmonics of the m in the bit set MASK, max(m, 1) <= l <= LMAX: slots ordered by l, m, part.
template <int LMAX_, unsigned MASK>
struct MSet {
    static constexpr int LMAX = LMAX_;
    __host__ __device__ static constexpr bool has(int m) { return (MASK >> m) & 1u; }
    // columns of Q the sums and the gradient read: m and m + 1
    __host__ __device__ static constexpr bool column(int m) { return m <= LMAX && (has(m) || (m > 0 && has(m - 1))); }
    __host__ __device__ static constexpr int first_l(int m) { return m > 1 ? m : 1; }
    // slots of the harmonics below l
    __host__ __device__ static constexpr int off(int l) {
        int o = 0;
        for (int k = 1; k < l; ++k)
            for (int m = 0; m <= k; ++m) o += has(m) ? (m ? 2 : 1) : 0;
        return o;
    }
    static constexpr int N = off(LMAX + 1);
    __host__ __device__ static constexpr int slot(int l, int m, int part) {
        int o = off(l) + part;
        for (int k = 0; k < m; ++k) o += has(k) ? (k ? 2 : 1) : 0;
        return o;
    }
    __host__ __device__ static constexpr int l_of(int s) {
        int l = 1;
        while (s >= off(l + 1)) ++l;
        return l;
    }
    __host__ __device__ static constexpr int m_of(int s) {
        int m = 0, o = off(l_of(s));
        for (;; ++m) {
            const int w = has(m) ? (m ? 2 : 1) : 0;
            if (s < o + w) return m;
            o += w;
        }
    }
    // K_lm^2 and the entry of l within dE/dg_ang[n] of slot s; zero and 0 past the last slot
    __host__ __device__ static constexpr float k2(int s) { return s < N ? K2Tab<LMAX>{}(l_of(s), m_of(s)) : 0.f; }
    __host__ __device__ static constexpr int row_of(int s) { return s < N ? l_of(s) - 1 : 0; }
};

// The columns of Q_l^m a set reads, and C_m, S_m (nepx_desc.h's Harm, column by column).
template <class MS>
struct HarmM {
    static constexpr int L = MS::LMAX;
    float Q[L + 1][L + 1];  // [m][l], the set's columns
    float C[L + 1], S[L + 1];
    __device__ __forceinline__ float q(int l, int m) const { return Q[m][l]; }
    __device__ __forceinline__ float z(int l, int m, int part) const {
        return m == 0 ? q(l, 0) : q(l, m) * (part ? S[m] : C[m]);
    }
    __device__ __forceinline__ void eval(float x, float y, float zz) {
        float qmm = 1.f;
#pragma unroll
        for (int m = 0; m <= L; ++m) {
            if (m > 0) qmm *= -(2.f * m - 1.f);
            if (MS::column(m)) {
                Q[m][m] = qmm;
                if (m < L) Q[m][m + 1] = (2.f * m + 1.f) * zz * qmm;
#pragma unroll
                for (int l = m + 2; l <= L; ++l) {
                    const float a = (2.f * l - 1.f) / (float)(l - m);
                    const float b = (float)(l + m - 1) / (float)(l - m);
                    Q[m][l] = a * zz * Q[m][l - 1] - b * Q[m][l - 2];
                }
            }
        }
        C[0] = 1.f;
        S[0] = 0.f;
#pragma unroll
        for (int m = 1; m <= L; ++m) {  // the powers past the set's last m are never read
            C[m] = x * C[m - 1] - y * S[m - 1];
            S[m] = x * S[m - 1] + y * C[m - 1];
        }
    }
};

// Groups of m, one wave each; the radial terms go with one of them.
template <int LMAX>
struct MGroups {  // all m on one wave
    static constexpr int COUNT = 1, RAD = 0;
    template <int G>
    using Set = MSet<LMAX, (2u << LMAX) - 1u>;
};
template <>
struct MGroups<10> {  // 30 harmonics each
    static constexpr int COUNT = 4, RAD = 2;
    static constexpr unsigned MASK[4] = {0x003, 0x024, 0x018, 0x7c0};
    template <int G>
    using Set = MSet<10, MASK[G]>;
};

// Largest number of 4-slot chunks among the sets.
template <class MG, int G = 0>
constexpr int max_chunks() {
    constexpr int n = (MG::template Set<G>::N + 3) / 4;
    if constexpr (G + 1 < MG::COUNT) {
        constexpr int r = max_chunks<MG, G + 1>();
        return n > r ? n : r;
    } else {
        return n;
    }
}

}  // namespace nepx
