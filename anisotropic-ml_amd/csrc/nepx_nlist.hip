// Neighbour list on the GPU: cell binning, half Verlet list within r_list
// (rows i<j sorted by j, reverse rows sorted by i), per-step COM filter with
// an FP64 predicate and deterministic compaction, and the deterministic
// gather of per-pair forces.
//
// Replaces the host cKDTree list (nep_simulator/Sim.py:85-92,192-198), the
// per-step COM filter (nep_simulator/DescriptorGenerator.py:168-185) and the
// index_add_ scatter (nep_simulator/ForceEvaluator.py:135-142).
//
// Pair predicate (all paths, bit-exact with the oracle): t = X_j - X_i per
// component, one wrap (t > L/2 -> t - L, t < -L/2 -> t + L), then
// d2 = (tx*tx + ty*ty) + tz*tz in FP64 with no fused multiply-add, d2 < r*r.
#include <mutex>

#include "nepx_common.h"

namespace nepx {

constexpr int kNB = 256;        // threads per block
constexpr int kScanBlock = 1024;
constexpr int kSortMax = 2048;  // longest row the sorts accept
constexpr int kSlotsPerBlock = 1024;

// One wrap of t: past L/2 either way, t moves L towards zero.  (The two tests t > L/2 -> t - L,
// t < -L/2 -> t + L in turn give the same bits: t - L cannot round below -L/2.)
__device__ __forceinline__ double wrap1(double t, double L) {
    return fabs(t) > 0.5 * L ? __dsub_rn(t, copysign(L, t)) : t;
}

// Squared minimum-image distance from (xi, yi, zi) to (xj, yj, zj); t = X_j - X_i.
__device__ __forceinline__ double pos_d2(double xi, double yi, double zi, double xj, double yj, double zj, double L,
                                         double& tx, double& ty, double& tz) {
    tx = wrap1(__dsub_rn(xj, xi), L);
    ty = wrap1(__dsub_rn(yj, yi), L);
    tz = wrap1(__dsub_rn(zj, zi), L);
    return __dadd_rn(__dadd_rn(__dmul_rn(tx, tx), __dmul_rn(ty, ty)), __dmul_rn(tz, tz));
}

__device__ __forceinline__ double pair_d2(const nepx_state& st, double L, int i, int j, double& tx,
                                          double& ty, double& tz) {
    return pos_d2(st.x[i], st.y[i], st.z[i], st.x[j], st.y[j], st.z[j], L, tx, ty, tz);
}

// Cell of coordinate x along one side: x is wrapped once, as the pair predicate wraps differences, so a
// configuration off the box (positions in [0, L), or moved and not folded back) has the cells of its image
// in the box.  Clamped to [0, nc): NaN and infinities (a faulted system's particles, between the step that
// went non-finite and its removal) land in the edge cells; the comparisons run in floating point so no
// out-of-range value is converted.
__device__ __forceinline__ int cell_coord(double x, double L, int nc) {
    const double f = floor((wrap1(x, L) + 0.5 * L) / L * (double)nc);
    if (!(f >= 0.0)) return 0;
    return f >= (double)nc ? nc - 1 : (int)f;
}

// A build runs when the list is stale (F_REBUILD) or due soon (F_SOON, set while it is still valid).
__device__ __forceinline__ bool want_build(const int32_t* flags) { return flags[F_REBUILD] != 0 || flags[F_SOON] != 0; }

// A particle takes part in the list when it belongs to an active system.
__device__ __forceinline__ bool live(const nepx_state& st, int i) {
    const int s = st.sys[i];
    return s >= 0 && st.sp[s].active;
}

// Start of a build step: clear the longest-row flag and, when a rebuild is due, the cell counters.  A
// forced build requests itself and clears a stale overflow (the flags it sets are not read here).
__global__ void k_build_begin(int32_t* flags, int32_t* cell_count, int32_t* cell_fill, int64_t nct, int force) {
    const bool build = force || want_build(flags);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        flags[F_MAXROW] = 0;
        flags[F_LONGSYS] = 0;
        if (force) {
            flags[F_REBUILD] = 1;
            flags[F_OVERFLOW] = 0;
        }
    }
    if (!build) return;
    for (int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; k < nct; k += (int64_t)gridDim.x * blockDim.x) {
        cell_count[k] = 0;
        cell_fill[k] = 0;
    }
}

__global__ void k_cells_count(nepx_state st, nepx_nlist nl) {
    if (!want_build(nl.flags)) return;
    const int i = blockIdx.x * kNB + threadIdx.x;
    if (i >= st.n) return;
    // positions at this build: the reference for the displacement test that requests the next one
    st.xb[i] = st.x[i];
    st.yb[i] = st.y[i];
    st.zb[i] = st.z[i];
    if (!live(st, i)) return;
    const int s = st.sys[i];
    const nepx_sysparam& sp = st.sp[s];
    if (sp.nc <= 0) return;
    const int cx = cell_coord(st.x[i], sp.L, sp.nc), cy = cell_coord(st.y[i], sp.L, sp.nc),
              cz = cell_coord(st.z[i], sp.L, sp.nc);
    const int c = sp.cell_off + (cx * sp.nc + cy) * sp.nc + cz;
    nl.cell_of[i] = c;
    atomicAdd(&nl.cell_count[c], 1);
}

// Exclusive scan of a[0..n) into out (which may be a); returns the total.  One block of kScanBlock
// threads, kScanPer consecutive entries a thread, the next entries loaded while these are summed.
constexpr int kScanPer = 8;
__device__ int block_exclusive_scan(const int32_t* a, int32_t* out, int n) {
    __shared__ int32_t wsum[kScanBlock / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int32_t v[kScanPer];
    auto load = [&](int base) {
        const int k0 = base + threadIdx.x * kScanPer;
#pragma unroll
        for (int r = 0; r < kScanPer; ++r) v[r] = k0 + r < n ? a[k0 + r] : 0;
    };
    int carry = 0;
    load(0);
    for (int base = 0; base < n; base += kScanBlock * kScanPer) {
        int32_t x[kScanPer], t = 0;
#pragma unroll
        for (int r = 0; r < kScanPer; ++r) {
            x[r] = t;
            t += v[r];
        }
        load(base + kScanBlock * kScanPer);  // past this chunk, so `out` may be `a`
        int inc = t;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int u = __shfl_up(inc, o, 64);
            inc += lane >= o ? u : 0;
        }
        if (lane == 63) wsum[w] = inc;
        __syncthreads();
        int before = carry, all = 0;
#pragma unroll
        for (int k = 0; k < kScanBlock / 64; ++k) {
            const int u = wsum[k];
            before += k < w ? u : 0;
            all += u;
        }
        before += inc - t;
        const int k0 = base + threadIdx.x * kScanPer;
#pragma unroll
        for (int r = 0; r < kScanPer; ++r)
            if (k0 + r < n) out[k0 + r] = before + x[r];
        carry += all;
        __syncthreads();  // wsum is read before the next chunk's sums
    }
    return carry;
}

// Cells are scanned up to the last one a system uses (the counters are also scratch of 2 n entries).
__global__ __launch_bounds__(kScanBlock) void k_scan_cells(nepx_state st, nepx_nlist nl) {
    if (!want_build(nl.flags)) return;
    __shared__ int used;
    if (threadIdx.x == 0) used = 0;
    __syncthreads();
    int m = 0;
    for (int s = threadIdx.x; s < st.n_sys; s += kScanBlock) {
        const int nc = st.sp[s].nc, e = nc > 0 ? st.sp[s].cell_off + nc * nc * nc : 0;
        m = e > m ? e : m;
    }
    if (m > 0) atomicMax(&used, m);
    __syncthreads();
    const int n = used < nl.n_cells_total ? used : nl.n_cells_total;
    const int total = block_exclusive_scan(nl.cell_count, nl.cell_start, n);
    if (threadIdx.x == 0) nl.cell_start[n] = total;
}

__global__ void k_cells_fill(nepx_state st, nepx_nlist nl) {
    if (!want_build(nl.flags)) return;
    const int i = blockIdx.x * kNB + threadIdx.x;
    if (i >= st.n || !live(st, i)) return;
    const int s = st.sys[i];
    if (st.sp[s].nc <= 0) return;
    const int c = nl.cell_of[i];
    const int pos = nl.cell_start[c] + atomicAdd(&nl.cell_fill[c], 1);
    nl.cell_list[pos] = i;
    // positions in cell order: the candidate walk reads a cell's positions contiguously
    reinterpret_cast<double4*>(nl.cell_pos)[pos] = make_double4(st.x[i], st.y[i], st.z[i], 0.0);
}

// The list build gives each particle a group of LG lanes.  The lanes walk the candidates j of particle
// i in rounds of LG: round r of a run of cells covers its entries r*LG + sub.  Every lane of a group sees
// the same runs and rounds (same i), so ballots inside a round are uniform over the group; f(j, valid, d2)
// is called for each round slot with the squared minimum-image distance d2, valid = false for slots past
// the end of a run and for j == i.
//
// Cells along z are neighbours in memory, so the cells of one (x, y) column that a particle reaches are one
// run (two where they wrap): 2 R + 1 cells, R = the cells that cover r_list (1 for cells of a side of
// r_list or more, 2 for half of that, ...), or the whole system when there are no cells.  Candidates'
// positions come from the cell-ordered copy (contiguous), the same FP64 values as st.x.
//
// LG: with 16 lanes a particle, 4,096 particles are one wave per SIMD and the walk waits for memory, so
// systems of up to kWideGroups particles take a wave per particle (4,097 tetrahedra, a list of 402,000 pairs:
// the two walks 254 -> 84 us, with the columns walked as runs).  nepx/system.py picks the cells' side by the
// lanes, so it holds this number as well.
constexpr int kWideGroups = 8192;

template <int LG>
__device__ __forceinline__ uint64_t group_mask(uint64_t ballot) {
    if constexpr (LG == 64) {
        return ballot;
    } else {
        const int gbase = (threadIdx.x & 63) & ~(LG - 1);
        return (ballot >> gbase) & ((1ull << LG) - 1ull);
    }
}

// Cells each way that cover r (at least one); nc = floor(L / r) gives 1 whatever the rounding.
__device__ __forceinline__ int cell_reach(double r, double L, int nc) {
    const double f = r * (double)nc / L;
    if (f <= 1.0 + 1e-9) return 1;
    return f < (double)nc ? (int)ceil(f - 1e-9) : nc;
}

template <int LG, class F>
__device__ __forceinline__ void for_candidates(const nepx_state& st, const nepx_nlist& nl, int i, int sub, F&& f) {
    const int s = st.sys[i];
    const nepx_sysparam& sp = st.sp[s];
    const double L = sp.L;
    const double xi = st.x[i], yi = st.y[i], zi = st.z[i];
    double tx, ty, tz;
    if (sp.nc <= 0) {
        for (int base = sp.p_start; base < sp.p_end; base += LG) {
            const int j = base + sub;
            const bool valid = j < sp.p_end && j != i && st.sys[j] == s;
            const int jj = valid ? j : i;
            const double d2 = pos_d2(xi, yi, zi, st.x[jj], st.y[jj], st.z[jj], L, tx, ty, tz);
            f(jj, valid, d2);
        }
        return;
    }
    const double4* cpos = reinterpret_cast<const double4*>(nl.cell_pos);
    const int nc = sp.nc, R = cell_reach(sp.r_list, L, nc);
    const int span = 2 * R + 1 < nc ? 2 * R + 1 : nc;  // distinct cells a side
    const int cx = cell_coord(st.x[i], L, nc), cy = cell_coord(st.y[i], L, nc), cz = cell_coord(st.z[i], L, nc);
    // the column's cells: [z0, z0 + span), of which those past nc wrap to the front
    const int z0 = span < nc ? (cz - R + nc) % nc : 0;
    const int first = z0 + span <= nc ? span : nc - z0;
    for (int dx = 0; dx < span; ++dx) {
        const int ax = (cx - R + dx + nc) % nc;
        for (int dy = 0; dy < span; ++dy) {
            const int col = sp.cell_off + (ax * nc + (cy - R + dy + nc) % nc) * nc;
            for (int run = 0; run < (first < span ? 2 : 1); ++run) {
                const int b = nl.cell_start[run ? col : col + z0];
                const int e = nl.cell_start[run ? col + span - first : col + z0 + first];
                for (int base = b; base < e; base += LG) {
                    const int k = base + sub;
                    const bool in = k < e;
                    const int j = in ? nl.cell_list[k] : i;
                    const double4 pj = in ? cpos[k] : make_double4(xi, yi, zi, 0.0);
                    const double d2 = pos_d2(xi, yi, zi, pj.x, pj.y, pj.z, L, tx, ty, tz);
                    f(j, j != i, d2);
                }
            }
        }
    }
}

template <int W>
__device__ __forceinline__ int group_sum(int v) {
#pragma unroll
    for (int o = W / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, W);
    return v;
}

// Row lengths.  row_start and rrow_start get each row's offset within its block's rows, row_count[b] and
// rrow_count[b] the block's totals, which k_scan_rows turns into the blocks' offsets.
template <int LG>
__global__ __launch_bounds__(kNB) void k_nbr_count(nepx_state st, nepx_nlist nl) {
    if (!want_build(nl.flags)) return;
    constexpr int ROWS = kNB / LG;
    __shared__ int len[2][ROWS];
    const int r = threadIdx.x / LG, i = blockIdx.x * ROWS + r;
    const int sub = threadIdx.x % LG;
    int nf = 0, nr = 0;
    if (i < st.n && live(st, i)) {  // uniform per group
        const nepx_sysparam& sp = st.sp[st.sys[i]];
        const double r2 = __dmul_rn(sp.r_list, sp.r_list);
        for_candidates<LG>(st, nl, i, sub, [&](int j, bool valid, double d2) {
            if (valid && d2 < r2) {
                if (j > i) ++nf;
                else ++nr;
            }
        });
    }
    nf = group_sum<LG>(nf);
    nr = group_sum<LG>(nr);
    if (sub == 0) {
        len[0][r] = nf;
        len[1][r] = nr;
        if (nf > kSortMax || nr > kSortMax) {
            atomicMax(&nl.flags[F_MAXROW], nf > nr ? nf : nr);
            nl.flags[F_LONGSYS] = st.sys[i] + 1;  // one system holding such a row (any, if several)
        }
    }
    __syncthreads();
    if (threadIdx.x < 2 * ROWS) {
        const int side = threadIdx.x / ROWS, k = threadIdx.x % ROWS;
        int o = 0;
        for (int u = 0; u < k; ++u) o += len[side][u];
        const int row = blockIdx.x * ROWS + k;
        int32_t* start = side ? nl.rrow_start : nl.row_start;
        if (row < st.n) start[row] = o;
        if (k == ROWS - 1) (side ? nl.rrow_count : nl.row_count)[blockIdx.x] = o + len[side][k];
    }
}

// Block 0 scans the forward rows, block 1 the reverse rows: the row counts into row starts (PER_ROW), or the
// blocks' totals in place.
template <bool PER_ROW>
__global__ __launch_bounds__(kScanBlock) void k_scan_rows(nepx_nlist nl, int m, int n) {
    if (!want_build(nl.flags)) return;
    if (blockIdx.x == 0) {
        const int total = block_exclusive_scan(nl.row_count, PER_ROW ? nl.row_start : nl.row_count, m);
        if (threadIdx.x == 0) {
            nl.row_start[n] = total;
            nl.flags[F_PL] = total;
            if ((int64_t)total > nl.cap || nl.flags[F_MAXROW] > kSortMax) nl.flags[F_OVERFLOW] = 1;
        }
    } else {
        const int total = block_exclusive_scan(nl.rrow_count, PER_ROW ? nl.rrow_start : nl.rrow_count, m);
        if (threadIdx.x == 0) nl.rrow_start[n] = total;
    }
}

// Same walk as k_nbr_count; each round's accepted candidates are placed by a
// ballot prefix within the group (no atomics).  The row order this gives
// depends on the cell lists; the sorts make it canonical.
template <int LG>
__global__ __launch_bounds__(kNB) void k_nbr_fill(nepx_state st, nepx_nlist nl) {
    if (!want_build(nl.flags)) return;
    const int i = (blockIdx.x * kNB + threadIdx.x) / LG;
    const int sub = threadIdx.x % LG;
    if (i >= st.n) return;  // uniform per group
    int pf = nl.row_count[blockIdx.x] + nl.row_start[i], pr = nl.rrow_count[blockIdx.x] + nl.rrow_start[i];
    if (sub == 0) {
        nl.row_start[i] = pf;
        nl.rrow_start[i] = pr;
    }
    if (nl.flags[F_OVERFLOW] || !live(st, i)) return;
    const nepx_sysparam& sp = st.sp[st.sys[i]];
    const double r2 = __dmul_rn(sp.r_list, sp.r_list);
    const uint64_t below = (1ull << sub) - 1ull;
    for_candidates<LG>(st, nl, i, sub, [&](int j, bool valid, double d2) {
        const bool in = valid && d2 < r2;
        const bool fwd = in && j > i, rev = in && j < i;
        const uint64_t mf = group_mask<LG>(__ballot(fwd)), mr = group_mask<LG>(__ballot(rev));
        if (fwd) {
            const int slot = pf + __popcll(mf & below);
            nl.nbr[slot] = j;
            nl.slot_row[slot] = i;
        }
        if (rev) nl.rnbr[pr + __popcll(mr & below)] = j;
        pf += __popcll(mf);
        pr += __popcll(mr);
    });
}

// ---- row sorts ----------------------------------------------------------------
// One wave sorts a row.  Up to 64 * kRegRow entries sit in registers, entry k * 64 + lane in register k of
// the lane: a bitonic network whose strides below 64 exchange lanes (DPP for 1, 2, 4 and 8) and the others
// registers, no LDS and no barriers (both sorts and the slots of 402,000 pairs: 152 -> 55 us against a
// network in LDS).  Longer rows (up to kSortMax) sort in the wave's part of LDS.
constexpr int kSortThreads = 256, kSortWaves = kSortThreads / 64, kRegRow = 8;

template <int STRIDE>
__device__ __forceinline__ int lane_xor(int v) {
    if constexpr (STRIDE == 1) return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true);   // quad 1,0,3,2
    else if constexpr (STRIDE == 2) return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, true);  // quad 2,3,0,1
    else if constexpr (STRIDE == 4)  // 7 - i within eight lanes, then 3 - i within four
        return __builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp(v, 0x141, 0xF, 0xF, true), 0x1B, 0xF, 0xF, true);
    else if constexpr (STRIDE == 8) return __builtin_amdgcn_mov_dpp(v, 0x128, 0xF, 0xF, true);  // rotate 16 by 8
    else return __shfl_xor(v, STRIDE, 64);
}

template <int K, int SIZE, int STRIDE>
__device__ __forceinline__ void bitonic_stage(int32_t (&v)[K], int lane) {
    if constexpr (STRIDE >= 64) {
        constexpr int RS = STRIDE / 64;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            if ((k & RS) == 0) {
                const bool up = (k & (SIZE / 64)) == 0;
                const int32_t a = v[k], b = v[k | RS], lo = a < b ? a : b, hi = a < b ? b : a;
                v[k] = up ? lo : hi;
                v[k | RS] = up ? hi : lo;
            }
        }
    } else {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const bool up = SIZE < 64 ? (lane & SIZE) == 0 : (k & (SIZE / 64)) == 0;
            const int32_t o = lane_xor<STRIDE>(v[k]);
            const bool low = ((lane & STRIDE) == 0) == up;  // this lane keeps the smaller
            v[k] = low ? (v[k] < o ? v[k] : o) : (v[k] < o ? o : v[k]);
        }
    }
}
template <int K, int SIZE, int STRIDE>
__device__ __forceinline__ void bitonic_strides(int32_t (&v)[K], int lane) {
    bitonic_stage<K, SIZE, STRIDE>(v, lane);
    if constexpr (STRIDE > 1) bitonic_strides<K, SIZE, STRIDE / 2>(v, lane);
}
template <int K, int SIZE = 2>
__device__ __forceinline__ void bitonic_sort(int32_t (&v)[K], int lane) {
    bitonic_strides<K, SIZE, SIZE / 2>(v, lane);
    if constexpr (SIZE < 64 * K) bitonic_sort<K, SIZE * 2>(v, lane);
}

// load(k) gives entry k of the row, store(k, v) takes the sorted entry k.
template <int K, class Load, class Store>
__device__ __forceinline__ void sort_in_registers(int len, int lane, Load&& load, Store&& store) {
    int32_t v[K];
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = k * 64 + lane < len ? load(k * 64 + lane) : 0x7fffffff;
    bitonic_sort<K>(v, lane);
#pragma unroll
    for (int k = 0; k < K; ++k)
        if (k * 64 + lane < len) store(k * 64 + lane, v[k]);
}

template <class Load, class Store>
__device__ __forceinline__ void sort_row(int len, int lane, int32_t* buf, Load&& load, Store&& store) {
    if (len <= 64) sort_in_registers<1>(len, lane, load, store);
    else if (len <= 128) sort_in_registers<2>(len, lane, load, store);
    else if (len <= 256) sort_in_registers<4>(len, lane, load, store);
    else if (len <= 64 * kRegRow) sort_in_registers<kRegRow>(len, lane, load, store);
    else {
        int p2 = 1;
        while (p2 < len) p2 <<= 1;
        for (int k = lane; k < p2; k += 64) buf[k] = k < len ? load(k) : 0x7fffffff;
        wave_lds_order();
        for (int size = 2; size <= p2; size <<= 1) {
            for (int stride = size >> 1; stride > 0; stride >>= 1) {
                for (int k = lane; k < p2; k += 64) {
                    const int partner = k ^ stride;
                    if (partner > k) {
                        const bool up = (k & size) == 0;
                        const int32_t a = buf[k], c = buf[partner];
                        if ((a > c) == up) {
                            buf[k] = c;
                            buf[partner] = a;
                        }
                    }
                }
                wave_lds_order();
            }
        }
        for (int k = lane; k < len; k += 64) store(k, buf[k]);
        wave_lds_order();
    }
}

// Forward rows ascending in j.  The grid is capped, so the launch costs little when no rebuild is due.
__global__ __launch_bounds__(kSortThreads) void k_sort_rows(nepx_nlist nl, int n) {
    if (!want_build(nl.flags) || nl.flags[F_OVERFLOW]) return;
    __shared__ int32_t buf[kSortWaves][kSortMax];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int i = blockIdx.x * kSortWaves + w; i < n; i += gridDim.x * kSortWaves) {
        const int b = nl.row_start[i], len = nl.row_start[i + 1] - b;
        if (len <= 1) continue;  // uniform per wave
        int32_t* row = nl.nbr + b;
        sort_row(len, lane, buf[w], [&](int k) { return row[k]; }, [&](int k, int32_t v) { row[k] = v; });
    }
}

// Reverse entries hold the partner i; each becomes the slot of (i, k) in row i (binary search in the sorted
// row), and the slots are sorted, which orders them by i as the rows are in slot order.  The last block to
// arrive marks the build done: every block has read the flags by then, and nothing else is handed over.
__global__ __launch_bounds__(kSortThreads) void k_rev_rows(nepx_nlist nl, int n) {
    if (!want_build(nl.flags)) return;
    __shared__ int32_t buf[kSortWaves][kSortMax];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool skip = nl.flags[F_OVERFLOW] != 0;
    for (int k = blockIdx.x * kSortWaves + w; k < n && !skip; k += gridDim.x * kSortWaves) {
        const int b = nl.rrow_start[k], len = nl.rrow_start[k + 1] - b;
        if (len <= 0) continue;  // uniform per wave
        int32_t* row = nl.rnbr + b;
        sort_row(
            len, lane, buf[w],
            [&](int e) {
                const int i = row[e];
                int lo = nl.row_start[i], hi = nl.row_start[i + 1] - 1, slot = -1;
                while (lo <= hi) {
                    const int mid = (lo + hi) >> 1;
                    const int v = nl.nbr[mid];
                    if (v == k) {
                        slot = mid;
                        break;
                    }
                    if (v < k) lo = mid + 1;
                    else hi = mid - 1;
                }
                if (slot < 0) nl.flags[F_OVERFLOW] = 2;  // inconsistent list: never expected
                return slot;
            },
            [&](int e, int32_t slot) {
                row[e] = slot;
                if (nl.rpos && slot >= 0) nl.rpos[slot] = b + e;  // where the reverse row of k holds this slot
            });
    }
    __syncthreads();
    if (threadIdx.x == 0 && atomicAdd(&nl.flags[F_DONE], 1) == (int)gridDim.x - 1) {
        nl.flags[F_DONE] = 0;
        nl.flags[F_REBUILD] = 0;
        nl.flags[F_SOON] = 0;
        nl.flags[F_BUILDS] += 1;
    }
}

// ---- whole build of a small list ------------------------------------------------
// A small list (n particles with padding) in one block and one launch instead of nine.  A build point that finds
// no rebuild due costs 2 us instead of 14 (in a row of them in a graph), and most do; a rebuild costs more,
// growing with n^2.  Rebuild in one block against the launches, cubes at packing 0.02 to 0.45: 256 particles
// 27 to 47 us against 43 to 27, 384 49 to 74 against 39 to 47, 512 75 to 98 against 43 to 47, 640 115 to 156
// against 44 to 48.  So a forced build, which always rebuilds, takes the block up to 256 particles (at 512,
// energies and forces of one configuration: 204 to 226 us in one block, 171 to 175 with the launches), and a
// conditional one up to 512, where three to four idle build points pay for a rebuild.
// Every distance within a system is taken once (each wave: one particle against 64 later ones, the ballot
// is a word of its row of the adjacency matrix in LDS; the words before the diagonal are then read off the
// columns), and rows, reverse rows and slots are read off the matrix in order, so nothing is sorted or
// searched.
constexpr int kOneBuild = 512, kOneBuildForced = 256;
__global__ __launch_bounds__(kScanBlock) void k_build_one(nepx_state st, nepx_nlist nl, int force) {
    static_assert(kScanBlock >= kOneBuild && kOneBuild % 64 == 0, "one thread per particle");
    __shared__ uint64_t adj[kOneBuild * (kOneBuild / 64 | 1)];  // rows of an odd number of words: columns on distinct banks
    __shared__ double pos[3 * kOneBuild];  // then the row starts
    __shared__ int16_t sysid[kOneBuild];
    __shared__ int32_t wsum[2][kScanBlock / 64];
    int32_t* const flags = nl.flags;
    const bool build = force || want_build(flags);
    const int stale_overflow = force ? 0 : flags[F_OVERFLOW];
    if (threadIdx.x == 0) {
        flags[F_MAXROW] = 0;
        flags[F_LONGSYS] = 0;
    }
    if (!build) return;  // uniform: F_REBUILD and F_SOON are written at the end only
    const int n = st.n, W = (n + 63) / 64, LD = W | 1, i = threadIdx.x;
    const int lane = i & 63, wv = __builtin_amdgcn_readfirstlane(i >> 6);
    if (i < n) {
        const double x = st.x[i], y = st.y[i], z = st.z[i];
        st.xb[i] = x;
        st.yb[i] = y;
        st.zb[i] = z;
        pos[i] = x;
        pos[kOneBuild + i] = y;
        pos[2 * kOneBuild + i] = z;
        const int s = st.sys[i];
        sysid[i] = (int16_t)(s >= 0 && st.sp[s].active ? s : -1);
    }
    __syncthreads();
    for (int r = wv; r < n; r += kScanBlock / 64) {  // uniform per wave
        const int s = __builtin_amdgcn_readfirstlane((int)sysid[r]);
        const nepx_sysparam& sp = st.sp[s < 0 ? 0 : s];
        const double L = sp.L, r2 = __dmul_rn(sp.r_list, sp.r_list);
        const double xr = pos[r], yr = pos[kOneBuild + r], zr = pos[2 * kOneBuild + r];
        for (int w = r >> 6; w < W; ++w) {
            const int j = 64 * w + lane;
            bool in = false;
            if (s >= 0 && j < n && j > r && sysid[j] == s) {
                double tx, ty, tz;
                in = pos_d2(xr, yr, zr, pos[j], pos[kOneBuild + j], pos[2 * kOneBuild + j], L, tx, ty, tz) < r2;
            }
            const uint64_t m = __ballot(in);
            if (lane == 0) adj[r * LD + w] = m;
        }
    }
    __syncthreads();
    // partners before r: bit r of their rows (a diagonal word's bits above the diagonal stay as they are)
    for (int r = wv; r < n; r += kScanBlock / 64) {
        const int wr = r >> 6;
        for (int w = 0; w <= wr; ++w) {
            const int j = 64 * w + lane;
            const uint64_t m = __ballot(j < r && ((adj[j * LD + wr] >> (r & 63)) & 1ull));
            if (lane == 0) adj[r * LD + w] = w < wr ? m : adj[r * LD + w] | m;
        }
    }
    __syncthreads();
    // row lengths (bits above and below the diagonal) and their exclusive scan over the block
    int len[2] = {0, 0}, inc[2];
    if (i < n) {
        for (int w = 0; w < W; ++w) {
            const uint64_t m = adj[i * LD + w];
            const uint64_t lo = w < (i >> 6) ? ~0ull : w > (i >> 6) ? 0ull : (1ull << (i & 63)) - 1ull;
            len[1] += __popcll(m & lo);
            len[0] += __popcll(m & ~lo);
        }
    }
#pragma unroll
    for (int side = 0; side < 2; ++side) {
        inc[side] = len[side];
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int u = __shfl_up(inc[side], o, 64);
            inc[side] += lane >= o ? u : 0;
        }
        if (lane == 63) wsum[side][wv] = inc[side];
    }
    __syncthreads();
    int32_t* const rs = reinterpret_cast<int32_t*>(pos);  // the positions are used up
    int total = 0;
#pragma unroll
    for (int side = 0; side < 2; ++side) {
        int before = 0, all = 0;
        for (int k = 0; k < kScanBlock / 64; ++k) {
            before += k < wv ? wsum[side][k] : 0;
            all += wsum[side][k];
        }
        const int start = before + inc[side] - len[side];
        int32_t* const out = side ? nl.rrow_start : nl.row_start;
        if (i < n) {
            rs[side * kOneBuild + i] = start;
            out[i] = start;
        }
        if (i == 0) out[n] = all;
        total = side ? total : all;
    }
    const bool over = (int64_t)total > nl.cap;
    __syncthreads();
    if (!over && stale_overflow == 0 && i < n) {  // each thread writes its particle's rows
        int pf = rs[i], pr = rs[kOneBuild + i];
        for (int w = 0; w < W; ++w) {
            uint64_t m = adj[i * LD + w];
            while (m) {
                const int j = 64 * w + __builtin_ctzll(m);
                m &= m - 1ull;
                if (j > i) {
                    nl.nbr[pf] = j;
                    nl.slot_row[pf] = i;
                    ++pf;
                } else {  // the slot of (j, i) is past row j's partners between j and i
                    int slot = rs[j];
                    for (int u = j >> 6; u <= (i >> 6); ++u) {
                        uint64_t q = adj[j * LD + u];
                        if (u == (j >> 6)) q &= ~((1ull << (j & 63)) - 1ull);
                        if (u == (i >> 6)) q &= (1ull << (i & 63)) - 1ull;
                        slot += __popcll(q);
                    }
                    nl.rnbr[pr] = slot;
                    if (nl.rpos) nl.rpos[slot] = pr;
                    ++pr;
                }
            }
        }
    }
    if (i == 0) {
        flags[F_PL] = total;
        flags[F_OVERFLOW] = over ? 1 : stale_overflow;
        flags[F_REBUILD] = 0;
        flags[F_SOON] = 0;
        flags[F_BUILDS] += 1;
    }
}

// ---- explicit pair list (API path) ----------------------------------------
// Requests a "build" so that the shared kernels run, clears the overflow, the row counts and the rows' fill
// counters (2 n entries of the cell scratch).
__global__ void k_pairs_begin(nepx_nlist nl, int n) {
    const int k = blockIdx.x * kNB + threadIdx.x;
    if (k == 0) {
        nl.flags[F_REBUILD] = 1;
        nl.flags[F_OVERFLOW] = 0;
        nl.flags[F_MAXROW] = 0;
        nl.flags[F_LONGSYS] = 0;
    }
    if (k <= n) {
        nl.row_count[k] = 0;
        nl.rrow_count[k] = 0;
    }
    if (k < 2 * n) nl.cell_fill[k] = 0;
}

__global__ void k_pairs_count(nepx_nlist nl, const int64_t* pairs, int64_t m, int n) {
    const int64_t k = blockIdx.x * (int64_t)kNB + threadIdx.x;
    if (k >= m) return;
    int a = (int)pairs[2 * k], b = (int)pairs[2 * k + 1];
    if (a == b || a < 0 || b < 0 || a >= n || b >= n) {
        nl.flags[F_OVERFLOW] = 3;
        return;
    }
    if (a > b) {
        const int t = a;
        a = b;
        b = t;
    }
    atomicAdd(&nl.row_count[a], 1);
    atomicAdd(&nl.rrow_count[b], 1);
}

__global__ void k_pairs_fill(nepx_nlist nl, const int64_t* pairs, int64_t m, int32_t* fill_f, int32_t* fill_r) {
    if (nl.flags[F_OVERFLOW]) return;
    const int64_t k = blockIdx.x * (int64_t)kNB + threadIdx.x;
    if (k >= m) return;
    int a = (int)pairs[2 * k], b = (int)pairs[2 * k + 1];
    if (a > b) {
        const int t = a;
        a = b;
        b = t;
    }
    const int pf = nl.row_start[a] + atomicAdd(&fill_f[a], 1);
    nl.nbr[pf] = b;
    nl.slot_row[pf] = a;
    const int pr = nl.rrow_start[b] + atomicAdd(&fill_r[b], 1);
    nl.rnbr[pr] = a;
}

__global__ void k_rows_maxlen(nepx_nlist nl, int n) {
    const int i = blockIdx.x * kNB + threadIdx.x;
    if (i >= n) return;
    const int nf = nl.row_count[i], nr = nl.rrow_count[i];
    if (nf > kSortMax || nr > kSortMax) atomicMax(&nl.flags[F_MAXROW], nf > nr ? nf : nr);
}

// ---- per-step filter and compaction ---------------------------------------
// Each thread evaluates kSlotsPerThread list slots (stride kNB within the
// block's kSlotsPerBlock), issuing every load of all its slots before the
// predicates so the gathers overlap.
constexpr int kSlotsPerThread = kSlotsPerBlock / kNB;

struct SlotEval {
    bool act[kSlotsPerThread];
    int i[kSlotsPerThread], j[kSlotsPerThread];
    double tx[kSlotsPerThread], ty[kSlotsPerThread], tz[kSlotsPerThread];
};

__device__ __forceinline__ void eval_slots(const nepx_state& st, const nepx_nlist& nl, int base, int PL,
                                           SlotEval& r) {
    bool in[kSlotsPerThread];
    int si[kSlotsPerThread], sj[kSlotsPerThread];
#pragma unroll
    for (int k = 0; k < kSlotsPerThread; ++k) {
        const int s = base + k * kNB + threadIdx.x;
        in[k] = s < PL;
        r.i[k] = in[k] ? nl.slot_row[s] : 0;
        r.j[k] = in[k] ? nl.nbr[s] : 0;
    }
    if (st.n_sys == 1) {  // one system: its particle range stands in for the system-id reads
        const int p0 = st.sp[0].p_start, p1 = st.sp[0].p_end;
#pragma unroll
        for (int k = 0; k < kSlotsPerThread; ++k) {
            si[k] = r.i[k] >= p0 && r.i[k] < p1 ? 0 : -1;
            sj[k] = r.j[k] >= p0 && r.j[k] < p1 ? 0 : -1;
        }
    } else {
#pragma unroll
        for (int k = 0; k < kSlotsPerThread; ++k) {
            si[k] = st.sys[r.i[k]];
            sj[k] = st.sys[r.j[k]];
        }
    }
#pragma unroll
    for (int k = 0; k < kSlotsPerThread; ++k) {
        // slots left over from a freed system, or of an inactive one, are not pairs
        const bool same = in[k] && si[k] >= 0 && si[k] == sj[k];
        const nepx_sysparam& sp = st.sp[same ? si[k] : 0];
        const bool live_sys = same && sp.active;
        const double d2 = pair_d2(st, sp.L, r.i[k], r.j[k], r.tx[k], r.ty[k], r.tz[k]);
        r.act[k] = live_sys && d2 < __dmul_rn(sp.rc, sp.rc);
    }
}

// A step whose list is stale (F_REBUILD still set: a step of a multi-step graph after the skin ran
// out) is frozen: the filter selects no pairs and flags F_FROZEN, so the gather and the integrator
// leave the state alone until the next build.
__global__ __launch_bounds__(kNB) void k_filter_count(nepx_state st, nepx_nlist nl) {
    const int PL = nl.flags[F_PL];
    const int base = blockIdx.x * kSlotsPerBlock;
    if (base >= PL || nl.flags[F_OVERFLOW] || nl.flags[F_REBUILD]) {
        if (threadIdx.x == 0) nl.blk_count[blockIdx.x] = 0;
        return;
    }
    SlotEval r;
    eval_slots(st, nl, base, PL, r);
    int cnt = 0;
#pragma unroll
    for (int k = 0; k < kSlotsPerThread; ++k) cnt += r.act[k] ? 1 : 0;
    __shared__ int red[kNB];
    red[threadIdx.x] = cnt;
    __syncthreads();
    for (int off = kNB / 2; off > 0; off >>= 1) {
        if (threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) nl.blk_count[blockIdx.x] = red[0];
}

// Sum of cnt[0..b) by one block (integer, so the order does not matter).
__device__ __forceinline__ int block_prefix(const int32_t* __restrict__ cnt, int b) {
    __shared__ int wpart[kNB / 64];
    int v = 0;
    for (int k = threadIdx.x; k < b; k += kNB) v += cnt[k];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) wpart[threadIdx.x >> 6] = v;
    __syncthreads();
    int t = 0;
#pragma unroll
    for (int w = 0; w < kNB / 64; ++w) t += wpart[w];
    return t;
}

// Each block finds its output offset by summing the counts of the blocks before it (one count per
// kSlotsPerBlock list slots, so few), and the block holding the last slot stores the pair count;
// no separate scan launch.
__global__ __launch_bounds__(kNB) void k_filter_write(nepx_state st, nepx_nlist nl) {
    const int PL = nl.flags[F_PL];
    const int base = blockIdx.x * kSlotsPerBlock;
    const int frozen = nl.flags[F_REBUILD] != 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) nl.flags[F_FROZEN] = frozen;
    if (nl.flags[F_OVERFLOW] || frozen || PL == 0) {
        if (blockIdx.x == 0 && threadIdx.x == 0) nl.flags[F_P] = 0;
        return;
    }
    // a new pass: the pair kernels tag the reverse-order records they write with it
    if (blockIdx.x == 0 && threadIdx.x == 0) nl.flags[F_TAG] = nl.flags[F_TAG] + 1;
    if (base >= PL) return;
    const int first = block_prefix(nl.blk_count, blockIdx.x);
    if (base + kSlotsPerBlock >= PL && threadIdx.x == 0) nl.flags[F_P] = first + nl.blk_count[blockIdx.x];
    __shared__ int wsum[kSlotsPerThread][kNB / 64];
    SlotEval r;
    eval_slots(st, nl, base, PL, r);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    uint64_t below[kSlotsPerThread];
#pragma unroll
    for (int k = 0; k < kSlotsPerThread; ++k) {
        const uint64_t mask = __ballot(r.act[k]);
        below[k] = mask & ((1ull << lane) - 1ull);
        if (lane == 0) wsum[k][wv] = __popcll(mask);
    }
    __syncthreads();
    int out = first;
#pragma unroll
    for (int k = 0; k < kSlotsPerThread; ++k) {
        const int s = base + k * kNB + threadIdx.x;
        int woff = 0, tot = 0;
#pragma unroll
        for (int w = 0; w < kNB / 64; ++w) {
            woff += w < wv ? wsum[k][w] : 0;
            tot += wsum[k][w];
        }
        if (s < PL) {
            if (r.act[k]) {
                const int c = out + woff + __popcll(below[k]);
                nl.cidx[s] = c;
                nl.pair_i[c] = r.i[k];
                nl.pair_j[c] = r.j[k];
                if (nl.pair_e) nl.pair_e[c] = nl.rpos[s];
                reinterpret_cast<float4*>(nl.pair_t)[c] =
                    make_float4((float)r.tx[k], (float)r.ty[k], (float)r.tz[k], 0.f);
            } else {
                nl.cidx[s] = -1;
            }
        }
        out += tot;
    }
}

// ---- gather ----------------------------------------------------------------
// GL lanes per particle (tuned; 16 by default): lanes stride over the
// particle's forward row (i-role: +F, +tau_i, +E) and reverse row (j-role:
// -F, +tau_j), accumulate in FP64 and reduce with a fixed butterfly, so the
// result is independent of timing (and, for one GL, of the launch).  The j side
// comes from the reverse-order records when this pass's pair kernel wrote them
// (the same values, so the same sums bit for bit), else through the slot ->
// compacted-index map from the per-pair records.
template <int GL>
__device__ __forceinline__ double red_lanes(double v) {
#pragma unroll
    for (int o = GL / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, GL);
    return v;
}

template <int GL>
__global__ __launch_bounds__(kNB) void k_gather(nepx_state st, nepx_nlist nl, const float4* __restrict__ out) {
    // particles of one XCD are contiguous, so the records that neighbouring rows share
    // (forward rows of i, reverse rows of its neighbours) are fetched into one L2
    const int k = (xcd_contiguous_block(blockIdx.x, gridDim.x) * kNB + threadIdx.x) / GL;
    const int sub = threadIdx.x % GL;
    if (k >= st.n) return;  // whole lane groups exit together
    if (nl.flags[F_OVERFLOW] || nl.flags[F_FROZEN]) return;  // skipped step: forces stay as they are
    // the pair kernel of this pass wrote reverse-order records (uniform: every thread reads the same flags)
    const int tag = nl.flags[F_TAG];
    const bool rev = nl.rrec != nullptr && nl.flags[F_RTAG] == tag;
    double fx = 0, fy = 0, fz = 0, tx = 0, ty = 0, tz = 0, u = 0;
    if (live(st, k)) {
        for (int s = nl.row_start[k] + sub; s < nl.row_start[k + 1]; s += GL) {
            const int c = nl.cidx[s];
            if (c < 0) continue;
            const float4 a = out[3 * (size_t)c], b = out[3 * (size_t)c + 1];
            fx += a.x;
            fy += a.y;
            fz += a.z;
            u += a.w;
            tx += b.x;
            ty += b.y;
            tz += b.z;
        }
        if (rev) {  // this pass's j-side records, in reverse-row order: read contiguously
            const float4* rr = reinterpret_cast<const float4*>(nl.rrec);
            for (int e = nl.rrow_start[k] + sub; e < nl.rrow_start[k + 1]; e += GL) {
                const float4 a = rr[2 * (size_t)e];
                if (__float_as_int(a.w) != tag) continue;  // no active pair at this entry this step
                const float4 b = rr[2 * (size_t)e + 1];
                fx -= a.x;
                fy -= a.y;
                fz -= a.z;
                tx += b.x;
                ty += b.y;
                tz += b.z;
            }
        } else {
            for (int e = nl.rrow_start[k] + sub; e < nl.rrow_start[k + 1]; e += GL) {
                const int c = nl.cidx[nl.rnbr[e]];
                if (c < 0) continue;
                const float4 a = out[3 * (size_t)c], b = out[3 * (size_t)c + 2];
                fx -= a.x;
                fy -= a.y;
                fz -= a.z;
                tx += b.x;
                ty += b.y;
                tz += b.z;
            }
        }
    }
    fx = red_lanes<GL>(fx);
    fy = red_lanes<GL>(fy);
    fz = red_lanes<GL>(fz);
    tx = red_lanes<GL>(tx);
    ty = red_lanes<GL>(ty);
    tz = red_lanes<GL>(tz);
    u = red_lanes<GL>(u);
    if (sub == 0) {
        st.fx[k] = fx;
        st.fy[k] = fy;
        st.fz[k] = fz;
        st.tx[k] = tx;
        st.ty[k] = ty;
        st.tz[k] = tz;
        st.upot[k] = u;
    }
}

// State and list buffers every entry point reads; blk_count (the compaction's
// per-block partials) is checked by the entry points that take it from the list.
static int check_state_core(const nepx_state* st, const nepx_nlist* nl) {
    NEPX_REQUIRE(st && nl, NEPX_EINVAL, "null state or list");
    NEPX_REQUIRE(st->n > 0 && st->n_sys > 0, NEPX_EINVAL, "empty state");
    NEPX_REQUIRE(st->x && st->y && st->z && st->sys && st->sp, NEPX_EINVAL, "null state buffer");
    NEPX_REQUIRE(nl->flags && nl->nbr && nl->slot_row && nl->rnbr && nl->row_start && nl->rrow_start &&
                     nl->row_count && nl->rrow_count && nl->cidx && nl->pair_i && nl->pair_j && nl->pair_t,
                 NEPX_EINVAL, "null list buffer");
    NEPX_REQUIRE(nl->cap > 0 && nl->cap < (int64_t)1 << 31, NEPX_ECAP, "list capacity %lld out of range",
                 (long long)nl->cap);
    NEPX_REQUIRE(!(nl->pair_e || nl->rrec) || (nl->rpos && nl->pair_e && nl->rrec), NEPX_EINVAL,
                 "reverse-order records need rpos, pair_e and rrec together");
    return NEPX_OK;
}

static int check_state(const nepx_state* st, const nepx_nlist* nl) {
    const int rc = check_state_core(st, nl);
    if (rc) return rc;
    NEPX_REQUIRE(nl->blk_count, NEPX_EINVAL, "null list buffer (blk_count)");
    return NEPX_OK;
}

static int blocks_for(int64_t n, int b) { return (int)((n + b - 1) / b); }

}  // namespace nepx

using namespace nepx;

extern "C" int nepx_nlist_build(nepx_state* st, nepx_nlist* nl, int32_t force, void* stream) {
    int rc = check_state(st, nl);
    if (rc) return rc;
    NEPX_REQUIRE(nl->cell_count && nl->cell_start && nl->cell_fill && nl->cell_list && nl->cell_of && nl->cell_pos,
                 NEPX_EINVAL, "null cell buffer");
    NEPX_REQUIRE(((uintptr_t)nl->cell_pos & 31) == 0, NEPX_EINVAL, "cell_pos must be 32-byte aligned");
    hipStream_t s = as_stream(stream);
    const int n = st->n;
    if (n <= (force ? kOneBuildForced : kOneBuild) && st->n_sys <= INT16_MAX) {
        hipLaunchKernelGGL(k_build_one, dim3(1), dim3(kScanBlock), 0, s, *st, *nl, force ? 1 : 0);
        NEPX_LAUNCH_CHECK();
        return NEPX_OK;
    }
    const int gb = blocks_for(n, kNB);
    const int nct = nl->n_cells_total > 0 ? nl->n_cells_total : 1;
    const int gs = blocks_for(n, kSortWaves) < 4096 ? blocks_for(n, kSortWaves) : 4096;
    hipLaunchKernelGGL(k_build_begin, dim3(blocks_for(nct, kNB)), dim3(kNB), 0, s, nl->flags, nl->cell_count,
                       nl->cell_fill, (int64_t)nct, force ? 1 : 0);
    hipLaunchKernelGGL(k_cells_count, dim3(gb), dim3(kNB), 0, s, *st, *nl);
    hipLaunchKernelGGL(k_scan_cells, dim3(1), dim3(kScanBlock), 0, s, *st, *nl);
    hipLaunchKernelGGL(k_cells_fill, dim3(gb), dim3(kNB), 0, s, *st, *nl);
#define NEPX_ROWS(LG)                                                                                     \
    const int gg = blocks_for((int64_t)n * LG, kNB);                                                      \
    hipLaunchKernelGGL(k_nbr_count<LG>, dim3(gg), dim3(kNB), 0, s, *st, *nl);                             \
    hipLaunchKernelGGL(k_scan_rows<false>, dim3(2), dim3(kScanBlock), 0, s, *nl, gg, n);                  \
    hipLaunchKernelGGL(k_nbr_fill<LG>, dim3(gg), dim3(kNB), 0, s, *st, *nl)
    if (n <= kWideGroups) {
        NEPX_ROWS(64);
    } else {
        NEPX_ROWS(16);
    }
#undef NEPX_ROWS
    hipLaunchKernelGGL(k_sort_rows, dim3(gs), dim3(kSortThreads), 0, s, *nl, n);
    hipLaunchKernelGGL(k_rev_rows, dim3(gs), dim3(kSortThreads), 0, s, *nl, n);
    NEPX_LAUNCH_CHECK();
    return NEPX_OK;
}

extern "C" int nepx_nlist_from_pairs(nepx_state* st, nepx_nlist* nl, const int64_t* pairs, int64_t m,
                                     void* stream) {
    int rc = check_state(st, nl);
    if (rc) return rc;
    NEPX_REQUIRE(m >= 0 && (m == 0 || pairs), NEPX_EINVAL, "bad pair array");
    NEPX_REQUIRE(m <= nl->cap, NEPX_ECAP, "%lld pairs exceed list capacity %lld", (long long)m,
                 (long long)nl->cap);
    NEPX_REQUIRE(nl->cell_fill && nl->cell_count, NEPX_EINVAL, "null scratch buffer");
    // per-row fill counters reuse the cell scratch
    NEPX_REQUIRE(nl->n_cells_total >= 2 * st->n, NEPX_ECAP, "cell scratch (%d) smaller than 2*n (%d)",
                 nl->n_cells_total, 2 * st->n);
    hipStream_t s = as_stream(stream);
    const int n = st->n;
    const int gs = blocks_for(n, kSortWaves) < 4096 ? blocks_for(n, kSortWaves) : 4096;
    hipLaunchKernelGGL(k_pairs_begin, dim3(blocks_for(2 * (int64_t)n + 1, kNB)), dim3(kNB), 0, s, *nl, n);
    if (m > 0)
        hipLaunchKernelGGL(k_pairs_count, dim3(blocks_for(m, kNB)), dim3(kNB), 0, s, *nl, pairs, m, n);
    hipLaunchKernelGGL(k_rows_maxlen, dim3(blocks_for(n, kNB)), dim3(kNB), 0, s, *nl, n);
    hipLaunchKernelGGL(k_scan_rows<true>, dim3(2), dim3(kScanBlock), 0, s, *nl, n, n);
    if (m > 0)
        hipLaunchKernelGGL(k_pairs_fill, dim3(blocks_for(m, kNB)), dim3(kNB), 0, s, *nl, pairs, m,
                           nl->cell_fill, nl->cell_fill + n);
    hipLaunchKernelGGL(k_sort_rows, dim3(gs), dim3(kSortThreads), 0, s, *nl, n);
    hipLaunchKernelGGL(k_rev_rows, dim3(gs), dim3(kSortThreads), 0, s, *nl, n);
    NEPX_LAUNCH_CHECK();
    return NEPX_OK;
}

extern "C" int nepx_pairs_filter(nepx_state* st, nepx_nlist* nl, void* stream) {
    int rc = check_state(st, nl);
    if (rc) return rc;
    hipStream_t s = as_stream(stream);
    const int nblk = blocks_for(nl->cap, kSlotsPerBlock);
    hipLaunchKernelGGL(k_filter_count, dim3(nblk), dim3(kNB), 0, s, *st, *nl);
    hipLaunchKernelGGL(k_filter_write, dim3(nblk), dim3(kNB), 0, s, *st, *nl);
    NEPX_LAUNCH_CHECK();
    return NEPX_OK;
}

// ---- allocation-free filter --------------------------------------------------
// Scratch of nepx_pairs_filter_noalloc: the compaction's per-block partial counts
// (one int per kSlotsPerBlock list slots), in place of the list's blk_count.
// A file-scope device array: each GPU the library runs on holds its own copy
// (256 KiB) until the process ends.  Host code never passes the array's name to
// a kernel; it uses the address hipGetSymbolAddress returns for the current
// device, looked up once per device on the first call there.
constexpr int kNoallocMaxBlocks = 1 << 16;   // list capacity up to 64 Mi slots
static __device__ __align__(256) int32_t scratch[kNoallocMaxBlocks];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
int32_t* g_scratch_dev[kMaxDevices] = {};

int scratch_for_current_device(int32_t** out) {
    int dev = -1;
    NEPX_HIP_CHECK(hipGetDevice(&dev));
    NEPX_REQUIRE(dev >= 0 && dev < kMaxDevices, NEPX_EINVAL, "device %d out of range", dev);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_dev[dev] == nullptr) {
        void* p = nullptr;
        NEPX_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        NEPX_REQUIRE(p != nullptr, NEPX_EHIP, "no device address for the filter scratch");
        g_scratch_dev[dev] = static_cast<int32_t*>(p);
    }
    *out = g_scratch_dev[dev];
    return NEPX_OK;
}
}  // namespace

extern "C" int nepx_pairs_filter_noalloc(nepx_state* st, nepx_nlist* nl, void* stream) {
    int rc = check_state_core(st, nl);
    if (rc) return rc;
    const int nblk = blocks_for(nl->cap, kSlotsPerBlock);
    NEPX_REQUIRE(nblk <= kNoallocMaxBlocks, NEPX_ECAP,
                 "list capacity %lld exceeds the %lld slots of the allocation-free filter's scratch",
                 (long long)nl->cap, (long long)kNoallocMaxBlocks * kSlotsPerBlock);
    int32_t* scr = nullptr;
    rc = scratch_for_current_device(&scr);
    if (rc) return rc;
    // k_filter_count writes every partial that k_filter_write reads (zero for empty blocks), so
    // what an earlier call left in the scratch is never read.
    nepx_nlist l = *nl;
    l.blk_count = scr;
    hipStream_t s = as_stream(stream);
    hipLaunchKernelGGL(k_filter_count, dim3(nblk), dim3(kNB), 0, s, *st, l);
    hipLaunchKernelGGL(k_filter_write, dim3(nblk), dim3(kNB), 0, s, *st, l);
    NEPX_LAUNCH_CHECK();
    return NEPX_OK;
}

extern "C" int nepx_forces_gather(nepx_state* st, nepx_nlist* nl, const float* pair_out, void* stream) {
    int rc = check_state(st, nl);
    if (rc) return rc;
    NEPX_REQUIRE(pair_out && st->fx && st->fy && st->fz && st->tx && st->ty && st->tz && st->upot, NEPX_EINVAL,
                 "null force buffer");
    const int gl = tuning().gather_lanes;
#define NEPX_GATHER(GL)                                                                                   \
    hipLaunchKernelGGL(k_gather<GL>, dim3(blocks_for((int64_t)st->n * GL, kNB)), dim3(kNB), 0,             \
                       as_stream(stream), *st, *nl, (const float4*)pair_out)
    switch (gl) {
        case 4: NEPX_GATHER(4); break;
        case 8: NEPX_GATHER(8); break;
        case 32: NEPX_GATHER(32); break;
        case 64: NEPX_GATHER(64); break;
        default: NEPX_GATHER(16); break;
    }
#undef NEPX_GATHER
    NEPX_LAUNCH_CHECK();
    return NEPX_OK;
}
