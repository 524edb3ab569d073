// Merged levels: consecutive levels of a sweep as one launch.
//
// A launched level costs about 3.5 us however little it holds (a launch, the
// layout load, the gather: two dependent round trips to memory another XCD
// wrote), and outside the trailing block an application still runs 20 to 40 of
// them per direction. Inside a run of levels G, with P the rows before it, the
// forward substitution y_i = (r_i - sum l_ij y_j) / d_i can be carried out
// symbolically for the dependencies inside G: every row becomes one sum
//   y_i = sum_{j in G} a_ij r_j + sum_{p in P} b_ip y_p,
// all of whose operands exist before the launch. Two levels merged hold 1.4 to
// 1.9 times their entries on grids and R-MAT graphs, four 2.2 to 5 times;
// kernels then take one launch instead of two to eight (the rule of what
// joins is in host/merge.cpp). The coefficients are fp64 sums of terms of one
// sign. An application is as accurate with them as without (energy-norm error
// against 80-bit arithmetic, N(0,1): 32^3 grid 7.6e-15 / 7.8e-15, 32^3 SDDM
// 1.0e-15 / 1.0e-15, R-MAT s13 9.7e-17 / 8.8e-17).
//
// Used by applications with fp64 vectors of factors with a trailing block, in
// every schedule. Sweep launches of an application and its time, before ->
// after: 48^3 grid 44 + 1 run -> 15, a solve 6.8 -> 3.9 ms; 63^3 SDDM 58 -> 27,
// an application 270 -> 167 us; 89^3 SDDM 80 -> 57, a solve 12.0 -> 10.4 ms;
// R-MAT s14 8 -> 3, 0.94 -> 0.76 ms. fp32 vectors keep their levels: merged,
// small components of an R-MAT s18 solve moved by 5e-7 of x's rms.
#include "common.hpp"

namespace apxchol_amd {

// One wave per batch. Each lane runs the fma chain of its entries, the lanes of
// a row combine as in the level kernels, and the row's first lane stores. CB
// columns (c0 ..) of kp vectors stored row by row at a time: an entry is loaded
// once and its CB operands are contiguous; a column's arithmetic does not
// depend on CB. Chunks past the first (rows of more than 256 entries) follow in
// order.
template <int CB>
__device__ __forceinline__ void sweep_merged_body(int vb, int c0, const merge_desc& g, int b0, int nb, int backward,
                                                  const double* __restrict__ rhs, double* out, const pcg_state* st, int kp,
                                                  const batch_state* bs) {
    const int w = vb * kWavesPerBlock + static_cast<int>(threadIdx.x) / kWave;
    if (w >= nb) return;
    const int lane = threadIdx.x & (kWave - 1);
    const int b = __builtin_amdgcn_readfirstlane(b0 + w);
    const merge_batch mb = g.batch[b];
    const lane_rec rc = g.rec[static_cast<size_t>(b) * kWave + lane];
    const size_t e0 = static_cast<size_t>(mb.chunk) * kEpl * kWave + lane;
    const double* __restrict__ val = g.val;
    int j[kEpl];
    double v[kEpl];
#pragma unroll
    for (int k = 0; k < kEpl; ++k) {
        j[k] = g.idx[e0 + static_cast<size_t>(k) * kWave];
        v[k] = val[e0 + static_cast<size_t>(k) * kWave];
    }
    asm volatile("" ::: "memory");
    if (bs ? bs->active == 0 : (st && st->done)) return;
    typedef double vec __attribute__((ext_vector_type(CB)));
    double shift[CB];
#pragma unroll
    for (int u = 0; u < CB; ++u) shift[u] = (st && !backward) ? st[c0 + u].shift : 0.0;
    const int n = static_cast<int>(rc.info >> 9);
    double part[CB];
#pragma unroll
    for (int u = 0; u < CB; ++u) part[u] = 0.0;
    for (int c = 0;;) {
        double x[kEpl][CB];
#pragma unroll
        for (int k = 0; k < kEpl; ++k) {
            if (c * kEpl + k < n) {
                if (j[k] >= 0) {
                    const vec q = *reinterpret_cast<const vec*>(out + static_cast<size_t>(j[k]) * kp + c0);
#pragma unroll
                    for (int u = 0; u < CB; ++u) x[k][u] = q[u];
                } else {
                    const vec q = *reinterpret_cast<const vec*>(rhs + static_cast<size_t>(~j[k]) * kp + c0);
#pragma unroll
                    for (int u = 0; u < CB; ++u)
                        x[k][u] = q[u] - shift[u];
                }
            } else {
#pragma unroll
                for (int u = 0; u < CB; ++u) x[k][u] = 0.0;
            }
        }
        double vc[kEpl];
#pragma unroll
        for (int k = 0; k < kEpl; ++k) vc[k] = v[k];
        const bool more = ++c < static_cast<int>(mb.chunks);
        if (more) {
            const size_t e = e0 + static_cast<size_t>(c) * kEpl * kWave;
#pragma unroll
            for (int k = 0; k < kEpl; ++k) {
                j[k] = g.idx[e + static_cast<size_t>(k) * kWave];
                v[k] = val[e + static_cast<size_t>(k) * kWave];
            }
        }
#pragma unroll
        for (int k = 0; k < kEpl; ++k)
#pragma unroll
            for (int u = 0; u < CB; ++u) part[u] = fma(vc[k], x[k][u], part[u]);
        if (!more) break;
    }
    const int G = 1 << (rc.info & 7u);
#pragma unroll
    for (int u = 0; u < CB; ++u) part[u] = group_tree_sum(part[u], G);
    if (rc.row >= 0 && ((rc.info >> 3) & 63u) == 0) {
        vec q;
#pragma unroll
        for (int u = 0; u < CB; ++u) q[u] = part[u];
        *reinterpret_cast<vec*>(out + static_cast<size_t>(rc.row) * kp + c0) = q;
    }
}
template <int CB>
__global__ __launch_bounds__(kBlock) void sweep_merged(merge_desc g, int b0, int nb, int backward,
                                                       const double* __restrict__ rhs, double* out, const pcg_state* st,
                                                       int kp, const batch_state* bs) {
    sweep_merged_body<CB>(static_cast<int>(blockIdx.x), static_cast<int>(blockIdx.y) * CB, g, b0, nb, backward,
                                  rhs, out, st, kp, bs);
}

}  // namespace apxchol_amd
