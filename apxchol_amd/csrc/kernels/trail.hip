// The trailing block of the preconditioner, applied through its explicit
// inverse.
//
// The last eliminations of an approximate Cholesky factor are its long, thin
// part: on an 89^3 grid 129 of the 169 dependent levels of a sweep hold 4,832
// of 704,969 rows, on an R-MAT graph of scale 18 1,934 of 1,964 hold 7,004 of
// 262,143. Walking them costs a launch or a barrier per level and direction
// (0.6 .. 4.5 us each) for almost no bytes. With the rows split as P (before
// the block) and T (the block), L = [L_PP 0; L_TP T_], the pair of sweeps is
//   y_P = L_PP^-1 r_P                      (forward levels of P)
//   c   = r_T - L_TP y_P                   (trail_couple)
//   z_T = T_^-T W T_^-1 c = S c            (trail_apply: one dense product)
//   z_P = L_PP^-T (W y_P - L_TP^T z_T)     (back levels of P)
// (W: the fp16 storage's inv_scale^2, else 1), so the whole chain of the
// block's levels in both directions is one coupling launch and one symmetric
// matrix-vector product. S is computed once per factor, in fp64 on the matrix
// cores, and kept in the sweeps' vector precision. Every entry of T_^-1 is a
// sum of terms of one sign (the factor's off-diagonals are never positive), so
// forming S cancels nothing; rounding its entries does hide what a much softer
// direction covers, and a factor where that could matter walks every level
// (trail_is_sound, host/trail.cpp). c and the product's sums are fp64
// for fp32 vectors too: fp32 sums of a few thousand terms of both signs lost
// digits the walked levels keep (256^2 grid, projected N(0,1), error of an
// application against fp64: walked 8.5e-7, fp32 sums 1.5e-6, fp64 sums 3.9e-7;
// the product stays bound by its bytes).
//
// The block's first row depends on the factor and the vector precision alone
// (there is none where device memory does not suffice), never on the schedule,
// and the kernels below give every column of a block
// and every member of a group the single application's arithmetic, so all
// schedules keep agreeing bit for bit.
#include "common.hpp"

#include <type_traits>

namespace apxchol_amd {

// ---- application ---------------------------------------------------------------

inline constexpr int kTrailWaves = kTrailThreads / kWave;

// c = r - L_TP y_P for the rows of the block. Rows of at most 64 * kEpl
// entries before the block come packed in the static lane layout of the
// launched levels (two dependent loads: layout, gathered values), a batch per
// wave; a longer row (the hubs of power-law graphs: up to 28,854 entries at
// R-MAT scale 18) is summed by a whole workgroup, each thread a strided chain,
// sixteen loads in flight, then wave trees and the waves in order. Column
// c = blockIdx.y of kp vectors stored row by row (kp = 1: one vector).
template <class TO, bool F16>
__device__ __forceinline__ void trail_couple_body(int vb, int col, const trail_desc& t, const sweep_desc& d,
                                                  const double* __restrict__ rhs, const TO* __restrict__ y,
                                                  double* __restrict__ c, const pcg_state* st, int kp,
                                                  const batch_state* bs) {
    __shared__ double sh[kCoupleThreads / kWave];
    const int lane = threadIdx.x & (kWave - 1);
    const int wv = static_cast<int>(threadIdx.x) / kWave;
    constexpr int kWaves = kCoupleThreads / kWave;
    const int packed = (t.npack + kWaves - 1) / kWaves;
    if (vb < packed) {
        const int b = vb * kWaves + wv;
        if (b >= t.npack) return;
        const lane_rec rc = t.rec[static_cast<size_t>(b) * kWave + lane];
        entry32 e[kEpl];
#pragma unroll
        for (int k = 0; k < kEpl; ++k) e[k] = t.ent[(static_cast<size_t>(b) * kEpl + k) * kWave + lane];
        asm volatile("" ::: "memory");
        if (bs ? bs->active == 0 : (st && st->done)) return;
        const double shift = st ? st[col].shift : 0.0;
        const int nv = static_cast<int>((rc.info >> 9) & 7u);
        const int G = 1 << (rc.info & 7u);
        const bool head = rc.row >= 0 && ((rc.info >> 3) & 63u) == 0;
        TO xv[kEpl];
#pragma unroll
        for (int k = 0; k < kEpl; ++k) xv[k] = k < nv ? y[static_cast<size_t>(e[k].idx) * kp + col] : static_cast<TO>(0);
        double r = 0.0;
        if (head) r = rhs[static_cast<size_t>(t.first + rc.row) * kp + col] - shift;
        double part = 0.0;
#pragma unroll
        for (int k = 0; k < kEpl; ++k) part = fma(static_cast<double>(e[k].val), static_cast<double>(xv[k]), part);
        part = group_tree_sum(part, G);
        if (head) c[static_cast<size_t>(rc.row) * kp + col] = r - part;
        return;
    }
    if (bs ? bs->active == 0 : (st && st->done)) return;
    const double shift = st ? st[col].shift : 0.0;
    const int4 q = t.longrow[vb - packed];   // block row, first entry, entries
    const unsigned rb = static_cast<unsigned>(q.y), len = static_cast<unsigned>(q.z);
    constexpr int U = 16;
    double part = 0.0;
    for (unsigned c0 = 0; c0 < len; c0 += kCoupleThreads * U) {
        int jj[U];
        float vv[U];
        TO xv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const unsigned p = c0 + static_cast<unsigned>(u) * kCoupleThreads + threadIdx.x;
            load_entry<F16>(d, p < len ? rb + p : rb, jj[u], vv[u]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const unsigned p = c0 + static_cast<unsigned>(u) * kCoupleThreads + threadIdx.x;
            xv[u] = p < len ? y[static_cast<size_t>(jj[u]) * kp + col] : static_cast<TO>(0);
            if (p >= len) vv[u] = 0.0f;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) part = fma(static_cast<double>(vv[u]), static_cast<double>(xv[u]), part);
    }
    part = group_tree_sum(part, kWave);
    if (lane == 0) sh[wv] = part;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = sh[0];
        for (int k = 1; k < kWaves; ++k) s += sh[k];
        const double r = rhs[static_cast<size_t>(t.first + q.x) * kp + col] - shift;
        c[static_cast<size_t>(q.x) * kp + col] = r - s;
    }
}
template <class TO, bool F16>
__global__ __launch_bounds__(kCoupleThreads) void trail_couple(trail_desc t, sweep_desc d,
                                                               const double* __restrict__ rhs,
                                                               const TO* __restrict__ y, double* __restrict__ c,
                                                               const pcg_state* st, int kp, const batch_state* bs) {
    trail_couple_body<TO, F16>(static_cast<int>(blockIdx.x), static_cast<int>(blockIdx.y), t, d, rhs, y, c, st, kp,
                               bs);
}

// One term of the product without the zeros of S, which join rows of different
// components: a workgroup one of whose sums is not finite sums again with it
// (the same chains, an entry at a time: few registers), so an infinity or NaN
// stays in its component as in the walk of the levels.
template <class TO>
__device__ __forceinline__ double trail_skip(TO v, double c, double acc) {
    return v == static_cast<TO>(0) ? acc : fma(static_cast<double>(v), c, acc);
}
__device__ __forceinline__ bool trail_finite(double v) { return fabs(v) <= 1.7976931348623157e308; }

// z_T = S c. HBM-bound: S is read once, n^2 values (R-MAT s18, 7,004 fp32 rows,
// 196 MB: 35.2 us, 5.6 TB/s; 48^3 grid, 3,773 fp64 rows, 114 MB: 20.1 us, 5.7
// TB/s; a plain copy moves 5.0). With the coupling launch (35.0 us there: hub rows)
// it replaces 12 tail runs of 115 us and their couplings an iteration. A workgroup of 16 waves
// owns kTrailLine / sizeof(TO) rows (one 128-byte line of every row of S,
// which is symmetric, so a row is read as a column) and cuts the sum over k
// into 1024 / rows chunks; a thread runs its row's fma chain over one chunk,
// sixteen loads in flight, with c in LDS. The chunk sums of a wave are added in
// order, then the 16 waves': one fixed order per row.
template <class TO>
__device__ __forceinline__ void trail_apply_body(int vb, unsigned char* lds, const trail_desc& t,
                                                 const double* __restrict__ c, TO* __restrict__ z, const pcg_state* st) {
    if (st && st->done) return;
    constexpr int R = kTrailLine / static_cast<int>(sizeof(TO));
    constexpr int kChunks = kTrailThreads / R;
    constexpr int kPerWave = kChunks / kTrailWaves;
    double* cs = reinterpret_cast<double*>(lds);
    const int ch = t.chunk;
    const auto product = [&](auto skip_zeros, int tid) {
        for (int q = tid; q < kChunks * ch; q += kTrailThreads) cs[q] = q < t.n ? c[q] : 0.0;
        __syncthreads();
        const int p = tid / R;
        const TO* __restrict__ s = static_cast<const TO*>(t.s) + static_cast<size_t>(p) * ch * t.ld + vb * R + tid % R;
        const double* cp = cs + p * ch;
        double acc = 0.0;
        if constexpr (decltype(skip_zeros)::value) {
#pragma unroll 1
            for (int k = 0; k < ch; ++k) acc = trail_skip(s[static_cast<size_t>(k) * t.ld], cp[k], acc);
        } else {
            int k = 0;
            for (; k + 16 <= ch; k += 16) {
                TO v[16];
#pragma unroll
                for (int u = 0; u < 16; ++u) v[u] = s[static_cast<size_t>(k + u) * t.ld];
#pragma unroll
                for (int u = 0; u < 16; ++u) acc = fma(static_cast<double>(v[u]), cp[k + u], acc);
            }
            for (; k < ch; k += 4) {
                TO v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) v[u] = s[static_cast<size_t>(k + u) * t.ld];
#pragma unroll
                for (int u = 0; u < 4; ++u) acc = fma(static_cast<double>(v[u]), cp[k + u], acc);
            }
        }
        __syncthreads();
        cs[tid] = acc;
        __syncthreads();
        // The rows' sums are wave 0's.
        static_assert(R <= kWave, "rows of a workgroup");
        bool finite = true;
        if (tid < R && vb * R + tid < t.n) {
            double sum = 0.0;
#pragma unroll
            for (int w = 0; w < kTrailWaves; ++w) {
                double q = cs[w * kWave + tid];
#pragma unroll
                for (int j = 1; j < kPerWave; ++j) q += cs[w * kWave + j * R + tid];
                sum = w == 0 ? q : sum + q;
            }
            z[t.first + vb * R + tid] = static_cast<TO>(sum);
            finite = trail_finite(sum);
        }
        return finite;
    };
    int tid = static_cast<int>(threadIdx.x);
    const bool finite = product(std::false_type{}, tid);
    // In cs, whose last reads are wave 0's too. (A variable of its own would
    // move cs off its alignment: 8 to 10 us a product.)
    int* again = reinterpret_cast<int*>(lds);
    if (tid < kWave) {
        const int any = __any(!finite);
        if (tid == 0) *again = any;
    }
    __syncthreads();
    if (*again) {
        __syncthreads();
        asm volatile("" : "+v"(tid));   // nothing of the first pass is kept for this one
        (void)product(std::true_type{}, tid);
    }
}
// (Eight waves a SIMD: two workgroups a compute unit, 64 registers.)
template <class TO>
__global__ __launch_bounds__(kTrailThreads, 8) void trail_apply(trail_desc t, const double* __restrict__ c,
                                                             TO* __restrict__ z, const pcg_state* st) {
    extern __shared__ unsigned char trail_smem[];
    trail_apply_body<TO>(static_cast<int>(blockIdx.x), trail_smem, t, c, z, st);
}

// The product for CT columns of a block [n][kp] at a time: a wave takes 64
// rows and the chunks w * kPerWave .. of the single kernel, so a value of S
// feeds CT fmas whose other operand is wave-uniform (scalar loads of c); the
// chunk sums combine as above, so each column has the single kernel's bits.
// Bound by the vector fmas: n^2 kp of them.
template <class TO, int CT>
__global__ __launch_bounds__(kTrailThreads) void trail_apply_k(trail_desc t, const double* __restrict__ c,
                                                               TO* __restrict__ z, int kp, const batch_state* bs) {
    if (bs && bs->active == 0) return;
    constexpr int R = kTrailLine / static_cast<int>(sizeof(TO));
    constexpr int kChunks = kTrailThreads / R;
    constexpr int kPerWave = kChunks / kTrailWaves;
    static_assert(kTrailWaves * kWave * CT * sizeof(double) <= 65536, "static LDS");
    __shared__ double red[kTrailWaves][CT][kWave];
    const int c0 = static_cast<int>(blockIdx.y) * CT;
    // Returns whether every output of this thread is finite.
    const auto product = [&](auto skip_zeros, int tid) {
        const int lane = tid & (kWave - 1);
        const int w = __builtin_amdgcn_readfirstlane(tid / kWave);
        const int i = static_cast<int>(blockIdx.x) * kWave + lane;   // < ld: rows past n are zero in S
        double q[CT];
#pragma unroll
        for (int j = 0; j < kPerWave; ++j) {
            const int k0 = (w * kPerWave + j) * t.chunk;
            const int k1 = min(k0 + t.chunk, t.n);
            double acc[CT];
#pragma unroll
            for (int u = 0; u < CT; ++u) acc[u] = 0.0;
            const TO* __restrict__ s = static_cast<const TO*>(t.s) + i;
            int k = k0;
            if constexpr (decltype(skip_zeros)::value) {
#pragma unroll 1
                for (; k < k1; ++k) {
                    const TO v = s[static_cast<size_t>(k) * t.ld];
                    const double* __restrict__ cr = c + static_cast<size_t>(k) * kp + c0;
#pragma unroll
                    for (int u = 0; u < CT; ++u) acc[u] = trail_skip(v, cr[u], acc[u]);
                }
            }
            for (; k + 4 <= k1; k += 4) {
                TO v[4];
#pragma unroll
                for (int b = 0; b < 4; ++b) v[b] = s[static_cast<size_t>(k + b) * t.ld];
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const double* __restrict__ cr = c + static_cast<size_t>(k + b) * kp + c0;
#pragma unroll
                    for (int u = 0; u < CT; ++u) acc[u] = fma(static_cast<double>(v[b]), cr[u], acc[u]);
                }
            }
            for (; k < k1; ++k) {
                const TO v = s[static_cast<size_t>(k) * t.ld];
                const double* __restrict__ cr = c + static_cast<size_t>(k) * kp + c0;
#pragma unroll
                for (int u = 0; u < CT; ++u) acc[u] = fma(static_cast<double>(v), cr[u], acc[u]);
            }
#pragma unroll
            for (int u = 0; u < CT; ++u) q[u] = j == 0 ? acc[u] : q[u] + acc[u];
        }
#pragma unroll
        for (int u = 0; u < CT; ++u) red[w][u][lane] = q[u];
        __syncthreads();
        bool finite = true;
        for (int o = tid; o < kWave * CT; o += kTrailThreads) {
            const int rl = o & (kWave - 1), u = o / kWave;
            const int row = static_cast<int>(blockIdx.x) * kWave + rl;
            if (row >= t.n) continue;
            double sum = red[0][u][rl];
#pragma unroll
            for (int v = 1; v < kTrailWaves; ++v) sum += red[v][u][rl];
            z[static_cast<size_t>(t.first + row) * kp + c0 + u] = static_cast<TO>(sum);
            finite = finite && trail_finite(sum);
        }
        return finite;
    };
    int tid = static_cast<int>(threadIdx.x);
    __shared__ int again;
    if (tid == 0) again = 0;   // (a barrier of the product follows)
    if (!product(std::false_type{}, tid)) again = 1;
    __syncthreads();
    if (again) {
        asm volatile("" : "+v"(tid));   // nothing of the first pass is kept for this one
        (void)product(std::true_type{}, tid);
    }
}

// ---- setup: S = T_^-T W T_^-1 in fp64 --------------------------------------------

// T_ (block rows and columns of L, diagonal included) into the zeroed dense
// np x np array a, one wave per row; rows past n get a unit diagonal.
template <bool F16>
__global__ __launch_bounds__(kBlock) void trail_scatter(sweep_desc d, int first, int n, int np, double* a) {
    const int i = static_cast<int>(blockIdx.x) * kWavesPerBlock + static_cast<int>(threadIdx.x) / kWave;
    if (i >= np) return;
    const int lane = threadIdx.x & (kWave - 1);
    double* row = a + static_cast<size_t>(i) * np;
    if (i >= n) {
        if (lane == 0) row[i] = 1.0;
        return;
    }
    const unsigned b = d.ptr[first + i], e = d.ptr[first + i + 1];
    for (unsigned p = b + lane; p < e; p += kWave) {
        int j;
        float v;
        load_entry<F16>(d, p, j, v);
        if (j >= first) row[j - first] = static_cast<double>(v);
    }
    if (lane == 0) row[i] = static_cast<double>(d.diag[first + i]);
}

__global__ __launch_bounds__(kBlock) void trail_zero(double* a, size_t count) {
    for (size_t q = blockIdx.x * static_cast<size_t>(kBlock) + threadIdx.x; q < count;
         q += static_cast<size_t>(gridDim.x) * kBlock)
        a[q] = 0.0;
}

// Inverses of the 64 x 64 diagonal blocks of a into x: thread j solves for
// column j by forward substitution, the block and the columns in LDS.
__global__ __launch_bounds__(kWave) void trail_invert_diag(int np, const double* __restrict__ a, double* x) {
    __shared__ double t[kWave][kWave];
    const int j = static_cast<int>(threadIdx.x);
    const size_t o = static_cast<size_t>(blockIdx.x) * kWave * (static_cast<size_t>(np) + 1);
    for (int i = 0; i < kWave; ++i) t[i][j] = a[o + static_cast<size_t>(i) * np + j];
    __syncthreads();
    double v[kWave];
#pragma unroll
    for (int i = 0; i < kWave; ++i) {
        double s = i == j ? 1.0 : 0.0;
#pragma unroll
        for (int k = 0; k < i; ++k) s = fma(-t[i][k], v[k], s);
        v[i] = i < j ? 0.0 : s / t[i][i];
    }
#pragma unroll
    for (int i = 0; i < kWave; ++i) x[o + static_cast<size_t>(i) * np + j] = v[i];
}

// One 64 x 64 tile of a product over k in [k0, k1) (multiples of 16) on the
// fp64 matrix cores: four waves, each a 32 x 32 quadrant of 2 x 2
// v_mfma_f64_16x16x4 tiles, operands staged 16 deep in LDS. A is element
// (i, k) at a[i * ai + k * ak], B element (k, j) at b[k * bk + j * bj]; the
// loads run along whichever of the two strides is 1. With w, row k < wn of B
// is scaled by w[k]^2.
typedef double f64x4 __attribute__((ext_vector_type(4)));
struct trail_tile {
    f64x4 acc[2][2];
};
inline constexpr int kTrailPad = 66;
__device__ __forceinline__ void trail_gemm_tile(const double* __restrict__ a, size_t ai, size_t ak,
                                                const double* __restrict__ b, size_t bk, size_t bj, int k0, int k1,
                                                const float* __restrict__ w, int wn, double (*la)[kTrailPad],
                                                double (*lb)[kTrailPad], trail_tile& t) {
    const int tid = static_cast<int>(threadIdx.x), lane = tid & (kWave - 1), wv = tid / kWave;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) t.acc[x][y] = f64x4{0.0, 0.0, 0.0, 0.0};
    // This thread's four elements of each operand's 64 x 16 slab: its row (or
    // column) and depth, by the unit stride.
    const bool a_k = ak == 1, b_k = bk == 1;
    int pi[4], pk[4], qj[4], qk[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int e = tid + u * kBlock;
        pi[u] = a_k ? e / 16 : e % 64;
        pk[u] = a_k ? e % 16 : e / 64;
        qj[u] = b_k ? e / 16 : e % 64;
        qk[u] = b_k ? e % 16 : e / 64;
    }
    double ra[4], rb[4];
    const auto fetch = [&](int k) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            ra[u] = a[pi[u] * ai + static_cast<size_t>(k + pk[u]) * ak];
            rb[u] = b[static_cast<size_t>(k + qk[u]) * bk + qj[u] * bj];
            if (w && k + qk[u] < wn) {
                const double s = static_cast<double>(w[k + qk[u]]);
                rb[u] *= s * s;
            }
        }
    };
    if (k0 < k1) fetch(k0);
    for (int k = k0; k < k1; k += 16) {
        __syncthreads();
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            la[pk[u]][pi[u]] = ra[u];
            lb[qk[u]][qj[u]] = rb[u];
        }
        __syncthreads();
        if (k + 16 < k1) fetch(k + 16);
        const int i0 = (wv >> 1) * 32 + (lane & 15), j0 = (wv & 1) * 32 + (lane & 15), kq = lane >> 4;
#pragma unroll
        for (int s = 0; s < 16; s += 4) {
            const double a0 = la[s + kq][i0], a1 = la[s + kq][i0 + 16];
            const double b0 = lb[s + kq][j0], b1 = lb[s + kq][j0 + 16];
            t.acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, t.acc[0][0], 0, 0, 0);
            t.acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, t.acc[0][1], 0, 0, 0);
            t.acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, t.acc[1][0], 0, 0, 0);
            t.acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, t.acc[1][1], 0, 0, 0);
        }
    }
}
// Visits this thread's 16 elements (row, column) of the tile: register v of
// a 16 x 16 tile holds row 4 v + lane / 16, column lane mod 16.
template <class F>
__device__ __forceinline__ void trail_tile_each(const trail_tile& t, F&& f) {
    const int lane = threadIdx.x & (kWave - 1), wv = static_cast<int>(threadIdx.x) / kWave;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                f((wv >> 1) * 32 + x * 16 + 4 * v + (lane >> 4), (wv & 1) * 32 + y * 16 + (lane & 15), t.acc[x][y][v]);
}

// The doubling step of the inverse: with the diagonal blocks of width s
// inverted in x, the block [2 p s + s, ..) x [2 p s, 2 p s + s) of the inverse
// is -X22 (T21 X11). Stage 0 forms T21 X11 and leaves it, transposed, in the
// unused upper triangle of a; stage 1 multiplies by -X22 into x. Grid: (column
// tiles s / 64, row tiles s / 64, pairs).
__global__ __launch_bounds__(kBlock) void trail_invert_step(int np, int s, int stage, double* a, double* x) {
    __shared__ double la[16][kTrailPad], lb[16][kTrailPad];
    const int a0 = static_cast<int>(blockIdx.z) * 2 * s, b0 = a0 + s;
    const int rows = min(s, np - b0);
    const int i0 = static_cast<int>(blockIdx.y) * kWave, j0 = static_cast<int>(blockIdx.x) * kWave;
    if (i0 >= rows) return;
    const size_t ld = static_cast<size_t>(np);
    trail_tile t;
    if (stage == 0) {
        // X11 is lower triangular: k from the column tile on.
        trail_gemm_tile(a + (b0 + i0) * ld + a0, ld, 1, x + a0 * ld + a0 + j0, ld, 1, j0, s, nullptr, 0, la, lb, t);
        trail_tile_each(t, [&](int i, int j, double v) { a[(a0 + j0 + j) * ld + b0 + i0 + i] = v; });
    } else {
        // X22 is lower triangular: k up to the row tile.
        trail_gemm_tile(x + (b0 + i0) * ld + b0, ld, 1, a + (a0 + j0) * ld + b0, 1, ld, 0, i0 + kWave, nullptr, 0, la, lb,
                        t);
        trail_tile_each(t, [&](int i, int j, double v) { x[(b0 + i0 + i) * ld + a0 + j0 + j] = -v; });
    }
}

// S = X^T W X, the lower tiles and their mirror image, in the sweeps' vector
// precision, with zeros in the padding (rows and columns past n), and S's
// diagonal as formed; raises bad on an entry that is not finite. Grid:
// (np / 64, np / 64).
template <class TO>
__global__ __launch_bounds__(kBlock) void trail_form(int n, int np, const double* __restrict__ x,
                                                     const float* __restrict__ w, TO* s, int ld, double* diag,
                                                     int* bad) {
    __shared__ double la[16][kTrailPad], lb[16][kTrailPad];
    const int i0 = static_cast<int>(blockIdx.y) * kWave, j0 = static_cast<int>(blockIdx.x) * kWave;
    if (j0 > i0) return;
    const size_t lx = static_cast<size_t>(np);
    trail_tile t;
    trail_gemm_tile(x + i0, 1, lx, x + j0, lx, 1, i0, np, w, n, la, lb, t);
    trail_tile_each(t, [&](int i, int j, double v) {
        const int r = i0 + i, c = j0 + j;
        if (c > r) return;   // the mirror of an element below the diagonal
        if (c == r && r < n) diag[r] = v;
        const TO o = (r < n && c < n) ? static_cast<TO>(v) : static_cast<TO>(0);
        if (!(fabs(static_cast<double>(o)) <= 1.0e300) || (sizeof(TO) == 4 && !(fabsf(static_cast<float>(o)) <= 3.0e38f)))
            atomicOr(bad, 1);
        s[static_cast<size_t>(r) * ld + c] = o;
        s[static_cast<size_t>(c) * ld + r] = o;
    });
}

}  // namespace apxchol_amd
