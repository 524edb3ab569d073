// Level tiles: J consecutive launched levels in one launch. What bounds a
// launched level is its chain of latencies -- the launch, the layout loads, the
// gather, the store (4.1 us for 1 to ~1000 batches, of which the arithmetic is
// a tenth) -- so levels are joined without any wait between workgroups: a tile
// recomputes every row of its levels that its last rows reach (tile_step; the
// host chooses which levels are joined, host/tile.cpp), and passes its outputs
// on in LDS. All layout loads of all J levels, then all gathers from before
// the first, are in flight together; a further level is a barrier, an LDS
// gather and the row sums. The per-row arithmetic is sweep_lanes' (same lane
// groups, fma chain and butterfly), so the bits are those of the levels'
// own launches, also where two tiles compute a row. Tiles of 4 waves where the
// shared rows allow it: with 16 a compute unit's gathers, a line a cycle, are
// the longest part (four levels of a 256^2 grid: 8.9 us, with 4 waves 6.7, as
// launches of their own 4 x 3.9).
// Solves without and with tiles: 256^2 fp64 7,180 / 6,060 us, 128^3 SDDM mixed
// 28,600 / 25,500 (148 / 86 launched levels an iteration), R-MAT scale 18 mixed
// 7,180 / 6,480 (60 / 43).
namespace apxchol_amd {

inline constexpr int kTileBlock = kTileWaves * kWave;

template <class TI, class TO, int J>
__device__ __forceinline__ void sweep_tile_body(int tile, unsigned char* tile_lds, const sweep_desc& d,
                                                const tile_step& t, const lane_rec* __restrict__ rec,
                                                const entry32* __restrict__ ent, const TI* __restrict__ rhs, TO* out,
                                                const pcg_state* st) {
    const int w = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
    const int lane = threadIdx.x & (kWave - 1);
    TO* lds = reinterpret_cast<TO*>(tile_lds);
    lane_rec rc[J];
    entry32 e[J][kEpl];
#pragma unroll
    for (int p = 0; p < J; ++p) {
        rc[p] = {-1, 0};
        if (w < t.width[p]) {
            const size_t b = static_cast<size_t>(t.base[p]) + static_cast<size_t>(tile) * t.width[p] + w;
            rc[p] = rec[b * kWave + lane];
#pragma unroll
            for (int k = 0; k < kEpl; ++k) e[p][k] = ent[(b * kEpl + k) * kWave + lane];
        } else {
#pragma unroll
            for (int k = 0; k < kEpl; ++k) e[p][k] = {0, 0.0f};
        }
    }
    asm volatile("" ::: "memory");
    if (st && st->done) return;
    const double shift = (st && !d.backward) ? st->shift : 0.0;
    TO xv[J][kEpl], r[J];
    float dg[J];
#pragma unroll
    for (int p = 0; p < J; ++p) {
        const int nv = static_cast<int>((rc[p].info >> 9) & 7u);
#pragma unroll
        for (int k = 0; k < kEpl; ++k)
            xv[p][k] = k < nv && e[p][k].idx >= 0 ? out[e[p][k].idx] : static_cast<TO>(0);
        r[p] = 0;
        dg[p] = 1.0f;
        if (rc[p].row >= 0 && ((rc[p].info >> 3) & 63u) == 0) {
            r[p] = row_rhs<TI, TO>(d, rhs, rc[p].row, shift);
            dg[p] = diag_operand<TO>(d, rc[p].row);
        }
    }
#pragma unroll
    for (int p = 0; p < J; ++p) {
        if (p > 0) {
            lds_barrier();
            const int nv = static_cast<int>((rc[p].info >> 9) & 7u);
#pragma unroll
            for (int k = 0; k < kEpl; ++k)
                if (k < nv && e[p][k].idx < 0) xv[p][k] = lds[~e[p][k].idx];
        }
        if (w < t.width[p]) {
            TO part = 0;
#pragma unroll
            for (int k = 0; k < kEpl; ++k) part = fma(static_cast<TO>(e[p][k].val), xv[p][k], part);
            part = group_tree_sum(part, 1 << (rc[p].info & 7u));
            if (rc[p].row >= 0 && ((rc[p].info >> 3) & 63u) == 0) {
                const TO v = finish_row<TO>(r[p] - part, dg[p]);
                if (p + 1 < J) lds[(rc[p].info >> kTileSlotShift) & 0xffffu] = v;
                if (rc[p].info & kTileOwn) out[rc[p].row] = v;
            }
        }
    }
}
template <class TI, class TO, int J>
__global__ __launch_bounds__(kTileBlock) void sweep_tiles(sweep_desc d, tile_step t, const lane_rec* __restrict__ rec,
                                                          const entry32* __restrict__ ent,
                                                          const TI* __restrict__ rhs, TO* out, const pcg_state* st) {
    extern __shared__ unsigned char tile_lds[];
    sweep_tile_body<TI, TO, J>(static_cast<int>(blockIdx.x), tile_lds, d, t, rec, ent, rhs, out, st);
}

}  // namespace apxchol_amd
