// Matrix-free row products by node tiles.
//
// A workgroup takes one tile (at most kTileRows compact nodes, cvfes_tile_rows) and one chunk of
// the samples.  Groups of `lanes` consecutive lanes own one row each, VW samples per lane.
//   1. Every group loads its row's own state, up to two halo columns, its elements' coefficients
//      and its unit blocks, all at once; the columns x and the unit blocks go to LDS.
//   2. After one barrier each group walks its row's fan entries (the operations of fan_product, in
//      the same order: the results are equal bit for bit) with x and the unit blocks from LDS.
// Two things bounded the row kernels.  Their unit blocks come through the scalar cache, where every
// 64-byte line of them is a miss (each is read once) and a cache, one per two CUs, takes a new line
// only every 38 ns or so: 0.28 TB/s for the chip, 0.48 ms for the 132 MB of 102,400 nodes.  And they
// gather every column from L1/L2 for each of its about 7 rows, 77 KB per row and 128 samples, which
// keeps the L1 path 73 % busy.  A tile of 16 rows has about 35 columns, so a row costs 2.2 column
// loads instead of 8, and one wait for memory instead of one per element; the unit blocks are
// coalesced loads.  The step at 102,400 nodes: 505 -> 328 us with 128 samples, 99 -> 41 us with 32 on
// 49,152 nodes, 52 -> 26 us with 1.  What bounds it now is memory traffic (1.51 GB with the columns
// that neighbouring tiles share) and the wait for it at the start of a workgroup: two of 512 threads
// and 74 KB fit a CU (128 registers, 16 rows x 64 samples), two thirds of whose cycles are waits.  Tiles of 8 rows (three workgroups) and
// chunks of 32 samples measured 4 % and 45 % slower.
#pragma once

#include "rowops.h"

namespace cvfes {

typedef int32_t word4_t __attribute__((ext_vector_type(4)));

constexpr int kTileThreads = 32 * kTileRows;      // half a wavefront per row at most

struct TileArgs {
    const CVFES_G word4_t *head;    // [T][kTileRows] node (-1: none), first fan entry, fan entries, cut | skip << 16
    const CVFES_G int32_t *cols;    // [T][kTileCols - kTileRows] halo nodes (-1: none)
    const CVFES_G word4_t *ents;    // [T][kTileRows][kTileElems / 2] two entries each: element; slots
                                    // p, q and where its blocks (a,p), (a,q) start
    int32_t chunks;        // chunks of the samples
    int32_t chunk;         // samples per chunk (a multiple of the lane width)
    int32_t lanes;         // lanes per row, chunk / VW
    int32_t groups;        // rows per wavefront
    int32_t n_tiles;
};

// Shape of a tile launch over n_smp samples: as few chunks as fit half a wavefront at two samples
// per lane (odd counts: one sample per lane), of nearly equal size.
struct TileShape {
    int vw, chunk, chunks, lanes, groups, waves;
};

inline TileShape tile_shape(int64_t n_smp) {
    TileShape t;
    t.vw = n_smp % 2 == 0 ? 2 : 1;
    const int64_t l = n_smp / t.vw;
    t.chunks = static_cast<int>((l + 31) / 32);
    t.lanes = static_cast<int>((l + t.chunks - 1) / t.chunks);
    t.chunk = t.lanes * t.vw;
    t.groups = 64 / t.lanes < kTileRows ? 64 / t.lanes : kTileRows;
    t.waves = (kTileRows + t.groups - 1) / t.groups;
    return t;
}

// Unit block values staged per row: the blocks (a,p) and (a,q) of its elements, and up to two values
// of the skipped blocks (a,a) (k_tile_lists keeps the copies in aligned pairs).
__host__ __device__ constexpr int tile_kh(int elems) { return 18 * elems + 2; }

inline size_t tile_lds(int chunk, int elems) {
    return sizeof(double) * (static_cast<size_t>(kTileCols) * 3 * chunk +
                             static_cast<size_t>(kTileRows) * tile_kh(elems));
}

inline TileArgs tile_args(const cvfes_system_t *sys, const TileShape &h) {
    return TileArgs{(const CVFES_G word4_t *)sys->tile_head, (const CVFES_G int32_t *)sys->tile_cols,
                    (const CVFES_G word4_t *)sys->tile_ents, h.chunks, h.chunk, h.lanes, h.groups,
                    static_cast<int32_t>(sys->n_tiles)};
}

// Workgroups of a launch over the mesh (chunk by chunk of each tile), padded for xcd_block.
inline unsigned tile_grid(const TileArgs &t) {
    const int64_t blocks = static_cast<int64_t>(t.n_tiles) * t.chunks;
    return static_cast<unsigned>((blocks + kNumXcd - 1) / kNumXcd * kNumXcd);
}

// Up to this many samples a wavefront holds so many rows that each has few lanes to stage its unit
// blocks with; they are then staged by all lanes of the wavefront (SMALL), 14 rounds in flight
// (102,400 nodes: 1 sample 26 us, 5 samples 33, 8 samples 42; with all 27 values an element 37, 48
// and 52, against 55, 53 and 58 staged by the row's lanes).
constexpr int kTileSmall = 8;

// Whether a launch of `blocks` workgroups stays below 2^32 threads, with room for tile_grid's padding.
inline bool launch_fits(int64_t blocks, int threads) { return blocks + kNumXcd <= ((int64_t(1) << 32) - 1) / threads; }

// Whether the matrix-free kernels of this system run by tiles.  Tiles of a wall whose rows have many
// columns are half empty, so their launch can have more threads than that of the rows.
inline bool tiles_apply(const cvfes_system_t *sys) {
    const TileShape h = tile_shape(sys->n_smp);
    return sys->n_tiles > 0 && sys->tile_head && sys->tile_cols && sys->tile_ents && sys->max_node_elems >= 1 &&
           sys->max_node_elems <= kTileElems && launch_fits(sys->n_tiles * h.chunks, 64 * h.waves);
}

// `early()` issues what the caller needs for its row's update, while the last elements are applied.
// Nothing before the barrier branches on the mesh: absent halo nodes and the tail of the unit
// blocks repeat a valid one.
template <int ELEMS, int VW, bool SMALL, class RA, class COL, class EARLY>
__device__ __forceinline__ void tile_product(const RA &k, const TileArgs &t, const COL &col, int32_t tile,
                                             int i, int l, bool in, word4_t rw, double (&acc)[3][VW], EARLY early) {
    extern __shared__ double s_tile[];
    const int pitch = 3 * t.chunk;                      // doubles per column
    double *s_kh = s_tile + i * tile_kh(ELEMS);
    double *s_x = s_tile + kTileRows * tile_kh(ELEMS);
    int32_t ew[ELEMS];
    Vec<VW> cf[ELEMS];
    const int32_t node = rw.x >= 0 ? rw.x : 0;
    double xa[3][VW];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int v = 0; v < VW; ++v) acc[r][v] = 0.0;
    // Unit blocks, two values a round, kAhead rounds in flight at a time: by the lanes of the row (all
    // its rounds at once when the row has half a wavefront), or, with one or two samples, by the
    // wavefront's lanes shared out over its rows.
    constexpr int kAhead = SMALL ? 14 : (tile_kh(ELEMS) / 2 + 31) / 32;
    int si = i, l0 = 2 * l, ls = 2 * t.lanes;
    word4_t sw = rw;
    if constexpr (SMALL) {
        const int n = 64 / t.groups, lane = threadIdx.x & 63;
        si = static_cast<int>(threadIdx.x >> 6) * t.groups + lane / n;
        l0 = 2 * (lane % n);
        ls = 2 * n;
        // n lanes for each of `groups` rows: the last lanes and rows may have none
        sw = word4_t{-1, 0, 0, 0};
        if (lane / n < t.groups && si < kTileRows) sw = t.head[static_cast<int64_t>(tile) * kTileRows + si];
        else si = 0;
    }
    // values from `cut` on are those `skip` further on in the row's blocks (k_tile_lists)
    const int cut = sw.w & 0xffff, skip = sw.w >> 16;
    const int nk = 27 * sw.z - skip - 2;       // the last round's first value; negative: nothing to stage
    const auto *kh = k.khat + 27 * static_cast<int64_t>(sw.y);
    double *s_st = s_tile + si * tile_kh(ELEMS);
    double kv[kAhead][2];
    auto fetch = [&](int at) {
#pragma unroll
        for (int j = 0; j < kAhead; ++j) {
            const int to = min(at + j * ls, nk);
            const auto *p = kh + (to < cut ? to : to + skip);
            kv[j][0] = p[0];
            kv[j][1] = p[1];
        }
    };
    auto stage = [&](int at) {
#pragma unroll
        for (int j = 0; j < kAhead; ++j) {
            double *p = s_st + min(at + j * ls, nk);
            p[0] = kv[j][0];
            p[1] = kv[j][1];
        }
    };
    if (in) {
        const auto *hc = t.cols + static_cast<int64_t>(tile) * (kTileCols - kTileRows) + i;
        const bool two = i < kTileCols - 2 * kTileRows;
        int32_t n1 = hc[0], n2 = hc[two ? kTileRows : 0];
        const auto *e4 = t.ents + (static_cast<int64_t>(tile) * kTileRows + i) * (kTileElems / 2);
        word4_t en[ELEMS / 2];
#pragma unroll
        for (int e = 0; e < ELEMS / 2; ++e) en[e] = e4[e];
        n1 = n1 >= 0 ? n1 : node;
        n2 = n2 >= 0 ? n2 : node;
        auto put = [&](int slot, const typename COL::Raw &r, double (&x)[3][VW]) {
            col.column(r, x);
            double *d = s_x + slot * pitch + l * VW;
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                Vec<VW> o;
#pragma unroll
                for (int v = 0; v < VW; ++v) o.v[v] = x[j][v];
                store_vec<VW>(d + j * t.chunk, o);
            }
        };
        double y[3][VW];
        const typename COL::Raw r0 = col.load(node), r1 = col.load(n1);
        typename COL::Raw r2;
        if (two) r2 = col.load(n2);
        if constexpr (!SMALL) {
            if (nk >= 0) fetch(l0);
        }
        __builtin_amdgcn_sched_barrier(0);
        put(i, r0, xa);
        put(kTileRows + i, r1, y);
        if (two) put(2 * kTileRows + i, r2, y);
        if constexpr (!SMALL) {
            if (nk >= 0) stage(l0);
        }
        __builtin_amdgcn_sched_barrier(0);
        // in the registers of the columns; in flight across the barrier
#pragma unroll
        for (int e = 0; e < ELEMS; ++e) {
            const int32_t id = e % 2 ? en[e / 2].z : en[e / 2].x;
            ew[e] = e % 2 ? en[e / 2].w : en[e / 2].y;
            cf[e] = load_lane<VW>(k.coef + static_cast<int64_t>(id) * k.n_smp, col.lane);
        }
    }
    for (int at = SMALL ? l0 : l0 + kAhead * ls; at <= nk + 1; at += kAhead * ls) {
        fetch(at);
        stage(at);
    }
    __syncthreads();
    if (!in) return;
    double xp[3][VW], xq[3][VW];
    auto get = [&](int slot, double (&x)[3][VW]) {
        const double *d = s_x + slot * pitch + l * VW;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const Vec<VW> r = load_vec<VW>(d + j * t.chunk);
#pragma unroll
            for (int v = 0; v < VW; ++v) x[j][v] = minus(r.v[v], xa[j][v]);
        }
    };
    // element e with its p column (less the row's own) in x0; its q column goes to x1
    auto apply = [&](int e, int before, double (&x0)[3][VW], double (&x1)[3][VW]) {
        const int w = ew[e];
        if ((w & 255) != before) get(w & 255, x0);
        get((w >> 8) & 255, x1);
        const double *kp = s_kh + ((w >> 16) & 255), *kq = s_kh + (static_cast<uint32_t>(w) >> 24);
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
            for (int v = 0; v < VW; ++v) {
                double y = kp[3 * r] * x0[0][v];
#pragma unroll
                for (int j = 1; j < 3; ++j) y = fma(kp[3 * r + j], x0[j][v], y);
#pragma unroll
                for (int j = 0; j < 3; ++j) y = fma(kq[3 * r + j], x1[j][v], y);
                acc[r][v] = fma(cf[e].v[v], y, acc[r][v]);
            }
    };
#pragma unroll
    for (int e = 0; e < ELEMS; e += 2) {
        if (e == ELEMS - 2) early(node);        // in the registers of the coefficients done with
        if (e < rw.z) apply(e, e ? (ew[e - 1] >> 8) & 255 : -1, xp, xq);
        if (e + 1 < rw.z) apply(e + 1, (ew[e] >> 8) & 255, xq, xp);
    }
}

// The lane's place in a tile launch: its tile, row slot i, lane l in the row and first sample s
// (clamped to the last lane's), whether it has a row slot, and whether it stores.
struct TilePlace {
    int64_t s;
    int32_t tile;
    int i, l;
    bool in, active;
    word4_t rw;
};

// Place in workgroup `b` (tile-major, chunk by chunk) of the mesh's launch.
template <int VW>
__device__ __forceinline__ bool tile_place(const TileArgs &t, int64_t n_smp, uint32_t b, TilePlace &p) {
    p.tile = static_cast<int32_t>(b / static_cast<uint32_t>(t.chunks));
    if (p.tile >= t.n_tiles) return false;
    const int32_t ch = static_cast<int32_t>(b) - p.tile * t.chunks;
    const int lane = threadIdx.x & 63, g = lane / t.lanes;
    p.l = lane - g * t.lanes;
    p.i = static_cast<int>(threadIdx.x >> 6) * t.groups + g;
    p.in = g < t.groups && p.i < kTileRows;
    p.rw = p.in ? t.head[static_cast<int64_t>(p.tile) * kTileRows + p.i] : word4_t{-1, 0, 0, 0};
    p.s = static_cast<int64_t>(ch) * t.chunk + p.l * VW;
    p.active = p.in && p.rw.x >= 0 && p.s < n_smp;
    if (p.s >= n_smp) p.s = n_smp - VW;
    return true;
}

// One forward step of the workgroup's rows; SA: StepArgs, or GStepArgs of a batched mesh.
template <bool BETA, bool DAMP, int VW, int ELEMS, bool SMALL, class SA>
__device__ __forceinline__ void tile_step(const SA &a, const TileArgs &t, uint32_t b, int64_t step) {
    TilePlace p;
    if (!tile_place<VW>(t, a.k.n_smp, b, p)) return;
    typedef StateCol<false, BETA, VW, decltype(a.u)> Col;
    const Col col{a.u, a.up, a.bdt, a.k.n_smp, static_cast<uint32_t>(p.s) * 8u};
    double acc[3][VW];
    typename Col::Own own;
    tile_product<ELEMS, VW, SMALL>(a.k, t, col, p.tile, p.i, p.l, p.in, p.rw, acc,
                            [&](int32_t node) { own = col.own(node); });
    if (p.active)
        step_update<DAMP, VW>(a, p.rw.x, p.s, true, step, row_load<VW>(a, p.rw.x, p.s), acc, own.u, own.up);
}

}  // namespace cvfes
