// Node tiles of the matrix-free tile kernels (tile.h): compact groups of at most kTileRows nodes
// found on the host by recursive bisection of the node cloud, and the per-tile lists the kernels
// read, built on the device from the fan entries.
#include <algorithm>
#include <cmath>
#include <limits>
#include <vector>

#include "rowops.h"

namespace cvfes {
namespace {

// Distinct columns of the block rows ids[0..n) that are not themselves among ids, counted row
// by row up to `most`: the halo columns of a tile of these rows.  (A node of no element has an empty
// row and is no column of it, so the halo is not the row's columns less n.)  `seen` [N] holds the
// last stamp a node was counted under.
int count_halo(const int32_t *ids, int n, const int32_t *indptr, const int32_t *indices, int most, int32_t *seen,
               int32_t stamp) {
    for (int i = 0; i < n; ++i) seen[ids[i]] = stamp;
    int m = 0;
    for (int i = 0; i < n && m <= most; ++i)
        for (int32_t p = indptr[ids[i]]; p < indptr[ids[i] + 1]; ++p) {
            if (seen[indices[p]] == stamp) continue;
            seen[indices[p]] = stamp;
            ++m;
        }
    return m;
}

// Halve the nodes across their longest extent, on a multiple of the tile size, until a part is a
// tile; a tile with too many halo columns is halved again.
int64_t bisect(const double *nodes, const int32_t *indptr, const int32_t *indices, int64_t n_nodes,
               int32_t *rows, int64_t cap) {
    std::vector<int32_t> ids(n_nodes);
    for (int64_t i = 0; i < n_nodes; ++i) ids[i] = static_cast<int32_t>(i);
    // Extents are counted in edges: on a wall whose mesh is finer along one axis than along the
    // others, parts of equal sides would be long strips of nodes with too many columns.
    double edge[3] = {0.0, 0.0, 0.0};
    for (int64_t i = 0; i < n_nodes; ++i)
        for (int32_t p = indptr[i]; p < indptr[i + 1]; ++p)
            for (int k = 0; k < 3; ++k) {
                const double d = std::abs(nodes[3 * static_cast<int64_t>(indices[p]) + k] - nodes[3 * i + k]);
                if (d < std::numeric_limits<double>::infinity()) edge[k] += d;
            }
    for (double &d : edge) d = d > 0.0 ? 1.0 / d : 0.0;
    std::vector<int32_t> seen(n_nodes, 0);
    int32_t stamp = 0;                     // fewer than 2 N parts are counted, N < 2^30
    std::vector<std::pair<double, int32_t>> keys(n_nodes);
    std::vector<std::pair<int64_t, int64_t>> todo{{0, n_nodes}};
    int64_t n_tiles = 0;
    while (!todo.empty()) {
        const auto [a, b] = todo.back();
        todo.pop_back();
        const int64_t n = b - a;
        const int halo = kTileCols - kTileRows;
        if (n == 1 || (n <= kTileRows &&
                       count_halo(&ids[a], static_cast<int>(n), indptr, indices, halo, seen.data(), ++stamp) <= halo)) {
            if (n_tiles == cap) return -1;
            std::sort(ids.begin() + a, ids.begin() + b);
            for (int i = 0; i < kTileRows; ++i) rows[n_tiles * kTileRows + i] = i < n ? ids[a + i] : -1;
            ++n_tiles;
            continue;
        }
        double lo[3], hi[3];
        for (int k = 0; k < 3; ++k) {
            lo[k] = std::numeric_limits<double>::infinity();
            hi[k] = -lo[k];
            for (int64_t i = a; i < b; ++i) {
                const double x = nodes[3 * static_cast<int64_t>(ids[i]) + k];
                if (x < lo[k]) lo[k] = x;
                if (x > hi[k]) hi[k] = x;
            }
        }
        int ax = 0;
        for (int k = 1; k < 3; ++k)
            if (edge[k] * (hi[k] - lo[k]) > edge[ax] * (hi[ax] - lo[ax])) ax = k;
        const int64_t whole = (n + kTileRows - 1) / kTileRows;
        const int64_t h = n > kTileRows ? whole / 2 * kTileRows : n / 2;
        for (int64_t i = a; i < b; ++i) {
            const double x = nodes[3 * static_cast<int64_t>(ids[i]) + ax];
            // NaN last: a strict order for any input
            keys[i] = {x == x ? x : std::numeric_limits<double>::infinity(), ids[i]};
        }
        std::nth_element(keys.begin() + a, keys.begin() + a + h, keys.begin() + b);
        for (int64_t i = a; i < b; ++i) ids[i] = keys[i].second;
        todo.push_back({a + h, b});
        todo.push_back({a, a + h});
    }
    return n_tiles;
}

// Last column slot of a tile whose rows name more columns or elements than the slots hold.
constexpr int32_t kTileOver = -2;

// One wavefront per tile: lane c holds the node of column slot c (rows first, then the halo in the
// order the entries name it); every node of the entries is looked up with a ballot.
__global__ __launch_bounds__(kBlock) void k_tile_lists(int64_t n_tiles, const int32_t *__restrict__ rows,
                                                       const int32_t *__restrict__ nptr,
                                                       const fan_t *__restrict__ fan, int4 *__restrict__ head,
                                                       int32_t *__restrict__ cols, int2 *__restrict__ ents) {
    const int64_t t = (static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x) >> 6;
    const int lane = threadIdx.x & 63;
    if (t >= n_tiles) return;
    const int32_t mine = lane < kTileRows ? rows[t * kTileRows + lane] : -1;
    int32_t held = mine;
    int m = kTileRows;
    bool over = false;
    for (int i = 0; i < kTileRows; ++i) {
        const int32_t a = __shfl(mine, i);
        const int32_t q0 = a >= 0 ? nptr[a] : 0;
        const int32_t ne = a >= 0 ? min(nptr[a + 1] - q0, kTileElems) : 0;
        over |= a >= 0 && nptr[a + 1] - q0 > kTileElems;
        // The row's contributions lie block by block, the ne of its own block (a,a) next to each other
        // from d0 on.  The kernels stage them in aligned pairs of values without those: as they lie up
        // to `cut`, then from `skip` further on, both even, so up to two values of (a,a) stay.
        int d0 = 3 * kTileElems;
        for (int k = 0; k < ne; ++k) d0 = min(d0, fan[q0 + k].w & 1023);
        const int cut = ne ? (9 * d0 + 1) & ~1 : 0;
        const int skip = ne ? (9 * (d0 + ne) & ~1) - cut : 0;
        const auto at = [&](int pos) { return 9 * pos - (pos > d0 ? skip : 0); };
        if (lane == 0) head[t * kTileRows + i] = make_int4(a, q0, ne, cut | skip << 16);
        int before = 0;
        for (int k = 0; k < ne; ++k) {
            const fan_t e = fan[q0 + k];
            int slot[2] = {before, 0};
            for (int s = e.x >= 0 ? 0 : 1; s < 2; ++s) {
                const int32_t node = s == 0 ? e.x : e.y;
                const unsigned long long hit = __ballot(held == node);
                slot[s] = hit ? __ffsll(static_cast<long long>(hit)) - 1 : min(m++, kTileCols - 1);
                if (lane == slot[s]) held = node;
            }
            before = slot[1];
            if (lane == 0)
                ents[(t * kTileRows + i) * kTileElems + k] = make_int2(
                    e.z, static_cast<int32_t>(slot[0] | slot[1] << 8 | at((e.w >> 10) & 1023) << 16 |
                                              static_cast<uint32_t>(at((e.w >> 20) & 1023)) << 24));
        }
        if (lane >= ne && lane < kTileElems) ents[(t * kTileRows + i) * kTileElems + lane] = make_int2(0, 0);
    }
    over |= m > kTileCols;
    if (lane >= kTileRows && lane < kTileCols)
        cols[t * (kTileCols - kTileRows) + lane - kTileRows] = over && lane == kTileCols - 1 ? kTileOver : held;
}

}  // namespace
}  // namespace cvfes

using namespace cvfes;

extern "C" int64_t cvfes_tile_rows(int64_t n_nodes, const double *nodes, const int32_t *indptr,
                                   const int32_t *indices, int32_t *rows, int64_t cap) {
    CVFES_REQUIRE(n_nodes >= 0 && n_nodes < (int64_t(1) << 31), "cvfes_tile_rows: bad sizes");
    if (n_nodes == 0) return 0;
    CVFES_REQUIRE(nodes && indptr && indices && rows, "cvfes_tile_rows: null pointer");
    int64_t n = -1;
    try {
        n = bisect(nodes, indptr, indices, n_nodes, rows, cap);
    } catch (...) {
        return fail(CVFES_ERR_ARG, "cvfes_tile_rows: out of host memory");
    }
    CVFES_REQUIRE(n >= 0, "cvfes_tile_rows: more than %lld tiles", static_cast<long long>(cap));
    return n;
}

extern "C" int cvfes_tile_lists(void *stream, int64_t n_tiles, const int32_t *rows, const int32_t *nptr,
                                const int32_t *fan, int64_t max_node_elems, int32_t *head, int32_t *cols,
                                int32_t *ents) {
    CVFES_REQUIRE(n_tiles >= 0 && n_tiles < (int64_t(1) << 30), "cvfes_tile_lists: bad sizes");
    if (n_tiles == 0) return CVFES_OK;
    CVFES_REQUIRE(max_node_elems >= 1 && max_node_elems <= kTileElems,
                  "cvfes_tile_lists: max_node_elems must be 1..%d", kTileElems);
    CVFES_REQUIRE(rows && nptr && fan && head && cols && ents, "cvfes_tile_lists: null pointer");
    const int64_t blocks = (n_tiles + kBlock / 64 - 1) / (kBlock / 64);
    hipLaunchKernelGGL(k_tile_lists, dim3(static_cast<unsigned>(blocks)), dim3(kBlock), 0,
                       static_cast<hipStream_t>(stream), n_tiles, rows, nptr,
                       reinterpret_cast<const fan_t *>(fan), reinterpret_cast<int4 *>(head), cols,
                       reinterpret_cast<int2 *>(ents));
    if (int rc = check_launch("k_tile_lists")) return rc;
    // a tile that does not fit is refused here: its rows would read another node's column
    const int64_t halo = kTileCols - kTileRows;
    std::vector<int32_t> held;
    try {
        held.resize(n_tiles * halo);
    } catch (...) {
        return fail(CVFES_ERR_ARG, "cvfes_tile_lists: out of host memory");
    }
    hipError_t err = hipMemcpyAsync(held.data(), cols, sizeof(int32_t) * held.size(), hipMemcpyDeviceToHost,
                                    static_cast<hipStream_t>(stream));
    if (err == hipSuccess) err = hipStreamSynchronize(static_cast<hipStream_t>(stream));
    if (err != hipSuccess) return fail(CVFES_ERR_HIP, "cvfes_tile_lists: %s", hipGetErrorString(err));
    for (int64_t t = 0; t < n_tiles; ++t)
        CVFES_REQUIRE(held[(t + 1) * halo - 1] != kTileOver,
                      "cvfes_tile_lists: the rows of tile %lld name more than %lld halo columns or a node of more than "
                      "%d elements",
                      static_cast<long long>(t), static_cast<long long>(halo), kTileElems);
    return CVFES_OK;
}
