// Row operations shared by the single-mesh and the batched step kernels: the gathered block-row
// product (stored blocks, or element unit blocks scaled by the element coefficients) and the fused
// central-difference update of one block row.
#pragma once

#include "common.h"

namespace cvfes {

// Lanes per block row.  Packed (UNIFORM = false): S/VW lanes, so a wave may span several rows.
// Wave-uniform (UNIFORM = true): S/VW rounded up to whole wavefronts; lanes past the last sample
// are inactive (they read the last sample group and do not store), which keeps every row on
// whole wavefronts for any S.
template <bool UNIFORM, int VW>
__host__ __device__ __forceinline__ int64_t lanes_per_row(int64_t n_smp) {
    const int64_t l = n_smp / VW;
    return UNIFORM ? (l + 63) / 64 * 64 : l;
}

template <bool UNIFORM, int VW>
__device__ __forceinline__ bool row_and_sample(int64_t n_nodes, int64_t n_smp, int32_t &row,
                                               int64_t &s, bool &active) {
    // a launch has fewer than 2^32 threads, so the division is one of 32 bits (of 64 it took some
    // hundred instructions of each short kernel)
    const uint32_t lpr = static_cast<uint32_t>(lanes_per_row<UNIFORM, VW>(n_smp));
    const uint32_t g = static_cast<uint32_t>(xcd_block() * kBlock + threadIdx.x);
    uint32_t r = g / lpr;
    s = static_cast<int64_t>(g - r * lpr) * VW;
    active = s < n_smp;
    if (!active) s = n_smp - VW;
    if constexpr (UNIFORM) r = __builtin_amdgcn_readfirstlane(static_cast<int32_t>(r));
    row = static_cast<int32_t>(r);
    return r < n_nodes;
}

// Wave-uniform rows pay off when they keep at least 3/4 of the lanes busy.
template <int VW>
inline bool use_uniform(int64_t n_smp) {
    const int64_t l = n_smp / VW, padded = (l + 63) / 64 * 64;
    return 4 * l >= 3 * padded;
}

// Samples per lane of the generic row kernels (step, product, adjoint, fused): two for even
// counts, except where only one keeps the rows wave-uniform (64 samples: 32 two-sample lanes
// would put two rows in a wave, and the element blocks would come in per lane instead of through
// scalar loads).  The per-sample arithmetic is the same either way.
inline int generic_vw(int64_t n_smp) {
    if (n_smp % 2 != 0) return 1;
    return (!use_uniform<2>(n_smp) && use_uniform<1>(n_smp)) ? 1 : 2;
}

// Operator forms of the row functions (template argument OP): stored values in full storage,
// matrix-free (element coefficients x unit element blocks), stored values in symmetric storage.
// kOpFan is the matrix-free operator walked element by element around the row node
// (cvfes_system_t.fan); kOpMatfree walks it block by block (systems without fan entries).
constexpr int kOpStored = 0;
constexpr int kOpMatfree = 1;
constexpr int kOpSym = 2;
constexpr int kOpFan = 3;

// One fan entry: the element e incident to the row node, its two other nodes p and q, and the
// positions of its blocks (row, row), (row, p), (row, q) among the row's contributions, 10 bits
// each (`pk`).  p is -1 where it is the previous entry's q.
typedef int32_t fan_t __attribute__((ext_vector_type(4)));

// Stored operator: full storage `values` [nnzb][9][S], or, when `values` is null, symmetric
// storage: the upper blocks `uvalues` [nnzu][9][S], block p of the row structure being
// uvalues[vblk[p]], read transposed when its column precedes its row.
struct RowArgs {
    int64_t n_nodes;
    int64_t n_smp;
    const int32_t *indptr;
    const int32_t *indices;
    const double *values;
    const int32_t *cptr;
    const int32_t *celem;
    const double *khat;
    const double *coef;
    const double *uvalues;
    const int32_t *vblk;
    const int32_t *nptr;
    const fan_t *fan;      // null: the matrix-free operator is walked block by block
};

// The fan entries a kernel may use: the byte offsets inside a node's samples are 31 bits.
inline const fan_t *fan_entries(const cvfes_system_t *sys) {
    return sys->nptr && sys->n_smp < (int64_t(1) << 31) / 24 ? reinterpret_cast<const fan_t *>(sys->fan) : nullptr;
}

constexpr int kRecordSlots = 7;

// Whether the kernels that read a row's structure from its record (seven block slots) take the symmetric
// storage; the others walk indptr, indices and vblk.  Byte offsets inside a block are 32-bit: 72 S.
// Records of ten slots, those of irregular walls, serve k_step_sym alone: slots behind a row's last
// block repeat it, a third more loads than the rows' seven or so blocks need (16,384 rows of 4 to 8
// elements, walk / records: 64 samples 80 / 93 us a step, 8 12.0 / 13.5; 102,400 rows, 2 samples: product
// 32 / 45 us, 33 287 / 331; few gained, 16,384 rows, 40 samples: 55 / 49).  Adjoint: the adjoint step with
// one sample per lane loses by records in wave-uniform rows (16,384 nodes of a regular wall, 48 samples:
// 66 / 76 us), and with one sample on large walls (102,400 nodes: 20.2 / 22.2; 16,384: 9.2 / 7.9).
inline bool use_records(const cvfes_system_t *sys, bool adjoint = false) {
    const int64_t S = sys->n_smp;
    if (!sys->row_records || !sys->uvalues || 72 * S > INT32_MAX || sys->record_width != 2 + 2 * kRecordSlots ||
        sys->max_row_blocks < 1 || sys->max_row_blocks > kRecordSlots)
        return false;
    if (!adjoint) return true;
    return S == 1 ? sys->n_nodes < (1 << 16) : generic_vw(S) == 2 || !use_uniform<1>(S);
}

// Node tiles (tile.h): rows per tile, column slots (39 of 64 samples and the unit blocks of 16
// rows of 6 elements fit half a CU's LDS), and most elements around a node.
constexpr int kTileRows = CVFES_TILE_ROWS;
constexpr int kTileCols = CVFES_TILE_COLS;
constexpr int kTileElems = CVFES_TILE_ELEMS;

struct StepArgs {
    RowArgs k;
    const double *u;      // u_n   [N][3][S]
    const double *up;     // u_n-1 [N][3][S]
    double *out;          // u_n+1 (step) or y = K u (spmv)
    const double *lm;
    int64_t lm_sstride;
    const double *f1;
    const uint8_t *fixed;
    cvfes_load_t load;    // load.p null: the pressure is p0
    double p0;
    double bdy_u;
    double dt2;
    double bdt;           // beta / dt
    double ddt;           // damp / dt
    const int32_t *order; // visiting order of the rows (wave-uniform kernels; null = natural)
    unsigned occ_lds;     // launch only: unused LDS per workgroup that caps the occupancy
    bool nt_out;          // write `out` with non-temporal stores (stream_out)
};

// The same arguments with global-address-space pointers (see CVFES_G); the generic row functions
// below take either form.
// Read-only per-row data (structure, unit blocks, masses, loads) is in the constant address space
// (CVFES_K); the per-sample streams (values, coefficients, states) are global.
struct GRowArgs {
    int64_t n_nodes;
    int64_t n_smp;
    const CVFES_K int32_t *indptr;
    const CVFES_K int32_t *indices;
    const CVFES_G double *values;
    const CVFES_K int32_t *cptr;
    const CVFES_K int32_t *celem;
    const CVFES_K double *khat;
    const CVFES_G double *coef;
    const CVFES_G double *uvalues;
    const CVFES_K int32_t *vblk;
    const CVFES_K int32_t *nptr;
    const CVFES_K fan_t *fan;
};

struct GLoad {
    const CVFES_K double *p, *ga, *qa, *gb, *qb;
};

struct GStepArgs {
    GRowArgs k;
    const CVFES_G double *u;
    const CVFES_G double *up;
    CVFES_G double *out;
    const CVFES_K double *lm;
    int64_t lm_sstride;
    const CVFES_K double *f1;
    const CVFES_K uint8_t *fixed;
    GLoad load;
    double bdy_u;
    double dt2;
    double bdt;
    double ddt;
    bool nt_out;
};

// One matrix-free step as cvfes_step launches it (bcsr.hip).
void launch_matfree_step(hipStream_t st, const cvfes_system_t *sys, const StepArgs &a, bool beta, bool damp);

// Entry of a stored upper block that gives entry ij of the block a row needs: `side` < 0 the block's
// column precedes its row (read transposed), 0 it is the row's diagonal block, > 0 neither.  The
// diagonal block of a symmetric matrix is symmetric itself, so only its upper six entries are read:
// a quarter of the stored blocks are diagonal ones, which is 8 % of the stream of values.
__device__ __forceinline__ constexpr int sym_entry(int ij, int side) {
    const int i = ij / 3, j = ij % 3;
    return side < 0 || (side == 0 && i > j) ? 3 * j + i : ij;
}

// Stored block p of the row: kv[ij][v] = K_p[ij] of sample s + v.  SYM: symmetric storage, the
// block is the upper block vblk[p] (`side`: sym_entry).
template <bool SYM, int VW, class RA>
__device__ __forceinline__ void stored_block(const RA &k, int32_t p, int side, int64_t s,
                                             double (&kv)[9][VW]) {
    if constexpr (!SYM) {
        const auto *base = k.values + (static_cast<int64_t>(p) * 9) * k.n_smp + s;
#pragma unroll
        for (int ij = 0; ij < 9; ++ij) {
            const Vec<VW> t = load_vec<VW>(base + ij * k.n_smp);
#pragma unroll
            for (int v = 0; v < VW; ++v) kv[ij][v] = t.v[v];
        }
    } else {
        // sym_entry as two offsets: the entries above the diagonal lie 2 or 4 rows further on where the
        // block is read transposed, those below it as far back where it is or is the diagonal block.
        // Chosen entry by entry, packed rows branch and wait for memory in both branches.
        const int64_t n = k.n_smp, up = side < 0 ? 2 * n : 0, down = side > 0 ? 0 : 2 * n;
        const auto *base = k.uvalues + (static_cast<int64_t>(k.vblk[p]) * 9) * n + s;
        const int64_t at[9] = {0,     n + up,           2 * (n + up), 3 * n - down, 4 * n,
                               5 * n + up, 2 * (3 * n - down), 7 * n - down, 8 * n};
#pragma unroll
        for (int ij = 0; ij < 9; ++ij) {
            const Vec<VW> t = load_vec<VW>(base + at[ij]);
#pragma unroll
            for (int v = 0; v < VW; ++v) kv[ij][v] = t.v[v];
        }
    }
}

// acc[i][v] += K_p (i, :) . x for block p of the row.  Stored: the 3x3 block is read.  Matrix-free:
// K_p = sum over the block's element contributions c of coef_e(c) * khat_c, applied as
// acc += coef_e (khat_c x), so the block itself is never formed and only the three sums per
// sample are live (khat_c is wave-uniform for wave-uniform rows: scalar loads).
// `side`: the block's column less its row, for the symmetric storage (sym_entry).
// PIN: all nine entries of a stored block in flight before the first is used; the compiler else waits
// for them a few at a time in some kernels (16,384 rows of up to 13 blocks, 8 samples: 23.0 -> 13.4 us a
// step with the other two forms of this walk, sym_entry's two offsets and the row's own state first;
// the adjoint step of one sample per lane is scheduled well as it is: 11.9 us, pinned 12.9).
template <int OP, int VW, bool PIN = VW == 2, class RA>
__device__ __forceinline__ void block_apply(const RA &k, int32_t p, int side, int64_t s,
                                            const double (&x)[3][VW], double (&acc)[3][VW]) {
    if constexpr (OP != kOpMatfree) {
        double kv[9][VW];
        stored_block<OP == kOpSym, VW>(k, p, side, s, kv);
        if constexpr (PIN) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j)
#pragma unroll
                for (int v = 0; v < VW; ++v) acc[i][v] = fma(kv[3 * i + j][v], x[j][v], acc[i][v]);
    } else {
        const int32_t c0 = k.cptr[p], c1 = k.cptr[p + 1];
        for (int32_t c = c0; c < c1; ++c) {
            const int64_t e = k.celem[c];
            const Vec<VW> cf = load_vec<VW>(k.coef + e * k.n_smp + s);
            const auto *kh = k.khat + 9 * static_cast<int64_t>(c);
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const double h0 = kh[3 * i], h1 = kh[3 * i + 1], h2 = kh[3 * i + 2];
#pragma unroll
                for (int v = 0; v < VW; ++v) {
                    const double t = fma(h2, x[2][v], fma(h1, x[1][v], h0 * x[0][v]));
                    acc[i][v] = fma(cf.v[v], t, acc[i][v]);
                }
            }
        }
    }
}

// Column term of the step's product at node col: x = u + bdt (u - up) when BETA, else u.
template <bool BETA, int VW, class DP>
__device__ __forceinline__ void state_column(DP u, DP up, double bdt, int64_t col, int64_t n_smp,
                                             int64_t s, double (&x)[3][VW]) {
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int64_t off = (col * 3 + j) * n_smp + s;
        const Vec<VW> xu = load_vec<VW>(u + off);
        if constexpr (BETA) {
            const Vec<VW> xp = load_vec<VW>(up + off);
#pragma unroll
            for (int v = 0; v < VW; ++v) x[j][v] = fma(bdt, xu.v[v] - xp.v[v], xu.v[v]);
        } else {
#pragma unroll
            for (int v = 0; v < VW; ++v) x[j][v] = xu.v[v];
        }
    }
}

// block_apply for two columns at once (the block is loaded once): acc += K_p x and acc2 += K_p x2,
// each with exactly the operations block_apply performs.
template <int OP, int VW, class RA>
__device__ __forceinline__ void block_apply2(const RA &k, int32_t p, int side, int64_t s,
                                             const double (&x)[3][VW], double (&acc)[3][VW],
                                             const double (&x2)[3][VW], double (&acc2)[3][VW]) {
    if constexpr (OP != kOpMatfree) {
        double kv[9][VW];
        stored_block<OP == kOpSym, VW>(k, p, side, s, kv);
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j)
#pragma unroll
                for (int v = 0; v < VW; ++v) {
                    acc[i][v] = fma(kv[3 * i + j][v], x[j][v], acc[i][v]);
                    acc2[i][v] = fma(kv[3 * i + j][v], x2[j][v], acc2[i][v]);
                }
    } else {
        const int32_t c0 = k.cptr[p], c1 = k.cptr[p + 1];
        for (int32_t c = c0; c < c1; ++c) {
            const int64_t e = k.celem[c];
            const Vec<VW> cf = load_vec<VW>(k.coef + e * k.n_smp + s);
            const auto *kh = k.khat + 9 * static_cast<int64_t>(c);
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const double h0 = kh[3 * i], h1 = kh[3 * i + 1], h2 = kh[3 * i + 2];
#pragma unroll
                for (int v = 0; v < VW; ++v) {
                    const double t = fma(h2, x[2][v], fma(h1, x[1][v], h0 * x[0][v]));
                    acc[i][v] = fma(cf.v[v], t, acc[i][v]);
                    const double t2 = fma(h2, x2[2][v], fma(h1, x2[1][v], h0 * x2[0][v]));
                    acc2[i][v] = fma(cf.v[v], t2, acc2[i][v]);
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Ext-vector forms (one value or two consecutive samples per lane) used by the row-load and
// LDS-staged kernels.
typedef double dbl2 __attribute__((ext_vector_type(2)));

template <int VW> struct VecT;
template <> struct VecT<1> { typedef double type; };
template <> struct VecT<2> { typedef dbl2 type; };

template <int VW, bool NT>
__device__ __forceinline__ typename VecT<VW>::type ldv(const double *p) {
    typedef typename VecT<VW>::type V;
    if constexpr (NT)
        return __builtin_nontemporal_load(reinterpret_cast<const V *>(p));
    else
        return *reinterpret_cast<const V *>(p);
}

// Buffer loads: a resource (base address and size in bytes, built in scalar registers from
// wave-uniform values) and a 32-bit per-lane byte offset.  Every load of a row then shares one
// per-lane address register (the sample offset) instead of holding a 64-bit address per load,
// which is what lets the symmetric step kernel keep four waves per SIMD.  Word 3 of the resource
// is the gfx9 raw-access form (32-bit data format, no swizzle).  AUX is the load's cache policy:
// 0 plain, kAuxNT non-temporal.  Every offset the kernels form lies inside its resource, so the
// hardware's range check (which would return zeros) never applies.
constexpr int kAuxNT = 2;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_rsrc(const double *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<double *>(base), static_cast<short>(0),
                                             static_cast<int>(bytes), 0x00020000);
}

template <int VW, int AUX>
__device__ __forceinline__ typename VecT<VW>::type ldb(__amdgpu_buffer_rsrc_t r, uint32_t lane_off,
                                                       uint32_t off) {
    if constexpr (VW == 2)
        return __builtin_bit_cast(dbl2, __builtin_amdgcn_raw_buffer_load_b128(
                                            r, static_cast<int>(lane_off), static_cast<int>(off), AUX));
    else
        return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(
                                              r, static_cast<int>(lane_off), static_cast<int>(off), AUX));
}

template <int VW>
__device__ __forceinline__ Vec<VW> to_vec(typename VecT<VW>::type t) {
    Vec<VW> r;
    if constexpr (VW == 2) {
        r.v[0] = t[0];
        r.v[1] = t[1];
    } else {
        r.v[0] = t;
    }
    return r;
}

// The three components of a node's state, VW consecutive samples per lane at the lane's byte offset
// `lane`.  Wave-uniform rows (UNI): buffer loads (below: one address register per lane).
template <bool UNI, int VW, class DP>
__device__ __forceinline__ void load_node(DP base, int32_t node, int64_t n_smp, uint32_t lane,
                                          Vec<VW> (&r)[3]) {
    if constexpr (UNI) {
        const uint32_t sb = static_cast<uint32_t>(n_smp) * 8u;
        const auto rs = buffer_rsrc((const double *)(base + static_cast<int64_t>(node) * 3 * n_smp), 3 * sb);
#pragma unroll
        for (int j = 0; j < 3; ++j) r[j] = to_vec<VW>(ldb<VW, 0>(rs, lane, j * sb));
    } else {
#pragma unroll
        for (int j = 0; j < 3; ++j)
            r[j] = load_lane<VW>(base + (static_cast<int64_t>(node) * 3 + j) * n_smp, lane);
    }
}

// lane `i`'s value, i wave-uniform
__device__ __forceinline__ double lane_value(double x, int i) {
    const int2 w = __builtin_bit_cast(int2, x);
    return __builtin_bit_cast(double, make_int2(__builtin_amdgcn_readlane(w.x, i), __builtin_amdgcn_readlane(w.y, i)));
}

// One value per sample of row `i` of an [..][S] array.
template <bool UNI, int VW, class DP>
__device__ __forceinline__ Vec<VW> load_entry(DP base, int64_t i, int64_t n_smp, uint32_t lane) {
    if constexpr (UNI) {
        const uint32_t sb = static_cast<uint32_t>(n_smp) * 8u;
        return to_vec<VW>(ldb<VW, 0>(buffer_rsrc((const double *)(base + i * n_smp), sb), lane, 0));
    } else {
        return load_lane<VW>(base + i * n_smp, lane);
    }
}

// Columns of the fan product: load() issues a node's loads, column() forms the column from them,
// own() issues what the update of a row needs of its own node.  kCols columns share every
// operator load (the fused forward + adjoint step applies two).
template <bool UNI, bool BETA, int VW, class DP>
struct StateCol {
    static constexpr int kCols = 1;
    struct Raw {
        Vec<VW> u[3], up[3];
    };
    typedef Raw Own;
    DP u, up;
    double bdt;
    int64_t n_smp;
    uint32_t lane;          // the lane's byte offset in every row (its first sample)

    __device__ __forceinline__ Raw load(int32_t node) const {
        Raw r;
        load_node<UNI, VW>(u, node, n_smp, lane, r.u);
        if constexpr (BETA) load_node<UNI, VW>(up, node, n_smp, lane, r.up);
        return r;
    }
    __device__ __forceinline__ Own own(int32_t node) const {
        Own o;
        load_node<UNI, VW>(u, node, n_smp, lane, o.u);
        load_node<UNI, VW>(up, node, n_smp, lane, o.up);
        return o;
    }
    __device__ __forceinline__ void column(const Raw &r, double (&x)[3][VW]) const {
#pragma unroll
        for (int j = 0; j < 3; ++j)
#pragma unroll
            for (int v = 0; v < VW; ++v)
                x[j][v] = BETA ? fma(bdt, r.u[j].v[v] - r.up[j].v[v], r.u[j].v[v]) : r.u[j].v[v];
    }
    __device__ __forceinline__ void value(const Raw &r, double (&x)[1][3][VW]) const { column(r, x[0]); }
};

// a - b as it stands: a column that is itself a product would else be fused into the difference in
// the kernels that form it in registers, and not in those that read it back from LDS.
__device__ __forceinline__ double minus(double a, double b) {
#pragma clang fp contract(off)
    return a - b;
}

// acc[c] = the row's matrix-free product with each column c: for every element e around the row
// node a, with p and q its other nodes, acc += coef_e (khat_e(a,p) (x_p - x_a) + khat_e(a,q) (x_q -
// x_a)): an element's rows sum to zero, so its block (a,a) is neither read nor applied.  Compared
// with the walk over blocks, the coefficient is read and applied once per element instead of once
// per contribution, and where the entries chain around the node each neighbour is read once.  The next element's loads are issued before the current one is applied.
// A row's contributions are contiguous, so its unit blocks start at contribution 3 nptr[row].
template <bool UNI, int VW, class COL, class RA>
__device__ __forceinline__ void fan_product(const RA &k, const COL &col, int32_t row,
                                            double (&acc)[COL::kCols][3][VW]) {
    constexpr int NC = COL::kCols;
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int v = 0; v < VW; ++v) acc[c][i][v] = 0.0;
    const int32_t q0 = k.nptr[row], q1 = k.nptr[row + 1];
    if (q0 == q1) return;
    const auto *kh0 = k.khat + 27 * static_cast<int64_t>(q0);
    double xa[NC][3][VW], xp[NC][3][VW], xq[NC][3][VW];     // xp, xq less xa
    auto relative = [&](const typename COL::Raw &raw, double (&x)[NC][3][VW]) {
        col.value(raw, x);
#pragma unroll
        for (int m = 0; m < NC; ++m)
#pragma unroll
            for (int j = 0; j < 3; ++j)
#pragma unroll
                for (int v = 0; v < VW; ++v) x[m][j][v] = minus(x[m][j][v], xa[m][j][v]);
    };
    fan_t e = k.fan[q0];
    typename COL::Raw r = col.load(e.y);
    Vec<VW> c = load_entry<UNI, VW>(k.coef, e.z, k.n_smp, col.lane);
    {
        const typename COL::Raw ra = col.load(row), rp = col.load(e.x);
        col.value(ra, xa);
        relative(rp, xp);
    }
    for (int32_t q = q0 + 1;; ++q) {
        const fan_t n = k.fan[q < q1 ? q : q1 - 1];
        relative(r, xq);
        const Vec<VW> cf = c;
        r = col.load(n.y);              // behind the last element: its own node again
        c = load_entry<UNI, VW>(k.coef, n.z, k.n_smp, col.lane);
        __builtin_amdgcn_sched_barrier(0);
        const auto *kp = kh0 + 9 * ((e.w >> 10) & 1023);
        const auto *kq = kh0 + 9 * ((e.w >> 20) & 1023);
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int m = 0; m < NC; ++m)
#pragma unroll
                for (int v = 0; v < VW; ++v) {
                    double t = kp[3 * i] * xp[m][0][v];
#pragma unroll
                    for (int j = 1; j < 3; ++j) t = fma(kp[3 * i + j], xp[m][j][v], t);
#pragma unroll
                    for (int j = 0; j < 3; ++j) t = fma(kq[3 * i + j], xq[m][j][v], t);
                    acc[m][i][v] = fma(cf.v[v], t, acc[m][i][v]);
                }
        if (q >= q1) break;
        if (n.x >= 0) {
            relative(col.load(n.x), xp);
        } else {
#pragma unroll
            for (int m = 0; m < NC; ++m)
#pragma unroll
                for (int j = 0; j < 3; ++j)
#pragma unroll
                    for (int v = 0; v < VW; ++v) xp[m][j][v] = xq[m][j][v];
        }
        e = n;
    }
}

// acc[c] = the row's product with each column c from the symmetric storage, the row's structure
// coming from its record `r` (cvfes_system_t.row_records): the operations of block_apply, block by
// block in the same order, with the next block's loads issued before the current one is applied.  The walk over
// indptr, indices and vblk puts two dependent loads in front of every block's values.  Slots behind
// the row's last block repeat it and are not added.
template <bool UNI, int VW, class COL>
__device__ __forceinline__ void sym_product(const RowArgs &k, const int32_t *r, const COL &col, int32_t row,
                                            double (&acc)[COL::kCols][3][VW]) {
    constexpr int NC = COL::kCols;
    const int32_t nb = r[1];
    const int64_t S = k.n_smp;
    const uint32_t sb = static_cast<uint32_t>(S) * 8u;
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int v = 0; v < VW; ++v) acc[c][i][v] = 0.0;
    // blocks in flight, this one included: as many as leave two waves per SIMD (one sample per lane:
    // 166 registers; all of a row's blocks at once, which is what the compiler makes of the plain
    // loop, run at one wave per SIMD)
    constexpr int D = VW == 1 ? (NC == 1 ? 6 : 4) : (NC == 1 ? 3 : 2);
    typename COL::Raw x[D];
    Vec<VW> kv[D][9];
    auto issue = [&](int b) {
        const int32_t node = r[2 + b];
        const int side = node - row;
        const double *base = k.uvalues + static_cast<int64_t>(r[2 + kRecordSlots + b]) * 9 * S;
        x[b % D] = col.load(node);
#pragma unroll
        for (int ij = 0; ij < 9; ++ij) {
            const uint32_t src = side < 0 ? sym_entry(ij, -1) : (side == 0 ? sym_entry(ij, 0) : ij);
            if constexpr (UNI) kv[b % D][ij] = to_vec<VW>(ldb<VW, 0>(buffer_rsrc(base, 9 * sb), col.lane, src * sb));
            else kv[b % D][ij] = load_lane<VW>(base, src * sb + col.lane);
        }
    };
#pragma unroll
    for (int b = 0; b < D - 1; ++b) issue(b);
#pragma unroll
    for (int b = 0; b < kRecordSlots; ++b) {
        if (b + D - 1 < kRecordSlots) issue(b + D - 1);
        __builtin_amdgcn_sched_barrier(0);
        double xv[NC][3][VW];
        col.value(x[b % D], xv);
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int v = 0; v < VW; ++v) {
                    double t = acc[c][i][v];
#pragma unroll
                    for (int j = 0; j < 3; ++j) t = fma(kv[b % D][3 * i + j].v[v], xv[c][j][v], t);
                    acc[c][i][v] = b < nb ? t : acc[c][i][v];
                    // the sums stay here: they would be moved behind the loads of all blocks
                    asm volatile("" : "+v"(acc[c][i][v]));
                }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// acc[i][v] = sum over the row's blocks of K_p (i, :) . x_col, with x = u + bdt (u - up) when BETA.
template <int OP, bool BETA, int VW, class RA, class DP>
__device__ __forceinline__ void row_product(const RA &k, DP u, DP up, double bdt, int32_t row,
                                            int64_t s, double (&acc)[3][VW]) {
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int v = 0; v < VW; ++v) acc[i][v] = 0.0;
    const int32_t p0 = k.indptr[row], p1 = k.indptr[row + 1];
    for (int32_t p = p0; p < p1; ++p) {
        const int64_t col = k.indices[p];
        double x[3][VW];
        state_column<BETA, VW>(u, up, bdt, col, k.n_smp, s, x);
        block_apply<OP, VW, true>(k, p, static_cast<int>(col) - row, s, x, acc);
    }
}

// What the update of a row reads besides its states: unit load, lumped mass, whether the node is
// fixed.
template <int VW>
struct RowLoad {
    double f1[3];
    Vec<VW> m;
    bool fixed;
};

template <int VW, class SA>
__device__ __forceinline__ RowLoad<VW> row_load(const SA &a, int32_t row, int64_t s) {
    RowLoad<VW> r;
    r.fixed = a.fixed != nullptr && a.fixed[row] != 0;
#pragma unroll
    for (int i = 0; i < 3; ++i) r.f1[i] = a.f1[3 * static_cast<int64_t>(row) + i];
    if (a.lm_sstride) {
        const auto *lmp = a.lm + (static_cast<int64_t>(row) * a.k.n_smp + s);
#pragma unroll
        for (int v = 0; v < VW; ++v) r.m.v[v] = lmp[v];
    } else {
        const double mr = a.lm[row];
#pragma unroll
        for (int v = 0; v < VW; ++v) r.m.v[v] = mr;
    }
    return r;
}

// Pressure of a step: from its table, or (the single-mesh step only) with the launch.  One load in
// either case, of an address that holds: behind a branch it would wait for the row's product.
__device__ __forceinline__ double step_pressure(const StepArgs &a, int64_t step) {
    const double p = *(a.load.p ? a.load.p + step : a.f1);
    return a.load.p ? p : a.p0;
}

template <class SA>
__device__ __forceinline__ double step_pressure(const SA &a, int64_t step) {
    return a.load.p[step];
}

// Central-difference update of one block row and VW consecutive samples from its product
// acc = K x and its own state uu = u_n, pp = u_{n-1}: load, damping, lumped mass and Dirichlet
// value; stores u_{n+1} when `active`.  Every product and sum that could be contracted is an
// explicit fma, so the rounding is the same in every kernel that uses it (single-mesh, batched,
// and the step fused with the adjoint).  Everything the update reads is read before its first
// store: behind a store the compiler no longer takes the row's masses and loads through scalar
// loads, and the three components would wait for memory one after the other.
template <bool DAMP, int VW, class SA>
__device__ __forceinline__ void step_update(const SA &a, int32_t row, int64_t s, bool active,
                                            int64_t step, const RowLoad<VW> &r,
                                            const double (&acc)[3][VW], const Vec<VW> (&uu)[3],
                                            const Vec<VW> (&pp)[3]) {
    const int64_t nsm = a.k.n_smp;
    const double pn = step_pressure(a, step);
    double fi[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) fi[i] = pn * r.f1[i];
    if (a.load.ga) {
        const double qa = a.load.qa[step];
#pragma unroll
        for (int i = 0; i < 3; ++i) fi[i] = fma(qa, a.load.ga[3 * static_cast<int64_t>(row) + i], fi[i]);
    }
    if (a.load.gb) {
        const double qb = a.load.qb[step];
#pragma unroll
        for (int i = 0; i < 3; ++i) fi[i] = fma(qb, a.load.gb[3 * static_cast<int64_t>(row) + i], fi[i]);
    }
    Vec<VW> o[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
#pragma unroll
        for (int v = 0; v < VW; ++v) {
            double force = fi[i];
            if constexpr (DAMP) force = fma(-a.ddt, uu[i].v[v] - pp[i].v[v], force);
            const double rhs = fma(a.dt2, force - acc[i][v], r.m.v[v] * fma(2.0, uu[i].v[v], -pp[i].v[v]));
            const double un = r.m.v[v] != 0.0 ? rhs / r.m.v[v] : 0.0;
            o[i].v[v] = r.fixed ? a.bdy_u : un;
        }
    }
    // u_{n+1} is not read again in this launch: large outputs are streamed past L2 (stream_out)
    if (active) {
        auto *out = a.out + static_cast<int64_t>(row) * 3 * nsm + s;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            if (a.nt_out) store_vec_nt<VW>(out + i * nsm, o[i]);
            else store_vec<VW>(out + i * nsm, o[i]);
        }
    }
}

// The row's own state.
template <int VW, class SA>
__device__ __forceinline__ void own_state(const SA &a, int32_t row, int64_t s, Vec<VW> (&uu)[3], Vec<VW> (&pp)[3]) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int64_t off = (static_cast<int64_t>(row) * 3 + i) * a.k.n_smp + s;
        uu[i] = load_vec<VW>(a.u + off);
        pp[i] = load_vec<VW>(a.up + off);
    }
}

// The same with the row's own state read here.
template <bool DAMP, int VW, class SA>
__device__ __forceinline__ void step_update(const SA &a, int32_t row, int64_t s, bool active,
                                            int64_t step, const double (&acc)[3][VW]) {
    Vec<VW> uu[3], pp[3];
    own_state<VW>(a, row, s, uu, pp);
    step_update<DAMP, VW>(a, row, s, active, step, row_load<VW>(a, row, s), acc, uu, pp);
}

// Block-row product and central-difference update of one block row and VW consecutive samples.
// UNI: the row is wave-uniform.
template <int OP, bool UNI, bool BETA, bool DAMP, int VW, class SA>
__device__ __forceinline__ void step_row(const SA &a, int32_t row, int64_t s, bool active,
                                         int64_t step) {
    if constexpr (OP == kOpFan) {
        typedef StateCol<UNI, BETA, VW, decltype(a.u)> Col;
        const Col col{a.u, a.up, a.bdt, a.k.n_smp, static_cast<uint32_t>(s) * 8u};
        double acc[1][3][VW];
        fan_product<UNI, VW>(a.k, col, row, acc);
        step_update<DAMP, VW>(a, row, s, active, step, acc[0]);
    } else {
        double acc[3][VW];
        if constexpr (!UNI && (VW == 1 || !BETA)) {
            // What the update reads is in flight during the product; with both states of two samples
            // it would take the registers of a wave (8 samples: 14.6 -> 19.1 us).  102,400 rows, one
            // sample: 27.2 -> 18.9 us a step, two 42.7 -> 33.8.
            Vec<VW> uu[3], pp[3];
            own_state<VW>(a, row, s, uu, pp);
            const RowLoad<VW> r = row_load<VW>(a, row, s);
            row_product<OP, BETA, VW>(a.k, a.u, a.up, a.bdt, row, s, acc);
            step_update<DAMP, VW>(a, row, s, active, step, r, acc, uu, pp);
        } else {
            row_product<OP, BETA, VW>(a.k, a.u, a.up, a.bdt, row, s, acc);
            step_update<DAMP, VW>(a, row, s, active, step, acc);
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Helpers of the row-load and LDS-staged kernels.
template <int VW>
__device__ __forceinline__ typename VecT<VW>::type splat(double x) {
    if constexpr (VW == 2) return dbl2{x, x};
    else return x;
}

template <int VW>
__device__ __forceinline__ typename VecT<VW>::type sel(bool keep, typename VecT<VW>::type v) {
    return keep ? v : splat<VW>(0.0);
}

// Central-difference update of one block row from its product acc = K (u + bdt (u - up)), with
// the row's own u/up already loaded; stores u_{n+1} when `active`, non-temporally when NTO (a
// compile-time choice: the row-load and symmetric kernels with non-temporal value loads, which
// are the forms for large problems, stream their output too).
template <bool DAMP, int VW, bool NTO = false>
__device__ __forceinline__ void finish_row(const StepArgs &a, int32_t row, int64_t s, bool active,
                                           int64_t step, const typename VecT<VW>::type (&uo)[3],
                                           const typename VecT<VW>::type (&po)[3],
                                           const typename VecT<VW>::type (&acc)[3]) {
    typedef typename VecT<VW>::type V;
    const int64_t S = a.k.n_smp;
    const double pn = step_pressure(a, step);
    const double qa = a.load.ga ? a.load.qa[step] : 0.0;
    const double qb = a.load.gb ? a.load.qb[step] : 0.0;
    const bool fixed = a.fixed != nullptr && a.fixed[row] != 0;
    const V m = a.lm_sstride ? ldv<VW, false>(a.lm + static_cast<int64_t>(row) * S + s)
                             : splat<VW>(a.lm[row]);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int64_t d = 3 * static_cast<int64_t>(row) + i;
        double fi = pn * a.f1[d];
        if (a.load.ga) fi += qa * a.load.ga[d];
        if (a.load.gb) fi += qb * a.load.gb[d];
        V force = splat<VW>(fi);
        if constexpr (DAMP) force -= a.ddt * (uo[i] - po[i]);
        const V rhs = a.dt2 * (force - acc[i]) + m * (2.0 * uo[i] - po[i]);
        V un;
        if constexpr (VW == 2) {
            un.x = m.x != 0.0 ? rhs.x / m.x : 0.0;
            un.y = m.y != 0.0 ? rhs.y / m.y : 0.0;
        } else {
            un = m != 0.0 ? rhs / m : 0.0;
        }
        if (fixed) un = splat<VW>(a.bdy_u);
        if (active) {
            V *dst = reinterpret_cast<V *>(a.out + (static_cast<int64_t>(row) * 3 + i) * S + s);
            if constexpr (NTO) __builtin_nontemporal_store(un, dst);
            else *dst = un;
        }
    }
}

// ---------------------------------------------------------------------------------------------
// Matrix-free row step with the row's element data staged in LDS.
//
// The generic matrix-free row walks blocks and, inside each block, element contributions, and
// every contribution is a dependent chain (element id -> coefficient load -> FMAs), about 25 memory
// round trips per row.  Here one wavefront owns one row (wave-uniform, 64*VW samples) and:
//   1. loads, all at once, the coefficient of every element incident to the row node (one
//      coalesced load per element), the unit element blocks and element slots of the row's
//      contributions (contiguous: one lane per value), and the neighbour states;
//   2. parks coefficients, element blocks and slots in its LDS slice;
//   3. rebuilds each block as sum_c coef[slot_c] * khat_c from LDS (element blocks and slots are
//      read at wave-uniform addresses, i.e. broadcast) and accumulates the product with the
//      neighbour state.
// A row node with ne incident elements has exactly 3*ne contributions (each element adds one to
// the blocks (row, b) of its three nodes b).  Limits (exact maxima, checked on the host): blocks
// per row <= MAXB, incident elements per node <= MAXE.
struct LdsArgs {
    const int32_t *nptr;    // [N+1] node -> incident (element, local) list
    const int32_t *nent;    // [3E]  e*3 + local
    const int32_t *cslot;   // [9E]  slot of contribution c's element in its row node's list
};

template <int VW, int MAXE>
struct LdsRow {
    typename VecT<VW>::type coef[MAXE][64];
    double khat[3 * MAXE * 9];
    int32_t slot[3 * MAXE];
};

// Orders this wavefront's LDS writes before its later reads (and earlier reads before later
// writes when a wavefront reuses its slice); only the own wavefront shares the slice.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <bool BETA, bool DAMP, int VW, int MAXB, int MAXE>
__device__ __forceinline__ void step_row_lds(const StepArgs &a, const LdsArgs &l, LdsRow<VW, MAXE> &sl,
                                             int32_t row, int64_t s, bool active, int64_t step) {
    constexpr int MAXC = 3 * MAXE;
    constexpr int KH = (MAXC * 9 + 63) / 64;     // element-block values per lane
    typedef typename VecT<VW>::type V;
    const int lane = threadIdx.x & 63;
    const RowArgs &k = a.k;
    const int64_t S = k.n_smp;
    const int32_t p0 = k.indptr[row];
    const int32_t nb = k.indptr[row + 1] - p0;
    const int32_t q0 = l.nptr[row];
    const int32_t ne = l.nptr[row + 1] - q0;
    V uo[3], po[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int64_t off = (static_cast<int64_t>(row) * 3 + i) * S + s;
        uo[i] = ldv<VW, false>(a.u + off);
        po[i] = ldv<VW, false>(a.up + off);
    }
    V acc[3] = {splat<VW>(0.0), splat<VW>(0.0), splat<VW>(0.0)};
    if (nb > 0 && ne > 0) {
        const int32_t c0 = k.cptr[p0];
        const int32_t nc = k.cptr[p0 + nb] - c0;
        // 1. every load of the row, issued together
        V cf[MAXE];
#pragma unroll
        for (int e = 0; e < MAXE; ++e) {
            const int64_t el = l.nent[q0 + (e < ne ? e : ne - 1)] / 3;
            cf[e] = ldv<VW, false>(k.coef + el * S + s);
        }
        double kh[KH];
#pragma unroll
        for (int j = 0; j < KH; ++j) {
            const int idx = lane + 64 * j;
            kh[j] = idx < 9 * nc ? k.khat[9 * static_cast<int64_t>(c0) + idx] : 0.0;
        }
        const int32_t slot = lane < nc ? l.cslot[c0 + lane] : 0;
        V w[MAXB][3];
#pragma unroll
        for (int b = 0; b < MAXB; ++b) {
            const int64_t col = k.indices[p0 + (b < nb ? b : nb - 1)];
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const int64_t off = (col * 3 + j) * S + s;
                const V xu = ldv<VW, false>(a.u + off);
                if constexpr (BETA) {
                    const V xp = ldv<VW, false>(a.up + off);
                    w[b][j] = xu + a.bdt * (xu - xp);
                } else {
                    w[b][j] = xu;
                }
            }
        }
        // 2. stage coefficients, element blocks and slots in this wavefront's LDS slice
        wave_lds_sync();
#pragma unroll
        for (int e = 0; e < MAXE; ++e) sl.coef[e][lane] = cf[e];
#pragma unroll
        for (int j = 0; j < KH; ++j) {
            const int idx = lane + 64 * j;
            if (idx < MAXC * 9) sl.khat[idx] = kh[j];
        }
        if (lane < MAXC) sl.slot[lane] = slot;
        wave_lds_sync();
        // 3. rebuild each block from LDS and accumulate its product
        int32_t cb = 0;
#pragma unroll
        for (int b = 0; b < MAXB; ++b) {
            if (b < nb) {
                const int32_t ce = k.cptr[p0 + b + 1] - c0;
                V kv[9];
#pragma unroll
                for (int ij = 0; ij < 9; ++ij) kv[ij] = splat<VW>(0.0);
                for (int32_t j = cb; j < ce; ++j) {
                    const V c = sl.coef[sl.slot[j]][lane];
                    const double *kb = &sl.khat[9 * j];
#pragma unroll
                    for (int ij = 0; ij < 9; ++ij) kv[ij] += c * kb[ij];
                }
                cb = ce;
#pragma unroll
                for (int i = 0; i < 3; ++i)
#pragma unroll
                    for (int j = 0; j < 3; ++j) acc[i] += kv[3 * i + j] * w[b][j];
            }
        }
    }
    finish_row<DAMP, VW>(a, row, s, active, step, uo, po, acc);
}

// ---------------------------------------------------------------------------------------------
// Matrix-free row step with the row node's element coefficients loaded once per row.
//
// In the generic matrix-free row every element contribution loads its coefficient again (a row
// has 3 contributions per incident element) and each load sits in a dependent chain.  Here the
// wavefront (one row, wave-uniform) first loads the coefficients of the node's incident elements
// (at most MAXE, all issued together), then walks the blocks; each contribution picks its
// element's coefficient from registers by its slot (cslot, uniform) and its unit block from the
// scalar cache, so no vector load remains inside the contribution loop.
template <bool BETA, bool DAMP, int VW, int MAXE>
__device__ __forceinline__ void step_row_cached(const StepArgs &a, const LdsArgs &l, int32_t row,
                                                int64_t s, bool active, int64_t step) {
    typedef typename VecT<VW>::type V;
    const RowArgs &k = a.k;
    const int64_t S = k.n_smp;
    const int32_t q0 = l.nptr[row];
    const int32_t ne = l.nptr[row + 1] - q0;
    V cf[MAXE];
#pragma unroll
    for (int e = 0; e < MAXE; ++e) cf[e] = splat<VW>(0.0);
    if (ne > 0) {                   // an isolated node has no elements and no blocks
#pragma unroll
        for (int e = 0; e < MAXE; ++e) {
            const int64_t el = l.nent[q0 + (e < ne ? e : ne - 1)] / 3;
            cf[e] = ldv<VW, false>(k.coef + el * S + s);
        }
    }
    V uo[3], po[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int64_t off = (static_cast<int64_t>(row) * 3 + i) * S + s;
        uo[i] = ldv<VW, false>(a.u + off);
        po[i] = ldv<VW, false>(a.up + off);
    }
    V acc[3] = {splat<VW>(0.0), splat<VW>(0.0), splat<VW>(0.0)};
    const int32_t p0 = k.indptr[row], p1 = k.indptr[row + 1];
    for (int32_t p = p0; p < p1; ++p) {
        const int64_t col = k.indices[p];
        V x[3];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const int64_t off = (col * 3 + j) * S + s;
            const V xu = ldv<VW, false>(a.u + off);
            if constexpr (BETA) {
                const V xp = ldv<VW, false>(a.up + off);
                x[j] = xu + a.bdt * (xu - xp);
            } else {
                x[j] = xu;
            }
        }
        V kv[9];
#pragma unroll
        for (int ij = 0; ij < 9; ++ij) kv[ij] = splat<VW>(0.0);
        for (int32_t c = k.cptr[p]; c < k.cptr[p + 1]; ++c) {
            const int32_t slot = l.cslot[c];
            V cfc = cf[0];
#pragma unroll
            for (int e = 1; e < MAXE; ++e)
                if (slot == e) cfc = cf[e];
            const double *kh = k.khat + 9 * static_cast<int64_t>(c);
#pragma unroll
            for (int ij = 0; ij < 9; ++ij) kv[ij] += cfc * kh[ij];
        }
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
            for (int j = 0; j < 3; ++j) acc[i] += kv[3 * i + j] * x[j];
    }
    finish_row<DAMP, VW>(a, row, s, active, step, uo, po, acc);
}

}  // namespace cvfes
