// Adjoint of the explicit central-difference step, and the gradient with respect to the element
// log-modulus.
//
// Forward step (per sample, A = dt^2 M^-1 diagonal, P zeroes fixed dofs, b1 = 1 + beta/dt,
// b0 = beta/dt, gamma = dt damp / m):
//   u_{n+1} = P[(2-gamma) u_n - (1-gamma) u_{n-1} - A K (b1 u_n - b0 u_{n-1}) + A f_n] + (I-P) g.
// For L = sum_n l_n(u_n) the adjoint recurrence, with mu_n = P lambda_n and K symmetric, is
//   lambda_n = dl_n/du_n + (2-gamma) mu_{n+1} - (1-gamma) mu_{n+2} - K A (b1 mu_{n+1} - b0 mu_{n+2}),
// the same gathered block product as the forward step with a column scale dt^2/m.  With
// coef_e = h E_e and K = sum_e coef_e khat_e, the derivative with respect to theta_e = log E_e is
//   dL/dtheta_e = -coef_e sum_n (A mu_{n+1})_e^T khat_e (b1 u_n - b0 u_{n-1})_e.
// u_{-1} depends on K through the initial acceleration; its adjoint
//   lambda_{-1} = -(1-gamma) mu_1 + b0 K A mu_1   (u_{-1} is not projected)
// adds -coef_e (dt^2/2 M^-1 lambda_{-1})_e^T khat_e (u0 + beta du0)_e.
#include "tile.h"

namespace cvfes {
namespace {

struct AdjArgs {
    RowArgs k;             // structure and operator (stored values or element data)
    const double *mu1;     // mu_{n+1}
    const double *mu2;     // mu_{n+2}
    double *out;           // mu_n (projected) or lambda_{-1} (unprojected)
    const double *lm;
    int64_t lm_sstride;
    const double *minv;    // 1/lm (0 where lm = 0), same layout; NULL = divide by lm
    const uint8_t *fixed;
    const double *obs_u;   // u_n      (observation term, may be NULL)
    const double *obs_ref; // u_obs    (NULL = 0)
    const double *obs_w;   // [S] weight of the observation term per sample (NULL = 1)
    double dt2, bdt, dtdamp;
    int project;
    unsigned occ_lds;      // launch only: unused LDS per workgroup that caps the occupancy
    bool nt_out;           // write `out` with non-temporal stores (stream_out)
};

template <int VW>
__device__ __forceinline__ Vec<VW> mass_at(const AdjArgs &a, int64_t node, int64_t s) {
    Vec<VW> m;
    if (a.lm_sstride) {
        m = load_vec<VW>(a.lm + node * a.k.n_smp + s);
    } else {
        const double mv = a.lm[node];
#pragma unroll
        for (int v = 0; v < VW; ++v) m.v[v] = mv;
    }
    return m;
}

// Column term of the adjoint product at node col: x = dt^2/m_col (b1 mu1 - b0 mu2) (0 where the
// mass is 0); K is symmetric, so the transposed product is the same gathered row product.  With the
// inverse masses (minv, 0 where m = 0) the scale is dt^2 * minv_col, one multiply per column
// instead of an FP64 division per column and sample (the division sequence costs the kernel about
// a sixth of its time at 256 samples).
template <bool BETA, int VW>
__device__ __forceinline__ void adj_column(const AdjArgs &a, int64_t col, int64_t s, double (&x)[3][VW]) {
    Vec<VW> q;
    if (a.minv) {
        if (a.lm_sstride) {
            q = load_vec<VW>(a.minv + col * a.k.n_smp + s);
#pragma unroll
            for (int v = 0; v < VW; ++v) q.v[v] *= a.dt2;
        } else {
            const double qc = a.dt2 * a.minv[col];
#pragma unroll
            for (int v = 0; v < VW; ++v) q.v[v] = qc;
        }
    } else {
        const Vec<VW> mc = mass_at<VW>(a, col, s);
#pragma unroll
        for (int v = 0; v < VW; ++v) q.v[v] = mc.v[v] != 0.0 ? a.dt2 / mc.v[v] : 0.0;
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int64_t off = (col * 3 + j) * a.k.n_smp + s;
        const Vec<VW> m1 = load_vec<VW>(a.mu1 + off);
        Vec<VW> m2;
        if constexpr (BETA) m2 = load_vec<VW>(a.mu2 + off);
#pragma unroll
        for (int v = 0; v < VW; ++v) {
            double comb = m1.v[v];
            if constexpr (BETA) comb = fma(a.bdt, m1.v[v] - m2.v[v], m1.v[v]);
            x[j][v] = comb * q.v[v];
        }
    }
}

// The same column for the fan product: the node's loads (load) and the column formed from them.
template <bool UNI, bool BETA, int VW>
struct AdjCol {
    static constexpr int kCols = 1;
    struct Raw {
        Vec<VW> m1[3], m2[3], q;      // q: inverse mass (or mass) of the node
    };
    struct Own {
        Vec<VW> m1[3], m2[3];
    };
    const AdjArgs &a;
    uint32_t lane;

    __device__ __forceinline__ Raw load(int32_t node) const {
        Raw r;
        const double *m = a.minv ? a.minv : a.lm;
        if (a.lm_sstride) {
            r.q = load_entry<UNI, VW>(m, node, a.k.n_smp, lane);
        } else {
            const double mv = m[node];
#pragma unroll
            for (int v = 0; v < VW; ++v) r.q.v[v] = mv;
        }
        load_node<UNI, VW>(a.mu1, node, a.k.n_smp, lane, r.m1);
        if constexpr (BETA) load_node<UNI, VW>(a.mu2, node, a.k.n_smp, lane, r.m2);
        return r;
    }
    __device__ __forceinline__ Own own(int32_t node) const {
        Own o;
        load_node<UNI, VW>(a.mu1, node, a.k.n_smp, lane, o.m1);
        load_node<UNI, VW>(a.mu2, node, a.k.n_smp, lane, o.m2);
        return o;
    }
    __device__ __forceinline__ void column(const Raw &r, double (&x)[3][VW]) const {
#pragma unroll
        for (int v = 0; v < VW; ++v) {
            const double q = a.minv ? r.q.v[v] * a.dt2 : (r.q.v[v] != 0.0 ? a.dt2 / r.q.v[v] : 0.0);
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                double comb = r.m1[j].v[v];
                if constexpr (BETA) comb = fma(a.bdt, r.m1[j].v[v] - r.m2[j].v[v], r.m1[j].v[v]);
                x[j][v] = comb * q;
            }
        }
    }
    __device__ __forceinline__ void value(const Raw &r, double (&x)[1][3][VW]) const { column(r, x[0]); }
};

// Forward and adjoint columns of the fused step, both applied with each operator load.
template <bool UNI, bool BETA, int VW>
struct FusedCol {
    static constexpr int kCols = 2;
    typedef StateCol<UNI, BETA, VW, const double *> F;
    typedef AdjCol<UNI, BETA, VW> A;
    struct Raw {
        typename F::Raw f;
        typename A::Raw a;
    };
    F f;
    A a;
    uint32_t lane;

    __device__ __forceinline__ Raw load(int32_t node) const { return Raw{f.load(node), a.load(node)}; }
    __device__ __forceinline__ void value(const Raw &r, double (&x)[2][3][VW]) const {
        f.column(r.f, x[0]);
        a.column(r.a, x[1]);
    }
};

// lambda_n of one block row from acc = K A (b1 mu1 - b0 mu2) and the observation term; stores
// mu_n = P lambda_n (or lambda when not projecting) when `active`.  Explicit fma throughout, so
// the rounding is the same in the separate and the fused kernels.
template <bool DAMP, int VW>
__device__ __forceinline__ void adj_finish(const AdjArgs &a, int32_t row, int64_t s, bool active,
                                           const double (&acc)[3][VW], const Vec<VW> (&m1)[3],
                                           const Vec<VW> (&m2)[3]) {
    const int64_t S = a.k.n_smp;
    const bool fixed = a.project && a.fixed != nullptr && a.fixed[row] != 0;
    const int64_t off = static_cast<int64_t>(row) * 3 * S + s;
    Vec<VW> gam;
#pragma unroll
    for (int v = 0; v < VW; ++v) gam.v[v] = 0.0;
    if constexpr (DAMP) {
        const Vec<VW> m = mass_at<VW>(a, row, s);
#pragma unroll
        for (int v = 0; v < VW; ++v) gam.v[v] = m.v[v] != 0.0 ? a.dtdamp / m.v[v] : 0.0;
    }
    Vec<VW> o[3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int v = 0; v < VW; ++v)
            o[i].v[v] = fma(2.0 - gam.v[v], m1[i].v[v], -fma(1.0 - gam.v[v], m2[i].v[v], acc[i][v]));
    if (a.obs_u) {
        Vec<VW> w;
#pragma unroll
        for (int v = 0; v < VW; ++v) w.v[v] = a.obs_w ? a.obs_w[s + v] : 1.0;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const Vec<VW> u = load_vec<VW>(a.obs_u + off + i * S);
            Vec<VW> ref;
#pragma unroll
            for (int v = 0; v < VW; ++v) ref.v[v] = a.obs_ref ? a.obs_ref[off + i * S + v] : 0.0;
#pragma unroll
            for (int v = 0; v < VW; ++v) o[i].v[v] = fma(w.v[v], u.v[v] - ref.v[v], o[i].v[v]);
        }
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
#pragma unroll
        for (int v = 0; v < VW; ++v) o[i].v[v] = fixed ? 0.0 : o[i].v[v];
        if (active) {   // not read again in this launch: large outputs are streamed (stream_out)
            if (a.nt_out) store_vec_nt<VW>(a.out + off + i * S, o[i]);
            else store_vec<VW>(a.out + off + i * S, o[i]);
        }
    }
}

// The same with the row's own adjoint states read here.
template <bool DAMP, int VW>
__device__ __forceinline__ void adj_finish(const AdjArgs &a, int32_t row, int64_t s, bool active,
                                           const double (&acc)[3][VW]) {
    Vec<VW> m1[3], m2[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int64_t off = (static_cast<int64_t>(row) * 3 + i) * a.k.n_smp + s;
        m1[i] = load_vec<VW>(a.mu1 + off);
        m2[i] = load_vec<VW>(a.mu2 + off);
    }
    adj_finish<DAMP, VW>(a, row, s, active, acc, m1, m2);
}

template <int OP, bool UNIFORM, bool BETA, bool DAMP, int VW>
__global__ __launch_bounds__(kBlock) void k_adjoint_step(AdjArgs a) {
    int32_t row;
    int64_t s;
    bool active;
    if (!row_and_sample<UNIFORM, VW>(a.k.n_nodes, a.k.n_smp, row, s, active)) return;
    if constexpr (OP == kOpFan) {
        typedef AdjCol<UNIFORM, BETA, VW> Col;
        double y[1][3][VW];
        fan_product<UNIFORM, VW>(a.k, Col{a, static_cast<uint32_t>(s) * 8u}, row, y);
        adj_finish<DAMP, VW>(a, row, s, active, y[0]);
        return;
    }
    double acc[3][VW];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int v = 0; v < VW; ++v) acc[i][v] = 0.0;
    for (int32_t p = a.k.indptr[row]; p < a.k.indptr[row + 1]; ++p) {
        const int64_t col = a.k.indices[p];
        double x[3][VW];
        adj_column<BETA, VW>(a, col, s, x);
        block_apply<OP, VW>(a.k, p, static_cast<int>(col) - row, s, x, acc);
    }
    adj_finish<DAMP, VW>(a, row, s, active, acc);
}

// The adjoint step on the symmetric storage with row records (sym_product; the bits are those of
// k_adjoint_step<kOpSym>).
template <bool UNIFORM, bool BETA, bool DAMP, int VW>
__global__ __launch_bounds__(kBlock) void k_adjoint_symrec(AdjArgs a, const int32_t *__restrict__ rec) {
    int32_t row;
    int64_t s;
    bool active;
    if (!row_and_sample<UNIFORM, VW>(a.k.n_nodes, a.k.n_smp, row, s, active)) return;
    const int32_t *r = rec + static_cast<int64_t>(row) * (2 + 2 * kRecordSlots);
    row = r[0];
    double acc[1][3][VW];
    sym_product<UNIFORM, VW>(a.k, r, AdjCol<UNIFORM, BETA, VW>{a, static_cast<uint32_t>(s) * 8u}, row, acc);
    adj_finish<DAMP, VW>(a, row, s, active, acc[0]);
}

// The matrix-free adjoint step by node tiles (tile.h); the bits are those of k_adjoint_step<kOpFan>.
template <bool BETA, bool DAMP, int VW, int ELEMS, bool SMALL>
__global__ __launch_bounds__(kTileThreads) __attribute__((amdgpu_waves_per_eu(4)))
void k_adjoint_tile(AdjArgs a, TileArgs t) {
    TilePlace p;
    if (!tile_place<VW>(t, a.k.n_smp, static_cast<uint32_t>(xcd_block()), p)) return;
    typedef AdjCol<false, BETA, VW> Col;
    const Col col{a, static_cast<uint32_t>(p.s) * 8u};
    double acc[3][VW];
    typename Col::Own own;
    tile_product<ELEMS, VW, SMALL>(a.k, t, col, p.tile, p.i, p.l, p.in, p.rw, acc,
                            [&](int32_t node) { own = col.own(node); });
    if (p.active) adj_finish<DAMP, VW>(a, p.rw.x, p.s, true, acc, own.m1, own.m2);
}

// One forward step (the generic row kernel's operations) and one adjoint step in a single pass
// over the operator: each block (stored values, or element coefficients and unit blocks) is
// loaded once and applied to both the forward column u + bdt (u - up) and the adjoint column
// dt^2/m (b1 mu1 - b0 mu2).  The products and updates are the operations of k_step and
// k_adjoint_step in the same order, so both outputs equal those of the separate launches bit for
// bit.  The forward and the adjoint may be at different time steps (the reverse sweep of one
// checkpoint segment runs with the recomputation of the segment before it).  (A register target
// of 5 waves per SIMD, 94 VGPRs instead of 100 for the stored two-sample instance, measured 2-3 %
// slower: the loads in flight per wave count for more here.)  By fan entries see fan_as_two.
template <int OP, bool UNIFORM, bool BETA, bool DAMP, int VW>
__global__ __launch_bounds__(kBlock) void k_fused_step(StepArgs f, AdjArgs a, int64_t step) {
    int32_t row;
    int64_t s;
    bool active;
    if (!row_and_sample<UNIFORM, VW>(f.k.n_nodes, f.k.n_smp, row, s, active)) return;
    if constexpr (OP == kOpFan) {
        const uint32_t lane = static_cast<uint32_t>(s) * 8u;
        typedef FusedCol<UNIFORM, BETA, VW> Col;
        const Col col{{f.u, f.up, f.bdt, f.k.n_smp, lane}, {a, lane}, lane};
        double y[2][3][VW];
        fan_product<UNIFORM, VW>(f.k, col, row, y);
        step_update<DAMP, VW>(f, row, s, active, step, y[0]);
        adj_finish<DAMP, VW>(a, row, s, active, y[1]);
        return;
    }
    double accf[3][VW], acca[3][VW];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int v = 0; v < VW; ++v) accf[i][v] = acca[i][v] = 0.0;
    for (int32_t p = f.k.indptr[row]; p < f.k.indptr[row + 1]; ++p) {
        const int64_t col = f.k.indices[p];
        double xf[3][VW], xa[3][VW];
        state_column<BETA, VW>(f.u, f.up, f.bdt, col, f.k.n_smp, s, xf);
        adj_column<BETA, VW>(a, col, s, xa);
        block_apply2<OP, VW>(f.k, p, static_cast<int>(col) - row, s, xf, accf, xa, acca);
    }
    step_update<DAMP, VW>(f, row, s, active, step, accf);
    adj_finish<DAMP, VW>(a, row, s, active, acca);
}

// The fused step on the symmetric storage with row records (the bits are those of
// k_fused_step<kOpSym>).
template <bool UNIFORM, bool BETA, bool DAMP, int VW>
__global__ __launch_bounds__(kBlock) void k_fused_symrec(StepArgs f, AdjArgs a, const int32_t *__restrict__ rec,
                                                        int64_t step) {
    int32_t row;
    int64_t s;
    bool active;
    if (!row_and_sample<UNIFORM, VW>(f.k.n_nodes, f.k.n_smp, row, s, active)) return;
    const int32_t *r = rec + static_cast<int64_t>(row) * (2 + 2 * kRecordSlots);
    row = r[0];
    const uint32_t lane = static_cast<uint32_t>(s) * 8u;
    const FusedCol<UNIFORM, BETA, VW> col{{f.u, f.up, f.bdt, f.k.n_smp, lane}, {a, lane}, lane};
    double acc[2][3][VW];
    sym_product<UNIFORM, VW>(f.k, r, col, row, acc);
    step_update<DAMP, VW>(f, row, s, active, step, acc[0]);
    adj_finish<DAMP, VW>(a, row, s, active, acc[1]);
}

struct GradArgs {
    int64_t n_elms, n_smp;
    const int32_t *elems, *cpos;
    const double *khat, *coef, *lm;
    int64_t lm_sstride;
    const double *minv;    // 1/lm (0 where lm = 0), same layout; NULL = divide by lm
    const double *mu, *xc, *xp;
    double bdt, nu_scale;
    double *grad;
};

// sum_{a,b} nu_a^T khat_e(a,b) x_b over the element's nodes, by the vectors relative to its node 0:
// an element's rows and columns sum to zero and its block is symmetric, so three of the nine 3 x 3
// unit blocks, (1,1), (1,2) and (2,2), 27 of the 81 entries, hold the form.
constexpr int kGradKh = 27;

__device__ __forceinline__ int grad_block(int r) { return r < 9 ? 4 : (r < 18 ? 5 : 8); }

template <int VW, class KH>
__device__ __forceinline__ void grad_form(const double (&nu)[2][3][VW], const double (&x)[2][3][VW], KH kh,
                                          double (&acc)[VW]) {
    double y[2][3][VW];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int v = 0; v < VW; ++v) y[0][i][v] = y[1][i][v] = 0.0;
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const double pp = kh(3 * i + j), pq = kh(9 + 3 * i + j), qq = kh(18 + 3 * i + j);
#pragma unroll
            for (int v = 0; v < VW; ++v) {
                y[0][i][v] = fma(pp, x[0][j][v], y[0][i][v]);
                y[0][i][v] = fma(pq, x[1][j][v], y[0][i][v]);
                y[1][i][v] = fma(qq, x[1][j][v], y[1][i][v]);
                y[1][j][v] = fma(pq, x[0][i][v], y[1][j][v]);
            }
        }
#pragma unroll
    for (int v = 0; v < VW; ++v) {
        acc[v] = 0.0;
#pragma unroll
        for (int i = 0; i < 3; ++i) acc[v] = fma(nu[0][i][v], y[0][i][v], fma(nu[1][i][v], y[1][i][v], acc[v]));
    }
}

// The same with all nine blocks and the vectors as they are: a system without fan entries makes no claim
// on its unit blocks.  Entry (3 p + b, 3 i + j) of the element's block is kh(9 (3 p + b) + 3 i + j).
constexpr int kGradAll = 81;

template <int VW, class KH>
__device__ __forceinline__ void grad_form_all(const double (&nu)[3][3][VW], const double (&x)[3][3][VW], KH kh,
                                              double (&acc)[VW]) {
#pragma unroll
    for (int v = 0; v < VW; ++v) acc[v] = 0.0;
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            double t[VW] = {};
#pragma unroll
            for (int b = 0; b < 3; ++b)
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    const double h = kh(9 * (3 * p + b) + 3 * i + j);
#pragma unroll
                    for (int v = 0; v < VW; ++v) t[v] = fma(h, x[b][j][v], t[v]);
                }
#pragma unroll
            for (int v = 0; v < VW; ++v) acc[v] = fma(nu[p][i][v], t[v], acc[v]);
        }
}

__device__ __forceinline__ double grad_scale(const GradArgs &a, double m) {
    return a.minv ? a.nu_scale * m : (m != 0.0 ? a.nu_scale / m : 0.0);
}

// grad[e,s] = fma(-coef[e,s], sum_{a,b} nu_a^T khat_e(a,b) x_b, grad[e,s]) for the lane's element e
// and VW samples at s, with nu = nu_scale * mu / m (nu_scale * minv with the inverse masses) and
// x = xc + bdt (xc - xp) (PREV; else x = xc).  `sc` holds nu_scale / m of the three nodes where the
// mass has no sample axis.  All loads are issued before the first is used.
template <bool PREV, bool LMS, int VW, bool ALL = false, class KH>
__device__ __forceinline__ void grad_update(const GradArgs &a, int64_t e, int64_t s, const int32_t (&ids)[3],
                                            const double (&sc)[3], KH kh) {
    Vec<VW> mu[3][3], c[3][3], p[3][3], m[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const int64_t nd = ids[q];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const int64_t off = (nd * 3 + j) * a.n_smp + s;
            mu[q][j] = load_vec<VW>(a.mu + off);
            c[q][j] = load_vec<VW>(a.xc + off);
            if constexpr (PREV) p[q][j] = load_vec<VW>(a.xp + off);
        }
        if constexpr (LMS) m[q] = load_vec<VW>((a.minv ? a.minv : a.lm) + nd * a.n_smp + s);
    }
    const int64_t idx = e * a.n_smp + s;
    const Vec<VW> cf = load_vec<VW>(a.coef + idx);
    Vec<VW> g = load_vec<VW>(a.grad + idx);
    __builtin_amdgcn_sched_barrier(0);
    double f[VW];
    if constexpr (ALL) {
        double nu[3][3][VW], x[3][3][VW];
#pragma unroll
        for (int q = 0; q < 3; ++q)
#pragma unroll
            for (int v = 0; v < VW; ++v) {
                const double scale = LMS ? grad_scale(a, m[q].v[v]) : sc[q];
#pragma unroll
                for (int j = 0; j < 3; ++j) {
                    const double u = c[q][j].v[v];
                    nu[q][j][v] = scale * mu[q][j].v[v];
                    x[q][j][v] = PREV ? fma(a.bdt, u - p[q][j].v[v], u) : u;
                }
            }
        grad_form_all<VW>(nu, x, kh, f);
#pragma unroll
        for (int v = 0; v < VW; ++v) g.v[v] = fma(-cf.v[v], f[v], g.v[v]);
        store_vec<VW>(a.grad + idx, g);
        return;
    }
    double nu0[3][VW], x0[3][VW], dn[2][3][VW], dx[2][3][VW];
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
        for (int v = 0; v < VW; ++v) {
            const double scale = LMS ? grad_scale(a, m[q].v[v]) : sc[q];
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                // products and differences as written, so that every form gives the same bits
                const double u = c[q][j].v[v], x = PREV ? fma(a.bdt, u - p[q][j].v[v], u) : u;
                if (q == 0) {
                    nu0[j][v] = scale * mu[q][j].v[v];
                    x0[j][v] = x;
                } else {
                    dn[q - 1][j][v] = fma(scale, mu[q][j].v[v], -nu0[j][v]);
                    dx[q - 1][j][v] = x - x0[j][v];
                }
            }
        }
    grad_form<VW>(dn, dx, kh, f);
#pragma unroll
    for (int v = 0; v < VW; ++v) g.v[v] = fma(-cf.v[v], f[v], g.v[v]);
    store_vec<VW>(a.grad + idx, g);
}

// Sample counts that are multiples of 128: each wave one element and 128 of its samples, two per
// lane.  What the samples share, node ids, node scales and unit blocks, comes in by one vector load
// each (lane r the r-th entry) and is broadcast from the registers: scalar loads of 648 B an element
// missed their cache ten times each and bound the kernel.  Waves run sample group first (all
// elements for samples 0-127, then 128-255, ...), which keeps the gathered node data of one group in
// L2 between the elements that share it.  The gather bounds it: the address unit takes a vector
// load's lanes at 4 a clock whatever their width, hence 16 bytes each.
template <bool PREV, bool LMS>
__global__ __launch_bounds__(kBlock) void k_grad_accum(GradArgs a) {
    const uint32_t w = static_cast<uint32_t>(xcd_block() * kBlock + threadIdx.x) >> 6;
    const uint32_t group = w / static_cast<uint32_t>(a.n_elms);
    if (group >= a.n_smp / 128) return;
    const int64_t e = __builtin_amdgcn_readfirstlane(static_cast<int32_t>(w - group * static_cast<uint32_t>(a.n_elms)));
    const int lane = threadIdx.x & 63;
    const int64_t s = (static_cast<int64_t>(group) * 64 + lane) * 2;
    const int r = lane < kGradKh ? lane : 0;
    const int32_t id = a.elems[3 * e + (lane < 3 ? lane : 0)];
    const double kh = a.khat[9 * static_cast<int64_t>(a.cpos[9 * e + grad_block(r)]) + r % 9];
    const double m = LMS ? 1.0 : grad_scale(a, (a.minv ? a.minv : a.lm)[id]);
    int32_t ids[3];
    double sc[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        ids[q] = __builtin_amdgcn_readlane(id, q);
        sc[q] = lane_value(m, q);
    }
    grad_update<PREV, LMS, 2>(a, e, s, ids, sc, [&](int i) { return lane_value(kh, i); });
}

// Any other sample count: lanes packed, VW samples of one element each, the ids, scales and unit
// blocks of the workgroup's elements staged in LDS first.  Two samples per lane for even counts from
// kGradPair (a workgroup then still has at most kGradElems elements; four waves per SIMD: a fifth
// waits on fewer registers, 56 us), one from kGradMin.  98,304 elements x 32 samples: 80 -> 52 us;
// 65,536 x 64 with the damped state: 114 -> 72 us (one wave an element with one sample per lane 89).
constexpr int kGradMin = 8, kGradPair = 16;
constexpr int kGradElems = (kBlock - 1) / kGradMin + 2;   // 33

template <bool PREV, bool LMS, int VW, bool ALL = false>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(VW == 2 && !LMS && !ALL ? 4 : 1))) void
k_grad_accum_lds(GradArgs a) {
    constexpr int KH = ALL ? kGradAll : kGradKh;
    __shared__ double sk[kGradElems * KH];
    __shared__ double ssc[kGradElems * 3];
    __shared__ int32_t sid[kGradElems * 3];
    const uint32_t lpr = static_cast<uint32_t>(a.n_smp / VW), g0 = static_cast<uint32_t>(xcd_block() * kBlock);
    const uint32_t e0 = g0 / lpr;
    uint32_t e1 = (g0 + (kBlock - 1)) / lpr;
    if (e1 >= a.n_elms) e1 = static_cast<uint32_t>(a.n_elms) - 1;
    const int nel = e0 <= e1 ? static_cast<int>(e1 - e0 + 1) : 0;    // <= kGradElems
    for (int q = threadIdx.x; q < nel * 3; q += kBlock) {
        const int32_t id = a.elems[3 * static_cast<int64_t>(e0) + q];
        sid[q] = id;
        ssc[q] = LMS ? 1.0 : grad_scale(a, (a.minv ? a.minv : a.lm)[id]);
    }
    for (int q = threadIdx.x; q < nel * KH; q += kBlock) {
        const int le = q / KH, r = q - le * KH;
        const int block = ALL ? r / 9 : grad_block(r);
        sk[q] = a.khat[9 * static_cast<int64_t>(a.cpos[9 * static_cast<int64_t>(e0 + le) + block]) + r % 9];
    }
    __syncthreads();
    const uint32_t g = g0 + threadIdx.x, e = g / lpr;
    if (e >= a.n_elms) return;
    const int le = static_cast<int>(e - e0);
    const int32_t ids[3] = {sid[3 * le], sid[3 * le + 1], sid[3 * le + 2]};
    const double sc[3] = {ssc[3 * le], ssc[3 * le + 1], ssc[3 * le + 2]};
    grad_update<PREV, LMS, VW, ALL>(a, e, static_cast<int64_t>(g - e * lpr) * VW, ids, sc,
                                    [&](int i) { return sk[KH * le + i]; });
}

// Fewer than 8 samples: everything read per lane.
template <bool PREV, bool LMS, bool ALL = false>
__global__ __launch_bounds__(kBlock) void k_grad_accum_lane(GradArgs a) {
    const int64_t g = xcd_block() * kBlock + threadIdx.x;
    if (g >= a.n_elms * a.n_smp) return;
    const int64_t e = g / a.n_smp;
    const int32_t ids[3] = {a.elems[3 * e], a.elems[3 * e + 1], a.elems[3 * e + 2]};
    constexpr int BLOCKS = ALL ? 9 : 3;
    double sc[3];
    const double *kh[BLOCKS];
#pragma unroll
    for (int q = 0; q < 3; ++q) sc[q] = LMS ? 1.0 : grad_scale(a, (a.minv ? a.minv : a.lm)[ids[q]]);
#pragma unroll
    for (int q = 0; q < BLOCKS; ++q)
        kh[q] = a.khat + 9 * static_cast<int64_t>(a.cpos[9 * e + (ALL ? q : grad_block(9 * q))]);
    grad_update<PREV, LMS, 1, ALL>(a, e, g - e * a.n_smp, ids, sc, [&](int i) { return kh[i / 9][i % 9]; });
}

template <int MF, bool UNI, int VW>
void adj_launch(hipStream_t st, const AdjArgs &a, bool beta, bool damp) {
    const dim3 g(grid_for(a.k.n_nodes * lanes_per_row<UNI, VW>(a.k.n_smp))), b(kBlock);
    if (beta) {
        if (damp) hipLaunchKernelGGL((k_adjoint_step<MF, UNI, true, true, VW>), g, b, a.occ_lds, st, a);
        else hipLaunchKernelGGL((k_adjoint_step<MF, UNI, true, false, VW>), g, b, a.occ_lds, st, a);
    } else {
        if (damp) hipLaunchKernelGGL((k_adjoint_step<MF, UNI, false, true, VW>), g, b, a.occ_lds, st, a);
        else hipLaunchKernelGGL((k_adjoint_step<MF, UNI, false, false, VW>), g, b, a.occ_lds, st, a);
    }
}

template <int VW, int ELEMS, bool SMALL>
void adj_tile_launch(hipStream_t st, const AdjArgs &a, const TileArgs &t, const TileShape &h, bool beta,
                     bool damp) {
    const dim3 g(tile_grid(t)), b(64 * h.waves);
    const size_t lds = tile_lds(h.chunk, ELEMS);
    if (beta) {
        if (damp) hipLaunchKernelGGL((k_adjoint_tile<true, true, VW, ELEMS, SMALL>), g, b, lds, st, a, t);
        else hipLaunchKernelGGL((k_adjoint_tile<true, false, VW, ELEMS, SMALL>), g, b, lds, st, a, t);
    } else {
        if (damp) hipLaunchKernelGGL((k_adjoint_tile<false, true, VW, ELEMS, SMALL>), g, b, lds, st, a, t);
        else hipLaunchKernelGGL((k_adjoint_tile<false, false, VW, ELEMS, SMALL>), g, b, lds, st, a, t);
    }
}

void adj_tile(hipStream_t st, const cvfes_system_t *sys, const AdjArgs &a, bool beta, bool damp) {
    const TileShape h = tile_shape(sys->n_smp);
    const TileArgs t = tile_args(sys, h);
    const bool six = sys->max_node_elems <= 6, small = sys->n_smp <= kTileSmall;
    if (h.vw == 2) {
        if (small) {
            if (six) adj_tile_launch<2, 6, true>(st, a, t, h, beta, damp);
            else adj_tile_launch<2, 8, true>(st, a, t, h, beta, damp);
        } else {
            if (six) adj_tile_launch<2, 6, false>(st, a, t, h, beta, damp);
            else adj_tile_launch<2, 8, false>(st, a, t, h, beta, damp);
        }
    } else {
        if (small) {
            if (six) adj_tile_launch<1, 6, true>(st, a, t, h, beta, damp);
            else adj_tile_launch<1, 8, true>(st, a, t, h, beta, damp);
        } else {
            if (six) adj_tile_launch<1, 6, false>(st, a, t, h, beta, damp);
            else adj_tile_launch<1, 8, false>(st, a, t, h, beta, damp);
        }
    }
}

// Lane width and row mapping as the generic forward kernel chooses them (generic_vw; wave-uniform
// rows when they keep 3/4 of the lanes busy).
template <int MF>
void adj_dispatch(hipStream_t st, const AdjArgs &a, bool beta, bool damp) {
    if (generic_vw(a.k.n_smp) == 2) {
        if (use_uniform<2>(a.k.n_smp)) adj_launch<MF, true, 2>(st, a, beta, damp);
        else adj_launch<MF, false, 2>(st, a, beta, damp);
    } else {
        if (use_uniform<1>(a.k.n_smp)) adj_launch<MF, true, 1>(st, a, beta, damp);
        else adj_launch<MF, false, 1>(st, a, beta, damp);
    }
}

template <bool UNI, int VW>
void adj_symrec_launch(hipStream_t st, const AdjArgs &a, const int32_t *rec, bool beta, bool damp) {
    const dim3 g(grid_for(a.k.n_nodes * lanes_per_row<UNI, VW>(a.k.n_smp))), b(kBlock);
    if (beta) {
        if (damp) hipLaunchKernelGGL((k_adjoint_symrec<UNI, true, true, VW>), g, b, a.occ_lds, st, a, rec);
        else hipLaunchKernelGGL((k_adjoint_symrec<UNI, true, false, VW>), g, b, a.occ_lds, st, a, rec);
    } else {
        if (damp) hipLaunchKernelGGL((k_adjoint_symrec<UNI, false, true, VW>), g, b, a.occ_lds, st, a, rec);
        else hipLaunchKernelGGL((k_adjoint_symrec<UNI, false, false, VW>), g, b, a.occ_lds, st, a, rec);
    }
}

template <bool UNI, int VW>
void fused_symrec_launch(hipStream_t st, const StepArgs &f, const AdjArgs &a, const int32_t *rec, bool beta,
                         bool damp) {
    const dim3 g(grid_for(f.k.n_nodes * lanes_per_row<UNI, VW>(f.k.n_smp))), b(kBlock);
    const int64_t step = 0;
    if (beta) {
        if (damp) hipLaunchKernelGGL((k_fused_symrec<UNI, true, true, VW>), g, b, f.occ_lds, st, f, a, rec, step);
        else hipLaunchKernelGGL((k_fused_symrec<UNI, true, false, VW>), g, b, f.occ_lds, st, f, a, rec, step);
    } else {
        if (damp) hipLaunchKernelGGL((k_fused_symrec<UNI, false, true, VW>), g, b, f.occ_lds, st, f, a, rec, step);
        else hipLaunchKernelGGL((k_fused_symrec<UNI, false, false, VW>), g, b, f.occ_lds, st, f, a, rec, step);
    }
}

// The adjoint step by row records, for the sample counts that use_records leaves it.
void adj_symrec(hipStream_t st, const AdjArgs &a, const int32_t *rec, bool beta, bool damp) {
    const int64_t S = a.k.n_smp;
    if (generic_vw(S) == 1) adj_symrec_launch<false, 1>(st, a, rec, beta, damp);
    else if (use_uniform<2>(S)) adj_symrec_launch<true, 2>(st, a, rec, beta, damp);
    else adj_symrec_launch<false, 2>(st, a, rec, beta, damp);
}

// The same fused with the forward step f.
void fused_symrec(hipStream_t st, const StepArgs &f, const AdjArgs &a, const int32_t *rec, bool beta, bool damp) {
    const int64_t S = a.k.n_smp;
    if (generic_vw(S) == 2) {
        if (use_uniform<2>(S)) fused_symrec_launch<true, 2>(st, f, a, rec, beta, damp);
        else fused_symrec_launch<false, 2>(st, f, a, rec, beta, damp);
    } else {
        if (use_uniform<1>(S)) fused_symrec_launch<true, 1>(st, f, a, rec, beta, damp);
        else fused_symrec_launch<false, 1>(st, f, a, rec, beta, damp);
    }
}

template <int MF, bool UNI, int VW>
void fused_launch(hipStream_t st, const StepArgs &f, const AdjArgs &a, bool beta, bool damp) {
    const dim3 g(grid_for(f.k.n_nodes * lanes_per_row<UNI, VW>(f.k.n_smp))), b(kBlock);
    if (beta) {
        if (damp) hipLaunchKernelGGL((k_fused_step<MF, UNI, true, true, VW>), g, b, f.occ_lds, st, f, a, int64_t(0));
        else hipLaunchKernelGGL((k_fused_step<MF, UNI, true, false, VW>), g, b, f.occ_lds, st, f, a, int64_t(0));
    } else {
        if (damp) hipLaunchKernelGGL((k_fused_step<MF, UNI, false, true, VW>), g, b, f.occ_lds, st, f, a, int64_t(0));
        else hipLaunchKernelGGL((k_fused_step<MF, UNI, false, false, VW>), g, b, f.occ_lds, st, f, a, int64_t(0));
    }
}

template <int MF>
void fused_dispatch(hipStream_t st, const StepArgs &f, const AdjArgs &a, bool beta, bool damp) {
    if (generic_vw(f.k.n_smp) == 2) {
        if (use_uniform<2>(f.k.n_smp)) fused_launch<MF, true, 2>(st, f, a, beta, damp);
        else fused_launch<MF, false, 2>(st, f, a, beta, damp);
    } else {
        if (use_uniform<1>(f.k.n_smp)) fused_launch<MF, true, 1>(st, f, a, beta, damp);
        else fused_launch<MF, false, 1>(st, f, a, beta, damp);
    }
}

// Whether the fused matrix-free step runs as its two launches: with both columns of two samples the
// fan walk holds the registers of two waves per SIMD, and reading the coefficients once saves less
// than that costs (16,384 nodes of a regular / irregular wall, fused against step + adjoint: 128 samples
// 130 / 141 against 85 / 97 us, 200 239 / 256 against 196 / 207; the walk over blocks took 139 / 131
// and 206 / 213).  Small systems are bound by the launches themselves (600 nodes x 128: 9.4 against
// 14.1 us, 96 x 2,048: 13.7 against 15.4, 2,052 x 128: 21.6 against 21.8).
bool fan_as_two(const cvfes_system_t *sys) {
    return generic_vw(sys->n_smp) == 2 && use_uniform<2>(sys->n_smp) && sys->n_nodes * sys->n_smp >= (1 << 18);
}

void launch_adjoint_fan(hipStream_t st, const cvfes_system_t *sys, const AdjArgs &a, bool beta, bool damp) {
    if (tiles_apply(sys)) adj_tile(st, sys, a, beta, damp);
    else adj_dispatch<kOpFan>(st, a, beta, damp);
}

// Operator form of the generic row kernels for this system and method (as the forward step's
// generic kernel chooses it: full values when present, else the symmetric upper blocks).
int operator_form(const cvfes_system_t *sys, int method) {
    if (method == CVFES_METHOD_MATFREE) return fan_entries(sys) ? kOpFan : kOpMatfree;
    return sys->values ? kOpStored : kOpSym;
}

int check_adjoint_args(const cvfes_system_t *sys, int method, const double *mu1, const double *mu2,
                       const double *mu_out, double dt, const char *who) {
    CVFES_REQUIRE(sys && sys->indptr && sys->indices && sys->n_nodes >= 1 && sys->n_smp >= 1,
                  "%s: empty system", who);
    CVFES_REQUIRE(method == CVFES_METHOD_STORED || method == CVFES_METHOD_MATFREE,
                  "%s: unknown method %d", who, method);
    CVFES_REQUIRE(method == CVFES_METHOD_MATFREE || sys->values || (sys->uvalues && sys->vblk),
                  "%s: no stored values (full or symmetric)", who);
    CVFES_REQUIRE(method == CVFES_METHOD_STORED || (sys->cptr && sys->celem && sys->khat && sys->coef),
                  "%s: matrix-free needs cptr/celem/khat/coef", who);
    CVFES_REQUIRE(mu1 && mu2 && mu_out && sys->lm, "%s: null pointer", who);
    CVFES_REQUIRE(mu_out != mu1 && mu_out != mu2, "%s: output aliases an input", who);
    CVFES_REQUIRE(dt > 0.0, "%s: dt must be positive", who);
    CVFES_REQUIRE(sys->waves_per_simd == 0 || (sys->waves_per_simd >= 2 && sys->waves_per_simd <= 7),
                  "%s: waves_per_simd must be 0 or 2..7", who);
    return CVFES_OK;
}

AdjArgs adjoint_args(const cvfes_system_t *sys, const double *mu1, const double *mu2, double *mu_out,
                     const double *obs_u, const double *obs_ref, const double *obs_w, double dt,
                     double beta, double damp, int project) {
    AdjArgs a{};
    a.k = RowArgs{sys->n_nodes, sys->n_smp, sys->indptr, sys->indices, sys->values,
                  sys->cptr, sys->celem, sys->khat, sys->coef, sys->uvalues, sys->vblk,
                  sys->nptr, fan_entries(sys)};
    a.mu1 = mu1;
    a.mu2 = mu2;
    a.out = mu_out;
    a.lm = sys->lm;
    a.lm_sstride = sys->lm_sstride;
    a.minv = sys->minv;
    a.fixed = sys->fixed;
    a.obs_u = obs_u;
    a.obs_ref = obs_ref;
    a.obs_w = obs_w;
    a.dt2 = dt * dt;
    a.bdt = beta / dt;
    a.dtdamp = dt * damp;
    a.project = project;
    a.occ_lds = occupancy_lds(sys->waves_per_simd);
    a.nt_out = stream_out(sys->n_nodes, sys->n_smp);
    return a;
}

// minv[i] = 1 / lm[i], 0 where lm[i] = 0.
__global__ __launch_bounds__(kBlock) void k_inverse_mass(int64_t n, const double *__restrict__ lm,
                                                         double *__restrict__ minv) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (i < n) minv[i] = lm[i] != 0.0 ? 1.0 / lm[i] : 0.0;
}
}  // namespace
}  // namespace cvfes

using namespace cvfes;

extern "C" int cvfes_adjoint_step(void *stream, const cvfes_system_t *sys, int method,
                                  const double *mu1, const double *mu2, double *mu_out,
                                  const double *obs_u, const double *obs_ref, const double *obs_w,
                                  double dt, double beta, double damp, int project) {
    if (int rc = check_adjoint_args(sys, method, mu1, mu2, mu_out, dt, "cvfes_adjoint_step")) return rc;
    const AdjArgs a = adjoint_args(sys, mu1, mu2, mu_out, obs_u, obs_ref, obs_w, dt, beta, damp, project);
    hipStream_t st = static_cast<hipStream_t>(stream);
    switch (operator_form(sys, method)) {
    case kOpFan: launch_adjoint_fan(st, sys, a, beta != 0.0, damp != 0.0); break;
    case kOpMatfree: adj_dispatch<kOpMatfree>(st, a, beta != 0.0, damp != 0.0); break;
    case kOpStored: adj_dispatch<kOpStored>(st, a, beta != 0.0, damp != 0.0); break;
    default:
        if (use_records(sys, true)) adj_symrec(st, a, sys->row_records, beta != 0.0, damp != 0.0);
        else adj_dispatch<kOpSym>(st, a, beta != 0.0, damp != 0.0);
        break;
    }
    return check_launch("k_adjoint_step");
}

extern "C" int cvfes_adjoint_fused_step(void *stream, const cvfes_system_t *sys, int method,
                                        double *const *state, const cvfes_load_t *load,
                                        const double *mu1, const double *mu2, double *mu_out,
                                        const double *obs_u, const double *obs_ref,
                                        const double *obs_w, double dt, double beta, double damp) {
    if (int rc = check_adjoint_args(sys, method, mu1, mu2, mu_out, dt, "cvfes_adjoint_fused_step"))
        return rc;
    CVFES_REQUIRE(state && state[0] && state[1] && state[2], "cvfes_adjoint_fused_step: null state buffer");
    const double *bufs[6] = {state[0], state[1], state[2], mu1, mu2, mu_out};
    for (int i = 0; i < 6; ++i)
        for (int j = i + 1; j < 6; ++j)
            CVFES_REQUIRE(bufs[i] != bufs[j] || (i == 3 && j == 4),
                          "cvfes_adjoint_fused_step: state and adjoint buffers must be distinct");
    CVFES_REQUIRE(sys->f1 && load && load->p && (!load->ga || load->qa) && (!load->gb || load->qb),
                  "cvfes_adjoint_fused_step: load tables");
    CVFES_REQUIRE(sys->lm_sstride == 0 || sys->lm_sstride == 1, "cvfes_adjoint_fused_step: lm_sstride");
    const int64_t kern = cvfes_step_kernel(sys, method);
    CVFES_REQUIRE(kern == CVFES_VARIANT_GENERIC,
                  "cvfes_adjoint_fused_step: the forward step of this system runs kernel variant "
                  "%lld, not the generic one the fused kernel replays",
                  static_cast<long long>(kern));
    StepArgs f{};
    f.k = RowArgs{sys->n_nodes, sys->n_smp, sys->indptr, sys->indices, sys->values,
                  sys->cptr, sys->celem, sys->khat, sys->coef, sys->uvalues, sys->vblk,
                  sys->nptr, fan_entries(sys)};
    f.u = state[0];
    f.up = state[1];
    f.out = state[2];
    f.lm = sys->lm;
    f.lm_sstride = sys->lm_sstride;
    f.f1 = sys->f1;
    f.fixed = sys->fixed;
    f.load = *load;
    f.bdy_u = sys->bdy_u;
    f.dt2 = dt * dt;
    f.bdt = beta / dt;
    f.ddt = damp / dt;
    f.order = nullptr;
    f.occ_lds = occupancy_lds(sys->waves_per_simd);
    f.nt_out = stream_out(sys->n_nodes, sys->n_smp);
    const AdjArgs a = adjoint_args(sys, mu1, mu2, mu_out, obs_u, obs_ref, obs_w, dt, beta, damp, 1);
    hipStream_t st = static_cast<hipStream_t>(stream);
    switch (operator_form(sys, method)) {
    case kOpFan:
        if (fan_as_two(sys)) {
            launch_matfree_step(st, sys, f, beta != 0.0, damp != 0.0);
            launch_adjoint_fan(st, sys, a, beta != 0.0, damp != 0.0);
        } else {
            fused_dispatch<kOpFan>(st, f, a, beta != 0.0, damp != 0.0);
        }
        break;
    case kOpMatfree: fused_dispatch<kOpMatfree>(st, f, a, beta != 0.0, damp != 0.0); break;
    case kOpStored: fused_dispatch<kOpStored>(st, f, a, beta != 0.0, damp != 0.0); break;
    default:
        if (use_records(sys)) fused_symrec(st, f, a, sys->row_records, beta != 0.0, damp != 0.0);
        else fused_dispatch<kOpSym>(st, f, a, beta != 0.0, damp != 0.0);
        break;
    }
    return check_launch("k_fused_step");
}

extern "C" int cvfes_grad_accum(void *stream, const cvfes_system_t *sys, const int32_t *elems,
                                const int32_t *cpos, const double *mu, const double *x_cur,
                                const double *x_prev, double dt, double beta, double nu_scale,
                                double *grad) {
    CVFES_REQUIRE(sys && sys->n_elms >= 1 && sys->n_smp >= 1, "cvfes_grad_accum: empty system");
    CVFES_REQUIRE(elems && cpos && sys->khat && sys->coef && sys->lm && mu && x_cur && grad,
                  "cvfes_grad_accum: null pointer");
    CVFES_REQUIRE(dt > 0.0, "cvfes_grad_accum: dt must be positive");
    const GradArgs a{sys->n_elms, sys->n_smp, elems, cpos, sys->khat, sys->coef, sys->lm,
                     sys->lm_sstride, sys->minv, mu, x_cur, x_prev, beta / dt, nu_scale, grad};
    const int64_t S = sys->n_smp, work = sys->n_elms * S;
    hipStream_t st = static_cast<hipStream_t>(stream);
    // two samples per lane need 16-byte alignment of every array with a sample axis
    const uintptr_t any = reinterpret_cast<uintptr_t>(mu) | reinterpret_cast<uintptr_t>(x_cur) |
                          reinterpret_cast<uintptr_t>(x_prev) | reinterpret_cast<uintptr_t>(grad) |
                          reinterpret_cast<uintptr_t>(a.coef) | reinterpret_cast<uintptr_t>(a.minv ? a.minv : a.lm);
    const bool pairs = S % 2 == 0 && any % 16 == 0;
    auto run = [&](auto prev, auto lms) {
        constexpr bool PREV = decltype(prev)::value, LMS = decltype(lms)::value;
        auto launch = [&](auto kernel, int vw) {
            hipLaunchKernelGGL(kernel, dim3(grid_for(work / vw)), dim3(kBlock), 0, st, a);
        };
        if (!sys->fan) {        // no claim on the unit blocks: all of them
            if (S >= kGradPair && pairs) launch(k_grad_accum_lds<PREV, LMS, 2, true>, 2);
            else if (S >= kGradMin) launch(k_grad_accum_lds<PREV, LMS, 1, true>, 1);
            else launch(k_grad_accum_lane<PREV, LMS, true>, 1);
        } else if (S % 128 == 0 && pairs) launch(k_grad_accum<PREV, LMS>, 2);
        else if (S >= kGradPair && pairs) launch(k_grad_accum_lds<PREV, LMS, 2>, 2);
        else if (S >= kGradMin) launch(k_grad_accum_lds<PREV, LMS, 1>, 1);
        else launch(k_grad_accum_lane<PREV, LMS>, 1);
    };
    if (x_prev) a.lm_sstride ? run(std::true_type{}, std::true_type{}) : run(std::true_type{}, std::false_type{});
    else a.lm_sstride ? run(std::false_type{}, std::true_type{}) : run(std::false_type{}, std::false_type{});
    return check_launch("k_grad_accum");
}

extern "C" int cvfes_inverse_mass(void *stream, int64_t n, const double *lm, double *minv) {
    CVFES_REQUIRE(n >= 0, "cvfes_inverse_mass: negative size");
    if (n == 0) return CVFES_OK;
    CVFES_REQUIRE(lm && minv, "cvfes_inverse_mass: null pointer");
    hipLaunchKernelGGL(k_inverse_mass, dim3(static_cast<unsigned>((n + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                       static_cast<hipStream_t>(stream), n, lm, minv);
    return check_launch("k_inverse_mass");
}
