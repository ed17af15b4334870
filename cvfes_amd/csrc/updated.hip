// Kernels on the per-sample geometry X + u_s: element stress recovery and the matrix-free step of
// the updated-geometry mode.
//
// Stress (optimizedSolidAssemble.pyx:1116-1223; physicsSolverGPUs.cl:443-589): per element and
// sample, the local strain B T u_e of the constant-strain triangle on the geometry X + ug_s, the
// local stress E D B T u_e (D the 5x5 membrane + transverse-shear matrix / (1 - nu^2)) as the
// symmetric tensor [[s0, s2, s3], [s2, s1, s4], [s3, s4, 0]], rotated to global axes T^T S T;
// output (xx, yy, xy, xz, yz) as stress[e][c][s].
//
// Updated-geometry step (physicsSolver.py:294-324 with optimizedSolidAssemble.pyx:710-819, the
// K(X+u) product of physicsSolverSDampGPUs.cl:232-391): the stiffness and the unit-traction load are
// those of the geometry X + ug_s, where ug is the displacement at the last re-formation.  Nothing
// is stored: each thread owns one (row node, sample), walks the elements incident to the node,
// forms each element's frame on the moved geometry and applies its three blocks in the local
// frame, T^T (k_ab (T x_b)), so the matrix is never formed.  The update of u is the fused
// central-difference update of the linear step.
#include "geometry.h"
#include "rowops.h"

namespace cvfes {
namespace {

struct GeomArgs {
    const double *nodes;     // [N][3] reference coordinates
    const int32_t *elems;    // [E][3]
    const double *ug;        // [N][3][S] geometry displacement (null: reference geometry)
    const int32_t *nptr;     // [N+1]
    const int32_t *nent;     // [3E]
    double nu, g, gk, inv_1mnu2;
    const fan_t *fan;        // [3E] (rowops.h); null: the elements are walked by nent
    const int32_t *head;     // [n_rows][4] the rows in the order of the node tiles (tile.h), -1: none;
    int64_t n_rows;          // null: in natural order
};

__device__ __forceinline__ void moved_points(const GeomArgs &g, const int32_t (&ids)[3], int64_t S,
                                             int64_t s, double (&X)[3][3]) {
#pragma unroll
    for (int b = 0; b < 3; ++b)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            X[b][k] = g.nodes[3 * static_cast<int64_t>(ids[b]) + k];
            if (g.ug) X[b][k] += g.ug[(static_cast<int64_t>(ids[b]) * 3 + k) * S + s];
        }
}

// FAST: reciprocal-normalised frames and one reciprocal for the element scale (results within a few
// ulp of the divided forms).  GEO_U: the geometry displacement is the current u (interval 1), so
// each node's u is loaded once for the geometry and the product.  VW samples per lane.
template <bool UNIFORM, bool BETA, bool DAMP, bool FAST, bool GEO_U, int VW>
__global__ __launch_bounds__(kBlock) void k_step_updated(StepArgs a, GeomArgs g, int64_t step) {
    int32_t row;
    int64_t s;
    bool active;
    if (!row_and_sample<UNIFORM, VW>(a.k.n_nodes, a.k.n_smp, row, s, active)) return;
    const int64_t S = a.k.n_smp;
    const uint32_t lo = static_cast<uint32_t>(s) * 8u;   // the lane's byte offset in every row
    const uint32_t sb = static_cast<uint32_t>(S) * 8u;   // bytes of one entry across the samples
    double acc[VW][3] = {};
    double fl[VW][3] = {};    // unit-traction load of the row node on the moved geometry
    for (int32_t q = g.nptr[row]; q < g.nptr[row + 1]; ++q) {
        const int32_t ent = g.nent[q];
        const int32_t e = ent / 3;
        const int la = ent - 3 * e;
        const int32_t ids[3] = {g.elems[3 * e], g.elems[3 * e + 1], g.elems[3 * e + 2]};
        double ref[3][3];
#pragma unroll
        for (int b = 0; b < 3; ++b)
#pragma unroll
            for (int k = 0; k < 3; ++k) ref[b][k] = g.nodes[3 * static_cast<int64_t>(ids[b]) + k];
        // per-sample state of the element's nodes: u (and up), the geometry displacement
        // (wave-uniform rows: buffer loads from scalar resources per node, one per-lane offset)
        double xu[VW][3][3], xg[VW][3][3];
#pragma unroll
        for (int b = 0; b < 3; ++b)
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const int64_t off = (static_cast<int64_t>(ids[b]) * 3 + k) * S + s;
                Vec<VW> uu, pp, gg;
                if constexpr (UNIFORM) {
                    const int64_t node = static_cast<int64_t>(ids[b]) * 3 * S;
                    uu = to_vec<VW>(ldb<VW, 0>(buffer_rsrc(a.u + node, 3 * sb), lo, k * sb));
                    if constexpr (BETA)
                        pp = to_vec<VW>(ldb<VW, 0>(buffer_rsrc(a.up + node, 3 * sb), lo, k * sb));
                } else {
                    uu = load_vec<VW>(a.u + off);
                    if constexpr (BETA) pp = load_vec<VW>(a.up + off);
                }
                if constexpr (!GEO_U) {
                    if (g.ug) gg = load_vec<VW>(g.ug + off);
                }
#pragma unroll
                for (int v = 0; v < VW; ++v) {
                    xu[v][b][k] = BETA ? uu.v[v] + a.bdt * (uu.v[v] - pp.v[v]) : uu.v[v];
                    if constexpr (GEO_U) xg[v][b][k] = uu.v[v];
                    else xg[v][b][k] = g.ug ? gg.v[v] : 0.0;
                }
            }
        Vec<VW> cf;
        if constexpr (UNIFORM) cf = to_vec<VW>(ldb<VW, 0>(buffer_rsrc(a.k.coef + static_cast<int64_t>(e) * S, sb), lo, 0));
        else cf = load_vec<VW>(a.k.coef + static_cast<int64_t>(e) * S + s);
#pragma unroll
        for (int v = 0; v < VW; ++v) {
            double X[3][3];
#pragma unroll
            for (int b = 0; b < 3; ++b)
#pragma unroll
                for (int k = 0; k < 3; ++k) X[b][k] = ref[b][k] + xg[v][b][k];
            const Frame f = frame_from_points<FAST>(X);
            const double bb[3] = {f.ly[1] - f.ly[2], f.ly[2] - f.ly[0], f.ly[0] - f.ly[1]};
            const double cc[3] = {f.lx[2] - f.lx[1], f.lx[0] - f.lx[2], f.lx[1] - f.lx[0]};
            const double scale = FAST ? cf.v[v] * g.inv_1mnu2 * (1.0 / (4.0 * f.area))
                                      : cf.v[v] * g.inv_1mnu2 / (4.0 * f.area);
            double L0 = 0.0, L1 = 0.0, L2 = 0.0;
#pragma unroll
            for (int b = 0; b < 3; ++b) {
                const double *x = xu[v][b];
                const double x0 = f.t[0][0] * x[0] + f.t[0][1] * x[1] + f.t[0][2] * x[2];
                const double x1 = f.t[1][0] * x[0] + f.t[1][1] * x[1] + f.t[1][2] * x[2];
                const double x2 = f.t[2][0] * x[0] + f.t[2][1] * x[1] + f.t[2][2] * x[2];
                const double ba = bb[la], ca = cc[la];
                L0 += (ba * bb[b] + g.g * ca * cc[b]) * x0 + (g.nu * ba * cc[b] + g.g * ca * bb[b]) * x1;
                L1 += (g.nu * ca * bb[b] + g.g * ba * cc[b]) * x0 + (ca * cc[b] + g.g * ba * bb[b]) * x1;
                L2 += g.gk * (ba * bb[b] + ca * cc[b]) * x2;
            }
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                acc[v][k] += scale * (f.t[0][k] * L0 + f.t[1][k] * L1 + f.t[2][k] * L2);
                fl[v][k] += (1.0 / 3.0) * f.area * f.t[2][k];
            }
        }
    }
    const double pn = a.load.p[step];
    const double qa = a.load.ga ? a.load.qa[step] : 0.0;
    const double qb = a.load.gb ? a.load.qb[step] : 0.0;
    const bool fixed = a.fixed != nullptr && a.fixed[row] != 0;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int64_t off = (static_cast<int64_t>(row) * 3 + i) * S + s;
        const Vec<VW> uu = load_vec<VW>(a.u + off);
        const Vec<VW> pp = load_vec<VW>(a.up + off);
        const int64_t d = 3 * static_cast<int64_t>(row) + i;
        Vec<VW> o;
#pragma unroll
        for (int v = 0; v < VW; ++v) {
            const double m = a.lm_sstride ? a.lm[static_cast<int64_t>(row) * S + s + v] : a.lm[row];
            double force = pn * fl[v][i];
            if (a.load.ga) force += qa * a.load.ga[d];
            if (a.load.gb) force += qb * a.load.gb[d];
            if constexpr (DAMP) force -= a.ddt * (uu.v[v] - pp.v[v]);
            const double rhs = a.dt2 * (force - acc[v][i]) + m * (2.0 * uu.v[v] - pp.v[v]);
            const double un = m != 0.0 ? rhs / m : 0.0;
            o.v[v] = fixed ? a.bdy_u : un;
        }
        if (active) store_vec<VW>(a.out + off, o);
    }
}

__device__ __forceinline__ double dot(const double (&x)[3], const double (&y)[3]) {
    return fma(x[2], y[2], fma(x[1], y[1], x[0] * y[0]));
}

__device__ __forceinline__ void cross(const double (&x)[3], const double (&y)[3], double (&z)[3]) {
    z[0] = fma(x[1], y[2], -(x[2] * y[1]));
    z[1] = fma(x[2], y[0], -(x[0] * y[2]));
    z[2] = fma(x[0], y[1], -(x[1] * y[0]));
}

// The same product by the fan entries and without element frames.  With the row's node a as origin,
// e_p and e_q the moved edges to an element's other nodes, n = e_p x e_q (twice the area vector) and
// G_p = e_q x n, G_q = n x e_p, G_a = -(G_p + G_q) the gradients of the shape functions times n.n,
// the in-plane isotropic law and the transverse shear, both independent of the direction of the
// in-plane axes, give the force of the relative displacements y_p, y_q on a as
//   f_a = coef / (1 - nu^2) / (2 |n|) [ g w + ((gk - g) (n.w) n + nu tau G_a + g (G_p (y_p.G_a) +
//         G_q (y_q.G_a))) / n.n ],
//   w = (e_p.d) y_q - (e_q.d) y_p,  d = e_q - e_p,  tau = y_p.G_p + y_q.G_q,
// and the unit-pressure load as n / 6.  That is one reciprocal square root and about 100 FP64
// instructions per element and sample; the frames (two square roots, three divisions, the local
// coordinates and the nine 3 x 3 blocks' rows) took about 250, and FP64 issue bounds this kernel.
// Neighbours chain around the node, so each is read once, its loads in flight while the element
// before is applied.  65,920 nodes x 200 samples, every step re-formed: 939 -> 560 us a step.
template <bool UNIFORM, bool BETA, bool DAMP, bool GEO_U, int VW>
__global__ __launch_bounds__(kBlock) void k_step_moved(StepArgs a, GeomArgs g, int64_t step) {
    int32_t row;
    int64_t s;
    bool active;
    if (!row_and_sample<UNIFORM, VW>(g.n_rows, a.k.n_smp, row, s, active)) return;
    if (g.head) {
        row = g.head[4 * static_cast<int64_t>(row)];
        if constexpr (UNIFORM) row = __builtin_amdgcn_readfirstlane(row);
        if (row < 0) return;
    }
    const int64_t S = a.k.n_smp;
    const uint32_t lane = static_cast<uint32_t>(s) * 8u;
    // y = x relative to the row's node is all the product needs of the displacement, and with
    // GEO_U and no beta the moved edge is the reference edge plus y
    constexpr bool ONE = GEO_U && !BETA;
    struct Raw {
        Vec<VW> u[3], up[3], ug[3];
        double ref[3];
    };
    struct Rel {
        double e[3][VW], y[3][VW], ee[VW];
    };
    auto load = [&](int32_t node) {
        Raw r;
        load_node<UNIFORM, VW>(a.u, node, S, lane, r.u);
        if constexpr (BETA) load_node<UNIFORM, VW>(a.up, node, S, lane, r.up);
        if constexpr (!GEO_U) {
            if (g.ug) load_node<UNIFORM, VW>(g.ug, node, S, lane, r.ug);
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) r.ref[k] = g.nodes[3 * static_cast<int64_t>(node) + k];
        return r;
    };
    auto disp = [&](const Raw &r, int k, int v) {
        return BETA ? fma(a.bdt, r.u[k].v[v] - r.up[k].v[v], r.u[k].v[v]) : r.u[k].v[v];
    };
    auto move = [&](const Raw &r, int k, int v) {
        if constexpr (GEO_U) return r.u[k].v[v];
        else return g.ug ? r.ug[k].v[v] : 0.0;
    };
    const Raw own = load(row);
    auto relative = [&](const Raw &r, Rel &o) {
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
            for (int v = 0; v < VW; ++v) {
                o.y[k][v] = disp(r, k, v) - disp(own, k, v);
                o.e[k][v] = (r.ref[k] - own.ref[k]) + (ONE ? o.y[k][v] : move(r, k, v) - move(own, k, v));
            }
#pragma unroll
        for (int v = 0; v < VW; ++v)
            o.ee[v] = fma(o.e[2][v], o.e[2][v], fma(o.e[1][v], o.e[1][v], o.e[0][v] * o.e[0][v]));
    };
    double acc[3][VW] = {};
    double fl[3][VW] = {};        // six times the unit-traction load of the row's node
    const double cg = g.g, cs = g.gk - g.g, half = 0.5 * g.inv_1mnu2;
    auto apply = [&](const Rel &p, const Rel &q, const Vec<VW> &cf) {
#pragma unroll
        for (int v = 0; v < VW; ++v) {
            const double ep[3] = {p.e[0][v], p.e[1][v], p.e[2][v]}, eq[3] = {q.e[0][v], q.e[1][v], q.e[2][v]};
            const double yp[3] = {p.y[0][v], p.y[1][v], p.y[2][v]}, yq[3] = {q.y[0][v], q.y[1][v], q.y[2][v]};
            double n[3], Gp[3], Gq[3];
            cross(ep, eq, n);
            const double r = rsqrt(dot(n, n));
            cross(eq, n, Gp);
            cross(n, ep, Gq);
            const double pq = dot(ep, eq), cp = q.ee[v] - pq, cq = pq - p.ee[v];
            double w[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) w[k] = fma(cq, yq[k], -(cp * yp[k]));
            // nu tau G_a + g (G_p (y_p.G_a) + G_q (y_q.G_a)) = fp G_p + fq G_q
            const double ypp = dot(yp, Gp), yqq = dot(yq, Gq), t = g.nu * (ypp + yqq);
            const double fp = -fma(cg, ypp + dot(yp, Gq), t), fq = -fma(cg, yqq + dot(yq, Gp), t);
            const double nw = cs * dot(n, w), sc = half * cf.v[v] * r, s1 = sc * cg, s2 = sc * (r * r);
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const double in = fma(nw, n[k], fma(fp, Gp[k], fq * Gq[k]));
                acc[k][v] = fma(s2, in, fma(s1, w[k], acc[k][v]));
                fl[k][v] += n[k];
            }
        }
    };
    const int32_t q0 = g.nptr[row], q1 = g.nptr[row + 1];
    if (q0 != q1) {
        Rel x0, x1;                     // the p and q columns, taking turns
        const fan_t e = g.fan[q0];
        fan_t n = g.fan[q0 + 1 < q1 ? q0 + 1 : q0];        // one entry ahead of the loads it names
        Raw rq = load(e.y);
        Vec<VW> c = load_entry<UNIFORM, VW>(a.k.coef, e.z, S, lane);
        int32_t q = q0 + 1;
        relative(load(e.x), x0);
        // one element: its q column into xq, the next one's loads, then the element itself; true
        // behind the last one
        auto element = [&](Rel &xp, Rel &xq) {
            relative(rq, xq);
            const Vec<VW> cf = c;
            const int32_t apart = n.x;
            rq = load(n.y);             // behind the last element: its own node again
            c = load_entry<UNIFORM, VW>(a.k.coef, n.z, S, lane);
            n = g.fan[q + 1 < q1 ? q + 1 : q1 - 1];
            __builtin_amdgcn_sched_barrier(0);
            apply(xp, xq, cf);
            if (q++ >= q1) return true;
            if (apart >= 0) relative(load(apart), xq);
            return false;
        };
        while (!element(x0, x1) && !element(x1, x0)) {}
    }
    Vec<VW> pp[3];
    if constexpr (BETA) {
#pragma unroll
        for (int k = 0; k < 3; ++k) pp[k] = own.up[k];
    } else {
        load_node<UNIFORM, VW>(a.up, row, S, lane, pp);
    }
    const RowLoad<VW> rl = row_load<VW>(a, row, s);
    const double pn = a.load.p[step];
    const double qa = a.load.ga ? a.load.qa[step] : 0.0;
    const double qb = a.load.gb ? a.load.qb[step] : 0.0;
    Vec<VW> o[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int64_t d = 3 * static_cast<int64_t>(row) + k;
        double more = 0.0;
        if (a.load.ga) more = qa * a.load.ga[d];
        if (a.load.gb) more = fma(qb, a.load.gb[d], more);
#pragma unroll
        for (int v = 0; v < VW; ++v) {
            double force = fma(pn, (1.0 / 6.0) * fl[k][v], more);
            if constexpr (DAMP) force -= a.ddt * (own.u[k].v[v] - pp[k].v[v]);
            const double m = rl.m.v[v];
            const double rhs = fma(a.dt2, force - acc[k][v], m * fma(2.0, own.u[k].v[v], -pp[k].v[v]));
            const double un = m != 0.0 ? rhs / m : 0.0;
            o[k].v[v] = rl.fixed ? a.bdy_u : un;
        }
    }
    if (active) {
#pragma unroll
        for (int k = 0; k < 3; ++k) store_vec<VW>(a.out + (static_cast<int64_t>(row) * 3 + k) * S + s, o[k]);
    }
}

// Element stresses from the gradient of the displacement, without element frames.  With node 0 as
// origin, e_p, e_q the edges to nodes 1 and 2, n = e_p x e_q, G_p = e_q x n and G_q = n x e_p (the
// shape gradients times n.n), H = y_p (x) G_p + y_q (x) G_q of the relative displacements and
// q = (y_p.n) G_p + (y_q.n) G_q, the plane-stress law and the transverse shear are
//   sigma = E / (1 - nu^2) / n.n [ nu tr H (I - nn / n.n) + g (H + H^T) + (gk - g) (n (x) q + q (x) n) / n.n ]
// whatever the in-plane axes are: one division where the frame took two square roots and seven.
// GEO: 0 the reference geometry (the gradients are the same for a lane's samples), 1 X + u itself,
// 2 X + ug.  The output is written once and read by no kernel, in 16-byte stores, past L2 (NT) where
// stream_stress says so.
// 131,840 elements x 100 samples (0.79 GB) on the reference geometry: the call 270 -> 178 us, of which this
// kernel takes 155 to 171.
template <bool UNIFORM, int GEO, int VW, bool NT>
__global__ __launch_bounds__(kBlock) void k_element_stress(int64_t n_elms, int64_t S, GeomArgs g,
                                                           const double *__restrict__ u,
                                                           const double *__restrict__ ave_E,
                                                           double *__restrict__ stress) {
    int32_t row;
    int64_t s;
    bool active;
    if (!row_and_sample<UNIFORM, VW>(n_elms, S, row, s, active)) return;
    const int64_t e = static_cast<uint32_t>(row);
    const int32_t ids[3] = {g.elems[3 * e], g.elems[3 * e + 1], g.elems[3 * e + 2]};
    Vec<VW> x[3][3], m[3][3];
    double X[3][3];
#pragma unroll
    for (int b = 0; b < 3; ++b) {
        const int64_t d = 3 * static_cast<int64_t>(ids[b]);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            x[b][k] = load_vec<VW>(u + (d + k) * S + s);
            if constexpr (GEO == 2) m[b][k] = load_vec<VW>(g.ug + (d + k) * S + s);
            X[b][k] = g.nodes[d + k];
        }
    }
    const Vec<VW> E = load_vec<VW>(ave_E + e * S + s);
    Vec<VW> o[5];
#pragma unroll
    for (int v = 0; v < VW; ++v) {
        double ep[3], eq[3], yp[3], yq[3], n[3], Gp[3], Gq[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            yp[k] = x[1][k].v[v] - x[0][k].v[v];
            yq[k] = x[2][k].v[v] - x[0][k].v[v];
            ep[k] = X[1][k] - X[0][k];
            eq[k] = X[2][k] - X[0][k];
            if constexpr (GEO == 1) {
                ep[k] += yp[k];
                eq[k] += yq[k];
            } else if constexpr (GEO == 2) {
                ep[k] += m[1][k].v[v] - m[0][k].v[v];
                eq[k] += m[2][k].v[v] - m[0][k].v[v];
            }
        }
        cross(ep, eq, n);
        cross(eq, n, Gp);
        cross(n, ep, Gq);
        const double r = 1.0 / dot(n, n);
        const double c = E.v[v] * g.inv_1mnu2 * r, cg = c * g.g, cs = c * (g.gk - g.g) * r;
        const double tr = c * g.nu * (dot(yp, Gp) + dot(yq, Gq)), tn = tr * r;
        const double pn = dot(yp, n), qn = dot(yq, n);
        double w[3];                     // cs q - tn n / 2: the n (x) ... + ... (x) n terms together
#pragma unroll
        for (int k = 0; k < 3; ++k) w[k] = fma(cs, fma(pn, Gp[k], qn * Gq[k]), -0.5 * tn * n[k]);
        auto sym = [&](int i, int j) {
            const double h = fma(yp[i], Gp[j], fma(yp[j], Gp[i], fma(yq[i], Gq[j], yq[j] * Gq[i])));
            return fma(cg, h, fma(n[i], w[j], n[j] * w[i]));
        };
        o[0].v[v] = tr + sym(0, 0);
        o[1].v[v] = tr + sym(1, 1);
        o[2].v[v] = sym(0, 1);
        o[3].v[v] = sym(0, 2);
        o[4].v[v] = sym(1, 2);
    }
    if (!active) return;
    double *out = stress + e * 5 * S + s;
#pragma unroll
    for (int k = 0; k < 5; ++k) {
        if constexpr (NT) store_vec_nt<VW>(out + k * S, o[k]);
        else store_vec<VW>(out + k * S, o[k]);
    }
}

// Past L2 where the rows are whole 64-byte sectors (65,280 elements, 16 samples: 10.2 us past L2, 12.5
// through it), or longer rows of an array that the Infinity Cache cannot hold beside the inputs: a store
// past L2 of part of a sector leaves in pieces (204,288 elements: 4 samples 30 / 13 us, 20 51 / 41, 33
// 99 / 136; 131,428: 33 samples, 174 MB, 63 / 73).
bool stream_stress(int64_t n_elms, int64_t S) {
    return S % 8 == 0 || (S >= 20 && 40 * n_elms * S >= (int64_t(162) << 20));
}

template <int GEO, int VW, bool NT>
void launch_stress(hipStream_t st, int64_t n_elms, int64_t S, const GeomArgs &g, const double *u,
                   const double *ave_E, double *stress) {
    // padding the rows to whole wavefronts may not push the launch past 2^32 threads
    if (use_uniform<VW>(S) && n_elms < (int64_t(1) << 31) / lanes_per_row<true, VW>(S))
        hipLaunchKernelGGL((k_element_stress<true, GEO, VW, NT>), dim3(grid_for(n_elms * lanes_per_row<true, VW>(S))),
                           dim3(kBlock), 0, st, n_elms, S, g, u, ave_E, stress);
    else
        hipLaunchKernelGGL((k_element_stress<false, GEO, VW, NT>), dim3(grid_for(n_elms * lanes_per_row<false, VW>(S))),
                           dim3(kBlock), 0, st, n_elms, S, g, u, ave_E, stress);
}

GeomArgs geom_args(const cvfes_geometry_t *geo, const cvfes_system_t *sys, const double *ug) {
    GeomArgs g{};
    g.nodes = geo->nodes;
    g.elems = geo->elems;
    g.ug = ug;
    g.nptr = sys ? sys->nptr : nullptr;
    g.nent = sys ? sys->nent : nullptr;
    g.fan = sys ? fan_entries(sys) : nullptr;
    g.n_rows = sys ? sys->n_nodes : 0;
    g.nu = geo->nu;
    g.g = 0.5 * (1.0 - geo->nu);
    g.gk = 0.5 * geo->kshear * (1.0 - geo->nu);
    g.inv_1mnu2 = 1.0 / (1.0 - geo->nu * geo->nu);
    return g;
}

template <bool UNIFORM, bool FAST, bool GEO_U, int VW>
void launch_updated_inst(hipStream_t st, const StepArgs &a, const GeomArgs &g, int64_t step, bool beta,
                         bool damp) {
    const int64_t work = a.k.n_nodes * lanes_per_row<UNIFORM, VW>(a.k.n_smp);
    const dim3 grid(grid_for(work)), block(kBlock);
    if (beta) {
        if (damp) hipLaunchKernelGGL((k_step_updated<UNIFORM, true, true, FAST, GEO_U, VW>), grid, block, 0, st, a, g, step);
        else hipLaunchKernelGGL((k_step_updated<UNIFORM, true, false, FAST, GEO_U, VW>), grid, block, 0, st, a, g, step);
    } else {
        if (damp) hipLaunchKernelGGL((k_step_updated<UNIFORM, false, true, FAST, GEO_U, VW>), grid, block, 0, st, a, g, step);
        else hipLaunchKernelGGL((k_step_updated<UNIFORM, false, false, FAST, GEO_U, VW>), grid, block, 0, st, a, g, step);
    }
}

template <bool UNIFORM, bool GEO_U, int VW>
void launch_moved_inst(hipStream_t st, const StepArgs &a, const GeomArgs &g, int64_t step, bool beta, bool damp) {
    const dim3 grid(grid_for(g.n_rows * lanes_per_row<UNIFORM, VW>(a.k.n_smp))), block(kBlock);
    if (beta) {
        if (damp) hipLaunchKernelGGL((k_step_moved<UNIFORM, true, true, GEO_U, VW>), grid, block, 0, st, a, g, step);
        else hipLaunchKernelGGL((k_step_moved<UNIFORM, true, false, GEO_U, VW>), grid, block, 0, st, a, g, step);
    } else {
        if (damp) hipLaunchKernelGGL((k_step_moved<UNIFORM, false, true, GEO_U, VW>), grid, block, 0, st, a, g, step);
        else hipLaunchKernelGGL((k_step_moved<UNIFORM, false, false, GEO_U, VW>), grid, block, 0, st, a, g, step);
    }
}

template <bool GEO_U, int VW>
void launch_moved(hipStream_t st, const StepArgs &a, const GeomArgs &g, int64_t step, bool beta, bool damp) {
    if (use_uniform<VW>(a.k.n_smp)) launch_moved_inst<true, GEO_U, VW>(st, a, g, step, beta, damp);
    else launch_moved_inst<false, GEO_U, VW>(st, a, g, step, beta, damp);
}

template <bool FAST, bool GEO_U, int VW>
void launch_updated_u(hipStream_t st, const StepArgs &a, const GeomArgs &g, int64_t step, bool beta,
                      bool damp) {
    if (use_uniform<VW>(a.k.n_smp)) launch_updated_inst<true, FAST, GEO_U, VW>(st, a, g, step, beta, damp);
    else launch_updated_inst<false, FAST, GEO_U, VW>(st, a, g, step, beta, damp);
}

// Rows by node tiles where u is larger than the L2s, a neighbour takes more than its u (the damped state
// or a saved geometry) and rows are long: in natural order the neighbouring rings' lines then leave L2
// between their rows.  Five steps, natural / by tiles, 16,384 nodes x 256 samples: with beta 876 / 811 us,
// a saved geometry 1,000 / 938, both 1,312 / 1,015 (irregular wall 879 / 845, 1,020 / 987, 1,264 / 1,035);
// 65,920 x 200: 3,078 / 2,984, 3,429 / 3,341, 3,886 / 3,672.  Shorter rows gain only with both and whole
// wavefronts (102,400 x 128: 3,957 / 3,187; beta alone 2,615 / 2,539, on an irregular wall 2,687 /
// 2,861), others lose by the tiles' empty slots and the wider spread of a workgroup's rows (102,400 x 64
// with both 2,016 / 2,189, 65,920 x 180 1.03 and 1.09 times as long).  With u alone natural order already
// moves little (102,400 x 128: 450 / 458 us a step), and a small system gains nothing (4,096 x 33: 13.1 /
// 13.4).
void order_by_tiles(GeomArgs &g, const cvfes_system_t *sys, bool beta, bool saved) {
    const int64_t S = sys->n_smp;
    if (!g.fan || sys->n_tiles <= 0 || !sys->tile_head || S % 2 != 0 || 24 * sys->n_nodes * S < (int64_t(32) << 20) ||
        sys->n_tiles * CVFES_TILE_ROWS > INT32_MAX)
        return;
    if (S >= 192 ? !(beta || saved) : !(beta && saved && S % 128 == 0)) return;
    // the tiles' empty slots count as rows of the launch, which stays below 2^32 threads
    if (sys->n_tiles * CVFES_TILE_ROWS * lanes_per_row<true, 1>(S) >= (int64_t(1) << 32) - kBlock * kNumXcd) return;
    g.head = sys->tile_head;
    g.n_rows = sys->n_tiles * CVFES_TILE_ROWS;
}

// Updated-geometry kernel forms (sys->variant): GENERIC the divided frames with one sample per
// lane; ROWLOAD1 one sample per lane, ROWLOAD (and AUTO) two for even sample counts, without frames
// by the fan entries (65,920 nodes x 200 samples: 560 us a step for two samples per lane, 564 for
// one), with reciprocal frames (939 us) for systems that hold none.  geo_u: the geometry
// displacement is the current u.
void launch_updated(hipStream_t st, const StepArgs &a, const GeomArgs &g, int64_t step, bool beta,
                    bool damp, int64_t variant, bool geo_u) {
    const bool two = (variant == CVFES_VARIANT_AUTO || variant == CVFES_VARIANT_ROWLOAD) &&
                     a.k.n_smp % 2 == 0;
    if (variant == CVFES_VARIANT_GENERIC) {
        launch_updated_u<false, false, 1>(st, a, g, step, beta, damp);
    } else if (g.fan) {
        if (two) {
            if (geo_u) launch_moved<true, 2>(st, a, g, step, beta, damp);
            else launch_moved<false, 2>(st, a, g, step, beta, damp);
        } else {
            if (geo_u) launch_moved<true, 1>(st, a, g, step, beta, damp);
            else launch_moved<false, 1>(st, a, g, step, beta, damp);
        }
    } else if (two) {
        if (geo_u) launch_updated_u<true, true, 2>(st, a, g, step, beta, damp);
        else launch_updated_u<true, false, 2>(st, a, g, step, beta, damp);
    } else {
        if (geo_u) launch_updated_u<true, true, 1>(st, a, g, step, beta, damp);
        else launch_updated_u<true, false, 1>(st, a, g, step, beta, damp);
    }
}

}  // namespace
}  // namespace cvfes

using namespace cvfes;

extern "C" int cvfes_element_stress(void *stream, int64_t n_elms, int64_t n_smp,
                                    const cvfes_geometry_t *geo, const double *u, const double *ug,
                                    const double *ave_E, double *stress) {
    CVFES_REQUIRE(n_elms >= 0 && n_smp >= 1, "cvfes_element_stress: bad sizes");
    CVFES_REQUIRE(geo && geo->nodes && geo->elems && u && ave_E && stress,
                  "cvfes_element_stress: null argument");
    CVFES_REQUIRE(geo->nu > -1.0 && geo->nu < 1.0, "cvfes_element_stress: nu out of range");
    if (n_elms == 0) return CVFES_OK;
    const GeomArgs g = geom_args(geo, nullptr, ug);
    // two samples per lane and 16-byte accesses where the count and every array allow it
    const uintptr_t any = reinterpret_cast<uintptr_t>(u) | reinterpret_cast<uintptr_t>(ug) |
                          reinterpret_cast<uintptr_t>(ave_E) | reinterpret_cast<uintptr_t>(stress);
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int geom = !ug ? 0 : ug == u ? 1 : 2;
    auto launch = [&](auto geo_c, auto vw_c) {
        constexpr int GEO = decltype(geo_c)::value, VW = decltype(vw_c)::value;
        if (stream_stress(n_elms, n_smp)) launch_stress<GEO, VW, true>(st, n_elms, n_smp, g, u, ave_E, stress);
        else launch_stress<GEO, VW, false>(st, n_elms, n_smp, g, u, ave_E, stress);
    };
    auto width = [&](auto geo_c) {
        if (n_smp % 2 == 0 && any % 16 == 0) launch(geo_c, std::integral_constant<int, 2>{});
        else launch(geo_c, std::integral_constant<int, 1>{});
    };
    if (geom == 0) width(std::integral_constant<int, 0>{});
    else if (geom == 1) width(std::integral_constant<int, 1>{});
    else width(std::integral_constant<int, 2>{});
    return check_launch("k_element_stress");
}

extern "C" int cvfes_step_updated(void *stream, const cvfes_system_t *sys, const cvfes_geometry_t *geo,
                                  cvfes_update_t *upd, double **state, const cvfes_load_t *load,
                                  int64_t nsteps, double dt, double beta, double damp) {
    CVFES_REQUIRE(sys && geo && upd && state && load, "cvfes_step_updated: null argument");
    CVFES_REQUIRE(sys->n_nodes >= 1 && sys->n_smp >= 1 && nsteps >= 0 && dt > 0.0,
                  "cvfes_step_updated: bad sizes");
    CVFES_REQUIRE(sys->n_nodes * 3 < (int64_t(1) << 31), "cvfes_step_updated: too many nodes");
    // buffer resources of 3*S doubles (a node's state) must fit 31 bits
    CVFES_REQUIRE(sys->n_smp < (int64_t(1) << 31) / 24, "cvfes_step_updated: too many samples");
    CVFES_REQUIRE(sys->nptr && sys->nent && sys->coef && sys->lm && geo->nodes && geo->elems,
                  "cvfes_step_updated: the system needs nptr, nent, coef, lm and the geometry");
    CVFES_REQUIRE(geo->nu > -1.0 && geo->nu < 1.0, "cvfes_step_updated: nu out of range");
    CVFES_REQUIRE(upd->interval >= 1, "cvfes_step_updated: interval must be >= 1");
    CVFES_REQUIRE(upd->interval == 1 || upd->ug, "cvfes_step_updated: interval > 1 needs the ug buffer");
    CVFES_REQUIRE(state[0] && state[1] && state[2], "cvfes_step_updated: null state buffer");
    CVFES_REQUIRE(load->p && (!load->ga || load->qa) && (!load->gb || load->qb),
                  "cvfes_step_updated: load tables");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int64_t S = sys->n_smp;
    double *cur = state[0], *prev = state[1], *nxt = state[2];
    for (int64_t n = 0; n < nsteps; ++n) {
        if (upd->counter >= upd->interval) {
            if (upd->interval > 1) {
                const hipError_t err = hipMemcpyAsync(upd->ug, cur, sizeof(double) * 3 * sys->n_nodes * S,
                                                      hipMemcpyDeviceToDevice, st);
                if (err != hipSuccess)
                    return fail(CVFES_ERR_HIP, "cvfes_step_updated: %s", hipGetErrorString(err));
            }
            upd->has_geometry = 1;
            upd->counter = 1;
        } else {
            upd->counter += 1;
        }
        const double *geom = upd->has_geometry ? (upd->interval == 1 ? cur : upd->ug) : nullptr;
        StepArgs a;
        a.k = RowArgs{sys->n_nodes, S, sys->indptr, sys->indices, sys->values, sys->cptr, sys->celem,
                      sys->khat, sys->coef, sys->uvalues, sys->vblk, sys->nptr, nullptr};
        a.u = cur;
        a.up = prev;
        a.out = nxt;
        a.lm = sys->lm;
        a.lm_sstride = sys->lm_sstride;
        a.f1 = sys->f1;
        a.fixed = sys->fixed;
        a.load = *load;
        a.bdy_u = sys->bdy_u;
        a.dt2 = dt * dt;
        a.bdt = beta / dt;
        a.ddt = damp / dt;
        a.order = nullptr;
        GeomArgs g = geom_args(geo, sys, geom);
        order_by_tiles(g, sys, beta != 0.0, geom != nullptr && geom != cur);
        launch_updated(st, a, g, n, beta != 0.0, damp != 0.0, sys->variant, geom != nullptr && geom == cur);
        if (int rc = check_launch("k_step_updated")) return rc;
        double *t = prev;
        prev = cur;
        cur = nxt;
        nxt = t;
    }
    state[0] = cur;
    state[1] = prev;
    state[2] = nxt;
    return CVFES_OK;
}
