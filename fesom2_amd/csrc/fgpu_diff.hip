// Explicit diffusion terms of diff_tracers_ale (oce_ale_tracer.F90:533-793),
// evaluated from T^n before any kernel of the step overwrites it:
//
//   k_hdiff_edge  diff_part_hor_redi (oce_ale_tracer.F90:1526-1689): per edge
//                 and level the flux Kh (grad T + isredi S T_z) through the
//                 edge's dual segments. The element gradients
//                 (tracer_gradient_elements) and T_z (tracer_gradient_z, on
//                 hnode) are formed on the fly.
//   k_zbar        under Redi: interface depths rebuilt from hnode, per column
//   k_vextra      per column: diff_ver_part_expl_ale (:841-902) for tracers
//                 with i_vert_diff off, and diff_ver_part_redi_expl
//                 (:1439-1522) under Redi.
//
// k_hdiff_edge and k_vextra give an edge or column to one wave: 2^sh lanes take
// its levels, 2^sh the smallest power of two above the number of layers (without
// Redi k_hdiff_edge's not below it) and at most 64, and the wave's 64 / 2^sh lane
// groups take a tracer each. What does not depend on the tracer is loaded once
// per level. Fewer tracers than groups leave the others to further edges or
// columns. Both are bound by the gathers of T. 20 thousand nodes, 47 layers, 4
// tracers: k_hdiff_edge 232 -> 124 us against one thread per (edge, level,
// tracer), which divided its index and loaded the edge's geometry for itself;
// k_zbar and k_vextra 1124 -> 113 us against one thread per column, whose
// neighbours in a wave read rows apart. 120 thousand nodes, 4 layers, 1 tracer,
// one edge or column to a wave and as many as fit: k_hdiff_edge with Redi 226 and
// 62 us, without 159 and 29, k_vextra 174 and 43.
//
// They write the increments' parts (t.hd, t.ve, t.vr); the node update of
// either step (k_node_update / k_tstar, kL_node) adds them to del_ttf in the
// reference's order: advection, edges in ascending order, explicit vertical,
// explicit Redi, then the T* update. Arithmetic keeps the reference's
// evaluation order, so the sums are bit-identical to a serial run.
#include <algorithm>

#include "fgpu_internal.h"

#define ZCOL 32   // columns per block of k_zbar

// T_z at interface k (oce_tracer_mod.F90:192-232), t0 and t1 the values above
// and below it, dz the distance of their levels: zero at the column's top and
// bottom interfaces and outside the column
__device__ __forceinline__ double grad_z(double t0, double t1, double dz, bool inner)
{
    return inner ? (t0 - t1) / dz : 0.0;
}

// an element's rows and geometry, wave-uniform
struct Elem {
    size_t r0, r1, r2;   // offsets of its nodes' rows
    double g[6];
};
__device__ __forceinline__ Elem load_elem(const DevMesh &m, int el)
{
    Elem E;
    const int *en = m.elem_nodes + 3 * (size_t)el;
    const double *gs = m.gsca + 6 * (size_t)el;
    E.r0 = (size_t)ldc(en) * m.L;
    E.r1 = (size_t)ldc(en + 1) * m.L;
    E.r2 = (size_t)ldc(en + 2) * m.L;
#pragma unroll
    for (int i = 0; i < 6; ++i) E.g[i] = ldc(gs + i);
    return E;
}
// tracer_gradient_elements at the level that T points at
__device__ __forceinline__ void grad_el(const Elem &E, const double *T, double &gx, double &gy)
{
    const double t0 = T[E.r0], t1 = T[E.r1], t2 = T[E.r2];
    gx = E.g[0] * t0 + E.g[1] * t1 + E.g[2] * t2;
    gy = E.g[3] * t0 + E.g[4] * t1 + E.g[5] * t2;
}

// MULTI: with fewer tracers than lane groups the groups go round 2^eg edges
// or columns, whose records the lanes then load for themselves
template <bool REDI, bool MULTI>
__global__ void __launch_bounds__(64) k_hdiff_edge(DevMesh m, DevDyn d, DevTracers t, int tr0, int ntr, int sh, int eg)
{
    const int L = m.L, idx = threadIdx.x & ((1 << sh) - 1), gt = 64 >> sh >> (MULTI ? eg : 0);
    const int g = (int)(threadIdx.x >> sh) & (gt - 1);
    const int je = MULTI ? (xcd_unit() << eg) + (int)(threadIdx.x >> sh) / gt : xcd_unit();
    if (je >= m.E2) return;
    const int *ri = m.erec_i + (size_t)je * ERI;
    const double *rd = m.erec_d + (size_t)je * ERD;
    const int n1 = ldc(ri + ER_N1), n2 = ldc(ri + ER_N2), el1 = ldc(ri + ER_EL1), el2 = ldc(ri + ER_EL2);
    const int nl1 = ldc(ri + ER_NL1), nu1 = ldc(ri + ER_NU1), nl2 = ldc(ri + ER_NL2), nu2 = ldc(ri + ER_NU2);
    const bool two = el2 >= 0;
    const int q2 = two ? el2 : el1;
    const int lo = two ? min(nu1, nu2) : nu1, hi = two ? max(nl1, nl2) : nl1;
    const double dX1 = ldc(rd + ER_DX1), dY1 = ldc(rd + ER_DY1), dX2 = ldc(rd + ER_DX2), dY2 = ldc(rd + ER_DY2);
    const Elem E1 = load_elem(m, el1), E2 = load_elem(m, q2);
    double *hd = t.hd + (size_t)ldc(ri + ER_E) * L;
    const int zt1 = ldc(m.ulevn + n1), zb1 = ldc(m.nlevn + n1), zt2 = ldc(m.ulevn + n2), zb2 = ldc(m.nlevn + n2);
    // with the slope terms the last lane only supplies T_z at its upper interface to the lane before
    for (int kb = lo; kb <= hi; kb += (1 << sh) - (REDI ? 1 : 0)) {
        const int k = kb + idx, kc = min(k, L), ku = max(kc - 1, 1);
        // cases (A)/(D): el1 alone, (B)/(E): el2 alone, (C): both. The levels without either keep the zeros
        // that the buffer starts with
        const bool p1 = k >= nu1 && k <= nl1, p2 = two && k >= nu2 && k <= nl2;
        // in a level gap between the elements both segments reach into it, where the reference's element
        // gradients are zero: the slope terms of both
        const bool gap = REDI && two && ((k > nl1 && k < nu2) || (k > nl2 && k < nu1));
        const bool out = (p1 || p2 || gap) && (!REDI || idx < (1 << sh) - 1);
        const size_t c1 = (size_t)n1 * L + kc - 1, c2 = (size_t)n2 * L + kc - 1;
        const double Kh = (d.Ki[c1] + d.Ki[c2]) / 2.0;
        const double h1 = m.helem[(size_t)el1 * L + kc - 1], h2 = m.helem[(size_t)q2 * L + kc - 1];
        const double dz = p1 ? (p2 ? (h1 + h2) / 2.0 : h1) : h2;
        const double a = p1 ? (p2 ? dX2 - dX1 : -dX1) : dX2, b = p1 ? (p2 ? dY2 - dY1 : -dY1) : dY2;
        double dz1 = 0.0, dz2 = 0.0, sx1 = 0.0, sy1 = 0.0, sx2 = 0.0, sy2 = 0.0;
        const bool in1 = k > zt1 && k < zb1, in2 = k > zt2 && k < zb2;
        const int up = kc - ku;
        if (REDI) {
            dz1 = 0.5 * (m.hnode[c1 - up] + m.hnode[c1]);
            dz2 = 0.5 * (m.hnode[c2 - up] + m.hnode[c2]);
            sx1 = d.slope[3 * c1]; sy1 = d.slope[3 * c1 + 1];
            sx2 = d.slope[3 * c2]; sy2 = d.slope[3 * c2 + 1];
        }
        for (int tb = g; tb < ntr; tb += gt) {
            const double *T = t.T + t.sN * (tr0 + tb);
            double sx = 0.0, sy = 0.0;
            if (REDI) {
                const double z1 = grad_z(T[c1 - up], T[c1], dz1, in1), z2 = grad_z(T[c2 - up], T[c2], dz2, in2);
                const double Tz1 = 0.5 * (z1 + lane_above(z1)), Tz2 = 0.5 * (z2 + lane_above(z2));
                sx = (Tz1 * sx1 + Tz2 * sx2) / 2.0;
                sy = (Tz1 * sy1 + Tz2 * sy2) / 2.0;
            }
            double gx1, gy1, gx2, gy2;
            grad_el(E1, T + kc - 1, gx1, gy1);
            grad_el(E2, T + kc - 1, gx2, gy2);
            const double Tx = p1 ? (p2 ? 0.5 * (gx1 + gx2) : gx1) : gx2, Ty = p1 ? (p2 ? 0.5 * (gy1 + gy2) : gy1) : gy2;
            const double Fx = Kh * (Tx + sx), Fy = Kh * (Ty + sy);
            double c = (a * Fy - b * Fx) * dz;
            if (REDI && gap) {
                const double gx = Kh * sx, gy = Kh * sy;
                c = (-dX1 * gy + dY1 * gx) * h1 + (dX2 * gy - dY2 * gx) * h2;
            }
            if (out) hd[t.sE * (tr0 + tb) + k - 1] = c;
        }
    }
}

// surface flux of the explicit vertical diffusion (oce_ale_tracer.F90:873-885)
__device__ __forceinline__ double expl_surface_flux(int id, const DevDyn &d, int n)
{
    if (id == 1) return -d.heat_flux[n] / 4.2e6;   // vcpw (oce_modules.F90)
    if (id == 2) return d.virtual_salt[n] + d.relax_salt[n] + d.real_salt_flux[n] * d.is_nonlinfs;
    return 0.0;
}

// zbar of every column from the bottom up on hnode (oce_ale_tracer.F90:1439-1522), a chain of sums of its own
// for each column: a tile of columns in LDS, one lane per column for the sums
__global__ void __launch_bounds__(64) k_zbar(DevMesh m, double *zb)
{
    extern __shared__ double zs[];   // ZCOL rows of an odd length
    const int L = m.L, NL = m.NL, P = NL | 1, n0 = blockIdx.x * ZCOL, nc = min(ZCOL, m.N2 - n0);
    for (int c = 0; c < nc; ++c)
        for (int k = threadIdx.x; k < L; k += 64) zs[c * P + k] = m.hnode[(size_t)(n0 + c) * L + k];
    __syncthreads();
    if ((int)threadIdx.x < nc) {
        const int n = n0 + threadIdx.x, ul1 = m.ulevn[n], nl1 = m.nlevn[n] - 1;
        double *z = zs + threadIdx.x * P;
        double s = m.zbar_n_bot[n];
        z[nl1] = s;
        for (int nz = nl1; nz >= ul1 + 1; --nz) {
            s = s + z[nz - 1];
            z[nz - 1] = s;
        }
    }
    __syncthreads();
    for (int c = 0; c < nc; ++c)
        for (int k = threadIdx.x; k < NL; k += 64) zb[(size_t)(n0 + c) * NL + k] = zs[c * P + k];
}

template <bool MULTI>
__global__ void __launch_bounds__(64) k_vextra(DevMesh m, DevDyn d, DevTracers t, int tr0, int ntr, int sh, int eg, double dt)
{
    const int L = m.L, NL = m.NL, lp = 1 << sh, idx = threadIdx.x & (lp - 1), gt = 64 >> sh >> (MULTI ? eg : 0);
    const int g = (int)(threadIdx.x >> sh) & (gt - 1);
    const int jn = MULTI ? (xcd_unit() << eg) + (int)(threadIdx.x >> sh) / gt : xcd_unit();
    if (jn >= m.N2) return;
    const int n = ldc(m.node_ord + jn), ul1 = ldc(m.ulevn + n), nl1 = ldc(m.nlevn + n) - 1;
    const int num = ldc(m.nie_num + n);
    const bool redi = d.redi != 0;
    // a column of more levels than lanes: the first and the last lane of a further pass only supply their
    // values to their neighbours
    for (int kb = ul1;; kb += lp - 2) {
        const int k = kb + idx, kc = min(k, nl1);
        const bool out = k <= nl1 && (idx > 0 || kb == ul1) && (idx < lp - 1 || k == nl1);
        const size_t c = (size_t)n * L + kc - 1, ci = (size_t)n * NL + kc - 1;
        const double ar = m.area[ci], av = m.areasvol[ci];
        const double kv = d.Kv[ci], zb0 = m.zbar3d[ci], zb1 = m.zbar3d[ci + 1];
        const double Z = m.Z3d[c], zinv1 = 1.0 / (lane_below(Z) - Z);
        double a = 0.0, b = 0.0, den = 1.0, ki = 0.0, kim = 0.0, s0 = 0.0, s1 = 0.0;
        if (redi) {
            const double zbn = t.zbh[ci], zn = t.zbh[ci + 1] + m.hnode[c] / 2.0, znm = lane_below(zn);
            a = znm - zbn;
            b = zbn - zn;
            den = znm - zn;
            ki = d.Ki[c];
            kim = lane_below(ki);
            s0 = d.slope[3 * c];
            s1 = d.slope[3 * c + 1];
        }
        for (int tb = g; tb < ntr; tb += gt) {
            const int tr = tr0 + tb;
            const double *T = t.T + t.sN * tr;
            if (!t.ivd[tr]) {   // diff_ver_part_expl_ale
                const double Tk = T[c], Tu = lane_below(Tk);
                const double vd = k == ul1 ? expl_surface_flux(t.id[tr], d, n) : kv * (Tu - Tk) * zinv1 * ar;
                const double va = lane_above(vd), vb = k >= nl1 ? 0.0 : va;   // all lanes exchange
                if (out) t.ve[t.sN * tr + c] = (vd - vb) / (zb0 - zb1) * dt / av;
            }
            if (redi) {   // diff_ver_part_redi_expl
                // node gradients: element gradients weighted by area / 3 / areasvol
                double Tx = 0.0, Ty = 0.0;
                for (int j = 0; j < num; ++j) {
                    const int el = ldc(m.nie + (size_t)n * m.kmax + j);
                    const Elem E = load_elem(m, el);
                    const double A = ldc(m.elem_area + el);
                    double gx, gy;
                    grad_el(E, T + kc - 1, gx, gy);
                    if (k <= ldc(m.nlev + el) - 1 && k >= ldc(m.ulev + el)) {
                        Tx = Tx + gx * A;
                        Ty = Ty + gy * A;
                    }
                }
                const double tx = Tx / 3.0 / av, ty = Ty / 3.0 / av;
                const double sg = s0 * tx + s1 * ty;
                double v = a * lane_below(sg) * kim;
                v = v + b * sg * ki;
                const double vd = k == ul1 ? 0.0 : v / den * ar;
                const double va = lane_above(vd), vb = k >= nl1 ? 0.0 : va;   // all lanes exchange
                if (out) t.vr[t.sN * tr + c] = (vd - vb) * dt / av;
            }
        }
        if (kb + lp - 1 >= nl1) break;
    }
}

// ==============================================================================
// host side
// ==============================================================================
static bool any_explicit_vertical(const fgpu_context *c)
{
    for (int v : c->h_ivd)
        if (!v) return true;
    return false;
}

// buffers of the explicit terms for every tracer slot; before any capture
int fgpu_ensure_diff(fgpu_context *c)
{
    DevTracers &t = c->t;
    const int nt = t.ntr;
    struct A { double **p; size_t n; bool need; } arrs[] = {
        {&t.hd, t.sE * nt, c->d.hdiff != 0}, {&t.ve, t.sN * nt, any_explicit_vertical(c)},
        {&t.vr, t.sN * nt, c->d.redi != 0}, {&t.zbh, t.sNI, c->d.redi != 0}};
    for (auto &a : arrs) {
        if (!a.need || *a.p) continue;
        int rc = fgpu_alloc(c, (void **)a.p, a.n * sizeof(double), true);
        if (rc) return rc;
        if ((rc = fgpu_zero(c, *a.p, a.n * sizeof(double)))) return rc;
        c->graph_valid = false;
    }
    return FGPU_OK;
}

// enqueue the explicit terms of tracers tr0..tr0+ntr-1 from the current T
int fgpu_launch_diff(fgpu_context *c, int tr0, int ntr, double dt)
{
    const DevMesh &m = c->m;
    bool ve = false;
    for (int i = tr0; i < tr0 + ntr; ++i) ve = ve || !c->h_ivd[i];
    // lanes per column: above the layer count where levels exchange values, so that the lane below the deepest
    // layer exists, else (1 << se) no fewer than it
    int sh = 3, se = 2;
    while (sh < 6 && (1 << sh) <= m.L) ++sh;
    while (se < 6 && (1 << se) < m.L) ++se;
    if (c->d.redi) se = sh;
    // 2^eg edges and 2^cg columns per wave, as many as leave a lane group to each tracer
    auto per_wave = [&](int s) {
        int g = 6 - s;
        while (g > 0 && (64 >> s >> g) < ntr) --g;
        return g;
    };
    const int eg = per_wave(se), cg = per_wave(sh);
    if (c->d.hdiff) {
        if (!c->t.hd) return fgpu_fail(FGPU_ERR_STATE, "diffusion buffers not allocated");
        ProfScope ps(c, "k_hdiff_edge");
        const dim3 g(xcd_grid((m.E2 + (1 << eg) - 1) >> eg)), b(64);
        if (c->d.redi && eg) hipLaunchKernelGGL((k_hdiff_edge<true, true>), g, b, 0, c->stream, m, c->d, c->t, tr0, ntr, se, eg);
        else if (c->d.redi) hipLaunchKernelGGL((k_hdiff_edge<true, false>), g, b, 0, c->stream, m, c->d, c->t, tr0, ntr, se, eg);
        else if (eg) hipLaunchKernelGGL((k_hdiff_edge<false, true>), g, b, 0, c->stream, m, c->d, c->t, tr0, ntr, se, eg);
        else hipLaunchKernelGGL((k_hdiff_edge<false, false>), g, b, 0, c->stream, m, c->d, c->t, tr0, ntr, se, eg);
        FGPU_HIP(hipGetLastError());
    }
    if (ve || c->d.redi) {
        if ((ve && !c->t.ve) || (c->d.redi && (!c->t.vr || !c->t.zbh)))
            return fgpu_fail(FGPU_ERR_STATE, "diffusion buffers not allocated");
        if (c->d.redi) {
            ProfScope ps(c, "k_zbar");
            hipLaunchKernelGGL(k_zbar, dim3((m.N2 + ZCOL - 1) / ZCOL), dim3(64), ZCOL * (m.NL | 1) * sizeof(double),
                               c->stream, m, c->t.zbh);
            FGPU_HIP(hipGetLastError());
        }
        ProfScope ps(c, "k_vextra");
        const dim3 g(xcd_grid((m.N2 + (1 << cg) - 1) >> cg)), b(64);
        if (cg) hipLaunchKernelGGL(k_vextra<true>, g, b, 0, c->stream, m, c->d, c->t, tr0, ntr, sh, cg, dt);
        else hipLaunchKernelGGL(k_vextra<false>, g, b, 0, c->stream, m, c->d, c->t, tr0, ntr, sh, cg, dt);
        FGPU_HIP(hipGetLastError());
    }
    return FGPU_OK;
}
