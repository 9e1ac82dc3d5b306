// Fused, batched tracer step for gfx950: six launches per step for all tracers.
//
//   K_G  node pass   area-weighted mean element gradient of T^n at the levels
//                    where an edge needs it (fill_up_dn_grad's non-shared levels)
//   K_A  edge pass   LO upwind flux (T^n) and antidiffusive flux HO(T^AB) - LO
//                    (MFCT/UPW1); the up/downwind element gradients and T^AB are
//                    evaluated on the fly
//   K_B  node pass   LO solution and antidiffusive vertical flux (QR4C/UPW1)
//   K_C  node pass   FCT bounds over the 1-ring (edge gather), P+/P-, R+/R-
//   K_L  node pass   limited vertical and horizontal fluxes, flux2dtracer, T*,
//                    valuesold rotation
//   K_V  column pass implicit vertical diffusion (Thomas), salinity clamp
//
// K_B..K_L are separated by the three global dependencies of FCT (LO of the
// neighbours, R+/R- of the neighbours, limited edge fluxes). One wave owns one
// column (an edge or a node) and every tracer of its block; lanes run over
// levels, so a column's topology and geometry are wave-uniform and its field
// accesses are contiguous column segments. Blocks are mapped to columns XCD by
// XCD (workgroups are dispatched to the XCDs round-robin), so neighbouring
// columns share an L2.
//
// Arithmetic is the same sequence of operations as the per-function kernels
// and the reference (no FMA contraction); edge->node sums run over the node's
// edges in ascending edge order. Results are bit-identical to a serial run of
// the reference's loops.
#include <algorithm>
#include <type_traits>

#include "fgpu_internal.h"
#include "fgpu_vert.h"

__device__ __forceinline__ double dmx(double a, double b) { return a > b ? a : b; }
__device__ __forceinline__ double dmn(double a, double b) { return a < b ? a : b; }

// ordering of LDS accesses between the lanes of one wave: prior LDS writes
// complete before later accesses, and the compiler keeps the order
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

__device__ __forceinline__ int rl(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ double rld(double v, int lane)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), lane);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// position of this block's column in the processing order (the node or edge
// is node_ord / edge_ord of it), XCD-contiguous: blocks b, b+8, ... run on one
// XCD and take consecutive positions
__device__ __forceinline__ int xcd_column(int ncol)
{
    const int per = (int)(gridDim.x / NXCD);
    return (int)(blockIdx.x % NXCD) * per + (int)(blockIdx.x / NXCD);
}

// ------------------------------------------------------------------------------
// K_G: mean gradient around a node (oce_muscl_adv.F90:388-401, 443-520) for
// levels kneed(n)..nlevels_nod2D-1
// ------------------------------------------------------------------------------
// One wave per node. The range is a handful of levels at the bottom of most
// columns, so the lanes take (tracer, level) pairs, as many tracers at a time
// as fit, instead of one tracer's levels.
__global__ void __launch_bounds__(64) kG_node(DevMesh m, DevTracers t, const int *kneed, int tpb)
{
    const int jn = xcd_column(m.N2);
    if (jn >= m.N2) return;
    const int n = ldc(m.node_ord + jn);
    const int k0 = ldc(kneed + n), nzmax = ldc(m.nlevn + n);
    if (k0 > nzmax - 1) return;
    const int L = m.L, lane = threadIdx.x;
    const int num = ldc(m.nie_num + n);
    int lo = 1, hi = 0, a0 = 0, a1 = 0, a2 = 0;
    double ar = 0.0, g0 = 0.0, g1 = 0.0, g2 = 0.0, g3 = 0.0, g4 = 0.0, g5 = 0.0;
    if (lane < num) {
        const int el = m.nie[(size_t)n * m.kmax + lane];
        lo = m.ulev[el];
        hi = m.nlev[el] - 1;
        ar = m.elem_area[el];
        a0 = m.elem_nodes[3 * el]; a1 = m.elem_nodes[3 * el + 1]; a2 = m.elem_nodes[3 * el + 2];
        const double *gs = m.gsca + 6 * (size_t)el;
        g0 = gs[0]; g1 = gs[1]; g2 = gs[2]; g3 = gs[3]; g4 = gs[4]; g5 = gs[5];
    }
    const int trb = blockIdx.y * tpb, tre = min(t.ntr, trb + tpb);
    for (int kb = k0; kb < nzmax; kb += 64) {   // one pass unless the range is deeper than the wave
        const int nk = min(64, nzmax - kb), tp = 64 / nk;   // levels, tracers at a time
        const int ti = (int)(((float)lane + 0.5f) / (float)nk), k = kb + lane - ti * nk;
        for (int tb = trb; tb < tre; tb += tp) {
            const int tr = tb + ti;
            // node means feed MFCT and MUSCL
            const bool act = ti < tp && tr < tre && t.hor[min(tr, tre - 1)] != HOR_UPW1;
            const double *T = t.T + t.sN * min(tr, tre - 1) + k - 1;
            double tvol = 0.0, tx = 0.0, ty = 0.0;
            for (int i = 0; i < num; ++i) {
                const int elo = rl(lo, i), ehi = rl(hi, i);
                const int b0 = rl(a0, i), b1 = rl(a1, i), b2 = rl(a2, i);
                const double a = rld(ar, i);
                const double s0 = rld(g0, i), s1 = rld(g1, i), s2 = rld(g2, i);
                const double s3 = rld(g3, i), s4 = rld(g4, i), s5 = rld(g5, i);
                if (act && k >= elo && k <= ehi) {
                    const double t0 = T[(size_t)b0 * L], t1 = T[(size_t)b1 * L], t2 = T[(size_t)b2 * L];
                    const double ex = s0 * t0 + s1 * t1 + s2 * t2;
                    const double ey = s3 * t0 + s4 * t1 + s5 * t2;
                    tvol = tvol + a;
                    tx = tx + ex * a;
                    ty = ty + ey * a;
                }
            }
            if (act) {
                double *o = t.gmean + t.sG * tr + ((size_t)n * L + k - 1) * 2;
                o[0] = tx / tvol;
                o[1] = ty / tvol;
            }
        }
    }
}

// ------------------------------------------------------------------------------
// Column waves: one wave per node column (or edge), NV adjacent levels per lane
// and GT tracers per wave, 64 / GT lanes each.
//
// These kernels are bound by the vector memory pipeline: at 1.3 million nodes,
// 70 layers, 10 tracers a CU's texture data unit is busy 97 to 99 % of the time
// in K_A to K_L, 46 to 63 % of that waiting for L2. Instruction issue is not far
// behind: a SIMD issues some instruction in 64 to 87 % of its cycles, VALU work in
// 46 to 69 %, and with 64-bit row addresses formed in scalar registers and
// branches around masked lanes the scalar instructions outnumbered the vector
// ones. So the rows' byte offsets are formed once per column in vector registers
// (the tracers of a block only change the scalar base), loads are not masked
// (lanes without a wet level read a valid row entry), and the level ranges of the
// edges are lane masks that select results.
// One wave per block: with four, a block's slots stay taken until its slowest
// wave is done (70 layers, 10 tracers: K_L 3 % slower).
// ------------------------------------------------------------------------------
// two adjacent levels of a row: 16 bytes at any 8-byte boundary
typedef double lv2 __attribute__((ext_vector_type(2), aligned(8)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x8 __attribute__((ext_vector_type(8)));

// row values at byte offset off from a wave-uniform base
template <int NV, typename OFF>
__device__ __forceinline__ void row_load(const double *p, OFF off, double (&x)[NV])
{
    const char *a = (const char *)p + off;
#pragma unroll
    for (int s = 0; s + 1 < NV; s += 2) {
        const lv2 v = *(const lv2 *)(a + 8 * s);
        x[s] = v.x;
        x[s + 1] = v.y;
    }
    if constexpr (NV % 2 == 1) x[NV - 1] = *(const double *)(a + 8 * (NV - 1));
}

template <int NV, typename OFF>
__device__ __forceinline__ void row_store(double *p, OFF off, const double (&x)[NV], const bool (&on)[NV])
{
    char *a = (char *)p + off;
#pragma unroll
    for (int s = 0; s + 1 < NV; s += 2) {
        if (on[s] && on[s + 1]) {
            lv2 v;
            v.x = x[s];
            v.y = x[s + 1];
            *(lv2 *)(a + 8 * s) = v;
        } else if (on[s]) {
            *(double *)(a + 8 * s) = x[s];
        } else if (on[s + 1]) {
            *(double *)(a + 8 * s + 8) = x[s + 1];
        }
    }
    if constexpr (NV % 2 == 1)
        if (on[NV - 1]) *(double *)(a + 8 * (NV - 1)) = x[NV - 1];
}

// a column's values one level up (k - 1) and one level down (k + 1)
template <int NV>
__device__ __forceinline__ void col_up(const double (&x)[NV], double (&y)[NV])
{
    y[0] = lane_below(x[NV - 1]);
#pragma unroll
    for (int s = 1; s < NV; ++s) y[s] = x[s - 1];
}
template <int NV>
__device__ __forceinline__ void col_down(const double (&x)[NV], double (&y)[NV])
{
    y[NV - 1] = lane_above(x[0]);
#pragma unroll
    for (int s = 0; s + 1 < NV; ++s) y[s] = x[s + 1];
}

// a / 3 and a / 6 with the constant's reciprocal in two parts, zh + zl: one
// rounding of a zh + (a zl). A quotient by 3 (or 6) is never nearer to a
// rounding boundary than a sixth of its last place and the two-part product is
// within 2^-104 of it, so this is the correctly rounded quotient wherever a zl
// does not underflow. The caller sends smaller numerators to the division.
#define TINY_NUM 1e-280
__device__ __forceinline__ double third(double a) { return fma(a, 0x1.5555555555555p-2, a * 0x1.5555555555555p-56); }
__device__ __forceinline__ double sixth(double a) { return fma(a, 0x1.5555555555555p-3, a * 0x1.5555555555555p-57); }
__device__ __forceinline__ bool tiny(double a) { return fabs(a) < TINY_NUM && a != 0.0; }

// the column of a wave and its edges: byte offsets of the other nodes' rows and
// of the edge rows, first level and level count - 1 of the edge. Lanes outside
// an edge's levels, and the missing edges of the last batch, read rows that
// exist: the column's own and the first edge's.
#define CE 8   // edges kept in registers; a node's further ones are read in place
template <typename OFF, int NV, int GT>
struct Column {
    int n, deg, p0, nzmin, nzmax;
    int g, kb, kc;       // tracer of the wave, first level of the lane, the same within the row
    bool wet[NV];
    OFF own, ownI;       // offsets of the lane in layer and interface rows of one tracer's field
    OFF on[CE], oe[CE];
    int a0[CE], len[CE], side[CE];
};

// x, or -x on the edge's second node (sgn: bit 63)
__device__ __forceinline__ double signed_by(double x, long long sgn)
{
    return __longlong_as_double(__double_as_longlong(x) ^ sgn);
}

// level kb + s is one of the edge's levels
__device__ __forceinline__ bool edge_has(int kb, int s, int a0, int len) { return (unsigned)(kb + s - a0) <= (unsigned)len; }

template <typename OFF, int NV, int GT>
__device__ __forceinline__ void edge_offsets(const DevMesh &m, const DevTracers &t, const Column<OFF, NV, GT> &c, int u,
                                             OFF &on, OFF &oe, int &a0, int &len, int &side)
{
    const i32x8 r = ldc((const i32x8 *)m.col_ne + c.p0 + u);
    const OFF lev = 8 * (OFF)(c.kc - 1);
    side = r[0] & 1;
    a0 = r[2];
    len = r[3] - r[2];
    bool some = false;
#pragma unroll
    for (int s = 0; s < NV; ++s) some = some || edge_has(c.kb, s, a0, len);
    on = some ? lev + 8 * (OFF)c.g * (OFF)t.sN + 8 * (OFF)r[1] * (OFF)m.L : c.own;
    oe = lev + 8 * (OFF)c.g * (OFF)t.sE + 8 * (OFF)(r[0] >> 1) * (OFF)m.L;
}

// the levels g0..g1 between the elements of a column's edge where those share none: none on most edges (g0 > g1)
__device__ __forceinline__ void edge_gap(const DevMesh &m, int p, int &g0, int &g1)
{
    const i32x8 r = ldc((const i32x8 *)m.col_ne + p);   // [4..7]: nl1, nu1, nl2, nu2
    g0 = min(r[4], r[6]) + 1;
    g1 = r[7] > 0 ? max(r[5], r[7]) - 1 : 0;
}

template <bool LANES_OFF, typename OFF, int NV, int GT>
__device__ __forceinline__ bool load_column(const DevMesh &m, const DevTracers &t, Column<OFF, NV, GT> &c)
{
    const int lane = threadIdx.x;
    const int jc = xcd_column(m.N2);
    if (jc >= m.N2) return false;
    const i32x8 r = ldc((const i32x8 *)m.col_rec + jc);
    c.n = r[0];
    c.p0 = r[1];
    c.deg = r[2];
    c.nzmin = r[3];
    c.nzmax = r[4];
    constexpr int LP = 64 / GT;
    c.g = lane / LP;
    c.kb = (lane % LP) * NV + 1;
    // LANES_OFF: the lanes without a level or interface of the column are off
    // throughout; a lane exchange only leaves the column's ends to them, which
    // have rules of their own
    if (LANES_OFF && (c.kb > c.nzmax || c.kb + NV - 1 < c.nzmin)) return false;
    c.kc = c.kb <= m.L ? c.kb : 1;
#pragma unroll
    for (int s = 0; s < NV; ++s) c.wet[s] = c.kb + s >= c.nzmin && c.kb + s <= c.nzmax - 1;
    c.own = 8 * ((OFF)(c.kc - 1) + (OFF)c.g * (OFF)t.sN + (OFF)c.n * (OFF)m.L);
    c.ownI = 8 * ((OFF)((LANES_OFF || c.kb <= m.NL ? c.kb : 1) - 1) + (OFF)c.g * (OFF)t.sNI + (OFF)c.n * (OFF)m.NL);
#pragma unroll
    for (int u = 0; u < CE; ++u) {
        c.on[u] = c.own;
        c.oe[u] = c.oe[0];
        c.a0[u] = 0x40000000;
        c.len[u] = 0;
        c.side[u] = 0;
        if (u < c.deg) edge_offsets<OFF, NV, GT>(m, t, c, u, c.on[u], c.oe[u], c.a0[u], c.len[u], c.side[u]);
    }
    return true;
}

// ------------------------------------------------------------------------------
// K_A: edge pass
// ------------------------------------------------------------------------------
// Per tracer it gathers T and the old level at the edge's nodes and T at the
// nodes of the upwind and downwind triangles: ten row loads and a store per
// tracer. The volume fluxes are stored once for all tracers instead of a LO flux
// per tracer. Against a block per edge, 126,858 nodes, 47 layers, 2 tracers: 670
// -> 506 us; 12 thousand nodes, 32 tracers: 886 -> 445; 40 thousand nodes, 70
// layers, 10 tracers: 1390 -> 730.
// GAP is the form for a mesh with a level gap across some edge: the reference's
// segments of both elements reach into the gap (oce_adv_tra_hor.F90:166-249),
// the upper element's first, so two fluxes follow each other there. K_B and K_C
// have the form too; other meshes do not carry its registers.
template <typename OFF, int NV, int GT, bool GAP>
__global__ void __launch_bounds__(64) kA_edge(DevMesh m, DevDyn d, DevTracers t, int tpb)
{
    const int lane = threadIdx.x;
    const int je = xcd_column(m.E2);
    if (je >= m.E2) return;
    constexpr int LP = 64 / GT;
    const int g = lane / LP, kb = (lane % LP) * NV + 1;
    const int L = m.L;
    const int *ri = m.erec_i + (size_t)je * ERI;
    const double *rd = m.erec_d + (size_t)je * ERD;
    const int nl1 = ldc(ri + ER_NL1), nu1 = ldc(ri + ER_NU1), nl2 = ldc(ri + ER_NL2), nu2 = ldc(ri + ER_NU2);
    if (kb + NV - 1 < min(nu1, nu2 > 0 ? nu2 : nu1) || kb > max(nl1, nl2)) return;
    const int e = ldc(ri + ER_E), el1 = ldc(ri + ER_EL1), el2 = ldc(ri + ER_EL2);
    const OFF lev = 8 * (OFF)(kb - 1);
    const OFF gN = lev + 8 * (OFF)g * (OFF)t.sN, gO = lev + 8 * (OFF)g * (OFF)t.sOld;
    // byte offsets of the rows of the edge's nodes and of its upwind and downwind triangle's nodes
    const OFF o1 = 8 * (OFF)ldc(ri + ER_N1) * (OFF)L, o2 = 8 * (OFF)ldc(ri + ER_N2) * (OFF)L;
    OFF ou[3], ow[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        ou[j] = gN + 8 * (OFF)ldc(ri + ER_UA0 + j) * (OFF)L;
        ow[j] = gN + 8 * (OFF)ldc(ri + ER_DA0 + j) * (OFF)L;
    }
    // volume flux per level: the elements with that level add up
    double vf[NV], vl[GAP ? NV : 1];   // vl: the lower element's at a gap's levels, vf the upper one's
    bool act[NV], mean[NV], gap[GAP ? NV : 1], any_mean = false;
    {
        const double dX1 = ldc(rd + ER_DX1), dY1 = ldc(rd + ER_DY1), dX2 = ldc(rd + ER_DX2), dY2 = ldc(rd + ER_DY2);
        double uv1[2 * NV], h1[NV], uv2[2 * NV], h2[NV];
        const size_t q1 = (size_t)el1 * L, q2 = (size_t)(el2 >= 0 ? el2 : el1) * L;
        row_load<2 * NV>(d.uv + 2 * q1, 16u * (unsigned)(kb - 1), uv1);
        row_load<NV>(m.helem + q1, 8u * (unsigned)(kb - 1), h1);
        row_load<2 * NV>(d.uv + 2 * q2, 16u * (unsigned)(kb - 1), uv2);
        row_load<NV>(m.helem + q2, 8u * (unsigned)(kb - 1), h2);
        const int s0 = ldc(ri + ER_NZMIN), s1 = ldc(ri + ER_NZMAX);
#pragma unroll
        for (int s = 0; s < NV; ++s) {
            const int k = kb + s;
            const bool in1 = k >= nu1 && k <= nl1, in2 = nu2 > 0 && k >= nu2 && k <= nl2;
            const double f1 = (-uv1[2 * s + 1] * dX1 + uv1[2 * s] * dY1) * h1[s];
            const double f2 = (uv2[2 * s + 1] * dX2 - uv2[2 * s] * dY2) * h2[s];
            vf[s] = in1 ? (in2 ? f1 + f2 : f1) : f2;
            act[s] = in1 || in2;
            if constexpr (GAP) {
                const bool under1 = nu2 > 0 && k > nl1 && k < nu2, under2 = nu2 > 0 && k > nl2 && k < nu1;
                gap[s] = under1 || under2;
                vf[s] = under1 ? f1 : vf[s];
                vl[s] = under1 ? f2 : f1;
                act[s] = act[s] || gap[s];
            }
            // fill_up_dn_grad (oce_muscl_adv.F90:375-520): the triangles' gradients at the levels their
            // nodes share (an empty range without both triangles), else the node means
            mean[s] = act[s] && !(k >= s0 && k <= s1 - 1);
            any_mean = any_mean || mean[s];
        }
    }
    double vp[NV], vm[NV];
#pragma unroll
    for (int s = 0; s < NV; ++s) {
        vp[s] = vf[s] + fabs(vf[s]);
        vm[s] = vf[s] - fabs(vf[s]);
    }
    const double edxa = ldc(rd + ER_EDX) * ldc(rd + ER_A), edyr = ldc(rd + ER_EDY) * FGPU_R_EARTH;
    const OFF oE = lev + 8 * (OFF)g * (OFF)t.sE;
    const int trb = blockIdx.y * tpb, tre = min(t.ntr, trb + tpb);
    if (trb == 0 && g == 0) {   // K_B forms the LO fluxes again from it
        row_store<NV>(t.vf + (size_t)e * L, lev, vf, act);
        if constexpr (GAP) row_store<NV>(t.vf2 + (size_t)e * L, lev, vl, gap);
    }
    for (int tb = trb; tb < tre; tb += GT) {
        if (GT > 1 && tb + g >= tre) return;   // the last group's missing tracers
        const double *T = t.T + t.sN * tb, *Told = t.Told + t.sOld * tb;
        const int abo = ldc(t.abo + tb), lim = ldc(t.lim + tb), hor = ldc(t.hor + tb);
        double T1[NV], T2[NV], A1[NV], A2[NV], ux[3][NV], wx[3][NV];
        row_load<NV>(T, gN + o1, T1);
        row_load<NV>(T, gN + o2, T2);
        if (abo == 2) {
            row_load<NV>(Told, gO + o1, A1);
            row_load<NV>(Told, gO + o2, A2);
        }
        if (hor != HOR_UPW1) {
#pragma unroll
            for (int j = 0; j < 3; ++j) row_load<NV>(T, ou[j], ux[j]);
#pragma unroll
            for (int j = 0; j < 3; ++j) row_load<NV>(T, ow[j], wx[j]);
        }
        if (abo == 2) {   // T^AB (oce_tracer_mod.F90:44-59)
#pragma unroll
            for (int s = 0; s < NV; ++s) {
                A1[s] = -(0.5 + FGPU_EPS_AB) * A1[s] + (1.5 + FGPU_EPS_AB) * T1[s];
                A2[s] = -(0.5 + FGPU_EPS_AB) * A2[s] + (1.5 + FGPU_EPS_AB) * T2[s];
            }
        } else {
            double q1[2 * NV], q2[2 * NV];
            row_load<2 * NV>(Told, lev + gO + 2 * o1, q1);
            row_load<2 * NV>(Told, lev + gO + 2 * o2, q2);
#pragma unroll
            for (int s = 0; s < NV; ++s) {
                A1[s] = (5.0 * q1[2 * s + 1] - 16.0 * q1[2 * s] + 23.0 * T1[s]) / 12.0;
                A2[s] = (5.0 * q2[2 * s + 1] - 16.0 * q2[2 * s] + 23.0 * T2[s]) / 12.0;
            }
        }
        double f[NV];
        if (lim == LIM_FCT) {
#pragma unroll
            for (int s = 0; s < NV; ++s) {
                f[s] = -0.5 * (T1[s] * vp[s] + T2[s] * vm[s]) - 0.0;
                if constexpr (GAP)
                    if (gap[s]) f[s] = -0.5 * (T1[s] * (vl[s] + fabs(vl[s])) + T2[s] * (vl[s] - fabs(vl[s]))) - f[s];
            }
        } else {
#pragma unroll
            for (int s = 0; s < NV; ++s) f[s] = 0.0;
        }
        if (hor != HOR_UPW1) {   // MFCT, MUSCL
            const double no = ldc(t.ph + tb);
            double gr[4][NV];
#pragma unroll
            for (int s = 0; s < NV; ++s) {
                gr[0][s] = ldc(rd + ER_GU0) * ux[0][s] + ldc(rd + ER_GU1) * ux[1][s] + ldc(rd + ER_GU2) * ux[2][s];
                gr[2][s] = ldc(rd + ER_GU3) * ux[0][s] + ldc(rd + ER_GU4) * ux[1][s] + ldc(rd + ER_GU5) * ux[2][s];
                gr[1][s] = ldc(rd + ER_GD0) * wx[0][s] + ldc(rd + ER_GD1) * wx[1][s] + ldc(rd + ER_GD2) * wx[2][s];
                gr[3][s] = ldc(rd + ER_GD3) * wx[0][s] + ldc(rd + ER_GD4) * wx[1][s] + ldc(rd + ER_GD5) * wx[2][s];
            }
            if (any_mean) {
                const double *gm = t.gmean + t.sG * tb;
                const OFF oG = 2 * lev + 8 * (OFF)g * (OFF)t.sG;
                double m1[2 * NV], m2[2 * NV];
                row_load<2 * NV>(gm, oG + 2 * o1, m1);
                row_load<2 * NV>(gm, oG + 2 * o2, m2);
#pragma unroll
                for (int s = 0; s < NV; ++s) {
                    gr[0][s] = mean[s] ? m1[2 * s] : gr[0][s];
                    gr[2][s] = mean[s] ? m1[2 * s + 1] : gr[2][s];
                    gr[1][s] = mean[s] ? m2[2 * s] : gr[1][s];
                    gr[3][s] = mean[s] ? m2[2 * s + 1] : gr[3][s];
                }
            }
            double x1[NV], x2[NV], c1[NV], c2[NV];
            bool small = false;
#pragma unroll
            for (int s = 0; s < NV; ++s) {
                const double dA = 2.0 * (A2[s] - A1[s]);
                x2[s] = dA + edxa * gr[1][s] + edyr * gr[3][s];
                x1[s] = dA + edxa * gr[0][s] + edyr * gr[2][s];
                c2[s] = sixth(x2[s]);
                c1[s] = sixth(x1[s]);
                small = small || tiny(x1[s]) || tiny(x2[s]);
            }
            if (__any(small)) {
#pragma unroll
                for (int s = 0; s < NV; ++s) {
                    c2[s] = x2[s] / 6.0;
                    c1[s] = x1[s] / 6.0;
                }
            }
            if (hor == HOR_MUSCL) {   // reconstruction only down to nboundary_lay (oce_adv_tra_hor.F90:356-367)
#pragma unroll
                for (int s = 0; s < NV; ++s) {
                    c1[s] = c1[s] * (kb + s <= ldc(ri + ER_NBL1) ? 1.0 : 0.0);
                    c2[s] = c2[s] * (kb + s <= ldc(ri + ER_NBL2) ? 1.0 : 0.0);
                }
            }
#pragma unroll
            for (int s = 0; s < NV; ++s) {
                const double Tmean2 = A2[s] - c2[s], Tmean1 = A1[s] + c1[s];
                const double cHO = vp[s] * Tmean1 + vm[s] * Tmean2;
                f[s] = -0.5 * (1.0 - no) * cHO - vf[s] * no * 0.5 * (Tmean1 + Tmean2) - f[s];
                if constexpr (GAP)
                    if (gap[s]) {
                        const double c = (vl[s] + fabs(vl[s])) * Tmean1 + (vl[s] - fabs(vl[s])) * Tmean2;
                        f[s] = -0.5 * (1.0 - no) * c - vl[s] * no * 0.5 * (Tmean1 + Tmean2) - f[s];
                    }
            }
        } else {
#pragma unroll
            for (int s = 0; s < NV; ++s) {
                f[s] = -0.5 * (A1[s] * vp[s] + A2[s] * vm[s]) - f[s];
                if constexpr (GAP)
                    if (gap[s]) f[s] = -0.5 * (A1[s] * (vl[s] + fabs(vl[s])) + A2[s] * (vl[s] - fabs(vl[s]))) - f[s];
            }
        }
        row_store<NV>(t.a_h + t.sE * tb + (size_t)e * L, oE, f, act);
    }
}

// ------------------------------------------------------------------------------
// K_B: LO solution and antidiffusive vertical flux per node column
// ------------------------------------------------------------------------------
// The edges' LO fluxes are formed again from the volume fluxes and the T of the
// neighbours, whose rows a node's edges share, where a stored LO flux is a row
// per edge and tracer, three times as many. Levels exchange values by wave
// shifts. Against a block per column, 12 thousand nodes, 47 layers, 32 tracers:
// 352 -> 281 us; 40 thousand nodes, 70 layers, 10 tracers: 537 -> 518; 126,858
// nodes, 47 layers, 2 tracers: 291 -> 298, against K_A's gain.
// KB_XV compiles in the CDIFF and PPM tracers; PPM reads up to four layers around
// an interface, from LDS. KB_WS compiles in the W split (use_wsplit), where the HO
// scheme is handed the upwind flux with the full W and the LO solution of FCT
// tracers takes the implicit upwind advection with w_i afterwards (K_V on it). Each
// has its own registers: 120 thousand nodes, 12 layers, 1 tracer 169 us with the W
// split and 305 with PPM (168 without either), 299 and 414 where one form carried
// both and ran two waves per SIMD. So one level per lane is held to the registers
// of four waves, three with PPM.
#define KB_XV 1    // CDIFF and PPM
#define KB_GAP 2
#define KB_WS 4    // the W split
template <typename OFF, int NV, int GT, int FORM>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(NV > 1 || (FORM & KB_GAP) ? 1 : (FORM & KB_XV ? 3 : 4))))
kB_cols(DevMesh m, DevDyn d, DevTracers t, double dt, int tpb)
{
    constexpr bool XV = (FORM & KB_XV) != 0, GAP = (FORM & KB_GAP) != 0, WS = (FORM & KB_WS) != 0;
    Column<OFF, NV, GT> c;
    if (!load_column<(NV > 1), OFF, NV, GT>(m, t, c)) return;
    static_assert(!XV || GT == 1, "one column's rows in LDS");
    __shared__ double sT[XV ? 64 * NV : 1], sHn[XV ? 64 * NV : 1], sHo[XV ? 64 * NV : 1];
    __shared__ double sW[XV ? 64 * NV : 1], sWe[XV ? 64 * NV : 1], sAr[XV ? 64 * NV : 1];
    const int nzmin = c.nzmin, nzmax = c.nzmax;
    const int L = m.L;
    bool first[NV], inner[NV], deep[NV], last[NV], face[NV];
    double W[NV], We[NV], ar[NV], hn[NV], hh[NV], av[NV], dz[NV], d1[NV], d2[NV];
    constexpr int NB = NV == 1 ? 8 : 3;   // edges whose loads are issued together
    constexpr bool VREG = NV == 1;        // the edges' volume fluxes stay in registers over the tracers
    double vf[VREG ? CE : NB][NV];
    {
        const size_t nL = (size_t)c.n * L, nNL = (size_t)c.n * m.NL;
        const unsigned oL = 8u * (unsigned)(c.kc - 1), oI = 8u * (unsigned)((c.kb <= m.NL ? c.kb : 1) - 1);
        double z[NV], zu[NV], zb[NV];
        row_load<NV>(d.w + nNL, oI, W);
        row_load<NV>(d.w_e + nNL, oI, We);
        row_load<NV>(m.area + nNL, oI, ar);
        row_load<NV>(m.zbar3d + nNL, oI, zb);
        row_load<NV>(m.areasvol + nNL, oI, av);
        row_load<NV>(m.hnode_new + nL, oL, hn);
        row_load<NV>(m.hnode + nL, oL, hh);
        row_load<NV>(m.Z3d + nL, oL, z);
        if constexpr (VREG) {
#pragma unroll
            for (int u = 0; u < CE; ++u)
                if (u < c.deg) row_load<NV>(t.vf, c.oe[u] - 8 * (OFF)c.g * (OFF)t.sE, vf[u]);
        }
        col_up<NV>(z, zu);
#pragma unroll
        for (int s = 0; s < NV; ++s) {
            const int k = c.kb + s;
            first[s] = k == nzmin;
            last[s] = k == nzmax;
            inner[s] = k >= nzmin + 1 && k <= nzmax - 1;
            deep[s] = k >= nzmin + 2 && k <= nzmax - 2;
            face[s] = k >= nzmin && k <= nzmax;
            dz[s] = zu[s] - z[s];
            d1[s] = zb[s] - z[s];
            d2[s] = zb[s] - zu[s];
            if constexpr (XV) {
                const int i = c.kb + s - 1;
                sHn[i] = hn[s];
                sHo[i] = hh[s];
                sW[i] = W[s];
                sWe[i] = We[s];
                sAr[i] = ar[s];
            }
        }
    }
    const int trb = blockIdx.y * tpb, tre = min(t.ntr, trb + tpb);
    for (int tb = trb; tb < tre; tb += GT) {
        if (GT > 1 && tb + c.g >= tre) return;   // the last group's missing tracers
        const int abo = ldc(t.abo + tb), lim = ldc(t.lim + tb), ver = ldc(t.ver + tb);
        const double pv = ldc(t.pv + tb);
        const bool fct = lim == LIM_FCT;
        const double *T = t.T + t.sN * tb, *Told = t.Told + t.sOld * tb;
        double Tk[NV], A[NV], Tu[NV], Au[NV], tm[NB][NV];
        row_load<NV>(T, c.own, Tk);
        const OFF oO = 8 * ((OFF)(c.kc - 1) + (OFF)c.g * (OFF)t.sOld);
        if (abo == 2) row_load<NV>(Told + (size_t)c.n * L, oO, A);
        if (abo == 2) {   // T^AB (oce_tracer_mod.F90:44-59)
#pragma unroll
            for (int s = 0; s < NV; ++s) A[s] = -(0.5 + FGPU_EPS_AB) * A[s] + (1.5 + FGPU_EPS_AB) * Tk[s];
        } else {
            double p[2 * NV];
            row_load<2 * NV>(Told + 2 * (size_t)c.n * L, oO + 8 * (OFF)(c.kc - 1), p);
#pragma unroll
            for (int s = 0; s < NV; ++s) A[s] = (5.0 * p[2 * s + 1] - 16.0 * p[2 * s] + 23.0 * Tk[s]) / 12.0;
        }
        col_up<NV>(Tk, Tu);
        col_up<NV>(A, Au);
        // LO flux at interface k: upwind with w_e
        double lk[NV], f[NV], lw[NV];   // lw: with the full W, what the HO flux has taken off
#pragma unroll
        for (int s = 0; s < NV; ++s) {
            const double a = -We[s] * Tk[s] * ar[s];
            const double b = -0.5 * (Tk[s] * (We[s] + fabs(We[s])) + Tu[s] * (We[s] - fabs(We[s]))) * ar[s];
            lk[s] = fct ? (first[s] ? a : (inner[s] ? b : 0.0)) : 0.0;
            lw[s] = lk[s];
            if (WS && d.wsplit) {
                const double x = -W[s] * Tk[s] * ar[s];
                const double y = -0.5 * (Tk[s] * (W[s] + fabs(W[s])) + Tu[s] * (W[s] - fabs(W[s]))) * ar[s];
                lw[s] = fct ? (first[s] ? x : (inner[s] ? y : 0.0)) : 0.0;
            }
        }
        // HO flux minus the LO one (oce_adv_tra_ver.F90:332-434, 244-328)
        if (ver == VER_QR4C) {
            double qc[NV], qu[NV], qd[NV], x1[NV], x2[NV], y1[NV], y2[NV];
#pragma unroll
            for (int s = 0; s < NV; ++s) qc[s] = (Au[s] - A[s]) / dz[s];   // the slope over interface k
            col_down<NV>(qc, qu);
            col_up<NV>(qc, qd);
            bool small = false;
#pragma unroll
            for (int s = 0; s < NV; ++s) {
                x1[s] = (2 * qc[s] + qu[s]) * d1[s];
                x2[s] = (2 * qc[s] + qd[s]) * d2[s];
                y1[s] = third(x1[s]);
                y2[s] = third(x2[s]);
                small = small || (deep[s] && (tiny(x1[s]) || tiny(x2[s])));
            }
            if (__any(small)) {
#pragma unroll
                for (int s = 0; s < NV; ++s) {
                    y1[s] = x1[s] / 3.0;
                    y2[s] = x2[s] / 3.0;
                }
            }
#pragma unroll
            for (int s = 0; s < NV; ++s) {
                const double ww = fct ? W[s] : We[s];
                const double Tmean1 = A[s] + y1[s], Tmean2 = Au[s] + y2[s];
                const double Tmean = (ww + fabs(ww)) * Tmean1 + (ww - fabs(ww)) * Tmean2;
                const double ho = (-0.5 * (1.0 - pv) * Tmean - pv * (0.5 * (Tmean1 + Tmean2)) * ww) * ar[s];
                const double top = -A[s] * ww * ar[s];
                const double near = -0.5 * (Au[s] + A[s]) * ww * ar[s];   // next to the surface and the bottom
                f[s] = (first[s] ? top : (deep[s] ? ho : (last[s] ? 0.0 : near))) - lw[s];
                if (nzmax - nzmin == 2 && inner[s]) f[s] = near - f[s];   // both rows at once
            }
        } else if (XV && ver == VER_PPM) {
            wave_sync();
#pragma unroll
            for (int s = 0; s < NV; ++s) sT[c.kb + s - 1] = A[s];
            wave_sync();
#pragma unroll
            for (int s = 0; s < NV; ++s)
                f[s] = face[s] ? ver_ppm(c.kb + s, nzmin, nzmax, sT, fct ? sW : sWe, sAr, sHn, sHo, dt, lw[s]) : 0.0;
        } else {
#pragma unroll
            for (int s = 0; s < NV; ++s) {
                const double ww = fct ? W[s] : We[s];
                const double a = -ww * A[s] * ar[s];
                if (XV && ver == VER_CDIFF) {   // adv_tra_ver_cdiff (oce_adv_tra_ver.F90:635-695)
                    const double b = -(0.5 * (Au[s] + A[s])) * ww * ar[s];
                    f[s] = first[s] ? a - lw[s] : (inner[s] ? b - lw[s] : lw[s]);
                } else {
                    const double b = -0.5 * (A[s] * (ww + fabs(ww)) + Au[s] * (ww - fabs(ww))) * ar[s];
                    f[s] = (first[s] ? a : (inner[s] ? b : 0.0)) - lw[s];
                }
            }
        }
        row_store<NV>(t.a_v + t.sNI * tb, c.ownI, f, face);
        if (!fct) continue;
        // the edges' LO fluxes, formed again from the volume fluxes, in ascending order
        double acc[NV];
#pragma unroll
        for (int s = 0; s < NV; ++s) acc[s] = 0.0;
        int kb = c.kb;
        if constexpr (NV > 1) asm volatile("" : "+v"(kb));   // the level masks are formed in place: they would not fit the scalar registers
        auto add = [&](int u, OFF oe, int side, const double (&v)[NV], const double (&to)[NV], int a0, int len)
            __attribute__((always_inline)) {
            if constexpr (GAP) {
                int g0, g1;
                edge_gap(m, c.p0 + u, g0, g1);
                if (g0 <= g1) {   // the edge's levels one by one, both fluxes in the gap
                    double w[NV];
                    row_load<NV>(t.vf2, oe - 8 * (OFF)c.g * (OFF)t.sE, w);
#pragma unroll
                    for (int s = 0; s < NV; ++s) {
                        const double x1 = side ? to[s] : Tk[s], x2 = side ? Tk[s] : to[s];
                        double z = -0.5 * (x1 * (v[s] + fabs(v[s])) + x2 * (v[s] - fabs(v[s]))) - 0.0;
                        const double zl = -0.5 * (x1 * (w[s] + fabs(w[s])) + x2 * (w[s] - fabs(w[s]))) - z;
                        z = kb + s >= g0 && kb + s <= g1 ? zl : z;
                        const double x = side ? acc[s] - z : acc[s] + z;
                        acc[s] = edge_has(kb, s, a0, len) ? x : acc[s];
                    }
                    return;
                }
            }
            // side 0: acc + -0.5 (Tk (v + |v|) + to (v - |v|)); side 1: acc - -0.5 (to (v + |v|) + Tk (v - |v|))
            const long long sgn = (long long)side << 63;
            const double half = side ? 0.5 : -0.5;
#pragma unroll
            for (int s = 0; s < NV; ++s) {
                const double a = signed_by(fabs(v[s]), sgn);
                const double x = acc[s] + half * (Tk[s] * (v[s] + a) + to[s] * (v[s] - a));
                acc[s] = edge_has(kb, s, a0, len) ? x : acc[s];
            }
        };
#pragma unroll
        for (int u0 = 0; u0 < CE; u0 += NB) {
            if (u0 < c.deg) {
#pragma unroll
                for (int u = 0; u < NB; ++u) {
                    if (u0 + u >= CE || u0 + u >= c.deg) break;
                    row_load<NV>(T, c.on[u0 + u], tm[u]);
                    if constexpr (!VREG) row_load<NV>(t.vf, c.oe[u0 + u] - 8 * (OFF)c.g * (OFF)t.sE, vf[u]);
                }
#pragma unroll
                for (int u = 0; u < NB; ++u)
                    if (u0 + u < CE && u0 + u < c.deg) add(u0 + u, c.oe[u0 + u], c.side[u0 + u], vf[VREG ? u0 + u : u], tm[u], c.a0[u0 + u], c.len[u0 + u]);
            }
        }
        for (int u = CE; u < c.deg; ++u) {
            OFF on, oe;
            int a0, len, side;
            edge_offsets<OFF, NV, GT>(m, t, c, u, on, oe, a0, len, side);
            double v[NV], to[NV];
            row_load<NV>(t.vf, oe - 8 * (OFF)c.g * (OFF)t.sE, v);
            row_load<NV>(T, on, to);
            add(u, oe, side, v, to, a0, len);
        }
        double ld[NV], o[NV];
        col_down<NV>(lk, ld);
#pragma unroll
        for (int s = 0; s < NV; ++s) o[s] = (Tk[s] * hh[s] + (acc[s] + (lk[s] - ld[s])) * dt / av[s]) / hn[s];
        row_store<NV>(t.fct_lo + t.sN * tb, c.own, o, c.wet);
    }
}

// ------------------------------------------------------------------------------
// K_C: FCT bounds, P+/P-, R+/R- per node column (oce_adv_tra_fct.F90:119-405)
// The element bound (max over the 3 nodes of max(LO, T^n)), maximised over the
// elements around the node, equals the maximum over the node and those edge
// neighbours m for which an element adjacent to edge (n, m) has the level,
// together with the padding -1e3 (max) / +1e3 (min) of every element around
// the node that lacks the level (oce_adv_tra_fct.F90:148-178).
// ------------------------------------------------------------------------------
// Against a block per column, 126,858 nodes, 47 layers, 2 tracers: 347 -> 315 us;
// 12 thousand nodes, 32 tracers: 482 -> 382; 40 thousand nodes, 70 layers, 10
// tracers: 745 -> 647.
// GAP: in a level gap neither element has the level, and the other node is no
// part of its bounds.
template <typename OFF, int NV, int GT, bool GAP>
__global__ void __launch_bounds__(64) kC_cols(DevMesh m, DevTracers t, double dt, int tpb)
{
    Column<OFF, NV, GT> c;
    if (!load_column<true, OFF, NV, GT>(m, t, c)) return;
    const int L = m.L;
    const int pad0 = ldc(m.fct_pad + 2 * (size_t)c.n), pad1 = ldc(m.fct_pad + 2 * (size_t)c.n + 1);
    double av[NV], hn[NV];
    row_load<NV>(m.areasvol + (size_t)c.n * m.NL, 8u * (unsigned)(c.kc - 1), av);
    row_load<NV>(m.hnode_new + (size_t)c.n * L, 8u * (unsigned)(c.kc - 1), hn);
    bool padded[NV], alone[NV];
#pragma unroll
    for (int s = 0; s < NV; ++s) {
        const int k = c.kb + s;
        padded[s] = k < pad0 || k >= pad1;   // an element around n lacks level k
        alone[s] = k == c.nzmax - 1 || k == c.nzmin;
    }
    const int trb = blockIdx.y * tpb, tre = min(t.ntr, trb + tpb);
    for (int tb = trb; tb < tre; tb += GT) {
        if (GT > 1 && tb + c.g >= tre) return;   // the last group's missing tracers
        if (ldc(t.lim + tb) != LIM_FCT) continue;
        const double *T = t.T + t.sN * tb, *LO = t.fct_lo + t.sN * tb, *ah = t.a_h + t.sE * tb;
        double lo[NV], tk[NV], f[NV], fd[NV], vmax[NV], vmin[NV], p[NV], q[NV];
        row_load<NV>(LO, c.own, lo);
        row_load<NV>(T, c.own, tk);
        row_load<NV>(t.a_v + t.sNI * tb, c.ownI, f);
        constexpr int NB = NV == 1 || GT == 1 ? 3 : 4;   // edges whose loads are issued together
        double lm[NB][NV], tm[NB][NV], fl[NB][NV];
        auto load = [&](int u0) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                if (u0 + u >= CE || u0 + u >= c.deg) break;
                row_load<NV>(LO, c.on[u0 + u], lm[u]);
                row_load<NV>(T, c.on[u0 + u], tm[u]);
                row_load<NV>(ah, c.oe[u0 + u], fl[u]);
            }
        };
        int kb = c.kb;
        if constexpr (NV > 1) asm volatile("" : "+v"(kb));   // see K_B
        auto add = [&](int u, int side, const double (&a)[NV], const double (&b)[NV], const double (&x)[NV], int a0, int len)
            __attribute__((always_inline)) {
            const long long sgn = (long long)side << 63;
            int g0 = 1, g1 = 0;
            if constexpr (GAP) edge_gap(m, c.p0 + u, g0, g1);
#pragma unroll
            for (int s = 0; s < NV; ++s) {
                const bool has = edge_has(kb, s, a0, len);
                if constexpr (NV == 1 && !GAP) {   // outside the edge's levels a and b are the column's own values
                    vmax[s] = dmx(vmax[s], dmx(a[s], b[s]));
                    vmin[s] = dmn(vmin[s], dmn(a[s], b[s]));
                } else {
                    const double hi = dmx(vmax[s], dmx(a[s], b[s])), lw = dmn(vmin[s], dmn(a[s], b[s]));
                    const bool in = has && !(GAP && kb + s >= g0 && kb + s <= g1);
                    vmax[s] = in ? hi : vmax[s];
                    vmin[s] = in ? lw : vmin[s];
                }
                const double y = has ? signed_by(x[s], sgn) : 0.0;
                p[s] = p[s] + dmx(0.0, y);
                q[s] = q[s] + dmn(0.0, y);
            }
        };
        load(0);
        col_down<NV>(f, fd);
#pragma unroll
        for (int s = 0; s < NV; ++s) {
            vmax[s] = dmx(lo[s], tk[s]);
            vmin[s] = dmn(lo[s], tk[s]);
            vmax[s] = padded[s] ? dmx(vmax[s], -1e3) : vmax[s];
            vmin[s] = padded[s] ? dmn(vmin[s], 1e3) : vmin[s];
            p[s] = 0.0 + (dmx(0.0, f[s]) + dmx(0.0, -fd[s]));
            q[s] = 0.0 + (dmn(0.0, f[s]) + dmn(0.0, -fd[s]));
        }
#pragma unroll
        for (int u0 = 0; u0 < CE; u0 += NB) {
            if (u0 < c.deg) {
                if (u0 > 0) load(u0);
#pragma unroll
                for (int u = 0; u < NB; ++u)
                    if (u0 + u < CE && u0 + u < c.deg) add(u0 + u, c.side[u0 + u], lm[u], tm[u], fl[u], c.a0[u0 + u], c.len[u0 + u]);
            }
        }
        for (int u = CE; u < c.deg; ++u) {
            OFF on, oe;
            int a0, len, side;
            edge_offsets<OFF, NV, GT>(m, t, c, u, on, oe, a0, len, side);
            double a[NV], b[NV], x[NV];
            row_load<NV>(LO, on, a);
            row_load<NV>(T, on, b);
            row_load<NV>(ah, oe, x);
            add(u, side, a, b, x, a0, len);
        }
        double mxu[NV], mxd[NV], mnu[NV], mnd[NV], rp[NV], rm[NV];
        col_up<NV>(vmax, mxu);
        col_down<NV>(vmax, mxd);
        col_up<NV>(vmin, mnu);
        col_down<NV>(vmin, mnd);
#pragma unroll
        for (int s = 0; s < NV; ++s) {
            const double hi = dmx(dmx(mxu[s], vmax[s]), mxd[s]), lw = dmn(dmn(mnu[s], vmin[s]), mnd[s]);
            const double bmax = (alone[s] ? vmax[s] : hi) - lo[s], bmin = (alone[s] ? vmin[s] : lw) - lo[s];
            rp[s] = dmn(1.0, bmax / (p[s] * dt / av[s] / hn[s] + 1e-16));
            rm[s] = dmn(1.0, bmin / (q[s] * dt / av[s] / hn[s] - 1e-16));
        }
        row_store<NV>(t.rp + t.sN * tb, c.own, rp, c.wet);
        row_store<NV>(t.rm + t.sN * tb, c.own, rm, c.wet);
    }
}

// ------------------------------------------------------------------------------
// K_L: limited fluxes, flux2dtracer and T* (oce_adv_tra_fct.F90:425-497,
// oce_adv_tra_driver.F90:494-646, oce_ale_tracer.F90:595-626); T* replaces T,
// T^n goes to valuesold. The implicit vertical diffusion follows in K_V: inside
// the column's wave its sweeps kept 2 to 10 of 64 lanes busy for most of the
// kernel's instructions. One kernel for both, a block per column, took 775 us at
// 126,858 nodes, 47 layers, 2 tracers (K_L 350 us, K_V 160), 988 us at 12 thousand
// nodes, 32 tracers (420, 150) and 1429 us at 40 thousand nodes, 70 layers, 10
// tracers (688, 309).
// ------------------------------------------------------------------------------
// DX compiles in the explicit diffusion increments (Ki, Redi, i_vert_diff off):
// 20 thousand nodes, 47 layers, 4 tracers: K_L 157 us and K_V 92, 361 for one
// kernel with a block per column.
template <typename OFF, int NV, int GT, bool DX>
__global__ void __launch_bounds__(64) kL_node(DevMesh m, DevDyn d, DevTracers t, double dt, int tpb)
{
    Column<OFF, NV, GT> c;
    if (!load_column<true, OFF, NV, GT>(m, t, c)) return;
    const int L = m.L;
    double av[NV], hn[NV], hh[NV];
    row_load<NV>(m.areasvol + (size_t)c.n * m.NL, 8u * (unsigned)(c.kc - 1), av);
    row_load<NV>(m.hnode_new + (size_t)c.n * L, 8u * (unsigned)(c.kc - 1), hn);
    row_load<NV>(m.hnode + (size_t)c.n * L, 8u * (unsigned)(c.kc - 1), hh);
    bool first[NV], lim_[NV];
#pragma unroll
    for (int s = 0; s < NV; ++s) {
        first[s] = c.kb + s == c.nzmin;
        lim_[s] = c.kb + s <= c.nzmax - 1;
    }
    const int trb = blockIdx.y * tpb, tre = min(t.ntr, trb + tpb);
    for (int tb = trb; tb < tre; tb += GT) {
        if (GT > 1 && tb + c.g >= tre) return;   // the last group's missing tracers
        const bool fct = ldc(t.lim + tb) == LIM_FCT;
        const int abo = ldc(t.abo + tb);
        double *T = t.T + t.sN * tb;
        const double *rpT = t.rp + t.sN * tb, *rmT = t.rm + t.sN * tb, *ah = t.a_h + t.sE * tb;
        double rp[NV], rm[NV], Tk[NV], lo[NV], f[NV], h[NV], v[NV];
#pragma unroll
        for (int s = 0; s < NV; ++s) rp[s] = rm[s] = lo[s] = 1.0;
        constexpr int NB = NV == 1 ? 4 : (NV == 2 ? 2 : 3);   // edges whose loads are issued together
        double fl[NB][NV], rpo[NB][NV], rmo[NB][NV];
        int kb = c.kb;
        if constexpr (NV > 1) asm volatile("" : "+v"(kb));   // see K_B
        row_load<NV>(t.a_v + t.sNI * tb, c.ownI, f);
        row_load<NV>(T, c.own, Tk);
        if (fct) {
            row_load<NV>(rpT, c.own, rp);
            row_load<NV>(rmT, c.own, rm);
            row_load<NV>(t.fct_lo + t.sN * tb, c.own, lo);
        }
        auto load = [&](int u0) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                if (u0 + u >= CE || u0 + u >= c.deg) break;
                row_load<NV>(ah, c.oe[u0 + u], fl[u]);
                if (fct) {
                    row_load<NV>(rpT, c.on[u0 + u], rpo[u]);
                    row_load<NV>(rmT, c.on[u0 + u], rmo[u]);
                }
            }
        };
        // node 1 takes R+ of an inflow, node 2 R- of the same flux, and the other way round
        auto add = [&](int side, const double (&x)[NV], const double (&po)[NV], const double (&mo)[NV], int a0, int len)
            __attribute__((always_inline)) {
            const long long sgn = (long long)side << 63;
#pragma unroll
            for (int s = 0; s < NV; ++s) {
                double y = x[s];
                if (fct) {
                    const bool plus = (x[s] >= 0.0) != (side != 0);
                    const double own = plus ? rp[s] : rm[s], oth = plus ? mo[s] : po[s];
                    // min(min(1, R of node 1), R of node 2), R <= 1
                    const bool mine = side ? !(oth < own) : own < oth;
                    y = (mine ? own : oth) * y;
                }
                const double hs = h[s] + signed_by(y * dt / av[s], sgn);
                h[s] = edge_has(kb, s, a0, len) ? hs : h[s];
            }
        };
        load(0);
        // limited vertical antidiffusive flux at interface k (oce_adv_tra_fct.F90:425-456)
        {
            double rpu[NV], rmu[NV], fd[NV];
            if (fct) {
                col_up<NV>(rp, rpu);
                col_up<NV>(rm, rmu);
#pragma unroll
                for (int s = 0; s < NV; ++s) {
                    const double flux = f[s];
                    const bool pos = flux >= 0.0;
                    // above the interface R- (R+) of the layer, below it R+ (R-); none above the top one
                    const double below = pos ? rp[s] : rm[s], above = pos ? rmu[s] : rpu[s];
                    double ae = first[s] ? 1.0 : dmn(1.0, above);
                    ae = dmn(ae, below);
                    f[s] = lim_[s] ? ae * flux : flux;
                }
            }
            col_down<NV>(f, fd);
#pragma unroll
            for (int s = 0; s < NV; ++s) {
                h[s] = 0.0;
                v[s] = 0.0;
                if (fct) v[s] = v[s] - Tk[s] * hh[s] + lo[s] * hn[s];
                v[s] = v[s] + (f[s] - fd[s]) * dt / av[s];
            }
        }
#pragma unroll
        for (int u0 = 0; u0 < CE; u0 += NB) {
            if (u0 < c.deg) {
                if (u0 > 0) load(u0);
#pragma unroll
                for (int u = 0; u < NB; ++u)
                    if (u0 + u < CE && u0 + u < c.deg) add(c.side[u0 + u], fl[u], rpo[u], rmo[u], c.a0[u0 + u], c.len[u0 + u]);
            }
        }
        for (int u = CE; u < c.deg; ++u) {
            OFF on, oe;
            int a0, len, side;
            edge_offsets<OFF, NV, GT>(m, t, c, u, on, oe, a0, len, side);
            double x[NV], po[NV], mo[NV];
            row_load<NV>(ah, oe, x);
            if (fct) {
                row_load<NV>(rpT, on, po);
                row_load<NV>(rmT, on, mo);
            }
            add(side, x, po, mo, a0, len);
        }
        double ts[NV], del[NV];
#pragma unroll
        for (int s = 0; s < NV; ++s) {
            del[s] = 0.0 + h[s] + v[s];
        }
        if constexpr (DX) {
            // in diff_tracers_ale's order (oce_ale_tracer.F90:595-626): edge fluxes of diff_part_hor_redi
            // ascending, then the vertical parts
            auto diff = [&](int side, const double (&x)[NV], int a0, int len) __attribute__((always_inline)) {
#pragma unroll
                for (int s = 0; s < NV; ++s) {
                    const double r = side ? 0.0 - x[s] : 0.0 + x[s];
                    const double y = del[s] + r * dt / av[s];
                    del[s] = edge_has(kb, s, a0, len) ? y : del[s];
                }
            };
            if (d.hdiff) {
                const double *hd = t.hd + t.sE * tb;
#pragma unroll
                for (int u0 = 0; u0 < CE; u0 += NB) {
                    if (u0 < c.deg) {
#pragma unroll
                        for (int u = 0; u < NB; ++u) {
                            if (u0 + u >= CE || u0 + u >= c.deg) break;
                            row_load<NV>(hd, c.oe[u0 + u], fl[u]);
                        }
#pragma unroll
                        for (int u = 0; u < NB; ++u)
                            if (u0 + u < CE && u0 + u < c.deg) diff(c.side[u0 + u], fl[u], c.a0[u0 + u], c.len[u0 + u]);
                    }
                }
                for (int u = CE; u < c.deg; ++u) {
                    OFF on, oe;
                    int a0, len, side;
                    edge_offsets<OFF, NV, GT>(m, t, c, u, on, oe, a0, len, side);
                    double x[NV];
                    row_load<NV>(hd, oe, x);
                    diff(side, x, a0, len);
                }
            }
            double x[NV];
            if (!t.ivd[tb + c.g]) {
                row_load<NV>(t.ve + t.sN * tb, c.own, x);
#pragma unroll
                for (int s = 0; s < NV; ++s) del[s] = del[s] + x[s];
            }
            if (d.redi) {
                row_load<NV>(t.vr + t.sN * tb, c.own, x);
#pragma unroll
                for (int s = 0; s < NV; ++s) del[s] = del[s] + x[s];
            }
        }
#pragma unroll
        for (int s = 0; s < NV; ++s) {
            del[s] = del[s] + Tk[s] * (hh[s] - hn[s]);
            ts[s] = Tk[s] + del[s] / hn[s];
        }
        row_store<NV>(T, c.own, ts, c.wet);
        // valuesold rotation (oce_tracer_mod.F90:94-123)
        double *Told = t.Told + t.sOld * (size_t)(GT == 1 ? tb : tb + c.g) + (size_t)(abo - 1) * ((size_t)c.n * L + c.kc - 1);
        if (abo == 2) {
            row_store<NV>(Told, 0u, Tk, c.wet);
        } else {
#pragma unroll
            for (int s = 0; s < NV; ++s) {
                if (!c.wet[s]) continue;
                Told[2 * s + 1] = Told[2 * s];
                Told[2 * s] = Tk[s];
            }
        }
    }
}

// ------------------------------------------------------------------------------
// K_V: implicit vertical diffusion of T* in place (diff_ver_part_impl_ale,
// oce_ale_tracer.F90:907-1435) and the salinity clamp. Bound by the latency of
// a block: three dependent loads, the rows, and two serial passes over the
// levels (about 200 cycles a level for the two dependent divisions).
// ------------------------------------------------------------------------------
// A block of up to eight waves takes NC columns x TB tracers, NC x TB <= 64 rows.
// Each wave forms the tridiagonal rows and right-hand sides of its columns with
// lanes over the levels, of 64 >> lsh columns at once (SH), and leaves them in LDS; one wave sweeps with one lane
// per row, and the waves add the result to T*. LDS rows have an odd length, so
// that the lanes of the sweep, each on its own row, use different banks. Eight
// waves per SIMD leave the plain form 64 registers, of which two levels per lane
// spill 7 (32 bytes a lane); several columns per wave need more, and six waves do.
// XF bit 0 (use_wsplit): the non-FCT tracers' rows also take the implicit part
// w_i of the split W, a second set of rows; bit 1: the K33 terms of Redi and
// tracers with i_vert_diff off, which are left as they are. KV_LO instead solves
// the implicit upwind advection with w_i on the LO solution of the FCT tracers
// (adv_tra_vert_impl, oce_adv_tra_ver.F90:90-240), between K_B and K_C.
#define KV_WS 1
#define KV_DX 2
#define KV_LO 4
#define KV_NW 8   // waves of a block at most
#define KV_TP 2   // tracers whose rows are loaded together
template <int NV, int XF, bool SH>
__global__ void __launch_bounds__(64 * KV_NW) __attribute__((amdgpu_waves_per_eu(XF == 0 ? (SH ? 6 : 8) : 4)))
kV_cols(DevMesh m, DevDyn d, DevTracers t, int tr0, int ntr, double dt, int all, int clamp_tracer, int NC, int TB, int lsh)
{
    extern __shared__ double lds[];
    const int L = m.L, NL = m.NL, RS = L | 1;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
    const int part = SH ? lane >> lsh : 0, step = (int)(blockDim.x >> 6) << (SH ? 6 - lsh : 0);
    const int col0 = xcd_unit() * NC;
    if (col0 >= m.N2) return;
    const int ncol = min(NC, m.N2 - col0);
    const int trb = tr0 + blockIdx.y * TB, ntb = min(TB, tr0 + ntr - trb);
    constexpr bool WS = (XF & KV_WS) != 0, LO = (XF & KV_LO) != 0;
    const bool redi = (XF & KV_DX) != 0 && d.redi != 0;
    const size_t set = 3 * (size_t)NC * RS;   // the rows' second set follows the first
    double *sa = lds, *sb = sa + (size_t)NC * RS, *sc = sb + (size_t)NC * RS, *sr = lds + (WS ? 2 : 1) * set;
    double *F = LO ? t.fct_lo : t.T;
    // does the solve take tracer tr, and with the second set?
    auto solved = [&](int tr) { return LO ? ldc(t.lim + tr) == LIM_FCT : (XF == 0 || all || ldc(t.ivd + tr) != 0); };
    auto second = [&](int tr) { return WS && ldc(t.lim + tr) != LIM_FCT; };
    // the block's columns, one per lane
    const int *rec = m.col_rec + 8 * (size_t)(col0 + min(lane, ncol - 1));
    const int nl_ = rec[0], z0l = rec[3], z1l = rec[4];
    const int kb = (SH ? lane & ((1 << lsh) - 1) : lane) * NV + 1;
    const unsigned off = 8u * (unsigned)(kb - 1);
    // the lane's column of the block, the wave's one without SH; past the last one a lane has no level
    auto column = [&](int c, int &n, int &nzmin, int &nzmax) __attribute__((always_inline)) {
        if constexpr (SH) {
            const int at = min(c, ncol - 1);
            n = __shfl(nl_, at);
            nzmin = __shfl(z0l, at);
            nzmax = __shfl(z1l, at);
            if (c >= ncol) nzmax = 0;
        } else {
            n = rl(nl_, c);
            nzmin = rl(z0l, c);
            nzmax = rl(z1l, c);
        }
    };
    for (int c0 = SH ? w << (6 - lsh) : w; c0 < ncol; c0 += step) {
        const int c = c0 + part;
        int n, nzmin, nzmax;
        column(c, n, nzmin, nzmax);
        const size_t nL = (size_t)n * L, nNL = (size_t)n * NL;
        double hn[NV], av[NV], zk[NV], kv[NV], ar[NV], zu[NV], zd[NV], kvd[NV], ard[NV], a_[NV], c_[NV], bd_[NV];
        double ts[KV_TP][NV], wi[NV], wid[NV], wa[WS ? NV : 1], wb[WS ? NV : 1], wc[WS ? NV : 1], k33[NV], k33u[NV];
#pragma unroll
        for (int s = 0; s < NV; ++s) {
            hn[s] = av[s] = zk[s] = kv[s] = ar[s] = 1.0;
            wi[s] = k33[s] = 0.0;
#pragma unroll
            for (int j = 0; j < KV_TP; ++j) ts[j][s] = 0.0;
        }
        const bool layer = kb <= nzmax - 1;
        if (kb <= nzmax) {   // interfaces to nzmax
            if (!LO) row_load<NV>(d.Kv + nNL, off, kv);
            if (WS || LO) row_load<NV>(d.w_i + nNL, off, wi);
            row_load<NV>(m.area + nNL, off, ar);
            row_load<NV>(m.areasvol + nNL, off, av);
        }
        if (layer) {
            row_load<NV>(m.hnode_new + nL, off, hn);
            if (!LO) row_load<NV>(m.zn_vd + nL, off, zk);
#pragma unroll
            for (int j = 0; j < KV_TP; ++j)
                if (j < ntb) row_load<NV>(F + t.sN * (trb + j) + nL, off, ts[j]);
        }
        col_up<NV>(zk, zu);
        col_down<NV>(zk, zd);
        col_down<NV>(kv, kvd);
        col_down<NV>(ar, ard);
        col_down<NV>(wi, wid);
        if (redi) {   // K33 = Kv + Ki S3^2 at the interface below a layer (oce_ale_tracer.F90:1105-1108, 1138-1144, 1181-1184)
            double s3[NV], ki[NV], zb[NV], s3d[NV], kid[NV], zbd[NV];
#pragma unroll
            for (int s = 0; s < NV; ++s) s3[s] = ki[s] = zb[s] = 0.0;
            if (kb <= nzmax) row_load<NV>(m.zbn_vd + nNL, off, zb);
            if (layer) {
                row_load<NV>(d.Ki + nL, off, ki);
#pragma unroll
                for (int s = 0; s < NV; ++s) s3[s] = d.slope[3 * (nL + kb - 1 + (kb + s <= L ? s : 0)) + 2];
            }
            col_down<NV>(s3, s3d);
            col_down<NV>(ki, kid);
            col_down<NV>(zb, zbd);
#pragma unroll
            for (int s = 0; s < NV; ++s) {
                const double zinv2 = 1.0 / (zk[s] - zd[s]);
                k33[s] = (zbd[s] - zd[s]) * zinv2 * (s3[s] * s3[s]) * ki[s] +
                         (zk[s] - zbd[s]) * zinv2 * (s3d[s] * s3d[s]) * kid[s];
            }
        }
        col_up<NV>(k33, k33u);
        // tridiagonal coefficients (oce_ale_tracer.F90:1098-1175)
#pragma unroll
        for (int s = 0; s < NV; ++s) {
            const int k = kb + s;
            a_[s] = c_[s] = bd_[s] = 0.0;
            if (k < nzmin || k > nzmax - 1) continue;
            const double zinv = 1.0 * dt;
            double a = 0.0, b, cc = 0.0;
            if constexpr (LO) {
                double v_adv = zinv * ar[s] / av[s];
                if (k == nzmin) {
                    b = hn[s] + wi[s] * v_adv;
                } else {
                    a = dmn(0.0, wi[s]) * v_adv;
                    b = hn[s] + dmx(0.0, wi[s]) * v_adv;
                }
                if (k <= nzmax - 2) {
                    v_adv = zinv * ard[s] / av[s];
                    b = b - dmn(0.0, wid[s]) * v_adv;
                    cc = -dmx(0.0, wid[s]) * v_adv;
                }
            } else {
                if (k > nzmin) {
                    const double zinv1 = 1.0 / (zu[s] - zk[s]);
                    a = -(redi ? kv[s] + k33u[s] : kv[s]) * zinv1 * zinv * (ar[s] / av[s]);
                }
                if (k <= nzmax - 2) {
                    const double zinv2 = 1.0 / (zk[s] - zd[s]);
                    cc = -(redi ? kvd[s] + k33[s] : kvd[s]) * zinv2 * zinv * ard[s] / av[s];
                }
                if (k == nzmin) b = -cc + hn[s];
                else if (k <= nzmax - 2) b = -a - cc + hn[s];
                else b = -a + hn[s];
            }
            if constexpr (WS) {   // oce_ale_tracer.F90:1118-1129, 1158-1172, 1194-1202
                double v_adv = zinv * (ar[s] / av[s]), a2 = a, b2 = b, c2 = cc;
                if (k == nzmin) {
                    b2 = b2 + wi[s] * v_adv;
                } else {
                    a2 = a2 + dmn(0.0, wi[s]) * v_adv;
                    b2 = b2 + dmx(0.0, wi[s]) * v_adv;
                }
                if (k <= nzmax - 2) {
                    v_adv = zinv * ard[s] / av[s];
                    b2 = b2 - dmn(0.0, wid[s]) * v_adv;
                    c2 = c2 - dmx(0.0, wid[s]) * v_adv;
                }
                sa[set + c * RS + k - 1] = a2;
                sb[set + c * RS + k - 1] = b2;
                sc[set + c * RS + k - 1] = c2;
                wa[s] = a2;
                wb[s] = b2 - hn[s];
                wc[s] = c2;
            }
            sa[c * RS + k - 1] = a;
            sb[c * RS + k - 1] = b;
            sc[c * RS + k - 1] = cc;
            a_[s] = a;
            c_[s] = cc;
            bd_[s] = b - hn[s];
        }
        // right-hand sides (oce_ale_tracer.F90:1206-1229, 1377-1383)
        for (int j0 = 0; j0 < ntb; j0 += KV_TP) {
            if (j0 > 0 && layer) {
#pragma unroll
                for (int j = 0; j < KV_TP; ++j)
                    if (j0 + j < ntb) row_load<NV>(F + t.sN * (trb + j0 + j) + nL, off, ts[j]);
            }
#pragma unroll
            for (int j = 0; j < KV_TP; ++j) {
                if (j0 + j >= ntb) break;
                const int id = ldc(t.id + trb + j0 + j);
                if (!solved(trb + j0 + j)) continue;
                const bool w2 = second(trb + j0 + j);
                double tu[NV], td[NV];
                col_up<NV>(ts[j], tu);
                col_down<NV>(ts[j], td);
#pragma unroll
                for (int s = 0; s < NV; ++s) {
                    const int k = kb + s;
                    if (k < nzmin || k > nzmax - 1) continue;
                    const double ra = WS && w2 ? wa[WS ? s : 0] : a_[s], rb = WS && w2 ? wb[WS ? s : 0] : bd_[s],
                                 rc = WS && w2 ? wc[WS ? s : 0] : c_[s];
                    double r;
                    if (k == nzmin) r = -rb * ts[j][s] - rc * td[s];
                    else if (k <= nzmax - 2) r = -ra * tu[s] - rb * ts[j][s] - rc * td[s];
                    else r = -ra * tu[s] - rb * ts[j][s];
                    if (LO) {
                    } else if (bc_every_layer(id, d)) r = r + bc_surface_dev(id, dt, d, m.N2, L, n, k, ts[j][s]);
                    else if (k == nzmin) r = r + bc_surface_dev(id, dt, d, m.N2, L, n, nzmin, ts[j][s]);
                    sr[(c * TB + j0 + j) * RS + k - 1] = r;
                }
            }
        }
    }
    __syncthreads();
    // Thomas sweeps (oce_ale_tracer.F90:1406-1430), one lane per row; the lanes
    // of a column all compute its pivots. c' replaces c.
    if (w == 0 && lane < ncol * ntb) {
        const int c = lane / ntb, j = lane % ntb;
        const int z0 = __shfl(z0l, c), z1 = __shfl(z1l, c);
        const size_t o = WS && t.lim[trb + j] != LIM_FCT ? set : 0;
        const double *pa = sa + o + c * RS - 1, *pb = sb + o + c * RS - 1;
        double *pc = sc + o + c * RS - 1, *pr = sr + (c * TB + j) * RS - 1;
        double cp = pc[z0] / pb[z0], tp = pr[z0] / pb[z0];
        pc[z0] = cp;
        pr[z0] = tp;
        double an = pa[z0 + 1], bn = pb[z0 + 1], cn = pc[z0 + 1], rn = pr[z0 + 1];
        for (int nz = z0 + 1; nz <= z1 - 1; ++nz) {
            const int nx = min(nz + 1, z1 - 1);   // the next level's rows, loaded ahead
            const double a1 = pa[nx], b1 = pb[nx], c1 = pc[nx], r1 = pr[nx];
            const double mm = bn - cp * an;
            cp = cn / mm;
            tp = (rn - tp * an) / mm;
            pc[nz] = cp;
            pr[nz] = tp;
            an = a1; bn = b1; cn = c1; rn = r1;
        }
        double x = tp;
        double r0 = pr[max(z1 - 2, z0)], c0 = pc[max(z1 - 2, z0)];
        for (int nz = z1 - 2; nz >= z0; --nz) {
            const int nx = max(nz - 1, z0);
            const double r1 = pr[nx], c1 = pc[nx];
            x = r0 - c0 * x;
            pr[nz] = x;
            r0 = r1; c0 = c1;
        }
    }
    __syncthreads();
    for (int c0 = SH ? w << (6 - lsh) : w; c0 < ncol; c0 += step) {
        const int c = c0 + part;
        int n, nzmin, nzmax;
        column(c, n, nzmin, nzmax);
        const size_t nL = (size_t)n * L;
        bool on[NV], any = false;
#pragma unroll
        for (int s = 0; s < NV; ++s) {
            on[s] = kb + s >= nzmin && kb + s <= nzmax - 1;
            any = any || on[s];
        }
        for (int j0 = 0; j0 < ntb; j0 += 2 * KV_TP) {
            double v[2 * KV_TP][NV];
#pragma unroll
            for (int j = 0; j < 2 * KV_TP; ++j)
                if (j0 + j < ntb && any) row_load<NV>(F + t.sN * (trb + j0 + j) + nL, off, v[j]);
#pragma unroll
            for (int j = 0; j < 2 * KV_TP; ++j) {
                if (j0 + j >= ntb) break;
                const int tr = trb + j0 + j;
                const bool add = solved(tr);
                if (LO && !add) continue;
#pragma unroll
                for (int s = 0; s < NV; ++s) {
                    if (on[s] && add) v[j][s] = v[j][s] + sr[(c * TB + j0 + j) * RS + kb + s - 1];
                    if (!LO && tr == clamp_tracer) {
                        if (v[j][s] > 45.0) v[j][s] = 45.0;
                        if (v[j][s] < 3.0) v[j][s] = 3.0;
                    }
                }
                row_store<NV>(F + t.sN * tr + nL, off, v[j], on);
            }
        }
    }
}

// Z levels of diff_ver_part_impl_ale rebuilt bottom-up from hnode_new and
// zbar_n_bot (oce_ale_tracer.F90:1088-1096), one thread per column
__global__ void k_zn_vdiff(DevMesh m, double *zn, double *zbn)
{
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= m.N2) return;
    const int L = m.L, nzmin = m.ulevn[n], nzmax = m.nlevn[n];
    const double *hn = m.hnode_new + (size_t)n * L;
    double *z = zn + (size_t)n * L, *zi = zbn + (size_t)n * m.NL;
    double zb = m.zbar_n_bot[n];
    zi[nzmax - 1] = zb;
    z[nzmax - 2] = zb + hn[nzmax - 2] / 2.0;
    for (int nz = nzmax - 1; nz >= nzmin + 1; --nz) {
        zb = zb + hn[nz - 1];
        zi[nz - 1] = zb;
        z[nz - 2] = zb + hn[nz - 2] / 2.0;
    }
}

// ==============================================================================
// host side
// ==============================================================================
int fgpu_compute_zn(fgpu_context *c)
{
    struct A { const double **p; size_t n; } arrs[] = {
        {&c->m.zn_vd, (size_t)c->N2 * (c->nl - 1)}, {&c->m.zbn_vd, (size_t)c->N2 * c->nl}};
    for (auto &a : arrs) {
        if (*a.p) continue;
        double *q = nullptr;
        int rc = fgpu_alloc(c, (void **)&q, sizeof(double) * a.n);
        if (rc) return rc;
        if ((rc = fgpu_zero(c, q, sizeof(double) * a.n))) return rc;
        *a.p = q;
    }
    hipLaunchKernelGGL(k_zn_vdiff, dim3((c->N2 + 255) / 256), dim3(256), 0, c->stream, c->m, (double *)c->m.zn_vd,
                       (double *)c->m.zbn_vd);
    FGPU_HIP(hipGetLastError());
    FGPU_HIP(hipStreamSynchronize(c->stream));
    return FGPU_OK;
}
// Extra terms compiled into K_L and K_V: bit 0 the W split (w_i rows of the
// implicit diffusion for non-FCT tracers), bit 1 explicit diffusion increments
// (Ki, Redi, i_vert_diff off) and the Redi K33 rows.
int fgpu_kd_extras(const fgpu_context *c)
{
    bool dx = c->d.hdiff || c->d.redi;
    for (int v : c->h_ivd) dx = dx || !v;
    return (c->d.wsplit ? 1 : 0) | (dx ? 2 : 0);
}

// The Thomas chunk and columns per block that fgpu_step_shape reports for the
// requested ones. They told forms of the former last kernel apart; K_L and K_V
// take their own from the column depth and the tracer count.
void fgpu_kd_shape(const fgpu_context *c, int *tch_out, int *cpb_out)
{
    int tch = (c->step_tch == 4 || c->step_tch == 5 || c->step_tch == 8) ? c->step_tch : 2;
    int cpb = c->step_cpb;
    if (fgpu_kd_extras(c)) {   // the W split or explicit diffusion terms: one lock-step shape
        tch = 2;
        cpb = 1;
    } else if (c->m.NL <= 64) {
        if (cpb == 8) tch = 2;
        else if (cpb == 4) tch = tch == 4 ? 4 : 2;
        else cpb = 1;
    } else if (c->step_kdp && cpb >= 3 && c->m.NL <= KDP_SHORT_NL) {
        cpb = cpb >= 4 ? 4 : 3;
        tch = 2;
    } else if (c->step_kdp && cpb >= 2) {
        cpb = 2;
        tch = tch == 4 ? 4 : 2;
    } else {
        cpb = 1;
    }
    *tch_out = tch;
    *cpb_out = cpb;
}

// The lanes of the column waves: NV levels per lane and GT tracers per wave, so
// that a lane group holds every interface of a column (NV x 64 / GT >= NL). Two
// tracers share a wave where they share its scheme branches and both rows lie
// within a 32-bit offset of the wave's base; from 65 to 96 interfaces on also
// beyond, with 64-bit offsets: at 1.3 million nodes, 70 layers, 10 tracers K_B
// takes 16.4 ms by <3,2> and 22.6 by <2,1> with 32-bit ones, K_L 21.9 and 22.1.
// The lines between the mappings were measured per kernel, in us, at 47 layers with 2 tracers (126,858 nodes) and 32
// tracers (12 thousand), and at 70 layers with 10 tracers (40 thousand):
//   K_A  <1,1> 507, 576; <2,2> 506, 440 | <2,1> 730, <3,2> 740
//   K_B  <1,1> 298, 271; <2,2> 469, 366 | <2,1> 710, <3,2> 518
//   K_C  <1,1> 315, 462; <2,2> 329, 396 | <2,1> 648, <3,2> 637
//   K_L  <1,1> 363, 491; <2,2> 351, 441 | <2,1> 700, <3,2> 687
// Two levels per lane halve a row's vector memory instructions, two tracers per
// wave form the offsets once for both; against that stand the registers (fewer
// waves per SIMD) and what a second tracer's lanes repeat of the first one's
// tracer-independent work. Rows of up to 32 interfaces leave half a wave free,
// which a second tracer takes at no cost.
struct ColLanes {
    bool pair;   // tracers two to a wave
    bool wide;   // row offsets need 64 bits
    bool far;    // those of a pair do
};
static ColLanes col_lanes(const fgpu_context *c, int tpb)
{
    const DevTracers &t = c->t;
    const size_t field = 8 * std::max(std::max(t.sE, t.sNI), std::max(t.sOld, t.sG)) + 4096, reach = 0xffffffffu;
    bool same = true;
    for (int i = 1; i < t.ntr; ++i)
        same = same && c->h_lim[i] == c->h_lim[0] && c->h_abo[i] == c->h_abo[0] && c->h_hor[i] == c->h_hor[0] &&
               c->h_ver[i] == c->h_ver[0] && c->h_ph[i] == c->h_ph[0] && c->h_pv[i] == c->h_pv[0];
    const bool wide = c->step_wide || field >= reach, far = wide || 2 * field >= reach;
    const bool deep = c->m.NL > 64 && c->m.NL <= 96;
    return {same && std::min(tpb, t.ntr) >= 2 && (!far || deep), wide, far};
}

#define COL_LAUNCH(kern, NV, GT, X, grid, ...)                                                                       \
    do {                                                                                                             \
        if (GT > 1 ? cl.far : cl.wide) hipLaunchKernelGGL((kern<size_t, NV, GT, X>), grid, dim3(64), 0, c->stream, __VA_ARGS__);            \
        else hipLaunchKernelGGL((kern<unsigned, NV, GT, X>), grid, dim3(64), 0, c->stream, __VA_ARGS__);             \
    } while (0)
// pairs of up to 64 interfaces, within 32-bit offsets
#define COL_NEAR(kern, NV, X, grid, ...)                                                                             \
    hipLaunchKernelGGL((kern<unsigned, NV, 2, X>), grid, dim3(64), 0, c->stream, __VA_ARGS__)

template <int XF>
static void launch_kv(fgpu_context *c, int tr0, int nt, double dt, int all, int clamp)
{
    const DevMesh &m = c->m;
    const int row = 8 * (m.L | 1), coef = XF & KV_WS ? 6 : 3;
    // tracers in equal groups of at most ten: a column's pivots are formed once
    // per group (70 layers, 10 tracers: 328 us in one group, 682 us by fours)
    const int groups = (nt + 9) / 10, TB = (nt + groups - 1) / groups;
    // columns: at most 64 sweep lanes, 40,000 bytes of LDS (four blocks per CU;
    // 47 layers, 2 tracers, 126,858 nodes: 159 us, 214 us at 65,536 bytes, 191
    // us at 26,000), and 1,024 blocks on a small mesh, where the blocks' serial
    // sweeps have to run side by side
    int NC = std::min(64 / TB, 40000 / (row * (coef + TB)));
    NC = std::max(1, std::min(NC, (int)((size_t)m.N2 * groups / 1024)));
    // up to 32 layers leave half a wave free, which further columns take: with one
    // column to a wave 120 thousand nodes, 4 layers, 1 tracer took 67 us (13), 60
    // thousand nodes, 16 layers 48 us (24)
    int lsh = 6;
    while (lsh > 1 && (1 << (lsh - 1)) >= m.L) --lsh;
    // no waves without a column: they held the slots of further blocks (3,000
    // nodes, 24 layers, 1 tracer: 22 us with eight waves, 15 with one)
    const int waves = std::min(KV_NW, (NC + (64 >> lsh) - 1) >> (6 - lsh));
    const size_t lds = (size_t)row * (coef + TB) * NC;
    const dim3 g(xcd_grid((m.N2 + NC - 1) / NC), (unsigned)groups), b(64 * waves);
    if (lsh < 6) hipLaunchKernelGGL((kV_cols<1, XF, true>), g, b, lds, c->stream, m, c->d, c->t, tr0, nt, dt, all, clamp, NC, TB, lsh);
    else if (m.NL <= 64) hipLaunchKernelGGL((kV_cols<1, XF, false>), g, b, lds, c->stream, m, c->d, c->t, tr0, nt, dt, all, clamp, NC, TB, lsh);
    else hipLaunchKernelGGL((kV_cols<2, XF, false>), g, b, lds, c->stream, m, c->d, c->t, tr0, nt, dt, all, clamp, NC, TB, lsh);
}

// K_V of tracers tr0..tr0+ntr-1; all: also of those with i_vert_diff off
void fgpu_launch_kv(fgpu_context *c, int tr0, int ntr, double dt, int all, int clamp)
{
    bool dx = c->d.redi != 0;
    for (int i = tr0; i < tr0 + ntr; ++i) dx = dx || (!all && !c->h_ivd[i]);
    if (c->d.wsplit && dx) launch_kv<KV_WS | KV_DX>(c, tr0, ntr, dt, all, clamp);
    else if (c->d.wsplit) launch_kv<KV_WS>(c, tr0, ntr, dt, all, clamp);
    else if (dx) launch_kv<KV_DX>(c, tr0, ntr, dt, all, clamp);
    else launch_kv<0>(c, tr0, ntr, dt, all, clamp);
}
void fgpu_launch_kv_lo(fgpu_context *c, int tr0, int ntr, double dt) { launch_kv<KV_LO>(c, tr0, ntr, dt, 0, -1); }

int fgpu_enqueue_fused_step(fgpu_context *c, double dt)
{
    const DevMesh &m = c->m;
    const int nt = c->t.ntr;
    const int clamp = nt >= 2 ? 1 : -1;
    if (m.NL > 128) return fgpu_fail(FGPU_ERR_ARG, "more than 127 layers");
    // tracers per block: 1 runs every tracer's chain in its own waves
    const int tpb = std::max(1, std::min(c->step_tpb, nt));
    const unsigned ny = (unsigned)((nt + tpb - 1) / tpb);
    bool xv = false;   // a CDIFF or PPM tracer
    for (int v : c->h_ver) xv = xv || v == VER_CDIFF || v == VER_PPM;
    const int xf = fgpu_kd_extras(c);
    {   // explicit diffusion terms from T^n (no-op without Ki, Redi or explicit vertical diffusion)
        int rc = fgpu_launch_diff(c, 0, nt, dt);
        if (rc) return rc;
    }
    const bool narrow = m.NL <= 64, slim = m.NL <= 32;
    const dim3 nodes(xcd_grid(m.N2), ny), edges(xcd_grid(m.E2), ny);
    const ColLanes cl = col_lanes(c, tpb);
    const bool pair = cl.pair, many = pair && std::min(tpb, nt) >= 4;
    {
        ProfScope ps(c, "kG_node");
        hipLaunchKernelGGL(kG_node, nodes, dim3(64), 0, c->stream, m, c->t, c->d_kneed, tpb);
    }
    {
        ProfScope ps(c, "kA_edge");
        if (c->edge_gap && narrow) COL_LAUNCH(kA_edge, 1, 1, true, edges, m, c->d, c->t, tpb);
        else if (c->edge_gap) COL_LAUNCH(kA_edge, 2, 1, true, edges, m, c->d, c->t, tpb);
        else if (!narrow) COL_LAUNCH(kA_edge, 2, 1, false, edges, m, c->d, c->t, tpb);
        else if (slim && pair) COL_NEAR(kA_edge, 1, false, edges, m, c->d, c->t, tpb);
        else if (many) COL_NEAR(kA_edge, 2, false, edges, m, c->d, c->t, tpb);
        else COL_LAUNCH(kA_edge, 1, 1, false, edges, m, c->d, c->t, tpb);
    }
    {
        ProfScope ps(c, "kB_node");
        const bool ws = c->d.wsplit != 0;
        if (c->edge_gap && narrow) COL_LAUNCH(kB_cols, 1, 1, KB_XV | KB_WS | KB_GAP, nodes, m, c->d, c->t, dt, tpb);
        else if (c->edge_gap) COL_LAUNCH(kB_cols, 2, 1, KB_XV | KB_WS | KB_GAP, nodes, m, c->d, c->t, dt, tpb);
        else if (xv && ws && narrow) COL_LAUNCH(kB_cols, 1, 1, KB_XV | KB_WS, nodes, m, c->d, c->t, dt, tpb);
        else if (xv && ws) COL_LAUNCH(kB_cols, 2, 1, KB_XV | KB_WS, nodes, m, c->d, c->t, dt, tpb);
        else if (xv && narrow) COL_LAUNCH(kB_cols, 1, 1, KB_XV, nodes, m, c->d, c->t, dt, tpb);
        else if (xv) COL_LAUNCH(kB_cols, 2, 1, KB_XV, nodes, m, c->d, c->t, dt, tpb);
        else if (ws && narrow) COL_LAUNCH(kB_cols, 1, 1, KB_WS, nodes, m, c->d, c->t, dt, tpb);
        else if (ws) COL_LAUNCH(kB_cols, 2, 1, KB_WS, nodes, m, c->d, c->t, dt, tpb);
        else if (pair && m.NL > 64 && m.NL <= 96) COL_LAUNCH(kB_cols, 3, 2, 0, nodes, m, c->d, c->t, dt, tpb);
        else if (!narrow) COL_LAUNCH(kB_cols, 2, 1, 0, nodes, m, c->d, c->t, dt, tpb);
        else if (slim && pair) COL_NEAR(kB_cols, 1, 0, nodes, m, c->d, c->t, dt, tpb);
        else COL_LAUNCH(kB_cols, 1, 1, 0, nodes, m, c->d, c->t, dt, tpb);
    }
    if (c->d.wsplit) {
        ProfScope ps(c, "kV_lo");
        fgpu_launch_kv_lo(c, 0, nt, dt);
    }
    {
        ProfScope ps(c, "kC_node");
        if (c->edge_gap && narrow) COL_LAUNCH(kC_cols, 1, 1, true, nodes, m, c->t, dt, tpb);
        else if (c->edge_gap) COL_LAUNCH(kC_cols, 2, 1, true, nodes, m, c->t, dt, tpb);
        else if (!narrow) COL_LAUNCH(kC_cols, 2, 1, false, nodes, m, c->t, dt, tpb);
        else if (slim && pair) COL_NEAR(kC_cols, 1, false, nodes, m, c->t, dt, tpb);
        else if (many) COL_NEAR(kC_cols, 2, false, nodes, m, c->t, dt, tpb);
        else COL_LAUNCH(kC_cols, 1, 1, false, nodes, m, c->t, dt, tpb);
    }
    {
        ProfScope ps(c, "kL_node");
        const bool dx = (xf & 2) != 0;
        auto launch = [&](auto DX) {
            constexpr bool X = decltype(DX)::value;
            if (pair && m.NL > 64 && m.NL <= 96) COL_LAUNCH(kL_node, 3, 2, X, nodes, m, c->d, c->t, dt, tpb);
            else if (!narrow) COL_LAUNCH(kL_node, 2, 1, X, nodes, m, c->d, c->t, dt, tpb);
            else if (slim && pair) COL_NEAR(kL_node, 1, X, nodes, m, c->d, c->t, dt, tpb);
            else if (pair) COL_NEAR(kL_node, 2, X, nodes, m, c->d, c->t, dt, tpb);
            else COL_LAUNCH(kL_node, 1, 1, X, nodes, m, c->d, c->t, dt, tpb);
        };
        if (dx) launch(std::true_type{});
        else launch(std::false_type{});
    }
    {
        ProfScope ps(c, "kV_cols");
        fgpu_launch_kv(c, 0, nt, dt, 0, clamp);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fgpu_fail(FGPU_ERR_HIP, std::string("fused step launch: ") + hipGetErrorString(e));
    return FGPU_OK;
}
