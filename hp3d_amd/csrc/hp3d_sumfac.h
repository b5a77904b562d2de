// hp3d_sumfac.h -- element matrices by sum factorisation (device code of
// libhp3d_gpu, included by hp3d_gpu.hip).
//
// Every hexahedral dof is +- a product of 1D functions chi_i or their
// derivatives (dof_row in hp3d_tables.h), so an element matrix is a sum of
// terms
//   sum_q  F_i0 F_j0 (q0)  F_i1 F_j1 (q1)  F_i2 F_j2 (q2)  g(q0, q1, q2),
// F = chi or chi', with g one of the point's symmetric metric fields: the
// nine (s, t) terms d_s u d_t v of the H1 form, and in H(curl), where a dof of
// component a is d_a of a product, the mass term (a, b) and the four curl
// terms (curl rows r != a, r' != b, derivatives in every direction but r).
// The sums run one direction after the other, A = y, then B = x, then C = z:
//   T(iA, jA; qB, qC) = sum_qA F F g     (LDS, for a chunk of columns jA)
//   S(I, J; qC) = sum_qB F F T           (registers, pencils I = (iA, iB), J)
//   K(I iC, J jC) = sum_qC F F S         (registers, all iC and jC at once)
// which is O(m^7) work for O(m^6) entries where the A A^T product is O(m^9).
// One thread owns one pencil pair: its M x M block of K is computed from four
// S vectors against compile-time 1D tables in scalar registers.  The element's
// other arithmetic is small beside writing K.
//
// Replaces the A_TEST fill and DSYRK of POISSON/GALERKIN/elem_opt.F90:88-137
// and the real form of MAXWELL/GALERKIN/elem_opt.F90:88-149.
#pragma once

__constant__ SfTables c_sf = make_sf_tables();

__host__ __device__ constexpr int sf_sym(int r, int s) { return r <= s ? r * (5 - r) / 2 + s : s * (5 - s) / 2 + r; }

// One element.  m[] and everything indexed like it goes by role: 0 = B, 1 = A,
// 2 = C, with dir[role] the element direction of the role and rol[] its
// inverse; components of H(curl) dofs are counted by role too (a cyclic
// relabelling of the directions leaves the curl terms alone, an odd one turns
// the sign of both curls).
struct SfElem {
    ElemOrders o;
    DofBases bs, bh; // of the space, and of H1 (geometry nodes)
    int n, nb, nh, m[3], dir[3], rol[3], nint, ok, negjac, np, mode;
};

// roles of the directions and the mode of one element (orders md[], n dofs)
template <int SPACE>
__device__ __forceinline__ void sf_choose(SfElem &es, const int (&md)[3], int n, SfFused fu)
{
    const SfRoles ro = sf_roles<SPACE>(md, n, es.nb, fu);
    es.mode = ro.mode;
    es.dir[0] = ro.b;
    es.dir[1] = ro.a;
    es.dir[2] = ro.c;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int r = d == ro.b ? 0 : d == ro.a ? 1 : 2;
        es.rol[d] = r;
        es.m[r] = md[d];
    }
}

// inclusive scan over lanes 0..31 by DPP moves (shifts within the rows of 16,
// then the first row's total to the second)
template <typename F>
__device__ __forceinline__ int sf_scan(int x, F f)
{
    x = f(x, __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false));
    x = f(x, __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false));
    x = f(x, __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false));
    x = f(x, __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false));
    return f(x, __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false));
}

// Orders, counts and dof bases of one element, decoded by the lanes of wave 0
// (lane l: header integer l; counts by a lane scan, quadrature sizes by an
// or-reduction of order bits), ending in an LDS barrier.  Returns false
// (uniformly) for an invalid element.
// The geometry nodes of maps with up to XS_MAX nodes and the coefficient are
// loaded beside the header, so that their latency is paid once.
template <int SPACE, int WGS>
__device__ __forceinline__ bool sf_setup(const ElemArgs &a, int e, SfElem &es, double *xg, int tid, SfFused fu = {0, 0, 0, 0, 0, 0})
{
    const int nx = a.ngeo <= XS_MAX ? 3 * a.ngeo : 0;
    constexpr int NX = WGS > 3 * XS_MAX ? 1 : 2;
    static_assert(NX * WGS > 3 * XS_MAX, "staged values");
    double xv[NX];
#pragma unroll
    for (int i = 0; i < NX; ++i) {
        const int k = tid + i * WGS;
        xv[i] = 0.0;
        if (k < nx) xv[i] = a.xnod[(size_t)3 * a.ngeo * e + k];
        else if (k == 3 * XS_MAX) xv[i] = a.coef ? a.coef[e] : 1.0;
    }
    if (tid < 64) {
        int v = 0;
        if (tid < 19) v = a.norder[19 * (size_t)e + tid];
        else if (tid < 31) v = a.nori_e[12 * (size_t)e + tid - 19];
        else if (tid < 37) v = a.nori_f[6 * (size_t)e + tid - 31];
        const int vf = __shfl(v, tid + 19); // lanes 12..17: their face's orientation code
        bool ok = true;
        int cnt = 0, cnt_h = 0, inner = 0;
        unsigned bits = 0;
        auto order_bit = [](int p, int d) { return (1u << (p & 7)) << (8 * d); };
        if (tid < 12) {
            ok = v >= 1 && v <= MAXP;
            es.o.pe[tid] = v;
            cnt_h = v - 1;
            cnt = SPACE == 0 ? v - 1 : v;
            bits = order_bit(v, tid >= 8 ? 2 : tid & 1);
        } else if (tid < 18) {
            const int f = tid - 12, h = v / MODORDER, w = v % MODORDER;
            ok = h >= 1 && h <= MAXP && w >= 1 && w <= MAXP;
            es.o.fh[f] = h;
            es.o.fv[f] = w;
            cnt_h = (h - 1) * (w - 1);
            cnt = SPACE == 0 ? cnt_h : h * (w - 1) + (h - 1) * w;
            const int ax0 = f == 3 || f == 5 ? 1 : 0, ax1 = f < 2 ? 1 : 2;
            const bool sw = face_swapped(vf) != 0;
            bits = order_bit(sw ? w : h, ax0) | order_bit(sw ? h : w, ax1);
        } else if (tid == 18) {
            const int b0 = v / 100, b1 = (v / 10) % 10, b2 = v % 10;
            ok = b0 >= 1 && b0 <= MAXP && b1 >= 1 && b1 <= MAXP && b2 >= 1 && b2 <= MAXP;
            es.o.b[0] = b0;
            es.o.b[1] = b1;
            es.o.b[2] = b2;
            cnt_h = (b0 - 1) * (b1 - 1) * (b2 - 1);
            inner = cnt = SPACE == 0 ? cnt_h : b0 * (b1 - 1) * (b2 - 1) + (b0 - 1) * b1 * (b2 - 1) + (b0 - 1) * (b1 - 1) * b2;
            bits = order_bit(b0, 0) | order_bit(b1, 1) | order_bit(b2, 2);
        } else if (tid < 31) {
            ok = v == 0 || v == 1;
            es.o.oe[tid - 19] = v;
        } else if (tid < 37) {
            ok = v >= 0 && v <= 7;
            es.o.of[tid - 31] = v;
        }
        const bool all_ok = __all(ok);
        // inclusive scans over lanes 0..18 (lane 18 ends with the totals):
        // both entity counts at once, and the order bits
        const int sc = sf_scan(cnt + (cnt_h << 16), [](int x, int y) { return x + y; });
        bits = sf_scan((int)bits, [](int x, int y) { return x | y; });
        const int base = (sc & 0xffff) - cnt + (SPACE == 0 ? 8 : 0);
        const int base_h = (sc >> 16) - cnt_h + 8;
        if (tid < 12) {
            es.bs.edge[tid] = (short)base;
            es.bh.edge[tid] = (short)base_h;
        } else if (tid < 18) {
            es.bs.face[tid - 12] = (short)base;
            es.bh.face[tid - 12] = (short)base_h;
        } else if (tid == 18) {
            es.bs.interior = (short)base;
            es.bh.interior = (short)base_h;
            es.n = base + cnt;
            es.nb = inner;
            es.nh = (sc >> 16) + 8;
            int md[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) md[d] = 32 - __clz((int)((bits >> (8 * d)) & 0x7eu));
            es.nint = md[0] * md[1] * md[2];
            es.negjac = 0;
            es.ok = all_ok && a.ngeo <= es.nh ? 1 : 0;
            sf_choose<SPACE>(es, md, base + cnt, fu);
        }
    }
#pragma unroll
    for (int i = 0; i < NX; ++i)
        if (tid + i * WGS < nx || tid + i * WGS == 3 * XS_MAX) xg[tid + i * WGS] = xv[i];
    lds_barrier();
    return es.ok != 0;
}

// the value of a role
__device__ __forceinline__ int sf_pick(int role, int b, int a, int c) { return role == 0 ? b : role == 1 ? a : c; }

// 1D tables of the three directions in LDS
struct SfTab {
    double f[3][2][SF_I * 8];
    double w[3][8];
};
template <int WGS>
__device__ __forceinline__ void sf_fill_tab(const int (&m)[3], SfTab &t, int tid)
{
    constexpr int LEN = 2 * SF_I * 8, NL = (3 * LEN + WGS - 1) / WGS;
    double v[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        const int k = min(tid + i * WGS, 3 * LEN - 1), d = k / LEN;
        v[i] = (&c_sf.f[sf_pick(d, m[0], m[1], m[2])][0][0][0])[k - d * LEN];
    }
    const int dw = min(tid >> 3, 2);
    const double w = c_sf.w[sf_pick(dw, m[0], m[1], m[2])][tid & 7];
#pragma unroll
    for (int i = 0; i < NL; ++i)
        if (tid + i * WGS < 3 * LEN) (&t.f[0][0][0])[tid + i * WGS] = v[i];
    if (tid < 24) t.w[dw][tid & 7] = w;
}

// dof rows by 1D indexes: row[((comp * 7 + iA) * 7 + iB) * 8 + iC], iA < m[1],
// iB < m[0]
template <int SPACE>
__device__ __forceinline__ void sf_fill_rows(const SfElem &es, short *row, int tid, int wgs)
{
    const int mA = es.m[1], mB = es.m[0], mC = es.m[2];
    for (int k = tid; k < sf_comps(SPACE) * mA * mB * 8; k += wgs) {
        const int iC = k & 7, k1 = k >> 3, k2 = div_small(k1, mB), iB = k1 - k2 * mB;
        const int c = SPACE == 0 ? 0 : (k2 >= mA) + (k2 >= 2 * mA), iA = k2 - c * mA;
        int r = -1;
        if (iC < mC)
            r = dof_row(SPACE, SPACE == 0 ? 0 : es.dir[c], sf_pick(es.rol[0], iB, iA, iC), sf_pick(es.rol[1], iB, iA, iC),
                        sf_pick(es.rol[2], iB, iA, iC), es.o, es.bs);
        row[((c * SF_I + iA) * SF_I + iB) * 8 + iC] = (short)r;
    }
}

// geometry node -> H1 1D indexes and sign, for maps beyond the trilinear one
__device__ __forceinline__ void sf_fill_gmap(const SfElem &es, int ngeo, unsigned short *gmap, int tid, int wgs)
{
    for (int k = tid; k < SF_I * SF_I * SF_I; k += wgs) {
        const int i0 = k % SF_I, i1 = (k / SF_I) % SF_I, i2 = k / (SF_I * SF_I);
        if (i0 >= es.m[es.rol[0]] || i1 >= es.m[es.rol[1]] || i2 >= es.m[es.rol[2]]) continue;
        const int r = dof_row(0, 0, i0, i1, i2, es.o, es.bh);
        if (r >= 0 && (r & ~ROW_NEG) < ngeo)
            gmap[r & ~ROW_NEG] = (unsigned short)(i0 | (i1 << 3) | (i2 << 6) | (r & ROW_NEG ? 512 : 0));
    }
}

// The map at the point with 1D indexes (q0, q1, q2) in x, y and z
// (geom3D.F90:77-91, geom.F90:57-113): x, J (jm[c][i] = d x_c / d xi_i), its
// inverse [reference, physical] and det J.
template <bool STAGED>
__device__ __forceinline__ double sf_map(const SfElem &es, const SfTab &tb, const unsigned short *gmap,
                                         const double *xn, int ngeo, int q0, int q1, int q2, double (&x)[3],
                                         double (&jm)[3][3], double (&inv)[3][3])
{
    const int r0 = es.rol[0], r1 = es.rol[1], r2 = es.rol[2]; // roles of x, y, z
#pragma unroll
    for (int c = 0; c < 3; ++c) x[c] = jm[c][0] = jm[c][1] = jm[c][2] = 0.0;
    auto node = [&](const double *xk, double v0, double v1, double v2, double g0, double g1, double g2) {
        const double ph = v0 * v1 * v2, h0 = g0 * v1 * v2, h1 = v0 * g1 * v2, h2 = v0 * v1 * g2;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const double xc = xk[c];
            x[c] += xc * ph;
            jm[c][0] += xc * h0;
            jm[c][1] += xc * h1;
            jm[c][2] += xc * h2;
        }
    };
    if (STAGED && ngeo == 8) {
        double v[3][2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            v[0][i] = tb.f[r0][0][8 * i + q0];
            v[1][i] = tb.f[r1][0][8 * i + q1];
            v[2][i] = tb.f[r2][0][8 * i + q2];
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int i0 = vtx_mu(k, 0), i1 = vtx_mu(k, 1), i2 = vtx_mu(k, 2);
            node(xn + 3 * k, v[0][i0], v[1][i1], v[2][i2], i0 ? 1.0 : -1.0, i1 ? 1.0 : -1.0, i2 ? 1.0 : -1.0);
        }
    } else {
        for (int k = 0; k < ngeo; ++k) {
            const int g = gmap[k], i0 = 8 * (g & 7) + q0, i1 = 8 * ((g >> 3) & 7) + q1, i2 = 8 * ((g >> 6) & 7) + q2;
            const double sg = g & 512 ? -1.0 : 1.0;
            node(xn + 3 * k, sg * tb.f[r0][0][i0], tb.f[r1][0][i1], tb.f[r2][0][i2], sg * tb.f[r0][1][i0],
                 tb.f[r1][1][i1], tb.f[r2][1][i2]);
        }
    }
    const double c00 = jm[1][1] * jm[2][2] - jm[2][1] * jm[1][2], c01 = jm[2][1] * jm[0][2] - jm[0][1] * jm[2][2],
                 c02 = jm[0][1] * jm[1][2] - jm[1][1] * jm[0][2];
    const double det = jm[0][0] * c00 + jm[1][0] * c01 + jm[2][0] * c02;
    const double rdet = 1.0 / det;
    inv[0][0] = c00 * rdet;
    inv[0][1] = c01 * rdet;
    inv[0][2] = c02 * rdet;
    inv[1][0] = (jm[2][0] * jm[1][2] - jm[1][0] * jm[2][2]) * rdet;
    inv[1][1] = (jm[0][0] * jm[2][2] - jm[2][0] * jm[0][2]) * rdet;
    inv[1][2] = (jm[1][0] * jm[0][2] - jm[0][0] * jm[1][2]) * rdet;
    inv[2][0] = (jm[1][0] * jm[2][1] - jm[2][0] * jm[1][1]) * rdet;
    inv[2][1] = (jm[2][0] * jm[0][1] - jm[0][0] * jm[2][1]) * rdet;
    inv[2][2] = (jm[0][0] * jm[1][1] - jm[1][0] * jm[0][1]) * rdet;
    return det;
}

// Metric fields and load of every quadrature point, q = (qA mB + qB) mC + qC,
// field f at d[f * nint + q], the weights folded in (elem_opt.F90:101-122).
// Returns true when a point of this thread has det < 0.
// The load and the metric of a point are evaluated by different waves, side by
// side (the lower half of the workgroup has the metric).
template <int SPACE, bool STAGED>
__device__ __forceinline__ bool sf_points_of(const SfElem &es, const SfTab &tb, const unsigned short *gmap,
                                             const double *xn, int ngeo, double coef, int load, double *d, int tid0,
                                             int wgs0)
{
    // waves of the load and of the metric (one wave alone: both, in turn)
    const int wl = wgs0 >= 128 ? wgs0 / 128 * 64 : 0, wm = wgs0 - wl;
    const bool half = tid0 >= wm;
    const int tid = half ? tid0 - wm : tid0, wgs = half ? wl : wm;
    const int Q = es.nint, mB = es.m[0], mC = es.m[2];
    const int r0 = es.rol[0], r1 = es.rol[1], r2 = es.rol[2]; // roles of x, y, z
    bool neg = false;
    for (int l = tid; l < Q; l += wgs) {
        const int l1 = div_small(l, mC), qC = l - l1 * mC, qA = div_small(l1, mB), qB = l1 - qA * mB;
        const int q0 = sf_pick(r0, qB, qA, qC), q1 = sf_pick(r1, qB, qA, qC), q2 = sf_pick(r2, qB, qA, qC);
        double x[3], jm[3][3], inv[3][3];
        const double det = sf_map<STAGED>(es, tb, gmap, xn, ngeo, q0, q1, q2, x, jm, inv);
        neg = neg || det < 0.0;
        const double rdet = 1.0 / det;
        const double wd = det * (tb.w[0][qB] * tb.w[1][qA] * tb.w[2][qC]);
        if (half || wl == 0) {
            double f[3];
            getf(load, x, f);
            if (SPACE == 0) {
                d[6 * Q + l] = f[0] * wd;
            } else {
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    d[(12 + es.rol[c]) * Q + l] = (inv[c][0] * f[0] + inv[c][1] * f[1] + inv[c][2] * f[2]) * wd;
            }
            if (wl > 0) continue;
        }
        // the square roots of the weights are taken and squared again so that
        // a negative weight gives NaN, as the reference's A_TEST factors do
        const double sm = sqrt(coef * wd);
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
            for (int c = 0; c < 3; ++c) inv[r][c] *= sm;
        constexpr int M0 = SPACE == 0 ? 0 : 6; // first mass / gradient field
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
            for (int s = r; s < 3; ++s)
                d[(M0 + sf_sym(es.rol[r], es.rol[s])) * Q + l] =
                    inv[r][0] * inv[s][0] + inv[r][1] * inv[s][1] + inv[r][2] * inv[s][2];
        if (SPACE == 1) {
            const double sc = sqrt(wd) * rdet;
#pragma unroll
            for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int r = 0; r < 3; ++r) jm[c][r] *= sc;
#pragma unroll
            for (int r = 0; r < 3; ++r)
#pragma unroll
                for (int s = r; s < 3; ++s)
                    d[sf_sym(es.rol[r], es.rol[s]) * Q + l] = jm[0][r] * jm[0][s] + jm[1][r] * jm[1][s] + jm[2][r] * jm[2][s];
        }
    }
    return neg;
}
template <int SPACE>
__device__ __forceinline__ bool sf_points(const SfElem &es, const SfTab &tb, const unsigned short *gmap,
                                          const ElemArgs &a, int e, const double *xg, double *d, int tid, int wgs)
{
    const double coef = xg[3 * XS_MAX];
    if (a.ngeo <= XS_MAX) return sf_points_of<SPACE, true>(es, tb, gmap, xg, a.ngeo, coef, a.load, d, tid, wgs);
    return sf_points_of<SPACE, false>(es, tb, gmap, a.xnod + 3 * (size_t)a.ngeo * e, a.ngeo, coef, a.load, d, tid, wgs);
}

// The pencils (comp, iA, iB) that carry a dof, in ascending order, and the
// first of every (comp, iA) in js[comp * 8 + iA] (js[comp * 8 + 7]: one past
// the component's last); one wave.
template <int SPACE>
__device__ __forceinline__ void sf_pencils(SfElem &es, const short *row, unsigned short *pl, short *js, int lane)
{
    constexpr int NP = sf_comps(SPACE) * SF_I * SF_I;
    int cnt = 0;
    for (int k0 = 0; k0 < NP; k0 += 64) {
        const int k = k0 + lane;
        bool any = false;
        if (k < NP && k % SF_I < es.m[0] && (k / SF_I) % SF_I < es.m[1]) {
            const int4 r = *reinterpret_cast<const int4 *>(row + 8 * k);
            any = (r.x & r.y & r.z & r.w) != -1; // -1 in all eight
        }
        const unsigned long long bal = __ballot(any);
        const int at = cnt + __popcll(bal & ((1ull << lane) - 1));
        if (k < NP) {
            const int iB = k % SF_I, iA = (k / SF_I) % SF_I, c = k / (SF_I * SF_I);
            if (any) pl[at] = (unsigned short)(c << 6 | iA << 3 | iB);
            if (iB == 0) {
                js[c * 8 + iA] = (short)at;
                if (iA == 0 && c > 0) js[c * 8 - 1] = (short)at;
            }
        }
        cnt += __popcll(bal);
    }
    if (lane == 0) {
        js[(sf_comps(SPACE) - 1) * 8 + 7] = (short)cnt;
        es.np = cnt;
    }
}

// one entry of a 1D transform: sum over the n points at `stride` of g f
__device__ __forceinline__ double sf_dot(const double *g, int stride, int n, const double *f)
{
    double a[SF_I], b[SF_I], s = 0.0;
#pragma unroll
    for (int q = 0; q < SF_I; ++q) {
        const int p = min(q, n - 1);
        a[q] = g[p * stride];
        b[q] = f[q];
    }
#pragma unroll
    for (int q = 0; q < SF_I; ++q) s = fma(q < n ? a[q] : 0.0, b[q], s);
    return s;
}

// Pair (il, jl) of T's rows and columns: rectangular, jl ni + il, or TRI (H1,
// each pair of pencils once): the rows up to the column's own index,
// jA (jA + 1) / 2 + iA from the chunk's first
template <bool TRI> __device__ __forceinline__ int sf_tpair(int iA, int jA, int i0, int j0, int ni)
{
    return TRI ? (jA * (jA + 1) - j0 * (j0 + 1)) / 2 + iA : (jA - j0) * ni + iA - i0;
}

// T tables of the columns jA in [j0, j0 + nj) against the rows iA in
// [i0, i0 + ni) (np pairs): t[tab * ts + (pair * mB + qB) * MCP + qC], in
// H(curl) for columns of component b, and of the next `nb` - 1 components at
// t + per each
template <int SPACE, int MC, bool TRI>
__device__ __forceinline__ void sf_build_t(const SfElem &es, const SfTab &tb, const double *d, double *t, int ts, int per,
                                           int j0, int np, int i0, int ni, int b0, int nb, int tid, int wgs)
{
    constexpr int MCP = (MC + 1) & ~1;
    const int mA = es.m[1], mB = es.m[0], Q = es.nint;
    const double *f0 = tb.f[1][0], *f1 = tb.f[1][1];
    const int one = np * mB * MC;
    for (int kk = tid; kk < nb * one; kk += wgs) {
        const int u = SPACE == 0 ? 0 : (kk >= one) + (kk >= 2 * one), k = kk - u * one, b = b0 + u;
        const int k1 = k / MC, qC = k - k1 * MC, k2 = div_small(k1, mB), qB = k1 - k2 * mB;
        int iA, jA;
        if (TRI) {
            const int m = k2 + j0 * (j0 + 1) / 2;
            jA = j0;
#pragma unroll
            for (int j = 1; j < SF_I; ++j) jA = m >= j * (j + 1) / 2 ? j : jA;
            iA = m - jA * (jA + 1) / 2;
        } else {
            const int jl = div_small(k2, ni);
            iA = i0 + k2 - jl * ni;
            jA = j0 + jl;
        }
        const double *g = d + qB * MC + qC;
        double v[sf_ttabs(SPACE)];
#pragma unroll
        for (int s = 0; s < sf_ttabs(SPACE); ++s) v[s] = 0.0;
        for (int qA = 0; qA < mA; ++qA, g += mB * MC) {
            const double i_0 = f0[8 * iA + qA], i_1 = f1[8 * iA + qA], j_0 = f0[8 * jA + qA], j_1 = f1[8 * jA + qA];
            if constexpr (SPACE == 0) {
                // A = y, B = x, C = z
                const double vv = i_0 * j_0, dv = i_1 * j_0, vd = i_0 * j_1, dd = i_1 * j_1;
                const double gab = g[sf_sym(0, 1) * Q], gac = g[sf_sym(1, 2) * Q];
                v[0] += dd * g[sf_sym(1, 1) * Q];
                v[1] += dv * gab;
                v[2] += vd * gab;
                v[3] += vv * g[sf_sym(0, 0) * Q];
                v[4] += dv * gac;
                v[5] += vd * gac;
                v[6] += vv * g[sf_sym(0, 2) * Q];
                v[7] += vv * g[sf_sym(2, 2) * Q];
            } else {
                const double jm = b == 1 ? j_1 : j_0; // mass: derivative in the component's direction
#pragma unroll
                for (int a = 0; a < 3; ++a) v[a] += (a == 1 ? i_1 : i_0) * jm * g[(6 + sf_sym(a, b)) * Q];
#pragma unroll
                for (int r2 = 0; r2 < 2; ++r2) {
                    const int rj = r2 == 0 ? (b == 0 ? 1 : 0) : (b == 2 ? 1 : 2); // curl rows other than b
                    const double jc = rj != 1 ? j_1 : j_0;
#pragma unroll
                    for (int r = 0; r < 3; ++r) v[3 + 2 * r + r2] += (r != 1 ? i_1 : i_0) * jc * g[sf_sym(r, rj) * Q];
                }
            }
        }
        double *o = t + u * per + k1 * MCP + qC;
#pragma unroll
        for (int s = 0; s < sf_ttabs(SPACE); ++s) o[s * ts] = v[s];
    }
}

// one T vector in registers (t 16-byte aligned, padded to an even length)
template <int MC> struct SfVec {
    typedef double d2_t __attribute__((ext_vector_type(2)));
    d2_t v[(MC + 1) / 2];
    __device__ __forceinline__ void load(const double *t)
    {
#pragma unroll
        for (int q = 0; q < (MC + 1) / 2; ++q) v[q] = reinterpret_cast<const d2_t *>(t)[q];
    }
    // s[q] += p * v[q]
    __device__ __forceinline__ void axpy(double (&s)[MC], double p) const
    {
#pragma unroll
        for (int q = 0; q < MC; ++q) s[q] = fma(p, v[q / 2][q % 2], s[q]);
    }
};

// The 1D tables of the last direction, in scalar registers (uniform loads).
// Gauss points and functions are symmetric about the middle of [0, 1]:
// chi_0(x) = chi_1(1 - x), chi_i(1 - x) = (-1)^i chi_i(x) for i >= 2 and the
// opposite for chi_i', with chi_0' = -1 and chi_1' = 1, so half of the values
// do and a sum over the points takes half of the products (of sums or
// differences of mirrored points).
template <int MC> struct SfRow {
    static constexpr int H = (MC + 1) / 2, NH = MC > 2 ? MC - 2 : 1;
    double f0[MC], g[H];       // chi_0, and chi_0 - 1/2 up to the middle point
    double e[NH][H], d[NH][H]; // chi_i and chi_i', i >= 2, up to the middle point
    __device__ __forceinline__ SfRow()
    {
        typedef const __attribute__((address_space(4))) double *kd_t;
        kd_t p = (kd_t)(uintptr_t)&c_sf.f[MC][0][0][0], pg = (kd_t)(uintptr_t)&c_sf.g[MC][0];
#if defined(__HIP_DEVICE_COMPILE__)
        __asm__ volatile("" : "+s"(p), "+s"(pg)); // loaded here, not held across the element
#endif
#pragma unroll
        for (int q = 0; q < MC; ++q) f0[q] = p[q];
#pragma unroll
        for (int q = 0; q < H; ++q) g[q] = pg[q];
#pragma unroll
        for (int i = 2; i < MC; ++i)
#pragma unroll
            for (int q = 0; q < H; ++q) {
                e[i - 2][q] = p[8 * i + q];
                d[i - 2][q] = p[SF_I * 8 + 8 * i + q];
            }
    }
    // chi_i' at point q times s, and chi_i at point q times s plus that of t
    __device__ __forceinline__ double der(int i, int q, double s) const
    {
        if (i == 0) return -s;
        if (i == 1) return s;
        return q < H ? d[i - 2][q] * s : (i & 1 ? d[i - 2][MC - 1 - q] : -d[i - 2][MC - 1 - q]) * s;
    }
    __device__ __forceinline__ double both(int i, int q, double s, double t) const
    {
        if (i == 0) return fma(f0[q], s, -t);
        if (i == 1) return fma(f0[MC - 1 - q], s, t);
        const double c = q < H ? e[i - 2][q] : (i & 1 ? -e[i - 2][MC - 1 - q] : e[i - 2][MC - 1 - q]);
        return fma(c, s, der(i, q, t));
    }
};

// The block of pencil pair (first, second) from its S vectors, emitted column
// by column as em.col(iG, values over iF).  S_xy: derivative in C on the first
// (x) and second (y) function.  KIND 0: all four, 1: S01 and S11 (the second's
// component is C), 2: S11 alone (both are).
template <int MC, int KIND, typename EM>
__device__ __forceinline__ void sf_block(const double (&s00)[MC], const double (&s01)[MC], const double (&s10)[MC],
                                         const double (&s11)[MC], const EM &em)
{
    constexpr int H = (MC + 1) / 2, L = MC / 2; // points up to and below the middle
    auto column = [&](int j, const SfRow<MC> &tab) __attribute__((always_inline)) {
        double r[MC];
#pragma unroll
        for (int i = 0; i < MC; ++i) r[i] = 0.0;
#pragma unroll
        for (int q = 0; q < H; ++q) {
            // the second function's sums at q and its mirror point (v0: the
            // first not differentiated, v1: differentiated), their sums e and
            // differences o
            const int m = MC - 1 - q;
            auto at = [&](const double (&s0)[MC], const double (&s1)[MC], int p) __attribute__((always_inline)) {
                return KIND == 0 ? tab.both(j, p, s0[p], s1[p]) : tab.der(j, p, s1[p]);
            };
            const double a1 = at(s10, s11, q), b1 = q < L ? at(s10, s11, m) : 0.0;
            const double e1 = q < L ? a1 + b1 : a1, o1 = a1 - b1;
            double e0 = 0.0, o0 = 0.0;
            if (KIND < 2) {
                const double a0 = at(s00, s01, q), b0 = q < L ? at(s00, s01, m) : 0.0;
                e0 = q < L ? a0 + b0 : a0;
                o0 = a0 - b0;
            }
            // chi_0 and chi_1: 1/2 +- g at q and 1/2 -+ g at its mirror point
            double c0 = -e1, c1 = e1;
            if (KIND < 2) {
                if (q < L) {
                    c0 = fma(tab.g[q], o0, c0);
                    c1 = fma(-tab.g[q], o0, c1);
                }
                c0 = fma(0.5, e0, c0);
                c1 = fma(0.5, e0, c1);
            }
            r[0] += c0;
            r[1] += c1;
#pragma unroll
            for (int i = 2; i < MC; ++i) {
                if (KIND < 2 && (i % 2 == 0 || q < L)) r[i] = fma(tab.e[i - 2][q], i % 2 ? o0 : e0, r[i]);
                if (i % 2 || q < L) r[i] = fma(tab.d[i - 2][q], i % 2 ? e1 : o1, r[i]);
            }
        }
        em.col(j, r);
    };
    // for MC <= 5 the tables fit the scalar registers for all columns
    if constexpr (MC <= 5) {
        const SfRow<MC> tab;
#pragma unroll
        for (int j = KIND == 0 ? 0 : 1; j < MC; ++j) column(j, tab);
    } else {
#pragma unroll
        for (int j = KIND == 0 ? 0 : 1; j < MC; ++j) column(j, SfRow<MC>());
    }
}

// What an item needs: its two pencils in canonical order (first = the lower
// pencil number, so that K(I, J) and K(J, I) are the same operations on the
// same numbers and K is symmetric to the bit) and where T holds its sums.
struct SfItem {
    int iBF, iBG, aF, aG; // B indexes and components of first and second
    bool swap;            // first is the column pencil
    const double *t;      // table 0 at (jl, il)
};

// H1: S from the nine (s, t) terms
template <int MC, typename EM>
__device__ __forceinline__ void sf_item_h1(const SfItem &it, const SfTab &tb, int mB, int ts, const EM &em)
{
    constexpr int MCP = (MC + 1) & ~1;
    const double *fF = tb.f[0][0] + 8 * it.iBF, *fG = tb.f[0][0] + 8 * it.iBG;
    constexpr int DER = SF_I * 8;
    const double *t = it.t;
    // tables with the A derivative on the first / the second function
    const int oF = it.swap ? 2 : 1, oG = 3 - oF;
    double s00[MC], s01[MC], s10[MC], s11[MC];
#pragma unroll
    for (int q = 0; q < MC; ++q) s00[q] = s01[q] = s10[q] = s11[q] = 0.0;
    for (int qB = 0; qB < mB; ++qB, t += MCP) {
        const double vF = fF[qB], dF = fF[DER + qB], vG = fG[qB], dG = fG[DER + qB];
        // half of the tables at a time in flight (pairs for MC = 7, which has
        // not the registers)
        constexpr bool ALL = MC < 7;
        SfVec<MC> a0, a1, a2, a3;
        a0.load(t);
        a1.load(t + oF * ts);
        if (!ALL) __builtin_amdgcn_sched_barrier(0);
        const double vv = vF * vG, vd = vF * dG, dv = dF * vG, dd = dF * dG;
        if (!ALL) {
            a0.axpy(s00, vv);
            a1.axpy(s00, vd);
        }
        a2.load(t + oG * ts);
        a3.load(t + 3 * ts);
        __builtin_amdgcn_sched_barrier(0);
        if (ALL) {
            a0.axpy(s00, vv);
            a1.axpy(s00, vd);
        }
        a2.axpy(s00, dv);
        a3.axpy(s00, dd);
        a0.load(t + (3 + oF) * ts);
        a1.load(t + (3 + oG) * ts);
        if (!ALL) {
            __builtin_amdgcn_sched_barrier(0);
            a0.axpy(s01, vv);
            a1.axpy(s10, vv);
        }
        a2.load(t + 6 * ts);
        a3.load(t + 7 * ts);
        __builtin_amdgcn_sched_barrier(0);
        if (ALL) {
            a0.axpy(s01, vv);
            a1.axpy(s10, vv);
        }
        a2.axpy(s01, dv);
        a2.axpy(s10, vd);
        a3.axpy(s11, vv);
    }
    sf_block<MC, 0>(s00, s01, s10, s11, em);
}

// H(curl), by the components of the pair: KIND 0 neither is z, 1 the second
// is, 2 both are.  The sign of curl row r of a component-a dof is + for
// r = a + 1 and - for r = a + 2 (mod 3); the derivative of curl row r in B = x
// is absent for r = 0, that of the mass term present for a = 0.
template <int MC, int KIND, typename EM>
__device__ __forceinline__ void sf_item_hcurl(const SfItem &it, const SfTab &tb, int mB, int ts, const EM &em)
{
    constexpr int MCP = (MC + 1) & ~1;
    const double *fF = tb.f[0][0] + 8 * it.iBF, *fG = tb.f[0][0] + 8 * it.iBG;
    constexpr int DER = SF_I * 8;
    const double *t = it.t;
    const bool sw = it.swap;
    const int aI = sw ? it.aG : it.aF; // component of the row pencil
    double s00[MC], s01[MC], s10[MC], s11[MC];
#pragma unroll
    for (int q = 0; q < MC; ++q) s00[q] = s01[q] = s10[q] = s11[q] = 0.0;
    if constexpr (KIND == 0) {
        // curl rows z (no C derivative) and o = 1 - a; tables (rI, rJ) at
        // 3 + 2 rI + (rJ is z)
        const int oI = 3 + 2 * (1 - aI), m = aI * ts, zz = 8 * ts, oo = oI * ts;
        const int zo = (sw ? oI + 1 : 7) * ts, oz = (sw ? 7 : oI + 1) * ts; // (first, second)
        const double eps = it.aF == it.aG ? 1.0 : -1.0;
        for (int qB = 0; qB < mB; ++qB, t += MCP) {
            const double vF = fF[qB], dF = fF[DER + qB], vG = fG[qB], dG = fG[DER + qB];
            const double mF = it.aF == 0 ? dF : vF, mG = it.aG == 0 ? dG : vG;
            const double emG = eps * mG, edG = eps * dG;
            SfVec<MC> am, azz, azo, aoz, aoo;
            am.load(t + m);
            azz.load(t + zz);
            if (MC > 6) __builtin_amdgcn_sched_barrier(0);
            azo.load(t + zo);
            aoz.load(t + oz);
            aoo.load(t + oo);
            __builtin_amdgcn_sched_barrier(0);
            am.axpy(s00, mF * mG);
            azz.axpy(s00, dF * edG);
            azo.axpy(s01, -dF * emG);
            aoz.axpy(s10, -mF * edG);
            aoo.axpy(s11, mF * emG);
        }
    } else if constexpr (KIND == 1) {
        // first: rows z and o; second (component z): rows 0 and 1
        const int m = aI * ts, z0 = (sw ? 4 : 7) * ts, z1 = (sw ? 6 : 8) * ts;
        const int oI = 3 + 2 * (1 - it.aF), o0 = (sw ? 3 : oI) * ts, o1 = (sw ? 5 : oI + 1) * ts;
        const double sg = it.aF == 0 ? -1.0 : 1.0;
        for (int qB = 0; qB < mB; ++qB, t += MCP) {
            const double vF = fF[qB], dF = fF[DER + qB], vG = fG[qB], dG = fG[DER + qB];
            const double mF = it.aF == 0 ? dF : vF, sd = sg * dF, sm = sg * mF;
            SfVec<MC> am, az0, az1, ao0, ao1;
            am.load(t + m);
            az0.load(t + z0);
            if (MC > 6) __builtin_amdgcn_sched_barrier(0);
            az1.load(t + z1);
            ao0.load(t + o0);
            ao1.load(t + o1);
            __builtin_amdgcn_sched_barrier(0);
            am.axpy(s01, mF * vG);
            az0.axpy(s01, sd * vG);
            az1.axpy(s01, -sd * dG);
            ao0.axpy(s11, -sm * vG);
            ao1.axpy(s11, sm * dG);
        }
    } else {
        const int r01 = (sw ? 5 : 4) * ts, r10 = (sw ? 4 : 5) * ts;
        for (int qB = 0; qB < mB; ++qB, t += MCP) {
            const double vF = fF[qB], dF = fF[DER + qB], vG = fG[qB], dG = fG[DER + qB];
            const double vv = vF * vG;
            SfVec<MC> am, a00, a01, a10, a11;
            am.load(t + 2 * ts);
            a00.load(t + 3 * ts);
            a01.load(t + r01);
            a10.load(t + r10);
            a11.load(t + 6 * ts);
            __builtin_amdgcn_sched_barrier(0);
            am.axpy(s11, vv);
            a00.axpy(s11, vv);
            a01.axpy(s11, -vF * dG);
            a10.axpy(s11, -dF * vG);
            a11.axpy(s11, dF * dG);
        }
    }
    sf_block<MC, KIND>(s00, s01, s10, s11, em);
}

// one of the eight packed rows of a pencil
__device__ __forceinline__ int sf_row_of(const int4 &r, int i)
{
    const int w = i < 2 ? r.x : i < 4 ? r.y : i < 6 ? r.z : r.w;
    return (int)(short)(i & 1 ? w >> 16 : w);
}

// v with the sign of the entry whose packed rows are f and g
__device__ __forceinline__ double sf_signed(int f, int g, double v)
{
    const unsigned hi = (unsigned)__double2hiint(v) ^ (((unsigned)(f ^ g) << 17) & 0x80000000u);
    return __hiloint2double((int)hi, __double2loint(v));
}

// Where the columns of a pencil pair's block go: an object made from the packed
// rows of the pair, with col(j, r): r[i] belongs to (first i, second j).  On the
// diagonal pair (diag) the block's upper half serves both halves.
//
// K in memory (any leading dimension): consecutive lanes hold consecutive row
// pencils of one column pencil, so a store writes pieces of one column.
template <typename T, int MC> struct SfColK {
    T *k;
    long long ld, aF, aG;
    int4 rF, rG;
    bool diag, full;
    __device__ __forceinline__ SfColK(T *k_, long long ld_, const int4 rI, const int4 rJ, bool swap, bool diag_)
        : k(k_), ld(ld_), aF(swap ? ld_ : 1), aG(swap ? 1 : ld_), rF(swap ? rJ : rI), rG(swap ? rI : rJ), diag(diag_)
    {
        bool ok = !diag;
#pragma unroll
        for (int i = 0; i < MC; ++i) ok = ok && sf_row_of(rF, i) >= 0 && sf_row_of(rG, i) >= 0;
        full = __all(ok); // no missing dof, no diagonal pair in the wave
    }
    __device__ __forceinline__ void col(int j, const double (&r)[MC]) const
    {
        const int eG = sf_row_of(rG, j);
        T *const kj = k + (eG & ~ROW_NEG) * aG;
        if (full) {
#pragma unroll
            for (int i = 0; i < MC; ++i) {
                const int eF = sf_row_of(rF, i);
                kj[(eF & ~ROW_NEG) * aF] = (T)sf_signed(eF, eG, r[i]);
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < MC; ++i) {
            const int eF = sf_row_of(rF, i);
            if (eF < 0 || eG < 0 || (diag && i > j)) continue;
            const T v = (T)sf_signed(eF, eG, r[i]);
            kj[(eF & ~ROW_NEG) * aF] = v;
            if (diag && i < j) k[(eF & ~ROW_NEG) * ld + (eG & ~ROW_NEG)] = v;
        }
    }
};
template <typename T> struct SfToK {
    T *k;
    long long ld;
    template <int MC> __device__ __forceinline__ SfColK<T, MC> pair(const int4 rI, const int4 rJ, bool swap, bool diag) const
    {
        return SfColK<T, MC>(k, ld, rI, rJ, swap, diag);
    }
};

// K in LDS (SfLay), every unordered pair visited once.  (On the diagonal pair
// both halves go to the same place, the upper half's value last.)
template <int MC> struct SfColPacked {
    double *o;
    SfLay ly;
    int4 rF, rG;
    int oF[MC];
    bool full;
    __device__ __forceinline__ SfColPacked(double *pk, const SfLay &l, const int4 f, const int4 g) : o(pk), ly(l), rF(f), rG(g)
    {
        bool ok = true;
#pragma unroll
        for (int i = 0; i < MC; ++i) {
            const int eF = sf_row_of(rF, i);
            ok = ok && eF >= 0 && sf_row_of(rG, i) >= 0;
            oF[i] = ly.row(eF & ~ROW_NEG);
        }
        full = __all(ok); // no dof is missing from any of the wave's pencils
    }
    __device__ __forceinline__ void col(int j, const double (&r)[MC]) const
    {
        const int eG = sf_row_of(rG, j), g = eG & ~ROW_NEG, og = ly.row(g);
        if (full) {
#pragma unroll
            for (int i = 0; i < MC; ++i) {
                const int eF = sf_row_of(rF, i), f = eF & ~ROW_NEG, lo = oF[i] + g, up = og + f;
                o[f >= g ? lo : up] = sf_signed(eF, eG, r[i]);
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < MC; ++i) {
            const int eF = sf_row_of(rF, i), f = eF & ~ROW_NEG, lo = oF[i] + g, up = og + f;
            if (eF >= 0 && eG >= 0) o[f >= g ? lo : up] = sf_signed(eF, eG, r[i]);
        }
    }
};
struct SfToPacked {
    double *pk;
    SfLay ly;
    template <int MC> __device__ __forceinline__ SfColPacked<MC> pair(const int4 rF, const int4 rG, bool, bool) const
    {
        return SfColPacked<MC>(pk, ly, rF, rG);
    }
};

// K in memory (when asked for) and, for an element that is condensed (aii), its
// bubble rows packed in LDS and its interface block, still without the
// condensation's update, in Aii's place
template <typename T> struct SfToSplit {
    T *k;
    long long ld;
    double *kb, *aii; // bubble rows, stride ldb
    int ni, ldb;
    template <int MC> struct Col {
        SfToSplit to;
        int4 rI, rJ;
        bool swap, diag;
        __device__ __forceinline__ void put(int a, int b, double v) const
        {
            if (to.k) to.k[a + b * to.ld] = (T)v;
            if (!to.aii) return;
            if (a < to.ni && b < to.ni) to.aii[a + (size_t)b * to.ni] = v;
            else if (a >= b) to.kb[(a - to.ni) * to.ldb + b] = v;
        }
        __device__ __forceinline__ void col(int j, const double (&r)[MC]) const
        {
#pragma unroll
            for (int i = 0; i < MC; ++i) {
                const int eI = sf_row_of(rI, swap ? j : i), eJ = sf_row_of(rJ, swap ? i : j);
                if (eI < 0 || eJ < 0 || (diag && i > j)) continue;
                const double v = sf_signed(eI, eJ, r[i]);
                put(eI & ~ROW_NEG, eJ & ~ROW_NEG, v);
                if (diag && i < j) put(eJ & ~ROW_NEG, eI & ~ROW_NEG, v);
            }
        }
    };
    template <int MC> __device__ __forceinline__ Col<MC> pair(const int4 rI, const int4 rJ, bool swap, bool diag) const
    {
        return Col<MC>{*this, rI, rJ, swap, diag};
    }
};

// The pencil pairs of the column chunks of `part` out of `nparts`: T for a
// chunk, then one pair per thread and step.  TRI: unordered pairs, the row
// pencil not above the column's; otherwise every row pencil.  d: the fields,
// t: `room` doubles for T.
template <int SPACE, int MC, bool TRI, typename TO>
__device__ __forceinline__ void sf_matrix(const SfElem &es, const SfTab &tb, const short *row,
                                          const unsigned short *pl, const short *js, const double *d, double *t,
                                          int room, const TO &to, int part, int nparts, int tid, int wgs)
{
    constexpr int MCP = (MC + 1) & ~1, NT = sf_ttabs(SPACE);
    const int mA = es.m[1], mB = es.m[0];
    // as many columns jA at a time as the pool holds; if it does not hold one
    // against all rows, the rows in pieces (elements whose 1D orders exceed
    // what their dof count suggests).  TT: pairs of T stored once.
    constexpr bool TT = TRI && SPACE == 0;
    const int one = NT * mB * MCP, have = room / one;
    const bool whole = have >= mA; // a column against all rows
    const int ni = whole ? mA : max(1, have);
    const int n01 = SPACE == 0 ? 0 : js[2 * 8]; // pencils of components x and y
    int w0 = 0;                                 // first wave of the next run: short runs take different waves
    // H(curl): several components at a time when they fit, whole each
    const int per = one * mA * mA;
    const int nbat = SPACE == 1 && nparts == 1 ? min(3, have / (mA * mA)) : 0;
    int part_at = 0;
    for (int b0 = 0; b0 < sf_comps(SPACE); b0 += max(nbat, 1)) {
        const int nb = nbat > 0 ? min(nbat, sf_comps(SPACE) - b0) : 1;
        for (int j0 = 0, njc; j0 < mA; j0 += njc) {
            // columns of this chunk
            if (nbat > 0) njc = mA;
            else if (nparts > 1 || !whole) njc = 1;
            else if (TT) {
                njc = 1;
                while (j0 + njc < mA && sf_tpair<true>(0, j0 + njc + 1, 0, j0, 0) <= have) ++njc;
            } else {
                njc = min(have / mA, mA - j0);
            }
            if (nparts > 1 && (part_at++ % nparts) != part) continue;
            for (int i0 = 0; i0 < mA; i0 += ni) {
                const int nic = min(ni, mA - i0);
                const bool tt = TT && whole;
                const int np = tt ? sf_tpair<true>(0, j0 + njc, 0, j0, 0) : njc * nic, ts = np * mB * MCP;
                if (tt) sf_build_t<SPACE, MC, TT>(es, tb, d, t, ts, per, j0, np, i0, nic, b0, nb, tid, wgs);
                else sf_build_t<SPACE, MC, false>(es, tb, d, t, ts, per, j0, np, i0, nic, b0, nb, tid, wgs);
                lds_barrier();
                for (int u = 0; u < nb; ++u) {
                    const int b = b0 + u;
                    const int pj0 = js[b * 8 + j0], pj1 = js[b * 8 + (j0 + njc < SF_I ? j0 + njc : SF_I)], npj = pj1 - pj0;
                    if (npj == 0) continue;
                    const double *const tu = t + u * per;
            // row pencils [pi0, pi1), with tri up to the column's own; KIND as
            // in sf_block
            auto run = [&](auto kind, int pi0, int pi1, bool tri) __attribute__((always_inline)) {
                constexpr int KIND = decltype(kind)::value;
                const int npi = pi1 - pi0, q0 = pj0 - pi0, q1 = pj1 - pi0;
                const int base = tri ? q0 * (q0 + 1) / 2 : 0;
                const int nit = tri ? q1 * (q1 + 1) / 2 - base : npi * npj;
                const float rn = 1.0f / (float)max(npi, 1);
                int k = tid - 64 * w0;
                if (k < 0) k += wgs;
                w0 += (nit + 63) >> 6;
                while (64 * w0 >= wgs) w0 -= wgs >> 6;
                for (; k < nit; k += wgs) {
                    int I, J;
                    if (tri) {
                        const int m = k + base;
                        int q = (int)((sqrtf(8.0f * (float)m + 1.0f) - 1.0f) * 0.5f);
                        if (q * (q + 1) / 2 > m) --q;
                        if ((q + 1) * (q + 2) / 2 <= m) ++q;
                        J = pi0 + q;
                        I = pi0 + m - q * (q + 1) / 2;
                    } else {
                        const int jx = (int)(((float)k + 0.5f) * rn);
                        I = pi0 + k - jx * npi;
                        J = pj0 + jx;
                    }
                    const int pI = pl[I], pJ = pl[J];
                    const int iAI = (pI >> 3) & 7, iBI = pI & 7, iAJ = (pJ >> 3) & 7, iBJ = pJ & 7;
                    if (TRI && (iAI < i0 || iAI >= i0 + nic)) continue; // (rows in pieces)
                    SfItem it;
                    it.swap = !TRI && I > J;
                    it.iBF = it.swap ? iBJ : iBI;
                    it.iBG = it.swap ? iBI : iBJ;
                    it.aF = it.swap ? pJ >> 6 : pI >> 6;
                    it.aG = it.swap ? pI >> 6 : pJ >> 6;
                    it.t = tu + (tt ? sf_tpair<true>(iAI, iAJ, 0, j0, 0) : sf_tpair<false>(iAI, iAJ, i0, j0, nic)) * mB * MCP;
                    const int4 rI = *reinterpret_cast<const int4 *>(row + 8 * (((pI >> 6) * SF_I + iAI) * SF_I + iBI));
                    const int4 rJ = *reinterpret_cast<const int4 *>(row + 8 * (((pJ >> 6) * SF_I + iAJ) * SF_I + iBJ));
                    const auto em = to.template pair<MC>(rI, rJ, it.swap, I == J);
                    if constexpr (SPACE == 0) sf_item_h1<MC>(it, tb, mB, ts, em);
                    else sf_item_hcurl<MC, KIND>(it, tb, mB, ts, em);
                }
            };
            typedef std::integral_constant<int, 0> k0_t;
            typedef std::integral_constant<int, 1> k1_t;
            typedef std::integral_constant<int, 2> k2_t;
            const int i1 = i0 + nic < SF_I ? i0 + nic : SF_I;
            if constexpr (SPACE == 0) {
                if (TRI) run(k0_t{}, 0, pj1, true);
                else run(k0_t{}, js[i0], js[i1], false);
            } else if (TRI) {
                if (b < 2) {
                    run(k0_t{}, 0, pj1, true);
                } else {
                    run(k1_t{}, 0, n01, false);
                    run(k2_t{}, n01, pj1, true);
                }
            } else {
                // components x and y together when all rows are at hand; z
                // starts on a whole wave
                for (int c = 0; c < 3; ++c) {
                    int pi0 = js[c * 8 + i0], pi1 = js[c * 8 + i1];
                    if (ni >= mA && c == 0) continue;
                    if (ni >= mA && c == 1) pi0 = 0;
                    if (c < 2 && b < 2) run(k0_t{}, pi0, pi1, false);
                    else if (c == 2 && b == 2) run(k2_t{}, pi0, pi1, false);
                    else run(k1_t{}, pi0, pi1, false);
                }
            }
                }
                lds_barrier();
            }
        }
    }
}

// Load vector, entry by entry as put(row, value): the load fields transformed
// in place, one direction after the other; ends with a barrier.
template <int SPACE, int WGS, typename PUT>
__device__ __forceinline__ void sf_load(const SfElem &es, const SfTab &tb, const short *row, double *g, const PUT &put,
                                        int tid)
{
    constexpr int U = (sf_comps(SPACE) * SF_I * SF_I * SF_I + WGS - 1) / WGS;
    const int mA = es.m[1], mB = es.m[0], mC = es.m[2], Q = es.nint, len = sf_comps(SPACE) * Q;
#pragma unroll
    for (int step = 0; step < 3; ++step) {
        double v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            // entry (c; a, b, z): line along A, B or C through its other two indexes
            if ((tid & ~63) + u * WGS >= len) continue; // (whole waves)
            const int k = min(tid + u * WGS, len - 1), c = SPACE == 0 ? 0 : (k >= Q) + (k >= 2 * Q), k0 = k - c * Q;
            const int l1 = div_small(k0, mC), z = k0 - l1 * mC, a = div_small(l1, mB), b = l1 - a * mB;
            const double *gc = g + c * Q;
            if (step == 0) v[u] = sf_dot(gc + b * mC + z, mB * mC, mA, tb.f[1][SPACE == 1 && c == 1] + 8 * a);
            if (step == 1) v[u] = sf_dot(gc + a * mB * mC + z, mC, mB, tb.f[0][SPACE == 1 && c == 0] + 8 * b);
            if (step == 2) v[u] = sf_dot(gc + l1 * mC, 1, mC, tb.f[2][SPACE == 1 && c == 2] + 8 * z);
            if (step == 2 && tid + u * WGS < len) {
                const int r = row[((c * SF_I + a) * SF_I + b) * 8 + z];
                if (r >= 0) put(r & ~ROW_NEG, r & ROW_NEG ? -v[u] : v[u]);
            }
        }
        lds_barrier();
        if (step == 2) break;
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (tid + u * WGS < len) g[tid + u * WGS] = v[u];
        lds_barrier();
    }
}

// Element matrices and loads: one workgroup per (element, part); the parts of
// an element share its column chunks, so that a few elements fill the chip.
// Bound by writing K (9.6 GB for 4,096 H(curl) p = 5 elements in FP64, at the
// rate of a large copy 2 ms): the element + condensation step of that mesh
// took 54.4 ms with the A A^T product on MFMA tiles (41 ms of it the product)
// and takes 15.7 ms (3.7 ms of it this kernel); element matrices of 990
// H(curl) p = 4 elements in FP32 1.53 -> 0.24 ms.
template <typename T, int SPACE, int WGS, int POOL, int WPE>
__global__ __launch_bounds__(WGS, WPE) void sf_elem_kernel(ElemArgs a)
{
    __shared__ SfElem es;
    __shared__ SfTab tb;
    __shared__ double xg[3 * XS_MAX + 1];
    __shared__ __align__(16) short row[sf_comps(SPACE) * SF_I * SF_I * 8];
    __shared__ unsigned short pl[sf_comps(SPACE) * SF_I * SF_I];
    __shared__ short js[sf_comps(SPACE) * 8];
    __shared__ unsigned short gmap[SF_I * SF_I * SF_I];
    __shared__ __align__(16) double pool[POOL];
    const int e = blockIdx.x, tid = threadIdx.x, part = blockIdx.y, nparts = gridDim.y;
    const bool ok = sf_setup<SPACE, WGS>(a, e, es, xg, tid);
    if (!ok || es.n > a.max_ndof) { // invalid codes, or above the caller's bound
        if (tid == 0 && part == 0 && a.status) a.status[e] = ok ? HP3D_E_ARG : HP3D_E_ORDER;
        return;
    }
    sf_fill_tab<WGS>(es.m, tb, tid);
    sf_fill_rows<SPACE>(es, row, tid, WGS);
    if (a.ngeo != 8) sf_fill_gmap(es, a.ngeo, gmap, tid, WGS);
    lds_barrier();
    if (sf_points<SPACE>(es, tb, gmap, a, e, xg, pool, tid, WGS)) es.negjac = 1;
    if (tid < 64) sf_pencils<SPACE>(es, row, pl, js, tid);
    lds_barrier();
    if (part == nparts - 1 && a.bout) {
        double *bo = a.bout + a.off_v[e];
        sf_load<SPACE, WGS>(es, tb, row, pool + (SPACE == 0 ? 6 : 12) * es.nint, [=](int r, double v) { bo[r] = v; }, tid);
    }
    const SfToK<T> to{(T *)a.kout + a.off_k[e], a.ld_k > 0 ? a.ld_k : es.n};
    const int dl = (SPACE == 0 ? 6 : 12) * es.nint; // T takes the load fields' place
    auto run = [&](auto mc) __attribute__((always_inline)) {
        sf_matrix<SPACE, decltype(mc)::value, false>(es, tb, row, pl, js, pool, pool + dl, POOL - dl, to, part, nparts,
                                                     tid, WGS);
    };
    switch (es.m[2]) {
    case 2: run(std::integral_constant<int, 2>{}); break;
    case 3: run(std::integral_constant<int, 3>{}); break;
    case 4: run(std::integral_constant<int, 4>{}); break;
    case 5: run(std::integral_constant<int, 5>{}); break;
    case 6: run(std::integral_constant<int, 6>{}); break;
    default: run(std::integral_constant<int, 7>{}); break;
    }
    if (tid == 0 && part == 0 && a.status) a.status[e] = es.negjac ? HP3D_NEG_JACOBIAN : 0;
}

// ------------------------------------------------------ fused condensation

template <int MC> struct SfColHold {
    double (&o)[MC][MC];
    __device__ __forceinline__ void col(int j, const double (&r)[MC]) const
    {
#pragma unroll
        for (int i = 0; i < MC; ++i) o[j][i] = r[i];
    }
};

// SF_HOLD: all pencil pairs of an H1 element at once, one (MC = 5) or two
// (MC = 4) per thread, their blocks in registers until every T has been read;
// then K packed over fields and T.
template <int MC, int NB>
__device__ __forceinline__ void sf_hold(const SfElem &es, const SfTab &tb, const short *row, const unsigned short *pl,
                                        double *pool, int dl, const SfLay &ly, int tid, int wgs)
{
    constexpr int MCP = (MC + 1) & ~1;
    const int mA = es.m[1], mB = es.m[0], np = mA * (mA + 1) / 2, ts = np * mB * MCP;
    double *t = pool + dl;
    sf_build_t<0, MC, true>(es, tb, pool, t, ts, 0, 0, np, 0, mA, 0, 1, tid, wgs);
    lds_barrier();
    const int nit = es.np * (es.np + 1) / 2;
    double out[NB][MC][MC];
    int ij[NB];
#pragma unroll
    for (int u = 0; u < NB; ++u) {
        const int k = tid + u * wgs;
        ij[u] = -1;
        if (k < nit) {
            int q = (int)((sqrtf(8.0f * (float)k + 1.0f) - 1.0f) * 0.5f);
            if (q * (q + 1) / 2 > k) --q;
            if ((q + 1) * (q + 2) / 2 <= k) ++q;
            const int pJ = pl[q], pI = pl[k - q * (q + 1) / 2];
            ij[u] = pI | pJ << 8;
            SfItem it;
            it.swap = false;
            it.aF = it.aG = 0;
            it.iBF = pI & 7;
            it.iBG = pJ & 7;
            it.t = t + sf_tpair<true>(pI >> 3, pJ >> 3, 0, 0, 0) * mB * MCP;
            sf_item_h1<MC>(it, tb, mB, ts, SfColHold<MC>{out[u]});
        }
    }
    lds_barrier(); // T and the fields are read
    const SfToPacked to{pool, ly};
#pragma unroll
    for (int u = 0; u < NB; ++u) {
        if (ij[u] < 0) continue;
        const int pI = ij[u] & 255, pJ = ij[u] >> 8;
        const int4 rI = *reinterpret_cast<const int4 *>(row + 8 * ((pI >> 3) * SF_I + (pI & 7)));
        const int4 rJ = *reinterpret_cast<const int4 *>(row + 8 * ((pJ >> 3) * SF_I + (pJ & 7)));
        const auto em = to.pair<MC>(rI, rJ, false, pI == pJ);
#pragma unroll
        for (int j = 0; j < MC; ++j) em.col(j, out[u][j]);
    }
}

// y = d^-1/2 for d > 0: the hardware estimate and two Newton steps
__device__ __forceinline__ double sf_rsqrt(double d)
{
    double y = __builtin_amdgcn_rsq(d);
    y = fma(0.5 * y, fma(-d * y, y, 1.0), y);
    return fma(0.5 * y, fma(-d * y, y, 1.0), y);
}

// Blocked Cholesky Abb = L L^T of the bubble block (nb <= 16 NBT) and W = L^-1 by
// one wave, 4 x 4 diagonal blocks, on FP64 MFMA.  [Abb | I] sits in the MFMA
// result layout (tile rows in registers: lane group q, register j: row q + 4j),
// in which block row s is register s of its tile: by symmetry the operand that
// a rank-4 update takes on both sides, so no value changes lanes.  Step s: the
// 4 x 4 block to every lane (readlane), its inverse Cholesky factor, the block
// row times it (a block row of L^T and of W) and the update.  W's lower tiles
// go to w (row k at k (16 NBT + 1)), padded from nb to whole blocks with the identity.
// Returns true when a pivot is not positive.
template <int NBT>
__device__ __forceinline__ bool sf_factor(const double *kb, int ldb, int ni, int nb, double *w, int lane)
{
    constexpr int WLD = 16 * NBT + 1;
    typedef Mfma<double> MD;
    const int lr = lane & 15, lq = lane >> 4;
    d4_t acc[NBT][NBT], id[NBT][NBT]; // Abb: tiles (r, c), c >= r; I: c <= r
#pragma unroll
    for (int r = 0; r < NBT; ++r)
#pragma unroll
        for (int c = 0; c < NBT; ++c)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int i = 16 * r + lq + 4 * j, k = 16 * c + lr, hi = max(i, k), lo = min(i, k);
                if (c >= r) {
                    const double v = kb[hi < nb ? hi * ldb + ni + lo : 0];
                    acc[r][c][j] = hi < nb ? v : (i == k ? 1.0 : 0.0);
                }
                id[r][c][j] = i == k ? 1.0 : 0.0;
            }
    bool bad = false;
#pragma unroll
    for (int s = 0; s < 4 * NBT; ++s) {
        if (4 * s >= nb) continue;
        const int tr = s / 4, j = s % 4;
        const double p = acc[tr][tr][j];
        double d[4][4];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b <= a; ++b) d[a][b] = readlane_f64(p, 16 * a + 4 * j + b);
        auto root = [&](double x) __attribute__((always_inline)) {
            const bool pos = x > 0.0;
            bad |= !pos;
            return pos ? sf_rsqrt(x) : 0.0;
        };
        const double r0 = root(d[0][0]);
        const double l10 = d[1][0] * r0, l20 = d[2][0] * r0, l30 = d[3][0] * r0;
        const double r1 = root(fma(-l10, l10, d[1][1]));
        const double l21 = fma(-l20, l10, d[2][1]) * r1, l31 = fma(-l30, l10, d[3][1]) * r1;
        const double r2 = root(fma(-l21, l21, fma(-l20, l20, d[2][2])));
        const double l32 = fma(-l31, l21, fma(-l30, l20, d[3][2])) * r2;
        const double r3 = root(fma(-l32, l32, fma(-l31, l31, fma(-l30, l30, d[3][3]))));
        const double m10 = -r1 * (l10 * r0), m21 = -r2 * (l21 * r1), m32 = -r3 * (l32 * r2);
        const double m20 = -r2 * fma(l21, m10, l20 * r0), m31 = -r3 * fma(l32, m21, l31 * r1);
        const double m30 = -r3 * fma(l32, m20, fma(l31, m10, l30 * r0));
        // operand row lr, column lq of the inverse factor
        const double c0 = lr == 0 ? r0 : lr == 1 ? m10 : lr == 2 ? m20 : m30;
        const double c1 = lr == 0 ? 0.0 : lr == 1 ? r1 : lr == 2 ? m21 : m31;
        const double c2 = lr < 2 ? 0.0 : lr == 2 ? r2 : m32;
        const double c3 = lr == 3 ? r3 : 0.0;
        const double cv = lq == 0 ? c0 : lq == 1 ? c1 : lq == 2 ? c2 : c3;
        const double av = lr < 4 ? cv : 0.0;
        const d4_t zero = {0.0, 0.0, 0.0, 0.0};
        double lt[NBT], ws[NBT];
#pragma unroll
        for (int c = 0; c < NBT; ++c) {
            lt[c] = c >= tr ? MD::mma(av, acc[tr][c][j], zero)[0] : 0.0;
            ws[c] = c <= tr ? MD::mma(av, id[tr][c][j], zero)[0] : 0.0;
            if (c <= tr) w[(4 * s + lq) * WLD + 16 * c + lr] = ws[c];
        }
        // (the update also runs over rows and columns that are done: what it
        // leaves there is not read again)
#pragma unroll
        for (int r = tr; r < NBT; ++r)
#pragma unroll
            for (int c = 0; c < NBT; ++c) {
                if (c >= r) acc[r][c] = MD::mma(-lt[r], lt[c], acc[r][c]);
                if (c <= tr) id[r][c] = MD::mma(4 * s + 3 < 16 * r + lr ? -lt[r] : 0.0, ws[c], id[r][c]);
            }
    }
    return bad;
}

template <int R> struct SfSmall {
    double b[R + 4]; // load vector, and zeros up to a multiple of four bubbles
    int fail;
};

// The symmetric n x n matrix in LDS (SfLay), written to memory by waves w of nw:
// lanes along the rows (16, 32 or 64 lanes a column, two rows a lane beyond
// 64), columns strided over the waves, four loads in flight.  What depends on
// the column alone is scalar when a wave has one column at a time.
template <typename S>
__device__ __forceinline__ void sf_unpack(const double *pk, const SfLay &ly, S *out, size_t ld, int n, int w, int nw,
                                          int lane)
{
    if (n > 64) { // two rows a lane
        const int r0 = lane, r1 = min(lane + 64, n - 1), b0 = ly.row(r0), b1 = ly.row(r1);
        const bool two = lane + 64 < n;
        S *o = out + w * ld;
        const size_t st = nw * ld;
        auto col = [&](int c, double &v0, double &v1) __attribute__((always_inline)) {
            const int oc = ly.row(c), l0 = b0 + c, u0 = oc + r0, l1 = b1 + c, u1 = oc + r1;
            v0 = pk[c <= r0 ? l0 : u0];
            v1 = pk[c <= r1 ? l1 : u1];
        };
        int c = w;
        for (; c + nw < n; c += 2 * nw, o += 2 * st) {
            double v0, v1, w0, w1;
            col(c, v0, v1);
            col(c + nw, w0, w1);
            o[r0] = (S)v0;
            (o + st)[r0] = (S)w0;
            if (two) {
                o[r1] = (S)v1;
                (o + st)[r1] = (S)w1;
            }
        }
        if (c < n) {
            double v0, v1;
            col(c, v0, v1);
            o[r0] = (S)v0;
            if (two) o[r1] = (S)v1;
        }
    } else if (n > 32) {
        const int r = lane;
        if (r >= n) return;
        const int rb = ly.row(r);
        auto at = [&](int c) __attribute__((always_inline)) {
            const int lo = rb + c, up = ly.row(c) + r;
            return c <= r ? lo : up;
        };
        int c = w;
        S *o = out + c * ld;
        const size_t st = nw * ld;
        for (; c + 3 * nw < n; c += 4 * nw, o += 4 * st) {
            const double v0 = pk[at(c)], v1 = pk[at(c + nw)], v2 = pk[at(c + 2 * nw)], v3 = pk[at(c + 3 * nw)];
            o[r] = (S)v0;
            (o + st)[r] = (S)v1;
            (o + 2 * st)[r] = (S)v2;
            (o + 3 * st)[r] = (S)v3;
        }
        for (; c < n; c += nw, o += st) o[r] = (S)pk[at(c)];
    } else {
        const int lg = n <= 16 ? 4 : 5, r = lane & ((1 << lg) - 1), cpw = 64 >> lg;
        if (r >= n) return;
        const int rb = ly.row(r);
        for (int c = w * cpw + (lane >> lg); c < n; c += nw * cpw) {
            const int lo = rb + c, up = ly.row(c) + r;
            out[c * ld + r] = (S)pk[c <= r ? lo : up];
        }
    }
}

// After K and the load are in LDS: K written out while one wave factors Abb,
// then, 16 columns of [Abi | Bb] a tile, S = W [Abi | Bb] and X = W^T S on FP64
// MFMA (stc_fwd_herm, stc.F90:338-416): S over the bubble rows with its load
// column at column ni (Abb is not needed any more), X straight to ASchur and
// BSchur; last [Aii; Bi] = [Kii; b] - S^T S, lower tiles of an (ni + 1)-row
// matrix.  The bubble rows are padded with zero rows to whole steps of four, so
// no step needs a mask.
// PACKED false (streamed elements): K has been written, its interface block
// waits in Aii's memory and only the bubble rows are in LDS.
template <typename T, int NBT, int R, int NW, bool PACKED>
__device__ __forceinline__ void sf_condense(const ElemArgs &a, const CondArgs &cd, int e, const SfElem &es, double *pk,
                                            double *kb, const SfLay &ly, double *w, SfSmall<R> &sm, size_t ldc, int tid)
{
    typedef Mfma<double> MD;
    constexpr int WLD = 16 * NBT + 1;
    const int lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lr = lane & 15, lq = lane >> 4;
    const int n = __builtin_amdgcn_readfirstlane(es.n), nb = __builtin_amdgcn_readfirstlane(es.nb), ni = n - nb;
    const int ldb = n | 1, nk = (nb + 3) >> 2, nk0 = min(nk, 4);
    const bool cond = nb <= 16 * NBT, fac = cond && nb > 0;
    if (fac && wv == 0) {
        if (sf_factor<NBT>(kb, ldb, ni, nb, w, lane) && lane == 0) sm.fail = 1;
    }
    // the other waves (all, if there is nothing to factor): K, both triangles
    if (PACKED && a.kout && (wv > 0 || !fac))
        sf_unpack(pk, ly, (T *)a.kout + a.off_k[e], a.ld_k > 0 ? (size_t)a.ld_k : (size_t)n, n, fac ? wv - 1 : wv,
                  fac ? NW - 1 : NW, lane);
    if (!cond) {
        // more bubbles than the caller declared
        if (tid == 0 && a.status) a.status[e] = HP3D_E_ARG;
        return;
    }
    double *aii = cd.aii + cd.off_c[e];
    double *bi = cd.bi + a.off_v[e];
    if (nb == 0) {
        for (int c = tid; c < ni; c += 64 * NW) bi[c] = sm.b[c];
    } else {
        // zero rows up to the next multiple of four (columns 0..ni are read)
        for (int k = nb; k < 4 * nk; ++k) {
            for (int c = tid; c < ldb; c += 64 * NW) kb[k * ldb + c] = 0.0;
            if (tid == 0) sm.b[ni + k] = 0.0;
        }
        lds_barrier();
        double *xs = cd.aschur + cd.off_s[e];
        double *xb = cd.bschur + a.off_v[e];
        const double *const pf = w + lr * WLD + lq, *const pb = w + lq * WLD + lr;
        for (int t = wv; t < (ni + 16) / 16; t += NW) {
            const int c = 16 * t + lr;
            // Z(4 s + lq, c): the bubble rows, or the load in column ni
            const double *src = c == ni ? sm.b + ni + lq : kb + lq * ldb + min(c, ni);
            const int stp = c == ni ? 4 : 4 * ldb;
            d4_t f0 = {0.0, 0.0, 0.0, 0.0}, f1 = f0, x0 = f0, x1 = f0;
#pragma unroll 4
            for (int s = 0; s < nk0; ++s) {
                const double z = src[s * stp];
                f0 = MD::mma(pf[4 * s], z, f0);
                if (NBT > 1) f1 = MD::mma(pf[16 * WLD + 4 * s], z, f1);
            }
            if (NBT > 1)
#pragma unroll 4
                for (int s = 4; s < nk; ++s) f1 = MD::mma(pf[16 * WLD + 4 * s], src[s * stp], f1);
            // S over [Abi | Bb]; its rows are X's operands
            double *so = kb + lq * ldb + min(c, ni);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (c <= ni && j < nk) so[4 * j * ldb] = f0[j];
                if (NBT > 1 && c <= ni && j + 4 < nk) so[(4 * j + 16) * ldb] = f1[j];
            }
            wave_sync_lds();
#pragma unroll 4
            for (int s = 0; s < nk0; ++s) x0 = MD::mma(pb[4 * s * WLD], so[4 * s * ldb], x0);
            if (NBT > 1)
#pragma unroll 4
                for (int s = 4; s < nk; ++s) {
                    const double z = so[4 * s * ldb];
                    x0 = MD::mma(pb[4 * s * WLD], z, x0);
                    x1 = MD::mma(pb[4 * s * WLD + 16], z, x1);
                }
            double *xo = c < ni ? xs + (size_t)c * nb + lq : xb + lq;
            if (c <= ni)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    if (4 * j + lq < nb) xo[4 * j] = x0[j];
                    if (NBT > 1 && 4 * j + 16 + lq < nb) xo[4 * j + 16] = x1[j];
                }
        }
        if (!PACKED) __threadfence_block(); // the interface block comes back from memory
        __syncthreads();
        // lower tiles (tr, tc) of [Aii; Bi], tile t of the triangle by wave t
        // mod NW
        const int nti = (ni + 16) / 16;
        int tr = 0, tc = wv;
        while (tc > tr) {
            tc -= tr + 1;
            ++tr;
        }
        while (tr < nti) {
            const int c = 16 * tc + lr, r0 = 16 * tr + lq;
            // (r0 + 4 j)(r0 + 4 j + 1) / 2 + c; what lies beyond the triangle
            // is read but not used
            const int at = (__mul24(r0, r0 + 1) >> 1) + c;
            d4_t acc;
            if (PACKED) {
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[j] = pk[at + j * 4 * r0 + 8 * j * j + 2 * j];
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int r = r0 + 4 * j;
                    acc[j] = aii[r < ni && c <= r ? r + c * ldc : 0];
                }
            }
            const double *pa = kb + lq * ldb + 16 * tr + lr, *pc = kb + lq * ldb + c;
            d4_t up = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 8
            for (int s = 0; s < nk; ++s) up = MD::mma(pa[4 * s * ldb], pc[4 * s * ldb], up);
            if (16 * tr + 16 <= ni && tr > tc) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const double v = acc[j] - up[j];
                    if (PACKED) {
                        pk[at + j * 4 * r0 + 8 * j * j + 2 * j] = v;
                    } else {
                        aii[r0 + 4 * j + c * ldc] = v;
                        aii[c + (r0 + 4 * j) * ldc] = v;
                    }
                }
            } else {
                const double bc = sm.b[min(c, ni - 1)];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int r = r0 + 4 * j;
                    const double v = acc[j] - up[j];
                    if (r < ni && c <= r) {
                        if (PACKED) {
                            pk[at + j * 4 * r0 + 8 * j * j + 2 * j] = v;
                        } else {
                            aii[r + c * ldc] = v;
                            aii[c + r * ldc] = v;
                        }
                    }
                    if (r == ni && c < ni) bi[c] = bc - up[j];
                }
            }
            tc += NW;
            while (tc > tr) {
                tc -= tr + 1;
                ++tr;
            }
        }
        lds_barrier();
    }
    if (PACKED) sf_unpack(pk, ly, aii, ldc, ni, wv, NW, lane);
    if (tid == 0 && a.status) a.status[e] = sm.fail ? HP3D_E_FACTOR : (es.negjac ? HP3D_NEG_JACOBIAN : 0);
}

// arguments of the fused kernel, as one kernel argument at offset 0
struct SingleArgs {
    ElemArgs a;
    CondArgs cd;
};
typedef const __attribute__((address_space(4))) SingleArgs *kargs_t;

// Element matrix, load and condensation of elements with at most R dofs and
// 16 NBT bubbles in one launch, a workgroup per element (or, with a smaller
// grid, per element of a grid stride): K in LDS (SfLay), half of it computed.
// Against the kernel it replaces, which formed A A^T on MFMA tiles and
// condensed them from registers: 4,199 H1 p = 4 elements without K 0.986 ->
// 0.331 ms, 32,768 with K in FP32 5.2 -> 2.6 ms, 13,824 p = 3 in FP64 0.631 ->
// 0.378 ms, 10,051 H(curl) p = 2 0.578 -> 0.316 ms.  What bounds it is not the
// memory (p = 4 in FP64: 2.5 TB/s) but the length of an element's chain of
// short phases between barriers and the instructions in them (VALU half busy),
// so what counts is how many elements a CU holds: see the launch.
template <typename T, int SPACE, int R, int NBT, int NW, int POOL, int WPE>
__global__ __launch_bounds__(64 * NW, WPE) void sf_fused_kernel(SingleArgs sa)
{
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int WGS = 64 * NW;
    constexpr SfShape SH{SPACE, R, NBT, NW, POOL, WPE, 0};
    constexpr SfFused FU = sf_limits(SH);
    constexpr int H5 = FU.h5, H4 = FU.h4;
    constexpr bool HOLD = H5 > 0, STREAM = sf_streams(SH);
    __shared__ SfElem es;
    __shared__ SfTab tb;
    __shared__ SfSmall<R> sm;
    // L^-1 of the bubble block; before that the staged geometry nodes.  With one
    // tile row of bubbles they have their places in the pool, after (nodes: at
    // the end of) what it holds then.
    __shared__ double wbuf[NBT > 1 ? 16 * NBT * (16 * NBT + 1) : 1];
    static_assert(16 * (16 + 1) >= SF_XG, "staged nodes");
    __shared__ __align__(16) short row[sf_comps(SPACE) * SF_I * SF_I * 8];
    __shared__ unsigned short pl[sf_comps(SPACE) * SF_I * SF_I];
    __shared__ short js[sf_comps(SPACE) * 8];
    __shared__ __align__(16) double pool[POOL];
    const int nel = sa.a.nel;
    for (int e = blockIdx.x; e < nel; e += gridDim.x) {
        if (e != (int)blockIdx.x) __syncthreads(); // the previous element is done with LDS
        // the arguments are read again (scalar loads) and the thread index
        // passes through an empty asm for every element, so that nothing
        // derived from them is held in registers across the element's body
        kargs_t kp = (kargs_t)__builtin_amdgcn_kernarg_segment_ptr();
        __asm__ volatile("" : "+s"(kp));
        const ElemArgs a = kp->a;
        const CondArgs cd = kp->cd;
        int tid = threadIdx.x;
        __asm__ volatile("" : "+v"(tid));
        double *const xg = NBT > 1 ? wbuf : pool + POOL - SF_XG;
        unsigned short *const gmap = reinterpret_cast<unsigned short *>(xg + 3 * XS_MAX + 1);
        const bool ok = sf_setup<SPACE, WGS>(a, e, es, xg, tid, FU);
        if (!ok || es.n > a.max_ndof || es.n > R) { // invalid codes, or above the caller's bound
            if (tid == 0 && a.status) a.status[e] = ok ? HP3D_E_ARG : HP3D_E_ORDER;
            continue;
        }
        if (tid == 0) sm.fail = 0;
        sf_fill_tab<WGS>(es.m, tb, tid);
        sf_fill_rows<SPACE>(es, row, tid, WGS);
        if (a.ngeo != 8) sf_fill_gmap(es, a.ngeo, gmap, tid, WGS);
        lds_barrier();
        const int n = es.n, mode = STREAM ? es.mode : SF_DIRECT;
        const SfLay ly(n, es.nb, 16 * NBT);
        double *const d = pool + (mode == SF_DIRECT ? ly.len : 0);
        if (sf_points<SPACE>(es, tb, gmap, a, e, xg, d, tid, WGS)) es.negjac = 1;
        if (tid < 64) sf_pencils<SPACE>(es, row, pl, js, tid);
        lds_barrier();
        {
            double *const bl = sm.b, *const bo = a.bout ? a.bout + a.off_v[e] : nullptr;
            sf_load<SPACE, WGS>(es, tb, row, d + (SPACE == 0 ? 6 : 12) * es.nint,
                                [=](int r, double v) {
                                    bl[r] = v;
                                    if (bo) bo[r] = v;
                                },
                                tid);
        }
        const int dl = (SPACE == 0 ? 6 : 12) * es.nint; // T takes the load fields' place
        if (mode == SF_DIRECT) {
            const SfToPacked to{pool, ly};
            auto run = [&](auto mc) __attribute__((always_inline)) {
                sf_matrix<SPACE, decltype(mc)::value, true>(es, tb, row, pl, js, d, d + dl, POOL - ly.len - dl, to, 0, 1,
                                                            tid, WGS);
            };
            switch (es.m[2]) {
            case 2: run(std::integral_constant<int, 2>{}); break;
            case 3: run(std::integral_constant<int, 3>{}); break;
            case 4: run(std::integral_constant<int, 4>{}); break;
            case 5: run(std::integral_constant<int, 5>{}); break;
            case 6: run(std::integral_constant<int, 6>{}); break;
            default: run(std::integral_constant<int, 7>{}); break;
            }
        } else if (HOLD && mode == SF_HOLD) {
            if constexpr (HOLD) {
                if (es.m[2] == 5) sf_hold<5, H5>(es, tb, row, pl, pool, dl, ly, tid, WGS);
                else sf_hold<4, H4>(es, tb, row, pl, pool, dl, ly, tid, WGS);
                lds_barrier();
            }
        } else if constexpr (STREAM) {
            // the bubble rows at the pool's end, T in between
            const int kl = ly.len - ((ly.kb + 1) & ~1);
            double *const kb = pool + POOL - kl;
            const SfToSplit<T> to{a.kout ? (T *)a.kout + a.off_k[e] : nullptr, a.ld_k > 0 ? a.ld_k : n, kb,
                                  es.nb <= 16 * NBT ? cd.aii + cd.off_c[e] : nullptr, n - es.nb, ly.ldb};
            // (with the pools of the launches, elements whose longest
            // direction has fewer functions never come here)
            if (HOLD && sf_stream_mc(SH, es.m[2]) == 6)
                sf_matrix<SPACE, 6, false>(es, tb, row, pl, js, d, d + dl, POOL - kl - dl, to, 0, 1, tid, WGS);
            else
                sf_matrix<SPACE, 7, false>(es, tb, row, pl, js, d, d + dl, POOL - kl - dl, to, 0, 1, tid, WGS);
            sf_condense<T, NBT, R, NW, false>(a, cd, e, es, nullptr, kb, ly, NBT > 1 ? wbuf : pool, sm, n - es.nb, tid);
            continue;
        }
        sf_condense<T, NBT, R, NW, true>(a, cd, e, es, pool, pool + ly.kb, ly, NBT > 1 ? wbuf : pool + ly.len, sm,
                                           n - es.nb, tid);
    }
#endif
}

// ------------------------------------------------------- field evaluation
//
// One workgroup per element evaluates finite-element fields from element dof
// vectors at the quadrature points (soleval, element/util/soleval.F90, with
// the dofs in element order) and integrates one of:
//   HP3D_FIELD_ERROR    element_error (element/util/compute_error.F90:226-400):
//                       set_3Dint rule with INTEGRATION = 2; out[2e] = errorH
//                       (int |grad(u - u_h)|^2 + |u - u_h|^2) or errorE (curl
//                       and value), out[2e+1] = the same norm of the exact u
//   HP3D_FIELD_ADJOINT  out[e] = -coef_e int grad v_h . grad u_h (H1) or
//                       -coef_e int v_h . u_h (H(curl)): lambda_e^T (dK_e /
//                       dlog coef_e) u_e with a minus sign, i.e. dJ/dtheta_e
//                       for coef = exp(theta), recomputed at the points of the
//                       element rule without forming K_e
//   HP3D_FIELD_L2       out[e] = int u_h . u_h and r[off_v[e] + k] = int
//                       phi_k . u_h (the element mass matrix times u_e)
// The dofs are summed one direction after the other (C, B, then A at the
// point), value and reference derivatives at once, and r goes the same way
// back: O(m^4) work where a sum over all dofs at every point is O(m^6).  What
// is left is mostly the points themselves (map, exact solution).  On 13,824
// H1 p = 3 elements (216 points, ERROR) 0.490 -> 0.117 ms, on 4,080 p = 4
// elements ADJOINT and L2 0.263 -> 0.040 ms each.
struct FieldArgs {
    int space, mode, nel, ngeo, exact;
    const int *norder, *nori_e, *nori_f;
    const double *xnod, *coef;
    const long long *off_v;
    const double *u, *v;
    double *out, *r;
    int *status;
};

// exact solutions of the manufactured problems (value, gradient); the
// selector is the load selector of the same problem
__device__ inline void exact_h1(int sel, const double *x, double &u, double *du)
{
    const double pi = 3.14159265358979323846;
    u = du[0] = du[1] = du[2] = 0.0;
    if (sel == HP3D_LOAD_SINSINSIN) {
        double s[3], c[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) sincospi(x[i], &s[i], &c[i]);
        u = s[0] * s[1] * s[2];
        du[0] = pi * c[0] * s[1] * s[2];
        du[1] = pi * s[0] * c[1] * s[2];
        du[2] = pi * s[0] * s[1] * c[2];
    } else if (sel == HP3D_LOAD_CONV) {
        double sx, cx;
        sincospi(x[0], &sx, &cx);
        const double sh = sinh(pi * x[1]), z2 = x[2] * x[2];
        u = sx * sh * z2;
        du[0] = pi * cx * sh * z2;
        du[1] = pi * sx * cosh(pi * x[1]) * z2;
        du[2] = 2.0 * sx * sh * x[2];
    } else if (sel == HP3D_LOAD_POLY2) {
        double a0 = x[0] * (1.0 - x[0]), a1 = x[1] * (1.0 - x[1]), a2 = x[2] * (1.0 - x[2]);
        u = a0 * a1 * a2;
        du[0] = (1.0 - 2.0 * x[0]) * a1 * a2;
        du[1] = a0 * (1.0 - 2.0 * x[1]) * a2;
        du[2] = a0 * a1 * (1.0 - 2.0 * x[2]);
    } else if (sel == HP3D_LOAD_XYZ) {
        u = x[0] * x[1] * x[2];
        du[0] = x[1] * x[2];
        du[1] = x[0] * x[2];
        du[2] = x[0] * x[1];
    }
}

__device__ inline void exact_hcurl(int sel, const double *x, double *e, double *curl)
{
    const double pi = 3.14159265358979323846;
    for (int i = 0; i < 3; ++i) e[i] = curl[i] = 0.0;
    if (sel == HP3D_LOAD_CURL_SIN) {
        double sy, cy, sz, cz;
        sincospi(x[1], &sy, &cy);
        sincospi(x[2], &sz, &cz);
        e[0] = sy * sz;
        curl[1] = pi * sy * cz;
        curl[2] = -pi * cy * sz;
    }
}

// points per direction (by role) of the set_3Dint brick rule with INTEGRATION
// = 2 (set_3D_int.F90:8-21,203-244): face orders as coded (no swap), orders
// raised by 2 and capped at MAXP; direction d by the calling lane
__device__ __forceinline__ int sf_rule_plain(const SfElem &es, int d)
{
    int m = es.o.b[d];
    for (int i = 0; i < 4; ++i) m = max(m, es.o.pe[d == 2 ? 8 + i : 2 * i + d]);
    // faces 0..5 have axes (0,1), (0,1), (0,2), (1,2), (0,2), (1,2)
    const int h = d == 0 ? 0x17 : d == 1 ? 0x28 : 0, v = d == 1 ? 0x03 : d == 2 ? 0x3c : 0;
    for (int f = 0; f < 6; ++f) {
        if (h >> f & 1) m = max(m, es.o.fh[f]);
        if (v >> f & 1) m = max(m, es.o.fv[f]);
    }
    return min(m + 2, MAXP) + 1;
}

// u_h's dofs summed over C, then B: y[3 (comp (mA nB nC) + (iA nB + qB) nC + qC) ..]
// = the value chain, the one with the derivative in B, the one in C; c may be y
template <int SPACE, int WGS>
__device__ __forceinline__ void sf_field_sums(const SfElem &es, const SfTab &tb, const int (&nq)[3], const short *row,
                                              const double *u, double *c, double *x, double *y, int tid)
{
    constexpr int NC = sf_comps(SPACE), DER = SF_I * 8;
    const int mA = es.m[1], mB = es.m[0], mC = es.m[2], nB = nq[0], nC = nq[2];
    for (int k = tid; k < NC * mA * mB * mC; k += WGS) {
        const int k1 = k / mC, iC = k - k1 * mC, k2 = k1 / mB, iB = k1 - k2 * mB, a = k2 / mA, iA = k2 - a * mA;
        const int r = row[((a * SF_I + iA) * SF_I + iB) * 8 + iC];
        const double v = r < 0 ? 0.0 : u[r & ~ROW_NEG];
        c[k] = r & ROW_NEG ? -v : v;
    }
    lds_barrier();
    for (int k = tid; k < NC * mA * mB * nC; k += WGS) {
        const int k1 = k / nC, qC = k - k1 * nC, a = SPACE == 0 ? -1 : k1 / (mA * mB);
        const double *f = tb.f[2][0] + qC, *ck = c + k1 * mC;
        const int v = a == 2 ? DER : 0;
        double s0 = 0.0, s1 = 0.0;
        for (int i = 0; i < mC; ++i) {
            s0 = fma(f[v + 8 * i], ck[i], s0);
            s1 = fma(f[DER + 8 * i], ck[i], s1);
        }
        x[2 * k] = s0;
        x[2 * k + 1] = s1;
    }
    lds_barrier();
    for (int k = tid; k < NC * mA * nB * nC; k += WGS) {
        const int k1 = k / nC, qC = k - k1 * nC, k2 = k1 / nB, qB = k1 - k2 * nB, a = SPACE == 0 ? -1 : k2 / mA;
        const double *f = tb.f[0][0] + qB, *xk = x + 2 * (k2 * mB * nC + qC);
        const int v = a == 0 ? DER : 0;
        double s0 = 0.0, s1 = 0.0, s2 = 0.0;
        for (int i = 0; i < mB; ++i) {
            const double x0 = xk[2 * i * nC], x1 = xk[2 * i * nC + 1];
            s0 = fma(f[v + 8 * i], x0, s0);
            s1 = fma(f[DER + 8 * i], x0, s1);
            s2 = fma(f[v + 8 * i], x1, s2);
        }
        y[3 * k] = s0;
        y[3 * k + 1] = s1;
        y[3 * k + 2] = s2;
    }
    lds_barrier();
}

// the field in reference form at point (qA, qB, qC): value and gradient (H1)
// or E and curl E (H(curl))
template <int SPACE>
__device__ __forceinline__ void sf_field_at(const SfElem &es, const SfTab &tb, const int (&nq)[3], const double *y, int qA,
                                            int qB, int qC, double (&f)[3], double (&g)[3])
{
    constexpr int DER = SF_I * 8;
    const int mA = es.m[1], nB = nq[0], nC = nq[2];
#pragma unroll
    for (int j = 0; j < 3; ++j) f[j] = g[j] = 0.0;
#pragma unroll
    for (int a = 0; a < sf_comps(SPACE); ++a) { // (the roles B, A, C are x, y, z)
        const double *t = tb.f[1][0] + qA, *ya = y + 3 * ((a * mA * nB + qB) * nC + qC);
        const int v = SPACE == 1 && a == 1 ? DER : 0;
        double s = 0.0, dx = 0.0, dy = 0.0, dz = 0.0;
        for (int i = 0; i < mA; ++i, ya += 3 * nB * nC) {
            const double y0 = ya[0], fa = t[v + 8 * i];
            s = fma(fa, y0, s);
            dy = fma(t[DER + 8 * i], y0, dy);
            dx = fma(fa, ya[1], dx);
            dz = fma(fa, ya[2], dz);
        }
        if (SPACE == 0) {
            f[0] = s;
            g[0] = dx;
            g[1] = dy;
            g[2] = dz;
        } else { // curl (s e_a) = grad s x e_a
            f[a] = s;
            if (a == 0) {
                g[1] += dz;
                g[2] -= dy;
            } else if (a == 1) {
                g[0] -= dz;
                g[2] += dx;
            } else {
                g[0] += dy;
                g[1] -= dx;
            }
        }
    }
}

// covariant transform: gradients of H1, values of H(curl)
__device__ __forceinline__ void sf_covariant(const double (&inv)[3][3], const double (&g)[3], double (&out)[3])
{
#pragma unroll
    for (int j = 0; j < 3; ++j) out[j] = g[0] * inv[0][j] + g[1] * inv[1][j] + g[2] * inv[2][j];
}

// PAIR: ADJOINT (two fields); otherwise ERROR or L2
template <int SPACE, bool PAIR>
__global__ __launch_bounds__(128, SPACE == 0 ? 3 : 2) void field_kernel(FieldArgs fa)
{
    constexpr int WGS = 128, NU = (MAXQ + WGS - 1) / WGS, NC = sf_comps(SPACE);
    __shared__ SfElem es;
    __shared__ SfTab tb;
    __shared__ __align__(16) short row[NC * SF_I * SF_I * 8];
    __shared__ double xg[SF_XG];
    __shared__ double x[2 * NC * MAXQ], y[3 * NC * MAXQ];
    __shared__ double red[2][WGS / 64];
    __shared__ int rule[3];
    unsigned short *const gmap = reinterpret_cast<unsigned short *>(xg + 3 * XS_MAX + 1);
    const int e = blockIdx.x, tid = threadIdx.x;
    ElemArgs a;
    a.ngeo = fa.ngeo;
    a.norder = fa.norder;
    a.nori_e = fa.nori_e;
    a.nori_f = fa.nori_f;
    a.xnod = fa.xnod;
    a.coef = fa.coef;
    if (!sf_setup<SPACE, WGS>(a, e, es, xg, tid)) {
        if (tid == 0 && fa.status) fa.status[e] = HP3D_E_ORDER;
        return;
    }
    const bool err = !PAIR && fa.mode == HP3D_FIELD_ERROR;
    if (tid < 3) rule[tid] = err ? sf_rule_plain(es, tid) : es.m[tid];
    sf_fill_rows<SPACE>(es, row, tid, WGS);
    if (fa.ngeo != 8) sf_fill_gmap(es, fa.ngeo, gmap, tid, WGS);
    lds_barrier();
    const int nq[3] = {rule[0], rule[1], rule[2]}, Q = nq[0] * nq[1] * nq[2];
    sf_fill_tab<WGS>(nq, tb, tid);
    lds_barrier();
    // of the pair, v's part (reference gradient or value) waits in registers
    double hv[PAIR ? NU : 1][3];
    if constexpr (PAIR) {
        sf_field_sums<SPACE, WGS>(es, tb, nq, row, fa.v + fa.off_v[e], y, x, y, tid);
#pragma unroll
        for (int i = 0; i < NU; ++i) {
            const int l = min(tid + i * WGS, Q - 1), l1 = l / nq[2], qC = l - l1 * nq[2], qA = l1 / nq[0];
            double f[3], g[3];
            sf_field_at<SPACE>(es, tb, nq, y, qA, l1 - qA * nq[0], qC, f, g);
#pragma unroll
            for (int j = 0; j < 3; ++j) hv[i][j] = SPACE == 0 ? g[j] : f[j];
        }
        lds_barrier();
    }
    sf_field_sums<SPACE, WGS>(es, tb, nq, row, fa.u + fa.off_v[e], y, x, y, tid);

    const bool staged = fa.ngeo <= XS_MAX;
    const double coef = xg[3 * XS_MAX];
    double acc0 = 0.0, acc1 = 0.0;
    bool neg = false;
    double *const pw = x; // weighted field of L2
    auto point = [&](int l, const double (&h)[3]) __attribute__((always_inline)) {
        const int l1 = l / nq[2], qC = l - l1 * nq[2], qA = l1 / nq[0], qB = l1 - qA * nq[0];
        double f[3], g[3], xp[3], jm[3][3], inv[3][3], t[3];
        sf_field_at<SPACE>(es, tb, nq, y, qA, qB, qC, f, g);
        const double det = staged ? sf_map<true>(es, tb, gmap, xg, fa.ngeo, qB, qA, qC, xp, jm, inv)
                                  : sf_map<false>(es, tb, gmap, fa.xnod + 3 * (size_t)fa.ngeo * e, fa.ngeo, qB, qA, qC,
                                                  xp, jm, inv);
        neg = neg || det < 0.0;
        const double wd = det * (tb.w[0][qB] * tb.w[1][qA] * tb.w[2][qC]);
        sf_covariant(inv, SPACE == 0 ? g : f, t);
        if constexpr (PAIR) {
            double tv[3];
            sf_covariant(inv, h, tv);
            acc0 -= coef * (t[0] * tv[0] + t[1] * tv[1] + t[2] * tv[2]) * wd;
        } else if (err) {
            double fe[3], ge[3], fu[3], gu[3];
            if (SPACE == 0) {
                exact_h1(fa.exact, xp, fe[0], ge);
                fe[1] = fe[2] = fu[1] = fu[2] = 0.0;
                fu[0] = f[0];
            } else {
                exact_hcurl(fa.exact, xp, fe, ge);
            }
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                if (SPACE == 0) {
                    gu[j] = t[j];
                } else {
                    fu[j] = t[j];
                    gu[j] = (jm[j][0] * g[0] + jm[j][1] * g[1] + jm[j][2] * g[2]) / det;
                }
                acc0 += ((ge[j] - gu[j]) * (ge[j] - gu[j]) + (fe[j] - fu[j]) * (fe[j] - fu[j])) * wd;
                acc1 += (ge[j] * ge[j] + fe[j] * fe[j]) * wd;
            }
        } else {
            // weighted field pulled back to reference components: phi_k . u_h w det
            if (SPACE == 0) {
                acc0 += f[0] * f[0] * wd;
                pw[l] = f[0] * wd;
            } else {
                acc0 += (t[0] * t[0] + t[1] * t[1] + t[2] * t[2]) * wd;
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    pw[i * Q + l] = (inv[i][0] * t[0] + inv[i][1] * t[1] + inv[i][2] * t[2]) * wd;
            }
        }
    };
    if constexpr (PAIR) {
#pragma unroll
        for (int i = 0; i < NU; ++i)
            if (tid + i * WGS < Q) point(tid + i * WGS, hv[i]);
    } else {
        for (int l = tid; l < Q; l += WGS) point(l, hv[0]);
    }
    if (neg) es.negjac = 1;
    // workgroup sums
    for (int off = 32; off > 0; off >>= 1) {
        acc0 += __shfl_down(acc0, off);
        acc1 += __shfl_down(acc1, off);
    }
    if ((tid & 63) == 0) {
        red[0][tid >> 6] = acc0;
        red[1][tid >> 6] = acc1;
    }
    lds_barrier();
    if (tid == 0) {
        if (err) {
            fa.out[2 * (size_t)e] = red[0][0] + red[0][1];
            fa.out[2 * (size_t)e + 1] = red[1][0] + red[1][1];
        } else {
            fa.out[e] = red[0][0] + red[0][1];
        }
        if (fa.status) fa.status[e] = es.negjac ? HP3D_NEG_JACOBIAN : 0;
    }
    if (!PAIR && fa.mode == HP3D_FIELD_L2 && fa.r) {
        double *re = fa.r + fa.off_v[e];
        sf_load<SPACE, WGS>(es, tb, row, pw, [=](int k, double v) { re[k] = v; }, tid);
    }
}
