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

constexpr int SF_I = MAXP + 1;                   // 1D functions per direction
__host__ __device__ constexpr int sf_comps(int space) { return space == 0 ? 1 : 3; }
// fields per point: metric (6 symmetric entries; H(curl) curl, then mass) and load
__host__ __device__ constexpr int sf_fields(int space) { return space == 0 ? 7 : 15; }
__host__ __device__ constexpr int sf_ttabs(int space) { return space == 0 ? 8 : 9; }
__host__ __device__ constexpr int sf_sym(int r, int s) { return r <= s ? r * (5 - r) / 2 + s : s * (5 - s) / 2 + r; }

struct SfElem {
    ElemOrders o;
    DofBases bs, bh; // of the space, and of H1 (geometry nodes)
    int n, nb, nh, m[3], nint, ok, negjac, np, npad[2];
};

// Orders, counts and dof bases of one element, decoded by the lanes of wave 0
// (lane l: header integer l; counts by a lane scan, quadrature sizes by an
// or-reduction of order bits), ending in an LDS barrier.  Returns false
// (uniformly) for an invalid element.
template <int SPACE>
__device__ __forceinline__ bool sf_setup(const ElemArgs &a, int e, SfElem &es, int tid)
{
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
        // inclusive scan of the entity counts over lanes 0..18, both counts at once
        int sc = cnt + (cnt_h << 16);
        for (int d = 1; d < 32; d <<= 1) {
            const int up = __shfl_up(sc, d);
            if (tid >= d) sc += up;
        }
        for (int d = 1; d < 32; d <<= 1) bits |= __shfl_xor(bits, d);
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
            int nint = 1;
            for (int d = 0; d < 3; ++d) {
                const int top = 31 - __clz((int)((bits >> (8 * d)) & 0x7eu));
                es.m[d] = top + 1;
                nint *= top + 1;
            }
            es.nint = nint;
            es.negjac = 0;
            es.ok = all_ok && a.ngeo <= es.nh ? 1 : 0;
        }
    }
    lds_barrier();
    return es.ok != 0;
}

// 1D tables of the three directions in LDS
struct SfTab {
    double f[3][2][SF_I * 8];
    double w[3][8];
};
__device__ __forceinline__ void sf_fill_tab(const SfElem &es, SfTab &t, int tid, int wgs)
{
    for (int k = tid; k < 3 * 2 * SF_I * 8; k += wgs) {
        const int d = k / (2 * SF_I * 8), r = k % (2 * SF_I * 8);
        (&t.f[0][0][0])[k] = (&c_sf.f[es.m[d]][0][0][0])[r];
    }
    if (tid < 24) t.w[tid >> 3][tid & 7] = c_sf.w[es.m[tid >> 3]][tid & 7];
}

// dof rows by 1D indexes: row[((comp * 7 + iA) * 7 + iB) * 8 + iC]
template <int SPACE>
__device__ __forceinline__ void sf_fill_rows(const SfElem &es, short *row, int tid, int wgs)
{
    const int mA = es.m[1], mB = es.m[0], mC = es.m[2];
    for (int k = tid; k < sf_comps(SPACE) * SF_I * SF_I * 8; k += wgs) {
        const int iC = k & 7, pen = k >> 3, iB = pen % SF_I, iA = (pen / SF_I) % SF_I, c = pen / (SF_I * SF_I);
        int r = -1;
        if (iA < mA && iB < mB && iC < mC) r = dof_row(SPACE, c, iB, iA, iC, es.o, es.bs);
        row[k] = (short)r;
    }
}

// geometry node -> H1 1D indexes and sign, for maps beyond the trilinear one
__device__ __forceinline__ void sf_fill_gmap(const SfElem &es, int ngeo, unsigned short *gmap, int tid, int wgs)
{
    for (int k = tid; k < SF_I * SF_I * SF_I; k += wgs) {
        const int i0 = k % SF_I, i1 = (k / SF_I) % SF_I, i2 = k / (SF_I * SF_I);
        if (i0 >= es.m[0] || i1 >= es.m[1] || i2 >= es.m[2]) continue;
        const int r = dof_row(0, 0, i0, i1, i2, es.o, es.bh);
        if (r >= 0 && (r & ~ROW_NEG) < ngeo)
            gmap[r & ~ROW_NEG] = (unsigned short)(i0 | (i1 << 3) | (i2 << 6) | (r & ROW_NEG ? 512 : 0));
    }
}

// Metric fields and load of every quadrature point, q = (qA mB + qB) mC + qC,
// field f at d[f * nint + q]: the map, its Jacobian and inverse as in
// point_map, with the weights folded in (geom3D.F90:77-91, geom.F90:57-113,
// elem_opt.F90:101-122).  Returns true when a point of this thread has det < 0.
template <int SPACE>
__device__ __forceinline__ bool sf_points(const SfElem &es, const SfTab &tb, const unsigned short *gmap,
                                          const double *xn, int ngeo, double coef, int load, double *d, int tid,
                                          int wgs)
{
    const int Q = es.nint, mB = es.m[0], mC = es.m[2];
    bool neg = false;
    for (int l = tid; l < Q; l += wgs) {
        const int r0 = div_small(l, mC), qC = l - r0 * mC, qA = div_small(r0, mB), qB = r0 - qA * mB;
        double x[3] = {0.0, 0.0, 0.0}, jm[3][3] = {{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};
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
        if (ngeo == 8) {
            double v[3][2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                v[0][i] = tb.f[0][0][8 * i + qB];
                v[1][i] = tb.f[1][0][8 * i + qA];
                v[2][i] = tb.f[2][0][8 * i + qC];
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const int i0 = vtx_mu(k, 0), i1 = vtx_mu(k, 1), i2 = vtx_mu(k, 2);
                node(xn + 3 * k, v[0][i0], v[1][i1], v[2][i2], i0 ? 1.0 : -1.0, i1 ? 1.0 : -1.0, i2 ? 1.0 : -1.0);
            }
        } else {
            for (int k = 0; k < ngeo; ++k) {
                const int g = gmap[k], i0 = 8 * (g & 7) + qB, i1 = 8 * ((g >> 3) & 7) + qA, i2 = 8 * ((g >> 6) & 7) + qC;
                const double sg = g & 512 ? -1.0 : 1.0;
                node(xn + 3 * k, sg * tb.f[0][0][i0], tb.f[1][0][i1], tb.f[2][0][i2], sg * tb.f[0][1][i0],
                     tb.f[1][1][i1], tb.f[2][1][i2]);
            }
        }
        const double c00 = jm[1][1] * jm[2][2] - jm[2][1] * jm[1][2], c01 = jm[2][1] * jm[0][2] - jm[0][1] * jm[2][2],
                     c02 = jm[0][1] * jm[1][2] - jm[1][1] * jm[0][2];
        const double det = jm[0][0] * c00 + jm[1][0] * c01 + jm[2][0] * c02;
        neg = neg || det < 0.0;
        const double rdet = 1.0 / det;
        double inv[3][3];
        inv[0][0] = c00 * rdet;
        inv[0][1] = c01 * rdet;
        inv[0][2] = c02 * rdet;
        inv[1][0] = (jm[2][0] * jm[1][2] - jm[1][0] * jm[2][2]) * rdet;
        inv[1][1] = (jm[0][0] * jm[2][2] - jm[2][0] * jm[0][2]) * rdet;
        inv[1][2] = (jm[1][0] * jm[0][2] - jm[0][0] * jm[1][2]) * rdet;
        inv[2][0] = (jm[1][0] * jm[2][1] - jm[2][0] * jm[1][1]) * rdet;
        inv[2][1] = (jm[2][0] * jm[0][1] - jm[0][0] * jm[2][1]) * rdet;
        inv[2][2] = (jm[0][0] * jm[1][1] - jm[1][0] * jm[0][1]) * rdet;
        const double wd = det * (tb.w[0][qB] * tb.w[1][qA] * tb.w[2][qC]);
        // the square roots of the weights are taken and squared again so that
        // a negative weight gives NaN, as the reference's A_TEST factors do
        const double sm = sqrt(coef * wd);
        double f[3];
        getf(load, x, f);
        if (SPACE == 0) {
            d[6 * Q + l] = f[0] * wd;
        } else {
#pragma unroll
            for (int c = 0; c < 3; ++c)
                d[(12 + c) * Q + l] = (inv[c][0] * f[0] + inv[c][1] * f[1] + inv[c][2] * f[2]) * wd;
        }
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
            for (int c = 0; c < 3; ++c) inv[r][c] *= sm;
        constexpr int M0 = SPACE == 0 ? 0 : 6; // first mass / gradient field
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
            for (int s = r; s < 3; ++s)
                d[(M0 + sf_sym(r, s)) * Q + l] = inv[r][0] * inv[s][0] + inv[r][1] * inv[s][1] + inv[r][2] * inv[s][2];
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
                    d[sf_sym(r, s) * Q + l] = jm[0][r] * jm[0][s] + jm[1][r] * jm[1][s] + jm[2][r] * jm[2][s];
        }
    }
    return neg;
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
        if (k < NP) {
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

// load vector: entry of the dof with 1D indexes (comp; iA, iB, iC), the
// point's load fields against the product of its functions
template <int SPACE>
__device__ __forceinline__ double sf_load_entry(const SfElem &es, const SfTab &tb, const double *d, int c, int iA,
                                                int iB, int iC)
{
    const int mA = es.m[1], mB = es.m[0], mC = es.m[2];
    const double *g = d + (SPACE == 0 ? 6 : 12 + c) * es.nint;
    const double *fB = tb.f[0][SPACE == 1 && c == 0] + 8 * iB, *fA = tb.f[1][SPACE == 1 && c == 1] + 8 * iA,
                 *fC = tb.f[2][SPACE == 1 && c == 2] + 8 * iC;
    double s = 0.0;
    for (int qA = 0; qA < mA; ++qA)
        for (int qB = 0; qB < mB; ++qB) {
            const double *gq = g + (qA * mB + qB) * mC;
            double t = 0.0;
            for (int qC = 0; qC < mC; ++qC) t += fC[qC] * gq[qC];
            s += fA[qA] * fB[qB] * t;
        }
    return s;
}

// T tables of the columns jA in [j0, j0 + nj) against the rows iA in
// [i0, i0 + ni): t[tab * ts + ((jl * ni + il) * mB + qB) * MCP + qC], in
// H(curl) for columns of component b
template <int SPACE, int MC>
__device__ __forceinline__ void sf_build_t(const SfElem &es, const SfTab &tb, const double *d, double *t, int ts, int j0,
                                           int nj, int i0, int ni, int b, int tid, int wgs)
{
    constexpr int MCP = (MC + 1) & ~1;
    const int mA = es.m[1], mB = es.m[0], Q = es.nint;
    const double *f0 = tb.f[1][0], *f1 = tb.f[1][1];
    for (int k = tid; k < nj * ni * mB * MC; k += wgs) {
        const int k1 = k / MC, qC = k - k1 * MC, k2 = div_small(k1, mB), qB = k1 - k2 * mB;
        const int jl = div_small(k2, ni), il = k2 - jl * ni;
        const int iA = i0 + il, jA = j0 + jl;
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
        double *o = t + (size_t)(k1 * MCP + qC);
#pragma unroll
        for (int s = 0; s < sf_ttabs(SPACE); ++s) o[s * ts] = v[s];
    }
}

// s[q] += p * t[q], q < MC (t 16-byte aligned, padded to an even length)
template <int MC>
__device__ __forceinline__ void sf_axpy(double (&s)[MC], double p, const double *t)
{
    typedef double d2_t __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int q = 0; q < MC; q += 2) {
        const d2_t v = *reinterpret_cast<const d2_t *>(t + q);
        s[q] = fma(p, v[0], s[q]);
        if (q + 1 < MC) s[q + 1] = fma(p, v[1], s[q + 1]);
    }
}

// The block of pencil pair (first, second) from its S vectors, emitted entry
// by entry as em(iF, iG, value).  S_xy: derivative in C on the first (x) and
// second (y) function.  KIND 0: all four, 1: S01 and S11 (the second is a
// z-component dof), 2: S11 alone (both are).
template <int MC, int KIND, typename EM>
__device__ __forceinline__ void sf_block(const double (&s00)[MC], const double (&s01)[MC], const double (&s10)[MC],
                                         const double (&s11)[MC], EM em)
{
    typedef const __attribute__((address_space(4))) double *kd_t;
#pragma unroll
    for (int j = KIND == 0 ? 0 : 1; j < MC; ++j) {
        // the 1D tables come in through the scalar cache, again for every j:
        // held for all j they would not fit the scalar registers
        kd_t f0 = (kd_t)(uintptr_t)&c_sf.f[MC][0][0][0];
#if defined(__HIP_DEVICE_COMPILE__)
        __asm__ volatile("" : "+s"(f0));
#endif
        const kd_t f1 = f0 + SF_I * 8;
        double v0[MC], v1[MC];
#pragma unroll
        for (int q = 0; q < MC; ++q) {
            const double g0 = f0[8 * j + q], g1 = f1[8 * j + q];
            v0[q] = KIND == 0 ? fma(g0, s00[q], g1 * s01[q]) : KIND == 1 ? g1 * s01[q] : 0.0;
            v1[q] = KIND == 0 ? fma(g0, s10[q], g1 * s11[q]) : g1 * s11[q];
        }
#pragma unroll
        for (int i = KIND == 2 ? 1 : 0; i < MC; ++i) {
            double r = 0.0;
#pragma unroll
            for (int q = 0; q < MC; ++q) {
                if (KIND < 2) r = fma(f0[8 * i + q], v0[q], r);
                r = fma(f1[8 * i + q], v1[q], r);
            }
            em(i, j, r);
        }
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
__device__ __forceinline__ void sf_item_h1(const SfItem &it, const SfTab &tb, int mB, int ts, EM em)
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
        const double vv = vF * vG, vd = vF * dG, dv = dF * vG, dd = dF * dG;
        sf_axpy<MC>(s00, vv, t);
        sf_axpy<MC>(s00, vd, t + oF * ts);
        sf_axpy<MC>(s00, dv, t + oG * ts);
        sf_axpy<MC>(s00, dd, t + 3 * ts);
        sf_axpy<MC>(s01, vv, t + (3 + oF) * ts);
        sf_axpy<MC>(s10, vv, t + (3 + oG) * ts);
        sf_axpy<MC>(s01, dv, t + 6 * ts);
        sf_axpy<MC>(s10, vd, t + 6 * ts);
        sf_axpy<MC>(s11, vv, t + 7 * ts);
    }
    sf_block<MC, 0>(s00, s01, s10, s11, em);
}

// H(curl), by the components of the pair: KIND 0 neither is z, 1 the second
// is, 2 both are.  The sign of curl row r of a component-a dof is + for
// r = a + 1 and - for r = a + 2 (mod 3); the derivative of curl row r in B = x
// is absent for r = 0, that of the mass term present for a = 0.
template <int MC, int KIND, typename EM>
__device__ __forceinline__ void sf_item_hcurl(const SfItem &it, const SfTab &tb, int mB, int ts, EM em)
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
            sf_axpy<MC>(s00, mF * mG, t + m);
            sf_axpy<MC>(s00, dF * edG, t + zz);
            sf_axpy<MC>(s01, -dF * emG, t + zo);
            sf_axpy<MC>(s10, -mF * edG, t + oz);
            sf_axpy<MC>(s11, mF * emG, t + oo);
        }
    } else if constexpr (KIND == 1) {
        // first: rows z and o; second (component z): rows 0 and 1
        const int m = aI * ts, z0 = (sw ? 4 : 7) * ts, z1 = (sw ? 6 : 8) * ts;
        const int oI = 3 + 2 * (1 - it.aF), o0 = (sw ? 3 : oI) * ts, o1 = (sw ? 5 : oI + 1) * ts;
        const double sg = it.aF == 0 ? -1.0 : 1.0;
        for (int qB = 0; qB < mB; ++qB, t += MCP) {
            const double vF = fF[qB], dF = fF[DER + qB], vG = fG[qB], dG = fG[DER + qB];
            const double mF = it.aF == 0 ? dF : vF, sd = sg * dF, sm = sg * mF;
            sf_axpy<MC>(s01, mF * vG, t + m);
            sf_axpy<MC>(s01, sd * vG, t + z0);
            sf_axpy<MC>(s01, -sd * dG, t + z1);
            sf_axpy<MC>(s11, -sm * vG, t + o0);
            sf_axpy<MC>(s11, sm * dG, t + o1);
        }
    } else {
        const int r01 = (sw ? 5 : 4) * ts, r10 = (sw ? 4 : 5) * ts;
        for (int qB = 0; qB < mB; ++qB, t += MCP) {
            const double vF = fF[qB], dF = fF[DER + qB], vG = fG[qB], dG = fG[DER + qB];
            const double vv = vF * vG;
            sf_axpy<MC>(s11, vv, t + 2 * ts);
            sf_axpy<MC>(s11, vv, t + 3 * ts);
            sf_axpy<MC>(s11, -vF * dG, t + r01);
            sf_axpy<MC>(s11, -dF * vG, t + r10);
            sf_axpy<MC>(s11, dF * dG, t + 6 * ts);
        }
    }
    sf_block<MC, KIND>(s00, s01, s10, s11, em);
}

// Stores of K: the entry of the pair and, on the diagonal pair's upper half,
// its mirror.  Lanes of a wave hold consecutive row pencils of one column
// pencil, so a store instruction writes pieces of one column.
template <typename T, int MC>
__device__ __forceinline__ auto sf_store_k(T *k, long long ld, const int4 rI4, const int4 rJ4, bool swap, bool diag)
{
    // the eight packed rows of either pencil; first = column pencil if swapped
    const int4 rF4 = swap ? rJ4 : rI4, rG4 = swap ? rI4 : rJ4;
    const long long aF = swap ? ld : 1, aG = swap ? 1 : ld;
    auto get = [](const int4 &r, int i) {
        const int w = i < 2 ? r.x : i < 4 ? r.y : i < 6 ? r.z : r.w;
        return (int)(short)(i & 1 ? w >> 16 : w);
    };
    return [=](int i, int j, double v) {
        const int eF = get(rF4, i), eG = get(rG4, j);
        if (eF < 0 || eG < 0 || (diag && i > j)) return;
        const int r = eF & ~ROW_NEG, c = eG & ~ROW_NEG;
        const double s = (eF ^ eG) & ROW_NEG ? -v : v;
        k[r * aF + c * aG] = (T)s;
        if (diag && i < j) k[r * ld + c] = (T)s;
    };
}

// All column pencils of this workgroup's chunks: T, then one pencil pair per
// thread and step.  `part` of `nparts` workgroups of the element.
template <typename T, int SPACE, int MC, int POOL>
__device__ __forceinline__ void sf_matrix(const SfElem &es, const SfTab &tb, const short *row,
                                          const unsigned short *pl, const short *js, double *pool, T *kout, long long ld,
                                          int part, int nparts, int tid, int wgs)
{
    constexpr int MCP = (MC + 1) & ~1, NT = sf_ttabs(SPACE);
    const int mA = es.m[1], mB = es.m[0];
    const int dlen = (sf_fields(SPACE) * es.nint + 1) & ~1;
    const double *d = pool;
    double *t = pool + dlen;
    // as many columns jA at a time as the pool holds; if it does not hold one
    // against all rows, the rows in pieces (H1 elements whose 1D orders exceed
    // what their dof count suggests)
    const int one = NT * mB * MCP, room = (POOL - dlen) / one;
    int nj = room / mA, ni = mA;
    if (nj < 1) {
        nj = 1;
        ni = room;
    }
    if (nj > mA) nj = mA;
    if (nparts > 1) nj = 1;
    const int nch = (mA + nj - 1) / nj;
    for (int ch = part; ch < sf_comps(SPACE) * nch; ch += nparts) {
        const int b = ch / nch, j0 = (ch - b * nch) * nj, njc = min(nj, mA - j0);
        const int pj0 = js[b * 8 + j0], pj1 = js[b * 8 + (j0 + njc < SF_I ? j0 + njc : SF_I)], npj = pj1 - pj0;
        if (npj == 0) continue;
        for (int i0 = 0; i0 < mA; i0 += ni) {
            const int nic = min(ni, mA - i0), ts = njc * nic * mB * MCP;
            sf_build_t<SPACE, MC>(es, tb, d, t, ts, j0, njc, i0, nic, b, tid, wgs);
            lds_barrier();
            // rows: H1 all pencils with iA in the piece; H(curl) components x
            // and y, then z from the next whole wave on
            for (int grp = 0; grp < (SPACE == 0 ? 1 : 2); ++grp) {
                int pi0, pi1;
                if (SPACE == 0) {
                    pi0 = js[i0];
                    pi1 = js[i0 + nic < SF_I ? i0 + nic : SF_I];
                } else {
                    pi0 = grp == 0 ? 0 : js[2 * 8];
                    pi1 = grp == 0 ? js[2 * 8] : es.np;
                }
                const int npi = pi1 - pi0, nit = npi * npj;
                const float rn = 1.0f / (float)max(npi, 1);
                for (int k = tid; k < nit; k += wgs) {
                    const int jx = (int)(((float)k + 0.5f) * rn), I = pi0 + k - jx * npi, J = pj0 + jx;
                    const int pI = pl[I], pJ = pl[J];
                    const int iAI = (pI >> 3) & 7, iBI = pI & 7, iAJ = (pJ >> 3) & 7, iBJ = pJ & 7;
                    SfItem it;
                    it.swap = I > J;
                    it.iBF = it.swap ? iBJ : iBI;
                    it.iBG = it.swap ? iBI : iBJ;
                    it.aF = it.swap ? pJ >> 6 : pI >> 6;
                    it.aG = it.swap ? pI >> 6 : pJ >> 6;
                    it.t = t + ((iAJ - j0) * nic + iAI - i0) * mB * MCP;
                    const int4 rI = *reinterpret_cast<const int4 *>(row + 8 * (((pI >> 6) * SF_I + iAI) * SF_I + iBI));
                    const int4 rJ = *reinterpret_cast<const int4 *>(row + 8 * (((pJ >> 6) * SF_I + iAJ) * SF_I + iBJ));
                    auto em = sf_store_k<T, MC>(kout, ld, rI, rJ, it.swap, I == J);
                    if constexpr (SPACE == 0) {
                        sf_item_h1<MC>(it, tb, mB, ts, em);
                    } else {
                        if (grp == 0 && b < 2) sf_item_hcurl<MC, 0>(it, tb, mB, ts, em);
                        else if (grp == 1 && b == 2) sf_item_hcurl<MC, 2>(it, tb, mB, ts, em);
                        else sf_item_hcurl<MC, 1>(it, tb, mB, ts, em);
                    }
                }
            }
            lds_barrier();
        }
    }
}

// Element matrices and loads: one workgroup per (element, part); the parts of
// an element share its column chunks, so that a few elements fill the chip.
// Bound by writing K (9.6 GB for 4,096 H(curl) p = 5 elements in FP64, at the
// rate of a large copy 2 ms): the element + condensation step of that mesh
// took 54.3 ms with the A A^T product on MFMA tiles (41 ms of it the product)
// and takes 17.1 ms; element matrices of 990 H(curl) p = 4 elements in FP32
// 1.53 -> 0.38 ms.
template <typename T, int SPACE, int WGS, int POOL, int WPE>
__global__ __launch_bounds__(WGS, WPE) void sf_elem_kernel(ElemArgs a)
{
    __shared__ SfElem es;
    __shared__ SfTab tb;
    __shared__ __align__(16) short row[sf_comps(SPACE) * SF_I * SF_I * 8];
    __shared__ unsigned short pl[sf_comps(SPACE) * SF_I * SF_I];
    __shared__ short js[sf_comps(SPACE) * 8];
    __shared__ unsigned short gmap[SF_I * SF_I * SF_I];
    __shared__ __align__(16) double pool[POOL];
    const int e = blockIdx.x, tid = threadIdx.x, part = blockIdx.y, nparts = gridDim.y;
    const bool ok = sf_setup<SPACE>(a, e, es, tid);
    if (!ok || es.n > a.max_ndof) { // invalid codes, or above the caller's bound
        if (tid == 0 && part == 0 && a.status) a.status[e] = ok ? HP3D_E_ARG : HP3D_E_ORDER;
        return;
    }
    sf_fill_tab(es, tb, tid, WGS);
    sf_fill_rows<SPACE>(es, row, tid, WGS);
    if (a.ngeo != 8) sf_fill_gmap(es, a.ngeo, gmap, tid, WGS);
    lds_barrier();
    if (sf_points<SPACE>(es, tb, gmap, a.xnod + 3 * (size_t)a.ngeo * e, a.ngeo, a.coef[e], a.load, pool, tid, WGS))
        es.negjac = 1;
    if (tid < 64) sf_pencils<SPACE>(es, row, pl, js, tid);
    lds_barrier();
    if (part == nparts - 1 && a.bout) {
        double *bo = a.bout + a.off_v[e];
        for (int k = tid; k < sf_comps(SPACE) * SF_I * SF_I * 8; k += WGS) {
            const int r = row[k], pen = k >> 3;
            if (r < 0) continue;
            const double v = sf_load_entry<SPACE>(es, tb, pool, pen / (SF_I * SF_I), (pen / SF_I) % SF_I, pen % SF_I, k & 7);
            bo[r & ~ROW_NEG] = r & ROW_NEG ? -v : v;
        }
    }
    T *kout = (T *)a.kout + a.off_k[e];
    const long long ld = a.ld_k > 0 ? a.ld_k : es.n;
    switch (es.m[2]) {
    case 2: sf_matrix<T, SPACE, 2, POOL>(es, tb, row, pl, js, pool, kout, ld, part, nparts, tid, WGS); break;
    case 3: sf_matrix<T, SPACE, 3, POOL>(es, tb, row, pl, js, pool, kout, ld, part, nparts, tid, WGS); break;
    case 4: sf_matrix<T, SPACE, 4, POOL>(es, tb, row, pl, js, pool, kout, ld, part, nparts, tid, WGS); break;
    case 5: sf_matrix<T, SPACE, 5, POOL>(es, tb, row, pl, js, pool, kout, ld, part, nparts, tid, WGS); break;
    case 6: sf_matrix<T, SPACE, 6, POOL>(es, tb, row, pl, js, pool, kout, ld, part, nparts, tid, WGS); break;
    default: sf_matrix<T, SPACE, 7, POOL>(es, tb, row, pl, js, pool, kout, ld, part, nparts, tid, WGS); break;
    }
    if (tid == 0 && part == 0 && a.status) a.status[e] = es.negjac ? HP3D_NEG_JACOBIAN : 0;
}
