// hp3d_sumfac_layout.h -- where the one-launch element kernel (sf_fused_kernel)
// keeps an element in LDS: its launch shapes, the storage of K and the choice of
// an element's mode.  Shared by the kernel, its launch and a host test that goes
// through every element the shapes admit.
#pragma once

#include "hp3d_tables.h"

namespace hp3d {

constexpr int SF_I = MAXP + 1; // 1D functions per direction
HP3D_HD constexpr int sf_comps(int space) { return space == 0 ? 1 : 3; }
// fields per point: metric (6 symmetric entries; H(curl) curl, then mass) and load
HP3D_HD constexpr int sf_fields(int space) { return space == 0 ? 7 : 15; }
HP3D_HD constexpr int sf_ttabs(int space) { return space == 0 ? 8 : 9; }

constexpr int XS_MAX = 27; // geometry nodes staged in LDS by the geometry code
// doubles of the staged geometry nodes, the coefficient and the node map
constexpr int SF_XG = 3 * XS_MAX + 1 + (SF_I * SF_I * SF_I + 3) / 4;

// One launch shape: elements of at most `rows` dofs and 16 nbt bubbles, `waves`
// waves with a pool of `pool` doubles, wpe waves per SIMD (launch bound), per_cu
// workgroups on a CU.  The waves are those that fill a CU with the workgroups
// that the pools let in.  Measured (workgroups x waves of a CU):
//   13,824 H1 p = 3 elements, FP64, and p = 2: 4 x 3 at 168 registers 0.386 and
//   0.228 ms; 4 x 4 at 128 0.385 and 0.246; 3 x 4 0.438 and 0.280; 4 x 2 0.417
//   and 0.228; 4 x 1 0.484 and 0.244;
//   8,000 H1 p = 4 elements, FP64 and FP32: 2 x 8 at 128 registers 0.612 and
//   0.612 ms; 2 x 4 at 256 0.662 and 0.650; 6 waves at 168 registers leave a CU
//   one workgroup (a SIMD would have to take four of their waves): 1.03 and 1.06;
//   8,000 H(curl) p = 2 elements: 3 x 4 0.281 ms, 3 x 3 0.305, 3 x 2 0.320, 2 x 4
//   (a pool of 8,000) 0.338.
// The 64-row H(curl) pool is the smallest in which every element with at most
// six functions a direction is direct (N = 64, nb = 9: 5,728), so that the one
// streamed template is of seven; the 128-row one the smallest in which every
// element is direct (N = 128, nb = 29 at 7 x 7 x 7 points: 14,223).  The 128-row
// H1 pool is about what two workgroups leave of a CU's LDS: the packed K of a
// whole p = 4 element; what is larger is streamed.
struct SfShape {
    int space, rows, nbt, waves, pool, wpe, per_cu;
};
enum { SF_H1_64 = 0, SF_H1_128 = 1, SF_HCURL_64 = 2, SF_HCURL_128 = 3, SF_SHAPES = 4 };
HP3D_HD constexpr SfShape sf_shape(int i)
{
    return i == SF_H1_64    ? SfShape{0, 64, 1, 3, 4500, 3, 4}
         : i == SF_H1_128   ? SfShape{0, 128, 2, 8, 8352, 4, 2}
         : i == SF_HCURL_64 ? SfShape{1, 64, 1, 4, 5728, 3, 3}
                            : SfShape{1, 128, 2, 8, 14224, 2, 1};
}

// How the block of K is kept while its entries are computed (sf_roles)
enum { SF_STREAM = 0, SF_DIRECT = 1, SF_HOLD = 2 };

// where a pool of doubles holds one element's packed K (PK), fields and T:
// which roles the directions take, and whether K's entries go straight to LDS
// (SF_DIRECT: packed K, fields and at least one row of T fit together), stay in
// registers until T is done with (SF_HOLD: all of T fits, and then the packed K
// in its place; one pencil pair per thread at MC = 5, two at MC = 4), or are
// recomputed (SF_STREAM)
struct SfFused {
    int pool, wgs, nbx; // nbx: the most bubbles it condenses
    int xg;             // pool doubles taken by the staged nodes
    int h5, h4;         // pencil pairs a thread holds at MC = 5 and 4 (0: never)
};
HP3D_HD constexpr SfFused sf_limits(const SfShape s)
{
    const int wgs = 64 * s.waves, h5 = s.space == 0 && s.rows > 64 ? (325 + wgs - 1) / wgs : 0;
    return SfFused{s.pool, wgs, 16 * s.nbt, s.nbt > 1 ? 0 : SF_XG, h5, h5 ? (666 + wgs - 1) / wgs : 0};
}
// the shapes with streamed elements (the pool of the 128-row H(curl) form holds
// every element's K, fields and T), and the 1D size that such an element's last
// direction is taken for
HP3D_HD constexpr bool sf_streams(const SfShape s) { return s.space == 0 || s.rows < 128; }
HP3D_HD constexpr int sf_stream_mc(const SfShape s, int mC) { return sf_limits(s).h5 > 0 && mC == 6 ? 6 : 7; }

// a b of 24-bit values
HP3D_HD inline int sf_mul24(int a, int b)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __mul24(a, b);
#else
    return a * b;
#endif
}
HP3D_HD inline int sf_min(int a, int b) { return a < b ? a : b; }
HP3D_HD inline int sf_max(int a, int b) { return a > b ? a : b; }

// Storage of one element's symmetric K in LDS: rows r < ni as a packed lower
// triangle, entry (r, c) at r (r + 1) / 2 + c, then the bubble rows at an odd
// stride, whole up to their diagonal, and zero rows up to a multiple of four
// (an element that is not condensed has all rows packed: ni = n)
struct SfLay {
    int ni, kb, ldb, len;
    HP3D_HD SfLay(int n, int nb, int nbx)
    {
        ni = nb <= nbx ? n - nb : n;
        kb = ni * (ni + 1) / 2;
        ldb = n | 1;
        len = (kb + ((n - ni + 3) & ~3) * ldb + 1) & ~1;
    }
    HP3D_HD inline int row(int r) const
    {
        const int t = sf_mul24(r, r + 1) >> 1, b = kb + sf_mul24(r - ni, ldb);
        return r < ni ? t : b;
    }
};

// Roles of the directions (which of x, y, z is B, A and C) and the mode of one
// element (1D sizes md[], n dofs, nb of them bubbles).  Without a pool (the
// streaming kernel): (B, A, C) = (x, y, z), so that consecutive lanes run along
// consecutive bubble rows.  A fused kernel takes the C that costs the fewest
// steps, counting whole passes of the workgroup over the pencil pairs, of those
// that fit its pool.
struct SfRoles {
    int mode, b, a, c;
};
template <int SPACE> HP3D_HD inline SfRoles sf_roles(const int (&md)[3], int n, int nb, const SfFused fu)
{
    int best = SF_STREAM, cC = 2, cA = 1, cost = 0x7fffffff;
    if (fu.pool > 0) {
        const int Q = md[0] * md[1] * md[2], pk = SfLay(n, nb, fu.nbx).len;
        const int dl = sf_fields(SPACE) * Q + fu.xg, dk = (SPACE == 0 ? 6 : 12) * Q; // with and without the load
        // SF_HOLD stores all of K over fields and sums: graded elements such as
        // orders (3, 4, 6) with N = 126, nb = 30 have room for those but not for K
        const bool room = pk <= fu.pool;
        if (md[0] == md[1] && md[1] == md[2]) { // nothing to choose but the mode
            const int m = md[0], one = sf_ttabs(SPACE) * m * ((m + 1) & ~1), P = m * m;
            if (pk + sf_max(dl, dk + one) <= fu.pool) best = SF_DIRECT;
            else if (room && sf_max(dl, dk + m * (m + 1) / 2 * one) <= fu.pool && P * (P + 1) / 2 <= (m == 5 ? fu.h5 : m == 4 ? fu.h4 : 0) * fu.wgs)
                best = SF_HOLD;
        } else {
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const int C = 2 - i, x = C == 0 ? 1 : 0, y = C == 2 ? 1 : 2; // the other two, x < y
                const int mC = md[C], mcp = (mC + 1) & ~1, mx = md[x], my = md[y], lo = sf_min(mx, my), hi = sf_max(mx, my);
                const int P = (SPACE == 0 ? 1 : 3) * mx * my, items = P * (P + 1) / 2;
                const int pass = ((items + fu.wgs - 1) / fu.wgs), tail = 2 * mC * mC * mC + 4 * mC * mC;
                // direct: B the shorter of the two (its sums are the inner loop)
                const bool direct = pk + sf_max(dl, dk + sf_ttabs(SPACE) * lo * mcp) <= fu.pool;
                const int cap = mC == 5 ? fu.h5 * fu.wgs : mC == 4 ? fu.h4 * fu.wgs : 0;
                const bool hold = room && items <= cap && sf_max(dl, dk + 4 * lo * (lo + 1) * hi * mcp) <= fu.pool;
                const int mode = direct ? SF_DIRECT : hold ? SF_HOLD : SF_STREAM;
                const int c = direct ? pass * (9 * lo * mC + tail) : hold ? pass * (9 * hi * mC + tail) : 0x7fffffff;
                if (mode != SF_STREAM && c < cost) {
                    cost = c;
                    best = mode;
                    cC = C;
                    cA = (mode == SF_DIRECT) == (my >= mx) ? y : x;
                    if (mx == my) cA = y;
                }
            }
        }
        if (best == SF_STREAM) { // the longest direction for C
            cC = md[2] >= md[0] && md[2] >= md[1] ? 2 : md[1] >= md[0] ? 1 : 0;
            cA = cC == 1 ? 2 : 1;
        }
    }
    return SfRoles{best, 3 - cC - cA, cA, cC};
}

} // namespace hp3d
