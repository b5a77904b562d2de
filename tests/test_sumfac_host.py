"""Host build of the shared topology header (hp3d_amd/csrc/hp3d_tables.h):
the tensor-side dof layout of the sum-factorised kernels (dof_row) is the
inverse of the hp3D-ordered descriptors (desc_h1, desc_hcurl), over random
anisotropic orders and all edge and face orientation codes, and its 1D tables
are the descriptors' tables.  Runs on the CPU with g++."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HEADER = os.path.join(HERE, "..", "hp3d_amd", "csrc", "hp3d_tables.h")

SRC = r"""
#define __host__
#define __device__
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include "%s"
using namespace hp3d;
// 1D index and sign of table entry t of a direction (P_{i-1} = chi_i')
static int index_of(int t, int &neg)
{
    if (t < 2) return t;
    if (t < 7) return t;
    if (t < 12) { neg ^= (t - 5) & 1; return t - 5; }
    if (t < 18) return t - 12 + 1;
    neg ^= (t - 18) & 1;
    return t - 18 + 1;
}
int main(int argc, char **argv)
{
    const int trials = atoi(argv[1]), space = atoi(argv[2]);
    srand(11 + space);
    long bad = 0, tot = 0;
    for (int it = 0; it < trials; ++it) {
        int hdr[37];
        for (int e = 0; e < 12; ++e) hdr[e] = 1 + rand() %% MAXP;
        for (int f = 0; f < 6; ++f) hdr[12 + f] = (1 + rand() %% MAXP) * MODORDER + 1 + rand() %% MAXP;
        hdr[18] = (1 + rand() %% MAXP) * 100 + (1 + rand() %% MAXP) * 10 + 1 + rand() %% MAXP;
        for (int e = 0; e < 12; ++e) hdr[19 + e] = rand() %% 2;
        for (int f = 0; f < 6; ++f) hdr[31 + f] = rand() %% 8;
        ElemOrders o;
        if (!decode_orders(hdr, hdr + 19, hdr + 31, o)) return 2;
        int n, nb;
        dof_counts(space, o, n, nb);
        DofBases b;
        dof_bases(space, o, b);
        bad += b.interior != n - nb;
        for (int k = 0; k < n; ++k) {
            const unsigned d = space == 0 ? desc_h1(k, o) : desc_hcurl(k, o);
            int neg = desc_neg(d), ix[3];
            for (int c = 0; c < 3; ++c) ix[c] = index_of(desc_ix(d, c), neg);
            const int r = dof_row(space, desc_comp(d), ix[0], ix[1], ix[2], o, b);
            ++tot;
            bad += r != k + (neg ? ROW_NEG : 0);
        }
        long rows = 0;
        for (int a = 0; a < (space ? 3 : 1); ++a)
            for (int i = 0; i < 343; ++i)
                rows += dof_row(space, a, i %% 7, i / 7 %% 7, i / 49, o, b) >= 0;
        bad += rows != n;
    }
    // the tables against table_at, to a few units of rounding
    static const SfTables t = make_sf_tables();
    const double gx[10][10] = HP3D_GAUSS_X;
    for (int n = 1; n <= MAXP + 1; ++n)
        for (int q = 0; q < n; ++q) {
            double v[NTAB], dv[NTAB];
            table_at(0.5 * (1.0 + gx[n - 1][q]), v, dv);
            for (int i = 0; i <= MAXP; ++i) {
                bad += std::fabs(t.f[n][0][i][q] - v[i]) > 4e-16;
                bad += std::fabs(t.f[n][1][i][q] - dv[i]) > 4e-16;
                if (i >= 1) bad += std::fabs(t.f[n][1][i][q] - v[t_leg(i - 1, 0)]) > 1e-15;
            }
        }
    printf("%%ld %%ld\n", tot, bad);
    return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("space", [0, 1])
def test_dof_rows_invert_the_descriptors(tmp_path, space):
    src = tmp_path / "rows.cpp"
    src.write_text(SRC % os.path.abspath(HEADER))
    exe = tmp_path / "rows"
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-o", str(exe), str(src)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    r = subprocess.run([str(exe), "4000", str(space)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    tot, bad = map(int, r.stdout.split())
    assert tot > 300_000 and bad == 0, (tot, bad)
