"""Where the one-launch element kernel keeps an element in LDS, over every
element its launch shapes admit: all 1D sizes, interior orders and dof counts,
for the constants the kernel is launched with (hp3d_sumfac_layout.h built for
the host).  Each must have packed K, point fields and sums inside the pool in
its mode, and a streamed one the template of its last direction's size.  Runs
on the CPU with g++."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HEADER = os.path.join(HERE, "..", "hp3d_amd", "csrc", "hp3d_sumfac_layout.h")

SRC = r"""
#define __host__
#define __device__
#include <cstdio>
#include <cstdlib>
#include "%s"
using namespace hp3d;
static long count[3], bad;
static void fail(const char *what, const int (&m)[3], int n, int nb, int mode)
{
    if (bad++ < 8) printf("# %%s: sizes %%d %%d %%d, n %%d, nb %%d, mode %%d\n", what, m[0], m[1], m[2], n, nb, mode);
}
template <int SPACE> static void element(const SfShape s, const int (&md)[3], int n, int nb)
{
    const SfFused fu = sf_limits(s);
    const SfRoles r = sf_roles<SPACE>(md, n, nb, fu);
    if (((1 << r.b) | (1 << r.a) | (1 << r.c)) != 7) return fail("roles", md, n, nb, r.mode);
    const int mB = md[r.b], mA = md[r.a], mC = md[r.c], mcp = (mC + 1) / 2 * 2, Q = mA * mB * mC;
    const SfLay ly(n, nb, fu.nbx);
    const bool cond = nb <= fu.nbx;
    ++count[r.mode];
    auto need = [&](const char *what, int doubles) { if (doubles > s.pool) fail(what, md, n, nb, r.mode); };
    // storage: the last entry of every row inside, the zero rows behind them
    if (ly.ni != (cond ? n - nb : n) || ly.len < ly.kb + (n - ly.ni + 3) / 4 * 4 * ly.ldb) fail("layout", md, n, nb, r.mode);
    for (int k = 0; k < n; ++k)
        if (ly.row(k) + k >= ly.len || (k > 0 && ly.row(k) <= ly.row(k - 1) + k - 1)) fail("row", md, n, nb, r.mode);
    const int fields = (SPACE == 0 ? 7 : 15) * Q + fu.xg, metric = (SPACE == 0 ? 6 : 12) * Q;
    const int tabs = SPACE == 0 ? 8 : 9, one = tabs * mB * mcp; // sums of a pair of 1D functions
    const int w = s.nbt == 1 && cond && nb > 0 ? 16 * 17 : 0;   // L^-1, where it has its place in the pool
    const int at = 16 * ((ly.ni + 16) / 16) - 1;                // last row of the update's tiles
    if (r.mode != SF_STREAM && cond && nb > 0) need("tiles of Aii", at * (at + 1) / 2 + at + 1);
    if (r.mode == SF_DIRECT) {
        need("K and fields", ly.len + fields);
        need("K and a row of sums", ly.len + metric + one);
        need("K and L^-1", ly.len + w);
    } else if (r.mode == SF_HOLD) {
        const int P = mA * mB, items = P * (P + 1) / 2, held = mC == 5 ? fu.h5 : mC == 4 ? fu.h4 : 0;
        if (SPACE != 0 || s.nbt == 1 || items > held * fu.wgs) fail("held pairs", md, n, nb, r.mode);
        need("fields", fields);
        need("all sums", metric + mA * (mA + 1) / 2 * one);
        need("K", ly.len);
    } else {
        if (!sf_streams(s) || sf_stream_mc(s, mC) != mC) fail("streamed template", md, n, nb, r.mode);
        const int rows = ly.len - (ly.kb + 1) / 2 * 2; // bubble rows at the pool's end
        need("fields", fields);
        need("bubble rows and a row of sums", rows + metric + one);
        need("bubble rows and L^-1", rows + w);
    }
}
template <int SPACE> static void shape(const SfShape s)
{
    int m[3];
    for (m[0] = 2; m[0] <= SF_I; ++m[0])
        for (m[1] = 2; m[1] <= SF_I; ++m[1])
            for (m[2] = 2; m[2] <= SF_I; ++m[2]) {
                // interface dofs of an element with these sizes, at least and at most
                const int least = SPACE == 0 ? 8 : 12;
                int most = SPACE == 0 ? 8 : 0;
                for (int d = 0; d < 3; ++d) {
                    const int p = m[d] - 1, q = m[(d + 1) %% 3] - 1;
                    most += SPACE == 0 ? 4 * (p - 1) + 2 * (p - 1) * (q - 1) : 4 * p + 2 * (p * (q - 1) + (p - 1) * q);
                }
                for (int i = 0; i < (m[0] - 1) * (m[1] - 1) * (m[2] - 1); ++i) {
                    const int x = i %% (m[0] - 1) + 1, y = i / (m[0] - 1) %% (m[1] - 1) + 1, z = i / ((m[0] - 1) * (m[1] - 1)) + 1;
                    const int nb = SPACE == 0 ? (x - 1) * (y - 1) * (z - 1)
                                              : x * (y - 1) * (z - 1) + (x - 1) * y * (z - 1) + (x - 1) * (y - 1) * z;
                    for (int n = nb + least; n <= nb + most && n <= s.rows; ++n) element<SPACE>(s, m, n, nb);
                }
            }
}
int main(int, char **argv)
{
    const SfShape s = sf_shape(atoi(argv[1]));
    if (s.space == 0) shape<0>(s);
    else shape<1>(s);
    printf("%%ld %%ld %%ld %%ld\n", count[SF_STREAM], count[SF_DIRECT], count[SF_HOLD], bad);
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    d = tmp_path_factory.mktemp("layout")
    src, exe = d / "layout.cpp", d / "layout"
    src.write_text(SRC % os.path.abspath(HEADER))
    r = subprocess.run(["g++", "-O2", "-std=c++17", "-o", str(exe), str(src)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return str(exe)


@pytest.mark.parametrize("shape", [0, 1, 2, 3], ids=["h1_64", "h1_128", "hcurl_64", "hcurl_128"])
def test_every_element_fits(program, shape):
    r = subprocess.run([program, str(shape)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    *_, last = r.stdout.splitlines()
    stream, direct, hold, bad = map(int, last.split())
    assert bad == 0, r.stdout
    assert direct > 10_000 and (shape != 1 or (stream > 100 and hold > 100)), r.stdout
