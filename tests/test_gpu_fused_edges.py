"""The one-launch element kernel at the elements where what an element keeps in
LDS comes to its pool's end, condensed against the oracle (tolerances of
condensed_against_oracle: the kernel and the reference both stay within about
sqrt(10^3) eps of K)."""
import numpy as np
import pytest

from hp3d_amd import mesh
from hp3d_amd.elem import ndof
from test_gpu_sumfac import FUSED, condensed_against_oracle

pytestmark = pytest.mark.gpu


def packed(n, nb):
    """doubles of the packed K: the interface's triangle, the bubble rows at an
    odd stride, padded to a multiple of four rows"""
    ni = n - nb
    return (ni * (ni + 1) // 2 + (nb + 3) // 4 * 4 * (n | 1) + 1) // 2 * 2


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("axis,mid,side,size", [(0, (3, 4, 6), (3, 3, 6), (126, 30)), (1, (4, 3, 6), (3, 3, 6), (126, 30)),
                                                (1, (6, 4, 3), (4, 4, 3), (124, 30)), (2, (3, 5, 5), (2, 4, 5), (126, 32)),
                                                (0, (5, 3, 5), (5, 4, 3), (128, 32)), (1, (5, 5, 3), (3, 5, 3), (128, 32))])
def test_graded_h1(gpu, axis, mid, side, size, precision):
    """Three elements in a row, the middle one of higher order: its K is larger
    than the 128-row pool, its fields and sums are not."""
    shape = [1, 1, 1]
    shape[axis] = 3
    m = mesh.structured(tuple(shape), porder=[side, mid, side], perm_seed=7 + axis, coef=[0.7, 1.9, 1.1])
    n, nb = ndof(0, m.norder)
    assert (n[1], nb[1]) == size and packed(*size) > 8352
    x = m.xnod() + 0.05 * np.random.default_rng(sum(mid)).uniform(-1, 1, (3, 8, 3))
    condensed_against_oracle(0, m.norder, m.nori_e, m.nori_f, x, m.coef, FUSED, precision)


def bounded_codes(rng, most, nel, least):
    """Codes with edge, face and interior orders of direction d in
    [least, most[d]], most of them and an edge of each direction at the bound;
    face orientations that do not swap the axes."""
    draw = lambda d, size: np.where(rng.random(size) < 0.75, most[d], rng.integers(least, most[d] + 1, size))
    no = np.zeros((nel, 19), np.int32)
    for k, d in enumerate(mesh.EDGE_DIR):
        no[:, k] = most[d] if k in (0, 1, 8) else draw(d, nel)
    for k, (s, t) in enumerate(mesh.FACE_AXES):
        no[:, 12 + k] = 10 * draw(s, nel) + draw(t, nel)
    no[:, 18] = 100 * draw(0, nel) + 10 * draw(1, nel) + draw(2, nel)
    oe = rng.integers(0, 2, (nel, 12)).astype(np.int32)
    return no, oe, rng.choice(np.array([0, 2, 5, 7], np.int32), (nel, 6))


def condensed_at_the_end(space, no, oe, of, seed):
    rng = np.random.default_rng(seed)
    v = mesh.VERT_XYZ[None] + 0.15 * rng.uniform(-1, 1, (len(no), 8, 3))
    condensed_against_oracle(space, no, oe, of, v, rng.uniform(0.5, 2.0, len(no)), FUSED)


@pytest.mark.parametrize("most", [(3, 4, 6), (6, 3, 4), (5, 3, 5), (5, 6, 3), (4, 5, 4)])
def test_edges_above_the_interior_h1(gpu, most):
    """The same pool, of elements whose interior orders are below the edges'."""
    no, oe, of = bounded_codes(np.random.default_rng(sum(most)), most, 20000, 2)
    n, nb = ndof(0, no)
    ok = np.nonzero((n >= 120) & (n <= 128) & (nb <= 32) & (nb > 0))[0]
    pick = np.array([e for e in ok if packed(int(n[e]), int(nb[e])) > 8352][:12])
    assert pick.size >= 4
    condensed_at_the_end(0, no[pick], oe[pick], of[pick], sum(most))


@pytest.mark.parametrize("interior,edges,faces,size", [(221, [5] * 12, [21] * 3 + [11] * 3, (64, 1)),
                                                       (122, [5] * 12, [12] * 3 + [11] * 3, (64, 1)),
                                                       (441, [4] * 5 + [5] * 7, [11] * 6, (64, 9)),
                                                       (144, [4] * 5 + [5] * 7, [11] * 6, (64, 9)),
                                                       (111, [5] * 12, [11] * 3 + [21] * 3, (63, 0)),
                                                       (111, [6] + [5] * 7 + [6] + [5] * 3, [11] * 6, (62, 0))])
def test_six_functions_a_direction_hcurl(gpu, interior, edges, faces, size):
    """64 rows in H(curl): K and the fields of 6 x 6 x 6 points just fit (and
    those of 7 x 6 x 7, the last, do not)."""
    no = np.array([edges + faces + [interior]] * 3, np.int32)
    assert (np.array(ndof(1, no[0])) == size).all()
    rng = np.random.default_rng(interior)
    oe = rng.integers(0, 2, (3, 12)).astype(np.int32)
    condensed_at_the_end(1, no, oe, rng.integers(0, 8, (3, 6)).astype(np.int32), interior)


@pytest.mark.parametrize("interior,faces,size", [(252, [33, 33, 23, 22, 11, 11], (128, 21)), (616, [33, 11, 23, 11, 33, 11], (128, 25)),
                                                 (226, [11, 13, 33, 33, 22, 11], (128, 26)), (234, [33, 33, 14, 11, 11, 11], (128, 29)),
                                                 (432, [11, 12, 11, 33, 33, 11], (126, 29)), (225, [33, 33, 23, 11, 11, 11], (124, 21))])
def test_seven_functions_a_direction_hcurl(gpu, interior, faces, size):
    """128 rows in H(curl), edges of order 6: K and the fields of 7 x 7 x 7
    points come to the pool's end."""
    no = np.array([[6] * 12 + faces + [interior]] * 3, np.int32)
    assert (np.array(ndof(1, no[0])) == size).all()
    rng = np.random.default_rng(interior)
    oe = rng.integers(0, 2, (3, 12)).astype(np.int32)
    condensed_at_the_end(1, no, oe, rng.integers(0, 8, (3, 6)).astype(np.int32), interior)
