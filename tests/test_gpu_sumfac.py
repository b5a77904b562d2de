"""The sum-factorised element matrices against the oracle, at the sizes and
codes where the kernel's splits change: every pair of pencil lengths and column
chunks (anisotropic orders), orders of edges and faces above the interior's,
isoparametric maps, a leading dimension above N and split elements (a few
elements run several workgroups each).

Tolerance: the reference sums O(10^3) products of magnitude |K|_F at most per
entry in FP64, as the kernel does in another order, so both stay within about
sqrt(10^3) eps of the exact value: 1e-13 of |K|_F covers both with room.  FP32
K is the FP64 value rounded once: 2^-24 relative to the largest entry, held
to 1e-7."""
import ctypes

import numpy as np
import pytest

import oracle
from hp3d_amd import mesh

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def random_codes(rng, nel, pmax):
    no = np.zeros((nel, 19), np.int32)
    no[:, :12] = rng.integers(1, pmax + 1, (nel, 12))
    no[:, 12:18] = 10 * rng.integers(1, pmax + 1, (nel, 6)) + rng.integers(1, pmax + 1, (nel, 6))
    b = rng.integers(1, pmax + 1, (nel, 3))
    no[:, 18] = 100 * b[:, 0] + 10 * b[:, 1] + b[:, 2]
    return no, rng.integers(0, 2, (nel, 12)).astype(np.int32), rng.integers(0, 8, (nel, 6)).astype(np.int32)


def check(space, no, oe, of, xnod, coef, precision=0):
    import torch

    import hp3d_amd

    load = oracle.LOAD_SINSINSIN if space == 0 else oracle.LOAD_CURL_SIN
    batch = hp3d_amd.ElementBatch(space, no, oe, of, xnod, coef, load=load, rules=({"path": "two_pass"},))
    out = batch.alloc_outputs(precision, want_stc=False)
    batch.element_matrices(out, precision)
    torch.cuda.synchronize()
    assert (batch.check_status() == 0).all()
    ref = oracle.element_loop(space, no, oe, of, xnod, coef, load, ldk=int(batch.n.max()), want_stc=False)
    for e in range(batch.nel):
        n = int(batch.n[e])
        k = batch.k_of(out, e)
        assert rel(k, ref["k"][e].T[:n, :n]) < (1e-13 if precision == 0 else 1e-7), (e, n)
        assert np.array_equal(k, k.T), e
        b = ref["b"][e][:n]
        assert np.linalg.norm(batch.vec_of(out, "b", e) - b) <= 1e-13 * max(np.linalg.norm(b), 1e-3)


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("space", [0, 1])
def test_any_codes(gpu, space, precision):
    rng = np.random.default_rng(50 + space)
    nel = 24
    no, oe, of = random_codes(rng, nel, 6)
    v = mesh.VERT_XYZ[None] + 0.15 * rng.uniform(-1, 1, (nel, 8, 3))
    check(space, no, oe, of, v, rng.uniform(0.5, 2.0, nel), precision)


@pytest.mark.parametrize("space", [0, 1])
@pytest.mark.parametrize("porder", [(6, 6, 6), (6, 5, 1), (1, 6, 6), (5, 1, 6), (2, 6, 4), (6, 3, 3), (4, 5, 2), (5, 5, 5)])
def test_anisotropic(gpu, space, porder):
    m = mesh.structured((2, 1, 1), porder=porder, perturb=0.0, perm_seed=3 + sum(porder), coef=[0.7, 1.9])
    x = m.xnod() + 0.05 * np.random.default_rng(sum(porder)).uniform(-1, 1, (2, 8, 3))
    check(space, m.norder, m.nori_e, m.nori_f, x, m.coef)


def condensed_against_oracle(space, no, oe, of, xnod, coef, rules, precision=0):
    """celem of one launch against the oracle (FP64: Aii and Bi 1e-12, the
    bubble solutions nb cond(Abb) eps; FP32 K only rounds K)."""
    import torch

    import hp3d_amd
    from test_gpu_elem import TOL64, compare

    load = oracle.LOAD_SINSINSIN if space == 0 else oracle.LOAD_CURL_SIN
    batch = hp3d_amd.ElementBatch(space, no, oe, of, xnod, coef, load=load, rules=rules)
    assert batch.bin_paths == ["fused"]
    out = batch.alloc_outputs(precision)
    for v in out.values():
        v.fill_(float("nan"))
    batch.celem(out, precision)
    bare = batch.run(precision, want_k=False)
    torch.cuda.synchronize()
    assert (batch.check_status() == 0).all()
    ref = oracle.element_loop(space, no, oe, of, xnod, coef, load, ldk=int(batch.n.max()), herm=True)
    compare(batch, out, ref, TOL64 if precision == 0 else 1e-7, TOL64)
    for e in range(batch.nel):
        k = batch.k_of(out, e)
        assert np.array_equal(k, k.T)
        a, b = batch.aii_of(out, e), batch.aii_of(bare, e)
        assert np.array_equal(a, a.T) and np.array_equal(a, b)
        ni = int(batch.ni[e])
        if batch.nb[e] == 0:
            assert rel(a, ref["k"][e].T[:ni, :ni]) < TOL64
            assert np.array_equal(batch.vec_of(out, "bi", e, ni), batch.vec_of(out, "b", e))


FUSED = ({"max_ndof": 128, "max_nbubble": 32, "path": "fused"}, {"path": "two_pass"})


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("space", [0, 1])
@pytest.mark.parametrize("most", [(64, 16), (128, 32)])
def test_fused_any_codes(gpu, space, most, precision):
    """Interior orders of at most 3 under edges and faces of up to 6: every
    storage mode of the one-launch kernel, the streamed one (seven functions in
    each direction) among them."""
    rng = np.random.default_rng(70 + space + most[0])
    no, oe, of = random_codes(rng, 4000, 6)
    b = rng.integers(1, 4 if space == 0 else 3, (4000, 3))
    no[:, 18] = 100 * b[:, 0] + 10 * b[:, 1] + b[:, 2]
    flat = rng.random(4000) < 0.8     # faces of order 1: mostly edges
    no[flat, 12:18] = 11
    from hp3d_amd.elem import ndof, nquad

    n, nb = ndof(space, no)
    ok = np.nonzero((n <= most[0]) & (nb <= most[1]) & (n > (0 if most[0] == 64 else 64)))[0]
    q = nquad(no[ok], of[ok]).min(1)
    pick = np.concatenate([ok[q == 7][:10], ok[q < 7][:14]])
    assert pick.size >= 16
    v = mesh.VERT_XYZ[None] + 0.15 * rng.uniform(-1, 1, (pick.size, 8, 3))
    condensed_against_oracle(space, no[pick], oe[pick], of[pick], v, rng.uniform(0.5, 2.0, pick.size), FUSED, precision)


@pytest.mark.parametrize("space,porder", [(0, (1, 1, 1)), (0, (2, 1, 2)), (0, (4, 4, 4)), (0, (3, 5, 4)), (0, (5, 4, 3)),
                                          (0, (6, 2, 2)), (0, (2, 6, 5)), (0, (6, 4, 2)), (0, (3, 3, 6)), (0, (1, 6, 6)),
                                          (1, (1, 1, 1)), (1, (2, 2, 2)), (1, (3, 3, 2)), (1, (1, 5, 2)), (1, (6, 1, 1))])
def test_fused_anisotropic(gpu, space, porder):
    m = mesh.structured((2, 1, 1), porder=porder, perm_seed=5 + sum(porder), coef=[0.7, 1.9])
    x = m.xnod() + 0.05 * np.random.default_rng(sum(porder)).uniform(-1, 1, (2, 8, 3))
    condensed_against_oracle(space, m.norder, m.nori_e, m.nori_f, x, m.coef, FUSED)


@pytest.mark.parametrize("space", [0, 1])
@pytest.mark.parametrize("ngeo", [8, 27, 343])
def test_field_any_codes(gpu, space, ngeo):
    """The field integrals at any orders and orientations (ngeo = 8) and with
    isoparametric maps, staged (27 nodes) and not (343).  Tolerance: the field
    at a point sums up to 343 products of O(1) dofs, 343 eps < 1e-13 of the
    field's own size; the integrals are quadratic in it and their weights carry
    a few eps more, so 1e-12 of their norms."""
    import torch

    import hp3d_amd
    from hp3d_amd import FIELD_ADJOINT, FIELD_ERROR, FIELD_L2
    from hp3d_amd.solve import field

    rng = np.random.default_rng(90 + space + ngeo)
    nel = 24 if ngeo == 8 else 4
    no, oe, of = random_codes(rng, nel, 6)
    if ngeo > 8:
        p = 2 if ngeo == 27 else 6
        no[:, :12], no[:, 12:18], no[:, 18] = p, 11 * p, 111 * p
    x = np.zeros((nel, ngeo, 3))
    x[:, :8] = mesh.VERT_XYZ[None] + 0.15 * rng.uniform(-1, 1, (nel, 8, 3))
    x[:, 8:] = 0.2 / ngeo * rng.uniform(-1, 1, (nel, ngeo - 8, 3))
    coef = rng.uniform(0.5, 2.0, nel)
    sel = oracle.LOAD_SINSINSIN if space == 0 else oracle.LOAD_CURL_SIN
    batch = hp3d_amd.ElementBatch(space, no, oe, of, x, coef, load=sel)
    u = torch.as_tensor(rng.normal(size=batch.size_v), device="cuda")
    v = torch.as_tensor(rng.normal(size=batch.size_v), device="cuda")
    err = field(batch, FIELD_ERROR, u, exact=sel)[0].cpu().numpy()
    l2, r = field(batch, FIELD_L2, u, with_r=True)
    adj = field(batch, FIELD_ADJOINT, u, v=v)[0].cpu().numpy()
    assert (batch.check_status() == 0).all()
    l2 = l2.cpu().numpy()
    for e in range(nel):
        i = int(batch.iperm[e])
        o, n = int(batch.off_v_h[i]), int(batch._n[i])
        ue, ve, re = (t[o:o + n].cpu().numpy() for t in (u, v, r))
        assert rel(err[i], np.array(oracle.element_error(space, no[e], oe[e], of[e], x[e].T, ue, sel))) < 1e-12, e
        mm = oracle.elem_mass(space, no[e], oe[e], of[e], x[e].T)
        assert abs(l2[i] - ue @ mm @ ue) < 1e-12 * (ue @ mm @ ue), e
        assert rel(re, mm @ ue) < 1e-12, e
        k = oracle.elem_h1(no[e], oe[e], of[e], x[e].T, kappa=coef[e])[0] if space == 0 else coef[e] * mm
        assert abs(adj[i] + ve @ k @ ue) < 1e-12 * np.sqrt((ve @ k @ ve) * (ue @ k @ ue)), e
