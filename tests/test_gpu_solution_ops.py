"""Back substitution, gather-sum and CSR product against numpy at the sizes
where their splits change: few and many elements (a workgroup or a wave each),
one bubble, as many as a wave and more, ragged tails and empty segments.

Tolerance: every result is an FP64 sum of at most 1,000 products in another
order; 1,000 eps of the sum of magnitudes is 2.3e-13, held to 1e-12."""
import ctypes

import numpy as np
import pytest

from hp3d_amd import mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("space,porder,shape", [(0, 2, (3, 2, 1)), (0, 2, (11, 10, 10)), (0, 5, (2, 2, 2)), (0, 6, (11, 10, 10)),
                                                (0, (6, 6, 2), (2, 2, 1)), (1, (2, 2, 1), (3, 3, 1)), (1, 4, (11, 10, 10)),
                                                (1, 6, (2, 1, 1)), (0, 0, (12, 11, 9))])
def test_back_substitute(gpu, space, porder, shape):
    import torch

    import hp3d_amd
    from hp3d_amd import solve

    rng = np.random.default_rng(sum(shape))
    nel = shape[0] * shape[1] * shape[2]
    m = mesh.structured(shape, porder=porder or rng.integers(1, 6, (nel, 3)), perm_seed=4)
    batch = hp3d_amd.ElementBatch.from_mesh(space, m)
    size = int((batch.off_s_h + batch._nb * batch._ni).max())
    out = {"aschur": torch.as_tensor(rng.normal(size=max(size, 1)), device="cuda"),
           "bschur": torch.as_tensor(rng.normal(size=batch.size_v), device="cuda")}
    u = torch.as_tensor(rng.normal(size=batch.size_v), device="cuda")
    before = u.cpu().numpy()
    got = solve.back_substitute(batch, out, u).cpu().numpy()
    a, b = out["aschur"].cpu().numpy(), out["bschur"].cpu().numpy()
    want, mag = before.copy(), np.ones_like(before)
    for i in range(nel):
        n, ni, nb, o = int(batch._n[i]), int(batch._ni[i]), int(batch._nb[i]), int(batch.off_v_h[i])
        s = a[batch.off_s_h[i]:batch.off_s_h[i] + nb * ni].reshape(ni, nb)
        want[o + ni:o + n] = b[o:o + nb] - before[o:o + ni] @ s
        mag[o + ni:o + n] += np.abs(before[o:o + ni]) @ np.abs(s) + np.abs(b[o:o + nb])
    assert (np.abs(got - want) <= 1e-12 * mag).all()


@pytest.mark.parametrize("n", [1, 255, 257, 32768, 32769, 70001])
def test_gather_and_spmv(gpu, n):
    import torch

    from hp3d_amd import _lib

    lib = _lib.load()
    rng = np.random.default_rng(n)
    cnt = rng.integers(0, 9, n)
    cnt[rng.integers(0, n)] = 300
    ptr = np.concatenate([[0], np.cumsum(cnt)])
    src = rng.integers(0, n, ptr[-1])
    vals, x = rng.normal(size=ptr[-1]), rng.normal(size=n)
    t = [torch.as_tensor(v, device="cuda") for v in (ptr, src, src.astype(np.int32), vals, x)]
    y = torch.full((2, n), float("nan"), dtype=torch.float64, device="cuda")
    p = lambda v: ctypes.c_void_p(v.data_ptr())
    assert lib.hp3d_gpu_gather_sum(n, p(t[0]), p(t[1]), p(t[4]), p(y[0]), None) == 0
    assert lib.hp3d_gpu_csr_spmv(n, p(t[0]), p(t[2]), p(t[3]), p(t[4]), p(y[1]), None) == 0
    torch.cuda.synchronize()
    row = np.repeat(np.arange(n), cnt)
    for got, terms in zip(y.cpu().numpy(), (x[src], vals * x[src])):
        want, mag = np.bincount(row, terms, n), np.bincount(row, np.abs(terms), n)
        assert (np.abs(got - want) <= 1e-12 * mag).all()


@pytest.mark.parametrize("n", [3, 16383, 16384])
@pytest.mark.parametrize("longest", [1, 16, 17, 32, 33, 130])
def test_spmv_row_lengths(gpu, n, longest):
    """Rows of up to one product a lane and beyond, few rows and many, empty
    ones among them."""
    import torch

    from hp3d_amd import _lib

    lib = _lib.load()
    rng = np.random.default_rng(n + longest)
    cnt = rng.integers(0, longest + 1, n)
    cnt[:: 7] = longest
    ptr = np.concatenate([[0], np.cumsum(cnt)])
    src = rng.integers(0, n, ptr[-1])
    vals, x = rng.normal(size=ptr[-1]), rng.normal(size=n)
    t = [torch.as_tensor(v, device="cuda") for v in (ptr, src.astype(np.int32), vals, x)]
    y = torch.full((n,), float("nan"), dtype=torch.float64, device="cuda")
    p = lambda v: ctypes.c_void_p(v.data_ptr())
    assert lib.hp3d_gpu_csr_spmv(n, *(p(v) for v in t), p(y), None) == 0
    torch.cuda.synchronize()
    row, terms = np.repeat(np.arange(n), cnt), vals * x[src]
    want, mag = np.bincount(row, terms, n), np.bincount(row, np.abs(terms), n)
    assert (np.abs(y.cpu().numpy() - want) <= 1e-12 * mag).all()


def codes(space, edge, face, body):
    """norder of equal edges and faces under a body code, and (n, nb)."""
    no = np.array([edge] * 12 + [face] * 6 + [body], np.int32)
    h, v, (x, y, z) = face // 10, face % 10, (int(c) for c in str(body))
    if space == 0:
        nb = (x - 1) * (y - 1) * (z - 1)
        n = 8 + 12 * (edge - 1) + 6 * (h - 1) * (v - 1) + nb
    else:
        nb = x * (y - 1) * (z - 1) + (x - 1) * y * (z - 1) + (x - 1) * (y - 1) * z
        n = 12 * edge + 6 * (h * (v - 1) + (h - 1) * v) + nb
    return no, n, nb


@pytest.mark.parametrize("space,bound,elements", [
    (0, (64, 16), [(1, 11, 111), (2, 22, 222), (3, 33, 333), (1, 22, 353), (5, 11, 333), (3, 33, 323)]),
    # interface and bubbles at and beyond what the kernel keeps on the chip (nb = 30 of N = 128)
    (0, (128, 32), [(4, 44, 444), (1, 46, 643), (1, 46, 422), (2, 44, 543), (5, 34, 111), (4, 44, 333)]),
    (1, (64, 16), [(1, 11, 111), (2, 22, 222), (4, 11, 122), (4, 11, 222)]),
    (1, (128, 32), [(2, 33, 222), (3, 22, 322), (1, 33, 332), (2, 33, 321)])])
@pytest.mark.parametrize("mode", ["packed", "strided", "inplace", "fp32"])
def test_condense_stored(gpu, space, bound, elements, mode):
    """stc_batch on random SPD systems with eigenvalues in [1, 5] (N cond eps
    of the norm is 128 * 5 * 2.2e-16 = 1.4e-13, held to 1e-12); with a leading
    dimension above N, in place, and K read as FP32."""
    import torch

    from hp3d_amd import _lib

    lib = _lib.load()
    rng = np.random.default_rng(sum(bound) + space)
    el = [codes(space, *x) for x in elements] * 3
    assert all(n <= bound[0] and nb <= bound[1] for _, n, nb in el)
    nel, ld = len(el), 0 if mode in ("packed", "fp32") else 131
    f32 = mode == "fp32"
    ks, off_k, off_v, off_c, off_s = [], [0], [0], [0], [0]
    for _, n, nb in el:
        q = np.linalg.qr(rng.normal(size=(n, n)))[0]
        k = (q * rng.uniform(1, 5, n)) @ q.T
        k = 0.5 * (k + k.T)
        ks.append(k.astype(np.float32).astype(np.float64) if f32 else k)
        off_k.append(off_k[-1] + (ld or n) * n)
        off_v.append(off_v[-1] + n)
        off_c.append(off_c[-1] + (n - nb) ** 2)
        off_s.append(off_s[-1] + (n - nb) * nb)
    kin = np.full(off_k[-1], np.nan)
    for k, o in zip(ks, off_k):
        kin[o:o + (ld or len(k)) * len(k)].reshape(len(k), -1)[:, :len(k)] = k
    b = rng.normal(size=off_v[-1])
    dev = lambda v, t=None: torch.as_tensor(np.asarray(v), dtype=t, device="cuda")
    kd, bd = dev(kin, torch.float32 if f32 else torch.float64), dev(b)
    inplace = mode == "inplace"
    aii = kd if inplace else torch.full((off_c[-1],), float("nan"), dtype=torch.float64, device="cuda")
    bi = bd if inplace else torch.full_like(bd, float("nan"))
    xs, xb = (torch.full((m,), float("nan"), dtype=torch.float64, device="cuda") for m in (max(off_s[-1], 1), off_v[-1]))
    no = dev(np.stack([x[0] for x in el]))
    offs = [dev(o, torch.int64) for o in (off_k, off_v, off_k if inplace else off_c, off_s)]
    st = dev(np.arange(nel) % 2, torch.int32)    # every other one with a warning to keep
    ws = torch.empty(max(lib.hp3d_gpu_stc_workspace(nel, *bound), 1), dtype=torch.uint8, device="cuda")
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    rc = lib.hp3d_gpu_stc_batch(space, int(f32), nel, p(no), p(offs[0]), ld, p(kd), p(offs[1]), p(bd), p(offs[2]),
                                ld if inplace else 0, p(aii), p(bi), p(offs[3]), p(xs), p(xb), p(ws), p(st), *bound, None)
    torch.cuda.synchronize()
    assert rc == 0 and np.array_equal(st.cpu().numpy(), np.arange(nel) % 2)
    aii, bi, xs, xb = (t.cpu().numpy().astype(np.float64) for t in (aii, bi, xs, xb))
    close = lambda x, y: np.linalg.norm(x - y) <= 1e-12 * max(np.linalg.norm(y), 1.0)
    for e, (_, n, nb) in enumerate(el):
        ni, k, be = n - nb, ks[e], b[off_v[e]:off_v[e] + n]
        x = np.linalg.solve(k[ni:, ni:], np.column_stack([k[ni:, :ni], be[ni:]])) if nb else np.zeros((0, ni + 1))
        o = off_k[e] if inplace else off_c[e]
        a = aii[o:o + (ld if inplace else ni) * ni].reshape(ni, -1)[:, :ni]
        assert close(a, k[:ni, :ni] - k[:ni, ni:] @ x[:, :ni]) and np.array_equal(a, a.T), (e, n, nb)
        assert close(bi[off_v[e]:off_v[e] + ni], be[:ni] - k[:ni, ni:] @ x[:, ni]), (e, n, nb)
        assert close(xs[off_s[e]:off_s[e] + ni * nb].reshape(ni, nb), x[:, :ni].T), (e, n, nb)
        assert close(xb[off_v[e]:off_v[e] + nb], x[:, ni]), (e, n, nb)


@pytest.mark.parametrize("space,bound,elements", [(0, (64, 16), [(1, 11, 111), (5, 11, 111), (2, 22, 231)]),
                                                  (0, (128, 32), [(1, 11, 111), (6, 33, 111), (5, 44, 166)]),
                                                  (1, (64, 16), [(1, 11, 111), (4, 12, 121), (5, 11, 161)]),
                                                  (1, (128, 32), [(1, 11, 111), (6, 11, 116), (4, 23, 111)])])
@pytest.mark.parametrize("mode", ["packed", "strided", "inplace", "fp32"])
def test_condense_without_bubbles(gpu, space, bound, elements, mode):
    """An element without bubbles comes through as it is, to the bit, also an
    unsymmetric one, among elements of a batch with other bounds."""
    import torch

    from hp3d_amd import _lib

    lib = _lib.load()
    rng = np.random.default_rng(sum(bound) + space + 1)
    el = [codes(space, *x) for x in elements] * 3
    assert all(n <= bound[0] and nb == 0 for _, n, nb in el)
    nel, ld = len(el), 0 if mode in ("packed", "fp32") else 131
    f32, inplace = mode == "fp32", mode == "inplace"
    off_k = np.concatenate([[0], np.cumsum([(ld or n) * n for _, n, _ in el])])
    off_v = np.concatenate([[0], np.cumsum([n for _, n, _ in el])])
    off_c = np.concatenate([[0], np.cumsum([n * n for _, n, _ in el])])
    dt = torch.float32 if f32 else torch.float64
    dev = lambda v, t=None: torch.as_tensor(np.asarray(v), dtype=t, device="cuda")
    kd, bd = dev(rng.normal(size=off_k[-1]), dt), dev(rng.normal(size=off_v[-1]))
    kin, b = kd.cpu().numpy().astype(np.float64), bd.cpu().numpy()
    aii = kd if inplace else torch.full((int(off_c[-1]),), float("nan"), dtype=torch.float64, device="cuda")
    bi = bd if inplace else torch.full_like(bd, float("nan"))
    none = torch.zeros(1, dtype=torch.float64, device="cuda")
    no = dev(np.stack([x[0] for x in el]))
    offs = [dev(o, torch.int64) for o in (off_k, off_v, off_k if inplace else off_c, [0] * nel)]
    st = dev(np.arange(nel) % 3, torch.int32)    # a warning to keep, and a stale code
    ws = torch.empty(lib.hp3d_gpu_stc_workspace(nel, *bound), dtype=torch.uint8, device="cuda")
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    rc = lib.hp3d_gpu_stc_batch(space, int(f32), nel, p(no), p(offs[0]), ld, p(kd), p(offs[1]), p(bd), p(offs[2]),
                                ld if inplace else 0, p(aii), p(bi), p(offs[3]), p(none), p(none), p(ws), p(st), *bound, None)
    torch.cuda.synchronize()
    assert rc == 0 and np.array_equal(st.cpu().numpy(), np.arange(nel) % 3 == 1)
    aii, bi = aii.cpu().numpy(), bi.cpu().numpy()
    assert np.array_equal(bi, b)
    for e, (_, n, _) in enumerate(el):
        k = kin[off_k[e]:off_k[e] + (ld or n) * n].reshape(n, -1)[:, :n]
        o = off_k[e] if inplace else off_c[e]
        a = aii[o:o + (ld if inplace else n) * n].reshape(n, -1)[:, :n]
        assert np.array_equal(a, k), (e, n)


@pytest.mark.parametrize("space,edge,body", [(0, 2, 455), (0, 5, 555), (0, 6, 666), (1, 3, 333), (1, 4, 444), (1, 6, 555), (1, 6, 666)])
def test_condense_in_place_by_strips(gpu, space, edge, body):
    """Systems of more than 32 bubbles condensed in place, as stc_fwd does on
    ALOC: the same bits as out of place, and within N cond eps (882 * 5 *
    2.2e-16 = 9.8e-13, held to 1e-11) of numpy."""
    import torch

    from hp3d_amd import _lib

    lib = _lib.load()
    rng = np.random.default_rng(edge + body)
    no, n, nb = codes(space, edge, 11 * edge, body)
    assert nb > 32
    nel, ld, ni = 6, n + 5, n - nb
    q = np.linalg.qr(rng.normal(size=(n, n)))[0]
    ks = [(q * rng.uniform(1, 5, n)) @ q.T for _ in range(nel)]
    kin = np.full((nel, n, ld), np.nan)
    for e, k in enumerate(ks):
        kin[e, :, :n] = 0.5 * (k + k.T)
    b = rng.normal(size=(nel, n))
    dev = lambda v, t=None: torch.as_tensor(np.ascontiguousarray(v), dtype=t, device="cuda")
    nod, off_k, off_v, off_s = (dev(v, t) for v, t in ((np.stack([no] * nel), torch.int32), (np.arange(nel) * n * ld, torch.int64),
                                                       (np.arange(nel) * n, torch.int64), (np.arange(nel) * nb * ni, torch.int64)))
    ws = torch.empty(lib.hp3d_gpu_stc_workspace(nel, n, nb), dtype=torch.uint8, device="cuda")
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    out = []
    for inplace in (False, True):
        kd, bd = dev(kin.reshape(-1)), dev(b.reshape(-1))
        aii, bi = (kd, bd) if inplace else (torch.full_like(kd, float("nan")), torch.full_like(bd, float("nan")))
        xs = torch.full((nel * nb * ni,), float("nan"), dtype=torch.float64, device="cuda")
        xb = torch.full_like(bd, float("nan"))
        st = torch.zeros(nel, dtype=torch.int32, device="cuda")
        rc = lib.hp3d_gpu_stc_batch(space, 0, nel, p(nod), p(off_k), ld, p(kd), p(off_v), p(bd), p(off_k), ld, p(aii),
                                    p(bi), p(off_s), p(xs), p(xb), p(ws), p(st), n, nb, None)
        torch.cuda.synchronize()
        assert rc == 0 and (st == 0).all()
        out.append([aii.view(nel, n, ld)[:, :ni, :ni].cpu().numpy(), bi.view(nel, n)[:, :ni].cpu().numpy(),
                    xs.view(nel, ni, nb).cpu().numpy(), xb.view(nel, n)[:, :nb].cpu().numpy()])
    for x, y in zip(*out):
        assert np.array_equal(x, y)
    close = lambda x, y: np.linalg.norm(x - y) <= 1e-11 * max(np.linalg.norm(y), 1.0)
    for e in range(nel):
        k, (aii, bi, xs, xb) = kin[e, :, :n], [v[e] for v in out[1]]
        x = np.linalg.solve(k[ni:, ni:], np.column_stack([k[ni:, :ni], b[e, ni:]]))
        assert close(aii, k[:ni, :ni] - k[:ni, ni:] @ x[:, :ni]) and close(bi, b[e, :ni] - k[:ni, ni:] @ x[:, ni]), e
        assert close(xs, x[:, :ni].T) and close(xb, x[:, ni]), e
