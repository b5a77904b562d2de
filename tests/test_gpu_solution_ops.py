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
