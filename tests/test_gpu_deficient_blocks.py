"""Plain method, more than 1024 rows and columns, on tensors whose blocks are exactly rank
deficient and not zero: constant, constant in blocks, a few entries, zero outside a box. Their
zeros and repeated entries survive FP32 products exactly, so a CholeskyQR pass meets a pivot that
is not positive and the block iteration is repeated with TSQR."""
import ctypes

import numpy as np
import pytest

import ht_tensor_learning_using_gpu_tensor_cores_amd as ht
from ht_tensor_learning_using_gpu_tensor_cores_amd import _lib
from oracle import ht_oracle as O

pytestmark = pytest.mark.gpu


def tensor(kind, n, rng):
    x = np.zeros((n,) * 4, np.float32)
    if kind == "const":
        x[:] = 3.0
    elif kind == "blocks":
        for m in range(4):
            x += rng.integers(-3, 4, 3)[np.arange(n) * 3 // n].reshape([n if a == m else 1 for a in range(4)])
    elif kind == "sparse":
        for _ in range(5):
            x[tuple(rng.integers(0, n, 4))] = rng.standard_normal()
    else:  # zero outside a box of `kind` entries a side
        x[(slice(0, kind),) * 4] = rng.standard_normal((kind,) * 4)
    return x.reshape(-1, order="F")


# Every HT rank of these tensors is below k, so the error is FP32 rounding: 2e-6 on it and on the
# bases' orthonormality, as for the other blocks of this size. (k = 33: Jacobi for the projected
# problem, blocks of 64.)
@pytest.mark.parametrize("n,k", [(33, 8), (34, 16), (34, 33)])
@pytest.mark.parametrize("kind", ["const", "blocks", "sparse", 2])
def test_plain_deficient(n, k, kind):
    import torch
    x = tensor(kind, n, np.random.default_rng(n + k))
    dims, tr, ranks = [n] * 4, ht.tree.balanced_4d(), [1, k, k] + [min(k, n)] * 4
    print(f"plain {n}^4 k={k} {kind}", flush=True)
    with ht.Handle(0) as h:
        xd = torch.from_numpy(x).cuda()
        a = ht.decompose(xd, dims, tr, ranks, method="plain", precision="fp32", handle=h)
        r = ht.reconstruct(a, handle=h).cpu().numpy().reshape(-1)
    assert a.rel_err <= 2e-6, a.rel_err
    assert np.linalg.norm(r - x) <= 4e-6 * np.linalg.norm(x)
    for t in range(tr.n_nodes):
        if tr.is_leaf(t):
            u = a.U[t].cpu().numpy().astype(np.float64)
            np.testing.assert_allclose(u.T @ u, np.eye(u.shape[1]), atol=2e-6)


# A box of 4 a side has interior rank 16, above k = 8: the truncation is the oracle's.
def test_plain_padded_truncated():
    import torch
    n, k = 33, 8
    x = tensor(4, n, np.random.default_rng(5))
    dims, tr, ranks = [n] * 4, ht.tree.balanced_4d(), [1, k, k, k, k, k, k]
    ref = O.rel_error(x, O.plain_ht(x, dims, O.Tree(tr.lo, tr.hi, tr.left, tr.right), ranks).reconstruct())
    a = ht.decompose(torch.from_numpy(x).cuda(), dims, tr, ranks, method="plain", precision="fp32")
    assert abs(a.rel_err - ref) <= 2e-6, (a.rel_err, ref)


# Blocks with a pivot that fails in the second pass: TSQR gives the basis, orthonormal whatever
# the columns, and Y lies in its span. 4e-6 as for every orthonormalisation here.
@pytest.mark.parametrize("m,b", [(1089, 16), (1089, 24), (2000, 33), (2000, 64)])
@pytest.mark.parametrize("kind", ["few", "repeated"])
def test_tall_orth_deficient(lib, handle, rng, m, b, kind):
    import torch
    Y = np.zeros((m, b), np.float32)
    if kind == "few":  # four rows hold it
        Y[:4] = rng.standard_normal((4, b))
    else:  # integers in three distinct rows
        Y[:] = rng.integers(-3, 4, (3, b))[np.arange(m) * 3 // m]
    Yd = torch.from_numpy(np.ascontiguousarray(Y.T)).cuda()
    Q = torch.empty_like(Yd)
    fb = ctypes.c_int32(-1)
    torch.cuda.synchronize()
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    print(f"tall_orth {kind} {m} x {b}", flush=True)
    _lib.check(lib.ht_tall_orth(handle.ptr, p(Yd), m, b, p(Q), ctypes.byref(fb)), "tall_orth")
    torch.cuda.synchronize()
    assert fb.value == 1
    q = Q.cpu().numpy().T.astype(np.float64)
    np.testing.assert_allclose(q.T @ q, np.eye(b), atol=4e-6)
    y = Y.astype(np.float64)
    assert np.linalg.norm(y - q @ (q.T @ y)) <= 4e-6 * np.linalg.norm(y)
