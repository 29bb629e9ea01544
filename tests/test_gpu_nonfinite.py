"""Eigen solvers on matrices that hold NaN or Inf: the Jacobi's order of the eigenvalues stays a
permutation (its entries address LDS), so such a problem ends like any other, says NaN, and
leaves its neighbours in a launch alone."""
import ctypes

import numpy as np
import pytest

import ht_tensor_learning_using_gpu_tensor_cores_amd as ht
from ht_tensor_learning_using_gpu_tensor_cores_amd import _lib

pytestmark = pytest.mark.gpu


# k <= 32: tridiagonal solver, refused, then Jacobi in the same kernel (n <= 32) or in its own;
# k > 32: Jacobi at once.
@pytest.mark.parametrize("n,k", [(1, 1), (5, 3), (16, 16), (17, 4), (32, 32), (33, 8), (64, 32), (64, 40)])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("everywhere", [False, True])
def test_topk_nonfinite(lib, handle, rng, n, k, bad, everywhere):
    import torch
    G = rng.standard_normal((n, n))
    G = G @ G.T
    if everywhere:
        G[:] = bad
    else:  # a row and a column, as one bad entry of X leaves its Gram
        G[n // 2, :] = G[:, n // 2] = bad
    U = torch.zeros(n * k, dtype=torch.float64, device="cuda")
    w = torch.zeros(k, dtype=torch.float64, device="cuda")
    it = ctypes.c_int32()
    Gd = torch.from_numpy(G).cuda()
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    print(f"topk n={n} k={k} {bad} {everywhere}", flush=True)
    _lib.check(lib.ht_sym_topk(handle.ptr, p(Gd), n, k, 1e-10, p(U), p(w), ctypes.byref(it)), "topk")
    assert not np.isfinite(w.cpu().numpy()[0])


# (10 tensors: one launch for every size class; 400: a launch for each)
@pytest.mark.parametrize("count", [10, 400])
def test_batch_nonfinite_member(count):
    import torch
    dims, core = ht.batch_shapes(count, 7)
    batch = ht.generate_batch(dims, core, 7, 1e-3)
    ranks = ht.batch_ranks(core)
    ref, err, _ = ht.decompose_batched(batch, ranks)
    bad = [1, count // 2, count - 1]
    for b, v in zip(bad, (float("nan"), float("inf"), float("nan"))):
        batch.member(b)[3] = v
    print(f"batch of {count}, members {bad} not finite", flush=True)
    res, err2, _ = ht.decompose_batched(batch, ranks)
    for b in range(count):
        if b not in bad:
            assert err2[b] == err[b] and torch.equal(res[b].packed, ref[b].packed), b
