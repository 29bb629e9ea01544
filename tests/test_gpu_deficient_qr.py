"""QR and eigen solvers on blocks of which a few rows are not zero: every further column is
exactly dependent, and what rounding leaves of it falls by 1e-16 from one to the next, down to the
subnormal numbers."""
import ctypes

import numpy as np
import pytest

from ht_tensor_learning_using_gpu_tensor_cores_amd import _lib

pytestmark = pytest.mark.gpu


def ptr(t):
    return ctypes.c_void_p(t.data_ptr())


# One leaf (m <= 4 b), one tree level and two. 4e-6 as for every orthonormalisation here; the
# product Q R is Y to FP32 rounding of entries below 4.
@pytest.mark.parametrize("m,b", [(100, 32), (1156, 24), (1156, 32), (1156, 64), (5000, 64)])
def test_tsqr_deficient(lib, handle, m, b):
    import torch
    for seed in range(24):
        rng = np.random.default_rng(seed)
        r = 1 + seed % 6
        Y = np.zeros((m, b), np.float32)
        Y[rng.choice(min(m, 3 * b), r, replace=False)] = rng.standard_normal((r, b))
        W = torch.from_numpy(np.ascontiguousarray(Y.T)).cuda()
        Q = torch.empty_like(W)
        R = torch.empty(b, b, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        _lib.check(lib.ht_tsqr(handle.ptr, ptr(W), m, b, ptr(Q), ptr(R)), "tsqr")
        q, r64 = Q.cpu().numpy().T.astype(np.float64), R.cpu().numpy().T
        np.testing.assert_allclose(q.T @ q, np.eye(b), atol=4e-6, err_msg=str(seed))
        np.testing.assert_allclose(q @ r64, Y, atol=1e-5, err_msg=str(seed))


# 65 to 256 rows: powers of the block, Householder QR, Rayleigh-Ritz; 64 rows, more than 32
# pairs: Jacobi of the matrix. Blocks of 48 columns and more leave Jacobi entries down to the
# subnormal numbers. Tolerances of the top-k tests: values to 1e-10 of the largest (the solver's
# own), orthonormal to 1e-10.
@pytest.mark.parametrize("n,k", [(64, 40), (65, 16), (96, 64), (100, 32), (127, 63), (128, 64), (200, 24), (256, 32)])
def test_topk_deficient(lib, handle, n, k):
    import torch
    for seed in range(24):
        rng = np.random.default_rng(seed)
        r = 1 + seed % 6
        o, A = rng.integers(0, n - r), rng.standard_normal((r, r))
        G = np.zeros((n, n))
        G[o:o + r, o:o + r] = A @ A.T
        U = torch.zeros(n * k, dtype=torch.float64, device="cuda")
        w = torch.zeros(k, dtype=torch.float64, device="cuda")
        it = ctypes.c_int32()
        Gd = torch.from_numpy(G).cuda()
        torch.cuda.synchronize()
        _lib.check(lib.ht_sym_topk(handle.ptr, ptr(Gd), n, k, 1e-10, ptr(U), ptr(w), ctypes.byref(it)), f"seed {seed}")
        u, lam = U.cpu().numpy().reshape((n, k), order="F"), np.linalg.eigvalsh(G)[::-1][:k]
        np.testing.assert_allclose(w.cpu().numpy(), lam, atol=1e-10 * lam[0], rtol=0, err_msg=str(seed))
        np.testing.assert_allclose(u.T @ u, np.eye(k), atol=1e-10, err_msg=str(seed))
