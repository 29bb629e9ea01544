"""Top-k of diagonal matrices of up to 64 rows: unit vectors in descending order, ties by index,
exactly, as a Jacobi solve without a rotation returns them."""
import ctypes

import numpy as np
import pytest

from ht_tensor_learning_using_gpu_tensor_cores_amd import _lib

pytestmark = pytest.mark.gpu


# both kernels (32 rows and less, more), full waves and not, all pairs and one
@pytest.mark.parametrize("n,k", [(1, 1), (7, 7), (16, 16), (31, 5), (32, 32), (33, 32), (63, 1), (64, 32)])
@pytest.mark.parametrize("kind", ["equal", "zero", "two", "mixed"])
def test_topk_diagonal(lib, handle, rng, n, k, kind):
    import torch
    d = {"equal": np.full(n, 2.5), "zero": np.zeros(n), "two": np.where(np.arange(n) % 2, 3.0, 1.0),
         "mixed": np.round(4 * rng.standard_normal(n)) / 4}[kind]
    U = torch.full((n * k,), 7.0, dtype=torch.float64, device="cuda")
    w = torch.full((k,), 7.0, dtype=torch.float64, device="cuda")
    it = ctypes.c_int32()
    Gd = torch.from_numpy(np.diag(d)).cuda()
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    _lib.check(lib.ht_sym_topk(handle.ptr, p(Gd), n, k, 1e-10, p(U), p(w), ctypes.byref(it)), "topk")
    order = np.argsort(-d, kind="stable")[:k]
    np.testing.assert_array_equal(w.cpu().numpy(), d[order])
    np.testing.assert_array_equal(U.cpu().numpy().reshape((n, k), order="F"), np.eye(n)[:, order])
