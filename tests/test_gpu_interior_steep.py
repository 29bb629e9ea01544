"""Interior spectra of the leaves-to-root method that fall by decades within the rank: the small
pairs, below the common residual test, decide the truncation error."""
import numpy as np
import pytest

import ht_tensor_learning_using_gpu_tensor_cores_amd as ht
from test_gpu_interior import core_matrix

pytestmark = pytest.mark.gpu


def reference_error(X, Xg, n, r, k):
    """Relative error in float64; Xg is X as the first two leaves' Grams read it."""
    top = lambda A, k: np.linalg.svd(A, full_matrices=False)[0][:, :k]
    unf = lambda T, m: np.moveaxis(T, m, 0).reshape(T.shape[m], -1)
    U = [top(unf(Xg, m), r) for m in (0, 1)]
    Z = np.einsum("abcd,ai,bj->ijcd", X, *U, optimize=True)
    U += [top(unf(Z, m), r) for m in (2, 3)]
    C = np.einsum("ijcd,ck,dl->ijkl", Z, U[2], U[3], optimize=True).reshape(r * r, r * r, order="F")
    P, Q = top(C, k), top(C.T, k)
    W = (P @ (P.T @ C @ Q) @ Q.T).reshape([r] * 4, order="F")
    return np.linalg.norm(X - np.einsum("abcd,ia,jb,kc,ld->ijkl", W, *U, optimize=True)) / np.linalg.norm(X)


# Spectrum i^-3, 144 and 256 rows: theta_k is 3e-7 and 6e-8 of theta_1, the reference errors 8e-4
# and 4e-4. A pair with a residual of 1e-4 theta_i loses 1e-8 of its energy; what is left is the
# FP32 rounding of the factors, 6e-8 of ||X||: 1e-7.
@pytest.mark.parametrize("n,r,k", [(24, 12, 12), (32, 16, 16)])
@pytest.mark.parametrize("precision", ["fp32", "bf16"])
def test_steep_spectra(n, r, k, precision):
    import torch
    rng = np.random.default_rng(r)
    C = core_matrix("steep", r * r, rng)
    U = [np.linalg.qr(rng.standard_normal((n, r)))[0] for _ in range(4)]
    x = (np.kron(U[1], U[0]) @ C @ np.kron(U[3], U[2]).T).reshape(-1, order="F")
    x += 1e-5 * np.linalg.norm(x) / np.sqrt(x.size) * rng.standard_normal(x.size)
    x = x.astype(np.float32)
    X = x.astype(np.float64).reshape([n] * 4, order="F")
    Xg = torch.from_numpy(x).bfloat16().double().numpy().reshape([n] * 4, order="F") if precision == "bf16" else X
    ref = reference_error(X, Xg, n, r, k)
    a = ht.decompose(torch.from_numpy(x).cuda(), [n] * 4, ht.tree.balanced_4d(), [1, k, k, r, r, r, r], method="ltr",
                     precision=precision)
    print(f"steep {r * r} rows, {precision}: {a.rel_err:.8e}, reference {ref:.8e}", flush=True)
    assert abs(a.rel_err - ref) <= 1e-7, (a.rel_err, ref)
    for t in (1, 2):
        B = a.B[t].cpu().numpy().astype(np.float64).reshape(-1, k, order="F")
        np.testing.assert_allclose(B.T @ B, np.eye(k), atol=2e-6)
