"""First round of the interior eigen problems where the spectrum ends between the wanted rank and
the block's width (32): the powers of the whole block converge in one round."""
import numpy as np
import pytest

import ht_tensor_learning_using_gpu_tensor_cores_amd as ht

pytestmark = pytest.mark.gpu


# 8 values at 6 pairs and 25 at 8, 12 and 16; 24 powers and the Rayleigh-Ritz product are 25
# products with G, a second round adds its own.
@pytest.mark.parametrize("n,r,k,values", [(32, 16, 6, 8), (20, 9, 8, 25), (24, 12, 12, 25), (32, 16, 16, 25)])
@pytest.mark.parametrize("precision", ["fp32", "bf16"])
def test_one_round(n, r, k, values, precision):
    import torch
    rng = np.random.default_rng(r)
    m = r * r
    s = np.where(np.arange(m) < values, 1.0 - 0.4 * np.arange(m) / values, 0.0)
    C = (np.linalg.qr(rng.standard_normal((m, m)))[0] * s) @ np.linalg.qr(rng.standard_normal((m, m)))[0].T
    U = [np.linalg.qr(rng.standard_normal((n, r)))[0] for _ in range(4)]
    x = (np.kron(U[1], U[0]) @ C @ np.kron(U[3], U[2]).T).reshape(-1, order="F")
    x += 1e-5 * np.linalg.norm(x) / np.sqrt(x.size) * rng.standard_normal(x.size)
    a = ht.decompose(torch.from_numpy(x.astype(np.float32)).cuda(), [n] * 4, ht.tree.balanced_4d(),
                     [1, k, k, r, r, r, r], method="ltr", precision=precision)
    # the noise (1e-5 of ||x||) and the leaves' tilt (1e-4) add in second order
    ref = np.sqrt(np.sum(s[k:] ** 2) / np.sum(s ** 2))
    assert abs(a.rel_err - ref) <= 1e-6, (a.rel_err, ref)
    assert a.stats["eig_iters_max"] == 25, a.stats
