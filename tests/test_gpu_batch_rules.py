"""Batched HT at the edges of its launch rules: a tensor's result does not depend on the handle, on
what was timed before, or (beyond rounding) on the number of tensors beside it."""
import numpy as np
import pytest

import ht_tensor_learning_using_gpu_tensor_cores_amd as ht

pytestmark = pytest.mark.gpu


def batch(dims, seed):
    import torch
    rng = np.random.default_rng(seed)
    offs = np.concatenate([[0], np.cumsum(dims.prod(1))]).astype(np.int64)
    return rng.standard_normal(offs[-1]).astype(np.float32), offs, torch


# 8 tensors: eight waves a projection; 511 and 512: the last with eight, the first with four; 1024:
# a wave per whole Gram. FP64 sums in another order, FP32 Grams in the same one: the factors are
# the same to FP32 rounding (2e-6, as for every batched comparison of factors against factors).
@pytest.mark.parametrize("count", [511, 512, 1024])
def test_same_in_larger_batch(count):
    few = np.array([[5, 7, 9], [16, 12, 17], [20, 16, 8], [12, 12, 12], [3, 24, 5], [9, 33, 4], [18, 2, 15], [16, 16, 16]])
    core = np.array([[2, 2, 3], [4, 3, 4], [5, 4, 2], [3, 3, 3], [2, 4, 2], [3, 5, 2], [3, 2, 4], [4, 4, 4]], np.int32)
    x, offs, torch = batch(few, 3)
    ranks = np.ascontiguousarray(ht.batch_ranks(core))
    xd = torch.from_numpy(x).cuda()
    ref, err, _ = ht.decompose_batched(ht.Batch(few.astype(np.int64), xd, offs[:-1]), ranks)
    pick = np.arange(count) % 8
    big = ht.Batch(few[pick].astype(np.int64), xd, offs[:-1][pick])  # members may share their data
    res, err2, _ = ht.decompose_batched(big, np.ascontiguousarray(ranks[pick]))
    for b in range(count):
        assert abs(err2[b] - err[b % 8]) <= 1e-9, b
        np.testing.assert_allclose(res[b].packed.cpu().numpy(), ref[b % 8].packed.cpu().numpy(), rtol=2e-6, atol=2e-6)


@pytest.mark.parametrize("count", [3, 40])
def test_same_in_every_handle(count):
    dims, core = ht.batch_shapes(count, 21)
    b = ht.generate_batch(dims, core, 21, 1e-3)
    ranks = ht.batch_ranks(core)
    first = None
    for _ in range(4):
        with ht.Handle(0) as h:
            for _ in range(3):  # launched, captured, replayed
                res, err, _ = ht.decompose_batched(b, ranks, handle=h)
                got = res[0].packed._base.cpu().numpy().copy()
                if first is None:
                    first = got, err
                assert np.array_equal(got, first[0]) and np.array_equal(err, first[1])


# Eigen problems of every size class, one launch for all (341 tensors) and a launch for each (342);
# without the two long classes the line is at 170. The classes differ in threads a problem, so in
# the order of the convergence test's sums: a sweep more or less, 1e-14 of the values.
@pytest.mark.parametrize("sizes,low,high", [((16, 30, 40, 64), 341, 342), ((5, 16, 24, 32), 170, 171)])
def test_eigen_launches(sizes, low, high):
    import torch
    rng = np.random.default_rng(9)
    shapes = np.array([[sizes[i], sizes[(i + 1) % 4], sizes[(i + 2) % 4]] for i in range(4)], dtype=np.int64)
    core = np.full((4, 3), 4, np.int32)
    offs = np.concatenate([[0], np.cumsum(shapes.prod(1))]).astype(np.int64)
    xd = torch.from_numpy(rng.standard_normal(offs[-1]).astype(np.float32)).cuda()
    got = []
    for count in (low, high):
        pick = np.arange(count) % 4
        res, err, _ = ht.decompose_batched(ht.Batch(shapes[pick], xd, offs[:-1][pick]),
                                           np.ascontiguousarray(ht.batch_ranks(core)[pick]))
        for b in range(4, count):
            assert err[b] == err[b % 4] and torch.equal(res[b].packed, res[b % 4].packed), b
        got.append(([r.packed.cpu().numpy() for r in res[:4]], err[:4]))
    for b in range(4):
        np.testing.assert_allclose(got[1][0][b], got[0][0][b], rtol=2e-6, atol=2e-6)
        assert abs(got[1][1][b] - got[0][1][b]) <= 1e-9
