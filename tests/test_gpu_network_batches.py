"""GPU checks of the network's batch kernels where their work split changes.

  forward   the small-batch kernel (32 rows per workgroup) and the one for large batches give the same
            bits for every row: predictions of a large batch against the same rows in small batches
            around the 16- and 32-row tiles and at the size where the rule switches
  backward  more than 1024 groups of 64 rows (a workgroup then takes several and adds to its gradient):
            the gradient of 2 m rows is the mean of the gradients of its halves. The factor 1/n of dZ
            halves exactly, so only the FP32 sums differ, in order: at most 2048 additions of relative
            error 2^-24 each, 1.3e-4 in the worst case, relative L2 1e-5 for their random part
  tail      rows past the batch's end contribute nothing: the gradient of 65 rows is the mean of that
            of 64 rows (weight 64) and of the last one, within the BF16 rounding of dZ (2^-8)
"""
import numpy as np
import pytest

from anisotropicelastoplasticity_amd import Solver

pytestmark = pytest.mark.gpu


def pairs(n, seed):
    g = np.random.default_rng(seed)
    eps = -np.sort(-g.normal(size=(n, 3)) * 0.01, axis=1)
    x = np.concatenate([eps, g.uniform(25, 40, (n, 1)), g.uniform(1.5, 3.0, (n, 1))], axis=1).astype(np.float32)
    return x, (x[:, :3] + 1e-3 * g.normal(size=(n, 3))).astype(np.float32)


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 31, 32, 33, 64, 2048, 16384, 16385])
def test_forward_kernels_agree(rows):
    x, _ = pairs(40000, 3)
    with Solver(0) as s:
        s.surrogate_init(5)
        whole = s.surrogate_predict(x)
        part = s.surrogate_predict(x[:rows])
    print("rows", rows, flush=True)
    assert np.array_equal(part, whole[:rows])


def test_gradient_of_many_groups():
    m = 65536
    x, H = pairs(2 * m, 4)
    with Solver(0) as s:
        s.surrogate_init(6)
        g, loss = s.surrogate_gradient(x, H)
        a, la = s.surrogate_gradient(x[:m], H[:m])
        b, lb = s.surrogate_gradient(x[m:], H[m:])
    mean = 0.5 * (a.astype(np.float64) + b)
    err = np.linalg.norm(g - mean) / np.linalg.norm(mean)
    print("relative L2", err, "loss", loss, 0.5 * (la + lb), flush=True)
    assert err <= 1e-5 and abs(loss - 0.5 * (la + lb)) <= 1e-5 * loss


def test_gradient_tail_rows():
    x, H = pairs(65, 7)
    with Solver(0) as s:
        s.surrogate_init(8)
        g, _ = s.surrogate_gradient(x, H)
        a, _ = s.surrogate_gradient(x[:64], H[:64])
        b, _ = s.surrogate_gradient(x[64:], H[64:])
    mean = (64 * a.astype(np.float64) + b) / 65
    assert np.linalg.norm(g - mean) / np.linalg.norm(mean) <= 2.0 ** -8
