"""The data pass of a fit (means, centring, variance, weights in one chain of launches) against fp64."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# rows beyond the one-launch sums (64), either side of a workgroup's stretch of a row (16 KB) and of the cap on
# workgroups, columns that leave values behind the last 128-bit load
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,d", [(1, 1), (3, 2), (257, 65), (4_096, 3), (4_099, 7), (70_001, 30), (20_000, 900), (300_002, 64)])
@pytest.mark.parametrize("copy_x", [True, False])
def test_centring_variance_and_weights(cuda, n, d, dtype, copy_x):
    import torch

    from sklearn_numba_dpex_amd.kmeans import drivers

    rng = np.random.default_rng(n + d)
    X = (rng.standard_normal((d, n)) + rng.uniform(-9, 9, (d, 1))).astype(dtype)
    w = rng.uniform(0.5, 1.5, n).astype(dtype)
    init = rng.standard_normal((d, 3)).astype(dtype)
    X_t, init_t = torch.as_tensor(X, device=cuda), torch.as_tensor(init, device=cuda)
    out, mean, init_out, tol, uniform = drivers.prepare_data_for_lloyd(X_t, init_t, 2.0, torch.as_tensor(w, device=cuda), copy_x)
    eps = np.finfo(dtype).eps
    exact = X.astype(np.float64).mean(axis=1)
    got = mean.cpu().numpy()
    # one rounding of the sum, one of the quotient (fp64: of the additions too)
    assert (np.abs(got - exact) <= 2 * eps * np.abs(exact) + 1e-14 * np.abs(X).max()).all()
    np.testing.assert_array_equal(out.cpu().numpy(), X - got[:, None])
    assert (out.data_ptr() == X_t.data_ptr()) == (not copy_x)
    if copy_x:
        np.testing.assert_array_equal(X_t.cpu().numpy(), X)
    np.testing.assert_array_equal(init_out.cpu().numpy(), init - got[:, None])
    assert tol == pytest.approx(2.0 * ((X - got[:, None]).astype(np.float64) ** 2).mean(), rel=2 * eps + 1e-13, abs=1e-30)
    assert uniform == (n == 1)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_means_of_zero_leave_the_data_alone(cuda, dtype):
    import torch

    from sklearn_numba_dpex_amd.kmeans import drivers

    half = np.random.default_rng(2).standard_normal((5, 301)).astype(dtype)
    X_t = torch.as_tensor(np.concatenate([half, -half], axis=1), device=cuda)
    before = X_t.cpu().numpy().copy()
    ones = torch.full((602,), 0.25, dtype=X_t.dtype, device=cuda)
    for copy_x in (True, False):
        out, mean, init, tol, uniform = drivers.prepare_data_for_lloyd(X_t, "random", 1.0, ones, copy_x)
        if mean is None:  # (the order of the additions decides whether opposite values cancel)
            assert out.data_ptr() == X_t.data_ptr() and uniform and init == "random"
            np.testing.assert_array_equal(out.cpu().numpy(), before)
            assert tol == pytest.approx((before.astype(np.float64) ** 2).mean(), rel=1e-6)
    zeros = torch.zeros((3, 77), dtype=X_t.dtype, device=cuda)
    assert drivers.prepare_data_for_lloyd(zeros, "random", 1.0, ones[:77].contiguous(), False)[1] is None
    # weights of another type or length than the data's are looked at by themselves
    assert drivers.prepare_data_for_lloyd(zeros, "random", 1.0, torch.ones(77, dtype=torch.float64, device=cuda).float(), True)[4]
