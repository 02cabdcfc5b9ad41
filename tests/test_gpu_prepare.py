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


@pytest.mark.parametrize("rows,cols", [(1, 1), (2, 70_001), (14, 1_000_003), (900, 20_000), (1_500, 40)])
def test_centring_stays_within_its_workspace(cuda, rows, cols):
    import torch

    from sklearn_numba_dpex_amd import _capi
    from sklearn_numba_dpex_amd._capi import lib, ptr

    X_t = torch.randn((rows, cols), device=cuda, dtype=torch.float64) + 3
    w, mean, stats = torch.ones(cols, device=cuda, dtype=X_t.dtype), X_t.new_empty(rows), X_t.new_empty(4)
    out, size = torch.empty_like(X_t), lib.kmx_center_workspace_bytes(rows, cols)
    ws = torch.full((size + 4096,), 0x5A, dtype=torch.uint8, device=cuda)
    args = (rows, cols, _capi.KMX_F64, _capi.current_stream())
    assert lib.kmx_center_rows(ptr(X_t), ptr(out), ptr(w), ptr(mean), ptr(stats), ptr(ws), size - 1, *args) != 0
    _capi.check(lib.kmx_center_rows(ptr(X_t), ptr(out), ptr(w), ptr(mean), ptr(stats), ptr(ws), size, *args), "kmx_center_rows")
    assert bool((ws[size:] == 0x5A).all())
    torch.testing.assert_close(mean, X_t.mean(1), rtol=1e-12, atol=1e-13)
    torch.testing.assert_close(out, X_t - mean[:, None], rtol=0, atol=0)
    assert float(stats[2]) == cols and float(stats[3]) == 1
    torch.testing.assert_close(stats[1], (out * out).sum(), rtol=1e-11, atol=1e-300)


# memory for the centred copy is asked for ahead of the means; means of zero do without it
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_means_of_zero_need_no_memory_for_a_copy(cuda, dtype, monkeypatch):
    import torch

    from sklearn_numba_dpex_amd.kmeans import drivers

    X_t = torch.as_tensor(np.tile(np.array([[3, -3], [1, -1]], dtype=dtype), (1, 100)), device=cuda)
    before, ones = X_t.clone(), torch.ones(200, dtype=X_t.dtype, device=cuda)

    def none_left(*args, **kwargs):
        raise torch.OutOfMemoryError("no memory for a copy")

    monkeypatch.setattr(torch, "empty_like", none_left)
    out, mean, _, tol, uniform = drivers.prepare_data_for_lloyd(X_t, "random", 1.0, ones, True)
    assert mean is None and out.data_ptr() == X_t.data_ptr() and torch.equal(X_t, before) and tol == 5.0 and uniform
    with pytest.raises(torch.OutOfMemoryError):
        drivers.prepare_data_for_lloyd(X_t + 1, "random", 1.0, ones, True)


@pytest.mark.parametrize("copy_x", [True, False])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_means_of_zero_leave_the_data_alone(cuda, dtype, copy_x):
    import torch

    from sklearn_numba_dpex_amd.kmeans import drivers

    # small whole numbers: the sums are exact in any order
    half = np.random.default_rng(2).integers(-9, 10, (5, 301)).astype(dtype)
    X_t = torch.as_tensor(np.concatenate([half, -half], axis=1), device=cuda)
    before = X_t.cpu().numpy().copy()
    ones = torch.full((602,), 0.25, dtype=X_t.dtype, device=cuda)
    out, mean, init, tol, uniform = drivers.prepare_data_for_lloyd(X_t, "random", 1.0, ones, copy_x)
    assert mean is None and out.data_ptr() == X_t.data_ptr() and uniform and init == "random"
    np.testing.assert_array_equal(X_t.cpu().numpy(), before)
    assert tol == pytest.approx((before.astype(np.float64) ** 2).mean(), rel=1e-6)


@pytest.mark.parametrize("dtype,other", [(np.float32, np.float64), (np.float64, np.float32)])
def test_weights_of_another_type_or_length_are_looked_at_by_themselves(cuda, dtype, other):
    import torch

    from sklearn_numba_dpex_amd.kmeans import drivers

    X_t = torch.as_tensor(np.random.default_rng(3).standard_normal((3, 77)).astype(dtype), device=cuda)
    same = drivers.prepare_data_for_lloyd(X_t, "random", 1.0, torch.ones(77, dtype=X_t.dtype, device=cuda), True)
    for weights, uniform in ((np.full(77, 0.5), True), (np.arange(1.0, 78.0), False), (np.arange(1.0, 6.0), False)):
        for w in (weights.astype(other), weights.astype(dtype)):
            got = drivers.prepare_data_for_lloyd(X_t, "random", 1.0, torch.as_tensor(w, device=cuda), True)
            assert got[4] == uniform and got[3] == same[3]
            assert torch.equal(got[0], same[0]) and torch.equal(got[1], same[1])
