"""GPU parity of the shared kernels (sums, argmin, top-k, elementwise, matmul, label helpers),
restating the reference's common/tests and kmeans/tests cases against numpy."""

import numpy as np
import pytest

from oracle import kmeans as ok

pytestmark = pytest.mark.gpu

DTYPES = [np.float32, np.float64]


def _dev(a, cuda):
    import torch

    return torch.as_tensor(np.ascontiguousarray(a), device=cuda)


# reference common/tests/test_reductions.py:16-68
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("axis", [0, 1])
@pytest.mark.parametrize("shape", [(1, 1), (1, 3), (3, 1), (3, 5), (5, 3), (3, 4), (4, 3), (3, 9), (7, 20011)])
def test_sum_reduction_2d(cuda, shape, axis, dtype):
    from sklearn_numba_dpex_amd.common.reductions import sum_reduction

    a = np.arange(shape[0] * shape[1], dtype=dtype).reshape(shape) % 1000
    got = sum_reduction(_dev(a, cuda), axis=axis).cpu().numpy()
    np.testing.assert_allclose(got, a.sum(axis=axis, dtype=np.float64), rtol=1e-6)


@pytest.mark.parametrize("dtype", DTYPES)
def test_sum_reduction_1d_square_and_determinism(cuda, dtype):
    from sklearn_numba_dpex_amd.common.reductions import sum_reduction

    for length, expected in [(4, 6), (5, 10)]:
        assert sum_reduction(_dev(np.arange(length, dtype=dtype), cuda)).cpu().numpy()[0] == pytest.approx(expected)
    rng = np.random.default_rng(0)
    v = rng.normal(size=3_000_017).astype(dtype)
    d = _dev(v, cuda)
    s1 = sum_reduction(d, square=True).cpu().numpy()[0]
    s2 = sum_reduction(d, square=True).cpu().numpy()[0]
    assert s1 == s2  # fixed summation order
    assert s1 == pytest.approx(float(np.sum(v.astype(np.float64) ** 2)), rel=1e-6)


# reference common/tests/test_reductions.py:109-133
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("values, expected", [([3.0, 1.0, 0.0, 2.0], 2), ([0.0, 1.0, 3.0, 2.0], 0),
                                              ([3.0, 1.0, 2.0, -1.0, -2.0], 4), ([5.0, 1.0, 1.0, 7.0], 1)])
def test_argmin(cuda, values, expected, dtype):
    import torch

    from sklearn_numba_dpex_amd.common.reductions import argmin_reduction

    out = argmin_reduction(_dev(np.array(values, dtype=dtype), cuda))
    assert out.dtype == torch.int32
    assert int(out.cpu()[0]) == expected
    rng = np.random.default_rng(1)
    big = rng.normal(size=50_000).astype(dtype)
    big[[123, 40_000]] = -100.0
    assert int(argmin_reduction(_dev(big, cuda)).cpu()[0]) == 123


TOPK_CASES = [
    [0, 1, -2, -3, 4, -5, 6, 7, 8, -9, 10],
    [0, 8, -2, -3, 4, -5, 6, 7, 8, -9, 10],
    [0, 8, -2, -3, 4, -5, 6, 7, 8, -9, 8],
    [0, 8, 8, -3, 4, -5, 6, 7, 8, -9, 10],
    [0, 8, 8, -3, 4, -5, 6, 7, 8, -9, 8],
    [8, 8, 8, 8, 8, 8, 8, 8, 8, 8, 8],
]


# reference common/tests/test_topk.py:28-59 (+ our deterministic order policy)
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("k", [1, 3, 11])
@pytest.mark.parametrize("case", range(len(TOPK_CASES)))
def test_topk_handcrafted(cuda, case, k, dtype):
    from sklearn_numba_dpex_amd.common.topk import topk, topk_idx

    a = np.array(TOPK_CASES[case], dtype=dtype)
    idx = topk_idx(_dev(a, cuda), k).cpu().numpy()
    np.testing.assert_array_equal(idx, ok.top_k_indices(a, k))  # descending value, ascending index
    np.testing.assert_array_equal(np.sort(a[idx]), np.sort(a)[-k:])
    np.testing.assert_array_equal(np.sort(topk(_dev(a, cuda), k).cpu().numpy()), np.sort(a)[-k:])


@pytest.mark.parametrize("dtype", DTYPES)
def test_topk_multirow_and_random(cuda, dtype):
    from sklearn_numba_dpex_amd.common.topk import topk, topk_idx

    a = np.array(TOPK_CASES, dtype=dtype)
    got = topk(_dev(a, cuda), 3).cpu().numpy()
    np.testing.assert_array_equal(got, -np.sort(-a, axis=1)[:, :3])  # descending
    rng = np.random.default_rng(123)
    # the reference's random case (common/tests/test_topk.py:62-80): 1000 rows of 1000 values;
    # 1001 columns here so that most rows start off a 16-byte boundary
    big = rng.normal(size=(1000, 1001)).astype(dtype)
    d_big = _dev(big, cuda)
    for k in (1, 3, 40):
        idx = topk_idx(d_big, k).cpu().numpy()
        assert idx.shape == (1000, k) and idx.dtype == np.int64
        want = np.stack([ok.top_k_indices(big[r], k) for r in range(big.shape[0])])
        np.testing.assert_array_equal(idx, want)
        vals = topk(d_big, k).cpu().numpy()
        np.testing.assert_array_equal(vals, np.take_along_axis(big, want, axis=1))


@pytest.mark.parametrize("dtype", DTYPES)
def test_topk_dense_threshold_bucket_and_signed_zeros(cuda, dtype):
    """Rows whose largest values share their leading digits: more candidates than the side
    buffer holds (all of [1, 1.25) and a constant row), a quarter-full one (uniform [0, 1)),
    and -0.0 / +0.0, which rank as equal (lowest index first)."""
    from sklearn_numba_dpex_amd.common.topk import topk, topk_idx

    rng = np.random.default_rng(77)
    n = 300_001
    rows = np.stack([
        rng.uniform(1.0, 1.25, n),
        np.full(n, 3.0),
        rng.uniform(0.0, 1.0, n),
        -rng.uniform(1.0, 1.25, n),
    ]).astype(dtype)
    d_rows = _dev(rows, cuda)
    for k in (1, 7, 2000):
        idx = topk_idx(d_rows, k).cpu().numpy()
        want = np.stack([ok.top_k_indices(rows[r], k) for r in range(rows.shape[0])])
        np.testing.assert_array_equal(idx, want)
        np.testing.assert_array_equal(topk(d_rows, k).cpu().numpy(), np.take_along_axis(rows, want, axis=1))
    z = np.array([-1.0, -0.0, 0.0, -0.0, 0.0, -2.0], dtype=dtype)
    np.testing.assert_array_equal(topk_idx(_dev(z, cuda), 3).cpu().numpy(), [1, 2, 3])
    got = topk(_dev(z, cuda), 3).cpu().numpy()
    np.testing.assert_array_equal(np.signbit(got), [True, False, True])  # the stored values, bit for bit


@pytest.mark.parametrize("dtype", DTYPES)
def test_topk_edges(cuda, dtype):
    """k = n, a single value, infinities, and more rows than one grid dimension holds."""
    from sklearn_numba_dpex_amd.common.topk import topk, topk_idx

    rng = np.random.default_rng(9)
    v = rng.normal(size=37).astype(dtype)
    np.testing.assert_array_equal(topk_idx(_dev(v, cuda), 37).cpu().numpy(), ok.top_k_indices(v, 37))
    np.testing.assert_array_equal(topk_idx(_dev(v[:1], cuda), 1).cpu().numpy(), [0])
    w = v.copy()
    w[[3, 20]] = np.inf
    w[[5, 6]] = -np.inf
    np.testing.assert_array_equal(topk_idx(_dev(w, cuda), 4).cpu().numpy(), ok.top_k_indices(w, 4))
    np.testing.assert_array_equal(topk(_dev(w, cuda), 37).cpu().numpy()[-2:], [-np.inf, -np.inf])
    many = rng.normal(size=(70_000, 5)).astype(dtype)  # 70 000 rows: two slices of the grid
    got = topk_idx(_dev(many, cuda), 2).cpu().numpy()
    want = np.argsort(-many, axis=1, kind="stable")[:, :2]
    np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("dtype", DTYPES)
def test_topk_large_with_ties_and_negatives(cuda, dtype):
    from sklearn_numba_dpex_amd.common.topk import topk_idx

    rng = np.random.default_rng(5)
    v = rng.normal(size=1_000_003).astype(dtype)
    v[rng.choice(v.size, 5000, replace=False)] = np.float32(2.5)  # many ties at the threshold
    v[::7] *= -1
    for k in (1, 16, 300):
        idx = topk_idx(_dev(v, cuda), k).cpu().numpy()
        np.testing.assert_array_equal(idx, ok.top_k_indices(v, k))
    with pytest.raises(ValueError, match="Expected k to be greater than or equal"):
        topk_idx(_dev(v[:5], cuda), 6)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n", [1, 63, 1_024, 4_097, 65_537, 262_145, 1_048_577, 4_200_003, 16_000_001])
def test_topk_of_one_row_for_small_k(cuda, dtype, n):
    """One row and k <= 64 take the path that reads the row once (per workgroup the k largest via
    the thread maxima, then one workgroup over the workgroups' results): every tier of elements
    per thread, rows that are sorted either way (all the large values in one thread or one in
    each), constant rows and rows of few distinct values (ties everywhere: lowest index first)."""
    from sklearn_numba_dpex_amd.common.topk import topk, topk_idx

    rng = np.random.default_rng(n)
    rows = {
        "random": rng.normal(size=n),
        "ascending": np.arange(n, dtype=np.float64),
        "descending": -np.arange(n, dtype=np.float64),
        "constant": np.full(n, -1.5),
        "few values": rng.integers(0, 3, n).astype(np.float64),
    }
    for name, v in rows.items():
        v = v.astype(dtype)
        d_v = _dev(v, cuda)
        for k in (1, 16, 64):
            if k > n:
                continue
            want = ok.top_k_indices(v, k)
            np.testing.assert_array_equal(topk_idx(d_v, k).cpu().numpy(), want, err_msg=f"{name}, k={k}")
        k = min(5, n)
        np.testing.assert_array_equal(topk(d_v, k).cpu().numpy(), v[ok.top_k_indices(v, k)], err_msg=name)


@pytest.mark.parametrize("dtype", DTYPES)
def test_elementwise_kernels(cuda, dtype):
    from sklearn_numba_dpex_amd.common import kernels

    rng = np.random.default_rng(2)
    a = rng.normal(size=(5, 1003)).astype(dtype)
    v_rows = rng.normal(size=5).astype(dtype)
    v_cols = rng.uniform(1, 2, 1003).astype(dtype)
    d = _dev(a, cuda)
    np.testing.assert_array_equal(kernels.half_l2_norm(d).cpu().numpy().shape, (1003,))
    np.testing.assert_allclose(kernels.half_l2_norm(d).cpu().numpy(), ok.half_sq_norms(a.T), rtol=1e-6)
    kernels.broadcast_rows(d, _dev(v_rows, cuda), "minus")
    np.testing.assert_array_equal(d.cpu().numpy(), a - v_rows[:, None])
    kernels.broadcast_rows(d, _dev(v_rows, cuda), "plus")
    np.testing.assert_allclose(d.cpu().numpy(), a, atol=1e-6)
    d = _dev(a, cuda)
    kernels.broadcast_division(d, _dev(v_cols, cuda))
    np.testing.assert_array_equal(d.cpu().numpy(), a / v_cols[None, :])
    d = _dev(a, cuda)
    kernels.divide_by(d, 7.0)
    np.testing.assert_array_equal(d.cpu().numpy(), a / dtype(7.0))
    b = rng.normal(size=(5, 1003)).astype(dtype)
    np.testing.assert_allclose(kernels.centroid_shifts(_dev(a, cuda), _dev(b, cuda)).cpu().numpy(),
                               ((a - b) ** 2).sum(axis=0), rtol=1e-6)
    kernels.initialize_to_zeros(d)
    assert float(d.abs().sum()) == 0.0


# reference common/tests/test_matmul.py:71-127
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 5, 2), (16, 16, 16), (65, 17, 130), (1999, 661, 563), (128, 4, 128),
                                   (257, 33, 129), (300, 70, 200), (1024, 256, 512)])
def test_matmul(cuda, shape, dtype):
    from sklearn_numba_dpex_amd.common.matmul import matmul

    m, p, q = shape
    rng = np.random.default_rng(0)
    X = rng.normal(size=(m, p)).astype(dtype)
    Y_t = rng.normal(size=(q, p)).astype(dtype)
    got = matmul(_dev(X, cuda), _dev(Y_t, cuda)).cpu().numpy()
    np.testing.assert_allclose(got, X.astype(np.float64) @ Y_t.astype(np.float64).T,
                               rtol=1e-4 if dtype == np.float32 else 1e-11, atol=1e-4 if dtype == np.float32 else 1e-11)


# the reference's small shapes with `arange` operands (common/tests/test_matmul.py:13-16,71-104)
@pytest.mark.parametrize("shapes", [((1, 1), (1, 1)), ((4, 4), (4, 4)), ((5, 5), (5, 5)), ((1, 4), (4, 1)),
                                    ((1, 5), (5, 1)), ((4, 1), (1, 4)), ((5, 1), (1, 5)), ((4, 5), (5, 4)),
                                    ((5, 4), (4, 5)), ((5, 4), (4, 8)), ((5, 4), (4, 10)), ((4, 5), (5, 10)),
                                    ((10, 4), (4, 5)), ((5, 10), (10, 4)), ((1999, 661), (661, 563))])
def test_matmul_arange(cuda, shapes):
    from sklearn_numba_dpex_amd.common.matmul import matmul

    (m, p), (_, q) = shapes
    X = np.arange(m * p, dtype=np.float32).reshape(m, p)
    Y = np.arange(p * q, dtype=np.float32).reshape(p, q)
    got = matmul(_dev(X, cuda), _dev(np.ascontiguousarray(Y.T), cuda)).cpu().numpy()
    np.testing.assert_allclose(got, np.matmul(X, Y), rtol=1e-5)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape", [(3, 5, 2), (65, 17, 130), (257, 33, 129), (1000, 70, 300)])
def test_matmul_fused_functions(cuda, shape, dtype):
    """multiply_fn and out_fused_elementwise_fn of make_matmul_2d_kernel (reference
    common/matmul.py:55-66) for the functions the reference predefines (common/_utils.py:17-33)."""
    from sklearn_numba_dpex_amd.common import _utils
    from sklearn_numba_dpex_amd.common.matmul import matmul

    m, p, q = shape
    rng = np.random.default_rng(3)
    X = rng.normal(size=(m, p)).astype(dtype)
    Y_t = rng.normal(size=(q, p)).astype(dtype)
    X64, Y64 = X.astype(np.float64), Y_t.astype(np.float64)
    tol = dict(rtol=1e-4, atol=1e-4) if dtype == np.float32 else dict(rtol=1e-11, atol=1e-11)
    dX, dY = _dev(X, cuda), _dev(Y_t, cuda)
    prod = X64 @ Y64.T
    np.testing.assert_allclose(matmul(dX, dY, out_fused_elementwise_fn=_utils._square).cpu().numpy(), prod**2, **tol)
    np.testing.assert_allclose(matmul(dX, dY, out_fused_elementwise_fn=_utils._divide_by(4.0)).cpu().numpy(),
                               prod / 4.0, **tol)
    minus = X64.sum(axis=1)[:, None] - Y64.sum(axis=1)[None, :]
    plus = X64.sum(axis=1)[:, None] + Y64.sum(axis=1)[None, :]
    np.testing.assert_allclose(matmul(dX, dY, multiply_fn=_utils._minus).cpu().numpy(), minus, **tol)
    np.testing.assert_allclose(matmul(dX, dY, multiply_fn=_utils._plus).cpu().numpy(), plus, **tol)
    np.testing.assert_allclose(
        matmul(dX, dY, multiply_fn=_utils._minus, out_fused_elementwise_fn=_utils._square).cpu().numpy(),
        minus**2, rtol=tol["rtol"] * 10, atol=tol["atol"] * 10)
    with pytest.raises(NotImplementedError, match="predefined functions"):
        matmul(dX, dY, multiply_fn=lambda x, y: x * y + 1)


def test_label_helpers(cuda):
    from sklearn_numba_dpex_amd.kmeans import drivers

    # reference kmeans/tests/test_kmeans.py:448-457
    labels = _dev(np.array([0, 1, 0, 2, 2, 7, 6, 5, 3, 3], dtype=np.int32), cuda)
    assert int(drivers.get_nb_distinct_clusters(labels, 8)) == 7
    rng = np.random.default_rng(0)
    a = rng.integers(0, 50, 200_000).astype(np.int32)
    perm = rng.permutation(50).astype(np.int32)
    b = perm[a]
    c = b.copy()
    c[77_777] = (c[77_777] + 1) % 50
    assert drivers.is_same_clustering(_dev(a, cuda), _dev(b, cuda), 50) is True
    assert drivers.is_same_clustering(_dev(a, cuda), _dev(c, cuda), 50) is False
    assert int(drivers.get_nb_distinct_clusters(_dev(a, cuda), 50)) == len(np.unique(a))


# either side of the clusters whose flags a workgroup keeps in LDS, vector loads with and without a
# remainder, a start off their alignment
@pytest.mark.parametrize("n,k,offset", [(1, 1, 0), (7, 3, 0), (4096 * 5 + 3, 10, 0), (100_001, 5, 1), (300_000, 32768, 0),
                                        (300_000, 32769, 0)])
def test_distinct_labels_are_counted(cuda, n, k, offset):
    from sklearn_numba_dpex_amd.kmeans import drivers

    rng = np.random.default_rng(n + k)
    kept = np.flatnonzero(rng.random(k) < 0.7) if k > 1 else np.zeros(1, dtype=np.int64)
    labels = rng.choice(kept, n + offset).astype(np.int32)
    got = drivers.get_nb_distinct_clusters(_dev(labels, cuda)[offset:], k)
    assert int(got) == len(np.unique(labels[offset:]))


# every instantiation of the distance and inertia kernels (register / tiled distances,
# centroids in LDS or not, 128-bit or scalar accesses) against numpy in fp64
@pytest.mark.parametrize("shape", [(1003, 14, 127, np.float32), (4096, 32, 7, np.float32), (777, 33, 5, np.float32),
                                   (1001, 16, 9, np.float64), (500, 17, 3, np.float64), (1000, 300, 50, np.float32),
                                   (3, 2, 2, np.float64), (1000, 70, 130, np.float64), (1028, 100, 64, np.float32),
                                   (515, 129, 67, np.float32), (1026, 48, 66, np.float64),
                                   # few clusters of wide samples: centroid tiles of 16 (one, two), then of 64
                                   (1001, 784, 10, np.float32), (1030, 200, 20, np.float64),
                                   (1000, 65, 32, np.float32), (1000, 65, 33, np.float32)])
def test_distances_and_inertia_kernels(cuda, shape):
    import torch

    from sklearn_numba_dpex_amd.kmeans import drivers

    n, d, k, dtype = shape
    rng = np.random.default_rng(n + d)
    X = rng.normal(size=(n, d)).astype(dtype)
    C = rng.normal(size=(k, d)).astype(dtype)
    w = rng.uniform(0.5, 2.0, n).astype(dtype)
    labels = rng.integers(0, k, n).astype(np.int32)
    X_t, C_t = _dev(X.T, cuda), _dev(C.T, cuda)
    rtol = 2e-5 if dtype == np.float32 else 1e-12
    exact = np.sqrt(((X.astype(np.float64)[:, None, :] - C.astype(np.float64)[None, :, :]) ** 2).sum(axis=2))
    got = drivers.get_euclidean_distances(X_t, C_t).cpu().numpy()
    assert got.shape == (n, k)
    np.testing.assert_allclose(got, exact, rtol=rtol, atol=rtol)
    per_sample = (exact[np.arange(n), labels] ** 2)
    lab_d = torch.as_tensor(labels, device=cuda)
    got_w = drivers._per_sample_inertia(X_t, _dev(w, cuda), C_t, lab_d).cpu().numpy()
    np.testing.assert_allclose(got_w, per_sample * w.astype(np.float64), rtol=rtol * 5, atol=rtol)
    # unit weights through the NULL-weights entry (what the relocation ranks samples by)
    from sklearn_numba_dpex_amd import _capi
    from sklearn_numba_dpex_amd._capi import lib, ptr

    out = torch.empty(n, dtype=X_t.dtype, device=cuda)
    _capi.check(lib.kmx_per_sample_inertia(ptr(X_t), None, ptr(C_t), ptr(lab_d), ptr(out), n, d, k,
                                           _capi.dtype_code(X.dtype), _capi.current_stream()), "inertia")
    np.testing.assert_allclose(out.cpu().numpy(), per_sample, rtol=rtol * 5, atol=rtol)
    # the same kernel with the sum folded in (no per-sample values written)
    total = drivers._inertia_array(X_t, _dev(w, cuda), C_t, lab_d)
    assert total.shape == (1,) and total.dtype == dtype
    np.testing.assert_allclose(total[0], (per_sample * w.astype(np.float64)).sum(), rtol=rtol)
    total_unit = drivers._inertia_array(X_t, None, C_t, lab_d)
    np.testing.assert_allclose(total_unit[0], per_sample.sum(), rtol=rtol)


# both layouts of X, at the edges of sample tiles (128), feature stages (32; 1 024 of the shift), centroid tiles
# (16, 32, 64) and the kernels kept per number of features
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,d,k", [(1, 1, 1), (5, 1, 5), (130, 2, 17), (1023, 5, 600), (257, 7, 9), (127, 8, 64), (128, 9, 16),
                                   (129, 15, 33), (1025, 16, 130), (4097, 16, 2100), (2049, 17, 1), (127, 31, 15),
                                   (128, 32, 16), (1153, 33, 32), (640, 36, 65), (129, 64, 64), (300, 100, 129),
                                   (200, 1023, 3), (131, 1056, 20), (70, 1500, 66), (70, 1793, 9)])
def test_distances_from_either_layout(cuda, n, d, k, dtype):
    import torch

    from sklearn_numba_dpex_amd.kmeans import drivers

    rng = np.random.default_rng(n + 7 * d + k)
    C = rng.uniform(-4, 4, (k, d)).astype(dtype)
    X = (C[rng.integers(0, k, n)] + rng.standard_normal((n, d))).astype(dtype)
    X[n // 2] = C[k // 2]  # distance exactly 0
    exact = np.sqrt(((X.astype(np.float64)[:, None, :] - C.astype(np.float64)[None, :, :]) ** 2).sum(axis=2))
    # d additions of non-negative terms, each rounded, and the root
    rtol = (d / 2 + 3) * np.finfo(dtype).eps if dtype == np.float64 or d <= 16 else 1.5 * np.finfo(dtype).eps
    not_finite = torch.empty(1, dtype=torch.int32, device=cuda)
    rows = drivers.get_euclidean_distances_rows(_dev(X, cuda), _dev(C.T, cuda), not_finite)
    assert int(not_finite) == 0
    for got in (rows, drivers.get_euclidean_distances(_dev(X.T, cuda), _dev(C.T, cuda))):
        got = got.cpu().numpy()
        assert got.shape == (n, k) and got.dtype == dtype
        np.testing.assert_allclose(got, exact, rtol=rtol)
        assert (got[exact == 0] == 0).all()
    for i, f, value in ((0, 0, np.nan), (n - 1, d - 1, np.inf), (n // 2, d // 2, -np.inf)):
        bad = X.copy()
        bad[i, f] = value
        drivers.get_euclidean_distances_rows(_dev(bad, cuda), _dev(C.T, cuda), not_finite)
        assert int(not_finite) == 1


# pairs that the inner products cannot settle: next to a centroid, far from the origin, tiny, and squares beyond
# fp32 (infinite in the difference form too)
@pytest.mark.parametrize("case", ["near", "offset", "tiny", "huge", "one far centroid"])
def test_fp32_distances_of_close_and_extreme_pairs(cuda, case):
    from sklearn_numba_dpex_amd.kmeans import drivers

    rng = np.random.default_rng(17)
    n, d, k = 700, 40, 70
    C = rng.uniform(-4, 4, (k, d))
    X = C[rng.integers(0, k, n)] + rng.standard_normal((n, d))
    if case == "near":
        X = C[rng.integers(0, k, n)] * (1 + 1e-6 * rng.standard_normal((n, d)))
    elif case == "offset":
        C, X = C + 1e6, X + 1e6
    elif case == "tiny":
        C, X = C * 1e-17, X * 1e-17
    elif case == "huge":
        C, X = C * 1e17, X * 1e17
    else:
        C[5] = 1e8
    C, X = C.astype(np.float32), X.astype(np.float32)
    exact = np.sqrt(((X.astype(np.float64)[:, None, :] - C.astype(np.float64)[None, :, :]) ** 2).sum(axis=2))
    got = drivers.get_euclidean_distances(_dev(X.T, cuda), _dev(C.T, cuda)).cpu().numpy()
    np.testing.assert_allclose(got, exact, rtol=(d / 2 + 3) * 1.2e-7)  # (redone pairs: d rounded additions)


# pairs lost against the kernel's shift, many or all of a tile's: centroids far from everything (the first of them one),
# two groups far apart (mixed, and in turn by 128 samples), an offset (the shift ends at 1 792 features), huge samples.
# 16, 32 and 64 centroids a workgroup, its operands resident (d <= 32) or not, partial tiles, several tiles a workgroup.
@pytest.mark.parametrize("case", ["far first", "far at both ends", "two groups", "groups by turns", "offset", "huge samples"])
@pytest.mark.parametrize("n,d,k", [(1, 17, 1), (129, 20, 16), (300, 32, 31), (257, 100, 64), (700, 40, 70), (131, 1900, 5),
                                   (200_003, 24, 20), (130_001, 33, 40)])
def test_fp32_distances_far_from_the_shift(cuda, n, d, k, case):
    import torch

    from sklearn_numba_dpex_amd.kmeans import drivers

    gen = torch.Generator(device=cuda).manual_seed(n + k)
    C = torch.rand(k, d, generator=gen, device=cuda) * 8 - 4
    lab = torch.randint(0, k, (n,), generator=gen, device=cuda)
    if case == "far first":
        C[0] = 1e6
    elif case == "far at both ends":
        C[0], C[-1] = 1e6, -2e6
    elif case in ("two groups", "groups by turns"):
        C[: (k + 1) // 2] += 1e6
        if case == "groups by turns":
            lab = torch.where(torch.arange(n, device=cuda) // 128 % 3 == 1, 0, k - 1)
    elif case == "offset":
        C += 1e5
    X = C[lab] + torch.randn(n, d, generator=gen, device=cuda)
    if case == "huge samples":
        X[::3] *= (1.1e38 / (6.3 * d)) ** 0.5  # squares about 2^126, below the largest fp32
    exact = torch.stack([(X.double() - c.double()).square().sum(1).sqrt() for c in C], dim=1)
    not_finite = torch.empty(1, dtype=torch.int32, device=cuda)
    for got in (drivers.get_euclidean_distances_rows(X, C.T.contiguous(), not_finite),
                drivers.get_euclidean_distances(X.T.contiguous(), C.T.contiguous())):
        # (redone pairs: d rounded additions)
        torch.testing.assert_close(got.double(), exact, rtol=(d / 2 + 3) * 1.2e-7, atol=0)
    assert int(not_finite) == 0


def test_fp32_distances_take_as_long_with_a_far_centroid(cuda):
    """The time does not hang on which centroid is an outlier, and not by more than a factor on how many pairs are redone
    (before: 25 times as long with a far centroid 0, 13 with two groups)."""
    import torch

    from sklearn_numba_dpex_amd.kmeans import drivers

    n, d, k = 200_000, 100, 64
    gen = torch.Generator(device=cuda).manual_seed(1)
    C = torch.rand(k, d, generator=gen, device=cuda) * 8 - 4
    lab = torch.randint(0, k, (n,), generator=gen, device=cuda)

    def least(C):
        X_t, C_t, times = (C[lab] + torch.randn(n, d, generator=gen, device=cuda)).T.contiguous(), C.T.contiguous(), []
        for _ in range(8):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            drivers.get_euclidean_distances(X_t, C_t)
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end))
        return min(times)

    usual = least(C)
    far, groups = C.clone(), C.clone()
    far[0] = 1e6
    groups[: k // 2] += 1e6
    assert least(far) < 1.5 * usual
    assert least(groups) < 6 * usual


@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("d,k,at", [(20, 5, 0), (40, 70, 0), (40, 70, 69), (17, 2, 1), (1100, 20, 0)])
def test_fp32_distances_to_a_centroid_with_nan(cuda, d, k, at, sign):
    import torch

    from sklearn_numba_dpex_amd.kmeans import drivers

    rng = np.random.default_rng(d)
    X, C = rng.standard_normal((300, d)).astype(np.float32), rng.standard_normal((k, d)).astype(np.float32)
    for f in (0, d // 2, d - 1):
        C[at, f] = np.copysign(np.float32(np.nan), np.float32(sign))
    exact = np.sqrt(((X.astype(np.float64)[:, None, :] - C.astype(np.float64)[None, :, :]) ** 2).sum(axis=2))
    not_finite = torch.empty(1, dtype=torch.int32, device=cuda)
    for got in (drivers.get_euclidean_distances_rows(_dev(X, cuda), _dev(C.T, cuda), not_finite),
                drivers.get_euclidean_distances(_dev(X.T, cuda), _dev(C.T, cuda))):
        np.testing.assert_allclose(got.cpu().numpy(), exact, rtol=1.5 * 1.2e-7)  # (NaN in the column of `at` alone)


# a total that a kernel writes to the host: the same bits call after call, from several streams at once, and as a graph
# that is replayed between other calls leaves it in device memory
@pytest.mark.parametrize("n,d,k,dtype", [(1, 3, 2, np.float32), (20_001, 14, 40, np.float32), (30_003, 70, 9, np.float32),
                                         (30_003, 20, 30, np.float64), (523_000, 3, 5, np.float64)])
def test_inertia_totals_repeat_themselves(cuda, n, d, k, dtype):
    import torch

    from sklearn_numba_dpex_amd import _capi
    from sklearn_numba_dpex_amd._capi import lib, ptr
    from sklearn_numba_dpex_amd.kmeans import drivers

    rng = np.random.default_rng(n)
    X, C = rng.standard_normal((n, d)).astype(dtype), rng.standard_normal((k, d)).astype(dtype)
    w = rng.uniform(0.5, 1.5, n).astype(dtype)
    X_t, C_t, w_d = _dev(X.T, cuda), _dev(C.T, cuda), _dev(w, cuda)
    labels, first = drivers.get_labels_inertia(X_t, C_t, w_d, True)
    lab = labels.cpu().numpy()
    exact = (w.astype(np.float64) * ((X.astype(np.float64) - C.astype(np.float64)[lab]) ** 2).sum(axis=1)).sum()
    np.testing.assert_allclose(first[0], exact, rtol=2e-5 if dtype == np.float32 else 1e-12)
    streams = [torch.cuda.Stream() for _ in range(3)]
    torch.cuda.synchronize()
    for _ in range(5):
        for s in streams:
            with torch.cuda.stream(s):
                assert drivers.get_labels_inertia(X_t, C_t, w_d, True)[1][0] == first[0]
    dc = _capi.dtype_code(X_t.dtype)
    ws_bytes = lib.kmx_assign_inertia_workspace_bytes(n, d, k, dc, 0)
    ws, out = torch.empty(ws_bytes, dtype=torch.uint8, device=cuda), torch.empty(1, dtype=X_t.dtype, device=cuda)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        _capi.check(lib.kmx_assign_labels_inertia(ptr(X_t), ptr(w_d), ptr(C_t), ptr(labels), ptr(out), ptr(ws), ws_bytes, n, d,
                                                  k, dc, 0, _capi.current_stream()), "captured")
    for _ in range(4):
        out.fill_(-1)
        graph.replay()
        assert drivers.get_labels_inertia(X_t, C_t, w_d, True)[1][0] == first[0]
        assert float(out[0]) == first[0]


def test_distances_with_few_samples_split_the_centroids(cuda):
    """With few samples the centroid range is split over the second grid dimension (ragged last
    share, k not a multiple of 4), and exact zeros / tiny distances go through the square root."""
    from sklearn_numba_dpex_amd.kmeans import drivers

    rng = np.random.default_rng(5)
    n, d, k = 2000, 14, 127
    X = rng.normal(size=(n, d)).astype(np.float32)
    C = rng.normal(size=(k, d)).astype(np.float32)
    C[3] = X[10]            # distance exactly 0
    C[4] = X[11] + 1e-20    # below the fast path's range
    exact = np.sqrt(((X.astype(np.float64)[:, None, :] - C.astype(np.float64)[None, :, :]) ** 2).sum(axis=2))
    got = drivers.get_euclidean_distances(_dev(X.T, cuda), _dev(C.T, cuda)).cpu().numpy()
    np.testing.assert_allclose(got, exact, rtol=1e-5, atol=1e-6)
    assert got[10, 3] == 0.0 and np.isfinite(got).all()


@pytest.mark.parametrize("shape", [(5_000, 14), (14, 5_000), (1, 1), (64, 64), (65, 129), (300, 1), (1, 300), (1_000, 784)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_transposed_copy(cuda, shape, dtype):
    import torch

    from sklearn_numba_dpex_amd.common.kernels import transposed_copy

    a = np.arange(shape[0] * shape[1], dtype=dtype).reshape(shape)
    got = transposed_copy(_dev(a, cuda))
    assert got.is_contiguous() and tuple(got.shape) == (shape[1], shape[0])
    np.testing.assert_array_equal(got.cpu().numpy(), a.T)


# (one value, one tile, tiles with remainders on both sides, few long rows, few columns, a start
# that is not aligned to 16 bytes)
@pytest.mark.parametrize("shape, skip", [((1, 1), 0), ((256, 32), 0), ((257, 33), 1), ((3, 20_001), 0), ((5_003, 14), 1),
                                         ((1_025, 129), 0)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_not_finite_values_are_seen(cuda, shape, skip, dtype):
    import torch

    from sklearn_numba_dpex_amd.common.kernels import all_finite, transposed_copy

    n = shape[0] * shape[1]
    a = _dev(np.full(n + skip, np.finfo(dtype).max, dtype), cuda)[skip:].reshape(shape)
    a.view(-1)[::2] = -float(np.finfo(dtype).max)
    flag = torch.full((1,), 7, dtype=torch.int32, device=cuda)
    for at in sorted({0, n // 2, n - 1}):
        for value, expected in [(np.nan, 1), (np.inf, 1), (-np.inf, 1), (0.0, 0)]:
            a.view(-1)[at] = value
            all_finite(a, flag)
            assert int(flag) == expected
            flag.fill_(7)
            got = transposed_copy(a, flag)
            assert int(flag) == expected
            np.testing.assert_array_equal(got.cpu().numpy(), a.cpu().numpy().T)
