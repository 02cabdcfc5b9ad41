"""Rows that start at no 16-byte boundary: sample counts of every remainder, and arrays that begin one element
into their buffer.  Every kernel family against fp64, by labels, sums, inertia, distances and seeding picks."""

import numpy as np
import pytest

from oracle import kmeans as ok
from tests._parity import RTOL, assert_centers_close, assert_labels_match

pytestmark = pytest.mark.gpu


def _offset(a, cuda, skip):
    """`a` on the device, `skip` elements into its buffer."""
    import torch

    a = np.ascontiguousarray(a)
    buf = torch.zeros(a.size + skip, dtype=torch.from_numpy(a[:0].reshape(-1)).dtype, device=cuda)
    buf[skip:] = torch.from_numpy(a.reshape(-1)).to(cuda)
    out = buf[skip:].view(a.shape)
    assert out.data_ptr() % 16 == (skip * a.itemsize) % 16
    return out


SHAPES = [
    (14, 40, np.float32), (33, 40, np.float32),   # screened step, one and three K steps
    (5, 40, np.float32), (4, 200, np.float32),    # fp32 matrix cores; sums beside the labels
    (14, 5, np.float32), (9, 5, np.float64),      # samples in registers
    (70, 12, np.float32), (150, 9, np.float32),   # few clusters of wide samples, row-major and not
    (67, 40, np.float32), (67, 40, np.float64),   # tiled product
    (66, 300, np.float32),                        # wide samples, bucketed sums in fixed point
    (32, 40, np.float64), (50, 150, np.float64),  # screened fp64 step; fp64 matrix cores
]


@pytest.mark.parametrize("d,k,dtype", SHAPES)
@pytest.mark.parametrize("n,skip", [(2_052, 1), (2_053, 0), (2_054, 3), (2_055, 1)])
def test_rows_off_16_byte_boundaries(cuda, n, skip, d, k, dtype):
    from sklearn_numba_dpex_amd.kmeans import drivers

    rng = np.random.default_rng(n + 31 * d + k)
    C = rng.uniform(-5, 5, (k, d)).astype(dtype)
    X = (C[rng.integers(0, k, n)] + rng.standard_normal((n, d))).astype(dtype)
    w = rng.uniform(0.5, 1.5, n).astype(dtype)
    X_t, w_d, C_t = _offset(X.T, cuda, skip), _offset(w, cuda, skip), _offset(C.T, cuda, skip)

    labels, inertia = drivers.get_labels_inertia(X_t, C_t, w_d, True)
    got = labels.cpu().numpy().astype(np.int64)
    assert_labels_match(got, ok.assign_labels(X, C), X, C)
    assert float(inertia[0]) == pytest.approx(float(ok.inertia(X, w, C, got)), rel=RTOL[X.dtype] * 5)

    dist = drivers.get_euclidean_distances(X_t, C_t).cpu().numpy()
    exact = np.sqrt(((X.astype(np.float64)[:, None, :] - C.astype(np.float64)[None, :, :]) ** 2).sum(axis=2))
    np.testing.assert_allclose(dist, exact, rtol=RTOL[X.dtype] * 2, atol=RTOL[X.dtype])

    _, _, centres, n_iter = drivers.lloyd(X_t, w_d, C_t, False, 1, False, 0.0)
    assert n_iter == 1
    sums = np.zeros((k, d))
    np.add.at(sums, got, X.astype(np.float64) * w[:, None].astype(np.float64))
    sizes = np.bincount(got, weights=w.astype(np.float64), minlength=k)
    assert (sizes > 0).all()
    assert_centers_close(centres.cpu().numpy().T, sums / sizes[:, None], dtype)


@pytest.mark.parametrize("n,skip", [(2_052, 1), (2_053, 0), (2_054, 3), (140_003, 1)])
@pytest.mark.parametrize("d,k,dtype", [(5, 6, np.float32), (9, 6, np.float64), (70, 6, np.float32), (70, 6, np.float64),
                                       (65, 40, np.float32)])
def test_seeding_picks_off_16_byte_boundaries(cuda, n, skip, d, k, dtype):
    """The oracle's picks, wherever the rows lie."""
    from sklearn_numba_dpex_amd.kmeans import drivers

    rng = np.random.default_rng(n + d)
    X = rng.standard_normal((n, d)).astype(dtype)
    w = rng.uniform(0.5, 1.5, n).astype(dtype)
    got = []
    for at in (0, skip, 2):
        centres, picks = drivers.kmeans_plusplus(_offset(X.T, cuda, at), _offset(w, cuda, at), k, 3)
        picks = picks.cpu().numpy()
        np.testing.assert_array_equal(centres.cpu().numpy().T, X[picks])
        got.append(picks)
    np.testing.assert_array_equal(got[0], got[1])
    np.testing.assert_array_equal(got[0], got[2])
    if n < 10_000:
        np.testing.assert_array_equal(got[0], ok.kmeans_plusplus(X, w, k, 3)[1])


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("rows,cols", [(3, 1), (2, 3), (5, 1_027), (3, 300_001), (70, 5_002)])
def test_row_sums_and_centring_off_16_byte_boundaries(cuda, rows, cols, dtype):
    from sklearn_numba_dpex_amd.common.kernels import broadcast_rows
    from sklearn_numba_dpex_amd.common.reductions import sum_reduction

    rng = np.random.default_rng(rows + cols)
    a, v = rng.standard_normal((rows, cols)).astype(dtype), rng.standard_normal(rows).astype(dtype)
    for skip in (0, 1):
        at = _offset(a, cuda, skip)
        for square in (False, True):
            exact = (a.astype(np.float64) ** (2 if square else 1)).sum(axis=1)
            bound = 2 * np.finfo(dtype).eps * np.abs(exact) + 1e-15 * cols * np.abs(a).max() ** 2
            assert (np.abs(sum_reduction(at, axis=1, square=square).cpu().numpy() - exact) <= bound).all()
        broadcast_rows(at, _offset(v, cuda, 0), "minus")
        np.testing.assert_array_equal(at.cpu().numpy(), a - v[:, None])
