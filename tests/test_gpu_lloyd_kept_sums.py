"""GPU tests of the sums that a run with the half-precision copy keeps and corrects for the samples that move
(csrc/lloyd_moves.hip): the centroids of corrected sums are those of rebuilt ones bit for bit (integers),
and both are the weighted means of the samples of a label."""

import numpy as np
import pytest

from tests.test_gpu_lloyd import _ResidentRun

pytestmark = pytest.mark.gpu

HEADER_SUMS = 7  # word of the copy's header: iterations behind the kept sums
HEADER_KEEP = 5  # whether the last iteration had sums to correct
HEADER_ENTRIES = 4
HEADER_FIXED = 6  # whether the sums are fixed point
KMX_NEED_RELOCATION = 4


def _words(run):
    import torch

    return run.resident[:32].view(torch.int32)


def _blobs(n, d, k, dtype, seed=0, spread=2.0):
    rng = np.random.default_rng(seed)
    blobs = k * 3 // 4  # (every third blob has two centroids: labels keep moving, and no cluster empties)
    centres = rng.uniform(-spread, spread, (blobs, d))
    X = (centres[np.arange(n) % blobs] + rng.standard_normal((n, d))).astype(dtype)
    w = rng.uniform(0.5, 1.5, n).astype(dtype)
    w[::17] = 0.0
    return X, w, X[:k].copy()


# rows of 16, 32 and 64 lanes in both types, features beyond one pass of the lanes, widths that are no multiple of
# a lane's values, stretches of the order that begin and end inside clusters, more clusters than stretches
@pytest.mark.parametrize("n,d,k,dtype", [
    (20_001, 16, 1300, np.float64), (20_011, 33, 620, np.float64), (65_603, 100, 100, np.float64), (20_001, 255, 130, np.float64),
    (20_063, 129, 288, np.float32), (30_001, 70, 300, np.float32), (66_001, 191, 1025, np.float32), (66_001, 66, 400, np.float32),
])
def test_corrected_sums_are_rebuilt_sums(cuda, n, d, k, dtype):
    X, w, init = _blobs(n, d, k, dtype, n + d)
    steps = 8
    corrected, rebuilt = _ResidentRun(cuda, X, w, init, steps), _ResidentRun(cuda, X, w, init, steps)
    n_corrected = 0
    for step in range(1, steps + 1):
        a = corrected.run(step)
        _words(rebuilt)[HEADER_SUMS] = 0
        b = rebuilt.run(step)
        if corrected.status.state not in (0, 3) or corrected.n_done < step:  # (KMX_RUNNING, KMX_MAX_ITER)
            break
        assert bool((a == b).all()) and bool((corrected.sizes == rebuilt.sizes).all())
        assert bool((corrected.labels[step % 2] == rebuilt.labels[step % 2]).all())
        keep, entries = int(_words(corrected)[HEADER_KEEP]), int(_words(corrected)[HEADER_ENTRIES])
        assert int(_words(rebuilt)[HEADER_KEEP]) == 0 and keep == (1 if step > 1 else 0)
        n_corrected += 1 if entries > 0 else 0
        lab = corrected.labels[step % 2].cpu().numpy()
        sizes = np.bincount(lab, weights=w.astype(np.float64), minlength=k)
        full = sizes > 0
        for f in (0, d // 2, d - 1):
            want = np.bincount(lab, weights=X[:, f].astype(np.float64) * w, minlength=k)[full] / sizes[full]
            got = a[f].cpu().numpy().astype(np.float64)[full]
            # (the rounding of the result, and of the comparison's own sums; weights down to one sample's)
            tol = 4 * np.finfo(dtype).eps if dtype == np.float32 else 1e-13
            np.testing.assert_allclose(got, want, rtol=tol, atol=tol * np.abs(X[:, f]).max())
    assert n_corrected >= 3


@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("weight", [1.0, 0.0])
@pytest.mark.parametrize("n,d,k,dtype", [(30_001, 100, 200, np.float64), (20_063, 129, 288, np.float32)])
def test_values_that_are_not_finite_stay_in_their_clusters(cuda, n, d, k, dtype, weight, value):
    """One infinite or undefined coordinate: the cluster that holds the sample has an infinite or undefined mean there
    (also with a weight of zero), every other mean is finite, and no iteration corrects sums with such values
    in them."""
    X, w, init = _blobs(n, d, k, dtype, 3)
    X[n - 5, 7] = value
    w[n - 5] = weight
    run = _ResidentRun(cuda, X, w, init, 3)
    for step in (1, 2):
        run.run(step, resident=True)
        assert int(_words(run)[HEADER_KEEP]) == 0
        if step == 1 or run.n_done == 2:
            lab = run.labels[run.n_done % 2].cpu().numpy()
            c = run.cent[run.n_done % 2].cpu().numpy()
            bad = ~np.isfinite(c)
            assert bad[7, lab[n - 5]] and set(np.nonzero(bad)[1]) <= {int(lab[n - 5])} and set(np.nonzero(bad)[0]) == {7}


@pytest.mark.parametrize("value", [np.inf, np.nan])
@pytest.mark.parametrize("n,d,k,dtype", [(30_001, 100, 200, np.float64), (20_063, 129, 288, np.float32)])
def test_weights_that_are_not_finite_stay_in_their_clusters(cuda, n, d, k, dtype, value):
    X, w, init = _blobs(n, d, k, dtype, 4)
    w[n - 5] = value
    run = _ResidentRun(cuda, X, w, init, 3)
    run.run(1)
    lab, c = run.labels[1].cpu().numpy(), run.cent[1].cpu().numpy()
    held = np.arange(k) == lab[n - 5]
    assert not np.isfinite(c[:, held]).any() and np.isfinite(c[:, ~held]).all()
    run.run(2)
    assert int(_words(run)[HEADER_KEEP]) == 0


# magnitudes that the fused steps' fixed point and the fp32 maxima do not hold; one feature far below the others
@pytest.mark.parametrize("scale,weight_scale,dtype", [
    (1e10, 1e20, np.float32), (1e-17, 1e-12, np.float32), (1e-35, 1.0, np.float64),
    (1e-80, 1.0, np.float64), (1e45, 1.0, np.float64), (1.0, 1e45, np.float64), (1.0, 1e-60, np.float64),
])
def test_sums_of_data_of_any_magnitude(cuda, scale, weight_scale, dtype):
    n, d, k = (30_001, 100, 200) if dtype == np.float64 else (20_063, 129, 288)
    X, w, init = _blobs(n, d, k, np.float64, 5)
    X[:, 3] *= 1e-20 if dtype == np.float64 else 1e-5
    X, w = (X * scale).astype(dtype), (w * weight_scale).astype(dtype)
    run = _ResidentRun(cuda, X, w, X[:k].copy(), 2)
    c = run.run(1).cpu().numpy().astype(np.float64)
    assert run.n_done == 1 and run.status.state in (0, 3)  # (no cluster is empty)
    lab = run.labels[1].cpu().numpy()
    sizes = np.bincount(lab, weights=w.astype(np.float64), minlength=k)
    full = sizes > 0
    for f in (0, 3, d - 1):
        want = np.bincount(lab, weights=X[:, f].astype(np.float64) * w, minlength=k)[full] / sizes[full]
        tol = 4 * np.finfo(dtype).eps if dtype == np.float32 else 1e-13  # (as above)
        np.testing.assert_allclose(c[f][full], want, rtol=tol, atol=tol * float(np.abs(X[:, f]).max()))


def test_all_sums_are_converted_when_the_gpu_is_busy(cuda):
    """An iteration that ends with empty clusters: the workgroup that finds them is the launch's first and does not wait
    for the 1 024 that convert the sums.  Another stream keeps the GPU busy with workgroups of a thousand threads, each
    on a long row, so that many of them start behind its end."""
    import torch

    n, d, k = 20_003, 256, 1024
    X, w, init = _blobs(n, d, k, np.float32, 6)
    init[-16:] = 1e4
    load = torch.rand(1024, 1 << 19, device=cuda)
    out = torch.empty_like(load)
    side = torch.cuda.Stream()
    expected = None
    for busy in [False] + [True] * 8:
        run = _ResidentRun(cuda, X, w, init, 2)
        run.cent[1].fill_(float("nan"))
        torch.cuda.synchronize()
        if busy:
            with torch.cuda.stream(side):
                for _ in range(20):
                    torch.softmax(load, 1, out=out)
        run.run(1)
        torch.cuda.synchronize()
        assert (run.status.state, run.status.n_empty, run.status.n_iter) == (KMX_NEED_RELOCATION, 16, 0)
        assert sorted(run.empty[:16].tolist()) == list(range(k - 16, k))
        sums = run.cent[1].cpu().numpy()
        assert np.isfinite(sums).all()
        if expected is None:
            lab, expected = run.labels[1].cpu().numpy(), sums
            for f in (0, d - 1):
                want = np.bincount(lab, weights=X[:, f].astype(np.float64) * w, minlength=k)
                np.testing.assert_allclose(sums[f], want, rtol=1e-6, atol=1e-6 * np.abs(X[:, f]).max())
        np.testing.assert_array_equal(sums, expected)


def _check_means(run, X, w, k, features, tol):
    """Centroids of the clusters that hold samples of some weight against fp64 means, relative to the mean magnitude of their
    terms; cluster sizes likewise."""
    lab = run.labels[run.n_done % 2].cpu().numpy()
    w64 = w.astype(np.float64)
    sizes = np.bincount(lab, weights=w64, minlength=k)
    full = sizes > 0
    np.testing.assert_allclose(run.sizes.cpu().numpy().astype(np.float64), sizes, rtol=tol)
    c = run.cent[run.n_done % 2].cpu().numpy().astype(np.float64)
    for f in features:
        x = X[:, f].astype(np.float64)
        want = np.bincount(lab, weights=x * w64, minlength=k)[full] / sizes[full]
        size_of = np.bincount(lab, weights=np.abs(x) * w64, minlength=k)[full] / sizes[full]
        assert np.abs((c[f][full] - want) / np.maximum(size_of, np.finfo(np.float64).tiny)).max() < tol


# a copy whose sums were fp64 additions before they were kept: the tiled product in fp32, all of fp64.  An outlier within
# the words of a sum and one beyond them; a cluster whose weights are that far below the others'
@pytest.mark.parametrize("outlier,weight,fixed", [
    (1e9, 1.0, True), (1e11, 1.0, True), (1e25, 1.0, False), (1.0, 1e-10, True), (1.0, 1e-30, False), (1e9, 1e-30, False),
])
@pytest.mark.parametrize("n,d,k,dtype", [(100_003, 129, 128, np.float32), (65_603, 100, 100, np.float64)])
def test_sums_beside_much_larger_ones(cuda, n, d, k, dtype, outlier, weight, fixed):
    X, w, init = _blobs(n, d, k, dtype, 8)
    X += np.sign(X) * 0.1  # (smallest magnitude 0.1: the line is that of the outlier and the weights)
    X[n // 2, 5] = 3.0 * outlier
    w[w > 0] = 1.0
    lightest = np.arange(n) % (k * 3 // 4) == 7
    w[lightest] = weight
    X = X.astype(dtype)
    # (samples of that blob stand apart, so that clusters are of one weight)
    X[lightest] += dtype(30.0)
    init = X[:k].copy()
    run = _ResidentRun(cuda, X, w, init, 3)
    for step in (1, 2):
        run.run(step)
        if step > 1 and run.n_done < step:
            break  # (the outlier's score is no number in fp32: a cluster is empty)
        assert run.n_done == step and run.status.state in (0, 3)
        assert int(_words(run)[HEADER_FIXED]) == int(fixed)
        assert int(_words(run)[HEADER_KEEP]) == int(fixed and step > 1)
        # (a term's own rounding, fp64 additions in some order and the result's)
        _check_means(run, X, w, k, (0, 5, d - 1), 4 * np.finfo(dtype).eps if dtype == np.float32 else 1e-13)


@pytest.mark.parametrize("n,d,k,dtype", [(20_001, 100, 300, np.float32), (100_003, 129, 128, np.float32),
                                         (65_603, 100, 100, np.float64)])
def test_sums_corrected_behind_a_relocation(cuda, n, d, k, dtype):
    """The iterations behind a relocation, which has moved samples between sums but not between the kept ones: the same
    bits as with sums rebuilt in every iteration; the run goes on without a look at its state."""
    import torch

    from sklearn_numba_dpex_amd._capi import check, lib, ptr
    from sklearn_numba_dpex_amd.kmeans import drivers

    X, w, init = _blobs(n, d, k, dtype, 9)
    w[w == 0] = 1.0
    init[[2, k // 2, k - 1]] = 1e4
    steps, seen = 6, {}
    for rebuilt in (False, True):
        run = _ResidentRun(cuda, X, w, init, steps)
        results, kept = [], []
        relocations, until = 0, 1
        while until <= steps:
            if rebuilt:
                _words(run)[HEADER_SUMS] = 0
            run.run(until)
            if run.status.state == KMX_NEED_RELOCATION:
                relocations += 1
                j = run.status.n_iter
                a, b = j % 2, (j + 1) % 2
                drivers._relocate_empty_clusters(run.status.n_empty, run.X_t, run.w, run.cent[b], run.sizes, run.labels[b],
                                                 run.empty, run.cent[a])
                check(lib.kmx_lloyd_finalize(run.plan, ptr(run.cent[a]), ptr(run.cent[b]), ptr(run.sizes), ptr(run.ws),
                                             run.ws_bytes, run.stream), "kmx_lloyd_finalize")
                run.n_done = j + 1
            kept.append(int(_words(run)[HEADER_KEEP]))
            results.append((run.cent[run.n_done % 2].clone(), run.labels[run.n_done % 2].clone(), run.sizes.clone()))
            until = run.n_done + 1
            if run.status.state not in (0, 3, KMX_NEED_RELOCATION):
                break
        assert relocations >= 1 and len(results) >= 4
        assert kept[1:] == [0 if rebuilt else 1] * (len(kept) - 1)
        seen[rebuilt] = results
    assert len(seen[False]) == len(seen[True])
    for step, (one, other) in enumerate(zip(seen[False], seen[True])):
        differ = [i for i in range(3) if not torch.equal(one[i], other[i])]
        assert not differ, step
