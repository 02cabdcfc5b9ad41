"""GPU parity of the Lloyd path (fused step, reduction/finalisation, full run, labels,
inertia) against the CPU oracle, through the C ABI and through the drivers."""

import ctypes

import numpy as np
import pytest

from oracle import datasets
from oracle import kmeans as ok
from tests._parity import RTOL, assert_centers_close, assert_labels_match

pytestmark = pytest.mark.gpu


def _dev(a, cuda):
    import torch

    return torch.as_tensor(np.ascontiguousarray(a), device=cuda)


# a step per kernel family; more runs at once than there are words to announce iterations in (64), so
# that some of them read the status instead
@pytest.mark.parametrize("n,d,k,dtype,runs", [(3_001, 14, 20, np.float32, 70), (3_001, 10, 5, np.float64, 3),
                                              (5_000, 70, 6, np.float32, 3), (5_003, 100, 40, np.float64, 3)])
def test_runs_in_several_threads_equal_iterations_one_by_one(cuda, n, d, k, dtype, runs):
    import threading

    import torch

    from sklearn_numba_dpex_amd import _capi
    from sklearn_numba_dpex_amd._capi import lib, ptr

    rng = np.random.default_rng(n + d)
    X_t, w = _dev(rng.standard_normal((d, n)).astype(dtype), cuda), _dev(rng.uniform(0.5, 1.5, n).astype(dtype), cuda)
    max_iter = 7

    def run(out, in_one_call):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            plan = _capi.lloyd_plan(n, d, k, _capi.dtype_code(X_t.dtype))
            cent = [X_t[:, :k].contiguous(), torch.empty(d, k, dtype=X_t.dtype, device=cuda)]
            labels = [torch.empty(n, dtype=torch.int32, device=cuda) for _ in range(2)]
            sizes, empty = torch.empty(k, dtype=X_t.dtype, device=cuda), torch.empty(k, dtype=torch.int32, device=cuda)
            ws, status = torch.empty(plan.workspace_bytes, dtype=torch.uint8, device=cuda), _capi.LloydStatus()
            _capi.check(lib.kmx_lloyd_init(plan, ptr(ws), plan.workspace_bytes, ptr(X_t), ptr(w), ptr(cent[0]),
                                           max_iter, 0.0, stream.cuda_stream), "init")
            if in_one_call:
                _capi.check(lib.kmx_lloyd_run(plan, ptr(X_t), None, ptr(w), ptr(cent[0]), ptr(cent[1]), ptr(labels[0]),
                                              ptr(labels[1]), ptr(sizes), ptr(empty), ptr(ws), plan.workspace_bytes,
                                              None, 0, 0, max_iter, status, stream.cuda_stream), "run")
            else:
                for it in range(max_iter):
                    a, b = it % 2, (it + 1) % 2
                    _capi.check(lib.kmx_lloyd_iter(plan, ptr(X_t), None, ptr(w), ptr(cent[a]), ptr(cent[b]),
                                                   ptr(labels[a]), ptr(labels[b]), ptr(sizes), ptr(empty), ptr(ws),
                                                   plan.workspace_bytes, stream.cuda_stream), "iter")
                _capi.check(lib.kmx_lloyd_status_read(ptr(ws), status, stream.cuda_stream), "status")
            stream.synchronize()
            b = status.n_iter % 2
            out.append((status.n_iter, status.state, status.shift_sum, cent[b].cpu().numpy(), labels[b].cpu().numpy()))

    expected, got = [], []
    torch.cuda.synchronize()
    run(expected, False)
    threads = [threading.Thread(target=run, args=(got, True)) for _ in range(runs)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(got) == runs
    tol = 1e-6 if dtype == np.float32 else 1e-13  # (fp64 sums by floating-point atomics: order of additions)
    for r in got:
        assert r[:2] == expected[0][:2]
        np.testing.assert_allclose(r[2], expected[0][2], rtol=10 * tol)
        np.testing.assert_allclose(r[3], expected[0][3], rtol=tol, atol=tol)
        np.testing.assert_array_equal(r[4], expected[0][4])


# every number of 16-feature steps (fp64 up to 64 features, both types beyond), one and two columns of samples per
# wave (from 65 536 samples on), centroid tiles resident in LDS and streamed, sample counts at the edges of tiles
# and of 128-bit loads, clusters at the edges of blocks of 32
@pytest.mark.parametrize("n,d,k,dtype,data", [
    (20_001, 16, 1300, np.float64, "blobs"), (20_032, 17, 1250, np.float64, "blobs"), (16_385, 48, 640, np.float64, "blobs"),
    (16_383, 64, 513, np.float64, "blobs"), (20_001, 65, 300, np.float32, "blobs"), (20_000, 96, 257, np.float32, "blobs"),
    (65_600, 100, 100, np.float64, "blobs"), (65_600, 112, 272, np.float32, "blobs"), (65_537, 128, 65, np.float64, "blobs"),
    (20_063, 129, 288, np.float32, "blobs"), (20_031, 160, 1000, np.float32, "blobs"), (66_049, 161, 320, np.float32, "blobs"),
    (20_001, 177, 200, np.float64, "blobs"), (66_001, 192, 1025, np.float32, "blobs"), (20_001, 208, 300, np.float32, "blobs"),
    (20_001, 224, 300, np.float32, "blobs"), (65_999, 240, 500, np.float32, "blobs"), (65_543, 256, 1100, np.float32, "blobs"),
    (20_001, 256, 130, np.float64, "blobs"), (20_001, 100, 300, np.float32, "integers"), (20_001, 100, 300, np.float64, "integers"),
    (20_001, 100, 300, np.float32, "far"), (20_001, 100, 300, np.float64, "outliers"), (20_001, 100, 300, np.float64, "few values"),
])
def test_labels_from_the_half_precision_copy(cuda, n, d, k, dtype, data):
    """Labels of a run and of its end against fp64 distances: the exact arg-min, or one whose distance is the same to
    the rounding of one score in the input type (2 (d + 2) ulp of |x| |c|)."""
    import torch

    from sklearn_numba_dpex_amd import _capi
    from sklearn_numba_dpex_amd._capi import lib
    from sklearn_numba_dpex_amd.kmeans import drivers

    rng = np.random.default_rng(n + d + k)
    X = (rng.uniform(-2, 2, (k, d))[rng.integers(0, k, n)] + rng.standard_normal((n, d)))
    if data == "integers":
        X = np.round(X)
    elif data == "few values":
        X = X[rng.integers(0, 500, n)]  # every centroid among the samples, most of them more than once
    elif data == "outliers":
        X[::97] *= 1e5
    X = X.astype(dtype)
    init = X[rng.choice(n, k, replace=False)].copy()
    if data == "far":
        init[3] = 1e4
    w = rng.uniform(0.5, 1.5, n).astype(dtype)
    plan = _capi.lloyd_plan(n, d, k, _capi.dtype_code(np.dtype(dtype)), 0)
    assert lib.kmx_lloyd_resident_bytes(plan) > 0
    labels, inertia, centroids_t, n_iter = drivers.lloyd(_dev(X.T, cuda), _dev(w, cuda), _dev(init.T, cuda), False,
                                                         max_iter=2, tol=0.0, flags=0)
    x, c = _dev(X, cuda).double(), centroids_t.double()
    half = (c * c).sum(0) / 2
    lab = labels.long()
    assert int(lab.min()) >= 0 and int(lab.max()) < k
    ulp = float(np.finfo(dtype).eps)
    own, total = torch.empty(n, dtype=torch.float64, device=cuda), 0.0
    for lo in range(0, n, 8192):
        hi = min(n, lo + 8192)
        scores = half[None] - x[lo:hi] @ c.contiguous()
        mine = scores.gather(1, lab[lo:hi, None])[:, 0]
        allowed = 2 * (d + 2) * ulp * (x[lo:hi].norm(dim=1) * c.norm(dim=0).max() + half.max())
        assert bool((mine - scores.min(1).values <= allowed).all())
        own[lo:hi] = ((x[lo:hi] - c.T[lab[lo:hi]]) ** 2).sum(1)
    expected = float((own * _dev(w, cuda).double()).sum())
    np.testing.assert_allclose(float(inertia), expected, rtol=1e-5 if dtype == np.float32 else 1e-12)
    # the first iteration's labels and sums, through the centroids of a run of one iteration
    labels1, _, first_t, n_iter = drivers.lloyd(_dev(X.T, cuda), _dev(w, cuda), _dev(init.T, cuda), False, max_iter=1,
                                                tol=0.0, flags=0)
    if data in ("blobs", "outliers"):
        d2 = [((x[lo:lo + 8192] @ _dev(init.T, cuda).double()) - (_dev(init, cuda).double() ** 2).sum(1) / 2).argmax(1)
              for lo in range(0, n, 8192)]
        start = torch.cat(d2)
        weights = torch.zeros(k, dtype=torch.float64, device=cuda).index_add_(0, start, _dev(w, cuda).double())
        sums = torch.zeros(k, d, dtype=torch.float64, device=cuda).index_add_(0, start, x * _dev(w, cuda).double()[:, None])
        full = weights > 0
        err = (first_t.T.double() - sums / weights[:, None])[full].abs().max() / sums[full].div(weights[full, None]).abs().max()
        assert float(err) <= (2e-5 if dtype == np.float32 else 1e-11)


class _ResidentRun:
    """A run with the half-precision copy, through the C ABI."""

    def __init__(self, cuda, X, w, init, max_iter):
        import torch

        from sklearn_numba_dpex_amd import _capi
        from sklearn_numba_dpex_amd._capi import lib, ptr

        n, d = X.shape
        k = len(init)
        dtype = _dev(X[:1], cuda).dtype
        self.lib, self.ptr, self.check, self.stream = lib, ptr, _capi.check, _capi.current_stream()
        self.n, self.max_iter, self.n_done = n, max_iter, 0
        self.plan = _capi.lloyd_plan(n, d, k, _capi.dtype_code(dtype), 0)
        self.X_t, self.w = _dev(X.T, cuda), _dev(w, cuda)
        self.X_rm = torch.empty(n, d, dtype=dtype, device=cuda)
        self.cent = [_dev(init.T, cuda), torch.empty(d, k, dtype=dtype, device=cuda)]
        self.labels = [torch.empty(n, dtype=torch.int32, device=cuda) for _ in range(2)]
        self.sizes, self.empty = torch.empty(k, dtype=dtype, device=cuda), torch.empty(k, dtype=torch.int32, device=cuda)
        self.ws_bytes, self.res_bytes = self.plan.workspace_bytes, lib.kmx_lloyd_resident_bytes(self.plan)
        assert self.res_bytes > 0
        self.ws = torch.empty(self.ws_bytes, dtype=torch.uint8, device=cuda)
        self.resident = torch.empty(self.res_bytes, dtype=torch.uint8, device=cuda)
        self.status = _capi.LloydStatus()
        self.init()

    def init(self):
        ptr = self.ptr
        self.check(self.lib.kmx_lloyd_init_resident(
            self.plan, ptr(self.ws), self.ws_bytes, ptr(self.X_t), ptr(self.w), ptr(self.cent[0]), self.max_iter, 0.0,
            ptr(self.X_rm), ptr(self.resident), self.res_bytes, self.stream), "kmx_lloyd_init_resident")

    def run(self, until, resident=True):
        ptr = self.ptr
        self.check(self.lib.kmx_lloyd_run(
            self.plan, ptr(self.X_t), ptr(self.X_rm), ptr(self.w), ptr(self.cent[0]), ptr(self.cent[1]),
            ptr(self.labels[0]), ptr(self.labels[1]), ptr(self.sizes), ptr(self.empty), ptr(self.ws), self.ws_bytes,
            ptr(self.resident) if resident else None, self.res_bytes, self.n_done, until, self.status, self.stream),
            "kmx_lloyd_run")
        self.n_done = self.status.n_iter
        return self.cent[self.n_done % 2]

    def labels_inertia(self):
        import torch

        ptr, centroids_t = self.ptr, self.cent[self.n_done % 2]
        labels, out = torch.full_like(self.labels[0], -1), torch.empty(1, dtype=centroids_t.dtype, device=centroids_t.device)
        area_bytes = self.lib.kmx_inertia_workspace_bytes(self.n)
        area = torch.empty(area_bytes, dtype=torch.uint8, device=centroids_t.device)
        self.check(self.lib.kmx_lloyd_labels_inertia(
            self.plan, ptr(self.X_t), ptr(self.X_rm), ptr(self.w), ptr(centroids_t), ptr(labels), ptr(out), ptr(self.ws),
            self.ws_bytes, ptr(self.resident), self.res_bytes, self.n_done, ptr(area), area_bytes, self.stream),
            "kmx_lloyd_labels_inertia")
        return labels.cpu().numpy(), out.cpu().numpy()

    def listed(self):
        """Samples of the last labelling without a certificate: the second word of the copy's header."""
        return self._header()[1]

    def left(self):
        """... of which so many had more candidates than are looked at one by one: the third word."""
        return self._header()[2]

    def _header(self):
        import torch

        return self.resident[:12].view(torch.int32).tolist()


@pytest.mark.parametrize("n,d,k,data", [(20_003, 128, 260, "offset"), (5_003, 128, 500, "blobs")])
def test_labels_of_a_resident_run_taken_twice_and_midway(cuda, n, d, k, data):
    """kmx_lloyd_labels_inertia again and between two halves of a run: each labelling starts its lists anew (three that
    list nearly all samples would run past their n entries otherwise), and the run goes on as if not interrupted."""
    rng = np.random.default_rng(d)
    X = rng.standard_normal((n, d))
    if data == "offset":
        X[:, 0] += 300  # no clusters, and a rounding to half precision of the order of the margins: little is certified
    else:
        X += rng.uniform(-2, 2, (k, d))[rng.integers(0, k, n)]
    X = X.astype(np.float32)
    w = rng.uniform(0.5, 1.5, n).astype(np.float32)
    init = X[rng.choice(n, k, replace=False)]
    whole = _ResidentRun(cuda, X, w, init, 6)
    expected = whole.run(6).cpu().numpy()
    parts = _ResidentRun(cuda, X, w, init, 6)
    parts.run(3)
    first, first_inertia = parts.labels_inertia()
    if data == "offset":
        assert parts.listed() > n // 2
    for _ in range(3):
        again, inertia = parts.labels_inertia()
        np.testing.assert_array_equal(again, first)
        np.testing.assert_array_equal(inertia, first_inertia)
    np.testing.assert_array_equal(parts.run(6).cpu().numpy(), expected)  # (sums in fixed point: whatever the order)
    assert parts.n_done == whole.n_done == 6
    for a, b in zip(parts.labels_inertia(), whole.labels_inertia()):
        np.testing.assert_array_equal(a, b)
    # another run on the same copy, begun with the plain initialisation
    again = _ResidentRun(cuda, X, w, init, 6)
    again.run(3)
    again.cent[0].copy_(_dev(init.T, cuda))
    ptr = again.ptr
    again.check(again.lib.kmx_lloyd_init(again.plan, ptr(again.ws), again.ws_bytes, ptr(again.X_t), ptr(again.w),
                                         ptr(again.cent[0]), 6, 0.0, again.stream), "kmx_lloyd_init")
    again.n_done = 0
    np.testing.assert_array_equal(again.run(6).cpu().numpy(), expected)


def test_recheck_count_of_a_resident_run(cuda):
    """The count of uncertified samples is that of the copy's labelling, where a run takes its labels from it."""
    import ctypes

    rng = np.random.default_rng(3)
    X = rng.standard_normal((20_003, 128)).astype(np.float32)
    run = _ResidentRun(cuda, X, np.ones(len(X), dtype=np.float32), X[:260], 2)
    run.run(2)
    assert run.status.uncertified_iter == 0
    count = ctypes.c_uint32(12345)
    run.check(run.lib.kmx_lloyd_recheck_count(run.plan, run.ptr(run.ws), ctypes.byref(count), run.stream), "recheck")
    assert 0 < count.value == run.listed() < len(X) // 8


@pytest.mark.parametrize("n,d,k,dtype,far", [(20_001, 100, 300, np.float32, 1e8), (65_600, 100, 100, np.float64, 1e8),
                                             (20_001, 129, 300, np.float32, -3e4), (20_001, 129, 300, np.float64, 1e200)])
def test_initial_centroids_far_from_all_samples(cuda, n, d, k, dtype, far):
    """The half-precision copy keeps the samples' digits whatever the initial centroids are: as soon as those have been
    relocated, the labelling certifies samples again."""
    from sklearn_numba_dpex_amd import _capi
    from sklearn_numba_dpex_amd.kmeans import drivers

    rng = np.random.default_rng(n + d)
    X = (rng.uniform(-2, 2, (k, d))[rng.integers(0, k, n)] + rng.standard_normal((n, d))).astype(dtype)
    init = X[:k].copy()
    init[1:4] = far
    run = _ResidentRun(cuda, X, np.ones(n, dtype=dtype), init, 6)
    run.run(6)
    assert (run.status.state, run.status.n_iter, run.status.n_empty) == (_capi.KMX_NEED_RELOCATION, 0, 3)
    run.cent[1] /= run.sizes.clamp(min=1)  # (the sums of the first iteration), and samples for the empty clusters
    run.cent[1][:, 1:4] = _dev(X[k:k + 3].T, cuda)
    centroids_t = run.cent[1].clone()
    run.sizes.fill_(1)
    run.check(run.lib.kmx_lloyd_finalize(run.plan, run.ptr(run.cent[0]), run.ptr(run.cent[1]), run.ptr(run.sizes),
                                         run.ptr(run.ws), run.ws_bytes, run.stream), "kmx_lloyd_finalize")
    np.testing.assert_array_equal(run.cent[1].cpu().numpy(), centroids_t.cpu().numpy())
    run.n_done = 1
    labels, _ = run.labels_inertia()
    assert run.listed() < n // 8
    expected, _ = drivers.get_labels_inertia(run.X_t, centroids_t, run.w, True)
    np.testing.assert_array_equal(labels, expected.cpu().numpy())


@pytest.mark.parametrize("n,d,k,dtype", [(20_001, 100, 300, np.float32), (20_003, 129, 300, np.float32),
                                         (65_601, 101, 100, np.float64)])
def test_data_that_half_precision_cannot_tell_apart(cuda, n, d, k, dtype):
    """One feature far wider than the others: the run leaves the copy after its first iteration, whatever pieces it is
    asked for in, and comes to what a run without the copy comes to."""
    from sklearn_numba_dpex_amd.kmeans import drivers

    rng = np.random.default_rng(n + d)
    X = rng.standard_normal((n, d))
    X[:, 0] *= 100
    X = X.astype(dtype)
    w, init = rng.uniform(0.5, 1.5, n).astype(dtype), X[rng.choice(n, k, replace=False)]
    plain = _ResidentRun(cuda, X, w, init, 8)
    expected = plain.run(8, resident=False).cpu().numpy()
    assert (plain.n_done, plain.status.uncertified_iter) == (8, 0)
    rtol = 0 if dtype == np.float32 else 1e-12  # (fp64 sums by floating-point atomics: order of additions)
    for stops in ([8], [1, 2, 5, 8]):
        run = _ResidentRun(cuda, X, w, init, 8)
        for until in stops:
            got = run.run(until)
            assert run.status.uncertified_iter == 1
        assert (run.n_done, run.status.state) == (plain.n_done, plain.status.state)
        np.testing.assert_allclose(got.cpu().numpy(), expected, rtol=rtol, atol=100 * rtol)
        last = run.n_done % 2
        np.testing.assert_array_equal(run.labels[last].cpu().numpy(), plain.labels[last].cpu().numpy())
    labels, inertia, centroids_t, _ = drivers.lloyd(run.X_t, run.w, _dev(init.T, cuda), False, 8, False, 0.0, flags=0)
    np.testing.assert_allclose(centroids_t.cpu().numpy(), expected, rtol=rtol, atol=100 * rtol)
    assigned, score = drivers.get_labels_inertia(run.X_t, centroids_t, run.w, True)
    np.testing.assert_array_equal(labels.cpu().numpy(), assigned.cpu().numpy())
    assert float(inertia) == float(score[0])


@pytest.mark.parametrize("n,d,k,dtype", [(20_003, 128, 260, np.float32), (65_601, 101, 100, np.float64)])
@pytest.mark.parametrize("branch", ["candidates", "too many candidates", "too many samples"])
def test_samples_without_a_certificate_take_each_way(cuda, n, d, k, dtype, branch):
    from sklearn_numba_dpex_amd.kmeans import drivers

    rng = np.random.default_rng(d)
    X = rng.standard_normal((n, d))
    if branch == "too many samples":
        X[:, 0] *= 100
    elif branch == "too many candidates":
        X += rng.uniform(-2, 2, (k, d))[np.arange(n) % k]
    X = X.astype(dtype)
    init = X[:k].copy()
    if branch == "too many candidates":
        init[k // 2:k // 2 + 12] = init[k // 2]  # a dozen equal ones
    run = _ResidentRun(cuda, X, np.ones(n, dtype=dtype), init, 1)
    labels, _ = run.labels_inertia()
    if branch == "candidates":
        assert 0 < run.listed() <= n // 8 and run.left() == 0
    elif branch == "too many candidates":
        assert 0 < run.left() <= run.listed() <= n // 8
        assert (labels == k // 2).any() and not np.isin(labels, np.arange(k // 2 + 1, k // 2 + 12)).any()
    else:
        assert run.listed() > n // 8
    expected, _ = drivers.get_labels_inertia(run.X_t, run.cent[0], run.w, True)
    np.testing.assert_array_equal(labels, expected.cpu().numpy())


# rows that 128-bit loads take and rows that they do not
@pytest.mark.parametrize("n,d,k,dtype", [(20_001, 100, 300, np.float32), (20_003, 129, 300, np.float32),
                                         (65_601, 100, 100, np.float64), (65_537, 65, 101, np.float64)])
def test_relocation_in_a_run_with_the_half_precision_copy(cuda, n, d, k, dtype):
    """The distances that rank the samples against fp64, and the centroids of an iteration that relocates three empty
    clusters against the oracle."""
    import torch

    from sklearn_numba_dpex_amd.kmeans import drivers

    rng = np.random.default_rng(n + d)
    X = (rng.uniform(-2, 2, (k, d))[rng.integers(0, k, n)] + rng.standard_normal((n, d))).astype(dtype)
    for i, stretch in ((7, 3), (n // 2, 4), (n - 1, 5)):  # the samples that are to be picked, far apart in rank
        X[i] *= stretch
    w = rng.uniform(0.5, 1.5, n).astype(dtype)
    init = X[rng.choice(n // 2 - 8, k, replace=False) + 8].copy()
    init[[2, k // 2, k - 1]] = 1e4
    run = _ResidentRun(cuda, X, w, init, 1)
    labels = torch.as_tensor(rng.integers(0, k, n).astype(np.int32), device=cuda)
    got = torch.full((n,), -1.0, dtype=run.w.dtype, device=cuda)
    run.check(run.lib.kmx_lloyd_sample_distances(run.plan, run.ptr(run.X_rm), run.ptr(labels), run.ptr(run.ws),
                                                 run.ptr(got), run.stream), "kmx_lloyd_sample_distances")
    exact = ((_dev(X, cuda).double() - _dev(init, cuda).double()[labels.long()]) ** 2).sum(1)
    # a difference, its square and d / 16 + 4 additions, each within an ulp of terms of one sign
    np.testing.assert_allclose(got.cpu().numpy(), exact.cpu().numpy(), rtol=(d / 16 + 8) * np.finfo(dtype).eps)
    for relocation in ("sklearn", "literal"):
        _, _, centroids_t, n_iter = drivers.lloyd(run.X_t, run.w, _dev(init.T, cuda), False, 1, False, 0.0,
                                                  relocation=relocation, flags=0)
        it = next(ok.lloyd_iterations(X, w, init, max_iter=1, tol=0.0, relocation=relocation))
        assert it["n_empty"] == 3 and n_iter == 1
        assert_centers_close(centroids_t.cpu().numpy().T, it["centers"], dtype, scale_rtol=2e-5 if dtype == np.float32 else 1e-11)


# whole-numbered features, many samples nearly as far from two centroids; the wide fp32 step, the tiled product, an
# odd number of features, the largest number of 16-feature steps, and data where the screen settles next to nothing
@pytest.mark.parametrize("n,d,k,values,offset", [(1_000_000, 100, 300, 3, 0), (400_000, 101, 64, 2, 0), (300_000, 256, 1000, 2, 0),
                                                 (200_003, 70, 300, 2, 0), (60_000, 100, 300, 3, 2000), (200_000, 129, 65, 3, 300)])
@pytest.mark.parametrize("seed", [1, 2])
def test_labels_of_a_run_are_those_of_its_centroids(cuda, n, d, k, values, offset, seed):
    """labels_ of a fit and predict() on the same data: equal, near ties included."""
    import torch

    from sklearn_numba_dpex_amd import _capi
    from sklearn_numba_dpex_amd._capi import lib
    from sklearn_numba_dpex_amd.kmeans import drivers

    gen = torch.Generator(device=cuda).manual_seed(seed)
    X = torch.randint(0, values, (n, d), generator=gen, device=cuda).float()
    X[:, 0] += offset
    w = torch.ones(n, device=cuda)
    assert lib.kmx_lloyd_resident_bytes(_capi.lloyd_plan(n, d, k, _capi.KMX_F32, 0)) > 0
    X_t = X.T.contiguous()
    for iters in (1, 3):
        labels, _, centroids_t, _ = drivers.lloyd(X_t, w, X[:k].T.contiguous(), True, iters, False, 0.0, flags=0)
        expected, _ = drivers.get_labels_inertia(X_t, centroids_t, w, True)
        assert int((labels != expected).sum()) == 0


def test_runs_that_are_refused_leave_the_words_of_others_free(cuda):
    """More runs that end with an error than there are words to announce iterations in (64): a run after them still
    announces itself (it then returns what it announced alone, and not the whole status)."""
    from sklearn_numba_dpex_amd import _capi

    rng = np.random.default_rng(0)
    X = rng.standard_normal((20_001, 100)).astype(np.float32)
    run = _ResidentRun(cuda, X, np.ones(len(X), dtype=np.float32), X[:300], 4)
    ptr, enough = run.ptr, run.ws_bytes
    for _ in range(70):
        rc = run.lib.kmx_lloyd_run(run.plan, ptr(run.X_t), ptr(run.X_rm), ptr(run.w), ptr(run.cent[0]), ptr(run.cent[1]),
                                   ptr(run.labels[0]), ptr(run.labels[1]), ptr(run.sizes), ptr(run.empty), ptr(run.ws),
                                   enough - 1, None, 0, 0, 4, run.status, run.stream)
        assert rc == -4  # KMX_ERR_WORKSPACE
    run.run(4)
    assert (run.status.n_iter, run.status.state) == (4, _capi.KMX_MAX_ITER)
    whole = _capi.LloydStatus()
    run.check(run.lib.kmx_lloyd_status_read(ptr(run.ws), whole, run.stream), "kmx_lloyd_status_read")
    assert whole.max_iter == 4 and whole.reserved[1] > 0  # (labels that the last iteration changed)
    assert run.status.reserved[1] == 0


@pytest.mark.parametrize("n,d,k,dtype", [(30_001, 14, 40, np.float32), (20_001, 100, 300, np.float32)])
def test_long_runs_come_back_to_the_interpreter(cuda, monkeypatch, n, d, k, dtype):
    """A run is several library calls of a bounded length, with Ctrl-C handled between them, and the same run."""
    from sklearn_numba_dpex_amd.kmeans import drivers

    assert drivers._iterations_per_call(100_000_000, 64, 1_000, 4) == 16
    assert drivers._iterations_per_call(1_000_000, 256, 1_024, 4) * 5e-3 <= 0.11
    X = np.random.default_rng(n).standard_normal((n, d)).astype(dtype)
    X_t, w, init = _dev(X.T, cuda), _dev(np.ones(n, dtype=dtype), cuda), _dev(X[:k].T, cuda)
    whole = drivers.lloyd(X_t, w, init, True, 50, False, 0.0, flags=0)
    assert whole[3] > 16
    asked, run = [], drivers.lib.kmx_lloyd_run

    def counted(*args):
        asked.append(args[15] - args[14])
        return run(*args)

    monkeypatch.setattr(drivers.lib, "kmx_lloyd_run", counted)
    monkeypatch.setattr(drivers, "_iterations_per_call", lambda *a: 8)
    pieces = drivers.lloyd(X_t, w, init, True, 50, False, 0.0, flags=0)
    assert len(asked) >= 3 and max(asked) == 8
    assert pieces[3] == whole[3]
    for a, b in zip(pieces[:3:2], whole[:3:2]):
        np.testing.assert_array_equal(a.cpu().numpy(), b.cpu().numpy())


@pytest.mark.parametrize("short_of", ["room", "the half-precision copy", "the row-major copy", "seeding"])
def test_runs_and_seedings_without_memory_for_copies(cuda, monkeypatch, short_of):
    """Copies of X are made where they leave as much memory again; without them the results are the same
    (up to near ties of the labels, which these data do not have)."""
    import torch

    from sklearn_numba_dpex_amd import _capi
    from sklearn_numba_dpex_amd.kmeans import drivers

    n, d, k = 400_001, 100, 300
    rng = np.random.default_rng(5)
    which = rng.integers(0, k, n)
    X = (rng.uniform(-5, 5, (k, d))[which] + rng.standard_normal((n, d))).astype(np.float32)
    X_t, w = _dev(X.T, cuda), _dev(np.ones(n, dtype=np.float32), cuda)
    init = _dev(X[np.unique(which, return_index=True)[1]].T, cuda)  # a sample of every blob: no near ties
    resident = _capi.lib.kmx_lloyd_resident_bytes(_capi.lloyd_plan(n, d, k, _capi.KMX_F32, 0))
    screen = _capi.lib.kmx_kpp_screen_bytes(n, d, 40, 5, _capi.KMX_F32)
    assert resident > 0 and screen > 0
    expected_seeds = drivers.kmeans_plusplus(X_t, w, 40, np.random.RandomState(0))
    expected = drivers.lloyd(X_t, w, init, True, 3, False, 0.0, flags=0)
    empty, refused = torch.empty, []

    def scarce(*size, **kwargs):
        want = size[0] if len(size) == 1 else size
        n_bytes = want if isinstance(want, int) and kwargs.get("dtype") == torch.uint8 else 0
        if (short_of == "the half-precision copy" and n_bytes == resident or short_of == "seeding" and n_bytes > screen or
                short_of == "the row-major copy" and want == (n, d)):
            refused.append(want)
            raise torch.cuda.OutOfMemoryError("as asked")
        return empty(*size, **kwargs)

    if short_of == "room":
        monkeypatch.setattr(drivers, "room_for", lambda n_bytes, device: refused.append(n_bytes) or False)
    else:
        monkeypatch.setattr(torch, "empty", scarce)
    seeds = drivers.kmeans_plusplus(X_t, w, 40, np.random.RandomState(0))
    got = drivers.lloyd(X_t, w, init, True, 3, False, 0.0, flags=0)
    monkeypatch.undo()
    assert refused
    np.testing.assert_array_equal(seeds[1].cpu().numpy(), expected_seeds[1].cpu().numpy())
    np.testing.assert_array_equal(got[0].cpu().numpy(), expected[0].cpu().numpy())
    np.testing.assert_allclose(got[2].cpu().numpy(), expected[2].cpu().numpy(), rtol=1e-6, atol=1e-6)
    np.testing.assert_allclose(float(got[1]), float(expected[1]), rtol=1e-6)


def test_copies_of_x_leave_as_much_memory_again(cuda, monkeypatch):
    import torch

    from sklearn_numba_dpex_amd.common import _buffers

    gib = 1 << 30
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device=None: (10 * gib, 300 * gib))
    monkeypatch.setattr(torch.cuda, "memory_reserved", lambda device=None: 7 * gib)
    monkeypatch.setattr(torch.cuda, "memory_allocated", lambda device=None: 5 * gib)
    assert _buffers.room_for(6 * gib, cuda) and not _buffers.room_for(6 * gib + 1, cuda)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device=None: (0, 300 * gib))
    assert not _buffers.room_for(gib + 1, cuda)
    assert _buffers.room_for(gib, cuda)  # (small ones are simply asked for)


# a kernel family each; the iterations enqueued behind one that stops for a relocation find label
# buffers that no iteration has written
@pytest.mark.parametrize("n,d,k,dtype", [(3_001, 14, 20, np.float32), (3_001, 40, 20, np.float64), (3_001, 10, 5, np.float64),
                                         (5_000, 70, 6, np.float32), (5_003, 100, 40, np.float64), (5_003, 100, 40, np.float32),
                                         (4_001, 128, 300, np.float32), (4_001, 14, 700, np.float32)])
def test_iterations_behind_a_stop_leave_everything_alone(cuda, n, d, k, dtype):
    import torch

    from sklearn_numba_dpex_amd import _capi
    from sklearn_numba_dpex_amd._capi import lib, ptr

    rng = np.random.default_rng(n + d)
    X = rng.standard_normal((n, d)).astype(dtype)
    init = X[:k].copy()
    init[1] = 1e3  # empty at once
    X_t, w = _dev(X.T, cuda), _dev(np.ones(n, dtype=dtype), cuda)
    plan = _capi.lloyd_plan(n, d, k, _capi.dtype_code(X_t.dtype))
    X_rm = _dev(X, cuda) if lib.kmx_lloyd_plan_reads_rowmajor(plan) else None
    cent = [_dev(init.T, cuda), torch.empty(d, k, dtype=X_t.dtype, device=cuda)]
    labels = [torch.full((n,), -16, dtype=torch.int32, device=cuda) for _ in range(2)]
    sizes, empty = torch.empty(k, dtype=X_t.dtype, device=cuda), torch.empty(k, dtype=torch.int32, device=cuda)
    ws, status = torch.empty(plan.workspace_bytes, dtype=torch.uint8, device=cuda), _capi.LloydStatus()
    stream = _capi.current_stream()
    _capi.check(lib.kmx_lloyd_init(plan, ptr(ws), plan.workspace_bytes, ptr(X_t), ptr(w), ptr(cent[0]), 9, 0.0, stream),
                "init")
    _capi.check(lib.kmx_lloyd_run(plan, ptr(X_t), ptr(X_rm), ptr(w), ptr(cent[0]), ptr(cent[1]), ptr(labels[0]),
                                  ptr(labels[1]), ptr(sizes), ptr(empty), ptr(ws), plan.workspace_bytes, None, 0, 0, 9,
                                  status, stream), "run")
    torch.cuda.synchronize()
    assert (status.state, status.n_iter, status.n_empty) == (_capi.KMX_NEED_RELOCATION, 0, 1)
    assert int(empty[0]) == 1
    assert bool((labels[0] == -16).all())
    got = labels[1].cpu().numpy().astype(np.int64)
    np.testing.assert_array_equal(sizes.cpu().numpy(), np.bincount(got, minlength=k))


# iterations that the step's last workgroup ends: either side of 16 384 partial sums (workgroups x (d + 1) k), of 256
# sums (several groups of threads per sum, several sums per thread), one and two clusters, a single workgroup; the kernels
# with the samples in registers (11), streaming them (1) and on the fp32 matrix cores (31), also at most of 64 KB of LDS
@pytest.mark.parametrize("n,d,k,dtype,flags,variant", [
    (418_816, 4, 8, np.float32, 0, 11), (418_817, 4, 8, np.float32, 0, 11), (65_536, 16, 15, np.float32, 0, 11),
    (65_537, 16, 15, np.float32, 0, 11), (32_768, 31, 8, np.float32, 0, 11), (32_769, 31, 8, np.float32, 0, 11),
    (5_000, 60, 12, np.float32, 0, 11), (6_000, 60, 12, np.float32, 0, 11), (700, 2, 1, np.float32, 0, 11),
    (32_768, 16, 15, np.float64, 0, 11), (32_769, 16, 15, np.float64, 0, 11), (9_001, 40, 8, np.float64, 0, 11),
    (700, 2, 2, np.float64, 0, 11), (100, 3, 4, np.float64, 0, 11), (20_001, 20, 8, np.float32, 1, 1),
    (7_000, 70, 8, np.float64, 1, 1), (7_700, 70, 8, np.float64, 1, 1), (20_001, 9, 45, np.float32, 0x10, 31),
    (129, 14, 16, np.float32, 0x10, 31), (9_001, 42, 126, np.float32, 0x10, 31)])
def test_iterations_ended_by_the_last_workgroup(cuda, n, d, k, dtype, flags, variant):
    """Runs of one to three iterations, the first with a relocation out of the step, against the oracle."""
    from sklearn_numba_dpex_amd import _capi
    from sklearn_numba_dpex_amd.kmeans import drivers

    assert _capi.lloyd_plan(n, d, k, _capi.dtype_code(dtype), flags).variant == variant
    rng = np.random.default_rng(n + d)
    y = np.arange(n) % k
    X = (rng.uniform(-50, 50, (k, d))[y] + rng.standard_normal((n, d))).astype(dtype)
    X[n // 2] *= 4  # the farthest sample
    init, w = X[:k].copy(), rng.uniform(0.5, 1.5, n).astype(dtype)
    if k > 2:
        init[k // 2] = 1e4
    X_t, w_d = _dev(X.T, cuda), _dev(w, cuda)
    for it in ok.lloyd_iterations(X, w, init, max_iter=3):
        assert it["n_empty"] == (1 if k > 2 and it["n_iter"] == 1 else 0)
        labels, _, centers_t, n_iter = drivers.lloyd(X_t, w_d, _dev(init.T, cuda), False, it["n_iter"], False, 0.0, flags=flags)
        assert n_iter == it["n_iter"]
        centers = centers_t.cpu().numpy().T
        assert_centers_close(centers, it["centers"], dtype)
        assert_labels_match(labels.cpu().numpy().astype(np.int64), ok.assign_labels(X, centers), X, centers)


def _small_configs():
    return {
        "C1": lambda: datasets.config1(n=100_000),
        "C2": lambda: datasets.config2(n=200_000),
        "C3": lambda: datasets.config3(n=20_000, d=256, k=1024),
        "C3s": lambda: datasets.config3(n=30_001, d=70, k=50),
        "C3m": lambda: datasets.config3(n=30_001, d=100, k=300),
        "C3w": lambda: datasets.config3(n=9_000, d=300, k=70),
        "C5": lambda: datasets.config5(n=100_000),
        "odd": lambda: _odd_config(),
        # shapes off the fast paths of the matrix-core kernels: n not a multiple of the tile or
        # of 4 (no 128-bit accesses), odd d, k not a multiple of the centroid block
        "F64a": lambda: _blob_config(10_007, 13, 37, np.float64, 11),
        "F64b": lambda: _blob_config(4_100, 30, 100, np.float64, 12),
        "F64c": lambda: _blob_config(50, 32, 16, np.float64, 13),
        "M32a": lambda: _blob_config(10_003, 9, 45, np.float32, 14),
        "M32b": lambda: _blob_config(5_000, 40, 20, np.float32, 15),
        "M32c": lambda: _blob_config(33, 14, 16, np.float32, 16),
        # wide fp32 path with very unequal clusters (bucket sizes from 0 to a third of n)
        "C3k": lambda: dict(_blob_config(40_000, 128, 64, np.float32, 17, skew=True), flags=0x3, variant=42),
        "C3k2": lambda: dict(_blob_config(40_000, 128, 64, np.float32, 17, skew=True), variant=63),
        # few features, many clusters: accumulators and centroid copies need more than 64 KB of
        # LDS, which only the screened step (one workgroup per compute unit) may take
        "M32d": lambda: dict(_blob_config(20_000, 14, 600, np.float32, 18), variant=61),
        # the same with the screen switched off, and a shape whose accumulators exceed what any
        # kernel keeps in LDS: the wide path with one chunk of features (d <= 32)
        "M32e": lambda: dict(_blob_config(20_000, 14, 600, np.float32, 18), flags=0x10, variant=42),
        # beyond the LDS of the fused screened step: its labels-only form with sums per bucket of
        # samples; the wide path on request
        "M32f": lambda: dict(_blob_config(20_000, 14, 700, np.float32, 20), variant=63),
        "M32g": lambda: dict(_blob_config(20_000, 14, 700, np.float32, 20), flags=0x3, variant=42),
        # accumulators beyond LDS off the wide fp32 path: a labels-only kernel (fp64 matrix cores
        # where the centroids fit, else vector ALU) and sums per bucket of samples
        "F64d": lambda: dict(_blob_config(20_000, 32, 500, np.float64, 19), variant=53),
        "B64a": lambda: dict(_blob_config(20_001, 100, 100, np.float64, 25), variant=63),
        "B64b": lambda: dict(_blob_config(30_000, 8, 5000, np.float64, 26), variant=63),
        "B64d": lambda: dict(_blob_config(30_000, 8, 5000, np.float64, 26), flags=0x2, variant=13),
        "B64e": lambda: dict(_blob_config(10_000, 100, 100, np.float64, 30), flags=0x1, variant=3),
        "B32a": lambda: dict(_blob_config(9_001, 300, 40, np.float32, 27, skew=True), variant=63),
        "B32b": lambda: dict(_blob_config(3_000, 784, 130, np.float32, 28), variant=63),
        "B64c": lambda: dict(_blob_config(2_999, 70, 260, np.float64, 29), variant=63),
        # the tiled product with one tile of 32 / 64 centroids
        "B32c": lambda: dict(_blob_config(5_001, 300, 20, np.float32, 31), variant=63),
        "B64f": lambda: dict(_blob_config(4_000, 100, 24, np.float64, 32), variant=63),
        "B64g": lambda: dict(_blob_config(4_003, 90, 50, np.float64, 33), variant=63),
        # cluster counts either side of where the tiled product widens its centroid tile (32, 64)
        "B32d": lambda: dict(_blob_config(3_001, 300, 32, np.float32, 68), variant=63),
        "B32e": lambda: dict(_blob_config(3_001, 300, 33, np.float32, 69), variant=63),
        "B32f": lambda: dict(_blob_config(2_000, 200, 64, np.float32, 70), variant=63),
        "B32g": lambda: dict(_blob_config(2_000, 200, 65, np.float32, 71), variant=63),
        "B64i": lambda: dict(_blob_config(2_001, 150, 32, np.float64, 72), variant=63),
        "B64j": lambda: dict(_blob_config(2_001, 150, 33, np.float64, 73), variant=63),
        "B64k": lambda: dict(_blob_config(1_500, 100, 64, np.float64, 74), variant=63),
        "B64l": lambda: dict(_blob_config(1_500, 100, 65, np.float64, 75), variant=63),
        # few clusters of wide fp64 samples: the finalisation with 64 lanes per cluster
        "B64h": lambda: dict(_blob_config(3_001, 300, 18, np.float64, 67, skew=True), variant=63),
        # few clusters: the register-resident and the streaming vector-ALU steps
        "R64a": lambda: dict(_blob_config(5_003, 50, 7, np.float64, 34), variant=11),
        "R32a": lambda: dict(_blob_config(5_003, 40, 8, np.float32, 35), variant=11),
        "S64a": lambda: dict(_blob_config(5_002, 90, 16, np.float64, 36), flags=0x1, variant=1),
        # (fp64 below a million samples leaves the streaming step to the tiled product by itself)
        "S64c": lambda: dict(_blob_config(5_002, 90, 16, np.float64, 36), variant=63),
        "S32a": lambda: dict(_blob_config(300_000, 70, 5, np.float32, 37), flags=0x1, variant=1),
        # enough samples for four (fp32) / two (fp64) consecutive samples per thread
        "S32b": lambda: dict(_blob_config(600_000, 70, 5, np.float32, 38), flags=0x1, variant=1),
        # fp32, up to 16 clusters, more than 64 features: a tile of samples in LDS serves the labels
        # and the sums (one read of X); tiles of 64, 32 and 16 samples, every unrolling of the
        # kernel, n below a tile, n not a multiple of 4, one cluster
        "K32a": lambda: dict(_blob_config(7_001, 784, 10, np.float32, 48), variant=81),
        "K32b": lambda: dict(_blob_config(20_000, 100, 10, np.float32, 49), variant=81),
        "K32c": lambda: dict(_blob_config(5_003, 65, 16, np.float32, 50), variant=81),
        "K32d": lambda: dict(_blob_config(3_002, 1216, 3, np.float32, 51), variant=81),
        "K32e": lambda: dict(_blob_config(40, 300, 2, np.float32, 52), variant=81),
        "K32f": lambda: dict(_blob_config(9_000, 257, 7, np.float32, 53), variant=81),
        "K32g": lambda: dict(_blob_config(300_000, 70, 5, np.float32, 37), variant=81),
        "K32h": lambda: dict(_blob_config(6_000, 513, 1, np.float32, 54), variant=81),
        "K32i": lambda: dict(_blob_config(8_000, 200, 12, np.float32, 55, skew=True), variant=81),
        # up to 128 features (a multiple of 4) with the row-major copy: every wave on tiles of its own
        "K32j": lambda: dict(_blob_config(50_001, 128, 16, np.float32, 56), variant=81),
        "K32k": lambda: dict(_blob_config(10_000, 68, 3, np.float32, 57), variant=81),
        "K32l": lambda: dict(_blob_config(30_003, 112, 9, np.float32, 58, skew=True), variant=81),
        # tiles that arrive in LDS directly (row-major copy, a multiple of 4 features beyond 128): four
        # waves per workgroup up to 512 features, eight beyond; fewer samples than a tile; rows of
        # exactly one, two and more than two load instructions of 64 pieces
        "K32m": lambda: dict(_blob_config(2_501, 384, 6, np.float32, 59), variant=81),
        "K32n": lambda: dict(_blob_config(9, 640, 4, np.float32, 60), variant=81),
        "K32o": lambda: dict(_blob_config(4_100, 512, 16, np.float32, 61), variant=81),
        "K32p": lambda: dict(_blob_config(1_030, 832, 5, np.float32, 62, skew=True), variant=81),
        "K32q": lambda: dict(_blob_config(777, 256, 11, np.float32, 63), variant=81),
        # the widest samples of this step: one workgroup per compute unit, with and without the row-major copy
        "K32r": lambda: dict(_blob_config(1_500, 1792, 4, np.float32, 64), variant=81),
        "K32s": lambda: dict(_blob_config(2_003, 1500, 16, np.float32, 65), variant=81),
        # enough samples for the labels-only kernel with a tile per wave, n odd (no 128-bit accesses)
        "K32t": lambda: dict(_blob_config(270_001, 96, 7, np.float32, 66), variant=81),
        "S64b": lambda: dict(_blob_config(300_000, 70, 5, np.float64, 39), flags=0x1, variant=1),
        # extremes of the tiled product: thousands of features (many passes of the bucketed sums),
        # more clusters than the bucket counts hold in LDS and than the wide path takes
        "X32a": lambda: dict(_blob_config(1_500, 3_000, 20, np.float32, 40), variant=63),
        "X32b": lambda: dict(_blob_config(30_000, 8, 9_000, np.float32, 41), variant=63),
        "X64a": lambda: dict(_blob_config(12_000, 3, 5_000, np.float64, 42), variant=63),
        # the tiled product screened on the fp16 matrix cores (on request), the uncertified
        # samples through the listed fp32 pass
        "G32s": lambda: dict(_blob_config(6_001, 100, 100, np.float32, 43), flags=0x20, variant=63),
        "G32t": lambda: dict(_blob_config(3_000, 784, 40, np.float32, 44, skew=True), flags=0x20, variant=63),
        "G32u": lambda: dict(_blob_config(5_000, 70, 20, np.float32, 45), flags=0x20, variant=63),
        # fp64 on the matrix cores beyond 32 features (no rows in flight for the next tile) and
        # with accumulators that need most of a compute unit's LDS
        # (fp64 inputs up to 64 features: labels screened on the fp16 matrix cores, the rest in
        # fp64 - variant 71; with the screen switched off the all-fp64 matrix-core step, 51)
        "F64e": lambda: dict(_blob_config(20_003, 48, 64, np.float64, 21), variant=71),
        # (64 features x 100 clusters: the fp64 and fp32 copies of the centroids do not both fit the LDS)
        "F64f": lambda: dict(_blob_config(8_000, 64, 100, np.float64, 22), variant=51),
        "F64g": lambda: dict(_blob_config(20_000, 32, 300, np.float64, 23), variant=51),
        "F64h": lambda: dict(_blob_config(6_001, 61, 33, np.float64, 24), variant=71),
        "F64e1": lambda: dict(_blob_config(20_003, 48, 64, np.float64, 21), flags=0x10, variant=51),
        "F64h1": lambda: dict(_blob_config(6_001, 61, 33, np.float64, 24), flags=0x10, variant=51),
        "C5f": lambda: dict(datasets.config5(n=100_000), flags=0x10, variant=51),
        # fp64 screened step, one K step of 16 features with and without a spare slot
        "F64i": lambda: dict(_blob_config(30_000, 16, 127, np.float64, 46), variant=71),
        "F64j": lambda: dict(_blob_config(30_004, 14, 127, np.float64, 47), variant=71),
    }


def _blob_config(n, d, k, dtype, seed, skew=False):
    rng = np.random.default_rng(seed)
    centers = rng.uniform(-10, 10, (k, d))
    p = rng.dirichlet(np.full(k, 0.15)) if skew else np.full(k, 1.0 / k)
    y = rng.choice(k, size=n, p=p)
    X = (centers[y] + rng.standard_normal((n, d))).astype(dtype)
    init = X[rng.choice(n, k, replace=False)].copy()
    w = rng.uniform(0.5, 1.5, n).astype(dtype)
    return dict(X=X, init=init, sample_weight=w, k=k, max_iter=20, tol=0.0, name=f"blob{seed}")


def _odd_config():
    """Ragged shapes: n not a multiple of anything, d = 3, k = 5, fp64."""
    rng = np.random.default_rng(7)
    X = rng.normal(size=(1237, 3))
    init = X[rng.choice(1237, 5, replace=False)].copy()
    return dict(X=X, init=init, sample_weight=rng.uniform(0.5, 2, 1237), k=5, max_iter=50, tol=0.0, name="odd")


@pytest.mark.parametrize("rowmajor", [False, True])
@pytest.mark.parametrize("name", ["C1", "C2", "C3", "C3s", "C3m", "C3w", "C5", "odd", "F64a", "F64b", "F64c",
                                  "M32a", "M32b", "M32c", "C3k", "M32d", "M32e", "M32f", "M32g", "F64d", "F64e", "F64f",
                                  "F64g", "F64h", "F64e1", "F64h1", "C5f", "F64i", "F64j", "B64a", "B64b", "B32a", "B32b", "B64c", "B64d", "B64e", "C3k2", "B32c", "B64f", "B64g", "B64h", "B32d", "B32e", "B32f", "B32g", "B64i", "B64j", "B64k", "B64l", "R64a", "R32a", "S64a", "S64c", "S32a", "S32b", "S64b", "X32a", "X32b", "X64a", "G32s", "G32t", "G32u",
                                  "K32a", "K32b", "K32c", "K32d", "K32e", "K32f", "K32g", "K32h", "K32i",
                                  "K32j", "K32k", "K32l", "K32m", "K32n", "K32o", "K32p", "K32q", "K32r", "K32s"])
def test_single_iteration_through_c_abi(cuda, name, rowmajor):
    import torch

    from sklearn_numba_dpex_amd import _capi
    from sklearn_numba_dpex_amd._capi import lib, ptr

    cfg = _small_configs()[name]()
    X, init, w, k = cfg["X"], cfg["init"], cfg["sample_weight"], cfg["k"]
    n, d = X.shape
    dc = _capi.dtype_code(X.dtype)
    X_t = _dev(X.T, cuda)
    w_d = _dev(w, cuda)
    c_in = _dev(init.T, cuda)
    c_out = torch.empty_like(c_in)
    labels_prev = torch.zeros(n, dtype=torch.int32, device=cuda)
    labels = torch.empty(n, dtype=torch.int32, device=cuda)
    sizes = torch.empty(k, dtype=X_t.dtype, device=cuda)
    empty = torch.empty(k, dtype=torch.int32, device=cuda)
    plan = _capi.lloyd_plan(n, d, k, dc, cfg.get("flags", 0))
    if "variant" in cfg:
        assert plan.variant == cfg["variant"]
    ws_bytes = plan.workspace_bytes
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=cuda)
    stream = _capi.current_stream()
    _capi.check(lib.kmx_lloyd_init(plan, ptr(ws), ws_bytes, ptr(X_t), ptr(w_d), ptr(c_in), 100, 0.0, stream), "init")
    if rowmajor and plan.variant not in (42, 3, 13, 53, 63, 81):
        pytest.skip("the row-major copy is only used by the wide fp32 path, the bucketed sums and the few-cluster step")
    X_rm = _dev(X, cuda) if rowmajor else None
    _capi.check(lib.kmx_lloyd_iter(plan, ptr(X_t), ptr(X_rm), ptr(w_d), ptr(c_in), ptr(c_out), ptr(labels_prev),
                                   ptr(labels), ptr(sizes), ptr(empty), ptr(ws), ws_bytes, stream), "iter")
    status = _capi.LloydStatus()
    _capi.check(lib.kmx_lloyd_status_read(ptr(ws), status, stream), "status")

    ref_labels = ok.assign_labels(X, init)
    n_ties = assert_labels_match(labels.cpu().numpy(), ref_labels, X, init)
    got_labels = labels.cpu().numpy().astype(np.int64)
    sums, ref_sizes = ok.weighted_sums(X, w, got_labels, k)
    n_empty = int(np.count_nonzero(ref_sizes == 0))
    assert status.n_empty == n_empty
    np.testing.assert_allclose(sizes.cpu().numpy(), ref_sizes, rtol=RTOL[X.dtype])
    if n_empty:
        assert status.state == _capi.KMX_NEED_RELOCATION
        assert status.n_iter == 0
        np.testing.assert_array_equal(empty.cpu().numpy()[:n_empty], np.flatnonzero(ref_sizes == 0))
        got = c_out.cpu().numpy().T
        assert_centers_close(got, sums, X.dtype)
    else:
        assert status.state == _capi.KMX_RUNNING
        assert status.n_iter == 1
        ref_centers = sums / ref_sizes[:, None]
        assert_centers_close(c_out.cpu().numpy().T, ref_centers, X.dtype)
        shift = float(np.sum((np.asarray(init, np.float64) - ref_centers.astype(np.float64)) ** 2))
        assert status.shift_sum == pytest.approx(shift, rel=1e-4)
        expected_changed = int(np.count_nonzero(got_labels != 0))
        assert status.reserved[1] == expected_changed
    print(f"{name}: near-tie label differences: {n_ties}")


@pytest.mark.parametrize("name", ["C2", "M32a", "M32b", "C3", "C3s", "C5", "C5f", "F64j", "F64d", "B64a", "B64d", "B64e", "odd", "S64a", "K32a", "K32b"])
def test_duplicate_and_identical_centroids_on_every_kernel_family(cuda, name):
    """Exact ties: with two centroids duplicated no sample may take the copy with the higher
    index, with all centroids identical every label is 0 (the reference's strict '<' in
    increasing centroid order), whichever label kernel the shape selects."""
    import torch

    from sklearn_numba_dpex_amd import _capi
    from sklearn_numba_dpex_amd._capi import lib, ptr

    cfg = _small_configs()[name]()
    X, w, k = cfg["X"], cfg["sample_weight"], cfg["k"]
    n, d = X.shape
    dc = _capi.dtype_code(X.dtype)
    X_t, w_d = _dev(X.T, cuda), _dev(w, cuda)
    labels_prev = torch.zeros(n, dtype=torch.int32, device=cuda)
    labels = torch.empty(n, dtype=torch.int32, device=cuda)
    sizes = torch.empty(k, dtype=X_t.dtype, device=cuda)
    empty = torch.empty(k, dtype=torch.int32, device=cuda)
    plan = _capi.lloyd_plan(n, d, k, dc, cfg.get("flags", 0))
    ws = torch.empty(plan.workspace_bytes, dtype=torch.uint8, device=cuda)
    stream = _capi.current_stream()

    def one_iteration(init):
        c_in = _dev(init.T, cuda)
        c_out = torch.empty_like(c_in)
        _capi.check(lib.kmx_lloyd_init(plan, ptr(ws), plan.workspace_bytes, ptr(X_t), ptr(w_d), ptr(c_in), 100, 0.0,
                                       stream), "init")
        _capi.check(lib.kmx_lloyd_iter(plan, ptr(X_t), None, ptr(w_d), ptr(c_in), ptr(c_out), ptr(labels_prev),
                                       ptr(labels), ptr(sizes), ptr(empty), ptr(ws), plan.workspace_bytes, stream),
                    "iter")
        return labels.cpu().numpy().astype(np.int64)

    init = cfg["init"].copy()
    init[k - 1] = init[0]
    init[k // 2] = init[1]
    got = one_iteration(init)
    assert not np.any(got == k - 1) and not np.any(got == k // 2)
    assert_labels_match(got, ok.assign_labels(X, init), X, init)

    init = cfg["init"].copy()
    init[:] = init[0]
    assert np.all(one_iteration(init) == 0)


@pytest.mark.parametrize("name", ["C1", "C2", "C3s", "C3w", "odd", "F64a", "F64b", "M32a", "M32b", "C3k", "M32d", "M32e", "F64d",
                                  "F64e", "F64f", "F64g", "F64h", "F64e1", "F64h1", "C5f", "F64i", "F64j", "B64a", "B64b", "B32a", "B32b", "B64c", "B64d", "B64e", "C3k2", "B32c", "B64f", "B64g", "B64h", "R64a", "R32a", "S64a", "S32a", "G32s", "G32t",
                                  # (not K32d: with 1216 features two fp32 evaluations of a score differ by up
                                  # to 2e-6 of its size, more than the near-tie rule's 1e-6 - one label in ten
                                  # iterations of 3002 samples)
                                  "K32a", "K32b", "K32c", "K32f", "K32i", "K32m", "K32o", "K32q"])
def test_lockstep_iterations_match_oracle(cuda, name):
    """Ten iterations, each compared from identical inputs: the oracle repeats every GPU
    iteration from the centroids the GPU started it with (a Lloyd trajectory at tol = 0 is
    chaotic, so free-running trajectories may only be compared until the first near-tie)."""
    import torch

    from sklearn_numba_dpex_amd import _capi
    from sklearn_numba_dpex_amd._capi import lib, ptr

    cfg = _small_configs()[name]()
    X, init, w, k = cfg["X"], cfg["init"], cfg["sample_weight"], cfg["k"]
    n, d = X.shape
    dc = _capi.dtype_code(X.dtype)
    X_t, w_d = _dev(X.T, cuda), _dev(w, cuda)
    cent = [_dev(init.T, cuda), None]
    cent[1] = torch.empty_like(cent[0])
    labels = [torch.zeros(n, dtype=torch.int32, device=cuda) for _ in range(2)]
    sizes = torch.empty(k, dtype=X_t.dtype, device=cuda)
    empty = torch.empty(k, dtype=torch.int32, device=cuda)
    plan = _capi.lloyd_plan(n, d, k, dc, cfg.get("flags", 0))
    ws_bytes = plan.workspace_bytes
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=cuda)
    stream = _capi.current_stream()
    status = _capi.LloydStatus()
    _capi.check(lib.kmx_lloyd_init(plan, ptr(ws), ws_bytes, ptr(X_t), ptr(w_d), ptr(cent[0]), 100, 0.0, stream), "init")
    prev = None
    for it in range(10):
        a, b = it % 2, (it + 1) % 2
        c_in = cent[a].cpu().numpy().T.copy()
        _capi.check(lib.kmx_lloyd_iter(plan, ptr(X_t), None, ptr(w_d), ptr(cent[a]), ptr(cent[b]), ptr(labels[a]),
                                       ptr(labels[b]), ptr(sizes), ptr(empty), ptr(ws), ws_bytes, stream),
                    "iter")
        _capi.check(lib.kmx_lloyd_status_read(ptr(ws), status, stream), "status")
        got = labels[b].cpu().numpy().astype(np.int64)
        assert_labels_match(got, ok.assign_labels(X, c_in), X, c_in)
        sums, ref_sizes = ok.weighted_sums(X, w, got, k)
        if status.n_empty > 0:
            # an empty cluster appeared: the iteration waits for the host's relocation
            assert status.state == _capi.KMX_NEED_RELOCATION and status.n_iter == it
            assert status.n_empty == int(np.count_nonzero(ref_sizes == 0))
            break
        assert status.n_iter == it + 1
        assert_centers_close(cent[b].cpu().numpy().T, sums / ref_sizes[:, None], X.dtype)
        if prev is not None:
            assert status.reserved[1] == int(np.count_nonzero(got != prev))
        prev = got
        if status.state != _capi.KMX_RUNNING:
            assert status.state == _capi.KMX_CONVERGED_STRICT and np.array_equal(got, prev)
            break


@pytest.mark.parametrize("name", ["C1", "C2", "C3s", "C3m", "C5", "odd"])
def test_full_lloyd_run_matches_oracle(cuda, name):
    from sklearn_numba_dpex_amd.kmeans import drivers

    cfg = _small_configs()[name]()
    if name == "C2":
        cfg = datasets.config2(n=50_000)
    X, init, w, k = cfg["X"], cfg["init"], cfg["sample_weight"], cfg["k"]
    max_iter = min(cfg["max_iter"], 30)
    Xc = X - X.mean(axis=0).astype(X.dtype)
    initc = init - X.mean(axis=0).astype(X.dtype)
    tol = 0.0
    labels, inertia, centers_t, n_iter = drivers.lloyd(
        _dev(Xc.T, cuda), _dev(w, cuda), _dev(initc.T, cuda), False, max_iter=max_iter, tol=tol
    )
    ref_labels, ref_inertia, ref_centers, ref_n_iter = ok.lloyd(Xc, w, initc, max_iter=max_iter, tol=tol)
    assert n_iter == ref_n_iter
    centers = centers_t.cpu().numpy().T
    got = labels.cpu().numpy().astype(np.int64)
    # the returned labels are the argmin for the returned centroids, whatever the trajectory
    assert_labels_match(got, ok.assign_labels(Xc, centers), Xc, centers)
    assert float(inertia) == pytest.approx(float(ok.inertia(Xc, w, centers, got)), rel=1e-5)
    if np.array_equal(got, ref_labels.astype(np.int64)):
        # same final partition: centroids must agree to rounding
        # (ten roundings of 1e-5 / 1e-12: the two runs agree iteration by iteration, each
        # within the per-iteration tolerance, and the iterations contract towards the fixed point)
        assert_centers_close(centers, ref_centers, X.dtype, scale_rtol=RTOL[X.dtype] * 10)
        assert float(inertia) == pytest.approx(float(ref_inertia), rel=1e-5)
    else:
        # a near-tie flipped somewhere along the run: a few samples at a boundary, not another
        # clustering (per-iteration parity is what the lockstep test above asserts)
        assert np.count_nonzero(got != ref_labels.astype(np.int64)) <= max(1, n_samples_differ_cap(X))
        assert float(inertia) == pytest.approx(float(ref_inertia), rel=1e-4)


def _converging_configs():
    """Cases whose Lloyd run at tol = 0 reaches strict convergence (an iteration that changes no
    label) well below max_iter = 100.  Per case: the data, the kernel variant the plan must
    choose, and the iteration count of the oracle (found on the CPU; scikit-learn's Cython loop
    takes the same number when run on 8 threads, but its own count moves with its thread count
    - 43 instead of 39 on C1 with 4 threads - because its per-thread partial sums round
    differently and a Lloyd trajectory at tol = 0 amplifies every flipped near-tie)."""
    return {
        # 100 000 x 14, 127 clusters at full size (fused screened step, sums corrected per moved sample)
        "C1": (lambda: datasets.config1(), 61, 39),
        # 14 features, 127 clusters (weighted, unequal blobs, one cluster empties and is relocated) and
        # 32 features, 64 clusters (fp64, sixteen clusters that empty on the first iteration) on fewer samples
        "C2_30k": (lambda: datasets.config2(n=30_000), 61, 38),
        "C5_100k": (lambda: datasets.config5(n=100_000), 71, 67),
        # screened labels with the sums taken straight from the labels, and with sums per bucket
        "direct": (lambda: _blob_config(20_000, 14, 700, np.float32, 20), 63, 8),
        "bucket": (lambda: _blob_config(20_000, 32, 500, np.float64, 19), 53, 8),
    }


@pytest.mark.parametrize("name", ["C1", "C2_30k", "C5_100k", "direct", "bucket"])
def test_n_iter_at_real_strict_convergence(cuda, name):
    """n_iter must be identical at tol = 0: whole runs with max_iter = 100 that stop because an
    iteration changed no label, not because of the cap, against the oracle, and against
    scikit-learn's own Lloyd loop wherever that one stayed on the oracle's trajectory."""
    from sklearn.cluster._kmeans import _kmeans_single_lloyd

    from sklearn_numba_dpex_amd import _capi
    from sklearn_numba_dpex_amd.kmeans import drivers

    make, variant, expected_n_iter = _converging_configs()[name]
    cfg = make()
    X, init, w, k = cfg["X"], cfg["init"], cfg["sample_weight"], cfg["k"]
    n, d = X.shape
    assert _capi.lloyd_plan(n, d, k, _capi.dtype_code(X.dtype), 0).variant == variant
    mean = X.mean(axis=0).astype(X.dtype)
    Xc, initc = X - mean, init - mean
    max_iter = 100
    labels, inertia, centers_t, n_iter = drivers.lloyd(
        _dev(Xc.T, cuda), _dev(w, cuda), _dev(initc.T, cuda), False, max_iter=max_iter, tol=0.0
    )
    ref_labels, ref_inertia, ref_centers, ref_n_iter = ok.lloyd(Xc, w, initc, max_iter=max_iter, tol=0.0)
    # the case is not decided by the cap
    assert ref_n_iter == expected_n_iter < max_iter
    assert n_iter == ref_n_iter
    centers = centers_t.cpu().numpy().T
    got = labels.cpu().numpy().astype(np.int64)
    # strict convergence: the returned labels are those of the last iteration and the argmin for
    # the returned centroids
    assert_labels_match(got, ok.assign_labels(Xc, centers), Xc, centers)
    assert float(inertia) == pytest.approx(float(ok.inertia(Xc, w, centers, got)), rel=RTOL[X.dtype] * 10)
    n_diff = np.count_nonzero(got != ref_labels.astype(np.int64))
    if n_diff == 0:
        # same final partition: the centroids are the same weighted means, 1e-5 / 1e-12
        assert_centers_close(centers, ref_centers, X.dtype)
        assert float(inertia) == pytest.approx(float(ref_inertia), rel=RTOL[X.dtype] * 10)
    else:
        # a near-tie went the other way in some iteration and the run ended in a neighbouring
        # fixed point after the same number of iterations: a few boundary samples (iteration by
        # iteration parity from identical inputs is what the lockstep tests assert)
        assert n_diff <= n_samples_differ_cap(X)
        assert float(inertia) == pytest.approx(float(ref_inertia), rel=1e-4)
    sk_labels, sk_inertia, sk_centers, sk_n_iter = _kmeans_single_lloyd(
        Xc, w, initc.copy(), max_iter=max_iter, tol=0.0, n_threads=8
    )
    if np.array_equal(sk_labels, ref_labels):
        # scikit-learn ended in the oracle's partition: it took the oracle's path
        assert n_iter == sk_n_iter
    assert float(inertia) == pytest.approx(float(sk_inertia), rel=1e-3)


def test_lockstep_to_strict_convergence_where_free_runs_part_ways(cuda):
    """configs[1] on 100 000 samples: at iteration 3 one sample lies within 4e-9 (relative) of a
    bisector, the kernel and the oracle label it differently, and from there the two free runs
    (and scikit-learn's) follow different trajectories: 69, 84 and 84 iterations.  What can be
    pinned there is every single iteration up to the end: the oracle repeats each iteration from
    the centroids the GPU started it with, through the relocation of the cluster that empties, and
    the run must stop at the first iteration whose labels equal the previous ones."""
    import torch

    from sklearn_numba_dpex_amd import _capi
    from sklearn_numba_dpex_amd._capi import lib, ptr
    from sklearn_numba_dpex_amd.kmeans import drivers

    cfg = datasets.config2(n=100_000)
    X, init, w, k = cfg["X"], cfg["init"], cfg["sample_weight"], cfg["k"]
    mean = X.mean(axis=0).astype(X.dtype)
    X, init = X - mean, init - mean
    n, d = X.shape
    dc = _capi.dtype_code(X.dtype)
    X_t, w_d = _dev(X.T, cuda), _dev(w, cuda)
    cent = [_dev(init.T, cuda), None]
    cent[1] = torch.empty_like(cent[0])
    labels = [torch.zeros(n, dtype=torch.int32, device=cuda) for _ in range(2)]
    sizes = torch.empty(k, dtype=X_t.dtype, device=cuda)
    empty = torch.empty(k, dtype=torch.int32, device=cuda)
    plan = _capi.lloyd_plan(n, d, k, dc, 0)
    assert plan.variant == 61
    ws_bytes = plan.workspace_bytes
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=cuda)
    stream = _capi.current_stream()
    status = _capi.LloydStatus()
    _capi.check(lib.kmx_lloyd_init(plan, ptr(ws), ws_bytes, ptr(X_t), ptr(w_d), ptr(cent[0]), 100, 0.0, stream), "init")
    prev = None
    n_relocations = 0
    for it in range(100):
        a, b = it % 2, (it + 1) % 2
        c_in = cent[a].cpu().numpy().T.copy()
        _capi.check(lib.kmx_lloyd_iter(plan, ptr(X_t), None, ptr(w_d), ptr(cent[a]), ptr(cent[b]), ptr(labels[a]),
                                       ptr(labels[b]), ptr(sizes), ptr(empty), ptr(ws), ws_bytes, stream), "iter")
        _capi.check(lib.kmx_lloyd_status_read(ptr(ws), status, stream), "status")
        got = labels[b].cpu().numpy().astype(np.int64)
        assert_labels_match(got, ok.assign_labels(X, c_in), X, c_in)
        sums, ref_sizes = ok.weighted_sums(X, w, got, k)
        if status.state == _capi.KMX_NEED_RELOCATION:
            n_relocations += 1
            assert status.n_empty == int(np.count_nonzero(ref_sizes == 0)) and status.n_iter == it
            drivers._relocate_empty_clusters(status.n_empty, X_t, w_d, cent[b], sizes, labels[b], empty, cent[a])
            _capi.check(lib.kmx_lloyd_finalize(plan, ptr(cent[a]), ptr(cent[b]), ptr(sizes), ptr(ws), ws_bytes, stream),
                        "finalize")
            _capi.check(lib.kmx_lloyd_status_read(ptr(ws), status, stream), "status")
            ok.relocate_empty_clusters(X, w, sums, ref_sizes, got, ok.sq_dist_to_assigned(X, c_in, got))
        assert status.n_iter == it + 1
        assert_centers_close(cent[b].cpu().numpy().T, sums / ref_sizes[:, None], X.dtype)
        strict = prev is not None and np.array_equal(got, prev)
        assert (status.state == _capi.KMX_CONVERGED_STRICT) == strict
        if strict:
            break
        assert status.state == _capi.KMX_RUNNING
        prev = got
    assert status.state == _capi.KMX_CONVERGED_STRICT and n_relocations >= 1
    # the driver's own loop (iterations enqueued ahead) stops at the same iteration
    n_iter = drivers.lloyd(X_t, w_d, _dev(init.T, cuda), False, max_iter=100, tol=0.0)[3]
    assert n_iter == status.n_iter


def n_samples_differ_cap(X):
    return X.shape[0] // 1000


@pytest.mark.parametrize("name", ["C3s", "C3w", "C3k2", "F64d", "F64e", "F64h", "F64i", "F64j", "C5", "B64a", "B64b", "B32a", "B32b", "B64c", "odd", "B32c", "B64f", "B64g", "B64h", "B32d", "B32e", "B32f", "B32g", "B64i", "B64j", "B64k", "B64l", "R64a", "R32a", "S64a", "S32a",
                                  # few clusters on wide samples: the labels-only matrix-core kernel that reads
                                  # the feature-major array directly (tiles of 32 and of 64 samples, every width
                                  # of its centroid registers, n odd, n below a tile) and the inertia summed
                                  # with the features split over workgroups
                                  "K32a", "K32b", "K32d", "K32e", "K32f", "K32g", "K32j", "K32m", "K32n", "K32o", "K32p", "K32r", "K32s", "K32t"])
def test_labels_and_score_paths_on_every_label_kernel(cuda, name):
    """kmx_assign_labels, labels + inertia in one call and the distances on the shapes of the
    tiled matrix-core product, of the labels-only fp64 matrix-core kernel, of the vector-ALU
    kernels and of the few-cluster kernels, against the oracle."""
    import torch

    from sklearn_numba_dpex_amd.kmeans import drivers

    cfg = _small_configs()[name]()
    X, init, w = cfg["X"], cfg["init"], cfg["sample_weight"]
    n = X.shape[0]
    X_t, C_t, w_d = _dev(X.T, cuda), _dev(init.T, cuda), _dev(w, cuda)
    ref = ok.assign_labels(X, init)
    labels = torch.full((n,), -1, dtype=torch.int32, device=cuda)
    drivers._assign(X_t, C_t, labels)
    got = labels.cpu().numpy().astype(np.int64)
    assert_labels_match(got, ref, X, init)
    labels2, inertia = drivers.get_labels_inertia(X_t, C_t, w_d, True)
    np.testing.assert_array_equal(labels2.cpu().numpy().astype(np.int64), got)
    assert float(inertia[0]) == pytest.approx(float(ok.inertia(X, w, init, got)), rel=RTOL[X.dtype] * 5)
    dist = drivers.get_euclidean_distances(X_t[:, :512].contiguous(), C_t).cpu().numpy()
    exact = np.sqrt(((X[:512].astype(np.float64)[:, None, :] - init.astype(np.float64)[None, :, :]) ** 2).sum(axis=2))
    np.testing.assert_allclose(dist, exact, rtol=RTOL[X.dtype] * 2, atol=RTOL[X.dtype])


@pytest.mark.parametrize("n,d,k", [
    (3_001, 4, 300),    # the fewest features that are screened; accumulators of the step beyond LDS
    (3_001, 3, 1_000),  # one feature fewer: fp64 products
    (2_000, 16, 700),   # no spare feature slot for the half norms
    (2_003, 17, 250), (2_004, 33, 230), (1_999, 50, 150),
    (130, 64, 128),     # two tiles of samples and a remainder
    (63, 63, 40),       # less than a tile
    (2_000, 64, 190),   # operands beyond LDS
    # either side of the lines between the screen and the product: few features, wide samples, odd sample counts
    (200_001, 4, 600), (199_999, 4, 600), (3_001, 6, 800), (2_001, 24, 260), (2_001, 23, 260), (65_537, 24, 260),
    (200_001, 17, 300), (100_001, 33, 230), (100_001, 56, 120), (100_001, 57, 115), (100_000, 64, 100), (99_996, 49, 140),
    (2_004, 48, 160),
])
def test_fp64_labels_where_only_the_labels_fit_the_lds(cuda, n, d, k):
    import torch

    from sklearn_numba_dpex_amd.kmeans import drivers

    rng = np.random.default_rng(n + d)
    C = rng.uniform(-5, 5, (k, d))
    C[k // 2] = C[3]  # of equal centroids the first
    X = C[rng.integers(0, k, n)] + 0.5 * rng.standard_normal((n, d))
    labels = torch.full((n,), -1, dtype=torch.int32, device=cuda)
    X_t, C_t = _dev(X.T, cuda), _dev(C.T, cuda)
    drivers._assign(X_t, C_t, labels)
    got = labels.cpu().numpy().astype(np.int64)
    assert_labels_match(got, ok.assign_labels(X, C), X, C)
    assert not (got == k // 2).any()
    w = rng.uniform(0.5, 1.5, n)
    labels2, inertia = drivers.get_labels_inertia(X_t, C_t, _dev(w, cuda), True)
    np.testing.assert_array_equal(labels2.cpu().numpy(), got)
    assert float(inertia[0]) == pytest.approx(float(ok.inertia(X, w, C, got)), rel=RTOL[X.dtype] * 5)
