"""GPU tests of the Lloyd iterations that look only at samples whose label can have changed
(csrc/lloyd_bounds.hip): whole runs with the memory they need and without it, which has every
iteration read all of X.  Labels, centroids, cluster sizes and the number of iterations are the same bit
for bit: sums are integers, and what is passed over is proven unchanged.  The screened steps
themselves are compared with the oracle in test_gpu_lloyd_screen.py."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MARK = 0xFF


def _drift_and_words(area, n, k):
    import torch

    # drift of the labels (two copies), then a word per sample
    return (area[:2 * k * 4].view(torch.float32).view(2, k),
            area[(2 * k * 4 + 255) // 256 * 256:][: 4 * n].view(torch.int32))


def _entered(area, n, k):
    """Whether a bounded iteration has written the area (all of its words: the entering one does), or none has."""
    # (conditions first: pytest iterates over the tensors of a comparison that an assert contains)
    _, words = _drift_and_words(area, n, k)
    written, labels_fit = bool((words != -1).all()), bool(((words & 0x7FF) < k).all())
    untouched = bool((area == MARK).all())
    assert untouched or (written and labels_fit)
    return not untouched


def _run(X_t, w, init_t, max_iter, with_bounds, must_enter=True):
    import torch

    from sklearn_numba_dpex_amd import _capi
    from sklearn_numba_dpex_amd._capi import check, lib, ptr

    (d, n), k, dev = X_t.shape, init_t.shape[1], X_t.device
    plan = _capi.lloyd_plan(n, d, k, _capi.dtype_code(X_t.dtype), 0)
    need = lib.kmx_lloyd_bounds_bytes(plan)
    assert need > 0
    area = torch.full((need,), MARK, dtype=torch.uint8, device=dev) if with_bounds else None
    ws = torch.empty(plan.workspace_bytes, dtype=torch.uint8, device=dev)
    cent = [init_t.clone(), torch.empty_like(init_t)]
    labels = [torch.empty(n, dtype=torch.int32, device=dev) for _ in range(2)]
    sizes, empty = torch.empty(k, dtype=X_t.dtype, device=dev), torch.empty(k, dtype=torch.int32, device=dev)
    status, stream = _capi.LloydStatus(), _capi.current_stream()
    check(lib.kmx_lloyd_init(plan, ptr(ws), ws.numel(), ptr(X_t), ptr(w), ptr(cent[0]), max_iter, 0.0, stream), "init")
    check(lib.kmx_lloyd_run(plan, ptr(X_t), None, ptr(w), ptr(cent[0]), ptr(cent[1]), ptr(labels[0]), ptr(labels[1]),
                            ptr(sizes), ptr(empty), ptr(ws), ws.numel(), ptr(area), need, 0, max_iter, status, stream), "run")
    torch.cuda.synchronize()
    uncertain = ctypes.c_uint32(0)
    check(lib.kmx_lloyd_recheck_count(plan, ptr(ws), ctypes.byref(uncertain), stream), "recheck")
    if with_bounds and must_enter is not None:
        assert _entered(area, n, k) == must_enter
    if with_bounds and must_enter:
        drift, words = _drift_and_words(area, n, k)
        # a drift above zero comes from an iteration behind the entering one; and words with a margin above the drift by now
        # are of samples that the next iteration passes over
        by_now = drift.max(0).values
        assert float(by_now.min()) > 0.0, "no iteration behind the entering one has run"
        passed = float(((words & ~0x7FF).view(torch.float32) > by_now[(words & 0x7FF).long()]).double().mean())
        assert passed > 0.5
    at = status.n_iter % 2
    return dict(n_iter=status.n_iter, state=status.state, labels=labels[at], cent=cent[at], sizes=sizes,
                uncertain=uncertain.value)


def _same(a, b):
    assert (a["n_iter"], a["state"]) == (b["n_iter"], b["state"])
    differ = [name for name in ("labels", "sizes", "cent") if not bool((a[name] == b[name]).all())]
    assert not differ


def _blobs(n, d, k, dtype, seed, cuda, spread=5.0):
    import torch

    gen = torch.Generator(device=cuda).manual_seed(seed)
    blobs = k * 3 // 4  # (every third blob has two centroids: labels keep moving, and no cluster empties)
    centres = (torch.rand(blobs, d, generator=gen, device=cuda) * 2 - 1) * spread
    std = 0.5 + 1.5 * torch.rand(blobs, generator=gen, device=cuda)
    which = torch.arange(n, device=cuda) % blobs
    X = centres[which] + std[which, None] * torch.randn(n, d, generator=gen, device=cuda)
    X_t = X.to(dtype).T.contiguous()
    w = 0.5 + torch.rand(n, generator=gen, device=cuda, dtype=dtype)
    init = X_t[:, :k].contiguous()
    return X_t, w, init


# feature counts on both sides of the steps of 16 and of rows of 8; clusters on both sides of 32 and 64; sample
# counts off every unit (128 words, 32 samples); each number of K steps in both types
@pytest.mark.parametrize("n, d, k, dtype", [
    (900_001, 14, 127, "float32"), (1_300_033, 16, 33, "float32"), (800_127, 17, 64, "float32"),
    (500_031, 33, 65, "float32"), (400_001, 48, 100, "float32"), (400_129, 49, 31, "float32"), (300_001, 64, 100, "float32"),
    (800_001, 13, 64, "float64"), (400_003, 32, 64, "float64"), (330_000, 33, 17, "float64"), (250_127, 49, 40, "float64"),
    (200_001, 64, 48, "float64"),
])
def test_same_as_iterations_over_all_samples(n, d, k, dtype, cuda):
    import torch

    X_t, w, init = _blobs(n, d, k, getattr(torch, dtype), 7, cuda)
    a = _run(X_t, w, init, 40, False)
    b = _run(X_t, w, init, 40, True)
    assert a["n_iter"] > 10
    _same(a, b)
    # samples without a certificate: a few of those looked at, none of the others (the bounds are nearly the same)
    assert b["uncertain"] <= 2 * a["uncertain"] + 16 and a["uncertain"] < n // 20


def test_samples_on_the_bisector_and_more_of_them_than_the_list_holds(cuda):
    """Two clusters that mirror each other exactly, and samples of weight zero on the plane between them: ties in
    every iteration, which go to the lower index; with 5e6 samples and 2.9 % on the plane a workgroup meets
    about 570 of them, beside some 200 that are close by themselves, and its list holds 640."""
    import torch

    n, d, k = 5_000_000, 10, 20
    X_t, w, init = _blobs(n, d, k, torch.float32, 3, cuda)
    half, on_plane = 200_000, int(0.029 * n)
    gen = torch.Generator(device=cuda).manual_seed(1)
    side = 40.0 + torch.randn(d, half, generator=gen, device=cuda)
    X_t[:, :half] = side
    X_t[:, half:2 * half] = side
    X_t[0, half:2 * half] *= -1.0
    w[half:2 * half] = w[:half]
    plane = slice(2 * half, 2 * half + on_plane)
    X_t[:, plane] = 40.0 + torch.randn(d, on_plane, generator=gen, device=cuda)
    X_t[0, plane] = 0.0
    w[plane] = 0.0
    order = torch.randperm(n, generator=gen, device=cuda)
    init[:, 3], init[:, 11] = X_t[:, 0], X_t[:, half]
    X_t, w = X_t[:, order].contiguous(), w[order].contiguous()
    a = _run(X_t, w, init, 24, False)
    b = _run(X_t, w, init, 24, True)
    _same(a, b)
    assert b["uncertain"] > 640 * torch.cuda.get_device_properties(cuda).multi_processor_count  # (some list is too short)
    tied = (X_t[0] == 0.0) & (w == 0.0)
    assert int(tied.sum()) == on_plane
    assert float(a["cent"][0, 3]) == -float(a["cent"][0, 11])  # the ties are exact
    assert bool((b["labels"][tied] == 3).all())


@pytest.mark.parametrize("dtype", ["float32", "float64"])
def test_run_with_relocated_clusters(dtype, cuda, monkeypatch):
    """Through the driver: relocations end a call to the library, and the run goes on with another."""
    import torch

    from sklearn_numba_dpex_amd import _capi
    from sklearn_numba_dpex_amd.kmeans import drivers

    n, k, seen = 600_001, 64, dict(areas=[], relocations=0)
    X_t, w, init = _blobs(n, 32, k, getattr(torch, dtype), 5, cuda)
    for j in range(8):
        init[:, 63 - j] = 1e3 * (1 + j * 1e-3)
    lib = drivers.lib

    class Torch:
        def __getattr__(self, name):
            return getattr(torch, name)

        def empty(self, *args, **kwargs):
            out = torch.empty(*args, **kwargs)
            if kwargs.get("dtype") is torch.uint8 and out.numel() > n:
                seen["areas"].append(out.fill_(MARK))
            return out

    class Lib:
        def __init__(self, with_bounds):
            self.with_bounds = with_bounds

        def __getattr__(self, name):
            if name == "kmx_lloyd_bounds_bytes" and not self.with_bounds:
                return lambda plan: 0
            return self.run if name == "kmx_lloyd_run" else getattr(lib, name)

        def run(self, *args):
            rc = lib.kmx_lloyd_run(*args)
            if args[-2].state == _capi.KMX_NEED_RELOCATION:
                seen["relocations"] += 1
                for area in seen["areas"]:  # (used within a call only: what is written from here on comes behind)
                    area.fill_(MARK)
            return rc

    monkeypatch.setattr(drivers, "torch", Torch())
    monkeypatch.setattr(drivers, "lib", Lib(True))
    with_bounds = drivers.lloyd(X_t, w, init, False, 25, False, 0.0)
    assert seen["relocations"] >= 1 and len(seen["areas"]) == 1 and _entered(seen["areas"][0], n, k)
    monkeypatch.setattr(drivers, "lib", Lib(False))
    without = drivers.lloyd(X_t, w, init, False, 25, False, 0.0)
    assert len(seen["areas"]) == 1
    assert with_bounds[3] == without[3] and with_bounds[1] == without[1]
    same = bool((with_bounds[0] == without[0]).all()), bool((with_bounds[2] == without[2]).all())
    assert same == (True, True)


@pytest.mark.parametrize("d, k, dtype", [(49, 133, "float32"), (49, 105, "float64")])
def test_queue_that_holds_one_load_of_words(d, k, dtype, cuda):
    """The largest operands that leave room for it: 2 048 and 1 024 entries, emptied behind every load of a workgroup's
    3 900 samples."""
    import torch

    from sklearn_numba_dpex_amd import _capi
    from sklearn_numba_dpex_amd._capi import lib

    n, code = 1_000_003, _capi.dtype_code(getattr(torch, dtype))
    assert lib.kmx_lloyd_bounds_bytes(_capi.lloyd_plan(n, d, k, code, 0)) > 0
    assert lib.kmx_lloyd_bounds_bytes(_capi.lloyd_plan(n, d, k + 1, code, 0)) == 0
    X_t, w, init = _blobs(n, d, k, getattr(torch, dtype), 13, cuda)
    _same(_run(X_t, w, init, 30, False), _run(X_t, w, init, 30, True))


@pytest.mark.parametrize("dtype", ["float32", "float64"])
def test_runs_of_every_length(dtype, cuda):
    import torch

    X_t, w, init = _blobs(800_001, 20, 48, getattr(torch, dtype), 17, cuda)
    for max_iter in range(4, 24):
        _same(_run(X_t, w, init, max_iter, False), _run(X_t, w, init, max_iter, True, max_iter > 20 or None))


@pytest.mark.parametrize("dtype", ["float32", "float64"])
def test_a_sample_that_is_no_number(dtype, cuda):
    """Its scores compare with none, which gives it the first label in every iteration, and no margin."""
    import torch

    X_t, w, init = _blobs(1_200_001, 14, 64, getattr(torch, dtype), 19, cuda)
    at = 777_777
    X_t[3, at] = float("nan")
    w[at] = 0.0
    a, b = _run(X_t, w, init, 30, False), _run(X_t, w, init, 30, True, None)
    for run in (a, b):
        assert int(run["labels"][at]) == 0
    a["cent"], b["cent"] = (run["cent"].nan_to_num(nan=-1e30) for run in (a, b))
    _same(a, b)


# from 6e-14 to 1e18 (the data are about 15 wide) labels are those of bounded iterations; beyond, an fp32 chain loses
# products that the screen keeps (7e-22: other labels than those of the screened step), and they are not entered
@pytest.mark.parametrize("scale, dtype, entered", [
    (1e-25, "float64", False), (1e-16, "float64", False), (1e-14, "float64", True), (3e16, "float64", True),
    (2e17, "float64", False), (1e25, "float64", False),
    (1e-22, "float32", False), (7e-22, "float32", False), (1e-16, "float32", False), (1e-14, "float32", True),
    (3e16, "float32", True), (2e17, "float32", False),
])
def test_data_of_any_magnitude(scale, dtype, entered, cuda):
    import torch

    n, d, k = 1_200_001, 14, 64
    X_t, w, init = _blobs(n, d, k, torch.float64, 11, cuda, spread=10.0)
    X_t, w, init = ((scale * X_t).to(getattr(torch, dtype)), w.to(getattr(torch, dtype)),
                    (scale * init).to(getattr(torch, dtype)))
    a = _run(X_t, w, init, 30, False)
    b = _run(X_t, w, init, 30, True, entered)
    _same(a, b)
