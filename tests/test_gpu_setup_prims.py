"""The setup's device primitives through hierarchies whose sizes reach their edges
(exact results: the hierarchy and V-cycle of the oracle): the median of the scaling
decision in one workgroup and over the whole device, product rows longer than a
sort's LDS classes, tiles at segment borders; and the reuse of a destroyed
hierarchy's memory by the next build, also from other threads and streams."""
import threading

import numpy as np
import pytest
import scipy.sparse as sp
import torch

from matrices import impes_like, laplacian_2d

pytestmark = pytest.mark.gpu


def _csr(A, dev):
    return (torch.tensor(A.indptr, dtype=torch.int32, device=dev), torch.tensor(A.indices, dtype=torch.int32, device=dev),
            torch.tensor(A.data, dtype=torch.float64, device=dev))


@pytest.mark.parametrize("n", [1, 2, 7, 64, 1000, 1025, 32767, 32768, 32769, 300001])
def test_median_scaling(dev, n):
    """dhalf_inv is 1/sqrt of the lower median of |a_ii| (spread over 30 orders)."""
    import impes_hip as H

    d = 10.0 ** np.random.default_rng(n).uniform(-32.0, -7.0, n)
    d[:: max(1, n // 5)] = d[0]  # ties
    A = sp.diags(d, format="csr")
    h = H.AmgHierarchy(max_levels=1, dense_max=1)
    h.setup_csr(*_csr(A, dev))
    mid = np.sort(np.maximum(np.abs(d), 1e-30))[(n - 1) // 2]
    assert float(h.dhalf_inv()[0]) == 1.0 / np.sqrt(mid)


@pytest.mark.parametrize("n", [511, 512, 513, 1024, 4097, 6000])
def test_long_rows_and_segment_borders(dev, n):
    """A hub coupled to every 13th row: product rows of thousands of terms, above and
    below the size at which a sort bins its segments."""
    import impes_hip as H
    from oracle import amg as oa

    A = sp.lil_matrix(sp.diags([np.full(n, 2.1), np.full(n - 1, -1.0), np.full(n - 1, -1.0)], [0, 1, -1]))
    hub = n // 2
    for j in range(0, n, 13):
        if abs(j - hub) > 1:
            A[hub, j] = A[j, hub] = -0.6
            A[j, j] = A[j, j] + 0.6
            A[hub, hub] = A[hub, hub] + 0.6
    A = sp.csr_matrix(A)
    A.sort_indices()
    kw = dict(coarsest_size=40)
    ho, h = oa.Hierarchy(A, **kw), H.AmgHierarchy(**kw)
    h.setup_csr(*_csr(A, dev))
    assert h.num_levels == len(ho.levels)
    b = np.random.default_rng(1).standard_normal(n)
    x = h.vcycle(torch.tensor(b, device=dev)).cpu().numpy()
    y = ho.vcycle(b)
    assert np.linalg.norm(x - y) <= 1e-11 * np.linalg.norm(y)


def test_memory_of_destroyed_hierarchies(dev):
    """Build, use and drop hierarchies from several threads on streams of their own:
    every result equals the first one's bits; the kept memory is given back."""
    import impes_hip as H

    sizes = [(20, 18, 9), (30, 20, 11), (25, 25, 4)]
    want = {}

    def once(dims):
        A, *_ = impes_like(*dims, seed=3)
        b = torch.tensor(np.random.default_rng(2).standard_normal(A.shape[0]), device=dev)
        h = H.AmgHierarchy()
        h.setup_csr(*_csr(A, dev))
        x = h.precondition(b, precision=32)
        h.close()
        return x

    for d in sizes:
        want[d] = once(d).cpu()
    bad = []

    def work(k):
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            for q in range(6):
                d = sizes[(k + q) % len(sizes)]
                try:
                    x = once(d)
                except Exception as e:  # noqa: BLE001 (a thread's exception fails no test by itself)
                    bad.append((k, q, d, e))
                    return
                st.synchronize()
                if not torch.equal(x.cpu(), want[d]):
                    bad.append((k, q, d))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not bad, bad
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    H.release_cached_memory()
    assert torch.cuda.mem_get_info()[0] > before


def test_update_after_a_reused_build(dev):
    """A numeric update of a hierarchy in reused memory equals a fresh one's."""
    import impes_hip as H

    A = laplacian_2d(70)
    A = (A + sp.identity(A.shape[0]) * 1e-3).tocsr()
    A.sort_indices()
    out = []
    for _ in range(2):
        h = H.AmgHierarchy()
        h.setup_csr(*_csr(A, dev))
        h.update_csr(_csr(A * 1.5, dev)[2])
        out.append(h.vcycle(torch.ones(A.shape[0], dtype=torch.float64, device=dev)))
        h.close()
    assert torch.equal(*out)


def test_builds_leave_other_threads_captures_alone(dev):
    """Hierarchies and simulators are built, used and destroyed while another thread
    records a graph of its own (the first preconditioner call of a hierarchy records one
    as well)."""
    import impes_hip as H
    from simulator.cases import baseline_case, build

    cfg, fields = baseline_case(1, dims=(8, 8, 3))
    A, *_ = impes_like(20, 18, 9, seed=3)
    csr = _csr(A, dev)
    b = torch.ones(A.shape[0], dtype=torch.float64, device=dev)
    errors = []

    def work(times):
        try:
            st = torch.cuda.Stream()
            with torch.cuda.stream(st):
                for _ in range(times):
                    h = H.AmgHierarchy()
                    h.setup_csr(*csr)
                    h.precondition(b, precision=32)
                    st.synchronize()
                    h.close()
                    assert build(cfg, fields, "cuda:0").run_step(86400.0)
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    work(2)  # code objects and streams are made
    x = torch.zeros(1000, device=dev)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, capture_error_mode="thread_local"):
        x += 1.0
        th = threading.Thread(target=work, args=(3,))
        th.start()
        th.join()
        x += 1.0
    for k in range(1, 4):
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(x, torch.full_like(x, 2.0 * k))
    threads = [threading.Thread(target=work, args=(30,)) for _ in range(4)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not errors, errors[0]


def test_threads_that_come_and_go_leave_nothing_behind(dev):
    """Hierarchies built by one short-lived thread after another: the process's mappings
    of device and pinned memory do not grow."""
    import impes_hip as H

    csr = _csr(impes_like(8, 8, 4, seed=3)[0], dev)

    def work():
        h = H.AmgHierarchy()
        h.setup_csr(*csr)
        h.close()

    def mappings():
        with open("/proc/self/maps") as f:
            return sum("renderD" in line or "kfd" in line for line in f)

    counts = []
    for _ in range(3):
        for _ in range(20):
            th = threading.Thread(target=work)
            th.start()
            th.join()
        counts.append(mappings())
    assert counts[-1] - counts[0] <= 4, counts  # one a thread would be 40


@pytest.mark.parametrize("first", [False, True])
def test_failed_setup_leaves_no_hierarchy(dev, first):
    """A pattern that is not symmetric is refused; so is every use of the handle until a
    setup succeeds, whether it had a hierarchy before or not."""
    import impes_hip as H

    A, *_ = impes_like(12, 10, 9, seed=3)
    good = _csr(A, dev)
    B = A.tolil()
    B[5, 700] = -1e-11
    B = sp.csr_matrix(B)
    B.sort_indices()
    b = torch.ones(A.shape[0], dtype=torch.float64, device=dev)
    h, ref = H.AmgHierarchy(), H.AmgHierarchy()
    ref.setup_csr(*good)
    z = ref.precondition(b)
    if first:
        h.setup_csr(*good)
        assert torch.equal(h.precondition(b), z)
    with pytest.raises(H.ImpesError):
        h.setup_csr(*_csr(B, dev))
    for use in (lambda: h.precondition(b), lambda: h.vcycle(b), lambda: h.cycles(b), lambda: h.update_csr(good[2])):
        with pytest.raises(H.ImpesError):
            use()
    h.setup_csr(*good)
    assert torch.equal(h.precondition(b), z)
