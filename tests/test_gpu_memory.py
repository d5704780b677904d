"""Device memory of released objects: kept for reuse within a bound, never
handed on before queued work on other streams has read it, and safe with
several threads."""

import gc
import threading

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

GIB = 1 << 30


def build(A, X, C):
    m = A.Mesh(3, X, C)
    b = A.BSRFormat(m, 1, use_csr=True)
    b.compute_sparsity()
    s = A.DoFLinearSystem(len(X))
    b.assemble_laplace(None, 1.0, s.rhs())
    return m, b, s


def test_kept_memory_is_bounded(afem_gpu):
    """Systems of growing sizes, 1.7 GiB of distinct buffers together, released
    one after the other: what stays allocated is within the bound of 1 GiB
    (and 64 MiB for the runtime's own chunks)."""
    print("[case] kept memory", flush=True)
    A = afem_gpu
    torch.cuda.synchronize()
    gc.collect()
    lib = A.lib()
    before = torch.cuda.mem_get_info()[0]
    for n in range(1 << 20, 20 << 20, 1 << 20):  # doubles in x, rhs and the elimination's arrays
        s = A.DoFLinearSystem(n)
        s.rhs().zero()
        del s
        gc.collect()
    after = torch.cuda.mem_get_info()[0]
    print(f"[result] {(before - after) / GIB:.3f} GiB kept", flush=True)
    assert before - after <= GIB + (64 << 20)
    assert lib is not None


def test_repeated_builds_agree(afem_gpu):
    """Buffers that held something else before: every build of a matrix and
    every solve gives the first one's numbers."""
    print("[case] reused memory", flush=True)
    A = afem_gpu
    meshes = [A.box_mesh(3, n, 0.15, n) for n in (9, 14, 10)]
    first = {}
    for turn in range(3):
        for k, (X, C) in enumerate(meshes):
            m, b, s = build(A, X, C)
            out = [a.copy() for a in b.download()] + [s.rhs().numpy()]
            for a, f in zip(out, first.setdefault(k, out)):
                assert np.array_equal(a, f), (turn, k)
            del m, b, s


def test_work_on_another_stream_meets_its_own_values(afem_gpu):
    """A view read on a torch stream behind a long queue, its owner released at
    once and its block asked for again and overwritten."""
    print("[case] view on another stream", flush=True)
    A = afem_gpu
    n = 1 << 22
    side = torch.cuda.Stream()
    s = A.DoFLinearSystem(n)
    s.rhs().upload(np.full(n, 3.0))

    class View:
        __cuda_array_interface__ = {"shape": (n,), "typestr": "<f8", "data": (s.rhs().ptr, False), "version": 3}

    v = torch.as_tensor(View(), device="cuda")
    busy = torch.ones(1 << 26, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        for _ in range(50):
            busy += 1.0
        total = v.sum()
    del s
    gc.collect()
    t = A.DoFLinearSystem(n)
    t.rhs().upload(np.full(n, 5.0))
    torch.cuda.synchronize()
    assert float(total) == 3.0 * n


def test_threads(afem_gpu):
    print("[case] threads", flush=True)
    A = afem_gpu
    meshes = [A.box_mesh(3, n, 0.15, n) for n in (6, 8, 11, 13)]
    want = []
    for X, C in meshes:
        m, b, s = build(A, X, C)
        want.append(b.download()[2].copy())
    errors = []
    lock = threading.Lock()  # the library has one stream: calls that build one matrix are not interleaved

    def work(k):
        try:
            for _ in range(5):
                with lock:
                    m, b, s = build(A, *meshes[k])
                    val = b.download()[2].copy()
                del m, b, s  # released while others build
                if not np.array_equal(val, want[k]):
                    errors.append(k)
        except Exception as e:  # noqa: BLE001
            errors.append(repr(e))

    th = [threading.Thread(target=work, args=(k,)) for k in range(len(meshes))]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not errors


@pytest.mark.parametrize("where", ["same thread, relaxed", "other thread, relaxed", "other thread, thread_local"])
def test_releases_during_a_capture(afem_gpu, where):
    """Another stream is being captured in a mode that allows allocations: a
    released object leaves the capture valid, and the graph replays."""
    print(f"[case] release during a capture: {where}", flush=True)
    A = afem_gpu
    n = 1 << 20
    x = torch.zeros(n, device="cuda")
    g = torch.cuda.CUDAGraph()
    held = []

    def work():
        held.clear()  # releases blocks that are kept
        gc.collect()
        held.append(A.DoFLinearSystem(n))  # and asks for them again
        held.append(A.DoFLinearSystem(n + 4096))  # these are new

    for _ in range(2):
        work()
    A.check(A.lib().afem_synchronize())
    torch.cuda.synchronize()
    gc.disable()
    try:
        with torch.cuda.graph(g, capture_error_mode=where.split(", ")[1]):
            x += 1.0
            if where.startswith("other"):
                t = threading.Thread(target=work)
                t.start()
                t.join()
            else:
                work()
            x += 2.0
    finally:
        gc.enable()
    for k in range(3):
        g.replay()
        held[0].rhs().upload(np.full(n, float(k)))
        torch.cuda.synchronize()
        assert float(x[0]) == 3.0 * (k + 1) and float(x[-1]) == 3.0 * (k + 1)
        assert held[0].rhs().numpy()[-1] == k
