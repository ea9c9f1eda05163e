"""Host code of libpagani on a stub HIP runtime (hip_stub.cpp): which device is
current at a launch, what happens when an allocation fails.  Kernels do not
run, so a network has no edges here; no GPU is needed."""
import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes as C, os, sys
stub = C.CDLL({stub!r}, mode=os.RTLD_GLOBAL)
sys.modules["torch"] = None  # its HIP runtime is not wanted
sys.path.insert(0, {pkg!r})
import numpy as np
import pagani_amd
from pagani_amd import lib as L
stub.stub_alloc.restype = C.c_void_p
stub.stub_alloc.argtypes = [C.c_size_t, C.c_int, C.c_int]
HOOK = C.CFUNCTYPE(None, C.c_char_p, C.c_int, C.c_int, C.POINTER(C.c_void_p))
launches, check = [], lambda name, args: None
@HOOK
def hook(name, current, device, args):
    launches.append((name.decode(), current, device))
    check(name.decode(), args)
stub.stub_hook(hook)
def misplaced():
    return [x for x in launches if x[1] != x[2]]
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("hip") / "libhipstub.so")
    subprocess.run(["g++", "-shared", "-fPIC", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "hip_stub.cpp"), "-o", out], check=True)
    return out


def run(stub, code):
    src = PRELUDE.format(stub=stub, pkg=os.path.join(ROOT, "pagani-toolkit_amd")) + textwrap.dedent(code)
    r = subprocess.run([sys.executable, "-c", src], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr + r.stdout


def test_corr_csr_on_its_own_device(stub):
    """pg_corr_csr of a context on device 1 while device 0 is current: its
    kernel runs on device 1, and only for arrays that lie there; other devices'
    and managed memory are copied to by the runtime."""
    run(stub, """
    ctx = pagani_amd.Context(1)
    n = 40
    ctx.corr_build(np.zeros((20, n), np.float32), n, 20, 0.3, weighted=True)
    assert launches and not misplaced()
    def take(device, managed):
        stub.hipSetDevice(0)
        launches.clear()
        before = stub.stub_copies()
        row, col, val = (C.c_void_p(stub.stub_alloc(4 * (n + 1), device, managed)) for _ in range(3))
        ctx._check(ctx._lib.pg_corr_csr(ctx._h, row, col, val))
        return len(launches), stub.stub_copies() - before
    assert take(1, 0) == (1, 0) and not misplaced()
    assert take(0, 0)[0] == 0 and take(0, 0)[1] >= 1
    assert take(1, 1)[0] == 0 and take(1, 1)[1] >= 1
    """)


def test_weighted_clustering_launches(stub):
    """A region-level call is its launches: the check, (Onnela) the maximum, the
    lists with the factors, the clustering, the mean."""
    run(stub, """
    n = 116
    row, col, val = np.zeros(n + 1, np.int32), np.zeros(200, np.int32), np.ones(200, np.float32)
    row[1:] = 200
    ctx = pagani_amd.Context(0)
    for kind, count in ((1, 4), (2, 5)):
        launches.clear()
        ctx.cp_weighted(row, col, val, kind)
        assert len(launches) == count, launches
    """)


def test_clustering_flag_after_a_failed_allocation(stub):
    """Each allocation of a context's first pg_cp_binary fails once: the next
    call finds its malformed-CSR flag clear."""
    run(stub, """
    n = 40
    row, col = np.zeros(n + 1, np.int32), np.zeros(0, np.int32)
    flags = []
    def check(name, args):
        if "csr_validate" in name:
            flags.append(C.cast(args[5], C.POINTER(C.POINTER(C.c_int)))[0][0])
    failed = 0
    for nth in range(1, 12):
        ctx = pagani_amd.Context(0)
        stub.stub_fail_malloc(nth)
        try:
            ctx.cp_binary(row, col)
        except pagani_amd.PgError as e:
            assert e.status == 2, e
            failed += 1
        stub.stub_fail_malloc(0)
        flags.clear()
        ctx.cp_binary(row, col)
        assert flags == [0], (nth, flags)
    assert failed >= 4
    """)


def test_weighted_build_allocations(stub):
    """Two buffers of a weighted build are only for speed: without either the
    scatter sums the weights itself, and no other request may fail."""
    run(stub, """
    n, t = 300, 100
    x = np.zeros((t, n), np.float32)
    summed, listed = "bucket_scatterILi2E", "bucket_scatterILi1E"
    spared = refused = 0
    live = []  # allocations after a build that summed
    for nth in range(1, 60):
        if nth > 1:
            ctx.close()
        ctx = pagani_amd.Context(0)
        launches.clear()
        stub.stub_fail_malloc(nth)
        status = 0
        try:
            ctx.corr_build(x, n, t, 0.3, weighted=True)
        except pagani_amd.PgError as e:
            status = e.status
        made = stub.stub_mallocs()
        stub.stub_fail_malloc(0)
        names = [x[0] for x in launches]
        if status == 2:
            refused += 1
            continue
        assert status == 0
        if made < nth:
            assert any(listed in x for x in names), names
            break
        assert any(summed in x for x in names) and not any(listed in x for x in names), (nth, names)
        spared += 1
        live.append(stub.stub_live())
    assert spared == 2 and refused >= 10, (spared, refused, nth)
    # the lists' weights are given back where the sort's buffer had no room
    assert live[0] == live[1], live
    # with the lists: a small network's values take one launch
    assert sum("edge_values" in x for x in names) == 1, names
    """)


def test_threshold_of_an_average_copies_nothing_back(stub):
    """What the host checks comes through pinned memory: no copy per number."""
    run(stub, """
    n = 116
    x = np.zeros((50, n), np.float32)
    ctx = pagani_amd.Context(0)
    ctx.cormat_begin(n)
    ctx.cormat_add(x, 50)
    ctx.cormat_finish()
    before = stub.stub_copies()
    assert ctx.cormat_threshold(0.3).nnz == 0
    assert stub.stub_copies() == before
    """)
