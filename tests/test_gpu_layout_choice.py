"""Which lane layout a call takes, read from the grid of its captured launch
(one workgroup per tile of 4 matrices in 16-lane rows, of 16 in quads; nothing
is run): forced layouts and the tuning table are honoured by the plain and the
refined inverse, on both sides of each line where rows replace the table's
quads."""
import ctypes
import os
import subprocess
import sys
from types import SimpleNamespace

import numpy as np
import pytest

import oracle
from tests.conftest import ROOT

pytestmark = pytest.mark.gpu

ROWS, QUADS = 4, 16  # matrices per tile
LAYOUT = {"auto": 0x0, "rows": 0x10, "quads": 0x20}


class _KernelNode(ctypes.Structure):  # hipKernelNodeParams
    _fields_ = [("block", ctypes.c_uint32 * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p),
                ("grid", ctypes.c_uint32 * 3), ("params", ctypes.c_void_p), ("shared", ctypes.c_uint32)]


def _grid(gpu, call):
    """Workgroups of the one kernel that call(stream) launches."""
    from matrixinversion_amd._native import lib

    hip = lib()  # its dependencies hold the runtime's entry points
    s = gpu.Stream()
    graph, count = ctypes.c_void_p(), ctypes.c_size_t()
    stream = ctypes.c_void_p(s.handle)
    try:
        assert hip.hipStreamBeginCapture(stream, 2) == 0
        try:
            call(s.handle)
        finally:
            assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
        assert hip.hipGraphGetNodes(graph, None, ctypes.byref(count)) == 0 and count.value == 1
        nodes = (ctypes.c_void_p * 1)()
        assert hip.hipGraphGetNodes(graph, nodes, ctypes.byref(count)) == 0
        p = _KernelNode()
        assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(nodes[0]), ctypes.byref(p)) == 0
        assert hip.hipGraphDestroy(graph) == 0
        return p.grid[0]
    finally:
        s.close()


def _per_tile(gpu, entry, n, flags, batch):
    from matrixinversion_amd._native import check, lib

    A, X = gpu.DeviceBuffer(batch * n * n * 4), gpu.DeviceBuffer(batch * n * n * 4)
    try:
        print(f"[case] layout {entry} n={n} flags={flags:#x} batch={batch}", flush=True)
        if entry == "plain":
            g = _grid(gpu, lambda s: check(lib().lu_batched_inverse_async64(A.ptr, None, n, batch, flags, s)))
        elif entry == "refined":
            g = _grid(gpu, lambda s: check(lib().lu_batched_inverse_refined(A.ptr, X.ptr, None, n, batch, flags, s)))
        else:
            g = _grid(gpu, lambda s: check(lib().lu_batched_refine(A.ptr, X.ptr, n, batch, s)))
    finally:
        A.close()
        X.close()
    return {-(-batch // ROWS): ROWS, -(-batch // QUADS): QUADS}[g]


@pytest.mark.parametrize("entry", ["plain", "refined"])
@pytest.mark.parametrize("rule", [0x0, 0x1, 0x2, 0x3, 0x4])
def test_forced_layouts(gpu, entry, rule):
    for n in (1, 5, 8, 9, 12, 13, 16):
        for batch in (100, 40000):
            assert _per_tile(gpu, entry, n, rule | LAYOUT["rows"], batch) == ROWS
            assert _per_tile(gpu, entry, n, rule | LAYOUT["quads"], batch) == QUADS


@pytest.mark.parametrize("entry,line", [("plain", 8192), ("refined", 16384), ("refine", 16384)])
def test_automatic_layout(gpu, entry, line):
    for n, rule, batch, want in ((8, 1, 50, QUADS), (9, 1, line, ROWS), (9, 1, line + 1, QUADS), (12, 3, line, ROWS),
                                 (12, 3, line + 1, QUADS), (12, 0, line, ROWS), (12, 0, line + 1, QUADS),
                                 (13, 1, 40000, ROWS), (17, 1, 40000, ROWS)):
        assert _per_tile(gpu, entry, n, rule, batch) == want
    if entry != "refine":
        assert _per_tile(gpu, entry, 8, 4, 40000) == QUADS and _per_tile(gpu, entry, 9, 4, 40000) == ROWS


@pytest.mark.parametrize("entry", ["plain", "refined"])
def test_table_is_honoured(gpu, entry):
    layout, grab = gpu.tuning_get()
    try:
        mine = layout.copy()
        mine[5], mine[14] = 0, 1
        gpu.tuning_set(mine, grab)
        assert _per_tile(gpu, entry, 5, 1, 40000) == ROWS
        assert _per_tile(gpu, entry, 14, 1, 40000) == QUADS
        assert _per_tile(gpu, entry, 14, 1, 100) == QUADS
    finally:
        gpu.tuning_set(layout, grab)


def ragged_direct(gpu):
    """(grid, inverses) of 1,500 mixed matrices, a batch that needs no plan."""
    ns = np.random.RandomState(3).randint(1, 33, 1500).astype(np.int32)
    flat = np.concatenate([oracle.dominant_matrices(80, 1, int(n))[0].ravel() for n in ns])
    offs = np.concatenate([[0], np.cumsum(ns.astype(np.int64) ** 2)[:-1]])
    A, O, NS = (gpu.DeviceBuffer.from_array(v) for v in (flat, offs, ns))
    with gpu.RaggedPlan(ns.size) as plan:
        print("[case] ragged without a plan, 1500 matrices", flush=True)
        grid = _grid(gpu, lambda s: gpu.lu_batched_inverse_ragged(A, O, NS, ns.size, 0x1, plan=plan,
                                                                  stream=SimpleNamespace(handle=s)))
        gpu.lu_batched_inverse_ragged(A, O, NS, ns.size, 0x1, plan=plan)
        gpu.synchronize()
        x = A.download(flat.shape, np.float32)
    for b in (A, O, NS):
        b.close()
    return grid, x


CHILD = """
import sys
import numpy as np
import matrixinversion_amd as mia
from tests.test_gpu_layout_choice import ragged_direct
grid, x = ragged_direct(mia)
np.savez(sys.argv[1], grid=grid, x=x)
"""


def test_persistent_waves_without_a_plan(gpu, tmp_path):
    """LUB_RAGGED_WAVES_PER_CU bounds the grid of a batch without a plan too;
    the variable is read once, so a child process sets it."""
    path = str(tmp_path / "direct.npz")
    env = dict(os.environ, LUB_RAGGED_WAVES_PER_CU="1", PYTHONPATH=ROOT)
    r = subprocess.run([sys.executable, "-u", "-c", CHILD, path], env=env, cwd=ROOT, timeout=100, capture_output=True,
                       text=True)
    print(r.stdout[-1000:], r.stderr[-1000:], flush=True)
    assert r.returncode == 0
    got = np.load(path)
    grid, x = ragged_direct(gpu)
    assert grid == 1501 and int(got["grid"]) == gpu.device_info(0).cu_count
    assert np.array_equal(got["x"].view(np.uint32), x.view(np.uint32))
