"""The refined inverse and the refinement of a given X at the edges of their
products (4, 2 or 1 matrices per matrix instruction up to n = 4, 8, 16; two by
two blocks above), of their tiles (16 or 4 matrices) and of alignment, for
every pivot rule: against one FP64-residual step of the plain inverse, with
the plain pivots, A untouched and nothing written past the batch."""
import numpy as np
import pytest

import oracle
from tests.test_gpu_refine import _step_reference, _within_step

pytestmark = pytest.mark.gpu

RULES = {"none": 0x0, "parallel": 0x1, "serial": 0x2, "tree": 0x3, "gepp": 0x4}


@pytest.mark.parametrize("rule", sorted(RULES))
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 8, 9, 11, 12, 13, 15, 16, 17, 23, 28, 31, 32])
def test_refined_inverse_every_rule(gpu, n, rule):
    from matrixinversion_amd._native import check, lib

    flags = RULES[rule]
    for batch, a_off, x_off in ((1, 0, 0), (5, 4, 0), (16, 0, 4), (35, 0, 0), (64, 0, 0)):
        a = oracle.dominant_matrices(700 + n, batch, n)
        x0, p0 = gpu.invert(a, flags)
        guard = np.full(8, np.float32(-7.25))
        A, X, P = gpu.DeviceBuffer(a.nbytes + 4), gpu.DeviceBuffer(a.nbytes + 36), gpu.DeviceBuffer(batch * n * 4)
        try:
            print(f"[case] refined n={n} rule={rule} batch={batch} offsets={a_off},{x_off}", flush=True)
            A.upload(a, offset=a_off)
            X.upload(guard, offset=x_off + a.nbytes)
            check(lib().lu_batched_inverse_refined(A.ptr + a_off, X.ptr + x_off, P.ptr, n, batch, flags, None))
            gpu.synchronize()
            x1, p1 = X.download(a.shape, np.float32, offset=x_off), P.download((batch, n), np.int32)
            assert np.array_equal(A.download(a.shape, np.float32, offset=a_off), a)
            assert np.array_equal(X.download((8,), np.float32, offset=x_off + a.nbytes), guard)
            assert np.array_equal(p1, p0)
            assert _within_step(a, x0, x1)
            # the separate step on the plain inverse gives the same bits
            X.upload(x0, offset=x_off)
            check(lib().lu_batched_refine(A.ptr + a_off, X.ptr + x_off, n, batch, None))
            gpu.synchronize()
            x2 = X.download(a.shape, np.float32, offset=x_off)
            assert np.array_equal(X.download((8,), np.float32, offset=x_off + a.nbytes), guard)
        finally:
            for b in (A, X, P):
                b.close()
        assert np.array_equal(x2.view(np.uint32), x1.view(np.uint32))


@pytest.mark.parametrize("n", [3, 8, 12, 16])
def test_rough_inverse_is_corrected(gpu, n):
    """A given X off by 1e-3 is corrected to the FP64 step's value, each matrix
    by its own A (neighbours in one product differ)."""
    rng = np.random.RandomState(n)
    a = oracle.dominant_matrices(800 + n, 37, n) * rng.uniform(0.5, 2.0, (37, 1, 1)).astype(np.float32)
    x = (np.linalg.inv(a.astype(np.float64)) * (1 + 1e-3 * rng.uniform(-1, 1, a.shape))).astype(np.float32)
    A, X = gpu.DeviceBuffer.from_array(a), gpu.DeviceBuffer.from_array(x)
    try:
        print(f"[case] refine rough n={n}", flush=True)
        gpu.refine(A, X, n, 37)
        got = X.download(a.shape, np.float32)
    finally:
        A.close()
        X.close()
    ref = _step_reference(a, x)
    scale = np.abs(ref).max(axis=(1, 2), keepdims=True)
    # the correction's n-term FP32 sums: n ulps of 1e-3 of the scale, and one rounding
    assert np.all(np.abs(got - ref) <= 2.0 ** -24 * np.abs(ref) + (n + 2) * 2.0 ** -24 * 4e-3 * scale)


@pytest.mark.parametrize("rule", sorted(RULES))
@pytest.mark.parametrize("n", range(1, 17))
def test_forced_layouts_agree(gpu, n, rule):
    """16-lane rows and quads, partial tiles and unaligned A and X: the same
    bits, within the FP64 step of the plain inverse."""
    from matrixinversion_amd._native import check, lib

    for batch, a_off, x_off in ((64, 0, 0), (37, 4, 0), (19, 0, 4), (1, 8, 12)):
        a = oracle.dominant_matrices(900 + n, batch, n)
        x0, p0 = gpu.invert(a, RULES[rule])
        guard = np.full(8, np.float32(-7.25))
        A, X, P = gpu.DeviceBuffer(a.nbytes + 16), gpu.DeviceBuffer(a.nbytes + 48), gpu.DeviceBuffer(batch * n * 4)
        got = []
        try:
            A.upload(a, offset=a_off)
            for layout in (0x10, 0x20):
                print(f"[case] refined n={n} rule={rule} layout={layout:#x} batch={batch} at {a_off},{x_off}", flush=True)
                X.upload(guard, offset=x_off + a.nbytes)
                check(lib().lu_batched_inverse_refined(A.ptr + a_off, X.ptr + x_off, P.ptr, n, batch,
                                                       RULES[rule] | layout, None))
                gpu.synchronize()
                got.append(X.download(a.shape, np.float32, offset=x_off))
                assert np.array_equal(P.download((batch, n), np.int32), p0)
                assert np.array_equal(X.download((8,), np.float32, offset=x_off + a.nbytes), guard)
        finally:
            for b in (A, X, P):
                b.close()
        assert _within_step(a, x0, got[0])
        assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))


@pytest.mark.parametrize("n", [9, 10, 11, 12])
def test_quads_above_the_small_batch_line(gpu, n):
    """From 16,385 matrices n = 9..12 take quads, in the refined inverse and in
    the refinement of a given X: the bits of a small batch (rows), also in a
    partial last tile and unaligned."""
    from matrixinversion_amd._native import check, lib

    block = oracle.dominant_matrices(950 + n, 512, n)
    for batch, off in ((16385, 0), (16389, 4), (16400, 0)):
        a = np.tile(block, (batch // 512 + 1, 1, 1))[:batch].copy()
        x0, _ = gpu.invert(block, 0x1)
        A, X = gpu.DeviceBuffer(a.nbytes + 4), gpu.DeviceBuffer(a.nbytes + 4)
        try:
            A.upload(a, offset=off)
            for given in (False, True):
                results = []
                for count in (512, batch):
                    print(f"[case] refined quads n={n} batch={count} offset={off} given={given}", flush=True)
                    if given:
                        X.upload(np.tile(x0, (batch // 512 + 1, 1, 1))[:batch].copy(), offset=off)
                        check(lib().lu_batched_refine(A.ptr + off, X.ptr + off, n, count, None))
                    else:
                        check(lib().lu_batched_inverse_refined(A.ptr + off, X.ptr + off, None, n, count, 0x1, None))
                    gpu.synchronize()
                    results.append(X.download((count, n, n), np.float32, offset=off))
                rows, quads = results
                assert _within_step(block, x0, rows)
                want = np.tile(rows, (batch // 512 + 1, 1, 1))[:batch]
                assert np.array_equal(quads.view(np.uint32), want.view(np.uint32))
        finally:
            A.close()
            X.close()
