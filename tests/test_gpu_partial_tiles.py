"""Partial and unaligned tiles of the plain path: any number of matrices at any
4-byte offset gives the bits of the same matrices in full, aligned tiles, and
nothing before or after the batch is written."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", range(1, 33))
def test_any_count_at_any_offset(gpu, n):
    from matrixinversion_amd._native import check, lib

    a = oracle.dominant_matrices(40 + n, 32, n)
    for flags in (0x0, 0x1, 0x3, 0x4, 0x11, 0x14) + ((0x21, 0x24) if n <= 16 else ()):
        x, p = gpu.invert(a, flags)
        for count, off in ((1, 0), (2, 1), (3, 0), (4, 3), (5, 2), (15, 0), (16, 1), (17, 0), (31, 3)):
            pad = np.full(4 + off, np.float32(-7.25))
            host = np.concatenate([pad, a[:count].ravel(), pad])
            A, P = gpu.DeviceBuffer.from_array(host), gpu.DeviceBuffer.from_array(np.full(count * n + 1, -5, np.int32))
            try:
                print(f"[case] partial n={n} flags={flags:#x} count={count} off={off}", flush=True)
                check(lib().lu_batched_inverse(A.ptr + 4 * pad.size, P.ptr, n, count, flags))
                got, piv = A.download(host.shape, np.float32), P.download((count * n + 1,), np.int32)
            finally:
                A.close()
                P.close()
            assert np.array_equal(got[:pad.size], pad) and np.array_equal(got[pad.size + count * n * n:], pad)
            mid = got[pad.size:pad.size + count * n * n].reshape(count, n, n)
            assert np.array_equal(mid.view(np.uint32), x[:count].view(np.uint32))
            assert np.array_equal(piv[:-1].reshape(count, n), p[:count]) and piv[-1] == -5
