"""The automatic lane layout (rows instead of quads for partial pivoting from
n = 9 and for small batches of n = 9..12) gives the same bits as either forced
layout, on both sides of each line, in the plain and refined inverse."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rule", [0x0, 0x1, 0x3, 0x4])
@pytest.mark.parametrize("n", [8, 9, 10, 11, 12, 13])
def test_auto_layout_matches_forced(gpu, n, rule):
    from matrixinversion_amd._native import check, lib

    gen = oracle.dominant_matrices if rule == 0 else oracle.uniform_matrices
    block = gen(60 + n, 512, n)
    for batch in (3, 8192, 8193, 16384, 16385):
        a = np.tile(block, (batch // 512 + 1, 1, 1))[:batch].copy()
        print(f"[case] layout n={n} rule={rule} batch={batch}", flush=True)
        x, p = gpu.invert(a, rule)
        for layout in (0x10, 0x20):
            xf, pf = gpu.invert(a, rule | layout)
            assert np.array_equal(x.view(np.uint32), xf.view(np.uint32)) and np.array_equal(p, pf)
        A, X, P = gpu.DeviceBuffer.from_array(a), gpu.DeviceBuffer(a.nbytes), gpu.DeviceBuffer(batch * n * 4)
        try:
            check(lib().lu_batched_inverse_refined(A.ptr, X.ptr, P.ptr, n, batch, rule, None))
            gpu.synchronize()
            r = X.download(a.shape, np.float32)
            assert np.array_equal(P.download((batch, n), np.int32), p)
        finally:
            for b in (A, X, P):
                b.close()
        # the tiled block: every repeat, and both sides of the lines, agree
        first = r[:min(batch, 512)]
        for lo in range(0, batch, 512):
            part = r[lo:lo + 512]
            assert np.array_equal(part.view(np.uint32), first[:part.shape[0]].view(np.uint32))
        if batch == 3:
            small = r
        else:
            assert np.array_equal(r[:3].view(np.uint32), small.view(np.uint32))
