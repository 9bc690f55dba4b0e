"""The device Q8_0 quantiser where its accesses differ: rows that start off a
16-byte boundary, outputs off theirs, remainders of a workgroup's 32 blocks.

Batch.quantizeBlock (nn/batch.go:109-143) against the oracle, bit for bit.
"""
import numpy as np
import pytest

from golem_amd import capi, synth
from tests.gpu_util import log, q16_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,pad,shift,qshift", [
    (1, 32, 0, 0, 0),        # one block
    (31, 32, 0, 0, 0),       # one short of a workgroup
    (33, 96, 4, 0, 0),       # one token past the fp16 copy's group, wide rows apart
    (33, 96, 3, 0, 0),       # rows off a 16-byte boundary
    (5, 2560, 0, 1, 0),      # the first row off it
    (5, 2560, 0, 0, 1),      # q off a 4-byte boundary
    (7, 704, 5, 3, 3),
])
def test_q8_0_layouts(dev, orc, M, K, pad, shift, qshift):
    log(f"q8_0 layouts M={M} K={K} pad={pad} shift={shift} qshift={qshift}")
    x = synth.activations(synth.rng(30 + M + pad), M, K)
    x[M // 2, :32] = 0.0
    b = orc.Batch(x).quantize()
    ldx = K + pad
    flat = np.full(shift + M * ldx, np.nan, np.float32)
    for m in range(M):
        flat[shift + m * ldx:shift + m * ldx + K] = x[m]
    xd = dev.put(flat)[shift:]
    q = dev.full((qshift + M * K + 4,), 77, np.int8)
    sc = dev.empty((M, K // 32), np.float32)
    qs = dev.empty((M, K // 32), np.int32)
    co = dev.empty((M, K // 32), np.float32)
    q16 = dev.empty((capi.q16_elems(M, K) + qshift,), np.int16)[qshift:]
    for out16 in (q16, None):
        capi.call("gx_quantize_q8_0", dev.ctx.ptr, capi.vp(xd), ldx, M, K, capi.vp(q[qshift:]), capi.vp(sc),
                  capi.vp(qs), capi.vp(co), capi.vp(out16))
        got = dev.get(q)
        np.testing.assert_array_equal(got[qshift:qshift + M * K].reshape(M, K), b.q_rows())
        assert np.all(got[:qshift] == 77) and np.all(got[qshift + M * K:] == 77)
        np.testing.assert_array_equal(dev.get(sc).view(np.uint32), b.scales_rows().view(np.uint32))
        np.testing.assert_array_equal(dev.get(qs), b.qsum_rows())
        np.testing.assert_array_equal(dev.get(co).view(np.uint32), b.corr_rows().view(np.uint32))
        q[:] = 77
    rows16 = q16_rows(dev.get(q16), M, K)
    np.testing.assert_array_equal(rows16[:M], b.q_rows().astype(np.float32))
    assert not np.any(rows16[M:])
