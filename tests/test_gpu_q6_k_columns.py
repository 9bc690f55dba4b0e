"""The Q6_K product of several columns, on the matrix cores and in the vector
kernel's wider forms: each column bit for bit what the one-column kernel gives
it, outputs and superblock integers."""
import numpy as np
import pytest

from golem_amd import capi, synth

pytestmark = pytest.mark.gpu

# rows, cols, M, first row, spare floats a row of y.  On the matrix cores:
# tiles' edges, one superblock, odd and past eight of them (a scale chunk), a
# second launch of one and of two columns, an odd number of column scales
# (columns times superblocks: 3 to 135), inputs of which fourteen columns fit
# the LDS, few columns of many rows.  On the vector kernel: 2, 3, 4, 6, 7 and 8
# columns, eight and nine of a row that only its four fit
CASES = [(64, 256, 3, 0, 0), (1000, 2560, 9, 0, 1), (129, 2816, 16, 3, 0), (257, 768, 17, 0, 0),
         (200, 2304, 18, 65, 4), (130, 512, 9, 0, 2), (130, 2816, 11, 0, 0), (200, 2304, 7, 0, 0),
         (257, 2304, 15, 3, 0), (65, 768, 5, 0, 1), (70, 5120, 16, 0, 0), (24600, 1280, 3, 5, 0),
         (24600, 1280, 8, 0, 0), (64, 256, 2, 0, 0), (1000, 2560, 6, 0, 1), (130, 2816, 3, 0, 0),
         (130, 2816, 4, 0, 0), (70, 2560, 8, 0, 0), (70, 5120, 7, 0, 0), (66, 8704, 8, 0, 0), (66, 8704, 9, 0, 0),
         (128, 6144, 16, 0, 0)]


@pytest.mark.parametrize("rows,cols,M,start,spare", CASES)
def test_columns_equal_one_at_a_time(dev, rows, cols, M, start, spare):
    g = synth.rng(rows + cols + M)
    w = dev.weight(synth.q6_k_weights(g, rows, cols), capi.Q6_K, rows, cols)
    x = synth.activations(g, M, cols)
    x[-1, :256] = 0.0  # a zero superblock
    x[0] *= 1e6
    q, ks, bs = dev.quantize_q8_k(x)
    bias = synth.activations(g, 1, rows)[0]
    end = rows - (3 if start else 0)
    y = dev.full((M, rows + spare), float("nan"))
    got = dev.get(dev.matmul_q6_k(w, (q, ks, bs), M, start, end, bias=bias, y=y))
    dots = dev.q6_k_block_dots(w, (q, ks, bs), M, start, end)
    for c in range(M):
        one = (q[c:c + 1], ks[c:c + 1].contiguous(), bs[c:c + 1].contiguous())
        want = dev.get(dev.matmul_q6_k(w, one, 1, start, end, bias=bias))
        assert np.array_equal(got[c, start:end].view(np.uint32), want[0, start:end].view(np.uint32)), c
        assert np.array_equal(dots[c], dev.q6_k_block_dots(w, one, 1, start, end)[0]), c
    assert np.isnan(got[:, :start]).all() and np.isnan(got[:, end:]).all()  # nothing else is written
    w.free()
