"""The batch product's three tile shapes at the edges of their tiles: each
column bit for bit what the few-column kernel (at most 16 columns a call)
gives it, and the block integers of both kernels the same."""
import numpy as np
import pytest

from golem_amd import capi, synth

from .gpu_util import Device

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    d = Device()
    yield d
    d.close()


# rows, cols, M, first row, spare floats a row of y: 128 x 64 tiles (three
# whole rounds of 256 CUs, the last row tile and the last token part full), 64 x
# 64, 128 x 32 (to 32 tokens, and where the others need another round); rows
# past a tile, one block, blocks past a stage and a stretch
CASES = [(98304 - 63, 64, 63, 0, 0), (6000, 64, 129, 5, 1), (98304 + 65, 64, 64, 0, 0), (49152, 32, 65, 31, 3), (65, 32, 33, 0, 0), (1000, 2080, 65, 3, 1),
         (192, 4128, 130, 0, 4), (64, 288, 64, 0, 0), (1000, 96, 32, 64, 2), (129, 2592, 17, 0, 0)]


@pytest.mark.parametrize("rows,cols,M,start,spare", CASES)
def test_shapes_equal_few_columns(dev, rows, cols, M, start, spare):
    g = synth.rng(rows + cols + M)
    w = dev.weight(synth.q4_0_weights(g, rows, cols), capi.Q4_0, rows, cols)
    act = dev.quantize_q8_0(synth.activations(g, M, cols), with_corr=False, with_q16=False)
    bias = synth.activations(g, 1, rows)[0]
    end = rows - (5 if start else 0)
    y = dev.full((M, rows + spare), float("nan"))
    dev.matmul_q4_0(w, act, M, start, end, bias=bias, y=y)
    got = dev.get(y)
    for c in range(0, M, 16):
        n = min(16, M - c)
        part = tuple(None if a is None else a[c:c + n].contiguous() for a in act[:3]) + (None,)
        want = dev.full((n, rows), float("nan"))
        dev.matmul_q4_0(w, part, n, start, end, bias=bias, y=want)
        want = dev.get(want)
        assert np.array_equal(got[c:c + n, start:end].view(np.uint32), want[:, start:end].view(np.uint32)), c
    assert np.isnan(got[:, :start]).all() and np.isnan(got[:, end:]).all()  # nothing else is written
    lo = max(start, end - 200)
    dots = dev.q4_0_block_dots(w, act, M, lo, end, 1)
    n = min(16, M)
    part = tuple(a[:n].contiguous() for a in act[:3]) + (None,)
    assert np.array_equal(dots[:n], dev.q4_0_block_dots(w, part, n, lo, end, 5))
    w.free()
