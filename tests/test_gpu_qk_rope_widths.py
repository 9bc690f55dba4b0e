"""The one-token head norm and rotation at head widths off its unrolled sizes:
a width under sixteen values, one that leaves a remainder of the sum's
sixteens, one with a part-full second pair a lane, the widest.  Bit for bit
against the oracle, as the widths 64 and 128 are.
"""
import pytest

from tests import test_gpu_qwen as base

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,heads,kv", [(8, 2, 1), (24, 3, 1), (96, 4, 2), (200, 2, 2), (256, 2, 1)])
def test_qk_rope_widths(dev, orc, hd, heads, kv):
    base.test_qk_rope_and_cache_bit_exact(dev, orc, hd, heads, kv, 6)
