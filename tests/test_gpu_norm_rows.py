"""The norm and quantiser at the row counts where a row's thread count
changes (one row a CU, three), at widths that leave threads idle and that do
not fill the sum's 512 partials.  Bit for bit against the oracle, as the few
rows of the other tests are.
"""
import pytest
import torch

from tests import test_gpu_qwen as base

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("times,more,K", [(1, 0, 96), (1, 1, 96), (1, 1, 2560), (3, 0, 1056), (3, 1, 32), (3, 1, 1056)])
def test_norm_quant_rows(dev, orc, times, more, K):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    base.test_norm_quant_bit_exact(dev, orc, times * cus + more, K)
