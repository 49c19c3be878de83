"""FP64 hdiff past 400 MiB of fields by the default rule: widths that fill just under and just over 60% of the 128-column strips,
odd ones among them; the bits of the oracle, so the tolerance is zero."""
import numpy as np
import pytest

from test_gpu_hdiff_flat import _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ni,nj,nk", [(76, 2950, 80), (77, 2910, 80), (131, 1710, 80), (153, 1470, 80), (154, 1460, 80)])
def test_default_rule(gpu, oracle, ni, nj, nk):
    _run(gpu, oracle, ni, nj, nk, np.float64, 0, "native")
