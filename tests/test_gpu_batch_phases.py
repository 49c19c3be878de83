"""The two-phase batching form at the sizes where its kernels split: the vertical phase's depth classes at both edges
of each, also with several items per wavefront crossing from one class to the next; the stencil phase's narrowest and
lowest domains, widths around a wavefront's 60 pairs and lists that end inside a chunk of 64 wavefronts.  FP64 and the native FP32 and mixed
forms equal the oracle chain bit for bit, so the tolerance is zero."""
import numpy as np
import pytest

from test_gpu_batch import check_batch

pytestmark = pytest.mark.gpu

FORMS = [(np.float64, 0), (np.float32, 1), (np.float32, 0)]
# one domain per class edge
EDGES = [(65, 2, nk) for nk in (2, 8, 9, 40, 41, 48, 49, 56, 57, 64, 65, 72, 73, 80, 81, 104, 105, 112, 113, 128, 129,
                                136, 137, 144)]
# 512 wavefronts (two per CU on 256 CUs) walk classes of fewer and of more items than that
MANY = [(130, 200, 120), (70, 90, 100), (64, 300, 75), (200, 150, 60), (33, 40, 50), (140, 250, 44), (66, 300, 10)]


@pytest.mark.parametrize("dtype,precision", FORMS)
def test_vertical_depth_classes(gpu, oracle, dtype, precision):
    check_batch(gpu, oracle, EDGES, dtype, precision, wg_per_cu=2, rounded_ustage=True)


@pytest.mark.parametrize("dtype,precision", FORMS)
def test_vertical_items_across_classes(gpu, oracle, dtype, precision):
    check_batch(gpu, oracle, MANY, dtype, precision, wg_per_cu=1, rounded_ustage=True)


# (1, ...) takes the one-column sweep, as do domains of fewer rows than a wavefront's
NARROW = [(1, 5, 4), (2, 1, 3), (3, 2, 5), (2, 4, 7), (4, 3, 2), (113, 3, 9), (116, 7, 6), (117, 33, 21), (118, 4, 40),
          (119, 5, 3), (120, 6, 3), (121, 9, 3), (240, 1, 5)]


@pytest.mark.parametrize("hjb", [8, 16, 32])
@pytest.mark.parametrize("dtype,precision", FORMS)
def test_stencil_widths(gpu, oracle, monkeypatch, dtype, precision, hjb):
    monkeypatch.setenv("GT355_TUNE_batch_hjb", str(hjb))
    check_batch(gpu, oracle, NARROW, dtype, precision, wg_per_cu=2, rounded_ustage=True)
