"""Inference on both sides of the size up to which a wave takes one group of 16
samples: the same outputs to the bit."""
import numpy as np
import pytest

from test_gpu_surrogate import _random_model
from walicxe2d_amd import surrogate as S

pytestmark = pytest.mark.gpu


def test_forms_agree():
    m = _random_model(11)
    x = np.random.default_rng(12).normal(size=(40000, 4)).astype(np.float32)
    y = S.infer(m, x)
    for n in (1, 15, 16, 17, 63, 64, 65, 16383, 16384, 16385, 16449):
        assert np.array_equal(S.infer(m, x[:n]).view(np.int32), y[:n].view(np.int32)), n
