"""BatchNormalization where a thread takes one to four vectors of its channel, chosen so that few channels do not leave the
chip in many small workgroups: shapes on both sides of each step of that choice, with the checks of the spans' own tests."""
import pytest
import torch

from daceml_amd import _lib as L
from tests import test_zx_batchnorm_spans as spans

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("act", [L.ACT_NONE, L.ACT_SWISH])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("shape", [(4, 20, 8192), (4, 21, 8192), (16, 24, 3136), (8, 64, 3136), (8, 64, 3135), (16, 96, 3136)])
def test_vectors_per_thread(shape, dtype, act, lib):
    spans.test_spans(shape, dtype, 0, act, lib)
