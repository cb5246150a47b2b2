"""GPU checks of the register-mix entanglement kernel's one-half form (8 positions per workgroup, rows of more than 256
channels) against the older kernels, bit for bit, at its edges; the check itself is test_gpu_ent_reg's."""
import pytest
import torch

from hip_helpers import need_gpu
from test_gpu_ent_reg import test_ent_reg_matches_older_kernels as _check

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _gpu():
    need_gpu()


# (B, L, R, D, W, cross): the narrowest and widest rows of the form and the row width next below it (both halves);
# lengths one below, at and one past the 8-position block and past two; a window of one; key rows of more items than
# the first staging round takes; a rank that is no multiple of 8
SHAPES = [(2, 7, 64, 320, 32, False), (1, 8, 96, 512, 32, True), (1, 9, 80, 512, 32, False), (3, 17, 128, 320, 32, True),
          (1, 25, 30, 448, 32, False), (1, 33, 256, 384, 1, False), (2, 50, 128, 256, 32, True)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "B{}xL{}_R{}_D{}_W{}{}".format(*s[:5], "_cross" if s[5] else ""))
def test_one_half_matches_older_kernels(shape, dtype, monkeypatch):
    _check(shape, dtype, monkeypatch)
