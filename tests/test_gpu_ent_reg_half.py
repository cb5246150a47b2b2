"""GPU checks of the register-mix entanglement kernel's one-half form (8 positions per workgroup, rows of more than 256
channels) against the older kernels, bit for bit, at its edges; the check itself is test_gpu_ent_reg's."""
import pytest
import torch

from hip_helpers import DEV, need_gpu
from tesm_amd import hip_ops
from test_gpu_ent_reg import _case
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


# (grid of both halves in sixteenths of the CUs, R, D, W, dtype, halves): on both sides of the rule's lines, a few
# positions short of whole workgroups: odd and even numbers of one-half workgroups per CU, rounds of both from which one
# half is taken by width, rank and window, the parts of a first and fourth round, forms of many registers
F32, BF16 = torch.float32, torch.bfloat16
FORMS = [(8, 96, 384, 32, F32, 1), (9, 96, 384, 32, F32, 2), (20, 96, 384, 32, F32, 1), (30, 96, 384, 32, F32, 2),
         (46, 64, 384, 32, F32, 2), (58, 64, 384, 32, F32, 1), (78, 64, 384, 32, F32, 1), (52, 128, 384, 16, F32, 2),
         (94, 128, 384, 16, F32, 2),
         (15, 64, 320, 32, F32, 1), (15, 80, 320, 32, F32, 2), (30, 80, 320, 32, F32, 1), (30, 192, 320, 32, F32, 2),
         (36, 192, 320, 32, BF16, 2), (9, 80, 512, 32, F32, 1), (11, 80, 512, 32, F32, 2), (9, 112, 512, 32, F32, 2),
         (30, 80, 512, 32, F32, 1), (30, 128, 448, 32, F32, 2), (15, 80, 512, 16, F32, 1), (11, 256, 512, 16, F32, 1),
         (15, 256, 512, 16, F32, 2), (46, 256, 448, 16, F32, 2), (9, 80, 512, 32, BF16, 2), (30, 80, 512, 32, BF16, 1),
         (30, 128, 448, 32, BF16, 2)]


@pytest.mark.parametrize("sixteenths,R,D,W,dtype,halves", FORMS)
def test_form_by_grid(sixteenths, R, D, W, dtype, halves, monkeypatch):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    L = 16 * (cus * sixteenths // 16) - 3
    q, k, S, bias, _ = _case(1, L, R, D, W, dtype, seed=L + D)
    rope = hip_ops.rope_table(L, R, dtype, DEV)
    with hip_ops.launch_log() as log:
        hip_ops.local_ent_quant(q, k, rope, S, bias, W, 0.08, 0.2)
    names = [n for n in log.kernels if n.startswith("ent_reg_kernel<")]
    assert len(names) == 1 and names[0].split(",")[5] == str(halves), log.kernels
    _check((1, L, R, D, W, False), dtype, monkeypatch)
