"""GPU checks of the one-pass global entanglement of bf16 single-head layers (global_mfma_kernel) against the oracle, at
the edges of its tiles, and of which layers take it.  Decisions and codes are compared as in test_gpu_global: a
decision may differ from the oracle's only next to the threshold, and the outputs are compared with the device's."""
import pytest
import torch

from hip_helpers import DEV, TOL, need_gpu, normwise
from oracle import tesm_torch as ot
from tesm_amd import TESM_SISO, hip_ops
from test_gpu_global import _siso, _siso_lockstep

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _gpu():
    need_gpu()


# (B, L, R, D, cross, one pass): lengths around the 16-query blocks, the 32-key steps, the 64-key halves and the
# 128-key blocks; widths of one 16-channel tile, a ragged last wave, whole rows (quantized in place) and two channel
# blocks; ranks at both ends and next to the 32-value steps; layers beside the range, which take the general kernels
SHAPES = [(2, 1, 16, 16, False, True), (1, 15, 34, 48, False, True), (1, 16, 32, 256, True, True),
          (3, 17, 64, 240, False, True), (2, 64, 66, 272, False, True), (1, 65, 128, 256, False, True),
          (2, 127, 48, 32, True, True), (1, 128, 16, 512, False, True), (1, 129, 64, 256, False, True),
          (1, 290, 62, 528, True, True), (1, 900, 64, 256, False, True),
          (1, 70, 14, 64, False, False), (1, 70, 130, 64, False, False), (2, 70, 32, 40, False, False)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "B{}xL{}_R{}_D{}{}".format(*s[:4], "_cross" if s[4] else ""))
def test_one_pass_global_matches_oracle(shape):
    B, L, R, D, cross, one_pass = shape
    dt, kw = torch.bfloat16, dict(d_state=D, ent_rank=R, max_seq_len=1024)
    ref = _siso(ot.TESM_SISO, L + R + D, dt, **kw)
    m = _siso(TESM_SISO, L + R + D, dt, **kw).to(DEV)
    gen = torch.Generator().manual_seed(L + D)
    u = torch.randn(B, L, 96, generator=gen).to(dt)
    cs = torch.randn(B, L, D, generator=gen).to(dt) if cross else None
    _, f, fr = _siso_lockstep(ref, m, u, cs, dt)
    assert normwise(f.cpu().numpy(), fr.numpy()) <= TOL[dt]
    # without the taps (no float outputs are written then): the same outputs, and the kernels expected
    with torch.no_grad(), hip_ops.launch_log() as log:
        args = dict(cross_layer_state=cs.to(DEV) if cross else None)
        y0 = m(u.to(DEV), **args)[0]
        y1 = m(u.to(DEV), **args)[0]
        torch.cuda.synchronize()
    names = [n.split("<")[0] for n in log.kernels]
    assert ("global_mfma_kernel" in names) == one_pass and ("global_scores_kernel" in names) != one_pass, names
    assert torch.equal(y0, y1)
