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


def test_longest_one_pass_against_the_general_kernels():
    """Positions of which many round to one bf16 value: the longest sequence the one-pass kernel takes against the same
    positions of one that is longer by a token, which takes the general kernels (the layer is causal).  The two add a
    score's products in another order, so a decision next to the threshold may differ, which moves its row's average by
    less than two parts in its decision count; a wrong bias entry would show as leaving the bias out does."""
    L, kw = 32768, dict(d_model=32, d_state=16, ent_rank=16, max_seq_len=33000)
    m = _siso(TESM_SISO, 3, torch.bfloat16, **kw).to(DEV)
    u = torch.randn(1, L + 1, 32, generator=torch.Generator().manual_seed(4)).to(torch.bfloat16).to(DEV)
    with torch.no_grad():
        with hip_ops.launch_log() as log:
            y = m(u[:, :L].contiguous())[0].float()
        with hip_ops.launch_log() as log1:
            long = m(u)[0][:, :L].float()
        m.global_rel_pos_scale.zero_()
        m.global_rel_pos_bias.zero_()
        plain = m(u)[0][:, :L].float()
    names, names1 = ([n.split("<")[0] for n in lg.kernels] for lg in (log, log1))
    assert "global_mfma_kernel" in names and "global_mfma_kernel" not in names1 and "global_scores_kernel" in names1
    for part in (slice(0, 4096), slice(4096, 16384), slice(16384, L)):  # (by how far positions round)
        d = float((y - long)[:, part].norm() / long[:, part].norm())
        without = float((plain - long)[:, part].norm() / long[:, part].norm())
        print(f"positions {part.start}-{part.stop}: rel. L2 {d:.2e}, without the bias {without:.2e}")
        assert d <= 2.0 ** -8 and d <= without / 10, (part, d, without)
