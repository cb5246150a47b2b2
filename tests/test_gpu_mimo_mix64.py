"""GPU checks of the window-64 form of the MIMO mix (mix64) at its edges, against the oracle: a last block of channels
that is not whole after whole ones, workgroups of fewer than their four blocks, lengths of one position, one below and
one past a workgroup's 64 and one past two of them, and widths on both sides of the line up to which it is taken."""
import pytest
import torch

from hip_helpers import DEV, need_gpu
from oracle import tesm_torch as ot
from tesm_amd import TESMMIMO_Optimized, hip_ops
from test_gpu_mimo import _prefill_lockstep, build

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _gpu():
    need_gpu()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("L,D,taken", [(129, 116, True), (65, 500, True), (64, 644, True), (100, 128, True), (1, 644, True),
                                       (63, 160, True), (70, 64, True), (70, 60, False), (129, 132, False)])
def test_window_64_mix(dtype, L, D, taken):
    meta = dict(seed=L + D, dm=64, D=D, H=2, Rm=2, R=16, W=64, thr=0.05, decay_bias=2.0, max_seq_len=160)
    ref = build(ot.TESMMIMO_Optimized, meta).to(dtype)
    m = build(TESMMIMO_Optimized, meta).to(DEV).to(dtype)
    u = torch.randn(2, L, 64, generator=torch.Generator().manual_seed(7)).to(dtype)
    with torch.no_grad(), hip_ops.launch_log() as log:
        m(u.to(DEV))
    names = [k for k in log.kernels if k.startswith("mimo_mix_kernel<")]
    assert len(names) == 1 and names[0].endswith(",true,64>") == taken, names
    _prefill_lockstep(ref, m, u, dtype)


def test_window_64_mix_of_more_workgroups_than_fit_at_once():
    """There narrower last blocks go to the general form, and both give one bit pattern (rows of a batch are alike)."""
    meta = dict(seed=5, dm=64, D=64, H=8, Rm=2, R=16, W=64, thr=0.05, decay_bias=2.0, max_seq_len=160)
    m = build(TESMMIMO_Optimized, meta).to(DEV)
    u = torch.randn(1, 130, 64, generator=torch.Generator().manual_seed(7)).to(DEV)
    out, form = [], []
    for B in (1, 2 * torch.cuda.get_device_properties(0).multi_processor_count // 24 + 1):
        with torch.no_grad(), hip_ops.launch_log() as log:
            out.append(m(u.expand(B, -1, -1).contiguous())[0])
        form += [k.endswith(",true,64>") for k in log.kernels if k.startswith("mimo_mix_kernel<")]
    assert form == [True, False]
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[1][0], out[1][-1])
