"""GPU checks of the window-64 form of the MIMO mix (mix64) at its edges, against the oracle: a last block of channels
that is not whole after whole ones, workgroups of fewer than their four blocks, and lengths of one position, one below
and one past a workgroup's 64 and one past two of them."""
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
@pytest.mark.parametrize("L,D", [(129, 132), (65, 516), (64, 644), (100, 128), (1, 644), (63, 132)])
def test_window_64_mix(dtype, L, D):
    meta = dict(seed=L + D, dm=64, D=D, H=2, Rm=2, R=16, W=64, thr=0.05, decay_bias=2.0, max_seq_len=160)
    ref = build(ot.TESMMIMO_Optimized, meta).to(dtype)
    m = build(TESMMIMO_Optimized, meta).to(DEV).to(dtype)
    u = torch.randn(2, L, 64, generator=torch.Generator().manual_seed(7)).to(dtype)
    with torch.no_grad(), hip_ops.launch_log() as log:
        m(u.to(DEV))
    assert any(k.startswith("mimo_mix_kernel<") and k.endswith(",true,64>") for k in log.kernels), log.kernels
    _prefill_lockstep(ref, m, u, dtype)
