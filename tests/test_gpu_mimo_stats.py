"""GPU checks of the sampled MIMO entanglement statistics (mimo_stats_kernel) at the edges of its work split, against the
oracle: rows staged whole and in slices, one and several heads side by side, more scores of a head than threads, and
score counts that leave threads idle, for the window and the global branch."""
import pytest
import torch

from hip_helpers import DEV, need_gpu
from oracle import tesm_torch as ot
from test_gpu_mimo import build
from tesm_amd import TESMMIMO_Optimized

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _gpu():
    need_gpu()


# (B, L, H, R, W): W 0 is the global branch (all heads' products in one score: 2 x 180 and 4 x 64)
CASES = [(1, 64, 4, 256, 64), (1, 20, 2, 300, 8), (2, 3, 1, 6, 2), (1, 70, 3, 64, 16), (2, 40, 5, 34, 9),
         (1, 1, 2, 16, 4), (1, 33, 2, 180, 0), (2, 9, 4, 64, 0)]
# rows of more than a slice (rank a multiple of 4 or not; the global branch's too), more than 1024 scores of a head,
# three heads of a group of two
CASES += [(1, 64, 1, 400, 1), (1, 64, 2, 402, 2), (1, 40, 2, 604, 0), (1, 64, 2, 20, 32), (1, 64, 3, 250, 64)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,L,H,R,W", CASES)
def test_stats_work_split(dtype, B, L, H, R, W):
    meta = dict(seed=L + R, dm=64, D=16, H=H, Rm=2, R=R, W=max(W, 1), thr=0.05, decay_bias=2.0, max_seq_len=128)

    def make(cls):
        if W:
            return build(cls, meta)
        torch.manual_seed(meta["seed"])
        return cls(d_model=64, d_state=16, n_heads=H, mimo_rank=2, ent_rank=R, entanglement_window=0,
                   entanglement_threshold=0.05, max_seq_len=128).eval()

    ref, m = make(ot.TESMMIMO_Optimized).to(dtype), make(TESMMIMO_Optimized).to(DEV).to(dtype)
    u = torch.randn(B, L, 64, generator=torch.Generator().manual_seed(9)).to(dtype)
    with torch.no_grad():
        ref(u)
        m(u.to(DEV))
    want, got = ref._stats_ternary_buffer, m._stats_ternary_buffer.cpu()
    assert got.dtype == dtype and got.shape == want.shape
    # A score one rounding step away (the order of its float32 sum, or of the projections before it) flips a decision
    # next to the threshold.  The scores spread over about their own size, and a step is 2^-8 of it in bf16, so a share
    # of up to p = 4 * 2^-8 * 0.4 = 0.6 % (two thresholds, both sides) may flip; p = 1 % (float32, whose sums alone
    # move: 0.2 %) as in test_gpu_mimo, and with few scores four standard deviations of that count.
    mean = (0.002 if dtype == torch.float32 else 0.01) * want.numel()
    flips = int((got != want).sum())
    assert flips <= mean + 4 * mean ** 0.5, flips
    n = got.numel()
    frac = {"positive": int((got > 0).sum()) / n, "negative": int((got < 0).sum()) / n, "zero": int((got == 0).sum()) / n}
    for k, v in m.last_entanglement_stats.items():  # the counts are those of the decisions
        assert abs(v - frac[k]) < 1e-6, (k, v, frac[k])
