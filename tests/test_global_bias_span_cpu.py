"""The slice of the global entanglement's bias table that global_mfma_kernel stages for a block of queries and keys holds
every entry the block's scores read, for every block up to the length the kernel takes: its index arithmetic
(positions and their difference rounded to bf16, as the layer dtype rounds them) enumerated on the CPU, with the sizes
read from the source."""
import os
import re

import torch

from conftest import ROOT


def _constants():
    with open(os.path.join(ROOT, "tesm_amd", "csrc", "global_mfma.hip")) as f:
        text = f.read()
    get = lambda name: int(re.search(rf"constexpr \w+ {name} = (\d+);", text).group(1))  # noqa: E731
    waves = int(re.search(r"constexpr int kGNW = (\d+), kGNT = 64 \* kGNW;", text).group(1))
    assert "constexpr int kGTab = kGNT;" in text
    return get("kGQ"), get("kGK"), 64 * waves, get("kGMaxL")


def _rel(x, y):
    bf = torch.bfloat16
    return (x.float().to(bf).float() - y.float().to(bf).float()).to(bf).float().to(torch.int64)


def test_a_blocks_bias_entries_fit_the_staged_slice():
    Q, K, staged, max_l = _constants()
    worst = 0
    for i0 in range(0, max_l, Q):
        k0 = torch.arange(0, i0 + Q, K)  # the key blocks these queries reach
        lo = _rel(torch.tensor(i0), k0 + K - 1).clamp(min=0)
        # the difference is monotone in both positions, so a block's entries lie between its corners'
        hi = _rel(torch.tensor(i0 + Q - 1), k0)
        assert bool((hi - lo < staged).all()), i0
        worst = max(worst, int((hi - lo).max()))
    assert worst == 256  # (257 entries; reached where positions round by up to 64)


def test_rounded_differences_are_monotone_and_causal():
    """What the corners stand on: rounding keeps order, and a key that is not past its query has a difference of zero
    or more and at least the slice's first entry."""
    _, K, _, max_l = _constants()
    pos = torch.arange(max_l)
    assert bool((pos.float().to(torch.bfloat16).float().diff() >= 0).all())
    for i in range(0, max_l, 997):
        d = _rel(torch.tensor(i), pos[:i + 1])
        assert bool((d >= 0).all()) and bool((d.diff() <= 0).all())
