"""The layers' descriptor plans, built without a GPU: the packed weights and the one kernel a plan may launch are stubbed
(what is tested is which of the module's parameters a plan holds, and when it is made anew), and a plan's parameters are
read back through the addresses in its descriptor."""
import ctypes

import numpy as np
import pytest
import torch
import torch.nn.utils.parametrize

from tesm_amd import TESM_SISO, TESMMIMO_Optimized, hip_ops
from tesm_amd.bitlinear import BitLinear, PackedWeight

KINDS = ["siso", "global", "mimo"]
D, H = 32, 2


@pytest.fixture(autouse=True)
def _stubs(monkeypatch):
    packs = {}

    def packed_weight(lin):
        z = torch.zeros(1)
        return packs.setdefault(id(lin), PackedWeight(torch.zeros(lin.out_features, 64, dtype=torch.uint8), z, z,
                                                      lin.out_features, lin.in_features))

    monkeypatch.setattr(BitLinear, "packed_weight", packed_weight)
    monkeypatch.setattr(hip_ops, "require_device", lambda *ts: None)
    monkeypatch.setattr(TESMMIMO_Optimized, "_make_coef",
                        staticmethod(lambda ts: (ts[0].float().sum(1), ts[1].float().sum(1))), raising=False)


class _Scale(torch.nn.Module):
    factor = 2.0

    def forward(self, x):
        return x * self.factor


def _make(kind, dtype=torch.float32):
    torch.manual_seed(0)
    kw = dict(d_model=64, d_state=D, ent_rank=8, entanglement_window=0 if kind == "global" else 8, max_seq_len=64)
    m = TESMMIMO_Optimized(n_heads=H, **kw) if kind == "mimo" else TESM_SISO(**kw)
    return m.to(dtype).eval()


def _prefill_plan(m, dtype=torch.float32):
    """(descriptor, what it keeps alive)"""
    if isinstance(m, TESMMIMO_Optimized):
        return m._mimo_layer_plan(dtype, torch.device("cpu"))
    return m._layer_plan(dtype, torch.device("cpu"), False)


def _floats(address, n):
    return np.array((ctypes.c_float * n).from_address(address))


@pytest.mark.parametrize("kind", KINDS)
def test_inference_tensors_count_as_changed(kind):
    """Under inference_mode a computed parameter is an inference tensor, which has no version to compare."""
    m = _make(kind)
    n = m.decay_bias.numel()
    rule = _Scale()
    torch.nn.utils.parametrize.register_parametrization(m, "decay_bias", rule)
    with torch.inference_mode():
        for factor in (2.0, -1.0, -1.0, 0.5):
            rule.factor = factor
            desc, keep = _prefill_plan(m)
            want = m.parametrizations.decay_bias.original.numpy().reshape(-1) * factor
            assert np.array_equal(_floats(desc.decay_bias, n), want), factor
