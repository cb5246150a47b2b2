"""The layers' descriptor plans, built without a GPU: the packed weights and the one kernel a plan may launch are stubbed
(what is tested is which of the module's parameters a plan holds, and when it is made anew), and a plan's parameters are
read back through the addresses in its descriptor."""
import copy
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
    if kind == "global":
        torch.nn.init.constant_(m.global_rel_pos_bias, 0.5)
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


class _Reused(torch.nn.Module):
    """A rule whose every value lies at one address and starts at version 0: what a caching allocator may hand out for
    values of one size that are computed anew and freed again."""

    def forward(self, x):
        if not hasattr(self, "buf"):
            self.buf = torch.empty_like(x)
        self.buf.copy_(x * self.factor)
        return self.buf.data

    factor = 2.0


# a plan's field for each parameter, and its values there: the module rounds them to its dtype, the plan holds floats
FIELDS = [("siso", "decay_bias", "decay_bias"), ("siso", "local_entanglement_bias", "local_bias"),
          ("global", "global_rel_pos_embed", "global_embed"), ("global", "global_rel_pos_scale", "global_scale"),
          ("global", "global_rel_pos_bias", "global_bias"), ("mimo", "local_entanglement_bias", "local_bias"),
          ("mimo", "mimo_x", "mimo_coef"), ("mimo", "mimo_o", "mimo_x0sq")]


@pytest.mark.parametrize("kind,name,field", FIELDS)
def test_computed_values_are_not_taken_for_older_ones(kind, name, field):
    """A value that a parametrization computes at an older one's address reaches the plan all the same."""
    dt = torch.float32 if name == "decay_bias" else torch.bfloat16  # (the plan holds a float32 copy of the others)
    m = _make(kind, dt)
    rule = _Reused()
    torch.nn.utils.parametrize.register_parametrization(m, name, rule, unsafe=True)
    for factor in (2.0, -1.0, 0.5, 4.0, 2.0, -3.0):
        rule.factor = factor
        with torch.no_grad():
            desc, keep = _prefill_plan(m, dt)
            want = getattr(m, name).to(torch.float32)
        want = want.sum(1) if name.startswith("mimo") else want
        assert np.array_equal(_floats(getattr(desc, field), want.numel()), want.numpy().reshape(-1)), factor


@pytest.mark.parametrize("kind", KINDS)
def test_copies_hold_no_derived_values(kind):
    m = _make(kind, torch.bfloat16)
    _prefill_plan(m, torch.bfloat16)
    held = [k for k, v in m.__dict__.items() if isinstance(v, tuple) and v and isinstance(v[0], tuple)]
    assert held
    twin = copy.deepcopy(m)
    assert not [k for k in held if twin.__dict__.get(k) is not None]
    assert _prefill_plan(twin, torch.bfloat16)[0].d_state == D


@pytest.mark.parametrize("kind,name", [("siso", "decay_bias"), ("siso", "local_entanglement_bias"), ("global", "decay_bias"),
                                       ("mimo", "decay_bias"), ("mimo", "local_entanglement_bias")])
@pytest.mark.parametrize("mode", [torch.no_grad, torch.inference_mode])
def test_decode_plans_take_computed_biases(kind, name, mode):
    dt, cpu = torch.float32 if name == "decay_bias" else torch.bfloat16, torch.device("cpu")
    m = _make(kind, dt)
    rule = _Reused()
    torch.nn.utils.parametrize.register_parametrization(m, name, rule, unsafe=True)
    args = (4, dt, cpu, torch.float32, 1 if kind == "global" else 8, False)
    field = "decay_bias" if name == "decay_bias" else "local_bias"
    for factor in (2.0, -1.0, 0.5, 2.0):
        rule.factor = factor
        with mode():
            desc, _, keep = m._mimo_step_plan(*args) if kind == "mimo" else m._step_plan(*args)
        want = (getattr(m.parametrizations, name).original * factor).detach().float().reshape(-1)
        assert np.array_equal(_floats(getattr(desc, field), want.numel()), want.numpy()), factor
