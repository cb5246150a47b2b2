"""The layers' descriptor plans (fields kept from call to call): every change a user can make to a module between
two calls reaches the next call, a copied or reloaded module does not use another's plan, and calls from several
threads on streams of their own do not disturb each other."""
import copy
import io
import threading

import pytest
import torch
import torch.nn.utils.parametrize

from hip_helpers import DEV, need_gpu
from tesm_amd import FeedForward, RMSNorm, TESM_SISO, TESMConfig, TESMMIMO_Optimized

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _gpu():
    need_gpu()


def _make(kind, dtype=torch.float32, seed=0):
    torch.manual_seed(seed)
    if kind == "ffn":
        m = FeedForward(TESMConfig(d_model=64, d_intermediate=128))
    elif kind == "mimo":
        m = TESMMIMO_Optimized(d_model=64, d_state=32, n_heads=2, ent_rank=8, entanglement_window=8,
                               entanglement_threshold=0.08, max_seq_len=64)
    else:
        m = TESM_SISO(d_model=64, d_state=32, ent_rank=8, entanglement_window=8 if kind == "siso" else 0,
                      entanglement_threshold=0.08, max_seq_len=64)
    return m.to(DEV).to(dtype).eval()


def _out(m, u):
    with torch.no_grad():
        out = m(u)
    return out[0] if isinstance(out, tuple) else out


def _u(dtype=torch.float32, L=40, seed=1):
    return torch.randn(2, L, 64, generator=torch.Generator().manual_seed(seed)).to(dtype).to(DEV)


KINDS = ["siso", "global", "mimo", "ffn"]


@pytest.mark.parametrize("kind", KINDS)
def test_weight_and_option_changes_reach_the_next_call(kind):
    """Each change is compared with a module that never had a plan."""
    m, u = _make(kind), _u()
    _out(m, u)
    other = _make(kind, seed=5)
    first = "gate_proj" if kind == "ffn" else "in_proj"
    edits = [lambda x: getattr(x, first).weight.data.mul_(-1.0).add_(0.01),        # in place through .data + version
             lambda x: setattr(x, first, copy.deepcopy(getattr(other, first))),       # a replaced submodule
             lambda x: getattr(x, first).__setattr__("weight", torch.nn.Parameter(getattr(other, first).weight * 0.5))]
    if kind != "ffn":
        edits += [lambda x: x.decay_bias.add_(0.5), lambda x: setattr(x, "entanglement_threshold", 0.3)]
    for i, edit in enumerate(edits):
        with torch.no_grad():
            edit(m)
            if i == 0:
                getattr(m, first).weight.add_(0.0)  # bump the version the packed cache follows
        fresh = _make(kind)
        fresh.load_state_dict(m.state_dict())
        if kind != "ffn":
            fresh.entanglement_threshold = m.entanglement_threshold
        assert torch.equal(_out(m, u), _out(fresh, u)), (kind, i)
        assert torch.equal(_out(m, _u(L=17, seed=9)), _out(fresh, _u(L=17, seed=9))), (kind, i)


@pytest.mark.parametrize("kind", KINDS)
def test_copied_and_reloaded_modules(kind):
    m, u = _make(kind), _u()
    want = _out(m, u)
    twin = copy.deepcopy(m)
    buf = io.BytesIO()
    torch.save(m, buf)
    buf.seek(0)
    loaded = torch.load(buf, weights_only=False)
    with torch.no_grad():
        for p in m.parameters():
            p.zero_()
    del m
    for x in (twin, loaded):
        assert torch.equal(_out(x, u), want)


@pytest.mark.parametrize("kind", KINDS)
def test_dtype_mismatch_still_refused(kind):
    m = _make(kind)
    _out(m, _u())
    with pytest.raises(RuntimeError, match="same dtype"):
        _out(m, _u(torch.bfloat16))


class _Scale(torch.nn.Module):
    factor = 2.0

    def forward(self, x):
        return x * self.factor


@pytest.mark.parametrize("kind", ["siso", "global", "mimo"])
def test_parametrized_decay_bias(kind):
    """A parameter that a parametrization computes anew for every access, and its later changes, reach the call."""
    m, plain, u = _make(kind), _make(kind), _u()
    rule = _Scale()
    torch.nn.utils.parametrize.register_parametrization(m, "decay_bias", rule)
    for factor in (2.0, -1.0, 0.5):
        rule.factor = factor
        with torch.no_grad():
            plain.decay_bias.copy_(m.parametrizations.decay_bias.original * factor)
        assert torch.equal(_out(m, u), _out(plain, u)), factor


def test_parametrized_norm_weight():
    m, plain, u = RMSNorm(64).to(DEV).eval(), RMSNorm(64).to(DEV).eval(), _u()
    torch.nn.utils.parametrize.register_parametrization(m, "weight", _Scale())
    with torch.no_grad():
        plain.weight.mul_(2.0)
    assert torch.equal(_out(m, u), _out(plain, u))


def test_threads_on_their_own_streams():
    m = _make("siso")
    us = [_u(L=8 + 7 * i, seed=20 + i) for i in range(4)]
    want = [_out(m, u) for u in us]
    torch.cuda.synchronize()
    got, errors = [None] * 4, []

    def work(i):
        try:
            s = torch.cuda.Stream()
            with torch.cuda.stream(s):
                for _ in range(20):
                    got[i] = _out(m, us[i])
            s.synchronize()
        except Exception as e:  # noqa: BLE001 - reported below
            errors.append(e)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in ts]
    [t.join(60) for t in ts]
    assert not errors
    for g, w in zip(got, want):
        assert torch.equal(g, w)


@pytest.mark.parametrize("kind", ["siso", "global", "mimo"])
def test_parametrized_decay_bias_under_inference_mode(kind):
    """There the computed bias is an inference tensor, which has no version a plan could compare."""
    m, plain, u = _make(kind), _make(kind), _u()
    rule = _Scale()
    torch.nn.utils.parametrize.register_parametrization(m, "decay_bias", rule)
    for factor in (2.0, -1.0, 0.5):
        rule.factor = factor
        with torch.no_grad():
            plain.decay_bias.copy_(m.parametrizations.decay_bias.original * factor)
        with torch.inference_mode():
            assert torch.equal(m(u)[0], plain(u)[0]), factor


@pytest.mark.parametrize("kind,name", [("siso", "local_entanglement_bias"), ("global", "global_rel_pos_embed"),
                                       ("global", "global_rel_pos_scale"), ("global", "global_rel_pos_bias"),
                                       ("mimo", "local_entanglement_bias"), ("mimo", "mimo_x"), ("mimo", "mimo_o")])
def test_parametrized_parameters_bf16(kind, name):
    """Values that are rounded or combined before a plan holds them: each of a row of changed ones reaches the call,
    though the allocator hands out the addresses of earlier ones again."""
    dt = torch.bfloat16
    m, plain, u = _make(kind, dt), _make(kind, dt), _u(dt)
    with torch.no_grad():
        for x in (m, plain):
            getattr(x, name).add_(0.25)
    rule = _Scale()
    torch.nn.utils.parametrize.register_parametrization(m, name, rule)
    for factor in (2.0, -1.0, 0.5, 4.0, 2.0, -3.0, 0.25):
        rule.factor = factor
        with torch.no_grad():
            getattr(plain, name).copy_(getattr(m.parametrizations, name).original * factor)
        assert torch.equal(_out(m, u), _out(plain, u)), factor


@pytest.mark.parametrize("kind,name", [("siso", "decay_bias"), ("siso", "local_entanglement_bias"), ("global", "decay_bias"),
                                       ("mimo", "decay_bias"), ("mimo", "local_entanglement_bias")])
def test_parametrized_biases_in_decode_steps(kind, name):
    m, plain, u = _make(kind), _make(kind), _u(L=12)
    rule = _Scale()
    torch.nn.utils.parametrize.register_parametrization(m, name, rule)
    caches = [{"state_cache": x.allocate_inference_cache(2, 64)} for x in (m, plain)]
    for t in range(9):
        rule.factor = (2.0, -1.0, 0.5)[t % 3]
        with torch.no_grad():
            getattr(plain, name).copy_(getattr(m.parametrizations, name).original * rule.factor)
            y, want = (x(u[:, t:t + 1], inference_params=c)[0] for x, c in zip((m, plain), caches))
        assert torch.equal(y, want), t
