"""GPU checks of the matrix-core window entanglement of wide bf16 layers (ent_mfma_kernel, d_state above 512).

It forms the same values as the scores + mix kernels and the activation quantization; only the order of the
float32 sums differs (the products of bf16 values are exact).  A sum of n terms reordered moves by at most
n * 2^-24 relative to its terms' magnitudes, far below a bf16 step (2^-8), so a rounded score or average may
move by one bf16 step where it lies next to a rounding boundary, and nothing else changes: a score's step
moves a ternary decision only next to the threshold, an average's step moves E and C by one step of E.
"""
import pytest
import torch

from hip_helpers import DEV, need_gpu
from tesm_amd import TESM_SISO, hip_ops

pytestmark = pytest.mark.gpu

THR, SCALE = 0.08, 0.2


@pytest.fixture(autouse=True)
def _gpu():
    need_gpu()


def _case(B, L, R, D, W, seed):
    g = torch.Generator().manual_seed(seed)
    make = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(DEV)  # noqa: E731
    return make(B, L, R), make(B, L, R), make(B, L, D), (torch.randn(W, generator=g) * 0.3).to(DEV), make(B, L, R)


# (B, L, R, D, W, cross): the large_40b layer's sizes; windows of 1 and at the edges of the 16-key tiles (17 / 18,
# 33 / 34); ranks that are no multiple of 8 or 32; widths at both ends of the range and with a last block of one
# 16-channel tile; lengths below the window, below and just past a 16-position block
SHAPES = [(1, 200, 256, 2048, 64, False), (2, 33, 64, 1024, 17, True), (1, 47, 80, 528, 18, False),
          (1, 64, 48, 784, 33, True), (1, 100, 30, 1040, 34, False), (2, 5, 16, 544, 64, False),
          (1, 17, 6, 640, 1, False), (1, 31, 256, 4096, 64, False), (3, 1, 32, 1024, 16, False)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "B{}xL{}_R{}_D{}_W{}{}".format(*s[:5], "_cross" if s[5] else ""))
def test_ent_mfma_matches_unfused(shape, monkeypatch):
    B, L, R, D, W, cross = shape
    q, k, S, bias, cq = _case(B, L, R, D, W, seed=L + R + D + W)
    qa = cq if cross else None
    rope = hip_ops.rope_table(L, R, torch.bfloat16, DEV)
    weff = min(W, L)
    with hip_ops.launch_log() as log:
        got = hip_ops.local_ent_quant(q, k, rope, S, bias, W, THR, SCALE, q_add=qa, want_floats=True, want_tern=True)
        torch.cuda.synchronize()
    assert any(n.startswith("ent_mfma_kernel<") for n in log.kernels), log.kernels
    monkeypatch.setenv("TESM_HIP_ENT_UNFUSED", "1")
    ref = hip_ops.local_ent(q, k, rope, S, bias[-weff:], weff, THR, SCALE, q_add=qa, outputs=("e_tanh", "c", "e"),
                            want_tern=True)
    tern, rt = got["tern"], ref["tern"][:, :, 0, :]
    same = (tern == rt).all(-1)
    assert same.float().mean() >= 0.999
    # rows with the same decisions: E within one bf16 step (2^-8 of its binade, at most 2^-7 relative)
    e = ref["e"].float()[same]
    step = e.abs() * 2.0 ** -7 + 2.0 ** -20
    dc = (got["c_float"].float()[same] - ref["c"].float()[same]).abs()
    dt = (got["e_tanh"].float()[same] - ref["e_tanh"].float()[same]).abs()
    assert bool((dc <= step).all()) and bool((dt <= step).all())
    assert float((dc > 0).float().mean()) <= 1e-2
    # the codes are the quantization of the kernel's own tanh(E) and C, bit for bit
    for name, fl in (("te", got["e_tanh"]), ("c", got["c_float"])):
        for a, b in zip(got[name], hip_ops.quant_act(fl.reshape(B * L, D))):
            assert torch.equal(a, b), name


def test_ent_mfma_unaligned_rows():
    """Rows that cannot be read in vectors (odd strides) give the bits of the aligned ones."""
    B, L, R, D, W = 1, 50, 64, 544, 16
    q, k, S, bias, _ = _case(B, L, R, D, W, seed=3)
    rope = hip_ops.rope_table(L, R, torch.bfloat16, DEV)
    a = hip_ops.local_ent_quant(q, k, rope, S, bias, W, THR, SCALE, want_tern=True)
    wide = torch.zeros(B, L, 2 * R + 3, dtype=torch.bfloat16, device=DEV)
    wide[..., 1:R + 1], wide[..., R + 1:2 * R + 1] = q, k
    b = hip_ops.local_ent_quant(wide[..., 1:R + 1], wide[..., R + 1:2 * R + 1], rope, S, bias, W, THR, SCALE,
                                want_tern=True)
    assert torch.equal(a["tern"], b["tern"])
    for name in ("te", "c"):
        for x, y in zip(a[name], b[name]):
            assert torch.equal(x, y), name


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_ent_mfma_nonfinite_state_stays_in_its_window(bad):
    """A state that is not finite reaches the positions whose window holds it and no others."""
    B, L, R, D, W, at = 1, 80, 32, 576, 16, 37
    q, k, S, bias, _ = _case(B, L, R, D, W, seed=5)
    rope = hip_ops.rope_table(L, R, torch.bfloat16, DEV)
    clean = hip_ops.local_ent_quant(q, k, rope, S, bias, W, THR, SCALE, want_floats=True)["c_float"]
    S2 = S.clone()
    S2[0, at, 100] = bad
    got = hip_ops.local_ent_quant(q, k, rope, S2, bias, W, THR, SCALE, want_floats=True)["c_float"]
    out = torch.ones(L, dtype=torch.bool)
    out[at:at + W] = False
    # the touched tile sums its slots in order, the clean one on the matrix cores: at most a step apart
    assert bool(torch.isfinite(got[0][out.to(DEV)].float()).all())
    d = (got[0].float() - clean[0].float())[out.to(DEV)].abs()
    assert bool((d <= 2.0 ** -6).all())
    assert torch.equal(got[0, :, :96], clean[0, :, :96])


def test_siso_layer_wide_state_runs_it():
    """A whole prefill of a wide bf16 layer: one launch for the entanglement, finite and causal."""
    torch.manual_seed(1)
    m = TESM_SISO(d_model=256, d_state=1024, ent_rank=64, entanglement_window=64, entanglement_threshold=THR,
                  max_seq_len=300).to(DEV).to(torch.bfloat16).eval()
    u = torch.randn(2, 150, 256, generator=torch.Generator().manual_seed(2)).to(torch.bfloat16).to(DEV)
    with torch.no_grad(), hip_ops.launch_log() as log:
        y, _ = m(u)
        y2, _ = m(u[:, :70].contiguous())
    assert any(n.startswith("ent_mfma_kernel<5,4,") for n in log.kernels), log.kernels
    assert not any(n.startswith(("ent_mix_kernel", "ent_scores_kernel")) for n in log.kernels), log.kernels
    assert bool(torch.isfinite(y.float()).all())
    assert torch.equal(y[:, :70], y2)
