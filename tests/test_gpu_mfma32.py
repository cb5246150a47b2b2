"""GPU checks of the 32x32x32 products (mfma32.hip) at the edges of their tiles and of the rules that choose them:
one row either side of a tile, columns and K tiles left over, K loops shorter than the pipeline, and K groups whose
last step has tiles for some groups only.  The integer sums are exact, so each output is compared with the product of
the codes in 64 bits, scaled as the kernels scale it (two float32 roundings, one more to the output dtype)."""
import pytest
import torch

from hip_helpers import DEV, need_gpu
from tesm_amd import FeedForward, TESMConfig, hip_ops

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _gpu():
    need_gpu()


def _codes(x):
    """Natural-order codes as float64, scales and sums, beside the product-order buffers the kernels read."""
    q1, s, rs = hip_ops.quant_act(x)
    q0, _, _ = hip_ops.quant_act(x, layout=0)
    return (q1, s, rs), q0[:, :x.shape[1]].double()


def _expect(acc, s, c_w, dtype):
    return ((acc.float() * (1.0 / s)[:, None]) * c_w.float()).to(dtype)


# (M, N, K, kernel): each rule of the dispatch, with M, N or K next to a tile edge
STORE = [(33, 65, 128, "mfma32_kernel<1,4,2,1,"), (129, 96, 384, "mfma32_kernel<1,4,2,1,"),
         (64, 4096, 4096, "mfma32k_kernel<1,2,1,1,4,3,"), (65, 1000, 2049, "mfma32k_kernel<1,2,1,1,4,3,"),
         (97, 70, 640, "mfma32k_kernel<1,2,1,1,2,3,"), (40, 300, 513, "mfma32k_kernel<1,2,1,1,2,3,"),
         (17, 16385, 500, "mfma32k_kernel<1,2,1,1,2,3,"), (17, 40001, 500, "mfma32_kernel<1,4,1,1,"), (513, 2944, 768, "mfma32_kernel<1,4,1,1,"),
         (2049, 2500, 700, "mfma32_kernel<1,4,2,1,"), (1025, 8200, 513, "mfma32_kernel<2,4,2,2,"),
         (1500, 4090, 1100, "mfma32_kernel<2,4,2,2,"), (520, 4090, 1100, "mfma32_kernel<1,4,2,1,"),
         (410, 4090, 1100, "mfma32k_kernel<1,4,1,1,2,3,"), (300, 4090, 1100, "mfma32k_kernel<1,2,1,1,2,3,"),
         (32, 40001, 1100, "mfma32k_kernel<1,2,1,1,2,3,"),
         (1300, 2432, 700, "mfma32_kernel<1,4,2,1,"), (1281, 4090, 4100, "mfma32_kernel<2,4,2,2,"),
         (513, 10900, 1100, "mfma32_kernel<2,4,2,2,"),
         (2100, 8200, 1100, "mfma32_kernel<2,4,2,2,"), (8190, 2401, 520, "mfma32_split_kernel<")]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,kernel", STORE)
def test_store_products_exact(M, N, K, kernel, dtype):
    g = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g).to(dtype).to(DEV)
    w = torch.randn(N, K, generator=g).to(dtype).to(DEV)
    s_w, c_w = hip_ops.absmean_scale(w)
    packed = hip_ops.pack_weight(w, s_w)
    (q, s, rs), qd = _codes(x)
    wd = hip_ops.unpack_weight(packed, K).double()
    want = _expect(qd @ wd.t(), s, c_w, dtype)
    with hip_ops.launch_log() as log:
        out = hip_ops.bitlinear(q, s, rs, packed, c_w, N, K, dtype)
    assert any(k.startswith(kernel) for k in log.kernels), log.kernels
    assert torch.equal(out, want)
    # rows of a wider output (vector stores where they are aligned, single ones where not)
    for pad in (8, 3):
        wide = torch.full((M, N + pad), 7.0, dtype=dtype, device=DEV)
        hip_ops.bitlinear(q, s, rs, packed, c_w, N, K, dtype, out=wide[:, :N])
        assert torch.equal(wide[:, :N], want) and bool((wide[:, N:] == 7.0).all())


# grids of one round: five M tiles are walked as one group (the kernel's last argument), others by fours
@pytest.mark.parametrize("M,N,order", [(512, 13053, 0), (513, 10900, 2), (640, 12800, 2), (641, 9200, 0), (1100, 7000, 0)])
def test_tile_walk_exact(M, N, order):
    K = 1100
    g = torch.Generator().manual_seed(M)
    x, w = (torch.randn(n, K, generator=g).to(torch.bfloat16).to(DEV) for n in (M, N))
    s_w, c_w = hip_ops.absmean_scale(w)
    packed = hip_ops.pack_weight(w, s_w)
    (q, s, rs), qd = _codes(x)
    with hip_ops.launch_log() as log:
        out = hip_ops.bitlinear(q, s, rs, packed, c_w, N, K, torch.bfloat16)
    assert log.kernels == [f"mfma32_kernel<2,4,2,2,0,1,{order}>"], log.kernels
    assert torch.equal(out, _expect(qd @ hip_ops.unpack_weight(packed, K).double().t(), s, c_w, torch.bfloat16))


# K loops of one to three tiles on both sides of the rule's lines: (M, N, K, bf16's kernel, float32's)
SHORT = [(512, 128, 384, "<1,4,2,1,", "<1,4,2,1,"), (513, 128, 384, "<1,4,1,1,", "<1,4,1,1,"),
         (33, 129, 60, "<1,4,1,1,", "<1,4,1,1,"), (4030, 1025, 130, "<1,4,2,1,", "<1,4,1,1,"),
         (3960, 1024, 256, "<1,4,1,1,", "<1,4,1,1,"), (4090, 2040, 300, "<2,4,2,2,", "<1,4,1,1,"),
         (8190, 2048, 384, "<2,4,2,2,", "<2,4,2,2,"), (64, 140000, 100, "<1,4,1,1,", "<1,4,1,1,"),
         (20, 140000, 100, "<1,4,1,1,", "<1,4,1,1,"), (65, 140000, 100, "<2,4,2,2,", "<2,4,2,2,")]
# under one 128x256 tile per CU, K to 2048 and past it: three 64x128 tiles per CU and fewer
SHORT += [(402, 12544, 1100, "<1,4,2,1,", "<1,4,2,1,"), (402, 12442, 2048, "<1,4,2,1,", "<1,4,2,1,"),
          (449, 12288, 1100, "<2,4,2,2,", "<2,4,2,2,"), (402, 12442, 2049, "<2,4,2,2,", "<2,4,2,2,")]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,K,bf16,f32", SHORT)
def test_short_products_exact(M, N, K, bf16, f32, dtype):
    g = torch.Generator().manual_seed(M + N)
    x, w = (torch.randn(n, K, generator=g).to(dtype).to(DEV) for n in (M, N))
    s_w, c_w = hip_ops.absmean_scale(w)
    packed = hip_ops.pack_weight(w, s_w)
    (q, s, rs), qd = _codes(x)
    with hip_ops.launch_log() as log:
        out = hip_ops.bitlinear(q, s, rs, packed, c_w, N, K, dtype)
    assert any(k.startswith("mfma32_kernel" + (bf16 if dtype == torch.bfloat16 else f32)) for k in log.kernels), log.kernels
    assert torch.equal(out, _expect(qd @ hip_ops.unpack_weight(packed, K).double().t(), s, c_w, dtype))


# outputs at each offset from 16 bytes, in rows of odd and even lengths: one per tile shape, K groups, the split kernel
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("M,N,K", [(97, 70, 640), (33, 65, 128), (600, 1001, 60), (1025, 8199, 513), (8190, 2402, 520)])
def test_unaligned_outputs(M, N, K, dtype):
    g = torch.Generator().manual_seed(M + K)
    x, w = (torch.randn(n, K, generator=g).to(dtype).to(DEV) for n in (M, N))
    s_w, c_w = hip_ops.absmean_scale(w)
    packed = hip_ops.pack_weight(w, s_w)
    (q, s, rs), qd = _codes(x)
    want = _expect(qd @ hip_ops.unpack_weight(packed, K).double().t(), s, c_w, dtype)
    for ld in (N + 8 - N % 8 + 8, N + 9 - N % 8 + 8, N + 10 - N % 8 + 8):
        for off in (0, 1, 2, 3, 5):
            wide = torch.full((M + 2, ld), 7.0, dtype=dtype, device=DEV)
            hip_ops.bitlinear(q, s, rs, packed, c_w, N, K, dtype, out=wide[1:M + 1, off:off + N])
            assert torch.equal(wide[1:M + 1, off:off + N], want), (ld, off)
            wide[1:M + 1, off:off + N] = 7.0
            assert bool((wide == 7.0).all()), (ld, off)


@pytest.mark.parametrize("M,N,K", [(65, 200, 2100), (2100, 2050, 1030)])
def test_bias_and_accumulators(M, N, K):
    """The general epilogue behind a K-group tile and a large one: bias and the accumulator dump."""
    g = torch.Generator().manual_seed(M)
    x, w = (torch.randn(n, K, generator=g).to(DEV) for n in (M, N))
    bias = torch.randn(N, generator=g).to(DEV)
    s_w, c_w = hip_ops.absmean_scale(w)
    packed = hip_ops.pack_weight(w, s_w)
    (q, s, rs), qd = _codes(x)
    acc = qd @ hip_ops.unpack_weight(packed, K).double().t()
    out, dump = hip_ops.bitlinear(q, s, rs, packed, c_w, N, K, torch.float32, bias=bias, acc_dump=True)
    assert torch.equal(dump.double(), acc)
    assert torch.equal(out, _expect(acc, s, c_w, torch.float32) + bias)


# (tokens, d_model, d_intermediate): 64 + 64 column tiles, 128 + 128 ones, a K loop of one tile, odd edges
FFN = [(33, 128, 70, "mfma32_kernel<2,2,1,1,2,"), (700, 200, 1111, "mfma32_kernel<2,2,1,1,2,"),
       (4097, 256, 2050, "mfma32_kernel<2,4,2,1,2,"), (500, 2100, 8193, "mfma32_kernel<2,4,2,1,2,")]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,dm,inner,kernel", FFN)
def test_swiglu_products(M, dm, inner, kernel, dtype):
    """SwiGLU's two products of one K loop: h is within the rounding of silu's device exponential of the same
    formula on the two products taken one by one, and down_proj of it follows."""
    torch.manual_seed(M)
    m = FeedForward(TESMConfig(d_model=dm, d_intermediate=inner)).to(DEV).to(dtype).eval()
    x = torch.randn(M, dm, generator=torch.Generator().manual_seed(1)).to(dtype).to(DEV)
    with torch.no_grad():
        with hip_ops.launch_log() as log:
            y = m(x)
        gate, up = m.gate_proj(x), m.up_proj(x)
        h = torch.nn.functional.silu(gate.float()).to(dtype) * up
        want = m.down_proj(h)
    assert any(k.startswith(kernel) for k in log.kernels), log.kernels
    # a silu one ulp off moves an int8 code of h by at most one, next to a rounding boundary only: under 1 % of them
    # in float32, and in bf16 (h itself has 8 bits) up to one code per rounding of silu
    rel = float((y.float() - want.float()).norm() / want.float().norm())
    assert rel <= (2e-3 if dtype == torch.float32 else 1e-2), rel


# (M, N, K): the gate's tile sizes and K groups, with edges and an odd number of steps per product
GATE = [(33, 1100, 4100, "mfma32k_kernel<1,1,1,1,8,3,1,"), (70, 8200, 4100, "mfma32k_kernel<1,2,1,1,4,3,1,"),
        (40, 70, 300, "mfma32_kernel<1,2,1,1,1,"), (1025, 2050, 300, "mfma32_kernel<2,4,1,1,1,"),
        (4100, 4100, 200, "mfma32_kernel<2,4,2,2,1,")]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,kernel", GATE)
def test_output_gate_products(M, N, K, kernel, dtype):
    """y = local + sigmoid(gate) * sp + ep with sp and ep the plain products: only the sigmoid may differ, by an ulp
    of float32 before its rounding, so y moves by at most one rounding of each of its three terms."""
    g = torch.Generator().manual_seed(M + K)
    te, cc = (torch.randn(M, K, generator=g).to(dtype).to(DEV) for _ in range(2))
    ws = [torch.randn(N, K, generator=g).to(dtype).to(DEV) for _ in range(2)]
    sc = [hip_ops.absmean_scale(w) for w in ws]
    pk = [hip_ops.pack_weight(w, s[0]) for w, s in zip(ws, sc)]
    lg = torch.randn(M, 2 * N + 5, generator=g).to(dtype).to(DEV)
    local, gate = lg[:, :N], lg[:, N + 5:]
    qt, qc = hip_ops.quant_act(te), hip_ops.quant_act(cc)
    with hip_ops.launch_log() as log:
        y, _ = hip_ops.output_gate(qt, qc, pk[0], sc[0][1], pk[1], sc[1][1], local, gate, K, quantize=False)
    assert any(k.startswith(kernel) for k in log.kernels), log.kernels
    sp = hip_ops.bitlinear(*qt, pk[0], sc[0][1], N, K, dtype)
    ep = hip_ops.bitlinear(*qc, pk[1], sc[1][1], N, K, dtype)
    gs = torch.sigmoid(gate.float()).to(dtype) * sp
    want = (local + gs) + ep
    eps = torch.finfo(dtype).eps
    bound = eps * (2 * gs.float().abs() + (local.float() + gs.float()).abs() + want.float().abs()) + 1e-6
    assert bool(((y.float() - want.float()).abs() <= bound).all())
    assert float((y != want).float().mean()) <= (0.5 if dtype == torch.float32 else 0.02)


# both sides of the rule's lines: (M, N, K, bf16's kernel, float32's) - rounds of 128x256 tiles nearly full or not, by K;
# float32's 64x128 tiles just past two per CU and beyond; long K with up to three 64x128 tiles per two CUs
GATE_LINES = [(1500, 4080, 2050, "<2,4,2,2,1,", "<1,4,2,1,1,"), (2047, 4000, 2050, "<2,4,2,2,1,", "<2,4,2,2,1,"),
              (2950, 4060, 2050, "<2,4,1,1,1,", "<1,4,2,1,1,"), (3000, 2430, 1280, "<2,4,2,2,1,", "<2,4,2,2,1,"),
              (4095, 2430, 1280, "<2,4,1,1,1,", "<1,4,2,1,1,"), (2048, 4000, 600, "<2,4,1,1,1,", "<2,4,2,2,1,"), (4095, 4000, 600, "<2,4,2,2,1,", "<2,4,2,2,1,"),
              (1500, 4080, 4100, "<2,4,2,2,1,", "<2,4,2,2,1,"), (2900, 2430, 1540, "<2,4,2,2,1,", "<2,4,2,2,1,"),
              (2048, 2430, 600, "<2,4,1,1,1,", "<1,2,1,1,1,"), (8190, 2050, 300, "<2,4,1,1,1,", "<1,4,2,1,1,"),
              (2900, 1024, 4100, "<1,2,1,1,1,", "<1,2,1,1,1,"), (3200, 1024, 4100, "<2,4,1,1,1,", "<2,4,1,1,1,")]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,bf16,f32", GATE_LINES)
def test_output_gate_lines(M, N, K, bf16, f32, dtype):
    test_output_gate_products(M, N, K, f"mfma32_kernel{bf16 if dtype == torch.bfloat16 else f32}", dtype)



# rows of whole 16-byte chunks take the inputs and outputs through LDS, others go one by one: the same results
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(33, 1104, 4100), (70, 8200, 4100), (40, 72, 300), (64, 8, 60), (1025, 2056, 300),
                                   (4100, 4104, 200), (8190, 2056, 300)])
def test_output_gate_aligned(M, N, K, dtype):
    g = torch.Generator().manual_seed(M + K)
    te, cc = (torch.randn(M, K, generator=g).to(dtype).to(DEV) for _ in range(2))
    ws = [torch.randn(N, K, generator=g).to(dtype).to(DEV) for _ in range(2)]
    sc = [hip_ops.absmean_scale(w) for w in ws]
    pk = [hip_ops.pack_weight(w, s[0]) for w, s in zip(ws, sc)]
    qt, qc = hip_ops.quant_act(te), hip_ops.quant_act(cc)
    local, gate = (torch.randn(M, N, generator=g).to(dtype).to(DEV) for _ in range(2))
    ys = []
    for ld, at in ((2 * N + 16, (8, N + 8)), (2 * N + 5, (0, N + 5)), (2 * N + 16, (4, N + 8)), (2 * N + 16, (8, N + 10))):
        lg = torch.full((M, ld), float("nan"), dtype=dtype, device=DEV)
        lg[:, at[0]:at[0] + N] = local
        lg[:, at[1]:at[1] + N] = gate
        y, _ = hip_ops.output_gate(qt, qc, pk[0], sc[0][1], pk[1], sc[1][1], lg[:, at[0]:at[0] + N],
                                   lg[:, at[1]:at[1] + N], K, quantize=False)
        ys.append(y)
    assert not bool(ys[0].isnan().any())
    for y in ys[1:]:
        assert torch.equal(ys[0], y)


# rows of odd lengths: single elements, the last one alone in its pair's place
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,kernel", [(41, 71, 300, "mfma32_kernel<1,2,1,1,1,"), (33, 1, 60, "mfma32_kernel<1,2,1,1,1,"),
                                          (33, 1103, 4100, "mfma32k_kernel<1,1,1,1,8,3,1,"),
                                          (1025, 2051, 300, "mfma32_kernel<2,4,1,1,1,"),
                                          (4099, 4097, 200, "mfma32_kernel<2,4,2,2,1,")])
def test_output_gate_odd_rows(M, N, K, kernel, dtype):
    test_output_gate_products(M, N, K, kernel, dtype)
