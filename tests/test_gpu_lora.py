"""LoRA side products (T = s X A^T, U = s dY B, dB = dY^T T, dA = U^T X) against
fp32 torch on the same inputs: relative error within the GEMM tolerance (1e-2
bf16, 5e-3 fp16), identical bits on a repeated call (fixed-order reduction),
ragged row and column counts, every supported rank, and empty problems."""

import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: 1e-2, torch.float16: 5e-3}
SHAPES = [
    (1, 8, 8),         # one row, one chunk of columns, rank 8 (padded to 16)
    (64, 256, 16),     # one step, one column block
    (65, 264, 16),     # one row past a step, 8 columns past a block
    (300, 520, 24),    # rank 24 (padded to 32), two column blocks + 8
    (130, 4104, 32),   # rank 32, 17 column blocks
    (2000, 4096, 16),  # several row blocks
    (513, 1000, 8),    # ragged in both directions
    (16, 4104, 32),    # decode size: lora_down's one-launch kernel, 8 columns past a 2048 sweep
    (40, 14336, 24),   # decode size, rank 24, long rows
]


def seeded(shape, seed, std, dtype, dev):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * std).to(dtype).to(dev)


def rel(a, b):
    a, b = a.float(), b.float()
    return ((a - b).norm() / b.norm().clamp_min(1e-30)).item()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,R", SHAPES)
def test_lora_down(cuda, dtype, M, K, R):
    from stratum_amd.functional import lora_down
    x = seeded((M, K), 1, 1.0, dtype, cuda)
    a = seeded((R, K), 2, 0.05, dtype, cuda)
    t = lora_down(x, a, 2.0)
    assert t.shape == (M, R) and t.dtype == dtype
    ref = 2.0 * (x.float() @ a.float().t().contiguous())
    assert rel(t, ref) <= TOL[dtype]
    assert torch.equal(t, lora_down(x, a, 2.0))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,N,R", SHAPES)
def test_lora_dy(cuda, dtype, M, N, R):
    from stratum_amd.functional import lora_dy
    dy = seeded((M, N), 3, 1.0, dtype, cuda)
    b = seeded((N, R), 4, 0.05, dtype, cuda)
    t = seeded((M, R), 5, 1.0, dtype, cuda)
    u, db = lora_dy(dy, b, t, 0.5)
    assert u.shape == (M, R) and db.shape == (N, R)
    assert rel(u, 0.5 * (dy.float() @ b.float())) <= TOL[dtype]
    assert rel(db, dy.float().t().contiguous() @ t.float()) <= TOL[dtype]
    u2, db2 = lora_dy(dy, b, t, 0.5)
    assert torch.equal(u, u2) and torch.equal(db, db2)
    # without T only U is computed, with the same bits
    u3, none = lora_dy(dy, b, None, 0.5)
    assert none is None and torch.equal(u, u3)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,R", SHAPES)
def test_lora_da(cuda, dtype, M, K, R):
    from stratum_amd.functional import lora_da
    u = seeded((M, R), 6, 1.0, dtype, cuda)
    x = seeded((M, K), 7, 1.0, dtype, cuda)
    da = lora_da(u, x)
    assert da.shape == (R, K)
    assert rel(da, u.float().t().contiguous() @ x.float()) <= TOL[dtype]
    assert torch.equal(da, lora_da(u, x))


def test_lora_at_the_lora_step_shape(cuda):
    """X [8192, 4096], dY [8192, 14336], rank 16: the products of one LoRA step."""
    from stratum_amd.functional import lora_da, lora_down, lora_dy
    dt = torch.bfloat16
    M, N, K, R = 8192, 14336, 4096, 16
    x = seeded((M, K), 8, 1.0, dt, cuda)
    dy = seeded((M, N), 9, 1.0, dt, cuda)
    a = seeded((R, K), 10, 0.01, dt, cuda)
    b = seeded((N, R), 11, 0.01, dt, cuda)
    t = lora_down(x, a, 1.0)
    assert rel(t, x.float() @ a.float().t().contiguous()) <= 1e-2
    u, db = lora_dy(dy, b, t, 1.0)
    assert rel(u, dy.float() @ b.float()) <= 1e-2
    assert rel(db, dy.float().t().contiguous() @ t.float()) <= 1e-2
    da = lora_da(u, x)
    assert rel(da, u.float().t().contiguous() @ x.float()) <= 1e-2


def test_lora_empty_problems(cuda):
    from stratum_amd.functional import lora_da, lora_down, lora_dy
    dt = torch.bfloat16
    x0 = torch.empty((0, 256), dtype=dt, device=cuda)
    a = seeded((16, 256), 12, 0.05, dt, cuda)
    assert lora_down(x0, a).shape == (0, 16)
    # no reduction (K = 0): zeros
    t = lora_down(torch.empty((5, 0), dtype=dt, device=cuda), torch.empty((16, 0), dtype=dt, device=cuda))
    assert t.shape == (5, 16) and not t.any()
    # no rows: U is empty, dB and dA are zero
    u, db = lora_dy(torch.empty((0, 64), dtype=dt, device=cuda), seeded((64, 16), 13, 0.05, dt, cuda),
                    torch.empty((0, 16), dtype=dt, device=cuda))
    assert u.shape == (0, 16) and db.shape == (64, 16) and not db.any()
    da = lora_da(torch.empty((0, 16), dtype=dt, device=cuda), x0)
    assert da.shape == (16, 256) and not da.any()


def test_lora_entry_points_replay_correctly_in_a_hip_graph(cuda):
    """T, U + dB and dA captured into one HIP graph: every replay, with eager
    LoRA work on other inputs and synchronisations between replays, matches the
    eager results bit for bit (the partial buffers are fully overwritten; no
    memset is recorded)."""
    from stratum_amd.functional import lora_da, lora_down, lora_dy
    dt = torch.bfloat16
    M, N, K, R = 300, 520, 264, 16
    x = seeded((M, K), 20, 1.0, dt, cuda)
    dy = seeded((M, N), 21, 1.0, dt, cuda)
    a = seeded((R, K), 22, 0.05, dt, cuda)
    b = seeded((N, R), 23, 0.05, dt, cuda)
    t_e = lora_down(x, a, 2.0)
    u_e, db_e = lora_dy(dy, b, t_e, 2.0)
    da_e = lora_da(u_e, x)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        lora_down(x, a, 2.0)  # warm-up on the capture stream
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        t_g = lora_down(x, a, 2.0)
        u_g, db_g = lora_dy(dy, b, t_g, 2.0)
        da_g = lora_da(u_g, x)
    for i in range(3):
        junk = lora_dy(dy.flip(0), b, t_e, 0.5)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(t_g, t_e), i
        assert torch.equal(u_g, u_e) and torch.equal(db_g, db_e), i
        assert torch.equal(da_g, da_e), i
        del junk


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,C,R", SHAPES + [(17, 64, 32), (33, 72, 16), (8192, 256, 16)])
def test_lora_up(cuda, dtype, M, C, R):
    """t @ lora^T (+ bias) in both layouts of lora: one rounding of an fp32 sum of at most 33
    products, so each value is within one unit in the last place of the result (2^-8 / 2^-11
    of it) plus the sum's own error, 34 * 2^-24 of the sum of magnitudes."""
    from stratum_amd.functional import lora_up
    t = seeded((M, R), 8, 1.0, dtype, cuda)
    b = seeded((C, R), 9, 0.05, dtype, cuda)
    bias = seeded((C,), 10, 0.1, dtype, cuda)
    for with_bias in (None, bias):
        exact = t.double() @ b.double().t().contiguous()
        scale = t.double().abs() @ b.double().abs().t().contiguous()
        if with_bias is not None:
            exact, scale = exact + bias.double(), scale + bias.double().abs()
        unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
        tiny = 0.0 if dtype == torch.bfloat16 else 2.0 ** -25  # half the spacing of fp16's subnormals
        limit = unit * exact.abs() + 34 * 2.0 ** -24 * scale + tiny
        for lora, transposed in ((b, False), (b.t().contiguous(), True)):
            y = lora_up(t, lora, with_bias, transposed=transposed)
            assert y.shape == (M, C) and y.dtype == dtype
            assert bool(((y.double() - exact).abs() <= limit).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,K,R", [(1, 64, 8), (65, 320, 24), (700, 1024, 16), (130, 4096, 32), (2000, 576, 16)])
def test_lora_down_aug(cuda, dtype, M, K, R):
    """The augmented left operand: x, lora_down's t and zeros, bit for bit."""
    from stratum_amd.functional import lora_down, lora_down_aug
    x = seeded((M, K), 11, 1.0, dtype, cuda)
    a = seeded((R, K), 12, 0.05, dtype, cuda)
    t, xa = lora_down_aug(x, a, 2.0)
    assert torch.equal(xa[:, :K], x) and torch.equal(xa[:, K:K + R], t) and not xa[:, K + R:].any()
    if M > 64:  # up to 64 rows lora_down sums in another order
        assert torch.equal(t, lora_down(x, a, 2.0))
    else:
        assert rel(t, 2.0 * (x.float() @ a.float().t().contiguous())) <= TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N,K,R,bs", [(1, 64, 8, 64), (33, 320, 24, 128), (3072, 1024, 16, 64), (9000, 4032, 32, 64)])
def test_dequantize_aug(cuda, dtype, N, K, R, bs):
    """The augmented right operand: dequantize_4bit's weight, lora_b and zeros, bit for bit."""
    from stratum_amd.functional import dequantize_4bit, dequantize_4bit_aug, quantize_4bit
    q, st = quantize_4bit(seeded((N, K), 13, 0.02, torch.float16, cuda), blocksize=bs)
    b = seeded((N, R), 14, 0.05, dtype, cuda)
    wa = dequantize_4bit_aug(q, st.absmax, (N, K), bs, b, dtype)
    assert torch.equal(wa[:, :K], dequantize_4bit(q, st, dtype=dtype))
    assert torch.equal(wa[:, K:K + R], b) and not wa[:, K + R:].any()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("keep", [True, False])
@pytest.mark.parametrize("N,K,rows,bias", [(768, 384, (3, 41), True), (704, 320, (1100,), False), (640, 384, (130,), True)])
def test_library_path_step_with_and_without_augmentation(cuda, dtype, keep, N, K, rows, bias, monkeypatch):
    """A LoRA step on the library path at N = 2 K (one product over K + 64 columns), above it
    and below it (the base product added to the rank-R term), 2-D and 3-D, against fp32."""
    from stratum_amd.functional import dequantize_4bit, quantize_4bit
    from stratum_amd.nf4_linear import NF4LoRALinear
    monkeypatch.setenv("STRATUM_NF4_FUSED_MAX_ROWS", "0")
    q, st = quantize_4bit(seeded((N, K), 15, 0.02, torch.float16, cuda))
    bv = seeded((N,), 16, 0.1, dtype, cuda) if bias else None
    lin = NF4LoRALinear(q, st, bv, r=16, lora_alpha=32.0, dtype=dtype)
    lin.keep_weight_for_backward = keep
    with torch.no_grad():
        lin.lora_A.copy_(seeded((16, K), 17, 0.05, dtype, cuda))
        lin.lora_B.copy_(seeded((N, 16), 18, 0.05, dtype, cuda))
    x = seeded((*rows, K), 19, 1.0, dtype, cuda).requires_grad_(True)
    dy = seeded((*rows, N), 20, 1.0, dtype, cuda)
    y = lin(x)
    y.backward(dy)
    w = dequantize_4bit(q, st, dtype=dtype).float()
    xf = x.detach().float().reshape(-1, K).requires_grad_(True)
    a, b = (p.detach().float().requires_grad_(True) for p in (lin.lora_A, lin.lora_B))
    ref = xf @ w.t() + 2.0 * (xf @ a.t()) @ b.t() + (bv.float() if bias else 0.0)
    ref.backward(dy.float().reshape(-1, N))
    for got, want in ((y, ref), (x.grad, xf.grad), (lin.lora_A.grad, a.grad), (lin.lora_B.grad, b.grad)):
        assert rel(got.detach().reshape(want.shape), want.detach()) <= TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("N,K,M,R", [(768, 384, 123, 32), (640, 320, 1100, 32), (704, 320, 65, 16), (2048, 1024, 1500, 16)])
def test_augmented_forward_is_one_rounding_of_one_sum(cuda, dtype, N, K, M, R, monkeypatch):
    """Y of the product over [x | t] and [W | B]: an fp32 sum of K + R products, rounded once. Each
    value is within one unit in the last place of the exact one plus 2^-23 (K + 64) of the sum of
    magnitudes (an addition is off by at most 2^-23 of it, whatever the order and the rounding)."""
    import importlib
    from stratum_amd.functional import dequantize_4bit, lora_down, quantize_4bit
    from stratum_amd.nf4_linear import NF4LoRALinear
    module, taken = importlib.import_module("stratum_amd.nf4_linear"), []
    real = module._augment
    monkeypatch.setattr(module, "_augment", lambda *args: taken.append(real(*args)) or taken[-1])
    monkeypatch.setenv("STRATUM_NF4_FUSED_MAX_ROWS", "0")
    q, st = quantize_4bit(seeded((N, K), 21, 0.02, torch.float16, cuda))
    lin = NF4LoRALinear(q, st, r=R, lora_alpha=float(R), dtype=dtype)
    with torch.no_grad():
        lin.lora_A.copy_(seeded((R, K), 22, 0.05, dtype, cuda))
        lin.lora_B.copy_(seeded((N, R), 23, 0.05, dtype, cuda))
        x = seeded((M, K), 24, 1.0, dtype, cuda)
        y = lin(x)
        assert torch.equal(y, lin(x)) and taken == [True, True]
        t = lora_down(x, lin.lora_A).double()
        w, b = (v.double().t().contiguous() for v in (dequantize_4bit(q, st, dtype=dtype), lin.lora_B))
        exact, scale = x.double() @ w + t @ b, x.double().abs() @ w.abs() + t.abs() @ b.abs()
    unit = 2.0 ** (-8 if dtype == torch.bfloat16 else -11)
    tiny = 0.0 if dtype == torch.bfloat16 else 2.0 ** -25  # half the spacing of fp16's subnormals
    assert bool(((y.double() - exact).abs() <= unit * exact.abs() + (K + 64) * 2.0 ** -23 * scale + tiny).all())
