"""Which route a LoRA layer's library-path step takes and what each route accepts, on the
CPU: the GPU operators are replaced by plain torch stand-ins with the same shapes (and the
same lack of a graph), so the autograd function's own decisions are what runs."""

import importlib

import pytest
import torch

nf4 = importlib.import_module("stratum_amd.nf4_linear")


@pytest.fixture
def operators(monkeypatch):
    """Stand-ins for the GPU operators; the list holds the names of those that ran."""
    ran = []

    def put(name, fn):
        def call(*args, **kwargs):
            ran.append(name)
            with torch.no_grad():
                return fn(*args, **kwargs)
        monkeypatch.setattr(nf4, name, call)

    def pad(t, cols):
        return torch.nn.functional.pad(t, (0, cols - t.shape[1]))

    def down_aug(x, a, scaling=1.0):
        t = scaling * x @ a.t()
        return t, torch.cat([x, pad(t, 64)], 1)

    def up(t, lora, bias=None, transposed=False):
        assert bias is None or tuple(bias.shape) == (lora.shape[1 if transposed else 0],)  # as the operator
        y = t @ lora if transposed else t @ lora.t()
        return y if bias is None else y + bias

    put("lora_up", up)
    put("lora_down", lambda x, a, scaling=1.0: scaling * x.reshape(-1, x.shape[-1]) @ a.t())
    put("lora_down_aug", down_aug)
    put("dequantize_4bit", lambda packed, **kw: packed.weight.to(kw["dtype"]))
    put("dequantize_4bit_aug", lambda packed, absmax, shape, bs, b, dtype: torch.cat([packed.weight.to(dtype), pad(b, 64)], 1))
    put("lora_dy", lambda dy, b, t, scaling=1.0: (scaling * dy @ b, dy.t() @ t if t is not None else None))
    put("lora_da", lambda u, x: u.t() @ x)
    return ran


class _Packed(torch.Tensor):
    """A packed weight that carries its dense values for the stand-ins."""
    weight: torch.Tensor


def layer(N, K, rank_a=16, rank_b=16, rows=70, seed=0, dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(seed)
    packed = torch.zeros(N * K // 2, 1, dtype=torch.uint8).as_subclass(_Packed)
    packed.weight = torch.randn(N, K, generator=g) * 0.1
    x, a, b, dy = (torch.randn(*s, generator=g).to(dtype) * f
                   for s, f in (((rows, K), 1), ((rank_a, K), 0.1), ((N, rank_b), 0.1), ((rows, N), 1)))
    return packed, torch.ones(N * K // 64), x, a, b, dy


def apply(packed, absmax, x, a, b, bias=None, scaling=2.0):
    shape = (packed.weight.shape[0], packed.weight.shape[1])
    return nf4._NF4LinearFn.apply(x, packed, absmax, shape, 64, bias, a, b, scaling, False)


def reference(packed, x, a, b, bias=None, scaling=2.0):
    w = packed.weight.to(x.dtype).float()
    y = x.float() @ w.t() + scaling * (x.float() @ a.float().t()) @ b.float().t()
    return y + bias.float() if bias is not None else y


def close(got, want):
    return float((got.float() - want).norm() / want.norm()) < 1e-2  # bf16 inputs and intermediates


@pytest.mark.parametrize("rank_a,rank_b", [(16, 32), (32, 16), (16, 8), (32, 64)])
def test_adapters_of_different_ranks_are_refused(operators, rank_a, rank_b):
    """N = 2 K, where one product over [x | t] and [W | B] would take any two ranks."""
    packed, absmax, x, a, b, _ = layer(256, 128, rank_a, rank_b)
    with pytest.raises((ValueError, RuntimeError)):
        apply(packed, absmax, x, a, b)


@pytest.mark.parametrize("rank", [16, 32])
def test_adapters_of_one_rank_take_the_augmented_product(operators, rank):
    packed, absmax, x, a, b, _ = layer(256, 128, rank, rank)
    y = apply(packed, absmax, x, a, b)
    assert "lora_down_aug" in operators and "dequantize_4bit_aug" in operators
    assert close(y, reference(packed, x, a, b))


@pytest.mark.parametrize("N,K", [(256, 128), (128, 128)])
@pytest.mark.parametrize("shape", [(1,), (), (1, "N"), ("rows", "N"), ("N",)])
def test_a_bias_that_broadcasts_is_added(operators, N, K, shape):
    """With the augmented product (N = 2 K) and with the rank-R term apart: a bias is whatever
    torch adds to [rows, N]."""
    packed, absmax, x, a, b, _ = layer(N, K)
    bias = torch.randn([{"N": N, "rows": x.shape[0]}.get(s, s) for s in shape]).bfloat16()
    assert close(apply(packed, absmax, x, a, b, bias), reference(packed, x, a, b, bias))


@pytest.mark.parametrize("N,K", [(256, 128), (128, 128)])
def test_input_gradient_stays_differentiable_in_lora_a(operators, N, K):
    """A gradient penalty: with create_graph, dX = dY W + U A keeps its graph to A."""
    packed, absmax, x, a, b, dy = layer(N, K)
    x.requires_grad_(True), a.requires_grad_(True)
    dx, = torch.autograd.grad(apply(packed, absmax, x, a, b), x, dy, create_graph=True)
    da, = torch.autograd.grad(dx, a, torch.ones_like(dx))
    u = 2.0 * dy.float() @ b.float()
    assert close(da, u.t() @ torch.ones(x.shape))
    del operators[:]
    torch.autograd.grad(apply(packed, absmax, x, a, b), (x, a), dy)
    assert "lora_up" in operators  # a plain backward runs the kernel
