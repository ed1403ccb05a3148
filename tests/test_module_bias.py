"""TrellisLinear's bias under function transforms (host side, the packed product replaced by fixed
values): vmap, forward-mode and reverse-mode differentiation over the bias give what y + bias,
rounded to the activations' dtype, gives."""
import importlib

import pytest
import torch

from conftest import PKG

Y = torch.linspace(-3, 3, 10).reshape(2, 5)


class _Product:
    k_in, n_out, K, V, codebook = 16, 5, 3, 1, "mcg"
    device = torch.device("cpu")

    def forward(self, x, out_dtype, mma_f16):
        return Y.to(out_dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_bias_under_transforms(dtype):
    layer = importlib.import_module(PKG + ".modules").TrellisLinear(_Product(), bias=torch.zeros(5))
    x = torch.zeros((2, 16), dtype=dtype)
    acc = torch.float16 if dtype == torch.float16 else torch.float32

    def f(b):
        return torch.func.functional_call(layer, {"bias": b}, (x,))

    def want(b):
        return (Y.to(acc) + b.to(acc)).to(dtype)

    biases = torch.linspace(-1, 1, 15).reshape(3, 5)
    assert torch.equal(f(biases[0]), want(biases[0])) and f(biases[0]).dtype == dtype
    assert torch.equal(torch.func.vmap(f)(biases), torch.stack([want(b) for b in biases]))
    y, t = torch.func.jvp(f, (biases[0],), (biases[1],))
    assert torch.equal(y, want(biases[0]))
    assert torch.equal(t, biases[1].to(dtype).expand(2, 5))
    g = torch.func.grad(lambda b: f(b).float().sum())(biases[0])
    assert torch.equal(g, torch.full((5,), 2.0))
    b = biases[2].clone().requires_grad_()
    f(b).float().sum().backward()
    assert torch.equal(b.grad, torch.full((5,), 2.0))
