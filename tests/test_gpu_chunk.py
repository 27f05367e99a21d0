"""Chunks of more than sixteen 16-bit tokens multiplied straight from the blocks (strata_dense_chunk): every type, one to
sixteen and more K steps over the waves, rows ending within a step, two to four tiles a workgroup and a last one cut
short, row groups cut short, against float64 products of the exact weights."""

import pytest
import torch

from strata_mlx_amd import blocks as B
from strata_mlx_amd import dense as D
from strata_mlx_amd import synth

pytestmark = pytest.mark.gpu

K_TYPES = ["Q3_K", "Q4_K", "Q5_K", "Q6_K", "IQ4_XS", "IQ3_S", "IQ3_XXS"]
SMALL = ["Q2_0", "IQ4_NL", "Q8_0", "Q4_0", "Q5_0"]
# the weights and the output rounded once each (a folded Q6_K weight is the file's integers' product rounded)
REL = {torch.float16: 2 * 2.0**-11, torch.bfloat16: 2.0**-8 + 2.0**-11}


def check(gpu, kind, rows, cols, tokens, dtype, spread=0):
    g = torch.Generator(device=gpu)
    g.manual_seed(rows + cols + tokens)
    data = synth.random_stack(kind, rows * cols, gpu, g)
    w = B.dequantize(data, kind, (rows, cols)).double()
    x = torch.randn((tokens, cols), device=gpu, generator=g) / (cols**0.5 * float(w.pow(2).mean().sqrt()))
    if spread:
        x *= torch.logspace(-spread, spread, tokens, device=gpu)[:, None]
    x = x.to(dtype)
    y = B.chunk_matmul(data, kind, rows, cols, x)
    want = x.double() @ w.T
    err = (y.double() - want).norm(dim=1) / want.norm(dim=1)
    assert y.shape == (tokens, rows) and float(err.max()) <= REL[dtype]
    return data, x, y


@pytest.mark.parametrize("kind", K_TYPES)
@pytest.mark.parametrize("rows, cols, tokens", [(100, 256, 17), (32, 2304, 33), (1000, 1536, 77), (96, 4608, 130)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_types_of_256_weight_blocks(gpu, kind, rows, cols, tokens, dtype):
    check(gpu, kind, rows, cols, tokens, dtype)


@pytest.mark.parametrize("kind", SMALL)
@pytest.mark.parametrize("rows, cols, tokens", [(33, 64, 1), (40, 640, 48), (1000, 2240, 77), (96, 4096, 64)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_types_of_smaller_blocks(gpu, kind, rows, cols, tokens, dtype):
    check(gpu, kind, rows, cols, tokens, dtype)


@pytest.mark.parametrize("kind", ["Q4_K", "Q6_K"])
def test_tokens_far_from_float16s_range(gpu, kind):
    check(gpu, kind, 256, 1024, 40, torch.bfloat16, spread=20)


def test_a_layers_chunk_takes_it(gpu):
    data, x, y = check(gpu, "Q4_K", 512, 1024, 50, torch.bfloat16)
    assert torch.equal(D.BlockLinear(data, "Q4_K", (512, 1024))(x), y)
    tall = torch.zeros((50 * 1024 + 1,), dtype=torch.bfloat16, device=gpu)[1:].reshape(50, 1024)  # 2 bytes past 16
    tall.copy_(x)
    assert torch.equal(D.BlockLinear(data, "Q4_K", (512, 1024))(tall), y)
