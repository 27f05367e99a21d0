"""Dense products with a window of tokens on MFMA (strata_dense_matvec at two to sixteen 16-bit tokens): every type, one
to sixteen K steps over the waves, rows ending within a step, row groups cut short, listed rows, against float64
products of the exact weights."""

import pytest
import torch

from strata_mlx_amd import blocks as B
from strata_mlx_amd import dense as D
from strata_mlx_amd import synth

pytestmark = pytest.mark.gpu

K_TYPES = ["Q3_K", "Q4_K", "Q5_K", "Q6_K", "IQ4_XS", "IQ3_S", "IQ3_XXS"]
SMALL = ["Q2_0", "IQ4_NL", "Q8_0", "Q4_0", "Q5_0"]
# the output rounded once and, in the types whose products exceed float16's 11 bits, the weights
REL = {torch.float16: 2 * 2.0**-11, torch.bfloat16: 2.0**-8 + 2.0**-11}


def layer(gpu, kind, rows, cols, seed):
    g = torch.Generator(device=gpu)
    g.manual_seed(seed)
    data = synth.random_stack(kind, rows * cols, gpu, g)
    return data, B.dequantize(data, kind, (rows, cols)).double(), g


def check(gpu, kind, rows, cols, tokens, dtype, spread=0):
    data, w, g = layer(gpu, kind, rows, cols, rows + cols + tokens)
    x = torch.randn((tokens, cols), device=gpu, generator=g) / (cols**0.5 * float(w.pow(2).mean().sqrt()))
    if spread:
        x *= torch.logspace(-spread, spread, tokens, device=gpu)[:, None]
    x = x.to(dtype)
    y = B.window_matvec(data, kind, rows, cols, x)
    want = x.double() @ w.T
    err = (y.double() - want).norm(dim=1) / want.norm(dim=1)
    assert float(err.max()) <= REL[dtype]
    ids = torch.tensor([rows - 1, 0, rows // 2, rows // 2, rows + 7, 17 % rows], device=gpu, dtype=torch.int32)
    some = B.window_matvec(data, kind, rows, cols, x, row_ids=ids)
    ok = ids < rows
    assert torch.equal(some[:, ok], y[:, ids[ok].long()]) and torch.isnan(some[:, ~ok]).all()


@pytest.mark.parametrize("kind", K_TYPES)
@pytest.mark.parametrize("rows, cols, tokens", [(600, 256, 2), (16, 1536, 5), (1000, 2560, 8), (4100, 4096, 16)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_types_of_256_weight_blocks(gpu, kind, rows, cols, tokens, dtype):
    check(gpu, kind, rows, cols, tokens, dtype)


@pytest.mark.parametrize("kind", SMALL)
@pytest.mark.parametrize("rows, cols, tokens", [(33, 64, 3), (520, 640, 16), (1000, 2240, 5), (4100, 4096, 7)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_types_of_smaller_blocks(gpu, kind, rows, cols, tokens, dtype):
    check(gpu, kind, rows, cols, tokens, dtype)


@pytest.mark.parametrize("kind", ["Q4_K", "Q6_K"])
def test_tokens_far_from_float16s_range(gpu, kind):
    check(gpu, kind, 256, 1024, 16, torch.bfloat16, spread=20)


def test_one_bfloat16_token(gpu):
    check(gpu, "Q6_K", 8192, 4096, 1, torch.bfloat16)


def test_a_layer_of_twelve_tokens_takes_the_window(gpu):
    data, w, g = layer(gpu, "Q6_K", 512, 1024, 9)
    x = (torch.randn((12, 1024), device=gpu, generator=g) / 8).to(torch.bfloat16)
    lin = D.BlockLinear(data, "Q6_K", (512, 1024))
    assert torch.equal(lin(x), B.window_matvec(data, "Q6_K", 512, 1024, x))
