"""Routed products of a few tokens on MFMA (rwin_kernel: gate/up with the SwiGLU and one matrix, strata_expert_*): every
type, one to sixteen K steps, rows ending within a step, row groups cut short, an expert named by more than 16 pairs,
pairs naming none, up to 128 pairs, against float64 products of the exact weights."""

import numpy as np
import pytest
import torch

from strata_mlx_amd import blocks as B
from strata_mlx_amd import synth

pytestmark = pytest.mark.gpu

K_TYPES = ["Q3_K", "Q4_K", "Q5_K", "Q6_K", "IQ4_XS", "IQ3_S", "IQ3_XXS"]
SMALL = ["Q2_0", "IQ4_NL", "Q8_0", "Q4_0", "Q5_0"]
U = 2.0**-8  # bfloat16's rounding


def stack(gpu, kind, experts, rows, cols, g):
    data = synth.random_stack(kind, experts * rows * cols, gpu, g)
    return B.BlockSwitchLinear(data, kind, (experts, rows, cols)), B.dequantize(data, kind, (experts, rows, cols)).double()


def rel(got, want):
    return float(((got.double() - want).norm(dim=-1) / want.norm(dim=-1)).max())


def check(gpu, kind, experts, rows, cols, tokens, k, seed=0, same=False):
    g = torch.Generator(device=gpu)
    g.manual_seed(seed + rows + cols)
    gate, wg = stack(gpu, kind, experts, rows, cols, g)
    up, wu = stack(gpu, kind, experts, rows, cols, g)
    x = (torch.randn((tokens, cols), device=gpu, generator=g) / (cols**0.5 * float(wg.pow(2).mean().sqrt()))).bfloat16()
    rng = np.random.default_rng(seed)
    idx = rng.integers(0, experts, tokens * k)
    if same:
        idx[:] = 1
    if tokens * k > 3:
        idx[2] = experts + 1
    ix = torch.from_numpy(idx).to(gpu)
    ok = ix < experts
    safe = ix.clamp(max=experts - 1)
    xs = x.double().repeat_interleave(k, 0)
    gw, uw = torch.einsum("pc,prc->pr", xs, wg[safe]), torch.einsum("pc,prc->pr", xs, wu[safe])
    gq, uq, h = B.gate_up_swiglu(gate, up, x, ix, k)
    assert rel(gq[ok], gw[ok]) <= U and rel(uq[ok], uw[ok]) <= U
    # the SwiGLU's four roundings (sigmoid, product, product, and g's and u's own)
    hw = gw * torch.sigmoid(gw) * uw
    assert rel(h[ok], hw[ok]) <= 6 * U
    for t in (gq, uq, h):
        assert torch.isnan(t[~ok]).all()
    g2, u2 = B.gate_up(gate, up, x, ix, k)
    assert rel(g2[ok], gw[ok]) <= U and rel(u2[ok], uw[ok]) <= U
    hx = (torch.randn((tokens * k, cols), device=gpu, generator=g) / 64).bfloat16()
    y = B.expert_matvec(gate, ix, hx)
    want = torch.einsum("pc,prc->pr", hx.double(), wg[safe])
    assert rel(y[ok], want[ok]) <= U and torch.isnan(y[~ok]).all()


@pytest.mark.parametrize("kind", K_TYPES)
@pytest.mark.parametrize("rows, cols, tokens, k", [(40, 256, 1, 1), (64, 1536, 8, 10), (100, 2560, 5, 3), (64, 4096, 2, 8)])
def test_types_of_256_weight_blocks(gpu, kind, rows, cols, tokens, k):
    check(gpu, kind, 7, rows, cols, tokens, k)


@pytest.mark.parametrize("kind", SMALL)
@pytest.mark.parametrize("rows, cols, tokens, k", [(40, 64, 3, 2), (64, 640, 8, 10), (100, 2240, 5, 3), (64, 4096, 1, 8)])
def test_types_of_smaller_blocks(gpu, kind, rows, cols, tokens, k):
    check(gpu, kind, 7, rows, cols, tokens, k)


@pytest.mark.parametrize("kind", ["IQ3_S", "Q4_K"])
def test_an_expert_of_many_pairs(gpu, kind):
    check(gpu, kind, 3, 48, 512, 16, 8, same=True)
    check(gpu, kind, 1, 48, 512, 64, 2, seed=1)


def test_a_bfloat16_layer_of_one_token(gpu):
    """switch_glu at one bfloat16 token takes these launches."""
    g = torch.Generator(device=gpu)
    g.manual_seed(5)
    gate, wg = stack(gpu, "IQ3_S", 16, 512, 1024, g)
    up, wu = stack(gpu, "IQ3_S", 16, 512, 1024, g)
    down, wd = stack(gpu, "IQ3_S", 16, 1024, 512, g)
    x = (torch.randn((1, 1024), device=gpu, generator=g) / 64).bfloat16()
    ix = torch.randperm(16, device=gpu, generator=g)[None, :4]
    _, _, h = B.gate_up_swiglu(gate, up, x, ix.reshape(-1), 4)
    y = B.expert_matvec(down, ix.reshape(-1), h)
    assert torch.equal(B.BlockSwitchGLU(gate, up, down)(x, ix).reshape(4, -1), y)
    want = torch.einsum("pc,prc->pr", h.double(), wd[ix[0]])
    assert rel(y, want) <= U
