"""The fused tile kernels over every block type (strata_tiles_gate_up_swiglu, strata_tiles_down through
switch_glu): experts of one to several chunks of tiles, rows ending within a 256-weight step, a ragged number of
tokens, pairs naming no expert, against float64 products of the exact weights."""

import numpy as np
import pytest
import torch

from strata_mlx_amd import blocks as B
from strata_mlx_amd import synth

pytestmark = pytest.mark.gpu

K_TYPES = ["Q3_K", "Q4_K", "Q5_K", "Q6_K", "IQ4_XS", "IQ3_S", "IQ3_XXS"]
SMALL = ["Q2_0", "IQ4_NL", "Q8_0", "Q4_0", "Q5_0"]
# h and the output are rounded once each and, in the types whose products exceed float16's 11 bits, the weights:
# three roundings of at most 2^-11 (bfloat16: two of 2^-8 and one of 2^-11), the first passed on by down
REL = {torch.float16: 3 * 2.0**-11, torch.bfloat16: 2 * 2.0**-8 + 2.0**-11}


def layer(kind, experts, hidden, inner, gpu, g):
    out = []
    for rows, cols in ((inner, hidden), (inner, hidden), (hidden, inner)):
        data = synth.random_stack(kind, experts * rows * cols, gpu, g)
        w = B.dequantize(data, kind, (experts, rows, cols)).double()
        out.append((B.BlockSwitchLinear(data, kind, (experts, rows, cols)), w))
    return out


def check(gpu, kind, hidden, inner, dtype, tokens=131, k=3, seed=0, missing=True):
    g = torch.Generator(device=gpu)
    g.manual_seed(seed)
    experts = 6
    (gate, wg), (up, wu), (down, wd) = layer(kind, experts, hidden, inner, gpu, g)
    rng = np.random.default_rng(seed)
    # expert 0 most tokens (several chunks of three tiles), expert 4 one tile, expert 5 none
    idx = np.stack([rng.permutation([0, 1 + t % 3, 4 if t < 9 else 1 + (t + 1) % 3])[:k] for t in range(tokens)])
    if missing:
        idx[7, 1] = experts
    x = (torch.randn((tokens, hidden), device=gpu, generator=g) / (hidden**0.5 * float(wg.pow(2).mean().sqrt()))).to(dtype)
    ix = torch.from_numpy(idx).to(gpu)
    old = B.TILES_FROM
    try:
        B.TILES_FROM = 1
        y = B.BlockSwitchGLU(gate, up, down)(x, ix)
    finally:
        B.TILES_FROM = old
    xd = x.double()
    want = torch.full((tokens, k, hidden), float("nan"), dtype=torch.float64, device=gpu)
    for e in range(experts):
        t, s = torch.nonzero(ix == e, as_tuple=True)
        p, q = xd[t] @ wg[e].T, xd[t] @ wu[e].T
        want[t, s] = (p * torch.sigmoid(p) * q) @ wd[e].T
    none = ix >= experts
    assert torch.isnan(y[none]).all()
    got = y.double()[~none]
    assert float((got - want[~none]).norm() / want[~none].norm()) <= REL[dtype]


@pytest.mark.parametrize("kind", K_TYPES)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_types_of_256_weight_blocks(gpu, kind, dtype):
    check(gpu, kind, 512, 768, dtype)


@pytest.mark.parametrize("kind", SMALL)
@pytest.mark.parametrize("inner", [64, 320, 640])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_rows_ending_within_a_step(gpu, kind, inner, dtype):
    check(gpu, kind, 448, inner, dtype, seed=inner)


def test_a_token_far_from_float16s_range(gpu):
    """A type with mins on bfloat16 rows of very different magnitudes: the runs' sums are scaled with the row."""
    g = torch.Generator(device=gpu)
    g.manual_seed(3)
    data = synth.random_stack("Q4_K", 2 * 64 * 512, gpu, g)
    w = B.dequantize(data, "Q4_K", (2, 64, 512)).double()
    h = torch.randn((40, 512), device=gpu, generator=g)
    h *= torch.logspace(-25, 25, 40, device=gpu)[:, None]
    h = h.to(torch.bfloat16)
    down = B.BlockSwitchLinear(data, "Q4_K", (2, 64, 512))
    idx = torch.arange(40, device=gpu, dtype=torch.int64)[:, None] % 2
    tiles, token, where, slot_pair, flat = B._route(idx, 2)
    slots = torch.zeros((token.numel(), 512), dtype=torch.bfloat16, device=gpu)
    slots[where.long()] = h
    h16, h_max, h_sum = B._tile_rows(slots, "Q4_K")
    y = torch.empty((40, 64), dtype=torch.bfloat16, device=gpu)
    lib = B._lib.library()
    B._lib.check(lib.strata_tiles_down(B._lib.kind_id("Q4_K"), data.data_ptr(), 2, 64, 512, h16.data_ptr(),
                                       h_max.data_ptr(), h_sum.data_ptr(), tiles.data_ptr(), tiles.numel(), 16,
                                       slot_pair.data_ptr(), flat.data_ptr(), 40, y.data_ptr(),
                                       B._lib.dtype_id(torch.bfloat16), B._lib.stream()), "down")
    want = torch.stack([w[i % 2] @ h[i].double() for i in range(40)])
    err = (y.double() - want).norm(dim=1) / want.norm(dim=1)
    assert float(err.max()) <= 2.0**-8


@pytest.mark.parametrize("pairs, experts", [(1, 1), (63, 5), (64, 256), (65, 1024), (1023, 7), (1025, 512), (2500, 3),
                                            (4096, 256), (4097, 256), (4000, 1025)])
def test_routes_of_one_workgroup_and_of_three_launches(gpu, pairs, experts):
    """tiles_of's layout with every slot's pair, at the sizes around the one-launch form's limits (4096 pairs, 1024
    experts) and a wave's chunks of 64, some pairs naming no expert."""
    rng = np.random.default_rng(pairs + experts)
    idx = rng.integers(0, experts, (pairs, 1))
    idx[rng.random(pairs) < 0.03] = experts + 3
    tiles, token, where, slot_pair, _ = (t.cpu().numpy() for t in B._route(torch.from_numpy(idx).to(gpu), experts))
    flat, tile = idx[:, 0], B.TOKENS_TILE
    counts = np.bincount(flat[flat < experts], minlength=experts)
    per = (counts + tile - 1) // tile
    first = np.concatenate([[0], np.cumsum(per)])
    assert np.array_equal(tiles, np.concatenate([np.repeat(np.arange(experts), per),
                                                 np.full(len(tiles) - first[-1], experts)]))
    slots = np.full(len(tiles) * tile, -1)
    for e in np.unique(flat[flat < experts]):
        at = np.nonzero(flat == e)[0]
        slots[first[e] * tile:first[e] * tile + len(at)] = at
        assert np.array_equal(where[at], first[e] * tile + np.arange(len(at)))
    assert np.array_equal(slot_pair, slots) and (where[flat >= experts] == -1).all()
    assert np.array_equal(token, np.where(slots >= 0, slots, 0))
