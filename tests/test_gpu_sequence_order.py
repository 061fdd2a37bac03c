"""Launches on both sides of the tile-order rules against the C oracle, byte for byte.

AdamW launches with BF16 parameters take their tiles in sequence from 5 * 2^21
elements on, or from 13 * 2^21 on where their formats have a cap on the
resident workgroups there; momentum SGD with FP16 or FP8 stochastic momentum
from 2^24 on.  One tile fewer, in the chunked order.  The rules count whole
tiles, so the sizes are chosen by tiles for each workgroup size.  The group
spreads them over three tensors, each with a partial last tile and a
remainder; the gradients start off 16-byte alignment.
"""

from __future__ import annotations

import pytest
import torch

from oracle import c_oracle, sr_oracle

pytestmark = pytest.mark.gpu

BF16, F16, E4M3 = torch.bfloat16, torch.float16, torch.float8_e4m3fn


@pytest.mark.parametrize("block_size", (128, 512))
@pytest.mark.parametrize("in_sequence", (False, True))
@pytest.mark.parametrize("moments,edge", [((BF16, BF16), 13 << 21), ((F16, E4M3), 5 << 21), ((E4M3,), 1 << 24)])
def test_both_sides_of_the_order_rule_equal_the_oracle(cuda, moments, edge, in_sequence, block_size):
    import sr_states

    formats = tuple((dtype, "stochastic") for dtype in moments)
    tile = 4 * block_size
    sizes = [1021, 4 * 1024 * 1024 + 1]
    tiles = edge // tile - (not in_sequence) - sum(-(-n // tile) for n in sizes)
    sizes.append((tiles - 1) * tile + 3)
    covered = sum(-(-n // tile) for n in sizes) * tile
    assert (covered >= edge) == in_sequence and edge - tile <= covered <= edge
    total = sum(sizes)
    generator = torch.Generator().manual_seed(total)
    params, grads = [], []
    for n in sizes:
        params.append(torch.randn(n, generator=generator).to(BF16))
        grads.append((torch.randn(n, generator=generator) * 0.1).to(BF16))
    flat = torch.zeros(total + 1, dtype=BF16, device=cuda)
    start, views = 1, []
    for n, g in zip(sizes, grads):
        views.append(flat[start:start + n].copy_(g))
        start += n
    device = [torch.nn.Parameter(p.to(cuda)) for p in params]
    adamw = len(moments) == 2
    names = ("exp_avg", "exp_avg_sq") if adamw else ("momentum_buffer",)
    options = dict(seed=7, block_size=block_size,
                   state_format={name: sr_states.StateFormat(*f) for name, f in zip(names, formats)})
    optimizer = (sr_states.AdamWHip(device, lr=3e-4, weight_decay=0.01, **options) if adamw else
                 sr_states.SGDMHip(device, lr=0.1, momentum=0.9, **options))
    for p, g in zip(device, views):
        p.grad = g
    optimizer.step()
    for index, (p, g, got) in enumerate(zip(params, grads, device)):
        expected = [torch.zeros(p.shape, dtype=dtype) for dtype in moments]
        key = dict(formats=formats, seed=sr_oracle.update_key(7, 1, index))
        if adamw:
            c_oracle.adamw_step_(p, g, *expected, lr=3e-4, beta1=0.9, beta2=0.999, eps=1e-8, weight_decay=0.01,
                                 step=1, **key)
        else:
            c_oracle.sgdm_step_(p, g, *expected, lr=0.1, momentum_factor=0.9, **key)
        state = optimizer.state[got]
        for have, want in ((got.detach(), p), *((state[name], e) for name, e in zip(names, expected))):
            assert torch.equal(have.cpu().view(torch.uint8), want.view(torch.uint8)), (index, total, moments)
