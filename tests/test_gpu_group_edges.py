"""Views that start anywhere and tiles that end anywhere, against the C oracle byte for byte.

A lane moves a group of four elements as one access whatever the group's
alignment, and the last lanes take the elements after the last whole group.
Sizes sit at the edges of a group, a wave and a tile (512 elements for an
update at 128 lanes, 2048 for a cast at 256); the elements around every
view must keep their bytes.
"""

from __future__ import annotations

import pytest
import torch

from oracle import c_oracle

pytestmark = pytest.mark.gpu

SIZES = (1, 2, 3, 4, 5, 7, 253, 255, 257, 508, 509, 511, 512, 513, 515, 1027)
CAST_SIZES = (1, 3, 4, 5, 1023, 1025, 2044, 2047, 2048, 2049, 4095, 4099)
F32, BF16, F16 = torch.float32, torch.bfloat16, torch.float16
E4M3, E5M2 = torch.float8_e4m3fn, torch.float8_e5m2
PAD = 8


def _bytes(t):
    return t.detach().contiguous().cpu().view(torch.uint8)


class _View:
    """``n`` seeded values of ``dtype`` starting ``start`` elements into a device buffer with other elements around."""

    def __init__(self, values, start):
        n = values.numel()
        self.host = torch.cat((torch.ones(start), values.float(), torch.ones(PAD))).to(values.dtype)
        self.device = self.host.cuda()
        self.view, self.expected = self.device[start:start + n], self.host[start:start + n]

    def check(self, what):
        assert torch.equal(_bytes(self.device), _bytes(self.host)), what


def _values(n, dtype, scale, seed):
    return (torch.randn(n, generator=torch.Generator().manual_seed(seed)) * scale).to(dtype)


@pytest.mark.parametrize("block_size", (128, 1024))
@pytest.mark.parametrize(
    "p_dtype,g_dtype,m,v",
    [(F32, F32, (BF16, "stochastic"), (BF16, "stochastic")), (F32, BF16, (F16, "stochastic"), (F32, "nearest")),
     (BF16, BF16, (E4M3, "stochastic"), (E5M2, "nearest"))],
)
def test_updates_at_any_alignment_and_size(cuda, p_dtype, g_dtype, m, v, block_size):
    from sr_states import StateFormat
    from sr_states.hip import hip_adamw_step_, hip_sgdm_step_

    adamw = dict(lr=3e-4, beta1=0.9, beta2=0.999, eps=1e-8, weight_decay=0.01, step=3)
    for k, n in enumerate(SIZES):
        for starts in ((0, 1, 0, 0), (1, 1, 1, 1), (3, 2, 1, 0), (0, 0, 3, 5)):
            p, g = _View(_values(n, p_dtype, 1.0, k), starts[0]), _View(_values(n, g_dtype, 0.1, k + 50), starts[1])
            a = _View(_values(n, m[0], 0.1, k + 100), starts[2])
            b = _View(_values(n, v[0], 0.1, k + 150).float().abs().to(v[0]), starts[3])
            options = dict(seed=77 + k, offset=2**32 - 5, formats=(m, v))
            c_oracle.adamw_step_(p.expected, g.expected, a.expected, b.expected, **adamw, **options)
            options["formats"] = tuple(StateFormat(*f) for f in (m, v))
            hip_adamw_step_(p.view, g.view, a.view, b.view, **adamw, **options, block_size=block_size)
            for view, name in ((p, "parameter"), (g, "gradient"), (a, "first moment"), (b, "second moment")):
                view.check(f"AdamW {name}, n={n}, starts={starts}")
            # A second update of the same views by momentum SGD.
            c_oracle.sgdm_step_(p.expected, g.expected, a.expected, lr=0.1, momentum_factor=0.9, seed=5, offset=9,
                                formats=(m,))
            hip_sgdm_step_(p.view, g.view, a.view, lr=0.1, momentum_factor=0.9, seed=5, offset=9,
                           formats=(StateFormat(*m),), block_size=block_size)
            for view, name in ((p, "parameter"), (g, "gradient"), (a, "momentum")):
                view.check(f"SGDM {name}, n={n}, starts={starts}")


@pytest.mark.parametrize("dtype,rounding", [(BF16, "stochastic"), (F16, "nearest"), (E4M3, "stochastic"), (F32, "nearest")])
def test_casts_at_any_alignment_and_size(cuda, dtype, rounding):
    from sr_states.hip.cast import native_cast
    from sr_states.rounding import native_codes

    rule = native_codes(dtype, rounding)[1]
    for k, n in enumerate(CAST_SIZES):
        for x_start, y_start in ((0, 1), (1, 0), (3, 2)):
            x, y = _View(_values(n, F32, 3.0, k), x_start), _View(_values(n, dtype, 1.0, k + 9), y_start)
            y.expected.copy_(c_oracle.cast(x.expected, dtype=dtype, rounding=rounding, seed=3, offset=2**32 - 100))
            native_cast(x.view, dtype=dtype, rule=rule, seed=3, offset=2**32 - 100, out=y.view)
            x.check(f"input, n={n}")
            y.check(f"output, n={n}, starts={(x_start, y_start)}")
