"""dK/dV of 16-bit inputs at head dim 128 on grids of up to one workgroup per CU (csrc/chill_tiles.h, dkdv_takes_small_row): the
4-wave and the 8-wave workgroup on either side of the line, with ragged ends, grouped heads and lengths, against the oracle."""
import pytest
import torch

import chill_attention as ca
from chill_attention import _lib
from chill_attention.tiles import tile_config
from conftest import make_mask
from oracle import chill_oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda"

# dtype, mask, B, H, H_kv, T, lens, waves
CASES = [
    (torch.bfloat16, ("CausalChillMask", ()), 1, 24, 8, 2057, None, 4),
    (torch.float16, ("PrefixLMChillMask", (300,)), 3, 17, 17, 513, (513, 64, 401), 4),
    (torch.bfloat16, ("CausalChillMask", ()), 2, 16, 16, 1000, (1000, 129), 8),
    (torch.bfloat16, ("FullChillMask", ()), 1, 9, 9, 2000, None, 8),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[1][0]}-{c[3]}-{c[5]}")
def test_against_the_oracle(case):
    dtype, m, B, H, H_kv, T, lens, waves = case
    mask = make_mask(m)
    cfg = tile_config(mask, 128, dtype, _lib.PASS_DKDV, seq_len=T, batch_heads=B * H_kv)
    assert cfg["waves"] == waves and cfg["rows"] in (64, 128), cfg
    g = torch.Generator(DEV).manual_seed(5)
    q, k, v, d_out = (torch.randn(B, h, T, 128, device=DEV, generator=g).to(dtype) for h in (H, H_kv, H_kv, H))
    lens_t = None if lens is None else torch.tensor(lens, dtype=torch.int32, device=DEV)
    leaves = [x.clone().requires_grad_() for x in (q, k, v)]
    ca.chill_attention(*leaves, mask=mask, lens=lens_t).backward(d_out)
    ref_leaves = [x.float().requires_grad_() for x in (q, k, v)]
    ref, inside = orc.reference_naive(m[0], m[1], *ref_leaves, lens_t)
    ref.backward(d_out.float() * inside)
    # relative 2-norm of rounding P and dS (8 or 11 bits) before the last products, and of rounding O before delta
    bound = 4e-3 if dtype == torch.bfloat16 else 6e-4
    for name, a, b in zip(("dk", "dv"), leaves[1:], ref_leaves[1:]):
        err = ((a.grad.double() - b.grad.double()).norm() / b.grad.double().norm()).item()
        assert err < bound, (name, err)
