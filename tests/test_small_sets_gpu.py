"""Small launches of 16-bit inputs whose workgroups give a tile two sets of waves (csrc/chill_tiles.h, small_takes_two_sets): sizes
on either side of the lines, ragged ends, grouped heads and lengths, against the oracle."""
import pytest
import torch

import chill_attention as ca
from chill_attention import _lib
from chill_attention.tiles import tile_config
from conftest import make_mask
from oracle import chill_oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda"

# id, dtype, mask, B, H, H_kv, T, D, lens, passes that take two sets
CASES = [
    ("either-side", torch.bfloat16, ("CausalChillMask", ()), 1, 4, 2, 257, 64, None, "fk"),
    ("below", torch.bfloat16, ("FullChillMask", ()), 1, 4, 4, 128, 64, None, ""),
    ("all-gqa-lens", torch.float16, ("CausalChillMask", ()), 2, 4, 1, 801, 64, (801, 33), "fqk"),
    ("all-32", torch.bfloat16, ("PrefixLMChillMask", (100,)), 1, 5, 5, 1025, 32, None, "fqk"),
    ("most-tiles-16", torch.float16, ("FullChillMask", ()), 1, 8, 8, 1024, 16, None, "fqk"),
    ("wide-rows", torch.bfloat16, ("CausalChillMask", ()), 1, 3, 1, 1090, 128, (1001,), "fq"),
    ("band", torch.float16, ("SlidingWindowChillMask", (200, 60)), 1, 4, 4, 1500, 64, None, "fk"),
    ("narrow-band", torch.bfloat16, ("ChunkwiseChillMask", (50, 1)), 1, 4, 4, 1500, 64, None, ""),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: c[0])
def test_against_the_oracle(case):
    _, dtype, m, B, H, H_kv, T, D, lens, sets = case
    mask = make_mask(m)
    for p, name, heads in ((_lib.PASS_FWD, "f", H), (_lib.PASS_DQ, "q", H), (_lib.PASS_DKDV, "k", H_kv)):
        cfg = tile_config(mask, D, dtype, p, seq_len=T, batch_heads=B * heads)
        if cfg["rows"] == 32:
            one = tile_config(mask, D, dtype, p, seq_len=32, batch_heads=1)["lds_bytes"]
            assert (cfg["lds_bytes"] == 2 * one) == (name in sets), (name, cfg)
        else:
            assert name not in sets
    g = torch.Generator(DEV).manual_seed(3)
    q, k, v, d_out = (torch.randn(B, h, T, D, device=DEV, generator=g).to(dtype) for h in (H, H_kv, H_kv, H))
    lens_t = None if lens is None else torch.tensor(lens, dtype=torch.int32, device=DEV)
    leaves = [x.clone().requires_grad_() for x in (q, k, v)]
    out = ca.chill_attention(*leaves, mask=mask, lens=lens_t)
    out.backward(d_out)
    ref_leaves = [x.float().requires_grad_() for x in (q, k, v)]
    ref, inside = orc.reference_naive(m[0], m[1], *ref_leaves, lens_t)
    ref.backward(d_out.float() * inside)
    # relative 2-norm of rounding P and dS (8 or 11 bits) before the last products: 2.6e-3 and 3.3e-4 at these sizes
    bound = 4e-3 if dtype == torch.bfloat16 else 6e-4
    for name, a, b in (("out", out.detach() * inside, ref.detach()), *((n, x.grad, y.grad) for n, x, y in zip(("dq", "dk", "dv"), leaves, ref_leaves))):
        err = ((a.double() - b.double()).norm() / b.double().norm()).item()
        assert err < bound, (name, err)
