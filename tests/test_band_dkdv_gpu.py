"""dK/dV of 16-bit inputs at head dim 128 under narrow bands and under masks whose rows grow (csrc/chill_tiles.h,
dkdv_takes_one_stage): 64-row workgroups with a ring of one stage, two to a CU, at ragged lengths, with grouped heads and padding,
either side of the widths, chunk sizes and grids that change the route, against the oracle."""
import pytest
import torch

import chill_attention as ca
from chill_attention import _lib
from chill_attention.tiles import tile_config
from conftest import make_mask
from oracle import chill_oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda"

# dtype, mask, B, H, H_kv, T, lens, rows and waves of the report (128, 8: two workgroups of the route, or one of the next kernel)
CASES = [
    (torch.float16, ("SlidingWindowChillMask", (16, 16)), 1, 12, 12, 1441, None, (128, 8)),
    (torch.bfloat16, ("SlidingWindowChillMask", (0, 0)), 2, 16, 8, 1100, None, (128, 8)),
    (torch.bfloat16, ("SlidingWindowChillMask", (100, 37)), 3, 8, 8, 1089, (1089, 0, 65), (128, 8)),
    (torch.float16, ("SlidingWindowChillMask", (2000, 47)), 1, 12, 6, 3001, None, (128, 8)),
    (torch.float16, ("SlidingWindowChillMask", (2000, 48)), 1, 10, 10, 2100, None, (128, 8)),
    (torch.bfloat16, ("ChunkwiseChillMask", (100, 3)), 2, 12, 12, 897, (800, 897), (128, 8)),
    (torch.float16, ("ChunkwiseChillMask", (16, 8)), 1, 24, 12, 1537, None, (128, 8)),
    (torch.bfloat16, ("ChunkwiseChillMask", (64, 2)), 1, 33, 33, 4097, None, (128, 8)),
    (torch.float16, ("ChunkwiseChillMask", (64, 2)), 1, 32, 32, 4096, None, (256, 4)),
    (torch.float16, ("ChunkwiseChillMask", (128, 1)), 1, 34, 34, 4100, None, (128, 8)),
    # as many 8-wave workgroups as CUs and a few more, up to four times that, and beyond with and without padding
    (torch.bfloat16, ("CausalChillMask", ()), 1, 16, 16, 2048, None, (128, 8)),
    (torch.float16, ("CausalChillMask", ()), 2, 16, 8, 2081, (2081, 65), (128, 8)),
    (torch.float16, ("PrefixLMChillMask", (300,)), 3, 8, 8, 1441, (1441, 0, 299), (128, 8)),
    (torch.bfloat16, ("PrefixLMChillMask", (100,)), 4, 16, 16, 1920, None, (128, 8)),
    (torch.bfloat16, ("CausalChillMask", ()), 4, 16, 16, 2033, None, (128, 8)),
    (torch.float16, ("CausalChillMask", ()), 4, 16, 16, 2033, (2033, 700, 64, 1), (128, 8)),
    (torch.bfloat16, ("CausalChillMask", ()), 1, 8, 8, 4100, None, (128, 8)),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[1][0]}-{c[1][1]}-{c[5]}")
def test_against_the_oracle(case):
    dtype, m, B, H, H_kv, T, lens, shape = case
    mask = make_mask(m)
    cfg = tile_config(mask, 128, dtype, _lib.PASS_DKDV, seq_len=T, batch_heads=B * H_kv)
    assert (cfg["rows"], cfg["waves"]) == shape, cfg
    g = torch.Generator(DEV).manual_seed(7)
    q, k, v, d_out = (torch.randn(B, T, h, 128, device=DEV, generator=g).to(dtype).transpose(1, 2) for h in (H, H_kv, H_kv, H))
    lens_t = None if lens is None else torch.tensor(lens, dtype=torch.int32, device=DEV)
    leaves = [x.clone().requires_grad_() for x in (q, k, v)]
    ca.chill_attention(*leaves, mask=mask, lens=lens_t).backward(d_out)
    # relative 2-norm of rounding P and dS (8 or 11 bits) before the last products, and of rounding O before delta; a GQA
    # group's sum is rounded once more
    bound = 5e-3 if dtype == torch.bfloat16 else 7e-4
    ref_leaves = [x.float().requires_grad_() for x in (q, k, v)]
    ref, inside = orc.reference_naive(m[0], m[1], *ref_leaves, lens_t)
    ref.backward(d_out.float() * inside)
    for name, a, b in zip(("dk", "dv"), leaves[1:], ref_leaves[1:]):
        got, want = a.grad.double(), b.grad.double()
        assert torch.isfinite(got).all(), name
        if m[1] == (0, 0) and name == "dk":  # (a row that sees one key has no score gradient)
            assert got.abs().max() < 2e-2
            continue
        err = ((got - want).norm() / want.norm()).item()
        assert err < bound, (name, err)
        if lens is not None:
            for i, n in enumerate(lens):
                assert (got[i, :, n:] == 0).all(), name
