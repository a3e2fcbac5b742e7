"""fp32 inputs through the fp16 matrix instructions (csrc/chill_f32_parts.h, csrc/chill_f32.h): every shape of workgroup that a
launch can take, at ragged sizes, against attention in 64 bits; inputs of any magnitude; infinities."""
import math

import pytest
import torch

import chill_attention as ca
from conftest import make_mask
from oracle import chill_oracle as orc

pytestmark = pytest.mark.gpu
DEV = "cuda"

# id, mask, B, H, H_kv, T, D, lens; the shape of the workgroups follows from the number of 32-row tiles and the mask
CASES = [
    ("eight-streams", ("CausalChillMask", ()), 1, 3, 3, 777, 64, None),
    ("eight-streams-gqa-lens", ("SlidingWindowChillMask", (100, 37)), 2, 4, 2, 517, 32, (517, 70)),
    ("eight-streams-16", ("ChunkwiseChillMask", (100, 1)), 1, 3, 1, 1025, 16, None),
    ("four-streams", ("CausalChillMask", ()), 1, 8, 4, 1024, 64, None),
    ("pairs-odd", ("PrefixLMChillMask", (200,)), 2, 4, 4, 1090, 64, (1090, 33)),
    ("pairs-neighbours-gqa", ("FullChillMask", ()), 1, 12, 3, 1001, 64, (970,)),
    ("pairs-16", ("CausalChillMask", ()), 3, 3, 3, 1057, 16, None),
    ("four-members", ("ChunkwiseChillMask", (77, 2)), 2, 16, 8, 1111, 64, (1000, 1111)),
    ("four-members-32", ("FullChillMask", ()), 4, 8, 8, 1030, 32, None),
    ("wide-four-streams", ("CausalChillMask", ()), 1, 2, 1, 600, 128, (599,)),
    ("wide-pairs", ("SlidingWindowChillMask", (64, 200)), 1, 10, 5, 1003, 128, None),
    ("wide-four-members", ("PrefixLMChillMask", (100,)), 2, 12, 4, 1100, 128, (1100, 65)),
]


def reference(m, q, k, v, d_out, lens):
    """Attention and its gradients in 64 bits (chill.py:498-544)."""
    B, H, T, D = q.shape
    G = H // k.shape[1]
    q, k, v = (x.detach().double().requires_grad_() for x in (q, k, v))
    seen = torch.as_tensor(orc.dense_mask(*m, T), device=DEV)
    pos = torch.arange(T, device=DEV)
    n = torch.full((B,), T, device=DEV) if lens is None else torch.tensor(lens, device=DEV)
    inside = pos < n[:, None]
    seen = seen & inside[:, None, :, None] & inside[:, None, None, :]
    s = (q @ k.repeat_interleave(G, 1).transpose(-1, -2).contiguous()) / math.sqrt(D)
    p = torch.softmax(s.masked_fill(~seen, -math.inf), -1).nan_to_num(0.0)
    out = (p @ v.repeat_interleave(G, 1)) * inside[:, None, :, None]
    out.backward(d_out.double())
    return out.detach(), q.grad, k.grad, v.grad


def inputs(B, H, H_kv, T, D, seed=0):
    g = torch.Generator(DEV).manual_seed(seed)
    return [torch.randn(B, T, h, D, device=DEV, generator=g).transpose(1, 2) for h in (H, H_kv, H_kv, H)]


def run(mask, q, k, v, d_out, lens):
    lens = None if lens is None else torch.tensor(lens, dtype=torch.int32, device=DEV)
    q, k, v = (x.detach().requires_grad_() for x in (q, k, v))
    out, lse = ca.chill_attention(q, k, v, mask=mask, lens=lens, return_lse=True)
    return (out.detach(), *torch.autograd.grad(out, (q, k, v), d_out)), lse


@pytest.mark.parametrize("case", CASES, ids=lambda c: c[0])
def test_against_64_bits(case):
    _, m, B, H, H_kv, T, D, lens = case
    mask = make_mask(m)
    q, k, v, d_out = inputs(B, H, H_kv, T, D)
    got, _ = run(mask, q, k, v, d_out, lens)
    for name, a, b in zip(("out", "dq", "dk", "dv"), got, reference(m, q, k, v, d_out, lens)):
        # relative 2-norm: the fp32 instruction gives 2e-7 .. 1e-6 at these sizes, the parts three quarters of that
        err = ((a.double() - b).norm() / b.norm()).item()
        assert err < 1e-6, (name, err)
        if lens is not None:
            for i, n in enumerate(lens):
                assert (a[i, :, n:] == 0).all(), name


# rows of few blocks, where the choice between the fp32 instruction (one or two sets of waves) and the parts lies: a mask and a T on
# either side of each limit, with ragged ends, shared heads and lengths
FEW_BLOCKS = [
    ("one-block", ("CausalChillMask", ()), 1, 1, 1, 31, 64, None),
    ("128-keys", ("FullChillMask", ()), 1, 2, 2, 128, 64, None),
    ("129-keys", ("FullChillMask", ()), 2, 2, 1, 129, 64, (129, 1)),
    ("two-sets-32", ("FullChillMask", ()), 1, 4, 2, 255, 32, (200,)),
    ("two-sets-16", ("SlidingWindowChillMask", (64, 64)), 2, 3, 3, 333, 16, (333, 40)),
    ("two-sets-all-units", ("SlidingWindowChillMask", (100, 60)), 1, 8, 4, 1023, 64, None),
    ("growing-rows-257", ("CausalChillMask", ()), 1, 3, 3, 257, 64, None),
    ("dq-385", ("PrefixLMChillMask", (30,)), 1, 3, 1, 385, 64, None),
    ("dq-513", ("CausalChillMask", ()), 1, 2, 2, 513, 64, (511,)),
    ("chunks", ("ChunkwiseChillMask", (32, 1)), 1, 4, 2, 700, 64, None),
    ("wide-256", ("CausalChillMask", ()), 1, 2, 1, 256, 128, (250,)),
    ("wide-385", ("FullChillMask", ()), 1, 2, 2, 385, 128, None),
    ("wide-window", ("SlidingWindowChillMask", (40, 0)), 1, 8, 2, 1001, 128, None),
]


@pytest.mark.parametrize("case", FEW_BLOCKS, ids=lambda c: c[0])
def test_few_blocks(case):
    _, m, B, H, H_kv, T, D, lens = case
    q, k, v, d_out = inputs(B, H, H_kv, T, D)
    got, _ = run(make_mask(m), q, k, v, d_out, lens)
    for name, a, b in zip(("out", "dq", "dk", "dv"), got, reference(m, q, k, v, d_out, lens)):
        # as above (a row of one key has a dQ and dK of rounding alone: the difference over that of the inputs then)
        err = ((a.double() - b).norm() / torch.maximum(b.norm(), 0.1 * q.double().norm())).item()
        assert err < 1e-6, (name, err)


@pytest.mark.parametrize("case", CASES[::2], ids=lambda c: c[0])
def test_any_magnitude(case):
    """Powers of two pass through the scaled parts exactly: inputs scaled by them give the same bits, scaled."""
    _, m, B, H, H_kv, T, D, lens = case
    mask = make_mask(m)
    q, k, v, d_out = inputs(B, H, H_kv, T, D, seed=1)
    want, lse = run(mask, q, k, v, d_out, lens)
    for a, b, c in ((40, 30, -50), (-45, -60, 20), (60, 5, 3)):
        got, lse2 = run(mask, q * 2.0**a, k * 2.0**-a, v * 2.0**b, d_out * 2.0**c, lens)
        assert torch.equal(lse, lse2)
        for x, y, e in zip(got, want, (b, b + c - a, b + c + a, c)):
            assert torch.equal(x, y * 2.0**e), e


@pytest.mark.parametrize("case", [c for c in CASES if c[-1] is not None], ids=lambda c: c[0])
def test_rows_past_the_lengths(case):
    """What the tensors hold behind a sequence, however large, does not reach the scales of the rows before it."""
    _, m, B, H, H_kv, T, D, lens = case
    mask = make_mask(m)
    x = inputs(B, H, H_kv, T, D, seed=4)
    want, lse = run(mask, *x, lens)
    for garbage in (1e30, math.nan):
        y = [t.clone() for t in x]
        for t in y[:3]:
            for i, n in enumerate(lens):
                t[i, :, n:] = garbage
        got, lse2 = run(mask, *y, lens)
        assert torch.equal(lse, lse2)
        for name, a, b in zip(("out", "dq", "dk", "dv"), got, want):
            assert torch.equal(a, b), (name, garbage)


@pytest.mark.parametrize("case", CASES[::3] + CASES[-1:], ids=lambda c: c[0])
def test_infinities(case):
    """Infinities have no parts: the waves that meet one compute their blocks with the fp32 instruction."""
    _, _, B, H, H_kv, T, D, _ = case
    mask, G, at = ca.CausalChillMask(), H // H_kv, T // 2
    q, k, v, d_out = inputs(B, H, H_kv, T, D, seed=2)
    # a value: the rows that see it are infinite in its column
    v_inf = v.clone()
    v_inf[0, 0, at, 3] = math.inf
    out = ca.chill_attention(q, k, v_inf, mask=mask)
    plain = ca.chill_attention(q, k, v, mask=mask)
    assert (out[0, :G, at:, 3] == math.inf).all()
    other = torch.ones(D, dtype=torch.bool, device=DEV)
    other[3] = False
    torch.testing.assert_close(out[..., other], plain[..., other], atol=2e-6, rtol=1e-4)
    before = 32 * (at // 32)  # (rows whose blocks stop short of it)
    torch.testing.assert_close(out[:, :, :before], plain[:, :, :before], atol=2e-6, rtol=1e-4)
    # a key whose score is -inf for every query is not seen
    q = q.abs() + 0.01
    k_inf = k.clone()
    k_inf[:, :, at] = -math.inf
    out = ca.chill_attention(q, k_inf, v, mask=mask)
    s = (q.double() @ k.double().repeat_interleave(G, 1).transpose(-1, -2).contiguous()) / math.sqrt(D)
    seen = torch.ones(T, T, dtype=torch.bool, device=DEV).tril()
    seen[:, at] = False
    want = torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ v.double().repeat_interleave(G, 1)
    assert torch.isfinite(out).all()
    torch.testing.assert_close(out.double(), want, atol=2e-6, rtol=1e-4)
    # NaN in a query stays in its row
    q_nan = q.clone()
    q_nan[0, 0, at] = math.nan
    out = ca.chill_attention(q_nan, k, v, mask=mask)
    assert torch.isnan(out[0, 0, at]).all()
    clean = torch.ones(T, dtype=torch.bool, device=DEV)
    clean[at] = False
    assert torch.isfinite(out[0, 0, clean]).all()
    # gradients: an infinite dO row reaches dV of the keys its query sees
    d_inf = d_out.clone()
    d_inf[0, 0, at, 5] = math.inf
    grads, _ = run(mask, q, k, v, d_inf, None)
    assert (grads[3][0, 0, :at + 1, 5] == math.inf).all() and torch.isfinite(grads[3][0, 0, :before, 6]).all()
