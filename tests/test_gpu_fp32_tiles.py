"""fp32 tiles of the HIP kernels at the lengths where their launches change shape, against the float64 oracle."""
import pytest
import torch

from oracle import fpa_oracle as O

pytestmark = pytest.mark.gpu

NAMES = ("o", "dq", "dk", "dv", "dphi", "dpsi", "dbeta")


@pytest.mark.parametrize("B,H,T,D", [
    (1, 1, 65, 64),      # one tile per side, one key past a block
    (1, 2, 385, 64),     # four tiles per side, the last of one row: the first length whose backward is split
    (1, 2, 449, 64),     # four tiles per side, one row in the last block
    (2, 4, 1000, 64),    # split, heads pinned to XCDs
    (1, 33, 512, 64),    # four tiles, 264 items: more than the one round that splits
    (1, 128, 512, 64),   # 512 tiles a side, two rounds: two launches
    (1, 1, 1, 64),       # one row: every other row of its tiles is a copy of it
    (1, 2, 129, 32),     # a second workgroup of one row
    (1, 2, 300, 16),     # half-width operands: columns 16 .. 31 of the tiles are never written
])
def test_fp32_gradients(B, H, T, D):
    """Largest difference over the largest value: within 1e-5, five times the largest of these shapes (1.9e-6); dbeta, whose
    terms cancel, within 2e-4, the bound the repository holds its fp32 path to."""
    import fpa
    a = O.make_inputs(B, H, T, D, dtype=torch.float32, seed=71, psi_noise=1.0)
    leaves = [t.cuda().requires_grad_() for t in a[:6]]
    o = fpa.first_passage_attention(*leaves, impl="hip")
    got = (o.detach(),) + torch.autograd.grad(o, leaves, a[6].cuda())
    ref = O.fpa_grads_chunked(*a, device="cuda")
    for name, x, r in zip(NAMES, got, ref):
        # an exactly zero gradient (dq, dk, dphi, ... of a single row) is checked absolutely: the operands are of order 1
        err = O.rel_err(x.cpu(), r) if r.abs().max() > 0 else x.abs().max().item()
        assert err <= (2e-4 if name == "dbeta" else 1e-5), name


@pytest.mark.parametrize("D", [16, 32, 64])
@pytest.mark.parametrize("scale", [1e-12, 1.0, 1e4])
def test_fp32_products_as_bf16_triples(D, scale):
    """P V runs on the bf16 matrix cores as sums of three-term splits, in which 2^-26 of a product is left out: o is
    within 2^-21 of the oracle, eight roundings of an fp32 result, as it is without them."""
    import fpa
    q, k, v, phi, psi, beta, do = O.make_inputs(1, 2, 500, D, dtype=torch.float32, seed=72, psi_noise=1.0)
    v = v * scale
    o = fpa.first_passage_attention(*(t.cuda() for t in (q, k, v, phi, psi, beta)), impl="hip")
    ref = O.fpa_grads(q, k, v, phi, psi, beta, do)[0]
    assert O.rel_err(o.cpu(), ref) <= 2.0 ** -21


def _forward(q, k, v, phi, psi, beta):
    """o from the kernels, and the oracle's in float64."""
    import fpa
    o = fpa.first_passage_attention(*(t.cuda() for t in (q, k, v, phi, psi, beta)), impl="hip").cpu()
    return o, O.fpa_forward(*(t.double() for t in (q, k, v, phi, psi, beta)))


@pytest.mark.parametrize("T", [200, 700])  # rows whole, and split in two parts
@pytest.mark.parametrize("D", [16, 32, 64])
@pytest.mark.parametrize("value", [2.0 ** 64, -1e30, 3.4e38, float("inf"), float("-inf")])
def test_fp32_huge_v(D, T, value):
    """One value of v at or past the end of what splits into bf16 triples: the rows that see it hold its share
    (an infinity for an infinity), every other output is as it is without it.  Key 128 starts a tile, so no
    row before it meets it, not even with weight 0.  The largest finite value takes equal weights, whose sums
    cannot overflow.  Bounds: 2^-20 for one weight (scores below 2: their rounding and exp2, the row sum, the
    division, each within 2^-22), 2^-21 of the largest output as above."""
    q, k, v, phi, psi, _, _ = O.make_inputs(1, 2, T, D, dtype=torch.float32, seed=73)
    q = q * (0.0 if value == 3.4e38 else 0.25)
    beta = torch.zeros(2)
    base, _ = _forward(q, k, v, phi, psi, beta)
    v[0, 1, 128, 5] = value
    o, ref = _forward(q, k, v, phi, psi, beta)
    seen = o[0, 1, 128:, 5]
    if abs(value) == float("inf"):
        assert (seen == value).all()
    else:
        want = ref[0, 1, 128:, 5]
        assert ((seen.double() - want).abs() <= 2.0 ** -20 * want.abs()).all()
    o[0, 1, 128:, 5] = base[0, 1, 128:, 5]
    v[0, 1, 128, 5] = 0.0
    assert torch.isfinite(o).all() and O.rel_err(o, base) <= 2.0 ** -21


@pytest.mark.parametrize("D", [16, 32, 64])
@pytest.mark.parametrize("scale", [1e-30, 1e-33, 1e-36])
def test_fp32_tiny_v(D, scale):
    """Values whose bf16 triples would be subnormal: o (down to 1e-37, still normal) is within the same 2^-21."""
    q, k, v, phi, psi, beta, _ = O.make_inputs(1, 2, 500, D, dtype=torch.float32, seed=74)
    o, ref = _forward(q, k, v * scale, phi, psi, beta)
    assert O.rel_err(o.double() / scale, ref / scale) <= 2.0 ** -21


@pytest.mark.parametrize("D", [16, 32, 64])
@pytest.mark.parametrize("value", [1.0, 2.0 ** 60, 2.0 ** 100])
def test_fp32_tiny_weight(D, value):
    """A weight of 2^-124 (score -86) on the only nonzero value: its share is o.  Bound 2^-15: the score, 124 in base 2,
    and its scaling round by 2^-17 each, which exp2 turns into a relative error."""
    q = torch.zeros(1, 1, 3, D)
    k, v = torch.zeros_like(q), torch.zeros_like(q)
    q[..., 0] = 8.0
    k[0, 0, 0, 0] = -86.0 * D ** 0.5 / 8.0
    v[0, 0, 0, 3] = value
    zero = torch.zeros(1, 1, 3)
    o, ref = _forward(q, k, v, zero, zero, torch.zeros(1))
    assert ((o.double() - ref)[0, 0, 2].abs() <= 2.0 ** -15 * ref[0, 0, 2].abs()).all()
