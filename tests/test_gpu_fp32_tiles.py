"""fp32 tiles of the HIP kernels at the lengths where their launches change shape, against the float64 oracle."""
import pytest
import torch

from oracle import fpa_oracle as O

pytestmark = pytest.mark.gpu

NAMES = ("o", "dq", "dk", "dv", "dphi", "dpsi", "dbeta")


@pytest.mark.parametrize("B,H,T,D", [
    (1, 1, 65, 64),      # one tile per side, one key past a block
    (1, 2, 449, 64),     # four tiles per side: the first length whose backward is split, one row in the last block
    (2, 4, 1000, 64),    # split, heads pinned to XCDs
    (1, 33, 512, 64),    # four tiles, 264 items: more than the one round that splits
    (1, 1, 1, 64),       # one row: every other row of its tiles is a copy of it
    (1, 2, 129, 32),     # a second workgroup of one row
    (1, 2, 300, 16),     # half-width operands: columns 16 .. 31 of the tiles are never written
])
def test_fp32_gradients(B, H, T, D):
    """All outputs within 2e-4 (2-norm), the bound the repository holds its fp32 path to; they are at 3e-6."""
    import fpa
    a = O.make_inputs(B, H, T, D, dtype=torch.float32, seed=71, psi_noise=1.0)
    leaves = [t.cuda().requires_grad_() for t in a[:6]]
    o = fpa.first_passage_attention(*leaves, impl="hip")
    got = (o.detach(),) + torch.autograd.grad(o, leaves, a[6].cuda())
    ref = O.fpa_grads_chunked(*a, device="cuda")
    for name, x, r in zip(NAMES, got, ref):
        # an exactly zero gradient (dq, dk, dphi, ... of a single row) is checked absolutely: the operands are of order 1
        err = O.rel_err(x.cpu(), r) if r.abs().max() > 0 else x.abs().max().item()
        assert err <= 2e-4, name


@pytest.mark.parametrize("D", [16, 32, 64])
@pytest.mark.parametrize("scale", [1e-12, 1.0, 1e4])
def test_fp32_products_as_bf16_triples(D, scale):
    """The fp32 products run on the bf16 matrix cores as sums of three-term splits, in each of which 2^-26 of a
    product is left out: o is within 2^-21 of the oracle, sixteen roundings of an fp32 result, at any size of v."""
    import fpa
    q, k, v, phi, psi, beta, do = O.make_inputs(1, 2, 500, D, dtype=torch.float32, seed=72, psi_noise=1.0)
    v = v * scale
    o = fpa.first_passage_attention(*(t.cuda() for t in (q, k, v, phi, psi, beta)), impl="hip")
    ref = O.fpa_grads(q, k, v, phi, psi, beta, do)[0]
    assert O.rel_err(o.cpu(), ref) <= 2.0 ** -21
