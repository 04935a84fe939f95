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
        assert O.rel_err(x.cpu(), r) <= 2e-4, name
