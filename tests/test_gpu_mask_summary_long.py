"""Mask summaries in the dword form with rows on and off 4-byte boundaries, up to
2048 tokens, and the byte form past that; holes in the last passes, the last
doc's last token kept; scores against the oracle (bf16 products, fp32 sums)."""

import numpy as np
import pytest
import torch

import lik_oracle as O
from conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lead", [0, 1, 3])
@pytest.mark.parametrize("L,pad", [(1, 0), (5, 0), (17, 0), (255, 0), (257, 2), (301, 0), (1024, 1), (1025, 3), (1030, 0), (1028, 0), (1030, 2), (1792, 0), (2048, 0), (2047, 1), (2052, 0)])
def test_masks(L, pad, lead):
    from late_interaction_kernels import maxsim

    g = torch.Generator().manual_seed(L)
    nd = 21
    Q = torch.randn(2, 8, 64, generator=g).to(torch.bfloat16)
    D = torch.randn(nd, L, 64, generator=g).to(torch.bfloat16)
    dm = torch.arange(L)[None] < torch.randint(0, L + 1, (nd,), generator=g)[:, None]
    dm[::4] = torch.rand(len(dm[::4]), L, generator=g) > 0.5
    dm[1], dm[2] = False, True
    dm[3] = False
    dm[3, L - 1] = True  # only the last token
    dm[-1, L - 1] = True
    # row stride L + pad, the first row `lead` bytes into its allocation
    flat = torch.ones(lead + nd * (L + pad), dtype=torch.bool, device="cuda")
    rows = flat[lead:].view(nd, L + pad)[:, :L]
    rows.copy_(dm)
    got = maxsim(Q.cuda(), D.cuda(), None, rows).cpu().numpy()
    ref = O.maxsim(Q.double().numpy(), D.double().numpy(), None, dm.numpy())
    assert np.isfinite(got).all() and rel_err(got, ref) < 1e-5
