"""PLAID scoring of larger query blocks (lik_plaid_block.hip): bitwise the tile
kernel's scores (plaid_variant 3 forces it), and the oracle's within the bf16
bar, over tile and stage remainders, empty docs, both layouts, all residual
widths and the sizes at which the column block or the group count changes."""

import numpy as np
import pytest
import torch

import lik_oracle as O
from conftest import rel_err
from late_interaction_kernels._lib import launch_options

pytestmark = pytest.mark.gpu


def _index(lens, d, nbits, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    T = int(sum(lens))
    cent = torch.nn.functional.normalize(torch.randn(300, d, generator=g), dim=-1).to(dtype)
    codes = torch.randint(-2, 303, (T,), generator=g, dtype=torch.int32)  # some out of range
    res = torch.randint(0, 256, (T, d * nbits // 8), generator=g, dtype=torch.uint8)
    bw = torch.linspace(-0.2, 0.2, 2**nbits - 1)  # one bucket code has no weight
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32)
    return cent, codes, res, bw, cu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Nq,Lq,d,nbits,R", [
    (8, 32, 128, 2, 0), (9, 32, 128, 2, 1), (16, 32, 128, 4, 3), (17, 32, 128, 2, 5), (33, 31, 128, 2, 7),
    (5, 17, 128, 8, 2), (1, 33, 128, 2, 4), (1, 512, 128, 2, 2), (2, 257, 96, 4, 3), (20, 32, 64, 2, 0),
    (7, 30, 64, 4, 4), (6, 32, 40, 8, 9), (70, 24, 128, 2, 16)])
def test_block_equals_tile_kernel(Nq, Lq, d, nbits, R, dtype):
    from late_interaction_kernels.plaid import maxsim_residual, maxsim_residual_varlen

    rng = np.random.default_rng(Nq * Lq + d)
    lens = [0, 1, 31, 32, 33, 128, 129, 0, 0, 5, 300, 96] + rng.integers(0, 140, 40).tolist() + [0]
    cent, codes, res, bw, cu = _index(lens, d, nbits, dtype, Nq + Lq)
    g = torch.Generator().manual_seed(7)
    Q = torch.nn.functional.normalize(torch.randn(Nq, Lq, d, generator=g), dim=-1).to(dtype).cuda()
    args = [t.cuda() for t in (codes, res, cu, cent, bw)] + [nbits]
    for normalize in (True, False):
        with launch_options(docs_per_wg=R, plaid_route="fused"):
            got = maxsim_residual_varlen(Q, *args, normalize=normalize)
        with launch_options(plaid_variant=3, plaid_route="fused"):
            want = maxsim_residual_varlen(Q, *args, normalize=normalize)
        assert torch.equal(got, want)
    # padded layout, lengths past the extent are clamped to it
    L, n = 70, len(lens)
    keep = np.minimum(lens, L)
    pc = torch.zeros(n, L, dtype=torch.int32)
    pr = torch.zeros(n, L, res.shape[1], dtype=torch.uint8)
    for j in range(n):
        a = int(cu[j])
        pc[j, : keep[j]], pr[j, : keep[j]] = codes[a : a + keep[j]], res[a : a + keep[j]]
    pargs = [pc.cuda(), pr.cuda(), torch.tensor(lens).cuda(), cent.cuda(), bw.cuda(), nbits]
    with launch_options(docs_per_wg=R):
        got = maxsim_residual(Q, *pargs)
    with launch_options(plaid_variant=3):
        want = maxsim_residual(Q, *pargs)
    assert torch.equal(got, want)


def test_block_against_oracle():
    from late_interaction_kernels.plaid import maxsim_residual_varlen

    lens = np.random.default_rng(3).integers(0, 200, 60).tolist()
    cent, codes, res, bw, cu = _index(lens, 128, 2, torch.bfloat16, 11)
    codes, bw = codes.clamp(0, 299), torch.linspace(-0.2, 0.2, 4)
    g = torch.Generator().manual_seed(5)
    Q = torch.nn.functional.normalize(torch.randn(12, 32, 128, generator=g), dim=-1).to(torch.bfloat16)
    got = maxsim_residual_varlen(Q.cuda(), codes.cuda(), res.cuda(), cu.cuda(), cent.cuda(), bw.cuda(), 2)
    ref = O.maxsim_residual_varlen(Q.float().numpy(), codes.numpy(), res.numpy(), cu.numpy(), cent.float().numpy(),
                                   bw.numpy(), 2)
    assert rel_err(got.cpu().numpy(), ref) < 1e-2
