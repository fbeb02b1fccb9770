"""Backward kernels for 16-bit rows of up to 128 dims, 16 bytes a lane
(grad_q_rows_kernel, grad_d_doc_kernel), at the pair counts and row counts
where their launch changes: against the oracle's gradients for the kernel's own
winners (outputs are rounded once to 16 bits, at most 2^-8 relative for
bf16; sums are fp32), and grad_D bit for bit against the radix-sorted kernel,
which takes the call when masked query tokens push it past the LDS sort."""

import numpy as np
import pytest
import torch

import lik_oracle as O
from conftest import rel_err

pytestmark = pytest.mark.gpu


def _inputs(Nq, Lq, Nd, Ld, d, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    Q = (torch.randn(Nq, Lq, d, generator=g) * 2).to(dtype)
    D = (torch.randn(Nd, Ld, d, generator=g) * 2).to(dtype)
    qm = torch.rand(Nq, Lq, generator=g) > 0.1
    dm = torch.arange(Ld)[None] < torch.randint(0, Ld + 1, (Nd,), generator=g)[:, None]
    dm[0] = True
    dm[-1] = torch.rand(Ld, generator=g) > 0.5
    G = torch.randn(Nq, Nd, generator=g)
    G[Nq // 2] = 0.0  # a query that adds nothing
    return Q, D, qm, dm, G


def _grads(Q, D, qm, dm, G, norm):
    from late_interaction_kernels._core import dense_maxsim_train, maxsim_backward

    _, am, Qp, Dp, qmi = dense_maxsim_train(Q.cuda(), D.cuda(), qm.cuda(), dm.cuda(), norm=norm, kd=False)
    gq, gd = maxsim_backward(G.cuda(), Qp, Dp, am, qmi, norm=norm, kd=False)
    return am, gq, gd


@pytest.mark.parametrize("norm", [0, 3])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Nq,Lq,Nd,Ld,d", [
    (5, 13, 3, 1, 128), (2, 33, 40, 31, 96), (64, 32, 9, 33, 128), (3, 683, 5, 300, 64), (256, 32, 4, 70, 128),
    (241, 34, 3, 1030, 40), (96, 128, 2, 1100, 128), (7, 30, 2, 2100, 128), (33, 7, 130, 65, 64)])
def test_rows_against_oracle(Nq, Lq, Nd, Ld, d, dtype, norm):
    Q, D, qm, dm, G = _inputs(Nq, Lq, Nd, Ld, d, dtype, Nq + Ld)
    am, gq, gd = _grads(Q, D, qm, dm, G, norm)
    wq, wd = O.maxsim_grads(G.numpy(), Q.float().numpy(), D.float().numpy(), am.view(Nq, Nd, Lq).cpu().numpy(),
                            qm.numpy(), normalize=bool(norm))
    assert rel_err(gq.float().cpu().numpy(), wq) < 2**-8
    assert rel_err(gd.float().cpu().numpy(), wd) < 2**-8
    _, gq2, gd2 = _grads(Q, D, qm, dm, G, norm)
    assert torch.equal(gq, gq2) and torch.equal(gd, gd2)


@pytest.mark.parametrize("norm", [0, 3])
@pytest.mark.parametrize("Nq,Lq,Nd,Ld,d", [(64, 32, 5, 300, 128), (256, 32, 3, 180, 128), (300, 40, 3, 90, 96),
                                           (128, 16, 4, 1030, 64), (9, 32, 33, 40, 128)])
def test_doc_kernel_equals_sorted_kernel(Nq, Lq, Nd, Ld, d, norm):
    Q, D, qm, dm, G = _inputs(Nq, Lq, Nd, Ld, d, torch.bfloat16, 3 * Nq + Ld)
    extra = 12288 // Nq + 1  # masked tokens: past the LDS sort's pair count
    g = torch.Generator().manual_seed(1)
    Qx = torch.cat([Q, torch.randn(Nq, extra, d, generator=g).to(Q.dtype)], 1)
    qmx = torch.cat([qm, torch.zeros(Nq, extra, dtype=torch.bool)], 1)
    _, gq, gd = _grads(Q, D, qm, dm, G, norm)
    _, gqx, gdx = _grads(Qx, D, qmx, dm, G, norm)
    assert torch.equal(gd, gdx)
    assert torch.equal(gq, gqx[:, :Lq]) and not gqx[:, Lq:].any()
