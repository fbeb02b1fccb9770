"""Pair-list gradients with the lists sorted in LDS (pair_lists_kernel) equal, bit
for bit, those with the device radix sort, which the same pairs take when unused
empty docs push the owner count past the LDS limit."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nq,nd,P", [(1, 1, 1), (3, 5, 64), (7, 2, 1000), (128, 1024, 4096), (2, 2048, 1023),
                                     (2048, 3, 1025), (40, 300, 16384), (40, 300, 16385), (600, 700, 9000)])
def test_lists_equal_radix_sort(nq, nd, P):
    from late_interaction_kernels._core import pairs_backward

    g = torch.Generator(device="cuda").manual_seed(P)
    dev = dict(generator=g, device="cuda")
    Lq, d = 5, 64
    dl = torch.randint(0, 9, (nd,), **dev)
    cq = torch.arange(nq + 1, device="cuda", dtype=torch.int32) * Lq
    cd = torch.nn.functional.pad(dl.cumsum(0), (1, 0)).to(torch.int32)
    Q = torch.randn(nq * Lq, d, **dev).bfloat16()
    D = torch.randn(max(int(dl.sum()), 1), d, **dev).bfloat16()
    pq = torch.randint(0, nq, (P,), **dev).to(torch.int32)
    pd = torch.randint(0, nd, (P,), **dev).to(torch.int32)
    pq[P // 3], pd[P // 2] = -1, nd + 6000  # out of range (there and with the unused docs): in no list
    ln = dl[pd.clamp(0, nd - 1).long()]
    am = (torch.rand(P, Lq, **dev) * ln[:, None]).to(torch.int32)
    am[ln == 0] = -1
    G = torch.randn(P, **dev)
    got = pairs_backward(G, Q, D, cq, cd, pq, pd, am, Lq, 9)
    cd2 = torch.cat([cd, cd[-1:].expand(5100)])
    want = pairs_backward(G, Q, D, cq, cd2, pq, pd, am, Lq, 9)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    # against fp64 sums
    ok = (pq >= 0) & (pd < nd)
    gq, gd = torch.zeros(nq * Lq, d, dtype=torch.float64, device="cuda"), torch.zeros(D.shape[0], d, dtype=torch.float64, device="cuda")
    rows_q = (pq.long()[:, None] * Lq + torch.arange(Lq, device="cuda"))[ok]
    a = am[ok].long()
    rows_d = cd[:-1].long()[pd[ok].long()][:, None] + a
    w = (G[ok][:, None] * (a >= 0)).double()
    rows_d = rows_d.clamp(0, D.shape[0] - 1)
    gq.index_add_(0, rows_q.reshape(-1), (w[..., None] * D[rows_d].double()).reshape(-1, d))
    gd.index_add_(0, rows_d.reshape(-1), (w[..., None] * Q[rows_q].double()).reshape(-1, d))
    for x, y in zip(got, (gq, gd)):
        assert ((x.double() - y).abs() <= 2**-8 * y.abs() + 1e-4).all()
