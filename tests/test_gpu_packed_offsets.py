"""Gradients against documents that lie far into a packed buffer: the calls take
a part of the buffer (``cu_seqlens_d[0] > 0``, include/lik.h), here one that
starts 64 GiB in, past 2**32 16-byte units, where a 32-bit row offset from the
buffer's start would wrap. The same documents at the start of a small buffer
give the same bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu

ROW0 = (1 << 28) - 300  # rows of 256 bytes: documents on both sides of the 64 GiB line


def _grad(call, Q):
    q = Q.clone().requires_grad_()
    s = call(q)
    w = torch.linspace(-1, 1, s.numel(), device="cuda").reshape(s.shape)
    (gq,) = torch.autograd.grad(s, q, w)
    return s.detach(), gq


@pytest.mark.parametrize("pairs", [False, True])
def test_grad_q_of_documents_beyond_64_gib(pairs):
    from late_interaction_kernels import maxsim_varlen
    from late_interaction_kernels.score_pairs import score_pairs_packed

    print(f"[case] grad_Q, packed docs 64 GiB into their buffer, pairs={pairs}", flush=True)
    if torch.cuda.mem_get_info()[0] < 80 << 30:
        pytest.skip("needs 80 GiB of free GPU memory")
    g = torch.Generator(device="cuda").manual_seed(3)
    lens = torch.tensor([70, 40, 130, 100, 33, 1], device="cuda")
    cu_d = torch.nn.functional.pad(lens.cumsum(0), (1, 0)).to(torch.int32)
    cu_q = torch.tensor([0, 20, 52, 60], device="cuda", dtype=torch.int32)
    Q = torch.nn.functional.normalize(torch.randn(60, 128, generator=g, device="cuda"), dim=-1).bfloat16()
    D = torch.nn.functional.normalize(torch.randn(int(lens.sum()), 128, generator=g, device="cuda"), dim=-1).bfloat16()
    big = torch.empty(ROW0 + D.shape[0], 128, device="cuda", dtype=torch.bfloat16)  # only the last rows are used
    big[ROW0:] = D
    pq = torch.tensor([0, 2, 1, 1, 0], device="cuda", dtype=torch.int32)
    pd = torch.tensor([5, 3, 2, 4, 0], device="cuda", dtype=torch.int32)

    def call(docs, cu):
        if pairs:
            return lambda q: score_pairs_packed(q, docs, cu_q, cu, pq, pd, max_seqlen_q=32, max_seqlen_d=130)
        return lambda q: maxsim_varlen(q, docs, cu_q, cu, max_seqlen_q=32, max_seqlen_d=130)

    s0, g0 = _grad(call(D, cu_d), Q)
    s1, g1 = _grad(call(big, cu_d + ROW0), Q)
    del big
    torch.cuda.empty_cache()
    assert torch.equal(s0, s1)
    assert torch.equal(g0, g1)
    assert g0.abs().sum() > 0
