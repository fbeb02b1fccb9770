"""The docs-per-workgroup rule of cross products with several query blocks:
scores and winners do not depend on it (bitwise, against forced values), at doc
counts around its one-round and many-round cases, for one- and two-workgroup
column blocks and packed docs."""

import pytest
import torch

from late_interaction_kernels._lib import launch_options

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("Nq,Nd", [(17, 1), (17, 7), (64, 129), (100, 300), (40, 3100), (1100, 20), (2100, 9)])
def test_scores_do_not_depend_on_docs_per_workgroup(Nq, Nd, dtype):
    from late_interaction_kernels import maxsim, maxsim_varlen
    from late_interaction_kernels.forward import maxsim_forward

    g = torch.Generator(device="cuda").manual_seed(Nq + Nd)
    Lq, Ld, d = 32, 40, 128
    Q = torch.nn.functional.normalize(torch.randn(Nq, Lq, d, generator=g, device="cuda"), dim=-1).to(dtype)
    D = torch.nn.functional.normalize(torch.randn(Nd, Ld, d, generator=g, device="cuda"), dim=-1).to(dtype)
    lens = torch.randint(1, Ld + 1, (Nd,), generator=g, device="cuda")
    dm = torch.arange(Ld, device="cuda")[None] < lens[:, None]
    cu = torch.nn.functional.pad(lens.cumsum(0), (1, 0)).to(torch.int32)
    cq = torch.arange(Nq + 1, device="cuda", dtype=torch.int32) * Lq
    calls = (lambda: maxsim(Q, D, d_mask=dm), lambda: maxsim_varlen(Q.view(-1, d), D[dm], cq, cu, Lq, Ld))
    for call in calls:
        got = call()
        for r in (1, 5, 512):
            with launch_options(docs_per_wg=r):
                assert torch.equal(got, call())
    if dtype == torch.bfloat16 and Nq <= 100:
        s, am = maxsim_forward(Q, D, d_mask=dm, save_argmax=True)
        q = Q[-1:].contiguous()  # alone: another column block and range split
        s1, am1 = maxsim_forward(q, D, d_mask=dm, save_argmax=True)
        assert torch.equal(am.view(Nq, Nd, Lq)[-1], am1.view(Nd, Lq))
        assert torch.allclose(s[-1], s1[0], rtol=0, atol=1e-5)  # another order of the 32-term column sum
