"""Few documents on the streaming kernel: four wavefronts share a doc. The tile
kernel's bits (a forced column block takes that one) at doc counts around the
limit, docs of fewer tiles than wavefronts, empty docs, masks, both layouts."""

import pytest
import torch

from late_interaction_kernels._lib import launch_options

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("normalize", [False, True])
@pytest.mark.parametrize("Nq,Lq,Nd,Ld,d", [(1, 32, 1, 1, 128), (1, 32, 50, 180, 128), (1, 9, 511, 33, 128),
                                           (1, 32, 512, 70, 128), (1, 32, 513, 70, 128), (2, 16, 37, 129, 128),
                                           (1, 32, 20, 1030, 64), (1, 20, 33, 300, 256), (1, 32, 9, 97, 96)])
def test_split_equals_tile_kernel(Nq, Lq, Nd, Ld, d, normalize, dtype):
    from late_interaction_kernels import maxsim, maxsim_varlen

    g = torch.Generator(device="cuda").manual_seed(Nd + Ld)
    Q = torch.randn(Nq, Lq, d, generator=g, device="cuda").to(dtype)
    D = torch.randn(Nd, Ld, d, generator=g, device="cuda").to(dtype)
    lens = torch.randint(0, Ld + 1, (Nd,), generator=g, device="cuda")
    dm = torch.arange(Ld, device="cuda")[None] < lens[:, None]
    holes = dm & (torch.rand(Nd, Ld, generator=g, device="cuda") > 0.3)
    cu = torch.nn.functional.pad(lens.cumsum(0), (1, 0)).to(torch.int32)
    cq = torch.arange(Nq + 1, device="cuda", dtype=torch.int32) * Lq
    calls = [lambda m=m: maxsim(Q, D, d_mask=m, normalize=normalize) for m in (None, dm, holes)]
    if not normalize and int(cu[-1]):
        calls.append(lambda: maxsim_varlen(Q.view(-1, d), D[dm], cq, cu, Lq, Ld))
    for call in calls:
        got = call()
        with launch_options(cfg=(4, 1)):
            assert torch.equal(got, call())


def test_split_kd_and_nan():
    from late_interaction_kernels import maxsim

    g = torch.Generator(device="cuda").manual_seed(2)
    Q = torch.randn(7, 24, 128, generator=g, device="cuda").bfloat16()
    D = torch.randn(7, 11, 150, 128, generator=g, device="cuda").bfloat16()
    D[1, 2, 149] = float("nan")  # scores 0: the last quarter carries the NaN
    D[2, 3, 0, 5] = float("inf")
    got = maxsim(Q, D)
    with launch_options(cfg=(4, 1)):
        assert torch.equal(got, maxsim(Q, D))
    assert got[1, 2] == 0 and torch.isfinite(got).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("P,Lq,Ld,d", [(1, 32, 1, 128), (7, 32, 300, 128), (512, 8, 70, 128), (300, 32, 1030, 64),
                                       (65, 20, 129, 256), (33, 32, 97, 512), (40, 31, 257, 96)])
def test_split_pairs_equal_whole_docs(P, Lq, Ld, d, dtype):
    """Pair lists of up to 512 pairs split their docs too: the bits of the same
    pairs in a list of more than 512, where a wavefront takes a whole doc."""
    from late_interaction_kernels.score_pairs import score_pairs_packed

    nq, nd = 5, 40
    g = torch.Generator(device="cuda").manual_seed(P + Ld)
    lens = torch.randint(0, Ld + 1, (nd,), generator=g, device="cuda")
    lens[:3] = torch.tensor([Ld, 0, 1])
    ql = torch.tensor([Lq, 1, 0, Lq, 5], device="cuda").clamp_max(Lq)
    cd, cq = (torch.nn.functional.pad(x.cumsum(0), (1, 0)).to(torch.int32) for x in (lens, ql))
    Q = torch.randn(int(cq[-1]), d, generator=g, device="cuda").to(dtype)
    D = torch.randn(int(cd[-1]), d, generator=g, device="cuda").to(dtype)
    D[int(cd[1]) - 1, 3] = float("nan")
    pq = torch.randint(-1, nq + 1, (P,), generator=g, device="cuda").to(torch.int32)  # ids out of range too
    pd = torch.randint(-1, nd + 1, (P,), generator=g, device="cuda").to(torch.int32)
    pq[0], pd[0] = 0, 0
    times = 512 // P + 1
    got = score_pairs_packed(Q, D, cq, cd, pq, pd, max_seqlen_q=Lq, max_seqlen_d=Ld)
    want = score_pairs_packed(Q, D, cq, cd, pq.repeat(times), pd.repeat(times), max_seqlen_q=Lq, max_seqlen_d=Ld)
    assert torch.equal(got, want[:P]) and torch.isfinite(got).all()
