"""The max_seqlen bounds check: exact against numpy, around the workgroup's
step, with one or two arrays, empty sequences and bounds equal to the longest."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _ok(a, ma, b, mb):
    from late_interaction_kernels import _lib

    ok = torch.empty((), device="cuda", dtype=torch.bool)
    _lib.check(_lib.load().lik_seqlens_cover(a.data_ptr(), a.numel() - 1, ma, b.data_ptr(), b.numel() - 1, mb,
                                             ok.data_ptr(), _lib.stream_of(ok)), "lik_seqlens_cover")
    return bool(ok)


@pytest.mark.parametrize("n", [1, 63, 1024, 1025, 4097, 20000])
def test_cover(n):
    rng = np.random.default_rng(n)
    lens = rng.integers(0, 50, n)
    at = int(rng.integers(0, n))
    lens[at] = 77  # the longest, at any place
    cu = torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32).cuda()
    short = torch.tensor([0, 3, 3, 9], dtype=torch.int32).cuda()
    assert _ok(cu, 77, short, 6) and _ok(short, 6, cu, 77) and _ok(cu, 1 << 40, cu, 77)
    assert not _ok(cu, 76, short, 6) and not _ok(cu, 77, short, 5) and not _ok(short, 6, cu, 76)
    assert not _ok(cu, -1, cu, 77)


def test_bounds_accepted_on_every_entry_point():
    """Covering bounds pass (equal to the longest, or larger) and change nothing."""
    from late_interaction_kernels import maxsim_varlen
    from late_interaction_kernels.score_pairs import score_pairs_packed

    g = torch.Generator(device="cuda").manual_seed(0)
    cq = torch.tensor([0, 5, 5, 32], dtype=torch.int32, device="cuda")
    cd = torch.tensor([0, 40, 41, 141], dtype=torch.int32, device="cuda")
    Q = torch.randn(32, 64, generator=g, device="cuda").bfloat16()
    D = torch.randn(141, 64, generator=g, device="cuda").bfloat16()
    want = maxsim_varlen(Q, D, cq, cd)
    for mq, md in ((27, 100), (27, None), (None, 100), (1000, 1000)):
        assert torch.equal(maxsim_varlen(Q, D, cq, cd, mq, md), want)
    i = torch.arange(3, device="cuda").repeat(3)
    s = score_pairs_packed(Q, D, cq, cd, i.sort().values, i, max_seqlen_q=27, max_seqlen_d=100)
    assert torch.allclose(s.view(3, 3), want, rtol=1e-6, atol=1e-5)  # another order of the column sum
    torch.cuda.synchronize()


@pytest.mark.parametrize("entry", ["varlen", "pairs"])
@pytest.mark.parametrize("mq,md,want", [(27, 100, set()), (26, 100, {"max_seqlen_q=26"}), (27, 99, {"max_seqlen_d=99"}),
                                        (1, 2, {"max_seqlen_q=1", "max_seqlen_d=2"}), (None, 99, {"max_seqlen_d=99"}),
                                        (26, None, {"max_seqlen_q=26"})])
def test_each_bound_has_its_own_message(monkeypatch, entry, mq, md, want):
    """The assert that fails names the bound that is too small, and no other. (The
    asserts are recorded on the host here, so none of them fires on the GPU; the
    calls stop at them.)"""
    from late_interaction_kernels import maxsim_varlen
    from late_interaction_kernels.score_pairs import score_pairs_packed

    cq = torch.tensor([0, 5, 5, 32], dtype=torch.int32, device="cuda")
    cd = torch.tensor([0, 40, 41, 141], dtype=torch.int32, device="cuda")
    Q, D = torch.zeros(32, 64, device="cuda").bfloat16(), torch.zeros(141, 64, device="cuda").bfloat16()
    seen = []
    monkeypatch.setattr(torch, "_assert_async", lambda ok, msg: seen.append((bool(ok), msg)))
    module = "late_interaction_kernels." + ("varlen" if entry == "varlen" else "score_pairs")

    class Stop(Exception):
        pass

    def stop(*a, **k):
        raise Stop

    monkeypatch.setattr(f"{module}.unify_dtype", stop)
    i = torch.zeros(1, device="cuda", dtype=torch.int32)
    with pytest.raises(Stop):
        if entry == "varlen":
            maxsim_varlen(Q, D, cq, cd, mq, md)
        else:
            score_pairs_packed(Q, D, cq, cd, i, i, max_seqlen_q=mq, max_seqlen_d=md)
    failed = {msg.split(" ")[0] for ok, msg in seen if not ok}
    assert failed == want
    assert all(msg.count("max_seqlen") == 1 for _, msg in seen)
