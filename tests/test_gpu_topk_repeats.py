"""Top-k over candidates that appear more than once (a window merged again over
the running list, a list padded with (-inf, -1)): every output slot is written
and each appearance counts, as a sort of all candidates gives it."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _sorted(s, i, k, largest):
    """Rows of (score, index) candidates by score, then lower index."""
    o = torch.sort(i, dim=-1, stable=True).indices
    s, i = torch.gather(s, 1, o), torch.gather(i, 1, o)
    o = torch.sort(s, dim=-1, descending=largest, stable=True).indices[:, :k]
    return torch.gather(s, 1, o), torch.gather(i, 1, o)


def _update(s, base, rs, ri, k, largest):
    """topk_update into a result whose memory held sentinels before."""
    from late_interaction_kernels.topk import topk_update

    width = min(k, s.shape[1] + rs.shape[1])
    for _ in range(2):  # (the allocator hands these blocks to the call's outputs)
        a = torch.full((s.shape[0], width), float("nan"), device="cuda")
        b = torch.full((s.shape[0], width), -7, device="cuda", dtype=torch.int64)
    del a, b
    return topk_update(s, base, rs, ri, k, largest)


@pytest.mark.parametrize("largest", [True, False])
@pytest.mark.parametrize("ties", [False, True])
@pytest.mark.parametrize("rows,n,k", [(3, 40, 1), (2, 200, 100), (2, 300, 256), (2, 3000, 257), (1, 4096, 1024),
                                      (1, 9000, 100), (1, 9000, 1500), (2, 300000, 100)])
def test_window_merged_twice(rows, n, k, ties, largest):
    from late_interaction_kernels.topk import topk_update

    print(f"[case] repeats rows={rows} n={n} k={k} ties={ties} largest={largest}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + k)
    s = torch.randn(rows, n, generator=g, device="cuda")
    if ties:
        s = (s * 2).round() + 0.0  # (no -0)
    idx = torch.arange(n, device="cuda").expand(rows, n)
    # a list shorter than k (all candidates compete) and a full one, then the window
    # again in full and in part
    for first in (min(k, n) // 2, k):
        rs, ri = topk_update(s, 0, None, None, first, largest) if first else (s[:, :0].contiguous(), idx[:, :0].contiguous())
        for lo in (0, n // 2):
            got_s, got_i = _update(s[:, lo:], lo, rs, ri, k, largest)
            want_s, want_i = _sorted(torch.cat([rs, s[:, lo:]], 1), torch.cat([ri, idx[:, lo:]], 1), k, largest)
            assert torch.equal(got_s, want_s), (first, lo)
            assert torch.equal(got_i, want_i), (first, lo)


@pytest.mark.parametrize("k", [5, 100, 300])
def test_padded_running_list(k):
    """A list padded with (-inf, -1): the pads fill what the candidates leave."""
    g = torch.Generator(device="cuda").manual_seed(k)
    s = torch.randn(2, 3, generator=g, device="cuda")
    rs = torch.full((2, k), float("-inf"), device="cuda")
    ri = torch.full((2, k), -1, device="cuda", dtype=torch.int64)
    got_s, got_i = _update(s, 50, rs, ri, k, True)
    order = torch.sort(s, dim=1, descending=True).indices
    assert torch.equal(got_s[:, :3], torch.gather(s, 1, order)) and torch.equal(got_i[:, :3], order + 50)
    assert bool((got_s[:, 3:] == float("-inf")).all())
    assert bool((got_i[:, 3:] == 0xFFFFFFFF).all())  # indices are 32-bit (include/lik.h)


@pytest.mark.parametrize("k", [3, 200, 700])
def test_one_candidate_many_times(k):
    """A full list of one candidate, the index word of its key 0 or not, and a
    window below it: all the keys that are compared are equal."""
    for index in (-1, 41):
        s = torch.full((2, 5), float("-inf"), device="cuda")
        ri = torch.full((2, k), index, device="cuda", dtype=torch.int64)
        got_s, got_i = _update(s, 50, torch.zeros(2, k, device="cuda"), ri, k, True)
        assert bool((got_s == 0).all()) and bool((got_i == index & 0xFFFFFFFF).all())
