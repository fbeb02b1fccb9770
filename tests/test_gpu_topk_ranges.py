"""Top-k selection against a stable sort (score, then lower index): score ranges
that put everything in one bin or one key per bin, heavy ties, infinities and
signed zeros, k around the rank / bitonic limit, rows of one and several levels."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _scores(kind, rows, n, g):
    x = torch.randn(rows, n, generator=g, device="cuda")
    if kind == "narrow":
        return 30.0 + x * 1e-6
    if kind == "wide":
        return x * torch.exp(torch.randn(rows, n, generator=g, device="cuda") * 30)
    if kind == "ties":
        return (x * 2).round()
    if kind == "equal":
        return torch.full((rows, n), -1.5, device="cuda")
    if kind == "special":
        x[:, ::7] = float("inf")
        x[:, 1::11] = float("-inf")
        x[:, 2::5] = 0.0
        x[:, 3::5] = -0.0
    return x


@pytest.mark.parametrize("largest", [True, False])
@pytest.mark.parametrize("kind", ["normal", "narrow", "wide", "ties", "equal", "special"])
@pytest.mark.parametrize("rows,n,k", [(3, 1, 1), (2, 100, 100), (4, 4096, 100), (2, 4097, 256), (1, 30000, 257),
                                      (2, 9000, 1024), (1, 20000, 1500), (16, 4096, 10), (1, 300000, 100)])
def test_select_equals_stable_sort(rows, n, k, kind, largest):
    from late_interaction_kernels.topk import topk_update

    g = torch.Generator(device="cuda").manual_seed(n + k)
    s = _scores(kind, rows, n, g)
    got_s, got_i = topk_update(s, 0, None, None, k, largest)
    order = torch.sort(s, dim=-1, descending=largest, stable=True).indices[:, :k]
    assert torch.equal(got_i, order) and torch.equal(got_s, torch.gather(s, 1, order))
    # in two chunks, with a running list
    if n > 1:
        cut = n // 3 + 1
        rs, ri = topk_update(s[:, :cut], 0, None, None, k, largest)
        rs, ri = topk_update(s[:, cut:], cut, rs, ri, k, largest) if cut < n else (rs, ri)
        assert torch.equal(ri, order)
