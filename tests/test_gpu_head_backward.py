"""Projection-head gradients (lik_head_backward) against float64 sums over the
winning rows, given grad_D and the winners: 16-bit outputs are rounded once
(2^-8 relative for bf16), fp32 sums are exact to ~1e-6; edges of the 32-row
blocks, the 64-column slices, the 384-column workgroups and the doc splits."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("Nq,Lq,Nd,Ld,d_out,dm", [
    (1, 1, 1, 1, 8, 8), (2, 32, 3, 31, 128, 768), (8, 32, 32, 257, 128, 384), (3, 17, 5, 64, 96, 392),
    (1, 32, 70, 500, 128, 776), (4, 32, 2, 8200, 40, 200), (2, 9, 600, 33, 64, 64), (40, 32, 2, 90, 120, 1032)])
def test_head_backward(Nq, Lq, Nd, Ld, d_out, dm, dtype):
    from late_interaction_kernels._core import head_backward

    g = torch.Generator(device="cuda").manual_seed(Nd + Ld)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda")
    am = torch.randint(-1, Ld, (Nq * Nd, Lq), generator=g, device="cuda", dtype=torch.int32)
    am.view(Nq, Nd, Lq)[:, Nd // 2] = -1  # a doc without winners
    won = torch.zeros(Nd, Ld + 1, dtype=torch.bool, device="cuda")
    won.scatter_(1, am.view(Nq, Nd, Lq).permute(1, 0, 2).reshape(Nd, -1).long().where(
        am.view(Nq, Nd, Lq).permute(1, 0, 2).reshape(Nd, -1) >= 0, torch.tensor(Ld, device="cuda")), True)
    won = won[:, :Ld]
    dp = (d_out + 7) // 8 * 8
    gd = rnd(Nd, Ld, dp) * won[..., None]
    gd[..., d_out:] = 0
    gd = gd.to(dtype)
    H = rnd(Nd, Ld + 1, dm).to(dtype)[:, 1:]  # strided docs
    H = torch.where(won[..., None], H, torch.full_like(H, float("nan")))[:, :, :]  # rows no query token won are not read
    W = rnd(d_out, dm).to(dtype)
    gh, gw, gb = head_backward(am, Nq, Lq, gd, H, W, need_h=True, need_w=True, need_b=True)
    r = gd[won][:, :d_out].double()
    wh = torch.zeros(Nd, Ld, dm, dtype=torch.float64, device="cuda")
    wh[won] = r @ W.double()
    ww, wb = r.t() @ H[won].double(), r.sum(0)
    tol = 2**-8 if dtype == torch.bfloat16 else 2**-11
    near = lambda a, b, t: ((a.double() - b).abs() <= t * b.abs() + 2e-5 * (b.abs().max() + 1e-30)).all()
    assert near(gh, wh, tol) and near(gw, ww, tol) and near(gb, wb, 1e-5)
    assert not gh[~won].any()
    again = head_backward(am, Nq, Lq, gd, H, W, need_h=True, need_w=True, need_b=True)
    assert all(torch.equal(a, b) for a, b in zip((gh, gw, gb), again))
    only = head_backward(am, Nq, Lq, gd, H, W, need_h=False, need_w=True, need_b=False)
    assert only[0] is None and only[2] is None and torch.equal(only[1], gw)


def test_calls_not_taken():
    from late_interaction_kernels._core import head_backward

    am = torch.zeros(2, 4, dtype=torch.int32, device="cuda")
    z = lambda *s, dt=torch.bfloat16: torch.zeros(*s, device="cuda", dtype=dt)
    kw = dict(need_h=True, need_w=True, need_b=True)
    assert head_backward(am, 1, 4, z(2, 9, 128, dt=torch.float32), z(2, 9, 64, dt=torch.float32),
                         z(128, 64, dt=torch.float32), **kw) is None
    assert head_backward(am, 1, 4, z(2, 9, 128), z(2, 9, 64, dt=torch.float16), z(128, 64), **kw) is None
    assert head_backward(am, 1, 4, z(2, 9, 136), z(2, 9, 64), z(136, 64), **kw) is None
    assert head_backward(am, 1, 4, z(2, 9, 128), z(2, 9, 60), z(128, 60), **kw) is None
