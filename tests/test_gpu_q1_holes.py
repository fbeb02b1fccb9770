"""Masks with holes on the streaming one-block kernel: the bits of the tile
kernel's masked launch (a forced column block takes that one), and the training
forward's winners against a plain float64 restatement; dropped rows hold NaN."""

import pytest
import torch

from late_interaction_kernels._lib import launch_options

pytestmark = pytest.mark.gpu


def _docs(n, Ld, d, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    D = torch.randn(n, Ld, d, generator=g)
    dm = torch.rand(n, Ld, generator=g) > 0.3
    dm[0] = torch.arange(Ld) < (Ld + 1) // 2  # a prefix
    dm[1] = False
    dm[2] = False
    dm[2, Ld - 1] = True  # only the last token
    D[~dm] = float("nan")
    return D.to(dtype), dm, g


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("normalize", [False, True])
@pytest.mark.parametrize("Nq,K,Lq,Ld,d", [(3, 5, 32, 33, 128), (1, 40, 17, 300, 128), (4, 6, 8, 1030, 128),
                                          (2, 9, 32, 64, 64), (2, 4, 30, 65, 256), (3, 3, 32, 31, 96)])
def test_holes_equal_tile_kernel(Nq, K, Lq, Ld, d, normalize, dtype):
    from late_interaction_kernels import maxsim

    D, dm, g = _docs(Nq * K, Ld, d, dtype, Nq * Ld + d)
    Q = torch.randn(Nq, Lq, d, generator=g).to(dtype).cuda()
    D, dm = D.view(Nq, K, Ld, d).cuda(), dm.view(Nq, K, Ld).cuda()
    got = maxsim(Q, D, d_mask=dm, normalize=normalize)
    with launch_options(cfg=(4, 1)):
        want = maxsim(Q, D, d_mask=dm, normalize=normalize)
    assert torch.equal(got, want) and torch.isfinite(got).all()


@pytest.mark.parametrize("Ld", [1, 32, 75, 300])
def test_holes_training_winners(Ld):
    """KD training forward (argmax on the streaming kernel): winners whose
    margin exceeds the bf16 products' error, -1 exactly for empty docs."""
    from late_interaction_kernels._core import dense_maxsim_train

    Nq, K, Lq, d = 3, 7, 32, 128
    D, dm, g = _docs(Nq * K, Ld, d, torch.bfloat16, Ld)
    Q = torch.randn(Nq, Lq, d, generator=g).to(torch.bfloat16)
    _, am, *_ = dense_maxsim_train(Q.cuda(), D.cuda(), None, dm.cuda(), norm=0, kd=True)
    am = am.view(Nq * K, Lq).cpu()
    for j in range(Nq * K):
        if not dm[j].any():
            assert (am[j] == -1).all()
            continue
        S = Q[j // K].double() @ D[j].nan_to_num().double().t()
        S[:, ~dm[j]] = -torch.inf
        top = S.topk(min(2, Ld), dim=1).values
        sure = (top[:, 0] - top[:, -1] > 1e-3) if Ld > 1 else torch.ones(Lq, dtype=torch.bool)
        assert torch.equal(am[j][sure].long(), S.argmax(1)[sure])
