"""fp8 scoring with per-token scales on the two-workgroup column blocks
(4 x 4, 4 x 6), against the oracle on the dequantised values (2e-3: the
sums are fp32) and against the 8 x 4 block (1e-5: another order of a query's
column sum)."""

import numpy as np
import pytest
import torch

import lik_oracle as O
from conftest import rel_err
from late_interaction_kernels._lib import launch_options

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [128, 96])
@pytest.mark.parametrize("Nq,Lq,Nd,Ld", [(24, 32, 9, 33), (32, 24, 5, 1030), (17, 30, 40, 64), (40, 32, 3, 31)])
def test_row_scales(Nq, Lq, Nd, Ld, d):
    from late_interaction_kernels.fp8 import maxsim_inference_fp8, quantize_fp8_per_token

    g = torch.Generator().manual_seed(Nq + Ld)
    Qf, sq = quantize_fp8_per_token(torch.randn(Nq, Lq, d, generator=g).cuda())
    Df, sd = quantize_fp8_per_token((torch.randn(Nd, Ld, d, generator=g) * torch.rand(Nd, Ld, 1, generator=g)).cuda())
    dm = torch.arange(Ld)[None] < torch.randint(1, Ld + 1, (Nd,), generator=g)[:, None]
    dm[0] = torch.rand(Ld, generator=g) > 0.3  # holes: the masked launch
    dm[1] = False
    # scales of rows that are not scored must not matter, whatever they are
    off = (~dm).nonzero()
    bad = torch.tensor([float("nan"), float("inf"), 0.0, -1.0])
    sdx = sd.clone()
    sdx[off[:, 0], off[:, 1]] = bad[torch.arange(len(off)) % 4].cuda()
    sdx[2, 0] = 0.0  # a scored row may have scale 0
    dm[2, 0] = True
    dmc = dm.cuda()
    got = maxsim_inference_fp8(Qf, Df, scale_Q=sq, scale_D=sdx, d_mask=dmc).cpu().numpy()
    Qd = Qf.float().cpu().numpy() * sq.cpu().numpy()[..., None]
    Dd = Df.float().cpu().numpy() * np.where(dm.numpy(), sdx.cpu().numpy(), 1.0)[..., None]
    assert rel_err(got, O.maxsim(Qd, Dd, None, dm.numpy())) < 2e-3
    for cfg in ((8, 4), (4, 4), (4, 6)):
        with launch_options(cfg=cfg):
            forced = maxsim_inference_fp8(Qf, Df, scale_Q=sq, scale_D=sdx, d_mask=dmc).cpu().numpy()
        assert rel_err(forced, got) < 1e-5
