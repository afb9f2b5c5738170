"""Sums of the colour network's gradients that are not ordinary numbers."""
import pytest
import torch
import torch.nn.functional as F

from srf_hip import color
from test_gpu_color import params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('value', [float('inf'), -float('inf'), 3e38, float('nan')])
@pytest.mark.parametrize('prec', ['fp32', 'bf16', 'bf16_split'])
def test_bias_sums_past_an_infinity(cuda, prec, value):
    """The last layer's bias gradient of one channel is the FP32 sum of its rows: infinite (not NaN) with one
    infinite upstream gradient among the first rows, or where finite ones overflow (rgb (1 - rgb) 3e38 of 2,000
    rows), NaN with a NaN.  The other channels' sums stay finite."""
    c = dict(C=72, Lf=0, Lv=0, view=True)
    n = 2000
    g = torch.Generator().manual_seed(40)
    prm = [t.to(cuda).requires_grad_(True) for t in params(c, 41)]
    app = (torch.randn(n, c['C'], generator=g) * 0.3).to(cuda)
    vd = F.normalize(torch.randn(n, 3, generator=g), dim=-1).to(cuda)
    gout = torch.randn(n, 3, generator=g).to(cuda)
    if value == 3e38:
        gout[:, 1] = value
    else:
        gout[3, 1] = value
    rgb = color.color_forward(color.ColorSpec(n_features=c['C'], prec=prec), app, prm[0], prm[1:], view_dirs=vd)
    db3 = torch.autograd.grad(rgb, prm[6], gout)[0].cpu()
    assert torch.isfinite(db3[[0, 2]]).all()
    want = torch.tensor(float('inf') if value == 3e38 else value)
    assert torch.equal(db3[1], want) or (want.isnan() and db3[1].isnan())
