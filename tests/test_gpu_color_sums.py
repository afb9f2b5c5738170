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


@pytest.mark.parametrize('prec,bar', [('fp32', 8.6e-7), ('bf16', 6.7e-7), ('bf16_split', 6.7e-7)])
def test_weight_gradients_of_many_rows(cuda, prec, bar):
    """The weight gradients of a call are the FP64 sum of those of its slices of 256 rows: a wave's running FP32
    sum ends after 1,024 points.  300,007 rows of the 72-component network, random signs, norm of the difference
    over the norm, largest over the weights: 6.1e-7 (FP32) and 4.1e-7 (BF16 modes), against 1.2e-6 and 1.1e-6 with
    sums of 16,384 points; the bars are the geometric means."""
    c = dict(C=72, Lf=0, Lv=0, view=True)
    n, part = 300007, 256
    g = torch.Generator(device=cuda).manual_seed(42)
    prm = [t.to(cuda).requires_grad_(True) for t in params(c, 43)]
    app = torch.randn(n, c['C'], generator=g, device=cuda) * 0.3
    vd = F.normalize(torch.randn(n, 3, generator=g, device=cuda), dim=-1)
    gout = torch.randn(n, 3, generator=g, device=cuda) * 0.1
    spec = color.ColorSpec(n_features=c['C'], prec=prec)
    leaves = [prm[i] for i in (0, 1, 3, 5)]

    def grads(q):
        rgb = color.color_forward(spec, app[q], prm[0], prm[1:], view_dirs=vd[q])
        return torch.autograd.grad(rgb, leaves, gout[q])
    ref = [torch.zeros_like(t, dtype=torch.float64) for t in leaves]
    for o in range(0, n, part):
        for r, t in zip(ref, grads(slice(o, o + part))):
            r += t.double()
    for x, r in zip(grads(slice(0, n)), ref):
        assert ((x.double() - r).norm() / r.norm()).item() < bar
