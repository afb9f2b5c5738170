"""FP32 sums of the MLP's weight gradients over many points.

A block's running sum ends after a few thousand points, however many points the block reduces: the gradients
of a call are the FP64 sum of the gradients of its slices of 256 points up to a bar that sums over whole
blocks of one round do not meet.  262,144 points, norm of the difference over the norm, largest over the
layers' weights: 1.7e-7 (FP32), 1.8e-7 (split BF16) and 1.4e-7 (BF16) with the short sums, 3.9e-7, 4.2e-7 and
2.8e-7 with those of whole blocks; the bars are the geometric means of the two.
"""
import pytest
import torch

from srf_hip import mlp as hm
from test_gpu_mlp import VARIANTS, make_params, points

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('prec,bar', [('fp32', 2.6e-7), ('bf16_split', 2.7e-7), ('bf16', 2.0e-7)])
def test_weight_gradients_of_many_points(cuda, prec, bar):
    n, part = 262144, 256
    spec = hm.MLPSpec(prec=prec, **VARIANTS['main']['spec'])
    ws, bs = make_params(spec, 50)
    w = [t.to(cuda).requires_grad_(True) for t in ws]
    b = [t.to(cuda) for t in bs]
    pts, dirs = (t.to(cuda) for t in points(n, 51))
    g = torch.Generator().manual_seed(52)
    gs = (torch.rand(n, generator=g) * 0.15 - 0.05).to(cuda)
    gc = (torch.rand(n, 3, generator=g) - 0.3).to(cuda)

    def grads(q):
        return torch.autograd.grad(hm.mlp_forward(spec, w, b, pts[q], dirs[q]), w, (gs[q], gc[q]))
    ref = [torch.zeros_like(t, dtype=torch.float64) for t in w]
    for o in range(0, n, part):
        for r, t in zip(ref, grads(slice(o, o + part))):
            r += t.double()
    for name, x, r in zip(hm.PARAM_NAMES, grads(slice(0, n)), ref):
        err = ((x.double() - r).norm() / r.norm()).item()
        assert err < bar, (name, err)
