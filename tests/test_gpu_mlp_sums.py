"""FP32 sums of the MLP's weight gradients over many points.

A block's running sum ends after a few thousand points, however many points the block reduces: the gradients
of a call are the FP64 sum of the gradients of its slices of 256 points up to a bar that sums over whole
blocks of one round do not meet.  262,144 points, norm of the difference over the norm, largest over the
layers' weights: 1.7e-7 (FP32), 1.8e-7 (split BF16) and 1.4e-7 (BF16) with the short sums, 3.9e-7, 4.2e-7 and
2.8e-7 with those of whole blocks; the bars are the geometric means of the two.
"""
import pytest
import torch

from srf_hip import autotune
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


@pytest.mark.parametrize('tuned', [0, 2048, 8192])
@pytest.mark.parametrize('prec,n', [('bf16', 1088), ('bf16', 20011), ('bf16', 300007), ('fp32', 60011), ('bf16_split', 93391)])
@pytest.mark.parametrize('variant', list(VARIANTS))
def test_points_at_the_ends_of_ranges(cuda, variant, prec, n, tuned):
    """Only the points on both sides of every multiple of 64 (1,024 where there are many), where the blocks'
    ranges and their segments end, and the last one have upstream gradients: the parameter gradients are those of
    a call with these m points alone, up to the FP32 sum of m terms (m 2^-24; a point lost or counted twice is
    1 / m)."""
    step = 1024 if n > 100000 else 64
    ends = torch.arange(step, n, step)
    ends = torch.cat([ends - 1, ends, torch.tensor([0, n - 1])]).unique()
    m = len(ends)
    spec = hm.MLPSpec(prec=prec, **VARIANTS[variant]['spec'])
    ws, bs = make_params(spec, 53)
    w = [None if t is None else t.to(cuda).requires_grad_(True) for t in ws]
    b = [None if t is None else t.to(cuda).requires_grad_(True) for t in bs]
    p = [t for t in w + b if t is not None]
    pts, dirs = (t.to(cuda) for t in points(n, 54))
    g = torch.Generator().manual_seed(55)
    gs, gc = torch.zeros(n), torch.zeros(n, 3)
    gs[ends] = torch.rand(m, generator=g) + 0.5
    gc[ends] = torch.rand(m, 3, generator=g) + 0.5
    gs, gc, ends = gs.to(cuda), gc.to(cuda), ends.to(cuda)
    old = autotune.get_knob('dw_chunk')
    autotune.set_knob('dw_chunk', tuned)
    try:
        whole = torch.autograd.grad(hm.mlp_forward(spec, w, b, pts, dirs), p, (gs, gc))
    finally:
        autotune.set_knob('dw_chunk', old)
    few = torch.autograd.grad(hm.mlp_forward(spec, w, b, pts[ends], dirs[ends]), p, (gs[ends], gc[ends]))
    for x, y in zip(whole, few):
        assert (x - y).norm() <= m * 2.0 ** -24 * y.norm()
