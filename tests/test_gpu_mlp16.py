"""The 16-bit MLP kernels at the edges of their tiles (32-point column blocks, 64-point waves, 256-point
blocks): a point's outputs do not depend on the call it is in, and neither do its gradients."""
import pytest
import torch

from srf_hip import mlp as hm
from test_gpu_mlp import VARIANTS, make_params, points

pytestmark = pytest.mark.gpu

COUNTS = [1, 31, 32, 33, 63, 64, 65, 255, 256, 257]


def leaves(spec, cuda, seed=21):
    ws, bs = make_params(spec, seed)
    return [None if w is None else w.to(cuda) for w in ws], [None if b is None else b.to(cuda) for b in bs]


@pytest.mark.parametrize('variant', list(VARIANTS))
@pytest.mark.parametrize('prec', ['bf16', 'fp16'])
def test_forward_of_a_prefix(cuda, variant, prec):
    spec = hm.MLPSpec(prec=prec, **VARIANTS[variant]['spec'])
    w, b = leaves(spec, cuda)
    pts, dirs = (t.to(cuda) for t in points(600, 22))
    with torch.no_grad():
        sig, rgb = hm.mlp_forward(spec, w, b, pts, dirs)
        for n in COUNTS:
            s, c = hm.mlp_forward(spec, w, b, pts[:n], dirs[:n])
            assert torch.equal(s, sig[:n]) and torch.equal(c, rgb[:n]), n


def test_a_nan_point_stays_alone(cuda):
    """The ReLUs turn NaN into 0 (as max(NaN, 0) does), and a point's column reaches no other point."""
    spec = hm.MLPSpec(prec='bf16')
    w, b = leaves(spec, cuda)
    pts, dirs = (t.to(cuda) for t in points(300, 23))
    bad = pts.clone()
    bad[70] = float('nan')
    with torch.no_grad():
        s0, c0 = hm.mlp_forward(spec, w, b, pts, dirs)
        s1, c1 = hm.mlp_forward(spec, w, b, bad, dirs)
    keep = torch.arange(300, device=cuda) != 70
    assert torch.equal(s0[keep], s1[keep]) and torch.equal(c0[keep], c1[keep])
    assert torch.isfinite(s1).all() and torch.isfinite(c1).all()


@pytest.mark.parametrize('variant', list(VARIANTS))
@pytest.mark.parametrize('n', COUNTS)
def test_gradients_of_a_prefix(cuda, variant, n):
    """Points whose outputs are not used add nothing: the parameter gradients of the first n of 600 points
    are those of a call with n points, up to the FP32 sum of at most 600 terms (600 x 2^-24 = 3.6e-5)."""
    spec = hm.MLPSpec(prec='bf16', **VARIANTS[variant]['spec'])
    w, b = leaves(spec, cuda)
    p = [t.requires_grad_(True) for t in w + b if t is not None]
    pts, dirs = (t.to(cuda) for t in points(600, 24))
    g = torch.Generator().manual_seed(25)
    gs = torch.rand(600, generator=g).to(cuda)
    gc = torch.rand(600, 3, generator=g).to(cuda)
    used = (torch.arange(600, device=cuda) < n).float()
    full = torch.autograd.grad(hm.mlp_forward(spec, w, b, pts, dirs), p, (gs * used, gc * used[:, None]))
    part = torch.autograd.grad(hm.mlp_forward(spec, w, b, pts[:n], dirs[:n]), p, (gs[:n], gc[:n]))
    for x, y in zip(part, full):
        assert (x - y).norm() <= 3.6e-5 * y.norm(), n


@pytest.mark.parametrize('variant', list(VARIANTS))
@pytest.mark.parametrize('n,cut', [(1025, 1024), (5000, 2437), (20011, 64)])
def test_gradients_add_up(cuda, variant, n, cut):
    """The weight gradients over several blocks' ranges of points: a call's are the sum of its two parts',
    up to the FP32 sum of n terms (n 2^-24)."""
    spec = hm.MLPSpec(prec='bf16', **VARIANTS[variant]['spec'])
    w, b = leaves(spec, cuda)
    p = [t.requires_grad_(True) for t in w + b if t is not None]
    pts, dirs = (t.to(cuda) for t in points(n, 26))
    g = torch.Generator().manual_seed(27)
    gs = torch.rand(n, generator=g).to(cuda)
    gc = torch.rand(n, 3, generator=g).to(cuda)

    def grads(q):
        return torch.autograd.grad(hm.mlp_forward(spec, w, b, pts[q], dirs[q]), p, (gs[q], gc[q]))
    whole, one, two = grads(slice(0, n)), grads(slice(0, cut)), grads(slice(cut, n))
    for x, y, z in zip(whole, one, two):
        assert (x - (y + z)).norm() <= n * 2.0 ** -24 * x.norm()


@pytest.mark.parametrize('variant', list(VARIANTS))
@pytest.mark.parametrize('prec', ['bf16', 'fp16'])
def test_few_points_as_many(cuda, variant, prec):
    """Inference of few points runs on 32-point waves while every block has a compute unit of its own (32,768
    points on 256), and on 64-point waves beyond: the same values, to the bit."""
    spec = hm.MLPSpec(prec=prec, **VARIANTS[variant]['spec'])
    w, b = leaves(spec, cuda)
    most = 128 * torch.cuda.get_device_properties(cuda).multi_processor_count
    pts, dirs = (t.to(cuda) for t in points(most + 300, 26))
    with torch.no_grad():
        sig, rgb = hm.mlp_forward(spec, w, b, pts, dirs)
        for n in (1, 33, 129, most - 1, most, most + 1):
            s, c = hm.mlp_forward(spec, w, b, pts[:n], dirs[:n])
            assert torch.equal(s, sig[:n]) and torch.equal(c, rgb[:n]), n
