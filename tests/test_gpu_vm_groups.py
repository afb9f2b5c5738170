"""Vector-matrix factor sampling at the edges of its groups, forward and cell-sorted backward.

A wave prepares 64 samples, packs the valid ones and reads their factors in groups of 4 or 8 lanes, up to
three quads of components a lane at once; a group width follows from the components.  Checked are sample
counts around a wave and a block, components of every group width, points on the faces of the box (whose
upper corners lie outside the factors) and, for the appearance rows, points outside it.  The bars are those
of the general tests: 1e-5 absolute against FP64 (sums of up to 72 products of N(0, 0.1) factors).
"""
import pytest
import torch

import oracle.tensorf as ot
from srf_hip import autotune, tensorf
from test_gpu_tensorf import BBOX, RES, factors, oracle_density, points, to_dev

pytestmark = pytest.mark.gpu

COMPS = [[4, 4, 4], [16, 4, 4], [16, 16, 16], [48, 12, 12], [64, 16, 32], [20, 8, 4]]


def edge_points(n, seed, outside):
    pts = points(n, BBOX, seed, outside=outside)
    g = torch.Generator().manual_seed(seed)
    # a quarter of the coordinates on a face of the box
    face = torch.where(torch.rand(n, 3, generator=g) < 0.5, BBOX[0], BBOX[1])
    return torch.where(torch.rand(n, 3, generator=g) < 0.25, face, pts)


@pytest.mark.parametrize('n', [1, 63, 65, 257, 4099])
@pytest.mark.parametrize('comps', COMPS)
def test_density_forward_groups(cuda, comps, n):
    planes, lines = factors(comps, RES, n)
    pts = edge_points(n, n + 1, 0.1)
    vol = (torch.rand(9, 10, 11, generator=torch.Generator().manual_seed(n)) < 0.5).float()
    s64, _ = oracle_density(planes, lines, pts, BBOX)
    P, L = to_dev(planes, cuda, True), to_dev(lines, cuda, True)
    box = BBOX.flatten().tolist()
    sig, valid = tensorf.vm_density(pts.to(cuda), P, L, box)
    # FP32 faces: a point on a face is inside for the comparison in FP32 that the kernel makes
    inside = ((pts >= BBOX[0]) & (pts <= BBOX[1])).all(-1)
    assert torch.equal(valid.cpu().bool(), inside)
    assert (sig.cpu().double() - s64).abs()[inside].max().item() < 1e-5 if inside.any() else True
    assert (sig.cpu()[~inside] == 0).all()
    # the alpha test packs fewer samples: the ones that stay have the same values, to the bit
    mask = tensorf.AlphaMask(vol.to(cuda), box)
    sig2, valid2 = tensorf.vm_density(pts.to(cuda), P, L, box, alpha=mask)
    keep = tensorf.alpha_mask_sample(mask, pts.to(cuda)) > 0
    assert torch.equal(valid2.bool(), valid.bool() & keep)
    assert torch.equal(sig2, torch.where(valid2.bool(), sig, torch.zeros_like(sig)))


@pytest.mark.parametrize('n', [1, 63, 65, 257, 4099])
@pytest.mark.parametrize('comps', COMPS)
def test_appearance_forward_groups(cuda, comps, n):
    planes, lines = factors(comps, RES, n)
    pts = edge_points(n, n + 2, 0.3)
    idx = torch.randperm(n, generator=torch.Generator().manual_seed(n))[:max(1, n - 3)].sort()[0].to(torch.int32)
    P, L = to_dev(planes, cuda, True), to_dev(lines, cuda, True)
    out = tensorf.vm_appearance(pts.to(cuda), P, L, BBOX.flatten().tolist(), idx=idx.to(cuda))
    ref = ot.vm_appearance_features([p.double() for p in planes], [q.double() for q in lines],
                                    ot.normalize_points(pts.double(), BBOX.double())[idx.long()])
    assert (out.cpu().double() - ref).abs().max().item() < 1e-5


# --- the cell-sorted backward: groups of max(c_p, c_line) / 4 lanes, 16 or more rows each, whose walks queue the
# texels they leave; bar: 1e-4 of the largest entry against FP64 autograd, as the general tests
def check_grads(got, ref):
    for a, b in zip(got, ref):
        scale = b.grad.abs().max().item()
        err = (a.grad.cpu().double() - b.grad).abs().max().item()
        assert err <= 1e-4 * scale, (err, scale)


@pytest.mark.parametrize('run', [0, 1, 256])
@pytest.mark.parametrize('n', [1, 17, 300, 9000])
@pytest.mark.parametrize('comps', [[4, 4, 4], [48, 12, 12], [16, 16, 16], [64, 16, 32], [20, 8, 4], [128, 64, 64]])
def test_appearance_backward_walks(cuda, comps, n, run):
    planes, lines = factors(comps, RES, n)
    pts = edge_points(n, n + 3, 0.2)
    # many rows in few cells (long runs within a cell) next to rows spread over the box
    crowd = torch.arange(n) % 3 == 0
    pts[crowd] = BBOX[0] + (BBOX[1] - BBOX[0]) * (0.41 + 0.02 * (pts[crowd] - BBOX[0]) / (BBOX[1] - BBOX[0]))
    P64 = [p.double().requires_grad_(True) for p in planes]
    L64 = [q.double().requires_grad_(True) for q in lines]
    ref = ot.vm_appearance_features(P64, L64, ot.normalize_points(pts.double(), BBOX.double()))
    gout = torch.randn(ref.shape, generator=torch.Generator().manual_seed(n))
    (ref * gout.double()).sum().backward()
    P, L = to_dev(planes, cuda, True), to_dev(lines, cuda, True)
    old = autotune.get_knob('gather_run')
    autotune.set_knob('gather_run', run)
    try:
        out = tensorf.vm_appearance(pts.to(cuda), P, L, BBOX.flatten().tolist())
        (out * gout.to(cuda)).sum().backward()
    finally:
        autotune.set_knob('gather_run', old)
    check_grads(P + L, P64 + L64)


@pytest.mark.parametrize('n', [1, 17, 300, 9000])
@pytest.mark.parametrize('comps', [[4, 4, 4], [16, 4, 4], [16, 16, 16], [24, 24, 24]])
def test_density_backward_walks(cuda, comps, n):
    planes, lines = factors(comps, RES, n)
    pts = edge_points(n, n + 4, 0.1)
    gs = torch.randn(n, generator=torch.Generator().manual_seed(n))
    gs[::5] = 0  # rows without a gradient are left out of the orders
    P64 = [p.double().requires_grad_(True) for p in planes]
    L64 = [q.double().requires_grad_(True) for q in lines]
    s64, _ = oracle_density(P64, L64, pts, BBOX, kind='SoftPlus', offset=-1.0)
    (s64 * gs.double()).sum().backward()
    P, L = to_dev(planes, cuda, True), to_dev(lines, cuda, True)
    sig, _ = tensorf.vm_density(pts.to(cuda), P, L, BBOX.flatten().tolist(), predictor=tensorf.predictor_code('SoftPlus'),
                                offset=-1.0)
    (sig * gs.to(cuda)).sum().backward()
    check_grads(P + L, P64 + L64)
