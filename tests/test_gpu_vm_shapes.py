"""Vector-matrix factors of unequal shapes, forward and cell-sorted backward: planes and lines without components,
of one texel, and lines of another length than the planes have texels along their axis.  An order of the backward
serves its own plane and another plane's line, so each of these meets both with and without a partner.  The bars are
those of the general tests: 1e-5 absolute against FP64, gradients 1e-4 of the largest entry."""
import pytest
import torch

import oracle.tensorf as ot
from srf_hip import tensorf
from test_gpu_tensorf import BBOX, oracle_density, to_dev
from test_gpu_vm_groups import check_grads, edge_points

pytestmark = pytest.mark.gpu

# components, (rows, columns) of the planes, lengths of the lines
SHAPES = {
    'first_plane': ([16, 0, 0], [(36, 40), (30, 40), (30, 36)], [30, 36, 40]),
    'second_plane': ([0, 8, 0], [(36, 40), (30, 40), (30, 36)], [30, 36, 40]),
    'third_plane': ([0, 0, 20], [(36, 40), (30, 40), (30, 36)], [30, 36, 40]),
    'without_first': ([0, 12, 48], [(36, 40), (30, 40), (30, 36)], [30, 36, 40]),
    'without_second': ([4, 0, 16], [(36, 40), (30, 40), (30, 36)], [30, 36, 40]),
    'without_third': ([48, 12, 0], [(36, 40), (30, 40), (30, 36)], [30, 36, 40]),
    'one_texel': ([4, 8, 4], [(1, 1), (1, 1), (1, 1)], [1, 1, 1]),
    'one_row': ([8, 4, 12], [(1, 40), (30, 1), (1, 36)], [30, 1, 40]),
    'two_texels': ([8, 8, 8], [(2, 2), (2, 2), (2, 2)], [2, 2, 2]),
    'longer_lines': ([16, 16, 16], [(9, 10), (8, 10), (8, 9)], [83, 97, 101]),
    'shorter_lines': ([20, 4, 8], [(36, 40), (30, 40), (30, 36)], [3, 2, 1]),
}


def factors(shape, seed):
    comps, sizes, lengths = SHAPES[shape]
    g = torch.Generator().manual_seed(seed)
    return ([0.1 * torch.randn(1, c, *hw, generator=g) for c, hw in zip(comps, sizes)],
            [0.1 * torch.randn(1, c, n, 1, generator=g) for c, n in zip(comps, lengths)])


def leaves(planes, lines):
    return [p.double().requires_grad_(True) for p in planes], [q.double().requires_grad_(True) for q in lines]


def check(P, L, P64, L64):
    pairs = [(a, b) for a, b in zip(P + L, P64 + L64) if b.numel() and b.grad.abs().max() > 0]
    assert pairs
    check_grads(*zip(*pairs))
    for a, b in zip(P + L, P64 + L64):
        assert b.numel() == 0 or torch.isfinite(a.grad).all()


@pytest.mark.parametrize('n', [1, 700, 9000])
@pytest.mark.parametrize('shape', list(SHAPES))
def test_density(cuda, shape, n):
    planes, lines = factors(shape, n)
    pts = edge_points(n, n + 1, 0.1)
    if n == 1:
        pts = BBOX.mean(0, keepdim=True)
    gs = torch.randn(n, generator=torch.Generator().manual_seed(n))
    P64, L64 = leaves(planes, lines)
    s64, _ = oracle_density(P64, L64, pts, BBOX, kind='SoftPlus', offset=-1.0)
    (s64 * gs.double()).sum().backward()
    P, L = to_dev(planes, cuda, True), to_dev(lines, cuda, True)
    sig, _ = tensorf.vm_density(pts.to(cuda), P, L, BBOX.flatten().tolist(), predictor=tensorf.predictor_code('SoftPlus'),
                                offset=-1.0)
    inside = ((pts >= BBOX[0]) & (pts <= BBOX[1])).all(-1)
    assert (sig.detach().cpu().double() - s64.detach()).abs()[inside].max().item() < 1e-5
    (sig * gs.to(cuda)).sum().backward()
    check(P, L, P64, L64)


@pytest.mark.parametrize('n', [1, 700, 9000])
@pytest.mark.parametrize('shape', list(SHAPES))
def test_appearance(cuda, shape, n):
    planes, lines = factors(shape, n)
    pts = edge_points(n, n + 2, 0.2)
    if n == 1:
        pts = BBOX.mean(0, keepdim=True)
    P64, L64 = leaves(planes, lines)
    ref = ot.vm_appearance_features(P64, L64, ot.normalize_points(pts.double(), BBOX.double()))
    gout = torch.randn(ref.shape, generator=torch.Generator().manual_seed(n))
    (ref * gout.double()).sum().backward()
    P, L = to_dev(planes, cuda, True), to_dev(lines, cuda, True)
    out = tensorf.vm_appearance(pts.to(cuda), P, L, BBOX.flatten().tolist())
    assert (out.detach().cpu().double() - ref.detach()).abs().max().item() < 1e-5
    (out * gout.to(cuda)).sum().backward()
    check(P, L, P64, L64)
