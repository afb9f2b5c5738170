"""Weight gradients of the colour network at the sizes where their kernel can go wrong.

A block reduces one of the four products over a range of points, whose length follows from the number
of rows (or the device-side count) and the products' numbers of 16-row tiles; waves take row and column
tiles by those numbers.  Checked are

* every number of column tiles against FP64 autograd of the oracle, on a few hundred rows whose
  pre-activations the oracle keeps 1e-4 away from zero (no ReLU can differ), to 1e-4 of the largest entry
  (the FP32 bar of the colour network);
* many rows against the sum over slices of 4,096 of them: each row's products are the same, so the two are
  FP32 sums in different orders of at most 40,000 terms, each about 2^-24 of the running sum apart; with
  random signs that stays below 2^-24 sqrt(40,000) = 1.2e-5 of the largest entry's own scale: 1e-4;
* a device-side count against the prefix of its rows, to the same bound.
"""
import pytest
import torch
import torch.nn.functional as F

from srf_hip import autotune, color
from test_gpu_color import _pe, oracle, params

pytestmark = pytest.mark.gpu

# components, PE levels -> 16-row tiles of the first layer's and the basis's inputs (FP32 / BF16 modes)
SHAPES = [dict(C=4, Lf=0, Lv=0, view=False), dict(C=20, Lf=0, Lv=1, view=True), dict(C=132, Lf=1, Lv=1, view=True),
          dict(C=144, Lf=2, Lv=0, view=True), dict(C=160, Lf=2, Lv=3, view=True), dict(C=244, Lf=3, Lv=1, view=True),
          dict(C=256, Lf=3, Lv=4, view=True)]


def grads(spec, prm, app, vd, gout, cuda, count=None):
    pd = [t.to(cuda).requires_grad_(True) for t in prm]
    rgb = color.color_forward(spec, app, pd[0], pd[1:], view_dirs=vd if spec.use_view_dirs else None, count=count)
    n = app.shape[0] if count is None else int(count.item())
    (rgb[:n] * gout[:n]).sum().backward()
    return [p.grad.double().cpu() for p in pd]


def close(a, b, tol=1e-4):
    for i, (x, y) in enumerate(zip(a, b)):
        e = (x - y).abs().max().item() / y.abs().max().item()
        assert e < tol, (i, e)


def spec_of(c, prec):
    return color.ColorSpec(n_features=c['C'], features_pe=c['Lf'], use_view_dirs=c['view'], views_pe=c['Lv'], prec=prec)


@pytest.mark.parametrize('prec', ['fp32', 'bf16_split'])
@pytest.mark.parametrize('i', range(len(SHAPES)))
def test_column_tiles(cuda, i, prec):
    c = SHAPES[i]
    g = torch.Generator().manual_seed(10 + i)
    prm = params(c, 20 + i)
    app = torch.randn(3000, c['C'], generator=g) * 0.3
    vd = F.normalize(torch.randn(3000, 3, generator=g), dim=-1)
    basis, w1, b1, w2, b2, _, _ = [t.double() for t in prm]
    x1 = _pe(app.double() @ basis.T, c['Lf'])
    if c['view']:
        x1 = torch.cat([x1, _pe(vd.double(), c['Lv'])], -1)
    z1 = x1 @ w1.T + b1
    z2 = z1.clamp_min(0) @ w2.T + b2
    keep = (torch.cat([z1, z2], -1).abs().min(-1)[0] > 1e-4).nonzero()[:, 0]
    keep = keep[:[1, 17, 255, 256, 257, 511, 513][i]]
    app, vd = app[keep], vd[keep]
    gout = torch.randn(len(keep), 3, generator=g)
    p64 = [t.double().requires_grad_(True) for t in prm]
    (oracle(c, p64, app.double(), vd.double()) * gout.double()).sum().backward()
    got = grads(spec_of(c, prec), prm, app.to(cuda), vd.to(cuda), gout.to(cuda), cuda)
    close(got, [p.grad for p in p64])


@pytest.mark.parametrize('tuned', [0, 2048])
@pytest.mark.parametrize('prec', ['fp32', 'bf16_split'])
def test_many_rows_and_counts(cuda, prec, tuned):
    c = dict(C=72, Lf=1, Lv=0, view=True)
    n, part = 40000, 4096
    g = torch.Generator().manual_seed(5)
    prm = params(c, 6)
    app = (torch.randn(n, c['C'], generator=g) * 0.3).to(cuda)
    vd = F.normalize(torch.randn(n, 3, generator=g), dim=-1).to(cuda)
    gout = torch.randn(n, 3, generator=g).to(cuda)
    spec = spec_of(c, prec)
    old = autotune.get_knob('color_dw_chunk')
    autotune.set_knob('color_dw_chunk', tuned)
    try:
        whole = grads(spec, prm, app, vd, gout, cuda)
        sums = [torch.zeros_like(t) for t in whole]
        for o in range(0, n, part):
            for s, t in zip(sums, grads(spec, prm, app[o:o + part], vd[o:o + part], gout[o:o + part], cuda)):
                s += t
        close(whole, sums)
        for m in (1, 300, 20001):
            count = torch.tensor([m], dtype=torch.int32, device=cuda)
            close(grads(spec, prm, app, vd, gout, cuda, count), grads(spec, prm, app[:m], vd[:m], gout[:m], cuda))
    finally:
        autotune.set_knob('color_dw_chunk', old)


# --- every number of column tiles of the first layer (1 .. 15) and of the basis (1 .. 16): D1 inputs by the basis
# outputs and encodings, C components; bar and rows as in test_column_tiles
WIDTHS = [(4, 14, 0, False), (16, 27, 0, True), (33 * 4, 20, 1, False), (48, 16, 1, False), (200, 27, 1, False),
          (80, 16, 2, False), (176, 32, 1, True), (96, 27, 2, False), (112, 29, 2, False), (240, 24, 2, False),
          (208, 24, 3, False), (224, 27, 3, False), (60, 29, 3, False), (64, 32, 3, False), (256, 26, 4, False)]


@pytest.mark.parametrize('prec', ['fp32', 'bf16_split'])
@pytest.mark.parametrize('i', range(len(WIDTHS)))
def test_every_width(cuda, i, prec):
    C, nb, Lf, view = WIDTHS[i]
    spec = color.ColorSpec(n_features=C, basis_dim=nb, features_pe=Lf, use_view_dirs=view, views_pe=0, prec=prec)
    if not spec.supported():
        pytest.skip('more than 240 inputs once padded to the BF16 k-unit')
    g = torch.Generator().manual_seed(60 + i)
    d1 = nb * (2 * Lf + 1) + (3 if view else 0)
    lin = lambda o, k: ((torch.rand(o, k, generator=g) * 2 - 1) / k ** 0.5, (torch.rand(o, generator=g) * 2 - 1) * 0.1)
    prm = [(torch.rand(nb, C, generator=g) * 2 - 1) / C ** 0.5, *lin(128, d1), *lin(128, 128), *lin(3, 128)]
    app = torch.randn(2600, C, generator=g) * 0.3
    vd = F.normalize(torch.randn(2600, 3, generator=g), dim=-1)
    basis, w1, b1, w2, b2, _, _ = [t.double() for t in prm]
    x1 = _pe(app.double() @ basis.T, Lf)
    if view:
        x1 = torch.cat([x1, vd.double()], -1)
    z1 = x1 @ w1.T + b1
    z2 = z1.clamp_min(0) @ w2.T + b2
    keep = (torch.cat([z1, z2], -1).abs().min(-1)[0] > 1e-4).nonzero()[:, 0][:600]
    app, vd = app[keep], vd[keep]
    gout = torch.randn(len(keep), 3, generator=g)
    p64 = [t.double().requires_grad_(True) for t in prm]
    (oracle(dict(Lf=Lf, Lv=0, view=view), p64, app.double(), vd.double()) * gout.double()).sum().backward()
    got = grads(spec, prm, app.to(cuda), vd.to(cuda), gout.to(cuda), cuda)
    close(got, [p.grad for p in p64])
