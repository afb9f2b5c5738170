"""Timed cases of the rendering hot path, through the package's public entry points.

The kinds follow the two models' steps:

  mlp         one NeRF MLP over rays x samples (``mlp_forward_rays``): inference, or forward and
              backward into the parameter gradients
  march       NeRF sampling and compositing around the MLPs: stratified depths, coarse weights, inverse-CDF
              fine depths, fine compositing and its backward
  density     TensoRF vector-matrix density of every sample, forward and backward
  appearance  TensoRF vector-matrix appearance rows of the surface samples, forward and backward
  color       TensoRF basis and colour network of the surface rows, forward and backward
  shade       TensoRF compositing: weights, surface list, colour sum, and the backward
  render      one whole evaluation call of the Simple-NeRF model

``exact`` restates each in float64 with plain torch.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch
import torch.nn.functional as F

_PKG = str(Path(__file__).resolve().parent.parent / 'simple-rf_amd')
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from models.ModelFactory02 import get_model  # noqa: E402
from srf_hip import color, compositing, configs, mlp, sampling, tensorf  # noqa: E402

DEV = 'cuda'
BBOX = (-1.5, -1.67, -1.0, 1.5, 1.67, 1.0)   # the TensoRF configuration's box (NDC)
RENDER_KEYS = ('rgb', 'acc', 'depth', 'depth_ndc')


def listed():
    return [
        # a preview tile of the viewer: the smallest useful MLP call, launches and latency count
        dict(name='nerf_preview', kind='mlp', variant='main', prec='bf16', train=False, rays=256, samples=64),
        # fine pass of an evaluation chunk
        dict(name='nerf_eval_fine', kind='mlp', variant='main', prec='bf16', train=False, rays=16384, samples=192),
        # coarse and fine passes of the training step on 4096 rays
        dict(name='nerf_coarse_train', kind='mlp', variant='main', prec='bf16', train=True, rays=4096, samples=64),
        dict(name='nerf_fine_train', kind='mlp', variant='main', prec='bf16', train=True, rays=4096, samples=192),
        # the points-augmented model at FP32-level rounding, an odd batch with an odd sample count
        dict(name='nerf_points_split_train', kind='mlp', variant='points', prec='bf16_split', train=True, rays=1531,
             samples=61),
        # what surrounds the MLPs in the same training step
        dict(name='nerf_march_train', kind='march', rays=4096, coarse=64, fine=128),
        # the 300^2 TensoRF step: 8192 rays x 443 samples, 64^3 occupancy mask
        dict(name='tensorf_density_train', kind='density', rays=8192, samples=443, grid=300, comps=16, mask=True),
        dict(name='tensorf_appearance_train', kind='appearance', rays=8192, samples=443, grid=300, comps=48),
        dict(name='tensorf_color_train', kind='color', rows=1400000, features=144, features_pe=2, prec='fp32'),
        # the shipped Simple-TensoRF configuration's colour network (72 features, no encoding) on BF16 operands
        dict(name='tensorf_color_bf16_train', kind='color', rows=300007, features=72, features_pe=0, prec='bf16'),
        dict(name='tensorf_shade_train', kind='shade', rays=8192, samples=443),
        # a whole evaluation call: coarse 64 + fine 192 samples, one chunk of the reference's 4096 rays
        dict(name='nerf_render', kind='render', prec='bf16', rays=4096),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(['mlp', 'mlp', 'mlp', 'march', 'density', 'appearance', 'color', 'color', 'shade', 'render'])
    if kind == 'mlp':
        prec = rng.choice(['bf16', 'bf16', 'bf16', 'bf16_split', 'fp32', 'fp16'])
        train = prec != 'fp16' and rng.random() < 0.6
        # points: at most the listed calls' time in the slower precisions
        most = {'bf16': 4096 * 192, 'fp16': 4096 * 192, 'bf16_split': 1 << 18, 'fp32': 1 << 16}[prec]
        samples = rng.randint(24, 192)
        return dict(kind='mlp', variant=rng.choice(['main', 'points', 'views']), prec=prec, train=train,
                    rays=_logint(rng, 64, most // samples), samples=samples)
    if kind == 'march':
        return dict(kind='march', rays=_logint(rng, 128, 4096), coarse=rng.randint(16, 64), fine=rng.randint(16, 128))
    if kind == 'density':
        return dict(kind='density', rays=_logint(rng, 256, 8192), samples=rng.randint(100, 443),
                    grid=rng.randint(64, 300), comps=rng.choice([4, 8, 16]), mask=rng.random() < 0.5)
    if kind == 'appearance':
        return dict(kind='appearance', rays=_logint(rng, 256, 8192), samples=rng.randint(100, 443),
                    grid=rng.randint(64, 300), comps=rng.choice([12, 24, 48]))
    if kind == 'color':
        return dict(kind='color', rows=_logint(rng, 2000, 1000000), features=rng.choice([36, 72, 144]),
                    features_pe=rng.choice([0, 2]), prec=rng.choice(['fp32', 'bf16', 'bf16_split']))
    if kind == 'shade':
        return dict(kind='shade', rays=_logint(rng, 256, 8192), samples=rng.randint(100, 443))
    return dict(kind='render', prec='bf16', rays=_logint(rng, 128, 4096))


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _rand(g, *shape, lo=0.0, hi=1.0):
    return torch.rand(shape, generator=g, device=DEV) * (hi - lo) + lo


def _randn(g, *shape, scale=1.0):
    return torch.randn(shape, generator=g, device=DEV) * scale


def _linear(g, out, inp, gain=1.0):
    """Weight and bias of a torch.nn.Linear as the models initialise it (Xavier uniform, small biases)."""
    a = gain * math.sqrt(6.0 / (inp + out))
    return _rand(g, out, inp, lo=-a, hi=a), _rand(g, out, lo=-0.05, hi=0.05)


def _rays(g, n):
    """Forward-facing rays in normalised device coordinates (z from -1 to 1 over [0, 1]), their world
    rays and view directions."""
    o = torch.cat([_rand(g, n, 2, lo=-0.9, hi=0.9), torch.full((n, 1), -1.0, device=DEV)], 1)
    d = torch.cat([_randn(g, n, 2, scale=0.15), torch.full((n, 1), 2.0, device=DEV)], 1)
    wo = _randn(g, n, 3, scale=0.05)
    wd = torch.cat([_rand(g, n, 2, lo=-0.6, hi=0.6), torch.full((n, 1), -1.0, device=DEV)], 1)
    return o, d, wo, wd, wd / wd.norm(dim=-1, keepdim=True)


def _sorted_z(g, n, s):
    """Stratified depths in [0, 1)."""
    return ((torch.arange(s, device=DEV) + _rand(g, n, s)) / s).contiguous()


def _spec(case):
    v = case['variant']
    return mlp.MLPSpec(sigma_pe_degree=3 if v == 'points' else None, view_dependent=v != 'views', prec=case['prec'])


def _prepare_mlp(case, seed):
    g = _gen(seed)
    spec = _spec(case)
    n, s = case['rays'], case['samples']
    weights, biases = [], []
    for shapes in spec.param_shapes():
        w, b = (None, None) if shapes is None else _linear(g, *shapes[0])
        weights.append(w)
        biases.append(b)
    weights[9][0] *= 4.0    # densities of a scene under training: part of the samples opaque
    o, d, _, _, vd = _rays(g, n)
    st = dict(case=case, spec=spec, weights=weights, biases=biases, o=o, d=d, z=_sorted_z(g, n, s),
              vd=vd if spec.view_dependent else None, noise=None)
    if case['train']:
        for t in weights + biases:
            if t is not None:
                t.requires_grad_(True)
        st['noise'] = _randn(g, n, s)
        # what a rendering loss sends back: a ray's residual, weighted by its samples' share of the pixel
        at = _rand(g, n, 1, lo=0.2, hi=0.9)
        share = torch.softmax(-((st['z'] - at) * 12.0) ** 2, 1)
        res = _rand(g, n, 3, lo=-0.3, hi=0.7) / n
        st['gr'] = (share[..., None] * res[:, None]).reshape(n * s, 3).contiguous()
        st['gs'] = (share * _rand(g, n, 1, lo=-0.05, hi=0.1) / n).reshape(n * s).contiguous()
    return st


def _prepare_march(case, seed):
    g = _gen(seed)
    n, c, f = case['rays'], case['coarse'], case['fine']
    o, d, wo, wd, _ = _rays(g, n)

    def field(s):   # a soft surface in front of empty space, and some fog
        k = torch.arange(s, device=DEV) / s
        at = _rand(g, n, 1, lo=0.2, hi=0.9)
        return (40.0 * torch.sigmoid((k - at) * 60.0) * _rand(g, n, s) + _rand(g, n, s)).contiguous()
    return dict(case=case, n=n, wo=wo, wd=wd, d=d, u=_rand(g, n, c), uf=_rand(g, n, f), sigma_c=field(c),
                rgb_c=_rand(g, n, c, 3), sigma_f=field(c + f).requires_grad_(True),
                rgb_f=_rand(g, n, c + f, 3).requires_grad_(True), g_rgb=_randn(g, n, 3, scale=1.0 / n),
                g_depth=_randn(g, n, scale=0.1 / n))


def _occupancy(g, size=64):
    """Blobs that fill 40 % of a size^3 volume."""
    v = F.interpolate(_rand(g, 1, 1, 9, 9, 9), size=(size,) * 3, mode='trilinear', align_corners=True)[0, 0]
    return (v > v.flatten().quantile(0.6)).float()


def _vm(g, grid, comps):
    planes = [tensorf.texel_major_param(comps, grid, grid, _randn(g, 1, comps, grid, grid, scale=0.3), DEV)
              for _ in range(3)]
    lines = [tensorf.texel_major_param(comps, grid, 1, _randn(g, 1, comps, grid, 1, scale=0.3), DEV) for _ in range(3)]
    return planes, lines


def _samples(g, case):
    o, d, _, _, _ = _rays(g, case['rays'])
    z = _sorted_z(g, case['rays'], case['samples'])
    return (o[:, None] + d[:, None] * z[..., None]).reshape(-1, 3).contiguous()


def _prepare_density(case, seed):
    g = _gen(seed)
    planes, lines = _vm(g, case['grid'], case['comps'])
    vol = _occupancy(g)
    pts = _samples(g, case)
    return dict(case=case, planes=planes, lines=lines, pts=pts, vol=vol if case['mask'] else None,
                mask=tensorf.AlphaMask(vol, BBOX) if case['mask'] else None,
                gs=_randn(g, pts.shape[0], scale=1e-2 / case['rays']))


def _prepare_appearance(case, seed):
    g = _gen(seed)
    planes, lines = _vm(g, case['grid'], case['comps'])
    vol = _occupancy(g)
    pts = _samples(g, case)
    lo = torch.tensor(BBOX[:3], device=DEV)
    hi = torch.tensor(BBOX[3:], device=DEV)
    vox = ((pts - lo) / (hi - lo) * 63.0).round().long().clamp(0, 63)
    # the surface list: 40 % of the samples, those in occupied voxels first
    hit = vol[vox[:, 2], vox[:, 1], vox[:, 0]] + 0.1 * _rand(g, pts.shape[0])
    idx = hit.topk(int(0.4 * pts.shape[0])).indices.sort().values.int().contiguous()
    return dict(case=case, planes=planes, lines=lines, pts=pts, idx=idx,
                ga=_randn(g, idx.shape[0], 3 * case['comps'], scale=1e-2 / case['rays']))


def _prepare_color(case, seed):
    g = _gen(seed)
    m, f, pe = case['rows'], case['features'], case['features_pe']
    views_pe = pe
    spec = color.ColorSpec(n_features=f, basis_dim=27, features_pe=pe, views_pe=views_pe, prec=case['prec'])
    d_in = 27 * (2 * pe + 1) + 3 * (2 * views_pe + 1)
    basis = _linear(g, 27, f)[0]
    w1, b1 = _linear(g, 128, d_in)
    w2, b2 = _linear(g, 128, 128)
    w3, b3 = _linear(g, 3, 128)
    per_ray = 443                              # samples of a ray; about 40 % of them are surface samples
    n = max(1, m // 177 + 1)
    keep = torch.rand((n * per_ray,), generator=g, device=DEV).topk(m).indices
    idx = keep.sort().values.int().contiguous()
    vd = F.normalize(_randn(g, n, 3), dim=-1)
    params = [t.requires_grad_(True) for t in (basis, w1, b1, w2, b2, w3, b3)]
    return dict(case=case, spec=spec, app=_randn(g, m, f, scale=0.3).requires_grad_(True), params=params, idx=idx,
                per_ray=per_ray, vd=vd, g_rgb=_randn(g, m, 3, scale=0.1 / n))


def _prepare_shade(case, seed):
    g = _gen(seed)
    n, s = case['rays'], case['samples']
    _, d, wo, wd, _ = _rays(g, n)
    k = torch.arange(s, device=DEV) / s
    at = _rand(g, n, 1, lo=0.1, hi=0.9)
    sigma = F.relu(_randn(g, n, s) + 3.0 * torch.sigmoid((k - at) * 40.0) - 1.0)
    return dict(case=case, wo=wo, wd=wd, d=d, z=_sorted_z(g, n, s), sigma=sigma.requires_grad_(True),
                rgb=_rand(g, n, s, 3).requires_grad_(True), g_rgb=_randn(g, n, 3, scale=1.0 / n),
                g_depth=_randn(g, n, scale=0.1 / n))


def _prepare_render(case, seed):
    g = _gen(seed)
    cfg = configs.simple_nerf_configs(precision=case['prec'], augmentations=False)
    mc = configs.model_configs()
    model = get_model(cfg, model_configs=mc).to(DEV).eval()
    with torch.no_grad():
        for net in (model.coarse_model, model.fine_model):
            for lin in net.modules():
                if isinstance(lin, torch.nn.Linear):
                    w, b = _linear(g, *lin.weight.shape)
                    lin.weight.copy_(w)
                    lin.bias.copy_(b)
            net.pts_output_linear.weight.mul_(4.0)
            net.pts_output_linear.bias.fill_(0.5)
    h, w = mc['resolution']
    n = case['rays']
    pid = torch.stack([torch.randint(0, k, (n,), generator=g, device=DEV) for k in (3, w, h)], 1).int()
    return dict(case=case, model=model, mc=mc, inp={'pixel_id': pid, 'num_frames': 3})


_PREPARE = dict(mlp=_prepare_mlp, march=_prepare_march, density=_prepare_density, appearance=_prepare_appearance,
                color=_prepare_color, shade=_prepare_shade, render=_prepare_render)


def prepare(case, seed):
    return _PREPARE[case['kind']](case, seed)


# -------------------------------------------------------------- one pass each
def _run_mlp(st):
    def forward():
        return mlp.mlp_forward_rays(st['spec'], st['weights'], st['biases'], st['o'], st['d'], st['z'], st['vd'],
                                    st['noise'])
    if not st['case']['train']:
        with torch.no_grad():
            return list(forward())
    sigma, rgb = forward()
    leaves = [t for t in st['weights'] + st['biases'] if t is not None]
    return [sigma, rgb, *torch.autograd.grad((sigma, rgb), leaves, (st['gs'], st['gr']))]


def _run_march(st):
    case = st['case']
    with torch.no_grad():
        z = sampling.stratified_z_vals(st['n'], case['coarse'], 0.0, 1.0, u=st['u'])
        c = compositing.composite(st['sigma_c'], st['rgb_c'], z, st['wo'], st['wd'], st['d'], ndc=True)
        zf = sampling.fine_z_vals(z, c['weights'], case['fine'], u=st['uf'])
    f = compositing.composite(st['sigma_f'], st['rgb_f'], zf, st['wo'], st['wd'], st['d'], ndc=True)
    grads = torch.autograd.grad((f['rgb'], f['depth_ndc']), (st['sigma_f'], st['rgb_f']), (st['g_rgb'], st['g_depth']))
    return [z, c['rgb'], c['weights'], zf, f['rgb'], f['acc'], f['depth_ndc'], f['weights'], *grads]


def _run_density(st):
    sigma, valid = tensorf.vm_density(st['pts'], st['planes'], st['lines'], BBOX, alpha=st['mask'])
    return [sigma, valid, *torch.autograd.grad(sigma, st['planes'] + st['lines'], st['gs'])]


def _run_appearance(st):
    app = tensorf.vm_appearance(st['pts'], st['planes'], st['lines'], BBOX, idx=st['idx'])
    return [app, *torch.autograd.grad(app, st['planes'] + st['lines'], st['ga'])]


def _run_color(st):
    rgb = color.color_forward(st['spec'], st['app'], st['params'][0], st['params'][1:], view_dirs=st['vd'],
                              idx=st['idx'], n_samples=st['per_ray'])
    return [rgb, *torch.autograd.grad(rgb, [st['app'], *st['params']], st['g_rgb'])]


def _run_shade(st):
    c = compositing.composite(st['sigma'], None, st['z'], st['wo'], st['wd'], st['d'], ndc=True, distance_scale=25.0)
    _, count = tensorf.threshold_compact(c['weights'], 1e-4)
    rgb = compositing.volume_render(st['rgb'], c['weights'])
    grads = torch.autograd.grad((rgb, c['depth_ndc']), (st['sigma'], st['rgb']), (st['g_rgb'], st['g_depth']))
    return [c['weights'], c['acc'], c['depth_ndc'], count, rgb, *grads]


def _run_render(st):
    with torch.no_grad():
        out = st['model'](st['inp'])
    return [out[f'{k}_{p}'] for p in ('coarse', 'fine') for k in RENDER_KEYS]


_RUN = dict(mlp=_run_mlp, march=_run_march, density=_run_density, appearance=_run_appearance, color=_run_color,
            shade=_run_shade, render=_run_render)


def run(state):
    return _RUN[state['case']['kind']](state)


# -------------------------------------------------------------- least work
_MACS = {'main': 593408, 'points': 577280, 'views': 492032}


def work(case):
    """Inputs read once, outputs written once; two operations per multiply-add."""
    k = case['kind']
    if k == 'mlp':
        n, macs = case['rays'] * case['samples'], _MACS[case['variant']]
        passes = 3 if case['train'] else 1
        return dict(bytes=n * (20 + (20 if case['train'] else 0)) + 4 * macs * (2 if case['train'] else 1),
                    flops=2.0 * macs * n * passes)
    if k == 'march':
        c, f = case['coarse'], case['coarse'] + case['fine']
        return dict(bytes=4.0 * case['rays'] * (c * 7 + case['fine'] + f * 10 + 40),
                    flops=case['rays'] * (c * 60.0 + f * 150.0))
    if k in ('density', 'appearance'):
        n = case['rays'] * case['samples']
        comps = 3 * case['comps']
        factors = 2 * 4 * comps * (case['grid'] ** 2 + case['grid'])
        if k == 'density':
            return dict(bytes=float(n * (12 + 5 + 4) + factors), flops=n * comps * 40.0 * (0.4 if case['mask'] else 1.0))
        m = int(0.4 * n)
        return dict(bytes=float(m * (16 + 8 * comps) + factors), flops=m * comps * 40.0)
    if k == 'color':
        d_in = 27 * (2 * case['features_pe'] + 1) + 3 * (2 * case['features_pe'] + 1)
        macs = 27 * case['features'] + 128 * (d_in + 128 + 3)
        return dict(bytes=float(case['rows'] * (8 * case['features'] + 28) + 8 * macs), flops=6.0 * macs * case['rows'])
    if k == 'shade':
        n = case['rays'] * case['samples']
        return dict(bytes=float(n * 4 * (2 + 1 + 3 + 1 + 3) + case['rays'] * 100), flops=n * 150.0)
    macs = _MACS['main'] * (64 + 192) * case['rays']
    return dict(bytes=float(case['rays'] * 76 + 8 * _MACS['main']), flops=2.0 * macs)


# ------------------------------------------------------------ float64 restatement
def _d(t):
    return None if t is None else t.detach().double()


def _encode(x, degree):
    out = [x]
    for m in range(degree):
        out += [torch.sin(x * 2.0 ** m), torch.cos(x * 2.0 ** m)]
    return torch.cat(out, -1)


def _mlp64(w, b, pts, dirs, noise, sigma_pe=None):
    """w, b: the 12 layers (trunk 0-7, feature, sigma / 4-channel head, view, rgb), None where absent."""
    enc = _encode(pts, 10)
    cut = 63 if sigma_pe is None else 3 * (2 * sigma_pe + 1)
    x = h = enc[:, :cut]
    for i in range(8):
        if i == 5:
            h = torch.cat([x, h], -1)
        h = F.relu(F.linear(h, w[i], b[i]))
    head = F.linear(h, w[9], b[9])
    raw = head[:, 0] if noise is None else head[:, 0] + noise
    if w[8] is None:
        return F.relu(raw), torch.sigmoid(head[:, 1:4])
    hv = torch.cat([F.linear(h, w[8], b[8]), enc[:, cut:], _encode(dirs, 4)], -1)
    hv = F.relu(F.linear(hv, w[10], b[10]))
    return F.relu(raw), torch.sigmoid(F.linear(hv, w[11], b[11]))


def _exact_mlp(case, seed):
    st = _prepare_mlp(case, seed)
    train, s = case['train'], case['samples']
    w = [None if t is None else _d(t).requires_grad_(train) for t in st['weights']]
    b = [None if t is None else _d(t).requires_grad_(train) for t in st['biases']]
    leaves = [t for t in w + b if t is not None]
    total = [torch.zeros_like(t) for t in leaves]
    o, d, z, vd = _d(st['o']), _d(st['d']), _d(st['z']), _d(st['vd'])
    sig, rgb = [], []
    step = max(1, 131072 // s)
    for r in range(0, case['rays'], step):
        q = slice(r, r + step)
        zz = z[q]
        pts = (o[q, None] + d[q, None] * zz[..., None]).reshape(-1, 3)
        dirs = None if vd is None else vd[q, None].expand(-1, s, 3).reshape(-1, 3)
        noise = None if st['noise'] is None else _d(st['noise'][q]).reshape(-1)
        with torch.set_grad_enabled(train):
            sg, cl = _mlp64(w, b, pts, dirs, noise, st['spec'].sigma_pe_degree)
        if train:
            p = slice(r * s, r * s + zz.numel())
            for t, gr in zip(total, torch.autograd.grad((sg, cl), leaves, (_d(st['gs'][p]), _d(st['gr'][p])))):
                t += gr
        sig.append(sg.detach())
        rgb.append(cl.detach())
    return [torch.cat(sig), torch.cat(rgb)] + (total if train else [])


def _composite64(sigma, rgb, z, d_ndc, scale=1.0):
    ones = torch.ones_like(z[:, :1])
    delta = (torch.cat([z, ones], 1)[:, 1:] - z) * d_ndc.norm(dim=-1, keepdim=True)
    alpha = 1.0 - torch.exp(-sigma * delta * scale)
    vis = torch.cumprod(torch.cat([ones, 1.0 - alpha + 1e-10], 1), 1)[:, :-1]
    wts = alpha * vis
    acc = wts.sum(1)
    depth = (wts * z).sum(1) / (acc + 1e-6)
    return dict(weights=wts, acc=acc, depth_ndc=depth, rgb=None if rgb is None else (wts[..., None] * rgb).sum(1))


def _stratified64(n, s, u):
    t = torch.linspace(0.0, 1.0, s, dtype=torch.float64, device=DEV).expand(n, s)
    if u is None:
        return t
    mid = 0.5 * (t[:, 1:] + t[:, :-1])
    lower, upper = torch.cat([t[:, :1], mid], 1), torch.cat([mid, t[:, -1:]], 1)
    return lower + (upper - lower) * u


def _fine64(z, wts, n_fine, u):
    bins = 0.5 * (z[:, 1:] + z[:, :-1])
    p = wts[:, 1:-1] + 1e-5
    cdf = torch.cumsum(p / p.sum(1, keepdim=True), 1)
    cdf = torch.cat([torch.zeros_like(cdf[:, :1]), cdf], 1)
    if u is None:
        u = torch.linspace(0.0, 1.0, n_fine, dtype=torch.float64, device=DEV).expand(z.shape[0], n_fine)
    i = torch.searchsorted(cdf, u.contiguous(), right=True)
    lo, hi = (i - 1).clamp(min=0), i.clamp(max=cdf.shape[1] - 1)
    c0, c1, b0, b1 = cdf.gather(1, lo), cdf.gather(1, hi), bins.gather(1, lo), bins.gather(1, hi)
    den = torch.where(c1 - c0 < 1e-5, torch.ones_like(c0), c1 - c0)
    return torch.cat([z, b0 + (u - c0) / den * (b1 - b0)], 1).sort(1).values


def _exact_march(case, seed):
    st = _prepare_march(case, seed)
    d = _d(st['d'])
    z = _stratified64(st['n'], case['coarse'], _d(st['u']))
    c = _composite64(_d(st['sigma_c']), _d(st['rgb_c']), z, d)
    zf = _fine64(z, c['weights'], case['fine'], _d(st['uf']))
    sf, rf = _d(st['sigma_f']).requires_grad_(True), _d(st['rgb_f']).requires_grad_(True)
    f = _composite64(sf, rf, zf, d)
    grads = torch.autograd.grad((f['rgb'], f['depth_ndc']), (sf, rf), (_d(st['g_rgb']), _d(st['g_depth'])))
    return [z, c['rgb'], c['weights'], zf, *(f[k].detach() for k in ('rgb', 'acc', 'depth_ndc', 'weights')), *grads]


_PLANE_AXES, _LINE_AXES = ([0, 1], [0, 2], [1, 2]), (2, 1, 0)


def _normalise64(pts):
    lo = torch.tensor(BBOX[:3], dtype=torch.float64, device=DEV)
    hi = torch.tensor(BBOX[3:], dtype=torch.float64, device=DEV)
    return (_d(pts) - lo) / (hi - lo) * 2.0 - 1.0


def _products64(planes, lines, x):
    for p in range(3):
        line = torch.stack([torch.zeros_like(x[:, 0]), x[:, _LINE_AXES[p]]], -1)
        pv = F.grid_sample(planes[p], x[None, :, None, _PLANE_AXES[p]], align_corners=True)[0, :, :, 0]
        lv = F.grid_sample(lines[p], line[None, :, None], align_corners=True)[0, :, :, 0]
        yield pv * lv


def _factor_leaves(st):
    planes = [_d(t).contiguous().requires_grad_(True) for t in st['planes']]
    lines = [_d(t).contiguous().requires_grad_(True) for t in st['lines']]
    return planes, lines, [torch.zeros_like(t) for t in planes + lines]


def _exact_density(case, seed):
    st = _prepare_density(case, seed)
    planes, lines, total = _factor_leaves(st)
    x = _normalise64(st['pts'])
    ok = (x.abs() <= 1.0).all(1)
    if st['vol'] is not None:
        ok &= F.grid_sample(_d(st['vol'])[None, None], x[None, :, None, None], align_corners=True).reshape(-1) > 0
    sigma = torch.zeros(x.shape[0], dtype=torch.float64, device=DEV)
    rows = ok.nonzero()[:, 0]
    for part in rows.split(1 << 18):
        sg = F.relu(sum(f.sum(0) for f in _products64(planes, lines, x[part])))
        for t, gr in zip(total, torch.autograd.grad(sg, planes + lines, _d(st['gs'][part]))):
            t += gr
        sigma[part] = sg.detach()
    return [sigma, None, *total]


def _exact_appearance(case, seed):
    st = _prepare_appearance(case, seed)
    planes, lines, total = _factor_leaves(st)
    out = []
    for k in range(0, st['idx'].shape[0], 1 << 17):
        app = torch.cat(list(_products64(planes, lines, _normalise64(st['pts'][st['idx'][k:k + (1 << 17)].long()])))).T.contiguous()
        for t, gr in zip(total, torch.autograd.grad(app, planes + lines, _d(st['ga'][k:k + (1 << 17)]))):
            t += gr
        out.append(app.detach())
    return [torch.cat(out), *total]


def _exact_color(case, seed):
    st = _prepare_color(case, seed)
    params = [_d(t).requires_grad_(True) for t in st['params']]
    basis, w1, b1, w2, b2, w3, b3 = params
    total = [torch.zeros_like(t) for t in params]
    pe = case['features_pe']
    rgb, g_app = [], []
    for k in range(0, case['rows'], 1 << 17):
        q = slice(k, k + (1 << 17))
        app = _d(st['app'][q]).requires_grad_(True)
        dirs = _d(st['vd'])[st['idx'][q].long() // st['per_ray']]
        h = torch.cat([_encode(F.linear(app, basis), pe), _encode(dirs, pe)], -1)
        h = F.relu(F.linear(F.relu(F.linear(h, w1, b1)), w2, b2))
        y = torch.sigmoid(F.linear(h, w3, b3))
        ga, *gp = torch.autograd.grad(y, [app, *params], _d(st['g_rgb'][q]))
        for t, gr in zip(total, gp):
            t += gr
        rgb.append(y.detach())
        g_app.append(ga)
    return [torch.cat(rgb), torch.cat(g_app), *total]


def _exact_shade(case, seed):
    st = _prepare_shade(case, seed)
    sg, cl = _d(st['sigma']).requires_grad_(True), _d(st['rgb']).requires_grad_(True)
    c = _composite64(sg, cl, _d(st['z']), _d(st['d']), 25.0)
    grads = torch.autograd.grad((c['rgb'], c['depth_ndc']), (sg, cl), (_d(st['g_rgb']), _d(st['g_depth'])))
    return [*(c[k].detach() for k in ('weights', 'acc', 'depth_ndc')), None, c['rgb'].detach(), *grads]


def _metric_depth64(wts, acc, z, o, d):
    oz, dz = o[:, 2:], d[:, 2:]
    tn = -(1.0 + oz) / dz
    at = torch.where(z == 1.0, torch.full_like(z, 1e-3), torch.zeros_like(z))
    zm = (oz + tn * dz) / dz * (1.0 / (1.0 - z + at) - 1.0) + tn
    return (wts * zm).sum(1) / (acc + 1e-6)


def _exact_render(case, seed):
    st = _prepare_render(case, seed)
    pid = st['inp']['pixel_id'].long()
    k = torch.as_tensor(st['mc']['intrinsics'], dtype=torch.float64, device=DEV)[pid[:, 0]]
    e = torch.as_tensor(st['mc']['extrinsics'], dtype=torch.float64, device=DEV)[pid[:, 0]]
    h, w = st['mc']['resolution']
    px = torch.stack([pid[:, 1].double(), pid[:, 2].double(), torch.ones_like(pid[:, 1]).double()], 1)
    cam = torch.linalg.solve(k, px[..., None])[..., 0] * torch.tensor([1.0, -1.0, -1.0], dtype=torch.float64, device=DEV)
    d, o = (cam[:, None] * e[:, :3, :3]).sum(-1), e[:, :3, 3]
    oo = o + (-(1.0 + o[:, 2:]) / d[:, 2:]) * d
    ax, ay = -2.0 * k[:, 0, 0] / w, -2.0 * k[:, 1, 1] / h
    o_ndc = torch.stack([ax * oo[:, 0] / oo[:, 2], ay * oo[:, 1] / oo[:, 2], 1.0 + 2.0 / oo[:, 2]], 1)
    d_ndc = torch.stack([ax * (d[:, 0] / d[:, 2] - oo[:, 0] / oo[:, 2]), ay * (d[:, 1] / d[:, 2] - oo[:, 1] / oo[:, 2]),
                         -2.0 / oo[:, 2]], 1)
    vd = d / d.norm(dim=-1, keepdim=True)
    out = []
    z = _stratified64(case['rays'], 64, None)
    with torch.no_grad():
        for net in (st['model'].coarse_model, st['model'].fine_model):
            sd = {n: _d(t) for n, t in net.state_dict().items()}
            wb = [[sd[f'{n}.{leaf}'] for n in mlp.PARAM_NAMES] for leaf in ('weight', 'bias')]
            sig, rgb = [], []
            for r in range(0, case['rays'], 512):
                q = slice(r, r + 512)
                pts = o_ndc[q, None] + d_ndc[q, None] * z[q][..., None]
                a, b = _mlp64(*wb, pts.reshape(-1, 3), vd[q, None].expand(pts.shape).reshape(-1, 3), None)
                sig.append(a.view(pts.shape[:2]))
                rgb.append(b.view(pts.shape))
            c = _composite64(torch.cat(sig), torch.cat(rgb), z, d_ndc)
            c['depth'] = _metric_depth64(c['weights'], c['acc'], z, o, d)
            out += [c[n] for n in RENDER_KEYS]
            z = _fine64(z, c['weights'], 128, None)
    return out


_EXACT = dict(mlp=_exact_mlp, march=_exact_march, density=_exact_density, appearance=_exact_appearance,
              color=_exact_color, shade=_exact_shade, render=_exact_render)


def exact(case, seed):
    """What ``run`` returns for these inputs, in float64."""
    return _EXACT[case['kind']](case, seed)
