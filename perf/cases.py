"""Timed cases: the work a reconstruction has this package do, through its public entry points.

An EMC iteration is one `Engine.maximize` call (or `EMCRecon.run_iteration`, which adds the
model update and the scale normalisation) on a detector, an orientation sampling, a set of
photon frames and a current model; a program calls it once per iteration on the same frames.
The cases cover what changes the work of that call: sparse and dense frames, the arithmetic
options (FP64, FP32 gathers, FP16 products of one and two terms), scaled and unscaled frames,
several modes, full searches and refinement subsets, a random start model (flat posterior) and
a developed one (sharp posterior). The learned orientation proposal (an MLP over polar photon
histograms) is timed in its two directions: features and logits, and loss and gradients.

Detector and model sizes are the ones of the benchmark configurations (151 x 151 with a 125^3
model, 260 x 257 with 251^3, the tests' 22 x 20 with 21^3) and odd ones between; frames are
simulated Poisson counts of a random-atom intensity at random orientations. Numbers of frames
and orientations are smaller than the benchmark's so that a pass stays under a second.
"""
import math

import numpy as np
import torch

import dragonfly_amd
from dragonfly_amd import _lib, proposal, synth
from dragonfly_amd.iterate import frame_counts, sum_log_factorials

DBL_MIN = float(np.finfo(np.float64).tiny)
PROB_MIN = 1e-6

# kind 'engine': one Engine.maximize; 'recon': one EMCRecon.run_iteration from the start model;
# 'logits' / 'grads': the proposal network. Keys of the EMC kinds: size (model), nx x ny
# (detector), gap (rows between its two panels), frames, photons (mean per frame), spread ('':
# same fluence; 'uniform': 0.5-1.5; 'lognormal': sigma 1, clipped to 20-20000 photons), div
# (orientations 10 (5 div^3 + div)), modes, model ('start': random, 'late': the intensity with
# 20% voxel noise), beta (0: the per-frame automatic value, times beta_factor), scaling,
# dense, precision, subset ('': full search; 'prior': cells around a prior; 'top': the cells
# nearest the true orientation, every 13th frame searched in full).
_EMC = dict(kind='engine', gap=0, spread='', modes=1, model='late', beta=0., beta_factor=1., scaling=False, dense=False,
            precision=0, subset='', coarse_div=0)


def _emc(name, **kw):
    return dict(_EMC, name=name, **kw)


def listed():
    return [
        # the smallest reconstruction (the quick-start size of the tests): launches and latency
        _emc('tiny', size=21, nx=22, ny=20, frames=60, photons=40., div=2, model='start', beta=1.),
        # a whole iteration of a small data set (the 3000-frame configuration), first iteration
        _emc('small_recon', kind='recon', size=125, nx=151, ny=151, frames=3000, photons=100., div=4, model='start',
             beta=1.),
        # two conformations refined at once (num_modes = 2), odd detector, sharp posterior
        _emc('two_modes', size=77, nx=93, ny=85, frames=2111, photons=150., div=4, modes=2, beta=0.5),
        # the plain FP64 search of the large detector: scaled frames, automatic beta, developed model
        _emc('scaled_fp64', size=251, nx=260, ny=257, gap=10, frames=30000, photons=200., spread='uniform', div=6,
             scaling=True),
        # the same search in its late, sharp iterations (beta raised as the schedule does)
        _emc('late_fp64', size=185, nx=201, ny=190, gap=7, frames=15013, photons=300., spread='uniform', div=6,
             scaling=True, beta_factor=4.),
        # first iterations from a random model: every orientation is kept by every frame
        _emc('start_fp64', size=125, nx=151, ny=151, frames=20000, photons=120., div=5, model='start'),
        # the FP32-gather option on the large detector
        _emc('fp32_gathers', size=251, nx=260, ny=257, gap=10, frames=40000, photons=200., spread='uniform', div=6,
             scaling=True, precision=3),
        # dense integer frames on the matrix cores, one FP16 term
        _emc('dense_fp16', size=251, nx=260, ny=257, gap=10, frames=4000, photons=5000., div=6, dense=True,
             precision=1),
        # dense integer frames, two FP16 terms, the smaller detector
        _emc('dense_fp16_two', size=125, nx=151, ny=151, frames=2999, photons=2000., div=6, dense=True, precision=2),
        # frames of very uneven photon counts, each searched around a prior orientation, FP64
        _emc('prior_subsets', size=251, nx=260, ny=257, gap=10, frames=40000, photons=150., spread='lognormal', div=8,
             scaling=True, subset='prior', coarse_div=3),
        # proposals: 16 cells per frame, some frames on the full search, FP32 gathers, sharp
        _emc('proposed_fp32', size=251, nx=260, ny=257, gap=10, frames=20000, photons=200., spread='uniform', div=8,
             scaling=True, precision=3, subset='top', coarse_div=3, beta_factor=4.),
        # the proposal network: gradients of one minibatch
        dict(name='network_grads', kind='grads', rows=1024, bins=4096, width=1024, depth=3, out=3240),
    ]


def _loguniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Another case of the same ranges; its (frames x orientations) work stays below the
    largest listed one's."""
    if rng.random() < 0.1:
        if rng.random() < 0.5:
            return dict(kind='grads', rows=_loguniform(rng, 100, 2048), bins=4096, width=rng.choice([512, 768, 1024]),
                        depth=rng.randint(2, 3), out=rng.choice([420, 1380, 3240]))
        return dict(kind='logits', rows=_loguniform(rng, 256, 20000), bins=4096, width=rng.choice([512, 1024]),
                    depth=rng.randint(2, 3), out=rng.choice([420, 1380, 3240]), size=125, nx=151, ny=151, photons=100.)
    size = 2 * (_loguniform(rng, 21, 251) // 2) + 1
    nx = max(18, int(size * rng.uniform(1.0, 1.25)))
    ny = max(18, nx + rng.randint(-5, 5))
    c = dict(_EMC, size=size, nx=nx, ny=ny, gap=rng.choice([0, 0, 4]) if nx > 40 else 0,
             spread=rng.choice(['', 'uniform', 'lognormal']), model=rng.choice(['start', 'late', 'late']),
             photons=float(_loguniform(rng, 40, 300)), div=rng.randint(2, 6),
             beta=rng.choice([0., 0., 1.]), beta_factor=rng.choice([1., 2., 4.]))
    most = 15000 if size > 150 else 20000
    c['frames'] = _loguniform(rng, 60, most)
    c['scaling'] = bool(c['spread'])
    how = rng.choice(['plain', 'plain', 'fp32', 'dense', 'prior', 'top', 'modes', 'recon'])
    if how == 'fp32':
        c['precision'] = 3
    elif how == 'dense':
        c.update(dense=True, precision=rng.choice([0, 1, 2]), spread='', scaling=False, model='late',
                 frames=min(c['frames'], 3000), photons=float(_loguniform(rng, 500, 5000)))
        if size < 61:
            c['photons'] = 500.
    elif how in ('prior', 'top'):
        c.update(subset=how, coarse_div=rng.choice([2, 3]), div=rng.randint(4, 8), precision=rng.choice([0, 3]))
    elif how == 'modes':
        c.update(modes=rng.randint(2, 3), div=rng.randint(2, 4), size=min(size, 151))
        if size > 151:
            c.update(nx=160, ny=157)
    elif how == 'recon':
        c.update(kind='recon', div=rng.randint(2, 5))
    return c


# ---- inputs ----------------------------------------------------------------------------------
def _dev():
    return torch.device('cuda', 0)


def _detector(case):
    return synth.flat_detector(case['nx'], case['ny'], qmax=(case['size'] - 3) / 2. - 0.05,
                               stoprad=5. if case['nx'] > 60 else 2., gap=case['gap'])


def _intensity(size, rng):
    """|F|^2 of 40 random atoms per 10^4 voxels^(2/3) (at most 400), Gaussian width 1.5."""
    n = max(6, min(400, size * size // 150))
    pos = synth.sphere_atoms(n, max(2., size / 8.4), rng)
    k = torch.arange(size, dtype=torch.float64, device=_dev()) - size // 2
    x = torch.as_tensor(pos, device=_dev())
    damp = torch.exp(-2. * (math.pi * 1.5 * k / size) ** 2)
    ph = [2. * math.pi / size * x[:, i, None] * k[None, :] for i in range(3)]
    c, s = [torch.cos(p) * damp for p in ph], [torch.sin(p) * damp for p in ph]
    cyz = (c[1][:, :, None] * c[2][:, None, :] - s[1][:, :, None] * s[2][:, None, :]).reshape(n, -1)
    syz = (s[1][:, :, None] * c[2][:, None, :] + c[1][:, :, None] * s[2][:, None, :]).reshape(n, -1)
    ct, st = c[0].t().contiguous(), s[0].t().contiguous()
    re, im = ct @ cyz - st @ syz, st @ cyz + ct @ syz
    return (re * re + im * im).reshape(size, size, size)


def _cells(rots, qv, size):
    """Trilinear cells of rotated pixels: (in grid (b, N), flat index of the 8 corners, weights)."""
    p = torch.matmul(rots.reshape(-1, 3), qv.t()).reshape(rots.shape[0], 3, -1) + float(size // 2)
    c = torch.trunc(p)
    ok = ((c >= 0) & (c <= size - 2)).all(1)
    f = p - c
    i = torch.where(ok[:, None], c, torch.zeros_like(c)).long()
    base = (i[:, 0] * size + i[:, 1]) * size + i[:, 2]
    for k in range(8):
        w = None
        off = 0
        for a, step in ((0, size * size), (1, size), (2, 1)):
            bit = (k >> (2 - a)) & 1
            fa = f[:, a] if bit else 1. - f[:, a]
            w = fa if w is None else w * fa
            off += bit * step
        yield ok, base + off, w


def _views(model, size, rots, qv, corr):
    """Trilinear views (b, N) at rotations rots, DBL_MIN outside the grid."""
    v = None
    for ok, at, w in _cells(rots, qv, size):
        t = w * model[at]
        v = t if v is None else v + t
    return torch.where(ok, v * corr, torch.full_like(v, DBL_MIN))


def _poisson_frames(case, intens, det, quats, fluence, gen):
    """Counts on mask <= 1 pixels of `intens` at quats: (frame, pixel, count) device arrays in
    frame order, and the factor that gives the mean photon count over views."""
    dev = _dev()
    size = case['size']
    model = intens.reshape(-1).float()
    qv = torch.as_tensor(det['qvals'], device=dev).float()
    corr = torch.as_tensor(det['corr'], device=dev).float()
    keep = torch.as_tensor(det['mask'] <= 1, device=dev)
    rots = torch.as_tensor(synth.rot_matrices(quats), device=dev).float()
    n = len(quats)
    batch = max(1, min(n, 24_000_000 // len(det['corr'])))
    tot = sum(float((_views(model, size, rots[b:b + batch], qv, corr) * keep).sum(dtype=torch.float64))
              for b in range(0, min(n, 1024), batch))
    rescale = case['photons'] / (tot / min(n, -(-min(n, 1024) // batch) * batch))
    fr, px, ct = [], [], []
    fl = torch.as_tensor(fluence, device=dev).float()
    for b in range(0, n, batch):
        lam = _views(model, size, rots[b:b + batch], qv, corr) * keep * (rescale * fl[b:b + batch, None])
        cnt = torch.poisson(lam, generator=gen)
        nz = cnt.nonzero()
        ct.append(cnt[nz[:, 0], nz[:, 1]].to(torch.int32))
        fr.append(nz[:, 0] + b)
        px.append(nz[:, 1])
    return torch.cat(fr), torch.cat(px), torch.cat(ct), rescale


def _inputs(case, seed):
    """Host arrays of one problem, made from the seed alone."""
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device=_dev())
    gen.manual_seed(int(seed))
    size, n = case['size'], case['frames']
    det = _detector(case)
    intens = _intensity(size, rng)
    quats = synth.random_quaternions(n, rng)
    spread = case['spread']
    if spread == 'lognormal':
        fluence = np.clip(rng.lognormal(np.log(case['photons']), 1., n), 20., 20000.) / case['photons']
    else:
        fluence = rng.uniform(0.5, 1.5, n) if spread == 'uniform' else np.ones(n)
    fr, px, ct, rescale = _poisson_frames(case, intens, det, quats, fluence, gen)
    mask = det['mask']
    num_pix = len(mask)
    inp = dict(det=det, quats=_lib.quat_gen(case['div']))
    if case['dense']:
        K = torch.zeros((n, num_pix), dtype=torch.int32, device=_dev())
        K[fr, px] = ct
        inp['dense'] = K.cpu().numpy()
        inp['fcounts'] = inp['dense'].sum(1).astype('i4')
        good = torch.as_tensor(mask < 1, device=_dev())
        inp['sum_fact'] = torch.zeros(n, dtype=torch.float64, device=_dev()).index_add_(
            0, fr, torch.lgamma(ct.double() + 1.) * good[px]).cpu().numpy()
    else:
        one = ct == 1
        f = {'ones': torch.bincount(fr[one], minlength=n), 'multi': torch.bincount(fr[~one], minlength=n),
             'place_ones': px[one], 'place_multi': px[~one], 'count_multi': ct[~one]}
        f = {k: v.cpu().numpy().astype('i4') for k, v in f.items()}
        f['ones_accum'] = np.concatenate([[0], np.cumsum(f['ones'], dtype='i8')[:-1]])
        f['multi_accum'] = np.concatenate([[0], np.cumsum(f['multi'], dtype='i8')[:-1]])
        inp['frames'] = f
        inp['fcounts'] = frame_counts(f['ones'], f['multi'], f['place_ones'], f['place_multi'], f['count_multi'], mask)
        inp['sum_fact'] = sum_log_factorials(f['multi'], f['place_multi'], f['count_multi'], mask)
    inp['mean_count'] = float(inp['fcounts'].astype('f8').sum() / n)
    if case['beta'] > 0:
        beta = np.full(n, case['beta'])
    elif case['scaling']:
        beta = np.exp(-6.5 * np.power(inp['fcounts'] * 1e-5, 0.15))
    else:
        beta = np.full(n, math.exp(-6.5 * math.pow(inp['mean_count'] * 1e-5, 0.15)))
    inp['beta'] = np.minimum(beta * case['beta_factor'], 1.)
    inp['scale'] = fluence / fluence.mean() * rng.uniform(0.9, 1.1, n) if case['scaling'] else np.ones(n)
    shape = (case['modes'],) + (size,) * 3 if case['modes'] > 1 else (size,) * 3
    if case['model'] == 'start':
        mean = inp['mean_count'] / max(1, int((mask == 0).sum())) * 2.
        inp['model'] = rng.random(shape) * mean
    else:
        noise = torch.rand(shape, generator=gen, device=_dev(), dtype=torch.float64) * 0.4 + 0.8
        inp['model'] = ((intens * rescale + 1e-9) * noise).cpu().numpy()
    if case['subset']:
        qc = _lib.quat_gen(case['coarse_div'])
        inp['cells'] = _lib.voronoi_subset(qc, inp['quats'])
        inp['num_coarse'] = len(qc)
        if case['subset'] == 'prior':
            hi = max(100, min(5000, len(inp['quats']) // 5))
            inp['rel_off'], inp['rel_quat'] = synth.prior_subsets(quats, qc, len(inp['quats']), (50, hi), 3.,
                                                                  seed=seed, device=_dev())
        else:
            k = min(16, len(qc) // 4)
            near = (torch.as_tensor(quats, device=_dev()) @ torch.as_tensor(qc[:, :4], device=_dev()).t()).abs()
            top = near.topk(k, dim=1).indices.to(torch.int32).cpu().numpy()
            full = np.arange(n) % 13 == 5
            inp['rel_off'], inp['rel_quat'] = proposal.refine_rows(np.arange(n + 1, dtype='i8') * k, top.reshape(-1),
                                                                   ~full)
    return inp


SPARSE = ('ones', 'multi', 'ones_accum', 'multi_accum', 'place_ones', 'place_multi', 'count_multi')


def prepare(case, seed):
    if case['kind'] in ('grads', 'logits'):
        return _prepare_network(case, seed)
    inp = _inputs(case, seed)
    det = inp['det']
    if case['kind'] == 'recon':
        itr = dragonfly_amd.Iterate()
        d = dragonfly_amd.CDetector.from_arrays(det['qvals'], det['corr'], det['mask'])
        itr.dets = [d]
        f = inp['frames']
        itr.set_data(dragonfly_amd.CDataset.from_arrays(d, f['ones'], f['multi'], f['place_ones'], f['place_multi'],
                                                        f['count_multi']))
        itr.set_quat(dragonfly_amd.Quaternion(num_div=case['div']))
        model = dragonfly_amd.Model(case['size'])
        model.model1 = inp['model']
        itr.set_model(model)
        itr.params.need_scaling = int(case['scaling'])
        itr.params.iteration = 2 if case['scaling'] else 1
        itr.params.update_scale, itr.params.verbosity = 1, 0
        itr.parse_scale('')
        itr.scale[:] = inp['scale']
        itr.calc_beta(case['beta'] if case['beta'] > 0 else None)
        itr.params.beta_factor = case['beta_factor']
        recon = dragonfly_amd.EMCRecon()
        recon.write_output = False
        recon.set_iterate(itr)
        return dict(case=case, recon=recon, itr=itr, model=inp['model'], scale=inp['scale'])
    eng = _lib.Engine(0)
    eng.set_precision(case['precision'])
    eng.set_detector(det['qvals'], det['corr'], det['mask'])
    eng.set_modes(case['modes'])
    eng.set_quats(inp['quats'])
    eng.set_model(inp['model'])
    if case['dense']:
        eng.set_frames_dense(inp['dense'])
    else:
        eng.set_frames(*[inp['frames'][k] for k in SPARSE])
    n = case['frames']
    eng.set_frame_params(inp['scale'], inp['beta'], np.zeros(n, 'u1'), inp['fcounts'], inp['sum_fact'],
                         inp['mean_count'], 0)
    if case['subset']:
        eng.set_refine(inp['num_coarse'], inp['cells'], inp['rel_off'], inp['rel_quat'])
    return dict(case=case, eng=eng, scale=inp['scale'])


def _fields(case):
    """Per-frame, per-orientation and volume results of one iteration. The index of the most
    likely orientation is read where the search is FP64 (ties of reduced-precision values are
    decided by their rounding)."""
    out = ['model2', 'inter_weight', 'likelihood', 'info', 'max_exp', 'psum_r']
    if case['precision'] == 0:
        out.append('rmax')
    if case['scaling']:
        out += ['scale', 'psum_d']
    if case['modes'] > 1:
        out.append('quat_norm')
    return out


def run(state):
    case = state['case']
    if case['kind'] == 'logits':
        X = state['net'].features(state['off'], state['pix'], state['cnt'], state['bins'])
        return dict(features=X, logits=state['net'].logits(X, case['rows']))
    if case['kind'] == 'grads':
        net = state['net']
        loss = net.loss_and_grads(state['X'], state['Y'], case['rows'])
        return dict(loss=loss, W=list(net.gW), b=list(net.gb))
    if case['kind'] == 'recon':
        itr, recon = state['itr'], state['recon']
        itr.model.model1 = state['model']
        if case['scaling']:
            itr.scale[:] = state['scale']
            recon.engine.set_scale(itr.scale)
        recon.run_iteration()
        return dict(model=itr.model.model1, weight=itr.model.inter_weight, rms=float(itr.rms_change),
                    likelihood=recon.likelihood, info=recon.info, rmax=recon.rmax, scale=itr.scale.copy(),
                    mean_likelihood=float(itr.likelihood), mutual_info=float(itr.mutual_info))
    eng = state['eng']
    scaling = int(case['scaling'])
    if scaling:
        eng.set_scale(state['scale'])
    st = eng.maximize(2 if scaling else 1, scaling, scaling, 0)
    out = {k: eng.get(k) for k in _fields(case)}
    out.update({k: float(st[k]) for k in ('avg_likelihood', 'mutual_info', 'rescale')})
    return out


# ---- the proposal network ----------------------------------------------------------------------
def _prepare_network(case, seed):
    rows = case['rows']
    net = proposal.OrientationProposal(case['out'], case['bins'], case['width'], case['depth'], 0, seed=seed % 1000003)
    gen = torch.Generator(device=_dev())
    gen.manual_seed(int(seed))
    st = dict(case=case, net=net)
    if case['kind'] == 'grads':
        # photon histograms: sparse, log(1 + 1000 x) of shares of ~200 photons
        B = -(-rows // 256) * 256
        lam = torch.rand((B, case['bins']), generator=gen, device=_dev()) ** 8 * 0.4
        X = torch.poisson(lam, generator=gen)
        X = torch.log1p(1000. * X / X.sum(1, keepdim=True).clamp(min=1.))
        X[rows:] = 0
        Y = torch.rand((B, case['out']), generator=gen, device=_dev()) ** 400
        Y /= Y.sum(1, keepdim=True).clamp(min=1e-30)
        st.update(X=X.to(torch.bfloat16), Y=Y.contiguous())
        return st
    c = dict(_EMC, frames=rows, div=2, size=case['size'], nx=case['nx'], ny=case['ny'], photons=case['photons'])
    inp = _inputs(c, seed)
    st['off'], st['pix'], st['cnt'] = proposal.photon_lists(inp['frames'], inp['det']['mask'])
    st['bins'] = proposal.polar_bins(inp['det']['qvals'], inp['det']['mask'])
    return st


def _network_exact(case, st):
    net = st['net']
    rows = case['rows']
    W = [w.double() for w in net.Wb]
    b = [x.double() for x in net.b]
    if case['kind'] == 'logits':
        off, pix, cnt = st['off'], st['pix'], st['cnt']
        fr = np.repeat(np.arange(rows), np.diff(off))
        bins = st['bins'][pix]
        H = np.zeros((rows, case['bins']))
        np.add.at(H, (fr[bins >= 0], bins[bins >= 0]), cnt[bins >= 0])
        tot = np.zeros(rows)
        np.add.at(tot, fr[bins >= 0], cnt[bins >= 0])
        X = torch.as_tensor(np.log1p(1000. * H / np.maximum(tot, 1e-300)[:, None]), device=_dev())
        X = X.to(torch.bfloat16).double()
    else:
        X = st['X'].double()[:rows]
    acts = [X]
    h = torch.zeros((X.shape[0], W[0].shape[1]), dtype=torch.float64, device=X.device)
    h[:, :X.shape[1]] = X
    acts = [h]
    for k in range(len(W)):
        h = h @ W[k].t() + b[k]
        if k < len(W) - 1:
            h = torch.relu(h)
        acts.append(h)
    if case['kind'] == 'logits':
        return dict(features=None, logits=h[:, :case['out']])
    Z = h[:, :case['out']]
    Y = st['Y'].double()[:rows]
    lp = torch.log_softmax(Z, 1)
    loss = float(-(Y * lp).sum() / rows)
    g = torch.zeros_like(h)
    g[:, :case['out']] = (lp.exp() - Y) / rows
    gW, gb = [None] * len(W), [None] * len(W)
    for k in range(len(W) - 1, -1, -1):
        gW[k] = g.t() @ acts[k]
        gb[k] = g.sum(0)[None]
        if k:
            g = (g @ W[k]) * (acts[k] > 0)
    return dict(loss=loss, W=gW, b=gb)


# ---- the same outputs in plain 64-bit torch ------------------------------------------------------
def exact(case, seed):
    if case['kind'] in ('grads', 'logits'):
        return _network_exact(case, _prepare_network(case, seed))
    inp = _inputs(case, seed)
    dev = _dev()
    det, size, n, M = inp['det'], case['size'], case['frames'], case['modes']
    mask = torch.as_tensor(det['mask'], device=dev)
    qv, corr = torch.as_tensor(det['qvals'], device=dev), torch.as_tensor(det['corr'], device=dev)
    P, Rn = len(mask), len(inp['quats']) * M
    wr = torch.as_tensor(inp['quats'][:, 4].copy(), device=dev).repeat_interleave(M)
    rots = torch.as_tensor(synth.rot_matrices(inp['quats'][:, :4]), device=dev).repeat_interleave(M, 0)
    model = torch.as_tensor(inp['model'], device=dev).reshape(M, -1)
    if case['dense']:
        K = torch.as_tensor(inp['dense'], device=dev).double()
    else:
        f = inp['frames']
        fr = torch.as_tensor(np.concatenate([np.repeat(np.arange(n), f['ones']), np.repeat(np.arange(n), f['multi'])]),
                             device=dev)
        px = torch.as_tensor(np.concatenate([f['place_ones'], f['place_multi']]), device=dev).long()
        ct = torch.as_tensor(np.concatenate([np.ones(len(f['place_ones'])), f['count_multi'].astype('f8')]), device=dev)
    step = 64 * M
    lik = mask < 1
    u = torch.empty(Rn, dtype=torch.float64, device=dev)
    R = torch.empty((n, Rn), dtype=torch.float64, device=dev)
    for r0 in range(0, Rn, step):
        sl = slice(r0, min(Rn, r0 + step))
        V = torch.empty((sl.stop - r0, P), dtype=torch.float64, device=dev)
        for m in range(M):
            V[m::M] = _views(model[m], size, rots[sl][m::M], qv, corr)
        u[sl] = V[:, lik].sum(1)
        L = torch.log(V)
        if case['dense']:
            R[:, sl] = K[:, lik] @ L[:, lik].t()
        else:
            good = lik[px]
            rows = L.t().contiguous()[px[good]] * ct[good, None]
            R[:, sl] = torch.zeros((n, sl.stop - r0), dtype=torch.float64, device=dev).index_add_(0, fr[good], rows)
    rescale = inp['mean_count'] / float((wr * u).sum()) * M
    scaling = case['scaling']
    scale = torch.as_tensor(inp['scale'], device=dev)
    phi = scale if scaling else torch.full((n,), rescale, dtype=torch.float64, device=dev)
    R += torch.log(wr)[None] - u[None] * phi[:, None]
    if case['dense']:
        R[torch.isnan(R)] = -math.inf
    if case['subset']:
        cells = torch.as_tensor(inp['cells'], device=dev).long()
        off, rq = inp['rel_off'], inp['rel_quat']
        allowed = torch.zeros((n, inp['num_coarse']), dtype=torch.bool, device=dev)
        owner = np.repeat(np.arange(n), np.diff(off))
        allowed[torch.as_tensor(owner[rq >= 0], device=dev), torch.as_tensor(rq[rq >= 0], device=dev).long()] = True
        allowed[torch.as_tensor(owner[rq < 0], device=dev)] = True
        for d0 in range(0, n, 2048):
            R[d0:d0 + 2048][~allowed[d0:d0 + 2048][:, cells]] = -math.inf
    beta = torch.as_tensor(inp['beta'], device=dev)
    sf = torch.as_tensor(inp['sum_fact'], device=dev)
    maxe, first = R.max(1)
    idx = torch.arange(Rn, device=dev)
    likelihood, info, psum_d = (torch.empty(n, dtype=torch.float64, device=dev) for _ in range(3))
    occ = torch.empty((n, M), dtype=torch.float64, device=dev)
    lw = torch.log(wr)
    for d0 in range(0, n, 1024):
        s = slice(d0, min(n, d0 + 1024))
        v, mx, rf, b = R[s], maxe[s, None], first[s, None], beta[s, None]
        c = 14. / b
        keep = torch.where(idx[None] > rf, v + c > mx, v > mx - c) | (idx[None] == rf)
        e = torch.where(keep, b * (v - mx), torch.full_like(v, -math.inf))
        p = torch.exp(e)
        pn = p.sum(1, keepdim=True)
        p = p / pn
        vv = torch.where(keep, v, torch.zeros_like(v))
        likelihood[s] = (p * (vv - sf[s, None])).sum(1)
        psum_d[s] = (p * u[None]).sum(1) * rescale
        big = p >= PROB_MIN
        info[s] = torch.where(big, p * (torch.log(p.clamp(min=1e-300)) - lw[None] + math.log(M)), torch.zeros_like(p)).sum(1)
        for m in range(M):
            occ[s, m] = torch.where(big, p, torch.zeros_like(p))[:, m::M].sum(1)
        R[s] = p
    psum_r = (R * (scale[:, None] if scaling else 1.)).sum(0)
    m2 = torch.zeros((M, size ** 3), dtype=torch.float64, device=dev)
    wt = torch.zeros((M, size ** 3), dtype=torch.float64, device=dev)
    merge = mask <= 1
    R[R <= PROB_MIN] = 0.
    fits = Rn * int(merge.sum()) <= 2_000_000_000  # the merge below within about 20 seconds
    for r0 in range(0, Rn if fits else 0, step):
        sl = slice(r0, min(Rn, r0 + step))
        if case['dense']:
            V = R[:, sl].t().contiguous() @ (K * (mask < 2))
        else:
            good = mask[px] < 2
            V = torch.zeros((P, sl.stop - r0), dtype=torch.float64, device=dev).index_add_(
                0, px[good], R[:, sl][fr[good]] * ct[good, None]).t()
        ps = psum_r[sl, None]
        V = (torch.where(ps > 0, V / ps, V) / corr)[:, merge]
        for m in range(M):
            for ok, at, w in _cells(rots[sl][m::M], qv[merge], size):
                w = w * (ok & (ps[m::M] > 0))
                at = at.reshape(-1)
                wt[m].index_add_(0, at, w.reshape(-1))
                m2[m].index_add_(0, at, (w * V[m::M]).reshape(-1))
    new_scale = torch.as_tensor(inp['fcounts'], device=dev) / psum_d
    shape = inp['model'].shape
    out = dict(model2=m2.reshape(shape) if fits else None, inter_weight=wt.reshape(shape) if fits else None,
               likelihood=likelihood, info=info, max_exp=maxe, psum_r=psum_r, rmax=None)
    if case['kind'] == 'recon':
        return _recon_exact(case, inp, out, m2, wt, rescale, new_scale, size) if fits else None
    if case['precision'] != 0:
        del out['rmax']
    if scaling:
        out.update(scale=new_scale, psum_d=psum_d)
    if M > 1:
        out['quat_norm'] = occ
    out.update(avg_likelihood=float(likelihood.mean()), mutual_info=float(info.mean()), rescale=rescale)
    return out


def _recon_exact(case, inp, out, m2, wt, rescale, new_scale, size):
    """The model update (Friedel average of the weighted sums, division, rms change) and the
    scale normalisation after the sums of exact()."""
    a, w = m2.reshape(size, size, size), wt.reshape(size, size, size)
    af, wf = a.flip(0, 1, 2), w.flip(0, 1, 2)
    ws = 0.5 * (w + wf)
    a = torch.where(ws > 0, 0.5 * (a * w + af * wf) / ws.clamp(min=1e-300), torch.zeros_like(a))
    a = torch.where(w > 0, a / w.clamp(min=1e-300), a)
    old = torch.as_tensor(inp['model'], device=a.device)
    rms = float(((a - old) ** 2).mean().sqrt())
    scale = torch.as_tensor(inp['scale'], device=a.device)
    if case['scaling']:
        mean = float(new_scale.mean())
        a, scale, rms = a * mean, new_scale / mean, rms * mean
    return dict(model=a, weight=w, rms=rms, likelihood=out['likelihood'], info=out['info'], rmax=None, scale=scale,
                mean_likelihood=float(out['likelihood'].mean()), mutual_info=float(out['info'].mean()))


# ---- the work of a pass ---------------------------------------------------------------------------
def work(case):
    """Bytes: the photon lists, the model and its two merged volumes, per-frame state. Operations:
    an interpolation (16) and a logarithm (10) per orientation and pixel, two multiply-adds per
    photon pixel and evaluated pair (likelihood and tomogram), ten per evaluated pair, 32 per
    merged pixel. Network: its three products per layer."""
    if case['kind'] in ('grads', 'logits'):
        dims = [case['bins']] + [case['width']] * case['depth'] + [case['out']]
        prod = sum(a * b for a, b in zip(dims, dims[1:]))
        rows = case['rows']
        times = 2. * (3. if case['kind'] == 'grads' else 1.)
        return dict(bytes=prod * (2 + (4 if case['kind'] == 'grads' else 0)) + rows * (dims[0] * 2 + dims[-1] * 4.),
                    flops=times * rows * prod)
    rot = 10 * (5 * case['div'] ** 3 + case['div']) * case['modes']
    pix = case['nx'] * case['ny']
    n, vol = case['frames'], case['modes'] * case['size'] ** 3
    mean = case['photons'] * (math.exp(0.5) if case['spread'] == 'lognormal' else 1.)
    lit = pix if case['dense'] else min(pix, mean)
    share = 1.
    if case['subset'] == 'prior':
        share = min(1., 1100. / rot)
    elif case['subset'] == 'top':
        share = min(1., 1. / 13 + 12. / 13 * 16 / (10 * (5 * case['coarse_div'] ** 3 + case['coarse_div'])))
    return dict(bytes=n * (lit * 4. if case['dense'] else lit * 5.) + n * 60. + vol * 24. + rot * 80. + pix * 40.,
                flops=rot * pix * (26. + 32.) + n * rot * share * (4. * lit + 10.))
