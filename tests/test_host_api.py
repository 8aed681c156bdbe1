"""Host side of the drop-in: parameters and config keys (dragonfly/params.pyx:16-128), the
config parser's ':::' chaining (read_config.py:9-24), the binary .emc format
(emcfile.c:3-57, emcfile.pyx:513-532), detector setters (detector.pyx:161-206) and the
per-frame precompute of dragonfly/src/iterate.c (frame counts, log-factorial sums, beta)."""
import math
import os

import numpy as np
import pytest

import dragonfly_amd as df
from dragonfly_amd import emcfile
from dragonfly_amd.iterate import frame_counts, lnfact, sum_log_factorials


def test_params_defaults_and_config(tmp_path):
    p = df.EMCParams()
    assert (p.need_scaling, p.alpha, p.beta_factor, p.num_modes, p.beta_jump, p.beta_period) == \
        (0, 0., -1., 1, 1., 100)
    assert (p.update_scale, p.save_prob, p.verbosity, p.output_folder, p.log_fname) == \
        (1, 0, 9, 'data/', 'EMC.log')
    cfg = tmp_path / 'config.ini'
    cfg.write_text('[emc]\nneed_scaling = 1\nalpha = 0.5\nbeta_schedule = 1.5 10\n'
                   'output_folder = out/\nlog_file = run.log\nnum_div = 6\n')
    p.from_config(str(cfg))
    assert p.need_scaling == 1 and p.alpha == 0.5 and p.beta_factor == 1.
    assert p.beta_jump == 1.5 and p.beta_period == 10
    assert p.output_folder == os.path.join(str(tmp_path), 'out/')
    assert p.log_fname == os.path.join(str(tmp_path), 'run.log')


def test_config_chaining(tmp_path):
    from dragonfly_amd.config import MyConfigParser
    cfg = tmp_path / 'c.ini'
    cfg.write_text('[make_data]\nout_photons_file = data/p.emc\n[emc]\n'
                   'in_photons_file = make_data:::out_photons_file\n')
    c = MyConfigParser()
    c.read(str(cfg))
    assert c.get_filename('emc', 'in_photons_file') == os.path.join(str(tmp_path), 'data/p.emc')


def test_emc_roundtrip(tmp_path):
    rng = np.random.default_rng(0)
    frames = rng.poisson(0.2, (30, 50)).astype('i4')
    fn = str(tmp_path / 'photons.emc')
    with df.EMCWriter(fn, 50) as w:
        for fr in frames:
            w.write_frame(fr)
    det = df.CDetector.from_arrays(np.zeros((50, 3)), np.ones(50), np.zeros(50, 'u1'))
    ds = df.CDataset(fn, det)
    assert ds.num_data == 30 and ds.num_pix == 50 and ds.ftype == 'sparse'
    raw = np.fromfile(fn, dtype='i4')
    assert raw[0] == 30 and raw[1] == 50 and (raw[2:256] == 0).all()
    back = np.zeros((30, 50), 'i4')
    for d in range(30):
        o, m = ds.ones_accum[d], ds.multi_accum[d]
        back[d, ds.place_ones[o:o + ds.ones[d]]] = 1
        back[d, ds.place_multi[m:m + ds.multi[d]]] = ds.count_multi[m:m + ds.multi[d]]
    assert np.array_equal(back, frames)
    assert (ds.place_multi.size == 0) or (ds.count_multi > 1).all()


def test_detector_setters_validate():
    det = df.CDetector()
    det.qvals = np.zeros((4, 3))
    with pytest.raises(ValueError):
        det.corr = np.ones(5)
    with pytest.raises(ValueError):
        det.raw_mask = np.zeros(4, 'i4')
    with pytest.raises(TypeError):
        det.qvals = np.zeros((4, 3), 'f4')
    det.corr = np.ones(4)
    det.raw_mask = np.zeros(4, 'u1')
    det.qvals = np.array([[3., 4., 0.], [0., 0., 1.], [1., 1., 1.], [0., 0., 0.]])
    assert det.num_pix == 4 and det.qmax() == 5.


def test_lnfact_closed_form():
    n = np.arange(0, 400)
    got = lnfact(n)
    want = np.array([math.lgamma(k + 1.) for k in n])
    assert np.allclose(got, want, rtol=1e-14, atol=1e-14)
    assert got[0] == 0. and got[1] == 0. and got[5] == math.log(120.)


def test_frame_precompute():
    rng = np.random.default_rng(1)
    P, D = 40, 25
    mask = rng.integers(0, 3, P).astype('u1')
    dense = rng.poisson(0.6, (D, P))
    ones = (dense == 1).sum(1)
    multi = (dense > 1).sum(1)
    po = np.concatenate([np.nonzero(r == 1)[0] for r in dense])
    pm = np.concatenate([np.nonzero(r > 1)[0] for r in dense])
    cm = np.concatenate([r[r > 1] for r in dense])
    fc = frame_counts(ones, multi, po, pm, cm, mask)
    assert np.array_equal(fc, (dense * (mask < 1)).sum(1))
    sf = sum_log_factorials(multi, pm, cm, mask)
    want = np.array([sum(math.lgamma(k + 1.) for k, m in zip(r, mask) if k > 1 and m < 1) for r in dense])
    assert np.allclose(sf, want, rtol=1e-13, atol=1e-13)


def _iterate(need_scaling, fcounts_like=None):
    rng = np.random.default_rng(2)
    P, D = 30, 12
    det = df.CDetector.from_arrays(rng.normal(size=(P, 3)), np.ones(P), np.zeros(P, 'u1'))
    dense = rng.poisson(2., (D, P))
    ones = (dense == 1).sum(1)
    multi = (dense > 1).sum(1)
    po = np.concatenate([np.nonzero(r == 1)[0] for r in dense])
    pm = np.concatenate([np.nonzero(r > 1)[0] for r in dense])
    cm = np.concatenate([r[r > 1] for r in dense])
    itr = df.Iterate()
    itr.params.need_scaling = need_scaling
    itr.dets = [det]
    itr.set_data(df.CDataset.from_arrays(det, ones, multi, po, pm, cm))
    return itr, dense


def test_beta_rules():
    itr, dense = _iterate(0)
    itr.calc_beta()
    m = dense.sum(1).mean()
    assert np.allclose(itr.beta_start, math.exp(-6.5 * math.pow(m * 1e-5, 0.15)))
    itr, dense = _iterate(1)
    itr.calc_beta()
    want = [math.exp(-6.5 * math.pow(f * 1e-5, 0.15)) for f in dense.sum(1)]
    assert np.array_equal(itr.beta_start, want)
    itr.calc_beta(0.3)
    assert (itr.beta_start == 0.3).all()


def test_blacklist_selection():
    itr, _ = _iterate(0)
    itr.blacklist[:] = 0
    itr.blacklist[3] = 1
    itr.parse_blacklist('', 'odd_only')
    # frames not already blacklisted alternate keep/drop starting with keep
    assert list(itr.blacklist) == [0, 1, 0, 1, 0, 1, 0, 1, 0, 1, 0, 1][:3] + [1] + \
        [1 - x for x in [0, 1, 0, 1, 0, 1, 0, 1]]
    with pytest.raises(ValueError):
        itr.parse_blacklist('', 'bad')


def test_update_beta_schedule():
    itr, _ = _iterate(0)
    itr.calc_beta(0.2)
    itr.params.beta_factor = 1.5
    itr.params.beta_jump = 2.
    itr.params.beta_period = 3

    class FakeEngine:
        def set_beta(self, b):
            self.b = b.copy()
    rec = df.EMCRecon()
    rec.iter = itr
    rec.engine = FakeEngine()
    itr.params.iteration = 7
    mean = rec.update_beta()
    assert np.allclose(itr.beta, min(0.2 * 2. ** 2 * 1.5, 1.))
    assert np.allclose(rec.engine.b, itr.beta) and abs(mean - 1.) < 1e-15


def test_calculate_size():
    assert df.Iterate.calculate_size(60.95) == 125
    assert df.Iterate.calculate_size(123.9) == 251
    assert df.Iterate.calculate_size(61.0) == 125


def test_parse_rel_quat_formats(tmp_path):
    """Per-frame coarse sets for refinement (legacy parse_rel_quat, src/iterate.c:364-525):
    the binary probs layout, an output file with sparse probabilities, and one with only the
    most likely orientations (rmax -1 gives an empty set); then the Voronoi map."""
    itr, _ = _iterate(0)
    itr.set_quat(df.Quaternion(2))
    D = itr.tot_num_data
    rng = np.random.default_rng(4)
    sets = [np.sort(rng.choice(60, rng.integers(0, 5), replace=False)).astype('i4') for _ in range(D)]
    hdr = np.zeros(256, 'i4')
    hdr[0], hdr[1] = D, 60
    fn = tmp_path / 'probs.bin'
    with open(fn, 'wb') as f:
        hdr.tofile(f)
        np.array([len(s) for s in sets], 'i4').tofile(f)
        for s in sets:
            s.tofile(f)
    got = itr.parse_rel_quat(str(fn), 1)
    assert all(np.array_equal(a, b) for a, b in zip(got, sets))
    hdr[1] = 61
    with open(fn, 'r+b') as f:
        hdr[:2].tofile(f)
    with pytest.raises(ValueError, match='num_rot_coarse'):
        itr.parse_rel_quat(str(fn), 1)
    npz = tmp_path / 'out.npz'
    np.savez(npz, **{'probabilities/num_prob': np.array([len(s) for s in sets], 'i4'),
                     'probabilities/place': np.concatenate(sets), 'orientations': np.arange(D)})
    got = itr.parse_rel_quat(str(npz), 1)
    assert all(np.array_equal(a, b) for a, b in zip(got, sets))
    orient = np.arange(D) - 1
    np.savez(npz, orientations=orient)
    got = itr.parse_rel_quat(str(npz), 1)
    assert len(got[0]) == 0 and all(list(g) == [o] for g, o in zip(got[1:], orient[1:]))
    itr.setup_refine(1, sets)
    assert itr.num_coarse == 60 and len(itr.quat_mapping) == itr.quat.num_rot
    assert itr.rel_off[-1] == sum(len(s) for s in sets)
    assert np.array_equal(itr.quat_mapping, df._lib.voronoi_subset(df._lib.quat_gen(1), itr.quat.quats))


def test_autotune_greedy_choice():
    """The tuner keeps, option by option, the value whose stages ran fastest, and leaves the
    engine set to it; scale factors are never updated while tuning."""
    from dragonfly_amd import autotune

    class FakeEngine:
        def __init__(self):
            self.opt = {'lik_unroll': 8, 'tomo_parts': 8}
            self.calls = []

        def set_option(self, name, value):
            self.opt[name] = value

        def maximize(self, iteration, need_scaling, update_scale, known_scale):
            self.calls.append(update_scale)
            lik = {4: 30., 8: 20., 16: 10.}[self.opt['lik_unroll']]
            tomo = {4: 9., 8: 7., 16: 8.}[self.opt['tomo_parts']]
            return {'stage_ms': {'likelihood': lik, 'tomogram': tomo, 'reduce': 1.}}

    eng = FakeEngine()
    space = (('lik_unroll', (8, 16, 4), ('likelihood',)), ('tomo_parts', (8, 16, 4), ('tomogram', 'reduce')))
    chosen, times = autotune.tune(eng, space=space)
    assert chosen == {'lik_unroll': 16, 'tomo_parts': 8}
    assert eng.opt == chosen
    assert times['tomo_parts'] == {8: 8., 16: 9., 4: 10.}
    assert not any(eng.calls)


def test_autotune_leaves_options_that_nothing_reads():
    """An option that the kernels in use do not read is not decided by the noise of equal runs."""
    from dragonfly_amd import autotune

    class FakeEngine:
        def __init__(self):
            self.opt = {'lik_xcd': 1, 'lik_unroll': 8}

        def set_option(self, name, value):
            self.opt[name] = value

        def option_in_use(self, name):
            return name != 'lik_unroll' or not self.hot  # as the bright-row likelihood

        def maximize(self, iteration, need_scaling, update_scale, known_scale):
            # the kernels of the last run count, and whatever is tried later looks a little faster
            self.hot = self.opt['lik_xcd'] == 1
            self.t = getattr(self, 't', 10.) - 0.01
            return {'stage_ms': {'likelihood': self.t + 5. * (self.opt['lik_xcd'] != 1)}}

    eng = FakeEngine()
    space = (('lik_xcd', (1, 2, 0), ('likelihood',)), ('lik_unroll', (8, 16, 4), ('likelihood',)))
    chosen, times = autotune.tune(eng, space=space)
    assert chosen == {'lik_xcd': 1, 'lik_unroll': 8} and eng.opt == chosen and list(times['lik_unroll']) == [8]


def test_refine_lists_match_refine_sets():
    """The flattened proposal lists equal the per-frame sets (top-k sorted, or every cell for
    a fall-back frame), and a reused buffer gives the same lists."""
    from dragonfly_amd import proposal
    rng = np.random.default_rng(4)
    top = np.stack([rng.choice(50, 5, replace=False) for _ in range(40)]).astype('i4')
    mass = rng.random(40)
    sets, fb = proposal.refine_sets(top, mass, 50, 0.5)
    off, rq, fb2, buf = proposal.refine_lists(top, mass, 50, 0.5)
    assert np.array_equal(fb, fb2)
    assert np.array_equal(off, np.concatenate([[0], np.cumsum([len(x) for x in sets])]))
    assert np.array_equal(rq, np.concatenate(sets))
    off3, rq3, _, buf3 = proposal.refine_lists(top, mass, 50, 0.5, buf)
    assert buf3 is buf and np.array_equal(rq3, rq)


def test_prior_subsets_sizes_and_nearest_cell():
    """Refinement sets around a prior: sizes follow the requested range of fine orientations
    (whole cells), the cells are distinct, and with no prior error the nearest cell to the
    true orientation is always in the set."""
    from dragonfly_amd import _lib, synth
    qc = _lib.quat_gen(2)
    nfine = _lib.num_rot(6)
    rng = np.random.default_rng(2)
    tq = rng.normal(size=(300, 4))
    tq /= np.linalg.norm(tq, axis=1, keepdims=True)
    off, rq = synth.prior_subsets(tq, qc, nfine, (50, 2000), 0., device='cpu')
    per_cell = nfine / len(qc)
    k = np.diff(off)
    assert k.min() >= 1 and (k * per_cell).max() <= 2000 + per_cell
    near = np.argmax(np.abs(tq @ qc[:, :4].T), axis=1)
    for d in range(300):
        cells = rq[off[d]:off[d + 1]]
        assert len(set(cells.tolist())) == len(cells)
        assert near[d] in cells


def test_modes_and_background_host_side(tmp_path):
    """num_modes from the config (params.pyx:104) gives a Model of that many volumes
    (model.pyx:58, random start drawn over the whole (modes, size^3) block); non-rotating
    modes are refused; a detector background (detector.pyx:101-104, 207-220) and the
    background scales (parse_scale(bg=True), iterate.pyx:284-315) are read back."""
    cfg = tmp_path / 'config.ini'
    cfg.write_text('[emc]\nnum_modes = 2\n')
    p = df.EMCParams()
    p.from_config(str(cfg))
    assert p.num_modes == 2 and p.nonrot_modes == 0
    cfg.write_text('[emc]\nnum_modes = 2\nnum_nonrot_modes = 1\n')
    with pytest.raises(NotImplementedError):
        df.EMCParams().from_config(str(cfg))
    m = df.Model(7, 2)
    m.allocate('', model_mean=3., fixed_seed=True)
    assert m.model1.shape == (2, 7, 7, 7) and m.model2.shape == (2, 7, 7, 7)
    want = np.random.RandomState(0x5EED).random_sample((2, 7, 7, 7)) * 3.
    assert np.array_equal(m.model1, want)
    itr, dense = _iterate(0)
    det = itr.dets[0]
    assert det.with_bg == 0 and det.background is None
    bg = np.linspace(0.1, 0.2, det.num_pix)
    np.savez(tmp_path / 'bg.npz', background=bg)
    det.parse_background(str(tmp_path / 'bg.npz'))
    assert det.with_bg == 1 and np.array_equal(det.background, bg)
    with pytest.raises(ValueError):
        det.background = bg[:-1]
    np.savez(tmp_path / 'bgscale.npz', scale=np.arange(1., 4.))
    itr.parse_scale(str(tmp_path / 'bgscale.npz'), bg=True)
    assert itr.bgscale.shape == (itr.tot_num_data,)
    assert np.array_equal(itr.bgscale[:3], [1., 2., 3.]) and (itr.bgscale[3:] == 1.).all()
    assert (itr.scale is None) or itr.scale.shape == (itr.tot_num_data,)


def test_from_config_background_selection_resume(tmp_path):
    """The config pipeline (iterate.pyx:40-182) on files written to disk: detector
    background from background_file or background_list (iterate.pyx:106-125), background
    scales from bgscale_file when need_scaling (:167-169, the file's 'scale' dataset),
    odd_only selection with num_blacklist left at 0 as the Cython path leaves it, the start
    model, refusal of axial_sym > 1, and resume from whichever of output_NNN.h5 / .npz
    exists (:141-151)."""
    import sys
    sys.path.insert(0, os.path.dirname(__file__))
    import problems as P
    p = P.build(P.tiny_config(num_data=30))
    P_ = len(p['det']['corr'])
    bg = np.linspace(0.01, 0.02, P_)
    np.savez(tmp_path / 'bg.npz', background=bg)
    np.savez(tmp_path / 'bgs.npz', scale=np.linspace(0.5, 1.5, 30))
    cfg = P.write_config(p, str(tmp_path), need_scaling=1, background_file='bg.npz',
                         bgscale_file='bgs.npz', selection='odd_only', beta=0.5)
    itr = df.Iterate(cfg)
    det = itr.dets[0]
    assert det.with_bg == 1 and np.array_equal(det.background, bg)
    assert np.array_equal(itr.bgscale, np.linspace(0.5, 1.5, 30))
    assert np.array_equal(itr.scale, np.ones(30))
    assert list(itr.blacklist) == [0, 1] * 15 and itr.num_blacklist == 0
    assert np.array_equal(itr.model.model1, p['model1']) and (itr.beta_start == 0.5).all()
    # background_list: one entry per detector, relative to the list's folder
    (tmp_path / 'bglist.txt').write_text('bg.npz\n')
    cfg = P.write_config(p, str(tmp_path), background_list='bglist.txt')
    assert np.array_equal(df.Iterate(cfg).dets[0].background, bg)
    cfg = P.write_config(p, str(tmp_path), background_list='bglist.txt', background_file='bg.npz')
    with pytest.raises(ValueError, match='Pick one'):
        df.Iterate(cfg)
    cfg = P.write_config(p, str(tmp_path), axial_sym=4)
    with pytest.raises(NotImplementedError):
        df.Iterate(cfg)
    # resume: the last logged iteration's output file gives model1 and the scales
    cfg = P.write_config(p, str(tmp_path), need_scaling=1)
    (tmp_path / 'EMC.log').write_text('header\n\nIter\ttime\n1\t0.1\n3\t0.1\n')
    with pytest.raises(FileNotFoundError):
        df.Iterate(cfg, resume=True)
    os.makedirs(tmp_path / 'out', exist_ok=True)
    intens = p['model1'][None] * 2.
    np.savez(tmp_path / 'out' / 'output_003.npz', intens=intens, scale=np.full(30, 1.25))
    itr = df.Iterate(cfg, resume=True)
    assert itr.params.start_iter == 4
    assert np.array_equal(itr.model.model1, intens[0]) and (itr.scale == 1.25).all()


def test_update_beta_mean_over_all_frames():
    """update_beta sums beta over frames that are not blacklisted and divides by
    tot_num_data - num_blacklist with num_blacklist never set, i.e. by every frame
    (recon.pyx:162-172)."""
    itr, _ = _iterate(0)
    itr.calc_beta(0.4)
    itr.parse_blacklist('', 'even_only')
    itr.params.beta_factor = 1.

    class FakeEngine:
        def set_beta(self, b):
            pass
    rec = df.EMCRecon()
    rec.iter = itr
    rec.engine = FakeEngine()
    itr.params.iteration = 1
    mean = rec.update_beta()
    kept = int((itr.blacklist == 0).sum())
    assert 0 < kept < itr.tot_num_data
    assert abs(mean - 0.4 * kept / itr.tot_num_data) < 1e-15


def test_reference_import_name_and_command():
    """The reference's import name and console command (pyproject.toml:69 and
    dragonfly/__init__.py there): `dragonfly` exposes the same objects, its submodules
    import, and the `dragonfly.emc` script resolves to the reconstruction's main()."""
    import configparser
    import subprocess
    import sys
    import dragonfly
    import dragonfly.iterate
    import dragonfly.recon
    from dragonfly.recon import EMCRecon, main
    assert dragonfly.EMCRecon is EMCRecon is df.EMCRecon
    assert dragonfly.iterate.Iterate is df.Iterate and main is df.recon.main
    for name in ('CDetector', 'CDataset', 'EMCWriter', 'Quaternion', 'Model', 'EMCParams', 'Iterate'):
        assert getattr(dragonfly, name) is getattr(df, name)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    cp = configparser.ConfigParser()
    cp.read(os.path.join(root, 'pyproject.toml'))
    target = cp.get('project.scripts', "'dragonfly.emc'").strip("'")
    mod, fn = target.split(':')
    assert (mod, fn) == ('dragonfly.recon', 'main')
    out = subprocess.run([sys.executable, '-m', 'dragonfly.recon', '--help'], cwd=root, capture_output=True,
                         text=True, timeout=120)
    assert out.returncode == 0 and 'niter' in out.stdout


def test_union_and_csr_refine_lists():
    """Proposal unions are each frame's distinct cells in ascending order; CSR refinement
    lists keep an accepted frame's cells and give a rejected frame the single entry -1 (every
    cell, emc_set_refine)."""
    from dragonfly_amd import proposal
    rng = np.random.default_rng(6)
    a, b = rng.integers(0, 40, (25, 5)), rng.integers(0, 40, (25, 3))
    off, cells = proposal.union_cells(a, b)
    for d in range(25):
        assert list(cells[off[d]:off[d + 1]]) == sorted(set(a[d]) | set(b[d]))
    acc = rng.random(25) < 0.6
    ro, rq = proposal.refine_lists_csr(off, cells, acc, 40)
    for d in range(25):
        want = cells[off[d]:off[d + 1]] if acc[d] else [-1]   # -1: every cell
        assert np.array_equal(rq[ro[d]:ro[d + 1]], want)


def test_widened_proposal_lists():
    """widen_lists_csr: kept frames keep their cells, widened ones get theirs followed by the
    added cells, full ones the single entry -1."""
    from dragonfly_amd import proposal
    rng = np.random.default_rng(7)
    n = rng.integers(1, 6, 40)
    off = np.zeros(41, 'i8')
    np.cumsum(n, out=off[1:])
    cells = rng.integers(0, 60, off[-1]).astype('i4')
    num_add = rng.choice([-1, 0, 0, 1, 3, 7], 40).astype('i4')
    add = rng.integers(0, 60, int(np.maximum(num_add, 0).sum())).astype('i4')
    ro, rq = proposal.widen_lists_csr(off, cells, num_add, add)
    a = 0
    for d in range(40):
        got = list(rq[ro[d]:ro[d + 1]])
        own = list(cells[off[d]:off[d + 1]])
        if num_add[d] < 0:
            assert got == [-1]
        else:
            k = int(num_add[d])
            assert got == own + list(add[a:a + k])
            a += k
    assert a == len(add)


def test_stacked_proposal_lists():
    """stack_cells keeps every row side by side (repeats allowed: the engine takes a frame's set
    as the union of its list); refine_rows gives refine_lists_csr's lists for them."""
    from dragonfly_amd import proposal
    rng = np.random.default_rng(4)
    a = rng.integers(0, 50, (30, 5)).astype('i4')
    b = rng.integers(0, 50, (30, 3)).astype('i4')
    off, cells = proposal.stack_cells(a, b)
    assert np.array_equal(off, np.arange(31) * 8)
    assert np.array_equal(cells.reshape(30, 8), np.concatenate([a, b], axis=1))
    acc = rng.random(30) > 0.3
    ro, rq = proposal.refine_rows(off, cells, acc)
    ro2, rq2 = proposal.refine_lists_csr(off, cells, acc, 50)
    assert np.array_equal(ro, ro2) and np.array_equal(rq, rq2)
    for d in range(30):
        got = rq[ro[d]:ro[d + 1]]
        if acc[d]:
            assert set(got) == set(a[d]) | set(b[d])
        else:
            assert list(got) == [-1]
