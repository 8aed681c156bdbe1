"""Photon gathers at the sizes where their lists are cut: frames of every photon count around the
64-entry stage, the two (FP32: two, and four for pairs) photon streams of a wavefront and the
rows in flight; frame counts that leave a block's wavefronts idle; orientation counts that end
inside a tile. Checked against the oracle: FP64 to 1e-9 as the other parity tests, FP32 log W to
the FP32-gather tests' bars (average log-likelihood 1e-6)."""
import numpy as np
import pytest
import torch  # noqa: F401  (its HIP runtime is loaded before the engine's library)

import problems as P
from dragonfly_amd import _lib

pytestmark = pytest.mark.gpu

COUNTS = (0, 1, 2, 3, 7, 8, 9, 15, 16, 17, 31, 33, 63, 64, 65, 66, 71, 72, 73, 127, 128, 129, 191, 200)


def counted_problem(counts, num_rot, seed=7):
    """The tiny geometry with frames of exactly counts[d] photon pixels (every fifth of them a
    multi-photon pixel), and the first num_rot orientations of the num_div 2 sampling."""
    p = P.build(P.tiny_config(num_data=len(counts)), quats=_lib.quat_gen(2)[:num_rot])
    rng = np.random.default_rng(seed)
    mask = p['det']['mask']
    good = np.flatnonzero(mask < 1)
    ones, multi, po, pm, cm = [], [], [], [], []
    for n in counts:
        px = rng.permutation(good)[:n]
        m = n // 5
        ones.append(n - m)
        multi.append(m)
        po.append(px[m:])
        pm.append(px[:m])
        cm.append(rng.integers(2, 9, m))
    f = dict(ones=np.array(ones, 'i4'), multi=np.array(multi, 'i4'), place_ones=np.concatenate(po).astype('i4'),
             place_multi=np.concatenate(pm).astype('i4'), count_multi=np.concatenate(cm).astype('i4'))
    f['ones_accum'] = np.concatenate([[0], np.cumsum(ones)[:-1]]).astype('i8')
    f['multi_accum'] = np.concatenate([[0], np.cumsum(multi)[:-1]]).astype('i8')
    p['frames'] = f
    fp = p['fparams']
    fp['fcounts'] = P.frame_counts(f['ones'], f['multi'], f['place_ones'], f['place_multi'], f['count_multi'], mask)
    fp['sum_fact'] = P.sum_log_factorials(f['multi'], f['place_multi'], f['count_multi'], mask)
    fp['mean_count'] = fp['fcounts'].astype('f8').mean()
    fp['beta'] = np.full(len(counts), 0.05)
    return p


@pytest.mark.parametrize('num_rot', (63, 129, 420))
@pytest.mark.parametrize('unroll', (4, 8, 16))
def test_likelihood_photon_counts(num_rot, unroll):
    p = counted_problem(COUNTS[:len(COUNTS) - (unroll == 8)], num_rot)
    o = P.run_oracle(p, dict(iteration=1))
    eng = P.engine_for(p)
    eng.set_option('lik_unroll', unroll)
    g = P.run_engine(eng, dict(iteration=1))
    for k in ('max_exp', 'p_norm', 'likelihood', 'prob', 'model2'):
        assert P.rel_err(g[k], o[k]) <= 1e-9, k
    # a frame without photons has R = log w - phi u alone, and the flat detector's two-fold symmetry
    # gives orientations 0 and 5 the same u to rounding: its arg-max is a tie
    seen = np.array(COUNTS[:len(g['rmax'])]) > 0
    assert np.array_equal(g['rmax'][seen], o['rmax'][seen])
    eng.set_precision(3)
    h = P.run_engine(eng, dict(iteration=1))
    assert abs(h['avg_likelihood'] / o['avg_likelihood'] - 1.) <= 1e-6
    assert P.rel_err(h['max_exp'], o['max_exp']) <= 1e-6
    eng.close()


@pytest.mark.parametrize('precision', (0, 3))
def test_likelihood_bright_pixels(precision):
    """The likelihood with the brightest pixels' rows in LDS (1536 frames x 3201 orientations: 12 parts of
    51 FP64 or 25.5 FP32 tiles, more than 256 blocks, the last tile short) against the gather through L2 alone (lik_xcd 2), with frames of
    every count around the stages, without photons and blacklisted: the same rows, summed in another
    order."""
    counts = COUNTS * 64
    p = counted_problem(counts, 3240)
    p['quats'] = _lib.quat_gen(4)[:3201]
    p['fparams']['blacklist'] = (np.arange(len(counts)) % 50 == 3).astype('u1')
    p['fparams']['num_blacklist'] = int(p['fparams']['blacklist'].sum())
    out = []
    for xcd in (1, 2):
        eng = P.engine_for(p)
        eng.set_precision(precision)
        eng.set_option('lik_xcd', xcd)
        out.append(P.run_engine(eng, dict(iteration=1)))
        assert (eng.get_option('lik_hot') > 0) == (xcd == 1)  # else the gather is compared with itself
        eng.close()
    for k in ('max_exp', 'p_norm', 'likelihood', 'prob'):
        assert P.rel_err(out[0][k], out[1][k]) <= 1e-9, k


@pytest.mark.parametrize('precision', (0, 3))
def test_pair_likelihood_photon_counts(precision):
    """The same lists on refinement subsets (pairs of frames and 64-slot tiles) against the
    masked full search of the engine."""
    p = counted_problem(COUNTS, 420)
    qc = _lib.quat_gen(1)
    cells = _lib.voronoi_subset(qc, p['quats'])
    rng = np.random.default_rng(3)
    sets = [np.sort(rng.permutation(len(qc))[:1 + d % 9]).astype('i4') for d in range(len(COUNTS))]
    off = np.concatenate([[0], np.cumsum([len(s) for s in sets])]).astype('i8')
    out = []
    for subset in (1, 0):
        eng = P.engine_for(p)
        eng.set_precision(precision)
        eng.set_option('subset', subset)
        eng.set_refine(len(qc), cells, off, np.concatenate(sets))
        out.append(P.run_engine(eng, dict(iteration=1)))
        eng.close()
    for k in ('max_exp', 'p_norm', 'likelihood', 'prob'):
        assert P.rel_err(out[0][k], out[1][k]) <= (1e-9 if precision == 0 else 1e-6), k


@pytest.mark.parametrize('frames, num_rot', ((1, 1), (3, 64), (65, 65), (257, 129), (16385, 20), (33000, 33)))
def test_tomogram_rows(frames, num_rot):
    """The tomogram's row tiles and frame ranges: one frame, fewer frames than streams, patches
    with few or no photons, orientation counts that end inside a 16- or 32-wide tile, two and
    three frame ranges (16,384 frames each). FP64 against the oracle to 1e-9, FP32 gathers to 1e-4
    (the FP32-gather tests' bars), orientation-major (brick merge) and tile-major (box merge)."""
    p = P.build(P.tiny_config(num_data=frames, mean_count=25.), quats=_lib.quat_gen(2)[:num_rot], num_ave=200)
    p['fparams']['beta'] = np.full(frames, 0.1)
    o = P.run_oracle(p, dict(iteration=1), dense_prob=False)
    eng = P.engine_for(p)
    for precision, merge_mode, bar in ((0, 1, 1e-9), (0, 0, 1e-9), (3, 1, 1e-4)):
        eng.set_precision(precision)
        eng.set_option('merge_mode', merge_mode)
        eng.maximize(1, 0, 1, 0)
        assert P.rel_err(eng.get('model2'), o['model2']) <= bar, (precision, merge_mode)
        assert P.rel_err(eng.get('inter_weight'), o['inter_weight']) <= 1e-9
    eng.close()


@pytest.mark.parametrize('frames, num_rot, mean_count', ((1, 20, 3000.), (3, 420, 3000.), (64, 129, 400.),
                                                         (65, 420, 400.), (700, 420, 150.), (17000, 33, 400.)))
def test_tomogram_marked_rows(frames, num_rot, mean_count):
    """The same with bright frames, whose posterior lies in a few orientations: tiles without any
    marked row, with few (taken by their marks) and with most of them, two frame ranges."""
    p = P.build(P.tiny_config(num_data=frames, mean_count=mean_count), quats=_lib.quat_gen(2)[:num_rot], num_ave=200)
    o = P.run_oracle(p, dict(iteration=1), dense_prob=False)
    eng = P.engine_for(p)
    for precision, merge_mode, bar in ((0, 1, 1e-9), (0, 0, 1e-9), (3, 1, 1e-4)):
        eng.set_precision(precision)
        eng.set_option('merge_mode', merge_mode)
        eng.maximize(1, 0, 1, 0)
        assert P.rel_err(eng.get('model2'), o['model2']) <= bar, (precision, merge_mode)
    eng.close()


@pytest.mark.parametrize('precision', (0, 3))
@pytest.mark.parametrize('part_frames', (12500, 7))
def test_full_frames_tomogram_ranges(precision, part_frames):
    """Refinement subsets with full frames: their sums (one launch or several frame ranges)
    taken over by the pair tomogram, against the masked full search."""
    p = counted_problem(COUNTS, 420)
    qc = _lib.quat_gen(1)
    cells = _lib.voronoi_subset(qc, p['quats'])
    rng = np.random.default_rng(5)
    sets = [np.array([-1], 'i4') if d % 2 else np.sort(rng.permutation(len(qc))[:5]).astype('i4')
            for d in range(len(COUNTS))]
    off = np.concatenate([[0], np.cumsum([len(s) for s in sets])]).astype('i8')
    out = []
    for subset in (1, 0):
        eng = P.engine_for(p)
        eng.set_precision(precision)
        eng.set_option('subset', subset)
        eng.set_option('sig_full_rows', 0)
        eng.set_option('full_part_frames', part_frames)
        eng.set_refine(len(qc), cells, off, np.concatenate(sets))
        out.append(P.run_engine(eng, dict(iteration=1)))
        eng.close()
    assert P.rel_err(out[0]['model2'], out[1]['model2']) <= (1e-9 if precision == 0 else 1e-4)


def test_full_frames_sums_over_ranges_keep_precision():
    """FP32 gathers, full frames in one and in 64 frame ranges: the sums pass from range to range without
    a rounding, so a view differs by the roundings of the single range's sum and of the two views: 2^-24
    each, whatever the number of ranges. Three orientations keep a voxel near one view's error."""
    n = 64 * len(COUNTS[4:])
    p = counted_problem(COUNTS[4:] * 64, 3)
    p['fparams']['beta'] = np.full(n, 1e-3)  # every orientation counts for every frame
    off, rq = np.arange(n + 1, dtype='i8'), np.full(n, -1, 'i4')
    out = []
    for part_frames in (12500, 20):
        eng = P.engine_for(p)
        eng.set_precision(3)
        eng.set_option('sig_full_rows', 0)
        eng.set_option('tomo_parts', 64)
        eng.set_option('full_part_frames', part_frames)
        eng.set_refine(1, np.zeros(3, 'i4'), off, rq)
        out.append(P.run_engine(eng, dict(iteration=1))['model2'])
        eng.close()
    on = out[0] > 0.
    assert on.sum() > 100 and np.array_equal(on, out[1] > 0.)
    assert np.abs(out[1][on] / out[0][on] - 1.).max() <= 3. * 2. ** -24


@pytest.mark.parametrize('precision', (0, 3))
@pytest.mark.parametrize('repeat, buckets', ((1, 1), (8, 1), (8, 0)))
@pytest.mark.parametrize('full', (False, True))
def test_pair_tomogram_photon_lists(precision, repeat, buckets, full):
    """The pair tomogram from its tiles' photon lists, by whole patches (24 frames) and by quarter
    patches (192 frames of the same counts; 440 pixels end inside a patch), with and without rows
    of full frames in the lists, and from the walk over the tiles' rows, against the masked full
    search."""
    counts = COUNTS * repeat
    p = counted_problem(counts, 420)
    qc = _lib.quat_gen(1)
    cells = _lib.voronoi_subset(qc, p['quats'])
    rng = np.random.default_rng(6)
    sets = [np.array([-1], 'i4') if full and d % 2 else np.sort(rng.permutation(len(qc))[:9]).astype('i4')
            for d in range(len(counts))]
    off = np.concatenate([[0], np.cumsum([len(s) for s in sets])]).astype('i8')
    out = []
    for subset in (1, 0):
        eng = P.engine_for(p)
        eng.set_precision(precision)
        eng.set_option('subset', subset)
        eng.set_option('tomo_buckets', buckets)
        eng.set_refine(len(qc), cells, off, np.concatenate(sets))
        out.append(P.run_engine(eng, dict(iteration=1)))
        eng.close()
    assert P.rel_err(out[0]['model2'], out[1]['model2']) <= (1e-9 if precision == 0 else 1e-4)
    assert P.rel_err(out[0]['inter_weight'], out[1]['inter_weight']) <= 1e-9


@pytest.mark.parametrize('size', (81, 128, 163))
def test_volume_readback(size):
    """Volumes of one piece and a remainder, whole pieces, and more pieces than copying threads
    come back byte for byte."""
    p = counted_problem((5,), 3)
    eng = P.engine_for(p)
    vol = np.random.default_rng(size).random((size,) * 3)
    eng.set_model(vol)
    for _ in range(2):
        assert np.array_equal(eng.get('model1').view('u8'), vol.view('u8'))
    assert not eng.get('model2').any()
    eng.close()


@pytest.mark.parametrize('frames', (1, 15, 17, 33, 700))
def test_psum_parts(frames):
    """psum_r (the divisor of the views) over one and several frame parts, the last one short, with
    blacklisted and scaled frames and 257 orientations (one past a block's)."""
    p = P.build(P.tiny_config(num_data=frames, mean_count=25.), quats=_lib.quat_gen(2)[:257], num_ave=200)
    fp = p['fparams']
    fp['beta'] = np.full(frames, 0.1)
    fp['scale'] = np.linspace(0.7, 1.4, frames)
    fp['blacklist'] = (np.arange(frames) % 3 == 1).astype('u1')
    fp['num_blacklist'] = int(fp['blacklist'].sum())
    flags = dict(iteration=2, need_scaling=1)
    o = P.run_oracle(p, flags)
    eng = P.engine_for(p)
    g = P.run_engine(eng, flags)
    eng.close()
    for k in ('likelihood', 'prob', 'model2', 'inter_weight'):
        assert P.rel_err(g[k], o[k]) <= 1e-9, k


@pytest.mark.parametrize('frames, beta', ((3, 1.), (40, 0.05)))
def test_merge_some_and_all_orientations(frames, beta):
    """Bright frames leave all but one orientation without any posterior, and so out of the merge;
    faint ones leave none out."""
    p = P.build(P.tiny_config(num_data=frames, mean_count=6000. if beta == 1. else 20.), num_ave=200)
    p['fparams']['beta'] = np.full(frames, beta)
    o = P.run_oracle(p, dict(iteration=1))
    assert (o['prob'].max(0) == 0.).any() == (beta == 1.)
    eng = P.engine_for(p)
    for merge_mode in (1, 0):
        eng.set_option('merge_mode', merge_mode)
        eng.maximize(1, 0, 1, 0)
        assert P.rel_err(eng.get('model2'), o['model2']) <= 1e-9, merge_mode
        assert P.rel_err(eng.get('inter_weight'), o['inter_weight']) <= 1e-9, merge_mode
    eng.close()


@pytest.mark.parametrize('size', (159, 160, 161, 162, 163))
def test_expand_from_brick_copy(size):
    """log W from model1 (159) and from its brick copy, with volumes that end at every place of a
    brick, with two models after one another."""
    # the problem builder makes detectors of odd sizes only: the detector is that of 159
    p = P.build(P.tiny_config(size=159, num_data=12, mean_count=60.), quats=_lib.quat_gen(2)[:70], num_ave=100)
    p['fparams']['beta'] = np.full(12, 0.05)
    eng = P.engine_for(p)
    rng = np.random.default_rng(size)
    for model in (rng.random((size,) * 3) + 0.1 for _ in range(2)):
        eng.set_model(model)
        o = P.run_oracle(p, dict(iteration=1), model1=model)
        g = P.run_engine(eng, dict(iteration=1))
        for k in ('u', 'max_exp', 'p_norm', 'likelihood', 'prob', 'model2'):
            assert P.rel_err(g[k], o[k]) <= 1e-9, k
    eng.close()
