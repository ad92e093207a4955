"""The inference renderer's one-ray-per-lane layout of fused and exact colours (samples queued per ray, evaluated cell by
cell) against the oracle and the group layout: T, traces and statistics bit-identical to the latter, rgb to rounding, at the
sizes and neighbourhoods where it branches: partial and several waves, neighbourhoods that are and are not multiples of four
and far beyond, rays whose queues fill at different times, no lit sample at all."""

import math

import numpy as np
import pytest
import torch

import oracle  # noqa: F401
from test_gpu_foam import compare, ref_foam
from test_gpu_foam_wide import HubField
from vgr import ext

pytestmark = pytest.mark.gpu

# indexed edge records, slot table, colour mode: exact colours (0) take this layout with both
CASES = [(False, False, 2), (False, True, 2), (True, False, 2), (True, True, 2), (True, True, 0)]


@pytest.fixture(scope='module')
def hub(gpu):
	f = HubField()
	sizes = np.diff(f.offsets) + 1
	assert sizes.max() > 32 and set(sizes % 4) == {0, 1, 2, 3}
	return f, f.rays(B=257, seed=11)


def run(dev, pk, deg, rays, tt, wt, mode, lanes=1, indexed=False, slots=False, cap=None, order=None, trace_cap=512,
		cut=math.inf):
	t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=dev)  # noqa: E731
	empty = torch.empty(0, dtype=torch.int32, device=dev)
	scene = [t(pk[k]) for k in ('points', 'offsets', 'nbr', 'edge', 'attr', 'sh')]
	orig = pk.get('orig')
	out = ext.foam_infer_extension().foam_infer(
		*scene, deg, *(t(a) for a in rays), tt, wt, cut, mode, 2, empty if cap is None else t(cap),
		t(orig) if orig is not None and len(orig) else empty, trace_cap=trace_cap, lanes=lanes,
		order=None if order is None else t(order), indexed=ext.index_pack(*scene[1:5]) if indexed else None,
		slots=ext.slot_table(scene[1], scene[2]) if slots else None)
	names = ('rgb', 'T', 'depth', 'stats', 'trace')[:len(out)]
	return {k: v.cpu().numpy() for k, v in zip(names, out)}


def check(g, two):
	"""Against two lanes per ray. The density of a cell is summed in another order there: T, and the samples' weights with it,
	agree to ulps (a ray that ends at a threshold may end one sample apart: none here)."""
	for k in ('stats', 'trace'):
		np.testing.assert_array_equal(g[k], two[k], err_msg=k)
	# colours of at most ~3, sums of at most ~50 terms in another order: a few ulps each
	for k in ('rgb', 'T', 'depth'):
		np.testing.assert_allclose(g[k], two[k], atol=1e-5, rtol=1e-6, err_msg=k)


@pytest.mark.parametrize('n_rays', [1, 63, 64, 65, 257])
@pytest.mark.parametrize('indexed,slots,mode', CASES)
def test_tile_layout(gpu, hub, n_rays, indexed, slots, mode):
	f, (o, d, start, near, _, far) = hub
	rays = tuple(a[:n_rays] for a in (o, d, start, near, far))
	pk = f.pack()
	for tt, wt in ((0.0, -1.0), (1e-4, 1e-4), (1e-4, 0.05), (1e-4, 2.0)):  # every segment lit ... none
		g = run(gpu, pk, 3, rays, tt, wt, mode, indexed=indexed, slots=slots)
		check(g, run(gpu, pk, 3, rays, tt, wt, mode, lanes=2))
		r = ref_foam(pk, 3, *rays, tt, wt, color_mode=mode, trace_cap=512)
		compare(g, r, exact_trace=tt == 0.0, stats_frac=1.0 if tt == 0.0 else 0.98, w_thresh=max(wt, 1e-4))
		if wt == 2.0:
			assert (g['rgb'] == 0).all() and (g['stats'][:, 1] == 0).all()


@pytest.mark.parametrize('sh_deg', [0, 1, 2, 3])
@pytest.mark.parametrize('sh_half', [False, True])
def test_tile_layout_degrees_orders_and_caps(gpu, hub, sh_deg, sh_half):
	"""SH degrees and types, a renumbered pack, sample caps, an order of the rays (bit-identical rays, whatever wave they fall
	in), starts outside the scene."""
	f, (o, d, start, near, _, far) = hub
	pk = f.pack(sh_half=sh_half, reorder=True)
	st = pk['inv'][start].astype(np.int32)
	st[:3] = [-1, f.n, 2 ** 30]
	rays = (o, d, st, near, far)
	cap = np.arange(len(o), dtype=np.int32) % 40 + 2
	order = np.random.default_rng(1).permutation(len(o)).astype(np.int32)
	for indexed, slots, mode in CASES:
		kw = dict(indexed=indexed, slots=slots, cap=cap)
		g = run(gpu, pk, sh_deg, rays, 1e-4, 1e-4, mode, **kw)
		check(g, run(gpu, pk, sh_deg, rays, 1e-4, 1e-4, mode, lanes=2, cap=cap))
		h = run(gpu, pk, sh_deg, rays, 1e-4, 1e-4, mode, order=order, **kw)
		for k in g:
			np.testing.assert_array_equal(h[k].view(np.int32), g[k].view(np.int32), err_msg=k)
		assert (g['T'][:3] == 1).all() and (g['rgb'][:3] == 0).all() and (g['stats'][:3] == 0).all()


@pytest.mark.parametrize('n_rays', [1, 65, 257])
@pytest.mark.parametrize('indexed', [False, True])
@pytest.mark.parametrize('sh_half', [False, True])
@pytest.mark.parametrize('cut', [0.0, 2.0, 2 * math.log(1e3)])
def test_tile_layout_cut_off(gpu, hub, n_rays, indexed, sh_half, cut):
	"""A finite cut-off admits a term against the running minimum of the terms before it: the counted lookups and the
	colours against the oracle and the 16-lane layout, which decide the same way in the same order."""
	f, (o, d, start, near, _, far) = hub
	rays = tuple(a[:n_rays] for a in (o, d, start, near, far))
	pk = f.pack(eps_density=1e-3, sh_half=sh_half)
	for tt, wt in ((0.0, -1.0), (1e-4, 0.05)):
		g = run(gpu, pk, 3, rays, tt, wt, 2, indexed=indexed, cut=cut)
		wide = run(gpu, pk, 3, rays, tt, wt, 2, lanes=None, cut=cut)
		for k in ('T', 'stats', 'trace'):
			np.testing.assert_array_equal(g[k].view(np.int32), wide[k].view(np.int32), err_msg=k)
		np.testing.assert_allclose(g['rgb'], wide['rgb'], atol=1e-5, rtol=0)  # as in check
		r = ref_foam(pk, 3, *rays, tt, wt, color_cut=cut, color_mode=2, trace_cap=512)
		compare(g, r, exact_trace=tt == 0.0, stats_frac=0.98, w_thresh=max(wt, 1e-4))


@pytest.mark.parametrize('sh_half', [False, True])
@pytest.mark.parametrize('indexed', [False, True])
def test_terms_left_out_add_nothing(gpu, hub, sh_half, indexed):
	"""A term left out of a blend adds nothing whatever its colour is: sites of infinite colour (fp16 SH past 65504) beyond
	the cut-off of a ray's samples, and cells whose terms are all left out (conics of infinities: distances NaN), whose
	colour is 0 / 0 as in the other layouts. Against 16 lanes per ray, which skip those terms."""
	f, (o, d, start, near, _, far) = hub
	rays = (o, d, start, near, far)
	pk = f.pack(eps_density=1e-3, sh_half=sh_half)
	pk['sh'] = pk['sh'].copy()  # the field's own array
	pk['sh'][::23, 0] = np.inf
	kw = dict(indexed=indexed, cut=0.5)
	g, wide = run(gpu, pk, 3, rays, 1e-4, 1e-3, 2, **kw), run(gpu, pk, 3, rays, 1e-4, 1e-3, 2, lanes=None, cut=0.5)
	ok = np.isfinite(wide['rgb'])  # the others: an infinite term that counts, as inf or, if its weight underflows, NaN
	assert not ok.all() and ok.all(1).sum() > 20
	np.testing.assert_array_equal(np.isfinite(g['rgb']), ok)
	np.testing.assert_allclose(g['rgb'][ok], wide['rgb'][ok], atol=1e-5, rtol=1e-6)  # as in check
	pk = f.pack(eps_density=1e-3, sh_half=sh_half)
	inside = np.abs(f.points).max(1) < 0.45  # whole neighbourhoods of these sites
	pk['attr'][inside, 8:14] = np.inf
	for cut in (math.inf, 2 * math.log(1e3)):
		kw = dict(indexed=indexed, cut=cut)
		g, wide = run(gpu, pk, 3, rays, 1e-4, 1e-3, 2, **kw), run(gpu, pk, 3, rays, 1e-4, 1e-3, 2, lanes=None, cut=cut)
		bad = np.isnan(wide['rgb']).any(1)
		assert bad.any() and not bad.all()
		np.testing.assert_allclose(g['rgb'], wide['rgb'], atol=1e-5, rtol=1e-6)


@pytest.mark.parametrize('indexed,slots,mode', CASES)
@pytest.mark.parametrize('reorder', [False, True])
def test_lookups_whose_distance_is_no_number(gpu, hub, indexed, slots, mode, reorder):
	"""Without a cut-off the counted lookups are the entries whose colour distance is a number: all, except beside sites of
	degenerate colour conics (all or one coefficient not finite, or finite ones whose distance overflows) and at samples so
	far out, or at no place at all, that distances overflow. The same counts as 16 lanes per ray, which look entry by entry,
	so that a batch's size does not change them; the oracle's for fused colours and the conics."""
	f, (o, d, start, near, _, far) = hub
	pk = f.pack(reorder=reorder)
	start = pk['inv'][start].astype(np.int32) if reorder else start
	pk['attr'][5::37, 8:14] = np.inf
	pk['attr'][7::41, 9] = np.nan
	pk['attr'][11::43, 8] = 3e38
	rays = (o, d, start, near, far)
	all_entries = run(gpu, f.pack(reorder=reorder), 3, rays, 0.0, -1.0, mode, indexed=indexed, slots=slots)['stats']
	for tt, wt in ((0.0, -1.0), (1e-4, 1e-3)):
		g = run(gpu, pk, 3, rays, tt, wt, mode, indexed=indexed, slots=slots)
		wide = run(gpu, pk, 3, rays, tt, wt, mode, lanes=None)
		np.testing.assert_array_equal(g['stats'], wide['stats'])
	g = run(gpu, pk, 3, rays, 0.0, -1.0, mode, indexed=indexed, slots=slots)
	assert (g['stats'][:, 4] < all_entries[:, 4]).sum() > 50
	if mode == 2:  # the oracle's two-pass exact colours take such a term in, and are NaN
		np.testing.assert_array_equal(g['stats'], ref_foam(pk, 3, *rays, 0.0, -1.0, color_mode=2)['stats'])
	out = far.copy()
	out[::3], out[1::5], out[2::7] = 3e19, np.inf, np.nan
	g = run(gpu, pk, 3, (o, d, start, near, out), 0.0, -1.0, mode, indexed=indexed, slots=slots)
	wide = run(gpu, pk, 3, (o, d, start, near, out), 0.0, -1.0, mode, lanes=None)
	np.testing.assert_array_equal(g['stats'], wide['stats'])
