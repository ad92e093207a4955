"""The inference renderer's 16-lanes-per-ray layout (the default of the full rendering for small batches) against the
oracle and against the one-ray-per-lane layout: T, traces and statistics bit-identical to the latter, rgb to rounding, at the
sizes and neighbourhoods where the layout branches (partial waves, neighbourhoods of up to 16, of 17 to 32 and beyond 32
entries, which the group loops over)."""

import math

import numpy as np
import pytest
import torch

import oracle  # noqa: F401
from helpers import Field, cKDTree
from test_gpu_foam import compare, gpu_foam, ref_foam
from vgr import render
from vgr.sites import delaunay_graph

pytestmark = pytest.mark.gpu

CUT = 2 * math.log(1e3)


class HubField(Field):
	"""A random field with hub sites: the centres of empty balls, each a neighbour of the ~50 sites on its sphere."""

	def __init__(self, seed=3, n=300):
		super().__init__(seed=seed, n=n)
		rng = np.random.default_rng(seed)
		centres = np.array([[0.0, 0.0, 0.0], [0.45, 0.4, -0.3]])
		pts = self.points[np.all(np.linalg.norm(self.points[:, None] - centres, axis=2) > 0.3, 1)].astype(np.float64)
		for c in centres:
			u = rng.normal(size=(50, 3))
			pts = np.concatenate([pts, c[None], c + 0.22 * u / np.linalg.norm(u, axis=1, keepdims=True)])
		keep = rng.permutation(len(pts))[:len(self.points)]
		hubs = [np.abs(pts - c).sum(1).argmin() for c in centres]
		keep = np.unique(np.concatenate([keep, hubs]))
		pts, _, self.offsets, self.adj = delaunay_graph(pts[keep].astype(np.float32).astype(np.float64))
		self.points = pts.astype(np.float32)
		n = len(pts)
		self.raw = (rng.normal(size=n) * 0.5 + 1.0).astype(np.float32)
		for name in ('d', 'c'):
			setattr(self, name + '_log_scale', (rng.normal(size=(n, 3)) * 0.3 - 1.8).astype(np.float32))
			setattr(self, name + '_quat', rng.normal(size=(n, 4)).astype(np.float32))
		self.sh = (rng.normal(size=(n, 16, 3)) * 0.3).astype(np.float32)
		self.tree = cKDTree(self.points)


@pytest.fixture(scope='module')
def hub(gpu):
	f = HubField()
	sizes = np.diff(f.offsets) + 1
	assert sizes.max() > 32 and (sizes <= 16).any() and ((sizes > 16) & (sizes <= 32)).any()
	o, d, start, near, _, far = f.rays(B=257, seed=7)
	return f, (o, d, start, near, far)


def baked(f, pk):
	v = f.points - np.array([0.1, 0.2, 2.5], np.float32)
	b = render.sh_basis(torch.from_numpy((v / np.linalg.norm(v, axis=1, keepdims=True)).astype(np.float32)), 3).numpy()
	return np.maximum((b[:, :, None] * f.sh).sum(1) + 0.5, 0)


@pytest.mark.parametrize('n_rays', [1, 3, 4, 5, 64, 257])
@pytest.mark.parametrize('mode,cut', [(0, math.inf), (2, math.inf), (1, math.inf), (0, CUT), (2, CUT), (1, CUT)])
def test_wide_layout(gpu, hub, n_rays, mode, cut):
	f, rays = hub
	o, d, start, near, far = (a[:n_rays] for a in rays)
	pk = f.pack(eps_density=0.0 if cut == math.inf else 1e-3)
	pk['attr'][:, 16:19] = baked(f, pk)
	for tt, wt in ((0.0, -1.0), (1e-4, 1e-4)):
		kw = dict(t_thresh=tt, w_thresh=wt, color_cut=cut, color_mode=mode, trace_cap=512)
		g = gpu_foam(gpu, pk, 3, o, d, start, near, far, **kw)
		one = gpu_foam(gpu, pk, 3, o, d, start, near, far, lanes=1, **kw)
		for k in ('T', 'stats', 'trace'):
			np.testing.assert_array_equal(g[k].view(np.int32), one[k].view(np.int32), err_msg=k)
		# colours of at most ~3, sums of at most ~50 terms in another order: a few ulps each
		np.testing.assert_allclose(g['rgb'], one['rgb'], atol=1e-5, rtol=0)
		np.testing.assert_allclose(g['depth'], one['depth'], atol=1e-5, rtol=1e-6)
		r = ref_foam(pk, 3, o, d, start, near, far, tt, wt, color_cut=cut, color_mode=mode, trace_cap=512)
		compare(g, r, exact_trace=tt == 0.0, stats_frac=1.0 if tt == 0.0 else 0.98)


@pytest.mark.parametrize('sh_deg', [0, 1, 2, 3])
@pytest.mark.parametrize('sh_half', [False, True])
def test_wide_layout_degrees_orders_and_caps(gpu, hub, sh_deg, sh_half):
	"""SH degrees and types, a renumbered pack, a sample cap, starts outside the scene and terms whose colour distance is
	NaN (a conic of infinities), which every layout leaves out of its colours and its count of lookups."""
	f, (o, d, start, near, far) = hub
	pk = f.pack(sh_half=sh_half, reorder=True)
	pk['attr'][5::37, 8:14] = np.inf
	st = pk['inv'][start].astype(np.int32)
	st[:3] = [-1, f.n, 2 ** 30]
	cap = np.arange(len(o), dtype=np.int32) % 40 + 2
	for mode in (0, 2):
		for c in (None, cap):
			kw = dict(color_mode=mode, cap=c, trace_cap=128)
			g = gpu_foam(gpu, pk, sh_deg, o, d, st, near, far, **kw)
			one = gpu_foam(gpu, pk, sh_deg, o, d, st, near, far, lanes=1, **kw)
			for k in ('T', 'stats', 'trace'):
				np.testing.assert_array_equal(g[k].view(np.int32), one[k].view(np.int32), err_msg=k)
			np.testing.assert_allclose(g['rgb'], one['rgb'], atol=1e-5, rtol=0)
			assert (g['T'][:3] == 1).all() and (g['rgb'][:3] == 0).all() and (g['stats'][:3] == 0).all()
