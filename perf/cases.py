"""The work that is timed: what a user of this framework has it do, through its public entry points.

A field is a cube of sites [-1, 1]^3 under a rotation of its own, with Delaunay neighbourhoods, anisotropic density and
colour Gaussians, and SH colours. Its geometry repeats one periodic Delaunay tile K x K x K times (K^3 * 2048 sites, so
that 2M sites need no triangulation of their own); rotation, site numbering, every attribute, the cameras and the rays
come from the seed. Sizes and distributions follow the benchmark scenes (scenes.py): clustered and uniform sites,
densities softplus(N(1, 1)) ("object"), opaque shells in thin air ("surface") and softplus(N(-4, 0.5)) ("thin"), SH
N(0, 0.5) and N(0, 0.05), orbit cameras of radius 3 and 60 degrees.

  infer     render_rays_foam_infer on a packed scene: evaluation and viewing (exact, fused, fast and baked colours)
  batch     foam_infer on an incoherent ray batch in ray_order, 8 lanes per ray: visibility and depth queries
  foam      render_rays_foam forward and backward: a training step's renderer
  uniform   render_rays_uniform forward and backward: the other training renderer
  march     render_rays_uniform without gradients: a view by the uniform march
  fields    walk, density and colour operators forward and backward: the NeRF-style sampler's layers
  pack      pack_foam: a model made ready for inference
  locate    nearest_sites: the start site of every ray of a batch
"""

import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'voronoi-gauss_amd'))

from vgr import ext, render, sites  # noqa: E402
from vgr.model import VoronoiGaussField  # noqa: E402

TILE = 2048  # sites of one periodic tile
NEAR, T_THRESH, W_THRESH, DT, N_BG, FAR = 0.02, 1e-4, 1e-4, 1 / 512, 64, 4.0
PARAMS = ('raw', 'd_log_scale', 'd_quat', 'c_log_scale', 'c_quat', 'sh_dc', 'sh_rest')


def listed():
	return [
		# one chunk of render_image (its default of 8192 rays), reference colours: the smallest rendering call
		dict(name='chunk-8192-exact', op='infer', k=4, geo='clusters', dens='object', deg=3, w=800, h=800, rays=8192,
			 colors='exact', half=False, eps=0.0, tiles=False),
		# evaluation of one 800 x 800 view of a medium object scene in the reference's default colour mode
		dict(name='view-800-exact', op='infer', k=6, geo='clusters', dens='object', deg=3, w=800, h=800, rays=640000,
			 colors='exact', half=False, eps=0.0, tiles=True),
		# one 1080p frame of a 2M-site surface scene, as the headline benchmark renders it
		dict(name='view-1080p-fused', op='infer', k=10, geo='clusters', dens='surface', deg=3, w=1920, h=1080,
			 rays=1920 * 1080, colors='fused', half=False, eps=0.0, tiles=True),
		# the fast settings (fp16 SH, cut-offs 1e-3) on an odd-sized photograph in pixel order
		dict(name='view-odd-fast', op='infer', k=8, geo='uniform', dens='surface', deg=3, w=1237, h=822,
			 rays=1237 * 822, colors='fused', half=True, eps=1e-3, tiles=False),
		# interactive viewing: a bake for the camera, then the view with baked colours
		dict(name='view-800-baked', op='infer', k=8, geo='clusters', dens='surface', deg=3, w=800, h=800, rays=640000,
			 colors='baked', half=False, eps=0.0, tiles=True),
		# incoherent rays through a thin scene without early termination (ambient visibility, depth queries)
		dict(name='batch-incoherent', op='batch', k=8, geo='uniform', dens='thin', deg=3, rays=500009),
		# a training step of the default renderer: 4096 random pixels, gradients of every parameter
		dict(name='train-foam-4096', op='foam', k=6, geo='clusters', dens='surface', deg=3, rays=4096),
		# the same with the uniform march, early in training: translucent everywhere, SH degree 1 in use
		dict(name='train-uniform-4096', op='uniform', k=5, geo='uniform', dens='object', deg=1, rays=4096),
		# the layers of the NeRF-style sampler on a training batch, 64 samples per ray
		dict(name='train-fields-4096', op='fields', k=6, geo='clusters', dens='object', deg=3, rays=4096, samples=64),
		# a view by the uniform march
		dict(name='march-400', op='march', k=8, geo='uniform', dens='surface', deg=3, w=400, h=400, rays=160000),
		# a trained model made ready for inference, renumbered
		dict(name='pack-2M', op='pack', k=10, geo='clusters', dens='surface', deg=3),
		# start sites of a million ray origins
		dict(name='locate-1M', op='locate', k=8, geo='uniform', dens='thin', deg=0, rays=1000003),
	]


def _log_int(rng, lo, hi):
	return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
	op = rng.choice(['infer', 'infer', 'infer', 'infer', 'batch', 'foam', 'foam', 'uniform', 'march', 'fields', 'pack',
					 'locate'])
	c = dict(op=op, k=rng.randint(2, 8), geo=rng.choice(['clusters', 'uniform']),
			 dens=rng.choice(['object', 'surface', 'thin']), deg=rng.choice([0, 1, 2, 3, 3, 3]))
	if op == 'infer':
		w, h = _log_int(rng, 64, 1400), _log_int(rng, 64, 1100)
		c.update(w=w, h=h, rays=rng.choice([w * h, min(w * h, 8192), _log_int(rng, 256, w * h)]),
				 colors=rng.choice(['exact', 'exact', 'fused', 'fused', 'baked']), half=rng.random() < 0.25,
				 eps=rng.choice([0.0, 0.0, 0.0, 1e-3]), tiles=rng.random() < 0.5)
	elif op == 'batch':
		c.update(rays=_log_int(rng, 4096, 400000))
	elif op in ('foam', 'uniform'):
		c.update(rays=_log_int(rng, 512, 16384 if op == 'foam' else 8192))
	elif op == 'march':
		w, h = _log_int(rng, 32, 400), _log_int(rng, 32, 400)
		c.update(w=w, h=h, rays=w * h)
	elif op == 'fields':
		c.update(rays=_log_int(rng, 256, 8192), samples=rng.choice([32, 64, 96]))
	elif op == 'locate':
		c.update(rays=_log_int(rng, 1000, 1000000))
	return c


# --------------------------------------------------------------------------------------------------------- scenes

@functools.lru_cache(maxsize=None)
def _tile(geo):
	"""One periodic tile in [0, 1)^3: points (n, 3), edges (i, j, s) of its periodic Delaunay graph sorted by i (site i
	neighbours site j of the tile at shift s in {-1, 0, 1}^3), both directions, and the mean distance to 3 neighbours."""
	rng = np.random.default_rng(7)
	p = rng.uniform(0, 1, (TILE, 3))
	if geo == 'clusters':
		m = int(0.6 * TILE)
		c = rng.integers(0, 6, m)
		p[:m] = rng.uniform(0, 1, (6, 3))[c] + rng.uniform(0.08, 0.25, 6)[c, None] * rng.normal(size=(m, 3))
		p = np.mod(p, 1.0)
	p = p.astype(np.float32).astype(np.float64)
	shifts = np.array([(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1)])
	q = (p[None] + shifts[:, None]).reshape(-1, 3)
	tag = np.stack([np.tile(np.arange(TILE), 27), np.repeat(np.arange(27), TILE)], 1)
	keep = np.all((q > -0.3) & (q < 1.3), 1)
	q, tag = q[keep], tag[keep]
	kept, idx, off, adj = sites.delaunay_graph(q)
	tag = tag[idx]
	own = np.repeat(np.arange(len(kept)), np.diff(off))
	base = tag[own, 1] == 13
	i, j, s = tag[own[base], 0], tag[adj[base], 0], shifts[tag[adj[base], 1]]
	both = np.concatenate([np.concatenate([i[:, None], j[:, None], s], 1), np.concatenate([j[:, None], i[:, None], -s], 1)])
	e = np.unique(both, axis=0)
	sp = np.full(TILE, np.inf)
	d = np.linalg.norm(p[e[:, 0]] - (p[e[:, 1]] + e[:, 2:]), axis=1)
	order = np.lexsort((d, e[:, 0]))
	rank = np.arange(len(e)) - np.searchsorted(e[:, 0], e[:, 0])
	near = np.zeros(TILE)
	np.add.at(near, e[order, 0], np.where(rank < 3, d[order], 0.0))
	sp = near / 3
	return p, e, sp


def _softplus(x):
	return torch.nn.functional.softplus(x)


def _gen(seed):
	g = torch.Generator(device='cuda')
	g.manual_seed(int(seed))
	return g


def _field(case, seed):
	"""-> points (N, 3), offsets, adj (CSR, int32), the parameters (PARAMS), all on the GPU."""
	g, dev, k = _gen(seed), 'cuda', case['k']
	p, e, sp = (torch.from_numpy(a).to(dev) for a in _tile(case['geo']))
	n_tiles, n = k ** 3, TILE * k ** 3

	def normal(*shape):
		return torch.randn(*shape, generator=g, device=dev)

	t = torch.arange(n_tiles, device=dev)
	tc = torch.stack([t // (k * k), t // k % k, t % k], 1)
	pts = ((p[None] + tc[:, None]).reshape(-1, 3) * (2.0 / k) - 1.0)
	rot = torch.linalg.qr(torch.randn(3, 3, generator=g, device=dev, dtype=torch.float64))[0]
	pts = (pts @ rot).float()
	spacing = (sp * (2.0 / k)).float().repeat(n_tiles)
	# the tiles' edges: inside the cube only
	nt = tc[:, None] + e[None, :, 2:]
	inside = ((nt >= 0) & (nt < k)).all(-1).reshape(-1)
	dst = (((nt[..., 0] * k + nt[..., 1]) * k + nt[..., 2]) * TILE + e[None, :, 1]).reshape(-1)[inside]
	src = (t[:, None] * TILE + e[None, :, 0]).reshape(-1)[inside]
	del nt, inside
	# a random numbering of the sites, as a point cloud comes
	perm = torch.randperm(n, generator=g, device=dev)  # new -> old
	inv = torch.empty_like(perm)
	inv[perm] = torch.arange(n, device=dev)
	deg = torch.bincount(src, minlength=n)
	first = torch.cumsum(deg, 0) - deg
	deg_new = deg[perm]
	off = torch.nn.functional.pad(torch.cumsum(deg_new, 0), (1, 0))
	row = torch.repeat_interleave(torch.arange(n, device=dev), deg_new, output_size=src.numel())
	order = torch.argsort(src, stable=True)  # tile-major edges, per old site
	adj = inv[dst[order[first[perm][row] + torch.arange(src.numel(), device=dev) - off[row]]]].int()
	del src, dst, row, order
	pts, spacing = pts[perm].contiguous(), spacing[perm]
	mean = 2.0 / n ** (1 / 3)
	if case['dens'] == 'object':
		rho = _softplus(normal(n) + 1.0) * (0.02 / mean)
	elif case['dens'] == 'thin':
		rho = _softplus(0.5 * normal(n) - 4.0)
	else:
		r = pts.norm(dim=1)
		ring = torch.sqrt((pts[:, :2].norm(dim=1) - 0.6) ** 2 + pts[:, 2] ** 2)
		on = ((r - 0.8).abs() < 2.5 * mean) & (pts[:, 0] > -0.3) | ((ring - 0.15).abs() < 2.5 * mean)
		rho = torch.where(on, _softplus(0.5 * normal(n) + 4.0) * (0.1 / mean), _softplus(0.5 * normal(n) - 3.0))
	log_s = spacing.log().unsqueeze(1)
	sh_rest = 0.05 * normal(n, 15, 3)
	sh_rest[:, (case['deg'] + 1) ** 2 - 1:] = 0
	par = {'raw': rho.log(), 'd_log_scale': log_s + 0.3 * normal(n, 3), 'd_quat': normal(n, 4),
		   'c_log_scale': log_s + 0.3 * normal(n, 3), 'c_quat': normal(n, 4), 'sh_dc': 0.5 * normal(n, 1, 3),
		   'sh_rest': sh_rest}
	return pts, off.int(), adj, {k_: v.contiguous() for k_, v in par.items()}


def _model(case, seed, grad=False):
	pts, off, adj, par = _field(case, seed)
	n = len(pts)
	m = VoronoiGaussField(pts, off, adj, torch.zeros(n, 3, device='cuda'), torch.ones(n, device='cuda'))
	with torch.no_grad():
		for name, v in par.items():
			getattr(m, name).copy_(v)
	m.sh_deg = case['deg']
	m.requires_grad_(grad)
	return m


def _camera(g):
	"""An orbit camera of radius 3 looking at the origin: eye (3,), axes (3, 3) as columns right, down, forward."""
	a, b = (torch.rand(2, generator=g, device='cuda', dtype=torch.float64) * torch.tensor([2 * math.pi, 0.8],
			device='cuda', dtype=torch.float64)).tolist()
	eye = 3.0 * np.array([math.cos(b) * math.cos(a), math.sin(b), math.cos(b) * math.sin(a)])
	f = -eye / 3.0
	r = np.cross(f, [0.0, 1.0, 0.0])
	r /= np.linalg.norm(r)
	return eye, np.stack([r, np.cross(f, r), f], 1)


def _pixels(cam, w, h, x, y):
	eye, axes = cam
	fx = 0.5 * w / math.tan(math.radians(30))
	v = torch.stack([(x + 0.5 - 0.5 * w) / fx, (y + 0.5 - 0.5 * h) / fx, torch.ones_like(x)], -1)
	d = v @ torch.from_numpy(axes.T.copy()).to(v.device)
	d = d / d.norm(dim=-1, keepdim=True)
	return torch.from_numpy(eye).to(d).expand_as(d).float().contiguous(), d.float().contiguous()


def _view(cam, w, h, count, tiles):
	"""`count` rays of a w x h view around its middle rows: in pixel order, or in 8 x 8 tiles along their Z-order."""
	i = torch.arange(w * h, device='cuda')
	if tiles:
		y, x = i // w, i % w
		key = torch.zeros_like(i)
		for b in range(9):
			key |= (((x // 8) >> b & 1) << 2 * b) | (((y // 8) >> b & 1) << (2 * b + 1))
		i = torch.argsort(key * 64 + (y % 8) * 8 + x % 8, stable=True)
	a = (w * h - count) // 2
	i = i[a:a + count]
	return _pixels(cam, w, h, (i % w).double(), (i // w).double())


def _nearest_one(pts, q):
	return int(((pts.double() - torch.as_tensor(q, device=pts.device, dtype=torch.float64)) ** 2).sum(1).argmin())


def _training_rays(case, seed, pts):
	"""Random pixels of 8 cameras of 800 x 800, mixed, each from the site nearest to its camera."""
	g, b = _gen(seed + 77), case['rays']
	cams = [_camera(g) for _ in range(8)]
	which = torch.randint(8, (b,), generator=g, device='cuda')
	x, y = (torch.randint(800, (b,), generator=g, device='cuda').double() for _ in range(2))
	o, d = torch.empty(b, 3, device='cuda'), torch.empty(b, 3, device='cuda')
	start = torch.empty(b, dtype=torch.int32, device='cuda')
	for c, cam in enumerate(cams):
		m = which == c
		o[m], d[m] = _pixels(cam, 800, 800, x[m], y[m])
		start[m] = _nearest_one(pts, cam[0])
	return o, d, start, torch.rand(b, 3, generator=g, device='cuda')


def _inside_rays(case, seed, pts):
	"""Origins and directions of an incoherent batch inside the cube: uniform in a ball of radius 0.9, on the sphere."""
	g, b = _gen(seed + 78), case['rays']
	o = torch.randn(b, 3, generator=g, device='cuda')
	o = 0.9 * o / o.norm(dim=1, keepdim=True) * torch.rand(b, 1, generator=g, device='cuda') ** (1 / 3)
	d = torch.randn(b, 3, generator=g, device='cuda')
	return o.contiguous(), (d / d.norm(dim=1, keepdim=True)).contiguous()


def _some_start(o, pts, g):
	"""A site near each origin: the nearest of 4096 spread sites (the renderer walks on from it)."""
	some = torch.randperm(len(pts), generator=g, device='cuda')[:4096]
	return torch.cat([some[torch.cdist(o[a:a + 65536], pts[some]).argmin(1)] for a in range(0, len(o), 65536)]).int()


# -------------------------------------------------------------------------------------------------- prepare and run

def prepare(case, seed):
	op = case['op']
	if op == 'locate':
		pts = _field(case, seed)[0]
		return dict(op=op, points=pts, queries=_inside_rays(case, seed, pts)[0])
	m = _model(case, seed, grad=op in ('foam', 'uniform', 'fields'))
	pts = m.graph.points
	st = dict(op=op, model=m, case=case)
	if op in ('infer', 'march'):
		cam = _camera(_gen(seed + 5))
		st['eye'] = torch.tensor(cam[0], dtype=torch.float32, device='cuda')
		st['o'], st['d'] = _view(cam, case['w'], case['h'], case['rays'], case.get('tiles', True))
		st['start'] = torch.full((case['rays'],), _nearest_one(pts, cam[0]), dtype=torch.int32, device='cuda')
	if op in ('infer', 'batch'):
		st['pack'] = render.pack_foam(m, eps_density=case.get('eps', 0.0), sh_half=case.get('half', False), reorder=True)
	if op == 'batch':
		o, d = _inside_rays(case, seed, pts)
		start = _some_start(o, pts, _gen(seed + 9))
		near, _, far = render.ray_bounds(o, d, NEAR, FAR)
		st.update(o=o, d=d, start=st['pack']['inv'][start.long()].int(), near=near.contiguous(), far=far.contiguous(),
				  empty=torch.empty(0, dtype=torch.int32, device='cuda'))
	if op in ('foam', 'uniform'):
		st['o'], st['d'], st['start'], st['gt'] = _training_rays(case, seed, pts)
	if op == 'fields':
		o, d, start, gt = _training_rays(case, seed, pts)
		g = _gen(seed + 6)
		b, s = case['rays'], case['samples']
		z = 2.0 + 2.0 * torch.sort(torch.rand(b, s, generator=g, device='cuda'), 1)[0]
		x = (o.unsqueeze(1) + d.unsqueeze(1) * z.unsqueeze(-1)).reshape(-1, 3).contiguous()
		# a third of the samples carry weight and get a colour
		lit = torch.sort(torch.randperm(b * s, generator=g, device='cuda')[:b * s // 3])[0]
		dirs = d.unsqueeze(1).expand(b, s, 3).reshape(-1, 3)[lit].contiguous()
		st.update(o=o, d=d, start=start, z=z, x=x, lit=lit, x_lit=x[lit].contiguous(), dirs=dirs, sh=m.sh().detach().requires_grad_(),
				  g_sigma=torch.randn(b * s, generator=g, device='cuda') / (b * s),
				  g_rgb=torch.randn(len(lit), 3, generator=g, device='cuda') / len(lit))
	return st


def _grads(m, names):
	return {n: getattr(m, n).grad for n in names}


def run(st):
	op = st['op']
	if op == 'locate':
		return sites.nearest_sites(st['points'], st['queries'])
	m, c = st['model'], st['case']
	if op == 'infer':
		if c['colors'] == 'baked':
			render.bake_colors(m, st['pack'], st['eye'])
		return render.render_rays_foam_infer(m, st['pack'], st['o'], st['d'], st['start'], near=NEAR, far_radius=FAR,
											 t_thresh=T_THRESH, w_thresh=W_THRESH, colors=c['colors'],
											 eps_color=c['eps'])
	if op == 'batch':
		p = st['pack']
		order = ext.ray_order(st['o'], st['d'])
		rgb, T, depth, stats = ext.foam_infer_extension().foam_infer(
			p['points'], p['offsets'], p['nbr'], p['edge'], p['attr'], p['sh'], m.sh_deg, st['o'], st['d'], st['start'],
			st['near'], st['far'], T_THRESH, W_THRESH, math.inf, 2, 2, st['empty'], p['orig'], lanes=8, order=order,
			indexed=(p['edge_i'], p['attr_i'], p['rows']))
		return {'rgb': rgb, 'T': T, 'depth': depth, 'stats': stats}
	if op == 'pack':
		p = render.pack_foam(m, reorder=True)
		bits = {k: p[k].view(torch.int32) for k in ('edge', 'edge_i', 'points')}
		return {**bits, **{k: p[k] for k in ('offsets', 'nbr', 'sh', 'slots', 'perm')}, 'conics': p['attr'][:, :14],
				'rows': p['rows'][:, :7]}
	if op == 'march':
		with torch.no_grad():
			r = render.render_rays_uniform(m, st['o'], st['d'], st['start'], dt=DT, n_bg=N_BG, near=NEAR, far_radius=FAR,
										   t_thresh=T_THRESH, w_thresh=W_THRESH)
		return {k: r[k] for k in ('rgb', 'acc', 'depth', 'samples')}
	m.zero_grad(set_to_none=True)
	if op == 'fields':
		st['sh'].grad = None
		site = m.walk(st['o'], st['d'], st['z'], st['start'])[0].reshape(-1)
		sigma = ext.density(m.graph, m.raw, m.d_log_scale, m.d_quat, st['x'], site)
		rgb = ext.color(m.graph, m.c_log_scale, m.c_quat, st['sh'], st['x_lit'], st['dirs'], site[st['lit']], m.sh_deg)
		torch.autograd.backward([sigma, rgb], [st['g_sigma'], st['g_rgb']])
		return {'site': site, 'sigma': sigma.detach(), 'rgb': rgb.detach(), 'g_sh': st['sh'].grad,
				**_grads(m, PARAMS[:5])}
	if op == 'foam':
		r = render.render_rays_foam(m, st['o'], st['d'], st['start'], near=NEAR, far_radius=FAR, t_thresh=T_THRESH,
									w_thresh=W_THRESH)
	else:
		r = render.render_rays_uniform(m, st['o'], st['d'], st['start'], dt=DT, n_bg=N_BG, near=NEAR, far_radius=FAR,
									   t_thresh=T_THRESH, w_thresh=W_THRESH)
	loss = torch.nn.functional.mse_loss(r['rgb'], st['gt'])
	loss.backward()
	return {'rgb': r['rgb'].detach(), 'acc': r['acc'].detach(), 'depth': r['depth'].detach(), 'loss': loss.detach(),
			'bg': m.bg_logit.grad, **_grads(m, PARAMS)}


# -------------------------------------------------------------------------------------------------- work, tolerance

def _samples(case):
	"""Samples that a ray of this case takes, roughly: the cells (or steps) along its path until it is opaque."""
	if case['op'] in ('uniform', 'march'):
		return 500.0
	path = {'object': 20.0, 'surface': 19.0, 'thin': 21.0}[case['dens']]
	return path * (0.5 if case['op'] == 'batch' else 1.0) * case['k']


def work(case):
	op, n = case['op'], TILE * case['k'] ** 3
	edges, nb = 16.4 * n, 3 * (case['deg'] + 1) ** 2
	if op == 'pack':
		# parameters, points and CSR read once; pack, indexed records, slot table and site blocks written once
		return {'bytes': n * 4.0 * (3 + 1 + 14 + 48) + 4.0 * edges + n * 4.0 * (4 + 20 + 48 + 20 + 16 + 64) + edges * 4.0 * 9,
				'flops': 250.0 * n}
	if op == 'locate':
		return {'bytes': 12.0 * n + 16.0 * case['rays'], 'flops': 40.0 * 8 * case['rays']}
	site = 4.0 * (3 + 1 + 14 + nb) * n + 4.0 * edges
	visits = case['rays'] * 16.4
	if op == 'fields':
		visits *= case['samples']
		return {'bytes': 2 * site + 40.0 * case['rays'] * case['samples'],
				'flops': visits * (3 * 60 + (2 * nb + 120))}
	visits *= _samples(case)
	per = 70 + (2 * nb + 20 if case.get('colors') != 'baked' else 20)
	if op in ('foam', 'uniform'):
		return {'bytes': 2 * site + 100.0 * case['rays'], 'flops': 3 * visits * per}
	return {'bytes': site + 60.0 * case['rays'], 'flops': visits * per}


def tolerance(case):
	"""32-bit sums in another order move colours by 1e-6; a segment whose weight lies within rounding of W_THRESH is
	coloured or not, which moves its ray by 1e-4 and a count by one. Gradients are sums with cancellation over Gaussians
	far narrower than the distance to the camera: 1e-4 of them is rounding of the sample points."""
	op = case['op']
	if op == 'locate':
		return 'exact'
	if op == 'pack':
		return {'rel': 2e-6, 'max': 1e-4, 'differ': 1e-5}
	if op in ('foam', 'uniform'):
		return {'rel': 2e-3, 'max': 0.1, 'differ': 1e-3}
	if op == 'fields':
		return {'rel': 5e-4, 'max': 5e-2, 'differ': 1e-6}
	return {'rel': 1e-4, 'max': 1e-2, 'differ': 1e-3}


# ------------------------------------------------------------------------------------------------------------ exact

class _Exact:
	"""The field in 64 bits: neighbourhoods as flat (sample, neighbour) pairs."""

	def __init__(self, case, seed):
		pts, off, adj, par = _field(case, seed)
		n, dev = len(pts), pts.device
		self.p = pts.double()
		deg = (off[1:] - off[:-1]).long()
		self.off = torch.nn.functional.pad(torch.cumsum(deg + 1, 0), (1, 0))
		nbr = torch.empty(n + len(adj), dtype=torch.long, device=dev)  # self first
		nbr[self.off[:-1]] = torch.arange(n, device=dev)
		at = torch.repeat_interleave(self.off[:-1] + 1 - off[:-1].long(), deg) + torch.arange(len(adj), device=dev)
		nbr[at] = adj.long()
		self.nbr = nbr
		self.par = {k: v.double() for k, v in par.items()}
		self.deg = case['deg']
		self.raw = self.par['raw'].clamp(max=30.0)
		self.dA, self.cA = self.conic('d', 0.0), self.conic('c', 0.0)
		self.sh = torch.cat([self.par['sh_dc'], self.par['sh_rest']], 1)

	def conic(self, which, floor):
		q = self.par[which + '_quat']
		q = q / q.norm(dim=1, keepdim=True)
		w, v = q[:, :1], q[:, 1:]
		eye = torch.eye(3, dtype=q.dtype, device=q.device)
		z = torch.zeros_like(w[:, 0])
		skew = torch.stack([z, -v[:, 2], v[:, 1], v[:, 2], z, -v[:, 0], -v[:, 1], v[:, 0], z], 1).view(-1, 3, 3)
		R = (w * w - (v * v).sum(1, keepdim=True))[..., None] * eye + 2 * v[:, :, None] * v[:, None] + 2 * w[..., None] * skew
		iv = 1 / (torch.exp(2 * self.par[which + '_log_scale']) + floor * floor)
		return (R * iv[:, None]) @ R.transpose(1, 2).contiguous()

	def pairs(self, cell):
		n = self.off[cell + 1] - self.off[cell]
		total = int(n.sum())
		seg = torch.repeat_interleave(torch.arange(len(cell), device=cell.device), n, output_size=total)
		rank = torch.arange(total, device=cell.device) - (torch.cumsum(n, 0) - n)[seg]
		return seg, self.nbr[self.off[cell][seg] + rank], rank

	@staticmethod
	def lowest(value, key, seg, n):
		"""Per sample the pair of smallest (value, key) -> value (inf without any), key."""
		best = torch.full((n,), math.inf, dtype=value.dtype, device=value.device).scatter_reduce(0, seg, value, 'amin')
		far = torch.full((n,), 1 << 60, dtype=torch.long, device=value.device)
		hit = (value == best[seg]) & torch.isfinite(value)
		return best, far.scatter_reduce(0, seg[hit], key[hit], 'amin')

	def walk(self, x, cell):
		cell, todo = cell.clone(), torch.arange(len(cell), device=cell.device)
		while len(todo):
			seg, k, _ = self.pairs(cell[todo])
			new = self.lowest(((x[todo][seg] - self.p[k]) ** 2).sum(1), k, seg, len(todo))[1]
			moved = new != cell[todo]
			cell[todo] = new
			todo = todo[moved]
		return cell

	def exit(self, o, d, cell):
		seg, k, rank = self.pairs(cell)
		a, b = self.p[cell][seg], self.p[k]
		nrm = b - a
		dn = (nrm * d[seg]).sum(1)
		t = ((0.5 * (a + b) - o[seg]) * nrm).sum(1) / dn
		t = torch.where((dn > 0) & (rank > 0), t, torch.full_like(t, math.inf))
		return self.lowest(t, k, seg, len(cell))

	@staticmethod
	def maha(A, v):
		return (v * (A * v[:, None]).sum(2)).sum(1)

	def basis(self, d):
		x, y, z = d.unbind(1)
		b = [torch.full_like(x, 0.28209479177387814), -0.4886025119029199 * y, 0.4886025119029199 * z,
			 -0.4886025119029199 * x, 1.0925484305920792 * x * y, -1.0925484305920792 * y * z,
			 0.31539156525252005 * (2 * z * z - x * x - y * y), -1.0925484305920792 * x * z,
			 0.5462742152960396 * (x * x - y * y), -0.5900435899266435 * y * (3 * x * x - y * y),
			 2.890611442640554 * x * y * z, -0.4570457994644658 * y * (4 * z * z - x * x - y * y),
			 0.3731763325901154 * z * (2 * z * z - 3 * x * x - 3 * y * y),
			 -0.4570457994644658 * x * (4 * z * z - x * x - y * y), 1.445305721320277 * z * (x * x - y * y),
			 -0.5900435899266435 * x * (x * x - 3 * y * y)]
		return torch.stack(b[:(self.deg + 1) ** 2], 1)

	def density(self, x, cell, r2=None):
		seg, k, _ = self.pairs(cell)
		v = x[seg] - self.p[k]
		e = torch.exp(self.raw[k] - 0.5 * self.maha(self.dA[k], v))
		if r2 is not None:
			e = torch.where((v * v).sum(1) <= r2[k], e, torch.zeros_like(e))
		return torch.zeros(len(cell), dtype=e.dtype, device=e.device).index_add(0, seg, e)

	def color(self, x, cell, basis, cut=math.inf, baked=None, two_pass=False):
		seg, k, rank = self.pairs(cell)
		n = len(cell)
		m = self.maha(self.cA[k], x[seg] - self.p[k])
		low = torch.full((n,), math.inf, dtype=m.dtype, device=m.device).scatter_reduce(0, seg, m.detach(), 'amin')
		a = torch.exp(-0.5 * (m - low[seg]))
		if cut < math.inf and two_pass:
			a = torch.where(m <= low[seg] + cut, a, torch.zeros_like(a))
		elif cut < math.inf:  # a term counts when m <= the minimum of the terms before it + cut, in neighbourhood order
			rows = torch.full((n, int(rank.max()) + 1), math.inf, dtype=m.dtype, device=m.device)
			rows[seg, rank] = m
			before = torch.nn.functional.pad(torch.cummin(rows, 1)[0][:, :-1], (1, 0), value=math.inf)
			a = torch.where(m <= before[seg, rank] + cut, a, torch.zeros_like(a))
		if baked is None:
			c = (self.sh[k, :basis.shape[1]] * basis[seg].unsqueeze(2)).sum(1).add(0.5).clamp_min(0)
		else:
			c = baked[k]
		z = torch.zeros(n, dtype=m.dtype, device=m.device)
		return torch.zeros(n, 3, dtype=m.dtype, device=m.device).index_add(0, seg, a[:, None] * c) / z.index_add(0, seg, a)[:, None]


def _bounds(o, d):
	od, oo = (o * d).sum(1), (o * o).sum(1)
	mid = torch.clamp((od * od - (oo - 1)).clamp_min(0).sqrt() - od, min=NEAR + 1e-3)
	far = torch.maximum((od * od - (oo - FAR * FAR)).clamp_min(0).sqrt() - od, mid + 1e-3)
	return mid, far


def _foam_samples(F, o, d, cell, far, density, color):
	"""The samples of the face-crossing renderer, step by step: (t, cell, weight of the segment before) per ray, the
	composited rgb, T, depth. color(t, cell, rays) is called for the samples of segments heavier than W_THRESH."""
	n = len(o)
	f = dict(dtype=torch.float64, device=o.device)
	rgb, T, depth = torch.zeros(n, 3, **f), torch.ones(n, **f), torch.zeros(n, **f)
	live = torch.arange(n, device=o.device)
	t = torch.full((n,), NEAR, **f)
	cell = F.walk(o + NEAR * d, cell)
	sig = density(o + t[:, None] * d, cell)
	C, has = torch.zeros(n, 3, **f), torch.zeros(n, dtype=torch.bool, device=o.device)
	steps = [(live, t.clone(), cell.clone())]
	while len(live):
		te, nx = F.exit(o[live], d[live], cell[live])
		last = ~(te < far[live])
		tq = torch.where(last, far[live], torch.maximum(te, t[live]))
		cq = torch.where(last, cell[live], nx)
		sq = density(o[live] + tq[:, None] * d[live], cq)
		alpha = -torch.expm1(-0.5 * (sig[live] + sq) * (tq - t[live]))
		w = T[live] * alpha
		lit = w > W_THRESH
		r = live[lit]
		need = r[~has[r]]
		C[need] = color(t[need], cell[need], need)
		Cq = torch.zeros(len(live), 3, **f)
		Cq[lit] = color(tq[lit], cq[lit], r)
		rgb[r] += (0.5 * w[lit])[:, None] * (C[r] + Cq[lit])
		depth[r] += 0.5 * w[lit] * (t[r] + tq[lit])
		T[live] *= 1 - alpha
		t[live], cell[live], sig[live], C[live], has[live] = tq, cq, sq, Cq, lit
		steps.append((live, tq, cq))
		live = live[~last & (T[live] >= T_THRESH)]
	return steps, rgb, T, depth


def _march_grid(o, d, mid, far):
	n_in = torch.ceil((mid - NEAR) / DT).long()
	k = torch.arange(int(n_in.max()) + N_BG, device=o.device)[None]
	t0 = NEAR + k * DT
	t1 = torch.minimum(t0 + DT, mid[:, None])
	i0, i1 = 1 / mid[:, None], 1 / far[:, None]
	u = (k - n_in[:, None]) / N_BG
	edge0, edge1 = 1 / (i0 + u * (i1 - i0)), 1 / (i0 + (u + 1 / N_BG) * (i1 - i0))
	inner = k < n_in[:, None]
	t = torch.where(inner, 0.5 * (t0 + t1), 1 / (i0 + (u + 0.5 / N_BG) * (i1 - i0)))
	return t, torch.where(inner, t1 - t0, edge1 - edge0), k < n_in[:, None] + N_BG


def _march_samples(F, o, d, cell, t, delta, valid, color):
	n, f = len(o), dict(dtype=torch.float64, device=o.device)
	rgb, T, depth = torch.zeros(n, 3, **f), torch.ones(n, **f), torch.zeros(n, **f)
	live, cell, steps = torch.arange(n, device=o.device), cell.clone(), []
	for k in range(t.shape[1]):
		live = live[valid[live, k]]
		if not len(live):
			break
		tk = t[live, k]
		x = o[live] + tk[:, None] * d[live]
		cell[live] = F.walk(x, cell[live])
		alpha = -torch.expm1(-F.density(x, cell[live]) * delta[live, k])
		w = T[live] * alpha
		lit = w > W_THRESH
		r = live[lit]
		rgb[r] += w[lit][:, None] * color(tk[lit], cell[r], r)
		depth[r] += w[lit] * tk[lit]
		T[live] *= 1 - alpha
		steps.append((live, tk, cell[live]))
		live = live[T[live] >= T_THRESH]
	return steps, rgb, T, depth


def _leaves_of(F, floor):
	"""Parameters that collect gradients, and the conics built from them again."""
	for v in F.par.values():
		v.requires_grad_(True)
	A = [F.conic(w, floor) for w in 'dc']
	F.dA, F.cA = (a.detach().requires_grad_(True) for a in A)
	F.raw = F.par['raw'].detach().clone().requires_grad_(True)
	F.sh = F.sh.detach().clone().requires_grad_(True)
	return A


def _finish(F, A):
	torch.autograd.backward(A, [F.dA.grad if F.dA.grad is not None else torch.zeros_like(A[0]),
								F.cA.grad if F.cA.grad is not None else torch.zeros_like(A[1])])
	g = {n: F.par[n].grad for n in PARAMS[1:5]}
	zero = torch.zeros_like
	gs = F.sh.grad if F.sh.grad is not None else zero(F.sh)
	return {'raw': F.raw.grad, **g, 'sh_dc': gs[:, :1].contiguous(), 'sh_rest': gs[:, 1:].contiguous()}


def _scatter_samples(F, o, d, basis, steps, g_sigma, g_C, chunk=60000):
	"""Adds the gradients of every sample's density and colour to the leaves of the field."""
	r, t, c = (torch.cat([s[i] for s in steps]) for i in range(3))
	for a in range(0, len(r), chunk):
		q = slice(a, a + chunk)
		x = o[r[q]] + t[q, None] * d[r[q]]
		F.density(x, c[q]).backward(g_sigma[q])
		lit = (g_C[q] != 0).any(1)
		if lit.any():
			F.color(x[lit], c[q][lit], basis[r[q]][lit]).backward(g_C[q][lit])


def _training(case, seed):
	foam = case['op'] == 'foam'
	F = _Exact(case, seed)
	floor = 0.0 if foam else DT / 2
	A = _leaves_of(F, floor)
	o, d, start, gt = _training_rays(case, seed, F.p.float())
	o, d, gt = o.double(), d.double(), gt.double()
	mid, far = _bounds(o, d)
	basis, start = F.basis(d), start.long()
	n, dev = len(o), o.device

	def color(t, cell, r):
		return F.color(o[r] + t[:, None] * d[r], cell, basis[r])

	with torch.no_grad():
		if foam:
			steps, rgb, T, depth = _foam_samples(F, o, d, start, far, F.density, color)
		else:
			grid = _march_grid(o, d, mid, far)
			steps, rgb, T, depth = _march_samples(F, o, d, start, *grid, color)
		# the samples as (step, ray) tables, and their densities and colours again
		S = len(steps)
		tab = torch.full((S, n), -1, dtype=torch.long, device=dev)
		at = 0
		for k, s in enumerate(steps):
			tab[k, s[0]] = torch.arange(at, at + len(s[0]), device=dev)
			at += len(s[0])
		r, t, c = (torch.cat([s[i] for s in steps]) for i in range(3))
		sig = torch.cat([F.density(o[r[a:a + 60000]] + t[a:a + 60000, None] * d[r[a:a + 60000]], c[a:a + 60000])
						 for a in range(0, at, 60000)])
		col = torch.cat([color(t[a:a + 60000], c[a:a + 60000], r[a:a + 60000]) for a in range(0, at, 60000)])
	sig.requires_grad_(True)
	col.requires_grad_(True)
	bg = torch.zeros(3, dtype=torch.float64, device=dev, requires_grad=True)
	Tr, acc = torch.ones(n, dtype=torch.float64, device=dev), torch.zeros(n, 3, dtype=torch.float64, device=dev)
	for k in range(1 if foam else 0, S):
		q = tab[k].clamp_min(0)
		on = tab[k] >= 0
		if foam:
			p = tab[k - 1].clamp_min(0)
			depth_k = 0.5 * (sig[p] + sig[q]) * (t[q] - t[p])
			shade = 0.5 * (col[p] + col[q])
		else:
			delta = grid[1][:, k]
			depth_k, shade = sig[q] * delta, col[q]
		alpha = torch.where(on, -torch.expm1(-depth_k), torch.zeros_like(depth_k))
		w = Tr * alpha
		acc = acc + torch.where(w > W_THRESH, w, torch.zeros_like(w))[:, None] * shade
		Tr = Tr * (1 - alpha)
	out = acc + Tr[:, None] * torch.sigmoid(bg)
	loss = torch.nn.functional.mse_loss(out, gt)
	loss.backward()
	_scatter_samples(F, o, d, basis, steps, sig.grad, col.grad)
	return {'rgb': out.detach(), 'acc': 1 - T, 'depth': depth, 'loss': loss.detach(), 'bg': bg.grad, **_finish(F, A)}


def _fields(case, seed):
	F = _Exact(case, seed)
	st = prepare(case, seed)
	A = _leaves_of(F, 0.0)
	b, s = case['rays'], case['samples']
	with torch.no_grad():
		cell, cells = st['start'].long(), []
		for k in range(s):
			cell = F.walk((st['o'] + st['d'] * st['z'][:, k:k + 1]).double(), cell)
			cells.append(cell)
		cell = torch.stack(cells, 1).reshape(-1)
	x, lit, dirs = st['x'].double(), st['lit'], st['dirs'].double()
	sigma, rgb = torch.empty(b * s, dtype=torch.float64, device=x.device), torch.empty(len(lit), 3, dtype=torch.float64,
																					   device=x.device)
	for a in range(0, b * s, 60000):
		q = slice(a, a + 60000)
		v = F.density(x[q], cell[q])
		v.backward(st['g_sigma'][q].double())
		sigma[q] = v.detach()
	for a in range(0, len(lit), 60000):
		q = slice(a, a + 60000)
		v = F.color(x[lit[q]], cell[lit[q]], F.basis(dirs[q]))
		v.backward(st['g_rgb'][q].double())
		rgb[q] = v.detach()
	g = _finish(F, A)
	return {'site': None, 'sigma': sigma, 'rgb': rgb, 'g_sh': torch.cat([g.pop('sh_dc'), g.pop('sh_rest')], 1), **g}


@torch.no_grad()
def _infer(case, seed):
	F = _Exact(case, seed)
	st = prepare(case, seed)
	o, d, deg = st['o'].double(), st['d'].double(), case['deg']
	start = (st['pack']['perm'][st['start'].long()] if case['op'] == 'batch' else st['start']).long()
	far = _bounds(o, d)[1]
	if case.get('half'):
		F.sh = F.sh.float().half().double()
	baked = r2 = None
	cut = 2 * math.log(1 / case['eps']) if case.get('eps') else math.inf
	if case.get('eps'):
		s2 = torch.exp(2 * F.par['d_log_scale'].float()).amax(1)
		r2 = (2 * s2 * (F.raw.float() - math.log(case['eps'])).clamp_min(0) * (1 + 2 ** -9)).half().double()
	if case.get('colors') == 'baked':
		v = F.p - st['eye'].double()
		F_basis = F.basis(v / v.norm(dim=1, keepdim=True))
		sh = torch.cat([F.par['sh_dc'], F.par['sh_rest']], 1)[:, :(deg + 1) ** 2]
		baked = (sh * F_basis.unsqueeze(2)).sum(1).add(0.5).clamp_min(0)
	rgb, T, depth = [], [], []
	for a in range(0, len(o), 200000):
		q = slice(a, a + 200000)
		oq, dq = o[q], d[q]
		basis = F.basis(dq)

		def color(t, cell, r):
			return F.color(oq[r] + t[:, None] * dq[r], cell, basis[r], cut, baked, case.get('colors') == 'exact')

		_, c, tr, z = _foam_samples(F, oq, dq, start[q], far[q], lambda x, cell: F.density(x, cell, r2), color)
		rgb.append(c), T.append(tr), depth.append(z)
	rgb, T, depth = torch.cat(rgb), torch.cat(T), torch.cat(depth)
	if case['op'] == 'batch':
		return {'rgb': rgb, 'T': T, 'depth': depth, 'stats': None}
	return {'rgb': rgb + 0.5 * T[:, None], 'acc': 1 - T, 'depth': depth, 'stats': None}


@torch.no_grad()
def _march(case, seed):
	F = _Exact(case, seed)
	F.dA, F.cA = F.conic('d', DT / 2), F.conic('c', DT / 2)
	st = prepare(case, seed)
	o, d = st['o'].double(), st['d'].double()
	mid, far = _bounds(o, d)
	basis = F.basis(d)
	t, delta, valid = _march_grid(o, d, mid, far)
	_, rgb, T, depth = _march_samples(F, o, d, st['start'].long(), t, delta, valid,
									  lambda tk, cell, r: F.color(o[r] + tk[:, None] * d[r], cell, basis[r]))
	return {'rgb': rgb + 0.5 * T[:, None], 'acc': 1 - T, 'depth': depth, 'samples': None}


@torch.no_grad()
def _pack(case, seed):
	F = _Exact(case, seed)
	p = F.p.float()
	lo, hi = p.amin(0), p.amax(0)
	q = ((p - lo) / (hi - lo).clamp_min(1e-12) * 1023).long()
	code = torch.zeros(len(p), dtype=torch.long, device=p.device)
	for b in range(10):
		for a in range(3):
			code |= (q[:, a] >> b & 1) << (3 * b + a)
	perm = torch.argsort(code)
	iu = [0, 0, 0, 1, 1, 2], [0, 1, 2, 1, 2, 2]
	dA, cA = F.dA[:, iu[0], iu[1]][perm], F.cA[:, iu[0], iu[1]][perm]
	raw, zero = F.raw[perm][:, None], torch.zeros(len(p), 1, dtype=torch.float64, device=p.device)
	return {'conics': torch.cat([dA, raw, zero, cA], 1), 'sh': F.sh[perm], 'rows': torch.cat([dA, raw], 1),
			**{k: None for k in ('edge', 'edge_i', 'points', 'offsets', 'nbr', 'slots', 'perm')}}


def exact(case, seed):
	"""What run() returns, in 64 bits; None for the whole numbers and where it would take too long."""
	op = case['op']
	if op == 'locate':
		return None
	if op == 'pack':
		return _pack(case, seed)
	if op == 'fields':
		return _fields(case, seed)
	pairs = case['rays'] * _samples(case)
	if pairs > (8e6 if op in ('foam', 'uniform') else 7e7):
		return None
	if op in ('foam', 'uniform'):
		return _training(case, seed)
	return _march(case, seed) if op == 'march' else _infer(case, seed)
