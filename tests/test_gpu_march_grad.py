"""GPU parity of the march backward (vgr_march_backward through the C ABI, and ext.march's autograd) against the C
oracle's sequential restatement of march.cu:264-345 on identical inputs, the oracle being pinned by float64 autograd
of the dense march. The kernel sums each pass's samples per neighbour in registers and adds them with fp32 atomics,
so the sums agree to rounding, not bitwise: the bar is a relative error (vector norm) of 2e-5 per gradient."""

import numpy as np
import pytest
import torch

import oracle
from helpers import Field
from test_oracle_grad import rel
from vgr import ext

pytestmark = pytest.mark.gpu

DT, NBG = 0.05, 8


def T(a, dev):
	return torch.as_tensor(np.ascontiguousarray(a), device=dev)


def case(dev, sh_deg, t_thresh, w_thresh, B=192, seed=5, lanes=0):
	f = Field(seed=seed, n=300, sh_deg=sh_deg)
	rays = f.rays(B=B, seed=seed)
	dA, cA = f.conics(0.01)
	fx = ext.march_extension()
	field = [T(a, dev) for a in (f.points, f.offsets, f.adj, f.raw, dA, cA, f.sh)]
	rt = [T(a, dev) for a in rays]
	rgb, Tt, _, _ = fx.march_forward(*field, sh_deg, *rt, DT, NBG, t_thresh, w_thresh, lanes=lanes)
	return f, rays, dA, cA, fx, field, rt, rgb, Tt


@pytest.mark.parametrize('lanes', [1, 16])
@pytest.mark.parametrize('t_thresh,w_thresh', [(0.0, -1.0), (1e-4, 1e-4)])
@pytest.mark.parametrize('sh_deg', [3, 2, 0])
def test_march_backward_matches_oracle(gpu, sh_deg, t_thresh, w_thresh, lanes):
	"""Both ray layouts (one ray per lane; 16 lanes per ray, one neighbour per lane), each replaying its own forward."""
	f, rays, dA, cA, fx, field, rt, rgb, Tt = case(gpu, sh_deg, t_thresh, w_thresh, lanes=lanes)
	rng = np.random.default_rng(3)
	g_rgb = rng.normal(size=(len(rays[0]), 3)).astype(np.float32)
	g_T = rng.normal(size=len(rays[0])).astype(np.float32)
	g_rgb[:7] = 0  # rays without an upstream colour gradient still pass dL/dT
	got = fx.march_backward(*field, sh_deg, *rt, DT, NBG, t_thresh, w_thresh, rgb, Tt, T(g_rgb, gpu), T(g_T, gpu),
							lanes=lanes)
	ref = oracle.march_backward(f.points, f.offsets, f.adj, f.raw, dA, cA, f.sh, sh_deg, *rays, DT, NBG,
								rgb.cpu().numpy(), Tt.cpu().numpy(), g_rgb, g_T, t_thresh, w_thresh)
	for name, a, r in zip(('raw', 'dA', 'cA', 'sh'), got, ref):
		assert rel(a.cpu().numpy(), r) < 2e-5, name
	assert (got[3][:, (sh_deg + 1) ** 2:] == 0).all()


def test_march_backward_wave_atomics_match_oracle(gpu):
	"""16,384 rays, where the launch shares each row of atomics across the wave: against the oracle, and against the
	per-lane atomics of the same rays in two launches of 8,192 (whose gradients add)."""
	B = 16384
	f, rays, dA, cA, fx, field, rt, rgb, Tt = case(gpu, 3, 1e-4, 1e-4, B=B, lanes=1)
	rng = np.random.default_rng(8)
	g_rgb = T(rng.normal(size=(B, 3)).astype(np.float32), gpu)
	g_T = T(rng.normal(size=B).astype(np.float32), gpu)
	got = fx.march_backward(*field, 3, *rt, DT, NBG, 1e-4, 1e-4, rgb, Tt, g_rgb, g_T, lanes=1)
	ref = oracle.march_backward(f.points, f.offsets, f.adj, f.raw, dA, cA, f.sh, 3, *rays, DT, NBG, rgb.cpu().numpy(),
								Tt.cpu().numpy(), g_rgb.cpu().numpy(), g_T.cpu().numpy())
	for name, a, r in zip(('raw', 'dA', 'cA', 'sh'), got, ref):
		assert rel(a.cpu().numpy(), r) < 2e-5, name
	halves = [fx.march_backward(*field, 3, *[x[s].contiguous() for x in rt], DT, NBG, 1e-4, 1e-4, rgb[s].contiguous(),
								Tt[s].contiguous(), g_rgb[s].contiguous(), g_T[s].contiguous(), lanes=1)
			  for s in (slice(0, B // 2), slice(B // 2, None))]
	for name, a, h0, h1 in zip(('raw', 'dA', 'cA', 'sh'), got, *halves):
		assert rel((h0 + h1).cpu().numpy(), a.cpu().numpy()) < 1e-5, name


def test_march_autograd_matches_oracle(gpu):
	"""ext.march with gradients on, as training calls it (ext.py:150-182): loss = <rgb, g_rgb> + <T, g_T>."""
	f, rays, dA, cA, fx, field, rt, rgb0, T0 = case(gpu, 3, 1e-4, 1e-4)
	graph = ext.Graph(*field[:3])
	params = [p.clone().requires_grad_() for p in field[3:]]
	rng = np.random.default_rng(4)
	g_rgb = rng.normal(size=(len(rays[0]), 3)).astype(np.float32)
	g_T = rng.normal(size=len(rays[0])).astype(np.float32)
	rgb, Tt, depth, stats = ext.march(graph, *params, 3, *rt, DT, NBG)
	assert torch.equal(rgb.detach(), rgb0) and torch.equal(Tt.detach(), T0)
	assert not depth.requires_grad and stats.dtype == torch.int32
	((rgb * T(g_rgb, gpu)).sum() + (Tt * T(g_T, gpu)).sum()).backward()
	ref = oracle.march_backward(f.points, f.offsets, f.adj, f.raw, dA, cA, f.sh, 3, *rays, DT, NBG,
								rgb0.cpu().numpy(), T0.cpu().numpy(), g_rgb, g_T)
	for name, p, r in zip(('raw', 'dA', 'cA', 'sh'), params, ref):
		assert rel(p.grad.cpu().numpy(), r) < 2e-5, name
	# a loss on T alone: autograd hands no colour gradient, which counts as zero
	params = [p.clone().requires_grad_() for p in field[3:]]
	_, Tt, _, _ = ext.march(graph, *params, 3, *rt, DT, NBG)
	Tt.sum().backward()
	ref = oracle.march_backward(f.points, f.offsets, f.adj, f.raw, dA, cA, f.sh, 3, *rays, DT, NBG,
								rgb0.cpu().numpy(), T0.cpu().numpy(), np.zeros((len(rays[0]), 3), np.float32),
								np.ones(len(rays[0]), np.float32))
	assert rel(params[0].grad.cpu().numpy(), ref[0]) < 2e-5
	assert not params[3].grad.any()


def test_march_backward_edge_cases(gpu):
	f, rays, dA, cA, fx, field, rt, rgb, Tt = case(gpu, 3, 1e-4, 1e-4, B=16)
	ones3, ones = torch.ones(16, 3, device=gpu), torch.ones(16, device=gpu)
	# untraced rays (start -1) have no samples and take no gradient
	start = rt[2].clone().fill_(-1)
	rays_u = rt[:2] + [start] + rt[3:]
	got = fx.march_backward(*field, 3, *rays_u, DT, NBG, 1e-4, 1e-4, rgb, Tt, ones3, ones)
	assert all(not g.any() for g in got)
	# no rays: zeroed gradients of the field's shapes
	e3, e = torch.empty(0, 3, device=gpu), torch.empty(0, device=gpu)
	got = fx.march_backward(*field, 3, e3, e3, torch.empty(0, dtype=torch.int32, device=gpu), e, e, e, DT, NBG, 1e-4,
							1e-4, e3, e, e3, e)
	assert [tuple(g.shape) for g in got] == [(f.n,), (f.n, 6), (f.n, 6), (f.n, 16, 3)]
	assert all(not g.any() for g in got)
	with pytest.raises(RuntimeError, match='sh_deg'):
		fx.march_backward(*field, 4, *rt, DT, NBG, 1e-4, 1e-4, rgb, Tt, ones3, ones)
	with pytest.raises(RuntimeError, match='g_rgb'):
		fx.march_backward(*field, 3, *rt, DT, NBG, 1e-4, 1e-4, rgb, Tt, ones3[:3], ones)


@pytest.mark.parametrize('n_rays', [1, 3, 65, 130])
@pytest.mark.parametrize('cap', [1, 24, 256])
@pytest.mark.parametrize('dt', [1 / 16, 1 / 256])
def test_backward_of_recorded_visits(gpu, n_rays, cap, dt):
	"""The backward from the forward's visit records (runs of up to 34 samples in a cell, replayed on their own) against the
	backward that marches every ray again: records that all fit, some and none, steps longer than a cell and many steps per
	cell. The samples replay with the forward's bits and the sums run in another order: 1e-5. The forward's outputs do not
	depend on the records."""
	f = Field(seed=9, n=300)
	o, d, start, near, mid, far = f.rays(B=n_rays, seed=9)
	start = start.copy()
	start[:1] = f.n if n_rays > 1 else start[:1]  # a ray that is not traced
	dA, cA = f.conics(0.01)
	t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=gpu)  # noqa: E731
	args = [t(a) for a in (f.points, f.offsets, f.adj, f.raw, dA, cA, f.sh)] + [3] + \
		[t(a) for a in (o, d, start, near, mid, far)] + [dt, 16, 1e-4, 1e-4]
	fx = ext.march_extension()
	visits = (torch.full((n_rays, cap, 8), float('nan'), device=gpu), torch.full((n_rays,), -1, dtype=torch.int32,
																				 device=gpu))
	outs = fx.march_forward(*args, lanes=16, visits=visits)
	plain = fx.march_forward(*args, lanes=16)
	for a, b in zip(outs, plain):
		assert torch.equal(a, b)
	assert (visits[1] >= 0).all()
	g = torch.Generator(device=gpu).manual_seed(2)
	up = torch.randn(n_rays, 3, device=gpu, generator=g), torch.randn(n_rays, device=gpu, generator=g)
	got = fx.march_backward(*args, outs[0], outs[1], *up, lanes=16, visits=visits, stats=outs[3])
	want = fx.march_backward(*args, outs[0], outs[1], *up, lanes=16)
	for a, b in zip(got, want):
		assert torch.isfinite(a).all() and (a.double() - b.double()).norm() <= 1e-5 * b.double().norm() + 1e-30


@pytest.mark.parametrize('n_rays', [1, 4099, (1 << 19) - 1, 1 << 19])
def test_march_without_gradients(gpu, n_rays):
	"""ext.march without gradients takes the layout by batch size and leaves no records: the bits of the forward under
	autograd below 2^19 rays (16 lanes per ray in both), and from there on one ray per lane, whose sums run in the order of
	the neighbourhood: the same samples, colours of at most ~3 by sums of at most ~30 terms each to a few ulps."""
	f = Field(seed=9, n=300)
	o, d, start, near, mid, far = f.rays(B=min(n_rays, 4099), seed=9)
	dA, cA = f.conics(0.01)
	rays = [torch.as_tensor(np.resize(a, (n_rays,) + a.shape[1:]), device=gpu) for a in (o, d, start, near, mid, far)]
	graph = ext.Graph(*[T(a, gpu) for a in (f.points, f.offsets, f.adj)])
	params = [T(a, gpu) for a in (f.raw, dA, cA, f.sh)]
	plain = ext.march(graph, *params, 3, *rays, DT, NBG)
	with torch.no_grad():
		off = ext.march(graph, *[p.clone().requires_grad_() for p in params], 3, *rays, DT, NBG)
	grad = ext.march(graph, *[p.clone().requires_grad_() for p in params], 3, *rays, DT, NBG)
	for a, b, c in zip(plain, off, grad):
		assert not a.requires_grad and torch.equal(a, b)
		if n_rays < 1 << 19:
			assert torch.equal(a, c.detach())
		elif a.dtype == torch.int32:
			assert (a == c).all(1).float().mean() > 0.999  # a weight within ulps of the threshold is coloured or not
		else:
			# such a segment moves its ray by its weight, 1e-4
			near_ = (a - c.detach()).abs()
			assert near_.max() < 5e-4 and (near_ < 1e-5).float().mean() > 0.999
