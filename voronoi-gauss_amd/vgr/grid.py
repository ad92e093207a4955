"""Start-cell locator on the GPU: a uniform grid over the sites and exact nearest-site queries (libvgr's
vgr_points_box, vgr_grid_build_points, vgr_grid_nearest_points, vgr_grid_nearest_binned).

It replaces the host-side cKDTree query of the reference's nearest_sites (sites.py:38-39), which finds the start
site of the traversal per camera centre (bench_infer.py:60, eval_scene.py:69) and per ray origin of a ray batch.
The answer is cKDTree's (float64 distances) up to exact distance ties, which go to the smaller site index."""

import ctypes
import math

import torch

from . import _lib


# Batches above this many queries, and of at least one query per BINNED_CELLS cells, are binned before they are answered. The
# binning clears and scans a counter per cell and writes the queries again; it pays where queries differ in how many cells
# they scan. One MI355X, ms query by query : binned, of a grid that is kept:
#   clustered sites, queries around them   20k sites 65537 queries 0.24 : 0.19, 1M sites 2.3 : 1.6, 1M queries 7.8 : 3.7
#   uniform sites, queries over the cube   1M sites 65537 queries 0.07 : 0.10, 1M 0.23 : 0.24, 4M 0.79 : 0.67; a batch of
#                                          near ones costs up to 0.1 more binned, one whose queries lie outside half
#   31M sites, 15.6M cells                 65537 queries 0.06 : 0.17 uniform, 4.4 : 4.7 clustered; 1M 0.34 : 0.47, 15.7 : 10.6
BINNED_QUERIES, BINNED_CELLS = 65536, 16


class SiteGrid:
	"""Sites binned into a uniform grid of about `per_cell` sites per cell (cubic cells over the bounding box).

	points: (N, 3) or (N, 4) float32 CUDA tensor (xyz first), kept by reference; the grid is built on its stream."""

	def __init__(self, points, per_cell=2.0):
		if not (isinstance(points, torch.Tensor) and points.is_cuda):
			raise RuntimeError('points must be a CUDA tensor')
		if points.dtype != torch.float32 or points.dim() != 2 or points.shape[1] < 3 or not points.is_contiguous():
			raise RuntimeError('points must be a contiguous float32 (N, 3) or (N, 4) tensor')
		n = len(points)
		if n == 0:
			raise RuntimeError('SiteGrid needs at least one site')
		self.points, self.stride, self.n = points, points.shape[1], n
		dev = points.device
		lib = _lib.load()
		box = torch.empty(int(lib.vgr_points_box_floats()), dtype=torch.float32, device=dev)
		_lib.call('vgr_points_box', _lib.ptr(points), n, self.stride, _lib.ptr(box), _lib.stream_of(dev))
		lo, hi = box[:6].cpu().double().view(2, 3)
		ext = torch.clamp(hi - lo, min=1e-6)
		lo = lo - 1e-6 * ext
		ext = ext * (1 + 2e-6)
		edge = (float(ext.prod()) * per_cell / n) ** (1.0 / 3.0)
		res = [int(min(max(math.ceil(float(e) / edge), 1), 1024)) for e in ext]
		while res[0] * res[1] * res[2] > 4096 * 4096:
			res = [max(r // 2, 1) for r in res]
		self.lo = [float(v) for v in lo]
		self.cell = [float(e) / r for e, r in zip(ext, res)]
		self.res = res
		n_cells = res[0] * res[1] * res[2]
		self.cell_start = torch.empty(n_cells + 1, dtype=torch.int32, device=dev)
		self.cell_sites = torch.empty(n, dtype=torch.int32, device=dev)
		work = torch.empty(int(lib.vgr_grid_work_size(n, n_cells)), dtype=torch.int32, device=dev)
		self._geom = (_floats(self.lo), _floats(self.cell), _ints(self.res))
		# the sites in cell order, (x, y, z, bits of the index) each, which the queries scan (a snapshot of points)
		self.cell_points = torch.empty(n, 4, dtype=torch.float32, device=dev)
		_lib.call('vgr_grid_build_points', _lib.ptr(points), n, self.stride, *self._geom, _lib.ptr(self.cell_start),
				  _lib.ptr(self.cell_sites), _lib.ptr(self.cell_points), _lib.ptr(work), _lib.stream_of(dev))
		self._work = work  # released once the asynchronous build has run (caching allocator, same stream)

	def nearest(self, queries, order=None):
		"""Index (int32) of the nearest site of every query point: queries (m, 3) float32 CUDA tensor. order:
		optional int32 (m,) permutation of 0 .. m - 1, the order in which the queries are answered (query_order
		gives a coherent one); the answers do not depend on it. Without an order, batches above 65,536 queries and
		a sixteenth of the grid's cells are binned into the cells first and answered cell by cell."""
		if not (isinstance(queries, torch.Tensor) and queries.is_cuda):
			raise RuntimeError('queries must be a CUDA tensor')
		if queries.dtype != torch.float32 or queries.dim() != 2 or queries.shape[1] != 3 or not queries.is_contiguous():
			raise RuntimeError('queries must be a contiguous float32 (m, 3) tensor')
		if order is not None and not (isinstance(order, torch.Tensor) and order.is_cuda and order.dtype == torch.int32
									  and order.shape == (len(queries),) and order.is_contiguous()):
			raise RuntimeError('order must be a contiguous int32 CUDA tensor of one entry per query')
		out = torch.empty(len(queries), dtype=torch.int32, device=queries.device)
		n_cells = len(self.cell_start) - 1
		if order is None and BINNED_QUERIES < len(queries) < 2 ** 31 and BINNED_CELLS * len(queries) >= n_cells:
			wb = int(_lib.load().vgr_grid_binned_work_size(len(queries), n_cells))
			work = torch.empty(wb, dtype=torch.uint8, device=queries.device)
			_lib.call('vgr_grid_nearest_binned', _lib.ptr(self.cell_points), self.n, *self._geom,
					  _lib.ptr(self.cell_start), _lib.ptr(queries), len(queries), _lib.ptr(work), wb, _lib.ptr(out),
					  _lib.stream_of(queries.device))
			return out
		_lib.call('vgr_grid_nearest_points', _lib.ptr(self.cell_points), self.n, *self._geom, _lib.ptr(self.cell_start),
				  _lib.ptr(queries), len(queries), _lib.ptr(order), _lib.ptr(out), _lib.stream_of(queries.device))
		return out

	def nearest_indexed(self, queries):
		"""nearest() reading the candidate sites through their indices into the point array (vgr_grid_nearest):
		the same answers."""
		if not (isinstance(queries, torch.Tensor) and queries.is_cuda):
			raise RuntimeError('queries must be a CUDA tensor')
		if queries.dtype != torch.float32 or queries.dim() != 2 or queries.shape[1] != 3 or not queries.is_contiguous():
			raise RuntimeError('queries must be a contiguous float32 (m, 3) tensor')
		out = torch.empty(len(queries), dtype=torch.int32, device=queries.device)
		_lib.call('vgr_grid_nearest', _lib.ptr(self.points), self.n, self.stride, *self._geom,
				  _lib.ptr(self.cell_start), _lib.ptr(self.cell_sites), _lib.ptr(queries), len(queries), _lib.ptr(out),
				  _lib.stream_of(queries.device))
		return out


def query_order(queries, pos_bits=8):
	"""A spatially coherent processing order of query points for SiteGrid.nearest: int32 (m,) permutation sorting
	them along the Z-order curve of pos_bits bits per axis over their bounding box (vgr_ray_order with one direction
	bin). The lanes of a wave then scan neighbouring cells."""
	from . import ext
	return ext.ray_order(queries, queries, dir_res=1, pos_bits=pos_bits)


def _floats(v):
	return (ctypes.c_float * 3)(*v)


def _ints(v):
	return (ctypes.c_int32 * 3)(*v)
