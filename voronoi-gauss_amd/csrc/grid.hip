// Uniform grid over the sites and exact nearest-site queries, gfx950: the start-cell locator of the traversals.
//
// The reference locates start cells on the host with scipy's cKDTree (sites.py:38-39, called per camera centre
// in bench_infer.py:60 and eval_scene.py:69, and per ray origin for ray batches). Here the sites are binned into a
// uniform grid by a counting sort on the GPU (histogram, exclusive scan, scatter), and each query scans Chebyshev
// rings of grid cells around its own cell until no unscanned cell can hold a closer site. Distances are computed in
// float64, as cKDTree computes them, and ties go to the smaller site index, so the answer is cKDTree's except
// where two sites are at exactly the same float64 distance.
#include <mutex>

#include "vgr_abi.h"
#include "vgr_device.h"
#include "vgr_scan.h"

namespace vgr {
namespace {

constexpr int kBlock = 256;
constexpr int64_t kMaxCells = int64_t(kScanTile) * kScanTile;

struct Geom {
    float lo[3];    // grid origin
    float cell[3];  // cell edge per axis
    int res[3];     // cells per axis
};

__device__ __forceinline__ int axis_cell(float x, float lo, float cell, int res) {
    const int c = static_cast<int>(floorf((x - lo) / cell));
    return min(max(c, 0), res - 1);
}

__device__ __forceinline__ const float* site_ptr(const float* pts, int stride, int64_t i) { return pts + stride * i; }

__device__ __forceinline__ int cell_index(const Geom& g, const float* p) {
    const int cx = axis_cell(p[0], g.lo[0], g.cell[0], g.res[0]);
    const int cy = axis_cell(p[1], g.lo[1], g.cell[1], g.res[1]);
    const int cz = axis_cell(p[2], g.lo[2], g.cell[2], g.res[2]);
    return (cz * g.res[1] + cy) * g.res[0] + cx;
}

// One more point in cell c: its place among the cell's points (any order). The lanes of a wave that share a cell take
// their places with one atomic, for the first two cells found in the wave: a batch of queries from one camera, or all
// outside the grid, would otherwise queue at one counter.
__device__ __forceinline__ int take_place(int* __restrict__ count, int c) {
    const int lane = static_cast<int>(threadIdx.x) & 63;
    uint64_t rest = __ballot(1);
    for (int u = 0; u < 2 && rest != 0; ++u) {
        const int leader = __builtin_amdgcn_readfirstlane(__ffsll(static_cast<unsigned long long>(rest)) - 1);
        const int shared = __builtin_amdgcn_readlane(c, leader);
        const uint64_t same = __ballot(c == shared) & rest;
        rest &= ~same;
        if (c == shared) {
            int first = 0;
            if (lane == leader) first = atomicAdd(count + c, __popcll(same));
            first = __builtin_amdgcn_readlane(first, leader);
            return first + __popcll(same & ((uint64_t(1) << lane) - 1));
        }
    }
    return atomicAdd(count + c, 1);
}

// The number of points per cell, and the place of every point in its cell.
__global__ void __launch_bounds__(kBlock) grid_count(const float* __restrict__ pts, int stride, int64_t n, Geom g,
                                                     int* __restrict__ place, int* __restrict__ count) {
    const int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= n) return;
    place[i] = take_place(count, cell_index(g, site_ptr(pts, stride, i)));
}

// Scatter: point i goes to slot start[its cell] + its place: its index to cell_sites and (x, y, z, bits of i) to cp,
// either of which may be null. The cell is computed again from the position (12 bytes) rather than kept (4 written, 4
// read); with the place known the scatter needs no second round of atomics: 1M sites 125 -> 76 us for both passes.
__global__ void __launch_bounds__(kBlock)
    grid_fill(const float* __restrict__ pts, int stride, int64_t n, Geom g, const int* __restrict__ start,
              const int* __restrict__ place, int* __restrict__ cell_sites, float4* __restrict__ cp) {
    const int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= n) return;
    const float* p = site_ptr(pts, stride, i);
    const int s = start[cell_index(g, p)] + place[i];
    if (cell_sites != nullptr) cell_sites[s] = static_cast<int>(i);
    if (cp != nullptr) cp[s] = make_float4(p[0], p[1], p[2], __int_as_float(static_cast<int>(i)));
}

// The build's cell-ordered copy of the sites: slot s of cell_sites gets (x, y, z, bits of the site index).
__global__ void __launch_bounds__(kBlock) grid_cell_points(const float* __restrict__ pts, int stride, int64_t n,
                                                           const int* __restrict__ cell_sites, float4* __restrict__ cp) {
    const int64_t s = int64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (s >= n) return;
    const int k = cell_sites[s];
    const float* p = site_ptr(pts, stride, k);
    cp[s] = make_float4(p[0], p[1], p[2], __int_as_float(k));
}

// Fills n ints with zero (the counters of a build; a kernel rather than hipMemsetAsync, so that a build is made of
// kernel launches only).
__global__ void __launch_bounds__(kBlock) zero_ints(int* __restrict__ a, int64_t n) {
    const int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (i < n) a[i] = 0;
}

// Scratch of vgr_grid_build_noalloc: 2^24 ints (64 MiB), enough for vgr_grid_work_size of 8M sites over 4M cells
// (the largest benchmark scene at two sites per cell is 12M ints). Each GPU that runs the library holds its own copy
// until the process ends. Host code never passes `scratch` itself to a kernel (in host code the name is only a
// stand-in for the symbol); it uses the device address from hipGetSymbolAddress, one per device.
constexpr int64_t kScratchInts = VGR_GRID_NOALLOC_MAX_WORK;
static __device__ __align__(256) int scratch[kScratchInts];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
int* g_scratch_ptr[kMaxDevices] = {};

// This device's address of `scratch`, looked up on the first call on each device (with that device current).
int scratch_on_current_device(int** out) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return launch_status("grid_build_noalloc: hipGetDevice");
    VGR_REQUIRE(dev >= 0 && dev < kMaxDevices, "grid_build_noalloc: device %d beyond the %d supported", dev,
                kMaxDevices);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
        void* p = nullptr;
        const hipError_t err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (err != hipSuccess)
            return fail(VGR_ERR_LAUNCH, "grid_build_noalloc: hipGetSymbolAddress(scratch): %s", hipGetErrorString(err));
        g_scratch_ptr[dev] = static_cast<int*>(p);
    }
    *out = g_scratch_ptr[dev];
    return VGR_OK;
}

// Nearest site of each query: lexicographic argmin of (float64 squared distance, site index).
//
// Rings r = 0, 1, ... of cells at Chebyshev distance r from the query's (clamped) cell are scanned. Every unscanned
// site lies in the grid box beyond a face of the scanned block that is not on the grid boundary, so after ring r
// no unscanned site is closer than the distance lb from the query to the nearest such region (for a query outside
// the grid, that includes its distance to the grid); the scan stops once the best distance is below lb (shrunk by
// a margin covering the float32 rounding of cell assignment), or when the block covers the grid.
// Before a row of cells is read, the distance from the query to the row's box (in y and z; the cells' faces widened by
// the margin of the float32 cell assignment) is compared with the best site so far: a row that starts beyond it holds no
// closer site, nor one as close. The cells of a row are consecutive, so a row is one range of sites.
// CP: the sites' positions come from the build's cell-ordered copy (the sites of a cell, and of a row of cells, share
// lines) instead of through the site index into the point array (a line per site). BINNED: the queries come in cell order
// with their index in the fourth word (grid_fill), so that the lanes of a wave scan the same cells.
template <bool CP, bool BINNED>
__global__ void __launch_bounds__(kBlock) grid_nearest(const float* __restrict__ pts, int stride, Geom g,
                                                       const int* __restrict__ cell_start,
                                                       const int* __restrict__ cell_sites,
                                                       const float4* __restrict__ cp, const float* __restrict__ q,
                                                       int64_t m, const int* __restrict__ order, double margin,
                                                       int* __restrict__ out) {
    const int64_t t = int64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (t >= m) return;
    int64_t i;
    float q0, q1, q2;
    if constexpr (BINNED) {
        const float4 v = reinterpret_cast<const float4*>(q)[t];
        q0 = v.x, q1 = v.y, q2 = v.z, i = __float_as_int(v.w);
    } else {
        i = order != nullptr ? order[t] : t;  // the query this lane answers (a permutation entry)
        if (i < 0 || i >= m) return;
        q0 = q[3 * i], q1 = q[3 * i + 1], q2 = q[3 * i + 2];
    }
    const double qx = q0, qy = q1, qz = q2;
    const int c[3] = {axis_cell(q0, g.lo[0], g.cell[0], g.res[0]), axis_cell(q1, g.lo[1], g.cell[1], g.res[1]),
                      axis_cell(q2, g.lo[2], g.cell[2], g.res[2])};
    const double qa[3] = {qx, qy, qz};
    double best = 1e300;
    int best_k = INT_MAX;
    const auto visit = [&](int x0, int x1, int y, int z) {  // cells x0 .. x1 of a row
        const int row = (z * g.res[1] + y) * g.res[0];
        for (int s = cell_start[row + x0], e = cell_start[row + x1 + 1]; s < e; ++s) {
            float px, py, pz;
            int k;
            if constexpr (CP) {
                const float4 v = cp[s];
                px = v.x, py = v.y, pz = v.z, k = __float_as_int(v.w);
            } else {
                k = cell_sites[s];
                const float* p = site_ptr(pts, stride, k);
                px = p[0], py = p[1], pz = p[2];
            }
            const double dx = qx - px, dy = qy - py, dz = qz - pz;
            const double d2 = dx * dx + dy * dy + dz * dz;
            if (d2 < best || (d2 == best && k < best_k)) best = d2, best_k = k;
        }
    };
    // a lower bound of the distance along axis a from the query to the sites of cell index v (a site outside the grid is
    // binned into the cells at its boundary, which therefore reach to infinity)
    const auto gap = [&](int a, int v) {
        const double lo = v == 0 ? -1e300 : double(g.lo[a]) + double(v) * g.cell[a] - margin;
        const double hi = v == g.res[a] - 1 ? 1e300 : double(g.lo[a]) + double(v + 1) * g.cell[a] + margin;
        return fmax(fmax(lo - qa[a], qa[a] - hi), 0.0);
    };
    const int r_max = max(max(g.res[0], g.res[1]), g.res[2]);
    for (int r = 0; r <= r_max; ++r) {
        // the cells at Chebyshev distance exactly r, clipped to the grid: whole rows where z or y is on the shell,
        // the two end cells of the other rows
        const int z0 = max(c[2] - r, 0), z1 = min(c[2] + r, g.res[2] - 1);
        const int y0 = max(c[1] - r, 0), y1 = min(c[1] + r, g.res[1] - 1);
        const int x0 = max(c[0] - r, 0), x1 = min(c[0] + r, g.res[0] - 1);
        for (int z = z0; z <= z1; ++z) {
            const double gz = gap(2, z), gz2 = gz * gz;
            if (gz2 > best) continue;
            for (int y = y0; y <= y1; ++y) {
                const double gy = gap(1, y);
                if (gy * gy + gz2 > best) continue;
                if (z == c[2] - r || z == c[2] + r || y == c[1] - r || y == c[1] + r) {
                    visit(x0, x1, y, z);
                } else {
                    if (c[0] - r >= 0) visit(c[0] - r, c[0] - r, y, z);
                    if (r > 0 && c[0] + r < g.res[0]) visit(c[0] + r, c[0] + r, y, z);
                }
            }
        }
        // unscanned sites lie in the grid box beyond an open face of the scanned block: the squared distance from
        // the query to each such region (an axis-aligned box) bounds theirs
        double lb2 = 1e300;
        bool open = false;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
#pragma unroll
            for (int side = 0; side < 2; ++side) {
                if (side == 0 ? c[a] - r <= 0 : c[a] + r >= g.res[a] - 1) continue;  // on the grid boundary
                open = true;
                double d2 = 0.0;
#pragma unroll
                for (int b = 0; b < 3; ++b) {
                    double lo = g.lo[b], hi = double(g.lo[b]) + double(g.res[b]) * g.cell[b];
                    if (b == a) {
                        if (side == 0) hi = double(g.lo[a]) + double(c[a] - r) * g.cell[a];
                        else lo = double(g.lo[a]) + double(c[a] + r + 1) * g.cell[a];
                    }
                    const double gap = fmax(fmax(lo - qa[b], qa[b] - hi), 0.0);
                    d2 += gap * gap;
                }
                lb2 = fmin(lb2, d2);
            }
        }
        if (!open) break;  // the scanned block covers the grid
        const double lb = sqrt(lb2) - margin;
        if (lb > 0.0 && best < lb * lb) break;
    }
    out[i] = best_k;
}

// float32 cell assignment can put a site one rounding step across a cell face: the stopping bound shrinks by a few
// float32 ulps of the grid's extent.
double nearest_margin(const float* lo, const float* cell, const int32_t* res) {
    double extent = 0.0;
    for (int a = 0; a < 3; ++a)
        extent = fmax(extent, fabs(double(lo[a])) + double(cell[a]) * res[a]);
    return extent * 1e-6;
}

Geom make_geom(const float* lo, const float* cell, const int32_t* res) {
    Geom g{};
    for (int a = 0; a < 3; ++a) g.lo[a] = lo[a], g.cell[a] = cell[a], g.res[a] = res[a];
    return g;
}

int check_geom(const float* lo, const float* cell, const int32_t* res, int64_t* n_cells) {
    VGR_REQUIRE(lo && cell && res, "grid: null geometry pointer");
    int64_t g = 1;
    for (int a = 0; a < 3; ++a) {
        VGR_REQUIRE(res[a] >= 1 && res[a] <= 65536, "grid: res[%d] must be in [1, 65536] (got %d)", a, res[a]);
        VGR_REQUIRE(cell[a] > 0.f, "grid: cell edge %d must be > 0", a);
        g *= res[a];
    }
    VGR_REQUIRE(g <= kMaxCells, "grid: at most %lld cells (got %lld)", static_cast<long long>(kMaxCells),
                static_cast<long long>(g));
    *n_cells = g;
    return VGR_OK;
}

}  // namespace
}  // namespace vgr

namespace vgr {
namespace {

// Bounding box of n points of `stride` floats, (min xyz, max xyz), NaN where a coordinate is NaN on that axis: kBoxBlocks
// blocks sweep the points, then one block reduces their boxes. (torch's amin and amax over the rows of an (N, 3) tensor
// take 0.76 ms for 1M points, this 12 us.)
constexpr int kBoxBlocks = 512;

__device__ __forceinline__ float nan_min(float a, float b) { return b < a || b != b ? b : a; }
__device__ __forceinline__ float nan_max(float a, float b) { return b > a || b != b ? b : a; }

__device__ __forceinline__ void block_box(float (&v)[6], float (*part)[6], float* __restrict__ out) {
#pragma unroll
    for (int a = 0; a < 6; ++a) {
        for (int off = 32; off > 0; off >>= 1) {
            const float u = __shfl_xor(v[a], off);
            v[a] = a < 3 ? nan_min(v[a], u) : nan_max(v[a], u);
        }
    }
    if ((threadIdx.x & 63) == 0)
        for (int a = 0; a < 6; ++a) part[threadIdx.x / 64][a] = v[a];
    __syncthreads();
    if (threadIdx.x < 6) {
        const int a = threadIdx.x;
        float r = part[0][a];
        for (int w = 1; w < kBlock / 64; ++w) r = a < 3 ? nan_min(r, part[w][a]) : nan_max(r, part[w][a]);
        out[a] = r;
    }
}

__global__ void __launch_bounds__(kBlock)
    points_box_blocks(const float* __restrict__ pts, int stride, int64_t n, float* __restrict__ box) {
    __shared__ float part[kBlock / 64][6];
    float v[6] = {pts[0], pts[1], pts[2], pts[0], pts[1], pts[2]};
    for (int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x; i < n; i += int64_t(gridDim.x) * kBlock) {
        const float* p = site_ptr(pts, stride, i);
#pragma unroll
        for (int a = 0; a < 3; ++a) v[a] = nan_min(v[a], p[a]), v[3 + a] = nan_max(v[3 + a], p[a]);
    }
    block_box(v, part, box + 6 * (1 + int64_t(blockIdx.x)));
}

__global__ void __launch_bounds__(kBlock) points_box_final(float* __restrict__ box, int blocks) {
    __shared__ float part[kBlock / 64][6];
    float v[6];
#pragma unroll
    for (int a = 0; a < 6; ++a) v[a] = box[6 + a];
    for (int b = threadIdx.x; b < blocks; b += kBlock) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            v[a] = nan_min(v[a], box[6 * (1 + b) + a]);
            v[3 + a] = nan_max(v[3 + a], box[6 * (1 + b) + 3 + a]);
        }
    }
    block_box(v, part, box);
}

}  // namespace
}  // namespace vgr

extern "C" int64_t vgr_points_box_floats(void) { return 6 * (1 + vgr::kBoxBlocks); }

extern "C" int vgr_points_box(const float* points, int64_t n, int32_t stride, float* box, void* stream) {
    using namespace vgr;
    VGR_REQUIRE(n >= 1, "points_box: n must be >= 1 (got %lld)", static_cast<long long>(n));
    VGR_REQUIRE(stride >= 3, "points_box: stride must be >= 3 floats (got %d)", stride);
    VGR_REQUIRE(points && box, "points_box: null pointer");
    const int64_t want = (n + kBlock - 1) / kBlock;
    const int blocks = static_cast<int>(want < kBoxBlocks ? want : kBoxBlocks);
    const hipStream_t s = as_stream(stream);
    hipLaunchKernelGGL(points_box_blocks, dim3(blocks), dim3(kBlock), 0, s, points, int(stride), n, box);
    hipLaunchKernelGGL(points_box_final, dim3(1), dim3(kBlock), 0, s, box, blocks);
    return launch_status("points_box");
}

extern "C" int64_t vgr_grid_work_size(int64_t n_sites, int64_t n_cells) {
    const int64_t tiles = (n_cells + vgr::kScanTile - 1) / vgr::kScanTile;
    return n_sites + n_cells + tiles + 1;
}

namespace vgr {
namespace {

// Counting sort of n points into the cells of g, with `work` (vgr_grid_work_size ints) for the place of every point in
// its cell, the per-cell counters and the scan's tile sums. The counters are cleared by a kernel (never hipMemsetAsync, so
// that a build can be captured in a graph).
int bin_points(const float* points, int64_t n, int32_t stride, const Geom& g, int64_t n_cells, int32_t* cell_start,
               int32_t* cell_sites, float4* cp, int32_t* work, hipStream_t s) {
    int* place = work;
    int* count = work + n;
    int* tile_sum = count + n_cells;
    hipLaunchKernelGGL(zero_ints, dim3(grid_for(n_cells, kBlock)), dim3(kBlock), 0, s, count, n_cells);
    if (int rc = launch_status("grid_build zero_ints")) return rc;
    if (n > 0) {
        hipLaunchKernelGGL(grid_count, dim3(grid_for(n, kBlock)), dim3(kBlock), 0, s, points, int(stride), n, g, place,
                           count);
        if (int rc = launch_status("grid_count")) return rc;
    }
    exclusive_scan(count, n_cells, cell_start, count, tile_sum, s);
    if (int rc = launch_status("grid_build scan")) return rc;
    if (n > 0) {
        hipLaunchKernelGGL(grid_fill, dim3(grid_for(n, kBlock)), dim3(kBlock), 0, s, points, int(stride), n, g,
                           cell_start, place, cell_sites, cp);
        return launch_status("grid_fill");
    }
    return VGR_OK;
}

int grid_build(const float* points, int64_t n_sites, int32_t stride, const float* lo, const float* cell,
               const int32_t* res, int32_t* cell_start, int32_t* cell_sites, float4* cp, int32_t* work, void* stream) {
    int64_t n_cells = 0;
    if (int rc = check_geom(lo, cell, res, &n_cells)) return rc;
    VGR_REQUIRE(n_sites >= 0 && n_sites <= INT_MAX, "grid_build: n_sites must be in [0, 2^31) (got %lld)",
                static_cast<long long>(n_sites));
    VGR_REQUIRE(stride >= 3, "grid_build: stride must be >= 3 floats (got %d)", stride);
    VGR_REQUIRE(cell_start && work && (n_sites == 0 || (points && cell_sites)), "grid_build: null pointer");
    return bin_points(points, n_sites, stride, make_geom(lo, cell, res), n_cells, cell_start, cell_sites, cp, work,
                      as_stream(stream));
}

}  // namespace
}  // namespace vgr

extern "C" int vgr_grid_build(const float* points, int64_t n_sites, int32_t stride, const float* lo, const float* cell,
                              const int32_t* res, int32_t* cell_start, int32_t* cell_sites, int32_t* work,
                              void* stream) {
    return vgr::grid_build(points, n_sites, stride, lo, cell, res, cell_start, cell_sites, nullptr, work, stream);
}

extern "C" int vgr_grid_build_points(const float* points, int64_t n_sites, int32_t stride, const float* lo,
                                     const float* cell, const int32_t* res, int32_t* cell_start, int32_t* cell_sites,
                                     float* cell_points, int32_t* work, void* stream) {
    VGR_REQUIRE(n_sites == 0 || cell_points, "grid_build_points: null pointer");
    VGR_REQUIRE(reinterpret_cast<uintptr_t>(cell_points) % 16 == 0, "grid_build_points: cell_points must be 16-byte "
                "aligned");
    return vgr::grid_build(points, n_sites, stride, lo, cell, res, cell_start, cell_sites,
                           reinterpret_cast<float4*>(cell_points), work, stream);
}

extern "C" int vgr_grid_build_noalloc(const float* points, int64_t n_sites, int32_t stride, const float* lo,
                                      const float* cell, const int32_t* res, int32_t* cell_start,
                                      int32_t* cell_sites, void* stream) {
    using namespace vgr;
    int64_t n_cells = 0;
    if (int rc = check_geom(lo, cell, res, &n_cells)) return rc;
    VGR_REQUIRE(n_sites >= 0 && n_sites <= INT_MAX, "grid_build_noalloc: n_sites must be in [0, 2^31) (got %lld)",
                static_cast<long long>(n_sites));
    const int64_t need = vgr_grid_work_size(n_sites, n_cells);
    VGR_REQUIRE(need <= kScratchInts,
                "grid_build_noalloc: %lld sites over %lld cells need %lld scratch ints, beyond the static %lld; use "
                "vgr_grid_build with a workspace",
                static_cast<long long>(n_sites), static_cast<long long>(n_cells), static_cast<long long>(need),
                static_cast<long long>(kScratchInts));
    int* work = nullptr;
    if (int rc = scratch_on_current_device(&work)) return rc;
    return grid_build(points, n_sites, stride, lo, cell, res, cell_start, cell_sites, nullptr, work, stream);
}

extern "C" int vgr_grid_nearest(const float* points, int64_t n_sites, int32_t stride, const float* lo,
                                const float* cell, const int32_t* res, const int32_t* cell_start,
                                const int32_t* cell_sites, const float* queries, int64_t n_queries, int32_t* site,
                                void* stream) {
    using namespace vgr;
    int64_t n_cells = 0;
    if (int rc = check_geom(lo, cell, res, &n_cells)) return rc;
    VGR_REQUIRE(n_queries >= 0, "grid_nearest: n_queries must be >= 0");
    if (n_queries == 0) return VGR_OK;
    VGR_REQUIRE(n_sites >= 1 && n_sites <= INT_MAX, "grid_nearest: n_sites must be in [1, 2^31) (got %lld)",
                static_cast<long long>(n_sites));
    VGR_REQUIRE(stride >= 3, "grid_nearest: stride must be >= 3 floats (got %d)", stride);
    VGR_REQUIRE(points && cell_start && cell_sites && queries && site, "grid_nearest: null pointer");
    const Geom g = make_geom(lo, cell, res);
    hipLaunchKernelGGL((grid_nearest<false, false>), dim3(grid_for(n_queries, kBlock)), dim3(kBlock), 0, as_stream(stream),
                       points, int(stride), g, cell_start, cell_sites, nullptr, queries, n_queries, nullptr,
                       nearest_margin(lo, cell, res), site);
    return launch_status("grid_nearest");
}

extern "C" int vgr_grid_cell_points(const float* points, int64_t n_sites, int32_t stride, const int32_t* cell_sites,
                                    float* cell_points, void* stream) {
    using namespace vgr;
    VGR_REQUIRE(n_sites >= 0 && n_sites <= INT_MAX, "grid_cell_points: n_sites must be in [0, 2^31) (got %lld)",
                static_cast<long long>(n_sites));
    VGR_REQUIRE(stride >= 3, "grid_cell_points: stride must be >= 3 floats (got %d)", stride);
    if (n_sites == 0) return VGR_OK;
    VGR_REQUIRE(points && cell_sites && cell_points, "grid_cell_points: null pointer");
    VGR_REQUIRE(reinterpret_cast<uintptr_t>(cell_points) % 16 == 0, "grid_cell_points: cell_points must be 16-byte "
                "aligned");
    hipLaunchKernelGGL(grid_cell_points, dim3(grid_for(n_sites, kBlock)), dim3(kBlock), 0, as_stream(stream), points,
                       int(stride), n_sites, cell_sites, reinterpret_cast<float4*>(cell_points));
    return launch_status("grid_cell_points");
}

extern "C" int vgr_grid_nearest_points(const float* cell_points, int64_t n_sites, const float* lo, const float* cell,
                                       const int32_t* res, const int32_t* cell_start, const float* queries,
                                       int64_t n_queries, const int32_t* order, int32_t* site, void* stream) {
    using namespace vgr;
    int64_t n_cells = 0;
    if (int rc = check_geom(lo, cell, res, &n_cells)) return rc;
    VGR_REQUIRE(n_queries >= 0, "grid_nearest_points: n_queries must be >= 0");
    if (n_queries == 0) return VGR_OK;
    VGR_REQUIRE(n_sites >= 1 && n_sites <= INT_MAX, "grid_nearest_points: n_sites must be in [1, 2^31) (got %lld)",
                static_cast<long long>(n_sites));
    VGR_REQUIRE(cell_points && cell_start && queries && site, "grid_nearest_points: null pointer");
    VGR_REQUIRE(reinterpret_cast<uintptr_t>(cell_points) % 16 == 0, "grid_nearest_points: cell_points must be "
                "16-byte aligned");
    const Geom g = make_geom(lo, cell, res);
    hipLaunchKernelGGL((grid_nearest<true, false>), dim3(grid_for(n_queries, kBlock)), dim3(kBlock), 0, as_stream(stream),
                       nullptr, 3, g, cell_start, nullptr, reinterpret_cast<const float4*>(cell_points), queries,
                       n_queries, order, nearest_margin(lo, cell, res), site);
    return launch_status("grid_nearest (cell points)");
}

extern "C" int64_t vgr_grid_binned_work_size(int64_t n_queries, int64_t n_cells) {
    return n_queries > 0 ? 16 * n_queries + 4 * (vgr_grid_work_size(n_queries, n_cells) + n_cells + 1) : 0;
}

extern "C" int vgr_grid_nearest_binned(const float* cell_points, int64_t n_sites, const float* lo, const float* cell,
                                       const int32_t* res, const int32_t* cell_start, const float* queries,
                                       int64_t n_queries, void* work, int64_t work_bytes, int32_t* site, void* stream) {
    using namespace vgr;
    int64_t n_cells = 0;
    if (int rc = check_geom(lo, cell, res, &n_cells)) return rc;
    VGR_REQUIRE(n_queries >= 0 && n_queries <= INT_MAX, "grid_nearest_binned: n_queries must be in [0, 2^31) (got %lld)",
                static_cast<long long>(n_queries));
    if (n_queries == 0) return VGR_OK;
    VGR_REQUIRE(n_sites >= 1 && n_sites <= INT_MAX, "grid_nearest_binned: n_sites must be in [1, 2^31) (got %lld)",
                static_cast<long long>(n_sites));
    VGR_REQUIRE(cell_points && cell_start && queries && site && work, "grid_nearest_binned: null pointer");
    VGR_REQUIRE(work_bytes >= vgr_grid_binned_work_size(n_queries, n_cells),
                "grid_nearest_binned: work must hold vgr_grid_binned_work_size(m, G) = %lld bytes",
                static_cast<long long>(vgr_grid_binned_work_size(n_queries, n_cells)));
    VGR_REQUIRE(reinterpret_cast<uintptr_t>(cell_points) % 16 == 0 && reinterpret_cast<uintptr_t>(work) % 16 == 0,
                "grid_nearest_binned: cell_points and work must be 16-byte aligned");
    const Geom g = make_geom(lo, cell, res);
    const hipStream_t s = as_stream(stream);
    float4* binned = static_cast<float4*>(work);
    int* start = reinterpret_cast<int*>(binned + n_queries);
    if (int rc = bin_points(queries, n_queries, 3, g, n_cells, start, nullptr, binned, start + n_cells + 1, s)) return rc;
    hipLaunchKernelGGL((grid_nearest<true, true>), dim3(grid_for(n_queries, kBlock)), dim3(kBlock), 0, s, nullptr, 3, g,
                       cell_start, nullptr, reinterpret_cast<const float4*>(cell_points),
                       reinterpret_cast<const float*>(binned), n_queries, nullptr, nearest_margin(lo, cell, res), site);
    return launch_status("grid_nearest (binned)");
}
