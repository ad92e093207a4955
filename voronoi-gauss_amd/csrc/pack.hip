// Records of the inference renderer from the model's tensors, gfx950: the step before foam_infer.
//
// Semantics follow pack_foam of the reference (render.py:179-225), with its optional Z-order renumbering
// (render.py:168-176; the permutation comes from the caller): self-first neighbourhoods (offsets of N + 1 entries,
// nbr of M + N), one float4 per edge = (p_j, half2(r2_j, lam_j)), the site records attr (N, 20) = (density conic,
// min(raw, 30), 0, colour conic, 0 x 6), the positions padded to float4, and the SH rows, all in the new numbering.
//   r2_j  = 2 max_k(s_jk^2 + floor^2) max(min(raw_j, 30) - ln eps_density, 0) (1 + 2^-9), or inf when eps_density = 0:
//           the squared distance beyond which rho_j G_j < eps_density (rounded up before the half conversion);
//   lam_j = min(1 / max_k(t_jk^2 + floor^2) (1 - 2^-9), 65000): the smallest eigenvalue of the colour conic,
//           rounded down; t the colour scales.
// Both halves are rounded to nearest even, as torch's half conversion does.
//
// Passes, all in the new numbering: the self-first row sizes and the inverse permutation, and the sizes' exclusive scan
// (the tile scan of vgr_scan.h); site records per site, staged in LDS so that every store is contiguous; SH rows per
// float4; edge rows with one lane per output entry. An edge record is read from the site records of the new numbering
// through inv[j]: spatial neighbours are close there, so only inv (4 bytes per site) is gathered at random, where records
// in the old numbering were 16. The derived records of an indexed pack (edge_i, attr_i, the slot table, the site rows) are
// written by the same passes, from registers and LDS. 2M sites renumbered,
// with the derived records (3.3 GB read and written at least, 0.69 ms at a copy's rate): 1.67 ms for the whole call, of which
// the edge rows 0.66 and the SH rows 0.34, against 2.89 ms with the derived records made by passes of their own.
//
// vgr_morton_codes gives the Z-order keys of the renumbering, with the arithmetic of morton_order (render.py:168-176):
// q = trunc((p - lo) / max(hi - lo, 1e-12) * 1023) per axis over the bounding box [lo, hi], bit b of axis a at
// bit 3 b + a of the key; vgr_morton_order also sorts them (30-bit keys, a stable radix sort) and gives the permutation.
#include <rocprim/device/device_radix_sort.hpp>

#include "vgr_abi.h"
#include "vgr_device.h"
#include "vgr_foam.h"
#include "vgr_scan.h"
#include "vgr_bbox.h"

#include <cmath>

namespace vgr {
namespace {

constexpr int kBlock = 256;

struct PackIn {
    const float* __restrict__ points;  // (N, 3)
    const int* __restrict__ offsets;   // (N + 1)
    const int* __restrict__ adj;       // (M)
    const float* __restrict__ raw;     // (N)
    const float* __restrict__ d_log_scale;  // (N, 3)
    const float* __restrict__ c_log_scale;  // (N, 3)
    const float* __restrict__ dA;      // (N, 6)
    const float* __restrict__ cA;      // (N, 6)
    const float4* __restrict__ sh;     // (N, 12) fp32
    const int* __restrict__ perm;      // (N) new -> old, or null (no renumbering)
    int n;
};

// Old index of new site i. perm is expected to be a permutation; an entry outside [0, N) is clamped so that no
// access leaves the arrays (the records are then meaningless, not out of bounds).
__device__ __forceinline__ int old_of(const PackIn& P, int i) {
    return P.perm != nullptr ? min(max(P.perm[i], 0), P.n - 1) : i;
}

// What the pack writes beside the reference's records (any of them may be null).
struct PackIndex {
    float4* __restrict__ edge_i;  // (E) p_j, the bits of j
    float4* __restrict__ attr_i;  // (N, 5) attr with column 7 = the site's cut-off word with its mark (kOddSite)
    int4* __restrict__ slots;     // (N, 4) slot table
    float4* __restrict__ rows;    // (N, row_vec) site rows: the first 16 columns of attr_i, then (row_vec 16) the SH row
    int row_vec;                  // 4 or 16 float4
};

// half2 cut-off word of old site o.
__device__ __forceinline__ float cut_word(const PackIn& P, int64_t o, float raw, float floor2, float log_eps, int eps_on) {
    float r2 = __builtin_huge_valf();
    if (eps_on) {
        float s_max2 = -kInf;
#pragma unroll
        for (int k = 0; k < 3; ++k)
            s_max2 = fmaxf(s_max2, expf(2.f * fminf(fmaxf(P.d_log_scale[3 * o + k], -20.f), 20.f)) + floor2);
        r2 = 2.f * s_max2 * fmaxf(raw - log_eps, 0.f) * (1.f + 0x1p-9f);
    }
    float c_max2 = -kInf;
#pragma unroll
    for (int k = 0; k < 3; ++k)
        c_max2 = fmaxf(c_max2, expf(2.f * fminf(fmaxf(P.c_log_scale[3 * o + k], -20.f), 20.f)) + floor2);
    const float lam = fminf(1.f / c_max2 * (1.f - 0x1p-9f), 65000.f);
    const uint16_t lo = __builtin_bit_cast(uint16_t, static_cast<_Float16>(r2));
    const uint16_t hi = __builtin_bit_cast(uint16_t, static_cast<_Float16>(lam));
    return __uint_as_float(static_cast<uint32_t>(lo) | (static_cast<uint32_t>(hi) << 16));
}

// Self-first row size of new site i, and inv[old] = new when renumbering.
__global__ void __launch_bounds__(kBlock) pack_size_kernel(PackIn P, int* __restrict__ size, int* __restrict__ inv) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= P.n) return;
    const int o = old_of(P, static_cast<int>(i));
    size[i] = P.offsets[o + 1] - P.offsets[o] + 1;
    if (P.perm != nullptr) inv[o] = static_cast<int>(i);
}

// Site records of new site i: position and cut-off word (the record of every edge that ends at it), padded position, attr
// row, and the derived rows. One lane per site gathers; the 20-float rows go through LDS (kSiteStride floats apart, odd, so
// that the lanes' writes hit distinct banks) and out contiguously.
constexpr int kSiteStride = 21;

__global__ void __launch_bounds__(kBlock)
    pack_sites_kernel(PackIn P, float floor2, float log_eps, int eps_on, float4* __restrict__ site4,
                      float4* __restrict__ pts4, float4* __restrict__ attr, PackIndex X) {
    __shared__ float rec[kBlock * kSiteStride];
    const int64_t i0 = static_cast<int64_t>(blockIdx.x) * kBlock, i = i0 + threadIdx.x;
    const int cnt = static_cast<int>(min(static_cast<int64_t>(kBlock), P.n - i0));
    if (i < P.n) {
        const int64_t o = old_of(P, static_cast<int>(i));
        const float raw = fminf(P.raw[o], 30.f);
        const float x = P.points[3 * o], y = P.points[3 * o + 1], z = P.points[3 * o + 2];
        const float cut = cut_word(P, o, raw, floor2, log_eps, eps_on);
        site4[i] = make_float4(x, y, z, cut);
        pts4[i] = make_float4(x, y, z, 0.f);
        float* a = rec + kSiteStride * threadIdx.x;
#pragma unroll
        for (int k = 0; k < 6; ++k) a[k] = P.dA[6 * o + k], a[8 + k] = P.cA[6 * o + k];
        a[6] = raw, a[7] = mark_site(cut, a + 8, x, y, z);
#pragma unroll
        for (int k = 14; k < 20; ++k) a[k] = 0.f;
    }
    __syncthreads();
    for (int t = threadIdx.x; t < 5 * cnt; t += kBlock) {
        const int s = t / 5, q = t - 5 * s;
        const float* a = rec + kSiteStride * s + 4 * q;
        float4 v = make_float4(a[0], a[1], a[2], a[3]);
        if (X.attr_i != nullptr) X.attr_i[5 * i0 + t] = v;
        if (X.rows != nullptr && q < 4) X.rows[X.row_vec * (i0 + s) + q] = v;
        if (q == 1) v.w = 0.f;
        attr[5 * i0 + t] = v;
    }
}

// SH rows in the new numbering, one float4 (of the 12 of a row) per lane, so that a wave writes 1 KB contiguously (fp32,
// fp16 when sh16 is given, and the SH part of 256-byte site rows). The rows come from P.sh, or, when it is null, from the
// model's own parts, the DC coefficients (N, 3) and the rest (N, 45).
__global__ void __launch_bounds__(kBlock)
    pack_sh_kernel(PackIn P, const float* __restrict__ dc, const float* __restrict__ rest, float4* __restrict__ sh32,
                   uint2* __restrict__ sh16, PackIndex X) {
    const int64_t t = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (t >= 12 * static_cast<int64_t>(P.n)) return;
    const int64_t i = t / 12;
    const int q = static_cast<int>(t - 12 * i);
    const int64_t o = old_of(P, static_cast<int>(i));
    float4 f;
    if (P.sh != nullptr) {
        f = P.sh[12 * o + q];
    } else {
        const float* r = rest + 45 * o + (4 * q - 3);
        f = q == 0 ? make_float4(dc[3 * o], dc[3 * o + 1], dc[3 * o + 2], r[3]) : make_float4(r[0], r[1], r[2], r[3]);
    }
    sh32[t] = f;
    if (sh16 != nullptr) {
        const uint32_t x = __builtin_bit_cast(uint16_t, static_cast<_Float16>(f.x)),
                       y = __builtin_bit_cast(uint16_t, static_cast<_Float16>(f.y)),
                       z = __builtin_bit_cast(uint16_t, static_cast<_Float16>(f.z)),
                       w = __builtin_bit_cast(uint16_t, static_cast<_Float16>(f.w));
        sh16[t] = make_uint2(x | (y << 16), z | (w << 16));
    }
    if (X.rows != nullptr && X.row_vec == 16) X.rows[16 * i + 4 + q] = f;
}

// The self-first rows of new sites i0 .. i0 + 63 (one wave): each site itself, then its neighbours in CSR order,
// renumbered. The rows are contiguous in the output, so the wave walks them with one lane per output entry (every
// store contiguous across the wave); a lane finds the site of its entry by a binary search over the 64 row starts,
// which lane s holds for site i0 + s. All lanes run every step (the shuffles read any lane).
//
// SLOTS: the slot table of the sites (their first and last entry of every slot j & 7, in CSR order) from 64-bit LDS
// minima and maxima of (entry, j), 16 per site.
template <bool SLOTS>
__global__ void __launch_bounds__(kBlock)
    pack_edges_kernel(PackIn P, const float4* __restrict__ site4, const int* __restrict__ inv,
                      const int* __restrict__ start, int* __restrict__ nbr, float4* __restrict__ edge, PackIndex X) {
    __shared__ unsigned long long ends[SLOTS ? kBlock * 16 : 1];
    const int lane = static_cast<int>(threadIdx.x) % 64;
    const int64_t i0 = (static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x) / 64 * 64;
    if (i0 >= P.n) return;  // whole waves; a wave's part of `ends` is its own
    unsigned long long* mine = ends + (SLOTS ? static_cast<int>(threadIdx.x) / 64 * (64 * 16) : 0);
    if (SLOTS)
        for (int t = lane; t < 64 * 16; t += 64) mine[t] = t % 16 < 8 ? ~0ull : 0ull;
    const int cnt = static_cast<int>(min(int64_t{64}, P.n - i0));
    const int64_t w_begin = start[i0], w_end = start[i0 + cnt];
    const bool has = lane < cnt;
    const int my_start = has ? start[i0 + lane] : static_cast<int>(w_end);  // past the rows: never <= an entry
    const int my_old = has ? old_of(P, static_cast<int>(i0 + lane)) : 0;
    const int my_e0 = has ? P.offsets[my_old] : 0;
    wave_sync();
    constexpr int U = 4;  // entries a lane has in flight: their loads (adj, inv, site4) depend on each other in turn
    for (int64_t base = w_begin; base < w_end; base += 64 * U) {
        int s[U], e[U], j[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t w = base + 64 * u + lane;
            s[u] = 0;  // the largest s with start[i0 + s] <= w
#pragma unroll
            for (int step = 32; step > 0; step >>= 1) {
                const int sm = __shfl(my_start, s[u] + step);
                if (sm <= w) s[u] += step;
            }
            const int row = __shfl(my_start, s[u]), e0 = __shfl(my_e0, s[u]);
            e[u] = static_cast<int>(w - row);
            j[u] = static_cast<int>(i0 + s[u]);
            if (w < w_end && e[u] > 0) j[u] = P.adj[e0 + e[u] - 1];
        }
        if (P.perm != nullptr) {
#pragma unroll
            for (int u = 0; u < U; ++u)  // in bounds whatever perm holds
                if (base + 64 * u + lane < w_end && e[u] > 0) j[u] = min(max(inv[j[u]], 0), P.n - 1);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t w = base + 64 * u + lane;
            if (w >= w_end) continue;
            const float4 v = site4[j[u]];
            nbr[w] = j[u];
            edge[w] = v;
            if (X.edge_i != nullptr) X.edge_i[w] = make_float4(v.x, v.y, v.z, __int_as_float(j[u]));
            if (SLOTS) {  // entry e + 1, so that 0 means none
                const unsigned long long key =
                    (static_cast<unsigned long long>(e[u] + 1) << 32) | static_cast<unsigned>(j[u]);
                atomicMin(mine + 16 * s[u] + (j[u] & 7), key);
                atomicMax(mine + 16 * s[u] + 8 + (j[u] & 7), key);
            }
        }
    }
    if (SLOTS) {
        wave_sync();
        for (int t = lane; t < 4 * cnt; t += 64) {  // one int4 (two slots) per lane
            const unsigned long long* m = mine + 16 * (t / 4) + 2 * (t % 4);
            const auto first = [](unsigned long long k) { return k == ~0ull ? -2 : static_cast<int>(k & 0xffffffffu); };
            const auto last = [](unsigned long long k) { return k == 0ull ? -2 : static_cast<int>(k & 0xffffffffu); };
            X.slots[4 * i0 + t] = make_int4(first(m[0]), last(m[8]), first(m[1]), last(m[9]));
        }
    }
}

// Scratch: float4 site4[N], int inv[N], int size[N], int tile_sum[tiles + 1] (sections 256-byte aligned).
constexpr int64_t align256p(int64_t b) { return (b + 255) / 256 * 256; }

int64_t pack_bytes(int64_t n) {
    return align256p(16 * n) + 2 * align256p(4 * n) + align256p(4 * (scan_tiles_of(n) + 1));
}


__global__ void __launch_bounds__(kBlock)
    morton_kernel(const float* __restrict__ points, int64_t n, const float* __restrict__ box, int bits,
                  int64_t* __restrict__ code, uint32_t* __restrict__ code32, int* __restrict__ idx) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= n) return;
    const float scale = static_cast<float>((1 << bits) - 1);
    int64_t key = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float lo = box[a], ext = fmaxf(box[3 + a] - lo, 1e-12f);
        const int64_t q = static_cast<int64_t>((points[3 * i + a] - lo) / ext * scale);
        for (int b = 0; b < bits; ++b) key |= ((q >> b) & 1) << (3 * b + a);
    }
    if (code != nullptr) code[i] = key;
    if (code32 != nullptr) code32[i] = static_cast<uint32_t>(key), idx[i] = static_cast<int>(i);
}

// The renumbering in the forms its users take: perm (new -> old) as int64, and its inverse.
__global__ void __launch_bounds__(kBlock) perm_forms_kernel(const int* __restrict__ perm32, int64_t n,
                                                            int64_t* __restrict__ perm, int64_t* __restrict__ inv) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= n) return;
    const int o = perm32[i];
    perm[i] = o;
    if (inv != nullptr) inv[o] = i;
}

size_t morton_sort_bytes(int64_t n) {
    size_t bytes = 0;
    (void)rocprim::radix_sort_pairs(nullptr, bytes, static_cast<const uint32_t*>(nullptr),
                                    static_cast<uint32_t*>(nullptr), static_cast<const int*>(nullptr),
                                    static_cast<int*>(nullptr), static_cast<size_t>(n), 0u, 30u);
    return bytes;
}

// Workspace of vgr_morton_order: per-block boxes, keys in and out, indices in, the sort's temporary storage.
int64_t order_work_bytes(int64_t n) {
    return align256p(4 * 6 * static_cast<int64_t>(grid_for(n, kBlock))) + 3 * align256p(4 * n) +
           align256p(static_cast<int64_t>(morton_sort_bytes(n)));
}

// Baked colour of site i for the view from c = (cx, cy, cz) (render.py:228-235): max(SH_i(d) + 1/2, 0) with
// d = (p_i - c) / max(|p_i - c|, 1e-12), written to attr[20 i + 16 .. 18]. The basis is sh_basis's; the
// coefficients of degree <= deg are summed in storage order, and only their float4 are read.
__global__ void __launch_bounds__(kBlock)
    bake_kernel(const float4* __restrict__ points4, const float4* __restrict__ sh32, int64_t n, int deg, float cx,
                float cy, float cz, float* __restrict__ attr) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= n) return;
    const float4 p = points4[i];
    float dx = p.x - cx, dy = p.y - cy, dz = p.z - cz;
    const float nrm = fmaxf(sqrtf(dx * dx + dy * dy + dz * dz), 1e-12f);
    dx /= nrm, dy /= nrm, dz /= nrm;
    float b[16];
    sh_basis(dx, dy, dz, deg, b);
    const int nb = (deg + 1) * (deg + 1);
    float c[3] = {0.f, 0.f, 0.f};
    const float4* s = sh32 + 12 * i;
#pragma unroll
    for (int q = 0; q < 12; ++q) {
        if (4 * q >= 3 * nb) break;
        const float4 f = s[q];
        const float fv[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = 4 * q + u;
            if (j / 3 < nb) c[j % 3] += b[j / 3] * fv[u];
        }
    }
    float* a = attr + 20 * i;
#pragma unroll
    for (int ch = 0; ch < 3; ++ch) a[16 + ch] = fmaxf(c[ch] + 0.5f, 0.f);
}

}  // namespace
}  // namespace vgr

extern "C" int vgr_bake_colors(const float* points4, const float* sh32, int64_t n_sites, int64_t sh_deg,
                               double cx, double cy, double cz, float* attr, void* stream) {
    using namespace vgr;
    VGR_REQUIRE(n_sites >= 0, "bake_colors: n_sites must be >= 0");
    VGR_REQUIRE(sh_deg >= 0 && sh_deg <= 3, "sh_deg must be in [0, 3] (got %lld)", static_cast<long long>(sh_deg));
    if (n_sites == 0) return VGR_OK;
    VGR_REQUIRE(points4 && sh32 && attr, "bake_colors: null pointer");
    hipLaunchKernelGGL(bake_kernel, dim3(grid_for(n_sites, kBlock)), dim3(kBlock), 0, as_stream(stream),
                       reinterpret_cast<const float4*>(points4), reinterpret_cast<const float4*>(sh32), n_sites,
                       int(sh_deg), float(cx), float(cy), float(cz), attr);
    return launch_status("bake_kernel");
}

extern "C" int64_t vgr_morton_work_size(int64_t n) {
    return n > 0 ? 4 * 6 * vgr::grid_for(n, vgr::kBlock) : 0;
}

extern "C" int vgr_morton_codes(const float* points, int64_t n, int32_t bits, int64_t* code, void* work,
                                int64_t work_bytes, void* stream) {
    using namespace vgr;
    VGR_REQUIRE(n >= 0, "morton_codes: n must be >= 0");
    VGR_REQUIRE(bits >= 1 && bits <= 21, "morton_codes: bits must be in [1, 21] (got %d)", bits);
    if (n == 0) return VGR_OK;
    VGR_REQUIRE(points && code, "morton_codes: null pointer");
    const int64_t blocks = grid_for(n, kBlock);
    VGR_REQUIRE(work != nullptr && work_bytes >= 4 * 6 * blocks, "morton_codes: work must hold %lld bytes",
                static_cast<long long>(4 * 6 * blocks));
    float* box = static_cast<float*>(work);
    const hipStream_t s = as_stream(stream);
    bounding_box(points, n, box, s);
    hipLaunchKernelGGL(morton_kernel, dim3(blocks), dim3(kBlock), 0, s, points, n, box, int(bits), code,
                       nullptr, nullptr);
    return launch_status("morton_codes");
}

extern "C" int64_t vgr_morton_order_work_size(int64_t n) { return n > 0 ? vgr::order_work_bytes(n) : 0; }

extern "C" int vgr_morton_order(const float* points, int64_t n, int32_t bits, int32_t* perm32, int64_t* perm, int64_t* inv,
                                void* work, int64_t work_bytes, void* stream) {
    using namespace vgr;
    VGR_REQUIRE(n >= 0 && n <= INT_MAX, "morton_order: n must be in [0, 2^31)");
    VGR_REQUIRE(bits >= 1 && bits <= 10, "morton_order: bits must be in [1, 10] (got %d)", bits);
    if (n == 0) return VGR_OK;
    VGR_REQUIRE(points && perm32 && perm, "morton_order: null pointer");
    const int64_t need = order_work_bytes(n);
    VGR_REQUIRE(work != nullptr && work_bytes >= need && reinterpret_cast<uintptr_t>(work) % 256 == 0,
                "morton_order: work must hold vgr_morton_order_work_size(n) = %lld bytes, 256-byte aligned",
                static_cast<long long>(need));
    char* w = static_cast<char*>(work);
    float* box = reinterpret_cast<float*>(w);
    w += align256p(4 * 6 * static_cast<int64_t>(grid_for(n, kBlock)));
    uint32_t* key = reinterpret_cast<uint32_t*>(w);
    w += align256p(4 * n);
    uint32_t* sorted = reinterpret_cast<uint32_t*>(w);
    w += align256p(4 * n);
    int* idx = reinterpret_cast<int*>(w);
    w += align256p(4 * n);
    size_t temp = morton_sort_bytes(n);
    const hipStream_t s = as_stream(stream);
    const dim3 grid(grid_for(n, kBlock)), block(kBlock);
    bounding_box(points, n, box, s);
    hipLaunchKernelGGL(morton_kernel, grid, block, 0, s, points, n, box, int(bits), nullptr, key, idx);
    if (int rc = launch_status("morton_order keys")) return rc;
    if (rocprim::radix_sort_pairs(w, temp, key, sorted, idx, perm32, static_cast<size_t>(n), 0u,
                                  static_cast<unsigned>(3 * bits), s) != hipSuccess)
        return launch_status("morton_order radix sort");
    hipLaunchKernelGGL(perm_forms_kernel, grid, block, 0, s, perm32, n, perm, inv);
    return launch_status("morton_order");
}

extern "C" int64_t vgr_pack_work_size(int64_t n_sites) { return n_sites > 0 ? vgr::pack_bytes(n_sites) : 0; }

namespace vgr {
namespace {

int pack_entry(const float* points, int64_t n_sites, const int32_t* offsets, const int32_t* adj, int64_t n_adj,
               const float* raw, const float* d_log_scale, const float* c_log_scale, const float* dA, const float* cA,
               const float* sh, const float* sh_dc, const float* sh_rest, const int32_t* perm, double scale_floor,
               double eps_density, float* points4, int32_t* offsets_sf, int32_t* nbr, float* edge, float* attr,
               float* sh32, void* sh16, const PackIndex& X, void* work, int64_t work_bytes, void* stream) {
    VGR_REQUIRE(n_sites > 0 && n_sites <= int64_t(kScanTile) * kScanTile,
                "pack_foam: n_sites must be in [1, %lld]", static_cast<long long>(int64_t(kScanTile) * kScanTile));
    VGR_REQUIRE(n_adj >= 0 && n_adj + n_sites <= INT_MAX, "pack_foam: n_adj + n_sites must be < 2^31");
    VGR_REQUIRE(points && offsets && (adj || n_adj == 0) && raw && d_log_scale && c_log_scale && dA && cA &&
                    (sh || (sh_dc && sh_rest)),
                "pack_foam: null input pointer");
    VGR_REQUIRE(points4 && offsets_sf && nbr && edge && attr && sh32, "pack_foam: null output pointer");
    VGR_REQUIRE(eps_density >= 0.0, "pack_foam: eps_density must be >= 0");
    VGR_REQUIRE(work != nullptr && work_bytes >= pack_bytes(n_sites) && reinterpret_cast<uintptr_t>(work) % 256 == 0,
                "pack_foam: work must hold vgr_pack_work_size(N) = %lld bytes, 256-byte aligned",
                static_cast<long long>(pack_bytes(n_sites)));
    const PackIn P{points, offsets, adj, raw, d_log_scale, c_log_scale, dA, cA, reinterpret_cast<const float4*>(sh),
                   perm, int(n_sites)};
    char* w = static_cast<char*>(work);
    float4* site4 = reinterpret_cast<float4*>(w);
    w += align256p(16 * n_sites);
    int* inv = reinterpret_cast<int*>(w);
    w += align256p(4 * n_sites);
    int* size = reinterpret_cast<int*>(w);
    w += align256p(4 * n_sites);
    int* tile_sum = reinterpret_cast<int*>(w);
    const hipStream_t s = as_stream(stream);
    const dim3 grid(grid_for(n_sites, kBlock)), block(kBlock);
    // ln(eps) in double, then fp32, as a Python float meets a float32 tensor
    const float log_eps = eps_density > 0.0 ? static_cast<float>(std::log(eps_density)) : 0.f;
    hipLaunchKernelGGL(pack_size_kernel, grid, block, 0, s, P, size, inv);
    exclusive_scan(size, n_sites, offsets_sf, size, tile_sum, s);  // offsets_sf[0 .. N]
    hipLaunchKernelGGL(pack_sites_kernel, grid, block, 0, s, P, static_cast<float>(scale_floor * scale_floor), log_eps,
                       eps_density > 0.0 ? 1 : 0, site4, reinterpret_cast<float4*>(points4),
                       reinterpret_cast<float4*>(attr), X);
    hipLaunchKernelGGL(pack_sh_kernel, dim3(grid_for(12 * n_sites, kBlock)), block, 0, s, P, sh_dc, sh_rest,
                       reinterpret_cast<float4*>(sh32), static_cast<uint2*>(sh16), X);
    if (X.slots != nullptr)
        hipLaunchKernelGGL(pack_edges_kernel<true>, grid, block, 0, s, P, site4, inv, offsets_sf, nbr,
                           reinterpret_cast<float4*>(edge), X);
    else
        hipLaunchKernelGGL(pack_edges_kernel<false>, grid, block, 0, s, P, site4, inv, offsets_sf, nbr,
                           reinterpret_cast<float4*>(edge), X);
    return launch_status("pack_foam");
}

}  // namespace
}  // namespace vgr

extern "C" int vgr_pack_foam(const float* points, int64_t n_sites, const int32_t* offsets, const int32_t* adj,
                             int64_t n_adj, const float* raw, const float* d_log_scale, const float* c_log_scale,
                             const float* dA, const float* cA, const float* sh, const int32_t* perm,
                             double scale_floor, double eps_density, float* points4, int32_t* offsets_sf,
                             int32_t* nbr, float* edge, float* attr, float* sh32, void* sh16, void* work,
                             int64_t work_bytes, void* stream) {
    return vgr::pack_entry(points, n_sites, offsets, adj, n_adj, raw, d_log_scale, c_log_scale, dA, cA, sh, nullptr,
                           nullptr, perm, scale_floor, eps_density, points4, offsets_sf, nbr, edge, attr, sh32, sh16,
                           vgr::PackIndex{}, work, work_bytes, stream);
}

extern "C" int vgr_pack_foam_indexed(const float* points, int64_t n_sites, const int32_t* offsets, const int32_t* adj,
                                     int64_t n_adj, const float* raw, const float* d_log_scale,
                                     const float* c_log_scale, const float* dA, const float* cA, const float* sh,
                                     const float* sh_dc, const float* sh_rest, const int32_t* perm, double scale_floor,
                                     double eps_density, float* points4, int32_t* offsets_sf, int32_t* nbr, float* edge,
                                     float* attr, float* sh32, void* sh16, float* edge_i, float* attr_i, int32_t* slots,
                                     float* rows, int64_t row_floats, void* work, int64_t work_bytes, void* stream) {
    VGR_REQUIRE(edge_i && attr_i && slots && rows, "pack_foam_indexed: null output pointer");
    VGR_REQUIRE(row_floats == 16 || row_floats == 64, "pack_foam_indexed: row_floats must be 16 or 64 (got %lld)",
                static_cast<long long>(row_floats));
    VGR_REQUIRE(reinterpret_cast<uintptr_t>(slots) % 16 == 0 && reinterpret_cast<uintptr_t>(rows) % 16 == 0,
                "pack_foam_indexed: slots and rows must be 16-byte aligned");
    const vgr::PackIndex X{reinterpret_cast<float4*>(edge_i), reinterpret_cast<float4*>(attr_i),
                           reinterpret_cast<int4*>(slots), reinterpret_cast<float4*>(rows), int(row_floats / 4)};
    return vgr::pack_entry(points, n_sites, offsets, adj, n_adj, raw, d_log_scale, c_log_scale, dA, cA, sh, sh_dc,
                           sh_rest, perm, scale_floor, eps_density, points4, offsets_sf, nbr, edge, attr, sh32, sh16, X,
                           work, work_bytes, stream);
}
