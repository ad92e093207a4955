// Inference renderer, one ray per lane with colours evaluated cell by cell on the matrix cores, gfx950: fused colours, and
// exact ones without a colour cut-off (+inf), for batches that fill the GPU with rays that share cells (the rule and what
// incoherent ones cost: default_lanes in foam_infer.hip).
//
// Same function as csrc/foam_infer.cu:286-361. A wave renders 64 consecutive rays (an 8 x 8 tile of the host's order). The
// walk, the exit faces and the density run one ray per lane, as in foam_infer.hip. A colour does not steer a ray: only the
// samples of segments heavier than w_thresh reach the image, each with the weight (w_before + w_after) / 2 of its two
// segments. So a lane queues those samples (position, weight, cell) in LDS, kDepth per ray, and when a ray's queue is full
// the wave evaluates all queued samples together (evaluate, blend_quads):
// - samples are sorted by cell into quads, four samples of one cell on four lanes (the rays of a tile cross the same cells
//   within a few steps), 64 samples at a time;
// - lane l of a quad reads the SH row of the cell's entry base + l; the colours of the quad's four samples at its four entries
//   are a product of rows (4 x 16) and SH bases (16 x 4), per channel 16 v_mfma_f32_4x4x1_f32 (fp32 in, fp32 sums, in the
//   order of the coefficients), each of which serves the wave's 16 quads at once and leaves a sample's four colours in its
//   own lane;
// - the lane clamps them, weighs them by exp(-(m_k - m_min) / 2) relative to its running minimum, and goes on with the
//   cell's next four entries: a sample's blend needs no other lane, and no value of it depends on the samples beside it;
// - every ray adds its queued contributions in the order of its samples, so a ray's colour does not depend on which rays
//   share its wave.
// An SH row is then read once per quad and its 48 multiply-adds run on the matrix cores, where a lookup per (sample,
// neighbour) through LDS took 12 LDS reads and 48 FMAs of every lane; samples of segments below w_thresh cost no colour.
//
// A finite cut-off (CUT) leaves a term out against the running minimum of the terms before it in edge order. A pass then
// also takes the colour distances, since the lookups they admit are counted (stats[:, 4]), and the evaluation, which visits
// a cell's entries in the same order with the same operations, admits the same terms.
//
// stats[:, 4], the reference's cache misses: without a cut-off a pass looks up all entries whose colour distance is a number,
// which but for degenerate sites is all of them, so that the count needs the cells: from the slot table with the ray's 8 tags
// in registers (count_lookups), or, without a table, from tags per lookup in LDS. EXACT: the exact
// (lazy) colour mode by the same one-pass blend. Its colour, sum_k exp(-(m_k - m_min) / 2) c_k / sum_k exp(-(m_k - m_min) / 2)
// over every neighbour, is the blend's two sums up to rounding; its statistics count a colour pass only where the reference
// runs one: for the far sample of a segment heavier than w_thresh and, when the segment before was not, its near sample.
//
// Bound by the texture data path, through which every gather returns: on the 2M-site scene below TD is busy 96 % of the
// launch, the L2 hits 97 %, and the VALU issues less than half of what the lookup per lane issued (4.7e10 against 1.0e11);
// in a view with fewer heavy segments the geometry pass is about half of the time (measured with the colours left out).
// One MI355X, ms of a render call, the one-ray-per-lane kernel of foam_infer.hip -> this one: 2M sites, 8.29M rays, fused,
// 69 % of the segments heavier than w_thresh, 179.9 -> 113.5; 1920 x 1080 rays of 2M sites, fused, 38 %, 78.4 -> 47.5;
// 800 x 800, exact, 29 %, 23.2 -> 11.5. With a cut-off of eps 1e-3: the first scene 169.8 -> 154.0, with fp16 SH 142.6 ->
// 125.5; 1237 x 822 rays, fp16, 40.1 -> 26.1.
// Not taken (two such views, 11.2 / 51.3 ms): 16 samples of a cell against 16 entries per v_mfma_f32_16x16x4_f32 13.7 /
// 60.2 (a cell's queue holds 6 samples on average, the rest is padding); the row's loads predicated on the entry instead of
// clamped to one of the cell's 16.8 / 81.6 (each becomes a branch with its own wait); the ray's state parked in LDS during the
// evaluation 11.7 / 53.5.
#include <cmath>
#include <type_traits>

#include "vgr_foam.h"

namespace vgr {
namespace {

constexpr int kBlock = 64;
constexpr int kRayTagSlots = 8;
// Queued samples per ray: 11.2 / 51.3 ms on the two views of the variants above; 3: 11.6 / 54.1 (smaller batches), 5: 12.0 /
// 55.1 (LDS).
constexpr int kDepth = 4;
// Waves per SIMD: 4 (128 VGPRs) hold the row, the basis and the ray with 13 spills (fp32, SH degree 3; none with fp16);
// 3 with 8 samples per ray 12.8 / 57.0, 5 spill: 19.9 / 86.7.
constexpr int kWaves = 4;

typedef float float4v __attribute__((ext_vector_type(4)));
typedef short short2v __attribute__((ext_vector_type(2), may_alias));  // two places of a queue's list

// LDS words as such (through a generic pointer they would be flat accesses, which wait for all outstanding loads).
typedef __attribute__((address_space(3))) volatile int lds_int;

constexpr int kQueued = kDepth * kBlock;  // samples of a wave's queue
constexpr int kHash = kQueued;            // entries of the hash table of their cells

struct Queue {
    float4 x[kQueued];  // position, weight; after evaluation weight * colour
    int cell[kQueued];
    int key[kHash];     // cells found (-1: free)
    int count[kHash];   // their samples, then the first place of the cell in `list`
    alignas(4) short list[4 * kQueued];  // samples by cell, every cell beginning a quad; -1: an empty place
};

// The walk of foam_infer.hip's one-ray-per-lane kernel.
template <bool IDX>
__device__ int walk(const FoamScene& S, int c, float x0, float x1, float x2, int& steps) {
    for (int it = 0; it < kWalkCap; ++it) {
        const float4 pc = S.points[c];
        float bd = (x0 - pc.x) * (x0 - pc.x) + (x1 - pc.y) * (x1 - pc.y) + (x2 - pc.z) * (x2 - pc.z);
        int bk = c;
        const int e0 = S.offsets[c], e1 = S.offsets[c + 1];
        for (int e = e0 + 1; e < e1; ++e) {
            const float4 ed = S.edge[e];
            const int k = IDX ? __float_as_int(ed.w) : S.nbr[e];
            const float v0 = x0 - ed.x, v1 = x1 - ed.y, v2 = x2 - ed.z;
            const float dk = v0 * v0 + v1 * v1 + v2 * v2;
            if (dk < bd || (dk == bd && before(S, k, bk))) bd = dk, bk = k;
        }
        if (bk == c) break;
        c = bk;
        ++steps;
    }
    return c;
}

struct Pass {
    float sigma, t_exit;
    int next;  // exit neighbour
    int n;     // entries of the cell; ~entries when the pass may not look all of them up (count_lookups)
};

// Every pass looks up the entries of its cell whose colour distance is a number (without a cut-off). That is every entry,
// except beside a site whose colour conic is not finite, or so far out that the distance overflows. Where distances are not
// taken, such a pass is told by vgr_foam.h's kOddSite, which the indexed records carry per site, and by the sample's position:
// no further bytes, config 3 113.2 ms (113.4 when every entry was counted). The reference records have no room for the mark,
// and tags per lookup need the distances in order, so those forms take them: 262144 rays of two scenes 5.0 -> 7.0 and 7.3 ->
// 9.8 ms without both (the lookup per lane before this layout: 7.0 and 17.3).
constexpr float kOddPosition = 1e9f;  // as kOddSite: 9 terms of at most 1e18 * (2e9)^2 stay below FLT_MAX

// Density at o + t d over the neighbourhood of c and, when want_exit, the exit face: foam_infer.hip's sequential pass (the
// same operations in the same order). The next edge record is requested while the current entry is evaluated.
// TAGS (no slot table): the lookups that miss the ray's tags, which start at `tags`, 64 ints apart. CUT: a finite colour
// cut-off, so a lookup is an entry within it of the running minimum of the entries before.
template <bool IDX, bool TAGS, bool CUT>
__device__ __forceinline__ Pass pass(const FoamScene& S, int c, float t, const float (&o)[3], const float (&d)[3],
                                     bool want_exit, int& n_dens, int& n_sh, lds_int* tags, float color_cut) {
    constexpr bool DIST = CUT || TAGS || !IDX;  // the pass takes the colour distances
    const int e0 = S.offsets[c], e1 = S.offsets[c + 1];
    float4 edn = S.edge[entry_in(e0, e1)];
    int kn = 0;
    if constexpr (!IDX) kn = S.nbr[entry_in(e0, e1)];
    const float4 pc = S.points[c];
    float x[3];
    sample_point(o, d, t, x);
    Pass R{0.f, kInf, INT_MAX, e1 - e0};
    float low = kInf;
    uint32_t words = 0;
    bool odd = !DIST && !(fabsf(x[0]) <= kOddPosition && fabsf(x[1]) <= kOddPosition && fabsf(x[2]) <= kOddPosition);
    for (int e = e0; e < e1; ++e) {
        const float4 ed = edn;
        const int k = IDX ? __float_as_int(ed.w) : kn;
        const float4* a = S.attr + 5 * static_cast<int64_t>(k);
        const float4 q0 = a[0], q1 = a[1];
        float4 q2, q3;
        if constexpr (DIST) q2 = a[2], q3 = a[3];
        const int en = min(e + 1, e1 - 1);
        edn = S.edge[en];
        if constexpr (!IDX) kn = S.nbr[en];
        if (want_exit && e > e0) {
            const float n0 = ed.x - pc.x, n1 = ed.y - pc.y, n2 = ed.z - pc.z;
            const float dn = n0 * d[0] + n1 * d[1] + n2 * d[2];
            if (dn > 0.f) {
                const float m0 = 0.5f * (ed.x + pc.x) - o[0], m1 = 0.5f * (ed.y + pc.y) - o[1],
                            m2 = 0.5f * (ed.z + pc.z) - o[2];
                const float tt = (m0 * n0 + m1 * n1 + m2 * n2) / dn;
                if (tt < R.t_exit || (tt == R.t_exit && (R.next == INT_MAX || before(S, k, R.next))))
                    R.t_exit = tt, R.next = k;
            }
        }
        float v0, v1, v2, r2;
        offset_of(x, ed, v0, v1, v2, r2);
        const float word = IDX ? q1.w : ed.w;
        const float2 cut = cutoffs(word);
        if (!DIST) words |= __float_as_uint(word);
        if (r2 <= (IDX ? fabsf(cut.x) : cut.x)) {
            R.sigma += density_term(q0, q1, v0, v1, v2);
            ++n_dens;
        }
        bool look = true;
        if constexpr (DIST) {
            const float lim = CUT ? low + color_cut : color_cut;
            look = r2 * cut.y <= lim;
            if (look) {
                const float m = maha_f(q2, q3, v0, v1, v2);
                look = m <= lim;
                if (CUT) low = look && m < low ? m : low;
            }
            odd = odd || !look;
        }
        if (TAGS && look) {
            lds_int* p = tags + (k & (kRayTagSlots - 1)) * kBlock;
            n_sh += *p != k ? 1 : 0;
            *p = k;
        }
    }
    if (!TAGS && (odd || (words & kOddSite) != 0)) R.n = ~R.n;
    return R;
}

// The lookups of a pass over cell c that hit the ray's tags (foam_infer.hip's table_hits, all 8 slots in one lane).
__device__ __forceinline__ int table_hits(const FoamScene& S, int c, int (&tag)[kRayTagSlots]) {
    const int4* row = S.slots + 4 * static_cast<int64_t>(c);
    int hits = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int4 v = row[q];
        hits += v.x == tag[2 * q] ? 1 : 0;
        tag[2 * q] = v.y >= 0 ? v.y : tag[2 * q];
        hits += v.z == tag[2 * q + 1] ? 1 : 0;
        tag[2 * q + 1] = v.w >= 0 ? v.w : tag[2 * q + 1];
    }
    return hits;
}

// The reference's cache misses of the pass over cell c at o + t d, without a cut-off: of all n entries by the slot table, or
// (n = ~entries, rare) of those whose colour distance is a number, entry by entry.
template <bool IDX>
__device__ __forceinline__ int count_lookups(const FoamScene& S, int c, int n, float t, const float (&o)[3],
                                             const float (&d)[3], int (&tag)[kRayTagSlots]) {
    if (n >= 0) return n - table_hits(S, c, tag);
    float x[3];
    sample_point(o, d, t, x);
    int misses = 0;
    const int e0 = S.offsets[c];
    for (int e = e0; e < e0 + ~n; ++e) {
        const float4 ed = S.edge[e];
        const int k = IDX ? __float_as_int(ed.w) : S.nbr[e];
        const float4* a = S.attr + 5 * static_cast<int64_t>(k);
        float v0, v1, v2, r2;
        offset_of(x, ed, v0, v1, v2, r2);
        const float lb = r2 * cutoffs(IDX ? a[1].w : ed.w).y, m = maha_f(a[2], a[3], v0, v1, v2);
        if (lb != lb || m != m) continue;
#pragma unroll
        for (int s = 0; s < kRayTagSlots; ++s) {
            const bool here = (k & (kRayTagSlots - 1)) == s;
            misses += here && tag[s] != k ? 1 : 0;
            tag[s] = here ? k : tag[s];
        }
    }
    return misses;
}

// Blends of 64 samples, one per lane, the four samples of a quad in one cell (`cell`, -1 for a quad without samples): lane l
// reads entry base + l % 4 of its quad's cell, the quad's four lanes share the four entries. `dir` is the sample's direction.
template <bool IDX, bool HALF, int DEG, bool CUT>
__device__ __forceinline__ void blend_quads(const FoamScene& S, float color_cut, int cell, const float (&x)[3],
                                            const float (&dir)[3], float (&C)[3]) {
    constexpr int NB = (DEG + 1) * (DEG + 1), NV = sh_vec4<HALF, DEG>();
    const int lane = static_cast<int>(threadIdx.x);
    float b[16];
    sh_basis(dir[0], dir[1], dir[2], DEG, b);
    int base = 0, e1 = 0;
    if (cell >= 0) base = S.offsets[cell], e1 = S.offsets[cell + 1];
    float m = kInf, A = 0.f, cr = 0.f, cg = 0.f, cb = 0.f;
    for (; wave_any(base < e1); base += 4) {
        const int e = entry_in(base + lane % 4, e1);  // an absent entry: another's records, left out
        const float4 ed = S.edge[e];
        const int k = IDX ? __float_as_int(ed.w) : S.nbr[e];
        const float4* row = S.sh + S.sh_stride * static_cast<int64_t>(k);
        float4 f[NV];
#pragma unroll
        for (int u = 0; u < NV; ++u) f[u] = row[u];
        const float4* at = S.attr + 5 * static_cast<int64_t>(k);
        const float4 q2 = at[2], q3 = at[3];
        const auto coef = [&](int i) {
            constexpr int PER = HALF ? 8 : 4;
            const float4 v = f[i / PER];
            if (HALF) {
                const int w = i % 8 / 2;
                const float2 h = cutoffs(w == 0 ? v.x : w == 1 ? v.y : w == 2 ? v.z : v.w);
                return i % 2 ? h.y : h.x;
            }
            return i % 4 == 0 ? v.x : i % 4 == 1 ? v.y : i % 4 == 2 ? v.z : v.w;
        };
        float4v c0 = {0.5f, 0.5f, 0.5f, 0.5f}, c1 = c0, c2 = c0;
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            c0 = __builtin_amdgcn_mfma_f32_4x4x1f32(coef(3 * j), b[j], c0, 0, 0, 0);
            c1 = __builtin_amdgcn_mfma_f32_4x4x1f32(coef(3 * j + 1), b[j], c1, 0, 0, 0);
            c2 = __builtin_amdgcn_mfma_f32_4x4x1f32(coef(3 * j + 2), b[j], c2, 0, 0, 0);
        }
        float lam = 0.f;  // the entry's bound: m >= lam r2
        if constexpr (CUT) lam = cutoffs(IDX ? at[1].w : ed.w).y;
        const auto distance = [&](auto perm, int r, float& lb) {  // of entry base + r, from the quad's lane r
            constexpr int P = decltype(perm)::value;
            const float4 p = make_float4(row_perm<P>(ed.x), row_perm<P>(ed.y), row_perm<P>(ed.z), 0.f);
            const float4 a = make_float4(row_perm<P>(q2.x), row_perm<P>(q2.y), row_perm<P>(q2.z), row_perm<P>(q2.w));
            const float4 c = make_float4(row_perm<P>(q3.x), row_perm<P>(q3.y), 0.f, 0.f);
            float v0, v1, v2, r2;
            offset_of(x, p, v0, v1, v2, r2);
            if constexpr (CUT) lb = r2 * row_perm<P>(lam);
            return maha_f(a, c, v0, v1, v2);
        };
        float lb[4], mk[4];
        mk[0] = distance(std::integral_constant<int, 0x00>{}, 0, lb[0]);
        mk[1] = distance(std::integral_constant<int, 0x55>{}, 1, lb[1]);
        mk[2] = distance(std::integral_constant<int, 0xAA>{}, 2, lb[2]);
        mk[3] = distance(std::integral_constant<int, 0xFF>{}, 3, lb[3]);
        float low = m;
#pragma unroll
        for (int r = 0; r < 4; ++r) {  // a term left out (absent, NaN, or beyond the cut-off): kInf, weight 0
            const float lim = CUT ? low + color_cut : kInf;
            const bool in = base + r < e1 && (!CUT || lb[r] <= lim) && mk[r] <= lim;
            mk[r] = in ? mk[r] : kInf;
            low = fminf(low, mk[r]);
        }
        const float keep = weight_of(m, low);
        A *= keep, cr *= keep, cg *= keep, cb *= keep, m = low;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            // max(c, 0); the colour of a term left out is also kept finite, lest 0 * inf make a NaN of the blend
            const float top = mk[r] < kInf ? __builtin_huge_valf() : kInf;
            const float c[3] = {__builtin_amdgcn_fmed3f(c0[r], 0.f, top), __builtin_amdgcn_fmed3f(c1[r], 0.f, top),
                                __builtin_amdgcn_fmed3f(c2[r], 0.f, top)};
            accumulate(A, cr, cg, cb, weight_of(mk[r], low), c);
        }
    }
    const float inv = m < kInf ? 1.f / A : __builtin_nanf("");  // every term left out: 0 / 0, as in the other layouts
    C[0] = cr * inv, C[1] = cg * inv, C[2] = cb * inv;
}

// Evaluates every queued sample (the whole wave takes part): `queued` of each ray, sample s of ray r at 64 s + r. The samples
// are grouped by cell through a hash table in LDS (a cell's entry counts its samples and gives each its rank; an exclusive
// scan of the counts, rounded up to quads, gives the cells their places), then evaluated 64 places at a time.
template <bool IDX, bool HALF, int DEG, bool CUT>
__device__ __forceinline__ void evaluate(const FoamScene& S, float color_cut, Queue& Q, int queued, const float (&d)[3]) {
    const int lane = static_cast<int>(threadIdx.x);
    constexpr int PER = kHash / kBlock;
#pragma unroll
    for (int u = 0; u < PER; ++u) Q.key[kBlock * u + lane] = -1, Q.count[kBlock * u + lane] = 0;
#pragma unroll
    for (int u = 0; u < 2 * kDepth; ++u) reinterpret_cast<short2v*>(Q.list)[kBlock * u + lane] = short2v{-1, -1};
    wave_sync();
    int slot[kDepth], rank[kDepth];
#pragma unroll
    for (int s = 0; s < kDepth; ++s) {
        slot[s] = rank[s] = 0;
        if (s < queued) {
            const int c = Q.cell[kBlock * s + lane];
            int h = static_cast<int>((static_cast<uint32_t>(c) * 2654435761u) >> 8) & (kHash - 1);
            for (int probe = 0; probe < kHash; ++probe) {  // at most kHash cells: a free entry or the cell's is found
                const int held = atomicCAS(Q.key + h, -1, c);
                if (held == -1 || held == c) break;
                h = (h + 1) & (kHash - 1);
            }
            slot[s] = h, rank[s] = atomicAdd(Q.count + h, 1);
        }
    }
    wave_sync();
    int places[PER], sum = 0;
#pragma unroll
    for (int u = 0; u < PER; ++u) places[u] = (Q.count[PER * lane + u] + 3) & ~3, sum += places[u];
    int run = sum;  // inclusive scan over the lanes
#pragma unroll
    for (int off = 1; off < kBlock; off <<= 1) {
        const int v = __shfl_up(run, off);
        if (lane >= off) run += v;
    }
    const int total = __builtin_amdgcn_readlane(run, kBlock - 1);
    run -= sum;
    wave_sync();
#pragma unroll
    for (int u = 0; u < PER; ++u) Q.count[PER * lane + u] = run, run += places[u];
    wave_sync();
#pragma unroll
    for (int s = 0; s < kDepth; ++s)
        if (s < queued) Q.list[Q.count[slot[s]] + rank[s]] = static_cast<short>(kBlock * s + lane);
    wave_sync();
    for (int first = 0; first < total; first += kBlock) {
        const int at = first + lane < total ? Q.list[first + lane] : -1;
        const int lead = row_perm<0x00>(at);  // the quad's first sample, there if any is
        const int from = at >= 0 ? at : max(lead, 0);
        const float4 q = Q.x[from];
        const float x[3] = {q.x, q.y, q.z};
        const int ray = from % kBlock;
        const float dir[3] = {__shfl(d[0], ray), __shfl(d[1], ray), __shfl(d[2], ray)};
        float C[3];
        blend_quads<IDX, HALF, DEG, CUT>(S, color_cut, lead >= 0 ? Q.cell[from] : -1, x, dir, C);
        if (at >= 0) Q.x[at] = make_float4(q.w * C[0], q.w * C[1], q.w * C[2], 0.f);
    }
    wave_sync();
}

// IDX: the indexed edge records (vgr_foam_index_pack). TABLE: cache misses from the slot table. EXACT: the exact colour
// mode's statistics (its colour passes: segments with weight > w_thresh, the far sample's cell and, when the segment before
// was not coloured, the near sample's); always with the table.
template <bool IDX, bool HALF, int DEG, bool CUT, bool TABLE, bool EXACT>
__global__ void __launch_bounds__(kBlock, kWaves) foam_tile_kernel(FoamScene S, FoamParams P, FoamRays R, FoamOut O) {
    __shared__ Queue Q;
    __shared__ int lds_tags[TABLE ? 1 : kRayTagSlots * kBlock];
    const int lane = static_cast<int>(threadIdx.x);
    lds_int* my_tags = (lds_int*)(lds_tags + (TABLE ? 0 : lane));
    if (!TABLE)
        for (int s = 0; s < kRayTagSlots; ++s) my_tags[s * kBlock] = -1;
    const int64_t i = xcd_block_id() * kBlock + lane;
    int64_t r = -1;
    if (i < R.n) {
        r = R.order != nullptr ? R.order[i] : i;
        if (r >= R.n) r = -1;
    }
    const bool ours = r >= 0;  // a lane without a ray stays for the wave's evaluations
    const int start = ours ? R.start[r] : -1;
    bool alive = start >= 0 && start < S.n_sites;
    float o[3] = {0.f, 0.f, 0.f}, d[3] = {0.f, 0.f, 1.f}, t_far = 0.f, tA = 0.f;
    int max_samples = INT_MAX;
    int walk_steps = 0, n_dens = 0, n_sh = 0, n_samples = 0, n_color = 0;
    int tag[kRayTagSlots];
#pragma unroll
    for (int s = 0; s < kRayTagSlots; ++s) tag[s] = -1;
    int cA = 0, nA = 0;
    Pass E{0.f, kInf, INT_MAX, 0};
    if (alive) {
#pragma unroll
        for (int a = 0; a < 3; ++a) o[a] = R.o[3 * r + a], d[a] = R.d[3 * r + a];
        t_far = R.t_far[r], tA = R.t_near[r];
        if (R.cap != nullptr) max_samples = R.cap[r];
        cA = walk<IDX>(S, start, o[0] + tA * d[0], o[1] + tA * d[1], o[2] + tA * d[2], walk_steps);
        E = pass<IDX, !TABLE, CUT>(S, cA, tA, o, d, true, n_dens, n_sh, my_tags, P.color_cut);
        nA = E.n;
        if (TABLE && !EXACT) n_sh += count_lookups<IDX>(S, cA, E.n, tA, o, d, tag);
        if (O.trace != nullptr) trace_cell<true>(S, O, r, 0, cA);
        n_samples = 1;
    }
    float T = 1.f, acc[3] = {0.f, 0.f, 0.f}, dep = 0.f, sA = E.sigma;
    float wA = 0.f;  // the near sample's share of the segment before
    bool lit_before = false, ended = false;  // ended: the last sample is still to be queued
    int queued = 0;
    for (;;) {
        float weight = 0.f, at[3] = {0.f, 0.f, 0.f};
        const int at_cell = cA;
        if (alive) {
            const bool last = E.next == INT_MAX || E.t_exit >= t_far || n_samples + 1 >= max_samples;
            const float tB = last ? t_far : fmaxf(E.t_exit, tA);
            const int cB = last ? cA : E.next;
            E = pass<IDX, !TABLE, CUT>(S, cB, tB, o, d, !last, n_dens, n_sh, my_tags, P.color_cut);
            if (TABLE && !EXACT) n_sh += count_lookups<IDX>(S, cB, E.n, tB, o, d, tag);
            if (O.trace != nullptr) trace_cell<true>(S, O, r, n_samples, cB);
            ++n_samples;
            const float delta = tB - tA;
            const float alpha = 1.f - fexp(-0.5f * (sA + E.sigma) * delta);
            const float w = T * alpha;
            const bool lit = w > P.w_thresh;
            const float half = lit ? 0.5f * w : 0.f;
            if (lit) {
                if constexpr (EXACT) {
#pragma unroll 1  // one copy of the rare part: two spill 17 more VGPRs
                    for (int far = lit_before ? 1 : 0; far < 2; ++far)
                        n_sh += count_lookups<IDX>(S, far ? cB : cA, far ? E.n : nA, far ? tB : tA, o, d, tag);
                }
                dep += w * 0.5f * (tA + tB);
                ++n_color;
            }
            T *= 1.f - alpha;
            weight = wA + half;
            sample_point(o, d, tA, at);
            cA = cB, nA = E.n, tA = tB, sA = E.sigma, wA = half, lit_before = lit;
            if (last || T < P.t_thresh || n_samples > kMaxCells) alive = false, ended = true;
        } else if (ended) {
            weight = wA, ended = false;
            sample_point(o, d, tA, at);
        }
        if (weight != 0.f) {
            Q.x[kBlock * queued + lane] = make_float4(at[0], at[1], at[2], weight);
            Q.cell[kBlock * queued + lane] = at_cell;
            ++queued;
        }
        const bool done = !wave_any(alive || ended);
        if (done || wave_any(queued == kDepth)) {
            wave_sync();
            evaluate<IDX, HALF, DEG, CUT>(S, P.color_cut, Q, queued, d);
            for (int s = 0; s < queued; ++s) {
                const float4 v = Q.x[kBlock * s + lane];
                acc[0] += v.x, acc[1] += v.y, acc[2] += v.z;
            }
            queued = 0;
        }
        if (done) break;
    }
    if (!ours) return;
#pragma unroll
    for (int a = 0; a < 3; ++a) O.rgb[3 * r + a] = acc[a];
    O.T[r] = T;
    O.depth[r] = dep;
    int* st = O.stats + 5 * r;
    st[0] = n_samples, st[1] = n_color, st[2] = walk_steps, st[3] = n_dens, st[4] = n_sh;
}

template <bool IDX, bool HALF, bool CUT, bool TABLE, bool EXACT>
void launch(const FoamScene& S, const FoamParams& P, const FoamRays& R, const FoamOut& O, hipStream_t stream) {
    const dim3 grid(grid_for(R.n, kBlock)), block(kBlock);
    const auto run = [&](auto deg) {
        hipLaunchKernelGGL((foam_tile_kernel<IDX, HALF, decltype(deg)::value, CUT, TABLE, EXACT>), grid, block, 0, stream, S, P,
                           R, O);
    };
    switch (P.sh_deg) {
        case 0: run(std::integral_constant<int, 0>{}); break;
        case 1: run(std::integral_constant<int, 1>{}); break;
        case 2: run(std::integral_constant<int, 2>{}); break;
        default: run(std::integral_constant<int, 3>{});
    }
}

template <bool HALF>
void launch_half(const FoamScene& S, const FoamParams& P, const FoamRays& R, const FoamOut& O, bool indexed, bool exact,
                 hipStream_t stream) {
    const bool table = S.slots != nullptr;
    if (!(std::isinf(P.color_cut) && P.color_cut > 0))  // lookups depend on the distances: tags per lookup
        indexed ? launch<true, HALF, true, false, false>(S, P, R, O, stream)
                : launch<false, HALF, true, false, false>(S, P, R, O, stream);
    else if (exact)  // always indexed, with the slot table
        launch<true, HALF, false, true, true>(S, P, R, O, stream);
    else if (indexed)
        table ? launch<true, HALF, false, true, false>(S, P, R, O, stream)
              : launch<true, HALF, false, false, false>(S, P, R, O, stream);
    else
        table ? launch<false, HALF, false, true, false>(S, P, R, O, stream)
              : launch<false, HALF, false, false, false>(S, P, R, O, stream);
}

}  // namespace

int launch_foam_tile(const FoamScene& S, const FoamParams& P, const FoamRays& R, const FoamOut& O, bool indexed,
                     bool exact, bool half, hipStream_t stream) {
    half ? launch_half<true>(S, P, R, O, indexed, exact, stream) : launch_half<false>(S, P, R, O, indexed, exact, stream);
    return launch_status("foam_tile_kernel");
}

}  // namespace vgr
