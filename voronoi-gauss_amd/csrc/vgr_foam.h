// What the kernels of the inference renderer share (foam_infer.hip, foam_wide.hip, foam_tile.hip): the scene, ray and output
// arguments, the field arithmetic and the tie order of the exit faces.
#pragma once

#include "vgr_abi.h"
#include "vgr_device.h"

namespace vgr {

constexpr int kLazy = VGR_COLOR_LAZY, kBaked = VGR_COLOR_BAKED, kFused = VGR_COLOR_FUSED;

struct FoamScene {
    const float4* __restrict__ points;  // (N) p, w unused
    const int* __restrict__ offsets;    // (N + 1) self-first
    const int* __restrict__ nbr;        // (E)
    const float4* __restrict__ edge;    // (E) p_j, half2(r2_j, lam_j)
    const float4* __restrict__ attr;    // (N, 5)
    const float4* __restrict__ sh;      // (N, 12) fp32 or (N, 6) fp16
    const int* __restrict__ orig;       // (N) or null
    const int4* __restrict__ slots;     // (N, 4) slot table (vgr_foam_slot_table) or null
    const float4* __restrict__ rows;    // site rows (the first 16 attr columns) or null, row_stride float4 apart
    int n_sites;
    int row_stride;  // float4 from one site row to the next: 4 (64-byte rows) or 16 (256-byte site blocks)
    int sh_stride;   // float4 from one SH row to the next: 12 (fp32), 6 (fp16) or 16 (the SH rows of site blocks)
};

// Mark of a site in its word of the indexed records (the sign of half2(r2, lam)'s r2, which is never negative): a colour
// distance to it need not be a number. Its colour conic is not finite or above 1e18, its position not finite or beyond 1e9, or
// its bound lam not a number; of every other site, from samples within 1e9, the distance and its bound are finite.
constexpr uint32_t kOddSite = 0x8000u;

__device__ __forceinline__ float mark_site(float word, const float* conic, float px, float py, float pz) {
    const uint32_t u = __float_as_uint(word), lam = u >> 16;
    bool even = (lam & 0x7c00u) != 0x7c00u && fabsf(px) <= 1e9f && fabsf(py) <= 1e9f && fabsf(pz) <= 1e9f;
#pragma unroll
    for (int q = 0; q < 6; ++q) even = even && fabsf(conic[q]) <= 1e18f;
    return __uint_as_float(even ? u : u | kOddSite);
}

struct FoamParams {
    float t_thresh, w_thresh, color_cut;
    int sh_deg;
};

struct FoamRays {
    const float* __restrict__ o;
    const float* __restrict__ d;
    const int* __restrict__ start;
    const float* __restrict__ t_near;
    const float* __restrict__ t_far;
    const int* __restrict__ cap;
    int64_t n;
    const int* __restrict__ order;  // processing order of the rays (a permutation of 0 .. n - 1), or null
};

struct FoamOut {
    float* __restrict__ rgb;
    float* __restrict__ T;
    float* __restrict__ depth;
    int* __restrict__ stats;
    int* __restrict__ trace;
    int64_t trace_cap;
};

// The whole rendering (stage 2) with 16 lanes per ray, for batches too small to fill the GPU with one ray per lane
// (foam_wide.hip).
int launch_foam_wide(const FoamScene& S, const FoamParams& P, const FoamRays& R, const FoamOut& O, int color_mode,
                     bool half, hipStream_t stream);

// Fused colours, one ray per lane, evaluated cell by cell on the matrix cores (foam_tile.hip); exact: the exact colour mode's
// statistics (colour cut-off +inf, indexed records and slot table). indexed: S.edge and S.attr are the indexed records.
int launch_foam_tile(const FoamScene& S, const FoamParams& P, const FoamRays& R, const FoamOut& O, bool indexed, bool exact,
                     bool half, hipStream_t stream);

namespace {

// Running normalised colour blend (fused / baked modes).
struct Blend {
    float m, a, r, g, b;
};

__device__ __forceinline__ void blend_init(Blend& B) { B.m = kInf, B.a = B.r = B.g = B.b = 0.f; }

// k precedes j in the tie-breaking order: the smaller original index.
__device__ __forceinline__ bool before(const FoamScene& S, int k, int j) {
    return S.orig != nullptr ? S.orig[k] < S.orig[j] : k < j;
}

// (r2, lam) half2 packed in the 4th component of an edge record.
__device__ __forceinline__ float2 cutoffs(float w) {
    const uint32_t u = __float_as_uint(w);
    const _Float16 lo = __builtin_bit_cast(_Float16, static_cast<uint16_t>(u & 0xffffu));
    const _Float16 hi = __builtin_bit_cast(_Float16, static_cast<uint16_t>(u >> 16));
    return make_float2(static_cast<float>(lo), static_cast<float>(hi));
}

// ------------------------------------------------------------------ field arithmetic (explicit FMA)
// The density, colour and blend arithmetic below fuses chosen products and sums into one FMA (fmaf), which rounds
// once where the CPU oracle rounds twice: each term moves by at most an ulp of its magnitude, and the colours and
// transmittances by a few ulps of 1 (about 1e-6), well inside the 1e-4 parity bar. The fusions are written out, not
// left to the compiler's contraction, so every kernel of this file that composes these terms rounds them the same
// way whatever the surrounding code and register schedule. The traversal arithmetic (walk distances, exit planes)
// is never fused, so the visited cells stay bit-exact.

__device__ __forceinline__ void blend_add(Blend& B, float m, float r, float g, float b) {
    if (m < B.m) {
        const float s = fexp(-0.5f * (B.m - m));
        B.a *= s, B.r *= s, B.g *= s, B.b *= s, B.m = m;
    }
    const float w = fexp(-0.5f * (m - B.m));
    B.a += w, B.r = fmaf(w, r, B.r), B.g = fmaf(w, g, B.g), B.b = fmaf(w, b, B.b);
}

// (vx, vy, vz) A (vx, vy, vz)^T for the symmetric conic A = (p.x p.y p.z / . p.w q.x / . . q.y)
__device__ __forceinline__ float maha_f(const float4& p, const float4& q, float vx, float vy, float vz) {
    const float diag = fmaf(p.x * vx, vx, fmaf(p.w * vy, vy, q.y * vz * vz));
    const float cross = fmaf(p.y * vx, vy, fmaf(p.z * vx, vz, q.x * vy * vz));
    return fmaf(2.f, cross, diag);
}

// Sample point o + t d, used by the field terms only (the traversal never reads it).
__device__ __forceinline__ void sample_point(const float (&o)[3], const float (&d)[3], float t, float (&x)[3]) {
    x[0] = fmaf(t, d[0], o[0]), x[1] = fmaf(t, d[1], o[1]), x[2] = fmaf(t, d[2], o[2]);
}

__device__ __forceinline__ void offset_of(const float (&x)[3], const float4& p, float& v0, float& v1, float& v2,
                                          float& r2) {
    v0 = x[0] - p.x, v1 = x[1] - p.y, v2 = x[2] - p.z;
    r2 = fmaf(v0, v0, fmaf(v1, v1, v2 * v2));
}

// rho_k G_k(x) from the density record (q0 = xx xy xz yy, q1 = yz zz min(raw, 30) 0).
__device__ __forceinline__ float density_term(const float4& q0, const float4& q1, float v0, float v1, float v2) {
    return fexp(fmaf(-0.5f, maha_f(q0, q1, v0, v1, v2), q1.z));
}

__device__ __forceinline__ float weight_of(float m, float mmin) { return fexp(-0.5f * (m - mmin)); }

__device__ __forceinline__ void accumulate(float& A, float& r, float& g, float& bl, float w, const float (&c)[3]) {
    A += w, r = fmaf(w, c[0], r), g = fmaf(w, c[1], g), bl = fmaf(w, c[2], bl);
}

// Adds blocks q0 .. q0 + 3 (those below nv) of a site's SH coefficients (fp32, or fp16 pairs) to c: the colour
// SH_k(d) accumulates over the coefficients in storage order, coefficient i of channel i mod 3 times basis i / 3.
template <bool HALF, int CH = 4>
__device__ __forceinline__ void sh_accumulate(const float4 (&f)[CH], int q0, int nv, const float (&b)[16],
                                              float (&c)[3]) {
#pragma unroll
    for (int uq = 0; uq < CH; ++uq) {
        const int q = q0 + uq;
        if (q >= nv) break;
        const float fv[4] = {f[uq].x, f[uq].y, f[uq].z, f[uq].w};
        if (HALF) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float2 p = cutoffs(fv[u]);
                const int i0 = 8 * q + 2 * u, i1 = i0 + 1;
                c[i0 % 3] = fmaf(b[i0 / 3], p.x, c[i0 % 3]);
                c[i1 % 3] = fmaf(b[i1 / 3], p.y, c[i1 % 3]);
            }
        } else {
#pragma unroll
            for (int u = 0; u < 4; ++u) c[(4 * q + u) % 3] = fmaf(b[(4 * q + u) / 3], fv[u], c[(4 * q + u) % 3]);
        }
    }
}

// Entry e of a neighbourhood [e0, e1) for a load issued ahead of the loop that may not run: clamped into the cell,
// and for an empty cell (no self entry, which no pack_foam pack has) to the entry before it, so the load stays in
// bounds whatever the offsets.
__device__ __forceinline__ int entry_in(int e, int e1) { return max(min(e, e1 - 1), 0); }

// Number of float4 a colour fetch reads: the blocks holding coefficients of degree <= DEG (the others multiply a
// zero basis value, so leaving them out changes no finite colour).
template <bool HALF, int DEG>
constexpr int sh_vec4() {
    return HALF ? sh_vec4_f16(DEG) : sh_vec4_f32(DEG);
}

template <bool TRACE>
__device__ __forceinline__ void trace_cell(const FoamScene& S, const FoamOut& O, int64_t r, int s, int c) {
    if (TRACE && s < O.trace_cap) O.trace[r * O.trace_cap + s] = S.orig != nullptr ? S.orig[c] : c;
}

__device__ __forceinline__ bool wave_any(bool p) { return __builtin_amdgcn_ballot_w64(p) != 0; }

// k precedes j in the tie order, INT_MAX (no face) after every site.
__device__ __noinline__ bool before_or_none(const FoamScene& S, int k, int j) {
    if (j == INT_MAX) return k != INT_MAX;
    if (k == INT_MAX) return false;
    return before(S, k, j);
}

// Keeps the lexicographic minimum of (t, k) and the candidate (u, j). Exact ties in t are rare: they take a
// wave-uniform branch, inside which only the tied lanes look up the tie order.
__device__ __forceinline__ void keep_min(const FoamScene& S, float u, int j, float& t, int& k) {
    bool take = u < t;
    const bool tie = u == t && j != k;
    if (wave_any(tie)) {
        if (tie) take = before_or_none(S, j, k);
    }
    if (take) t = u, k = j;
}

template <int CTRL>
__device__ __forceinline__ void min_step(const FoamScene& S, float& t, int& k) {
    const float u = row_perm<CTRL>(t);
    const int j = row_perm<CTRL>(k);
    keep_min(S, u, j, t, k);
}

}  // namespace
}  // namespace vgr
