// Inference renderer with 16 lanes per ray, gfx950: the layout for batches too small to fill the GPU.
//
// Same function as foam_infer.hip's kernels in stage 2 (csrc/foam_infer.cu:286-361). A ray is a chain of cells, each
// known only once the cell before has been read, so a launch of few waves lasts as long as its longest chain and its
// time is the latency of one cell times the cells of a ray. One ray per lane reads a cell's neighbourhood (mean 16.5
// entries) entry by entry, about 16 dependent rounds; here a group of 16 lanes (one DPP row, 4 rays per wave) reads it
// in one or two: two dependent reads per cell (its edge records; its neighbours' site records and CSR offsets, which the
// exit's lane hands on to the next cell) and, where the segment is coloured, a third (SH rows).
//
// What the batch size decides and what does not:
// - the cells visited are those of every other layout: the exit is the lexicographic minimum of (t, tie order);
// - density is summed in neighbourhood order (row_newbcast: every lane adds lane 0's term, then lane 1's, ...), so
//   sigma, alpha and T have the bits of the one-ray-per-lane kernels;
// - colours are evaluated for the samples of segments heavier than w_thresh only, in fused and baked mode too: only
//   those reach the image. The blend's weights are relative to the smallest Mahalanobis distance of the neighbourhood,
//   where the sequential blend rescales to its running minimum: the same sums to rounding;
// - a finite colour cut-off of fused and baked colours compares with the minimum of the entries before in neighbourhood
//   order, as the sequential blend does: an exclusive prefix minimum over the row. (An entry the blend skips never lowers
//   its running minimum.)
// - the reference's cache misses (stats[:, 4]): lane s < 8 of the group holds the ray's tag of slot s; the first and the
//   last lookup of a slot in a round come from ballots of the low bits of the sites (colour_tags).
//
// Bound: the chain of cells for a few thousand rays, then the vector-memory path (every lane of a wave reads its own site:
// 16 loads of 16 bytes per entry of a coloured sample). 8192 rays in rows of pixels over 131k sites, exact colours, fp32 SH
// (2 waves per SIMD, 0.40 ms of GPU time): the texture data path is busy 78 % of it, waves wait 46 % of their cycles, the
// VALU issues 44 % of the time, the L2 hits 97.5 % and DRAM moves 55 MB. The rule at kWideRays (foam_infer.hip) holds the
// comparison with the other layouts.
#include <cmath>

#include "vgr_foam.h"

namespace vgr {
namespace {

constexpr int kBlock = 64;       // one wave, 4 rays
constexpr int kRayTagSlots = 8;  // the reference's per-ray colour cache

constexpr int kLanes = 16;       // lanes per ray: one DPP row
constexpr int kSlots = 2;        // entries of a neighbourhood that a lane holds at once (longer ones loop)

// The group's first lane in the wave, and its lanes' bits of a ballot.
__device__ __forceinline__ int group_base() { return static_cast<int>(threadIdx.x) & (64 - kLanes); }

__device__ __forceinline__ unsigned group_bits(uint64_t ballot) {
    return static_cast<unsigned>(ballot >> group_base()) & ((1u << kLanes) - 1);
}

// Value of the row's lane J in every lane of the row (row_newbcast).
template <int J>
__device__ __forceinline__ float row_bcast(float v) {
    return row_perm<0x150 | J>(v);
}

// Lane g gets lane g - N's value, kInf where there is none (row_shr).
template <int N>
__device__ __forceinline__ float row_shr(float v) {
    return __int_as_float(
        __builtin_amdgcn_update_dpp(__float_as_int(kInf), __float_as_int(v), 0x110 | N, 0xF, 0xF, false));
}

// sum + v of lane 0 + v of lane 1 + ..., in that order, in every lane of the row.
__device__ __forceinline__ float ordered_sum(float sum, float v) {
    sum += row_bcast<0>(v), sum += row_bcast<1>(v), sum += row_bcast<2>(v), sum += row_bcast<3>(v);
    sum += row_bcast<4>(v), sum += row_bcast<5>(v), sum += row_bcast<6>(v), sum += row_bcast<7>(v);
    sum += row_bcast<8>(v), sum += row_bcast<9>(v), sum += row_bcast<10>(v), sum += row_bcast<11>(v);
    sum += row_bcast<12>(v), sum += row_bcast<13>(v), sum += row_bcast<14>(v), sum += row_bcast<15>(v);
    return sum;
}

template <typename V>
__device__ __forceinline__ V row_sum(V v) {
    v = v + row_perm<kXor1>(v);
    v = v + row_perm<kXor2>(v);
    v = v + row_perm<kHalfMirror>(v);
    return v + row_perm<kMirror>(v);
}

__device__ __forceinline__ float row_min(float v) {
    v = fminf(v, row_perm<kXor1>(v));
    v = fminf(v, row_perm<kXor2>(v));
    v = fminf(v, row_perm<kHalfMirror>(v));
    return fminf(v, row_perm<kMirror>(v));
}

__device__ __forceinline__ void row_exit(const FoamScene& S, float& t, int& k) {
    min_step<kXor1>(S, t, k);
    min_step<kXor2>(S, t, k);
    min_step<kHalfMirror>(S, t, k);
    min_step<kMirror>(S, t, k);
}

__device__ __forceinline__ const float4* record(const FoamScene& S, int k) { return S.attr + 5 * static_cast<int64_t>(k); }

// One entry of a neighbourhood: its edge record and site, and whether the lane has one.
struct Entry {
    float4 ed;
    int k;
    bool on;
};

__device__ __forceinline__ Entry entry_at(const FoamScene& S, int e, int e1) {
    Entry E;
    E.on = e < e1;
    E.ed = make_float4(0.f, 0.f, 0.f, 0.f), E.k = 0;
    if (E.on) E.ed = S.edge[e], E.k = S.nbr[e];
    return E;
}

// The reference's colour-cache lookups of one round, in neighbourhood order (lane 0, 1, ...): lane s < 8 returns 1 if
// the first lookup of slot s (k & 7) in the round is the site its tag holds, and then holds the last. The sites of a
// round are distinct, so no other lookup of the slot can hit. All lanes of the group take part.
__device__ __forceinline__ int colour_tags(bool look, int k, int g, int& tag) {
    const int row = group_base();
    const unsigned all = group_bits(__ballot(look)), b0 = group_bits(__ballot(k & 1)),
                   b1 = group_bits(__ballot(k & 2)), b2 = group_bits(__ballot(k & 4));
    const unsigned mine = all & (g & 1 ? b0 : ~b0) & (g & 2 ? b1 : ~b1) & (g & 4 ? b2 : ~b2);
    const int first = mine ? __ffs(mine) - 1 : g, last = mine ? 31 - __clz(mine) : g;
    const int kf = __shfl(k, row + first), kl = __shfl(k, row + last);
    if (g >= kRayTagSlots || mine == 0) return 0;
    const int hit = kf == tag ? 1 : 0;
    tag = kl;
    return hit;
}

// A sample's cell and the group's view of its neighbourhood: the lane's entries, their colour Mahalanobis distances and
// whether the colour cut-off keeps them (decided in the pass for fused and baked colours, in the colour pass for exact).
struct Sample {
    int c, e0, e1;
    float t, sigma;
    int k[kSlots];
    float m[kSlots], lb[kSlots];
    bool on[kSlots];
};

// Exclusive prefix minimum of m over the neighbourhood order; `carry` is the minimum of the rounds before.
__device__ __forceinline__ float min_before(float m, float& carry) {
    float v = m;
    v = fminf(v, row_shr<1>(v));
    v = fminf(v, row_shr<2>(v));
    v = fminf(v, row_shr<4>(v));
    v = fminf(v, row_shr<8>(v));
    const float before = fminf(row_shr<1>(v), carry);
    carry = fminf(carry, row_bcast<15>(v));
    return before;
}

// The pass over the neighbourhood of sample Q (c, e0, e1, t set): density, the entries' colour distances, and, when
// want_exit, the exit face with the next cell's CSR range. COUNT: the lookups of a fused colour pass, which counts at
// every sample.
template <bool COUNT, bool EXACT, bool CUT>
__device__ __forceinline__ void pass(const FoamScene& S, const FoamParams& P, int g, const float (&o)[3],
                                     const float (&d)[3], bool want_exit, Sample& Q, float& t_exit, int& next, int& f0,
                                     int& f1, int& n_dens, int& n_sh, int& tag) {
    Entry E[kSlots];
#pragma unroll
    for (int s = 0; s < kSlots; ++s) E[s] = entry_at(S, Q.e0 + g + kLanes * s, Q.e1);
    float x[3];
    sample_point(o, d, Q.t, x);
    // the cell's own entry comes first and holds its position
    const float p0 = row_bcast<0>(E[0].ed.x), p1 = row_bcast<0>(E[0].ed.y), p2 = row_bcast<0>(E[0].ed.z);
    float best = kInf, sigma = 0.f, carry = kInf;
    int bk = INT_MAX, of0[kSlots] = {}, of1[kSlots] = {};
    const auto visit = [&](const Entry& N, bool self, float& m, float& lb, int& a, int& b) {
        float4 q0, q1, q2, q3;
        m = kInf, lb = kInf;
        float term = 0.f;
        if (N.on) {
            const float4* r = record(S, N.k);
            q0 = r[0], q1 = r[1], q2 = r[2], q3 = r[3];
            a = S.offsets[N.k], b = S.offsets[N.k + 1];
            if (want_exit && !self) {
                const float n0 = N.ed.x - p0, n1 = N.ed.y - p1, n2 = N.ed.z - p2;
                const float dn = n0 * d[0] + n1 * d[1] + n2 * d[2];
                if (dn > 0.f) {
                    const float m0 = 0.5f * (N.ed.x + p0) - o[0], m1 = 0.5f * (N.ed.y + p1) - o[1],
                                m2 = 0.5f * (N.ed.z + p2) - o[2];
                    keep_min(S, (m0 * n0 + m1 * n1 + m2 * n2) / dn, N.k, best, bk);
                }
            }
            float v0, v1, v2, r2;
            offset_of(x, N.ed, v0, v1, v2, r2);
            const float2 cut = cutoffs(N.ed.w);
            if (r2 <= cut.x) {
                term = density_term(q0, q1, v0, v1, v2);
                ++n_dens;
            }
            m = maha_f(q2, q3, v0, v1, v2), lb = r2 * cut.y;
        }
        sigma = ordered_sum(sigma, term);
    };
    const auto look_up = [&](bool on, int k, float m, float lb) {
        if (EXACT) return on;
        const float lim = CUT ? min_before(m, carry) + P.color_cut : P.color_cut;  // +inf: all but NaN
        const bool look = on && lb <= lim && m <= lim;
        if (COUNT) n_sh += (look ? 1 : 0) - colour_tags(look, k, g, tag);
        return look;
    };
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
        Q.k[s] = E[s].k, Q.on[s] = false, Q.m[s] = Q.lb[s] = kInf;
        if (s == 0 || wave_any(E[s].on)) {
            visit(E[s], s == 0 && g == 0, Q.m[s], Q.lb[s], of0[s], of1[s]);
            Q.on[s] = look_up(E[s].on, E[s].k, Q.m[s], Q.lb[s]);
        }
    }
    for (int e = Q.e0 + kLanes * kSlots; e < Q.e1; e += kLanes) {
        const Entry N = entry_at(S, e + g, Q.e1);
        float m, lb;
        int a, b;
        visit(N, false, m, lb, a, b);
        look_up(N.on, N.k, m, lb);
    }
    Q.sigma = sigma;
    if (want_exit) {
        row_exit(S, best, bk);
        // the CSR range of the next cell, from the lane that holds it (a neighbour beyond the slots is read again)
        bool have = false;
        int a = 0, b = 0;
#pragma unroll
        for (int s = 0; s < kSlots; ++s)
            if (E[s].on && E[s].k == bk) have = true, a = of0[s], b = of1[s];
        const unsigned who = group_bits(__ballot(have));
        const int from = group_base() + (who ? __ffs(who) - 1 : 0);
        f0 = __shfl(a, from), f1 = __shfl(b, from);
        if (who == 0 && bk != INT_MAX) f0 = S.offsets[bk], f1 = S.offsets[bk + 1];
    }
    t_exit = best, next = bk;
}

// max(SH_k(d) + 1/2, 0), or the baked colour of site k.
template <bool BAKED, bool HALF, int DEG>
__device__ __forceinline__ void site_colour(const FoamScene& S, int k, const float (&b)[16], float (&c)[3]) {
    if (BAKED) {
        const float4 q = S.attr[5 * static_cast<int64_t>(k) + 4];
        c[0] = q.x, c[1] = q.y, c[2] = q.z;
    } else {
        constexpr int NV = sh_vec4<HALF, DEG>();
        const float4* row = S.sh + S.sh_stride * static_cast<int64_t>(k);
        float4 f[NV];
#pragma unroll
        for (int q = 0; q < NV; ++q) f[q] = row[q];
        c[0] = c[1] = c[2] = 0.5f;
        sh_accumulate<HALF, NV>(f, 0, NV, b, c);
        c[0] = fmaxf(c[0], 0.f), c[1] = fmaxf(c[1], 0.f), c[2] = fmaxf(c[2], 0.f);
    }
}

// Colour of sample Q. REUSE: the pass over Q's cell left the lane's entries in Q; else they are read again.
// EXACT: the exact mode's cut-off (against the smallest distance of all entries) and its count of lookups.
template <bool REUSE, bool EXACT, bool BAKED, bool HALF, int DEG, bool CUT>
__device__ __forceinline__ void colour(const FoamScene& S, const FoamParams& P, int g, const float (&o)[3],
                                       const float (&d)[3], const float (&b)[16], Sample& Q, float (&C)[3], int& n_sh,
                                       int& tag) {
    float x[3];
    sample_point(o, d, Q.t, x);
    const auto distance = [&](const Entry& N, float& m, float& lb) {
        m = lb = kInf;
        if (N.on) {
            const float4* r = record(S, N.k);
            const float4 q2 = r[2], q3 = r[3];
            float v0, v1, v2, r2;
            offset_of(x, N.ed, v0, v1, v2, r2);
            m = maha_f(q2, q3, v0, v1, v2), lb = r2 * cutoffs(N.ed.w).y;
        }
    };
    float carry = kInf;
    const auto kept = [&](bool on, float m, float lb) {  // fused and baked colours' cut-off
        if (EXACT) return on;
        const float lim = CUT ? min_before(m, carry) + P.color_cut : P.color_cut;
        return on && lb <= lim && m <= lim;
    };
    if (!REUSE) {
        Entry E[kSlots];
#pragma unroll
        for (int s = 0; s < kSlots; ++s) E[s] = entry_at(S, Q.e0 + g + kLanes * s, Q.e1);
#pragma unroll
        for (int s = 0; s < kSlots; ++s) {
            distance(E[s], Q.m[s], Q.lb[s]);
            Q.k[s] = E[s].k, Q.on[s] = kept(E[s].on, Q.m[s], Q.lb[s]);
        }
    } else if (CUT && !EXACT) {  // the prefix minimum after the slots
#pragma unroll
        for (int s = 0; s < kSlots; ++s) carry = fminf(carry, Q.m[s]);
        carry = row_min(carry);
    }
    float mmin = kInf;
#pragma unroll
    for (int s = 0; s < kSlots; ++s) mmin = fminf(mmin, Q.m[s]);
    for (int e = Q.e0 + kLanes * kSlots; e < Q.e1; e += kLanes) {
        float m, lb;
        distance(entry_at(S, e + g, Q.e1), m, lb);
        mmin = fminf(mmin, m);
    }
    mmin = row_min(mmin);
    float A = 0.f, cr = 0.f, cg = 0.f, cb = 0.f;
    const auto add = [&](bool on, int k, float m, float lb) {
        const bool look = on && (!EXACT || (lb <= mmin + P.color_cut && m <= mmin + P.color_cut));
        if (EXACT) n_sh += (look ? 1 : 0) - colour_tags(look, k, g, tag);
        if (look) {
            float c[3];
            site_colour<BAKED, HALF, DEG>(S, k, b, c);
            accumulate(A, cr, cg, cb, weight_of(m, mmin), c);
        }
    };
#pragma unroll
    for (int s = 0; s < kSlots; ++s)
        if (s == 0 || wave_any(Q.on[s])) add(Q.on[s], Q.k[s], Q.m[s], Q.lb[s]);
    for (int e = Q.e0 + kLanes * kSlots; e < Q.e1; e += kLanes) {
        const Entry N = entry_at(S, e + g, Q.e1);
        float m, lb;
        distance(N, m, lb);
        add(kept(N.on, m, lb), N.k, m, lb);
    }
    const float inv = 1.f / row_sum(A);
    C[0] = row_sum(cr) * inv, C[1] = row_sum(cg) * inv, C[2] = row_sum(cb) * inv;
}

// Greedy walk to the lexicographic argmin of (|x - p|^2, tie order) over {c} U adj(c), repeated.
__device__ __forceinline__ int walk(const FoamScene& S, int c, int g, float x0, float x1, float x2, int& steps) {
    for (int it = 0; it < kWalkCap; ++it) {
        const float4 pc = S.points[c];
        float bd = (x0 - pc.x) * (x0 - pc.x) + (x1 - pc.y) * (x1 - pc.y) + (x2 - pc.z) * (x2 - pc.z);
        int bk = c;
        const int e0 = S.offsets[c], e1 = S.offsets[c + 1];
        for (int e = e0 + 1 + g; e < e1; e += kLanes) {
            const float4 ed = S.edge[e];
            const int k = S.nbr[e];
            const float v0 = x0 - ed.x, v1 = x1 - ed.y, v2 = x2 - ed.z;
            keep_min(S, v0 * v0 + v1 * v1 + v2 * v2, k, bd, bk);
        }
        row_exit(S, bd, bk);
        if (bk == c) break;
        c = bk;
        ++steps;
    }
    return c;
}

template <int COLOR, bool HALF, int DEG, bool CUT>
__global__ void __launch_bounds__(kBlock) foam_wide_kernel(FoamScene S, FoamParams P, FoamRays R, FoamOut O) {
    constexpr bool EXACT = COLOR == kLazy, BAKED = COLOR == kBaked, COUNT = COLOR == kFused;
    const int g = static_cast<int>(threadIdx.x) % kLanes;
    const int64_t i = xcd_block_id() * (kBlock / kLanes) + threadIdx.x / kLanes;
    if (i >= R.n) return;  // whole groups leave together
    const int64_t r = R.order != nullptr ? R.order[i] : i;
    if (r < 0 || r >= R.n) return;
    const int start = R.start[r];
    if (start < 0 || start >= S.n_sites) {  // not traced: empty foreground
        if (g == 0) {
            O.rgb[3 * r] = O.rgb[3 * r + 1] = O.rgb[3 * r + 2] = 0.f;
            O.T[r] = 1.f, O.depth[r] = 0.f;
#pragma unroll
            for (int u = 0; u < 5; ++u) O.stats[5 * r + u] = 0;
        }
        return;
    }
    const float o[3] = {R.o[3 * r], R.o[3 * r + 1], R.o[3 * r + 2]};
    const float d[3] = {R.d[3 * r], R.d[3 * r + 1], R.d[3 * r + 2]};
    const float t_far = R.t_far[r];
    const int max_samples = R.cap != nullptr ? R.cap[r] : INT_MAX;
    const bool trace = O.trace != nullptr && g == 0;
    float b[16];
    if (!BAKED) sh_basis(d[0], d[1], d[2], DEG, b);

    int walk_steps = 0, n_dens = 0, n_sh = 0, tag = -1;
    Sample A, B;
    A.t = R.t_near[r];
    A.c = walk(S, start, g, o[0] + A.t * d[0], o[1] + A.t * d[1], o[2] + A.t * d[2], walk_steps);
    A.e0 = S.offsets[A.c], A.e1 = S.offsets[A.c + 1];
    float t_exit;
    int next, f0 = 0, f1 = 0;
    pass<COUNT, EXACT, CUT>(S, P, g, o, d, true, A, t_exit, next, f0, f1, n_dens, n_sh, tag);
    if (trace) trace_cell<true>(S, O, r, 0, A.c);
    float T = 1.f, acc[3] = {0.f, 0.f, 0.f}, dep = 0.f, CA[3] = {0.f, 0.f, 0.f};
    bool lit_before = false;
    int n_samples = 1, n_color = 0;
    for (int it = 0; it < kMaxCells; ++it) {
        const bool last = next == INT_MAX || t_exit >= t_far || n_samples + 1 >= max_samples;
        B.t = last ? t_far : fmaxf(t_exit, A.t);
        B.c = last ? A.c : next, B.e0 = last ? A.e0 : f0, B.e1 = last ? A.e1 : f1;
        pass<COUNT, EXACT, CUT>(S, P, g, o, d, !last, B, t_exit, next, f0, f1, n_dens, n_sh, tag);
        if (trace) trace_cell<true>(S, O, r, n_samples, B.c);
        ++n_samples;
        const float delta = B.t - A.t;
        const float alpha = 1.f - fexp(-0.5f * (A.sigma + B.sigma) * delta);
        const float w = T * alpha;
        const bool lit = w > P.w_thresh;
        float CB[3] = {0.f, 0.f, 0.f};
        if (lit) {
            if (!lit_before) colour<false, EXACT, BAKED, HALF, DEG, CUT>(S, P, g, o, d, b, A, CA, n_sh, tag);
            colour<true, EXACT, BAKED, HALF, DEG, CUT>(S, P, g, o, d, b, B, CB, n_sh, tag);
#pragma unroll
            for (int a = 0; a < 3; ++a) acc[a] += w * 0.5f * (CA[a] + CB[a]);
            dep += w * 0.5f * (A.t + B.t);
            ++n_color;
        }
        T *= 1.f - alpha;
        A.c = B.c, A.e0 = B.e0, A.e1 = B.e1, A.t = B.t, A.sigma = B.sigma, lit_before = lit;
#pragma unroll
        for (int a = 0; a < 3; ++a) CA[a] = CB[a];
        if (last || T < P.t_thresh) break;
    }
    n_dens = row_sum(n_dens), n_sh = row_sum(n_sh);
    if (g == 0) {
#pragma unroll
        for (int a = 0; a < 3; ++a) O.rgb[3 * r + a] = acc[a];
        O.T[r] = T;
        O.depth[r] = dep;
        int* st = O.stats + 5 * r;
        st[0] = n_samples, st[1] = n_color, st[2] = walk_steps, st[3] = n_dens, st[4] = n_sh;
    }
}

template <int COLOR, bool HALF, int DEG>
void launch(const FoamScene& S, const FoamParams& P, const FoamRays& R, const FoamOut& O, hipStream_t stream) {
    const dim3 grid(grid_for(R.n, kBlock / kLanes)), block(kBlock);
    if (std::isinf(P.color_cut) && P.color_cut > 0)
        hipLaunchKernelGGL((foam_wide_kernel<COLOR, HALF, DEG, false>), grid, block, 0, stream, S, P, R, O);
    else
        hipLaunchKernelGGL((foam_wide_kernel<COLOR, HALF, DEG, true>), grid, block, 0, stream, S, P, R, O);
}

template <int COLOR, bool HALF>
void launch_deg(const FoamScene& S, const FoamParams& P, const FoamRays& R, const FoamOut& O, hipStream_t stream) {
    switch (P.sh_deg) {
        case 0: launch<COLOR, HALF, 0>(S, P, R, O, stream); break;
        case 1: launch<COLOR, HALF, 1>(S, P, R, O, stream); break;
        case 2: launch<COLOR, HALF, 2>(S, P, R, O, stream); break;
        default: launch<COLOR, HALF, 3>(S, P, R, O, stream);
    }
}

}  // namespace

int launch_foam_wide(const FoamScene& S, const FoamParams& P, const FoamRays& R, const FoamOut& O, int color_mode,
                     bool half, hipStream_t stream) {
    if (color_mode == kBaked)
        launch<kBaked, false, 0>(S, P, R, O, stream);
    else if (color_mode == kLazy)
        half ? launch_deg<kLazy, true>(S, P, R, O, stream) : launch_deg<kLazy, false>(S, P, R, O, stream);
    else
        half ? launch_deg<kFused, true>(S, P, R, O, stream) : launch_deg<kFused, false>(S, P, R, O, stream);
    return launch_status("foam_wide_kernel");
}

}  // namespace vgr
