// What the mixed form's symmetry-function, force and tangent kernels share:
// an atom's staging in LDS, the angular pair walks, and the choice of the
// kernel instance for a model and system.
#pragma once

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "mixed.hpp"
#include "nnpx.h"
#include "stage.hpp"

namespace nnpx {
namespace {

// Cutoff function in FP32, branch-light.  CT_COS uses the hardware sine and
// cosine on x in [0, 1] (arguments in revolutions) and sin(pi x) for the
// derivative (the reference's sqrt(1 - cos^2) form cancels in single
// precision).
// COS: the model's cutoff is the cosine one (without the others' code the
// walks need 15 to 20 registers less).
template <bool COS>
__device__ inline void cutoff32(int type, float rc, float rci, float iw, float rcinv, float tanhPre,
                                float r, float& fc, float& dfc)
{
    if (COS || type == 1) {
        const float x = fminf(fmaxf((r - rci) * iw, 0.f), 1.f);
        const float c = __builtin_amdgcn_cosf(0.5f * x);
        const float s = __builtin_amdgcn_sinf(0.5f * x);
        const bool in = r < rc;
        fc = in ? 0.5f * (c + 1.f) : 0.f;
        dfc = in ? -0.5f * iw * (float)M_PI * s : 0.f;
        return;
    }
    if (r >= rc) { fc = 0.f; dfc = 0.f; return; }
    if (type == 2 || type == 3) {
        const float t = tanhf(1.f - r * rcinv);
        const float t2 = t * t;
        const float pre = type == 3 ? tanhPre : 1.f;
        fc = pre * t * t2;
        dfc = 3.f * pre * t2 * (t2 - 1.f) * rcinv;
        return;
    }
    if (type == 0) { fc = 1.f; dfc = 0.f; return; }
    if (r < rci) { fc = 1.f; dfc = 0.f; return; }
    const float x = (r - rci) * iw;
    if (type == 4) {
        const float t = 1.f / (x * x - 1.f);
        const float t2 = __expf(t);
        fc = (float)M_E * t2;
        dfc = -2.f * (float)M_E * x * t * t * t2;
    } else if (type == 5) {
        fc = (2.f * x - 3.f) * x * x + 1.f;
        dfc = x * (6.f * x - 6.f);
    } else if (type == 6) {
        const float x2 = x * x;
        fc = ((15.f - 6.f * x) * x - 10.f) * x * x2 + 1.f;
        dfc = x2 * ((60.f - 30.f * x) * x - 30.f);
    } else if (type == 7) {
        const float x2 = x * x;
        fc = (x * (x * (20.f * x - 70.f) + 84.f) - 35.f) * x2 * x2 + 1.f;
        dfc = x2 * x * (x * (x * (140.f * x - 420.f) + 420.f) - 140.f);
    } else {
        float x4 = x * x;
        x4 *= x4;
        fc = (x * (x * ((315.f - 70.f * x) * x - 540.f) + 420.f) - 126.f) * x * x4 + 1.f;
        dfc = x4 * (x * (x * ((2520.f - 630.f * x) * x - 3780.f) + 2520.f) - 630.f);
    }
    // The polynomials vanish at x = 1; in FP32 they can round to tiny
    // negative values just below it, which the log2 form of the angular
    // terms must not see.
    fc = fmaxf(fc, 0.f);
    dfc *= iw;
}

struct GroupF {
    float rc, rc2, rci, iw, rcinv;
};

__device__ inline GroupF group_f(const GroupT& g)
{
    return GroupF{(float)g.rc, (float)g.rc2, (float)g.rci, (float)g.iw, (float)g.rcinv};
}

constexpr int kRadChunk = 8;  // radial members accumulated per pass
constexpr int kRadBatch = 32;  // radial sums scaled per batch (fits the smallest triplet buffer)

// LDS staging of one atom's neighbours (FP32 geometry) and the compacted
// triplet buffer.
struct Stage {
    float4* g;       // x, y, z, |dr|
    float4* c;       // 1/|dr|, fc, dfc (cutoff of the current group), unused
    unsigned char* el;  // neighbour element
    unsigned short* la; unsigned short* lb;  // group lists
    unsigned* tjk;   // this wave's [trip + kWave] compacted pairs (j | k << 16)
                     // and up to a wave's worth past them; r_jk^2 is
                     // recomputed from g
    unsigned* tj0;   // the first wave's (each wave's sums pass through its own)
    float4* mp;      // [mpn] per-group constants (member constants or power-path terms)
    int* eoff;       // [kMaxElem + 1] first staged slot of each neighbour element
    int trip;        // capacity of the triplet buffer
};

// A group's neighbour list: the staged slots base .. base + n - 1 (contig:
// every staged neighbour of the element lies inside the group's cutoff) or
// the n slots listed in S.la / S.lb.
struct List {
    int base, n;
    bool contig;
};

// A wave-uniform value held in a scalar register (values read from LDS or
// shuffled are uniform but not known to be by the compiler).
__device__ inline int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }

// Slot of list entry a (CONTIG: base + a, else l[a]).
template <bool CONTIG>
__device__ inline int slot(const unsigned short* l, int base, int a)
{
    if constexpr (CONTIG) return base + a;
    else return l[a];
}


template <int W>
__device__ inline Stage carve(float* base, int capL, int trip, int mpn)
{
    Stage S;
    S.trip = trip;
    S.g = reinterpret_cast<float4*>(base);
    S.c = S.g + capL;
    S.tj0 = reinterpret_cast<unsigned*>(S.c + capL);
    S.tjk = S.tj0 + wave_id() * (trip + kWave);
    S.mp = reinterpret_cast<float4*>(S.tj0 + W * (trip + kWave));
    S.la = reinterpret_cast<unsigned short*>(S.mp + mpn);
    S.lb = S.la + capL;
    S.el = reinterpret_cast<unsigned char*>(S.lb + capL);
    S.eoff = reinterpret_cast<int*>(S.el + capL);
    return S;
}

// |b - a|^2 of two staged positions, one fixed operation order for the
// candidate test and the terms
__device__ inline float dist2(const float4& a, const float4& b)
{
    const float dx = b.x - a.x, dy = b.y - a.y, dz = b.z - a.z;
    return fmaf(dz, dz, fmaf(dy, dy, dx * dx));
}

// Stages the atom's in-cutoff list entries (stage_by_element).  idx, when
// given, receives each staged slot's list entry; keep, when given, a copy of
// the staging for the force kernel.
template <int W>
__device__ inline int stage_atom(const ModelT* __restrict__ M, const SysView& s, int i, int capL, const Stage& S,
                                 unsigned short* idx = nullptr, const StageKeep* keep = nullptr)
{
    const size_t base = (size_t)i * s.cap;
    // the counts use the pair buffers, free until the first walk
    const int n = stage_by_element<W>(
        M, s, i, capL, reinterpret_cast<int*>(S.tj0), S.eoff, [&](int pos, int k, const double* dr, double d, int el) {
            const float4 g = make_float4((float)dr[0], (float)dr[1], (float)dr[2], (float)d);
            const float id = (float)(1.0 / d);
            S.g[pos] = g;
            // .w: the neighbour's atomic number, the weight of types 12 and 13
            S.c[pos] = make_float4(id, 0.f, 0.f, (float)M->Zel[el]);
            S.el[pos] = (unsigned char)el;
            if (idx) idx[pos] = (unsigned short)k;
            if (keep) {
                const size_t q = (size_t)i * keep->ld + pos;
                keep->g[q] = g;
                keep->rinv[q] = id;
                keep->nbr[q] = s.nb_j[base + k];
                keep->el[q] = (unsigned char)el;
            }
        });
    if (keep && threadIdx.x <= M->nelem) keep->off[(size_t)i * (kMaxElem + 1) + threadIdx.x] = S.eoff[threadIdx.x];
    return n;
}

// The staging of atom i as the SF kernel kept it (same slots, same values
// as stage_atom gives); returns the slot count.
template <int W>
__device__ inline int load_stage(const ModelT* __restrict__ M, const StageKeep& K, int i, const Stage& S)
{
    const int tid = threadIdx.x;
    const int ne = M->nelem;
    const int* off = K.off + (size_t)i * (kMaxElem + 1);
    if (tid <= ne) S.eoff[tid] = off[tid];
    const int n = uni(off[ne]);
    const size_t b = (size_t)i * K.ld;
    for (int k = tid; k < n; k += W * kWave) {
        const int el = K.el[b + k];
        S.g[k] = K.g[b + k];
        S.c[k] = make_float4(K.rinv[b + k], 0.f, 0.f, (float)M->Zel[el]);
        S.el[k] = (unsigned char)el;
    }
    __syncthreads();
    return n;
}

// Neighbours of element `elem` (all elements: elem < 0) inside the group's
// cutoff rc.  full: rc is the model's largest cutoff, so every staged
// neighbour of the element qualifies and the list is its slot range;
// otherwise the qualifying slots are listed in `out`.  Ends with a barrier.
template <int W>
__device__ inline List make_list(const Stage& S, int n, int elem, float rc, bool full, unsigned short* out)
{
    const int lane = lane_id();
    const int lo = uni(elem < 0 ? 0 : S.eoff[elem]), hi = uni(elem < 0 ? n : S.eoff[elem + 1]);
    List L{lo, hi - lo, true};
    if (!full) {
        // every wave counts, the first one writes
        int cnt = 0;
        for (int b = lo; b < hi; b += kWave) {
            const int k = b + lane;
            const unsigned long long m = __ballot(k < hi && S.g[k].w < rc);
            if (wave_id() == 0 && ((m >> lane) & 1))
                out[cnt + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                         __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u))] =
                    (unsigned short)k;
            cnt += __popcll(m);
        }
        L = List{0, uni(cnt), false};
    }
    __syncthreads();
    return L;
}

// Whether a group's cutoff covers every staged neighbour.
__device__ inline bool full_cutoff(const ModelT* __restrict__ M, const GroupT& G) { return G.rc >= M->maxCutoff; }

// Cutoff values of every staged neighbour for one radius (elements whose
// groups all share it compute them once per atom).
template <int W, bool COS>
__device__ inline void all_cutoffs(const Stage& S, int n, int ctype, const GroupF& g, float tanhPre)
{
    for (int k = threadIdx.x; k < n; k += W * kWave) {
        float f = 0.f, df = 0.f;
        cutoff32<COS>(ctype, g.rc, g.rci, g.iw, g.rcinv, tanhPre, S.g[k].w, f, df);
        S.c[k].y = f;
        S.c[k].z = df;
    }
    __syncthreads();
}

template <int W, bool COS>
__device__ inline void group_cutoffs(const Stage& S, int n, int e1, int e2, int ctype, const GroupF& g,
                                     float tanhPre)
{
    for (int k = threadIdx.x; k < n; k += W * kWave) {
        float f = 0.f, df = 0.f;
        if (e1 < 0 || S.el[k] == e1 || S.el[k] == e2)
            cutoff32<COS>(ctype, g.rc, g.rci, g.iw, g.rcinv, tanhPre, S.g[k].w, f, df);
        S.c[k].y = f;
        S.c[k].z = df;
    }
    __syncthreads();
}

__device__ inline float powi(float x, int n) { return pow_int<float>(x, n); }

// Compensated summation step (Fast2Sum error term accumulated in c; the
// terms are non-negative, so the running sum dominates after the first).
__device__ inline void kahan(float& s, float& c, float x)
{
    const float t = s + x;
    c += (s - t) + x;
    s = t;
}

// Value of a per-triplet table at a wave-uniform index.
template <int MAXS>
__device__ inline float pick(const float* v, int s)
{
    float r = v[0];
    if (MAXS > 1) r = s == 1 ? v[1] : r;
    if (MAXS > 2) r = s == 2 ? v[2] : r;
    if (MAXS > 3) r = s == 3 ? v[3] : r;
    return r;
}

template <int MAXS>
__device__ inline float pickb(const float* v, unsigned b1, unsigned b2)
{
    if (MAXS <= 2) return b1 ? v[1] : v[0];
    const float lo = b1 ? v[1] : v[0];
    const float hi = b1 ? v[3] : v[2];
    return b2 ? hi : lo;
}

// Member constants of one group: flags as wave-uniform bit masks, values
// staged in LDS (mp[q] = zeta, eta log2 e, rs; mp[32+q] = the force-pass
// weights w zeta lambda, w, 2 eta w), read as broadcasts in the triplet loops.
struct MemberMasks {
    unsigned calc, s1, s2;
};

__device__ inline MemberMasks load_members(const Stage& S, const MemberF* __restrict__ mf, int nmem,
                                           const float* w)
{
    const int lane = lane_id();
    if (threadIdx.x < nmem) {
        const MemberF m = mf[lane];
        const float wq = w ? w[m.sf] : 0.f;
        S.mp[lane] = make_float4(m.zeta, m.etaL, m.rs, (float)(m.sidx & 1));
        S.mp[kMaxMembersExp + lane] = make_float4(wq * m.zetaLambda, wq, wq * m.twoEta, (float)((m.sidx >> 1) & 1));
    }
    MemberMasks R;
    R.calc = (unsigned)__ballot(lane < nmem && mf[min(lane, nmem - 1)].calcExp);
    R.s1 = (unsigned)__ballot(lane < nmem && (mf[min(lane, nmem - 1)].sidx & 1));
    R.s2 = (unsigned)__ballot(lane < nmem && (mf[min(lane, nmem - 1)].sidx & 2));
    __syncthreads();
    return R;
}

__device__ inline float fexp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ inline float flog2(float x) { return __builtin_amdgcn_logf(x); }

// `flush` runs after each buffer of triplets (a few per lane), so callers can
// keep short FP32 partial sums and fold them into their long accumulators.
struct NoFlush {
    __device__ void operator()() const {}
};

// Runs `work` over the first cnt buffered pairs, each lane a contiguous
// chunk, so a lane sees runs of one first atom j (j's geometry stays in
// registers over the run and the force kernel keeps j's contribution there).
template <typename Work>
__device__ inline void run_buffer(const Stage& S, int cnt, Work&& work)
{
    const int per = (cnt + kWave - 1) / kWave;
    const int x0 = lane_id() * per, x1 = min(cnt, x0 + per);
    for (int x = x0; x < x1; ++x) work(S.tjk[x] & 0xffffu, S.tjk[x] >> 16);
}

// The angular walk: each row a of list A pairs with its columns c -- for one
// list b = (a + c + 1) mod nA with c < (nA - 1) / 2, and for even nA one
// more column (b = a + nA / 2) on the rows a < nA / 2, so every unordered
// pair appears once; for two lists b = c, c < nB.  A step tests a block of
// rows x columns (lane = row * width + column, fixed per group), so a
// candidate's indices cost a few adds, and the row's geometry stays in
// registers.  Passing pairs are compacted through LDS in block order; the
// pairs run in buffers of exactly S.trip (the last one shorter), the pairs
// a step adds past a full buffer being carried to the next, so the buffers
// depend only on the pair sequence.  `flush` runs after each buffer.
// GATHER: gB holds the partners' geometry in list order (gB[b] =
// S.g[lb[b]]), so a candidate's index and position load together.
// src: the walk's nsrc pairs as stored by an earlier walk (same sequence,
// same buffers), read instead of tested.  dst: the pairs are stored there
// too while they fit in `room` entries.  Returns the walk's pair count.
// Wave w of the block's W takes the row blocks w, w + W, ... (its own buffer,
// src and dst); the waves do not wait for each other.
template <int W, bool CONTIG, bool GATHER, typename Work, typename Flush = NoFlush>
__device__ inline int for_each_triplet_blocks(const Stage& S, const float4* gB, const List& A, const List& B,
                                              bool same, float rc2, const unsigned* src, int nsrc, unsigned* dst,
                                              int room, Work&& work, Flush&& flush = Flush{})
{
    const int lane = lane_id();
    const int nA = A.n, nB = B.n;
    const int R = same ? (nA - 1) / 2 : nB;          // regular columns per row
    const int Rx = same && nA % 2 == 0 ? R + 1 : R;  // with the half-way column (rows a < nA / 2 only)
    const int half = nA / 2;
    // a row's columns split into nearly equal blocks of at most 8: the
    // blocks fill the wave's lanes closely, and the passing partners of one
    // row still form runs in the buffer
    const int nblk = (Rx + 7) >> 3;
    const int cw = nblk > 0 ? (Rx + nblk - 1) / nblk : 1, rh = kWave / cw;
    const int lr = lane / cw, lc = lane - lr * cw;  // lanes with lr >= rh stay idle
    const bool live = lr < rh;
    const unsigned short* lb = same ? S.la : S.lb;
    const int bB = same ? A.base : B.base;
    // contiguous partners are already in list order
    const float4* gp = CONTIG ? S.g + bB : gB;
    // no candidates: the fill loop never runs
    int a0 = src || nA == 0 || Rx == 0 ? nA : wave_id() * rh, c0 = 0;
    // the lane's row atom and its geometry, reloaded when the block moves down
    int ja = slot<CONTIG>(S.la, A.base, a0 + lr < nA ? a0 + lr : 0);
    float4 ga = a0 < nA ? S.g[ja] : make_float4(0.f, 0.f, 0.f, 0.f);
    int cnt = 0, done = 0;  // pairs in the buffer, pairs run so far
    // stored pairs are loaded a buffer ahead (buffers of up to kAhead per
    // lane), so the loads overlap the previous buffer's work
    constexpr int kAhead = 6;
    unsigned ahead[kAhead];
    const bool pre = src && S.trip <= kAhead * kWave;
    auto load_ahead = [&](int from) {
        const int m = min(S.trip, nsrc - from);
#pragma unroll
        for (int q = 0; q < kAhead; ++q) {
            const int x = q * kWave + lane;
            ahead[q] = x < m ? src[from + x] : 0u;
        }
    };
    if (pre) load_ahead(0);
    for (;;) {
        if (src) {
            cnt = min(S.trip, nsrc - done);
            if (pre) {
#pragma unroll
                for (int q = 0; q < kAhead; ++q)
                    if (q * kWave + lane < cnt) S.tjk[q * kWave + lane] = ahead[q];
                if (done + cnt < nsrc) load_ahead(done + cnt);
            } else {
                for (int x = lane; x < cnt; x += kWave) S.tjk[x] = src[done + x];
            }
        } else {
            while (a0 < nA && cnt < S.trip) {
                // branch-free: lanes outside the block test column 0 and fail
                const int a = a0 + lr, c = c0 + lc;
                const bool valid = live && a < nA && c < Rx && (c < R || a < half);
                int b = same ? a + c + 1 : c;
                b = same && b >= nA ? b - nA : b;
                b = valid ? b : 0;
                const int k = slot<CONTIG>(lb, bB, b);
                const float d2 = dist2(ga, (GATHER || CONTIG) ? gp[b] : S.g[k]);  // in bounds for every lane
                const bool ok = valid & (d2 < rc2);
                const unsigned long long m = __ballot(ok);
                // passing pairs to the next entries (at most a wave past the buffer)
                if (ok)
                    S.tjk[cnt + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                               __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u))] =
                        (unsigned)ja | ((unsigned)k << 16);
                cnt += __popcll(m);
                c0 += cw;
                if (c0 >= Rx) {
                    c0 = 0;
                    a0 += W * rh;
                    const int an = a0 + lr;
                    ja = slot<CONTIG>(S.la, A.base, an < nA ? an : 0);
                    ga = S.g[ja];
                }
            }
        }
        const int m = min(cnt, S.trip);
        if (m <= 0) break;
        wave_fence();
        if (dst && done + m <= room)
            for (int x = lane; x < m; x += kWave) dst[done + x] = S.tjk[x];
        run_buffer(S, m, work);
        flush();
        done += m;
        wave_fence();
        // pairs past the buffer move to its front (disjoint ranges)
        const int rest = cnt - m;
        if (lane < rest) S.tjk[lane] = S.tjk[S.trip + lane];
        cnt = rest;
        wave_fence();
    }
    return done;
}

// Row-major walk (the force kernel without pair lists): candidates are
// enumerated a-major from a linear index (all partners of la[a]
// consecutively), compacted the same way, and each lane takes a contiguous
// chunk of the compacted buffer.  Its partner atoms k differ more across the
// lanes of one step than in the block walk, which keeps the force kernel's
// LDS atomics on k from colliding; the block walk, whose lists the SF kernel
// can keep, tests candidates more cheaply.  `flush` runs after each buffer.
// Wave w takes every W-th 64 candidates.
template <int W, bool CONTIG, typename Work, typename Flush = NoFlush>
__device__ inline void for_each_triplet_rows(const Stage& S, const List& A, const List& B, bool same, float rc2,
                                             Work&& work, Flush&& flush = Flush{})
{
    const int lane = lane_id();
    constexpr int kStep = W * kWave;
    const int nA = A.n, nB = B.n;
    int full, total, R;
    if (same) {
        R = (nA - 1) / 2;
        full = nA * R;
        total = full + ((nA % 2 == 0) ? nA / 2 : 0);
    } else {
        R = nB;
        full = nA * nB;
        total = full;
    }
    if (total == 0) return;
    const unsigned short* lb = same ? S.la : S.lb;
    const int bB = same ? A.base : B.base;
    // the lane's linear index t = q R + r, advanced by kStep = dq R + dr per
    // step (decoded once per buffer, so only t0 lives across the work)
    const int dq = R > 0 ? kStep / R : 0, dr = R > 0 ? kStep - dq * R : kStep;
    int t0 = wave_id() * kWave;
    while (t0 < total) {
        int cnt = 0;
        int t = t0 + lane, q = 0, r = t;
        if (R > 0) {
            q = t / R;
            r = t - q * R;
        }
        while (t0 < total && cnt <= S.trip - kWave) {
            // branch-free: rows q (t < full) or the half-way column of row
            // t - full; lanes past the end test slot 0 and fail
            const bool valid = t < total, tail = t >= full;
            int b = same ? q + r + 1 : r;
            b = same && b >= nA ? b - nA : b;
            const int a = valid ? (tail ? t - full : q) : 0;
            b = valid ? (tail ? a + (nA >> 1) : b) : 0;
            const int j = slot<CONTIG>(S.la, A.base, a), k = slot<CONTIG>(lb, bB, b);
            const float d2 = dist2(S.g[j], S.g[k]);  // in bounds for every lane
            const bool ok = valid & (d2 < rc2);
            const unsigned long long m = __ballot(ok);
            if (ok)
                S.tjk[cnt + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                           __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u))] =
                    (unsigned)j | ((unsigned)k << 16);
            cnt += __popcll(m);
            t0 += kStep;
            t += kStep;
            q += dq;
            r += dr;
            if (r >= R) { r -= R; ++q; }
        }
        wave_fence();
        run_buffer(S, cnt, work);
        flush();
        wave_fence();
    }
}

// Copies the partner list's geometry into list order for the block walk
// (listed partners only: a slot range is in list order already).
template <int W>
__device__ inline void gather_partners(const Stage& S, const List& A, const List& B, bool same, float4* gB)
{
    if (A.contig) return;
    const unsigned short* lb = same ? S.la : S.lb;
    const int nB = same ? A.n : B.n;
    for (int b = threadIdx.x; b < nB; b += W * kWave) gB[b] = S.g[lb[b]];
    __syncthreads();
}

template <int W, typename Work, typename Flush = NoFlush>
__device__ inline void walk_rows(const Stage& S, const List& A, const List& B, bool same, float rc2, Work&& work,
                                 Flush&& flush = Flush{})
{
    if (A.contig) for_each_triplet_rows<W, true>(S, A, B, same, rc2, work, flush);
    else for_each_triplet_rows<W, false>(S, A, B, same, rc2, work, flush);
}

// Cursor over the stored pair lists of an atom's walks: each wave has its
// share of the atom's entries and a count per walk.
struct TripCursor {
    unsigned* p;   // the next walk's pairs
    int room;      // entries left for them (0: none kept)
    int* counts;   // this atom's counts (nullptr: no list)
    int ld;        // walks with a count
    int w;         // walks so far
    int total;     // pairs of all walks so far
    bool rows;     // force kernel: the row-major walk (no lists)
};

template <int W>
__device__ inline TripCursor trip_cursor(const TripList& T, int i)
{
    TripCursor c{nullptr, 0, nullptr, 0, 0, 0, T.rows};
    if (T.list) {
        c.room = T.cap / W;
        c.p = T.list + (size_t)i * T.cap + wave_id() * c.room;
        c.counts = T.counts + ((size_t)i * kListWaves + wave_id()) * T.ld;
        c.ld = T.ld;
    }
    return c;
}

// The walk for slot-range lists and for listed slots.  Storing side (the SF
// kernel, store): the pairs go to the cursor's list while they fit and the
// walk's count is recorded.  Reading side (the force kernel, read): a walk
// with a recorded count reads its pairs back instead of testing candidates.
template <int W, bool GATHER, typename Work, typename Flush = NoFlush>
__device__ inline void walk_blocks(const Stage& S, const float4* gB, const List& A, const List& B, bool same,
                                   float rc2, TripCursor& tc, bool store, Work&& work, Flush&& flush = Flush{})
{
    const int w = tc.w++;
    const bool listed = tc.counts && w < tc.ld;
    const unsigned* src = nullptr;
    int nsrc = 0;
    if (listed && !store) {
        nsrc = uni(tc.counts[w]);
        if (nsrc >= 0) {
            src = tc.p;
            tc.p += nsrc;
        }
    }
    unsigned* dst = listed && store ? tc.p : nullptr;
    const int room = dst ? tc.room : 0;
    const int n = A.contig ? for_each_triplet_blocks<W, true, GATHER>(S, gB, A, B, same, rc2, src, nsrc, dst, room, work, flush)
                           : for_each_triplet_blocks<W, false, GATHER>(S, gB, A, B, same, rc2, src, nsrc, dst, room, work, flush);
    tc.total += n;
    if (dst) {
        const bool kept = n <= room;
        if (lane_id() == 0) tc.counts[w] = kept ? n : -1;
        if (kept) {
            tc.p += n;
            tc.room -= n;
        }
    }
}

// ------------------------------------------------------------ power path --
// Angular groups whose members are exp(-eta_h sum r^2) (1 + lambda_s cos)^zeta
// with zeta = 2^b (b <= 4), at most two distinct eta and two lambda, rs = 0:
// per triplet one exponential per eta and the powers p, p^2, p^4, ... of the
// two bases by repeated squaring (the reference's integer-zeta pow_int,
// utility.h, also multiplies) stand in for one exp2/log2 per member.  Terms
// are indexed beta = s NB0 + b (first eta) and 2 NB0 + s NB1 + b (second).

// LDS of a merged walk: the pair map, then per (merged group, term) one
// 8-byte entry (each wave's FP64 term sum, or the FP32 weights wb, wa).
__host__ __device__ constexpr size_t merge_bytes(int ng, int nbas, int waves)
{
    return (size_t)kMaxElem * kMaxElem + (size_t)waves * ng * nbas * 8;
}

// Calls f(integral_constant MAXM, bool_constant FAST) for the kernel
// instance matching the model: exact member counts {4, 8, 10, 16} on the fast
// path, powers of two up to 32 on the general one.
template <typename F>
inline void dispatch_members(int exact, int maxm, F&& f)
{
    using std::integral_constant;
    switch (exact) {
    case 4: f(integral_constant<int, 4>{}, std::true_type{}); return;
    case 8: f(integral_constant<int, 8>{}, std::true_type{}); return;
    case 10: f(integral_constant<int, 10>{}, std::true_type{}); return;
    case 16: f(integral_constant<int, 16>{}, std::true_type{}); return;
    default: break;
    }
    if (maxm <= 8) f(integral_constant<int, 8>{}, std::false_type{});
    else if (maxm <= 16) f(integral_constant<int, 16>{}, std::false_type{});
    else f(integral_constant<int, 32>{}, std::false_type{});
}

// Calls f(MAXM, FAST, NB0, NB1, COS) for the SF, force and tangent kernels'
// instance of the model: the power path when it applies, with the cosine
// cutoff or any, else as dispatch_members.
template <typename F>
inline void dispatch_angular(const MixedModel& mm, const ModelT& t, int maxm, F&& f)
{
    using std::integral_constant;
    using I0 = integral_constant<int, 0>;
    using I1 = integral_constant<int, 1>;
    using I3 = integral_constant<int, 3>;
    using I4 = integral_constant<int, 4>;
    using I5 = integral_constant<int, 5>;
    if (mm.powNB[0] > 0) {
        const std::true_type fast{};
        auto power = [&](auto n0, auto n1) {
            if (t.cutoffType == 1) f(I4{}, fast, n0, n1, std::true_type{});
            else f(I4{}, fast, n0, n1, std::false_type{});
        };
        switch (mm.powNB[0] * 10 + mm.powNB[1]) {
        case 30: power(I3{}, I0{}); return;
        case 33: power(I3{}, I3{}); return;
        case 50: power(I5{}, I0{}); return;
        case 51: power(I5{}, I1{}); return;
        case 55: power(I5{}, I5{}); return;
        default: throw Error{NNPX_ERR_STATE, "no kernel built for this power-path shape"};
        }
    }
    dispatch_members(mm.fastM, maxm, [&](auto m, auto fs) { f(m, fs, I0{}, I0{}, std::false_type{}); });
}

// Waves per atom: one where the atoms alone fill the chip (1,024 SIMDs, four to
// six waves each), more where they leave it short of waves and one atom's
// serial walk decides.  Values + forces in us for one, two and four waves:
// water 192 atoms 110, 79, 66; 768: 145, 107, 95; 1,536: 148, 132, 147; 3,072:
// 224, 223, 239; 12,288: 493, 552, 707 (the buffers of several waves fill less).
// Crystal of 256 atoms (merged walk) 91, 69, 61; 2,048: 128, 117, 132; 6,912:
// 268, 260, 320.  30 functions of many eta (member path): 192 atoms 153, 96, 71;
// 1,536: 181, 147, 150.
// Fewer where the staging with the smallest buffers does not fit beside them
// (from 961 slots on), for all kernels alike: the SF and the force kernel share
// pair lists per wave.
constexpr int kFewAtoms = 1024, kSomeAtoms = 4096;
inline int waves_per_atom(const MixedModel& mm, const SysView& s)
{
    const int nbas = 2 * (mm.powNB[0] + mm.powNB[1]);
    auto fits = [&](int w) {
        const size_t st = stage_bytes(s.stage_cap, w, kWave, stage_mp(mm.powNB[0], mm.powNB[1], w));
        return st + merge_bytes(mm.merge_ng, nbas, w) <= 65536 &&
               st + merge_bytes(mm.merge_ng, nbas, 1) + (sizeof(double) * 3 + 2) * (size_t)s.stage_cap <= 65536;
    };
    int w = s.natoms <= kFewAtoms ? 4 : s.natoms <= kSomeAtoms ? 2 : 1;
    while (w > 1 && !fits(w)) w /= 2;
    return w;
}

// Entries of each wave's triplet buffer: the tuned size, less where the
// staging of capL neighbours (fixed bytes beside the buffers) leaves no room.
inline int wave_trip(int tuned, int waves, size_t fixed)
{
    int trip = tuned;
    while (trip > kWave && fixed + (size_t)waves * (trip + kWave) * 4 > 65536) trip -= kWave;
    return trip;
}

template <typename F>
inline void dispatch_waves(int waves, F&& f)
{
    if (waves == 4) f(std::integral_constant<int, 4>{});
    else if (waves == 2) f(std::integral_constant<int, 2>{});
    else f(std::integral_constant<int, 1>{});
}

inline int pow2_members(const ModelT& t)
{
    const int m = std::max(std::max(t.max_mem_ang, t.max_mem_rad), 1);
    return m <= 4 ? 4 : m <= 8 ? 8 : m <= 16 ? 16 : 32;
}

}  // namespace
}  // namespace nnpx
