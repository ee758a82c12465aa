// k_sf32: symmetry-function values of the mixed form in FP32, compensated sums
// per lane, lanes combined in FP64, FP64 scaling (SymGrpExpRad::calculate /
// SymGrpExpAngn::calculate without derivatives, SymGrpExpRad.cpp:144-239,
// SymGrpExpAngn.cpp:156-403); keeps each atom's staging, and optionally its
// angular pairs, in device memory for the force kernel of the same evaluation.
#include <map>
#include <mutex>

#include "mixed_device.hpp"

namespace nnpx {
namespace {

// SF values of one power-path group: FP32 partial sums per term over a
// triplet buffer folded into compensated sums, one FP64 wave reduction per
// used term, then each member takes its term (times 2^(1-zeta)) and is scaled.
template <int W, int NB0, int NB1, bool GATHER, bool COS>
__device__ inline void sf32_power_group(const ModelT* __restrict__ M, const Stage& S, float4* gB,
                                        const MemberF* __restrict__ mf, const GroupMixF& gm, const GroupT& GT,
                                        const GroupF& g, int n, int ctype, float tanhPre, int sf0,
                                        double* __restrict__ Gi, float* __restrict__ Ii, TripCursor& tc)
{
    constexpr int NBAS = 2 * (NB0 + NB1);
    constexpr int NBM = NB0 > NB1 ? NB0 : NB1;
    const int lane = lane_id();
    const bool same = GT.e1 == GT.e2;
    const bool wide = GT.type == 9;  // no r_jk cutoff or exponent term (SymGrpExpAngw.cpp:156-380)
    const bool wt = GT.type == 13;
    const bool full = full_cutoff(M, GT);
    const List A = make_list<W>(S, n, GT.e1, g.rc, full, S.la);
    const List B = same ? A : make_list<W>(S, n, GT.e2, g.rc, full, S.lb);
    if constexpr (GATHER) gather_partners<W>(S, A, B, same, gB);
    float acc[NBAS], cmp[NBAS], part[NBAS];
#pragma unroll
    for (int b = 0; b < NBAS; ++b) { acc[b] = 0.f; cmp[b] = 0.f; part[b] = 0.f; }
    const float ce0 = -gm.etaL[0], ce1 = -gm.etaL[1];
    const float lam0 = gm.lam[0], lam1 = gm.lam[1];
    int jc = -1;  // j of the cached geometry (runs of one j per lane)
    float4 gj = make_float4(0.f, 0.f, 0.f, 0.f), cj = gj;
    walk_blocks<W, GATHER>(S, gB, A, B, same, wide ? INFINITY : g.rc2, tc, true, [&](int j, int k) {
        if (j != jc) {
            gj = S.g[j];
            cj = S.c[j];
            jc = j;
        }
        const float4 gk = S.g[k];
        const float4 ck = S.c[k];
        const float r2jk = dist2(gj, gk);
        float fcjk = 1.f, dfcjk = 0.f;
        if (!wide) cutoff32<COS>(ctype, g.rc, g.rci, g.iw, g.rcinv, tanhPre, __builtin_amdgcn_sqrtf(r2jk), fcjk, dfcjk);
        const float cost = (gj.x * gk.x + gj.y * gk.y + gj.z * gk.z) * cj.x * ck.x;
        // type 13: times Z_j Z_k (SymGrpExpAngnWeighted.cpp)
        const float pfc = cj.y * ck.y * fcjk * (wt ? cj.w * ck.w : 1.f);
        const float r2sum = gj.w * gj.w + gk.w * gk.w + (wide ? 0.f : r2jk);
        const float E0 = fexp2(ce0 * r2sum) * pfc;
        const float E1 = NB1 > 0 ? fexp2(ce1 * r2sum) * pfc : 0.f;
#pragma unroll
        for (int sl = 0; sl < 2; ++sl) {
            const float pl = fmaf(sl ? lam1 : lam0, cost, 1.f);
            float p = pl > 0.f ? pl : 0.f;  // the reference's zero term for 1 + lambda cos <= 0
#pragma unroll
            for (int b = 0; b < NBM; ++b) {
                if (b < NB0) part[sl * NB0 + b] = fmaf(E0, p, part[sl * NB0 + b]);
                if (b < NB1) part[2 * NB0 + sl * NB1 + b] = fmaf(E1, p, part[2 * NB0 + sl * NB1 + b]);
                p *= p;
            }
        }
    }, [&]() {
#pragma unroll
        for (int b = 0; b < NBAS; ++b) {
            kahan(acc[b], cmp[b], part[b]);
            part[b] = 0.f;
        }
    });
    double* red = reinterpret_cast<double*>(S.mp);  // [W][NBAS], the waves' sums added in order
    double v[NBAS];
#pragma unroll
    for (int b = 0; b < NBAS; ++b) v[b] = (gm.used >> b) & 1 ? wave_sum((double)acc[b] + (double)cmp[b]) : 0.0;
    if (lane == 0) {
#pragma unroll
        for (int b = 0; b < NBAS; ++b) red[wave_id() * NBAS + b] = v[b];
    }
    __syncthreads();
    if (threadIdx.x < GT.nmem) {
        const MemberT& mt = M->mem[GT.mem0 + lane];
        double sum = 0.0;
#pragma unroll
        for (int w = 0; w < W; ++w) sum += red[w * NBAS + mf[lane].beta];
        const double gs = scale_sf(M->scale[sf0 + mt.sf], sum * mt.gnorm);
        Gi[mt.sf] = gs;
        Ii[mt.sf] = (float)gs;
    }
    __syncthreads();
}

// SF values of all power-path angular groups of an element in one triplet
// walk over the element-ordered in-cutoff list: FP32 partial sums per term
// over a lane's run of one group, folded into FP64 LDS sums per (group,
// term) when the group changes and after each buffer; then every member
// takes its group's term (times 2^(1-zeta)) and is scaled.
template <int W, int NB0, int NB1, bool GATHER, bool COS>
__device__ inline void sf32_power_merged(const ModelT* __restrict__ M, const Stage& S, float4* gB,
                                         const MemberF* __restrict__ MF, const GroupMixF* __restrict__ GM,
                                         const AngMergeF& am, const ElementT& E, int n, int ctype, float tanhPre,
                                         char* mbase, double* __restrict__ Gi, float* __restrict__ Ii,
                                         TripCursor& tc)
{
    constexpr int NBAS = 2 * (NB0 + NB1);
    constexpr int NBM = NB0 > NB1 ? NB0 : NB1;
    const int tid = threadIdx.x;
    const GroupT& G0 = M->grp[am.grp[0]];
    const GroupF g = group_f(G0);
    const GroupMixF gm = GM[am.grp[0]];
    const bool wide = G0.type == 9;
    const int ng = am.ng, used = am.used;
    signed char* pmap = reinterpret_cast<signed char*>(mbase);
    double* red = reinterpret_cast<double*>(mbase + kMaxElem * kMaxElem);
    for (int x = tid; x < kMaxElem * kMaxElem; x += W * kWave) pmap[x] = am.pair[x];
    for (int x = tid; x < W * ng * NBAS; x += W * kWave) red[x] = 0.0;
    double* mine = red + wave_id() * ng * NBAS;  // this wave's sums
    // all elements' in-cutoff neighbours, element by element (staging order)
    const List A = make_list<W>(S, n, -1, g.rc, full_cutoff(M, G0), S.la);  // its barrier orders the fills above
    if constexpr (GATHER) gather_partners<W>(S, A, A, true, gB);
    float part[NBAS];
#pragma unroll
    for (int b = 0; b < NBAS; ++b) part[b] = 0.f;
    int gc = -1;  // group of the partial sums
    auto flush = [&]() {
        if (gc >= 0) {
#pragma unroll
            for (int b = 0; b < NBAS; ++b)
                if ((used >> b) & 1) lds_add(mine + gc * NBAS + b, (double)part[b]);
        }
#pragma unroll
        for (int b = 0; b < NBAS; ++b) part[b] = 0.f;
        gc = -1;
    };
    const float ce0 = -gm.etaL[0], ce1 = -gm.etaL[1];
    const float lam0 = gm.lam[0], lam1 = gm.lam[1];
    int jc = -1, rowj = 0;
    float4 gj = make_float4(0.f, 0.f, 0.f, 0.f), cj = gj;
    walk_blocks<W, GATHER>(S, gB, A, A, true, wide ? INFINITY : g.rc2, tc, true, [&](int j, int k) {
        if (j != jc) {
            gj = S.g[j];
            cj = S.c[j];
            rowj = S.el[j] * kMaxElem;
            jc = j;
        }
        const int q = pmap[rowj + S.el[k]];
        if (q != gc) {
            flush();
            gc = q;
        }
        if (q < 0) return;
        const float4 gk = S.g[k];
        const float4 ck = S.c[k];
        const float r2jk = dist2(gj, gk);
        float fcjk = 1.f, dfcjk = 0.f;
        if (!wide) cutoff32<COS>(ctype, g.rc, g.rci, g.iw, g.rcinv, tanhPre, __builtin_amdgcn_sqrtf(r2jk), fcjk, dfcjk);
        const float cost = (gj.x * gk.x + gj.y * gk.y + gj.z * gk.z) * cj.x * ck.x;
        const float pfc = cj.y * ck.y * fcjk;
        const float r2sum = gj.w * gj.w + gk.w * gk.w + (wide ? 0.f : r2jk);
        const float E0 = fexp2(ce0 * r2sum) * pfc;
        const float E1 = NB1 > 0 ? fexp2(ce1 * r2sum) * pfc : 0.f;
#pragma unroll
        for (int sl = 0; sl < 2; ++sl) {
            const float pl = fmaf(sl ? lam1 : lam0, cost, 1.f);
            float p = pl > 0.f ? pl : 0.f;
#pragma unroll
            for (int b = 0; b < NBM; ++b) {
                if (b < NB0) part[sl * NB0 + b] = fmaf(E0, p, part[sl * NB0 + b]);
                if (b < NB1) part[2 * NB0 + sl * NB1 + b] = fmaf(E1, p, part[2 * NB0 + sl * NB1 + b]);
                p *= p;
            }
        }
    }, flush);
    __syncthreads();
    for (int q = 0; q < ng; ++q) {
        const GroupT& GT = M->grp[am.grp[q]];
        for (int x = tid; x < GT.nmem; x += W * kWave) {
            const MemberT& mt = M->mem[GT.mem0 + x];
            double sum = 0.0;
#pragma unroll
            for (int w = 0; w < W; ++w) sum += red[(w * ng + q) * NBAS + MF[GT.mem0 + x].beta];
            const double gs = scale_sf(M->scale[E.sf0 + mt.sf], sum * mt.gnorm);
            Gi[mt.sf] = gs;
            Ii[mt.sf] = (float)gs;
        }
    }
    __syncthreads();
}

// SF values of an element's radial groups when all its groups share one
// cutoff (staged cutoff values in S.c): all groups at once, each member on
// L = 64 W / members lanes (at least one) that sum every L-th neighbour of its
// group in FP32 with compensation; the L partial sums are added in FP64 in
// lane order through LDS (the idle triplet buffer), and the member's first
// lane scales and stores the value.
template <int W>
__device__ inline void radial_lanes(const ModelT* __restrict__ M, const Stage& S, const MemberF* __restrict__ MF,
                                    const ElementT& E, int n, double* __restrict__ Gi, float* __restrict__ Ii)
{
    constexpr int kLanes = W * kWave;
    const int lane = threadIdx.x;
    int nrad = 0;
    for (int gi = 0; gi < E.ngrp; ++gi) {
        const GroupT& GT = M->grp[E.grp0 + gi];
        if (GT.type == 2 || GT.type == 12) nrad += GT.nmem;
    }
    const int L = nrad > 0 && nrad < kLanes ? kLanes / nrad : 1;  // lanes per member
    const int sub = lane % L;
    double* part = reinterpret_cast<double*>(S.tj0);  // kLanes doubles fit the smallest buffers
    for (int base = 0; base < nrad; base += kLanes / L) {
        // the lane's member: the (base + lane / L)-th radial member of the element
        int rem = base + lane / L, gsel = -1;
        if (lane / L < kLanes / L)
            for (int gi = 0; gi < E.ngrp && gsel < 0; ++gi) {
                const GroupT& GT = M->grp[E.grp0 + gi];
                if (GT.type != 2 && GT.type != 12) continue;
                if (rem < GT.nmem) gsel = gi;
                else rem -= GT.nmem;
            }
        float acc = 0.f, cmp = 0.f;
        if (gsel >= 0) {
            const GroupT& GT = M->grp[E.grp0 + gsel];
            const MemberF mq = MF[GT.mem0 + rem];
            // type 2: the slots of neighbour element e1; type 12: every slot,
            // each term times its atomic number (SymGrpExpRadWeighted.cpp)
            const bool wt = GT.type == 12;
            const float rc = (float)GT.rc;
            const int lo = wt ? 0 : S.eoff[GT.e1], hi = wt ? n : S.eoff[GT.e1 + 1];
            for (int k = lo + sub; k < hi; k += L) {
                const float r = S.g[k].w;
                if (!(r < rc)) continue;
                const float4 ck = S.c[k];
                const float dr = r - mq.rs;
                kahan(acc, cmp, __expf(-mq.eta * dr * dr) * (wt ? ck.y * ck.w : ck.y));
            }
        }
        double v = (double)acc + (double)cmp;
        if (L > 1) {
            part[lane] = v;
            __syncthreads();
            if (sub == 0 && gsel >= 0)
                for (int t = 1; t < L; ++t) v += part[lane + t];
            __syncthreads();
        }
        if (gsel >= 0 && sub == 0) {
            const GroupT& GT = M->grp[E.grp0 + gsel];
            const MemberT& mt = M->mem[GT.mem0 + rem];
            const double gs = scale_sf(M->scale[E.sf0 + mt.sf], v);
            Gi[mt.sf] = gs;
            Ii[mt.sf] = (float)gs;
        }
    }
}

// ------------------------------------------------------------- SF values --
// Angular terms: vexp * pfc * pl^zeta evaluated as one exp2 of
// zeta * log2(pl) + log2(pfc) - eta log2(e) * sum(r - rs)^2, with log2(pl)
// shared by all members with the same lambda (pl <= 0 gives log2 = -inf, the
// reference's zero term).
// FAST: every angular group has exactly MAXM members, at most two distinct
// lambda and rs = 0 -- the member loop is then branch-free.  Otherwise the
// general loop handles shifted Gaussians and up to four lambda values.
// MERGE: the element's angular groups go through one merged walk when it
// has one (AngMergeF::ng > 0).
template <int W, int MAXM, bool FAST, int NB0, int NB1, bool GATHER, bool MERGE, bool COS>
__global__ __launch_bounds__(W * kWave) void k_sf32(const ModelT* __restrict__ M, const MemberF* __restrict__ MF,
                                             const GroupMixF* __restrict__ GM, const AngMergeF* __restrict__ AM,
                                             SysView s, double* __restrict__ G, float* __restrict__ Gin, int ldG,
                                             int ldK, int capL, int trip, TripList T, StageKeep K)
{
    extern __shared__ float sm[];
    const Stage S = carve<W>(sm, capL, trip, stage_mp(NB0, NB1, W));
    float4* gB = reinterpret_cast<float4*>(reinterpret_cast<char*>(sm) + stage_bytes(capL, W, trip, stage_mp(NB0, NB1, W)));
    char* mbase = reinterpret_cast<char*>(gB) + (GATHER ? sizeof(float4) * (size_t)capL : 0);
    const int i = blockIdx.x;
    const int tid = threadIdx.x, lane = lane_id();
    const int e = s.elem[i];
    const ElementT& E = M->el[e];
    const int ctype = M->cutoffType;
    const float tanhPre = (float)M->tanhPre;
    const int n = stage_atom<W>(M, s, i, capL, S, nullptr, K.g ? &K : nullptr);
    TripCursor tc = trip_cursor<W>(T, i);
    double* Gi = G + (size_t)i * ldG;
    float* Ii = Gin + (size_t)i * ldK;
    for (int q = E.nsf + tid; q < ldK; q += W * kWave) Ii[q] = 0.f;
    const bool merged = MERGE && AM[e].ng > 0;
    // one cutoff for all of the element's groups: the cutoff values once,
    // and every radial member at once, one lane each
    if (E.ucut && E.ngrp > 0) {
        all_cutoffs<W, COS>(S, n, ctype, group_f(M->grp[E.grp0]), tanhPre);
        radial_lanes<W>(M, S, MF, E, n, Gi, Ii);
    }

    for (int gi = 0; gi < E.ngrp; ++gi) {
        const GroupT& GT = M->grp[E.grp0 + gi];
        const GroupF g = group_f(GT);
        const int nmem = GT.nmem;
        const MemberF* mf = MF + GT.mem0;
        if (!E.ucut) group_cutoffs<W, COS>(S, n, GT.e1, GT.type == 2 ? GT.e1 : GT.e2, ctype, g, tanhPre);
        if (sf_compact(GT.type)) continue;  // the compact kernel's
        if (merged && GT.type != 2 && GT.type != 12) continue;  // the merged walk's
        if (GT.type == 2 || GT.type == 12) {
            if (E.ucut) continue;  // radial_lanes did it
            // radial members in chunks of kRadChunk (any member count);
            // type 12: every neighbour, each term times its atomic number
            // (SymGrpExpRadWeighted.cpp)
            const bool wt = GT.type == 12;
            // the wave sums go through LDS (the triplet buffer, >= kRadBatch
            // doubles) so a batch of members is scaled and stored by one lane
            // each, not one after another by lane 0
            double* red = reinterpret_cast<double*>(S.tjk);
            // the waves take the batches of kRadBatch members in turn
            for (int q0 = wave_id() * kRadBatch; q0 < nmem;
                 q0 += (q0 + kRadChunk) % kRadBatch == 0 ? kRadChunk + (W - 1) * kRadBatch : kRadChunk) {
                float acc[kRadChunk], cmp[kRadChunk];
#pragma unroll
                for (int q = 0; q < kRadChunk; ++q) { acc[q] = 0.f; cmp[q] = 0.f; }
                // type 2: the slots of neighbour element e1; type 12: every slot
                const int lo = wt ? 0 : S.eoff[GT.e1], hi = wt ? n : S.eoff[GT.e1 + 1];
                for (int k = lo + lane; k < hi; k += kWave) {
                    const float r = S.g[k].w;
                    if (!(r < g.rc)) continue;
                    const float fc = wt ? S.c[k].y * S.c[k].w : S.c[k].y;
#pragma unroll
                    for (int q = 0; q < kRadChunk; ++q)
                        if (q0 + q < nmem) {
                            const float dr = r - mf[q0 + q].rs;
                            kahan(acc[q], cmp[q], __expf(-mf[q0 + q].eta * dr * dr) * fc);
                        }
                }
                double v[kRadChunk];
#pragma unroll
                for (int q = 0; q < kRadChunk; ++q)
                    v[q] = q0 + q < nmem ? wave_sum((double)acc[q] + (double)cmp[q]) : 0.0;
                if (lane == 0) {
#pragma unroll
                    for (int q = 0; q < kRadChunk; ++q) red[(q0 + q) % kRadBatch] = v[q];
                }
                const int q1 = q0 + kRadChunk;
                if (q1 % kRadBatch == 0 || q1 >= nmem) {
                    wave_fence();
                    const int qm = q0 - q0 % kRadBatch + lane;  // this batch's members
                    if (lane < kRadBatch && qm < min(q1, nmem)) {
                        const MemberT& mt = M->mem[GT.mem0 + qm];
                        const double gs = scale_sf(M->scale[E.sf0 + mt.sf], red[qm % kRadBatch]);
                        Gi[mt.sf] = gs;
                        Ii[mt.sf] = (float)gs;
                    }
                    wave_fence();
                }
            }
            __syncthreads();
            continue;
        }
        if constexpr (NB0 > 0) {
            sf32_power_group<W, NB0, NB1, GATHER, COS>(M, S, gB, mf, GM[E.grp0 + gi], GT, g, n, ctype, tanhPre, E.sf0, Gi, Ii,
                                               tc);
            continue;
        }
        float acc[MAXM], cmp[MAXM];
#pragma unroll
        for (int q = 0; q < MAXM; ++q) { acc[q] = 0.f; cmp[q] = 0.f; }
        {
            const bool same = GT.e1 == GT.e2;
            const bool wide = GT.type == 9;  // no r_jk cutoff or exponent term (SymGrpExpAngw.cpp:156-380)
            const bool wt = GT.type == 13;
            const bool full = full_cutoff(M, GT);
            const List A = make_list<W>(S, n, GT.e1, g.rc, full, S.la);
            const List B = same ? A : make_list<W>(S, n, GT.e2, g.rc, full, S.lb);
            if constexpr (GATHER) gather_partners<W>(S, A, B, same, gB);
            const GroupMixF gm = GM[E.grp0 + gi];
            const MemberMasks R = load_members(S, mf, nmem, nullptr);
            // FAST: zeta and -eta log2 e in registers for the whole group;
            // terms summed in FP32 over one triplet buffer (a few per lane),
            // then folded into the compensated sums
            constexpr int NC = FAST ? MAXM : 1;
            float cz[NC], ce[NC], part[NC];
            if constexpr (FAST) {
#pragma unroll
                for (int q = 0; q < MAXM; ++q) {
                    cz[q] = S.mp[q].x;
                    ce[q] = -S.mp[q].y;
                    part[q] = 0.f;
                }
            }
            int jc = -1;  // j of the cached geometry (runs of one j per lane)
            float4 gj = make_float4(0.f, 0.f, 0.f, 0.f), cj = gj;
            walk_blocks<W, GATHER>(S, gB, A, B, same, wide ? INFINITY : g.rc2, tc, true, [&](int j, int k) {
                if (j != jc) {
                    gj = S.g[j];
                    cj = S.c[j];
                    jc = j;
                }
                const float4 gk = S.g[k];
                const float4 ck = S.c[k];
                const float r2jk = dist2(gj, gk);
                const float rjk = __builtin_amdgcn_sqrtf(r2jk);
                float fcjk, dfcjk;
                fcjk = 1.f;
                dfcjk = 0.f;
                if (!wide) cutoff32<COS>(ctype, g.rc, g.rci, g.iw, g.rcinv, tanhPre, rjk, fcjk, dfcjk);
                const float cost = (gj.x * gk.x + gj.y * gk.y + gj.z * gk.z) * cj.x * ck.x;
                const float lpfc = flog2(cj.y * ck.y * fcjk * (wt ? cj.w * ck.w : 1.f));  // type 13: Z_j Z_k
                const float r2sum = gj.w * gj.w + gk.w * gk.w + (wide ? 0.f : r2jk);
                constexpr int MAXS = FAST ? 2 : 4;
                float L[MAXS];
#pragma unroll
                for (int t = 0; t < MAXS; ++t) {
                    const float pl = 1.f + gm.lam[t] * cost;
                    L[t] = pl > 0.f ? flog2(pl) : -INFINITY;
                }
                if constexpr (FAST) {
#pragma unroll
                    for (int q = 0; q < MAXM; ++q) {
                        const bool s1 = (R.s1 >> q) & 1u;
                        const float ec = fmaf(ce[q], r2sum, lpfc);
                        part[q] += fexp2(fmaf(cz[q], s1 ? L[1] : L[0], ec));
                    }
                } else {
                    float ec = 0.f;
#pragma unroll
                    for (int q = 0; q < MAXM; ++q)
                        if (q < nmem) {
                            const float4 mq = S.mp[q];
                            const float4 mw = S.mp[kMaxMembersExp + q];
                            if ((R.calc >> q) & 1u) {
                                float arg = r2sum;
                                if (mq.z > 0.f) {
                                    const float a = gj.w - mq.z, b = gk.w - mq.z, c = rjk - mq.z;
                                    arg = a * a + b * b + (wide ? 0.f : c * c);
                                }
                                ec = fmaf(-mq.y, arg, lpfc);
                            }
                            const float lo = mq.w != 0.f ? L[1] : L[0];
                            const float hi = mq.w != 0.f ? L[3] : L[2];
                            const float Ls = mw.w != 0.f ? hi : lo;
                            kahan(acc[q], cmp[q], fexp2(fmaf(mq.x, Ls, ec)));
                        }
                }
            }, [&]() {
                if constexpr (FAST) {
#pragma unroll
                    for (int q = 0; q < MAXM; ++q) {
                        kahan(acc[q], cmp[q], part[q]);
                        part[q] = 0.f;
                    }
                }
            });
        }
        // wave sums through LDS, then one lane per member scales and stores
        double* red = reinterpret_cast<double*>(S.tjk);
        const int stride = (S.trip + kWave) / 2;  // doubles from a wave's buffer to the next
        static_assert(MAXM <= 32, "member sums must fit the smallest triplet buffer");
        double v[MAXM];
#pragma unroll
        for (int q = 0; q < MAXM; ++q) v[q] = q < nmem ? wave_sum((double)acc[q] + (double)cmp[q]) : 0.0;
        if (lane == 0) {
#pragma unroll
            for (int q = 0; q < MAXM; ++q) red[q] = v[q];
        }
        __syncthreads();
        if (tid < nmem) {
            const MemberT& mt = M->mem[GT.mem0 + lane];
            double sum = 0.0;
#pragma unroll
            for (int w = 0; w < W; ++w) sum += reinterpret_cast<double*>(S.tj0)[w * stride + lane];
            const double gs = scale_sf(M->scale[E.sf0 + mt.sf], sum * mt.gnorm);
            Gi[mt.sf] = gs;
            Ii[mt.sf] = (float)gs;
        }
        __syncthreads();
    }
    if constexpr (MERGE && NB0 > 0) {
        if (merged)
            sf32_power_merged<W, NB0, NB1, GATHER, COS>(M, S, gB, MF, GM, AM[e], E, n, ctype, tanhPre, mbase, Gi, Ii, tc);
    }
    // the largest pair count per atom sizes the lists (the waves' equal shares
    // by the fullest of them)
    if (T.count && lane == 0 &&
        W * tc.total > __hip_atomic_load(&s.flags[3], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
        atomicMax(&s.flags[3], W * tc.total);
}

}  // namespace

// Resident blocks per CU of a kernel instance at a dynamic LDS size, from the
// HIP occupancy calculator, cached per (instance, size).
static int blocks_per_cu(const void* kernel, int threads, size_t lds)
{
    static std::mutex mu;
    static std::map<std::pair<const void*, size_t>, int> cache;
    std::lock_guard<std::mutex> lock(mu);
    auto it = cache.find({kernel, lds});
    if (it != cache.end()) return it->second;
    int occ = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kernel, threads, lds) != hipSuccess)
        throw Error{NNPX_ERR_HIP, "hipOccupancyMaxActiveBlocksPerMultiprocessor"};
    cache[{kernel, lds}] = occ;
    return occ;
}

void launch_sf32(const MixedModel& mm, const ModelT& t, const ModelT* d_model, const SysView& s,
                 const MixedBuffers& b, const TripList& T, const StageKeep& KS, bool merge_sf, hipStream_t stream)
{
    const int capL = s.stage_cap;
    const int P = pow2_members(t);
    const int tsf = mm.tune.trip_sf;
    dispatch_waves(waves_per_atom(mm, s), [&](auto wc) {
          dispatch_angular(mm, t, P, [&](auto m, auto fast, auto nb0, auto nb1, auto cs) {
            constexpr int W = decltype(wc)::value;
            constexpr int cm = decltype(m)::value, c0 = decltype(nb0)::value, c1 = decltype(nb1)::value;
            constexpr bool cf = decltype(fast)::value, cc = decltype(cs)::value;
            constexpr bool cmg = c0 > 0;  // merged instances exist on the power path only
            const bool mg = cmg && merge_sf;
            const size_t extra = mg ? merge_bytes(mm.merge_ng, 2 * (c0 + c1), W) : 0;
            constexpr int mp = stage_mp(c0, c1, W);
            // the partner gather costs 16 B of LDS per slot: taken only when
            // it leaves the blocks per CU unchanged
            const int trip = wave_trip(tsf, W, stage_bytes(capL, 0, 0, mp) + extra);
            const size_t lds0 = stage_bytes(capL, W, trip, mp) + extra;
            const size_t lds1 = lds0 + sizeof(float4) * (size_t)capL;
            if (lds0 > 65536) throw Error{NNPX_ERR_UNSUPPORTED, "neighbour count too large for the mixed kernels' LDS"};
            auto launch = [&](auto gather, auto merge) {
                constexpr bool cg = decltype(gather)::value, cmm = decltype(merge)::value;
                hipLaunchKernelGGL((k_sf32<W, cm, cf, c0, c1, cg, cmm, cc>), dim3(s.natoms), dim3(W * kWave),
                                   cg ? lds1 : lds0, stream, d_model, mm.d_mem, mm.d_gmix, mm.d_amerge, s, b.G, b.Gin,
                                   b.ldG, mm.ldK, capL, trip, T, KS);
            };
            auto pick = [&](auto merge) {
                constexpr bool cmm = decltype(merge)::value;
                int occ0 = 0, occ1 = 0;
                const int want = mm.tune.sf_gather;
                if (lds1 <= 65536 && want != 0) {
                    occ0 = blocks_per_cu(reinterpret_cast<const void*>(&k_sf32<W, cm, cf, c0, c1, false, cmm, cc>),
                                         W * kWave, lds0);
                    occ1 = blocks_per_cu(reinterpret_cast<const void*>(&k_sf32<W, cm, cf, c0, c1, true, cmm, cc>),
                                         W * kWave, lds1);
                }
                if (occ1 > 0 && (occ1 >= occ0 || want == 1))
                    launch(std::true_type{}, merge);
                else
                    launch(std::false_type{}, merge);
            };
            if (mg) pick(std::integral_constant<bool, cmg>{});
            else pick(std::false_type{});
          });
        });
}

}  // namespace nnpx
