// k_force32: the mixed form's fused dG/dr backward: recomputes each pair and
// triplet term and contracts it with dE/dG (Mode::calculateForces semantics,
// Mode.cpp:1922-1984) without storing dG/dr; FP64 accumulation in LDS per
// neighbour entry, pushed with FP64 atomics.
#include "mixed_device.hpp"

namespace nnpx {
namespace {

// Force weights of one power-path group: wb[beta] = sum of the members'
// dE/dG weights w on term beta, wa[beta] = sum of zeta lambda w.
template <int NBAS>
__device__ inline void power_weights(const Stage& S, const MemberF* __restrict__ mf, int nmem,
                                     const float* __restrict__ w, float* wb, float* wa)
{
    const int lane = lane_id();
    // one member per lane (nmem <= kMaxMembersExp < kWave), so its constants
    // and its weight are loaded once, all members at the same time
    int beta = -1;
    float wq = 0.f, wz = 0.f;
    if (lane < nmem) {
        const MemberF m = mf[lane];
        beta = m.beta;
        wq = w[m.sf];
        wz = wq * m.zetaLambda;
    }
    // lane b sums the weights of term b in member order
    float sb = 0.f, sa = 0.f;
    for (int q = 0; q < nmem; ++q) {
        const int bq = lane_value(beta, q);
        const float x = lane_value(wq, q), y = lane_value(wz, q);
        if (lane == bq) {
            sb += x;
            sa += y;
        }
    }
    if (threadIdx.x < NBAS) S.mp[lane] = make_float4(sb, sa, 0.f, 0.f);
    __syncthreads();
    // uniform: held in scalar registers
#pragma unroll
    for (int b = 0; b < NBAS; ++b) {
        const float4 v = S.mp[b];
        wb[b] = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v.x)));
        wa[b] = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v.y)));
    }
}

// --------------------------------------------------- fused force backward --
// One triplet's force terms, P1 r_ij + P2 r_ik + P3 (r_ik - r_ij) in the
// form (P1 - P3) r_ij + P3 r_ik for j and (P2 - P3) r_ik + P3 r_ij for k:
// the atom's own and j's parts summed in FP32 over the lane's run of j, k's
// part added to its FP64 LDS sum.
__device__ inline void force_terms(float P1, float P2, float P3, const float4& gj, const float4& gk, float& sx,
                                   float& sy, float& sz, float& rx, float& ry, float& rz, double* kx, double* ky,
                                   double* kz)
{
    const float d1 = P1 - P3, d2 = P2 - P3;
    sx = fmaf(P1, gj.x, fmaf(P2, gk.x, sx));
    sy = fmaf(P1, gj.y, fmaf(P2, gk.y, sy));
    sz = fmaf(P1, gj.z, fmaf(P2, gk.z, sz));
    rx = fmaf(d1, gj.x, fmaf(P3, gk.x, rx));
    ry = fmaf(d1, gj.y, fmaf(P3, gk.y, ry));
    rz = fmaf(d1, gj.z, fmaf(P3, gk.z, rz));
    lds_add(kx, (double)fmaf(d2, gk.x, P3 * gj.x));
    lds_add(ky, (double)fmaf(d2, gk.y, P3 * gj.y));
    lds_add(kz, (double)fmaf(d2, gk.z, P3 * gj.z));
}

// Forces of all power-path angular groups of an element in one triplet walk
// over the element-ordered in-cutoff list: each triplet takes the term
// weights (wb, wa) of its pair's group from LDS; the geometry and the
// accumulation are those of the per-group walk in k_force32.
template <int W, int NB0, int NB1, bool COS>
__device__ inline void force32_power_merged(const ModelT* __restrict__ M, const Stage& S,
                                            const MemberF* __restrict__ MF, const GroupMixF* __restrict__ GM,
                                            const AngMergeF& am, int n, int ctype, float tanhPre, char* mbase,
                                            const float* __restrict__ wi, double* ax, double* ay, double* az,
                                            double& fx, double& fy, double& fz, TripCursor& tc)
{
    constexpr int NBAS = 2 * (NB0 + NB1);
    constexpr int NBM = NB0 > NB1 ? NB0 : NB1;
    const int tid = threadIdx.x;
    const GroupT& G0 = M->grp[am.grp[0]];
    const GroupF g = group_f(G0);
    const GroupMixF gm = GM[am.grp[0]];
    const bool wide = G0.type == 9;
    const int ng = am.ng;
    signed char* pmap = reinterpret_cast<signed char*>(mbase);
    float2* wtab = reinterpret_cast<float2*>(mbase + kMaxElem * kMaxElem);
    for (int x = tid; x < kMaxElem * kMaxElem; x += W * kWave) pmap[x] = am.pair[x];
    // wb = sum of the members' w on term b, wa = sum of zeta lambda w
    for (int x = tid; x < ng * NBAS; x += W * kWave) {
        const int q = x / NBAS, b = x - q * NBAS;
        const GroupT& GT = M->grp[am.grp[q]];
        const MemberF* mf = MF + GT.mem0;
        float sb = 0.f, sa = 0.f;
        for (int m = 0; m < GT.nmem; ++m)
            if (mf[m].beta == b) {
                const float wq = wi[mf[m].sf];
                sb += wq;
                sa += wq * mf[m].zetaLambda;
            }
        wtab[x] = make_float2(sb, sa);
    }
    // all elements' in-cutoff neighbours, element by element (staging order)
    const List A = make_list<W>(S, n, -1, g.rc, full_cutoff(M, G0), S.la);  // its barrier orders the tables above
    int cur = -1, rowj = 0;
    float rx = 0.f, ry = 0.f, rz = 0.f, sx = 0.f, sy = 0.f, sz = 0.f;
    auto flush = [&]() {
        if (cur >= 0) {
            lds_add(ax + cur, (double)rx);
            lds_add(ay + cur, (double)ry);
            lds_add(az + cur, (double)rz);
            fx -= (double)sx;
            fy -= (double)sy;
            fz -= (double)sz;
        }
        cur = -1;
    };
    float4 gj = make_float4(0.f, 0.f, 0.f, 0.f), cj = gj;
    auto work = [&](int j, int k) {
        if (j != cur) {
            flush();
            cur = j;
            rx = 0.f; ry = 0.f; rz = 0.f;
            sx = 0.f; sy = 0.f; sz = 0.f;
            gj = S.g[j];
            cj = S.c[j];
            rowj = S.el[j] * kMaxElem;
        }
        const int q = pmap[rowj + S.el[k]];
        if (q < 0) return;
        const float2* wq = wtab + q * NBAS;
        const float4 gk = S.g[k];
        const float4 ck = S.c[k];
        const float r2jk = dist2(gj, gk);
        const float ijk = __builtin_amdgcn_rsqf(r2jk);
        const float rjk = r2jk * ijk;
        float fcjk = 1.f, dfcjk = 0.f;
        if (!wide) cutoff32<COS>(ctype, g.rc, g.rci, g.iw, g.rcinv, tanhPre, rjk, fcjk, dfcjk);
        const float rinvijik = cj.x * ck.x;
        const float cost = (gj.x * gk.x + gj.y * gk.y + gj.z * gk.z) * rinvijik;
        const float pfc = cj.y * ck.y * fcjk;
        const float r2sum = gj.w * gj.w + gk.w * gk.w + (wide ? 0.f : r2jk);
        const float pr1 = ck.y * fcjk * cj.z * cj.x;
        const float pr2 = cj.y * fcjk * ck.z * ck.x;
        const float pr3 = cj.y * ck.y * dfcjk * ijk;
        const float E0 = fexp2(-gm.etaL[0] * r2sum);
        const float E1 = NB1 > 0 ? fexp2(-gm.etaL[1] * r2sum) : 0.f;
        // (1 + lambda cos)^(2^b - 1) carried beside the power: no division
        float Q0 = 0.f, Q1 = 0.f, qa0 = 0.f, qa1 = 0.f;
#pragma unroll
        for (int sl = 0; sl < 2; ++sl) {
            const float pl = fmaf(gm.lam[sl], cost, 1.f);
            const bool pos = pl > 0.f;
            float p = pos ? pl : 0.f, pq = pos ? 1.f : 0.f;
#pragma unroll
            for (int b = 0; b < NBM; ++b) {
                if (b < NB0) {
                    const float2 w = wq[sl * NB0 + b];
                    Q0 = fmaf(w.x, p, Q0);
                    qa0 = fmaf(w.y, pq, qa0);
                }
                if (b < NB1) {
                    const float2 w = wq[2 * NB0 + sl * NB1 + b];
                    Q1 = fmaf(w.x, p, Q1);
                    qa1 = fmaf(w.y, pq, qa1);
                }
                pq *= p;
                p *= p;
            }
        }
        const float A = E0 * qa0 + E1 * qa1;
        const float B0 = E0 * Q0, B1 = E1 * Q1;
        const float B = B0 + B1;
        const float C0 = gm.twoEta[0] * B0 + gm.twoEta[1] * B1;
        const float C3 = wide ? 0.f : C0;
        const float P1 = pfc * (A * (rinvijik - cost * cj.x * cj.x) - C0) + B * pr1;
        const float P2 = pfc * (A * (rinvijik - cost * ck.x * ck.x) - C0) + B * pr2;
        const float P3 = pfc * (A * rinvijik + C3) - B * pr3;
        force_terms(P1, P2, P3, gj, gk, sx, sy, sz, rx, ry, rz, ax + k, ay + k, az + k);
    };
    if (tc.rows) walk_rows<W>(S, A, A, true, wide ? INFINITY : g.rc2, work, flush);
    else walk_blocks<W, false>(S, nullptr, A, A, true, wide ? INFINITY : g.rc2, tc, false, work, flush);
    flush();
    __syncthreads();
}

// Forces on the atom's neighbours are accumulated per neighbour entry in LDS
// (FP64) and pushed to the force array with FP64 atomics; contributions to
// the atom's own periodic images are dropped in the pull form
// (Mode::calculateForces skips them, Mode.cpp:1957) and kept in the push form.
// Bound by instruction issue and LDS.  W waves share an atom (waves_per_atom);
// COS drops the other cutoff types' code, 15 registers, which the crystal's
// merged walk had spare waves for (131,072 atoms, one wave each: 1,798 -> 1,672
// us) and water's did not (12,288 atoms: 240 us either way).
template <int W, int MAXM, bool FAST, int NB0, int NB1, bool MERGE, bool COS>
__global__ __launch_bounds__(W * kWave) void k_force32(const ModelT* __restrict__ M, const MemberF* __restrict__ MF,
                                                const GroupMixF* __restrict__ GM, const AngMergeF* __restrict__ AM,
                                                SysView s, const float* __restrict__ fw, int ldG,
                                                double* __restrict__ F, int push, int capL, int trip, TripList T,
                                                StageKeep K)
{
    extern __shared__ float sm[];
    const Stage S = carve<W>(sm, capL, trip, stage_mp(NB0, NB1, W));
    double* ax = reinterpret_cast<double*>(reinterpret_cast<char*>(sm) + stage_bytes(capL, W, trip, stage_mp(NB0, NB1, W)));
    double* ay = ax + capL;
    double* az = ay + capL;
    unsigned short* idx = reinterpret_cast<unsigned short*>(az + capL);
    char* mbase = reinterpret_cast<char*>(idx + capL);
    const int i = blockIdx.x;
    const int tid = threadIdx.x, lane = lane_id();
    const int e = s.elem[i];
    const ElementT& E = M->el[e];
    const int ctype = M->cutoffType;
    const float tanhPre = (float)M->tanhPre;
    const int n = K.g ? load_stage<W>(M, K, i, S) : stage_atom<W>(M, s, i, capL, S, idx);
    TripCursor tc = trip_cursor<W>(T, i);
    for (int k = tid; k < n; k += W * kWave) { ax[k] = 0.0; ay[k] = 0.0; az[k] = 0.0; }
    const float* wi = fw + (size_t)i * ldG;
    double fx = 0.0, fy = 0.0, fz = 0.0;
    const bool merged = MERGE && AM[e].ng > 0;
    __syncthreads();

    for (int gi = 0; gi < E.ngrp; ++gi) {
        const GroupT& GT = M->grp[E.grp0 + gi];
        const GroupF g = group_f(GT);
        const int nmem = GT.nmem;
        const MemberF* mf = MF + GT.mem0;
        if (E.ucut) {
            if (gi == 0) all_cutoffs<W, COS>(S, n, ctype, g, tanhPre);
        } else {
            group_cutoffs<W, COS>(S, n, GT.e1, GT.type == 2 ? GT.e1 : GT.e2, ctype, g, tanhPre);
        }
        if (sf_compact(GT.type)) continue;  // the compact kernel's
        if (merged && GT.type != 2 && GT.type != 12) continue;  // the merged walk's
        if (GT.type == 2 || GT.type == 12) {
            // radial: each thread owns its neighbours, no conflicts; type 12
            // weights every neighbour by its atomic number
            const bool wt = GT.type == 12;
            // type 2: the slots of neighbour element e1; type 12: every slot
            const int lo = wt ? 0 : S.eoff[GT.e1], hi = wt ? n : S.eoff[GT.e1 + 1];
            for (int k = lo + tid; k < hi; k += W * kWave) {
                const float4 gk = S.g[k];
                if (!(gk.w < g.rc)) continue;
                const float4 ck = S.c[k];
                float P = 0.f;
#pragma unroll 2
                for (int q = 0; q < nmem; ++q) {
                    const float dr = gk.w - mf[q].rs;
                    const float ex = __expf(-mf[q].eta * dr * dr);
                    P += wi[mf[q].sf] * (ck.z - mf[q].twoEta * dr * ck.y) * ex;
                }
                P *= wt ? ck.x * ck.w : ck.x;
                const double vx = (double)(P * gk.x), vy = (double)(P * gk.y), vz = (double)(P * gk.z);
                fx -= vx; fy -= vy; fz -= vz;
                ax[k] += vx; ay[k] += vy; az[k] += vz;
            }
            __syncthreads();
            continue;
        }
        const bool same = GT.e1 == GT.e2;
        const bool wide = GT.type == 9;  // no r_jk cutoff or exponent term (SymGrpExpAngw.cpp:156-380)
        const bool wt = GT.type == 13;    // Z_j Z_k weights (SymGrpExpAngnWeighted.cpp)
        const bool full = full_cutoff(M, GT);
        const List A = make_list<W>(S, n, GT.e1, g.rc, full, S.la);
        const List B = same ? A : make_list<W>(S, n, GT.e2, g.rc, full, S.lb);
        const GroupMixF gm = GM[E.grp0 + gi];
        constexpr bool POW = NB0 > 0;
        constexpr int NBAS = POW ? 2 * (NB0 + NB1) : 1;
        constexpr int NBM = NB0 > NB1 ? NB0 : NB1;
        float pwb[NBAS], pwa[NBAS];
        MemberMasks R{0u, 0u, 0u};
        if constexpr (POW) power_weights<NBAS>(S, mf, nmem, wi, pwb, pwa);
        else R = load_members(S, mf, nmem, wi);
        // FAST: the member constants stay in registers for the whole group
        // (zeta, -eta log2 e, the weights of B and C, and the weight of A
        // split by lambda index so A needs no per-member select)
        constexpr int NC = FAST && !POW ? MAXM : 1;
        float cz[NC], ce[NC], cA0[NC], cA1[NC], cB[NC], cC[NC];
        if constexpr (FAST && !POW) {
#pragma unroll
            for (int q = 0; q < MAXM; ++q) {
                const float4 mq = S.mp[q];
                const float4 wq = S.mp[kMaxMembersExp + q];
                const bool s1 = (R.s1 >> q) & 1u;
                cz[q] = mq.x;
                ce[q] = -mq.y;
                cB[q] = wq.y;
                cC[q] = wq.z;
                cA0[q] = s1 ? 0.f : wq.x;
                cA1[q] = s1 ? wq.x : 0.f;
            }
        }
        // Contributions to the row atom j and to the atom itself are summed
        // in FP32 over the lane's run of equal j (a few triplets) and added
        // in FP64 when j changes.
        int cur = -1;
        float rx = 0.f, ry = 0.f, rz = 0.f, sx = 0.f, sy = 0.f, sz = 0.f;
        auto flush = [&]() {
            if (cur >= 0) {
                lds_add(ax + cur, (double)rx);
                lds_add(ay + cur, (double)ry);
                lds_add(az + cur, (double)rz);
                fx -= (double)sx;
                fy -= (double)sy;
                fz -= (double)sz;
            }
        };
        float4 gj = make_float4(0.f, 0.f, 0.f, 0.f), cj = gj;  // geometry of the run's j
        auto work = [&](int j, int k) {
            if (j != cur) {
                flush();
                cur = j;
                rx = 0.f; ry = 0.f; rz = 0.f;
                sx = 0.f; sy = 0.f; sz = 0.f;
                gj = S.g[j];
                cj = S.c[j];
            }
            const float4 gk = S.g[k];
            const float4 ck = S.c[k];
            const float r2jk = dist2(gj, gk);
            const float ijk = __builtin_amdgcn_rsqf(r2jk);
            const float rjk = r2jk * ijk;
            float fcjk, dfcjk;
            fcjk = 1.f;
            dfcjk = 0.f;
            if (!wide) cutoff32<COS>(ctype, g.rc, g.rci, g.iw, g.rcinv, tanhPre, rjk, fcjk, dfcjk);
            const float rinvijik = cj.x * ck.x;
            const float cost = (gj.x * gk.x + gj.y * gk.y + gj.z * gk.z) * rinvijik;
            const float pfc = cj.y * ck.y * fcjk;
            const float r2sum = gj.w * gj.w + gk.w * gk.w + (wide ? 0.f : r2jk);
            const float pr1 = ck.y * fcjk * cj.z * cj.x;
            const float pr2 = cj.y * fcjk * ck.z * ck.x;
            const float pr3 = cj.y * ck.y * dfcjk * ijk;
            // per distinct lambda: log2(pl) (-inf where pl <= 0) and 1/pl
            constexpr int MAXS = FAST ? 2 : 4;
            float L[MAXS], Rp[MAXS];
#pragma unroll
            for (int t = 0; t < MAXS; ++t) {
                const float pl = 1.f + gm.lam[t] * cost;
                const bool pos = pl > 0.f;
                L[t] = pos ? flog2(pl) : -INFINITY;
                Rp[t] = pos ? __builtin_amdgcn_rcpf(pl) : 0.f;
            }
            // t_q = vexp * pl^zeta: u_q * pl = w t_q and u_q = w t_q / pl,
            // u_q = w vexp pl^(zeta-1) being the reference's fg times w
            float A = 0.f, B = 0.f, C0 = 0.f, C1 = 0.f, C2 = 0.f, C3 = 0.f;
            if constexpr (POW) {
                // B_h = E_h sum wb P, A_s = sum_h E_h sum wa P (powers of lambda s)
                const float E0 = fexp2(-gm.etaL[0] * r2sum);
                const float E1 = NB1 > 0 ? fexp2(-gm.etaL[1] * r2sum) : 0.f;
                // (1 + lambda cos)^(2^b - 1) is carried beside the power, so
                // A needs no division
                float Q0 = 0.f, Q1 = 0.f, qa0 = 0.f, qa1 = 0.f;
#pragma unroll
                for (int sl = 0; sl < 2; ++sl) {
                    const float pl = fmaf(gm.lam[sl], cost, 1.f);
                    const bool pos = pl > 0.f;
                    float p = pos ? pl : 0.f, pq = pos ? 1.f : 0.f;
#pragma unroll
                    for (int b = 0; b < NBM; ++b) {
                        if (b < NB0) {
                            Q0 = fmaf(pwb[sl * NB0 + b], p, Q0);
                            qa0 = fmaf(pwa[sl * NB0 + b], pq, qa0);
                        }
                        if (b < NB1) {
                            Q1 = fmaf(pwb[2 * NB0 + sl * NB1 + b], p, Q1);
                            qa1 = fmaf(pwa[2 * NB0 + sl * NB1 + b], pq, qa1);
                        }
                        pq *= p;
                        p *= p;
                    }
                }
                const float B0 = E0 * Q0, B1 = E1 * Q1;
                B = B0 + B1;
                C0 = gm.twoEta[0] * B0 + gm.twoEta[1] * B1;
                A = E0 * qa0 + E1 * qa1;
            } else if constexpr (FAST) {
                float A0 = 0.f, A1 = 0.f;
#pragma unroll
                for (int q = 0; q < MAXM; ++q) {
                    const bool s1 = (R.s1 >> q) & 1u;
                    const float t = fexp2(fmaf(cz[q], s1 ? L[1] : L[0], ce[q] * r2sum));
                    B = fmaf(cB[q], t, B);
                    C0 = fmaf(cC[q], t, C0);
                    A0 = fmaf(cA0[q], t, A0);
                    A1 = fmaf(cA1[q], t, A1);
                }
                A = A0 * Rp[0] + A1 * Rp[1];
            } else {
                float ec = 0.f, fij = 1.f, fik = 1.f, fjk = 1.f;
                bool shifted = false;
#pragma unroll
                for (int q = 0; q < MAXM; ++q)
                    if (q < nmem) {
                        const float4 mq = S.mp[q];
                        const float4 wq = S.mp[kMaxMembersExp + q];
                        if ((R.calc >> q) & 1u) {
                            float arg = r2sum;
                            shifted = mq.z > 0.f;
                            if (shifted) {
                                const float a = gj.w - mq.z, b = gk.w - mq.z, c = rjk - mq.z;
                                arg = a * a + b * b + (wide ? 0.f : c * c);
                                fij = a * cj.x;
                                fik = b * ck.x;
                                fjk = wide ? 0.f : c * ijk;
                            }
                            ec = -mq.y * arg;
                        }
                        const bool s1 = mq.w != 0.f, s2 = wq.w != 0.f;
                        const float Ls = s2 ? (s1 ? L[3] : L[2]) : (s1 ? L[1] : L[0]);
                        const float Rs = s2 ? (s1 ? Rp[3] : Rp[2]) : (s1 ? Rp[1] : Rp[0]);
                        const float t = fexp2(fmaf(mq.x, Ls, ec));
                        B = fmaf(wq.y, t, B);
                        const float c = wq.z * t;
                        if (shifted) {
                            C1 = fmaf(c, fij, C1);
                            C2 = fmaf(c, fik, C2);
                            C3 = fmaf(c, fjk, C3);
                        } else {
                            C0 += c;
                        }
                        A = fmaf(wq.x, t * Rs, A);
                    }
            }
            C1 += C0; C2 += C0;
            if (!wide) C3 += C0;
            const float zw = wt ? cj.w * ck.w : 1.f;
            const float P1 = zw * (pfc * (A * (rinvijik - cost * cj.x * cj.x) - C1) + B * pr1);
            const float P2 = zw * (pfc * (A * (rinvijik - cost * ck.x * ck.x) - C2) + B * pr2);
            const float P3 = zw * (pfc * (A * rinvijik + C3) - B * pr3);
            force_terms(P1, P2, P3, gj, gk, sx, sy, sz, rx, ry, rz, ax + k, ay + k, az + k);
        };
        if (tc.rows) walk_rows<W>(S, A, B, same, wide ? INFINITY : g.rc2, work);
        else walk_blocks<W, false>(S, nullptr, A, B, same, wide ? INFINITY : g.rc2, tc, false, work);
        flush();
        __syncthreads();
    }
    if constexpr (MERGE && NB0 > 0) {
        if (merged)
            force32_power_merged<W, NB0, NB1, COS>(M, S, MF, GM, AM[e], n, ctype, tanhPre, mbase, wi, ax, ay, az, fx, fy, fz,
                                           tc);
    }
    fx = wave_sum(fx);
    fy = wave_sum(fy);
    fz = wave_sum(fz);
    double* red = reinterpret_cast<double*>(S.tj0);
    if (lane == 0) {
        red[wave_id() * 3] = fx;
        red[wave_id() * 3 + 1] = fy;
        red[wave_id() * 3 + 2] = fz;
    }
    __syncthreads();
    if (tid < 3) {
        double v = 0.0;
#pragma unroll
        for (int w = 0; w < W; ++w) v += red[w * 3 + tid];
        atomicAdd(F + 3 * (size_t)i + tid, v);
    }
    const size_t base = (size_t)i * s.cap;
    for (int k = tid; k < n; k += W * kWave) {
        const int j = K.g ? K.nbr[(size_t)i * K.ld + k] : s.nb_j[base + idx[k]];
        if (j == i && !push) continue;
        atomicAdd(F + 3 * (size_t)j, ax[k]);
        atomicAdd(F + 3 * (size_t)j + 1, ay[k]);
        atomicAdd(F + 3 * (size_t)j + 2, az[k]);
    }
}


}  // namespace

void launch_force32(const MixedModel& mm, const ModelT& t, const ModelT* d_model, const SysView& s,
                    const MixedBuffers& b, const TripList& T, const StageKeep& KS, bool merge_f, bool push,
                    hipStream_t stream)
{
    const int capL = s.stage_cap;
    const int P = pow2_members(t);
    const int tf = mm.tune.trip_force;
    const int ps = push ? 1 : 0;
    dispatch_waves(waves_per_atom(mm, s), [&](auto wc) {
          dispatch_angular(mm, t, P, [&](auto m, auto fast, auto nb0, auto nb1, auto cs) {
            constexpr int W = decltype(wc)::value;
            constexpr int cm = decltype(m)::value, c0 = decltype(nb0)::value, c1 = decltype(nb1)::value;
            constexpr bool cf = decltype(fast)::value, cc = decltype(cs)::value;
            const bool mg = c0 > 0 && merge_f;
            constexpr int mp = stage_mp(c0, c1, W);
            const size_t extra = (sizeof(double) * 3 + 2) * (size_t)capL +
                                 (mg ? merge_bytes(mm.merge_ng, 2 * (c0 + c1), 1) : 0);
            const int trip = wave_trip(tf, W, stage_bytes(capL, 0, 0, mp) + extra);
            const size_t lds_f = stage_bytes(capL, W, trip, mp) + extra;
            if (lds_f > 65536) throw Error{NNPX_ERR_UNSUPPORTED, "neighbour count too large for the mixed kernels' LDS"};
            if (mg)
                hipLaunchKernelGGL((k_force32<W, cm, cf, c0, c1, (c0 > 0), cc>), dim3(s.natoms), dim3(W * kWave), lds_f,
                                   stream, d_model, mm.d_mem, mm.d_gmix, mm.d_amerge, s, b.dEdGf, b.ldG, b.F, ps, capL,
                                   trip, T, KS);
            else
                hipLaunchKernelGGL((k_force32<W, cm, cf, c0, c1, false, cc>), dim3(s.natoms), dim3(W * kWave), lds_f,
                                   stream, d_model, mm.d_mem, mm.d_gmix, mm.d_amerge, s, b.dEdGf, b.ldG, b.F, ps, capL,
                                   trip, T, KS);
          });
        });
}

}  // namespace nnpx
