// k_tangent32: tangent of the symmetry functions along a field in the mixed
// form.
#include "mixed_device.hpp"

namespace nnpx {
namespace {

// ------------------------------------------- tangent of G along a field --
// dG_i/dx . u for every SF of every atom (the contraction of
// Training::collectDGdxia with a displacement field u), recomputing the
// radial and angular terms: per triplet the three geometric scalars
// s1 = r_ij.(u_i - u_j), s2 = r_ik.(u_i - u_k), s3 = r_jk.(u_k - u_j) are
// combined into three coefficients, and each member adds t_q times their
// member-weighted sum.  FP32 compensated sums per lane, FP64 across lanes,
// scaled like the SFs themselves (scaling factor and angular normalisation).
// Power path (NB0 > 0): per triplet one exponential per eta and the powers of
// the two bases, a term's tangent being E (p^(2^b) x + 2^b p^(2^b - 1) y) with
// x, y shared by the terms; FP64 sums per lane (the terms have both signs; a
// conversion and an addition, less than compensation).  Bound by instruction
// issue like the force kernel; 41,000 atoms, 30 angular functions per element:
// 1,342 us with an exponential per member, 972 us so (932 with FP32 sums over
// a buffer, which differ by up to 2e-7 with its size).
template <int W, int MAXM, bool FAST, int NB0, int NB1, bool COS>
__global__ __launch_bounds__(W * kWave) void k_tangent32(const ModelT* __restrict__ M, const MemberF* __restrict__ MF,
                                                         const GroupMixF* __restrict__ GM, SysView s,
                                                         const double* __restrict__ u, const float* __restrict__ sffac,
                                                         double* __restrict__ Gdot, int ldG, int capL, int trip)
{
    extern __shared__ float sm[];
    constexpr int MP = stage_mp(NB0, NB1, W);
    const Stage S = carve<W>(sm, capL, trip, MP);
    float4* du = reinterpret_cast<float4*>(reinterpret_cast<char*>(sm) + stage_bytes(capL, W, trip, MP));
    unsigned short* idx = reinterpret_cast<unsigned short*>(du + capL);
    const int i = blockIdx.x;
    const int tid = threadIdx.x, lane = lane_id();
    const int e = s.elem[i];
    const ElementT& E = M->el[e];
    const int ctype = M->cutoffType;
    const float tanhPre = (float)M->tanhPre;
    const int n = stage_atom<W>(M, s, i, capL, S, idx);
    {
        const double ux = u[3 * (size_t)i], uy = u[3 * (size_t)i + 1], uz = u[3 * (size_t)i + 2];
        const size_t base = (size_t)i * s.cap;
        for (int k = tid; k < n; k += W * kWave) {
            const int j = s.nb_j[base + idx[k]];
            const float dx = (float)(ux - u[3 * (size_t)j]);
            const float dy = (float)(uy - u[3 * (size_t)j + 1]);
            const float dz = (float)(uz - u[3 * (size_t)j + 2]);
            const float4 g = S.g[k];
            du[k] = make_float4(dx, dy, dz, g.x * dx + g.y * dy + g.z * dz);
        }
    }
    double* Gi = Gdot + (size_t)i * ldG;
    auto put = [&](int sf, double v) { Gi[sf] = v * (double)sffac[e * kMaxSF + sf]; };
    TripCursor tc{nullptr, 0, nullptr, 0, 0, 0, false};
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
        if (GT.type == 2 || GT.type == 12) {
            const bool wt = GT.type == 12;  // every neighbour, times its atomic number
            constexpr int CH = kRadChunk / 2;
            for (int q0 = wave_id() * CH; q0 < nmem; q0 += W * CH) {
                float acc[CH], cmp[CH];
#pragma unroll
                for (int q = 0; q < CH; ++q) { acc[q] = 0.f; cmp[q] = 0.f; }
                // type 2: the slots of neighbour element e1; type 12: every slot
                const int lo = wt ? 0 : S.eoff[GT.e1], hi = wt ? n : S.eoff[GT.e1 + 1];
                for (int k = lo + lane; k < hi; k += kWave) {
                    const float4 gk = S.g[k];
                    if (!(gk.w < g.rc)) continue;
                    const float4 ck = S.c[k];
                    const float sk = du[k].w * (wt ? ck.x * ck.w : ck.x);  // (r_ij / r).(u_i - u_j)
#pragma unroll
                    for (int q = 0; q < CH; ++q)
                        if (q0 + q < nmem) {
                            const float dr = gk.w - mf[q0 + q].rs;
                            const float ex = __expf(-mf[q0 + q].eta * dr * dr);
                            kahan(acc[q], cmp[q], (ck.z - mf[q0 + q].twoEta * dr * ck.y) * ex * sk);
                        }
                }
#pragma unroll
                for (int q = 0; q < CH; ++q)
                    if (q0 + q < nmem) {
                        const double v = wave_sum((double)acc[q] + (double)cmp[q]);
                        if (lane == 0) put(mf[q0 + q].sf, v);
                    }
            }
            __syncthreads();
            continue;
        }
        constexpr bool POW = NB0 > 0;
        constexpr int NBAS = POW ? 2 * (NB0 + NB1) : 1;
        constexpr int NBM = NB0 > NB1 ? NB0 : NB1;
        constexpr int NACC = POW ? NBAS : MAXM;
        // sums of terms of both signs: FP64, or FP32 with compensation per member
        using Sum = std::conditional_t<POW, double, float>;
        Sum acc[NACC];
        float cmp[POW ? 1 : MAXM];
#pragma unroll
        for (int q = 0; q < NACC; ++q) {
            acc[q] = 0;
            if (!POW) cmp[q] = 0.f;
        }
        const bool same = GT.e1 == GT.e2;
        const bool wide = GT.type == 9;  // no r_jk cutoff or exponent term (SymGrpExpAngw.cpp:156-380)
        const bool wt = GT.type == 13;    // Z_j Z_k weights (SymGrpExpAngnWeighted.cpp)
        const bool full = full_cutoff(M, GT);
        const List A = make_list<W>(S, n, GT.e1, g.rc, full, S.la);
        const List B = same ? A : make_list<W>(S, n, GT.e2, g.rc, full, S.lb);
        const GroupMixF gm = GM[E.grp0 + gi];
        MemberMasks R{0u, 0u, 0u};
        if constexpr (!POW) R = load_members(S, mf, nmem, nullptr);
        int jc = -1;  // j of the cached geometry (runs of one j per lane)
        float4 gj = make_float4(0.f, 0.f, 0.f, 0.f), cj = gj, uj = gj;
        walk_blocks<W, false>(S, nullptr, A, B, same, wide ? INFINITY : g.rc2, tc, true, [&](int j, int k) {
            if (j != jc) {
                gj = S.g[j];
                cj = S.c[j];
                uj = du[j];
                jc = j;
            }
            const float4 gk = S.g[k], ck = S.c[k], uk = du[k];
            const float r2jk = dist2(gj, gk);
            const float ijk = __builtin_amdgcn_rsqf(r2jk);
            const float rjk = r2jk * ijk;
            float fcjk = 1.f, dfcjk = 0.f;
            if (!wide) cutoff32<COS>(ctype, g.rc, g.rci, g.iw, g.rcinv, tanhPre, rjk, fcjk, dfcjk);
            const float rinvijik = cj.x * ck.x;
            const float cost = (gj.x * gk.x + gj.y * gk.y + gj.z * gk.z) * rinvijik;
            // type 13: every term and derivative times Z_j Z_k
            const float zw = wt ? cj.w * ck.w : 1.f;
            const float pfc = cj.y * ck.y * fcjk * zw;
            const float r2sum = gj.w * gj.w + gk.w * gk.w + (wide ? 0.f : r2jk);
            const float pr1 = ck.y * fcjk * cj.z * cj.x * zw;
            const float pr2 = cj.y * fcjk * ck.z * ck.x * zw;
            const float pr3 = cj.y * ck.y * dfcjk * ijk * zw;
            // geometric scalars of the field
            const float s1 = uj.w, s2 = uk.w;
            const float s3 = (gk.x - gj.x) * (uj.x - uk.x) + (gk.y - gj.y) * (uj.y - uk.y) +
                             (gk.z - gj.z) * (uj.z - uk.z);
            const float al = pfc * ((rinvijik - cost * cj.x * cj.x) * s1 + (rinvijik - cost * ck.x * ck.x) * s2 +
                                    rinvijik * s3);
            const float be = pr1 * s1 + pr2 * s2 - pr3 * s3;
            const float ga = pfc * ((wide ? 0.f : s3) - s1 - s2);
            if constexpr (POW) {
                const float E0 = fexp2(-gm.etaL[0] * r2sum);
                const float E1 = NB1 > 0 ? fexp2(-gm.etaL[1] * r2sum) : 0.f;
                const float x0 = E0 * fmaf(gm.twoEta[0], ga, be), x1 = E1 * fmaf(gm.twoEta[1], ga, be);
#pragma unroll
                for (int sl = 0; sl < 2; ++sl) {
                    const float pl = fmaf(gm.lam[sl], cost, 1.f);
                    const bool pos = pl > 0.f;
                    float p = pos ? pl : 0.f, pq = pos ? 1.f : 0.f;  // pl^(2^b), pl^(2^b - 1)
                    float y0 = E0 * al * gm.lam[sl], y1 = E1 * al * gm.lam[sl];  // times zeta = 2^b
#pragma unroll
                    for (int b = 0; b < NBM; ++b) {
                        if (b < NB0) acc[sl * NB0 + b] += (double)fmaf(x0, p, y0 * pq);
                        if (b < NB1) acc[2 * NB0 + sl * NB1 + b] += (double)fmaf(x1, p, y1 * pq);
                        pq *= p;
                        p *= p;
                        y0 += y0;
                        y1 += y1;
                    }
                }
            } else {
                constexpr int MAXS = FAST ? 2 : 4;
                float L[MAXS], Rp[MAXS];
#pragma unroll
                for (int t = 0; t < MAXS; ++t) {
                    const float pl = 1.f + gm.lam[t] * cost;
                    const bool pos = pl > 0.f;
                    L[t] = pos ? flog2(pl) : -INFINITY;
                    Rp[t] = pos ? __builtin_amdgcn_rcpf(pl) : 0.f;
                }
                if constexpr (FAST) {
#pragma unroll
                    for (int q = 0; q < MAXM; ++q) {
                        const float4 mq = S.mp[q];
                        const bool s1b = mq.w != 0.f;
                        const float t = fexp2(fmaf(mq.x, s1b ? L[1] : L[0], -mq.y * r2sum));
                        const float zl = mq.x * gm.lam[s1b ? 1 : 0];
                        const float c = fmaf(zl * (s1b ? Rp[1] : Rp[0]), al, be);
                        kahan(acc[q], cmp[q], t * fmaf(2.f * mq.y * 0.69314718f, ga, c));
                    }
                } else {
                    float ec = 0.f, fij = 1.f, fik = 1.f, fjk = 1.f;
                    bool shifted = false;
#pragma unroll
                    for (int q = 0; q < MAXM; ++q)
                        if (q < nmem) {
                            const float4 mq = S.mp[q];
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
                            const unsigned b1 = (R.s1 >> q) & 1u, b2 = (R.s2 >> q) & 1u;
                            const int sidx = (int)b1 | ((int)b2 << 1);
                            const float Ls = pickb<MAXS>(L, b1, b2);
                            const float Rs = pickb<MAXS>(Rp, b1, b2);
                            const float t = fexp2(fmaf(mq.x, Ls, ec));
                            const float zl = mq.x * pick<MAXS>(gm.lam, sidx);
                            const float twoEta = 2.f * mq.y * 0.69314718f;
                            float v = fmaf(zl * Rs, al, be);
                            if (shifted) v += twoEta * pfc * (fjk * s3 - fij * s1 - fik * s2);
                            else v += twoEta * ga;
                            kahan(acc[q], cmp[q], t * v);
                        }
                }
            }
        });
        // the waves' sums pass through their own buffers
        double* red = reinterpret_cast<double*>(S.tjk);
        const int stride = (S.trip + kWave) / 2;
#pragma unroll
        for (int q = 0; q < NACC; ++q)
            if (POW || q < nmem) {
                double v = (double)acc[q];
                if constexpr (!POW) v += (double)cmp[q];
                v = wave_sum(v);
                if (lane == 0) red[q] = v;
            }
        __syncthreads();
        if (tid < nmem) {
            const int at = POW ? mf[tid].beta : tid;
            double v = 0.0;
#pragma unroll
            for (int w = 0; w < W; ++w) v += reinterpret_cast<double*>(S.tj0)[w * stride + at];
            put(mf[tid].sf, v);
        }
        __syncthreads();
    }
}

}  // namespace

void launch_tangent32(const MixedModel& mm, const ModelT& t, const ModelT* d_model, const SysView& s,
                      const double* u, double* Gdot, int ldG, hipStream_t stream)
{
    if (!mm.ready) throw Error{NNPX_ERR_STATE, "mixed-precision tables not set up"};
    if (s.natoms == 0) return;
    const int capL = s.stage_cap;
    const int tt = mm.tune.trip_tangent;
    const size_t extra = (sizeof(float4) + 2) * (size_t)capL;
    if (stage_bytes(capL, 1, tt, stage_mp(0, 0, 1)) + extra > 65536)
        throw Error{NNPX_ERR_UNSUPPORTED, "neighbour count too large for the mixed kernels' LDS"};
    if (t.has_exp) dispatch_waves(waves_per_atom(mm, s), [&](auto wc) {
        dispatch_angular(mm, t, pow2_members(t), [&](auto m, auto fast, auto nb0, auto nb1, auto cs) {
            constexpr int W = decltype(wc)::value, c0 = decltype(nb0)::value, c1 = decltype(nb1)::value;
            constexpr int mp = stage_mp(c0, c1, W);
            const int trip = wave_trip(tt, W, stage_bytes(capL, 0, 0, mp) + extra);
            const size_t lds = stage_bytes(capL, W, trip, mp) + extra;
            if (lds > 65536) throw Error{NNPX_ERR_UNSUPPORTED, "neighbour count too large for the mixed kernels' LDS"};
            hipLaunchKernelGGL((k_tangent32<W, decltype(m)::value, decltype(fast)::value, c0, c1, decltype(cs)::value>),
                               dim3(s.natoms), dim3(W * kWave), lds, stream, d_model, mm.d_mem, mm.d_gmix, s, u,
                               mm.d_sffac, Gdot, ldG, capL, trip);
        });
    });
    launch_tangentcomp32(d_model, t, s, u, Gdot, ldG, stream);
}

}  // namespace nnpx
