// Compact symmetry-function groups in factored form (types 20, 22, 23, 25).
//
// The members of a wide compact group are products: a radial function at each
// of the two neighbours times an angular function of the triplet
// (SymGrpCompAngw::calculate, SymGrpCompAngw.cpp:117-341, evaluates them member
// by member; published models hold 54 members on 9 radial and 6 angular
// functions).  Here every radial function is evaluated once per neighbour
// and kept in LDS, every angular function once per triplet, and
//   G_uv     = sum_jk R_u(r_ij) R_u(r_ik) A_v(theta)
// takes one multiply-add per member and triplet, in FP64.  The force mode
// folds the members' weights w_uv first: with a_u = sum_v w_uv A_v and
// b_u = sum_v w_uv A_v',
//   X  = sum_u R_u(j) R_u(k) b_u,  Y1 = sum_u R_u'(j) R_u(k) a_u,
//   Y2 = sum_u R_u(j) R_u'(k) a_u
// give the members' summed p1, p2, p3 of the reference; the tangent mode takes
// two multiply-adds per member.  Radial groups (SymGrpCompRad.cpp:129-199 and
// SymGrpCompRadWeighted.cpp:120-200) are here too, with the element-weighted
// forms (23, 25: every neighbour, times its atomic number).  Narrow groups
// (21, 24: a third radial factor at r_jk, taken over between members) and
// groups with more functions stay in sfcomp64.hip.
//
// Mapping: four waves per atom, neighbours staged by element in the term
// precision with their radial tables.  Every pair of a group counts (no r_jk
// cutoff), so its pairs are dealt out evenly, each thread a run of
// neighbouring pairs: the first atom j's geometry, table row and force sum stay
// in registers over the run, partner k's force goes through LDS FP64 atomics.
// Radial members: a wave each (values, tangent); threads own neighbours
// (force).
//   Bound by instruction issue (294 vector instructions per triplet for 54
// values, 480 for their forces) with few waves to hide the rest: the registers
// allow two per SIMD for the values (64 FP64 sums take 128) and three for the
// forces; 1,152 atoms, 4.5 blocks per CU, keep 1.3 and 1.8 resident, which issue
// 43% and 63% of the time.  For those, 184 functions and 185 neighbours each,
// FP32 terms: values 4,344 us member by member -> 335 us, forces 4,872 -> 377
// us (647 and 639 with a switch over the cores and a window test per function
// in the walk; forces 370 with a run's sums in FP32, which cost up to 8e-7 of a
// sum of 392 like terms, against 1.8e-7 for the terms alone).
#include <type_traits>

#include "nnpx.h"
#include "sfcomp.hpp"
#include "stage.hpp"

namespace nnpx {
namespace {

constexpr int kFW = 4;                      // waves per atom
constexpr int kFT = kFW * kWave;
constexpr int kCells = kCompU * kCompV;
constexpr size_t kFLds = 65536;
static_assert(kCells <= kWave, "the wave reduction leaves one cell per lane");

template <typename T>
struct Vec4;
template <>
struct Vec4<float> {
    using type = float4;
};
template <>
struct Vec4<double> {
    using type = double4;
};

// Row of a slot's radial values (padded to 16-byte loads).
template <typename T>
constexpr int kRow = std::is_same<T, float>::value ? 12 : 10;
static_assert(kCompU <= 10 && kCompU <= 12, "a row holds every radial function");

template <typename T>
__device__ inline void load_row(const T* p, T* v)
{
    if constexpr (std::is_same<T, float>::value) {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const float4 x = reinterpret_cast<const float4*>(p)[q];
            v[4 * q] = x.x;
            v[4 * q + 1] = x.y;
            v[4 * q + 2] = x.z;
            v[4 * q + 3] = x.w;
        }
    } else {
#pragma unroll
        for (int q = 0; q < 5; ++q) {
            const double2 x = reinterpret_cast<const double2*>(p)[q];
            v[2 * q] = x.x;
            v[2 * q + 1] = x.y;
        }
    }
}

// LDS bytes: per slot the geometry, 1/r, list entry and element, the radial
// table and (not for values) its derivatives, and three FP64 sums (force) or
// the tangent's field; the weights and the waves' sums; the element offsets.
template <typename T>
__host__ __device__ constexpr size_t fac_bytes(int capL, bool der)
{
    return (size_t)capL * (4 * sizeof(T) + sizeof(T) + 2 + 1 + kRow<T> * sizeof(T) * (der ? 2 : 1) + (der ? 24 : 0)) +
           (size_t)kFW * kWave * 8 + 64 * sizeof(T) + kCompV * 4 * sizeof(T) + 48 + 64;
}

// A window's function and derivative at x: its polynomial core at
// min(|x - cen| scl, 1), where the polynomials and their slopes vanish, so the
// window needs no test; the exponential core does.  POLY2: every core of the
// model's factored groups is the second polynomial (no switch in the walk).
template <bool POLY2, typename T>
__device__ inline void window_fdf(int core, bool asym, T cen, T scl, T x, T& f, T& df)
{
    const T a = (x - cen) * scl;
    T y = a < T(0) ? -a : a;
    if (!POLY2 && core == 0 && !(y < T(1))) {
        f = df = T(0);
        return;
    }
    y = y < T(1) ? y : T(1);
    const T z = asym ? (T(2) - y) * y : y;
    if constexpr (POLY2) {
        const T z2 = z * z;
        f = ((T(15) - T(6) * z) * z - T(10)) * z * z2 + T(1);
        df = z2 * ((T(60) - T(30) * z) * z - T(30));
    } else {
        core_fdf(core, z, f, df);
    }
    if (asym) df *= T(2) - T(2) * y;
    df *= a < T(0) ? -scl : scl;
}

// Sums v[0 .. 2H - 1] over the wave's lanes for H = 32: lane l receives the
// total of v[bits of l reversed] by exchanging halves (63 exchanges for 64
// sums).  Recursive, so that every index is a constant (registers).
template <int H>
__device__ inline double reduce_cells(double* v)
{
    constexpr int m = 32 / H;
    const bool up = lane_id() & m;
#pragma unroll
    for (int k = 0; k < H; ++k) {
        const double give = up ? v[k] : v[k + H], keep = up ? v[k + H] : v[k];
        v[k] = keep + __shfl_xor(give, m);
    }
    if constexpr (H > 1) return reduce_cells<H / 2>(v);
    else return v[0];
}

template <typename T, int MODE, bool POLY2>
__global__ __launch_bounds__(kFT) void k_sfcomp_fac(const ModelT* __restrict__ M, SysView s, CompMix c, int capL)
{
    constexpr bool FORCE = MODE == CM_FORCE, TANGENT = MODE == CM_TANGENT, DER = FORCE || TANGENT;
    using V4 = typename Vec4<T>::type;
    extern __shared__ double4 fsm[];
    double* red = reinterpret_cast<double*>(fsm);      // [kFW][kWave]
    double* ax = red + kFW * kWave;                    // [3][capL] force sums, or u_j - u_i
    V4* g = reinterpret_cast<V4*>(ax + (DER ? 3 * capL : 0));
    T* ri = reinterpret_cast<T*>(g + capL);
    constexpr int RW = kRow<T>;
    T* R = ri + capL;                                  // [capL][RW]
    T* dR = R + (size_t)RW * capL;
    T* wl = dR + (DER ? (size_t)RW * capL : 0);        // [kCells] weights of the group's members
    V4* aw = reinterpret_cast<V4*>(wl + 64);           // [kCompV] centre and scale of the angular windows
    int* eoff = reinterpret_cast<int*>(aw + kCompV);
    unsigned short* idx = reinterpret_cast<unsigned short*>(eoff + 12);
    unsigned char* el = reinterpret_cast<unsigned char*>(idx + capL);

    const int i = blockIdx.x, tid = threadIdx.x, lane = lane_id(), wv = wave_id();
    const int e = s.elem[i];
    const ElementT& E = M->el[e];
    // the staging counts use the sums' area, which is free until the first walk
    const int n = stage_by_element<kFW>(M, s, i, capL, reinterpret_cast<int*>(red), eoff,
                                        [&](int pos, int k, const double* dr, double d, int ek) {
                                            g[pos] = V4{(T)dr[0], (T)dr[1], (T)dr[2], (T)d};
                                            ri[pos] = (T)(1.0 / d);
                                            idx[pos] = (unsigned short)k;
                                            el[pos] = (unsigned char)ek;
                                        });
    const size_t ebase = (size_t)i * s.cap;
    if constexpr (FORCE)
        for (int k = tid; k < 3 * capL; k += kFT) ax[k] = 0.0;
    if constexpr (TANGENT)
        for (int k = tid; k < n; k += kFT) {
            const size_t j = s.nb_j[ebase + idx[k]];
            for (int x = 0; x < 3; ++x) ax[x * capL + k] = c.u[3 * j + x] - c.u[3 * (size_t)i + x];
        }
    __syncthreads();

    double* Gi = FORCE ? nullptr : c.G + (size_t)i * c.ldG;
    float* Ii = c.Gin ? c.Gin + (size_t)i * c.ldK : nullptr;
    if (MODE == CM_VALUES && Ii)  // the network input's padding
        for (int q = E.nsf + tid; q < c.ldK; q += kFT) Ii[q] = 0.f;
    auto weight = [&](int sf) -> T {
        if constexpr (std::is_same<T, double>::value) return c.fw64[(size_t)i * c.ldG + sf];
        else return (T)c.fw[(size_t)i * c.ldG + sf];
    };
    auto put = [&](const MemberT& mb, double v) {
        if (TANGENT) {
            Gi[mb.sf] = v * mb.sfac;
            return;
        }
        const double gs = scale_sf(M->scale[E.sf0 + mb.sf], v);
        Gi[mb.sf] = gs;
        if (Ii) Ii[mb.sf] = (float)gs;
    };
    double fx = 0.0, fy = 0.0, fz = 0.0;  // force mode: this thread's part of the atom's own force

    // ---------------------------------------------------------- radial groups
    for (int gi = 0; gi < E.nrad; ++gi) {
        const GroupT& G = M->grp[E.grp0 + gi];
        if (G.type != 20 && G.type != 23) continue;
        const bool wt = G.type == 23;  // every neighbour, times its atomic number
        const int lo = wt ? 0 : eoff[G.e1], hi = wt ? n : eoff[G.e1 + 1];
        if constexpr (FORCE) {
            for (int k = lo + tid; k < hi; k += kFT) {
                const V4 gk = g[k];
                T P = T(0);
                for (int q = 0; q < G.nmem; ++q) {
                    const MemberT& mb = M->mem[G.mem0 + q];
                    if (!(gk.w > (T)mb.rl && gk.w < (T)mb.rcm)) continue;
                    T f, df;
                    compact_fdf(mb.core, mb.asym, (T)mb.cen, (T)mb.scl, gk.w, f, df);
                    P += weight(mb.sf) * df;
                }
                P *= (wt ? (T)M->Zel[el[k]] : T(1)) * ri[k];
                const double vx = (double)(P * gk.x), vy = (double)(P * gk.y), vz = (double)(P * gk.z);
                fx -= vx; fy -= vy; fz -= vz;
                ax[k] += vx; ax[capL + k] += vy; ax[2 * capL + k] += vz;
            }
            __syncthreads();
        } else {
            for (int q = wv; q < G.nmem; q += kFW) {
                const MemberT& mb = M->mem[G.mem0 + q];
                double sum = 0.0;
                for (int k = lo + lane; k < hi; k += kWave) {
                    const V4 gk = g[k];
                    if (!(gk.w > (T)mb.rl && gk.w < (T)mb.rcm)) continue;
                    T f, df;
                    compact_fdf(mb.core, mb.asym, (T)mb.cen, (T)mb.scl, gk.w, f, df);
                    const T Z = wt ? (T)M->Zel[el[k]] : T(1);
                    if constexpr (TANGENT)
                        sum -= (double)(Z * df * ri[k]) * ((double)gk.x * ax[k] + (double)gk.y * ax[capL + k] +
                                                           (double)gk.z * ax[2 * capL + k]);
                    else sum += (double)(Z * f);
                }
                sum = wave_sum(sum);
                if (lane == 0) put(mb, sum);
            }
        }
    }

    // --------------------------------------------------------- angular groups
    for (int gi = E.nrad; gi < E.ngrp; ++gi) {
        const GroupT& G = M->grp[E.grp0 + gi];
        if (!G.fac) continue;
        const CompFactorT& C = M->cfac[G.fac - 1];
        const bool wt = G.type == 25;  // all neighbour pairs, the angular factor times Z_j Z_k
        const bool same = G.e1 == G.e2;
        const int lo1 = wt ? 0 : eoff[G.e1], hi1 = wt ? n : eoff[G.e1 + 1];
        const int lo2 = wt ? 0 : eoff[G.e2], hi2 = wt ? n : eoff[G.e2 + 1];
        const int nA = hi1 - lo1, nB = hi2 - lo2;
        const int U = C.U, V = C.V;
        // radial tables of the group's neighbours and the members' weights
        for (int x = tid; x < n; x += kFT) {
            if (!((x >= lo1 && x < hi1) || (x >= lo2 && x < hi2))) continue;
            const T r = g[x].w;
            for (int u = 0; u < RW; ++u) {
                T f = T(0), df = T(0);
                if (u < U)
                    window_fdf<POLY2>(C.rad[u].core, C.rad[u].asym, (T)C.rad[u].cen, (T)C.rad[u].scl, r, f, df);
                R[x * RW + u] = f;
                if (DER) dR[x * RW + u] = df;
            }
        }
        if (tid < V) aw[tid] = V4{(T)C.ang[tid].cen, (T)C.ang[tid].scl, T(0), T(0)};
        if (FORCE && tid < kCells) wl[tid] = C.cell[tid] >= 0 ? weight(M->mem[G.mem0 + C.cell[tid]].sf) : T(0);
        __syncthreads();
        // pairs: row a with b = a + 1 .. a + cols (mod nA), for even nA the
        // half-way column on half the rows; unlike elements the full product
        const int cols = same ? (nA - 1) / 2 : nB;
        const int full = nA * cols, total = full + (same && nA % 2 == 0 ? nA / 2 : 0);
        const int per = (total + kFT - 1) / kFT;
        const int t0 = tid * per, t1 = min(total, t0 + per);
        // the weights in registers (FP32; in FP64 they would fill them)
        constexpr bool FLOATW = FORCE && std::is_same<T, float>::value;
        T wr[FLOATW ? kCells : 1];
        if constexpr (FLOATW) {
#pragma unroll
            for (int q = 0; q < kCells; ++q) wr[q] = wl[q];
        }
        double acc[FORCE ? 1 : 64];
#pragma unroll
        for (int q = 0; q < (FORCE ? 1 : 64); ++q) acc[q] = 0.0;
        int a = cols > 0 ? t0 / cols : 0, col = cols > 0 ? t0 - a * cols : 0;
        int cur = -1;
        V4 gj{};
        T rij = T(0), Rj[RW], dRj[DER ? RW : 1];
        double sx = 0.0, sy = 0.0, sz = 0.0, hx = 0.0, hy = 0.0, hz = 0.0;  // sums of a run of one j
        T wjx = T(0), wjy = T(0), wjz = T(0);
        auto flush = [&] {
            if constexpr (FORCE) {
                if (cur >= 0) {
                    lds_add(ax + cur, hx);
                    lds_add(ax + capL + cur, hy);
                    lds_add(ax + 2 * capL + cur, hz);
                    fx -= sx;
                    fy -= sy;
                    fz -= sz;
                }
            }
        };
        for (int t = t0; t < t1; ++t) {
            int b;
            if (t < full) {
                b = same ? a + col + 1 : col;
                b = same && b >= nA ? b - nA : b;
            } else {
                a = t - full;
                b = a + nA / 2;
            }
            const int j = lo1 + a, k = lo2 + b;
            if (j != cur) {
                flush();
                cur = j;
                gj = g[j];
                rij = ri[j];
                load_row(R + j * RW, Rj);
                if constexpr (DER) load_row(dR + j * RW, dRj);
                sx = sy = sz = hx = hy = hz = 0.0;
                if (TANGENT) {
                    wjx = (T)ax[j];
                    wjy = (T)ax[capL + j];
                    wjz = (T)ax[2 * capL + j];
                }
            }
            if (++col == cols) {
                col = 0;
                ++a;
            }
            const V4 gk = g[k];
            const T rik = ri[k];
            // FP64 as the member kernel forms it: whether a collinear pair's
            // cosine rounds to -1 decides if its triplet counts below
            const T rinvijik = std::is_same<T, double>::value ? T(1) / (gj.w * gk.w) : rij * rik;
            const T cost = (gj.x * gk.x + gj.y * gk.y + gj.z * gk.z) * rinvijik;
            T th, dacos;
            if constexpr (std::is_same<T, double>::value) {
                // the angular functions vanish at 0 and 180 degrees
                if (cost <= T(-1) || cost >= T(1)) continue;
                th = acos(cost);
                dacos = T(-1) / sqrt(T(1) - cost * cost);
            } else {
                // FP32: the angle from the sine (cross product) and cosine,
                // accurate at both ends where acos(cos) is not
                const T cx = gj.y * gk.z - gj.z * gk.y;
                const T cy = gj.z * gk.x - gj.x * gk.z;
                const T cz = gj.x * gk.y - gj.y * gk.x;
                const T sint = sqrt(cx * cx + cy * cy + cz * cz) * rinvijik;
                if (!(sint > T(0))) continue;
                th = atan2f(sint, cost);
                dacos = T(-1) / sint;
            }
            const T z = wt ? (T)(M->Zel[el[j]] * M->Zel[el[k]]) : T(1);
            T A[kCompV], dA[kCompV];
#pragma unroll
            for (int v = 0; v < kCompV; ++v) {
                A[v] = dA[v] = T(0);
                if (v < V) {
                    const V4 w = aw[v];
                    window_fdf<POLY2>(POLY2 ? 2 : C.ang[v].core, false, w.x, w.y, th, A[v], dA[v]);
                    A[v] *= z;
                    dA[v] *= dacos * z;
                }
            }
            T Rk[RW], dRk[DER ? RW : 1];
            load_row(R + k * RW, Rk);
            if constexpr (DER) load_row(dR + k * RW, dRk);
            if constexpr (FORCE) {
                T X = T(0), Y1 = T(0), Y2 = T(0);
#pragma unroll
                for (int u = 0; u < kCompU; ++u)
                    if (u < U) {
                        T au = T(0), bu = T(0);
#pragma unroll
                        for (int v = 0; v < kCompV; ++v) {
                            const T w = FLOATW ? wr[u * kCompV + v] : wl[u * kCompV + v];
                            au += w * A[v];
                            bu += w * dA[v];
                        }
                        X += Rj[u] * Rk[u] * bu;
                        Y1 += dRj[u] * Rk[u] * au;
                        Y2 += Rj[u] * dRk[u] * au;
                    }
                // P1 r_ij + P2 r_ik on the atom, P1 r_ij + P3 r_jk on j,
                // P2 r_ik - P3 r_jk on k (r_jk = r_ik - r_ij)
                const T P3 = rinvijik * X;
                const T P1 = rij * (rik - rij * cost) * X + rij * Y1;
                const T P2 = rik * (rij - rik * cost) * X + rik * Y2;
                const T d1 = P1 - P3, d2 = P2 - P3;
                sx += (double)(P1 * gj.x + P2 * gk.x);
                sy += (double)(P1 * gj.y + P2 * gk.y);
                sz += (double)(P1 * gj.z + P2 * gk.z);
                hx += (double)(d1 * gj.x + P3 * gk.x);
                hy += (double)(d1 * gj.y + P3 * gk.y);
                hz += (double)(d1 * gj.z + P3 * gk.z);
                lds_add(ax + k, (double)(d2 * gk.x + P3 * gj.x));
                lds_add(ax + capL + k, (double)(d2 * gk.y + P3 * gj.y));
                lds_add(ax + 2 * capL + k, (double)(d2 * gk.z + P3 * gj.z));
            } else if constexpr (TANGENT) {
                const T wkx = (T)ax[k], wky = (T)ax[capL + k], wkz = (T)ax[2 * capL + k];
                const T a1 = gj.x * wjx + gj.y * wjy + gj.z * wjz;
                const T a2 = gk.x * wkx + gk.y * wky + gk.z * wkz;
                const T a3 = (gk.x - gj.x) * (wjx - wkx) + (gk.y - gj.y) * (wjy - wky) + (gk.z - gj.z) * (wjz - wkz);
                const T D = rij * (rik - rij * cost) * a1 + rik * (rij - rik * cost) * a2 + rinvijik * a3;
                const T y1 = rij * a1, y2 = rik * a2;
#pragma unroll
                for (int u = 0; u < kCompU; ++u)
                    if (u < U) {
                        const double x = (double)(Rj[u] * Rk[u] * D);
                        const double y = (double)(dRj[u] * Rk[u] * y1 + Rj[u] * dRk[u] * y2);
#pragma unroll
                        for (int v = 0; v < kCompV; ++v)
                            acc[u * kCompV + v] -= x * (double)dA[v] + y * (double)A[v];
                    }
            } else {
#pragma unroll
                for (int u = 0; u < kCompU; ++u)
                    if (u < U) {
                        const double p = (double)(Rj[u] * Rk[u]);
#pragma unroll
                        for (int v = 0; v < kCompV; ++v) acc[u * kCompV + v] += p * (double)A[v];
                    }
            }
        }
        flush();
        if constexpr (!FORCE) {
            // lane l of each wave holds cell (bits of l reversed); the waves' sums in order
            red[wv * kWave + (int)(__brev((unsigned)lane) >> 26)] = reduce_cells<32>(acc);
            __syncthreads();
            if (tid < kCells && C.cell[tid] >= 0) {
                double v = 0.0;
#pragma unroll
                for (int w = 0; w < kFW; ++w) v += red[w * kWave + tid];
                put(M->mem[G.mem0 + C.cell[tid]], v);
            }
        }
        __syncthreads();
    }

    if constexpr (FORCE) {
        // the atom's own force, then its neighbours' (the pull form drops
        // the atom's own periodic images, Mode.cpp:1957)
        fx = wave_sum(fx);
        fy = wave_sum(fy);
        fz = wave_sum(fz);
        if (lane == 0) {
            red[wv * 3] = fx;
            red[wv * 3 + 1] = fy;
            red[wv * 3 + 2] = fz;
        }
        __syncthreads();
        if (tid < 3) {
            double v = 0.0;
#pragma unroll
            for (int w = 0; w < kFW; ++w) v += red[w * 3 + tid];
            atomicAdd(c.F + 3 * (size_t)i + tid, v);
        }
        for (int k = tid; k < n; k += kFT) {
            const int j = s.nb_j[ebase + idx[k]];
            if (j == i && !c.push) continue;
            atomicAdd(c.F + 3 * (size_t)j, ax[k]);
            atomicAdd(c.F + 3 * (size_t)j + 1, ax[capL + k]);
            atomicAdd(c.F + 3 * (size_t)j + 2, ax[2 * capL + k]);
        }
    }
}

}  // namespace

template <typename T>
bool sfcomp_factored_fits(CompMode mode, int capL)
{
    return fac_bytes<T>(capL, mode != CM_VALUES) <= kFLds;
}

template <typename T>
void launch_sfcomp_factored(const ModelT* m, const ModelT& hm, const SysView& s, const CompMix& c, CompMode mode,
                            int capL, hipStream_t stream)
{
    if (s.natoms == 0 || !hm.has_comp) return;
    const size_t lds = fac_bytes<T>(capL, mode != CM_VALUES);
    const dim3 grid(s.natoms), block(kFT);
    auto launch = [&](auto md) {
        constexpr int MD = decltype(md)::value;
        if (hm.fac_poly2) hipLaunchKernelGGL((k_sfcomp_fac<T, MD, true>), grid, block, lds, stream, m, s, c, capL);
        else hipLaunchKernelGGL((k_sfcomp_fac<T, MD, false>), grid, block, lds, stream, m, s, c, capL);
    };
    switch (mode) {
    case CM_VALUES: launch(std::integral_constant<int, CM_VALUES>{}); break;
    case CM_FORCE: launch(std::integral_constant<int, CM_FORCE>{}); break;
    case CM_TANGENT: launch(std::integral_constant<int, CM_TANGENT>{}); break;
    default: throw Error{NNPX_ERR_STATE, "the factored compact kernel does not store dG/dr"};
    }
}

template bool sfcomp_factored_fits<float>(CompMode, int);
template bool sfcomp_factored_fits<double>(CompMode, int);
template void launch_sfcomp_factored<float>(const ModelT*, const ModelT&, const SysView&, const CompMix&, CompMode, int,
                                            hipStream_t);
template void launch_sfcomp_factored<double>(const ModelT*, const ModelT&, const SysView&, const CompMix&, CompMode,
                                             int, hipStream_t);

}  // namespace nnpx
