// FP64 fused force backward of the plain form.
//
// The forces Mode::calculateForces computes from the stored Atom::dGdr and
// Atom::Neighbor::dGdr (Mode.cpp:1922-1984, Atom.cpp:371-401), without
// storing them: every radial pair term and angular triplet term of
// SymGrpExpRad::calculate / SymGrpExpAngn::calculate (SymGrpExpRad.cpp:
// 144-239, SymGrpExpAngn.cpp:156-403, and the wide and element-weighted
// groups SymGrpExpAngw.cpp:156-380, SymGrpExpRadWeighted.cpp:137-231,
// SymGrpExpAngnWeighted.cpp:165-395) is recomputed in FP64 and contracted on
// the fly with w = dE/dG times the member's derivative scale (angular
// 2^(1-zeta) times the scaling factor, radial the scaling factor).  Per
// triplet the members reduce to three sums, A = sum u zeta lambda,
// B = sum u (1 + lambda cos), C = sum u 2 eta (1 + lambda cos) with
// u = w exp(...) (1 + lambda cos)^(zeta-1), which give the reference's
// p1, p2, p3 summed over the members:
//   P1 = pfc (A (1/(rij rik) - cos/rij^2) - C) + B pr1
//   P2 = pfc (A (1/(rij rik) - cos/rik^2) - C) + B pr2
//   P3 = pfc (A /(rij rik) + C) - B pr3
// (shifted and weighted members carry (r - rs)/r factors into C per
// distance), and the atom receives -(P1 r_ij + P2 r_ik), neighbour j
// +(P1 r_ij + P3 r_jk), neighbour k +(P2 r_ik - P3 r_jk).
//
// Mapping: W waves per atom (one block), neighbour geometry and cutoff values
// staged once in LDS in FP64 for all of them.  Radial groups: threads own
// neighbours (force) or waves own members (values, tangent).  Angular groups:
// the group's neighbour pairs are walked in row x column blocks, each wave
// taking every W-th block of rows; a wave tests (r_jk^2 < rc^2 in FP64),
// compacts the passing pairs in its own LDS buffer and each lane takes a
// contiguous chunk of it, so it sees runs of one first atom j: j's geometry
// and its force contribution stay in registers over the run, the atom's own
// contribution too, and only partner k's goes through an LDS FP64 atomic.
// Neighbour sums are pushed to the force array with FP64 device atomics;
// the pull form drops the atom's own periodic images (Mode.cpp:1957).
//
// Bound by FP64 instruction issue (75% of the time in the values, 58% in the
// forces), which wants four waves per SIMD: one wave per atom left 2.1 and 1.8
// (its 12 KB of staging fills the LDS first), two that share it 4.2 and 3.3; the
// registers allow five and four once the other cutoff types' code and the
// series' coefficients are out of the walks (cutoff_fdf64, in_place; the forces
// still spill 34 at their 128).  Water of 12,288 atoms, two eta, 30 angular
// functions per element: values 506 -> 368 us, forces 665 -> 580 us between the
// bench line's markers (with four waves the forces take 40% more: the waves'
// last buffers are filled less).  5,100 atoms: the tangent 255 us and 212 us of
// values where storing dG/dr took 2,694 us and its tangent 152 us.
#include <string>
#include <type_traits>

#include "kernels.hpp"
#include "mixed.hpp"
#include "nnpx.h"
#include "stage.hpp"

namespace nnpx {
namespace {

// Pairs in a wave's buffer, fewer where LDS is short (water, 12,288 atoms,
// kernel trace: values 355 us at 256 pairs, 377 at 384; forces 553, 551).
constexpr int kWalk64 = 256;
constexpr int kMinWalk64 = 128;  // ... at least
constexpr size_t kLds64 = 65536;
// Atoms up to which four waves share one, else two: 4,096 atoms give every SIMD
// eight waves of two per atom.  1,300 atoms: four waves 88 + 128 us (values,
// forces), 192 atoms likewise bound by one atom's time; 5,100 atoms: two waves
// 211 + 297 us, four 215 + 383.
constexpr int kFew64 = 4096;

struct Stage64 {
    double4* g;          // x, y, z, |dr|
    double4* c;          // 1/|dr|, fc, dfc (current group's cutoff), atomic number
    double* ax;          // [capL] force sums per neighbour entry (force), u_i - u_j (tangent)
    double* ay;
    double* az;
    unsigned* tjk;       // this wave's compacted pairs (j | k << 16)
    int* cnt;            // [kStagePasses][kMaxElem] staging counts (before the walks, in the waves' pair buffers)
    unsigned short* la;  // group lists
    unsigned short* lb;
    unsigned char* el;   // neighbour element
    unsigned short* idx; // list entry of each staged slot
    int* eoff;           // [kMaxElem + 1] first staged slot of each neighbour element
    double* red;         // [W][32] per-wave sums, or the power path's term weights
    int walk;            // pairs a wave's buffer takes
};

// A group's neighbour list: staged slots base .. base + n - 1 (contig: the
// group's cutoff covers every staged neighbour of its element) or the n
// slots listed in S.la / S.lb.
struct List64 {
    int base, n;
    bool contig;
};

template <bool CONTIG>
__device__ inline int slot64(const unsigned short* l, int base, int a)
{
    if constexpr (CONTIG) return base + a;
    else return l[a];
}

constexpr int kRed64 = 32;  // per-wave sums (members of a group, or its terms)

__host__ __device__ constexpr size_t stage64_bytes(int capL, int waves, int walk)
{
    return (size_t)waves * kRed64 * 8 + (size_t)capL * (32 + 32 + 24 + 2 + 2 + 1 + 2) +
           (size_t)waves * (walk + kWave) * 4 + 48;
}

template <int W>
__device__ inline Stage64 carve64(double4* base, int capL, int walk)
{
    Stage64 S;
    S.walk = walk;
    S.red = reinterpret_cast<double*>(base);
    S.g = reinterpret_cast<double4*>(S.red + W * kRed64);
    S.c = S.g + capL;
    S.ax = reinterpret_cast<double*>(S.c + capL);
    S.ay = S.ax + capL;
    S.az = S.ay + capL;
    unsigned* t = reinterpret_cast<unsigned*>(S.az + capL);
    S.cnt = reinterpret_cast<int*>(t);
    S.tjk = t + wave_id() * (walk + kWave);
    S.la = reinterpret_cast<unsigned short*>(t + W * (walk + kWave));
    S.lb = S.la + capL;
    S.el = reinterpret_cast<unsigned char*>(S.lb + capL);
    S.idx = reinterpret_cast<unsigned short*>(S.el + capL);
    S.eoff = reinterpret_cast<int*>(S.idx + capL);
    return S;
}

// Stages the atom's in-cutoff list entries (stage_by_element): geometry, each
// slot's list entry in idx and, for the force kernel, zeroed neighbour force
// sums.
template <int W>
__device__ inline int stage64(const ModelT* __restrict__ M, const SysView& s, int i, int capL, const Stage64& S,
                              bool zero_sums)
{
    return stage_by_element<W>(M, s, i, capL, S.cnt, S.eoff, [&](int pos, int k, const double* dr, double d, int el) {
        S.g[pos] = make_double4(dr[0], dr[1], dr[2], d);
        S.c[pos] = make_double4(1.0 / d, 0.0, 0.0, M->Zel[el]);
        S.el[pos] = (unsigned char)el;
        S.idx[pos] = (unsigned short)k;
        if (zero_sums) {
            S.ax[pos] = 0.0;
            S.ay[pos] = 0.0;
            S.az[pos] = 0.0;
        }
    });
}

// sqrt(x) and 1/sqrt(x): the hardware's reciprocal square root (about 2^-28)
// refined by one coupled Goldschmidt step and a residual correction of each,
// half the instructions of sqrt and a division and as close (at most 0.50 and
// 1.47 ulp on 2^20 arguments).  x = 0 gives 0 and infinity.
__device__ inline void root64(double x, double& r, double& ri)
{
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double e = fma(-h, g, 0.5);
    g = fma(g, e, g);
    h = fma(h, e, h);
    g = fma(fma(-g, g, x), h, g);
    h += h;
    h = fma(h, fma(-g, h, 1.0), h);
    const bool zero = !(x > 0.0);
    r = zero ? 0.0 : g;
    ri = zero ? y : h;
}

// A constant made in scalar registers where it is used: kept over a walk, the
// series' coefficients would take 70 vector registers and a wave per SIMD.
__device__ inline double in_place(double c)
{
    asm volatile("" : "+s"(c));
    return c;
}

// exp(x) for x <= 0: x = k ln 2 + f with |f| <= ln 2 / 2 (ln 2 in two parts),
// the power series of exp(f) to f^13 (remainder 4e-18), times 2^k.  At most 0.86
// ulp off on 2^20 arguments (exp: 0.85).
__device__ inline double exp_neg64(double x)
{
    x = fmax(x, -800.0);
    const double k = rint(x * in_place(1.4426950408889634));
    double f = fma(-k, in_place(0.6931471805599453), x);
    f = fma(-k, in_place(2.3190468138462996e-17), f);
    double p = in_place(1.0 / 6227020800.0);
    p = fma(p, f, in_place(1.0 / 479001600.0));
    p = fma(p, f, in_place(1.0 / 39916800.0));
    p = fma(p, f, in_place(1.0 / 3628800.0));
    p = fma(p, f, in_place(1.0 / 362880.0));
    p = fma(p, f, in_place(1.0 / 40320.0));
    p = fma(p, f, in_place(1.0 / 5040.0));
    p = fma(p, f, in_place(1.0 / 720.0));
    p = fma(p, f, in_place(1.0 / 120.0));
    p = fma(p, f, in_place(1.0 / 24.0));
    p = fma(p, f, in_place(1.0 / 6.0));
    p = fma(p, f, 0.5);
    p = fma(p, f, 1.0);
    p = fma(p, f, 1.0);
    return ldexp(p, (int)k);
}

// cos(pi x) and sin(pi x) for x in [0, 1): with t = x - 1/2 they are
// -sin(pi t) and cos(pi t), |t| <= 1/2, from their power series (coefficients
// pi^n / n!; remainders below 2e-18).  At most 2.8 and 3.0 x 2^-53 off on 2^20
// arguments (sincospi 0.86): a cutoff value is 1.4 x 2^-53 off, from cos(M_PI x)
// 1.5.  The series on quarters of the range are 0.8 off, cost the values 9% and
// the forces 4% (12,288 atoms) and do not bring results nearer to 64-bit references.
__device__ inline void cossin_pi64(double x, double& cs, double& sn)
{
    const double t = x - 0.5, u = t * t;
    double a = in_place(5.392664662608129e-10);  // pi^21 / 21!
    a = fma(a, u, in_place(-2.2948428997269873e-08));
    a = fma(a, u, in_place(7.952054001475513e-07));
    a = fma(a, u, in_place(-2.1915353447830217e-05));
    a = fma(a, u, in_place(0.00046630280576761255));
    a = fma(a, u, in_place(-0.0073704309457143504));
    a = fma(a, u, in_place(0.08214588661112823));
    a = fma(a, u, in_place(-0.5992645293207921));
    a = fma(a, u, in_place(2.5501640398773455));
    a = fma(a, u, in_place(-5.16771278004997));
    a = fma(a, u, in_place(3.141592653589793));
    cs = -a * t;
    double b = in_place(-7.700707130601354e-11);  // -pi^22 / 22!
    b = fma(b, u, in_place(3.604730797462501e-09));
    b = fma(b, u, in_place(-1.3878952462213771e-07));
    b = fma(b, u, in_place(4.303069587032947e-06));
    b = fma(b, u, in_place(-0.0001046381049248457));
    b = fma(b, u, in_place(0.0019295743094039231));
    b = fma(b, u, in_place(-0.02580689139001406));
    b = fma(b, u, in_place(0.2353306303588932));
    b = fma(b, u, in_place(-1.3352627688545895));
    b = fma(b, u, in_place(4.0587121264167685));
    b = fma(b, u, in_place(-4.934802200544679));
    sn = fma(b, u, 1.0);
}

// Cutoff value and derivative; the cosine cutoff through cossin_pi64, the
// others as CutoffFunction::fdf.  COS: the model's cutoff is the cosine one
// (the others' code, never run, would cost the walks 20 registers).
template <bool COS>
__device__ inline void cutoff_fdf64(int type, const GroupT& g, double tanhPre, double r, double& fc, double& dfc)
{
    if (COS || type == 1) {
        const double x = fmin(fmax((r - g.rci) * g.iw, 0.0), 1.0);
        double sn, cs;
        cossin_pi64(x, cs, sn);
        const bool in = r < g.rc, flat = r < g.rci;
        fc = in ? flat ? 1.0 : 0.5 * (cs + 1.0) : 0.0;
        dfc = in && !flat ? -0.5 * g.iw * M_PI * sn : 0.0;
        return;
    }
    cutoff_fdf(type, g, tanhPre, r, fc, dfc);
}

// Cutoffs of the staged neighbours for one group (every slot when all the
// element's groups share one radius).  Ends with a barrier.
template <int W, bool COS>
__device__ inline void stage_cutoffs64(const Stage64& S, int n, int ctype, const GroupT& G, bool every, double tanhPre)
{
    for (int k = threadIdx.x; k < n; k += W * kWave) {
        double f = 0.0, df = 0.0;
        const int ek = S.el[k];
        if ((every || ek == G.e1 || ek == G.e2) && S.g[k].w < G.rc)
            cutoff_fdf64<COS>(ctype, G, tanhPre, S.g[k].w, f, df);
        S.c[k].y = f;
        S.c[k].z = df;
    }
    __syncthreads();
}

// Neighbours of element `elem` (all elements: elem < 0) inside the group's
// cutoff: the element's slot range when the group's cutoff is the model's
// largest, else the qualifying slots listed in `out` (by the first wave).
// Ends with a barrier.
template <int W>
__device__ inline List64 make_list64(const ModelT* __restrict__ M, const Stage64& S, int n, const GroupT& G, int elem,
                                     unsigned short* out)
{
    const int lane = lane_id();
    const int lo = __builtin_amdgcn_readfirstlane(elem < 0 ? 0 : S.eoff[elem]);
    const int hi = __builtin_amdgcn_readfirstlane(elem < 0 ? n : S.eoff[elem + 1]);
    List64 L{lo, hi - lo, true};
    if (!(G.rc >= M->maxCutoff)) {
        int cnt = 0;
        for (int b = lo; b < hi; b += kWave) {
            const int k = b + lane;
            const unsigned long long m = __ballot(k < hi && S.g[k].w < G.rc);
            if (wave_id() == 0 && (m >> lane) & 1)
                out[cnt + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                         __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u))] =
                    (unsigned short)k;
            cnt += __popcll(m);
        }
        L = List64{0, __builtin_amdgcn_readfirstlane(cnt), false};
    }
    __syncthreads();
    return L;
}

// Calls work(j, k) for every unordered pair of the group's lists with
// r_jk^2 < rc2 (like elements: row a pairs with b = a + c + 1 mod nA,
// c < (nA - 1) / 2, plus b = a + nA / 2 for even nA on rows a < nA / 2;
// unlike elements: the full product).  A step tests a block of rows x columns
// (lane = row * width + column), the row's geometry staying in registers; wave
// w takes the row blocks w, w + W, ...  The passing pairs are compacted in
// block order and run in buffers of S.walk, the pairs past a full buffer being
// carried over; flush() after each buffer.  Waves do not wait for each other.
template <int W, bool CONTIG, typename Work, typename Flush>
__device__ inline void triplets64(const Stage64& S, const List64& A, const List64& B, bool same, double rc2,
                                 Work&& work, Flush&& flush)
{
    const int lane = lane_id();
    const int nA = A.n, nB = B.n;
    const int R = same ? (nA - 1) / 2 : nB;          // regular columns per row
    const int Rx = same && nA % 2 == 0 ? R + 1 : R;  // with the half-way column (rows a < nA / 2 only)
    const int half = nA / 2;
    if (nA == 0 || Rx == 0) return;
    const int nblk = (Rx + 7) >> 3;
    const int cw = (Rx + nblk - 1) / nblk, rh = kWave / cw;
    const int lr = lane / cw, lc = lane - lr * cw;  // lanes with lr >= rh stay idle
    const bool live = lr < rh;
    const unsigned short* lb = same ? S.la : S.lb;
    const int bB = same ? A.base : B.base;
    int a0 = wave_id() * rh, c0 = 0;
    int ja = 0;
    double gx = 0.0, gy = 0.0, gz = 0.0;
    auto row = [&] {
        const int a = a0 + lr;
        ja = slot64<CONTIG>(S.la, A.base, a < nA ? a : 0);
        const double4 g = S.g[ja];
        gx = g.x;
        gy = g.y;
        gz = g.z;
    };
    row();
    int cnt = 0;
    for (;;) {
        while (a0 < nA && cnt < S.walk) {
            // lanes outside the block test column 0 and fail
            const int a = a0 + lr, c = c0 + lc;
            const bool valid = live && a < nA && c < Rx && (c < R || a < half);
            int b = same ? a + c + 1 : c;
            b = same && b >= nA ? b - nA : b;
            b = valid ? b : 0;
            const int k = slot64<CONTIG>(lb, bB, b);
            const double dx = S.g[k].x - gx, dy = S.g[k].y - gy, dz = S.g[k].z - gz;
            const bool ok = valid & (dx * dx + dy * dy + dz * dz < rc2);
            const unsigned long long m = __ballot(ok);
            if (ok)
                S.tjk[cnt + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                           __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u))] =
                    (unsigned)ja | ((unsigned)k << 16);
            cnt += __popcll(m);
            c0 += cw;
            if (c0 >= Rx) {
                c0 = 0;
                a0 += W * rh;
                row();
            }
        }
        const int m = min(cnt, S.walk);
        if (m <= 0) break;
        wave_fence();
        const int per = (m + kWave - 1) / kWave;
        const int x0 = lane * per, x1 = min(m, x0 + per);
        for (int x = x0; x < x1; ++x) {
            const unsigned jk = S.tjk[x];
            work((int)(jk & 0xffffu), (int)(jk >> 16));
        }
        flush();
        wave_fence();
        const int rest = cnt - m;
        if (lane < rest) S.tjk[lane] = S.tjk[S.walk + lane];
        cnt = rest;
        wave_fence();
    }
}

template <int W, typename Work, typename Flush>
__device__ inline void for_each_triplet64(const Stage64& S, const List64& A, const List64& B, bool same, double rc2,
                                          Work&& work, Flush&& flush)
{
    if (A.contig) triplets64<W, true>(S, A, B, same, rc2, work, flush);
    else triplets64<W, false>(S, A, B, same, rc2, work, flush);
}

// Geometry of one triplet: what every term needs.
struct Trip64 {
    double4 gj, gk, cj, ck;
    double x3, y3, z3, rjk, ijk, fcjk, dfcjk, rinvijik, cost, zw, r2sum;
};

template <bool COS>
__device__ inline void triplet_geometry(Trip64& t, const double4& gj, const double4& cj, const double4& gk,
                                        const double4& ck, bool wide, bool wt, int ctype, const GroupT& G,
                                        double tanhPre)
{
    t.gj = gj;
    t.gk = gk;
    t.cj = cj;
    t.ck = ck;
    t.x3 = gk.x - gj.x;
    t.y3 = gk.y - gj.y;
    t.z3 = gk.z - gj.z;
    const double r2jk = t.x3 * t.x3 + t.y3 * t.y3 + t.z3 * t.z3;
    t.rjk = 0.0;
    t.ijk = 0.0;
    t.fcjk = 1.0;
    t.dfcjk = 0.0;
    if (!wide) {
        root64(r2jk, t.rjk, t.ijk);
        cutoff_fdf64<COS>(ctype, G, tanhPre, t.rjk, t.fcjk, t.dfcjk);
    }
    t.rinvijik = cj.x * ck.x;
    t.cost = (gj.x * gk.x + gj.y * gk.y + gj.z * gk.z) * t.rinvijik;
    t.zw = wt ? cj.w * ck.w : 1.0;
    t.r2sum = gj.w * gj.w + gk.w * gk.w + (wide ? 0.0 : r2jk);
}

// Exponential of a member (shared by members of equal eta and rs): updates
// vexp and, for shifted or weighted members, the (r - rs)/r factors.
struct Exp64 {
    double vexp = 0.0, fij = 0.0, fik = 0.0, fjk = 0.0;
    bool shifted = false;
};

__device__ inline void member_exp(Exp64& x, const MemberT& mb, const Trip64& t, bool wide, bool wt)
{
    if (!mb.calcExp) return;
    x.shifted = mb.rs > 0.0 || wt;
    if (x.shifted) {
        const double a = t.gj.w - mb.rs, b = t.gk.w - mb.rs, c = t.rjk - mb.rs;
        x.vexp = exp_neg64(-mb.eta * (a * a + b * b + (wide ? 0.0 : c * c)));
        x.fij = a * t.cj.x;
        x.fik = b * t.ck.x;
        x.fjk = wide ? 0.0 : c * t.ijk;
    } else {
        x.vexp = exp_neg64(-mb.eta * t.r2sum);
    }
}

// NB0 > 0: the power path (angular groups whose members are
// exp(-eta_h sum r^2) (1 + lambda_s cos)^(2^b), b < NB0 resp. NB1, rs = 0):
// per triplet one exponential per eta and the powers by repeated squaring;
// the members' weights are folded per term (wb = sum w, wa = sum zeta lambda
// w), and (1 + lambda cos)^(2^b - 1) is carried beside the power so A needs
// no division.
template <int W, int MAXM, int NB0, int NB1, bool COS>
__global__ __launch_bounds__(kWave * W) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_force64f(const ModelT* __restrict__ M, const MemberF* __restrict__ MF,
                                                         const GroupPow64* __restrict__ GP, SysView s,
                                                         const double* __restrict__ fw, int ldG,
                                                         double* __restrict__ F, int push, int capL, int walk)
{
    extern __shared__ double4 sm64[];
    const Stage64 S = carve64<W>(sm64, capL, walk);
    const int i = blockIdx.x;
    const int lane = lane_id();
    const int e = s.elem[i];
    const ElementT& E = M->el[e];
    const int ctype = M->cutoffType;
    const double tanhPre = M->tanhPre;
    const int n = stage64<W>(M, s, i, capL, S, true);
    const size_t base = (size_t)i * s.cap;
    const double* wi = fw + (size_t)i * ldG;
    double fx = 0.0, fy = 0.0, fz = 0.0;
    bool cut_done = false;  // the cutoffs of a uniform-cutoff element are staged

    for (int gi = 0; gi < E.ngrp; ++gi) {
        const GroupT& G = M->grp[E.grp0 + gi];
        const int type = G.type;
        if (type != 2 && type != 12 && type != 3 && type != 9 && type != 13) continue;  // compact: k_sfcomp
        const bool radial = type == 2 || type == 12;
        const bool wt = type == 12 || type == 13;
        if (!E.ucut || !cut_done) stage_cutoffs64<W, COS>(S, n, ctype, G, E.ucut || wt, tanhPre);
        cut_done = true;
        const int nmem = G.nmem;
        const MemberT* mem = M->mem + G.mem0;
        if (radial) {
            // threads own neighbours: sum_q w_q sfac_q (dfc - 2 eta (r - rs) fc) exp(-eta (r - rs)^2);
            // type 2: the slots of element e1, type 12: every slot
            const int lo = wt ? 0 : S.eoff[G.e1], hi = wt ? n : S.eoff[G.e1 + 1];
            for (int k = lo + threadIdx.x; k < hi; k += W * kWave) {
                const double4 gk = S.g[k];
                if (!(gk.w < G.rc)) continue;
                const double4 ck = S.c[k];
                double P = 0.0;
                for (int q = 0; q < nmem; ++q) {
                    const MemberT& mb = mem[q];
                    const double dr = gk.w - mb.rs;
                    P += wi[mb.sf] * (ck.z - 2.0 * mb.eta * dr * ck.y) * exp_neg64(-mb.eta * dr * dr);
                }
                P *= wt ? ck.x * ck.w : ck.x;
                const double px = P * gk.x, py = P * gk.y, pz = P * gk.z;
                fx -= px; fy -= py; fz -= pz;
                S.ax[k] += px; S.ay[k] += py; S.az[k] += pz;
            }
            __syncthreads();
            continue;
        }
        const bool same = G.e1 == G.e2;
        const bool wide = type == 9;
        const List64 A = make_list64<W>(M, S, n, G, G.e1, S.la);
        const List64 B = same ? A : make_list64<W>(M, S, n, G, G.e2, S.lb);
        GroupPow64 gp{};
        double2* pw = reinterpret_cast<double2*>(S.red);
        if constexpr (NB0 > 0) {
            gp = GP[E.grp0 + gi];
            // term weights: wb = sum of the members' w, wa = sum of zeta lambda w
            if (threadIdx.x < 2 * (NB0 + NB1)) {
                double sb = 0.0, sa = 0.0;
                for (int q = 0; q < nmem; ++q)
                    if (MF[G.mem0 + q].beta == lane) {
                        const double wq = wi[mem[q].sf];
                        sb += wq;
                        sa += wq * mem[q].zetaLambda;
                    }
                pw[lane] = make_double2(sb, sa);
            }
            __syncthreads();
        }
        int cur = -1;
        double rx = 0.0, ry = 0.0, rz = 0.0, sx = 0.0, sy = 0.0, sz = 0.0;
        double4 gj = make_double4(0.0, 0.0, 0.0, 0.0), cj = gj;
        auto flush = [&]() {
            if (cur >= 0) {
                lds_add(S.ax + cur, rx);
                lds_add(S.ay + cur, ry);
                lds_add(S.az + cur, rz);
                fx -= sx;
                fy -= sy;
                fz -= sz;
                cur = -1;
            }
        };
        for_each_triplet64<W>(S, A, B, same, wide ? INFINITY : G.rc2, [&](int j, int k) {
            if (j != cur) {
                flush();
                cur = j;
                rx = 0.0; ry = 0.0; rz = 0.0;
                sx = 0.0; sy = 0.0; sz = 0.0;
                gj = S.g[j];
                cj = S.c[j];
            }
            Trip64 t;
            triplet_geometry<COS>(t, gj, cj, S.g[k], S.c[k], wide, wt, ctype, G, tanhPre);
            const double4 &gk = t.gk, &ck = t.ck;
            const double cost = t.cost, rinvijik = t.rinvijik;
            const double pfc = t.zw * cj.y * ck.y * t.fcjk;
            const double pr1 = t.zw * ck.y * t.fcjk * cj.z * cj.x;
            const double pr2 = t.zw * cj.y * t.fcjk * ck.z * ck.x;
            const double pr3 = t.zw * cj.y * ck.y * t.dfcjk * t.ijk;
            double A = 0.0, B = 0.0, C0 = 0.0, C1 = 0.0, C2 = 0.0, C3 = 0.0;
            if constexpr (NB0 > 0) {
                constexpr int NBM = NB0 > NB1 ? NB0 : NB1;
                const double E0 = exp_neg64(-gp.eta[0] * t.r2sum);
                const double E1 = NB1 > 0 ? exp_neg64(-gp.eta[1] * t.r2sum) : 0.0;
                double Q0 = 0.0, Q1 = 0.0;
#pragma unroll
                for (int sl = 0; sl < 2; ++sl) {
                    const double pl = 1.0 + gp.lam[sl] * cost;
                    const bool pos = pl > 0.0;
                    double pp = pos ? pl : 0.0;   // pl^(2^b)
                    double qq = pos ? 1.0 : 0.0;  // pl^(2^b - 1)
                    double qa0 = 0.0, qa1 = 0.0;
#pragma unroll
                    for (int b = 0; b < NBM; ++b) {
                        if (b < NB0) {
                            const double2 wv = pw[sl * NB0 + b];
                            Q0 += wv.x * pp;
                            qa0 += wv.y * qq;
                        }
                        if (b < NB1) {
                            const double2 wv = pw[2 * NB0 + sl * NB1 + b];
                            Q1 += wv.x * pp;
                            qa1 += wv.y * qq;
                        }
                        qq *= pp;
                        pp *= pp;
                    }
                    A += E0 * qa0 + E1 * qa1;
                }
                const double B0 = E0 * Q0, B1 = E1 * Q1;
                B = B0 + B1;
                C0 = gp.twoEta[0] * B0 + gp.twoEta[1] * B1;
            } else {
                Exp64 x;
#pragma unroll
                for (int q = 0; q < MAXM; ++q) {
                    if (q < nmem) {
                        const MemberT& mb = mem[q];
                        member_exp(x, mb, t, wide, wt);
                        const double pl = 1.0 + mb.lambda * cost;
                        if (pl > 0.0) {
                            const double pw = mb.useIntPow ? pow_int(pl, mb.zetaInt - 1) : pow(pl, mb.zeta - 1.0);
                            const double u = wi[mb.sf] * x.vexp * pw;
                            A += u * mb.zetaLambda;
                            const double v = u * pl;
                            B += v;
                            const double c2 = 2.0 * mb.eta * v;
                            if (x.shifted) {
                                C1 += c2 * x.fij;
                                C2 += c2 * x.fik;
                                C3 += c2 * x.fjk;
                            } else {
                                C0 += c2;
                            }
                        }
                    }
                }
            }
            C1 += C0;
            C2 += C0;
            C3 += C0;
            const double P1 = pfc * (A * (rinvijik - cost * cj.x * cj.x) - C1) + B * pr1;
            const double P2 = pfc * (A * (rinvijik - cost * ck.x * ck.x) - C2) + B * pr2;
            const double P3 = wide ? pfc * A * rinvijik : pfc * (A * rinvijik + C3) - B * pr3;
            const double p1x = P1 * gj.x, p1y = P1 * gj.y, p1z = P1 * gj.z;
            const double p2x = P2 * gk.x, p2y = P2 * gk.y, p2z = P2 * gk.z;
            const double p3x = P3 * t.x3, p3y = P3 * t.y3, p3z = P3 * t.z3;
            sx += p1x + p2x;
            sy += p1y + p2y;
            sz += p1z + p2z;
            rx += p1x + p3x;
            ry += p1y + p3y;
            rz += p1z + p3z;
            lds_add(S.ax + k, p2x - p3x);
            lds_add(S.ay + k, p2y - p3y);
            lds_add(S.az + k, p2z - p3z);
        }, flush);
        flush();
        __syncthreads();
    }
    fx = wave_sum(fx);
    fy = wave_sum(fy);
    fz = wave_sum(fz);
    if (lane == 0) {
        double* r = S.red + wave_id() * 3;
        r[0] = fx;
        r[1] = fy;
        r[2] = fz;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        double v = 0.0;
#pragma unroll
        for (int w = 0; w < W; ++w) v += S.red[w * 3 + threadIdx.x];
        atomicAdd(F + 3 * (size_t)i + threadIdx.x, v);
    }
    for (int k = threadIdx.x; k < n; k += W * kWave) {
        const int j = s.nb_j[base + S.idx[k]];
        if (j == i && !push) continue;
        atomicAdd(F + 3 * (size_t)j, S.ax[k]);
        atomicAdd(F + 3 * (size_t)j + 1, S.ay[k]);
        atomicAdd(F + 3 * (size_t)j + 2, S.az[k]);
    }
}

// Scaled SF values of the plain form (what k_sf64 computes without
// derivatives), or (TANGENT) the derivatives contracted with a field u,
// Gdot = sum_a dG/dx_a . u_a (Training::collectDGdxia, Training.cpp:3586-3625,
// contracted with u; the atom's own images included), on the same staging and
// triplet walk as the force kernel: radial members summed by lanes owning the
// neighbours (waves owning members), angular members per lane over its chunk
// of compacted triplets, one wave reduction per member and wave.  Terms follow
// the reference's expressions (SymGrpExpRad.cpp:190-196, SymGrpExpAngn.cpp:
// 260-300): exp(-eta (r - rs)^2) fc, and vexp (1 + lambda cos)^(zeta - 1)
// (1 + lambda cos) fc_ij fc_ik fc_jk with the exponential shared by members
// of equal (eta, rs).
//   The tangent of a term t = vexp (1 + lambda cos)^zeta fc_ij fc_ik fc_jk
// along the field is, with s1 = r_ij.(u_i - u_j), s2 = r_ik.(u_i - u_k),
// s3 = r_jk.(u_k - u_j) and p = 1 + lambda cos,
//   vexp p^(zeta - 1) (zeta lambda al + p (be + 2 eta ga)),
// al, be, ga being shared by the members (shifted and weighted ones carry their
// (r - rs)/r factors in ga).
template <int W, bool TANGENT, int MAXM, int NB0, int NB1, bool COS>
__global__ __launch_bounds__(kWave * W) void k_values64(const ModelT* __restrict__ M, const MemberF* __restrict__ MF,
                                                         const GroupPow64* __restrict__ GP, SysView s,
                                                         const double* __restrict__ u, const double* __restrict__ fac,
                                                         double* __restrict__ G, int ldG, int capL, int walk)
{
    extern __shared__ double4 sm64[];
    const Stage64 S = carve64<W>(sm64, capL, walk);
    const int i = blockIdx.x;
    const int lane = lane_id(), wv = wave_id();
    const int e = s.elem[i];
    const ElementT& E = M->el[e];
    const int ctype = M->cutoffType;
    const double tanhPre = M->tanhPre;
    const int n = stage64<W>(M, s, i, capL, S, false);
    if constexpr (TANGENT) {
        const double ux = u[3 * (size_t)i], uy = u[3 * (size_t)i + 1], uz = u[3 * (size_t)i + 2];
        for (int k = threadIdx.x; k < n; k += W * kWave) {
            const size_t j = s.nb_j[(size_t)i * s.cap + S.idx[k]];
            S.ax[k] = ux - u[3 * j];
            S.ay[k] = uy - u[3 * j + 1];
            S.az[k] = uz - u[3 * j + 2];
        }
    }
    double* Gi = G + (size_t)i * ldG;
    // member mb's value or tangent from its sum
    auto put = [&](const MemberT& mb, double v, bool angular) {
        if (TANGENT) Gi[mb.sf] = v * fac[e * kMaxSF + mb.sf];
        else Gi[mb.sf] = scale_sf(M->scale[E.sf0 + mb.sf], angular ? v * mb.gnorm : v);
    };
    auto along = [&](const double4& g, int k) { return g.x * S.ax[k] + g.y * S.ay[k] + g.z * S.az[k]; };
    bool cut_done = false;  // the cutoffs of a uniform-cutoff element are staged

    for (int gi = 0; gi < E.ngrp; ++gi) {
        const GroupT& GR = M->grp[E.grp0 + gi];
        const int type = GR.type;
        if (type != 2 && type != 12 && type != 3 && type != 9 && type != 13) continue;  // compact: k_sfcomp
        const bool radial = type == 2 || type == 12;
        const bool wt = type == 12 || type == 13;
        if (!E.ucut || !cut_done) stage_cutoffs64<W, COS>(S, n, ctype, GR, E.ucut || wt, tanhPre);
        cut_done = true;
        const int nmem = GR.nmem;
        const MemberT* mem = M->mem + GR.mem0;
        if (radial) {
            constexpr int CH = W >= 4 ? 3 : 4;  // members per wave and pass
            const int lo = wt ? 0 : S.eoff[GR.e1], hi = wt ? n : S.eoff[GR.e1 + 1];
            for (int q0 = wv * CH; q0 < nmem; q0 += W * CH) {
                double acc[CH];
#pragma unroll
                for (int q = 0; q < CH; ++q) acc[q] = 0.0;
                for (int k = lo + lane; k < hi; k += kWave) {
                    const double4 gk = S.g[k];
                    const double r = gk.w;
                    if (!(r < GR.rc)) continue;
                    const double4 ck = S.c[k];
                    const double sk = TANGENT ? along(gk, k) * (wt ? ck.x * ck.w : ck.x) : 0.0;
#pragma unroll
                    for (int q = 0; q < CH; ++q)
                        if (q0 + q < nmem) {
                            const MemberT& mb = mem[q0 + q];
                            const double dr = r - mb.rs;
                            double pexp = exp_neg64(-mb.eta * dr * dr);
                            if constexpr (TANGENT) {
                                acc[q] += (ck.z - 2.0 * mb.eta * dr * ck.y) * pexp * sk;
                            } else {
                                if (wt) pexp = ck.w * pexp;
                                acc[q] += pexp * ck.y;
                            }
                        }
                }
#pragma unroll
                for (int q = 0; q < CH; ++q)
                    if (q0 + q < nmem) {
                        const double v = wave_sum(acc[q]);
                        if (lane == 0) put(mem[q0 + q], v, false);
                    }
            }
            __syncthreads();
            continue;
        }
        const bool same = GR.e1 == GR.e2;
        const bool wide = type == 9;
        const List64 A = make_list64<W>(M, S, n, GR, GR.e1, S.la);
        const List64 B = same ? A : make_list64<W>(M, S, n, GR, GR.e2, S.lb);
        // the tangent's member-independent factors
        struct Along {
            double s1, s2, s3, al, be, ga, pfc;
        };
        auto tangent = [&](const Trip64& t, int j, int k, double pfc) {
            Along a;
            const double4 &cj = t.cj, &ck = t.ck;
            a.s1 = along(t.gj, j);
            a.s2 = along(t.gk, k);
            a.s3 = t.x3 * (S.ax[j] - S.ax[k]) + t.y3 * (S.ay[j] - S.ay[k]) + t.z3 * (S.az[j] - S.az[k]);
            const double pr1 = t.zw * ck.y * t.fcjk * cj.z * cj.x;
            const double pr2 = t.zw * cj.y * t.fcjk * ck.z * ck.x;
            const double pr3 = t.zw * cj.y * ck.y * t.dfcjk * t.ijk;
            a.al = pfc * ((t.rinvijik - t.cost * cj.x * cj.x) * a.s1 + (t.rinvijik - t.cost * ck.x * ck.x) * a.s2 +
                          t.rinvijik * a.s3);
            a.be = pr1 * a.s1 + pr2 * a.s2 - pr3 * a.s3;
            a.ga = pfc * ((wide ? 0.0 : a.s3) - a.s1 - a.s2);
            a.pfc = pfc;
            return a;
        };
        if constexpr (NB0 > 0) {
            // power path: term sums pfc E_h (1 + lambda_s cos)^(2^b) per lane,
            // one wave reduction per used term, members take their term
            constexpr int NBAS = 2 * (NB0 + NB1);
            constexpr int NBM = NB0 > NB1 ? NB0 : NB1;
            const GroupPow64 gp = GP[E.grp0 + gi];
            double part[NBAS];
#pragma unroll
            for (int b = 0; b < NBAS; ++b) part[b] = 0.0;
            for_each_triplet64<W>(S, A, B, same, wide ? INFINITY : GR.rc2, [&](int j, int k) {
                Trip64 t;
                triplet_geometry<COS>(t, S.g[j], S.c[j], S.g[k], S.c[k], wide, wt, ctype, GR, tanhPre);
                const double pfc = t.zw * t.cj.y * t.ck.y * t.fcjk;
                const double E0 = exp_neg64(-gp.eta[0] * t.r2sum);
                const double E1 = NB1 > 0 ? exp_neg64(-gp.eta[1] * t.r2sum) : 0.0;
                if constexpr (TANGENT) {
                    const Along a = tangent(t, j, k, pfc);
                    const double x0 = E0 * (a.be + gp.twoEta[0] * a.ga), x1 = E1 * (a.be + gp.twoEta[1] * a.ga);
#pragma unroll
                    for (int sl = 0; sl < 2; ++sl) {
                        const double pl = 1.0 + gp.lam[sl] * t.cost;
                        const bool pos = pl > 0.0;
                        double p = pos ? pl : 0.0;   // pl^(2^b)
                        double q = pos ? 1.0 : 0.0;  // pl^(2^b - 1)
                        // zeta lambda E_h al, zeta = 2^b
                        double y0 = E0 * a.al * gp.lam[sl], y1 = E1 * a.al * gp.lam[sl];
#pragma unroll
                        for (int b = 0; b < NBM; ++b) {
                            if (b < NB0) part[sl * NB0 + b] += x0 * p + y0 * q;
                            if (b < NB1) part[2 * NB0 + sl * NB1 + b] += x1 * p + y1 * q;
                            q *= p;
                            p *= p;
                            y0 += y0;
                            y1 += y1;
                        }
                    }
                } else {
                    const double x0 = E0 * pfc, x1 = E1 * pfc;
#pragma unroll
                    for (int sl = 0; sl < 2; ++sl) {
                        const double pl = 1.0 + gp.lam[sl] * t.cost;
                        double p = pl > 0.0 ? pl : 0.0;
#pragma unroll
                        for (int b = 0; b < NBM; ++b) {
                            if (b < NB0) part[sl * NB0 + b] += x0 * p;
                            if (b < NB1) part[2 * NB0 + sl * NB1 + b] += x1 * p;
                            p *= p;
                        }
                    }
                }
            }, [] {});
            static_assert(NBAS <= kRed64, "the terms need a slot each");
#pragma unroll
            for (int b = 0; b < NBAS; ++b)
                if ((gp.used >> b) & 1) {
                    const double v = wave_sum(part[b]);
                    if (lane == 0) S.red[wv * kRed64 + b] = v;
                }
            __syncthreads();
            for (int q = threadIdx.x; q < nmem; q += W * kWave) {
                double v = 0.0;
#pragma unroll
                for (int w = 0; w < W; ++w) v += S.red[w * kRed64 + MF[GR.mem0 + q].beta];
                put(mem[q], v, true);
            }
            __syncthreads();
            continue;
        }
        double acc[MAXM];
#pragma unroll
        for (int q = 0; q < MAXM; ++q) acc[q] = 0.0;
        for_each_triplet64<W>(S, A, B, same, wide ? INFINITY : GR.rc2, [&](int j, int k) {
            Trip64 t;
            triplet_geometry<COS>(t, S.g[j], S.c[j], S.g[k], S.c[k], wide, wt, ctype, GR, tanhPre);
            const double pfc = t.zw * t.cj.y * t.ck.y * t.fcjk;
            Along a{};
            if constexpr (TANGENT) a = tangent(t, j, k, pfc);
            Exp64 x;
#pragma unroll
            for (int q = 0; q < MAXM; ++q)
                if (q < nmem) {
                    const MemberT& mb = mem[q];
                    member_exp(x, mb, t, wide, wt);
                    const double plambda = 1.0 + mb.lambda * t.cost;
                    if (plambda > 0.0) {
                        const double fg =
                            x.vexp * (mb.useIntPow ? pow_int(plambda, mb.zetaInt - 1) : pow(plambda, mb.zeta - 1.0));
                        if constexpr (TANGENT) {
                            const double ga = x.shifted ? pfc * (x.fjk * a.s3 - x.fij * a.s1 - x.fik * a.s2) : a.ga;
                            acc[q] += fg * (mb.zetaLambda * a.al + plambda * (a.be + 2.0 * mb.eta * ga));
                        } else {
                            acc[q] += fg * plambda * pfc;
                        }
                    }
                }
        }, [] {});
        static_assert(MAXM <= kRed64, "the members need a slot each");
#pragma unroll
        for (int q = 0; q < MAXM; ++q)
            if (q < nmem) {
                const double v = wave_sum(acc[q]);
                if (lane == 0) S.red[wv * kRed64 + q] = v;
            }
        __syncthreads();
        for (int q = threadIdx.x; q < nmem; q += W * kWave) {
            double v = 0.0;
#pragma unroll
            for (int w = 0; w < W; ++w) v += S.red[w * kRed64 + q];
            put(mem[q], v, true);
        }
        __syncthreads();
    }
}

// w[i][q] = dE/dG[i][q] times the member's derivative scale.
__global__ void k_weights64(const int* __restrict__ elem, const double* __restrict__ dEdG,
                            const double* __restrict__ fac, int ldG, size_t total, double* __restrict__ w)
{
    for (size_t x = blockIdx.x * (size_t)blockDim.x + threadIdx.x; x < total; x += (size_t)gridDim.x * blockDim.x) {
        const size_t i = x / ldG;
        const int q = (int)(x - i * ldG);
        w[x] = dEdG[x] * fac[elem[i] * kMaxSF + q];
    }
}

__global__ void k_zero_f64(double* p, size_t n)
{
    for (size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
        p[q] = 0.0;
}

}  // namespace

// Kernel instance by the model's angular shape: the power path (NB0, NB1)
// when every angular group qualifies (MixedModel::powNB), with the cosine
// cutoff or any, else the member loop unrolled to the largest group.
template <typename F>
static void dispatch64(const ModelT& hm, const MixedModel& mm, F&& f)
{
    using std::integral_constant;
    using I0 = integral_constant<int, 0>;
    using I1 = integral_constant<int, 1>;
    using I3 = integral_constant<int, 3>;
    using I4 = integral_constant<int, 4>;
    using I5 = integral_constant<int, 5>;
    using std::false_type;
    if (mm.powNB[0] > 0) {
        auto power = [&](auto n0, auto n1) {
            if (hm.cutoffType == 1) f(I4{}, n0, n1, std::true_type{});
            else f(I4{}, n0, n1, false_type{});
        };
        switch (mm.powNB[0] * 10 + mm.powNB[1]) {
        case 30: power(I3{}, I0{}); return;
        case 33: power(I3{}, I3{}); return;
        case 50: power(I5{}, I0{}); return;
        case 51: power(I5{}, I1{}); return;
        case 55: power(I5{}, I5{}); return;
        default: break;
        }
    }
    const int mam = std::max(hm.max_mem_ang, 1);
    if (mam <= 4) f(integral_constant<int, 4>{}, I0{}, I0{}, false_type{});
    else if (mam <= 8) f(integral_constant<int, 8>{}, I0{}, I0{}, false_type{});
    else if (mam <= 16) f(integral_constant<int, 16>{}, I0{}, I0{}, false_type{});
    else f(integral_constant<int, 32>{}, I0{}, I0{}, false_type{});
}

// Calls f(waves per atom, walk buffer, LDS bytes): four waves where two would
// leave the chip short of them (see kFew64), the largest buffer that fits.
template <typename F>
static void shape64(const SysView& s, int capL, const char* what, F&& f)
{
    const int waves = s.natoms <= kFew64 && stage64_bytes(capL, 4, kMinWalk64) <= kLds64 ? 4 : 2;
    int walk = kWalk64;
    while (walk > kMinWalk64 && stage64_bytes(capL, waves, walk) > kLds64) walk -= 128;
    const size_t lds = stage64_bytes(capL, waves, walk);
    if (lds > kLds64)
        throw Error{NNPX_ERR_UNSUPPORTED, std::string("neighbour count too large for the ") + what + " kernel's LDS"};
    if (waves == 4) f(std::integral_constant<int, 4>{}, walk, lds);
    else f(std::integral_constant<int, 2>{}, walk, lds);
}

static int stage_slots(const SysView& s) { return ((std::max(s.stage_cap, 1) + 31) / 32) * 32; }

void launch_values64(const ModelT* m, const ModelT& hm, const MixedModel& mm, const SysView& s, double* G, int ldG,
                     hipStream_t stream)
{
    if (s.natoms == 0) return;
    if (!G || !s.nb_n || !s.nb_j) throw Error{NNPX_ERR_STATE, "FP64 SF values: a buffer is missing"};
    const int capL = stage_slots(s);
    shape64(s, capL, "FP64 SF value", [&](auto w, int walk, size_t lds) {
        if (!hm.has_exp) return;
        dispatch64(hm, mm, [&](auto mx, auto n0, auto n1, auto cs) {
            constexpr int W = decltype(w)::value;
            hipLaunchKernelGGL((k_values64<W, false, decltype(mx)::value, decltype(n0)::value, decltype(n1)::value, decltype(cs)::value>),
                               dim3(s.natoms), dim3(kWave * W), lds, stream, m, mm.d_mem, mm.d_gpow64, s, nullptr,
                               nullptr, G, ldG, capL, walk);
        });
    });
}

void launch_tangent64_fused(const ModelT* m, const ModelT& hm, const MixedModel& mm, const SysView& s,
                            const double* u, const double* fac, double* Gdot, int ldG, hipStream_t stream)
{
    if (s.natoms == 0) return;
    if (!u || !fac || !Gdot || !s.nb_n || !s.nb_j)
        throw Error{NNPX_ERR_STATE, "fused FP64 tangent: a buffer is missing"};
    const int capL = stage_slots(s);
    shape64(s, capL, "FP64 tangent", [&](auto w, int walk, size_t lds) {
        if (!hm.has_exp) return;
        dispatch64(hm, mm, [&](auto mx, auto n0, auto n1, auto cs) {
            constexpr int W = decltype(w)::value;
            hipLaunchKernelGGL((k_values64<W, true, decltype(mx)::value, decltype(n0)::value, decltype(n1)::value, decltype(cs)::value>),
                               dim3(s.natoms), dim3(kWave * W), lds, stream, m, mm.d_mem, mm.d_gpow64, s, u, fac,
                               Gdot, ldG, capL, walk);
        });
    });
    launch_tangentcomp64(m, hm, s, u, Gdot, ldG, stream);
}

size_t fused64_lds(int cap) { return stage64_bytes(((std::max(cap, 1) + 31) / 32) * 32, 2, kMinWalk64); }

void launch_force64_fused(const ModelT* m, const ModelT& hm, const MixedModel& mm, const SysView& s,
                          const double* dEdG, const double* fac, double* w, int ldG, double* F, bool push,
                          hipStream_t stream)
{
    if (s.natoms == 0) return;
    if (!dEdG || !fac || !w || !F || !s.nb_n || !s.nb_j)
        throw Error{NNPX_ERR_STATE, "fused FP64 forces: a buffer is missing"};
    const int capL = stage_slots(s);
    shape64(s, capL, "FP64 fused force", [&](auto wc, int walk, size_t lds) {
        const size_t total = (size_t)s.natoms * ldG;
        hipLaunchKernelGGL(k_weights64, dim3((unsigned)std::min<size_t>((total + 255) / 256, 4096)), dim3(256), 0,
                           stream, s.elem, dEdG, fac, ldG, total, w);
        const size_t n3 = (size_t)3 * s.nforce;
        hipLaunchKernelGGL(k_zero_f64, dim3((unsigned)std::min<size_t>((n3 + 255) / 256, 4096)), dim3(256), 0, stream,
                           F, n3);
        const int ps = push ? 1 : 0;
        if (hm.has_exp)
            dispatch64(hm, mm, [&](auto mx, auto n0, auto n1, auto cs) {
                constexpr int W = decltype(wc)::value;
                hipLaunchKernelGGL((k_force64f<W, decltype(mx)::value, decltype(n0)::value, decltype(n1)::value, decltype(cs)::value>),
                                   dim3(s.natoms), dim3(kWave * W), lds, stream, m, mm.d_mem, mm.d_gpow64, s, w, ldG,
                                   F, ps, capL, walk);
            });
    });
    launch_sfcomp64_force(m, hm, s, w, ldG, F, push, stream);
}

}  // namespace nnpx
