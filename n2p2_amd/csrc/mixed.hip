// Mixed-precision form of the energy/force path (see mixed.hpp).
//
// k_sf32     symmetry-function values (mixed_sf.hip)
// k_nnbf16   NeuralNetwork::propagate (NeuralNetwork.cpp:761-896) for a
//            16-atom tile per block (four waves) as v_mfma_f32_16x16x16_bf16
//            tiles, and the adjoint dE/dG as the transposed GEMMs (replacing
//            the reference's forward-mode NeuralNetwork::calculateDEdG,
//            NeuralNetwork.cpp:396-442).
// k_force32  fused dG/dr backward (mixed_force.hip)
#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>
#include <vector>

#include "mixed.hpp"
#include "nnpx.h"
#include "sfcomp.hpp"

namespace nnpx {
namespace {

typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kNNRows = 16;  // atoms per tile of the NN kernel
constexpr int kNNWaves = 4;  // waves per tile

// float -> bf16, round to nearest even
__host__ __device__ inline uint16_t to_bf16(float f)
{
    uint32_t u;
#ifdef __HIP_DEVICE_COMPILE__
    u = __float_as_uint(f);
#else
    std::memcpy(&u, &f, 4);
#endif
    u += 0x7FFFu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__host__ __device__ inline float from_bf16(uint16_t h)
{
    uint32_t u = (uint32_t)h << 16;
#ifdef __HIP_DEVICE_COMPILE__
    return __uint_as_float(u);
#else
    float f;
    std::memcpy(&f, &u, 4);
    return f;
#endif
}

// ------------------------------------------------------------ BF16 MFMA NN --
struct NNMix {
    const uint16_t* w;
    const float* b;
    const float* sffac;
    const int* atoms;
    int blk_off[kMaxElem + 1];
    int atom_off[kMaxElem + 1];
    int wW[kMaxElem][kMaxLayers], wT[kMaxElem][kMaxLayers], bo[kMaxElem][kMaxLayers];
    int pin[kMaxElem][kMaxLayers], pout[kMaxElem][kMaxLayers];
    int nelem, ldK, ldG, terms;
    int stride_in;  // LDS row length of the input tile (padded input width + 4)
    int stride;     // ... of the hidden/output tiles (padded layer width + 4)
    double* zero;   // cleared by the blocks in a grid-stride loop (the force
    size_t nzero;   // array of the force kernel that follows), nzero doubles
};

__device__ inline float act32(int a, float x, float& d)
{
    float v;
    switch (a) {
    case AF_IDENTITY: d = 1.f; return x;
    case AF_TANH: v = tanhf(x); d = 1.f - v * v; return v;
    case AF_LOGISTIC:
        if (x > 35.f) { d = 0.f; return 1.f; }
        if (x < -35.f) { d = 0.f; return 0.f; }
        v = 1.f / (1.f + __expf(-x)); d = v * (1.f - v); return v;
    case AF_SOFTPLUS:
        if (x > 35.f) { d = 1.f; return x; }
        if (x < -35.f) { d = 0.f; return 0.f; }
        { const float t = __expf(x); d = 1.f / (1.f + 1.f / t); return log1pf(t); }
    case AF_RELU: if (x > 0.f) { d = 1.f; return x; } d = 0.f; return 0.f;
    case AF_GAUSSIAN: { const float t = __expf(-0.5f * x * x); d = -x * t; return t; }
    case AF_COS: d = -sinf(x); return cosf(x);
    case AF_REVLOGISTIC: v = 1.f / (1.f + __expf(-x)); d = v * (v - 1.f); return 1.f - v;
    case AF_EXP: v = __expf(-x); d = -v; return v;
    case AF_HARMONIC: d = 2.f * x; return x * x;
    }
    d = 0.f;
    return 0.f;
}

// A fragment: rows = atoms (lane % 16), k = k0 + 4*(lane/16) + 0..3 from an
// LDS row-major [16][stride] FP32 tile, split into bf16 hi and lo.
__device__ inline void a_frag(const float* tile, int stride, int k0, s4& hi, s4& lo)
{
    const int lane = threadIdx.x & (kWave - 1);
    const float* p = tile + (lane & 15) * stride + k0 + 4 * (lane >> 4);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const uint16_t h = to_bf16(p[v]);
        hi[v] = (short)h;
        lo[v] = (short)to_bf16(p[v] - from_bf16(h));
    }
}

// B fragment: B[k][n] = Wt[n][k] for n = n0 + lane % 16, k = k0 + 4*(lane/16)
// + 0..3, from a row-major bf16 matrix with row length ld (hi; lo at +lo_off).
__device__ inline void b_frag(const uint16_t* __restrict__ w, int ld, int lo_off, int n0, int k0, s4& hi, s4& lo)
{
    const int lane = threadIdx.x & (kWave - 1);
    const uint16_t* p = w + (size_t)(n0 + (lane & 15)) * ld + k0 + 4 * (lane >> 4);
    const uint2 h = *reinterpret_cast<const uint2*>(p);
    const uint2 l = *reinterpret_cast<const uint2*>(p + lo_off);
    hi = __builtin_bit_cast(s4, h);
    lo = __builtin_bit_cast(s4, l);
}

__device__ inline f4 mma(f4 c, const s4& ah, const s4& al, const s4& bh, const s4& bl, int terms)
{
    c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ah, bh, c, 0, 0, 0);
    if (terms > 1) {
        c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(ah, bl, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(al, bh, c, 0, 0, 0);
    }
    return c;
}

// kNNWaves waves share one tile of 16 atoms: each takes every kNNWaves-th
// 16-column block of a layer, so the chain of dependent MFMA steps per wave
// is that much shorter (the network kernel is latency-bound: a few waves
// per CU).
__global__ __launch_bounds__(kWave * kNNWaves) void k_nnbf16(const ModelT* __restrict__ M, NNMix a,
                                                            const float* __restrict__ Gin,
                                                            double* __restrict__ Eatom, double* __restrict__ dEdG,
                                                            float* __restrict__ dEdGf)
{
    extern __shared__ float sm[];
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < a.nzero; q += (size_t)gridDim.x * blockDim.x)
        a.zero[q] = 0.0;
    const int lane = threadIdx.x & (kWave - 1);
    const int wv = threadIdx.x / kWave;
    int e = 0;
    while (e + 1 < a.nelem && (int)blockIdx.x >= a.blk_off[e + 1]) ++e;
    const NNT& N = M->el[e].nn;
    const int nl = N.nl;
    const int st = a.stride;
    float* bufI = sm;                           // [16][stride_in] network input
    float* bufA = bufI + kNNRows * a.stride_in;  // hidden/output tiles [16][st]
    float* bufB = bufA + kNNRows * st;
    float* dfd = bufB + kNNRows * st;  // [layer][16][st]
    const int tile = (int)blockIdx.x - a.blk_off[e];
    const int first = a.atom_off[e] + tile * kNNRows;
    const int cnt = min(kNNRows, a.atom_off[e + 1] - first);

    // layer-0 input rows
    const int pin0 = a.pin[e][1];
    for (int x = threadIdx.x; x < kNNRows * pin0; x += kWave * kNNWaves) {
        const int r = x / pin0, k = x % pin0;
        bufI[r * a.stride_in + k] = r < cnt ? Gin[(size_t)a.atoms[first + r] * a.ldK + k] : 0.f;
    }
    __syncthreads();
    float* in = bufI;
    float* out = bufA;
    int sin = a.stride_in;
    for (int l = 1; l < nl; ++l) {
        const int pi = a.pin[e][l], po = a.pout[e][l];
        const uint16_t* W = a.w + a.wW[e][l];
        const float* bias = a.b + a.bo[e][l];
        const float norm = N.normalize ? 1.f / N.n[l - 1] : 1.f;
        for (int n0 = 16 * wv; n0 < po; n0 += 16 * kNNWaves) {
            f4 c = {0.f, 0.f, 0.f, 0.f};
            // the next weight fragment is loaded while this one multiplies
            s4 bh, bl;
            b_frag(W, pi, po * pi, n0, 0, bh, bl);
            for (int k0 = 0; k0 < pi; k0 += 16) {
                s4 ah, al, nh = bh, nl_ = bl;
                if (k0 + 16 < pi) b_frag(W, pi, po * pi, n0, k0 + 16, nh, nl_);
                a_frag(in, sin, k0, ah, al);
                c = mma(c, ah, al, bh, bl, a.terms);
                bh = nh;
                bl = nl_;
            }
            const int n = n0 + (lane & 15);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = 4 * (lane >> 4) + v;
                float d;
                const float x = (c[v] + bias[n]) * norm;
                const float y = act32(N.act[l], x, d);
                out[r * st + n] = n < N.n[l] ? y : 0.f;
                dfd[(l * kNNRows + r) * st + n] = n < N.n[l] ? d : 0.f;
            }
        }
        __syncthreads();
        // the hidden and output tiles alternate between bufA and bufB
        in = out;
        out = in == bufA ? bufB : bufA;
        sin = st;
    }
    if (threadIdx.x < cnt) Eatom[a.atoms[first + threadIdx.x]] = (double)in[threadIdx.x * st];
    // adjoint: delta of the output layer is f'_out for the energy neuron
    float* dl = out;
    const int pl = a.pout[e][nl - 1];
    for (int x = threadIdx.x; x < kNNRows * pl; x += kWave * kNNWaves) {
        const int r = x / pl, n = x % pl;
        dl[r * st + n] = n == 0 ? dfd[((nl - 1) * kNNRows + r) * st] : 0.f;
    }
    __syncthreads();
    float* dn = in;
    for (int l = nl - 1; l >= 1; --l) {
        const int pi = a.pin[e][l], po = a.pout[e][l];
        const uint16_t* WT = a.w + a.wT[e][l];
        const float norm = N.normalize ? 1.f / N.n[l - 1] : 1.f;
        for (int m0 = 16 * wv; m0 < pi; m0 += 16 * kNNWaves) {
            f4 c = {0.f, 0.f, 0.f, 0.f};
            s4 bh, bl;
            b_frag(WT, po, po * pi, m0, 0, bh, bl);
            for (int k0 = 0; k0 < po; k0 += 16) {
                s4 ah, al, nh = bh, nl_ = bl;
                if (k0 + 16 < po) b_frag(WT, po, po * pi, m0, k0 + 16, nh, nl_);
                a_frag(dl, st, k0, ah, al);
                c = mma(c, ah, al, bh, bl, a.terms);
                bh = nh;
                bl = nl_;
            }
            const int m = m0 + (lane & 15);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = 4 * (lane >> 4) + v;
                float g = c[v] * norm;
                if (l > 1) {
                    dn[r * st + m] = g * dfd[((l - 1) * kNNRows + r) * st + m];
                } else if (r < cnt && m < N.n[0]) {
                    const size_t at = (size_t)a.atoms[first + r];
                    dEdG[at * a.ldG + m] = (double)g;
                    dEdGf[at * a.ldG + m] = g * a.sffac[e * kMaxSF + m];
                }
            }
        }
        __syncthreads();
        float* t = dl; dl = dn; dn = t;
    }
}

__global__ void k_zero(double* p, size_t n)
{
    for (size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
        p[q] = 0.0;
}

__global__ void k_mfma_probe(const float* A, const float* B, float* D)
{
    // A, B: 16x16 row-major; D = A * B (16x16 row-major)
    const int lane = threadIdx.x;
    s4 ah, al, bh, bl;
    a_frag(A, 16, 0, ah, al);
    // B fragment from B^T (row n, column k)
    float bt[4];
    for (int v = 0; v < 4; ++v) bt[v] = B[(4 * (lane >> 4) + v) * 16 + (lane & 15)];
    for (int v = 0; v < 4; ++v) {
        const uint16_t h = to_bf16(bt[v]);
        bh[v] = (short)h;
        bl[v] = (short)to_bf16(bt[v] - from_bf16(h));
    }
    f4 c = {0.f, 0.f, 0.f, 0.f};
    c = mma(c, ah, al, bh, bl, 3);
    for (int v = 0; v < 4; ++v) D[(4 * (lane >> 4) + v) * 16 + (lane & 15)] = c[v];
}

// Power-path shapes (NB0, NB1) with kernels built for them: terms per
// lambda of the first and second eta.
constexpr int kPowShapes[][2] = {{3, 0}, {3, 3}, {5, 0}, {5, 1}, {5, 5}};
constexpr int kNumPowShapes = sizeof(kPowShapes) / sizeof(kPowShapes[0]);

// b with zeta == 2^b, 0 <= b <= 4; -1 otherwise.
int pow2_exponent(double zeta)
{
    for (int b = 0; b <= 4; ++b)
        if (zeta == (double)(1 << b)) return b;
    return -1;
}

}  // namespace

static void pack_weights(MixedModel& mm, const HostModel& hm, std::vector<uint16_t>& w, std::vector<float>& b)
{
    // bf16 weights, padded to 16: W [out][in] and WT [in][out], hi then lo.
    const ModelT& t = hm.t;
    w.clear();
    b.clear();
    auto pad16 = [](int x) { return (x + 15) / 16 * 16; };
    mm.maxpad = 16;
    mm.maxpadh = 16;
    mm.ldK = 16;
    for (int e = 0; e < t.nelem; ++e) {
        const NNT& N = t.el[e].nn;
        mm.ldK = std::max(mm.ldK, pad16(N.n[0]));
        for (int l = 1; l < N.nl; ++l) {
            const int nin = N.n[l - 1], nout = N.n[l];
            const int pi = pad16(nin), po = pad16(nout);
            mm.pin[e][l] = pi;
            mm.pout[e][l] = po;
            mm.maxpad = std::max(mm.maxpad, std::max(pi, po));
            mm.maxpadh = std::max(mm.maxpadh, po);
            std::vector<float> W((size_t)po * pi, 0.f);
            for (int k = 0; k < nout; ++k)
                for (int j = 0; j < nin; ++j) W[(size_t)k * pi + j] = (float)hm.weights[N.woff[l] + (size_t)k * nin + j];
            mm.wW[e][l] = (int)w.size();
            std::vector<uint16_t> hi(W.size()), lo(W.size());
            for (size_t q = 0; q < W.size(); ++q) {
                hi[q] = to_bf16(W[q]);
                lo[q] = to_bf16(W[q] - from_bf16(hi[q]));
            }
            w.insert(w.end(), hi.begin(), hi.end());
            w.insert(w.end(), lo.begin(), lo.end());
            mm.wT[e][l] = (int)w.size();
            for (int j = 0; j < pi; ++j)
                for (int k = 0; k < po; ++k) hi[(size_t)j * po + k] = to_bf16(W[(size_t)k * pi + j]);
            for (int j = 0; j < pi; ++j)
                for (int k = 0; k < po; ++k) {
                    const float x = W[(size_t)k * pi + j];
                    lo[(size_t)j * po + k] = to_bf16(x - from_bf16(to_bf16(x)));
                }
            w.insert(w.end(), hi.begin(), hi.end());
            w.insert(w.end(), lo.begin(), lo.end());
            mm.bo[e][l] = (int)b.size();
            for (int k = 0; k < po; ++k) b.push_back(k < nout ? (float)hm.weights[N.boff[l] + k] : 0.f);
        }
    }
}

void setup_mixed(MixedModel& mm, const HostModel& hm)
{
    free_mixed(mm);
    const ModelT& t = hm.t;
    std::vector<MemberF> mf(std::max(t.nmembers, 1));
    std::vector<GroupMixF> gmix(std::max(t.ngroups, 1));
    std::vector<GroupPow64> gp64(std::max(t.ngroups, 1), GroupPow64{});
    std::vector<float> sffac((size_t)kMaxElem * kMaxSF, 0.f);
    mm.maxS = 1;
    mm.hasRs = false;
    for (int e = 0; e < t.nelem; ++e) {
        const ElementT& E = t.el[e];
        for (int g = E.grp0; g < E.grp0 + E.ngrp; ++g) {
            const GroupT& G = t.grp[g];
            GroupMixF& gm = gmix[g];
            gm = GroupMixF{};
            for (int q = G.mem0; q < G.mem0 + G.nmem; ++q) {
                const MemberT& M = t.mem[q];
                MemberF& f = mf[q];
                f.eta = (float)M.eta;
                f.rs = (float)M.rs;
                f.lambda = (float)M.lambda;
                f.zeta = (float)M.zeta;
                f.gnorm = (G.type == 3 || G.type == 9 || G.type == 13) ? (float)M.gnorm : 1.f;
                f.twoEta = (float)(2.0 * M.eta);
                f.zetaLambda = (float)M.zetaLambda;
                f.etaL = (float)(M.eta * 1.4426950408889634);  // eta * log2(e)
                f.sf = M.sf;
                f.calcExp = M.calcExp;
                f.sidx = 0;
                f.beta = -1;
                if (G.type == 3 || G.type == 9 || G.type == 13) {
                    if (M.rs > 0.0) mm.hasRs = true;
                    int k = 0;
                    while (k < gm.nlam && gm.lam[k] != f.lambda) ++k;
                    if (k == gm.nlam) {
                        if (gm.nlam == 4) throw Error{NNPX_ERR_UNSUPPORTED, "more than 4 distinct lambda per SF group"};
                        gm.lam[gm.nlam++] = f.lambda;
                    }
                    f.sidx = k;
                }
                sffac[(size_t)e * kMaxSF + M.sf] =
                    (float)((G.type == 3 || G.type == 9 || G.type == 13) ? M.factorNorm : M.sfac);
            }
            mm.maxS = std::max(mm.maxS, gm.nlam);
            // unused table slots repeat the first lambda (evaluated, never picked)
            for (int k = gm.nlam; k < 4; ++k) gm.lam[k] = gm.nlam ? gm.lam[0] : 0.f;
        }
    }
    mm.maxS = mm.maxS <= 2 ? 2 : 4;
    // fast path: all angular groups share one member count, <= 2 lambda, rs = 0
    mm.fastM = 0;
    if (mm.maxS == 2 && !mm.hasRs) {
        int cnt = -1;
        bool same = true;
        for (int g = 0; g < t.ngroups; ++g)
            if (t.grp[g].type == 3 || t.grp[g].type == 9 || t.grp[g].type == 13) {
                if (cnt < 0) cnt = t.grp[g].nmem;
                same = same && t.grp[g].nmem == cnt;
            }
        if (same && (cnt == 4 || cnt == 8 || cnt == 10 || cnt == 16)) mm.fastM = cnt;
    }
    // power path: every angular group has zeta in {1, 2, 4, 8, 16}, at most
    // two distinct eta and two lambda, rs = 0
    mm.powNB[0] = mm.powNB[1] = 0;
    if (mm.maxS == 2 && !mm.hasRs) {
        bool ok = true;
        int need[2] = {0, 0};
        std::vector<std::array<double, 2>> heta(std::max(t.ngroups, 1));
        std::vector<std::array<int, 2>> hnb(std::max(t.ngroups, 1));
        for (int g = 0; g < t.ngroups && ok; ++g) {
            const GroupT& G = t.grp[g];
            if (G.type != 3 && G.type != 9 && G.type != 13) continue;
            int nh = 0;
            int nb[2] = {0, 0};
            double eta[2] = {0.0, 0.0};
            for (int q = G.mem0; q < G.mem0 + G.nmem && ok; ++q) {
                const MemberT& M = t.mem[q];
                int h = 0;
                while (h < nh && eta[h] != M.eta) ++h;
                if (h == nh) {
                    if (nh == 2) { ok = false; break; }
                    eta[nh++] = M.eta;
                }
                const int b = pow2_exponent(M.zeta);
                if (b < 0) { ok = false; break; }
                nb[h] = std::max(nb[h], b + 1);
            }
            if (!ok) break;
            // the eta with the higher powers takes the larger block
            if (nb[1] > nb[0]) {
                std::swap(nb[0], nb[1]);
                std::swap(eta[0], eta[1]);
            }
            heta[g] = {eta[0], eta[1]};
            hnb[g] = {nb[0], nb[1]};
            need[0] = std::max(need[0], nb[0]);
            need[1] = std::max(need[1], nb[1]);
        }
        int best = -1;
        for (int k = 0; k < kNumPowShapes; ++k)
            if (kPowShapes[k][0] >= need[0] && kPowShapes[k][1] >= need[1] &&
                (best < 0 || kPowShapes[k][0] + kPowShapes[k][1] < kPowShapes[best][0] + kPowShapes[best][1]))
                best = k;
        if (ok && need[0] > 0 && best >= 0) {
            const int NB0 = kPowShapes[best][0], NB1 = kPowShapes[best][1];
            mm.powNB[0] = NB0;
            mm.powNB[1] = NB1;
            for (int g = 0; g < t.ngroups; ++g) {
                const GroupT& G = t.grp[g];
                if (G.type != 3 && G.type != 9 && G.type != 13) continue;
                GroupMixF& gm = gmix[g];
                GroupPow64& gp = gp64[g];
                for (int h = 0; h < 2; ++h) {
                    gm.etaL[h] = (float)(heta[g][h] * 1.4426950408889634);
                    gm.twoEta[h] = (float)(2.0 * heta[g][h]);
                    gp.eta[h] = heta[g][h];
                    gp.twoEta[h] = 2.0 * heta[g][h];
                }
                gm.used = 0;
                for (int q = G.mem0; q < G.mem0 + G.nmem; ++q) {
                    const MemberT& M = t.mem[q];
                    const int h = M.eta == heta[g][0] ? 0 : 1;
                    const int b = pow2_exponent(M.zeta);
                    mf[q].beta = h == 0 ? mf[q].sidx * NB0 + b : 2 * NB0 + mf[q].sidx * NB1 + b;
                    gm.used |= 1 << mf[q].beta;
                    gp.lam[mf[q].sidx] = M.lambda;
                }
                gp.used = gm.used;
            }
        }
    }
    // merged angular walks: per element, every angular group on the power
    // path, one type (3 or 9), the element's single cutoff radius, identical
    // term constants and distinct neighbour element pairs
    std::vector<AngMergeF> amerge(std::max(t.nelem, 1));
    mm.merge_ng = 0;
    mm.merge_avg = 0.0;
    int merged_elements = 0;
    for (int e = 0; e < t.nelem && mm.powNB[0] > 0; ++e) {
        AngMergeF& am = amerge[e];
        std::memset(&am, 0, sizeof(am));
        std::memset(am.pair, -1, sizeof(am.pair));
        const ElementT& E = t.el[e];
        std::vector<int> ang;
        for (int gi = 0; gi < E.ngrp; ++gi) {
            const int g = E.grp0 + gi;
            const int ty = t.grp[g].type;
            if (ty == 3 || ty == 9 || ty == 13) ang.push_back(g);
        }
        bool ok = E.ucut && ang.size() >= 2 && (int)ang.size() <= kMaxMerge;
        for (size_t q = 0; q < ang.size() && ok; ++q) {
            const GroupT& G = t.grp[ang[q]];
            const GroupT& G0 = t.grp[ang[0]];
            const GroupMixF& a = gmix[ang[q]];
            const GroupMixF& a0 = gmix[ang[0]];
            ok = G.type != 13 && G.type == G0.type && G.rc == G0.rc && a.nlam == a0.nlam && a.lam[0] == a0.lam[0] &&
                 a.lam[1] == a0.lam[1] && a.etaL[0] == a0.etaL[0] && a.etaL[1] == a0.etaL[1] &&
                 a.twoEta[0] == a0.twoEta[0] && a.twoEta[1] == a0.twoEta[1] &&
                 am.pair[G.e1 * kMaxElem + G.e2] < 0;
            if (!ok) break;
            am.grp[q] = ang[q];
            am.used |= a.used;
            am.pair[G.e1 * kMaxElem + G.e2] = (signed char)q;
            am.pair[G.e2 * kMaxElem + G.e1] = (signed char)q;
        }
        if (!ok) {
            std::memset(&am, 0, sizeof(am));
            std::memset(am.pair, -1, sizeof(am.pair));
            continue;
        }
        am.ng = (int)ang.size();
        mm.merge_ng = std::max(mm.merge_ng, am.ng);
        mm.merge_avg += am.ng;
        ++merged_elements;
    }
    if (merged_elements) mm.merge_avg /= merged_elements;
    // angular walks per element (an upper bound: every non-radial group, and
    // the merged walk)
    mm.max_walks = 0;
    for (int e = 0; e < t.nelem; ++e) {
        int nw = 1;
        for (int gi = 0; gi < t.el[e].ngrp; ++gi) {
            const int ty = t.grp[t.el[e].grp0 + gi].type;
            if (ty != 2 && ty != 12) ++nw;
        }
        mm.max_walks = std::max(mm.max_walks, nw);
    }
    std::vector<uint16_t> w;
    std::vector<float> b;
    pack_weights(mm, hm, w, b);
    auto up = [](void** dst, const void* src, size_t bytes) {
        if (hipMalloc(dst, std::max<size_t>(bytes, 16)) != hipSuccess) throw Error{NNPX_ERR_HIP, "hipMalloc mixed"};
        if (hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice) != hipSuccess) throw Error{NNPX_ERR_HIP, "hipMemcpy"};
    };
    up((void**)&mm.d_mem, mf.data(), sizeof(MemberF) * mf.size());
    up((void**)&mm.d_gmix, gmix.data(), sizeof(GroupMixF) * gmix.size());
    up((void**)&mm.d_gpow64, gp64.data(), sizeof(GroupPow64) * gp64.size());
    up((void**)&mm.d_amerge, amerge.data(), sizeof(AngMergeF) * amerge.size());
    up((void**)&mm.d_sffac, sffac.data(), sizeof(float) * sffac.size());
    up((void**)&mm.d_w, w.data(), sizeof(uint16_t) * w.size());
    up((void**)&mm.d_b, b.data(), sizeof(float) * b.size());
    mm.ready = true;
}

// New weights for the model that setup_mixed() saw: the networks' tables keep
// their sizes, nothing else depends on the weights.
void update_mixed_weights(MixedModel& mm, const HostModel& hm)
{
    if (!mm.ready) throw Error{NNPX_ERR_STATE, "mixed-precision tables not set up"};
    std::vector<uint16_t> w;
    std::vector<float> b;
    pack_weights(mm, hm, w, b);
    if (hipMemcpy(mm.d_w, w.data(), sizeof(uint16_t) * w.size(), hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(mm.d_b, b.data(), sizeof(float) * b.size(), hipMemcpyHostToDevice) != hipSuccess)
        throw Error{NNPX_ERR_HIP, "hipMemcpy"};
}

void free_mixed(MixedModel& mm)
{
    if (mm.d_mem) (void)hipFree(mm.d_mem);
    if (mm.d_gmix) (void)hipFree(mm.d_gmix);
    if (mm.d_gpow64) (void)hipFree(mm.d_gpow64);
    if (mm.d_amerge) (void)hipFree(mm.d_amerge);
    if (mm.d_sffac) (void)hipFree(mm.d_sffac);
    if (mm.d_w) (void)hipFree(mm.d_w);
    if (mm.d_b) (void)hipFree(mm.d_b);
    const int terms = mm.terms;
    const Tuning tune = mm.tune;
    mm = MixedModel{};
    mm.terms = terms;
    mm.tune = tune;
}

// Merged angular walk on or off: a tuning value of 0 or 1 decides, -1 takes
// it where the model merges at least four groups per element on average
// (fewer groups have enough triplets each to fill the per-group walks).
static bool use_merge(const MixedModel& mm, int want)
{
    if (mm.merge_ng == 0 || mm.powNB[0] == 0) return false;
    if (want >= 0) return want == 1;
    return mm.merge_avg >= 4.0;
}

void run_mixed(const MixedModel& mm, const ModelT& t, const ModelT* d_model, const SysView& s,
               const MixedBuffers& b, bool forces, bool push, hipStream_t stream, const TimedFn& timed)
{
    if (!mm.ready) throw Error{NNPX_ERR_STATE, "mixed-precision tables not set up"};
    if (s.natoms == 0) return;
    const int capL = s.stage_cap;
    const int tsf = mm.tune.trip_sf, tf = mm.tune.trip_force;
    // LDS of the largest kernel instances (the member paths' constant area)
    const size_t lds_sf_max = stage_bytes(capL, 1, tsf, stage_mp(0, 0, 1));
    const size_t lds_f_max = stage_bytes(capL, 1, tf, stage_mp(0, 0, 1)) + (sizeof(double) * 3 + 2) * (size_t)capL;
    if (lds_f_max > 65536 || lds_sf_max > 65536)
        throw Error{NNPX_ERR_UNSUPPORTED, "neighbour count too large for the mixed kernels' LDS"};
    const bool merge_sf = use_merge(mm, mm.tune.merge_sf), merge_f = use_merge(mm, mm.tune.merge_force);
    // with pair lists on, the angular pairs pass from the SF to the force
    // kernel when both make the same walks (the SF kernel also counts them,
    // which sizes the lists of later evaluations); off, the force kernel
    // walks rows
    const bool lists = keep_lists(mm.tune, s.natoms);
    TripList T{};
    if (forces && lists && merge_sf == merge_f) {
        T = b.trips;
        T.count = true;
    }
    // lists not set by the caller and not there (the first evaluation only counts
    // the pairs): rows, the faster walk of the two
    T.rows = !lists || (mm.tune.pair_lists < 0 && !T.list);
    // the staging passes from the SF to the force kernel (identical values)
    const StageKeep KS = forces && b.keep.ld >= capL ? b.keep : StageKeep{};
    // a model of compact functions alone leaves these kernels nothing: its
    // values (and the input rows' padding) come from the factored kernel
    const bool gauss_sf = t.has_exp || !sfcomp_factored_fits<float>(CM_VALUES, capL);
    timed("sf32", [&] {
        if (gauss_sf) launch_sf32(mm, t, d_model, s, b, T, KS, merge_sf, stream);
        launch_sfcomp32(d_model, t, s, b.G, b.Gin, b.ldG, mm.ldK, nullptr, nullptr, false, false, stream);
    });
    NNMix a{};
    a.w = mm.d_w;
    a.b = mm.d_b;
    a.sffac = mm.d_sffac;
    a.atoms = b.elem_atoms;
    a.nelem = t.nelem;
    a.ldK = mm.ldK;
    a.ldG = b.ldG;
    a.stride = mm.maxpadh + 4;
    a.stride_in = mm.ldK + 4;
    a.terms = mm.terms;
    int blocks = 0;
    for (int e = 0; e < t.nelem; ++e) {
        a.blk_off[e] = blocks;
        a.atom_off[e] = b.elem_off[e];
        blocks += (b.elem_off[e + 1] - b.elem_off[e] + kNNRows - 1) / kNNRows;
        for (int l = 0; l < kMaxLayers; ++l) {
            a.wW[e][l] = mm.wW[e][l];
            a.wT[e][l] = mm.wT[e][l];
            a.bo[e][l] = mm.bo[e][l];
            a.pin[e][l] = mm.pin[e][l];
            a.pout[e][l] = mm.pout[e][l];
        }
    }
    a.blk_off[t.nelem] = blocks;
    a.atom_off[t.nelem] = b.elem_off[t.nelem];
    const size_t lds_nn = sizeof(float) * (size_t)kNNRows * (a.stride_in + (size_t)a.stride * (2 + kMaxLayers));
    if (lds_nn > 65536) throw Error{NNPX_ERR_UNSUPPORTED, "network too wide for the mixed NN kernel's LDS"};
    // the NN blocks clear the forces of the force kernel (one launch fewer)
    const size_t n3 = forces ? (size_t)3 * s.nforce : 0;
    const bool nn_zero = blocks > 0;
    a.zero = nn_zero ? b.F : nullptr;
    a.nzero = nn_zero ? n3 : 0;
    timed("nnbf16", [&] {
        hipLaunchKernelGGL(k_nnbf16, dim3(blocks), dim3(kWave * kNNWaves), lds_nn, stream, d_model, a, b.Gin, b.Eatom,
                           b.dEdG, b.dEdGf);
    });
    timed("energy", [&] { launch_energy(b.Eatom, b.atom_off, b.nstruct, b.E, stream); });
    if (!forces) return;
    timed("force32", [&] {
        if (!nn_zero && n3 > 0)
            hipLaunchKernelGGL(k_zero, dim3((unsigned)std::min<size_t>((n3 + 255) / 256, 4096)), dim3(256), 0,
                               stream, b.F, n3);
        if (t.has_exp) launch_force32(mm, t, d_model, s, b, T, KS, merge_f, push, stream);
        launch_sfcomp32(d_model, t, s, nullptr, nullptr, b.ldG, mm.ldK, b.dEdGf, b.F, push, true, stream);
    });
}

double mfma_selftest()
{
    std::vector<float> A(256), B(256), D(256, 0.f);
    for (int i = 0; i < 16; ++i)
        for (int k = 0; k < 16; ++k) {
            A[i * 16 + k] = (float)((i * 7 + k * 3) % 11) - 5.f;
            B[i * 16 + k] = (float)((i * 5 + k * 13) % 9) - 4.f;
        }
    float *dA, *dB, *dD;
    if (hipMalloc(&dA, 1024) != hipSuccess || hipMalloc(&dB, 1024) != hipSuccess || hipMalloc(&dD, 1024) != hipSuccess)
        throw Error{NNPX_ERR_HIP, "hipMalloc"};
    (void)hipMemcpy(dA, A.data(), 1024, hipMemcpyHostToDevice);
    (void)hipMemcpy(dB, B.data(), 1024, hipMemcpyHostToDevice);
    hipLaunchKernelGGL(k_mfma_probe, dim3(1), dim3(64), 0, 0, dA, dB, dD);
    (void)hipMemcpy(D.data(), dD, 1024, hipMemcpyDeviceToHost);
    (void)hipFree(dA);
    (void)hipFree(dB);
    (void)hipFree(dD);
    double err = 0.0;
    for (int i = 0; i < 16; ++i)
        for (int j = 0; j < 16; ++j) {
            double ref = 0.0;
            for (int k = 0; k < 16; ++k) ref += (double)A[i * 16 + k] * B[k * 16 + j];
            err = std::max(err, std::fabs(ref - D[i * 16 + j]));
        }
    return err;
}

}  // namespace nnpx
