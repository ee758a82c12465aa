// Training gradient of the energy+force loss with respect to the network
// connections:
//   L = sum_s (E_s - E_ref,s)^2 / N_s + wF sum_{a,c} (F_ac - F_ref,ac)^2.
// The force term is differentiated through the forces' own derivative
// (second order): with u = dL/dF, sum_a u_a . dF_a/dw = -sum_i d/dw [dE_i/dG_i
// . Gdot_i], where Gdot_i = sum_a dG_i/dx_a . u_a is the tangent of atom i's
// SFs along u (the contraction of Training::collectDGdxia,
// Training.cpp:3586-3625).  Per atom, the network is run forward with that
// tangent and reversed once for both terms (the reference's calculateDEdc and
// calculateDFdc, NeuralNetwork.cpp:444-527, compute the same quantities per
// force component).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "train.hpp"
#include "nnpx.h"

namespace nnpx {
namespace {

constexpr int kBlock = 256;
constexpr size_t kGradLds = 65536;  // LDS a gradient block may use
constexpr int kGradTile = 16;       // atoms of its largest tile
constexpr int kGradBlocks = 512;    // blocks worth making: two per CU

// Activation, first and second derivative (NeuralNetwork::propagateLayer,
// NeuralNetwork.cpp:761-896).
template <typename T>
__device__ inline T act2(int a, T x, T& d1, T& d2)
{
    const T EXP_LIMIT = (T)35.0;
    T v;
    switch (a) {
    case AF_IDENTITY: d1 = 1; d2 = 0; return x;
    case AF_TANH: v = tanh(x); d1 = 1 - v * v; d2 = -2 * v * (1 - v * v); return v;
    case AF_LOGISTIC:
        if (x > EXP_LIMIT) { d1 = 0; d2 = 0; return 1; }
        if (x < -EXP_LIMIT) { d1 = 0; d2 = 0; return 0; }
        v = 1 / (1 + exp(-x)); d1 = v * (1 - v); d2 = v * (1 - v) * (1 - 2 * v); return v;
    case AF_SOFTPLUS:
        if (x > EXP_LIMIT) { d1 = 1; d2 = 0; return x; }
        if (x < -EXP_LIMIT) { d1 = 0; d2 = 0; return 0; }
        {
            const T t = exp(x);
            const T s = 1 / (1 + 1 / t);
            d1 = s; d2 = s * (1 - s);
            return log(1 + t);
        }
    case AF_RELU:
        d2 = 0;
        if (x > 0) { d1 = 1; return x; }
        d1 = 0; return 0;
    case AF_GAUSSIAN: { const T t = exp(-(T)0.5 * x * x); d1 = -x * t; d2 = (x * x - 1) * t; return t; }
    case AF_COS: { const T t = cos(x); d1 = -sin(x); d2 = -t; return t; }
    case AF_REVLOGISTIC:
        v = 1 / (1 + exp(-x)); d1 = v * (v - 1); d2 = v * (v - 1) * (1 - 2 * v); return 1 - v;
    case AF_EXP: v = exp(-x); d1 = -v; d2 = v; return v;
    case AF_HARMONIC: d1 = 2 * x; d2 = 2; return x * x;
    }
    d1 = 0; d2 = 0;
    return 0;
}

// u = 2 wF (F - F_ref); cE_s = 2 (E_s - E_ref,s) / N_s; loss terms.
__global__ __launch_bounds__(kBlock) void k_residual(const double* __restrict__ F, const double* __restrict__ Fref,
                                                     const double* __restrict__ E, const double* __restrict__ Eref,
                                                     const int* __restrict__ atom_off, int natoms, int nstruct,
                                                     double wF, double* __restrict__ u, double* __restrict__ cE,
                                                     double* __restrict__ loss)
{
    __shared__ double part[kBlock / 64];
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    double sq = 0.0;
    if (t < natoms)
        for (int k = 0; k < 3; ++k) {
            const size_t q = 3 * (size_t)t + k;
            const double d = F[q] - Fref[q];
            u[q] = 2.0 * wF * d;
            sq += d * d;
        }
    sq = wave_sum(sq);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = sq;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0.0;
        for (int w = 0; w < kBlock / 64; ++w) s += part[w];
        atomicAdd(loss + 2, wF * s);
    }
    if (t < nstruct) {
        const double n = (double)(atom_off[t + 1] - atom_off[t]);
        const double r = E[t] - Eref[t];
        cE[t] = n > 0 ? 2.0 * r / n : 0.0;
        if (n > 0) atomicAdd(loss + 1, r * r / n);
    }
}

// Tangent from the stored dG/dr: Gdot_iq = dGself_iq . u_i + sum over i's
// neighbour entries (self images included) of dGnbr . u_j.  One wave per
// atom, lanes over SFs.
__global__ __launch_bounds__(64) void k_tangent64(const ModelT* __restrict__ M, SysView s,
                                                  const double* __restrict__ dGself, const double* __restrict__ dGnbr,
                                                  int S, const int* __restrict__ islot, const double* __restrict__ u,
                                                  double* __restrict__ Gdot, int ldG)
{
    const int i = blockIdx.x;
    const int e = s.elem[i];
    const int nsf = M->el[e].nsf;
    const int n = s.nb_n[i];
    const size_t base = (size_t)i * s.cap;
    const double* ui = u + 3 * (size_t)i;
    for (int q = threadIdx.x; q < nsf; q += kWave) {
        const double* ds = dGself + ((size_t)i * ldG + q) * 3;
        double acc = ds[0] * ui[0] + ds[1] * ui[1] + ds[2] * ui[2];
        for (int k = 0; k < n; ++k) {
            const int j = s.nb_j[base + k];
            const int t = islot[(e * kMaxElem + s.elem[j]) * kMaxSF + q];
            if (t < 0) continue;
            const double* d = dGnbr + ((base + k) * S + t) * 3;
            const double* uj = u + 3 * (size_t)j;
            acc += d[0] * uj[0] + d[1] * uj[1] + d[2] * uj[2];
        }
        Gdot[(size_t)i * ldG + q] = acc;
    }
}

// Atoms of one 16-byte LDS load, and the padded row length of a neuron's atoms
// (rows stay 16-byte aligned).
template <typename T>
__host__ __device__ constexpr int vec_atoms(int ta)
{
    return ta < (int)(16 / sizeof(T)) ? ta : (int)(16 / sizeof(T));
}
template <typename T>
__host__ __device__ constexpr int tile_row(int ta)
{
    return ta + vec_atoms<T>(ta);
}

// Network forward with the tangent and one reverse pass for
// Phi_i = cE_s E_i - dE_i/dG . Gdot_i, and dPhi/dw summed over atoms in FP64.
//
// A block of four waves takes a.per_block atoms of one element in tiles of TA
// atoms: every (neuron, atom) pair of a layer is a thread's, so the layers'
// dependent steps are shared by TA atoms.  The tile's activations stay in LDS
// ([neuron][atom], padded rows: the connection sums read neighbouring neurons'
// atoms, 16 bytes a load), and the element's weights beside them where they
// fit (WLDS; 16 lanes share each read).  Then each connection is a thread's
// and sums its TA atoms in order in registers.
//   One summed gradient (ldgrad = 0): the sums over the block's tiles are kept
// in LDS (acc_lds) or, for networks too large for it, in the block's own row of
// a.part; k_grad_sum adds the rows in block order (no atomics, the same sum on
// every run).
//   One gradient per structure: a connection's sum goes to the structure's row
// with an atomic when the structure changes (the atoms of a tile are in index
// order, so each structure's are contiguous).
// Bound by latency (LDS reads; 50-25-25-1 networks need only 23 kFLOP per
// atom).  41,000 atoms in FP32: 664 us with one wave taking 32 atoms in series,
// 189 us in tiles with the weights read through L1, 133 us with them in LDS;
// 5,100 atoms in FP64: 542 -> 57 us; 1,300 atoms: 535 -> 26 us.
template <typename T, int TA, bool WLDS>
__global__ __launch_bounds__(kBlock) void k_grad(const ModelT* __restrict__ M, GradArgs a)
{
    constexpr int LD = tile_row<T>(TA);
    constexpr int NG = kBlock / TA;  // neurons a pass of the block covers
    constexpr int V = vec_atoms<T>(TA);
    typedef T vec __attribute__((ext_vector_type(V)));
    extern __shared__ double gsm[];
    const int tid = threadIdx.x;
    const int ta = tid % TA, tg = tid / TA;
    int e = 0;
    while (e + 1 < a.nelem && (int)blockIdx.x >= a.blk_off[e + 1]) ++e;
    const NNT& N = M->el[e].nn;
    const int nl = N.nl;
    const int nconn = a.nconn[e];
    double* acc = a.acc_lds ? gsm : a.part ? a.part + (size_t)blockIdx.x * a.nconn_max : nullptr;
    // LDS: the input layer's h and hdot; per layer h, hdot, f' and f'' adot;
    // the adjoints of the current layer (ab, ad) and of the one below (hb, hd)
    T* p = reinterpret_cast<T*>(gsm + (a.acc_lds ? (a.nconn_max + 1) / 2 * 2 : 0));  // 16-byte aligned
    T *H[kMaxLayers], *Hd[kMaxLayers], *D1[kMaxLayers], *D2[kMaxLayers];
    for (int l = 0; l < nl; ++l) {
        const int w = N.n[l] * LD;
        H[l] = p;
        Hd[l] = p + w;
        D1[l] = p + 2 * w;
        D2[l] = p + 3 * w;
        p += (l ? 4 : 2) * w;
    }
    T* hb = p;
    T* hd = hb + a.max_hidden * LD;
    T* ab = hd + a.max_hidden * LD;
    T* ad = ab + a.max_hidden * LD;
    T* wl = ad + a.max_hidden * LD;  // WLDS: the element's connections, in their order
    const double* wt = a.w + a.nweights;  // transposed copy [in][out]
    const int first = a.atom_off[e] + ((int)blockIdx.x - a.blk_off[e]) * a.per_block;
    const int last = min(first + a.per_block, a.atom_off[e + 1]);
    if (a.ldgrad == 0)
        for (int x = tid; x < nconn; x += kBlock) acc[x] = 0.0;
    if constexpr (WLDS) {
        int o = 0;
        for (int l = 1; l < nl; ++l) {
            const int nw = N.n[l - 1] * N.n[l];
            for (int x = tid; x < nw; x += kBlock) wl[o + x] = (T)wt[N.woff[l] + x];
            for (int x = tid; x < N.n[l]; x += kBlock) wl[o + nw + x] = (T)a.w[N.boff[l] + x];
            o += nw + N.n[l];
        }
    }
    for (int t0 = first; t0 < last; t0 += TA) {
        const int cnt = min(TA, last - t0);
        // rows past the tile's atoms repeat the last atom; their sums are not used
        const int mine = a.atoms[t0 + min(ta, cnt - 1)];
        __syncthreads();  // the previous tile's activations are read
        for (int k = tg; k < N.n[0]; k += NG) {
            H[0][k * LD + ta] = (T)a.G[(size_t)mine * a.ldG + k];
            Hd[0][k * LD + ta] = (T)a.Gdot[(size_t)mine * a.ldG + k];
        }
        __syncthreads();
        int cw = 0;  // the layer's first connection (NeuralNetwork::setConnections, NeuralNetwork.cpp:147-169)
        for (int l = 1; l < nl; ++l) {
            const int nin = N.n[l - 1], nout = N.n[l];
            const double* w = wt + N.woff[l];
            const double* b = a.w + N.boff[l];
            const T* wc = wl + cw;
            cw += (nin + 1) * nout;
            const T* hin = H[l - 1] + ta;
            const T* hdin = Hd[l - 1] + ta;
            // two neurons per thread and pass share the loads of h and hdot
            for (int k = tg; k < nout; k += 2 * NG) {
                const bool two = k + NG < nout;
                const int k2 = two ? k + NG : k;
                T x = 0, xd = 0, y = 0, yd = 0;
#pragma unroll 4
                for (int j = 0; j < nin; ++j) {
                    const T w1 = WLDS ? wc[j * nout + k] : (T)w[(size_t)j * nout + k];
                    const T w2 = WLDS ? wc[j * nout + k2] : (T)w[(size_t)j * nout + k2];
                    const T h = hin[j * LD], q = hdin[j * LD];
                    x += w1 * h;
                    xd += w1 * q;
                    y += w2 * h;
                    yd += w2 * q;
                }
                auto put = [&](int n, T v, T vd) {
                    v += WLDS ? wc[nin * nout + n] : (T)b[n];
                    if (N.normalize) { v /= (T)nin; vd /= (T)nin; }
                    T d1, d2;
                    H[l][n * LD + ta] = act2<T>(N.act[l], v, d1, d2);
                    D1[l][n * LD + ta] = d1;
                    D2[l][n * LD + ta] = d2 * vd;
                    Hd[l][n * LD + ta] = d1 * vd;
                };
                put(k, x, xd);
                if (two) put(k2, y, yd);
            }
            __syncthreads();
        }
        // seeds: dPhi/dE = cE, dPhi/d(dE/dG . Gdot) = -1
        if (tg == 0) {
            hb[ta] = (T)a.cE[a.sid[mine]];
            hd[ta] = (T)-1;
        }
        __syncthreads();
        for (int l = nl - 1; l >= 1; --l) {
            const int nin = N.n[l - 1], nout = N.n[l];
            cw -= (nin + 1) * nout;
            const T inv = N.normalize ? (T)1 / (T)nin : (T)1;
            for (int k = tg; k < nout; k += NG) {
                const int x = k * LD + ta;
                ab[x] = (hb[x] * D1[l][x] + hd[x] * D2[l][x]) * inv;
                ad[x] = hd[x] * D1[l][x] * inv;
            }
            __syncthreads();
            // connections: weights (j, k), then the biases (a unit input)
            for (int x = tid; x < (nin + 1) * nout; x += kBlock) {
                const int j = x / nout, k = x - j * nout;
                const bool bias = j == nin;
                const T* hin = H[l - 1] + (bias ? 0 : j) * LD;
                const T* hdin = Hd[l - 1] + (bias ? 0 : j) * LD;
                const T* bk = ab + k * LD;
                const T* dk = ad + k * LD;
                auto term = [&](int r) { return bias ? (double)bk[r] : (double)(bk[r] * hin[r] + dk[r] * hdin[r]); };
                double sum = 0.0;
                if (a.ldgrad == 0) {
                    if (cnt == TA && !bias) {
#pragma unroll
                        for (int r = 0; r < TA; r += V) {
                            const vec h = *reinterpret_cast<const vec*>(hin + r), q = *reinterpret_cast<const vec*>(hdin + r);
                            const vec b = *reinterpret_cast<const vec*>(bk + r), d = *reinterpret_cast<const vec*>(dk + r);
#pragma unroll
                            for (int v = 0; v < V; ++v) sum += (double)(b[v] * h[v] + d[v] * q[v]);
                        }
                    } else {
                        for (int r = 0; r < cnt; ++r) sum += term(r);
                    }
                    acc[cw + x] += sum;
                } else {
                    int cur = a.sid[a.atoms[t0]];
                    for (int r = 0; r < cnt; ++r) {
                        const int si = a.sid[a.atoms[t0 + r]];
                        if (si != cur) {
                            atomicAdd(a.grad + (size_t)cur * a.ldgrad + a.coff[e] + cw + x, sum);
                            sum = 0.0;
                            cur = si;
                        }
                        sum += term(r);
                    }
                    atomicAdd(a.grad + (size_t)cur * a.ldgrad + a.coff[e] + cw + x, sum);
                }
            }
            if (l > 1) {
                const double* w = a.w + N.woff[l];  // [out][in]
                const T* wc = wl + cw;              // [in][out]
                for (int j = tg; j < nin; j += 2 * NG) {
                    const bool two = j + NG < nin;
                    const int j2 = two ? j + NG : j;
                    T sb = 0, sd = 0, ub = 0, ud = 0;
#pragma unroll 4
                    for (int k = 0; k < nout; ++k) {
                        const T w1 = WLDS ? wc[j * nout + k] : (T)w[(size_t)k * nin + j];
                        const T w2 = WLDS ? wc[j2 * nout + k] : (T)w[(size_t)k * nin + j2];
                        const T vb = ab[k * LD + ta], vd = ad[k * LD + ta];
                        sb += w1 * vb;
                        sd += w1 * vd;
                        ub += w2 * vb;
                        ud += w2 * vd;
                    }
                    hb[j * LD + ta] = sb;
                    hd[j * LD + ta] = sd;
                    if (two) {
                        hb[j2 * LD + ta] = ub;
                        hd[j2 * LD + ta] = ud;
                    }
                }
                __syncthreads();
            }
        }
    }
    if (a.ldgrad == 0 && a.acc_lds) {
        double* row = a.part + (size_t)blockIdx.x * a.nconn_max;
        __syncthreads();
        for (int x = tid; x < nconn; x += kBlock) row[x] = acc[x];
    }
}

// Adds the blocks' rows of each element, in block order per slice and the
// slices in order: 64 connections per block, sixteen slices of the rows.
__global__ __launch_bounds__(1024) void k_grad_sum(GradArgs a)
{
    constexpr int kSlices = 16;
    __shared__ double sl[kSlices][kWave];
    const int e = blockIdx.y;
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const int x = blockIdx.x * kWave + lane;
    const int b0 = a.blk_off[e], nb = a.blk_off[e + 1] - b0;
    const int per = (nb + kSlices - 1) / kSlices;
    double v = 0.0;
    if (x < a.nconn[e]) {
        const double* row = a.part + (size_t)b0 * a.nconn_max + x;
        const int q1 = min(nb, (w + 1) * per);
#pragma unroll 8
        for (int q = w * per; q < q1; ++q) v += row[(size_t)q * a.nconn_max];
    }
    sl[w][lane] = v;
    __syncthreads();
    if (w == 0 && x < a.nconn[e]) {
        for (int q = 1; q < kSlices; ++q) v += sl[q][lane];
        a.grad[a.coff[e] + x] = v;
    }
}

}  // namespace

void launch_residual(const double* F, const double* Fref, const double* E, const double* Eref, const int* atom_off,
                     int natoms, int nstruct, double wF, double* u, double* cE, double* loss, hipStream_t stream)
{
    const int n = std::max(natoms, nstruct);
    hipLaunchKernelGGL(k_residual, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, stream, F, Fref, E, Eref,
                       atom_off, natoms, nstruct, wF, u, cE, loss);
}

void launch_tangent64(const ModelT* m, const SysView& s, const double* dGself, const double* dGnbr, int S,
                      const int* islot, const double* u, double* Gdot, int ldG, hipStream_t stream)
{
    if (s.natoms == 0) return;
    hipLaunchKernelGGL(k_tangent64, dim3(s.natoms), dim3(kWave), 0, stream, m, s, dGself, dGnbr, S, islot, u, Gdot,
                       ldG);
}

size_t grad_act_bytes(const GradArgs& a, bool fp32)
{
    const size_t t = fp32 ? sizeof(float) : sizeof(double);
    return t * ((size_t)5 * kMaxLayers * a.maxw + 6 * (size_t)a.maxw);
}

namespace {

// LDS bytes of a tile of ta atoms.
size_t tile_bytes(const GradArgs& a, int ta, size_t t)
{
    const size_t row = t == sizeof(float) ? tile_row<float>(ta) : tile_row<double>(ta);
    return t * row * (2 * (size_t)a.max_in + 4 * (size_t)a.sum_hidden + 4 * (size_t)a.max_hidden);
}

}  // namespace

int plan_grad(GradArgs& a, const ModelT& t, const int* elem_count, const int* elem_off, int per_block)
{
    a.nelem = t.nelem;
    a.maxw = std::max(t.max_width, t.max_sf);
    a.nweights = t.nweights;
    a.ldG = t.max_sf;
    int total = 0, natoms = 0;
    for (int e = 0; e < t.nelem; ++e) {
        const NNT& N = t.el[e].nn;
        int n = 0, hidden = 0;
        for (int l = 1; l < N.nl; ++l) {
            n += (N.n[l - 1] + 1) * N.n[l];
            hidden += N.n[l];
            a.max_hidden = std::max(a.max_hidden, N.n[l]);
        }
        a.max_in = std::max(a.max_in, N.n[0]);
        a.sum_hidden = std::max(a.sum_hidden, hidden);
        a.coff[e] = total;
        a.nconn[e] = n;
        a.nconn_max = std::max(a.nconn_max, n);
        total += n;
        natoms += elem_count[e];
    }
    // at most per_block atoms per block, fewer (whole tiles) while that makes
    // no more than two blocks per CU; the tile itself shrinks where one of 16
    // would leave CUs without a block
    int ta = kGradTile;
    while (ta > 1 && natoms < ta * kGradBlocks / 2) ta /= 2;
    const int target = (natoms + kGradBlocks - 1) / kGradBlocks;
    a.per_block = std::min(per_block, std::max(1, (target + ta - 1) / ta) * ta);
    int blocks = 0;
    for (int e = 0; e < t.nelem; ++e) {
        a.blk_off[e] = blocks;
        a.atom_off[e] = elem_off[e];
        blocks += (elem_count[e] + a.per_block - 1) / a.per_block;
    }
    a.blk_off[t.nelem] = blocks;
    a.atom_off[t.nelem] = elem_off[t.nelem];
    return blocks;
}

void launch_grad(const ModelT* m, GradArgs a, int blocks, bool fp32, hipStream_t stream)
{
    if (a.ldgrad == 0 && !a.part) throw Error{NNPX_ERR_STATE, "gradient: no buffer for the blocks' sums"};
    const size_t t = fp32 ? sizeof(float) : sizeof(double);
    if (grad_act_bytes(a, fp32) > kGradLds)
        throw Error{NNPX_ERR_UNSUPPORTED, "network too wide for the gradient kernel's LDS staging"};
    // the largest tile, no larger than a block's atoms (the next power of
    // two), whose activations fit with the weights, and without them where
    // no tile does; then the block's sums beside them if they fit
    const size_t wts = t * (size_t)a.nconn_max;
    const bool wlds = tile_bytes(a, 1, t) + wts <= kGradLds;
    const size_t extra = wlds ? wts : 0;
    int ta = kGradTile;
    while (ta > 1 && (tile_bytes(a, ta, t) + extra > kGradLds || ta / 2 >= a.per_block)) ta /= 2;
    size_t lds = tile_bytes(a, ta, t) + extra;
    if (lds > kGradLds) throw Error{NNPX_ERR_UNSUPPORTED, "network too wide for the gradient kernel's LDS staging"};
    const size_t sums = sizeof(double) * (size_t)((a.nconn_max + 1) / 2 * 2);
    a.acc_lds = a.ldgrad == 0 && lds + sums <= kGradLds ? 1 : 0;
    if (a.acc_lds) lds += sums;
    if (blocks > 0) {
        auto launch = [&](auto ty, auto n) {
            using T = decltype(ty);
            constexpr int TA = decltype(n)::value;
            if (wlds) hipLaunchKernelGGL((k_grad<T, TA, true>), dim3(blocks), dim3(kBlock), lds, stream, m, a);
            else hipLaunchKernelGGL((k_grad<T, TA, false>), dim3(blocks), dim3(kBlock), lds, stream, m, a);
        };
        auto pick = [&](auto ty) {
            switch (ta) {
            case 16: launch(ty, std::integral_constant<int, 16>{}); break;
            case 8: launch(ty, std::integral_constant<int, 8>{}); break;
            case 4: launch(ty, std::integral_constant<int, 4>{}); break;
            case 2: launch(ty, std::integral_constant<int, 2>{}); break;
            default: launch(ty, std::integral_constant<int, 1>{}); break;
            }
        };
        if (fp32) pick(0.f);
        else pick(0.0);
    }
    if (a.ldgrad == 0)
        hipLaunchKernelGGL(k_grad_sum, dim3((a.nconn_max + kWave - 1) / kWave, a.nelem), dim3(1024), 0, stream, a);
}

}  // namespace nnpx
