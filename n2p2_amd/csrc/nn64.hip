// FP64 atomic neural networks and per-structure energies (plain form).
//
// NeuralNetwork::propagate / propagateLayer (NeuralNetwork.cpp:386-394,
// 761-896) for every atom of an element, and dE/dG by reverse-mode
// (adjoint) accumulation instead of the reference's forward-mode
// NeuralNetwork::calculateDEdG (NeuralNetwork.cpp:396-442); both give
// dE/dG_k = sum over paths of W * f' products, the adjoint in one backward
// sweep.
//
// Bound by issue (a load, an LDS read and an FMA per weight and atom) and, for
// few atoms, by the chain of layers; the weights stay in the caches.  Teams of
// 16, 32 or 64 threads (the widest hidden layer) take one or two atoms each,
// threads over neurons: with 25 neurons a wave serves two to four atoms at
// once instead of one on 25 of its lanes, and a weight loaded serves them all.
// Sums run in the order of one atom alone.  50-25-25-1 networks, with dE/dG:
// 192 atoms 19.9 -> 11.5 us, 12,288 atoms 89.8 -> 24.9 us (27,783: 162 -> 48).
// Weights are read in two layouts: W^T ([in][out]) so lanes read consecutive
// outputs in the forward sweep, W ([out][in]) for the backward sweep.
#include "kernels.hpp"
#include "nnpx.h"

namespace nnpx {
namespace {

constexpr int kNNThreads = 256;
constexpr int kNNWaves = kNNThreads / kWave;
// One atom per team below, two from here on: 1,536 atoms 12.0 against 14.3 us,
// 3,000 15.9 against 14.7, 12,288 40.7 against 24.9; four are no faster at any
// size and 12 us slower for wide inputs.
constexpr int kNNTwo = 2048;
// LDS per block up to which a team takes two atoms (four blocks per CU)
constexpr size_t kNNLds = 40 * 1024;

__device__ inline double act_fwd(int a, double x, double& dfdx)
{
    const double EXP_LIMIT = 35.0;  // NeuralNetwork.cpp EXP_LIMIT
    double v;
    switch (a) {
    case AF_IDENTITY: dfdx = 1.0; return x;
    case AF_TANH: v = tanh(x); dfdx = 1.0 - v * v; return v;
    case AF_LOGISTIC:
        if (x > EXP_LIMIT) { dfdx = 0.0; return 1.0; }
        if (x < -EXP_LIMIT) { dfdx = 0.0; return 0.0; }
        v = 1.0 / (1.0 + exp(-x)); dfdx = v * (1.0 - v); return v;
    case AF_SOFTPLUS:
        if (x > EXP_LIMIT) { dfdx = 1.0; return x; }
        if (x < -EXP_LIMIT) { dfdx = 0.0; return 0.0; }
        { const double t = exp(x); dfdx = 1.0 / (1.0 + 1.0 / t); return log(1.0 + t); }
    case AF_RELU:
        if (x > 0.0) { dfdx = 1.0; return x; }
        dfdx = 0.0; return 0.0;
    case AF_GAUSSIAN: { const double t = exp(-0.5 * x * x); dfdx = -x * t; return t; }
    case AF_COS: dfdx = -sin(x); return cos(x);
    case AF_REVLOGISTIC: v = 1.0 / (1.0 + exp(-x)); dfdx = v * (v - 1.0); return 1.0 - v;
    case AF_EXP: v = exp(-x); dfdx = -v; return v;
    case AF_HARMONIC: dfdx = 2.0 * x; return x * x;
    }
    dfdx = 0.0;
    return 0.0;
}

// Doubles per atom in LDS.
__host__ __device__ inline int nn_stride(int maxw, int maxh, int layers)
{
    return (2 * maxw + (layers - 1) * maxh) | 1;
}

struct NNArgs {
    const double* w;    // [o][i] weights + biases (model layout)
    const double* wt;   // [i][o] transposed weights
    const int* atoms;   // atom indices sorted by element
    int blk_off[kMaxElem + 1];  // first block of each element
    int atom_off[kMaxElem + 1]; // first atom (in atoms[]) of each element
    int nelem;
    int layers;         // most layers of any element's network
};

template <int WIDTH, int A>
__global__ __launch_bounds__(kNNThreads) void k_nn64(const ModelT* __restrict__ M, NNArgs a,
                                                      NNIO io, int maxw, int maxh)
{
    extern __shared__ double sm[];
    const int team = threadIdx.x / WIDTH, lane = threadIdx.x & (WIDTH - 1);
    int e = 0;
    while (e + 1 < a.nelem && (int)blockIdx.x >= a.blk_off[e + 1]) ++e;
    const NNT& N = M->el[e].nn;
    const int nl = N.nl;
    // per atom in LDS: two activation buffers (any layer, input included) and
    // f' of every hidden/output layer; odd strides keep the atoms of a wave on
    // different banks
    const int stride = nn_stride(maxw, maxh, a.layers);
    double* base = sm + (size_t)team * A * stride;
    const int first = a.atom_off[e] + (((int)blockIdx.x - a.blk_off[e]) * (kNNThreads / WIDTH) + team) * A;
    const int cnt = min(A, a.atom_off[e + 1] - first);  // <= 0: a team past the last atom computes nothing
    if (cnt <= 0) return;
    int atom[A];
#pragma unroll
    for (int m = 0; m < A; ++m) {
        atom[m] = a.atoms[first + min(m, cnt - 1)];  // past the last: the last again, not stored
        const double* g = io.G + (size_t)atom[m] * io.ldG;
        for (int k = lane; k < N.n[0]; k += WIDTH) base[m * stride + k] = g[k];
    }
    wave_fence();
    int vin = 0, vout = maxw;           // offsets of the buffers
    const int dfd = 2 * maxw - maxh;    // [layer][maxh], from layer 1
    for (int l = 1; l < nl; ++l) {
        const int nin = N.n[l - 1], nout = N.n[l];
        const double* wt = a.wt + N.woff[l];
        const double* b = a.w + N.boff[l];
        for (int k = lane; k < nout; k += WIDTH) {
            double x[A];
#pragma unroll
            for (int m = 0; m < A; ++m) x[m] = 0.0;
#pragma unroll 5
            for (int j = 0; j < nin; ++j) {
                const double w = wt[(size_t)j * nout + k];
#pragma unroll
                for (int m = 0; m < A; ++m) x[m] += w * base[m * stride + vin + j];
            }
#pragma unroll
            for (int m = 0; m < A; ++m) {
                x[m] += b[k];
                if (N.normalize) x[m] /= nin;
                double df;
                base[m * stride + vout + k] = act_fwd(N.act[l], x[m], df);
                base[m * stride + dfd + l * maxh + k] = df;
            }
        }
        wave_fence();
        const int t = vin; vin = vout; vout = t;
    }
#pragma unroll
    for (int m = 0; m < A; ++m)
        if (lane == 0 && m < cnt) io.energy[atom[m]] = base[m * stride + vin];
    if (!io.dEdG) return;
    // Backward: delta_l = dE/dx_l (pre-activation), delta_{L-1} = f'_out.
    int din = vout;  // free buffer
    int dout = vin;
    wave_fence();
#pragma unroll
    for (int m = 0; m < A; ++m)
        if (lane == 0) base[m * stride + din] = base[m * stride + dfd + (nl - 1) * maxh];
    wave_fence();
    for (int l = nl - 1; l >= 1; --l) {
        const int nin = N.n[l - 1], nout = N.n[l];
        const double* w = a.w + N.woff[l];
        const double norm = N.normalize ? 1.0 / nin : 1.0;
        for (int j = lane; j < nin; j += WIDTH) {
            double s[A];
#pragma unroll
            for (int m = 0; m < A; ++m) s[m] = 0.0;
#pragma unroll 5
            for (int k = 0; k < nout; ++k) {
                const double x = w[(size_t)k * nin + j];
#pragma unroll
                for (int m = 0; m < A; ++m) s[m] += x * base[m * stride + din + k];
            }
#pragma unroll
            for (int m = 0; m < A; ++m) {
                if (N.normalize) s[m] *= norm;
                if (l - 1 >= 1) s[m] *= base[m * stride + dfd + (l - 1) * maxh + j];
                if (l > 1) base[m * stride + dout + j] = s[m];
                else if (m < cnt) io.dEdG[(size_t)atom[m] * io.ldG + j] = s[m];
            }
        }
        wave_fence();
        const int t = din; din = dout; dout = t;
    }
}

// One block per structure, fixed-order tree sum.
// Per-structure sum of the atomic energies, one block per structure: four
// independent strided partial sums per thread keep several loads in flight,
// then a fixed-order tree in LDS (deterministic from run to run).
constexpr int kEnergyThreads = 1024;
__global__ __launch_bounds__(kEnergyThreads) void k_energy(const double* atomE, const int* off, double* E)
{
    __shared__ double red[kEnergyThreads];
    const int st = blockIdx.x;
    const int b = off[st], e = off[st + 1];
    const int t = (int)threadIdx.x;
    double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
    int q = b + t;
    for (; q + 3 * kEnergyThreads < e; q += 4 * kEnergyThreads) {
        s0 += atomE[q];
        s1 += atomE[q + kEnergyThreads];
        s2 += atomE[q + 2 * kEnergyThreads];
        s3 += atomE[q + 3 * kEnergyThreads];
    }
    for (; q < e; q += kEnergyThreads) s0 += atomE[q];
    red[t] = (s0 + s1) + (s2 + s3);
    __syncthreads();
    for (int o = kEnergyThreads / 2; o > 0; o >>= 1) {
        if (t < o) red[t] += red[t + o];
        __syncthreads();
    }
    if (t == 0) E[st] = red[0];
}

}  // namespace

void launch_nn64(const ModelT* m, const ModelT& hm, const double* w, const int* elem_atoms,
                 const int* elem_count_host, const int* elem_off_host, const NNIO& io,
                 hipStream_t stream)
{
    NNArgs a{};
    a.w = w;
    a.wt = w + hm.nweights;
    a.atoms = elem_atoms;
    a.nelem = hm.nelem;
    for (int e = 0; e < hm.nelem; ++e) a.layers = std::max(a.layers, hm.el[e].nn.nl);
    const int maxw = hm.max_width, maxh = hm.max_hidden;
    const size_t atom_bytes = sizeof(double) * nn_stride(maxw, maxh, a.layers);
    // what was refused stays refused: four atoms' buffers, with all layers
    if (sizeof(double) * (size_t)kNNWaves * (2 * maxw + kMaxLayers * maxh) > 65536)
        throw Error{NNPX_ERR_UNSUPPORTED, "network too wide for the FP64 NN kernel's LDS staging"};
    int total = 0;
    for (int e = 0; e < hm.nelem; ++e) total += elem_count_host[e];
    int width = maxh <= 16 ? 16 : maxh <= 32 ? 32 : 64;
    while (width < kWave && kNNThreads / width * atom_bytes > 65536) width *= 2;
    const int A = total >= kNNTwo && kNNThreads / width * 2 * atom_bytes <= kNNLds ? 2 : 1;
    const int tile = kNNThreads / width * A;
    const size_t lds = tile * atom_bytes;
    int blocks = 0;
    for (int e = 0; e < hm.nelem; ++e) {
        a.blk_off[e] = blocks;
        a.atom_off[e] = elem_off_host[e];
        blocks += (elem_count_host[e] + tile - 1) / tile;
    }
    a.blk_off[hm.nelem] = blocks;
    a.atom_off[hm.nelem] = elem_off_host[hm.nelem];
    if (blocks == 0) return;
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kNNThreads), lds, stream, m, a, io, maxw, maxh);
    };
    switch (width * 8 + A) {
    case 16 * 8 + 1: go(k_nn64<16, 1>); break;
    case 16 * 8 + 2: go(k_nn64<16, 2>); break;
    case 32 * 8 + 1: go(k_nn64<32, 1>); break;
    case 32 * 8 + 2: go(k_nn64<32, 2>); break;
    case 64 * 8 + 1: go(k_nn64<64, 1>); break;
    default: go(k_nn64<64, 2>); break;
    }
}

void launch_energy(const double* atomE, const int* atom_off, int nstruct, double* E,
                   hipStream_t stream)
{
    if (nstruct == 0) return;
    hipLaunchKernelGGL(k_energy, dim3(nstruct), dim3(kEnergyThreads), 0, stream, atomE, atom_off, E);
}

}  // namespace nnpx
