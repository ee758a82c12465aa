// Staging of one atom's neighbours shared by the kernels that put several
// waves on an atom.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace nnpx {

// 64-entry passes of a list with counts of their own (1,024 entries).  A longer
// list (MD lists with a skin: the limit is checked where a list is fitted, and a
// fitted capacity leaves room for more) has the rest of its passes in the last one.
constexpr int kStagePasses = 16;

// Lane of the wave, and the wave's number in the block as a scalar.
__device__ inline int lane_id() { return threadIdx.x & (kWave - 1); }
__device__ inline int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x / kWave); }

// Places the atom's list entries closer than the model's largest cutoff
// (entries beyond it contribute nothing; MD lists built with a skin carry
// them) in slots grouped by neighbour element and in list order within an
// element, so element e's neighbours are the slots eoff[e] .. eoff[e + 1] - 1:
// store(slot, entry, vector, distance, element) for each.  The block's wave w
// (of W) takes the list's 64-entry passes w, w + W, ..., and the one with the
// last of kStagePasses all that follow it; cnt is LDS for kStagePasses *
// kMaxElem counts.  More such entries than capL: only slots
// below capL are stored, flag bit 4 is set (the caller repeats with the full
// capacity) and flags[2] keeps the largest count met.  Returns the slots in
// use; starts and ends with the block in step.
template <int W, typename Store>
__device__ inline int stage_by_element(const ModelT* __restrict__ M, const SysView& s, int i, int capL, int* cnt,
                                       int* eoff, Store&& store)
{
    const int lane = lane_id(), wv = wave_id();
    const StructT& St = s.st[s.sid[i]];
    const int nl = s.nb_n[i];
    const int ne = M->nelem;
    constexpr int kLast = kStagePasses - 1;
    const int passes = (nl + kWave - 1) / kWave, npass = min(passes, kStagePasses);
    const int mine = kLast % W == wv ? passes : npass;  // end of this wave's passes
    const size_t base = (size_t)i * s.cap;
    const double rmax = M->maxCutoff;
    struct Entry {
        double dr[3], d;
        int el;
    };
    auto entry = [&](int p) {
        Entry x{{0.0, 0.0, 0.0}, 0.0, -1};
        const int k = p * kWave + lane;
        if (k < nl) {
            entry_vector(s, i, base + k, St, x.dr);
            x.d = sqrt(x.dr[0] * x.dr[0] + x.dr[1] * x.dr[1] + x.dr[2] * x.dr[2]);
            if (x.d < rmax) x.el = s.elem[s.nb_j[base + k]];
        }
        return x;
    };
    // in-cutoff entries per pass and element; a wave's first passes stay in
    // registers for the placing (lists up to kKeep * W * 64 entries)
    constexpr int kKeep = W >= 4 ? 1 : 4 / W;
    Entry keep[kKeep];
    auto count = [&](int p, int el) {
        for (int e = 0; e < ne; ++e) {
            const int c = __popcll(__ballot(el == e));
            if (lane == 0) {
                int& row = cnt[min(p, kLast) * kMaxElem + e];
                row = p > kLast ? row + c : c;
            }
        }
    };
#pragma unroll
    for (int q = 0; q < kKeep; ++q) {
        const int p = wv + q * W;
        keep[q].el = -1;
        if (p < npass) {
            keep[q] = entry(p);
            count(p, keep[q].el);
        }
    }
    for (int p = wv + kKeep * W; p < mine; p += p < kLast ? W : 1) count(p, entry(p).el);
    __syncthreads();
    // lane e: element e's entries, its first slot, and the next of this wave's pass
    int tot = 0;
    if (lane < ne)
        for (int p = 0; p < npass; ++p) tot += cnt[p * kMaxElem + lane];
    const int incl = wave_incl_scan(tot);
    const int total = lane_value(incl, kWave - 1);
    int next = incl - tot, seen = 0;
    if (wv == 0 && lane <= ne) eoff[lane] = min(lane < ne ? next : total, capL);
    auto place = [&](int p, const Entry& x) {
        for (; seen < p; ++seen)
            if (lane < ne) next += cnt[seen * kMaxElem + lane];
        int pos = -1;
        for (int e = 0; e < ne; ++e) {
            const unsigned long long m = __ballot(x.el == e);
            const int at = lane_value(next, e);
            if (x.el == e)
                pos = at + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                          __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
        }
        if (pos >= 0 && pos < capL) store(pos, p * kWave + lane, x.dr, x.d, x.el);
    };
#pragma unroll
    for (int q = 0; q < kKeep; ++q)
        if (wv + q * W < npass) place(wv + q * W, keep[q]);
    for (int p = wv + kKeep * W; p < mine; p += p < kLast ? W : 1) {
        const Entry x = entry(p);
        place(p, x);
        if (p >= kLast) {  // for the passes that share its row
            for (int e = 0; e < ne; ++e) {
                const int c = __popcll(__ballot(x.el == e));
                if (lane == e) next += c;
            }
            seen = p + 1;
        }
    }
    if (threadIdx.x == 0) {
        if (total > capL) atomicOr(&s.flags[0], 4);
        if (total > __hip_atomic_load(&s.flags[2], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMax(&s.flags[2], total);
    }
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(min(total, capL));
}

}  // namespace nnpx
