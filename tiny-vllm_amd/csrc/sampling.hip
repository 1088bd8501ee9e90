// Token sampling over [rows, vocab] logits: greedy argmax, and temperature /
// top-k / top-p sampling by the exponential race.
//
// Reference behaviour: tinyvllm/sampling.py:21-72 (TorchSampler.sample:
// greedy rows use logits.argmax) and :75-164 (_sample_batch):
//   s = (logit.float() - rowmax) / T; optional top-k; stable descending sort;
//   softmax; drop every token whose preceding cumulative probability exceeds
//   top_p (the first token crossing top_p is kept); choice = argmax p / E,
//   E ~ Exp(1).
//
// MI355X design: no sort of a row. Probability masses are 2^-40 fixed point,
// so every sum is exact and independent of how it is split, and ties on s
// are resolved by token index, which is exactly the stable sort's order.
// With the split workspace the vocabulary is cut into spans over the whole
// chip: row maxima, 2048 bins of the score, the race over the tokens above
// the cut's bin, and an exact cut of that one bin. Rows that the split does
// not take, and calls without its workspace, run one 1024-thread workgroup
// per row: radix selection over an order-preserving 32-bit key of s (four
// 8-bit digit passes, histograms in LDS, three more for ties). Both keep the
// same set and draw the same token. The noise is a counter-based
// Philox4x32-10 stream (Salmon et al., SC'11) keyed by the request seed and
// its sample counter, so a step is reproducible and graph-capturable.
#include "common.h"

namespace tvllm {
namespace {

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / 64;

template <typename T>
__device__ __forceinline__ float load_logit(const T* row, int64_t i) {
    return to_f<T>(row[i]);
}

// Better = larger value; NaN beats numbers; ties go to the lower index.
__device__ __forceinline__ bool better(float a, int64_t ia, float b, int64_t ib) {
    const bool na = a != a, nb = b != b;
    if (na || nb) return na && (!nb || ia < ib);
    return a > b || (a == b && ia < ib);
}

__device__ __forceinline__ void wave_argmax(float& v, int64_t& idx) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const float ov = __shfl_xor(v, off, 64);
        const int64_t oi = __shfl_xor(idx, off, 64);
        if (better(ov, oi, v, idx)) { v = ov; idx = oi; }
    }
}

// Block-wide argmax over W waves; every thread gets the result.
template <int W>
__device__ void block_argmax_w(float& v, int64_t& idx) {
    __shared__ float sv[W];
    __shared__ int64_t si[W];
    wave_argmax(v, idx);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) { sv[w] = v; si[w] = idx; }
    __syncthreads();
    v = sv[0];
    idx = si[0];
    for (int i = 1; i < W; ++i)
        if (better(sv[i], si[i], v, idx)) { v = sv[i]; idx = si[i]; }
    __syncthreads();
}

template <typename T, bool VEC>
__global__ void __launch_bounds__(kThreads)
argmax_kernel(const T* __restrict__ logits, int64_t vocab, int64_t stride,
              int64_t* __restrict__ out);

// ------------------------------------------------------------ sampling ----

// Philox4x32-10 (Salmon, Moraes, Dror, Shaw: "Parallel random numbers: as
// easy as 1, 2, 3", SC'11): 10 rounds of the 4x32 multiply-xor bijection.
__device__ __forceinline__ uint4 philox4x32_10(uint4 ctr, uint2 key) {
    constexpr uint32_t kM0 = 0xD2511F53u, kM1 = 0xCD9E8D57u;
    constexpr uint32_t kW0 = 0x9E3779B9u, kW1 = 0xBB67AE85u;
#pragma unroll
    for (int round = 0; round < 10; ++round) {
        const uint32_t hi0 = __umulhi(kM0, ctr.x), lo0 = kM0 * ctr.x;
        const uint32_t hi1 = __umulhi(kM1, ctr.z), lo1 = kM1 * ctr.z;
        ctr = make_uint4(hi1 ^ ctr.y ^ key.x, lo1, hi0 ^ ctr.w ^ key.y, lo0);
        key.x += kW0;
        key.y += kW1;
    }
    return ctr;
}

// Order-preserving map float -> uint32 (larger float, larger key).
__device__ __forceinline__ uint32_t fkey(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

constexpr double kMassScale = 1099511627776.0;  // 2^40 fixed point

struct RowCtx {
    float mx;     // row max of the logits
    float temp;   // temperature
};

template <typename T>
__device__ __forceinline__ float score_of(const T* row, int64_t i, const RowCtx& c) {
    return (load_logit(row, i) - c.mx) / c.temp;
}

__device__ __forceinline__ uint64_t mass_of(float s) {
    return static_cast<uint64_t>(static_cast<double>(expf(s)) * kMassScale);
}

// Selection result: kept = key > k or (key == k and index <= idx).
struct Cut {
    uint32_t key;
    int64_t idx;
    bool all;  // total weight never exceeds the target: keep everything
};

__device__ __forceinline__ bool kept(const Cut& c, uint32_t key, int64_t i) {
    return c.all || key > c.key || (key == c.key && i <= c.idx);
}

// Finds the first element, in (key descending, index ascending) order among
// elements with in(i), whose inclusive cumulative weight exceeds `target`.
// weight(i) is 1 (MASS = false) or the fixed-point probability mass.
template <typename T, bool MASS, int NT, typename In>
__device__ Cut radix_cut(const T* row, int64_t vocab, const RowCtx& ctx,
                         uint64_t target, In&& in) {
    __shared__ uint64_t hist[256];
    __shared__ uint32_t s_prefix;
    __shared__ uint64_t s_above;
    __shared__ int s_found;
    uint32_t prefix = 0;
    uint64_t above = 0;
    for (int shift = 24; shift >= 0; shift -= 8) {
        for (int b = threadIdx.x; b < 256; b += NT) hist[b] = 0;
        __syncthreads();
        for (int64_t i = threadIdx.x; i < vocab; i += NT) {
            if (!in(i)) continue;
            const float s = score_of(row, i, ctx);
            const uint32_t k = fkey(s);
            if (shift < 24 && ((k ^ prefix) >> (shift + 8)) != 0) continue;
            atomicAdd(reinterpret_cast<unsigned long long*>(&hist[(k >> shift) & 255]),
                      static_cast<unsigned long long>(MASS ? mass_of(s) : 1));
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            uint64_t cum = above;
            int found = -1;
            for (int b = 255; b >= 0; --b) {
                if (cum + hist[b] > target) { found = b; break; }
                cum += hist[b];
            }
            s_found = found;
            s_prefix = found >= 0 ? prefix | (uint32_t(found) << shift) : prefix;
            s_above = cum;
        }
        __syncthreads();
        if (s_found < 0) {
            Cut c{0u, 0, true};
            __syncthreads();
            return c;
        }
        prefix = s_prefix;
        above = s_above;
        __syncthreads();
    }
    // prefix is the boundary key; every tie there has the same weight w.
    // The boundary is the j-th tie in index order, j = (target - above) / w.
    uint64_t w = 1;
    if constexpr (MASS) {
        w = 0;
        // All ties share s, hence the same mass; recompute from any of them.
        __shared__ uint64_t s_w;
        if (threadIdx.x == 0) s_w = 0;
        __syncthreads();
        for (int64_t i = threadIdx.x; i < vocab; i += NT) {
            if (!in(i)) continue;
            const float s = score_of(row, i, ctx);
            if (fkey(s) == prefix) { s_w = mass_of(s); break; }
        }
        __syncthreads();
        w = s_w;
        __syncthreads();
    }
    const uint64_t j = w ? (target - above) / w : 0;
    // Ascending radix select of the j-th tie index (indices < 2^24).
    __shared__ uint32_t ihist[256];
    __shared__ uint32_t s_iprefix;
    __shared__ uint64_t s_ibelow;
    uint32_t iprefix = 0;
    uint64_t below = 0;
    for (int shift = 16; shift >= 0; shift -= 8) {
        for (int b = threadIdx.x; b < 256; b += NT) ihist[b] = 0;
        __syncthreads();
        for (int64_t i = threadIdx.x; i < vocab; i += NT) {
            if (!in(i)) continue;
            const uint32_t ui = static_cast<uint32_t>(i);
            if (shift < 16 && ((ui ^ iprefix) >> (shift + 8)) != 0) continue;
            if (fkey(score_of(row, i, ctx)) != prefix) continue;
            atomicAdd(&ihist[(ui >> shift) & 255], 1u);
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            uint64_t cum = below;
            int found = 255;
            for (int b = 0; b < 256; ++b) {
                if (cum + ihist[b] > j) { found = b; break; }
                cum += ihist[b];
            }
            s_iprefix = iprefix | (uint32_t(found) << shift);
            s_ibelow = cum;
        }
        __syncthreads();
        iprefix = s_iprefix;
        below = s_ibelow;
        __syncthreads();
    }
    return Cut{prefix, static_cast<int64_t>(iprefix), false};
}

// Per-thread running argmax over a row (16-byte vector loads when VEC).
template <typename T, bool VEC>
__device__ __forceinline__ void thread_argmax(const T* row, int64_t vocab, float& best,
                                              int64_t& bi) {
    int64_t tail = 0;
    if constexpr (VEC) {
        const int64_t nvec = vocab / 8;
        const U16x8* rv = reinterpret_cast<const U16x8*>(row);
        // Rows of up to kOnePass * kThreads vectors (vocabularies up to
        // 163840): every load of the thread is issued at once - out-of-range
        // ones read vector 0 and are skipped - so the row costs one memory
        // round trip instead of one per loop iteration.
        constexpr int kOnePass = 20;
        if (nvec <= int64_t(kOnePass) * kThreads) {
            U16x8 raw[kOnePass];
            const uint32_t n32 = uint32_t(nvec);
#pragma unroll
            for (int u = 0; u < kOnePass; ++u) {  // 32-bit offsets from the row base
                const uint32_t c = threadIdx.x + uint32_t(u) * kThreads;
                raw[u] = rv[c < n32 ? c : 0u];
            }
            // Two cheap passes over the registers instead of a NaN-aware
            // compare per element (which left the row scan VALU-bound): the
            // maximum, then the first index holding it. A thread that saw a
            // NaN redoes its elements with the exact compare.
            float m = -INFINITY;
            bool nan = false;
#pragma unroll
            for (int u = 0; u < kOnePass; ++u) {
                const uint32_t c = threadIdx.x + uint32_t(u) * kThreads;
                if (c >= n32) break;
                float x[8];
                unpack8<T>(raw[u], x);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    m = fmaxf(m, x[e]);
                    nan |= x[e] != x[e];
                }
            }
            if (!nan) {
                uint32_t first = UINT32_MAX;
#pragma unroll
                for (int u = 0; u < kOnePass; ++u) {
                    const uint32_t c = threadIdx.x + uint32_t(u) * kThreads;
                    if (c >= n32) break;
                    float x[8];
                    unpack8<T>(raw[u], x);
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        first = x[e] == m ? min(first, c * 8u + uint32_t(e)) : first;
                }
                if (first != UINT32_MAX) {
                    best = m;
                    bi = first;
                }
            } else {
#pragma unroll
                for (int u = 0; u < kOnePass; ++u) {
                    const int64_t c = threadIdx.x + int64_t(u) * kThreads;
                    if (c >= nvec) break;
                    float x[8];
                    unpack8<T>(raw[u], x);
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (better(x[e], c * 8 + e, best, bi)) { best = x[e]; bi = c * 8 + e; }
                }
            }
        } else {
        // Four independent 16-byte loads in flight per thread, then compare
        // in index order (ties keep the lower index either way).
        constexpr int U = 4;
        int64_t c = threadIdx.x;
        for (; c + (U - 1) * kThreads < nvec; c += U * kThreads) {
            U16x8 raw[U];
#pragma unroll
            for (int u = 0; u < U; ++u) raw[u] = rv[c + u * kThreads];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                float x[8];
                unpack8<T>(raw[u], x);
                const int64_t base = (c + u * kThreads) * 8;
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (better(x[e], base + e, best, bi)) { best = x[e]; bi = base + e; }
            }
        }
        for (; c < nvec; c += kThreads) {
            float x[8];
            unpack8<T>(rv[c], x);
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (better(x[e], c * 8 + e, best, bi)) { best = x[e]; bi = c * 8 + e; }
        }
        }
        tail = nvec * 8;
    }
    for (int64_t i = tail + threadIdx.x; i < vocab; i += kThreads) {
        const float x = load_logit(row, i);
        if (better(x, i, best, bi)) { best = x; bi = i; }
    }
}

// Greedy scan split over workgroups: row r's span s (kPartSpan elements)
// is scanned by one 256-thread workgroup, 4 vectors per thread in flight at
// once; the sampling kernel combines the spans. One 1024-thread workgroup
// per row left the scan VALU-bound on one CU (28 us per 151936-wide row);
// spans of 4 / 8 / 16 vectors per thread measured 14.1 / 15.6 / 21.1 us at
// 64 rows.
constexpr int kPartThreads = 256;
constexpr int kPartVecs = 4;
constexpr int64_t kPartSpan = int64_t(kPartThreads) * kPartVecs * 8;

struct ArgPart {
    float v;
    int32_t i;  // -1: empty span
};

// Bins of width 1/64 over s in (-32, 0]. Monotonic in s (a product with a
// power of two, truncated), so bins respect the key order. The last bin takes
// everything below: its masses are 0 in 2^-40 fixed point (e^-31.9 = 1.4e-14),
// and it is not counted. 16-bit logits of a trained or random head put tens
// to a few hundred tokens in a bin; 4096 list entries hold bins of heads with
// a standard deviation down to about 0.25.
constexpr int kBins = 2048;
constexpr float kBinScale = 64.f;
constexpr int kListCap = 4096;

__device__ __forceinline__ int bin_of(float s) {
    return int(fminf(-s * kBinScale, float(kBins - 1)));
}

struct alignas(16) RowState {
    unsigned long long bins[kBins];
    unsigned long long list[kListCap];  // key << 32 | ~index
    unsigned long long rest;            // weight that the list's kept part must exceed
    uint32_t listed;                    // tokens offered to the list
    uint32_t whole;                     // the row is drawn by one workgroup
    int cut;                            // bin that holds the cut (kBins: none)
};

template <typename T, bool VEC>
__global__ void __launch_bounds__(kPartThreads)
argmax_part_kernel(const T* __restrict__ logits, int64_t vocab, int64_t stride, int nparts,
                   const float* __restrict__ temperature, ArgPart* __restrict__ parts,
                   RowState* __restrict__ states) {
    const int r = blockIdx.x / nparts;
    const int span = blockIdx.x - r * nparts;
    // The spans share the clearing of a sampled row's state.
    if (states != nullptr && temperature[r] > 0.f) {
        for (int b = span * kPartThreads + threadIdx.x; b < kBins; b += nparts * kPartThreads)
            states[r].bins[b] = 0;
        if (span == 0 && threadIdx.x == 0) states[r].listed = 0;
    }
    const T* row = logits + int64_t(r) * stride;
    const int64_t begin = int64_t(span) * kPartSpan;
    const int64_t end = min(vocab, begin + kPartSpan);
    float best = -INFINITY;
    int64_t bi = INT64_MAX;
    int64_t tail = begin;
    if constexpr (VEC) {
        const U16x8* rv = reinterpret_cast<const U16x8*>(row);
        const uint32_t v0 = uint32_t(begin / 8), v1 = uint32_t(end / 8);  // whole vectors
        U16x8 raw[kPartVecs];
#pragma unroll
        for (int u = 0; u < kPartVecs; ++u) {
            const uint32_t c = v0 + threadIdx.x + uint32_t(u) * kPartThreads;
            raw[u] = rv[c < v1 ? c : v0];
        }
        float m = -INFINITY;
        bool nan = false;
#pragma unroll
        for (int u = 0; u < kPartVecs; ++u) {
            const uint32_t c = v0 + threadIdx.x + uint32_t(u) * kPartThreads;
            if (c >= v1) break;
            float x[8];
            unpack8<T>(raw[u], x);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                m = fmaxf(m, x[e]);
                nan |= x[e] != x[e];
            }
        }
#pragma unroll
        for (int u = 0; u < kPartVecs; ++u) {
            const uint32_t c = v0 + threadIdx.x + uint32_t(u) * kPartThreads;
            if (c >= v1) break;
            float x[8];
            unpack8<T>(raw[u], x);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int64_t i = int64_t(c) * 8 + e;
                if (nan ? better(x[e], i, best, bi) : (x[e] == m && i < bi)) {
                    best = x[e];
                    bi = i;
                }
            }
        }
        tail = int64_t(v1) * 8;
    }
    for (int64_t i = tail + threadIdx.x; i < end; i += kPartThreads) {
        const float x = load_logit(row, i);
        if (better(x, i, best, bi)) { best = x; bi = i; }
    }
    block_argmax_w<kPartThreads / 64>(best, bi);
    if (threadIdx.x == 0)
        parts[blockIdx.x] = ArgPart{best, bi == INT64_MAX ? -1 : int32_t(bi)};
}

// One element's race value s - log(E), E ~ Exp(1) from word i % 4 of the
// Philox block i / 4 of the row's (seed, counter) stream.
__device__ __forceinline__ float race_value(float s, uint32_t bits) {
    const float u = (float(bits >> 8) + 0.5f) * (1.0f / 16777216.0f);
    const float e = -logf(u);
    return s - logf(e);
}

struct Noise {
    uint2 key;
    uint64_t step;
    __device__ __forceinline__ uint4 block(int64_t i) const {
        return philox4x32_10(
            make_uint4(static_cast<uint32_t>(i >> 2), static_cast<uint32_t>(i >> 34),
                       static_cast<uint32_t>(step), static_cast<uint32_t>(step >> 32)),
            key);
    }
    __device__ __forceinline__ uint32_t bits(int64_t i) const {
        const uint4 r = block(i);
        const int w = int(i & 3);
        return w == 0 ? r.x : w == 1 ? r.y : w == 2 ? r.z : r.w;
    }
};

__device__ __forceinline__ Noise noise_of(int64_t seed, int64_t counter) {
    return Noise{make_uint2(static_cast<uint32_t>(seed),
                            static_cast<uint32_t>(uint64_t(seed) >> 32)),
                 static_cast<uint64_t>(counter)};
}

// One row's draw by one workgroup of NT threads, whatever the row holds
// (radix selection over the whole row): rows without a workspace, and those
// whose boundary bin holds more tokens than the gathered list.
template <typename T, int NT>
__device__ int64_t sample_row(const T* row, int64_t vocab, const RowCtx& ctx, int64_t k, float p,
                              const Noise& noise) {
    Cut kcut{0u, 0, true};
    if (k > 0 && k < vocab) {
        kcut = radix_cut<T, false, NT>(row, vocab, ctx, uint64_t(k - 1),
                                       [](int64_t) { return true; });
    }
    auto in_k = [&](int64_t i) {
        return kcut.all || kept(kcut, fkey(score_of(row, i, ctx)), i);
    };

    Cut pcut{0u, 0, true};
    if (p < 1.f) {
        // Z = total mass of the top-k candidates (the softmax denominator).
        __shared__ unsigned long long s_z;
        if (threadIdx.x == 0) s_z = 0;
        __syncthreads();
        unsigned long long z = 0;
        for (int64_t i = threadIdx.x; i < vocab; i += NT)
            if (in_k(i)) z += mass_of(score_of(row, i, ctx));
        atomicAdd(&s_z, z);
        __syncthreads();
        const uint64_t target = static_cast<uint64_t>(static_cast<double>(p) *
                                                      static_cast<double>(s_z));
        pcut = radix_cut<T, true, NT>(row, vocab, ctx, target, in_k);
    }

    // Exponential race over the kept set: argmax s_i - log(E_i).
    float bv = -INFINITY;
    int64_t bidx = INT64_MAX;
    for (int64_t i = threadIdx.x; i < vocab; i += NT) {
        const float s = score_of(row, i, ctx);
        const uint32_t kk = fkey(s);
        if (!kcut.all && !kept(kcut, kk, i)) continue;
        if (!pcut.all && !kept(pcut, kk, i)) continue;
        const float g = race_value(s, noise.bits(i));
        if (better(g, i, bv, bidx)) { bv = g; bidx = i; }
    }
    block_argmax_w<NT / 64>(bv, bidx);
    return bidx;
}

template <typename T, bool VEC>
__global__ void __launch_bounds__(kThreads)
sample_kernel(const T* __restrict__ logits, int64_t vocab, int64_t stride,
              const float* __restrict__ temperature, const int64_t* __restrict__ top_k,
              const float* __restrict__ top_p, const int64_t* __restrict__ seeds,
              const int64_t* __restrict__ counters, int64_t* __restrict__ out,
              const ArgPart* __restrict__ parts, int nparts) {
    const int r = blockIdx.x;
    const T* row = logits + int64_t(r) * stride;

    // Row max (also the greedy answer): from the per-span partials of
    // argmax_part_kernel when given, else scanned here.
    float best = -INFINITY;
    int64_t bi = INT64_MAX;
    if (parts != nullptr) {
        for (int i = threadIdx.x; i < nparts; i += kThreads) {
            const ArgPart p = parts[int64_t(r) * nparts + i];
            const int64_t pi = p.i < 0 ? INT64_MAX : int64_t(p.i);
            if (better(p.v, pi, best, bi)) { best = p.v; bi = pi; }
        }
    } else {
        thread_argmax<T, VEC>(row, vocab, best, bi);
    }
    block_argmax_w<kWaves>(best, bi);
    const float temp = temperature[r];
    if (temp > 0.f)
        bi = sample_row<T, kThreads>(row, vocab, RowCtx{best, temp}, top_k[r], top_p[r],
                                     noise_of(seeds[r], counters[r]));
    if (threadIdx.x == 0) out[r] = bi;
}

// ------------------------------------------- sampling split over spans ----
// With a workspace, a row's passes are spread over its spans (kPartSpan
// elements each, one 256-thread workgroup): three launches of rows x spans
// workgroups that each read the row once, and a short one per row, where the
// one-workgroup kernel reads the row about fifteen times from one CU. 64 rows
// x 151936 bf16 with mixed filters: 1965 -> 71 us (in a trace race 26, finish
// 17, bins 16, maxima 9: four dependent launches of one or two waves per SIMD;
// 19 MB is 3 us of memory. Two changes left the race where it is: ruling
// tokens out by a bound of one exponential before the two logarithms and a
// rolled loop of a quarter of its 58 KB of instructions). A batch of greedy
// rows pays 0.6 us (bf16) to 1.5 us (fp32) for the two launches that find
// nothing to do.
//
//   argmax_part_kernel  each span's maximum; clears the row's bins.
//   bins_kernel         the row maximum from the spans (greedy rows are done);
//                       adds the span's tokens to the row's bins of s: their
//                       number (rows with a top-k) or their mass (top-p only).
//   race_kernel         finds the bin that holds the cut. Tokens in better
//                       bins are kept whatever happens inside that bin: with
//                       top-p only they race right here; the cut's own bin
//                       (with top-k: every bin up to it) is gathered into the
//                       row's list.
//   finish_kernel       sorts the list, cuts it exactly, races what is kept
//                       of it against the spans' winners.
//
// The finish is a launch of its own: with the row's last workgroup to finish
// doing it, the device-wide fence in front of each arrival (1216 of them)
// cost more than everything else (64 sampled rows: 64-120 us of fences).
//
// The sums are integers, so neither the order of the workgroups nor that of
// the list changes the result: it is the one-workgroup kernel's.

__device__ __forceinline__ ArgPart row_max(const ArgPart* __restrict__ parts, int nparts) {
    float best = -INFINITY;
    int64_t bi = INT64_MAX;
    for (int i = threadIdx.x & 63; i < nparts; i += 64) {
        const ArgPart p = parts[i];
        const int64_t pi = p.i < 0 ? INT64_MAX : int64_t(p.i);
        if (better(p.v, pi, best, bi)) { best = p.v; bi = pi; }
    }
    wave_argmax(best, bi);  // every wave on its own
    return ArgPart{best, bi == INT64_MAX ? -1 : int32_t(bi)};
}

// What a row needs: its list and bins hold counts (top-k) or masses (top-p
// only); a row that keeps everything needs neither. To the one-workgroup draw
// go rows whose maximum or temperature is not finite (their scores may be NaN)
// and those with a top-k beyond the list.
enum class Draw { kGreedy, kAll, kTopK, kTopP, kWhole };

__device__ __forceinline__ Draw draw_of(float temp, float mx, int64_t k, float p, int64_t vocab) {
    if (!(temp > 0.f)) return Draw::kGreedy;
    if (!(fabsf(mx) < INFINITY && temp < INFINITY)) return Draw::kWhole;
    if (k > 0 && k < vocab) return k <= kListCap ? Draw::kTopK : Draw::kWhole;
    return p < 1.f ? Draw::kTopP : Draw::kAll;
}

// f(i, logit) for every element of the thread's share of span [begin, end),
// aligned groups of 8 consecutive elements per vector load when VEC (`end` is
// a multiple of 8 except in a row's last span).
template <typename T, bool VEC, typename F>
__device__ __forceinline__ void for_span(const T* row, int64_t begin, int64_t end, F&& f) {
    int64_t tail = begin;
    if constexpr (VEC) {
        const U16x8* rv = reinterpret_cast<const U16x8*>(row);
        const uint32_t v0 = uint32_t(begin / 8), v1 = uint32_t(end / 8);
        if (v0 < v1) {
        U16x8 raw[kPartVecs];
#pragma unroll
        for (int u = 0; u < kPartVecs; ++u) {
            const uint32_t c = v0 + threadIdx.x + uint32_t(u) * kPartThreads;
            raw[u] = rv[c < v1 ? c : v0];
        }
#pragma unroll
        for (int u = 0; u < kPartVecs; ++u) {
            const uint32_t c = v0 + threadIdx.x + uint32_t(u) * kPartThreads;
            if (c >= v1) break;
            float x[8];
            unpack8<T>(raw[u], x);
#pragma unroll
            for (int e = 0; e < 8; ++e) f(int64_t(c) * 8 + e, x[e]);
        }
        }
        tail = int64_t(v1) * 8;
    }
    for (int64_t i = tail + threadIdx.x; i < end; i += kPartThreads) f(i, load_logit(row, i));
}

template <typename T, bool VEC>
__global__ void __launch_bounds__(kPartThreads)
bins_kernel(const T* __restrict__ logits, int64_t vocab, int64_t stride,
            const float* __restrict__ temperature, const int64_t* __restrict__ top_k,
            const float* __restrict__ top_p, int64_t* __restrict__ out,
            const ArgPart* __restrict__ parts, int nparts, RowState* __restrict__ states) {
    __shared__ unsigned long long bins[kBins];
    const int r = blockIdx.x / nparts;
    const int span = blockIdx.x - r * nparts;
    const float temp = temperature[r];
    if (!(temp > 0.f) && span != 0) return;
    const ArgPart top = row_max(parts + int64_t(r) * nparts, nparts);
    const Draw draw = draw_of(temp, top.v, top_k[r], top_p[r], vocab);
    if (draw == Draw::kGreedy && threadIdx.x == 0) out[r] = top.i;
    if (draw != Draw::kTopK && draw != Draw::kTopP) return;
    for (int b = threadIdx.x; b < kBins; b += kPartThreads) bins[b] = 0;
    __syncthreads();
    const bool mass = draw == Draw::kTopP;
    const int64_t begin = int64_t(span) * kPartSpan;
    for_span<T, VEC>(logits + int64_t(r) * stride, begin, min(vocab, begin + kPartSpan),
                     [&](int64_t, float x) {
        const float s = (x - top.v) / temp;
        const int b = bin_of(s);
        if (b < kBins - 1) {
            const unsigned long long w = mass ? mass_of(s) : 1ull;
            if (w != 0) atomicAdd(&bins[b], w);
        }
    });
    __syncthreads();
    unsigned long long* const sum = states[r].bins;
    for (int b = threadIdx.x; b < kBins; b += kPartThreads)
        if (bins[b] != 0) atomicAdd(&sum[b], bins[b]);
}

// Exclusive prefix sum over the NT threads of the workgroup; `total` for all.
template <int NT>
__device__ uint64_t block_scan(uint64_t v, uint64_t& total) {
    __shared__ uint64_t wave_total[NT / 64];
    uint64_t incl = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint64_t o = __shfl_up(incl, off, 64);
        if (int(threadIdx.x & 63) >= off) incl += o;
    }
    if ((threadIdx.x & 63) == 63) wave_total[threadIdx.x >> 6] = incl;
    __syncthreads();
    uint64_t before = 0;
    total = 0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) {
        if (w < int(threadIdx.x >> 6)) before += wave_total[w];
        total += wave_total[w];
    }
    __syncthreads();
    return before + incl - v;
}

// First position (of n, thread t owning the run [t * per, (t + 1) * per))
// whose inclusive sum of weight(i) exceeds target: that position and the sum
// before it, or n and the whole sum where none does.
template <int NT, typename W>
__device__ uint64_t first_over(int n, int per, uint64_t target, int& pos, W&& weight) {
    __shared__ int s_pos;
    __shared__ uint64_t s_above;
    const int i0 = min(n, int(threadIdx.x) * per), i1 = min(n, i0 + per);
    uint64_t mine = 0, total;
    for (int i = i0; i < i1; ++i) mine += weight(i);
    uint64_t cum = block_scan<NT>(mine, total);
    if (threadIdx.x == 0) { s_pos = n; s_above = total; }
    __syncthreads();
    if (cum <= target && cum + mine > target) {  // at most one thread
        int i = i0;
        for (; i < i1; ++i) {
            const uint64_t w = weight(i);
            if (cum + w > target) break;
            cum += w;
        }
        s_pos = i;
        s_above = cum;
    }
    __syncthreads();
    pos = s_pos;
    const uint64_t above = s_above;
    __syncthreads();
    return above;
}

__device__ __forceinline__ float key_value(uint32_t key) {  // inverse of fkey
    return __uint_as_float((key & 0x80000000u) ? key ^ 0x80000000u : ~key);
}

template <typename T, bool VEC>
__global__ void __launch_bounds__(kPartThreads)
race_kernel(const T* __restrict__ logits, int64_t vocab, int64_t stride,
            const float* __restrict__ temperature, const int64_t* __restrict__ top_k,
            const float* __restrict__ top_p, const int64_t* __restrict__ seeds,
            const int64_t* __restrict__ counters, const ArgPart* __restrict__ parts, int nparts,
            RowState* __restrict__ states, ArgPart* __restrict__ races) {
    __shared__ unsigned long long listed[kListCap];  // the span's share of the row's list
    __shared__ uint32_t s_listed, s_at;
    const int r = blockIdx.x / nparts;
    const int span = blockIdx.x - r * nparts;
    const float temp = temperature[r];
    if (!(temp > 0.f)) return;  // greedy: answered by bins_kernel
    if (threadIdx.x == 0) s_listed = 0;
    __syncthreads();
    const T* row = logits + int64_t(r) * stride;
    const int64_t k = top_k[r];
    const float p = top_p[r];
    const Noise noise = noise_of(seeds[r], counters[r]);
    const RowCtx ctx{row_max(parts + int64_t(r) * nparts, nparts).v, temp};
    const Draw draw = draw_of(temp, ctx.mx, k, p, vocab);
    RowState& state = states[r];

    int cut = kBins;  // tokens of the bins below it are kept
    bool whole = draw == Draw::kWhole;
    uint64_t rest = 0;
    if (draw == Draw::kTopK || draw == Draw::kTopP) {
        constexpr int kPer = kBins / kPartThreads;
        unsigned long long w[kPer];
        uint64_t z = 0, total;
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            w[i] = state.bins[threadIdx.x * kPer + i];
            z += w[i];
        }
        auto weight = [&](int i) -> uint64_t {
            uint64_t v = 0;
#pragma unroll
            for (int j = 0; j < kPer; ++j) v = (i & (kPer - 1)) == j ? w[j] : v;
            return v;
        };
        block_scan<kPartThreads>(z, total);
        const uint64_t target = draw == Draw::kTopK
            ? uint64_t(k - 1)
            : static_cast<uint64_t>(static_cast<double>(p) * static_cast<double>(total));
        rest = target - first_over<kPartThreads>(kBins, kPer, target, cut, weight);
        // Top-k beyond the bins' range: the whole row decides. (Top-p always
        // finds its bin unless the target rounds to the whole mass: then
        // everything is kept.)
        whole = draw == Draw::kTopK && cut == kBins;
    }
    if (span == 0 && threadIdx.x == 0) {
        state.rest = rest;
        state.whole = whole;
        state.cut = cut;
    }
    if (whole) return;

    float best = -INFINITY;
    int64_t bi = INT64_MAX;
    const int64_t begin = int64_t(span) * kPartSpan;
    const bool gather_all = draw == Draw::kTopK;  // every candidate into the list
    uint4 words{};
    int64_t held = -1;  // Philox block in `words`
    for_span<T, VEC>(row, begin, min(vocab, begin + kPartSpan), [&](int64_t i, float x) {
        const float s = (x - ctx.mx) / temp;
        const int b = cut == kBins ? -1 : bin_of(s);
        if (b > cut) return;
        if (gather_all || b == cut) {
            const uint32_t at = atomicAdd(&s_listed, 1u);
            if (at < uint32_t(kListCap))
                listed[at] = (static_cast<unsigned long long>(fkey(s)) << 32) |
                             (0xffffffffu - static_cast<uint32_t>(i));
            return;
        }
        if (held != (i >> 2)) {
            held = i >> 2;
            words = noise.block(i);
        }
        const int e = int(i & 3);
        const float g = race_value(s, e == 0 ? words.x : e == 1 ? words.y
                                                       : e == 2 ? words.z : words.w);
        if (better(g, i, best, bi)) { best = g; bi = i; }
    });
    block_argmax_w<kPartThreads / 64>(best, bi);
    if (threadIdx.x == 0) {
        races[blockIdx.x] = ArgPart{best, bi == INT64_MAX ? -1 : int32_t(bi)};
        s_at = s_listed ? atomicAdd(&state.listed, s_listed) : 0;
    }
    __syncthreads();
    if (s_at + s_listed <= uint32_t(kListCap))  // else the row is drawn whole
        for (uint32_t i = threadIdx.x; i < s_listed; i += kPartThreads)
            state.list[s_at + i] = listed[i];
}

// The draw among the n > 0 listed tokens of a row: sorts them (in `order`, which
// may be `list` itself), cuts them exactly, and races what is kept against the
// best so far. `rest`: the mass that the list's kept part must exceed (top-p
// without top-k).
__device__ void finish_list(const unsigned long long* list, unsigned long long* order, uint32_t n,
                            int64_t k, float p, int64_t vocab, uint64_t rest, const Noise& noise,
                            float& best, int64_t& bi) {
    // Descending (key, then ascending index) order: a bitonic sort in
    // LDS. Steps of up to 64 stay inside the 128 entries that a wave
    // owns in all of them, so only the wider ones need the workgroup's
    // barrier: at 1024 entries 6 of 55 steps.
    int m = 2;
    while (m < int(n)) m *= 2;
    for (int i = threadIdx.x; i < m; i += kThreads)
        order[i] = i < int(n) ? list[i] : 0ull;
    __syncthreads();
    for (int size = 2; size <= m; size <<= 1)
        for (int step = size >> 1; step > 0; step >>= 1) {
            for (int t = threadIdx.x; t < m / 2; t += kThreads) {
                const int i = 2 * t - (t & (step - 1)), j = i + step;
                const unsigned long long a = order[i], b = order[j];
                if ((a < b) == ((i & size) == 0)) {
                    order[i] = b;
                    order[j] = a;
                }
            }
            const int next = step > 1 ? step >> 1 : size;
            if (step > 64 || next > 64) {
                __syncthreads();
            } else {
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            }
        }
    __syncthreads();
    auto mass = [&](int i) { return mass_of(key_value(uint32_t(order[i] >> 32))); };
    const bool counted = k > 0 && k < vocab;  // the list holds every top-k candidate
    int keep = counted ? int(k) : int(n);
    if (p < 1.f) {
        if (counted) {
            uint64_t z = 0, total;
            for (int i = threadIdx.x; i < keep; i += kThreads) z += mass(i);
            block_scan<kThreads>(z, total);
            rest = static_cast<uint64_t>(static_cast<double>(p) * static_cast<double>(total));
        }
        int pos;
        first_over<kThreads>(keep, (keep + kThreads - 1) / kThreads, rest, pos, mass);
        keep = min(keep, pos + 1);
    }
    for (int t = threadIdx.x; t < keep; t += kThreads) {
        const int64_t i = int64_t(0xffffffffu - static_cast<uint32_t>(order[t]));
        const float g = race_value(key_value(uint32_t(order[t] >> 32)), noise.bits(i));
        if (better(g, i, best, bi)) { best = g; bi = i; }
    }
}

template <typename T>
__global__ void __launch_bounds__(kThreads)
finish_kernel(const T* __restrict__ logits, int64_t vocab, int64_t stride,
              const float* __restrict__ temperature, const int64_t* __restrict__ top_k,
              const float* __restrict__ top_p, const int64_t* __restrict__ seeds,
              const int64_t* __restrict__ counters, int64_t* __restrict__ out,
              const ArgPart* __restrict__ parts, int nparts,
              const RowState* __restrict__ states, const ArgPart* __restrict__ races) {
    __shared__ unsigned long long order[kListCap];
    const int r = blockIdx.x;
    const float temp = temperature[r];
    if (!(temp > 0.f)) return;
    const RowState& state = states[r];
    const int64_t k = top_k[r];
    const float p = top_p[r];
    const Noise noise = noise_of(seeds[r], counters[r]);
    const uint32_t n = state.listed;
    const T* const row = logits + int64_t(r) * stride;
    const bool counted = k > 0 && k < vocab;
    const bool overflow = n > uint32_t(kListCap);
    if (state.whole || (overflow && counted)) {
        const RowCtx ctx{row_max(parts + int64_t(r) * nparts, nparts).v, temp};
        const int64_t token = sample_row<T, kThreads>(row, vocab, ctx, k, p, noise);
        if (threadIdx.x == 0) out[r] = token;
        return;
    }
    float best = -INFINITY;
    int64_t bi = INT64_MAX;
    for (int i = threadIdx.x; i < nparts; i += kThreads) {
        const ArgPart q = races[int64_t(r) * nparts + i];
        if (q.i >= 0 && better(q.v, q.i, best, bi)) { best = q.v; bi = q.i; }
    }
    if (overflow) {  // the cut's bin holds more than the list: select inside it, from the row
        const RowCtx ctx{row_max(parts + int64_t(r) * nparts, nparts).v, temp};
        auto in_bin = [&](int64_t i) { return bin_of(score_of(row, i, ctx)) == state.cut; };
        const Cut cut = radix_cut<T, true, kThreads>(row, vocab, ctx, state.rest, in_bin);
        for (int64_t i = threadIdx.x; i < vocab; i += kThreads) {
            const float s = score_of(row, i, ctx);
            if (bin_of(s) != state.cut || !kept(cut, fkey(s), i)) continue;
            const float g = race_value(s, noise.bits(i));
            if (better(g, i, best, bi)) { best = g; bi = i; }
        }
        block_argmax_w<kWaves>(best, bi);
        if (threadIdx.x == 0) out[r] = bi;
        return;
    }
    if (n > 0) finish_list(state.list, order, n, k, p, vocab, state.rest, noise, best, bi);
    block_argmax_w<kWaves>(best, bi);
    if (threadIdx.x == 0) out[r] = bi;
}

// Rows of one span: all of it in one launch, a workgroup per row, with the bins
// and the list in LDS. Against the four launches, us for 64 rows of 8192 bf16
// tokens: greedy 12.5 -> 11.3, no filter 29.9 -> 23.7, top-k 36 -> 29, top-p 48
// -> 37; of 100 tokens without a filter 17.5 -> 9.0 (their own time, four
// launches of next to nothing).
template <typename T, bool VEC>
__global__ void __launch_bounds__(kThreads)
sample_span_kernel(const T* __restrict__ logits, int64_t vocab, int64_t stride,
                   const float* __restrict__ temperature, const int64_t* __restrict__ top_k,
                   const float* __restrict__ top_p, const int64_t* __restrict__ seeds,
                   const int64_t* __restrict__ counters, int64_t* __restrict__ out) {
    __shared__ unsigned long long shared[kListCap];  // the bins, then the list
    __shared__ uint32_t s_listed;
    static_assert(kBins <= kListCap && kBins % kThreads == 0, "the bins fit");
    const int r = blockIdx.x;
    const T* row = logits + int64_t(r) * stride;
    float best = -INFINITY;
    int64_t bi = INT64_MAX;
    thread_argmax<T, VEC>(row, vocab, best, bi);
    block_argmax_w<kWaves>(best, bi);
    const float temp = temperature[r];
    const int64_t k = top_k[r];
    const float p = top_p[r];
    const RowCtx ctx{best, temp};
    const Noise noise = noise_of(seeds[r], counters[r]);
    const Draw draw = draw_of(temp, best, k, p, vocab);
    bool whole = draw == Draw::kAll || draw == Draw::kWhole;
    if (draw == Draw::kTopK || draw == Draw::kTopP) {
        const bool mass = draw == Draw::kTopP;
        for (int b = threadIdx.x; b < kBins; b += kThreads) shared[b] = 0;
        if (threadIdx.x == 0) s_listed = 0;
        __syncthreads();
        for (int64_t i = threadIdx.x; i < vocab; i += kThreads) {
            const float s = score_of(row, i, ctx);
            const int b = bin_of(s);
            if (b < kBins - 1) {
                const unsigned long long w = mass ? mass_of(s) : 1ull;
                if (w != 0) atomicAdd(&shared[b], w);
            }
        }
        __syncthreads();
        constexpr int kPer = kBins / kThreads;
        uint64_t z = 0, total;
        for (int i = 0; i < kPer; ++i) z += shared[threadIdx.x * kPer + i];
        block_scan<kThreads>(z, total);
        const uint64_t target = mass
            ? static_cast<uint64_t>(static_cast<double>(p) * static_cast<double>(total))
            : uint64_t(k - 1);
        int cut;
        const uint64_t rest = target - first_over<kThreads>(
            kBins, kPer, target, cut, [&](int i) -> uint64_t { return shared[i]; });
        // (first_over's last barrier: the bins may become the list.)
        whole = !mass && cut == kBins;  // top-k beyond the bins' range
        if (!whole) {
            best = -INFINITY;
            bi = INT64_MAX;
            for (int64_t i = threadIdx.x; i < vocab; i += kThreads) {
                const float s = score_of(row, i, ctx);
                const int b = cut == kBins ? -1 : bin_of(s);
                if (b > cut) continue;
                if (!mass || b == cut) {
                    const uint32_t at = atomicAdd(&s_listed, 1u);
                    if (at < uint32_t(kListCap))
                        shared[at] = (static_cast<unsigned long long>(fkey(s)) << 32) |
                                     (0xffffffffu - static_cast<uint32_t>(i));
                    continue;
                }
                const float g = race_value(s, noise.bits(i));
                if (better(g, i, best, bi)) { best = g; bi = i; }
            }
            __syncthreads();
            const uint32_t n = s_listed;
            whole = n > uint32_t(kListCap);
            if (!whole) {
                if (n > 0) finish_list(shared, shared, n, k, p, vocab, rest, noise, best, bi);
                block_argmax_w<kWaves>(best, bi);
            }
        }
    }
    if (whole) bi = sample_row<T, kThreads>(row, vocab, ctx, k, p, noise);
    if (threadIdx.x == 0) out[r] = bi;
}

template <typename T, bool VEC>
__global__ void __launch_bounds__(kThreads)
argmax_kernel(const T* __restrict__ logits, int64_t vocab, int64_t stride,
              int64_t* __restrict__ out) {
    const T* row = logits + int64_t(blockIdx.x) * stride;
    float best = -INFINITY;
    int64_t bi = INT64_MAX;
    thread_argmax<T, VEC>(row, vocab, best, bi);
    block_argmax_w<kWaves>(best, bi);
    if (threadIdx.x == 0) out[blockIdx.x] = bi;
}

}  // namespace
}  // namespace tvllm

using namespace tvllm;

extern "C" int tvllm_argmax(const void* logits, int64_t rows, int64_t vocab,
                            int64_t row_stride, int64_t* out, int dtype,
                            tvllm_stream_t stream) {
    TVLLM_CHECK(rows >= 0 && vocab > 0 && row_stride >= vocab,
                "argmax: invalid logits geometry");
    TVLLM_CHECK(rows <= INT32_MAX, "argmax: too many rows");
    if (rows == 0) return TVLLM_OK;
    TVLLM_CHECK(logits && out, "argmax: null pointer");
    hipStream_t s = as_hip(stream);
    return dispatch_float(dtype, [&]<int DT>() {
        using T = typename Elem<DT>::T;
        const bool vec = row_stride % 8 == 0 && aligned16(logits);
        if constexpr (sizeof(T) == 2) {
            if (vec) {
                argmax_kernel<T, true><<<int(rows), kThreads, 0, s>>>(
                    static_cast<const T*>(logits), vocab, row_stride, out);
                return launch_status("argmax");
            }
        }
            argmax_kernel<T, false><<<int(rows), kThreads, 0, s>>>(
                static_cast<const T*>(logits), vocab, row_stride, out);
        return launch_status("argmax");
    });
}

extern "C" int64_t tvllm_sample_workspace_size(int64_t rows, int64_t vocab) {
    // One (value, index) partial per kPartSpan-wide span of each row.
    if (rows <= 0 || vocab <= 0) return 0;
    return rows * ((vocab + kPartSpan - 1) / kPartSpan) * int64_t(sizeof(ArgPart));
}

extern "C" int64_t tvllm_sample_split_workspace_size(int64_t rows, int64_t vocab) {
    // Each row's bins and list, and two (value, index) partials per span.
    if (rows <= 0 || vocab <= 0) return 0;
    return rows * int64_t(sizeof(RowState)) + 2 * tvllm_sample_workspace_size(rows, vocab);
}

extern "C" int tvllm_sample(const void* logits, int64_t rows, int64_t vocab,
                            int64_t row_stride, const float* temperature,
                            const int64_t* top_k, const float* top_p,
                            const int64_t* seeds, const int64_t* counters,
                            int64_t* out, void* workspace, int64_t workspace_bytes,
                            int dtype, tvllm_stream_t stream) {
    TVLLM_CHECK(rows >= 0 && vocab > 0 && row_stride >= vocab,
                "sample: invalid logits geometry");
    TVLLM_CHECK(vocab < (int64_t(1) << 24), "sample: vocab must be < 2^24");
    TVLLM_CHECK(rows <= INT32_MAX, "sample: too many rows");
    if (rows == 0) return TVLLM_OK;
    TVLLM_CHECK(logits && temperature && top_k && top_p && seeds && counters && out,
                "sample: null pointer");
    TVLLM_CHECK(workspace_bytes >= 0 && (workspace_bytes == 0 || workspace != nullptr),
                "sample: null workspace");
    hipStream_t s = as_hip(stream);
    // A workspace of tvllm_sample_split_workspace_size bytes spreads every
    // pass over spans, one of tvllm_sample_workspace_size bytes the search for
    // the row maximum only; without one each row's workgroup draws alone.
    const int64_t nparts = (vocab + kPartSpan - 1) / kPartSpan;
    const bool fits = aligned16(workspace) && rows * nparts <= INT32_MAX;
    const bool split = fits && workspace_bytes >= tvllm_sample_split_workspace_size(rows, vocab);
    const bool scan = fits && workspace_bytes >= tvllm_sample_workspace_size(rows, vocab);
    RowState* const states = split ? static_cast<RowState*>(workspace) : nullptr;
    ArgPart* const parts = split ? reinterpret_cast<ArgPart*>(states + rows)
                                 : scan ? static_cast<ArgPart*>(workspace) : nullptr;
    return dispatch_float(dtype, [&]<int DT>() {
        using T = typename Elem<DT>::T;
        const bool vec = sizeof(T) == 2 && row_stride % 8 == 0 && aligned16(logits);
        auto go = [&]<bool V>() {
            const T* const x = static_cast<const T*>(logits);
            const int grid = int(rows * nparts), np = int(nparts);
            if (split && nparts == 1) {
                sample_span_kernel<T, V><<<int(rows), kThreads, 0, s>>>(
                    x, vocab, row_stride, temperature, top_k, top_p, seeds, counters, out);
                return launch_status("sample");
            }
            if (parts != nullptr) {
                argmax_part_kernel<T, V><<<grid, kPartThreads, 0, s>>>(x, vocab, row_stride, np,
                                                                       temperature, parts, states);
                const int status = launch_status("sample");
                if (status != TVLLM_OK) return status;
            }
            if (!split) {
                sample_kernel<T, V><<<int(rows), kThreads, 0, s>>>(
                    x, vocab, row_stride, temperature, top_k, top_p, seeds, counters, out, parts,
                    np);
                return launch_status("sample");
            }
            bins_kernel<T, V><<<grid, kPartThreads, 0, s>>>(x, vocab, row_stride, temperature, top_k,
                                                            top_p, out, parts, np, states);
            int status = launch_status("sample");
            if (status != TVLLM_OK) return status;
            ArgPart* const races = parts + rows * nparts;
            race_kernel<T, V><<<grid, kPartThreads, 0, s>>>(x, vocab, row_stride, temperature, top_k,
                                                            top_p, seeds, counters, parts, np,
                                                            states, races);
            status = launch_status("sample");
            if (status != TVLLM_OK) return status;
            finish_kernel<T><<<int(rows), kThreads, 0, s>>>(x, vocab, row_stride, temperature, top_k,
                                                            top_p, seeds, counters, out, parts, np,
                                                            states, races);
            return launch_status("sample");
        };
        if constexpr (sizeof(T) == 2) {
            if (vec) return go.template operator()<true>();
        }
        return go.template operator()<false>();
    });
}

// ------------------------------------------------ pipelined input tokens ----

namespace tvllm {
namespace {

// tokens[i] = prev[src[i]] where 0 <= src[i] < prev_count, else unchanged.
__global__ void __launch_bounds__(256)
resolve_tokens_kernel(int64_t* __restrict__ tokens, const int64_t* __restrict__ src,
                      const int64_t* __restrict__ prev, int64_t n, int64_t prev_count) {
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n) return;
    const int64_t s = src[i];
    if (s >= 0 && s < prev_count) tokens[i] = prev[s];
}

}  // namespace
}  // namespace tvllm

extern "C" int tvllm_resolve_tokens(int64_t* tokens, const int64_t* src,
                                    const int64_t* prev, int64_t n, int64_t prev_count,
                                    tvllm_stream_t stream) {
    using namespace tvllm;
    TVLLM_CHECK(n >= 0 && prev_count >= 0, "resolve_tokens: negative size");
    TVLLM_CHECK(n <= (int64_t(INT32_MAX) - 255), "resolve_tokens: too many tokens");
    if (n == 0) return TVLLM_OK;
    TVLLM_CHECK(tokens && src && (prev || prev_count == 0), "resolve_tokens: null pointer");
    resolve_tokens_kernel<<<int((n + 255) / 256), 256, 0, as_hip(stream)>>>(
        tokens, src, prev, n, prev_count);
    return launch_status("resolve_tokens");
}
