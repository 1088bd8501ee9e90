// Paged attention for any head dim up to 256: the decode rows and prefill
// chunks that the MFMA kernels (head_dim 128, GQA groups <= 16, 16-byte
// aligned rows) do not take.
//
// Reference behaviour: tinyvllm/kernels/paged_decode.cu:572-666 dispatches
// head dims 32, 64, 128 and 256 to one templated kernel; chunked prefill is
// SDPA with a lower-right causal mask (tinyvllm/runtime/attention.py:102-151,
// 176-214). Output = softmax(scale * q.K^T) V over each row's cached tokens
// in logical order (a padded decode row of length 0 gives zeros).
//
// Head dims 32, 64, 128 and 256 with vector-aligned cache rows run on the
// matrix cores (rows_attention_kernel for few query rows, decode above all;
// tiles_attention_kernel for prefill chunks). Everything else - other head
// dims, unaligned rows - takes general_attention_kernel: one wave per (query
// token, KV head, group of up to 16 query heads of that KV head), so the
// query heads of a KV head share every K/V load. The wave walks its keys in
// chunks of 64: lane j scores key j of the chunk against all of the wave's
// heads (the query rows sit in LDS, read as broadcasts), the online softmax
// runs per head across the wave, and P.V runs with the lanes over the head
// dims (lane l: dims l, l + 64, ...), the chunk's probabilities read back
// from LDS. That kernel is fp32 throughout, without matrix cores.
#include "general_attention.h"

#include <algorithm>
#include <type_traits>

namespace tvllm {
namespace {

constexpr int GH = 16;     // query heads per wave
constexpr int DMAX = 256;  // largest head dim
constexpr float kLog2eG = 1.4426950408889634f;
constexpr int kRowWaves = 4;  // waves per workgroup of the matrix-core kernels (or half of one)

// Eight elements of a cache row starting at element e (FP8: bytes), as
// floats; elements at or past `left` read as 0.
template <typename T, bool F8, bool VEC>
__device__ __forceinline__ void load8(const void* __restrict__ base, int64_t e, int left,
                                      float (&x)[8]) {
    if constexpr (F8) {
        const uint8_t* b = static_cast<const uint8_t*>(base) + e;
        if constexpr (VEC) {
            fp8x8_unpack(*reinterpret_cast<const uint2*>(b), x);
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                x[i] = i < left ? __builtin_amdgcn_cvt_f32_fp8(int(b[i]), 0) : 0.f;
        }
    } else {
        const T* p = static_cast<const T*>(base) + e;
        if constexpr (VEC) {
            unpack8<T>(*reinterpret_cast<const U16x8*>(p), x);
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = i < left ? to_f<T>(p[i]) : 0.f;
        }
    }
}

template <typename T, bool F8>
__device__ __forceinline__ float load1(const void* __restrict__ base, int64_t e) {
    if constexpr (F8) {
        return __builtin_amdgcn_cvt_f32_fp8(int(static_cast<const uint8_t*>(base)[e]), 0);
    } else {
        return to_f<T>(static_cast<const T*>(base)[e]);
    }
}

template <typename T, bool F8, bool VEC>
__global__ void __launch_bounds__(64) general_attention_kernel(GeneralAttention a) {
    __shared__ __align__(16) float qs[GH][DMAX];
    __shared__ float ps[GH][64];
    const int lane = threadIdx.x;
    const int group = a.heads / a.kv_heads;
    const int chunks = (group + GH - 1) / GH;
    const int64_t bx = blockIdx.x;
    const int hc = int(bx % chunks);
    const int64_t ik = bx / chunks;
    const int kvh = int(ik % a.kv_heads);
    const int64_t item = ik / a.kv_heads;
    const int64_t qi = blockIdx.y;

    int64_t tok, qlen;
    if (a.rows) {
        tok = a.rows[item];
        qlen = 1;
    } else {
        const int64_t qb = a.q_offsets[item];
        qlen = a.q_offsets[item + 1] - qb;
        if (qi >= qlen) return;  // uniform per wave
        tok = qb + qi;
    }
    const int64_t ctx = a.lengths[item];
    const int64_t kv_end = ctx - qlen + qi + 1;  // decode: ctx
    const int g0 = hc * GH;
    const int gw = min(GH, group - g0);
    const int h0 = kvh * group + g0;
    const int D = a.head_dim;
    const int D8 = (D + 7) & ~7;
    T* const out = static_cast<T*>(a.out) + tok * a.ots;

    if (kv_end <= 0) {  // nothing to attend (a padded row): zeros
        for (int g = 0; g < gw; ++g)
            for (int d = lane; d < D; d += 64) out[(h0 + g) * a.ohs + d] = static_cast<T>(0.f);
        return;
    }

    const float qscale = a.scale * kLog2eG * a.k_scale;
    const T* const q = static_cast<const T*>(a.q) + tok * a.qts;
    for (int g = 0; g < gw; ++g)
        for (int d = lane; d < D8; d += 64)
            qs[g][d] = d < D ? to_f<T>(q[(h0 + g) * a.qhs + d]) * qscale : 0.f;
    __syncthreads();

    float m[GH], l[GH], acc[GH][4];
#pragma unroll
    for (int g = 0; g < GH; ++g) {
        m[g] = -INFINITY;
        l[g] = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[g][i] = 0.f;
    }
    const int64_t table = a.offsets[item];
    const int bs = a.block_size;
    const int64_t head_off = int64_t(kvh) * a.chs;

    for (int64_t t0 = 0; t0 < kv_end; t0 += 64) {
        const bool valid = t0 + lane < kv_end;
        const int64_t t = min(t0 + lane, kv_end - 1);  // masked lanes read a valid row
        const int64_t page = t / bs;
        const int64_t slot = a.blocks[table + page] * bs + (t - page * bs);
        const int64_t kb = slot * a.css + head_off;

        float s[GH];
#pragma unroll
        for (int g = 0; g < GH; ++g) s[g] = 0.f;
        for (int d = 0; d < D8; d += 8) {
            float x[8];
            load8<T, F8, VEC>(a.k, kb + d, D - d, x);
#pragma unroll
            for (int g = 0; g < GH; ++g) {
                if (g >= gw) continue;  // uniform
                const float4 qa = *reinterpret_cast<const float4*>(&qs[g][d]);
                const float4 qb = *reinterpret_cast<const float4*>(&qs[g][d + 4]);
                float v = s[g];
                v = fmaf(qa.x, x[0], v);
                v = fmaf(qa.y, x[1], v);
                v = fmaf(qa.z, x[2], v);
                v = fmaf(qa.w, x[3], v);
                v = fmaf(qb.x, x[4], v);
                v = fmaf(qb.y, x[5], v);
                v = fmaf(qb.z, x[6], v);
                v = fmaf(qb.w, x[7], v);
                s[g] = v;
            }
        }
        // Online softmax per head (base 2); lane 0's key is always valid, so
        // every chunk maximum is finite.
#pragma unroll
        for (int g = 0; g < GH; ++g) {
            if (g >= gw) continue;
            const float sg = valid ? s[g] : -INFINITY;
            const float mn = fmaxf(m[g], wave_max(sg));
            const float alpha = exp2f(m[g] - mn);
            const float p = exp2f(sg - mn);
            l[g] = l[g] * alpha + wave_sum(p);
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[g][i] *= alpha;
            m[g] = mn;
            ps[g][lane] = p;
        }
        __syncthreads();
        const int n = int(min<int64_t>(64, kv_end - t0));
        const uint32_t slo = uint32_t(slot), shi = uint32_t(uint64_t(slot) >> 32);
#pragma unroll 4
        for (int j = 0; j < n; ++j) {
            const int64_t sj = int64_t((uint64_t(uint32_t(__shfl(int(shi), j, 64))) << 32) |
                                       uint32_t(__shfl(int(slo), j, 64)));
            const int64_t vb = sj * a.css + head_off;
            float vv[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int d = lane + 64 * i;
                vv[i] = d < D ? load1<T, F8>(a.v, vb + d) : 0.f;
            }
#pragma unroll
            for (int g = 0; g < GH; ++g) {
                if (g >= gw) continue;
                const float p = ps[g][j];
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[g][i] = fmaf(p, vv[i], acc[g][i]);
            }
        }
        __syncthreads();  // ps is rewritten by the next chunk
    }

#pragma unroll
    for (int g = 0; g < GH; ++g) {
        if (g >= gw) continue;
        const float inv = a.v_scale / l[g];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int d = lane + 64 * i;
            if (d < D) out[(h0 + g) * a.ohs + d] = static_cast<T>(acc[g][i] * inv);
        }
    }
}

// ------------------------------------------------- matrix-core kernels ----
// The reference's head dims (32, 64, 128, 256) with vector-aligned cache
// rows, on 16x16x32 MFMAs. Both kernels compute S^T = K Q^T (a lane holds the
// scores of query row lane % 16) and O^T = V^T P^T, whose B operand is exactly
// the lane's own scores and whose accumulators belong to the same query row:
// the softmax, its rescaling and the output are lane-local, with two shuffles
// per reduction over the keys. The k index of P.V runs over 32 keys in the
// order (quad, tile, i) of the score layout: key 16 * tile + 4 * quad + i at
// k = 8 * quad + 4 * tile + i.
//
// Precision: Q.K^T takes the stored 16-bit values (their products are exact
// in fp32) and the scale is applied in fp32; P enters P.V as two terms of the
// storage type (P rounded, and the rounded remainder: 16 bits for bf16, 22
// for fp16), the denominator sums the unrounded P, accumulation is fp32.
// fp16 has no exponents below 2^-14 and no values below 2^-24: its weights
// are carried times 2^kLift, which puts the rounding of any of them below
// 2^-36 of the row's largest (2^-25 without; a row whose largest weight meets
// V = 0, as attention sinks have it, then came out wrong: its other keys 2^22
// below the largest 0.3 % off, 2^26 below it zero).

typedef f32x4_t gf32x4;

// Elements 2 * w and 2 * w + 1 of words a (first) and b: the even (or odd)
// elements of the two side by side.
__device__ __forceinline__ uint32_t pair_lo(uint32_t a, uint32_t b) {
    return __builtin_amdgcn_perm(b, a, 0x05040100u);
}
__device__ __forceinline__ uint32_t pair_hi(uint32_t a, uint32_t b) {
    return __builtin_amdgcn_perm(b, a, 0x07060302u);
}

// Two FP8 elements (the low or high half of w) widened exactly to one word of T.
template <typename T, bool HI>
__device__ __forceinline__ uint32_t widen2(uint32_t w) {
    if constexpr (std::is_same_v<T, __bf16>) {
        return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.f, HI));
    } else {
        return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.f, HI));
    }
}

// P of a 32-key group (8 scores' weights, k order) as the two B operands.
template <typename T>
__device__ __forceinline__ void split_p(const float (&p)[8], U16x8& hi, U16x8& lo) {
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        hi.w[w] = pack2<T>(p[2 * w], p[2 * w + 1]);
        lo.w[w] = pack2<T>(p[2 * w] - half_lo<T>(hi.w[w]), p[2 * w + 1] - half_hi<T>(hi.w[w]));
    }
}

// 16 bytes at an 8-byte boundary.
struct alignas(8) U16x8Half {
    uint32_t w[4];
};

// Max / sum over the four quads that share a query row.
__device__ __forceinline__ float quad_max(float v) {
    v = fmaxf(v, __shfl_xor(v, 16, 64));
    return fmaxf(v, __shfl_xor(v, 32, 64));
}
__device__ __forceinline__ float quad_sum(float v) {
    v += __shfl_xor(v, 16, 64);
    return v + __shfl_xor(v, 32, 64);
}

// Weights are 2^(score - m + kLift): fp16's largest, 2^15, are below its
// 65504. Partial results that leave the kernel (sums and accumulators) state
// m - kLift as their reference, so that they merge with unlifted ones.
template <typename T>
constexpr float kLift = std::is_same_v<T, _Float16> ? 11.f : 0.f;
template <typename T>
constexpr float kSlack = std::is_same_v<T, _Float16> ? 4.f : 8.f;

// The online softmax of one step: x holds the lane's scores (base 2, masked
// ones -inf) and becomes the weights 2^(x - m + kLift). The reference m
// follows the running maximum only once some row of the wave exceeds it by
// kSlack: until then the weights stay below 2^(kSlack + kLift) and nothing
// needs rescaling. Returns whether it moved; `alpha` is then the factor of
// what was summed before. Rows with no key yet keep m = -inf and weights 0.
template <typename T, int N>
__device__ __forceinline__ bool softmax_step(float (&x)[N], float& m, float& l, float& alpha) {
    float top = x[0];
#pragma unroll
    for (int i = 1; i < N; ++i) top = fmaxf(top, x[i]);
    top = quad_max(top);
    const bool moved = __any(top > m + kSlack<T>);  // m = -inf: any key at all
    if (moved) {
        const float mn = fmaxf(m, top);
        alpha = mn == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - mn);
        m = mn;
        l *= alpha;
    }
    const float base = m == -INFINITY ? 0.f : m - kLift<T>;
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        x[i] = __builtin_amdgcn_exp2f(x[i] - base);
        sum += x[i];
    }
    l += sum;  // this lane's share of the denominator
    return moved;
}

// Eight elements of a query row as an operand piece.
template <typename T>
__device__ __forceinline__ U16x8 load_query(const T* p, bool vec) {
    if (vec) return *reinterpret_cast<const U16x8*>(p);
    U16x8 r;
#pragma unroll
    for (int w = 0; w < 4; ++w)
        r.w[w] = uint32_t(__builtin_bit_cast(uint16_t, p[2 * w])) |
                 uint32_t(__builtin_bit_cast(uint16_t, p[2 * w + 1])) << 16;
    return r;
}

// Writes n (a multiple of 4) consecutive elements, rounded to T.
template <typename T, int N>
__device__ __forceinline__ void store_row(T* o, const float (&x)[N], float inv, bool vec) {
    if (vec) {
#pragma unroll
        for (int i = 0; i < N; i += 4)
            *reinterpret_cast<uint2*>(o + i) =
                make_uint2(pack2<T>(x[i] * inv, x[i + 1] * inv),
                           pack2<T>(x[i + 2] * inv, x[i + 3] * inv));
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i) o[i] = static_cast<T>(x[i] * inv);
    }
}

// V with infinities or NaNs. They meet zero weights above - masked and repeated
// keys, the remainder of an exact P - and 0 * inf is NaN where the sum over a
// row's own keys may be an infinity, or finite. So a workgroup whose
// accumulators end non-finite goes through its keys once more, EXACT: such
// elements enter P.V as 0, for each output dim the first key with a positive
// and with a negative one is noted (NaNs count as both), and the rows that see
// that key take the infinity, or the two as a NaN. Other rows keep their bits.
// In us, calls with one infinity against the same in fp32 on the vector units:
// 64 x 2048 decode rows, heads of 64 165 -> 70; 4 x 512 queries over 2048 tokens,
// heads of 64 / 256 2241 / 3298 -> 191 / 440; with NaNs throughout, 16 x 2048
// decode rows, heads of 64 / 256 54 / 87 -> 54 / 268. (The second pass called out
// of line cost every call scratch memory, 5 us and more.)

template <typename T>
__device__ __forceinline__ bool non_finite(uint32_t h) {  // of the low 16 bits
    constexpr uint32_t kExp = std::is_same_v<T, __bf16> ? 0x7f80u : 0x7c00u;
    return (h & kExp) == kExp;
}

// Zeroes the non-finite ones of a word's two elements: those whose magnitude,
// as an integer, exceeds the largest finite one's. Returns 0xffff in their halves.
template <typename T>
__device__ __forceinline__ uint32_t drop_non_finite(uint32_t& w) {
    typedef int16_t i16x2 __attribute__((ext_vector_type(2)));
    constexpr int16_t kMax = std::is_same_v<T, __bf16> ? 0x7f7f : 0x7bff;
    const i16x2 over = (i16x2{kMax, kMax} - __builtin_bit_cast(i16x2, w & 0x7fff7fffu)) >> 15;
    const uint32_t mask = __builtin_bit_cast(uint32_t, over);
    w &= ~mask;
    return mask;
}

// The same for the NaNs (0x7f, 0xff) of four FP8 elements; a bit for any.
__device__ __forceinline__ uint32_t drop_fp8_nan(uint32_t& w) {
    uint32_t any = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (((w >> (8 * i)) & 0x7f) == 0x7f) {
            w &= ~(0xffu << (8 * i));
            any = 1;
        }
    return any;
}

template <int D>
struct FirstSpecial {
    int plus[D], minus[D];  // key index, by output dim
    __device__ __forceinline__ void clear(int thread, int threads) {
        for (int i = thread; i < D; i += threads) plus[i] = minus[i] = INT32_MAX;
    }
    // Notes element h of `dim` at `key` if it is not finite.
    template <typename T>
    __device__ __forceinline__ void note(uint32_t h, int dim, int key) {
        constexpr uint32_t kMant = std::is_same_v<T, __bf16> ? 0x7fu : 0x3ffu;
        if (!non_finite<T>(h)) return;
        const bool nan = (h & kMant) != 0, neg = (h & 0x8000u) != 0;
        if (nan || !neg) atomicMin(&plus[dim], key);
        if (nan || neg) atomicMin(&minus[dim], key);
    }
    // What a row that sees keys below `bound` adds to its sum.
    __device__ __forceinline__ float value(int dim, int64_t bound) const {
        return (plus[dim] < bound ? INFINITY : 0.f) + (minus[dim] < bound ? -INFINITY : 0.f);
    }
};

// Few query rows against many keys: decode, and prefill calls of a few
// queries. A workgroup serves up to 16 (query token, query head) rows of one
// KV head: one query's group of heads (up to 16), or for groups below 16
// several consecutive queries of one prefill item, each row with its own
// causal bound. Its four waves take interleaved chunks of CH keys straight
// from the cache into operand registers, with no LDS on the way: lane (col,
// quad) holds the K pieces of key col as the A operand, and of V the dims
// VE * col .. of the keys 4 * quad + i, which gathered by element (v_perm)
// are the A operand of one MFMA per element. The next chunk's K loads are
// issued right after Q.K^T, its V loads after P.V. The waves' (max, sum,
// accumulator) merge through LDS at the end.
//
// Bound by the rate of its loads at many rows, by their latency along the
// longest row at few. In us, against fp32 arithmetic on the vector units
// (K and V broadcast to the query rows' lanes): 64 rows x 2048 tokens, 32
// query and 8 KV heads of 64 165 -> 46 (268 MB in graph replay, some of them
// left in the 256 MB memory-side cache), of 256 362 -> 177 (6.1 TB/s); 256 / 8
// heads of 128 888 -> 159; 33 rows of 1-4096 tokens, heads of 64 170 -> 52 with
// the merge. Two tiles per chunk rather than four (148 registers at head dim
// 64, three waves per SIMD): 1-7 % there.
// Waves per SIMD at most. Two for fp16 at head dim 64: rows of mixed lengths run
// faster with their workgroups spread over the CUs (33 rows of 1-4096 tokens,
// 32 / 8 heads, 41.5 us against 46.6 with the three that registers allow), short
// ones slower (128 x 100 12.0 against 11.4).
template <typename T, bool F8, int D>
constexpr int kRowsWavesMax = D == 64 && !F8 && std::is_same_v<T, _Float16> ? 2 : 8;

template <typename T, bool F8, int D>
__global__ void __launch_bounds__(64 * kRowWaves)
    __attribute__((amdgpu_waves_per_eu(1, kRowsWavesMax<T, F8, D>)))
rows_attention_kernel(GeneralAttention a) {
    constexpr int NT = 2;                // 16-key tiles per chunk
    constexpr int CH = 16 * NT;
    constexpr int KS = D / 32;           // Q.K^T steps
    constexpr int VE = D / 16;           // dims per lane and key of V
    constexpr int NW = kRowWaves;
    constexpr int EB = F8 ? 1 : 2;       // cache bytes per element
    constexpr int VW = VE / 2;           // V words per key, widened
    __shared__ float part_acc[(NW - 1) * VE * 4 * 64];
    __shared__ float part_ml[NW - 1][2][64];
    __shared__ FirstSpecial<D> special;
    __shared__ bool again[NW];
    const int wave = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    const int col = lane & 15, quad = lane >> 4;

    const int group = a.heads / a.kv_heads;
    const int hpq = group >= GH ? GH : group;       // heads per query
    const int qpw = group >= GH ? 1 : GH / group;   // queries per workgroup
    const int chunks = (group + GH - 1) / GH;
    const int64_t bx = blockIdx.x;
    const int hc = int(bx % chunks);
    const int64_t ik = bx / chunks;
    const int kvh = int(ik % a.kv_heads);
    const int64_t item = ik / a.kv_heads;
    // Prefill: y is the workgroup's tile of queries. Decode: its split of
    // the row's keys (one query).
    const int64_t q0 = a.rows ? 0 : int64_t(blockIdx.y) * qpw;
    const int64_t split = a.rows ? int64_t(blockIdx.y) : 0;

    int64_t tok0, qlen;
    if (a.rows) {
        tok0 = a.rows[item];
        qlen = 1;
    } else {
        tok0 = a.q_offsets[item];
        qlen = a.q_offsets[item + 1] - tok0;
        if (q0 >= qlen) return;  // uniform per workgroup
        tok0 += q0;
    }
    const int64_t nq = min<int64_t>(qpw, qlen - q0);
    const int g0 = hc * GH;
    const int hw = min(hpq, group - g0);
    const int nrows = int(nq) * hw;
    const int64_t ctx = a.lengths[item];
    const int64_t first_end = ctx - qlen + q0 + 1;  // causal bound of the first query
    const int64_t kv_max = first_end + nq - 1;       // ... and of the last
    T* const out = static_cast<T*>(a.out);
    // Keys [k_begin, k_end) of this split (all of them when unsplit). The
    // last split also takes any keys past splits * split_keys (a row longer
    // than the max_context the plan was sized for): slow, never wrong.
    const int64_t k_begin = split * a.split_keys;
    const int64_t k_end = a.splits > 1 && split + 1 < a.splits
        ? min(kv_max, k_begin + a.split_keys) : kv_max;
    const int row = min(col, nrows - 1);  // this lane's query row
    const int64_t token = tok0 + row / hw;
    const int head = kvh * group + g0 + row % hw;
    const int64_t part = (item * a.heads + head) * a.splits + split;

    if (a.splits > 1 && k_begin >= k_end) {  // no key of the row in this split
        if (wave == 0 && quad == 0 && col < nrows) {
            a.part_ml[2 * part] = -INFINITY;  // the merge skips it
            a.part_ml[2 * part + 1] = 0.f;
        }
        return;  // uniform per workgroup
    }
    if (kv_max <= 0) {  // no key for any row (a padded decode row): zeros, and
                        // no read of its block table, which may hold no entry
        for (int i = threadIdx.x; i < nrows * D; i += 64 * NW) {
            const int r = i / D;
            out[(tok0 + r / hw) * a.ots + (kvh * group + g0 + r % hw) * a.ohs + i % D] =
                static_cast<T>(0.f);
        }
        return;  // uniform per workgroup
    }
    U16x8 qb[KS];
    const T* const q = static_cast<const T*>(a.q) + token * a.qts + head * a.qhs + 8 * quad;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        qb[s] = load_query<T>(q + 32 * s, a.q_vec);
        if (col >= nrows) qb[s] = U16x8{};
    }
    // Keys this lane's row attends: none beyond the group's rows.
    const int64_t bound = col < nrows ? min(first_end + row / hw, k_end) : 0;
    const float qscale = a.scale * kLog2eG * a.k_scale;

    const int64_t table = a.offsets[item];
    const uint32_t bs = uint32_t(a.block_size);
    const char* const kc = static_cast<const char*>(a.k) + int64_t(kvh) * a.chs * EB;
    const char* const vc = static_cast<const char*>(a.v) + int64_t(kvh) * a.chs * EB;
    // The cache row of chunk key t0 + lane % CH (past the end: the row's last
    // key, a valid row that the mask drops), in two steps: its block id, whose
    // load is issued a chunk ahead of its use, and its byte offset.
    auto load_id = [&](int64_t t0) -> int64_t {
        return a.blocks[table + uint32_t(min(t0 + lane % CH, kv_max - 1)) / bs];
    };
    auto resolve = [&](int64_t t0, int64_t id) -> int64_t {
        const uint32_t t = uint32_t(min(t0 + lane % CH, kv_max - 1));
        return (id * bs + t % bs) * a.css * EB;
    };
    auto at = [&](int64_t off, int key) -> int64_t {
        const uint32_t lo = uint32_t(__shfl(int(uint32_t(off)), key, 64));
        const uint32_t hi = uint32_t(__shfl(int(uint32_t(uint64_t(off) >> 32)), key, 64));
        return int64_t(uint64_t(hi) << 32 | lo);
    };
    using KPiece = std::conditional_t<F8, uint2, U16x8>;
    KPiece kreg[NT][KS];
    constexpr int VB = VE * EB;  // V bytes per lane and key
    uint32_t vreg[NT][4][(VB + 3) / 4];
    auto load_k = [&](int64_t off) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const char* const p = kc + at(off, 16 * j + col) + 8 * quad * EB;
#pragma unroll
            for (int s = 0; s < KS; ++s)
                kreg[j][s] = *reinterpret_cast<const KPiece*>(p + 32 * s * EB);
        }
    };
    auto load_v = [&](int64_t off) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const char* const p = vc + at(off, 16 * j + 4 * quad + i) + col * VB;
                if constexpr (VB == 2) {
                    vreg[j][i][0] = *reinterpret_cast<const uint16_t*>(p);
                } else if constexpr (VB == 4) {
                    vreg[j][i][0] = *reinterpret_cast<const uint32_t*>(p);
                } else if constexpr (VB == 8) {
                    const uint2 x = *reinterpret_cast<const uint2*>(p);
                    vreg[j][i][0] = x.x;
                    vreg[j][i][1] = x.y;
                } else {
                    // FP8 rows are 8-byte aligned only.
                    using V16 = std::conditional_t<F8, U16x8Half, U16x8>;
#pragma unroll
                    for (int w = 0; w < VB / 16; ++w) {
                        const V16 x = *reinterpret_cast<const V16*>(p + 16 * w);
#pragma unroll
                        for (int y = 0; y < 4; ++y) vreg[j][i][4 * w + y] = x.w[y];
                    }
                }
            }
    };
    // Word w (elements 2w, 2w + 1) of the lane's V piece of key (j, i), in T.
    auto v_word = [&](int j, int i, int w) -> uint32_t {
        if constexpr (F8) {
            return (w & 1) ? widen2<T, true>(vreg[j][i][w / 2])
                           : widen2<T, false>(vreg[j][i][w / 2]);
        } else {
            return vreg[j][i][w];
        }
    };

    gf32x4 acc[VE];  // acc[e][v]: dim VE * (4 * quad + v) + e of the lane's row
    float m = -INFINITY, l = 0.f;
#pragma unroll
    for (int e = 0; e < VE; ++e) acc[e] = gf32x4{0.f, 0.f, 0.f, 0.f};
    float x[4 * NT];
    auto scores = [&](int64_t t0) {
        // Keys of the chunk from this quad's first on that the row sees.
        const int left = int(max<int64_t>(min<int64_t>(bound - t0, CH), 0)) - 4 * quad;
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            gf32x4 sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < KS; ++s) {
                if constexpr (F8) sc = mfma32<T>(fp8x8_widen<T>(kreg[j][s]), qb[s], sc);
                else sc = mfma32<T>(kreg[j][s], qb[s], sc);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
                x[4 * j + i] = 16 * j + i < left ? sc[i] * qscale : -INFINITY;
        }
    };
    auto attend = [&]<bool EXACT>(std::bool_constant<EXACT>, int64_t t0, int64_t off) {
        float alpha;
        if (softmax_step<T>(x, m, l, alpha)) {
#pragma unroll
            for (int e = 0; e < VE; ++e) acc[e] *= alpha;
        }
        if constexpr (EXACT) {
            static_assert(NT == 2, "one group of 32 keys");
            uint32_t flagged = 0;
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    uint32_t any = 0;
#pragma unroll
                    for (int w = 0; w < (VB + 3) / 4; ++w) {
                        if constexpr (F8) any |= drop_fp8_nan(vreg[j][i][w]);
                        else any |= drop_non_finite<T>(vreg[j][i][w]);
                    }
                    flagged |= uint32_t(any != 0) << (4 * j + i);
                }
#pragma unroll 1
            for (int e = 0; e < 8; ++e) {
                const bool mine = (flagged >> e) & 1;
                if (!__any(mine)) continue;
                const int key = 16 * (e / 4) + 4 * quad + e % 4;
                const char* const vk = vc + at(off, key) + col * VB;
                if (!mine || t0 + key >= k_end) continue;
#pragma unroll 1
                for (int n = 0; n < VE; ++n) {
                    uint32_t h;
                    if constexpr (F8) {
                        const uint32_t x = reinterpret_cast<const uint8_t*>(vk)[n];
                        h = (x & 0x7f) == 0x7f ? 0x7fffu : 0u;
                    } else {
                        h = reinterpret_cast<const uint16_t*>(vk)[n];
                    }
                    special.template note<T>(h, VE * col + n, int(t0) + key);
                }
            }
        }
#pragma unroll
        for (int g = 0; g < NT / 2; ++g) {
            float p[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) p[i] = x[8 * g + i];
            U16x8 hi, lo;
            split_p<T>(p, hi, lo);
#pragma unroll
            for (int w = 0; w < VW; ++w) {
                U16x8 even, odd;
#pragma unroll
                for (int y = 0; y < 4; ++y) {
                    const int j = 2 * g + y / 2, i = 2 * (y & 1);
                    const uint32_t v0 = v_word(j, i, w), v1 = v_word(j, i + 1, w);
                    even.w[y] = pair_lo(v0, v1);
                    odd.w[y] = pair_hi(v0, v1);
                }
                acc[2 * w] = mfma32<T>(even, hi, acc[2 * w]);
                acc[2 * w + 1] = mfma32<T>(odd, hi, acc[2 * w + 1]);
                acc[2 * w] = mfma32<T>(even, lo, acc[2 * w]);
                acc[2 * w + 1] = mfma32<T>(odd, lo, acc[2 * w + 1]);
            }
        }
    };

    // Wave w takes chunks w, w + NW, ... of the keys.
    int64_t t0 = k_begin + int64_t(wave) * CH;
    if (t0 < k_end) {
        constexpr int64_t kStep = NW * CH;
        int64_t off = resolve(t0, load_id(t0));
        int64_t id = load_id(t0 + kStep);
        load_k(off);
        load_v(off);
        asm volatile("" ::: "memory");  // see below
        for (; t0 < k_end; t0 += kStep) {
            off = resolve(t0 + kStep, id);
            id = load_id(t0 + 2 * kStep);
            scores(t0);
            load_k(off);
            // The scheduler would gather V's operands ahead of these loads,
            // and wait for V there.
            __builtin_amdgcn_sched_barrier(0);
            attend(std::false_type{}, t0, off);
            load_v(off);
            // Nothing is written; but a possible write keeps the compiler from
            // turning the loaded values carried into the next iteration into
            // loads there, right in front of their uses.
            asm volatile("" ::: "memory");
        }
    }
    l = quad_sum(l);

    // Merge the waves' partial results: out = sum_w 2^(m_w - M) acc_w /
    // sum_w 2^(m_w - M) l_w per row (M the largest m_w); a row with no key
    // in any wave gives zeros.
    auto publish = [&] {
        if (wave == 0) return;
#pragma unroll
        for (int e = 0; e < VE; ++e)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                part_acc[((wave - 1) * VE * 4 + 4 * e + v) * 64 + lane] = acc[e][v];
        part_ml[wave - 1][0][lane] = m;
        part_ml[wave - 1][1][lane] = l;
    };
    publish();
    gf32x4 sums = acc[0];  // four chains
#pragma unroll
    for (int e = 1; e < VE; ++e) sums += acc[e];
    const float sum = l + ((sums[0] + sums[1]) + (sums[2] + sums[3]));
    const bool bad = __any(col < nrows && !(fabsf(sum) < INFINITY));
    if (lane == 0) again[wave] = bad;
    __syncthreads();
    // Unlikely, said so to have what follows it next in line.
    if (__builtin_expect(again[0] || again[1] || again[2] || again[3], 0)) {  // uniform
#pragma unroll
        for (int e = 0; e < VE; ++e) acc[e] = gf32x4{0.f, 0.f, 0.f, 0.f};
        m = -INFINITY;
        l = 0.f;
        special.clear(threadIdx.x, 64 * NW);
        __syncthreads();
        for (int64_t t = k_begin + int64_t(wave) * CH; t < k_end; t += NW * CH) {
            const int64_t off = resolve(t, load_id(t));
            load_k(off);
            scores(t);
            load_v(off);
            attend(std::true_type{}, t, off);
        }
        l = quad_sum(l);
        publish();
        __syncthreads();
        if (wave == 0) {
#pragma unroll
            for (int e = 0; e < VE; ++e)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[e][v] += special.value(VE * (4 * quad + v) + e, bound);
        }
    }
    if (wave > 0) return;
    float mx = m;
#pragma unroll
    for (int w = 0; w < NW - 1; ++w) mx = fmaxf(mx, part_ml[w][0][lane]);
    const float w0 = mx == -INFINITY ? 0.f : exp2f(m - mx);
    float den = w0 * l;
#pragma unroll
    for (int e = 0; e < VE; ++e) acc[e] *= w0;
    for (int w = 0; w < NW - 1; ++w) {
        const float ww = mx == -INFINITY ? 0.f : exp2f(part_ml[w][0][lane] - mx);
        den += ww * part_ml[w][1][lane];
        if (ww == 0.f) continue;
#pragma unroll
        for (int e = 0; e < VE; ++e)
#pragma unroll
            for (int v = 0; v < 4; ++v)
                acc[e][v] += ww * part_acc[(w * VE * 4 + 4 * e + v) * 64 + lane];
    }
    float o[4 * VE];  // the lane's 4 * VE consecutive dims
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int e = 0; e < VE; ++e) o[v * VE + e] = acc[e][v];
    if (col >= nrows) return;
    if (a.splits > 1) {  // the split's partials, merged by general_merge
        float* const po = a.part_o + part * D + 4 * VE * quad;
#pragma unroll
        for (int i = 0; i < 4 * VE; i += 4)
            *reinterpret_cast<float4*>(po + i) = make_float4(o[i], o[i + 1], o[i + 2], o[i + 3]);
        if (quad == 0) {
            a.part_ml[2 * part] = mx - kLift<T>;
            a.part_ml[2 * part + 1] = den;
        }
        return;
    }
    store_row<T>(out + token * a.ots + head * a.ohs + 4 * VE * quad, o,
                 den > 0.f ? a.v_scale / den : 0.f, a.out_vec);
}

// Many query rows: prefill chunks. A workgroup of four waves serves up to
// 64 * RT consecutive (query, head) rows of one KV head and item (row r is
// query r / group, head r % group), 16 * RT per wave, each row with its own
// causal bound. All waves walk the same keys, KC at a time, staged in LDS
// for all of them: K as stored, V transposed into the k order of P.V, so
// that every operand is one 16-byte LDS read. Two buffers, the next chunk's
// global loads in flight while this one computes, one barrier per chunk.
// With HV = 2 a second set of four waves takes every other chunk of the same
// rows' keys through buffers of its own, and the two merge at the end.
//
// Bound by the instruction stream of a SIMD's waves (softmax and staging
// against 48 MFMAs per 32 keys at head dim 256) and by LDS bandwidth at RT = 1
// (1 KiB of operand per 16-cycle MFMA and wave). Registers are held to 256, so
// that two waves share a SIMD. In us, against the vector-unit kernel: 4 x 512
// queries over 2048 tokens, 32 query and 8 KV heads of 64 2241 -> 81 (370
// TFLOP/s), of 256 6520 -> 303 (397 TFLOP/s); 2 x 256 over 1033, 16 / 8 heads
// of 256 482 -> 50.
template <typename T, bool F8, int D, int RT, int HV>
__global__ void __launch_bounds__(64 * kRowWaves * HV, 2)
tiles_attention_kernel(GeneralAttention a) {
    constexpr int KC = D > 128 ? 32 : 64;  // keys per chunk
    constexpr int KS = D / 32;             // Q.K^T steps
    constexpr int DT = D / 16;             // 16-dim tiles of the output
    constexpr int G = KC / 32;             // P.V steps
    constexpr int NT = 64 * kRowWaves;
    // Row strides padded by 16 bytes: the 16 rows that a quarter wave reads
    // at once start 4 banks apart.
    constexpr int KSTR = D * 2 + 16, VSTR = KC * 2 + 16;
    constexpr int kBuf = KC * KSTR + D * VSTR;
    __shared__ __align__(16) unsigned char smem_all[HV * 2 * kBuf];
    __shared__ int64_t row_offs[HV][2][KC];  // byte offsets of a chunk's cache rows
    __shared__ FirstSpecial<D> special;
    __shared__ bool again[HV * kRowWaves];
    // (Uniform per wave, said so to keep them in scalar registers.)
    const int half = HV == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
    int tid = threadIdx.x % NT;  // within the half
    unsigned char* const smem = smem_all + half * 2 * kBuf;
    int64_t (*const row_off)[KC] = row_offs[half];
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int lane = tid & 63, col = lane & 15, quad = lane >> 4;

    const int group = a.heads / a.kv_heads;
    const int kvh = int(blockIdx.x % a.kv_heads);
    const int64_t item = blockIdx.x / a.kv_heads;
    const int64_t tok0 = a.q_offsets[item];
    const int64_t qlen = a.q_offsets[item + 1] - tok0;
    const int64_t total = qlen * group;
    const int64_t r0 = int64_t(blockIdx.y) * (64 * RT);
    if (r0 >= total) return;  // uniform per workgroup
    const int64_t ctx = a.lengths[item];
    const int64_t before = ctx - qlen;
    const int64_t last = min(r0 + 64 * RT, total) - 1;  // the workgroup's last row
    const int64_t kv_max = before + last / group + 1;   // and the keys it sees
    T* const out = static_cast<T*>(a.out);
    const int64_t wr0 = r0 + wave * 16 * RT;  // the wave's first row

    U16x8 qb[RT][KS];
    int64_t bound[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        const int64_t r = wr0 + 16 * t + col;
        const bool has = r < total;
        const int64_t query = (has ? r : 0) / group;
        const int head = kvh * group + int((has ? r : 0) % group);
        bound[t] = has ? before + query + 1 : 0;
        const T* const q = static_cast<const T*>(a.q) + (tok0 + query) * a.qts + head * a.qhs +
                           8 * quad;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            qb[t][s] = load_query<T>(q + 32 * s, a.q_vec);
            if (!has) qb[t][s] = U16x8{};
        }
    }
    // Keys beyond the wave's last row's bound are none of its business.
    const int64_t wave_end = wr0 < total
        ? before + min(wr0 + 16 * RT - 1, total - 1) / group + 1 : 0;
    const float qscale = a.scale * kLog2eG * a.k_scale;

    gf32x4 acc[RT][DT];  // acc[t][d][v]: dim 16 * d + 4 * quad + v of row 16 * t + col
    float m[RT], l[RT];

    // Staging. K: 8-element pieces, a key's pieces side by side in the lanes.
    // V: 4 keys x 8 dims per task, transposed in registers; 8 lanes hold 64
    // dims of the same keys (one 128-byte line each), 8 groups of lanes the
    // keys of a 32-key step.
    constexpr int kPieces = KC * (D / 8);
    constexpr int kPer = (kPieces + NT - 1) / NT;
    constexpr int kTasks = (KC / 4) * (D / 8);
    constexpr int kVPer = (kTasks + NT - 1) / NT;
    using Piece = std::conditional_t<F8, uint2, U16x8>;
    constexpr int EB = F8 ? 1 : 2;
    Piece kst[kPer], vst[kVPer][4];
    const int64_t table = a.offsets[item];
    const uint32_t bs = uint32_t(a.block_size);
    const char* const kc = static_cast<const char*>(a.k) + int64_t(kvh) * a.chs * EB;
    const char* const vc = static_cast<const char*>(a.v) + int64_t(kvh) * a.chs * EB;
    // Thread x < KC resolves key x of each chunk (past the end: the last key, a
    // valid row): its block id two chunks ahead of the chunk's loads, its
    // byte offset into LDS one chunk ahead, for all threads.
    auto load_id = [&](int64_t t0) -> int64_t {
        return a.blocks[table + uint32_t(min(t0 + tid % KC, kv_max - 1)) / bs];
    };
    auto put_offset = [&](int64_t t0, int64_t id, int slot) {
        const uint32_t t = uint32_t(min(t0 + tid % KC, kv_max - 1));
        if (tid < KC) row_off[slot][tid] = (id * bs + t % bs) * a.css * EB;
    };
    // Task x: 8-dim piece `oct` of keys 4 * kq .. + 3.
    auto v_task = [&](int x, int& oct, int& kq) {
        constexpr int OW = D / 8 < 8 ? D / 8 : 8;  // pieces side by side in the lanes
        const int inner = x % (OW * (KC / 4));
        oct = x / (OW * (KC / 4)) * OW + inner % OW;
        kq = inner / OW;
    };
    auto load_stage = [&](int slot) {
        const int64_t* const ro = row_off[slot];
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            const int x = tid + u * NT;
            if (kPieces % NT != 0 && x >= kPieces) break;
            kst[u] = *reinterpret_cast<const Piece*>(kc + ro[x / (D / 8)] +
                                                     (x % (D / 8)) * 8 * EB);
        }
#pragma unroll
        for (int u = 0; u < kVPer; ++u) {
            const int x = tid + u * NT;
            if (kTasks % NT != 0 && x >= kTasks) break;
            int oct, kq;
            v_task(x, oct, kq);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                vst[u][i] = *reinterpret_cast<const Piece*>(vc + ro[4 * kq + i] +
                                                            oct * 8 * EB);
        }
    };
    auto widen = [&](const Piece& x) -> U16x8 {
        if constexpr (F8) return fp8x8_widen<T>(x);
        else return x;
    };
    auto store_stage = [&](unsigned char* buf) {
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            const int x = tid + u * NT;
            if (kPieces % NT != 0 && x >= kPieces) break;
            *reinterpret_cast<U16x8*>(buf + (x / (D / 8)) * KSTR + (x % (D / 8)) * 16) =
                widen(kst[u]);
        }
#pragma unroll
        for (int u = 0; u < kVPer; ++u) {
            const int x = tid + u * NT;
            if (kTasks % NT != 0 && x >= kTasks) break;
            int oct, kq;
            v_task(x, oct, kq);
            const U16x8 r0v = widen(vst[u][0]), r1v = widen(vst[u][1]);
            const U16x8 r2v = widen(vst[u][2]), r3v = widen(vst[u][3]);
            // Keys 4 * kq .. + 3 of 32-key group kq / 8: tile (kq % 8) / 4,
            // quad kq % 4, so k = 8 * quad + 4 * tile + i.
            const int pos = 32 * (kq / 8) + 8 * (kq & 3) + 4 * ((kq & 7) >> 2);
            unsigned char* const vt = buf + KC * KSTR + oct * 8 * VSTR + pos * 2;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                *reinterpret_cast<uint2*>(vt + (2 * w) * VSTR) =
                    make_uint2(pair_lo(r0v.w[w], r1v.w[w]), pair_lo(r2v.w[w], r3v.w[w]));
                *reinterpret_cast<uint2*>(vt + (2 * w + 1) * VSTR) =
                    make_uint2(pair_hi(r0v.w[w], r1v.w[w]), pair_hi(r2v.w[w], r3v.w[w]));
            }
        }
    };

    constexpr int kStep = HV * KC;
    const int64_t first = half * KC;
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        m[t] = -INFINITY;
        l[t] = 0.f;
#pragma unroll
        for (int d = 0; d < DT; ++d) acc[t][d] = gf32x4{0.f, 0.f, 0.f, 0.f};
    }
    auto attend = [&]<bool EXACT>(std::bool_constant<EXACT>, int64_t t0,
                                  const unsigned char* buf) {
        const unsigned char* const ks = buf + col * KSTR + quad * 16;
        const unsigned char* const vs = buf + KC * KSTR + col * VSTR + quad * 16;
        // Operands are read ahead of the MFMAs that take them, all of K's at
        // once and V's behind Q.K^T: the compiler's own order reads one or two
        // ahead and waits out the LDS latency 32 times per chunk.
        auto k_at = [&](int j, int s) {
            return *reinterpret_cast<const U16x8*>(ks + 16 * j * KSTR + 64 * s);
        };
        auto v_at = [&](int d, int g) {
            return *reinterpret_cast<const U16x8*>(vs + 16 * d * VSTR + 64 * g);
        };
        U16x8 kk[2 * G][KS], vv[DT][G];  // (exact: read where they are taken)
        if constexpr (!EXACT) {
#pragma unroll
            for (int j = 0; j < 2 * G; ++j)
#pragma unroll
                for (int s = 0; s < KS; ++s) kk[j][s] = k_at(j, s);
            __builtin_amdgcn_sched_barrier(0);
        }
        gf32x4 sc[RT][2 * G];
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int j = 0; j < 2 * G; ++j) sc[t][j] = gf32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 2 * G; ++j) {
            if constexpr (EXACT) asm volatile("" ::: "memory");  // a few registers at a time
#pragma unroll
            for (int s = 0; s < KS; ++s)
#pragma unroll
                for (int t = 0; t < RT; ++t)
                    sc[t][j] = mfma32<T>(EXACT ? k_at(j, s) : kk[j][s], qb[t][s], sc[t][j]);
        }
        if constexpr (!EXACT) {
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
                for (int g = 0; g < G; ++g) vv[d][g] = v_at(d, g);
            __builtin_amdgcn_sched_barrier(0);
        }
        U16x8 hi[RT][G], lo[RT][G];
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            float x[8 * G];
            const int left = int(max<int64_t>(min<int64_t>(bound[t] - t0, KC), 0)) - 4 * quad;
#pragma unroll
            for (int j = 0; j < 2 * G; ++j)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    x[4 * j + i] = 16 * j + i < left ? sc[t][j][i] * qscale : -INFINITY;
            float alpha;
            if (softmax_step<T>(x, m[t], l[t], alpha)) {
#pragma unroll
                for (int d = 0; d < DT; ++d) acc[t][d] *= alpha;
            }
#pragma unroll
            for (int g = 0; g < G; ++g) {
                float p[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) p[i] = x[8 * g + i];
                split_p<T>(p, hi[t][g], lo[t][g]);
            }
        }
        [[maybe_unused]] uint32_t flagged[G] = {};  // by tile of the output dims
#pragma unroll
        for (int d = 0; d < DT; ++d)
#pragma unroll
            for (int g = 0; g < G; ++g) {
                if constexpr (EXACT) {
                    asm volatile("" ::: "memory");
                    vv[d][g] = v_at(d, g);
#pragma unroll
                    for (int w = 0; w < 4; ++w)
                        if (drop_non_finite<T>(vv[d][g].w[w])) flagged[g] |= 1u << d;
                }
#pragma unroll
                for (int t = 0; t < RT; ++t) {
                    acc[t][d] = mfma32<T>(vv[d][g], hi[t][g], acc[t][d]);
                    acc[t][d] = mfma32<T>(vv[d][g], lo[t][g], acc[t][d]);
                }
            }
        if constexpr (EXACT) {
#pragma unroll
            for (int g = 0; g < G; ++g)
#pragma unroll 1
                for (int d = 0; d < DT; ++d) {
                    if (!((flagged[g] >> d) & 1)) continue;
#pragma unroll 1
                    for (int e = 0; e < 8; ++e) {
                        const int key = int(t0) + 32 * g + 16 * (e / 4) + 4 * quad + e % 4;
                        const uint32_t h = *reinterpret_cast<const uint16_t*>(
                            vs + 16 * d * VSTR + 64 * g + 2 * e);
                        if (key < kv_max) special.template note<T>(h, 16 * d + col, key);
                    }
                }
        }
    };

    int64_t id = 0;
    if (kv_max > 0) {  // uniform per workgroup
        put_offset(first, load_id(first), 0);
        id = load_id(first + kStep);
        __syncthreads();
        load_stage(0);
    }
    asm volatile("" ::: "memory");  // keeps carried loads where they are issued
    int cur = 0;
    for (int64_t step = 0; step < kv_max; step += kStep, cur ^= 1) {
        const int64_t t0 = step + first;  // this half's chunk
        unsigned char* const buf = smem + cur * kBuf;
        store_stage(buf);
        put_offset(t0 + kStep, id, cur ^ 1);
        // After it, every wave is also past the reads of what the next
        // iteration overwrites (the other buffer, these offsets' predecessors).
        __syncthreads();
        id = load_id(t0 + 2 * kStep);
        load_stage(cur ^ 1);
        if (t0 < wave_end) attend(std::false_type{}, t0, buf);
    }
    // The lane's place once more, from the hardware: not kept through the loop.
    lane = int(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)));
    asm volatile("" : "+v"(lane));
    col = lane & 15;
    quad = lane >> 4;
    tid = 64 * wave + lane;
    bool bad = false;
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        gf32x4 sums = acc[t][0];  // four chains
#pragma unroll
        for (int d = 1; d < DT; ++d) sums += acc[t][d];
        const float sum = l[t] + ((sums[0] + sums[1]) + (sums[2] + sums[3]));
        bad = bad || (wr0 + 16 * t + col < total && !(fabsf(sum) < INFINITY));
    }
    bad = __any(bad);
    if (lane == 0) again[half * kRowWaves + wave] = bad;
    __syncthreads();  // also: every wave is past its reads of the buffers
    bad = false;
#pragma unroll
    for (int w = 0; w < HV * kRowWaves; ++w) bad = bad || again[w];
    if (__builtin_expect(bad, 0)) {  // uniform
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            m[t] = -INFINITY;
            l[t] = 0.f;
#pragma unroll
            for (int d = 0; d < DT; ++d) acc[t][d] = gf32x4{0.f, 0.f, 0.f, 0.f};
        }
        special.clear(threadIdx.x, HV * NT);
        for (int64_t step = 0; step < kv_max; step += kStep) {
            const int64_t t0 = step + first;
            put_offset(t0, load_id(t0), 0);
            __syncthreads();
            load_stage(0);
            store_stage(smem);
            __syncthreads();
            if (t0 < wave_end) attend(std::true_type{}, t0, smem);
            __syncthreads();  // every wave is past its reads of both
        }
        if (half == 0) {  // once, where the halves merge
#pragma unroll
            for (int t = 0; t < RT; ++t)
#pragma unroll
                for (int d = 0; d < DT; ++d)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        acc[t][d][v] += special.value(16 * d + 4 * quad + v, bound[t]);
        }
    }
    if constexpr (HV > 1) {
        // The second half's (max, sum, accumulators) join the first's, lane by
        // lane, through the staging buffers.
        float* const part = reinterpret_cast<float*>(smem_all) + wave * 64 + lane;
        constexpr int kStride = 64 * kRowWaves;
        static_assert((RT * (4 * DT + 2)) * kStride * 4 <= HV * 2 * kBuf, "merge fits the buffers");
        if (half == 1) {
#pragma unroll
            for (int t = 0; t < RT; ++t) {
                float* const p = part + t * (4 * DT + 2) * kStride;
                p[0] = m[t];
                p[kStride] = l[t];
#pragma unroll
                for (int d = 0; d < DT; ++d)
#pragma unroll
                    for (int v = 0; v < 4; ++v) p[(2 + 4 * d + v) * kStride] = acc[t][d][v];
            }
        }
        __syncthreads();
        if (half == 1) return;
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            const float* const p = part + t * (4 * DT + 2) * kStride;
            const float mx = fmaxf(m[t], p[0]);
            const float w0 = mx == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m[t] - mx);
            const float w1 = mx == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(p[0] - mx);
            l[t] = w0 * l[t] + w1 * p[kStride];
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    acc[t][d][v] = w0 * acc[t][d][v] + w1 * p[(2 + 4 * d + v) * kStride];
        }
    }
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        const float den = quad_sum(l[t]);
        const float inv = den > 0.f ? a.v_scale / den : 0.f;
        const int64_t r = wr0 + 16 * t + col;
        if (r >= total) continue;
        T* const o = out + (tok0 + r / group) * a.ots +
                     (kvh * group + int(r % group)) * a.ohs + 4 * quad;
#pragma unroll
        for (int d = 0; d < DT; ++d) {
            const float x[4] = {acc[t][d][0], acc[t][d][1], acc[t][d][2], acc[t][d][3]};
            store_row<T>(o + 16 * d, x, inv, a.out_vec);
        }
    }
}

// Merge a split decode: out = v_scale * sum_s 2^(m_s - M) o_s / sum_s
// 2^(m_s - M) l_s, M the largest m_s; splits with no key (m_s = -inf) are
// skipped, so their o_s is never read, and a row with none gives zeros. One
// wave per (row, query head): lane s holds split s's (max, sum) (splits <=
// 64), lane l the output dims l, l + 64, ...
template <typename T, int D>
__global__ void __launch_bounds__(64)
general_merge(const float* __restrict__ part_o, const float* __restrict__ part_ml,
              T* __restrict__ out, const int64_t* __restrict__ rows, int64_t ots, int64_t ohs,
              int heads, int splits, float v_scale) {
    constexpr int DI = (D + 63) / 64;
    const int id = blockIdx.x;
    const int r = id / heads;
    const int h = id - r * heads;
    const int lane = threadIdx.x;
    const int64_t base = (int64_t(r) * heads + h) * splits;
    float m = -INFINITY, l = 0.f;
    if (lane < splits) {
        m = part_ml[2 * (base + lane)];
        l = part_ml[2 * (base + lane) + 1];
    }
    const float mx = wave_max(m);
    T* const o = out + rows[r] * ots + h * ohs;
    float acc[DI];
#pragma unroll
    for (int i = 0; i < DI; ++i) acc[i] = 0.f;
    float inv = 0.f;
    if (mx != -INFINITY) {  // uniform
        const float w = m == -INFINITY ? 0.f : exp2f(m - mx);
        inv = v_scale / wave_sum(w * l);
        for (int s0 = 0; s0 < splits; ++s0) {
            const float ws = __shfl(w, s0, 64);
            if (ws == 0.f) continue;  // uniform: an empty split (or a negligible one)
            const float* const po = part_o + (base + s0) * D;
#pragma unroll
            for (int i = 0; i < DI; ++i) {
                const int d = lane + 64 * i;
                if (d < D) acc[i] = fmaf(ws, po[d], acc[i]);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < DI; ++i) {
        const int d = lane + 64 * i;
        if (d < D) o[d] = static_cast<T>(acc[i] * inv);
    }
}

// The unit of keys that decode splits are planned in: 64 up to head dim 64, 32
// at 128, 16 at 256. Fixed, as callers size workspaces by the plan; the kernel's
// own chunks are of 32 keys at every head dim.
int64_t split_unit(int64_t D) { return D > 64 ? 64 / (D / 64) : 64; }

bool rows_kernel_dim(int64_t D) { return D == 32 || D == 64 || D == 128 || D == 256; }

}  // namespace

GeneralSplits general_decode_splits(int64_t rows, int64_t heads, int64_t kv_heads,
                                    int64_t head_dim, int64_t max_context) {
    GeneralSplits p{1, max_context};
    if (rows <= 0 || kv_heads <= 0 || heads % kv_heads != 0 || max_context <= 0 ||
        !rows_kernel_dim(head_dim))
        return p;
    // Aim for 512 workgroups (two of four waves per CU). A split keeps at
    // least eight units: of the kernel's rounds (a 32-key chunk for each of
    // four waves) four up to head dim 64, two at 128, one at 256, where it may
    // also end inside a chunk. One merge lane per split.
    constexpr int64_t kTarget = 512, kMaxSplits = 64;
    const int64_t units = rows * kv_heads * ((heads / kv_heads + GH - 1) / GH);
    const int64_t unit = split_unit(head_dim);
    const int64_t min_keys = 8 * unit;
    int64_t s = std::min((kTarget + units - 1) / units, kMaxSplits);
    s = std::min(s, (max_context + min_keys - 1) / min_keys);
    if (s <= 1) return p;
    // Exactly s splits (a trailing one may hold no key: it writes an empty
    // partial), so the workspace never shrinks as max_context grows.
    p.splits = s;
    p.keys = ((max_context + s - 1) / s + unit - 1) / unit * unit;
    return p;
}

int64_t general_decode_workspace(int64_t rows, int64_t heads, int64_t kv_heads,
                                 int64_t head_dim, int64_t max_context) {
    const GeneralSplits p = general_decode_splits(rows, heads, kv_heads, head_dim, max_context);
    return p.splits > 1 ? rows * heads * p.splits * (head_dim + 2) * int64_t(sizeof(float)) : 0;
}

int launch_general_attention(const GeneralAttention& g_in, hipStream_t stream) {
    GeneralAttention g = g_in;
    TVLLM_CHECK(g.head_dim > 0 && g.head_dim <= DMAX, "attention: head_dim must be in 1..256");
    TVLLM_CHECK(g.heads > 0 && g.kv_heads > 0 && g.heads % g.kv_heads == 0,
                "attention: query heads must be a multiple of the KV heads");
    if (g.num_items == 0) return TVLLM_OK;
    const int64_t chunks = (g.heads / g.kv_heads + GH - 1) / GH;
    const int64_t gx = g.num_items * g.kv_heads * chunks;
    const int64_t gy = g.rows ? 1 : g.max_query_len;
    TVLLM_CHECK(gx <= INT32_MAX && gy >= 1 && gy <= 65535,
                "attention: launch grid out of range (query chunks of at most 65535 tokens)");
    const bool f8 = g.cache_dtype == TVLLM_FP8_E4M3;
    const bool vec = g.head_dim % 8 == 0 && g.css % 8 == 0 && g.chs % 8 == 0 &&
                     (f8 ? aligned8(g.k) && aligned8(g.v) : aligned16(g.k) && aligned16(g.v));
    const int D = g.head_dim;
    const bool rows_kernel = vec && rows_kernel_dim(D);
    const int group = g.heads / g.kv_heads;
    const int64_t qpw = rows_kernel && group < GH ? GH / group : 1;
    g.q_vec = g.qts % 8 == 0 && g.qhs % 8 == 0 && aligned16(g.q);
    g.out_vec = g.ots % 4 == 0 && g.ohs % 4 == 0 && aligned8(g.out);
    // Prefill (head dim 128 has its own kernel): the tiled kernel above 32 rows
    // per item and KV head (where three of its waves have rows); up to there,
    // four waves share the keys of 16 rows.
    const int64_t item_rows = g.max_query_len * group;
    const int64_t units = g.num_items * g.kv_heads;
    // 128 rows per workgroup where that leaves one for every CU (4 x 512
    // queries over 2048 tokens, 32 / 8 heads of 64: 81 us against 94 with 64
    // rows; where tiles are few they lose, 41 against 38 us for 3 x 300 over
    // 1300, 62 against 34 for 8 x 40 over 2040). Heads of 256 have no registers
    // for a second row tile.
    const bool wide = D <= 64 && units * ((item_rows + 127) / 128) >= 256;
    const int64_t ty = (item_rows + (wide ? 127 : 63)) / (wide ? 128 : 64);
    const bool tiles = rows_kernel && D != 128 && !g.rows && item_rows > 2 * GH && ty <= 65535;
    g.splits = 1;
    g.split_keys = 0;
    g.part_o = g.part_ml = nullptr;
    if (g.rows && rows_kernel) {
        TVLLM_CHECK(g.max_context > 0, "attention: decode needs a positive max_context");
        const GeneralSplits p = general_decode_splits(g.num_items, g.heads, g.kv_heads, D,
                                                      g.max_context);
        if (p.splits > 1) {
            const int64_t need = g.num_items * g.heads * p.splits * (D + 2) * int64_t(sizeof(float));
            TVLLM_CHECK(g.workspace_bytes >= need && g.workspace != nullptr,
                        "paged_decode: workspace of %lld bytes required, %lld given",
                        (long long)need, (long long)g.workspace_bytes);
            TVLLM_CHECK(aligned16(g.workspace), "paged_decode: workspace must be 16-byte aligned");
            g.splits = p.splits;
            g.split_keys = p.keys;
            g.part_o = static_cast<float*>(g.workspace);
            g.part_ml = g.part_o + g.num_items * g.heads * p.splits * D;
        }
    }
    const int64_t gy_rows = g.rows ? g.splits : (g.max_query_len + qpw - 1) / qpw;
    const dim3 grid{static_cast<uint32_t>(gx), static_cast<uint32_t>(rows_kernel ? gy_rows : gy),
                    1u};
    return dispatch_half(g.dtype, [&]<int DT>() {
        using T = typename Elem<DT>::T;
        if (tiles) {
            // Where the tiles do not fill the CUs, two halves of a workgroup
            // share the keys (2 x 256 over 1033, heads of 256: 59 -> 50 us; 8
            // x 40 over 2040, FP8, heads of 64: 42 -> 34 us); at full grids
            // the halves only add their merge (4 x 512 over 2048 in tiles of
            // 64 rows, heads of 64 / 256: 94 -> 109, 303 -> 318 us).
            const bool halves = units * ty < 256;
            const dim3 tg{static_cast<uint32_t>(units), static_cast<uint32_t>(ty), 1u};
            auto go = [&]<int DD, int RT, int HV>() {
                constexpr int threads = 64 * kRowWaves * HV;
                if (f8) tiles_attention_kernel<T, true, DD, RT, HV><<<tg, threads, 0, stream>>>(g);
                else tiles_attention_kernel<T, false, DD, RT, HV><<<tg, threads, 0, stream>>>(g);
            };
            auto rt = [&]<int DD>() {
                if constexpr (DD <= 64) {
                    if (wide) {
                        go.template operator()<DD, 2, 1>();
                        return;
                    }
                }
                if (halves) go.template operator()<DD, 1, 2>();
                else go.template operator()<DD, 1, 1>();
            };
            if (D == 32) rt.template operator()<32>();
            else if (D == 64) rt.template operator()<64>();
            else rt.template operator()<256>();
        } else if (rows_kernel) {
            auto go = [&]<int DD>() {
                constexpr int threads = 64 * kRowWaves;
                if (f8) rows_attention_kernel<T, true, DD><<<grid, threads, 0, stream>>>(g);
                else rows_attention_kernel<T, false, DD><<<grid, threads, 0, stream>>>(g);
            };
            if (D == 32) go.template operator()<32>();
            else if (D == 64) go.template operator()<64>();
            else if (D == 128) go.template operator()<128>();
            else go.template operator()<256>();
            if (g.splits > 1) {
                const int st = launch_status("attention (general head dims)");
                if (st != TVLLM_OK) return st;
                auto merge = [&]<int DD>() {
                    general_merge<T, DD><<<int(g.num_items * g.heads), 64, 0, stream>>>(
                        g.part_o, g.part_ml, static_cast<T*>(g.out), g.rows, g.ots, g.ohs,
                        g.heads, int(g.splits), g.v_scale);
                };
                if (D == 32) merge.template operator()<32>();
                else if (D == 64) merge.template operator()<64>();
                else if (D == 128) merge.template operator()<128>();
                else merge.template operator()<256>();
                return launch_status("attention merge (general head dims)");
            }
        } else if (f8 && vec) general_attention_kernel<T, true, true><<<grid, 64, 0, stream>>>(g);
        else if (f8) general_attention_kernel<T, true, false><<<grid, 64, 0, stream>>>(g);
        else if (vec) general_attention_kernel<T, false, true><<<grid, 64, 0, stream>>>(g);
        else general_attention_kernel<T, false, false><<<grid, 64, 0, stream>>>(g);
        return launch_status("attention (general head dims)");
    });
}

}  // namespace tvllm
