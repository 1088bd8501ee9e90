// Linear layers of few rows (a decode batch) and small weights, on MFMA.
//
// Reference behaviour: F.linear (tinyvllm/layers.py:80-125), and for the MLP's
// packed gate | up projection the SiLU-and-multiply that follows it
// (pointwise.cu:260-321), with that op's rounding points.
//
// These products read each weight once and do next to nothing with it, so they
// are bound by how soon the weights stream in. The library's GEMMs take one
// tile per workgroup over the whole reduction, which at these sizes leaves most
// CUs without work and pays one latency per step of a long chain. Here:
//  * a workgroup owns 16 * NT output columns (weight rows); its waves split
//    the reduction (and the grid's y, where the caller takes partial sums), so
//    even 1024 columns make 256 workgroups' worth of loads in flight;
//  * operands go straight from memory to MFMA registers: A = 16 weight rows x
//    32, B = the input rows (padded to 16 * MT by repeating the last), D[column]
//    [row], U steps of both loaded ahead of the MFMAs of the U before;
//  * weights are read non-temporally (once); the input stays in the caches;
//  * the waves' sums meet in LDS, each wave finishing its share of the tiles:
//    rounded to the storage type, kept as fp32 partial sums (the consumer adds
//    the slices up), or gate and up rounded, activated and multiplied.
//
// Measured in graph replay over cold weights, us, library -> here (1 / 16 / 64
// rows), bf16:
//   1024 -> 4096  7.5 / 7.6 / 11.6 -> 4.2 / 4.6 / 7.4 (the library's four-slice
//       batched product 7.3 at 64 rows, and its sum in the decode kernel 2.5)
//   1024 -> 6144 with SiLU  10.5 / 10.9 / 14.7 -> 5.7 / 6.3 / 8.9
//   2048 -> 1024 partials   4.6 / 6.0 / 5.9 -> 3.2 / 3.5 / 5.0
//   3072 -> 1024 partials   5.5 / 8.0 / 7.9 -> 3.8 / 4.1 / 6.0
//   8192 -> 5120 partials   47.6 / 47.6 / 44.5 -> 20.1 / 23.4 / not taken
//   25600 -> 5120 partials  79.3 / 81.5 / 76.0 -> 60.8 / 71.3 / not taken
//   4096 -> 24576 with SiLU  47.2 / 46.1 / 50.9 -> 37.2 / 44.4 / 69
// The last line shows the limit: every workgroup reads the whole input, which
// past about 16 rows costs large weights more than it saves. The rules of
// which calls come here stand in layers.py.
#include "common.h"

#include <type_traits>

namespace tvllm {
namespace {

typedef f32x4_t lf32x4;

__device__ __forceinline__ U16x8 load_once(const U16x8* p) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const u32x4 t = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
    return U16x8{{t[0], t[1], t[2], t[3]}};
}

enum Epilogue { kRounded, kPartials, kSilu };

// Grid: x = groups of 16 * NT columns (kSilu: 8 * NT gate columns and the up
// columns beside them, tiles alternating), y = slices of the reduction
// (kPartials only), each cut further over the NW waves.
template <typename T, int MT, int NT, int U, int NW, Epilogue EP>
__global__ void __launch_bounds__(64 * NW)
few_rows_linear(const T* __restrict__ x, int64_t x_stride, const T* __restrict__ w, int rows,
                int n, int k, void* __restrict__ out) {
    static_assert(EP != kSilu || NT % 2 == 0, "gate and up tiles come in pairs");
    constexpr int R = MT * NT;
    __shared__ lf32x4 sums[NW][R][64];
    const int wave = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    const int col = lane & 15, quad = lane >> 4;

    const int64_t steps = k / 32, slices = int64_t(NW) * gridDim.y;
    const int64_t slice = int64_t(blockIdx.y) * NW + wave;
    const int s0 = int(steps * slice / slices);
    const int mine = int(steps * (slice + 1) / slices) - s0;
    const U16x8* wp[NT];
    const U16x8* xp[MT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int64_t row = EP == kSilu
            ? int64_t(j % 2) * (n / 2) + int64_t(blockIdx.x) * (8 * NT) + 16 * (j / 2) + col
            : int64_t(blockIdx.x) * (16 * NT) + 16 * j + col;
        wp[j] = reinterpret_cast<const U16x8*>(w + row * k + s0 * 32 + 8 * quad);
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
        xp[i] = reinterpret_cast<const U16x8*>(x + min(16 * i + col, rows - 1) * x_stride +
                                               s0 * 32 + 8 * quad);
    lf32x4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = lf32x4{0.f, 0.f, 0.f, 0.f};

    U16x8 wr[U][NT], xr[U][MT];
    auto load = [&](int s) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < MT; ++i) xr[u][i] = xp[i][4 * (s + u)];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int j = 0; j < NT; ++j) wr[u][j] = load_once(wp[j] + 4 * (s + u));
    };
    int s = 0;
    if (mine >= U) {
        load(0);
        // A possible write between a load and the end of its block keeps the
        // compiler from carrying the address into the loop instead of the value.
        asm volatile("" ::: "memory");
        for (; s + U <= mine; s += U) {
            U16x8 wc[U][NT], xc[U][MT];
#pragma unroll
            for (int u = 0; u < U; ++u) {
#pragma unroll
                for (int j = 0; j < NT; ++j) wc[u][j] = wr[u][j];
#pragma unroll
                for (int i = 0; i < MT; ++i) xc[u][i] = xr[u][i];
            }
            if (s + 2 * U <= mine) load(s + U);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);  // the loads go out first
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int j = 0; j < NT; ++j)
#pragma unroll
                    for (int i = 0; i < MT; ++i)
                        acc[i][j] = mfma32<T>(wc[u][j], xc[u][i], acc[i][j]);
        }
    }
    for (; s < mine; ++s)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const U16x8 a = load_once(wp[j] + 4 * s);
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[i][j] = mfma32<T>(a, xp[i][4 * s], acc[i][j]);
        }

#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) sums[wave][i * NT + j][lane] = acc[i][j];
    __syncthreads();
    // Lane (col, quad) finishes columns 4 * quad .. + 3 of a tile for row col.
    constexpr int NO = EP == kSilu ? NT / 2 : NT;  // output tiles per row tile
    for (int t = wave; t < MT * NO; t += NW) {
        const int i = t / NO, j = t % NO, row = 16 * i + col;
        const int a0 = i * NT + (EP == kSilu ? 2 * j : j);
        lf32x4 a = sums[0][a0][lane];
#pragma unroll
        for (int v = 1; v < NW; ++v) a += sums[v][a0][lane];
        if constexpr (EP == kSilu) {
            lf32x4 b = sums[0][a0 + 1][lane];
#pragma unroll
            for (int v = 1; v < NW; ++v) b += sums[v][a0 + 1][lane];
            float y[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float g = rnd<T>(a[e]);
                y[e] = rnd<T>(g / (1.0f + expf(-g))) * rnd<T>(b[e]);
            }
            if (row < rows)
                *reinterpret_cast<uint2*>(static_cast<T*>(out) + int64_t(row) * (n / 2) +
                                          int64_t(blockIdx.x) * (8 * NT) + 16 * j + 4 * quad) =
                    make_uint2(pack2<T>(y[0], y[1]), pack2<T>(y[2], y[3]));
        } else {
            const int64_t at = int64_t(row) * n + int64_t(blockIdx.x) * (16 * NT) + 16 * j +
                               4 * quad;
            if (row < rows) {
                if constexpr (EP == kPartials)
                    *reinterpret_cast<lf32x4*>(static_cast<float*>(out) +
                                               int64_t(blockIdx.y) * rows * n + at) = a;
                else
                    *reinterpret_cast<uint2*>(static_cast<T*>(out) + at) =
                        make_uint2(pack2<T>(a[0], a[1]), pack2<T>(a[2], a[3]));
            }
        }
    }
}

}  // namespace
}  // namespace tvllm

using namespace tvllm;

extern "C" int tvllm_few_rows_linear(const void* x, int64_t x_row_stride, const void* weight,
                                     int64_t rows, int64_t columns, int64_t width, void* out,
                                     int64_t slices, int silu, int dtype,
                                     tvllm_stream_t stream) {
    TVLLM_CHECK(rows >= 0 && rows <= 64, "few_rows_linear: at most 64 rows");
    TVLLM_CHECK(width > 0 && width % 32 == 0 && width <= INT32_MAX,
                "few_rows_linear: the input width must be a multiple of 32");
    TVLLM_CHECK(columns > 0 && columns % 32 == 0 && columns <= INT32_MAX,
                "few_rows_linear: the output width must be a multiple of 32");
    TVLLM_CHECK(slices >= 0 && slices <= 64 && (slices == 0 || !silu),
                "few_rows_linear: 0 to 64 partial slices, none with SiLU");
    TVLLM_CHECK(x_row_stride % 8 == 0, "few_rows_linear: input rows in 16-byte units");
    if (rows == 0) return TVLLM_OK;
    TVLLM_CHECK(x && weight && out, "few_rows_linear: null pointer");
    TVLLM_CHECK(aligned16(x) && aligned16(weight) && aligned16(out),
                "few_rows_linear: 16-byte aligned tensors");
    hipStream_t s = as_hip(stream);
    const int m = int(rows), n = int(columns), k = int(width);
    return dispatch_half(dtype, [&]<int DT>() {
        using T = typename Elem<DT>::T;
        const T* const xt = static_cast<const T*>(x);
        const T* const wt = static_cast<const T*>(weight);
        auto go = [&]<int MT, int NT, int U, int NW, Epilogue EP>() {
            const dim3 grid{uint32_t(n / (16 * NT)), uint32_t(EP == kPartials ? slices : 1), 1u};
            few_rows_linear<T, MT, NT, U, NW, EP><<<grid, 64 * NW, 0, s>>>(xt, x_row_stride, wt, m,
                                                                           n, k, out);
            return launch_status("few_rows_linear");
        };
        // Tile shapes by measurement (the head of this file's sizes): 16
        // columns per workgroup for rounded results, so that 4096 make 256
        // workgroups; 32 with partial sums, whose slices fill the grid, and
        // with SiLU (a gate and an up tile). More steps ahead where fewer
        // input tiles leave the registers for them.
        if (silu) {
            if (m <= 16) return go.template operator()<1, 2, 4, 8, kSilu>();
            if (m <= 32) return go.template operator()<2, 2, 4, 4, kSilu>();
            return go.template operator()<4, 2, 2, 4, kSilu>();
        }
        if (slices > 0 && n > 2048) {  // enough columns for four waves a workgroup
            if (m <= 16) return go.template operator()<1, 2, 2, 4, kPartials>();
            if (m <= 32) return go.template operator()<2, 2, 2, 4, kPartials>();
        }
        if (slices > 0) {
            if (m <= 16) return go.template operator()<1, 2, 2, 8, kPartials>();
            if (m <= 32) return go.template operator()<2, 2, 2, 8, kPartials>();
            return go.template operator()<4, 2, 2, 8, kPartials>();
        }
        if (m <= 16) return go.template operator()<1, 1, 4, 4, kRounded>();
        if (m <= 32) return go.template operator()<2, 1, 4, 4, kRounded>();
        return go.template operator()<4, 1, 2, 4, kRounded>();
    });
}
