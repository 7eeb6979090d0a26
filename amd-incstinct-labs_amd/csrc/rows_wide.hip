// RMSNorm, two-pass LayerNorm and row softmax for the rows the wave-per-row kernels of norms.hip do
// not suit (gfx950): rows of more than 4,096 columns, rows whose start is not 16-byte aligned (any
// width that is no multiple of 4), and calls of few rows, where one wave per row leaves the chip
// idle.
//
// Reference behaviour restated: forward.hpp:34-56 (rmsnorm_f32_kernel), bench_layernorm.hip:51-114,
// bench_softmax.hip:59-105, the same arithmetic per element as norms.hip.
//
// What bounds these is the stream of X and Y through HBM, or, for few rows, the latency of one row.
// Measured (us, inputs rotating through memory; before: norms.hip's element-wise kernels): softmax
// 512 x 32000 503 -> 30.5 (4.3 TB/s), 4096 x 8192 156 -> 43.6 (6.2 TB/s), 1 x 32000 162 -> 5.4;
// LayerNorm 1024 x 12345 204 -> 27.5, 4096 x 3001 59.4 -> 23.8.
// The row is held in registers between the passes, as 16-byte vectors (NV per lane) over TPR
// threads: one wave for narrow rows (four rows per workgroup), a workgroup of 256 or 1,024 threads
// for wide ones. The wave totals of a workgroup row meet in one LDS line per pass (a write per wave,
// one read each, a barrier), everything else is the wave butterfly.
// Vectors need no alignment beyond the element's 4 bytes (global_load_dwordx4 takes dword-aligned
// addresses), and the last vector of a row whose width is no multiple of 4 is moved back to end at
// the row's end: its first `skip` elements then repeat its neighbour's, take no part in the row's
// sums, and are stored twice with the same value.
#include "common.hpp"
#include "rows_wide.hpp"
#include "wave_primitives/detail/xlane.hpp"

namespace cdna4 {
namespace {

using wave::xlane::allreduce;
using wave::xlane::Max;
using wave::xlane::row_allreduce;
using wave::xlane::Sum;

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef f32x4 f32x4_u __attribute__((aligned(4)));
typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
typedef u16x4 u16x4_u __attribute__((aligned(2)));

template <bool kNT>
__device__ __forceinline__ f32x4 ld4(const float* p) {
    if constexpr (kNT) return __builtin_nontemporal_load((const f32x4_u*)p);
    else return *(const f32x4_u*)p;
}
template <bool kNT>
__device__ __forceinline__ void st4(float* p, f32x4 v) {
    if constexpr (kNT) __builtin_nontemporal_store(v, (f32x4_u*)p);
    else *(f32x4_u*)p = v;
}

// Combined value over the TPR threads of a row, on every one of them. `slot` is an LDS line of its
// own per use, so one barrier (between its writes and its reads) is enough.
template <int TPR, class Op>
__device__ __forceinline__ float row_combine(float v, Op op, float* slot) {
    v = allreduce(v, op);
    if constexpr (TPR > 64) {
        const int wave = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63;
        if (lane == 0) slot[wave] = v;
        __syncthreads();
        if constexpr (TPR == 1024) {
            v = row_allreduce(slot[lane & 15], op);
        } else {
            static_assert(TPR == 256, "four or sixteen waves per row");
            const f32x4 w = *(const f32x4*)slot;
            v = op(op(w[0], w[1]), op(w[2], w[3]));
        }
    }
    return v;
}

// A vector's own elements (those from sk on; 0 in the place of the others) less `mean`.
__device__ __forceinline__ f32x4 own(f32x4 v, int sk, float mean = 0.f) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = e >= sk ? v[e] - mean : 0.f;
    return v;
}
// A vector added to a thread's sum. Rows of one wave add its elements in pairs, as the wave-per-row
// kernels do, whose results unaligned rows then give bit for bit: in sequence they were further from 64
// bits than the element-wise kernels (softmax of 2,047 columns 6.5e-8 relative, in pairs 5.6e-8,
// element-wise 6.1e-8; a little above 64 or 128 columns 2-6 % over those remain, 67: 6.4e-8 -> 6.7e-8: the
// last vector is alone in its 16 lanes, one more addition at the row's full size). Rows of a workgroup
// have short sums per thread and add in sequence (32,000 columns: 4.9e-8, in pairs 5.0e-8, element-wise
// 6.4e-8).
template <int TPR>
__device__ __forceinline__ void add4(float& s, f32x4 v, int sk) {
    if constexpr (TPR == 64) {
        v = own(v, sk);
        s += (v[0] + v[1]) + (v[2] + v[3]);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) s += e >= sk ? v[e] : 0.f;
    }
}
template <int TPR>
__device__ __forceinline__ void add4_squares(float& s, f32x4 v, int sk, float mean) {
    if constexpr (TPR == 64) {
        v = own(v, sk, mean);
        s += (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float d = v[e] - mean;
            s += e >= sk ? d * d : 0.f;
        }
    }
}

constexpr int kBlock = 256;

// One row per TPR threads: workgroups of 256 threads (TPR 64: four rows each; 256: one), or of 1,024.
// kOp: kRowsRms (W fp16 gain), kRowsLayer (G, B fp32), kRowsSoftmax (X may equal Y: every load of a
// row is used in its sums, before the barrier or in the same wave, ahead of its first store).
template <int kOp, int TPR, int NV, bool kNT>
__global__ __launch_bounds__(TPR > kBlock ? TPR : kBlock) void rows_kernel(const float* X, const void* G, const float* B,
                                                                          float* Y, int M, int H, float eps) {
    constexpr int kRows = TPR < kBlock ? kBlock / TPR : 1;
    __shared__ __attribute__((aligned(16))) float slots[2][16];
    const int t = (int)threadIdx.x % TPR;
    const int row = (int)blockIdx.x * kRows + (int)threadIdx.x / TPR;
    if (row >= M) return;   // TPR 64 only: whole waves, which meet no barrier
    const float* x = X + (size_t)row * H;
    float* y = Y + (size_t)row * H;
    // Vector k of thread t covers columns c .. c + 3, c = 4 (t + k TPR); past the row's last whole
    // vector it is read at H - 4 and its first c - (H - 4) elements (all four past the end) are not
    // its own.
    f32x4 v[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = ld4<kNT>(x + min((t + k * TPR) * 4, H - 4));
    auto skip = [&](int k) { return (t + k * TPR) * 4 - min((t + k * TPR) * 4, H - 4); };

    if constexpr (kOp == kRowsSoftmax) {
        float m = -INFINITY;   // the repeated elements do not change a maximum
#pragma unroll
        for (int k = 0; k < NV; ++k) m = fmaxf(fmaxf(m, fmaxf(v[k][0], v[k][1])), fmaxf(v[k][2], v[k][3]));
        m = row_combine<TPR>(m, Max{}, slots[0]);
        float s = 0.f;
#pragma unroll
        for (int k = 0; k < NV; ++k) {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[k][e] = __expf(v[k][e] - m);
            add4<TPR>(s, v[k], skip(k));
        }
        const float inv = 1.f / row_combine<TPR>(s, Sum{}, slots[1]);
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const int c = (t + k * TPR) * 4;
            if (c < H) st4<kNT>(y + min(c, H - 4), v[k] * inv);
        }
    } else {
        float mean = 0.f;
        if constexpr (kOp == kRowsLayer) {
            float s = 0.f;
#pragma unroll
            for (int k = 0; k < NV; ++k) add4<TPR>(s, v[k], skip(k));
            mean = row_combine<TPR>(s, Sum{}, slots[0]) / (float)H;
        }
        float q = 0.f;
#pragma unroll
        for (int k = 0; k < NV; ++k) add4_squares<TPR>(q, v[k], skip(k), mean);
        const float inv = rsqrtf(row_combine<TPR>(q, Sum{}, slots[1]) / (float)H + eps);
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const int c = (t + k * TPR) * 4;
            if (c >= H) continue;
            const int cl = min(c, H - 4);
            f32x4 o;
            if constexpr (kOp == kRowsLayer) {
                const f32x4 g = *(const f32x4_u*)((const float*)G + cl), b = *(const f32x4_u*)(B + cl);
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = (v[k][e] - mean) * inv * g[e] + b[e];
            } else {
                const u16x4 g = *(const u16x4_u*)((const uint16_t*)G + cl);
#pragma unroll
                for (int e = 0; e < 4; ++e) o[e] = v[k][e] * inv * f16_bits_to_f32(g[e]);
            }
            st4<kNT>(y + cl, o);
        }
    }
}

template <int kOp, int TPR, int NV>
int launch_rows(const float* X, const void* G, const float* B, float* Y, int M, int H, float eps, bool nt,
                hipStream_t s) {
    const unsigned grid = TPR < kBlock ? ceil_div((size_t)M, kBlock / TPR) : (unsigned)M;
    const unsigned block = TPR > kBlock ? TPR : kBlock;
    if (nt) rows_kernel<kOp, TPR, NV, true><<<grid, block, 0, s>>>(X, G, B, Y, M, H, eps);
    else rows_kernel<kOp, TPR, NV, false><<<grid, block, 0, s>>>(X, G, B, Y, M, H, eps);
    return launch_status();
}

template <int kOp>
int launch_op(const float* X, const void* G, const float* B, float* Y, int M, int H, float eps, bool nt,
              hipStream_t s) {
#define CDNA4_ROWS(TPR, NV) \
    if (H <= 4 * TPR * NV) return launch_rows<kOp, TPR, NV>(X, G, B, Y, M, H, eps, nt, s);
    if (!rows_few(M, H)) {   // a wave per row up to 2,048 columns (32 VGPRs of row)
        CDNA4_ROWS(64, 1) CDNA4_ROWS(64, 2) CDNA4_ROWS(64, 4) CDNA4_ROWS(64, 8)
    }
    CDNA4_ROWS(256, 1) CDNA4_ROWS(256, 2) CDNA4_ROWS(256, 4) CDNA4_ROWS(256, 8)
    CDNA4_ROWS(1024, 4) CDNA4_ROWS(1024, 8) CDNA4_ROWS(1024, 16)
#undef CDNA4_ROWS
    return CDNA4_ERR_INVALID_VALUE;   // wider than kRowsWideMax: the caller's rule does not come here
}

}  // namespace

int rows_wide(int op, const float* X, const void* G, const float* B, float* Y, int M, int H, float eps, bool nt,
              hipStream_t s) {
    switch (op) {
        case kRowsRms: return launch_op<kRowsRms>(X, G, B, Y, M, H, eps, nt, s);
        case kRowsLayer: return launch_op<kRowsLayer>(X, G, B, Y, M, H, eps, nt, s);
        default: return launch_op<kRowsSoftmax>(X, G, B, Y, M, H, eps, nt, s);
    }
}

}  // namespace cdna4
