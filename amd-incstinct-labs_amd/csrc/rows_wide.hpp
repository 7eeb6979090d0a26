// Row norms and softmax of wide, unaligned or few rows (rows_wide.hip), and the rule that sends a
// call there (norms.hip keeps the wave-per-row kernels for everything else).
#pragma once
#include <stdint.h>

typedef struct ihipStream_t* hipStream_t;   // as in HIP's own headers: the rules below are plain C++

namespace cdna4 {

enum { kRowsRms = 0, kRowsLayer = 1, kRowsSoftmax = 2 };

constexpr int kRowsWideMin = 4;       // one whole vector
constexpr int kRowsWideMax = 65536;   // 1,024 threads x 16 vectors

// Few rows, each wide enough for a workgroup: with one wave per row such a call leaves CUs idle or
// waits on one wave's loads. Wave / workgroup per row, LayerNorm, us: 16 x 768 2.71 / 2.41,
// 256 x 1024 3.14 / 2.52, 1024 x 1024 4.05 / 3.84, 1024 x 4096 11.3 / 8.6; beyond the line the wave
// is level or ahead (1024 x 768 3.65 / 3.51 but softmax 3.40 / 3.49, 4096 x 2048 13.4 / 14.7).
inline bool rows_few(int M, int H) { return H >= 768 && M <= (H >= 1024 ? 1024 : 512); }

// Threads per row of a call of many rows (rows_wide.hip, launch_op), and whether its grid stays below
// the 2^32 threads that one launch can have: past that (16.8 million rows of more than 2,048 columns,
// 4.2 million of more than 8,192) the element-wise kernels take the call, with 64 threads per row.
inline int rows_threads(int H) { return H <= 2048 ? 64 : H <= 8192 ? 256 : 1024; }
inline bool rows_fit(int M, int H) { return (uint64_t)M * (uint64_t)rows_threads(H) < (1ull << 32); }

// Whether a call goes to rows_wide. vec is norms.hip's own rule (16-byte aligned rows, H % 4 == 0,
// H <= 4,096): a call outside it otherwise runs element by element, one wave per row (softmax
// 512 x 32000 503 us, here 30.5; LayerNorm 4096 x 3001 59.4 / 23.8, 16384 x 101 7.6 / 5.7).
inline bool rows_wide_takes(int M, int H, bool vec) {
    return H >= kRowsWideMin && H <= kRowsWideMax && (vec ? rows_few(M, H) : rows_fit(M, H));
}

// G: the gain (fp16 for kRowsRms, fp32 for kRowsLayer), B: fp32 beta (kRowsLayer). nt: non-temporal
// loads and stores of X and Y. 4 <= H <= 65,536; X, Y, G and B aligned to their elements.
int rows_wide(int op, const float* X, const void* G, const float* B, float* Y, int M, int H, float eps, bool nt,
              hipStream_t s);

}  // namespace cdna4
