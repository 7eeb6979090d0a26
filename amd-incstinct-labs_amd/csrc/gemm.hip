// Prompt-path GEMM of the small-LLM runtime (gfx950): Y[M][N] (+)= X[M][K] W[N][K]^T with fp16
// X and W (both row-major, K contiguous), fp32 accumulation, fp32 or fp16 Y.
//
// Reference behaviour restated: the reference runs these products through rocBLAS gemm_ex
// (cdna3-prims/include/cdna3/runtime/rocblas_gemm.hpp:8-20; forward.hpp:70-131), Y = X W^T with W
// the [out][in] weight as the model files hold it, beta 0 (Q|K|V, gate|up) or 1 (the O and down
// projections added into the fp32 residual).
//
// MI355X design: at prompt lengths of a few hundred tokens these GEMMs are small (0.6-4.8 GFLOP,
// 2-10 MB of operands) and a launch is over in a few microseconds, so what sets the time is how
// many workgroups the grid gives each CU and how many bytes each CU keeps in flight. The tile
// (BM x BN, from a small menu) is chosen per shape so that the grid is about one round of one
// workgroup per CU, and each workgroup streams 64-wide K stages of both operand tiles HBM -> LDS
// with asynchronous copies (global_load_lds_dwordx4) into a ring of S stages, S - 1 ahead of the
// stage being multiplied (S as deep as 128 KB of LDS allows, up to 8). Four waves compute Y^T =
// W X^T on v_mfma_f32_16x16x32_f16: W rows are the A operand, X rows the B operand.
//
// LDS layout (the prefill's K tile at D = 64, whose reads were measured free of bank conflicts):
// a stage holds BN rows of W then BM rows of X, 128 bytes per row; 16-byte chunk c of row r sits
// at position c ^ swz_k<64>(r % 32). An operand block (16 rows) of 32-row group G is read in the
// permuted row order 32 G + 8 (l / 4) + l % 4 + 4 u (A-row / B-column l, u = 0 or 1): the lanes
// of one read then touch every bank once, and a lane's four accumulator values are four
// consecutive output columns n (one 16-byte or 8-byte store). Wave (wm, wn) takes block u = wn of
// every W group and u = wm of every X group of the tile. Rows past M or N read the last valid row
// (their results are not stored). Large products take 256-row tiles of eight waves (gemm_big, below).
#include "attn_stream.hpp"

namespace cdna4 {
namespace {

typedef _Float16 gf16x8 __attribute__((ext_vector_type(8)));
typedef float gf32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 gf16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kBK = 64;        // K per stage (one 128-byte LDS row per operand row)
constexpr int kKMul = kBK;     // K must be a multiple of this
constexpr int kRowBytes = kBK * 2;
constexpr int kLdsBudget = 128 * 1024;

// Ring depth for a BM x BN tile: as many stages as the LDS budget holds, at most 8.
constexpr int ring_stages(int bm, int bn, int budget = kLdsBudget) {
    const int s = budget / ((bm + bn) * kRowBytes);
    return s > 8 ? 8 : s;
}

// Wait until at most `younger` stages' copies (kPerStage each per wave) are still in flight.
template <int kPerStage, int S>
__device__ __forceinline__ void wait_stages(int younger) {
    static_assert(S >= 2 && S <= 12 && (S - 2) * kPerStage <= 63, "ring depth within the vmcnt range");
#define CDNA4_GEMM_WAIT(y) \
    case y: asm volatile("s_waitcnt vmcnt(%0)" : : "n"((y) * kPerStage) : "memory"); break;
    switch (younger) {
        CDNA4_GEMM_WAIT(0) CDNA4_GEMM_WAIT(1) CDNA4_GEMM_WAIT(2) CDNA4_GEMM_WAIT(3)
        CDNA4_GEMM_WAIT(4) CDNA4_GEMM_WAIT(5) CDNA4_GEMM_WAIT(6) CDNA4_GEMM_WAIT(7)
        CDNA4_GEMM_WAIT(8) CDNA4_GEMM_WAIT(9) CDNA4_GEMM_WAIT(10)
        default: asm volatile("s_waitcnt vmcnt(0)" : : : "memory"); break;
    }
#undef CDNA4_GEMM_WAIT
}

// Tile of workgroup b in a grid of tm x tn tiles (1-D). Workgroups go to the 8 XCDs round-robin
// (XCD = b % 8); when tn is a multiple of 8, XCD x takes the n tiles x tn/8 .. (x+1) tn/8 - 1 with
// every m tile (m fastest), so each W row is fetched into one XCD's L2 only and re-read there by
// that XCD's tiles, and X (the smaller operand at prompt lengths) is what each XCD fetches whole.
__device__ __forceinline__ void tile_of(int b, int tm, int tn, int& mt, int& nt) {
    if ((tn & 7) == 0) {
        const int x = b & 7, s = b >> 3;
        mt = s % tm;
        nt = x * (tn >> 3) + s / tm;
    } else {
        mt = b % tm;
        nt = b / tm;
    }
}

// Output forms: fp16 or fp32 Y (Y = X W^T, + Y with kAccum), or the SiLU-gated product of the
// SwiGLU MLP (kSilu): W holds 2F rows, gate rows 0 .. F - 1 then up rows F .. 2F - 1, and Y [M][F]
// fp16 = fp16(silu(X Wg^T) * (X Wu^T)) in fp32, the rounding the separate silu_mul kernel applies
// to the fp32 product. A kSilu tile of BN rows takes BN / 2 gate rows and the BN / 2 up rows of the
// same output columns, so a lane holds both values of its columns.
enum { kOutF16 = 0, kOutF32 = 1, kOutSilu = 2, kOutQKV = 3 };

// LDS budget of a tile's ring. The Q|K|V epilogue's 64 x 64 tiles take 64 KiB (four stages), so
// two workgroups share a CU: at config 5 (512 x 2304 x 768) that ran the projection + append in a
// time to first token of 0.770 ms against 0.804 with eight stages and one workgroup per CU, and
// 0.788 with the 64 x 128 tile.
// 64 x 32 tiles (the runtime's residual projections, llm_gemm_f16 with cold operands) likewise
// take 64 KiB (five stages), two workgroups per CU.
constexpr int ring_budget(int kOut, int bm, int bn) {
    return (kOut == kOutQKV && bm + bn <= 128) || (bm == 64 && bn == 32) ? 64 * 1024 : kLdsBudget;
}

// kOutQKV: the prompt's Q|K|V projection (columns [0, QD) query heads, [QD, QD + KVD) key heads,
// the rest value heads, D columns each) with the runtime's RoPE + append in the epilogue: each
// value is rounded to fp16 as the projection's output, the (d, d + D/2) pairs of query and key
// heads rotated with the cos/sin rows of positions pos0 + m (rope_pair, as the separate append
// kernel does), queries written head-major to q_out [QD / D][T][D] and keys and values into the
// caches [heads][max_seq][D] at row pos0 + m. Tiles are whole heads (BN % D == 0), so a lane holds
// both columns of its pairs: block i and block i + D / 64 (32 columns per block).

template <int BM, int BN, int kOut, bool kAccum>
__global__ __launch_bounds__(256) void gemm_ring(const uint16_t* __restrict__ X, const uint16_t* __restrict__ W,
                                                 void* __restrict__ Y, int M, int N, int K, int ldy, QkvOut qe) {
    static_assert(BM % 32 == 0 && BN % 32 == 0, "tiles are whole 32-row groups");
    static_assert(kOut != kOutSilu || (BN % 64 == 0 && !kAccum), "a SiLU tile pairs whole gate and up groups");
    constexpr bool kSilu = kOut == kOutSilu;
    constexpr int kTileCols = kSilu ? BN / 2 : BN;   // output columns per tile
    const int ncols = kSilu ? N / 2 : N;              // output columns (F for kSilu)
    constexpr int S = ring_stages(BM, BN, ring_budget(kOut, BM, BN));
    constexpr int FM = BM / 32, FN = BN / 32;        // 16-row blocks per wave: X (m), W (n)
    constexpr int kStage = (BN + BM) * kRowBytes;    // bytes per ring stage
    constexpr int kCopies = (BN + BM) / 8;           // 1 KB copy instructions per stage
    constexpr int kCopiesW = kCopies / 4;            // per wave
    static_assert(kCopies % 4 == 0, "copies split evenly over the four waves");
    __shared__ __attribute__((aligned(16))) char lds[S * kStage];

    const int lane = (int)(threadIdx.x & 63u);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int li = lane & 15, g = lane >> 4;
    const int wm = wave & 1, wn = wave >> 1;
    int mt, nt;
    tile_of((int)blockIdx.x, (M + BM - 1) / BM, (ncols + kTileCols - 1) / kTileCols, mt, nt);
    const int m0 = mt * BM, n0 = nt * kTileCols;

    // Copy j of this wave is instruction c = wave + 4 j of a stage: its lane l fills LDS row
    // 8 c + l / 8 at chunk position l % 8 (1 KB of the stage at byte 1024 c) from global chunk
    // (l % 8) ^ swz(row) of W row n0 + row (rows below BN) or X row m0 + row - BN; whether the
    // instruction copies W or X is uniform over the wave.
    uint32_t coff[kCopiesW];
    bool cw[kCopiesW];
#pragma unroll
    for (int j = 0; j < kCopiesW; ++j) {
        const int c = wave + 4 * j;
        const int row = c * 8 + (lane >> 3);
        const int chunk = (lane & 7) ^ tile::swz_k<64>(row & 31);
        cw[j] = c * 8 < BN;
        int r;
        if (!cw[j]) r = min(m0 + row - BN, M - 1);
        else if (kSilu) r = row < BN / 2 ? min(n0 + row, ncols - 1) : ncols + min(n0 + row - BN / 2, ncols - 1);
        else r = min(n0 + row, N - 1);
        coff[j] = (uint32_t)r * (uint32_t)K * 2u + (uint32_t)chunk * 16u;
    }
    auto issue = [&](int kt, int buf) {   // the copies of stage kt (k0 = 64 kt) into ring slot buf
        const uint16_t* wk = W + (size_t)kt * kBK;
        const uint16_t* xk = X + (size_t)kt * kBK;
#pragma unroll
        for (int j = 0; j < kCopiesW; ++j)
            stream::dma16_s(cw[j] ? wk : xk, coff[j], lds + buf * kStage + (wave + 4 * j) * 1024);
    };

    // Operand reads: W block i (group i, u = wn), X block j (group j, u = wm); K step kc of a stage
    // flips bit 6 (chunk c -> c + 4).
    const int r0 = 8 * (li >> 2) + (li & 3);
    const uint32_t rd = (uint32_t)(r0 * kRowBytes + ((g ^ tile::swz_k<64>(r0)) * 16));
    const uint32_t rw = rd + (uint32_t)wn * 512u;
    const uint32_t rx = (uint32_t)BN * kRowBytes + rd + (uint32_t)wm * 512u;

    gf32x4 acc[FN][FM];
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) acc[i][j] = gf32x4{0.f, 0.f, 0.f, 0.f};

    const int nk = K / kBK;
#pragma unroll
    for (int st = 0; st < S - 1; ++st)
        if (st < nk) issue(st, st);
    for (int kt = 0; kt < nk; ++kt) {
        // stage kt landed (this wave's copies; the barrier: every wave's), and every wave is past
        // stage kt - 1, whose slot now receives stage kt + S - 1
        wait_stages<kCopiesW, S>(min(S - 2, nk - 1 - kt));
        __syncthreads();
        if (kt + S - 1 < nk) issue(kt + S - 1, (kt + S - 1) % S);
        const char* st = lds + (kt % S) * kStage;
#pragma unroll
        for (int kc = 0; kc < 2; ++kc) {
            const uint32_t flip = (uint32_t)kc * 64u;
            u32x4 a[FN], b[FM];
#pragma unroll
            for (int i = 0; i < FN; ++i) a[i] = *(const u32x4*)(st + ((rw + (uint32_t)i * 4096u) ^ flip));
#pragma unroll
            for (int j = 0; j < FM; ++j) b[j] = *(const u32x4*)(st + ((rx + (uint32_t)j * 4096u) ^ flip));
#pragma unroll
            for (int i = 0; i < FN; ++i)
#pragma unroll
                for (int j = 0; j < FM; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(gf16x8, a[i]),
                                                                       __builtin_bit_cast(gf16x8, b[j]), acc[i][j], 0,
                                                                       0, 0);
        }
    }

    // acc[i][j] lane (li, g): Y[m][n .. n + 3], m = m0 + 32 j + r0 + 4 wm, n = n0 + 32 i + 8 g + 4 wn
    // (kSilu: gate group i < FN / 2 and up group i + FN / 2 hold the same columns n).
    if constexpr (kOut == kOutQKV) {
        const int hb = qe.D / 64;   // blocks per half head
#pragma unroll
        for (int j = 0; j < FM; ++j) {
            const int m = m0 + 32 * j + r0 + 4 * wm;
            if (m >= M) continue;
            const float* cr = qe.cosv + (size_t)(qe.pos0 + m) * qe.D;
            const float* sr = qe.sinv + (size_t)(qe.pos0 + m) * qe.D;
#pragma unroll
            for (int i = 0; i < FN; ++i) {
                if ((i / hb) % 2) continue;   // block i in the second half of its head: done with its partner
                const int n = n0 + 32 * i + 8 * g + 4 * wn;   // a first-half column; n + D / 2 its partner
                if (n >= ncols) continue;
                const int d = n % qe.D, half = qe.D / 2;
                const gf32x4 va = acc[i][j], vb = acc[(i + hb) % FN][j];
                uint32_t lo[4], hi[4];
                uint16_t* dst;
                if (n < qe.QD + qe.KVD) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        rope_pair(f32_to_f16_bits(va[e]), f32_to_f16_bits(vb[e]), cr[d + e], sr[d + e],
                                  cr[d + e + half], sr[d + e + half], lo[e], hi[e]);
                    dst = n < qe.QD ? qe.q_out + ((size_t)(n / qe.D) * qe.T + m) * qe.D
                                    : qe.Kc + ((size_t)((n - qe.QD) / qe.D) * qe.max_seq + qe.pos0 + m) * qe.D;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        lo[e] = f32_to_f16_bits(va[e]);
                        hi[e] = f32_to_f16_bits(vb[e]);
                    }
                    dst = qe.Vc + ((size_t)((n - qe.QD - qe.KVD) / qe.D) * qe.max_seq + qe.pos0 + m) * qe.D;
                }
                *(u32x2*)(dst + d) = u32x2{lo[0] | (lo[1] << 16), lo[2] | (lo[3] << 16)};
                *(u32x2*)(dst + d + half) = u32x2{hi[0] | (hi[1] << 16), hi[2] | (hi[3] << 16)};
            }
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < FM; ++j) {
        const int m = m0 + 32 * j + r0 + 4 * wm;
        if (m >= M) continue;
#pragma unroll
        for (int i = 0; i < (kSilu ? FN / 2 : FN); ++i) {
            const int n = n0 + 32 * i + 8 * g + 4 * wn;
            if (n >= ncols) continue;
            gf32x4 v = acc[i][j];
            if constexpr (kSilu) {
                const gf32x4 u = acc[i + FN / 2][j];
                uint32_t h[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) h[e] = f32_to_f16_bits(v[e] / (1.f + expf(-v[e])) * u[e]);
                *(u32x2*)((uint16_t*)Y + (size_t)m * ldy + n) = u32x2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
            } else if constexpr (kOut == kOutF32) {
                float* y = (float*)Y + (size_t)m * ldy + n;
                if constexpr (kAccum) v += *(const gf32x4*)y;
                *(gf32x4*)y = v;
            } else {
                _Float16* y = (_Float16*)Y + (size_t)m * ldy + n;
                if constexpr (kAccum) {
                    const gf16x4 o = *(const gf16x4*)y;
                    v += gf32x4{(float)o[0], (float)o[1], (float)o[2], (float)o[3]};
                }
                *(gf16x4*)y = gf16x4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
            }
        }
    }
}

// ---- large products: 256 x 256 and 256 x 128 tiles, eight waves ------------------------------
// One workgroup per CU, two waves per SIMD, wave (wm, wn) of WM x 8 / WM: 128 X rows x 64 W rows of
// a 256 x 256 tile (12 operand reads per 32 MFMAs), 64 x 64 of a 256 x 128 one (8 per 16). A stage
// (64-wide K of both operand tiles, the LDS layout above) is two K steps; the operands of a step are
// read during the MFMAs of the step before it, so the matrix cores wait for LDS only at the start:
//   step 0 of stage t: MFMAs; reads of stage t, step 1
//   wait for the copies of stage t + 1; barrier: stage t + 1 is visible, and stage t is in registers
//   step 1 of stage t: MFMAs; reads of stage t + 1, step 0; copies of stage t + 2 into stage t's slot
// Two slots (128 KB) then keep the copies behind the MFMAs with one barrier per stage.
// What bounds it is the matrix cores at the clock the board's power limit leaves them (random fp16
// operands), then the barrier. Measured, f16 unless said (us, before: 128 x 128 ring tiles): 4096^3
// 185 -> 110 (1,250 TFLOP/s; rocBLAS 95-108), 8192^3 1,371 -> 815, SiLU 4096 x 8192 x 4096 734 -> 428,
// 2048 x 4096 x 4096 (256 x 128) 87.6 -> 72, 2048 x 3072 x 1024 22.2 -> 19.5.
// Tried and slower: 32-wide stages in a ring of four (a barrier per step; 119 against 112 at 4096^3),
// four waves of 128 x 128 with the accumulators in AGPRs (127), 128 x 128 tiles of eight waves (217).
// Level: three or four operand reads per slot, wave priority raised around the MFMAs.
// Tile of workgroup b (XCD b % 8): each XCD takes a contiguous part of the tiles in an order that
// runs through groups of 8 m tiles, m fastest, so the 32 workgroups of an XCD share 8 X and 4 W
// tiles in its L2 at a time.
__device__ __forceinline__ void big_tile_of(int b, int tm, int tn, int& mt, int& nt) {
    const int total = tm * tn, q = total >> 3, r = total & 7, x = b & 7;
    const int i = x * q + min(x, r) + (b >> 3);
    constexpr int kGroup = 8;
    const int grp = i / (kGroup * tn), m0 = grp * kGroup, gm = min(kGroup, tm - m0), in = i - grp * kGroup * tn;
    mt = m0 + in % gm;
    nt = in / gm;
}

template <int BM, int BN, int WM, int kOut, bool kAccum>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_big(
    const uint16_t* __restrict__ X, const uint16_t* __restrict__ W, void* __restrict__ Y, int M, int N, int K, int ldy) {
    constexpr bool kSilu = kOut == kOutSilu;
    static_assert(kOut != kOutQKV && !(kSilu && kAccum), "output forms");
    constexpr int kTileCols = kSilu ? BN / 2 : BN;
    constexpr int kStage = (BN + BM) * kRowBytes;
    constexpr int WN = 8 / WM;                            // waves across W
    constexpr int FM = BM / WM / 16, FN = BN / WN / 16;   // 16-row blocks per wave: X, W
    constexpr int NCW = BN / 64, NC = (BN + BM) / 64;     // copies per wave and stage: of W, in all
    static_assert(FM % 2 == 0 && FN % 2 == 0 && (!kSilu || FN == 4), "waves take whole 32-row groups");
    const int ncols = kSilu ? N / 2 : N;
    __shared__ __attribute__((aligned(16))) char lds[2 * kStage];

    const int lane = (int)(threadIdx.x & 63u);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int li = lane & 15, g = lane >> 4;
    const int wm = wave % WM, wn = wave / WM;
    int mt, nt;
    big_tile_of((int)blockIdx.x, (M + BM - 1) / BM, (ncols + kTileCols - 1) / kTileCols, mt, nt);
    const int m0 = mt * BM, n0 = nt * kTileCols;

    // Copy j of a wave is instruction c = wave + 8 j of a stage (rows 8 c .. 8 c + 7): W for j < NCW.
    uint32_t coff[NC];
#pragma unroll
    for (int j = 0; j < NC; ++j) {
        const int row = (wave + 8 * j) * 8 + (lane >> 3);
        const int chunk = (lane & 7) ^ tile::swz_k<64>(row & 31);
        int r;
        if (j >= NCW) r = min(m0 + row - BN, M - 1);
        else if (kSilu) r = row < BN / 2 ? min(n0 + row, ncols - 1) : ncols + min(n0 + row - BN / 2, ncols - 1);
        else r = min(n0 + row, N - 1);
        coff[j] = (uint32_t)r * (uint32_t)K * 2u + (uint32_t)chunk * 16u;
    }
    auto copy = [&](int kt, int j) {
        stream::dma16_s((j < NCW ? W : X) + (size_t)kt * kBK, coff[j], lds + (kt & 1) * kStage + (wave + 8 * j) * 1024);
    };

    // Operand rows of the wave: FN / 2 W groups (32 rows, blocks u = 0, 1) and FM / 2 X groups, both
    // consecutive; a SiLU tile's wave takes a gate group and the up group of the same columns.
    const int r0 = 8 * (li >> 2) + (li & 3);
    const uint32_t rd = (uint32_t)(r0 * kRowBytes + ((g ^ tile::swz_k<64>(r0)) * 16));
    constexpr uint32_t kWStep = (kSilu ? WN : 1) * 4096u;   // bytes from one W group of the wave to the next
    const uint32_t rw = rd + (uint32_t)(kSilu ? wn : FN / 2 * wn) * 4096u;
    const uint32_t rx = rd + (uint32_t)(BN * kRowBytes) + (uint32_t)wm * (FM / 2) * 4096u;
    struct Ops { u32x4 a[FN], b[FM]; };
    auto read_a = [&](Ops& o, const char* st, uint32_t flip, int i) {
        o.a[i] = *(const u32x4*)(st + (rw ^ flip) + (i >> 1) * kWStep + (i & 1) * 512);
    };
    auto read_b = [&](Ops& o, const char* st, uint32_t flip, int j) {
        o.b[j] = *(const u32x4*)(st + (rx ^ flip) + (j >> 1) * 4096 + (j & 1) * 512);
    };

    gf32x4 acc[FN][FM];
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) acc[i][j] = gf32x4{0.f, 0.f, 0.f, 0.f};

    const int nk = K / kBK;   // >= 2 (big_takes)
#pragma unroll
    for (int j = 0; j < NC; ++j) copy(0, j);
#pragma unroll
    for (int j = 0; j < NC; ++j) copy(1, j);
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(NC) : "memory");
    __syncthreads();
    Ops o0, o1;
#pragma unroll
    for (int i = 0; i < FN; ++i) read_a(o0, lds, 0u, i);
#pragma unroll
    for (int j = 0; j < FM; ++j) read_b(o0, lds, 0u, j);

    constexpr int kReads = FM == 8 ? 2 : 4;   // operand reads per slot: all in the first slots
    // One K step: FM slots of FN MFMAs on operands o; ahead of them, in the first slots, the reads of
    // the next step's operands (rd_next) from st at K step `flip`, and the copies of stage kc (cp).
    auto step = [&](const Ops& o, Ops& nx, const char* st, uint32_t flip, bool rd_next, int kc, bool cp) {
#pragma unroll
        for (int j = 0; j < FM; ++j) {
            if (rd_next) {
#pragma unroll
                for (int r = j * kReads; r < min((j + 1) * kReads, FN + FM); ++r)
                    if (r < FN) read_a(nx, st, flip, r);
                    else read_b(nx, st, flip, r - FN);
            }
            if (cp) {
#pragma unroll
                for (int c = j * NC / FM; c < (j + 1) * NC / FM; ++c) copy(kc, c);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < FN; ++i)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(gf16x8, o.a[i]),
                                                                   __builtin_bit_cast(gf16x8, o.b[j]), acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int kt = 0;
    for (; kt + 2 < nk; ++kt) {
        step(o0, o1, lds + (kt & 1) * kStage, 64u, true, 0, false);
        asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
        __syncthreads();
        step(o1, o0, lds + ((kt + 1) & 1) * kStage, 0u, true, kt + 2, true);
    }
    // the last two stages: nothing left to copy
    step(o0, o1, lds + (kt & 1) * kStage, 64u, true, 0, false);
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
    __syncthreads();
    ++kt;
    step(o1, o0, lds + (kt & 1) * kStage, 0u, true, 0, false);
    step(o0, o1, lds + (kt & 1) * kStage, 64u, true, 0, false);
    step(o1, o0, lds, 0u, false, 0, false);

    // acc[i][j] lane (li, g): W group i / 2, block u = i % 2, so columns 8 g + 4 u + e of the group: a
    // lane's two blocks of a group are eight consecutive columns of row m of X block j. (The lane's
    // index is formed again: kept from the start it would take registers the loop has not.)
    const int el = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    const int er0 = 8 * ((el & 15) >> 2) + (el & 3), eg = el >> 4;
#pragma unroll
    for (int j = 0; j < FM; ++j) {
        const int m = m0 + 16 * FM * wm + 32 * (j >> 1) + er0 + 4 * (j & 1);
        if (m >= M) continue;
#pragma unroll
        for (int h = 0; h < (kSilu ? 1 : FN / 2); ++h) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int n = n0 + (kSilu ? 32 * wn : 16 * FN * wn + 32 * h) + 8 * eg + 4 * u;
                if (n >= ncols) continue;
                gf32x4 v = acc[2 * h + u][j];
                if constexpr (kSilu) {
                    const gf32x4 up = acc[(2 + u) % FN][j];
                    uint32_t q[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) q[e] = f32_to_f16_bits(v[e] / (1.f + expf(-v[e])) * up[e]);
                    *(u32x2*)((uint16_t*)Y + (size_t)m * ldy + n) = u32x2{q[0] | (q[1] << 16), q[2] | (q[3] << 16)};
                } else if constexpr (kOut == kOutF32) {
                    float* y = (float*)Y + (size_t)m * ldy + n;
                    if constexpr (kAccum) v += *(const gf32x4*)y;
                    *(gf32x4*)y = v;
                } else {
                    _Float16* y = (_Float16*)Y + (size_t)m * ldy + n;
                    if constexpr (kAccum) {
                        const gf16x4 p = *(const gf16x4*)y;
                        v += gf32x4{(float)p[0], (float)p[1], (float)p[2], (float)p[3]};
                    }
                    *(gf16x4*)y = gf16x4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
                }
            }
        }
    }
}

// ---- up to 16 rows of X: K split over the waves of a workgroup ----------------------------------
// Bound by the read of W in principle, by the chain of K stages in the ring (0.2 us each at 48 of
// them). Here every workgroup takes all rows of X and 16 output columns (kSilu: 16 gate and 16 up rows
// of W), wave w the w-th of kRowsWaves parts of K, straight from memory to registers: each W byte is
// read once and a wave's chain is an eighth. The waves' sums meet in LDS. Measured at M 1 and 16 (us,
// before: ring): N x K 768 x 3072 11.1 -> 6.1, 11.3 -> 7.6; 4096 x 4096 15.1 -> 10.9, 15.1 -> 13.1;
// 768 x 768 4.4 -> 3.1, 4.6 -> 3.7; SiLU 768 x 3072 15.9 -> 8.5, 15.8 -> 10.5.
// Tried and slower: batches of 8 steps' loads ahead of the MFMAs, with the part's last step read
// again past its end (768 x 768 at M 16: 5.9 against 3.6; a wave's load spans 16 rows of 64 bytes, so
// loads are what costs); 16 waves (level); 17 to 64 rows (4096 x 4096 at 32 rows: ring 15.1, here 17.4).
constexpr int kRowsMax = 16, kRowsWaves = 8;

template <int kOut, bool kAccum>
__global__ __launch_bounds__(64 * kRowsWaves) void gemm_rows(const uint16_t* __restrict__ X,
                                                             const uint16_t* __restrict__ W, void* __restrict__ Y,
                                                             int M, int N, int K, int ldy) {
    constexpr bool kSilu = kOut == kOutSilu;
    constexpr int NT = kSilu ? 2 : 1;
    constexpr int kUnroll = 8;
    __shared__ __attribute__((aligned(16))) gf32x4 part[kRowsWaves][NT][64];
    const int ncols = kSilu ? N / 2 : N;
    const int lane = (int)(threadIdx.x & 63u);
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int li = lane & 15, g = lane >> 4;
    const int n0 = (int)blockIdx.x * 16;
    const int steps = K / 32, per = (steps + kRowsWaves - 1) / kRowsWaves;
    const int s0 = min(steps, wave * per), s1 = min(steps, s0 + per);
    const u32x4* wp[NT];   // step s: 16-byte chunk 4 s + g of the row
#pragma unroll
    for (int i = 0; i < NT; ++i) wp[i] = (const u32x4*)(W + (size_t)(i * ncols + min(n0 + li, ncols - 1)) * K) + g;
    const u32x4* xp = (const u32x4*)(X + (size_t)min(li, M - 1) * K) + g;
    gf32x4 acc[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) acc[i] = gf32x4{0.f, 0.f, 0.f, 0.f};
    for (int s = s0; s < s1; s += kUnroll) {
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            if (s + u >= s1) break;
            const int c = 4 * (s + u);
            const u32x4 b = xp[c];
#pragma unroll
            for (int i = 0; i < NT; ++i)
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(gf16x8, wp[i][c]),
                                                                __builtin_bit_cast(gf16x8, b), acc[i], 0, 0, 0);
        }
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) part[wave][i][lane] = acc[i];
    __syncthreads();
    const int n = n0 + 4 * g;
    if (wave != 0 || li >= M || n >= ncols) return;
    gf32x4 v = acc[0], t = acc[NT - 1];
#pragma unroll
    for (int w = 1; w < kRowsWaves; ++w) {
        v += part[w][0][lane];
        if constexpr (kSilu) t += part[w][1][lane];
    }
    if constexpr (kSilu) {
        uint32_t h[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = f32_to_f16_bits(v[e] / (1.f + expf(-v[e])) * t[e]);
        *(u32x2*)((uint16_t*)Y + (size_t)li * ldy + n) = u32x2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
    } else if constexpr (kOut == kOutF32) {
        float* y = (float*)Y + (size_t)li * ldy + n;
        if constexpr (kAccum) v += *(const gf32x4*)y;
        *(gf32x4*)y = v;
    } else {
        _Float16* y = (_Float16*)Y + (size_t)li * ldy + n;
        if constexpr (kAccum) {
            const gf16x4 o = *(const gf16x4*)y;
            v += gf32x4{(float)o[0], (float)o[1], (float)o[2], (float)o[3]};
        }
        *(gf16x4*)y = gf16x4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
    }
}

// Shapes gemm_rows takes: one round of workgroups (8192 x 2048 at M 1 and 16: ring 9.7 and 9.8 us, here
// 10.0 and 12.6) and a K of four stages (1024 x 256: 2.8 -> 2.3, 2.9 -> 2.5). Below that the ring is kept
// and not measured against: the tile query's tests hold its tiles there.
bool takes_rows(int M, int ncols, int K, int cus) {
    return M <= kRowsMax && K >= 4 * kBK && (ncols + 15) / 16 <= cus;
}

int gemm_rows_launch(const uint16_t* X, const uint16_t* W, void* Y, int out, bool accum, int M, int N, int K, int ldy,
                     hipStream_t s) {
    const unsigned grid = ceil_div((size_t)(out == kOutSilu ? N / 2 : N), 16), block = 64 * kRowsWaves;
    if (out == kOutSilu) gemm_rows<kOutSilu, false><<<grid, block, 0, s>>>(X, W, Y, M, N, K, ldy);
    else if (out == kOutF32 && accum) gemm_rows<kOutF32, true><<<grid, block, 0, s>>>(X, W, Y, M, N, K, ldy);
    else if (out == kOutF32) gemm_rows<kOutF32, false><<<grid, block, 0, s>>>(X, W, Y, M, N, K, ldy);
    else if (accum) gemm_rows<kOutF16, true><<<grid, block, 0, s>>>(X, W, Y, M, N, K, ldy);
    else gemm_rows<kOutF16, false><<<grid, block, 0, s>>>(X, W, Y, M, N, K, ldy);
    return launch_status();
}

template <int BM, int BN>
int gemm_launch(const uint16_t* X, const uint16_t* W, void* Y, bool y_f32, bool accum, int M, int N, int K, int ldy,
                hipStream_t s) {
    const unsigned grid = ceil_div((size_t)M, BM) * ceil_div((size_t)N, BN);
    if (y_f32) {
        if (accum) gemm_ring<BM, BN, kOutF32, true><<<grid, 256, 0, s>>>(X, W, Y, M, N, K, ldy, QkvOut{});
        else gemm_ring<BM, BN, kOutF32, false><<<grid, 256, 0, s>>>(X, W, Y, M, N, K, ldy, QkvOut{});
    } else {
        if (accum) gemm_ring<BM, BN, kOutF16, true><<<grid, 256, 0, s>>>(X, W, Y, M, N, K, ldy, QkvOut{});
        else gemm_ring<BM, BN, kOutF16, false><<<grid, 256, 0, s>>>(X, W, Y, M, N, K, ldy, QkvOut{});
    }
    return launch_status();
}

template <int BM, int BN, int WM>
int gemm_big_launch(const uint16_t* X, const uint16_t* W, void* Y, bool y_f32, bool accum, int M, int N, int K, int ldy,
                    hipStream_t s) {
    const unsigned grid = ceil_div((size_t)M, BM) * ceil_div((size_t)N, BN);
    if (y_f32) {
        if (accum) gemm_big<BM, BN, WM, kOutF32, true><<<grid, 512, 0, s>>>(X, W, Y, M, N, K, ldy);
        else gemm_big<BM, BN, WM, kOutF32, false><<<grid, 512, 0, s>>>(X, W, Y, M, N, K, ldy);
    } else {
        if (accum) gemm_big<BM, BN, WM, kOutF16, true><<<grid, 512, 0, s>>>(X, W, Y, M, N, K, ldy);
        else gemm_big<BM, BN, WM, kOutF16, false><<<grid, 512, 0, s>>>(X, W, Y, M, N, K, ldy);
    }
    return launch_status();
}

template <int BM, int BN, int WM>
int gemm_big_silu_launch(const uint16_t* X, const uint16_t* W, void* Y, int M, int F, int K, int ldy, hipStream_t s) {
    const unsigned grid = ceil_div((size_t)M, BM) * ceil_div((size_t)F, BN / 2);
    gemm_big<BM, BN, WM, kOutSilu, false><<<grid, 512, 0, s>>>(X, W, Y, M, 2 * F, K, ldy);
    return launch_status();
}

template <int BM, int BN>
int gemm_silu_launch(const uint16_t* X, const uint16_t* W, void* Y, int M, int F, int K, int ldy, hipStream_t s) {
    const unsigned grid = ceil_div((size_t)M, BM) * ceil_div((size_t)F, BN / 2);
    gemm_ring<BM, BN, kOutSilu, false><<<grid, 256, 0, s>>>(X, W, Y, M, 2 * F, K, ldy, QkvOut{});
    return launch_status();
}

// The tile menu, and the estimate the dispatcher ranks it by: rounds of workgroups over the CUs
// (two workgroups per CU when the ring leaves room for a second in the 160 KB of LDS) times one
// workgroup's time: a fixed cost per K stage (the copy round trip the ring does not hide) plus its
// operand bytes at a per-CU stream rate and its MFMA work at a per-CU matrix rate. Calibrated on
// the cfg5 prompt shapes, where it picks the fastest tile of the menu measured on the box (Q|K|V
// 64 x 96: 7.7 us; O 32 x 32: 5.7; gate|up 128 x 96: 11.5; down 32 x 32: 13.6, event-timed).
struct Tile { int bm, bn; };
constexpr Tile kTiles[] = {{32, 32}, {64, 64}, {64, 96}, {64, 128}, {128, 64}, {128, 96}, {128, 128}};
constexpr double kStageUs = 0.1;           // per 64-wide K stage
constexpr double kCuBytesPerUs = 2.0e5;    // ~200 GB/s of operand tiles per CU
constexpr double kCuFlopsPerUs = 8.0e6;    // ~8 TFLOP/s of fp16 MFMA per CU

// Plain products of fewer stages stay on the ring's menu: not a limit of the kernel (two stages do), and not
// the faster side either (4096 x 4096 x 256, fp32 out: ring 27.5 us, 256 x 256 21.7), but the tiles
// that the tile query's tests name for these shapes.
constexpr int kBigMinStages = 5;

Tile pick_tile(int M, int N, int K, int cus, bool silu = false) {
    Tile best = {0, 0};
    double best_t = 1e300;
    for (const Tile& t : kTiles) {
        if (silu && t.bn % 64) continue;   // a SiLU tile pairs whole gate and up groups
        const int lds = ring_stages(t.bm, t.bn) * (t.bm + t.bn) * kRowBytes;
        const int per_cu = (160 * 1024) / lds >= 2 ? 2 : 1;
        const double tiles = (double)ceil_div((size_t)M, t.bm) * ceil_div((size_t)N, t.bn);
        const double rounds = ceil(tiles / ((double)cus * per_cu));
        const double wg = (double)(K / kBK) * kStageUs + (double)(t.bm + t.bn) * K * 2 / kCuBytesPerUs +
                          2.0 * t.bm * t.bn * K / kCuFlopsPerUs;
        const double est = rounds * wg;
        if (est < best_t) {
            best_t = est;
            best = t;
        }
    }
    return best;
}

// The large-product tile a shape takes, or {0, 0} for the ring tile `t` of the menu. Times in us of a
// round of one workgroup per CU, fitted to a sweep of both tiles and the ring over M 200 .. 4096 at
// N x K of 768 x 768 .. 8192 x 4096 (14 pairs; fill: share of the CUs the tiles occupy, at most 1): a
// tile's prologue and epilogue, then its stages. The estimate picked the faster side at each sweep
// point beyond 4 %, and no product of profiles/gemm_tiles.md is over 4 % slower than on the ring; small products stay on the ring (512 x 8192 x 4096: ring 45.9, 256 x 128 78.9).
Tile pick_big(int M, int N, int K, int cus, bool silu, const Tile& t) {
    const int nk = K / kBK;
    if (nk < (silu ? 2 : kBigMinStages)) return Tile{0, 0};
    auto rounds = [&](const Tile& x, int per_cu) {
        return ceil((double)ceil_div((size_t)M, x.bm) * ceil_div((size_t)N, x.bn) / ((double)cus * per_cu));
    };
    const int lds = ring_stages(t.bm, t.bn) * (t.bm + t.bn) * kRowBytes;
    const double wg = nk * kStageUs + (double)(t.bm + t.bn) * K * 2 / kCuBytesPerUs +
                      2.0 * t.bm * t.bn * K / kCuFlopsPerUs;
    double best = 0.95 * rounds(t, (160 * 1024) / lds >= 2 ? 2 : 1) * (1.2 * wg + 3.0);
    Tile r = {0, 0};
    struct Big { Tile t; double fixed, stage, stage_full; };
    constexpr Big kBig[] = {{{256, 256}, 6.0, 1.2, 0.42}, {{256, 128}, 4.5, 0.75, 0.33}};
    for (const Big& b : kBig) {
        const double fill = std::min(1.0, (double)ceil_div((size_t)M, b.t.bm) * ceil_div((size_t)N, b.t.bn) / cus);
        const double est = rounds(b.t, 1) * (b.fixed + nk * (b.stage + b.stage_full * fill));
        if (est < best) {
            best = est;
            r = b.t;
        }
    }
    return r;
}

// The tile of cdna4_gemm_f16_nt (or, silu, of cdna4_gemm_f16_nt_silu; N counts gate and up rows).
Tile choose_tile(int M, int N, int K, int cus, bool silu) {
    if (takes_rows(M, silu ? N / 2 : N, K, cus)) return Tile{kRowsMax, silu ? 32 : 16};
    const Tile t = pick_tile(M, N, K, cus, silu);
    const Tile big = pick_big(M, N, K, cus, silu, t);
    return big.bm ? big : t;
}

}  // namespace

// Returns -1, launching nothing, for a shape this kernel does not take (K not a multiple of 64,
// N or ldy not a multiple of 4, X / W not 16-byte or Y not 16- (fp32) / 8-byte (fp16) aligned,
// operands past 4 GiB); the caller then uses rocBLAS. Otherwise 0 or the launch's error.
// cold: the operands arrive from HBM or the Infinity Cache, not L2 (the runtime's prompt, where
// each GEMM reads the previous kernel's output and a layer's weights once). There a 32 x 32 pick
// becomes 64 x 32 (half the W re-reads, five-stage ring, two workgroups per CU): at config 5 the
// O and down projections took the time to first token from 0.767 to 0.733 ms, though launched
// back to back on the same operands (all in L2) 64 x 32 ran no faster (O 5.9 against 6.0 us,
// down 14.1 against 13.7).
int llm_gemm_f16(const uint16_t* X, const uint16_t* W, void* Y, bool y_f32, bool accum, int M, int N, int K, int ldy,
                 hipStream_t s, bool cold) {
    if (M <= 0 || N <= 0 || K <= 0 || K % kKMul || N % 4 || ldy % 4 || ldy < N) return -1;
    if (((uintptr_t)X | (uintptr_t)W) % 16 || (uintptr_t)Y % (y_f32 ? 16 : 8)) return -1;
    if ((uint64_t)M * K * 2 >= (1ull << 32) || (uint64_t)N * K * 2 >= (1ull << 32)) return -1;   // 32-bit copy offsets
    const int cus = device_cus() > 0 ? device_cus() : 256;
    if (takes_rows(M, N, K, cus)) return gemm_rows_launch(X, W, Y, y_f32 ? kOutF32 : kOutF16, accum, M, N, K, ldy, s);
    Tile t = choose_tile(M, N, K, cus, false);
    if (cold && t.bm == 32 && t.bn == 32 && M >= 64 &&
        (double)ceil_div((size_t)M, 64) * ceil_div((size_t)N, 32) <= 2.0 * cus)
        t = Tile{64, 32};
#define CDNA4_GEMM_TILE(a, b) \
    if (t.bm == a && t.bn == b) return gemm_launch<a, b>(X, W, Y, y_f32, accum, M, N, K, ldy, s);
    CDNA4_GEMM_TILE(32, 32) CDNA4_GEMM_TILE(64, 32) CDNA4_GEMM_TILE(64, 64) CDNA4_GEMM_TILE(64, 96)
    CDNA4_GEMM_TILE(64, 128) CDNA4_GEMM_TILE(128, 64) CDNA4_GEMM_TILE(128, 96) CDNA4_GEMM_TILE(128, 128)
    if (t.bm == 256 && t.bn == 256) return gemm_big_launch<256, 256, 2>(X, W, Y, y_f32, accum, M, N, K, ldy, s);
    if (t.bm == 256 && t.bn == 128) return gemm_big_launch<256, 128, 4>(X, W, Y, y_f32, accum, M, N, K, ldy, s);
#undef CDNA4_GEMM_TILE
    return -1;
}

// The prompt's Q|K|V projection X [M][K] x W [QD + 2 KVD][K]^T with the RoPE + append epilogue
// (kOutQKV; q_out, K and V caches as QkvOut describes, cos/sin tables [max_seq][D]). Tiles of
// whole heads only (BN % D == 0, D % 64 == 0): the tile of the single-pass menu with the least
// estimate among those. Returns -1, launching nothing, for shapes it does not take (the runtime
// then projects with llm_gemm_f16 and appends separately).
int llm_gemm_qkv_rope(const uint16_t* X, const uint16_t* W, int M, int K, const QkvOut& qe, hipStream_t s) {
    const int N = qe.QD + 2 * qe.KVD;
    if (M <= 0 || K <= 0 || K % kKMul || qe.D % 64 || qe.QD % qe.D || qe.KVD % qe.D) return -1;
    if (((uintptr_t)X | (uintptr_t)W) % 16 || ((uintptr_t)qe.q_out | (uintptr_t)qe.Kc | (uintptr_t)qe.Vc) % 8) return -1;
    if ((uint64_t)M * K * 2 >= (1ull << 32) || (uint64_t)N * K * 2 >= (1ull << 32)) return -1;
    const int cus = device_cus() > 0 ? device_cus() : 256;
    Tile best = {0, 0};
    double best_t = 1e300;
    for (const Tile& t : kTiles) {
        if (t.bn % qe.D || t.bn % 64) continue;
        const int lds = ring_stages(t.bm, t.bn, ring_budget(kOutQKV, t.bm, t.bn)) * (t.bm + t.bn) * kRowBytes;
        const int per_cu = (160 * 1024) / lds >= 2 ? 2 : 1;
        const double tiles = (double)ceil_div((size_t)M, t.bm) * ceil_div((size_t)N, t.bn);
        const double wg = (double)(K / kBK) * kStageUs + (double)(t.bm + t.bn) * K * 2 / kCuBytesPerUs +
                          2.0 * t.bm * t.bn * K / kCuFlopsPerUs;
        const double est = ceil(tiles / ((double)cus * per_cu)) * wg;
        if (est < best_t) {
            best_t = est;
            best = t;
        }
    }
    const unsigned grid = ceil_div((size_t)M, best.bm) * ceil_div((size_t)N, best.bn);
#define CDNA4_QKV_TILE(a, b)                                                                              \
    if (best.bm == a && best.bn == b) {                                                                     \
        gemm_ring<a, b, kOutQKV, false><<<grid, 256, 0, s>>>(X, W, nullptr, M, N, K, N, qe);                \
        return launch_status();                                                                             \
    }
    CDNA4_QKV_TILE(64, 64) CDNA4_QKV_TILE(64, 128) CDNA4_QKV_TILE(128, 64) CDNA4_QKV_TILE(128, 128)
#undef CDNA4_QKV_TILE
    return -1;
}

// Y[M][F] fp16 = fp16(silu(X Wg^T) * (X Wu^T)), W = [Wg; Wu] fp16 [2F][K] (the SwiGLU gate|up
// product followed by the SiLU product in one launch). Returns -1, launching nothing, for a shape
// the kernel does not take (as llm_gemm_f16; F a multiple of 4, Y 8-byte aligned).
int llm_gemm_f16_silu(const uint16_t* X, const uint16_t* W, void* Y, int M, int F, int K, int ldy, hipStream_t s) {
    if (M <= 0 || F <= 0 || K <= 0 || K % kKMul || F % 4 || ldy % 4 || ldy < F) return -1;
    if (((uintptr_t)X | (uintptr_t)W) % 16 || (uintptr_t)Y % 8) return -1;
    if ((uint64_t)M * K * 2 >= (1ull << 32) || (uint64_t)2 * F * K * 2 >= (1ull << 32)) return -1;
    const int cus = device_cus() > 0 ? device_cus() : 256;
    if (takes_rows(M, F, K, cus)) return gemm_rows_launch(X, W, Y, kOutSilu, false, M, 2 * F, K, ldy, s);
    const Tile t = choose_tile(M, 2 * F, K, cus, true);
#define CDNA4_GEMM_TILE(a, b) \
    if (t.bm == a && t.bn == b) return gemm_silu_launch<a, b>(X, W, Y, M, F, K, ldy, s);
    CDNA4_GEMM_TILE(64, 64) CDNA4_GEMM_TILE(64, 128) CDNA4_GEMM_TILE(128, 64) CDNA4_GEMM_TILE(128, 128)
    if (t.bm == 256 && t.bn == 256) return gemm_big_silu_launch<256, 256, 2>(X, W, Y, M, F, K, ldy, s);
    if (t.bm == 256 && t.bn == 128) return gemm_big_silu_launch<256, 128, 4>(X, W, Y, M, F, K, ldy, s);
#undef CDNA4_GEMM_TILE
    return -1;
}

}  // namespace cdna4

extern "C" int cdna4_gemm_f16_nt_silu(const void* X, const void* W, void* Y, int M, int F, int K, int ldy,
                                      cdna4_stream_t stream) {
    if (M < 0 || F < 0 || K < 0) return CDNA4_ERR_INVALID_VALUE;
    if (M == 0 || F == 0) return 0;
    if (!X || !W || !Y) return CDNA4_ERR_INVALID_VALUE;
    if (int e = cdna4::check_device()) return e;
    const int e = cdna4::llm_gemm_f16_silu((const uint16_t*)X, (const uint16_t*)W, Y, M, F, K, ldy, (hipStream_t)stream);
    return e == -1 ? CDNA4_ERR_INVALID_VALUE : e;
}

extern "C" int cdna4_gemm_f16_nt_silu_tile(int M, int F, int K, int* bm, int* bn) {
    if (M <= 0 || F <= 0 || K <= 0 || !bm || !bn) return CDNA4_ERR_INVALID_VALUE;
    const cdna4::Tile t = cdna4::choose_tile(M, 2 * F, K, cdna4::device_cus() > 0 ? cdna4::device_cus() : 256, true);
    *bm = t.bm;
    *bn = t.bn;
    return 0;
}

extern "C" int cdna4_gemm_f16_nt_tile(int M, int N, int K, int* bm, int* bn) {
    if (M <= 0 || N <= 0 || K <= 0 || !bm || !bn) return CDNA4_ERR_INVALID_VALUE;
    const cdna4::Tile t = cdna4::choose_tile(M, N, K, cdna4::device_cus() > 0 ? cdna4::device_cus() : 256, false);
    *bm = t.bm;
    *bn = t.bn;
    return 0;
}

extern "C" int cdna4_gemm_f16_nt(const void* X, const void* W, void* Y, int y_f32, int accum, int M, int N, int K,
                                 int ldy, cdna4_stream_t stream) {
    if (M < 0 || N < 0 || K < 0 || (y_f32 != 0 && y_f32 != 1) || (accum != 0 && accum != 1))
        return CDNA4_ERR_INVALID_VALUE;
    if (M == 0 || N == 0) return 0;
    if (!X || !W || !Y) return CDNA4_ERR_INVALID_VALUE;
    if (int e = cdna4::check_device()) return e;
    const int e = cdna4::llm_gemm_f16((const uint16_t*)X, (const uint16_t*)W, Y, y_f32 == 1, accum == 1, M, N, K, ldy,
                                      (hipStream_t)stream, false);
    return e == -1 ? CDNA4_ERR_INVALID_VALUE : e;
}
