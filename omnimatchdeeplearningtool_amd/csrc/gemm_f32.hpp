// gemm_f32.hpp — host-side interface of the fp32 MFMA GEMM shared by the GEMM
// and conv entry points.
#pragma once

#include <cstddef>
#include <cstdint>

namespace omhip {

struct GemmPlan {
    int cfg;      // 0: 256x256, 1: 128x128, 2: 64x64
    int splits;   // K splits (1: none)
    bool plain = false;   // cfg 2: on the fp32 MFMA instead of through the pieces
};

// The K pieces a plan's launch actually uses: K in chunks of a whole number of
// 16-deep slices (the last chunk may be shorter), so fewer than plan.splits
// pieces when K is short.
inline int splitPieces(int K, int splits, int* kChunk = nullptr) {
    const int bk = 16;
    const int chunk = ((K + splits - 1) / splits + bk - 1) / bk * bk;
    if (kChunk) *kChunk = chunk;
    return (K + chunk - 1) / chunk;
}

// Whether 64x64 tiles run on the fp32 MFMA instead of through the pieces (`chunk`:
// the K of one piece of a split, else K). The pieces cost a split of each operand
// element per 64 products and a stage of two slices, which only long products of
// tiles that share a CU pay back; K past the last whole stage waits for memory. A sum of
// one product is correctly rounded on the fp32 MFMA alone. Measured on MI355X, us,
// pieces / fp32 MFMA (NN, NT, TN):
//   a tile per CU at most, K not split: 64x64x64 4.9 / 4.8, 87x444x108 6.9 / 5.6, 300^3 10.1 / 8.8,
//     9.8 / 8.5, 11.0 / 8.6; 1024x1024x256 8.3 / 8.1, 8.2 / 7.9, 9.1 / 8.2; x1000 23.1 / 22.1, 22.7 / 21.3, 25.9 / 22.4;
//   split: 128x256x784 10.3 / 10.0, 10.8 / 9.9, 11.1 / 10.0; 256x256x512 8.5 / 8.9, 9.1 / 8.8, 9.1 / 8.9; x4096 (16
//     pieces) 17.4 / 18.9, 19.4 / 18.8, 18.2 / 19.5; 8x4096x4096 (pieces of 512) 21.8 / 25.1, 23.0 / 24.8, 23.9 / 25.6;
//     87x108x3284 (of 416) 15.0 / 15.5, 15.9 / 15.2, 16.3 / 15.6; 19x1212x1160 (of 304)
//     12.7 / 12.1, 12.8 / 11.9, 13.9 / 13.1; 128x4000x2100 TN (8 of 272, 1008 workgroups) 28.6 / 25.8;
//   more tiles than CUs: 1024x2048x64 6.8 / 6.4, x100 9.1 / 8.0, x160 9.5 / 9.3, x256 11.6 / 12.2; 600 of 64x64x32
//     7.8 / 6.4, x128 13.1 / 11.2.
// Rows of an operand stored K first that are no multiple of four (`ragged`) load element by element there.
constexpr bool smallTilePlain(long long tiles, int K, int chunk, bool ta, bool tb, bool ragged, long long cus) {
    if (tiles > cus) return K <= (K % 32 ? 320 : 192);
    if (ragged && chunk > 320) return false;
    if (chunk >= K) return true;
    if (chunk >= 512) return false;
    if (tiles * ((K + chunk - 1) / chunk) > 2 * cus) return true;   // the pieces' LDS holds two workgroups per CU
    return tb && !ta ? true : K < 2048 && (ta || chunk % 32 != 0);
}

// Tile and split-K choice on a device of `cus` compute units. A launch takes as
// long as its busiest CU: tiles per CU times the time of one tile's 16-deep
// slice, in us measured on MI355X (4096^3 forced onto each tile, divided by its
// rounds; a lone small tile per CU from 1 x 1 rounds): 256x256 2.25, 128x128 0.66,
// 64x64 0.23 (0.305 alone). Per 64x64 of C that is 0.141, 0.165, 0.23: the larger
// tile splits each operand element for more products; the smaller one wins where
// it fills the last round (4608^3: 324 tiles of 256x256 are two rounds, 4.5 against
// 4.0 for 1296 of 128x128). Ties go to the larger tile. A short K is fill and stores:
// small tiles on the fp32 MFMA (1500x1500x32 7.6 us on 128x128, 6.3; x100 11.2, 10.0; 2048x2048x32
// 8.6, 8.0, x64 9.6, 9.8; 1024 of 128x128x16 16.4, 18.3).
// When 64x64 tiles give fewer than two workgroups per CU and K is long (few rows
// or columns: 128 x 4096 x 4096, weight gradients), K is split over the 64x64
// tile: the smallest power of two (at most 64) that gives every CU two workgroups
// while each split keeps >= 256 of K. The partials cost one fp32 write and read
// of C per split. 128 x 4096 x 4096 measured (us): 1 split 78, 2 43, 4 38, 8 39.
// With 512 <= K < 1024 only grids of at most CUs / 4 tiles split (pieces of >= 128
// of K: 128 x 256 x 784, the MLP's first layer, 1 split 19.4, 2 13.4, 4 11.0,
// 8 10.8); shorter K runs faster unsplit. A split plan stops doubling once the grid
// holds 2 x CUs workgroups, so its partials cover fewer than 4 x CUs tiles of
// 64 x 64 floats (16 MiB on 256 CUs). Host-only, so a CPU test checks that bound.
inline GemmPlan planGemmFor(int M, int N, int K, int batch, bool wsOk, long long cus, bool ta = false, bool tb = false) {
    auto tiles = [&](int bm, int bn) { return (long long)((M + bm - 1) / bm) * ((N + bn - 1) / bn) * batch; };
    const long long t = tiles(64, 64);
    auto rounds = [&](long long n) { return (double)((n + cus - 1) / cus); };
    auto small = [&](int splits) {
        int chunk;
        splitPieces(K, splits, &chunk);
        const bool ragged = (ta && M % 4) || (!tb && N % 4);
        return GemmPlan{2, splits, smallTilePlain(t, K, chunk, ta, tb, ragged, cus)};
    };
    if (K < 4 || (K <= 32 && t <= 4 * cus) || (K <= 128 && tiles(128, 128) < cus)) return small(1);
    const double costL = 2.25 * rounds(tiles(256, 256)), costM = 0.66 * rounds(tiles(128, 128));
    const double costS = t <= cus ? 0.305 : 0.23 * rounds(t);
    if (costL <= costM && costL <= costS) return {0, 1};
    if (costM <= costS) return {1, 1};
    if (t >= 2 * cus || !wsOk || K < 512 || (K < 1024 && t * 4 > cus)) return small(1);
    int s = 1;
    if (K < 1024) {   // very few tiles (at most CUs / 4): splits of >= 128 of K
        while (s < 64 && t * s < 2 * cus && K / (2 * s) >= 128) s *= 2;
        return small(s);
    }
    // with one tile per CU already, a split must keep >= 1024 of K: shorter ones gain
    // little (1024^3 22.1 us unsplit, 21.3 split in two), and a split needs a workspace, which
    // a stream that records a graph cannot grow
    const int minK = t >= cus ? 1024 : 256;
    while (s < 64 && t * s < 2 * cus && K / (2 * s) >= minK) s *= 2;
    return small(s);
}

// Bytes of the fixed device array behind omHipGemmStridedBatchedNoAlloc: twice
// the bound above for a 256-CU device. Its last kNoAllocCounterBytes hold the
// tiles' split-K arrival counters (zero at load, and every launch leaves them
// zero); the partials use the rest.
constexpr size_t kNoAllocScratchBytes = (size_t)32 << 20;
constexpr size_t kNoAllocCounterBytes = (size_t)64 << 10;

// The buffer views of the operands and of C reach almost 2^32 bytes past their
// first element; a lane whose offset is kSplitOOB reads zero and writes nothing
// beside any scalar offset that lies inside the view (the range check is
// kSplitOOB >= kSplitView - scalar offset).
constexpr uint32_t kSplitView = 0xffffff00u, kSplitOOB = 0xffffff80u;

// Scalar byte offset of the C rows `ro` past a wave block's first, of which
// `rowsLeft` exist: 0 for rows that no lane writes, whose own offset could be any
// value mod 2^32 (a matrix of few rows may have a row stride of 2^30).
constexpr uint32_t storeRowOffset(int ro, int rowsLeft, long long ldc) {
    return ro < rowsLeft ? (uint32_t)(ro * ldc * 4) : 0u;
}

// Scalar byte offset of a tile's part `s` of `splits` among the split-K partials:
// 0 for parts past the last, whose lanes are marked out of range (their own offset
// lies past the view, where the range check's difference would wrap).
constexpr uint32_t splitPartOffset(int s, int splits, uint32_t base, uint32_t stride) {
    return s < splits ? base + (uint32_t)s * stride : 0u;
}

struct GemmF32Params {
    const float* A;
    const float* B;
    float* C;
    int M, N, K;
    long long lda, ldb, ldc;
    long long sA, sB, sC;   // per-batch element offsets (0 shares the operand)
    int tilesM, tilesN;
    int kChunk;             // split-K: split s covers k in [s*kChunk, min(K, (s+1)*kChunk))
    float* ws;              // split-K partials [split][batch][tile], each tile in its registers' order (null: write C)
    unsigned* ctr;          // split-K: per (batch, tile) arrival counters, zero at rest
    int splits;             // split-K: pieces of K (the last arrival of a tile sums them)
    const float* bias;      // [N] added to every row of C, or null
    int act;                // 0 identity, 1 ReLU (after the bias)
    const float* gate;      // Linear backward: C kept where gate > 0 (row stride ldg)
    long long ldg;
};

// C[b] = op(A[b]) * op(B[b]); ta: A stored [K,M]; tb: B stored [N,K].
// Enqueues on the library stream; returns 0 or -1 (message via fail()).
// bias ([N], nullable) and act (0 identity, 1 ReLU) are applied to every
// element of C as it is written: C = act(op(A) * op(B) + bias).
int gemmF32(bool ta, bool tb, int batch, int M, int N, int K,
            const float* A, long long lda, long long sA,
            const float* B, long long ldb, long long sB,
            float* C, long long ldc, long long sC,
            const float* bias = nullptr, int act = 0);

// Zeroes C (batch x M x N, row stride ldc, batch stride sC) on the stream.
int zeroOutput(float* C, int batch, int M, int N, long long ldc, long long sC);

}  // namespace omhip
