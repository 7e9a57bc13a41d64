// CPU test of the fp32 GEMM's tile / split-K plan (omhip::planGemmFor): the
// split-K partial sums of every plan fit the no-allocation entry's fixed array
// (kNoAllocScratchBytes less its arrival counters), the tiles' counters fit
// theirs (kNoAllocCounterBytes), and the partials stay below the stated bound of 4 x CUs tiles of
// 64 x 64 floats, over the GEMM sweep, the MLP and ResNet weight-gradient
// shapes, the shapes that reach the bound, and a dense grid of small M / N. And of
// the C store's offsets: whatever the row stride, a row past the matrix stays out of
// the buffer view and a row inside it keeps its offset.
// Exit status 0 = all checks passed.
#include <cstdint>
#include <cstdio>
#include <vector>

#include "../../omnimatchdeeplearningtool_amd/csrc/gemm_f32.hpp"

static int g_fail = 0;
static long long g_maxBytes = 0;

static void check(int M, int N, int K, int batch, long long cus) {
    // the layouts share tile and splits and differ in the unit that computes a small tile alone; sums of one
    // product are always the fp32 MFMA's
    for (int l = 0; l < 4; ++l) {
        const omhip::GemmPlan a = omhip::planGemmFor(M, N, K, batch, true, cus, l & 1, l & 2);
        const omhip::GemmPlan b = omhip::planGemmFor(M, N, K, batch, true, cus);
        const omhip::GemmPlan one = omhip::planGemmFor(M, N, 1, batch, true, cus, l & 1, l & 2);
        if (a.cfg != b.cfg || a.splits != b.splits || (a.plain && a.cfg != 2) || one.cfg != 2 || !one.plain) {
            std::printf("FAIL layout %d M=%d N=%d K=%d batch=%d cus=%lld\n", l, M, N, K, batch, cus);
            ++g_fail;
        }
    }
    const long long small = (long long)((M + 63) / 64) * ((N + 63) / 64) * batch;
    if (small >= cus && K < 2048 && omhip::planGemmFor(M, N, K, batch, true, cus).splits != 1) {
        std::printf("FAIL M=%d N=%d K=%d batch=%d cus=%lld: a split where every CU has a tile\n", M, N, K, batch, cus);
        ++g_fail;
    }
    // the wsOk rule of gemmF32: 64 splits of the batch's C within 256 MiB
    const bool wsOk = (long long)64 * batch * M * N * 4 <= (256LL << 20);
    const omhip::GemmPlan p = omhip::planGemmFor(M, N, K, batch, wsOk, cus);
    if (p.splits <= 1) return;
    const int pieces = omhip::splitPieces(K, p.splits);
    const long long tiles = (long long)((M + 63) / 64) * ((N + 63) / 64) * batch;
    const long long bytes = (long long)pieces * tiles * 64 * 64 * 4;   // partials in whole 64 x 64 tiles
    if (g_maxBytes < bytes && cus == 256) g_maxBytes = bytes;
    if (p.cfg != 2 || bytes > (long long)(omhip::kNoAllocScratchBytes - omhip::kNoAllocCounterBytes) ||
        tiles * 4 > (long long)omhip::kNoAllocCounterBytes || tiles * p.splits >= 4 * cus ||
        bytes > 4 * cus * 64LL * 64 * 4) {
        std::printf("FAIL M=%d N=%d K=%d batch=%d cus=%lld: cfg %d splits %d (%d pieces) %lld bytes\n", M, N, K, batch,
                    cus, p.cfg, p.splits, pieces, bytes);
        ++g_fail;
    }
}

// Range check of a raw buffer access: the lane's offset against the view's bytes less the scalar offset, all 32 bits.
static bool outOfRange(uint32_t lane, uint32_t scalar) { return lane >= (uint32_t)(omhip::kSplitView - scalar); }

static void checkStore(int M, long long ldc) {
    // the host takes the buffer views only while a 64-row tile's existing rows lie inside one
    if (((M < 64 ? M : 64) - 1) * ldc * 4 + 512 >= (long long)omhip::kSplitView) return;
    for (int block = 0; block < 64; block += 32)
        for (int r = 0; r < 16; ++r) {
            const int ro = 8 * (r >> 2) + (r & 3), left = M - block;
            const uint32_t off = omhip::storeRowOffset(ro, left, ldc);
            if (!outOfRange(omhip::kSplitOOB, off) || (ro < left && off != (uint64_t)ro * ldc * 4)) {
                std::printf("FAIL store M=%d ldc=%lld block %d row %d: offset %u\n", M, ldc, block, ro, off);
                ++g_fail;
            }
        }
}

// Every read of the partials: four parts at a time, those past the last out of range.
static void checkParts(int splits, uint32_t tiles) {
    const uint32_t view = tiles * splits * 64 * 64 * 4, stride = tiles * 64 * 64 * 4;
    for (uint32_t slot : {0u, tiles - 1})
        for (int s = 0; s < (splits + 3) / 4 * 4; ++s) {
            const uint32_t off = omhip::splitPartOffset(s, splits, slot * 64 * 64 * 4, stride);
            const uint32_t lane = s < splits ? 64 * 64 * 4 - 16 : 0x40000000u;   // kOOB
            const bool out = lane >= (uint32_t)(view - off);
            if (out == (s < splits) || (s < splits && (uint64_t)lane + off + 16 > view)) {
                std::printf("FAIL parts splits=%d tiles=%u slot %u part %d: offset %u\n", splits, tiles, slot, s, off);
                ++g_fail;
            }
        }
}

int main() {
    for (int splits = 2; splits <= 64; ++splits)
        for (uint32_t tiles : {1u, 3u, 64u, 511u}) checkParts(splits, tiles);
    for (int M : {1, 2, 3, 9, 17, 28, 31, 33, 60, 64, 200}) {
        for (long long ldc : {1LL, 64LL, 4096LL, 1LL << 24, (1LL << 30) - 1, 1LL << 30}) checkStore(M, ldc);
        // strides whose multiples fall just past the view's end, mod 2^32
        for (int ro = 1; ro < 28; ++ro)
            for (uint64_t at = 0xfffffe80u; at < 0x100000080u; at += 4)
                for (uint64_t w = 0; w < 4; ++w) checkStore(M, (long long)((at + (w << 32)) / 4 / ro));
    }
    const int sq[] = {512, 1024, 2048, 4096, 8192};
    for (int s : sq) check(s, s, s, 1, 256);
    check(128, 4096, 4096, 1, 256);
    check(8192, 256, 2048, 1, 256);
    check(448, 4672, 2048, 1, 256);   // 511 tiles split in two: the largest plan on 256 CUs
    check(128, 256, 784, 1, 256);     // MLP layers and their gradients
    check(784, 256, 128, 1, 256);
    check(256, 128, 128, 1, 256);
    check(64, 4096, 4096, 1, 256);
    // a dense grid of small outputs with long K, single and batched, on 256 and 304 CUs
    for (long long cus : {256LL, 304LL, 80LL})
        for (int b : {1, 2, 3, 8})
            for (int M = 16; M <= 1024; M += 48)
                for (int N = 16; N <= 5000; N += 112)
                    for (int K : {512, 784, 1000, 1024, 2048, 4096, 16384, 65536}) check(M, N, K, b, cus);
    std::printf("largest split plan on 256 CUs: %lld bytes\n", g_maxBytes);
    std::printf(g_fail ? "FAILED %d\n" : "ALL PASSED\n", g_fail);
    return g_fail ? 1 : 0;
}
