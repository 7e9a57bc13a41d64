// split_tile.hpp — fp32 products on the bf16 matrix cores (gfx950).
//
// An fp32 value x is the sum of three bf16 values: h = bf16(x), m = bf16(x - h),
// l = bf16(x - h - m) (round to nearest even; both differences are exact, and
// 3 x 8 significand bits hold all 24 of x). A product a * b is accumulated in
// fp32 from six of the nine piece products, smallest first within each 16-deep
// slice of K: al bh, ah bl, am bm, am bh, ah bm, ah bh. The three left out
// are together below 2^-24 |a b| (2^-26 typically): less than the rounding of
// one fp32 product. Each piece product is exact, and one MFMA adds 16 of them
// per rounding where v_mfma_f32_32x32x2_f32 adds 2, so sums of dense operands are
// closer to the exact ones than the fp32 MFMA's. Measured against float64
// (2-norm, N(0,1) operands): K = 16 3.4e-8 (fp32 MFMA 7.0e-8), K = 576 3.6e-7
// (4.3e-7), K = 4096 9.9e-7 (1.14e-6); uniform [0,1) operands, K = 4096: 5.3e-7
// (8.5e-7). The nine-product sum measures the same; big pieces first is worse
// at small K (8.2e-8 at K = 16).
// Where most products are zero, that turns: a slice rounds its sums six times
// however few of its products count, and the bf16 MFMA's rounding is not always to
// nearest. A row with one non-zero element, correctly rounded on the fp32 MFMA, is
// off by up to 1.45 units in the last place here (21 % of its outputs not the
// nearest float, 3.5e-8 for 2.5e-8); with n of 2048 elements non-zero, n = 4 7.7e-8
// (4.0e-8), n = 64 2.9e-7 (1.45e-7). Products of K < 4 run on the fp32 MFMA; rows
// of zeros in longer ones are not looked for. Adding each slice up on its own and then
// to the sums (n = 64: 1.5e-7) took 7 to 14 % more time on the smaller tiles and more
// registers than the large one has.
//
// Why: six v_mfma_f32_32x32x16_bf16 take 192 cycles for the 16 k that take
// v_mfma_f32_32x32x2_f32 512, and the bf16 MFMA runs beside VALU work (the
// splitting), which the fp32 MFMA does not.
//
// The operands are split times 2^16, exactly, and the sums taken back by 2^-32:
// then every bit of every fp32 value down to the smallest denormal (2^-149)
// lies in the pieces' range (2^-133). What the pieces cannot carry leaves a
// non-finite sum in every output it takes part in (x - h of an infinite or NaN
// h is NaN): infinities, NaN, |x| from 2^112 - 2^103 on (a scaled value that
// rounds past the largest bf16) and sums of 2^96 and more. A tile with such a sum
// is computed again on the fp32 MFMA.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

#include "buffer_io.hpp"
#include "gemm_f32.hpp"
#include "mfma_f32_tile.hpp"

namespace omhip {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr float kSplitScale = 65536.0f;              // 2^16 on each operand
constexpr float kSplitUnscale = 0x1p-32f;            // off the sums

__device__ __forceinline__ uint32_t packBf16(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}

// The three pieces of two values times kSplitScale, packed as bf16 pairs (a in
// the low half): 13 vector instructions.
__device__ __forceinline__ void splitPair(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
    a *= kSplitScale;
    b *= kSplitScale;
    h = packBf16(a, b);
    const float ra = a - __uint_as_float(h << 16), rb = b - __uint_as_float(h & 0xffff0000u);
    m = packBf16(ra, rb);
    l = packBf16(ra - __uint_as_float(m << 16), rb - __uint_as_float(m & 0xffff0000u));
}

// LDS image of one operand's 16-deep slice: per piece, two groups (k 0..7 and
// 8..15) of R rows x 8 bf16, so that a fragment (32 rows, one group per half
// wave) is two contiguous 512-byte runs. The 128 bytes between the groups keep
// 8-byte stores of 8 rows x 4 k quads on distinct banks.
template <int R>
struct SplitLds {
    static constexpr int BK = 16;
    static constexpr int GROUP = R * 16 + 128;
    static constexpr int PIECE = 2 * GROUP;
    static constexpr int SIZE = 3 * PIECE;   // bytes
};

// Loader of a K-contiguous operand: element (r, k) at P[r * ld + k], in
// 4-float vectors (any 4-byte alignment). Per-lane byte offsets are fixed for
// the K walk and each slice re-bases the buffer view; rows past the matrix read
// zeros. Slices that end past kEnd load element by element unless kEnd is a multiple of four. In-tile offsets
// must stay below kSplitView (splitViewOk).
template <int R, int NT>
struct SplitLoaderK {
    static constexpr int PER_T = R * 4 / NT;
    static_assert(R * 4 % NT == 0, "slice must divide over the threads");
    using Lds = SplitLds<R>;
    const float* tile;
    uint32_t voff[PER_T];
    f32x4 v[PER_T];

    __device__ __forceinline__ void init(const float* p, long long ld, int rows, int r0, int tid) {
        tile = p + (long long)r0 * ld;
#pragma unroll
        for (int i = 0; i < PER_T; ++i) {
            const int e = tid + i * NT, r = e / 4, k = (e % 4) * 4;
            voff[i] = r0 + r < rows ? (uint32_t)((r * ld + k) * 4) : kSplitOOB;
        }
    }

    // Loads and stores come in PARTS pieces, so that the splitting spreads over a slice's products.
    static constexpr int PARTS = PER_T;

    template <bool FULL>
    __device__ __forceinline__ void loadPart(int i, int k0, int kEnd, int tid) {
        const auto rs = bufferRsrc(tile + k0, kSplitView);
        if (FULL || k0 + Lds::BK <= kEnd) {
            v[i] = bufLoad4(rs, voff[i], 0);
        } else if (kEnd % 4 == 0) {   // whole vectors inside or past the end
            v[i] = bufLoad4(rs, k0 + ((tid + i * NT) % 4) * 4 < kEnd ? voff[i] : kSplitOOB, 0);
        } else {
            const int k = k0 + ((tid + i * NT) % 4) * 4;
#pragma unroll
            for (int j = 0; j < 4; ++j) v[i][j] = bufLoad1(rs, k + j < kEnd ? voff[i] + 4u * j : kSplitOOB, 0);
        }
    }

    __device__ __forceinline__ void storePart(int i, char* s, int tid) {
        const int e = tid + i * NT, r = e / 4, q = e % 4;
        u32x2 h, m, l;
        uint32_t a, b, c;
        splitPair(v[i][0], v[i][1], a, b, c);
        h[0] = a; m[0] = b; l[0] = c;
        splitPair(v[i][2], v[i][3], a, b, c);
        h[1] = a; m[1] = b; l[1] = c;
        char* d = s + (q >> 1) * Lds::GROUP + r * 16 + (q & 1) * 8;
        *reinterpret_cast<u32x2*>(d) = h;
        *reinterpret_cast<u32x2*>(d + Lds::PIECE) = m;
        *reinterpret_cast<u32x2*>(d + 2 * Lds::PIECE) = l;
    }

    template <bool FULL>
    __device__ __forceinline__ void load(int k0, int kEnd, int tid) {
#pragma unroll
        for (int i = 0; i < PARTS; ++i) loadPart<FULL>(i, k0, kEnd, tid);
    }
    __device__ __forceinline__ void store(char* s, int tid) {
#pragma unroll
        for (int i = 0; i < PARTS; ++i) storePart(i, s, tid);
    }
    // The slice as it is, for the fp32 MFMA: [R][16 + 4] (PLAIN_KMAJOR) or [16][R + 4].
    static constexpr bool PLAIN_KMAJOR = true;
    __device__ __forceinline__ void storePlain(float* s, int tid) const {
#pragma unroll
        for (int i = 0; i < PER_T; ++i) {
            const int e = tid + i * NT;
            *reinterpret_cast<f32x4*>(s + e / 4 * LdsShape<R, 16>::LD + e % 4 * 4) = v[i];
        }
    }
};

// Loader of an R-contiguous operand: element (r, k) at P[k * ld + r]. A thread
// owns one row r and KU consecutive k, loaded as single floats (a wave reads a
// contiguous run of each k row; no alignment needed), so the pieces pack along
// k without a transpose and leave as one 8- or 16-byte store each.
template <int R, int NT>
struct SplitLoaderR {
    static constexpr int KU = R * 16 / NT;
    static_assert(NT % R == 0 && (KU == 4 || KU == 8), "one unit of 4 or 8 k per thread");
    using Lds = SplitLds<R>;
    const float* tile;
    long long ld;
    uint32_t voff;
    float v[KU];
    uint32_t h[KU / 2], m[KU / 2], l[KU / 2];   // pieces of the unit being stored

    __device__ __forceinline__ void init(const float* p, long long ld_, int rows, int r0, int tid) {
        ld = ld_;
        tile = p + r0;
        const int r = tid % R, k = tid / R * KU;
        voff = r0 + r < rows ? (uint32_t)((k * ld + r) * 4) : kSplitOOB;
    }

    static constexpr int PARTS = KU / 4;   // four k each

    template <bool FULL>
    __device__ __forceinline__ void loadPart(int i, int k0, int kEnd, int tid) {
        const auto rs = bufferRsrc(tile + (long long)k0 * ld, kSplitView);
        // the k rows' offset is the scalar one: added to a marked row's kSplitOOB it would wrap into range
        const uint32_t step = (uint32_t)ld * 4u;
        if (FULL || k0 + Lds::BK <= kEnd) {
#pragma unroll
            for (int j = 4 * i; j < 4 * i + 4; ++j) v[j] = bufLoad1(rs, voff, j * step);
        } else {
            const int k = k0 + tid / R * KU;
#pragma unroll
            for (int j = 4 * i; j < 4 * i + 4; ++j) v[j] = bufLoad1(rs, k + j < kEnd ? voff : kSplitOOB, j * step);
        }
    }

    __device__ __forceinline__ void storePart(int i, char* s, int tid) {
        splitPair(v[4 * i], v[4 * i + 1], h[2 * i], m[2 * i], l[2 * i]);
        splitPair(v[4 * i + 2], v[4 * i + 3], h[2 * i + 1], m[2 * i + 1], l[2 * i + 1]);
        const int r = tid % R, u = tid / R;
        if constexpr (KU == 8) {
            if (i == 0) return;   // the unit leaves whole
            char* d = s + u * Lds::GROUP + r * 16;
            *reinterpret_cast<u32x4*>(d) = u32x4{h[0], h[1], h[2], h[3]};
            *reinterpret_cast<u32x4*>(d + Lds::PIECE) = u32x4{m[0], m[1], m[2], m[3]};
            *reinterpret_cast<u32x4*>(d + 2 * Lds::PIECE) = u32x4{l[0], l[1], l[2], l[3]};
        } else {
            char* d = s + (u >> 1) * Lds::GROUP + r * 16 + (u & 1) * 8;
            *reinterpret_cast<u32x2*>(d) = u32x2{h[0], h[1]};
            *reinterpret_cast<u32x2*>(d + Lds::PIECE) = u32x2{m[0], m[1]};
            *reinterpret_cast<u32x2*>(d + 2 * Lds::PIECE) = u32x2{l[0], l[1]};
        }
    }

    template <bool FULL>
    __device__ __forceinline__ void load(int k0, int kEnd, int tid) {
#pragma unroll
        for (int i = 0; i < PARTS; ++i) loadPart<FULL>(i, k0, kEnd, tid);
    }
    __device__ __forceinline__ void store(char* s, int tid) {
#pragma unroll
        for (int i = 0; i < PARTS; ++i) storePart(i, s, tid);
    }
    static constexpr bool PLAIN_KMAJOR = true;
    __device__ __forceinline__ void storePlain(float* s, int tid) const {
#pragma unroll
        for (int i = 0; i < PARTS; ++i)
            *reinterpret_cast<f32x4*>(s + tid % R * LdsShape<R, 16>::LD + tid / R * KU + 4 * i) =
                f32x4{v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]};
    }
};

// Loader of an R-contiguous operand for the fp32 MFMA whose row count is a
// multiple of four: four consecutive rows of one k in a 16-byte word (any 4-byte
// alignment), as they lie in memory.
template <int R, int NT>
struct PlainLoaderR {
    static constexpr int PER_T = R * 4 / NT;
    static_assert(R * 4 % NT == 0, "slice must divide over the threads");
    const float* tile;
    long long ld;
    uint32_t voff[PER_T];
    f32x4 v[PER_T];

    __device__ __forceinline__ void init(const float* p, long long ld_, int rows, int r0, int tid) {
        ld = ld_;
        tile = p + r0;
#pragma unroll
        for (int i = 0; i < PER_T; ++i) {
            const int e = tid + i * NT, r = e % (R / 4) * 4, k = e / (R / 4);
            voff[i] = r0 + r < rows ? (uint32_t)((k * ld + r) * 4) : kSplitOOB;
        }
    }
    template <bool FULL>
    __device__ __forceinline__ void load(int k0, int kEnd, int tid) {
        const auto rs = bufferRsrc(tile + (long long)k0 * ld, kSplitView);
#pragma unroll
        for (int i = 0; i < PER_T; ++i)
            v[i] = bufLoad4(rs, FULL || k0 + (tid + i * NT) / (R / 4) < kEnd ? voff[i] : kSplitOOB, 0);
    }
    static constexpr bool PLAIN_KMAJOR = false;
    __device__ __forceinline__ void storePlain(float* s, int tid) const {
#pragma unroll
        for (int i = 0; i < PER_T; ++i) {
            const int e = tid + i * NT;
            *reinterpret_cast<f32x4*>(s + e / (R / 4) * LdsShape<R, 16, false>::LD + e % (R / 4) * 4) = v[i];
        }
    }
};

// Loader of either layout by 64-bit addresses, one element at a time, for strides
// beyond the buffer views.
template <bool KMAJOR, int R, int NT>
struct FarLoader {
    static constexpr int KU = R * 16 / NT, UNITS = KU / 4;
    const float* tile;
    long long ld;
    int rowsLeft;
    f32x4 v[UNITS];

    // Row and first k of the thread's i-th four elements.
    static __device__ __forceinline__ int rowOf(int i, int tid) { return KMAJOR ? (tid + i * NT) / 4 : tid % R; }
    static __device__ __forceinline__ int kOf(int i, int tid) {
        return KMAJOR ? (tid + i * NT) % 4 * 4 : tid / R * KU + 4 * i;
    }

    __device__ __forceinline__ void init(const float* p, long long ld_, int rows, int r0, int) {
        ld = ld_;
        tile = KMAJOR ? p + r0 * ld : p + r0;
        rowsLeft = rows - r0;
    }
    template <bool FULL>
    __device__ __forceinline__ void load(int k0, int kEnd, int tid) {
#pragma unroll
        for (int i = 0; i < UNITS; ++i) {
            const int r = rowOf(i, tid);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int k = k0 + kOf(i, tid) + j;
                v[i][j] = r < rowsLeft && (FULL || k < kEnd) ? tile[KMAJOR ? r * ld + k : k * ld + r] : 0.f;
            }
        }
    }
    static constexpr bool PLAIN_KMAJOR = true;
    __device__ __forceinline__ void storePlain(float* s, int tid) const {
#pragma unroll
        for (int i = 0; i < UNITS; ++i)
            *reinterpret_cast<f32x4*>(s + rowOf(i, tid) * LdsShape<R, 16>::LD + kOf(i, tid)) = v[i];
    }
};

// Vector instructions of one loader part: two splitPair.
constexpr int kSideValu = 26;

template <bool KMAJOR, int R, int NT>
using SplitLoader = std::conditional_t<KMAJOR, SplitLoaderK<R, NT>, SplitLoaderR<R, NT>>;

// The fp32 MFMA's loaders. VEC: the rows of R-contiguous operands are multiples of four.
template <bool KMAJOR, int R, int NT, bool FAR, bool VEC>
using PlainLoader = std::conditional_t<FAR, FarLoader<KMAJOR, R, NT>,
                                       std::conditional_t<KMAJOR || !VEC, SplitLoader<KMAJOR, R, NT>, PlainLoaderR<R, NT>>>;

template <int R>
__device__ __forceinline__ void readSplit(const char* s, int row, int half, bf16x8 (&f)[3]) {
    const char* p = s + half * SplitLds<R>::GROUP + row * 16;
#pragma unroll
    for (int i = 0; i < 3; ++i) f[i] = *reinterpret_cast<const bf16x8*>(p + i * SplitLds<R>::PIECE);
}

// One 16-deep slice of a wave's WM x WN tile from LDS, a 32-column block of B
// at a time (its fragments are read while the block before is multiplied).
// side(i), i < SIDES, is work of the next slices that runs beside the products
// of column block i * FN / SIDES: splitting, LDS stores, global loads, at most
// SIDE_VALU vector instructions each. The schedule groups deal that work out
// between the MFMAs (issued together in front of them, as the compiler orders
// it by itself, it would leave the matrix cores idle), and the barriers keep
// each load right behind the split that frees its registers, a whole slice
// ahead of its use.
template <class Cfg, int SIDES, int SIDE_VALU, class Side>
__device__ __forceinline__ void mmaSplitSlice(const char* sA, const char* sB, f32x16 (&acc)[Cfg::FM][Cfg::FN], int wm,
                                              int wn, int lane, Side&& side) {
    const int li = lane & 31, h = lane >> 5;
    constexpr int P[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};
    constexpr int PER_FN = (SIDES + Cfg::FN - 1) / Cfg::FN;   // sides per column block
    constexpr int NV = (PER_FN * SIDE_VALU + 6 * Cfg::FM - 1) / (6 * Cfg::FM);   // their VALU per MFMA
    bf16x8 a[Cfg::FM][3], b[2][3];
#pragma unroll
    for (int fm = 0; fm < Cfg::FM; ++fm) readSplit<Cfg::BM>(sA, wm * Cfg::WM + fm * 32 + li, h, a[fm]);
    readSplit<Cfg::BN>(sB, wn * Cfg::WN + li, h, b[0]);
#pragma unroll
    for (int fn = 0; fn < Cfg::FN; ++fn) {
        if (fn + 1 < Cfg::FN) readSplit<Cfg::BN>(sB, wn * Cfg::WN + (fn + 1) * 32 + li, h, b[(fn + 1) & 1]);
#pragma unroll
        for (int i = fn * PER_FN; i < (fn + 1) * PER_FN; ++i)
            if (i < SIDES) side(i);
#pragma unroll
        for (int i = 0; i < 6; ++i)
#pragma unroll
            for (int fm = 0; fm < Cfg::FM; ++fm)
                acc[fm][fn] =
                    __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[fm][P[i][0]], b[fn & 1][P[i][1]], acc[fm][fn], 0, 0, 0);
        // fragment reads, then one MFMA and NV of the side's VALU at a time; the rest (LDS stores, loads) as it falls
        constexpr int HEAD_READS = 3 * Cfg::FM + (Cfg::FN > 1 ? 6 : 3);
        if (fn == 0) __builtin_amdgcn_sched_group_barrier(0x100, HEAD_READS, 0);
        else __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
#pragma unroll
        for (int i = 0; i < 6 * Cfg::FM; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, NV, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// SUB consecutive slices of a wave tile of one 32x32 block: every fragment is
// read first, so that only the first slice waits for LDS, and each slice's
// products have the sides of its own (side(u, i)) between them.
template <class Cfg, int SUB, int SIDES, int SIDE_VALU, class Side>
__device__ __forceinline__ void mmaSplitSub(const char* sA, const char* sB, int sliceBytes, f32x16& acc, int wm, int wn,
                                            int lane, Side&& side) {
    static_assert(Cfg::FM == 1 && Cfg::FN == 1, "one block per wave");
    const int li = lane & 31, h = lane >> 5;
    constexpr int P[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};
    constexpr int NV = (SIDES * SIDE_VALU + 5) / 6;
    bf16x8 a[SUB][3], b[SUB][3];
#pragma unroll
    for (int u = 0; u < SUB; ++u) {
        readSplit<Cfg::BM>(sA + u * sliceBytes, wm * Cfg::WM + li, h, a[u]);
        readSplit<Cfg::BN>(sB + u * sliceBytes, wn * Cfg::WN + li, h, b[u]);
    }
#pragma unroll
    for (int u = 0; u < SUB; ++u) {
#pragma unroll
        for (int i = 0; i < SIDES; ++i) side(u, i);
#pragma unroll
        for (int i = 0; i < 6; ++i)
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[u][P[i][0]], b[u][P[i][1]], acc, 0, 0, 0);
        if (u == 0) __builtin_amdgcn_sched_group_barrier(0x100, 6 * SUB, 0);
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, NV, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}

// Takes the scale off a lane's sums; whether any of them is not finite (0 * x
// is then NaN).
template <int FM, int FN>
__device__ __forceinline__ bool unscaleSums(f32x16 (&acc)[FM][FN]) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                s = __builtin_fmaf(acc[i][j][r], 0.f, s);
                acc[i][j][r] *= kSplitUnscale;
            }
    return !(s == 0.f);
}

}  // namespace omhip
