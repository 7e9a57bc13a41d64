// gemm_f32.hip — fp32 GEMM on gfx950 matrix cores: every product through its
// bf16 pieces (split_tile.hpp), with the fp32 MFMA for the data and strides
// that path does not take.
//
// Entry points: omHipMatmul / MatmulTransB / MatmulTransA / BatchedMatmul /
// BatchedMatmulTransB / GemmStridedBatched. They replace the reference's
// omCudaMatmul (src/cuda/cuda_kernels.cu:768-804) and omCudaBatchedMatmul
// (:843-878) and compute what CPUBackend::matmul / batchedMatmul compute
// (src/hal/om.hal.cpu_backend.ixx:239-286, :1520-1532); the transposed
// variants replace the reference's explicit transpose2d + matmul compositions
// (src/engine/om.engine.autograd.ixx:261-286).
#include "omhip_internal.hpp"
#include "mfma_f32_tile.hpp"
#include "split_tile.hpp"
#include "buffer_io.hpp"
#include "gemm_f32.hpp"
#include "../../include/omhip.h"

#include <algorithm>
#include <mutex>
#include <type_traits>

namespace omhip {

// Split-K arrival of one piece of a tile. The piece's accumulators go to its
// slot of ws in the tile's own register layout ([split][batch][tile] blocks of
// BM x BN floats, a lane's 16 values of a fragment as four 16-byte words), with
// device-coherent (sc1) stores; once every wave's stores have completed (each
// waits on its own, the block barrier orders them before the add), thread 0
// bumps the tile's counter. The piece that arrives last replaces acc by
// 0 + part 0 + part 1 + ... in split order (device-coherent loads, four splits
// in flight), resets the counter for the next launch and returns true; the
// others return false. The sum order does not depend on which piece arrives
// last, so the result is deterministic.
//
// Ordering. Every access to the exchanged data is an sc1 buffer access, the
// encoding of a monotonic agent-scope atomic load / store in the gfx942 /
// gfx950 memory model: it is performed at the device coherence point, past
// the per-XCD L2s. A piece's stores have completed there (vmcnt 0) before its
// counter add is issued, and the last piece's loads are issued after its add
// has returned, so they read every piece's data. An agent-scope release /
// acquire on the counter would add an L2 write-back (buffer_wbl2 sc1) to every
// arrival and an L2 invalidate (buffer_inv sc1) to the last one; both exist to
// make non-coherent (non-sc1) accesses visible, and none cross between the
// pieces here. Measured on MI355X, they cost 128 x 4096 x 4096 42.5 -> 52.6 us
// (release on the add and acquire in the last piece: 50.5) and 512^3 11.3 ->
// 13.6 us.
typedef uint32_t u32x4s __attribute__((ext_vector_type(4)));

template <class Cfg>
__device__ __forceinline__ bool splitArrive(const GemmF32Params& p, f32x16 (&acc)[Cfg::FM][Cfg::FN], float* smem,
                                            int lane, long long batch, int split, int bid) {
    constexpr int TILE = Cfg::BM * Cfg::BN;   // floats per tile and split
    constexpr int LANE_FLOATS = Cfg::FM * Cfg::FN * 16;
    const long long tiles = (long long)p.tilesM * p.tilesN * gridDim.z;
    const long long slot = batch * p.tilesM * p.tilesN + bid;
    // byte offset of this lane's first word in split 0's block of the tile
    const uint32_t laneOff = (uint32_t)((threadIdx.x >> 6) * 64 * LANE_FLOATS + lane * 4) * 4u;
    const auto rw = bufferRsrc(p.ws, (uint32_t)(tiles * p.splits * TILE * 4));
    const uint32_t own = (uint32_t)(((long long)split * tiles + slot) * TILE * 4);
#pragma unroll
    for (int fm = 0; fm < Cfg::FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < Cfg::FN; ++fn)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const f32x4 v = {acc[fm][fn][4 * q], acc[fm][fn][4 * q + 1], acc[fm][fn][4 * q + 2], acc[fm][fn][4 * q + 3]};
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4s, v), rw,
                                                       laneOff + (uint32_t)((fm * Cfg::FN + fn) * 4 + q) * 1024u, own,
                                                       kCpolAgent);
            }
    __builtin_amdgcn_s_waitcnt(0);   // this wave's partial stores have completed
    int* flag = reinterpret_cast<int*>(smem);
    __syncthreads();                 // every wave's have (and the LDS stages are free)
    unsigned* ctr = p.ctr + slot;
    if (threadIdx.x == 0)
        *flag = __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(p.splits - 1);
    __syncthreads();
    if (!*flag) return false;
#pragma unroll
    for (int fm = 0; fm < Cfg::FM; ++fm)
#pragma unroll
        for (int fn = 0; fn < Cfg::FN; ++fn)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[fm][fn][r] = 0.f;
    const uint32_t stride = (uint32_t)(tiles * TILE * 4);   // bytes from one split's block of the tile to the next
    const uint32_t base = (uint32_t)(slot * TILE * 4);
    for (int s0 = 0; s0 < p.splits; s0 += 4) {
        f32x4 w[4][Cfg::FM * Cfg::FN * 4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < Cfg::FM * Cfg::FN * 4; ++i)   // splits past the last are out of range: zero, no access
                w[j][i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                    rw, s0 + j < p.splits ? laneOff + (uint32_t)i * 1024u : kOOB,
                    splitPartOffset(s0 + j, p.splits, base, stride), kCpolAgent));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (s0 + j >= p.splits) break;
#pragma unroll
            for (int fm = 0; fm < Cfg::FM; ++fm)
#pragma unroll
                for (int fn = 0; fn < Cfg::FN; ++fn)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc[fm][fn][4 * q + e] += w[j][(fm * Cfg::FN + fn) * 4 + q][e];
        }
    }
    if (threadIdx.x == 0) __hip_atomic_store(ctr, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

// acc = op(A) * op(B) over [kBeg, kEnd) on the fp32 MFMA: the tiles whose
// operands the pieces cannot carry, and with FAR (64-bit addresses) strides
// beyond the buffer views. Two slices are in flight: while slice t is multiplied
// from LDS, slice t + 1, loaded one slice earlier, goes to the other stage and
// slice t + 2 is loaded. smem: two stages of both operands' slices. VEC: the row
// counts of the operands stored K first are multiples of four, and they are loaded
// four rows at a time (with a test per load instead, 448 of K took 12.2 us for 11.2).
template <class Cfg, bool TA, bool TB, bool FAR, bool VEC>
__device__ __forceinline__ void plainLoop(const GemmF32Params& p, float* smem, f32x16 (&acc)[Cfg::FM][Cfg::FN], int m0,
                                          int n0, long long batch, int kBeg, int kEnd, int wm, int wn, int lane,
                                          int tid) {
    using LA = PlainLoader<!TA, Cfg::BM, Cfg::NT, FAR, VEC>;
    using LB = PlainLoader<TB, Cfg::BN, Cfg::NT, FAR, VEC>;
    constexpr int OFF_B = LdsShape<Cfg::BM, 16, LA::PLAIN_KMAJOR>::SIZE;
    constexpr int STAGE = OFF_B + LdsShape<Cfg::BN, 16, LB::PLAIN_KMAJOR>::SIZE;
    LA la[2];
    LB lb[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        la[j].init(p.A + batch * p.sA, p.lda, p.M, m0, tid);
        lb[j].init(p.B + batch * p.sB, p.ldb, p.N, n0, tid);
    }
#pragma unroll
    for (int i = 0; i < Cfg::FM; ++i)
#pragma unroll
        for (int j = 0; j < Cfg::FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    const int nk = (kEnd - kBeg + 15) / 16, nFull = (kEnd - kBeg) / 16;
    la[0].template load<false>(kBeg, kEnd, tid);
    lb[0].template load<false>(kBeg, kEnd, tid);
    if (nk > 1) {
        la[1].template load<false>(kBeg + 16, kEnd, tid);
        lb[1].template load<false>(kBeg + 16, kEnd, tid);
    }
    la[0].storePlain(smem, tid);
    lb[0].storePlain(smem + OFF_B, tid);
    __syncthreads();
    // FULL: slices t + 1 and t + 2 exist and are whole
    auto step = [&](auto full, int t, int j) {
        constexpr bool FULL = decltype(full)::value;
        if (FULL || t + 2 < nk) {
            la[j].template load<FULL>(kBeg + (t + 2) * 16, kEnd, tid);
            lb[j].template load<FULL>(kBeg + (t + 2) * 16, kEnd, tid);
        }
        __builtin_amdgcn_sched_barrier(0);
        const float* cur = smem + j * STAGE;
        float* oth = smem + (j ^ 1) * STAGE;
        mma_slice_split<Cfg, LA::PLAIN_KMAJOR, LB::PLAIN_KMAJOR>(cur, cur + OFF_B, acc, wm, wn, lane, [&] {
            if (FULL || t + 1 < nk) {
                la[j ^ 1].storePlain(oth, tid);
                lb[j ^ 1].storePlain(oth + OFF_B, tid);
            }
        });
        __syncthreads();
    };
    int t = 0;
#pragma unroll 1
    for (; t + 3 < nFull; t += 2) {
        step(std::true_type{}, t, 0);
        step(std::true_type{}, t + 1, 1);
    }
#pragma unroll 1
    for (; t < nk; t += 2) {
        step(std::false_type{}, t, 0);
        if (t + 1 < nk) step(std::false_type{}, t + 1, 1);
    }
}

// 16-deep slices per LDS stage, and so per block barrier. The 64x64 tile has six
// MFMAs per wave and slice: with one slice per barrier their time is less than the
// fragment reads', the LDS stores' and the barrier's that every slice then waits for.
template <class Cfg>
constexpr int kSub = Cfg::FM * Cfg::FN == 1 ? 2 : 1;

template <class Cfg>
constexpr int kSliceBytes = SplitLds<Cfg::BM>::SIZE + SplitLds<Cfg::BN>::SIZE;

// The main loop of one tile: stage T & 1 (SUB slices) is multiplied from LDS
// while stage T + 1 goes from its registers to the other half of LDS and stage
// T + 2 is loaded.
template <class Cfg, bool TA, bool TB>
__device__ __forceinline__ void splitLoop(const GemmF32Params& p, char* smem, f32x16 (&acc)[Cfg::FM][Cfg::FN], int m0,
                                          int n0, long long batch, int kBeg, int kEnd, int wm, int wn, int lane,
                                          int tid) {
    constexpr int SUB = kSub<Cfg>, SLICE = kSliceBytes<Cfg>, STAGE = SUB * SLICE, OFF_B = SplitLds<Cfg::BM>::SIZE;
    using LA = SplitLoader<!TA, Cfg::BM, Cfg::NT>;
    using LB = SplitLoader<TB, Cfg::BN, Cfg::NT>;
    LA la[SUB];
    LB lb[SUB];
    la[0].init(p.A + batch * p.sA, p.lda, p.M, m0, tid);
    lb[0].init(p.B + batch * p.sB, p.ldb, p.N, n0, tid);
#pragma unroll
    for (int u = 1; u < SUB; ++u) {
        la[u] = la[0];
        lb[u] = lb[0];
    }
    const int nk = (kEnd - kBeg + 15) / 16, nFull = (kEnd - kBeg) / 16;
    const int nt = (nk + SUB - 1) / SUB;   // stages; slices past nk are loaded as zeros
    // FULL: stages T + 1 and T + 2 exist and are whole
    auto step = [&](auto full, int T, int j) {
        constexpr bool FULL = decltype(full)::value;
        const char* cur = smem + j * STAGE;
        char* oth = smem + (j ^ 1) * STAGE;
        const bool st = FULL || T + 1 < nt, ld = FULL || T + 2 < nt;
        auto side = [&](int u, int i) {
            const int k0 = kBeg + ((T + 2) * SUB + u) * 16;
            if (i < LA::PARTS) {
                if (st) la[u].storePart(i, oth + u * SLICE, tid);
                if (ld) la[u].template loadPart<FULL>(i, k0, kEnd, tid);
            } else {
                if (st) lb[u].storePart(i - LA::PARTS, oth + u * SLICE + OFF_B, tid);
                if (ld) lb[u].template loadPart<FULL>(i - LA::PARTS, k0, kEnd, tid);
            }
        };
        constexpr int SIDES = LA::PARTS + LB::PARTS;
        if constexpr (SUB > 1)
            mmaSplitSub<Cfg, SUB, SIDES, kSideValu>(cur, cur + OFF_B, SLICE, acc[0][0], wm, wn, lane, side);
        else
            mmaSplitSlice<Cfg, SIDES, kSideValu>(cur, cur + OFF_B, acc, wm, wn, lane, [&](int i) { side(0, i); });
        __syncthreads();
    };
    // Stages 0 and 1 are loaded together (one memory latency before the first products, not
    // two). The main loop's own first loads test nothing: its waits then count the same loads
    // on every path (after a guarded load the compiler waits for all of them on each trip).
    auto fill = [&](auto full) {
        constexpr bool FULL = decltype(full)::value;
        LA fa[SUB];
        LB fb[SUB];
#pragma unroll
        for (int u = 0; u < SUB; ++u) {
            fa[u] = la[0];
            fb[u] = lb[0];
            fa[u].template load<FULL>(kBeg + u * 16, kEnd, tid);
            fb[u].template load<FULL>(kBeg + u * 16, kEnd, tid);
        }
        if (FULL || nt > 1) {
#pragma unroll
            for (int u = 0; u < SUB; ++u) {
                la[u].template load<FULL>(kBeg + (SUB + u) * 16, kEnd, tid);
                lb[u].template load<FULL>(kBeg + (SUB + u) * 16, kEnd, tid);
            }
        }
#pragma unroll
        for (int u = 0; u < SUB; ++u) {
            fa[u].store(smem + u * SLICE, tid);
            fb[u].store(smem + u * SLICE + OFF_B, tid);
        }
        __syncthreads();
    };
    int T = 0;
    if (nFull >= 4 * SUB) {
        fill(std::true_type{});
        for (; (T + 4) * SUB <= nFull; T += 2) {
            step(std::true_type{}, T, 0);
            step(std::true_type{}, T + 1, 1);
        }
    } else {
        fill(std::false_type{});
    }
#pragma unroll 1
    for (; T < nt; T += 2) {
        step(std::false_type{}, T, 0);
        if (T + 1 < nt) step(std::false_type{}, T + 1, 1);
    }
}

// How a tile's products are computed: through the pieces, on the fp32 MFMA
// (smallTilePlain), or on the fp32 MFMA with 64-bit addresses (strides beyond
// the buffer views).
enum class Path { Pieces, Plain, Far };

// LDS: two stages of both operands' slices, as pieces or as they are; a tile of
// the pieces that is computed again uses its stages for the plain slices.
template <class Cfg, Path PATH>
constexpr size_t ldsBytes() {
    constexpr size_t plain = sizeof(float) * (LdsShape<Cfg::BM, 16>::SIZE + LdsShape<Cfg::BN, 16>::SIZE);
    static_assert(kSliceBytes<Cfg> >= plain);
    return 2 * (PATH == Path::Pieces ? kSub<Cfg> * kSliceBytes<Cfg> : plain);
}

// One output tile (bid: the tile's linear index, batch, split) of C =
// op(A) * op(B). GATE: each element of C is kept where p.gate (same shape, row
// stride p.ldg) is > 0 and set to 0 elsewhere (a ReLU's backward applied to the
// product). A tile in which any sum is not finite is computed again on the fp32
// MFMA, whole, so the last bits of its finite elements depend on such neighbours
// (and on which tile the plan chose); where all sums of a tile are finite, every
// tile adds a product's terms in the same order.
// Computing again costs that unit's time after the pieces', us, finite / one NaN
// element / all NaN: 4096^3 568 / 1465 / 1352 (952 on the fp32 MFMA alone), 2048^3
// 106 / 217 / 213, 128 x 4096 x 4096 41.6 / 55 / 64; 1024^3 runs on the fp32 MFMA
// anyway. Read from memory by each wave for its own block, without LDS, 4096^3 took
// 3385 and 5309.
template <class Cfg, bool TA, bool TB, Path PATH, bool GATE = false>
__device__ __forceinline__ void gemmF32Tile(const GemmF32Params& p, char* smem, int bid, long long batch, int split) {
    static_assert(Cfg::BK == 16, "one MFMA step per slice");
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / Cfg::WAVES_N;
    const int wn = wave % Cfg::WAVES_N;

    int tm, tn;
    tile_coords(bid, p.tilesM * p.tilesN, p.tilesM, p.tilesN, 8, tm, tn);
    const int m0 = tm * Cfg::BM;
    const int n0 = tn * Cfg::BN;
    // This split's K range; the loaders treat kEnd as the end of K.
    const int kBeg = split * p.kChunk;
    const int kEnd = min(p.K, kBeg + p.kChunk);

    f32x16 acc[Cfg::FM][Cfg::FN];
#pragma unroll
    for (int i = 0; i < Cfg::FM; ++i)
#pragma unroll
        for (int j = 0; j < Cfg::FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    // Small tiles (short main loops) load the epilogue's bias and gate values before the
    // first slice, so that their latency passes under the main loop instead of in front
    // of the C stores; the large tiles' registers are spoken for, and their main loops
    // are long, so they load the bias in the epilogue.
    constexpr bool PRE = Cfg::BM * Cfg::BN <= 128 * 128;
    float biasv[Cfg::FN];
    if constexpr (PRE) {
#pragma unroll
        for (int fn = 0; fn < Cfg::FN; ++fn) {
            const int col = n0 + wn * Cfg::WN + fn * 32 + (lane & 31);
            biasv[fn] = (p.bias && col < p.N) ? p.bias[col] : 0.f;
        }
    }
    static_assert(!GATE || PRE, "gated tiles prefetch their gate");
    float gatev[GATE ? Cfg::FM : 1][GATE ? Cfg::FN : 1][GATE ? 16 : 1];
    if constexpr (GATE) {
#pragma unroll
        for (int fm = 0; fm < Cfg::FM; ++fm)
#pragma unroll
            for (int fn = 0; fn < Cfg::FN; ++fn) {
                const int col = n0 + wn * Cfg::WN + fn * 32 + (lane & 31);
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int row = m0 + wm * Cfg::WM + fm * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                    gatev[fm][fn][r] = (row < p.M && col < p.N) ? p.gate[(long long)row * p.ldg + col] : 0.f;
                }
            }
    }

    auto plain = [&] {
        float* const s = reinterpret_cast<float*>(smem);
        if constexpr (PATH == Path::Far) {
            plainLoop<Cfg, TA, TB, true, false>(p, s, acc, m0, n0, batch, kBeg, kEnd, wm, wn, lane, tid);
        } else {
            if ((TA || !TB) && (!TA || p.M % 4 == 0) && (TB || p.N % 4 == 0))
                plainLoop<Cfg, TA, TB, false, true>(p, s, acc, m0, n0, batch, kBeg, kEnd, wm, wn, lane, tid);
            else
                plainLoop<Cfg, TA, TB, false, false>(p, s, acc, m0, n0, batch, kBeg, kEnd, wm, wn, lane, tid);
        }
    };
    if constexpr (PATH != Path::Pieces) {
        plain();
    } else {
        splitLoop<Cfg, TA, TB>(p, smem, acc, m0, n0, batch, kBeg, kEnd, wm, wn, lane, tid);
        int* const bad = reinterpret_cast<int*>(smem);   // a word per wave; the stages are free
        const bool mine = __any(unscaleSums(acc));
        if (lane == 0) bad[wave] = mine;
        __syncthreads();
        int any = 0;
#pragma unroll
        for (int w = 0; w < Cfg::NWAVES; ++w) any |= bad[w];
        // laid out behind the epilogue: a jump over its 600 instructions at the end of every tile cost
        // 1001 x 765 x 1537 TN 0.6 us of 29.8 (128 x 4096 x 4096 and 4096^3: nothing)
        if (__builtin_amdgcn_readfirstlane(any)) [[unlikely]] {
            __syncthreads();
            plain();
        }
    }

    const int li = lane & 31, h = lane >> 5;
    if constexpr (Cfg::BM * Cfg::BN <= 64 * 64) {   // the plans split K over the small tile only
        // Split-K: the last piece of the tile to arrive sums every piece's
        // partial product in split order and writes C.
        if (p.ws && !splitArrive<Cfg>(p, acc, reinterpret_cast<float*>(smem), lane, batch, split, bid)) return;
    }
    // A lane's 16 rows of a block are 8 (r / 4) + r % 4 past its first one: a wave-uniform
    // byte offset past its own. Rows and columns past the matrix get an offset out of the
    // view's range and store nothing. (Far: ldc may be beyond the view, 64-bit addresses.)
    float* C = p.C + batch * p.sC + (long long)m0 * p.ldc + n0;
    const auto rc = bufferRsrc(C, kSplitView);
    const bool bias = p.bias != nullptr;
    const bool relu = p.act == 1;
#pragma unroll
    for (int fm = 0; fm < Cfg::FM; ++fm) {
        const int rl = wm * Cfg::WM + fm * 32 + 4 * h;   // the lane's first row in the tile
        const int rowsLeft = p.M - m0 - wm * Cfg::WM - fm * 32;
#pragma unroll
        for (int fn = 0; fn < Cfg::FN; ++fn) {
            const int cl = wn * Cfg::WN + fn * 32 + li;
            const bool colOk = n0 + cl < p.N;
            float b = 0.f;
            if constexpr (PRE) b = biasv[fn];
            else b = bias && colOk ? p.bias[n0 + cl] : 0.f;
            const uint32_t voff = (uint32_t)((rl * p.ldc + cl) * 4);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int ro = 8 * (r >> 2) + (r & 3);
                float v = acc[fm][fn][r];
                if (bias) v += b;
                if (relu) v = v > 0.f ? v : 0.f;
                if constexpr (GATE) v = gatev[fm][fn][r] > 0.f ? v : 0.f;
                const bool in = colOk && m0 + rl + ro < p.M;
                if constexpr (PATH == Path::Far) {
                    if (in) C[(long long)(rl + ro) * p.ldc + cl] = v;
                } else {
                    bufStore1(rc, in ? voff : kSplitOOB, storeRowOffset(ro, rowsLeft, p.ldc), v);
                }
            }
        }
    }
}

template <class Cfg, bool TA, bool TB, Path PATH>
__global__ __launch_bounds__(Cfg::NT, 2) void gemm_f32_kernel(GemmF32Params p) {
    extern __shared__ __align__(16) char smem[];
    gemmF32Tile<Cfg, TA, TB, PATH>(p, smem, blockIdx.x, blockIdx.z, blockIdx.y);
}

template <class Cfg, bool TA, bool TB, Path PATH>
static int launchOne(const GemmF32Params& prm, int batch, int splits) {
    auto kern = gemm_f32_kernel<Cfg, TA, TB, PATH>;
    constexpr size_t lds = ldsBytes<Cfg, PATH>();
    OMHIP_CHECK(OMHIP_SET_MAX_DYNAMIC_LDS_ONCE(kern, lds));
    dim3 grid(prm.tilesM * prm.tilesN, splits, batch);
    hipLaunchKernelGGL(kern, grid, dim3(Cfg::NT), lds, stream(), prm);
    OMHIP_CHECK_LAUNCH();
    return 0;
}

// In-tile byte offsets of an operand's buffer view stay in range: R rows (at
// most `rows` of them exist) of a 16-deep slice.
static bool splitViewOk(bool kMajor, int R, int rows, long long ld) {
    const long long maxOff = kMajor ? ((long long)(std::min(R, rows) - 1) * ld + 16) * 4 : (15 * ld + R) * 4;
    return maxOff < (long long)kSplitView;
}

// The large tile runs 8 waves of 64 x 128 (two per SIMD, 128 accumulators
// each): while one wave splits its share of the next slice or waits on its
// fragment reads and the block barrier, the other keeps the matrix core busy.
// It is bound by power: 4096^3 takes 551-605 us (227-249 TFLOP/s = 1.36-1.50
// PFLOP/s of bf16 MFMA, what a library bf16 product of 8192^3 reaches on this
// card, 1.37); on the fp32 MFMA it took 951-961 us (0.92 of that unit's peak).
// Beside it: 8192^3 7.49 -> 4.74 ms, 3072^3 (128x128 tiles) 538 -> 345 us, 2048^3
// 135 -> 100 us, 1001 x 765 x 1537 (TN, odd rows) 38.4 -> 29.7 us.
using CfgL = TileCfg<256, 256, 16, 64, 128>;
using CfgM = TileCfg<128, 128, 16, 64, 64>;
using CfgS = TileCfg<64, 64, 16, 32, 32>;

template <class Cfg, bool TA, bool TB>
static int launchTile(GemmF32Params prm, int batch, int splits, bool plain) {
    prm.tilesM = (prm.M + Cfg::BM - 1) / Cfg::BM;
    prm.tilesN = (prm.N + Cfg::BN - 1) / Cfg::BN;
    if (splitViewOk(!TA, Cfg::BM, prm.M, prm.lda) && splitViewOk(TB, Cfg::BN, prm.N, prm.ldb) &&
        splitViewOk(true, Cfg::BM, prm.M, prm.ldc + Cfg::BN)) {
        if constexpr (Cfg::BM == CfgS::BM)
            if (plain) return launchOne<Cfg, TA, TB, Path::Plain>(prm, batch, splits);
        return launchOne<Cfg, TA, TB, Path::Pieces>(prm, batch, splits);
    }
    prm.tilesM = (prm.M + CfgS::BM - 1) / CfgS::BM;
    prm.tilesN = (prm.N + CfgS::BN - 1) / CfgS::BN;
    return launchOne<CfgS, TA, TB, Path::Far>(prm, batch, splits);
}

// Tile and split-K choice (planGemmFor in gemm_f32.hpp) for this device.
static GemmPlan planGemm(bool ta, bool tb, int M, int N, int K, int batch, bool wsOk) {
    return planGemmFor(M, N, K, batch, wsOk, cuCount(), ta, tb);
}

template <bool TA, bool TB>
static int launchCfg(const GemmF32Params& prm, int batch, int splits, const GemmPlan& plan) {
    if (plan.cfg == 0) return launchTile<CfgL, TA, TB>(prm, batch, splits, false);
    if (plan.cfg == 1) return launchTile<CfgM, TA, TB>(prm, batch, splits, false);
    return launchTile<CfgS, TA, TB>(prm, batch, splits, plan.plain);
}

// Launches the GEMM (split-K: partials to ws, summed in the same launch by
// each tile's last piece).
static int gemmF32Run(bool ta, bool tb, int batch, int M, int N, int K, const float* A, long long lda, long long sA,
                      const float* B, long long ldb, long long sB, float* C, long long ldc, long long sC,
                      GemmPlan plan, const float* bias, int act, float* fixedWs = nullptr, size_t fixedBytes = 0) {
    GemmF32Params prm{};
    prm.A = A; prm.B = B; prm.C = C;
    prm.bias = bias; prm.act = act;
    prm.M = M; prm.N = N; prm.K = K;
    prm.lda = lda; prm.ldb = ldb; prm.ldc = ldc;
    prm.sA = sA; prm.sB = sB; prm.sC = sC;
    const int splits = splitPieces(K, plan.splits, &prm.kChunk);
    prm.splits = splits;
    if (splits > 1) {
        const size_t tiles = (size_t)((M + 63) / 64) * ((N + 63) / 64) * batch;   // the split plans' 64 x 64 tiles
        const size_t need = (size_t)splits * tiles * 64 * 64 * sizeof(float);
        if (need >= kMaxBufferBytes) return fail("gemm: %zu bytes of split-K partial products exceed 2^30", need);
        if (fixedWs) {
            if (need > fixedBytes - kNoAllocCounterBytes || tiles * sizeof(unsigned) > kNoAllocCounterBytes)
                return fail("gemm: %d split-K partial products need %zu bytes of scratch; the fixed scratch holds %zu",
                            splits, need, fixedBytes - kNoAllocCounterBytes);
            prm.ws = fixedWs;
            prm.ctr = reinterpret_cast<unsigned*>(reinterpret_cast<char*>(fixedWs) + fixedBytes - kNoAllocCounterBytes);
        } else {
            prm.ws = static_cast<float*>(workspace(need));
            if (!prm.ws) return -1;   // workspace() recorded the cause
            prm.ctr = static_cast<unsigned*>(workspace(tiles * sizeof(unsigned), kWsCounters));
            if (!prm.ctr) return -1;
        }
    }
    int rc;
    if (!ta && !tb) rc = launchCfg<false, false>(prm, batch, splits, plan);
    else if (!ta && tb) rc = launchCfg<false, true>(prm, batch, splits, plan);
    else if (ta && !tb) rc = launchCfg<true, false>(prm, batch, splits, plan);
    else rc = launchCfg<true, true>(prm, batch, splits, plan);
    return rc;
}

// Split-K partials are kept to at most this many bytes of workspace.
constexpr size_t kMaxSplitWorkspace = (size_t)256 << 20;

int gemmF32(bool ta, bool tb, int batch, int M, int N, int K,
            const float* A, long long lda, long long sA,
            const float* B, long long ldb, long long sB,
            float* C, long long ldc, long long sC, const float* bias, int act) {
    const bool wsOk = (size_t)64 * batch * M * N * sizeof(float) <= kMaxSplitWorkspace;
    const GemmPlan plan = planGemm(ta, tb, M, N, K, batch, wsOk);
    return gemmF32Run(ta, tb, batch, M, N, K, A, lda, sA, B, ldb, sB, C, ldc, sC, plan, bias, act);
}

__global__ void zero_rows_kernel(float* C, int rows, int cols, long long ldc, long long sC) {
    const long long b = blockIdx.z;
    const long long n = (long long)rows * cols;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x) {
        const long long r = i / cols, c = i % cols;
        C[b * sC + r * ldc + c] = 0.f;
    }
}

// Degenerate shapes: C is zeroed when its extent is valid (cpu_backend.ixx:246-251).
int zeroOutput(float* C, int batch, int M, int N, long long ldc, long long sC) {
    if (!C || M <= 0 || N <= 0 || batch <= 0) return 0;
    const long long n = (long long)M * N;
    const int blocks = (int)std::min<long long>((n + 255) / 256, 4096);
    hipLaunchKernelGGL(zero_rows_kernel, dim3(blocks, 1, batch), dim3(256), 0, stream(), C, M, N, ldc, sC);
    OMHIP_CHECK_LAUNCH();
    return 0;
}

int gemmF32Checked(const char* name, bool ta, bool tb, int batch, int M, int N, int K,
                   const float* A, long long lda, long long sA,
                   const float* B, long long ldb, long long sB,
                   float* C, long long ldc, long long sC) {
    clearError();
    if (batch <= 0 || M <= 0 || N <= 0) return 0;
    if (!C) return fail("%s: null output", name);
    if (!A || !B || K <= 0) return zeroOutput(C, batch, M, N, ldc, sC);
    if (batch > 65535) return fail("%s: batch %d exceeds 65535", name, batch);
    return gemmF32(ta, tb, batch, M, N, K, A, lda, sA, B, ldb, sB, C, ldc, sC);
}

// ---- Linear backward in one launch -------------------------------------------
// Workgroups [0, tilesW) compute dW = X^T G over 64 x 64 tiles, the next tilesX
// dX = G W^T, kept where the gate is > 0 when one is given (GATE), and the last
// ones G's column sums into db, a thread per column. K is not split, so every
// element is the same sum, in the same order, as the separate products compute
// whenever they do not split K either (e.g. every layer of the 784-256-128-10
// MLP at batch 128).

// colSum[col] = the sum of column col of G [rows, cols], row after row from 0.
// Sixty-four rows are read at a time (each batch costs one memory latency: with
// sixteen the sums of 128 rows outlasted the product tiles) and then added in row
// order; rows past the end add -0.0f, which leaves every sum unchanged. The sums
// have workgroups of their own: a product tile that also added its columns took
// twice as long as its neighbours.
__device__ __forceinline__ void columnSum(const float* G, float* colSum, int rows, int cols, int col) {
    if (col >= cols) return;
    float s = 0.f;
    for (int k0 = 0; k0 < rows; k0 += 64) {
        float v[64];
#pragma unroll
        for (int k = 0; k < 64; ++k) v[k] = G[(long long)min(k0 + k, rows - 1) * cols + col];
#pragma unroll
        for (int k = 0; k < 64; ++k) s += k0 + k < rows ? v[k] : -0.0f;
    }
    colSum[col] = s;
}

constexpr int kSumCols = 64;   // columns per workgroup of the sums: many workgroups, one wave each

template <Path PATHW, Path PATHX, bool GATE>
__global__ __launch_bounds__(CfgS::NT) void linear_backward_kernel(GemmF32Params pw, GemmF32Params pa, int tilesW,
                                                                  int tilesX, float* db) {
    extern __shared__ __align__(16) char smem[];
    const int b = blockIdx.x;
    if (b < tilesW)
        gemmF32Tile<CfgS, true, false, PATHW>(pw, smem, b, 0, 0);
    else if (b < tilesW + tilesX)
        gemmF32Tile<CfgS, false, true, PATHX, GATE>(pa, smem, b - tilesW, 0, 0);
    else if (threadIdx.x < kSumCols)
        columnSum(pw.B, db, pw.K, pw.N, (b - tilesW - tilesX) * kSumCols + threadIdx.x);
}

template <Path PATHW, Path PATHX, bool GATE>
static int launchLinearBackward(const GemmF32Params& pw, const GemmF32Params& pa, int tilesW, int tilesX, float* db) {
    auto kern = linear_backward_kernel<PATHW, PATHX, GATE>;
    constexpr size_t lds = std::max(ldsBytes<CfgS, PATHW>(), ldsBytes<CfgS, PATHX>());
    OMHIP_CHECK(OMHIP_SET_MAX_DYNAMIC_LDS_ONCE(kern, lds));
    const int sums = db ? (pw.N + kSumCols - 1) / kSumCols : 0;
    hipLaunchKernelGGL(kern, dim3(tilesW + tilesX + sums), dim3(CfgS::NT), lds, stream(), pw, pa,
                       tilesW, tilesX, db);
    OMHIP_CHECK_LAUNCH();
    return 0;
}

static int linearBackward(const float* X, const float* G, const float* W, const float* gate, float* dW, float* db,
                          float* dX, int B, int I, int O) {
    GemmF32Params pw{}, pa{};
    // dW [I, O] = X^T G: A = X stored [K = B, M = I], B = G stored [K = B, N = O]
    pw.A = X; pw.B = G; pw.C = dW; pw.M = I; pw.N = O; pw.K = B;
    pw.lda = I; pw.ldb = O; pw.ldc = O; pw.kChunk = B;
    pw.tilesM = (I + CfgS::BM - 1) / CfgS::BM; pw.tilesN = (O + CfgS::BN - 1) / CfgS::BN;
    // dX [B, I] = G W^T: A = G stored [M = B, K = O], B = W stored [N = I, K = O]
    pa.A = G; pa.B = W; pa.C = dX; pa.M = B; pa.N = I; pa.K = O;
    pa.lda = O; pa.ldb = O; pa.ldc = I; pa.kChunk = O; pa.gate = gate; pa.ldg = I;
    pa.tilesM = (B + CfgS::BM - 1) / CfgS::BM; pa.tilesN = (I + CfgS::BN - 1) / CfgS::BN;
    const long long tilesW = (long long)pw.tilesM * pw.tilesN, tilesX = dX ? (long long)pa.tilesM * pa.tilesN : 0;
    if (tilesW + tilesX + (O + kSumCols - 1) / kSumCols > 0x7fffffffLL) return fail("omHipLinearBackward: %lld tiles exceed the grid", tilesW + tilesX);
    // X and G are walked along the batch, G and W along nOut
    const bool views = splitViewOk(false, CfgS::BM, I, I) && splitViewOk(false, CfgS::BN, O, O) &&
                       splitViewOk(true, CfgS::BM, B, O) && splitViewOk(true, CfgS::BN, I, O) &&
                       splitViewOk(true, CfgS::BM, B, I + CfgS::BN);
    auto launch = [&](auto w, auto x) {
        constexpr Path PW = decltype(w)::value, PX = decltype(x)::value;
        return gate ? launchLinearBackward<PW, PX, true>(pw, pa, (int)tilesW, (int)tilesX, db)
                    : launchLinearBackward<PW, PX, false>(pw, pa, (int)tilesW, (int)tilesX, db);
    };
    using Pieces = std::integral_constant<Path, Path::Pieces>;
    using Plain = std::integral_constant<Path, Path::Plain>;
    using Far = std::integral_constant<Path, Path::Far>;
    if (!views) return launch(Far{}, Far{});
    const bool plainW = smallTilePlain(tilesW, B, B, true, false, I % 4 || O % 4, cuCount()), plainX = !dX || smallTilePlain(tilesX, O, O, false, true, false, cuCount());
    if (plainW) return plainX ? launch(Plain{}, Plain{}) : launch(Plain{}, Pieces{});
    return plainX ? launch(Pieces{}, Plain{}) : launch(Pieces{}, Pieces{});
}

// ---- fixed scratch of the no-allocation entry ---------------------------------
// Split-K partial sums of omHipGemmStridedBatchedNoAlloc live in this array,
// so that entry never allocates. A plan splits K only over 64 x 64 tiles and
// only while the grid holds fewer than 2 x CUs workgroups, and stops doubling
// the split count once it has reached them, so its partials cover fewer than
// 4 x CUs tiles of 64 x 64 floats: 16 MiB on a 256-CU device (the array holds
// twice that). Each device the library runs on holds its own copy until the
// process ends.
constexpr int kMaxDevices = 64;
static __device__ __align__(256) float scratch[kNoAllocScratchBytes / sizeof(float)];

static std::once_flag g_scratchOnce[kMaxDevices];
static float* g_scratchPtr[kMaxDevices];
static hipError_t g_scratchErr[kMaxDevices];
// Ordering of the calls that use a device's array: the stream of the last such
// call and an event recorded after its kernels. A call on another stream first
// makes its stream wait for that event (no host wait, no device memory).
static std::mutex g_scratchMutex[kMaxDevices];
static hipEvent_t g_scratchEvent[kMaxDevices];
static hipStream_t g_scratchLast[kMaxDevices];
static bool g_scratchRecorded[kMaxDevices];

// Device address of this device's `scratch` (the array's name is a host-side
// stand-in), looked up once per device with that device current.
static float* noAllocScratch() {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) {
        (void)fail("no-allocation GEMM: hipGetDevice: %s", hipGetErrorString(hipGetLastError()));
        return nullptr;
    }
    if (dev < 0 || dev >= kMaxDevices) {
        (void)fail("no-allocation GEMM: device %d beyond the %d supported", dev, kMaxDevices);
        return nullptr;
    }
    std::call_once(g_scratchOnce[dev], [dev] {
        void* ptr = nullptr;
        g_scratchErr[dev] = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        g_scratchPtr[dev] = g_scratchErr[dev] == hipSuccess ? static_cast<float*>(ptr) : nullptr;
    });
    if (!g_scratchPtr[dev]) {
        (void)fail("no-allocation GEMM: hipGetSymbolAddress(scratch): %s", hipGetErrorString(g_scratchErr[dev]));
        return nullptr;
    }
    return g_scratchPtr[dev];
}

// Runs `launch` (kernels that use the device's array) ordered after the last
// call that used it, whatever stream that call ran on. A stream that records a
// graph neither waits nor records: ordering a replay against other streams is
// the caller's.
template <class F>
static int withScratchOrder(F&& launch) {
    int dev = 0;
    OMHIP_CHECK(hipGetDevice(&dev));
    const hipStream_t s = stream();
    if (capturing(s)) return launch();
    std::lock_guard<std::mutex> lock(g_scratchMutex[dev]);
    if (!g_scratchEvent[dev]) OMHIP_CHECK(hipEventCreateWithFlags(&g_scratchEvent[dev], hipEventDisableTiming));
    if (g_scratchRecorded[dev] && g_scratchLast[dev] != s) OMHIP_CHECK(hipStreamWaitEvent(s, g_scratchEvent[dev], 0));
    const int rc = launch();
    if (rc) return rc;
    OMHIP_CHECK(hipEventRecord(g_scratchEvent[dev], s));
    g_scratchLast[dev] = s;
    g_scratchRecorded[dev] = true;
    return 0;
}

}  // namespace omhip

using namespace omhip;

extern "C" {

int omHipMatmul(const float* pA, const float* pB, float* pC, int nM, int nK, int nN) {
    return gemmF32Checked("omHipMatmul", false, false, 1, nM, nN, nK, pA, nK, 0, pB, nN, 0, pC, nN, 0);
}

int omHipMatmulTransB(const float* pA, const float* pB, float* pC, int nM, int nK, int nN) {
    return gemmF32Checked("omHipMatmulTransB", false, true, 1, nM, nN, nK, pA, nK, 0, pB, nK, 0, pC, nN, 0);
}

int omHipMatmulTransA(const float* pA, const float* pB, float* pC, int nM, int nK, int nN) {
    return gemmF32Checked("omHipMatmulTransA", true, false, 1, nM, nN, nK, pA, nM, 0, pB, nN, 0, pC, nN, 0);
}

int omHipLinearBiasAct(const float* pA, const float* pW, const float* pBias, float* pOut, int nM, int nK, int nN,
                       int nAct) {
    clearError();
    if (nAct != 0 && nAct != 1) return fail("omHipLinearBiasAct: unknown activation %d", nAct);
    if (nM <= 0 || nN <= 0) return 0;
    if (!pOut) return fail("omHipLinearBiasAct: null output");
    if (!pA || !pW || nK <= 0) {
        // a product with no terms: act(0 + bias), as the unfused chain computes it
        if (zeroOutput(pOut, 1, nM, nN, nN, 0)) return -1;
        if (pBias && omHipAddBias(pOut, pBias, pOut, nM, nN, 1)) return -1;
        if (nAct == 1) {
            // omHipReLU takes an int count: walk M*N (up to 2^62 elements) in 2^30 pieces
            const long long total = (long long)nM * nN;
            for (long long off = 0; off < total; off += 1LL << 30)
                if (omHipReLU(pOut + off, pOut + off, (int)std::min(total - off, 1LL << 30))) return -1;
        }
        return 0;
    }
    return gemmF32(false, false, 1, nM, nN, nK, pA, nK, 0, pW, nN, 0, pOut, nN, 0, pBias, nAct);
}

int omHipLinearBackward(const float* pInput, const float* pGradOut, const float* pWeight, const float* pGate,
                        float* pGradWeight, float* pGradBias, float* pGradInput, int nBatch, int nIn, int nOut) {
    clearError();
    if (nBatch < 0 || nIn < 0 || nOut < 0) return fail("omHipLinearBackward: negative size");
    if (!pGradWeight && nIn > 0 && nOut > 0) return fail("omHipLinearBackward: null weight gradient");
    if (pGradInput && nBatch > 0 && nIn > 0 && nOut > 0 && !pWeight) return fail("omHipLinearBackward: null weight");
    if (nBatch == 0 || nIn == 0 || nOut == 0 || !pInput || !pGradOut) {
        // some product has no terms or no elements: the separate entries, whose degenerate cases match the chain's
        if (omHipMatmulTransA(pInput, pGradOut, pGradWeight, nIn, nBatch, nOut)) return -1;
        if (pGradBias && omHipAddBiasBackward(pGradOut, pGradBias, nBatch, nOut, 1)) return -1;
        if (pGradInput) {
            if (omHipMatmulTransB(pGradOut, pWeight, pGradInput, nBatch, nOut, nIn)) return -1;
            if (pGate) {
                const long long total = (long long)nBatch * nIn;
                for (long long off = 0; off < total; off += 1LL << 30)
                    if (omHipReLUBackward(pGate + off, pGradInput + off, pGradInput + off,
                                          (int)std::min(total - off, 1LL << 30)))
                        return -1;
            }
        }
        return 0;
    }
    return linearBackward(pInput, pGradOut, pWeight, pGate, pGradWeight, pGradBias, pGradInput, nBatch, nIn, nOut);
}

int omHipBatchedMatmul(const float* pA, const float* pB, float* pC, int nBatch, int nM, int nK, int nN) {
    return gemmF32Checked("omHipBatchedMatmul", false, false, nBatch, nM, nN, nK,
                          pA, nK, (long long)nM * nK, pB, nN, (long long)nK * nN, pC, nN, (long long)nM * nN);
}

int omHipBatchedMatmulTransB(const float* pA, const float* pB, float* pC, int nBatch, int nM, int nK, int nN) {
    return gemmF32Checked("omHipBatchedMatmulTransB", false, true, nBatch, nM, nN, nK,
                          pA, nK, (long long)nM * nK, pB, nK, (long long)nN * nK, pC, nN, (long long)nM * nN);
}

int omHipGemmStridedBatched(int bTransA, int bTransB, int nBatch, int nM, int nN, int nK,
                            const float* pA, long long nLda, long long nStrideA,
                            const float* pB, long long nLdb, long long nStrideB,
                            float* pC, long long nLdc, long long nStrideC) {
    clearError();
    if (nBatch > 0 && nM > 0 && nN > 0 && nK > 0) {
        if (nLda < (bTransA ? nM : nK) || nLdb < (bTransB ? nK : nN) || nLdc < nN)
            return fail("omHipGemmStridedBatched: leading dimension smaller than the row length");
        if (nStrideA < 0 || nStrideB < 0 || nStrideC < 0)
            return fail("omHipGemmStridedBatched: negative batch stride");
    }
    return gemmF32Checked("omHipGemmStridedBatched", bTransA != 0, bTransB != 0, nBatch, nM, nN, nK,
                          pA, nLda, nStrideA, pB, nLdb, nStrideB, pC, nLdc, nStrideC);
}

int omHipGemmStridedBatchedNoAlloc(int bTransA, int bTransB, int nBatch, int nM, int nN, int nK,
                                   const float* pA, long long nLda, long long nStrideA,
                                   const float* pB, long long nLdb, long long nStrideB,
                                   float* pC, long long nLdc, long long nStrideC) {
    clearError();
    const char* name = "omHipGemmStridedBatchedNoAlloc";
    if (nBatch <= 0 || nM <= 0 || nN <= 0) return 0;
    if (!pC) return fail("%s: null output", name);
    if (nK > 0 && pA && pB) {
        if (nLda < (bTransA ? nM : nK) || nLdb < (bTransB ? nK : nN) || nLdc < nN)
            return fail("%s: leading dimension smaller than the row length", name);
        if (nStrideA < 0 || nStrideB < 0 || nStrideC < 0) return fail("%s: negative batch stride", name);
    }
    if (!pA || !pB || nK <= 0) return zeroOutput(pC, nBatch, nM, nN, nLdc, nStrideC);
    if (nBatch > 65535) return fail("%s: batch %d exceeds 65535", name, nBatch);
    float* ws = noAllocScratch();
    if (!ws) return -1;
    // the same plan as omHipGemmStridedBatched, so the results are the same bits
    const bool wsOk = (size_t)64 * nBatch * nM * nN * sizeof(float) <= kMaxSplitWorkspace;
    const GemmPlan plan = planGemm(bTransA != 0, bTransB != 0, nM, nN, nK, nBatch, wsOk);
    auto run = [&] {
        return gemmF32Run(bTransA != 0, bTransB != 0, nBatch, nM, nN, nK, pA, nLda, nStrideA, pB, nLdb, nStrideB, pC,
                          nLdc, nStrideC, plan, nullptr, 0, ws, kNoAllocScratchBytes);
    };
    if (plan.splits <= 1) return run();   // the array is not touched
    return withScratchOrder(run);
}

}  // extern "C"
