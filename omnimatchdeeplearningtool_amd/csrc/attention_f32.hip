// attention_f32.hip — the fp32 attention core of the engine's ViT branch in one kernel: split of the
// QKV projection into heads, Q * scale, scores, row softmax, P x V and the merge of the heads.
//
// Reference: MultiHeadAttention::forward (src/engine/om.engine.vit.ixx:150-239) and CPUBackend::softmax
// (src/hal/om.hal.cpu_backend.ixx:352-370).
//
// Composed of a scale pass and, per head, a product, a softmax and a product, ViT-B/16 at batch 16
// (197 tokens, 12 heads) took 37 launches of a few us each, 250 us, and passed the scores through
// memory four times; its 1.9 GFLOP are 12 us of fp32 MFMA. This kernel takes 32 us (few
// workgroups at hd 64: 4.6 us and 3.5 us more per 64 keys): 13 of each head's 16 wave slots hold queries and the
// MFMAs wait on the softmax of their own wave. LDS reads hoisted to the front of a trip spilled (82 against 50
// us), and context stores through a descriptor per lane were loops of one lane a turn (50 against 32 us; 16
// tokens 14 against 4.6 us). Here a workgroup of four waves holds 64
// queries of one head and walks the keys 64 at a time:
//  * K and V rows pass memory -> registers -> LDS, the next 64 keys loading under this 64's math;
//  * scores^T = K . Q^T with v_mfma_f32_16x16x4_f32. Lane (l16, g = lane / 16) supplies k = g of each
//    step; step (u, r) takes d = 16 u + 4 g + r, so both operands are read four d at a time. The lane
//    then holds the scores of query l16 with keys 16 t + 4 g + r;
//  * softmax with a running maximum: weights e = exp(s - max), earlier sums scaled when the maximum
//    grows. The weights carry a power of two below 1 / S, so that no sum of weights times V overflows
//    where the weighted mean does not;
//  * context^T = V^T . e^T: step (t, r) takes keys 16 t + 4 g + r, which is the weight the lane holds,
//    so the weights never leave their registers. The lane ends with four consecutive d of its query.
// LDS rows are 16 DT + 4 floats: 16 consecutive rows' 16-byte words (K) and rows 4 apart (V) fall on
// distinct banks.
#include "omhip_internal.hpp"
#include "buffer_io.hpp"
#include "mfma_f32_tile.hpp"
#include "attention_f32.hpp"

#include <cmath>
#include <type_traits>

namespace omhip {

namespace {

typedef uint32_t u32x4s __attribute__((ext_vector_type(4)));

constexpr int kKeys = 64;      // keys per trip
constexpr int kQueries = kAttnF32Queries;   // queries per workgroup, 16 per wave
constexpr int kThreads = 256;

struct AttnF32Params {
    const float* qkv;   // [B * S][3 * H * hd]
    float* out;         // [B * S][H * hd]
    int S, H, hd, qBlocks;
    long long ldq, ldo;
    float scale;
    float weightScale;  // a power of two, at most 1 / S
};

// Head dimension at most 16 * DT, a multiple of 4; elements past it read as zeros.
template <int DT>
__global__ __launch_bounds__(kThreads, DT <= 4 ? 3 : 2) void attention_f32_kernel(AttnF32Params p) {
    constexpr int DP = 16 * DT, LD = DP + 4, VECS = DP / 4, PER_T = kKeys * VECS / kThreads;
    static_assert(kKeys * VECS % kThreads == 0, "a tile divides over the threads");
    __shared__ __attribute__((aligned(16))) float sK[kKeys * LD];
    __shared__ __attribute__((aligned(16))) float sV[kKeys * LD];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, g = lane >> 4;
    // the query blocks of a head share an XCD's L2
    const int id = xcd_remap(blockIdx.x, gridDim.x);
    const int qb = id % p.qBlocks, bh = id / p.qBlocks, b = bh / p.H, h = bh % p.H;
    const float* const head = p.qkv + (long long)b * p.S * p.ldq + (long long)h * p.hd;
    const long long toK = (long long)p.H * p.hd;
    const uint32_t ldq4 = (uint32_t)p.ldq * 4u;
    const uint32_t rowBytes = (uint32_t)p.hd * 4u;

    // A view covers one tile's rows from their first to the last element of the last row inside S.
    auto view = [&](const float* base, int row0) {
        const int rows = min(kKeys, p.S - row0);
        return bufferRsrc(base + (long long)row0 * p.ldq, (uint32_t)(rows - 1) * ldq4 + rowBytes);
    };
    f32x4 q[DT];
    {
        const auto r = view(head, qb * kQueries);
        const int row = wave * 16 + l16;
        const bool ok = qb * kQueries + row < p.S;
#pragma unroll
        for (int u = 0; u < DT; ++u) {
            const int d = 16 * u + 4 * g;
            q[u] = bufLoad4(r, ok && d < p.hd ? row * ldq4 + d * 4u : kOOB, 0) * p.scale;
        }
    }

    f32x4 rk[PER_T], rv[PER_T];
    auto load = [&](int key0) {
        const auto vk = view(head + toK, key0), vv = view(head + 2 * toK, key0);
        const int rows = p.S - key0;
#pragma unroll
        for (int i = 0; i < PER_T; ++i) {
            const int e = tid + i * kThreads, row = e / VECS, d = e % VECS * 4;
            const uint32_t off = row < rows && d < p.hd ? row * ldq4 + d * 4u : kOOB;
            rk[i] = bufLoad4(vk, off, 0);
            rv[i] = bufLoad4(vv, off, 0);
        }
    };

    f32x4 o[DT];
#pragma unroll
    for (int i = 0; i < DT; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, sum = 0.f;   // sum: this lane's keys only
    const bool active = qb * kQueries + wave * 16 < p.S;   // a wave past the last query only moves tiles
    // One trip over T blocks of 16 keys, `rows` of them real. The schedule barriers keep one step's LDS reads
    // in registers at a time: all hoisted to the front they cost 80 registers, a third of the resident waves.
    auto trip = [&](auto count, int rows) {
        constexpr int T = decltype(count)::value;
        f32x4 s[T];
#pragma unroll
        for (int t = 0; t < T; ++t) s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < DT; ++u) {
            f32x4 k[T];
#pragma unroll
            for (int t = 0; t < T; ++t) k[t] = *reinterpret_cast<const f32x4*>(sK + (16 * t + l16) * LD + 16 * u + 4 * g);
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int t = 0; t < T; ++t) s[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[t][r], q[u][r], s[t], 0, 0, 0);
            if (u & 1) __builtin_amdgcn_sched_barrier(0);
        }
        float top = m;
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (16 * t + 4 * g + r >= rows) s[t][r] = -INFINITY;
                top = fmaxf(top, s[t][r]);
            }
        top = fmaxf(top, __shfl_xor(top, 16, 64));
        top = fmaxf(top, __shfl_xor(top, 32, 64));
        const float base = top == -INFINITY ? 0.f : top;   // only -inf so far: weights 0, not NaN
        const float keep = expf(m - base);
        m = top;
        sum *= keep;
#pragma unroll
        for (int i = 0; i < DT; ++i) o[i] *= keep;
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                s[t][r] = expf(s[t][r] - base) * p.weightScale;
                sum += s[t][r];
            }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < T; ++t) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int i = 0; i < DT; ++i)
                    o[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(sV[(16 * t + 4 * g + r) * LD + 16 * i + l16], s[t][r], o[i],
                                                                0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    load(0);
    for (int key0 = 0; key0 < p.S; key0 += kKeys) {
#pragma unroll
        for (int i = 0; i < PER_T; ++i) {
            const int e = tid + i * kThreads, at = e / VECS * LD + e % VECS * 4;
            *reinterpret_cast<f32x4*>(sK + at) = rk[i];
            *reinterpret_cast<f32x4*>(sV + at) = rv[i];
        }
        __syncthreads();
        if (key0 + kKeys < p.S) load(key0 + kKeys);
        if (active) {
            const int rows = p.S - key0;   // keys from here on
            if (rows > 48) trip(std::integral_constant<int, 4>{}, rows);
            else if (rows > 32) trip(std::integral_constant<int, 3>{}, rows);
            else if (rows > 16) trip(std::integral_constant<int, 2>{}, rows);
            else trip(std::integral_constant<int, 1>{}, rows);
        }
        __syncthreads();
    }
    if (!active) return;
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    // One view of the block's rows: a descriptor is uniform over a wave (from one per lane the compiler makes a
    // loop that stores a lane a turn).
    const int rows = min(kQueries, p.S - qb * kQueries), row = wave * 16 + l16;
    const uint32_t ldo4 = (uint32_t)p.ldo * 4u;
    const auto w = bufferRsrc(p.out + ((long long)b * p.S + qb * kQueries) * p.ldo + (long long)h * p.hd,
                              (uint32_t)(rows - 1) * ldo4 + rowBytes);
#pragma unroll
    for (int i = 0; i < DT; ++i) {
        const int d = 16 * i + 4 * g;
        const f32x4 v = o[i] / sum;
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4s, v), w,
                                               row < rows && d < p.hd ? row * ldo4 + d * 4u : kOOB, 0, 0);
    }
}

template <int DT>
int launchAttnF32(const AttnF32Params& p, int blocks) {
    hipLaunchKernelGGL(attention_f32_kernel<DT>, dim3(blocks), dim3(kThreads), 0, stream(), p);
    OMHIP_CHECK_LAUNCH();
    return 0;
}

}  // namespace

bool attentionF32Fits(int B, int S, int H, int hd) {
    const long long blocks = (long long)B * H * (((long long)S + kQueries - 1) / kQueries);
    // 16-byte loads of four d; a tile's rows in one buffer view
    return hd % 4 == 0 && hd <= kAttnF32MaxHeadDim && blocks <= 0x7fffffffLL &&
           3LL * H * hd * 4 * kKeys <= (long long)kMaxBufferBytes;
}

int attentionF32(const float* qkv, float* out, int B, int S, int H, int hd, float scale) {
    AttnF32Params p{};
    p.qkv = qkv;
    p.out = out;
    p.S = S;
    p.H = H;
    p.hd = hd;
    p.qBlocks = (int)(((long long)S + kQueries - 1) / kQueries);
    p.ldq = 3LL * H * hd;
    p.ldo = (long long)H * hd;
    p.scale = scale;
    p.weightScale = ldexpf(1.0f, -(S > 1 ? 32 - __builtin_clz((unsigned)(S - 1)) : 0));
    const int blocks = B * H * p.qBlocks;
    switch ((hd + 15) / 16) {
        case 1: return launchAttnF32<1>(p, blocks);
        case 2: return launchAttnF32<2>(p, blocks);
        case 3: return launchAttnF32<3>(p, blocks);
        case 4: return launchAttnF32<4>(p, blocks);
        case 5: return launchAttnF32<5>(p, blocks);
        case 6: return launchAttnF32<6>(p, blocks);
        case 7: return launchAttnF32<7>(p, blocks);
        default: return launchAttnF32<8>(p, blocks);
    }
}

}  // namespace omhip
