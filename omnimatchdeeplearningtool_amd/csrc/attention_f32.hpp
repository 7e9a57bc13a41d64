// attention_f32.hpp — host-side interface of the fused fp32 attention core.
#pragma once

namespace omhip {

constexpr int kAttnF32MaxHeadDim = 128;
constexpr int kAttnF32Queries = 64;   // per workgroup; keys per trip as well

// Whether the fused kernel takes these sizes: head dimensions that are multiples of 4 up to 128 (its
// accumulators are registers) and rows whose 64-key tiles fit a buffer view.
bool attentionF32Fits(int B, int S, int H, int hd);

// Whether the fused kernel is the faster path. One workgroup walks all keys of its 64 queries alone, so its
// time is trips times a trip's (1.5 us at head dimension 16, 2.15 at 32, 3.5 at 64, 4.2 at 80, 6.3 at
// 128; 1.6 and 2.2 times that with two and three rounds of workgroups per CU). The composed path runs three
// launches for each of min(B, H) steps, which spread few heads over the whole card. Fitted to 746 sizes
// (1-8 images, 1-16 heads, 128-4096 tokens, head dimensions 16-128), us: 1 x 12 heads x 197 x 64 composed 23,
// fused 15; 1 x 3 x 384 x 64 23.9, 24.1; 1 x 3 x 512 x 64 25.0, 31.1; 1 x 12 x 512 x 64 35.2, 31.4; 1 x 1 x 2048 x 64 56,
// 116; 1 x 16 x 2048 x 64 407, 187; 2 x 3 x 1024 x 64 79, 60. On average the choice costs 0.35 % over the better
// path of each size, 28 % at worst.
constexpr bool attentionF32Faster(int B, int S, int H, int hd, long long cus) {
    const long long trips = ((long long)S + kAttnF32Queries - 1) / kAttnF32Queries;
    const long long rounds = ((long long)B * H * trips + cus - 1) / cus;
    const double steps = B < H ? B : H, perStep = B < H ? H : B, s = S;
    const double fused = (double)trips * (0.75 + 0.043 * hd) * (0.38 + 0.62 * (double)rounds);
    const double composed = steps * (9.0 + 0.0165 * s + 5e-6 * perStep * s * s);
    return fused <= composed;
}

// out [B * S][H * hd] = softmax(scale Q K^T) V per head of qkv [B * S][3 * H * hd]. Enqueues on the
// library stream; 0 or -1.
int attentionF32(const float* qkv, float* out, int B, int S, int H, int hd, float scale);

}  // namespace omhip
