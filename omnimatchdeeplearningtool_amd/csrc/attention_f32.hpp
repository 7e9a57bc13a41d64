// attention_f32.hpp — host-side interface of the fused fp32 attention core.
#pragma once

namespace omhip {

constexpr int kAttnF32MaxHeadDim = 128;

// Whether the fused kernel takes these sizes: head dimensions that are multiples of 4 up to 128 (its
// accumulators are registers), rows whose 64-key tiles fit a buffer view, and up to 512 tokens or a
// workgroup for every CU.
bool attentionF32Fits(int B, int S, int H, int hd);

// out [B * S][H * hd] = softmax(scale Q K^T) V per head of qkv [B * S][3 * H * hd]. Enqueues on the
// library stream; 0 or -1.
int attentionF32(const float* qkv, float* out, int B, int S, int H, int hd, float scale);

}  // namespace omhip
