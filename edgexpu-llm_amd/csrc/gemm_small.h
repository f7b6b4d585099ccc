// Activation-pack geometry of the few-token GEMM (gemm_small.hip).
#pragma once

namespace exq {
constexpr int kSmPackK = 4096 + 512 + 64;  // codes, 16-element sums, scales of (super-block, 16 tokens)
constexpr int kSmPack0 = 1024 + 128;       // codes and scales of (pair of 32-element blocks, 16 tokens)
}  // namespace exq
