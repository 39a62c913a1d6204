// Streaming GEMM for tiny K and M and many columns (gemm_stream.hip).
#pragma once
#include "common.hpp"

namespace dmrg {
namespace stream {
constexpr int MAX_K = 64, MAX_M = 64;
// Whether the kernel takes g: K and M in range, no accumulation, B's offsets (non-negative) below 2 GiB.
bool takes(const GemmDesc &g);
void launch(const GemmDesc &g, int cus, hipStream_t s);
} // namespace stream
} // namespace dmrg
