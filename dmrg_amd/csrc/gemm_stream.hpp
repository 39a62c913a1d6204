// Streaming GEMM for tiny K and M and many columns (gemm_stream.hip).
#pragma once
#include "common.hpp"

namespace dmrg {
namespace stream {
constexpr int MAX_K = 64, MAX_M = 64;

struct Desc {
    const void *A, *B;
    void       *C;
    Idx2        am, ak;                 // element strides
    int64_t     a_batch, b_batch, c_batch; // bytes for b_batch, elements otherwise
    Idx2        bk, bn;                 // byte strides
    Idx2        cm, cn;                 // element strides
    uint32_t    nmul, nsh, cmul, csh;   // i / bn.c and i / cn.c for i < 2^31
    uint32_t    mmul, msh, kmul, ksh, qmul, qsh; // i / am.c, i / ak.c and i / (K steps)
    int32_t     M, N, K, blocks, per_wave;
    float       sa, sb;                 // -1: conjugate
};

// Whether the kernel takes g: K and M in range, no accumulation, B's offsets (non-negative) below 2 GiB.
bool takes(const GemmDesc &g);
void launch(const GemmDesc &g, int cus, hipStream_t s);
// Grouped launches: each GEMM's description (its columns cut for about `waves` wavefronts), the workgroups it takes and the
// LDS it needs; n descriptions and n + 1 workgroup offsets in device memory, max_k and lds the largest of the group.
Desc   describe(const GemmDesc &g, int64_t waves);
int    workgroups(const Desc &d);
size_t lds_bytes(const GemmDesc &g);
void   launch_grouped(dmrg_dtype t, const Desc *d, const int *start, int n, int groups, int max_k, size_t lds, hipStream_t s);
} // namespace stream
} // namespace dmrg
