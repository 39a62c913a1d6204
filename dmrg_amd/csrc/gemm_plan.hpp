// Host side of the pipelined GEMM (gemm_pipe.hpp): its tile shapes, and the description of a GemmDesc for one of them.
#pragma once
#include "gemm_pipe.hpp"

#include <algorithm>

namespace dmrg {
namespace pipe {

constexpr uint32_t PLAIN = 0x7fffffffu;

// The same map over an extent, with a chunk only where it is one.
inline Idx2 normal(Idx2 x, int64_t ext) {
    if(x.c == 1) x = Idx2{x.s1, 0, PLAIN};
    if(ext <= static_cast<int64_t>(x.c) || x.s1 == x.s0 * static_cast<int64_t>(x.c)) x = Idx2{x.s0, 0, PLAIN};
    return x;
}
// umulhi(i, mul) >> sh = i / c for i < 2^31 and c > 1 (Granlund and Montgomery, Division by invariant integers using
// multiplication, 1994).
inline void magic(uint32_t c, uint32_t &mul, uint32_t &sh) {
    uint32_t l = 0;
    while((uint64_t(1) << l) < c) ++l;
    mul = static_cast<uint32_t>(((uint64_t(1) << (31 + l)) + c - 1) / c);
    sh  = l - 1;
}
// The largest offset of a map with non-negative strides over an extent.
inline int64_t span(const Idx2 &x, int64_t ext) {
    if(ext <= 0) return 0;
    return std::min<int64_t>(x.c - 1, ext - 1) * x.s0 + (ext - 1) / x.c * x.s1;
}

// Tile shapes per element type. Stages hold 4 KiB (32 rows) to 16 KiB per operand tile, so that two workgroups (two
// wavefronts per SIMD) or more fit a CU's 160 KiB of LDS; BK is at least two K positions of an MFMA fragment unit.
enum Shape { S128x64 = 0, S64x64 = 1, S64x32 = 2, S32x32 = 3, N_SHAPES = 4 };
struct ShapeInfo {
    int BM, BN, BK, NS, TM, TN, resident; // resident: workgroups a CU holds; BM = 0: no such shape for the type
};
inline ShapeInfo shape_info(dmrg_dtype t, Shape s) {
    static const ShapeInfo none{0, 0, 0, 0, 0, 0, 0};
    switch(t) {
        case DMRG_FP64: {
            static const ShapeInfo v[] = {{128, 64, 16, 3, 4, 2, 2}, {64, 64, 16, 4, 2, 2, 2}, {64, 32, 16, 4, 2, 1, 3}, {32, 32, 16, 4, 1, 1, 5}};
            return v[s];
        }
        case DMRG_CX64: {
            static const ShapeInfo v[] = {none, {64, 64, 8, 4, 2, 2, 2}, {64, 32, 16, 3, 2, 1, 2}, {32, 32, 8, 4, 1, 1, 4}};
            return v[s];
        }
        case DMRG_FP32: {
            static const ShapeInfo v[] = {none, {64, 64, 32, 4, 2, 2, 2}, none, {32, 32, 32, 4, 1, 1, 5}};
            return v[s];
        }
        case DMRG_CX32: {
            static const ShapeInfo v[] = {none, {64, 64, 16, 4, 2, 2, 2}, {64, 32, 16, 4, 2, 1, 3}, {32, 32, 16, 4, 1, 1, 5}};
            return v[s];
        }
    }
    return none;
}

struct Launch {
    Desc d;
    bool ar, br; // orientation of A's and B's units
    int  W;      // bytes per lane and load
};
// Describes g (already oriented: consecutive m should be consecutive in C) for a tile shape; false where the pipelined
// kernel does not take it (negative strides, K chunks that differ between the operands, operand tiles spanning 2 GiB).
// k_units: units along K only, as grouped launches take them.
bool describe(const GemmDesc &g, const ShapeInfo &s, int ksplit, Launch &out, bool k_units = false);
// Bytes per lane and load that describe would give g (4 where it refuses), at a fraction of its time.
int load_bytes(const GemmDesc &g, const ShapeInfo &s);
// Launches on the grid of l.d.
void launch_f64(const Launch &l, Shape s, dim3 grid, hipStream_t st);
void launch_c128(const Launch &l, Shape s, dim3 grid, hipStream_t st);
void launch_f32(const Launch &l, Shape s, dim3 grid, hipStream_t st);
void launch_c64(const Launch &l, Shape s, dim3 grid, hipStream_t st);

// Grouped launches: n descriptions and n + 1 tile offsets in device memory.
void launch_grouped_f64(const Desc *d, const int *start, int n, int tiles, Shape s, hipStream_t st);
void launch_grouped_c128(const Desc *d, const int *start, int n, int tiles, Shape s, hipStream_t st);
void launch_grouped_f32(const Desc *d, const int *start, int n, int tiles, Shape s, hipStream_t st);
void launch_grouped_c64(const Desc *d, const int *start, int n, int tiles, Shape s, hipStream_t st);

template <typename R, bool CPLX, int BM, int BN, int BK, int WM, int WN, int NS>
void launch_grouped_shape(const Desc *d, const int *start, int n, int tiles, hipStream_t st) {
    hipLaunchKernelGGL((grouped_kernel<R, CPLX, BM, BN, BK, WM, WN, NS>), dim3(tiles), dim3(64 * WM * WN), 0, st, d, start, n);
}

template <typename R, bool CPLX, int BM, int BN, int BK, int WM, int WN, int NS>
void launch_shape(const Launch &l, dim3 grid, hipStream_t st) {
    using E             = std::conditional_t<CPLX, cpx<R>, R>;
    constexpr int  U    = 16 / static_cast<int>(sizeof(E));
    constexpr bool RA   = U > 1 && (BM / (16 * WM)) % U == 0, RB = U > 1 && (BN / (16 * WN)) % U == 0;
    const dim3     block(64 * WM * WN);
    if(l.W == 4) hipLaunchKernelGGL((kernel<R, CPLX, BM, BN, BK, WM, WN, NS, false, false, 4>), grid, block, 0, st, l.d);
    else if(!l.ar && !l.br) hipLaunchKernelGGL((kernel<R, CPLX, BM, BN, BK, WM, WN, NS, false, false, 16>), grid, block, 0, st, l.d);
    else if(l.ar && !l.br) {
        if constexpr(RA) hipLaunchKernelGGL((kernel<R, CPLX, BM, BN, BK, WM, WN, NS, true, false, 16>), grid, block, 0, st, l.d);
    } else if(!l.ar) {
        if constexpr(RB) hipLaunchKernelGGL((kernel<R, CPLX, BM, BN, BK, WM, WN, NS, false, true, 16>), grid, block, 0, st, l.d);
    } else {
        if constexpr(RA && RB) hipLaunchKernelGGL((kernel<R, CPLX, BM, BN, BK, WM, WN, NS, true, true, 16>), grid, block, 0, st, l.d);
    }
}

} // namespace pipe
} // namespace dmrg
