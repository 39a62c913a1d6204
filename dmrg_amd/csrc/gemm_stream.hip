// Streaming GEMM for K and M of at most 64 and many columns, such as the MPO leg of a matvec or an environment update
// (K = d D, M = d D', N = chi chi'):  C[b][m,n] = sum_k op(A)[b][m,k] op(B)[b][k,n].
//
// Bound by HBM: every element of B is read and every element of C written once, and the matrix cores need a quarter to a
// half of that time. A wavefront takes 16 columns at a time straight from memory into the MFMA's operand layout (no LDS,
// no barrier; all of its K in flight at once), and walks over the 16-row blocks of A, whose fragments sit in LDS. Complex
// products take four real ones: there are matrix cores to spare, and the sums of the three-product form would cost
// accuracy in single precision and vector instructions.
//
// Measured (MI355X, us; before: 16x128 or 64x64 tiles, or one column per thread): 
// chi = 512, D = 5 (10x10 on 262144 columns) complex FP64 21.3 -> 16.9, FP32 18.2 -> 11.8 (among 200 matvecs in a row 16.0,
// 5.2 TB/s, the rate of a large copy, and 11.0);
// 173x211 complex 9.0 -> 5.9; D = 8, 8 vectors of 120x88 real 12.5 -> 7.4; chi = 24, D = 3 real 5.8 -> 3.4; D = 25 (50x50 on 32964
// columns) real 25.2 -> 16.2.
#include "gemm_plan.hpp"
#include "gemm_stream.hpp"

namespace dmrg {
namespace stream {
using pipe::magic;
using pipe::normal;
using pipe::span;

// MFMA steps over K, at least two (the divisions by multiplication below have no divisor 1).
__host__ __device__ inline int ksteps(int K) { return K <= 8 ? 2 : (K + 3) / 4; }

namespace {

template <typename R>
using acc_t = typename pipe::mma<R>::acc;

// Workgroup x of a GEMM, batch entry b. lds: A's fragments [16-row block][K step][lane], then the row offsets of C.
template <typename R, bool CPLX, int KST>
__device__ __forceinline__ void body(const Desc &g, int x, int b, char *lds) {
    using E  = std::conditional_t<CPLX, cpx<R>, R>;
    using MM = pipe::mma<R>;
    const int tid = threadIdx.x, lane = tid & 63, lg = lane >> 4, ll = lane & 15;
    const int mb = (g.M + 15) / 16, kst = ksteps(g.K);
    E        *fa   = reinterpret_cast<E *>(lds);
    int64_t  *coff = reinterpret_cast<int64_t *>(lds + static_cast<size_t>(mb) * kst * 64 * sizeof(E));
    const E  *A    = static_cast<const E *>(g.A) + b * g.a_batch;
    const int wave = static_cast<int>(pipe::uni(static_cast<uint32_t>(tid >> 6)));
    const int first = (x * 4 + wave) * g.per_wave, last = min(g.blocks, first + g.per_wave);

    const auto rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(static_cast<const char *>(g.B) + b * g.b_batch), static_cast<short>(0),
                                                      0x7fffffff, 0x00020000);
    uint32_t   kv[KST];
#pragma unroll
    for(int q = 0; q < KST; ++q) {
        const uint32_t k = 4 * q + lg;
        kv[q]            = k < static_cast<uint32_t>(g.K) ? (k % g.bk.c) * static_cast<uint32_t>(g.bk.s0) + (k / g.bk.c) * static_cast<uint32_t>(g.bk.s1) : pipe::OOB;
    }
    auto load = [&](int blk, E (&f)[KST]) { // columns [16 blk, 16 blk + 16); zeros outside the matrix
        const uint32_t n = 16 * blk + ll, d = __umulhi(n, g.nmul) >> g.nsh;
        const uint32_t v = (n - d * g.bn.c) * static_cast<uint32_t>(g.bn.s0) + d * static_cast<uint32_t>(g.bn.s1);
        const bool     in = n < static_cast<uint32_t>(g.N);
#pragma unroll
        for(int q = 0; q < KST; ++q) {
            const int o = static_cast<int>(in && kv[q] != pipe::OOB ? v + kv[q] : pipe::OOB);
            if constexpr(sizeof(E) == 16) f[q] = __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b128(rs, o, 0, 0));
            else if constexpr(sizeof(E) == 8) f[q] = __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b64(rs, o, 0, 0));
            else f[q] = __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b32(rs, o, 0, 0));
        }
    };
    E f[2][KST];
    if(first < last) load(first, f[0]); // in flight while A's fragments are laid out
    // Eight elements of A in flight per thread; one at a time, a 50 x 50 A took longer than its columns.
    auto off = [](const Idx2 &x, uint32_t mul, uint32_t sh, uint32_t i) {
        const uint32_t d = __umulhi(i, mul) >> sh;
        return static_cast<int64_t>(i - d * x.c) * x.s0 + static_cast<int64_t>(d) * x.s1;
    };
    auto element = [&](uint32_t i) {
        const uint32_t f = i >> 6, fm = __umulhi(f, g.qmul) >> g.qsh, m = fm * 16 + (i & 15), k = (f - fm * kst) * 4 + (i >> 4 & 3);
        E              v{};
        if(m < static_cast<uint32_t>(g.M) && k < static_cast<uint32_t>(g.K)) v = A[off(g.am, g.mmul, g.msh, m) + off(g.ak, g.kmul, g.ksh, k)];
        if constexpr(CPLX) v.im *= static_cast<R>(g.sa);
        return v;
    };
    const int total = mb * kst * 64;
    if(total <= 256) {
        if(tid < total) fa[tid] = element(tid);
    } else {
        for(int i0 = tid; i0 < total; i0 += 8 * 256) {
            E v[8];
#pragma unroll
            for(int u = 0; u < 8; ++u) v[u] = element(i0 + u * 256); // zeros past the last row block
#pragma unroll
            for(int u = 0; u < 8; ++u)
                if(i0 + u * 256 < total) fa[i0 + u * 256] = v[u];
        }
    }
    for(int m = tid; m < mb * 16; m += 256) coff[m] = idx_off(g.cm, static_cast<uint32_t>(m));
    __syncthreads();

    E *C = static_cast<E *>(g.C) + b * g.c_batch;
    for(int blk = first; blk < last; ++blk) {
        E(&cur)[KST] = f[0];
        if(blk + 1 < last) load(blk + 1, f[1]);
        const uint32_t n = 16 * blk + ll, d = __umulhi(n, g.cmul) >> g.csh;
        E             *col = C + static_cast<int64_t>(n - d * g.cn.c) * g.cn.s0 + static_cast<int64_t>(d) * g.cn.s1;
        for(int i = 0; i < mb; ++i) {
            acc_t<R> re{0, 0, 0, 0}, ii{0, 0, 0, 0}, im{0, 0, 0, 0};
            // Lane l: column l % 16 of B (n) and rows row(l / 16, v) of A's block (m).
#pragma unroll
            for(int q = 0; q < KST; ++q)
                if(q < kst) {
                    const E a = fa[(i * kst + q) * 64 + lane];
                    if constexpr(CPLX) {
                        re = MM::op(a.re, cur[q].re, re);
                        ii = MM::op(a.im, cur[q].im, ii);
                        im = MM::op(a.im, cur[q].re, im);
                    } else {
                        re = MM::op(a, cur[q], re);
                    }
                }
            if constexpr(CPLX) {
                acc_t<R> ri{0, 0, 0, 0};
#pragma unroll
                for(int q = 0; q < KST; ++q)
                    if(q < kst) ri = MM::op(fa[(i * kst + q) * 64 + lane].re, cur[q].im, ri);
                const R sb = static_cast<R>(g.sb);
#pragma unroll
                for(int v = 0; v < 4; ++v) {
                    const int m = i * 16 + MM::row(lg, v);
                    if(m < g.M && n < static_cast<uint32_t>(g.N)) col[coff[m]] = E{re[v] - sb * ii[v], im[v] + sb * ri[v]};
                }
            } else {
#pragma unroll
                for(int v = 0; v < 4; ++v) {
                    const int m = i * 16 + MM::row(lg, v);
                    if(m < g.M && n < static_cast<uint32_t>(g.N)) col[coff[m]] = re[v];
                }
            }
        }
#pragma unroll
        for(int q = 0; q < KST; ++q) f[0][q] = f[1][q];
    }
}

template <typename R, bool CPLX, int KST>
__global__ __launch_bounds__(256) void kernel(const Desc g) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    body<R, CPLX, KST>(g, blockIdx.x, blockIdx.y, lds);
}
// Several independent GEMMs in one launch; workgroup x belongs to the one whose range [start[i], start[i + 1]) holds x.
template <typename R, bool CPLX, int KST>
__global__ __launch_bounds__(256) void grouped_kernel(const Desc *descs, const int *start, int n) {
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int  i = pipe::group_of(start, n, blockIdx.x);
    const Desc g = descs[i];
    body<R, CPLX, KST>(g, blockIdx.x - start[i], 0, lds);
}

template <typename R, bool CPLX>
void run(const Desc &d, dim3 grid, size_t lds, hipStream_t s) {
    if(d.K <= 8) hipLaunchKernelGGL((kernel<R, CPLX, 2>), grid, dim3(256), lds, s, d);
    else if(d.K <= 12) hipLaunchKernelGGL((kernel<R, CPLX, 3>), grid, dim3(256), lds, s, d);
    else if(d.K <= 16) hipLaunchKernelGGL((kernel<R, CPLX, 4>), grid, dim3(256), lds, s, d);
    else if(d.K <= 32) hipLaunchKernelGGL((kernel<R, CPLX, 8>), grid, dim3(256), lds, s, d);
    else hipLaunchKernelGGL((kernel<R, CPLX, 16>), grid, dim3(256), lds, s, d);
}
template <typename R, bool CPLX>
void run_grouped(const Desc *d, const int *start, int n, int groups, int max_k, size_t lds, hipStream_t s) {
    const dim3 grid(groups), block(256);
    if(max_k <= 16) hipLaunchKernelGGL((grouped_kernel<R, CPLX, 4>), grid, block, lds, s, d, start, n);
    else if(max_k <= 32) hipLaunchKernelGGL((grouped_kernel<R, CPLX, 8>), grid, block, lds, s, d, start, n);
    else hipLaunchKernelGGL((grouped_kernel<R, CPLX, 16>), grid, block, lds, s, d, start, n);
}

} // namespace

size_t lds_bytes(const GemmDesc &g) {
    return static_cast<size_t>((g.M + 15) / 16) * (static_cast<size_t>(ksteps(g.K)) * 64 * dtype_size(g.dtype) + 16 * sizeof(int64_t));
}

bool takes(const GemmDesc &g) {
    if(g.K <= 0 || g.K > MAX_K || g.M > MAX_M || g.accumulate || lds_bytes(g) > 65536) return false;
    const int64_t es = static_cast<int64_t>(dtype_size(g.dtype));
    for(const Idx2 &x : {g.bk, g.bn})
        if(x.s0 < 0 || x.s1 < 0) return false;
    return (span(normal(g.bk, g.K), g.K) + span(normal(g.bn, g.N), g.N) + 1) * es < static_cast<int64_t>(0x7fffffff);
}

Desc describe(const GemmDesc &g, int64_t waves) {
    const int64_t es = static_cast<int64_t>(dtype_size(g.dtype));
    Desc          d;
    d.A = g.A, d.B = g.B, d.C = g.C;
    d.am = normal(g.am, g.M), d.ak = normal(g.ak, g.K);
    d.a_batch = g.a_batch, d.b_batch = g.b_batch * es, d.c_batch = g.c_batch;
    d.bk = normal(g.bk, g.K), d.bn = normal(g.bn, g.N);
    d.cm = g.cm, d.cn = normal(g.cn, g.N);
    magic(d.bn.c, d.nmul, d.nsh);
    magic(d.cn.c, d.cmul, d.csh);
    magic(d.am.c, d.mmul, d.msh);
    magic(d.ak.c, d.kmul, d.ksh);
    magic(static_cast<uint32_t>(ksteps(g.K)), d.qmul, d.qsh);
    d.bk.s0 *= es, d.bk.s1 *= es, d.bn.s0 *= es, d.bn.s1 *= es;
    d.M = g.M, d.N = g.N, d.K = g.K;
    d.sa = g.conjA ? -1.0f : 1.0f, d.sb = g.conjB ? -1.0f : 1.0f;
    d.blocks = (g.N + 15) / 16;
    d.per_wave          = static_cast<int32_t>(std::max<int64_t>(1, (static_cast<int64_t>(d.blocks) * g.batch + waves - 1) / waves));
    return d;
}
int workgroups(const Desc &d) { return (d.blocks + 4 * d.per_wave - 1) / (4 * d.per_wave); }

void launch(const GemmDesc &g, int cus, hipStream_t s) {
    // Enough workgroups to fill every CU with as many wavefronts as it holds, each wavefront walking consecutive columns.
    const Desc d = describe(g, static_cast<int64_t>(cus) * 16);
    const dim3 grid(static_cast<unsigned>(workgroups(d)), g.batch);
    const size_t lds = lds_bytes(g);
    switch(g.dtype) {
        case DMRG_FP64: run<double, false>(d, grid, lds, s); break;
        case DMRG_CX64: run<double, true>(d, grid, lds, s); break;
        case DMRG_FP32: run<float, false>(d, grid, lds, s); break;
        case DMRG_CX32: run<float, true>(d, grid, lds, s); break;
    }
    if(g.ev_after_main) DMRG_HIP_CHECK(hipEventRecord(static_cast<hipEvent_t>(g.ev_after_main), s));
}

void launch_grouped(dmrg_dtype t, const Desc *d, const int *start, int n, int groups, int max_k, size_t lds, hipStream_t s) {
    switch(t) {
        case DMRG_FP64: run_grouped<double, false>(d, start, n, groups, max_k, lds, s); break;
        case DMRG_CX64: run_grouped<double, true>(d, start, n, groups, max_k, lds, s); break;
        case DMRG_FP32: run_grouped<float, false>(d, start, n, groups, max_k, lds, s); break;
        case DMRG_CX32: run_grouped<float, true>(d, start, n, groups, max_k, lds, s); break;
    }
}

} // namespace stream
} // namespace dmrg
