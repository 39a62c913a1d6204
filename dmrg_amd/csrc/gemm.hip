// Generic batched GEMM on CDNA4 matrix cores (gfx950), FP64 and FP32, real and complex.
//
//   C[b][m,n] (+)= sum_k op(A)[b][m,k] * op(B)[b][k,n]
//
// Every operand index maps to memory through a two-level stride (Idx2), so the
// column-major tensors of the H_eff contraction (theta (d,chiL,chiR), env (chi,chi,D),
// MPO (DL,DR,d,d)) are read and written in place: no transposes or reshapes are
// materialised between the legs of a contraction.
//
// The GEMMs of the contractions run in the pipelined kernels of gemm_pipe.hpp. The kernel here stages tiles through
// registers (global -> registers -> LDS, double buffered, one barrier per K step; per-element 64-bit offsets where the
// index maps are not separable). It serves outputs of at most 16 rows that the streaming kernel (gemm_stream.hip) does not
// take, the block Jacobi steps, and single or grouped GEMMs whose index maps the pipelined kernels do not take. Each wave owns a (BM/WM) x (BN/WN) sub-tile of 16x16 blocks:
//   FP64: v_mfma_f64_16x16x4_f64,  FP32: v_mfma_f32_16x16x4_f32.
// Complex products use the 3-real-product (Gauss) form, 3 MFMAs per block per k-step:
//   P1 = sum ar br, P2 = sum ai bi, P3 = sum (ar + ai)(br + bi);  re = P1 - P2, im = P3 - P1 - P2.
// Its rounding error is bounded by a small multiple of eps * sum |a||b|, as for the 4-product form.
// The "swap" variant feeds B as the MFMA's first operand so that the lane index
// of the accumulator runs along M; it is picked when C is unit-stride in M, so
// the epilogue stores are coalesced either way.
#include "common.hpp"
#include "gemm_plan.hpp"
#include "gemm_stream.hpp"

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <type_traits>
#include <unordered_map>
#include <vector>

namespace dmrg {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float  v4f __attribute__((ext_vector_type(4)));

template <typename R>
struct mfma_t;
template <>
struct mfma_t<double> {
    using acc                                  = v4d;
    __device__ static inline acc op(double a, double b, acc c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
};
template <>
struct mfma_t<float> {
    using acc                                = v4f;
    __device__ static inline acc op(float a, float b, acc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
};

template <typename R, bool CPLX>
using elem_t = std::conditional_t<CPLX, cpx<R>, R>;

// LDS row padding (in elements) that makes the MFMA fragment reads conflict free:
// a fragment read puts 16 consecutive elements of one row on each group of 16 lanes;
// the groups that the LDS serves in one pass must land on disjoint bank ranges.
constexpr int lds_pad(int row_elems, int elem_bytes) {
    const int seg_bytes = 16 * elem_bytes;                 // bytes one 16-lane group reads
    const int groups    = seg_bytes >= 256 ? 1 : 256 / seg_bytes; // groups per 256-byte pass
    for(int p = 0; p <= 64; ++p) {
        const int row_bytes = (row_elems + p) * elem_bytes;
        if(row_bytes % 16 != 0 && elem_bytes >= 16) continue;
        bool ok = true;
        for(int g = 0; g < groups && ok; ++g)
            for(int h = 0; h < g && ok; ++h) {
                const int og = (g * row_bytes) % 256, oh = (h * row_bytes) % 256;
                const int d  = og > oh ? og - oh : oh - og;
                if(d < seg_bytes || 256 - d < seg_bytes) ok = false;
            }
        if(ok) return p;
    }
    return 0;
}

// LDS row pads (elements) per load direction. A tile stored [k][r] is written by lanes that walk r
// (operand contiguous along r: rows stay contiguous, the read-friendly pad applies) or k (operand contiguous
// along K: consecutive lanes write consecutive rows, so the row pitch must spread them over the banks).
// 16-byte elements: one pad of 1 serves both. The K-direction pads were chosen with a bank model of
// 64 banks x 4 bytes (and 32 x 4) over the fragment reads and the tile writes.
constexpr int pad_rfast(int row_elems, int elem_bytes) { return elem_bytes >= 16 ? 1 : lds_pad(row_elems, elem_bytes); }
constexpr int pad_kfast(int row_elems, int elem_bytes) { return (elem_bytes == 4 && row_elems >= 64) ? 9 : 1; }
constexpr int imax(int a, int b) { return a > b ? a : b; }

template <typename E>
__device__ inline E zero_elem() {
    if constexpr(std::is_same_v<E, cpx<double>> || std::is_same_v<E, cpx<float>>) return E{0, 0};
    else return E(0);
}

// Element loads that never wait: the aligned loader reads through a raw buffer resource whose base is
// the tile origin; an element outside the matrix gets an offset past the buffer's range, which the
// hardware answers with zero and without touching memory. No branch or use of the value follows the
// load, so the wait for it lands at the LDS store, after the MFMA work of the current K step.
constexpr uint32_t BUF_RANGE = 0x7fffffffu; // bytes addressable through one tile resource
constexpr uint32_t BUF_OOB   = 0x80000000u; // offset that reads as zero
constexpr int      BUF_FLAGS = 0x00020000;  // dword 3 of a gfx9 buffer resource (32-bit data format)

__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(const void *base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), static_cast<short>(0), static_cast<int>(BUF_RANGE), BUF_FLAGS);
}
template <typename E>
__device__ __forceinline__ E buffer_load_elem(__amdgpu_buffer_rsrc_t r, uint32_t off_bytes) {
    if constexpr(sizeof(E) == 16) return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b128(r, static_cast<int>(off_bytes), 0, 0));
    else if constexpr(sizeof(E) == 8) return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b64(r, static_cast<int>(off_bytes), 0, 0));
    else return __builtin_bit_cast(E, __builtin_amdgcn_raw_buffer_load_b32(r, static_cast<int>(off_bytes), 0, 0));
}
// Conjugation by a sign mask (0 or the sign bit of the imaginary part's high word): one XOR per element.
template <typename E>
__device__ __forceinline__ E conj_by_mask(E v, uint32_t imsign) {
    if constexpr(std::is_same_v<E, cpx<double>>) {
        const uint64_t b = __builtin_bit_cast(uint64_t, v.im) ^ (static_cast<uint64_t>(imsign) << 32);
        v.im             = __builtin_bit_cast(double, b);
    } else if constexpr(std::is_same_v<E, cpx<float>>) {
        v.im = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v.im) ^ imsign);
    }
    return v;
}
template <typename E>
__device__ __forceinline__ E conj_elem(E v, bool conj) {
    if constexpr(std::is_same_v<E, cpx<double>> || std::is_same_v<E, cpx<float>>) v.im = conj ? -v.im : v.im;
    return v;
}

// Walks the K index of one loaded element tile by tile without divisions:
// holds gk, gk % c and the element offset (gk % c) * s0 + (gk / c) * s1.
struct KCursor {
    int32_t  gk;
    uint32_t r;
    int64_t  off;
};
struct KStep {
    uint32_t dr, c;
    int64_t  delta, wrap;
};
__device__ inline KStep make_kstep(const Idx2 &x, int bk) {
    KStep st;
    st.c     = x.c;
    st.dr    = static_cast<uint32_t>(bk) % x.c;
    const int64_t dq = static_cast<int64_t>(static_cast<uint32_t>(bk) / x.c);
    st.delta = st.dr * x.s0 + dq * x.s1;
    st.wrap  = x.s1 - static_cast<int64_t>(x.c) * x.s0;
    return st;
}
__device__ inline KCursor make_kcursor(const Idx2 &x, int gk) {
    KCursor k;
    k.gk  = gk;
    k.r   = static_cast<uint32_t>(gk) % x.c;
    k.off = idx_off(x, static_cast<uint32_t>(gk));
    return k;
}
__device__ inline void advance(KCursor &k, const KStep &st, int bk) {
    k.gk += bk;
    k.r += st.dr;
    k.off += st.delta;
    if(k.r >= st.c) {
        k.r -= st.c;
        k.off += st.wrap;
    }
}

// Loads one operand tile (RT rows of the non-K dimension x BK) per K step into registers and
// then into LDS laid out [k][r]. Two address schemes:
//  ALIGNED: every chunk of the operand's index maps is a multiple or a divisor of the tile
//           extent, so offset(r0 + rr, k0 + kk) = offset(r0, k0) + offset(rr, kk): the per-element
//           part is a static 32-bit value and the tile base is uniform (scalar registers).
//  generic: per-element K cursors (KCursor) for arbitrary chunked index maps and ragged edges.
template <typename E, int RT, int BK, int NT, bool ALIGNED>
struct TileLoader {
    static constexpr int L = (RT * BK + NT - 1) / NT;
    int                  rr[L], kk[L];
    bool                 rval[L];
    bool                 lval[L];  // generic: validity of the element loaded last
    uint32_t             eoff[L];  // ALIGNED: static in-tile offset (bytes)
    uint32_t             eoffv[L]; // ALIGNED: eoff, or the zero-reading offset for rows outside the matrix
    int64_t              roff[L];  // generic: offset of the non-K coordinate
    KCursor              cur[L];   // generic: K cursors
    KCursor              kc;       // ALIGNED: K position of the next tile (uniform)
    KStep                st;
    const E             *tile_base; // ALIGNED: operand + offset of (r0, 0)
    Idx2                 kdim;
    int                  kbase;

    __device__ __forceinline__ void init(const E *src, const Idx2 &rdim, const Idx2 &kd, int r0, int rmax, int kbeg, bool fast_r, int tid) {
        kdim  = kd;
        kbase = kbeg;
#pragma unroll
        for(int e = 0; e < L; ++e) {
            const int  idx  = tid + e * NT;
            const bool used = idx < RT * BK;
            rr[e]           = fast_r ? idx % RT : (idx / BK) % RT;
            kk[e]           = fast_r ? (idx / RT) % BK : idx % BK;
            rval[e]         = used && (r0 + rr[e]) < rmax;
            if constexpr(ALIGNED) {
                eoff[e]  = static_cast<uint32_t>((idx_off(rdim, rr[e]) + idx_off(kd, kk[e])) * static_cast<int64_t>(sizeof(E)));
                eoffv[e] = rval[e] ? eoff[e] : BUF_OOB;
            } else {
                roff[e] = rval[e] ? idx_off(rdim, r0 + rr[e]) : 0;
                cur[e]  = make_kcursor(kd, kbeg + kk[e]);
            }
        }
        st = make_kstep(kd, BK);
        if constexpr(ALIGNED) {
            tile_base = src + idx_off(rdim, r0);
            kc        = make_kcursor(kd, kbeg);
        } else {
            tile_base = src;
        }
    }

    // Issues the loads of the next tile (K offset k0; tiles are loaded in K order from kbeg on) and advances.
    // Elements outside the matrix read as zero (ALIGNED) or are zeroed at store (generic). ALIGNED: the tile
    // origin advances by a cursor (no division per step) and each element costs one compare against the K
    // extent left (row validity is folded into its offset at init).
    __device__ __forceinline__ void load(E (&reg)[L], int k0, int kend) {
        if constexpr(ALIGNED) {
            const auto rs  = tile_rsrc(tile_base + kc.off);
            const int  rem = kend - k0;
            advance(kc, st, BK);
#pragma unroll
            for(int e = 0; e < L; ++e) reg[e] = buffer_load_elem<E>(rs, kk[e] < rem ? eoffv[e] : BUF_OOB);
        } else {
#pragma unroll
            for(int e = 0; e < L; ++e) {
                const bool v = rval[e] && cur[e].gk < kend;
                lval[e]      = v;
                reg[e]       = tile_base[v ? roff[e] + cur[e].off : 0];
                advance(cur[e], st, BK);
            }
        }
    }

    // Writes the tile into LDS laid out [k][r] with a row pitch of `pitch` elements.
    // The registers are updated in place (conjugation), so that each element goes to LDS without a copy.
    __device__ __forceinline__ void store(E *lds, int pitch, E (&reg)[L], int tid, uint32_t imsign) const {
#pragma unroll
        for(int e = 0; e < L; ++e)
            if(L * NT == RT * BK || tid + e * NT < RT * BK) {
                if constexpr(!ALIGNED) reg[e] = lval[e] ? reg[e] : zero_elem<E>();
                reg[e]                     = conj_by_mask(reg[e], imsign);
                lds[kk[e] * pitch + rr[e]] = reg[e];
            }
    }
};

// One output tile of g: bx is the tile's position in the launch (before the XCD remap), split the K slice
// and b the batch index.
template <typename R, bool CPLX, int BM, int BN, int BK, int WM, int WN, bool SWAP, bool ALIGNED>
__device__ __forceinline__ void gemm_body(const GemmDesc &g, int bx, int split, int b) {
    using E               = elem_t<R, CPLX>;
    using MF              = mfma_t<R>;
    using acc_t           = typename MF::acc;
    constexpr int NT      = 64 * WM * WN;
    constexpr int TM      = BM / (16 * WM);
    constexpr int TN      = BN / (16 * WN);
    constexpr int EB      = static_cast<int>(sizeof(E));
    constexpr int LDA     = BM + imax(pad_rfast(BM, EB), pad_kfast(BM, EB)); // allocated row length of A's tile
    constexpr int LDB     = BN + imax(pad_rfast(BN, EB), pad_kfast(BN, EB));
    constexpr int NACC    = CPLX ? 3 : 1; // complex: sum ar*br, sum ai*bi, sum (ar+ai)*(br+bi)
    static_assert(TM >= 1 && TN >= 1, "wave tile too small");
    static_assert(BK % 4 == 0, "BK must be a multiple of the MFMA k");

    __shared__ E As[2][BK * LDA];
    __shared__ E Bs[2][BK * LDB];

    const int tid  = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm   = wave % WM;
    const int wn   = wave / WM;

    // Tile index. Workgroups are dealt round-robin over the 8 XCDs (workgroup x runs on XCD x % 8), each with its
    // own L2. When the tile grid splits into 2 x 4 blocks, XCD x takes block (x / 4, x % 4): half of the tile rows
    // and a quarter of the tile columns, walked column by column, so that the operand panels an XCD reads are half
    // of A and a quarter of B. (Giving each XCD a range of whole tile columns instead makes every XCD stream all of
    // A; at chi = 512 that fetched 2.2x the HBM bytes for leg 1 at the same kernel time.) Otherwise each XCD
    // takes a contiguous range of tiles.
    const int tilesM = (g.M + BM - 1) / BM;
    const int tilesN = (g.N + BN - 1) / BN;
    const int total  = tilesM * tilesN;
    int       mt, nt;
    if(g.xcd_remap && (tilesM % 2) == 0 && (tilesN % 4) == 0) {
        const int x = bx % 8, j = bx / 8, rm = tilesM / 2;
        mt = (x / 4) * rm + j % rm;
        nt = (x % 4) * (tilesN / 4) + j / rm;
    } else {
        int bid = bx;
        if(g.xcd_remap && (total % 8) == 0) bid = (bid % 8) * (total / 8) + bid / 8;
        mt = bid % tilesM;
        nt = bid / tilesM;
    }
    const int m0 = mt * BM;
    const int n0 = nt * BN;

    // K range of this workgroup (split-K slice).
    const int kbeg  = split * g.kchunk;
    const int kend  = min(g.K, kbeg + g.kchunk);

    // Row pitches: A is loaded along M when g.a_fast_m, B along N when !g.b_fast_k.
    const int pa = g.a_fast_m ? BM + pad_rfast(BM, EB) : BM + pad_kfast(BM, EB);
    const int pb = !g.b_fast_k ? BN + pad_rfast(BN, EB) : BN + pad_kfast(BN, EB);
    TileLoader<E, BM, BK, NT, ALIGNED> la;
    TileLoader<E, BN, BK, NT, ALIGNED> lb;
    la.init(static_cast<const E *>(g.A) + b * g.a_batch, g.am, g.ak, m0, g.M, kbeg, g.a_fast_m, tid);
    lb.init(static_cast<const E *>(g.B) + b * g.b_batch, g.bn, g.bk, n0, g.N, kbeg, !g.b_fast_k, tid);
    E ra[TileLoader<E, BM, BK, NT, ALIGNED>::L], rb[TileLoader<E, BN, BK, NT, ALIGNED>::L];

    acc_t acc[NACC][TM][TN];
#pragma unroll
    for(int c = 0; c < NACC; ++c)
#pragma unroll
        for(int i = 0; i < TM; ++i)
#pragma unroll
            for(int j = 0; j < TN; ++j) acc[c][i][j] = acc_t{0, 0, 0, 0};

    const int      numK = kend > kbeg ? (kend - kbeg + BK - 1) / BK : 0;
    const uint32_t sgnA = g.conjA ? 0x80000000u : 0u, sgnB = g.conjB ? 0x80000000u : 0u; // conjugation masks
    const int lrow = lane >> 4; // k row within the 4-deep MFMA step
    const int lcol = lane & 15; // m (or n) within a 16-wide block
    if(numK > 0) {
        la.load(ra, kbeg, kend);
        lb.load(rb, kbeg, kend);
        la.store(As[0], pa, ra, tid, sgnA);
        lb.store(Bs[0], pb, rb, tid, sgnB);
        __syncthreads();
    }
    for(int kt = 0; kt < numK; ++kt) {
        const int buf = kt & 1;
        if(kt + 1 < numK) {
            la.load(ra, kbeg + (kt + 1) * BK, kend);
            lb.load(rb, kbeg + (kt + 1) * BK, kend);
        }
#pragma unroll
        for(int ks = 0; ks < BK / 4; ++ks) {
            const int kr = ks * 4 + lrow;
            E         fa[TM], fb[TN];
#pragma unroll
            for(int i = 0; i < TM; ++i) fa[i] = As[buf][kr * pa + (wm * TM + i) * 16 + lcol];
#pragma unroll
            for(int j = 0; j < TN; ++j) fb[j] = Bs[buf][kr * pb + (wn * TN + j) * 16 + lcol];
            R sa[CPLX ? TM : 1], sb[CPLX ? TN : 1];
            if constexpr(CPLX) {
#pragma unroll
                for(int i = 0; i < TM; ++i) sa[i] = fa[i].re + fa[i].im;
#pragma unroll
                for(int j = 0; j < TN; ++j) sb[j] = fb[j].re + fb[j].im;
            }
#pragma unroll
            for(int i = 0; i < TM; ++i)
#pragma unroll
                for(int j = 0; j < TN; ++j) {
                    if constexpr(CPLX) {
                        // (ar + i ai)(br + i bi): P1 += ar br, P2 += ai bi, P3 += (ar + ai)(br + bi).
                        if constexpr(!SWAP) {
                            acc[0][i][j] = MF::op(fa[i].re, fb[j].re, acc[0][i][j]);
                            acc[1][i][j] = MF::op(fa[i].im, fb[j].im, acc[1][i][j]);
                            acc[2][i][j] = MF::op(sa[i], sb[j], acc[2][i][j]);
                        } else {
                            acc[0][i][j] = MF::op(fb[j].re, fa[i].re, acc[0][i][j]);
                            acc[1][i][j] = MF::op(fb[j].im, fa[i].im, acc[1][i][j]);
                            acc[2][i][j] = MF::op(sb[j], sa[i], acc[2][i][j]);
                        }
                    } else {
                        if constexpr(!SWAP) acc[0][i][j] = MF::op(fa[i], fb[j], acc[0][i][j]);
                        else acc[0][i][j] = MF::op(fb[j], fa[i], acc[0][i][j]);
                    }
                }
        }
        if(kt + 1 < numK) {
            la.store(As[buf ^ 1], pa, ra, tid, sgnA);
            lb.store(Bs[buf ^ 1], pb, rb, tid, sgnB);
        }
        __syncthreads();
    }

    // Epilogue. 16x16 accumulator layout (measured on gfx950): lane l, register v holds column l%16 of
    // row 4*(l/16)+v for v_mfma_f32_16x16x4_f32 and of row (l/16)+4*v for v_mfma_f64_16x16x4_f64.
    // Without swap rows run along M; with swap they run along N.
    // Split-K partials go to g.part as plain column-major M x N slabs, one per (batch, split).
    E *C = static_cast<E *>(g.C) + b * g.c_batch;
    E *P = g.ksplit > 1 ? static_cast<E *>(g.part) + (static_cast<int64_t>(b) * g.ksplit + split) * g.M * g.N : nullptr;
#pragma unroll
    for(int i = 0; i < TM; ++i)
#pragma unroll
        for(int j = 0; j < TN; ++j)
#pragma unroll
            for(int v = 0; v < 4; ++v) {
                const int row = std::is_same_v<R, double> ? (lrow + 4 * v) : (4 * lrow + v);
                int       gm, gn;
                if constexpr(!SWAP) {
                    gm = m0 + (wm * TM + i) * 16 + row;
                    gn = n0 + (wn * TN + j) * 16 + lcol;
                } else {
                    gm = m0 + (wm * TM + i) * 16 + lcol;
                    gn = n0 + (wn * TN + j) * 16 + row;
                }
                if(gm < g.M && gn < g.N) {
                    E val;
                    if constexpr(CPLX) {
                        const R p1 = acc[0][i][j][v], p2 = acc[1][i][j][v];
                        val        = E{p1 - p2, acc[2][i][j][v] - p1 - p2};
                    }
                    else val = acc[0][i][j][v];
                    if(P) {
                        P[gm + static_cast<int64_t>(g.M) * gn] = val;
                    } else {
                        const int64_t off = idx_off(g.cm, gm) + idx_off(g.cn, gn);
                        if(g.accumulate) {
                            const E old = C[off];
                            if constexpr(CPLX) {
                                val.re += old.re;
                                val.im += old.im;
                            } else {
                                val += old;
                            }
                        }
                        C[off] = val;
                    }
                }
            }
}

template <typename R, bool CPLX, int BM, int BN, int BK, int WM, int WN, bool SWAP, bool ALIGNED>
__global__ __launch_bounds__(64 * WM *WN) void gemm_kernel(const GemmDesc g) {
    gemm_body<R, CPLX, BM, BN, BK, WM, WN, SWAP, ALIGNED>(g, blockIdx.x, blockIdx.y, blockIdx.z);
}

// Grouped launches of the GEMMs that the pipelined kernel does not take (gemm_pipe.hpp holds its grouped form).
template <typename R, bool CPLX, int BM, int BN, int BK, int WM, int WN, bool SWAP>
__global__ __launch_bounds__(64 * WM *WN) void gemm_grouped_kernel(const GemmDesc *descs, const int *tile_start, int ngemm) {
    const int i = pipe::group_of(tile_start, ngemm, blockIdx.x);
    gemm_body<R, CPLX, BM, BN, BK, WM, WN, SWAP, false>(descs[i], blockIdx.x - tile_start[i], 0, 0);
}

// Sums the split-K partial slabs in a fixed order and writes C through its index map.
template <typename E>
__global__ void splitk_reduce(const GemmDesc g) {
    const int64_t MN    = static_cast<int64_t>(g.M) * g.N;
    const int64_t total = MN * g.batch;
    const E      *P     = static_cast<const E *>(g.part);
    for(int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < total;
        t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int64_t b   = t / MN;
        const int64_t mn  = t - b * MN;
        const int     m   = static_cast<int>(mn % g.M);
        const int     n   = static_cast<int>(mn / g.M);
        const E      *src = P + b * g.ksplit * MN + mn;
        E             s   = src[0];
        for(int k = 1; k < g.ksplit; ++k) {
            const E v = src[k * MN];
            if constexpr(std::is_same_v<E, cpx<double>> || std::is_same_v<E, cpx<float>>) {
                s.re += v.re;
                s.im += v.im;
            } else {
                s += v;
            }
        }
        E            *C   = static_cast<E *>(g.C) + b * g.c_batch;
        const int64_t off = idx_off(g.cm, m) + idx_off(g.cn, n);
        if(g.accumulate) {
            const E old = C[off];
            if constexpr(std::is_same_v<E, cpx<double>> || std::is_same_v<E, cpx<float>>) {
                s.re += old.re;
                s.im += old.im;
            } else {
                s += old;
            }
        }
        C[off] = s;
    }
}

// ---------------------------------------------------------------------------------------
// Host launcher

struct CfgShape {
    int BM, BN;
};
static CfgShape cfg_shape(TileCfg c) {
    switch(c) {
        case TileCfg::T64x64: return {64, 64};
        case TileCfg::T32x64: return {32, 64};
        case TileCfg::T64x32: return {64, 32};
        case TileCfg::T16x128: return {16, 128};
        case TileCfg::T128x64: return {128, 64};
        case TileCfg::T32x32: return {32, 32};
        case TileCfg::T32x32K: return {32, 32};
        default: return {64, 64};
    }
}

int device_cu_count() {
    static int cus = [] {
        int dev = 0, n = 0;
        if(hipGetDevice(&dev) != hipSuccess) return 256;
        if(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) return 256;
        return n;
    }();
    return cus;
}

// A plan: tile configuration and K slices; with nsplit > 0 the columns [0, nsplit) run as one launch without
// K slicing and the tail [nsplit, N) as a second launch with ksplit2 K slices, so that the tail (the part of
// the grid that would occupy the GPU only partially) is spread over all CUs.
struct LaunchPlan {
    TileCfg cfg;
    int     ksplit;
    int     nsplit  = 0;
    int     ksplit2 = 1;
};

// The orientation in which consecutive m are (if anything is) consecutive in C: the pipelined kernel's lanes run along M.
static int      fast_score(const Idx2 &x) { return x.s0 == 1 ? static_cast<int>(std::min<uint32_t>(x.c, 1u << 20)) : 0; }
static GemmDesc oriented(const GemmDesc &g) {
    if(fast_score(g.cn) <= fast_score(g.cm)) return g;
    GemmDesc t = g;
    std::swap(t.A, t.B);
    std::swap(t.am, t.bn);
    std::swap(t.ak, t.bk);
    std::swap(t.a_batch, t.b_batch);
    std::swap(t.conjA, t.conjB);
    std::swap(t.M, t.N);
    std::swap(t.cm, t.cn);
    return t;
}

// The pipelined shape that a tile configuration stands for, or N_SHAPES.
static pipe::Shape shape_of(TileCfg c, dmrg_dtype t) {
    pipe::Shape s = pipe::N_SHAPES;
    switch(c) {
        case TileCfg::T128x64: s = pipe::S128x64; break;
        case TileCfg::T64x64: s = pipe::S64x64; break;
        case TileCfg::T32x64:
        case TileCfg::T64x32: s = pipe::S64x32; break;
        case TileCfg::T32x32:
        case TileCfg::T32x32K: s = pipe::S32x32; break;
        default: return s;
    }
    while(pipe::shape_info(t, s).BM == 0) s = static_cast<pipe::Shape>(s + 1); // the next smaller shape of the type
    return s;
}

// Microseconds that the pipelined kernel takes for g in shape s with ks K slices, with loads of W bytes per lane: a CU's
// workgroups share its matrix cores, so r of them advance one stage in r stage times of MFMA work, but none of them faster
// than its own chain of barrier, LDS read and MFMA (about 170 clocks beyond its MFMAs), and all of them together no faster
// than their loads, about 17 clocks each. Real stages are too short for workgroups to hide that chain of one another (32x32
// FP64: 0.165 us a stage with one workgroup on a CU, 0.33 with two; counted so, FP64 300x280 at D = 5 takes 39.1 us instead
// of 41.2); complex ones hide it (counted alike, 173x211 would take 42.9 us instead of 41.5). Over 360 legs 1 and 3 of random
// operators (bonds 12 to 840, d 2 and 4, D 3 to 8; 78 to 104 of each type) the cheapest plan takes 2.8 % longer than the best
// of 13 forced ones in the geometric mean (2.1 % complex FP64, 3.9 % complex FP32), 94 % are within 10 %, the worst 24 %.
static double pipe_cost_us(const GemmDesc &g, pipe::Shape s, int ks, int W) {
    const pipe::ShapeInfo i = pipe::shape_info(g.dtype, s);
    const bool   cplx = dtype_is_complex(g.dtype), sp = dtype_is_single(g.dtype);
    const double clk = 2300.0, cus = device_cu_count();
    const double stages = std::ceil((g.K + i.BK - 1) / i.BK / static_cast<double>(ks));
    const double mfma   = i.TM * i.TN * (i.BK / 4) * (cplx ? 3 : 1) * (sp ? 32.0 : 64.0);
    const double loads  = (i.BM + i.BN) * i.BK * static_cast<double>(dtype_size(g.dtype)) / (64.0 * W) * 17.0;
    const double tiles  = static_cast<double>((g.M + i.BM - 1) / i.BM) * ((g.N + i.BN - 1) / i.BN) * g.batch * ks;
    auto         round  = [&](double r) {
        return stages * (cplx ? std::max({r * mfma * 1.04, r * loads, mfma + 170.0}) : r * std::max(mfma + 150.0, loads));
    };
    const double per_cu = std::ceil(tiles / cus), full = std::floor(per_cu / i.resident), rest = per_cu - full * i.resident;
    double       us     = 3.0 + (full * (round(i.resident) + 1500.0) + (rest > 0 ? round(rest) : 0.0)) / clk;
    const double out    = static_cast<double>(g.M) * g.N * g.batch * static_cast<double>(dtype_size(g.dtype));
    us += out / 4.0e6;                                     // the results at 4 TB/s
    if(ks > 1) us += 3.5 + out * (ks + 1) / 3.0e6;         // the slices' sums
    return us;
}

// All pipelined plans of g, the cheapest first.
static std::vector<std::pair<double, LaunchPlan>> ranked_plans(const GemmDesc &g0) {
    const GemmDesc g = oriented(g0);
    std::vector<std::pair<double, LaunchPlan>> v;
    for(TileCfg c : {TileCfg::T128x64, TileCfg::T64x64, TileCfg::T64x32, TileCfg::T32x32}) {
        const pipe::Shape s = shape_of(c, g.dtype);
        if((c == TileCfg::T128x64 && s != pipe::S128x64) || (c == TileCfg::T64x32 && s != pipe::S64x32)) continue;
        const int    bk = pipe::shape_info(g.dtype, s).BK;
        const int    W = pipe::load_bytes(g, pipe::shape_info(g.dtype, s));
        for(int ks : {1, 2, 3, 4, 6, 8}) {
            if(ks > 1 && (g.K < 4 * bk * ks || !g.part || g.part_capacity < static_cast<int64_t>(g.M) * g.N * g.batch * ks)) continue;
            v.emplace_back(pipe_cost_us(g, s, ks, W), LaunchPlan{c, ks});
        }
    }
    std::stable_sort(v.begin(), v.end(), [](const auto &a, const auto &b) { return a.first < b.first; });
    return v;
}

static LaunchPlan heuristic_plan(const GemmDesc &g) {
    // The streaming kernel where the columns dominate: below 8 columns per row the tiles' reuse of B is worth more. Past 256
    // fragments, laying A out in LDS takes 2 to 7 us, which real GEMMs win back from three 32x32 tiles per CU on and complex
    // ones (four products against the tiles' three) hardly ever: K = M = 50, N = 960 complex 16.1 us, tiles 6.3; FP64 8.9
    // against 6.0, at N = 32964 16 against 26. Over K = M of 10 to 64 and 576 to 65536 columns (70 sizes of each type) the
    // choice takes 0.1 % longer than the best of streaming, 32x32 and 64x64 tiles in the geometric mean, 96 % are within
    // 10 %, the worst 18 % (FP32, K = M = 64; complex FP32, K = M = 18).
    if(stream::takes(g) && (g.M <= 16 || g.N >= 8 * g.M)) {
        const int64_t fragments = static_cast<int64_t>((g.M + 15) / 16) * ((g.K + 3) / 4) * 64;
        const int64_t tiles     = static_cast<int64_t>((g.M + 31) / 32) * ((g.N + 31) / 32) * g.batch;
        if(g.M <= 16 || fragments <= 256 || (!dtype_is_complex(g.dtype) && tiles >= 3 * static_cast<int64_t>(device_cu_count())))
            return LaunchPlan{TileCfg::SMALLK, 1};
    }
    if(g.M <= 16) return LaunchPlan{TileCfg::T16x128, 1};
    return ranked_plans(g).front().second;
}

// Tile-separable index map: offset(t0 + t) = offset(t0) + offset(t) for every tile origin t0 (a multiple
// of ext) and 0 <= t < ext, which holds when each chunk is a multiple or a divisor of ext.
static bool separable(const Idx2 &x, int ext) {
    return x.c >= 0x7fffffffu || (x.c % static_cast<uint32_t>(ext)) == 0 || (static_cast<uint32_t>(ext) % x.c) == 0;
}
// Largest in-tile offset (bytes) must stay inside the aligned loader's buffer range.
static bool small_tile_offsets(const Idx2 &r, int rt, const Idx2 &k, int bk, int elem_bytes) {
    auto mx = [](const Idx2 &x, int ext) {
        int64_t m = 0;
        for(int t = 0; t < ext; ++t) m = std::max<int64_t>(m, std::llabs(idx_off(x, t)));
        return m;
    };
    return (mx(r, rt) + mx(k, bk)) * elem_bytes < static_cast<int64_t>(BUF_RANGE) && r.s0 >= 0 && r.s1 >= 0 && k.s0 >= 0 &&
           k.s1 >= 0;
}

static void splitk_sum(const GemmDesc &g, hipStream_t s);

template <typename R, bool CPLX, int BM, int BN, int BK, int WM, int WN>
static void launch_cfg(const GemmDesc &g, bool swap, hipStream_t s) {
    const int  tiles = ((g.M + BM - 1) / BM) * ((g.N + BN - 1) / BN);
    const dim3 grid(tiles, g.ksplit, g.batch);
    const dim3 block(64 * WM * WN);
    const bool aligned = separable(g.am, BM) && separable(g.ak, BK) && separable(g.bn, BN) && separable(g.bk, BK) &&
                         (g.kchunk % BK) == 0 && small_tile_offsets(g.am, BM, g.ak, BK, static_cast<int>(sizeof(elem_t<R, CPLX>))) &&
                         small_tile_offsets(g.bn, BN, g.bk, BK, static_cast<int>(sizeof(elem_t<R, CPLX>)));
    if(aligned) {
        if(swap) hipLaunchKernelGGL((gemm_kernel<R, CPLX, BM, BN, BK, WM, WN, true, true>), grid, block, 0, s, g);
        else hipLaunchKernelGGL((gemm_kernel<R, CPLX, BM, BN, BK, WM, WN, false, true>), grid, block, 0, s, g);
    } else {
        if(swap) hipLaunchKernelGGL((gemm_kernel<R, CPLX, BM, BN, BK, WM, WN, true, false>), grid, block, 0, s, g);
        else hipLaunchKernelGGL((gemm_kernel<R, CPLX, BM, BN, BK, WM, WN, false, false>), grid, block, 0, s, g);
    }
    if(g.ev_after_main) DMRG_HIP_CHECK(hipEventRecord(static_cast<hipEvent_t>(g.ev_after_main), s));
    if(g.ksplit > 1) splitk_sum(g, s);
}

static void splitk_sum(const GemmDesc &g, hipStream_t s) {
    const int64_t total = static_cast<int64_t>(g.M) * g.N * g.batch;
    const dim3    rg(static_cast<unsigned>(std::min<int64_t>((total + 255) / 256, 8192)));
    switch(g.dtype) {
        case DMRG_FP64: hipLaunchKernelGGL((splitk_reduce<double>), rg, dim3(256), 0, s, g); break;
        case DMRG_CX64: hipLaunchKernelGGL((splitk_reduce<cpx<double>>), rg, dim3(256), 0, s, g); break;
        case DMRG_FP32: hipLaunchKernelGGL((splitk_reduce<float>), rg, dim3(256), 0, s, g); break;
        case DMRG_CX32: hipLaunchKernelGGL((splitk_reduce<cpx<float>>), rg, dim3(256), 0, s, g); break;
    }
}

// A GEMM described for a pipelined shape, all but its pointers fixed.
struct Prepared {
    pipe::Launch l;
    pipe::Shape  shape;
    dim3         grid;
};

// Describes g (oriented) for a shape with up to ksplit K slices; false where the pipelined kernel does not take it.
static bool prepare_pipelined(const GemmDesc &g, pipe::Shape shape, int ksplit, Prepared &p) {
    const pipe::ShapeInfo i = pipe::shape_info(g.dtype, shape);
    if(!pipe::describe(g, i, ksplit, p.l)) return false;
    p.shape = shape;
    p.grid  = dim3(static_cast<unsigned>((g.M + i.BM - 1) / i.BM) * static_cast<unsigned>((g.N + i.BN - 1) / i.BN), p.l.d.ksplit, g.batch);
    return true;
}

// g: oriented, with the pointers of p's description.
static void run_pipelined(GemmDesc g, const Prepared &p, hipStream_t s) {
    switch(g.dtype) {
        case DMRG_FP64: pipe::launch_f64(p.l, p.shape, p.grid, s); break;
        case DMRG_CX64: pipe::launch_c128(p.l, p.shape, p.grid, s); break;
        case DMRG_FP32: pipe::launch_f32(p.l, p.shape, p.grid, s); break;
        case DMRG_CX32: pipe::launch_c64(p.l, p.shape, p.grid, s); break;
    }
    if(g.ev_after_main) DMRG_HIP_CHECK(hipEventRecord(static_cast<hipEvent_t>(g.ev_after_main), s));
    if(p.l.d.ksplit > 1) {
        g.ksplit = p.l.d.ksplit;
        splitk_sum(g, s);
    }
    DMRG_HIP_CHECK(hipGetLastError());
}

template <typename R, bool CPLX>
static void launch_typed(const GemmDesc &g, TileCfg cfg, bool swap, hipStream_t s) {
    // The kernels beside the pipelined ones: tall outputs of at most 16 rows, tiny K, and 64x64 tiles with 64-bit offsets
    // per element for the index maps that the pipelined kernel does not take.
    constexpr int E  = static_cast<int>(sizeof(elem_t<R, CPLX>));
    constexpr int BK = E == 4 ? 32 : 16;
    constexpr int BH = E == 16 ? 8 : BK;
    if(cfg == TileCfg::SMALLK && !stream::takes(g)) cfg = TileCfg::T64x64;
    switch(cfg) {
        case TileCfg::T16x128: launch_cfg<R, CPLX, 16, 128, BH, 1, 4>(g, swap, s); break;
        case TileCfg::SMALLK: stream::launch(g, device_cu_count(), s); break;
        case TileCfg::AUTO: throw Error(DMRG_ERR_ARG, "bad tile config");
        default: {
            const dim3 grid(((g.M + 63) / 64) * ((g.N + 63) / 64), g.ksplit, g.batch), block(256);
            if(swap) hipLaunchKernelGGL((gemm_kernel<R, CPLX, 64, 64, BK, 2, 2, true, false>), grid, block, 0, s, g);
            else hipLaunchKernelGGL((gemm_kernel<R, CPLX, 64, 64, BK, 2, 2, false, false>), grid, block, 0, s, g);
            if(g.ev_after_main) DMRG_HIP_CHECK(hipEventRecord(static_cast<hipEvent_t>(g.ev_after_main), s));
            if(g.ksplit > 1) splitk_sum(g, s);
        }
    }
}

// ---------------------------------------------------------------------------------------
// Autotuner: times candidate (tile configuration, K slices) plans of a GEMM with HIP events on
// its own stream and caches the fastest per problem signature (dtype, sizes, index maps).

static std::mutex                        g_tune_mu;
static std::map<std::string, LaunchPlan> g_tuned;
static int                               g_autotune     = 1;
// GEMMs below this many (complex or real) multiply-adds, and with fewer than a sixteenth as many bytes of operands,
// take the size heuristic instead of being tuned.
static int64_t                           g_tune_min_macs = int64_t(1) << 29;
static std::atomic<uint64_t>             g_plan_state{0}; // counts the changes that can change a plan
static int                               g_override_cfg = -1, g_override_ks = 0;
static int                               g_override_nsplit = 0, g_override_ks2 = 1;

static std::string tune_key(const GemmDesc &g) {
    char buf[512];
    auto I = [](const Idx2 &x) { return std::to_string(x.s0) + "," + std::to_string(x.s1) + "," + std::to_string(x.c); };
    std::snprintf(buf, sizeof(buf), "%d|%d|%d|%d|%d|%d|%d|", static_cast<int>(g.dtype), g.M, g.N, g.K, g.batch,
                  g.part ? 1 : 0, static_cast<int>(std::min<int64_t>(g.part_capacity / std::max<int64_t>(1, int64_t(g.M) * g.N * g.batch), 8)));
    return std::string(buf) + I(g.am) + "|" + I(g.ak) + "|" + I(g.bk) + "|" + I(g.bn) + "|" + I(g.cm) + "|" + I(g.cn);
}

static void launch_plan_single(GemmDesc g, const LaunchPlan &p0, hipStream_t stream);

// Columns [n0, n0 + nn) of g as a GEMM of their own (valid when the B and C column maps are separable at n0).
static GemmDesc column_slice(const GemmDesc &g, int n0, int nn) {
    GemmDesc h     = g;
    const size_t es = dtype_size(g.dtype);
    h.B            = static_cast<const char *>(g.B) + idx_off(g.bn, static_cast<uint32_t>(n0)) * static_cast<int64_t>(es);
    h.C            = static_cast<char *>(g.C) + idx_off(g.cn, static_cast<uint32_t>(n0)) * static_cast<int64_t>(es);
    h.N            = nn;
    h.ev_after_main = nullptr;
    return h;
}
static bool column_separable(const Idx2 &x, int n0) { return x.c >= 0x7fffffffu || (static_cast<uint32_t>(n0) % x.c) == 0; }

static void launch_plan(const GemmDesc &g, const LaunchPlan &p, hipStream_t stream) {
    if(p.nsplit > 0 && p.nsplit < g.N && g.batch == 1 && column_separable(g.bn, p.nsplit) && column_separable(g.cn, p.nsplit)) {
        GemmDesc head = column_slice(g, 0, p.nsplit), tail = column_slice(g, p.nsplit, g.N - p.nsplit);
        launch_plan_single(head, LaunchPlan{p.cfg, 1}, stream);
        tail.ev_after_main = g.ev_after_main;
        launch_plan_single(tail, LaunchPlan{p.cfg, p.ksplit2}, stream);
        return;
    }
    launch_plan_single(g, LaunchPlan{p.cfg, p.ksplit}, stream);
}

static void launch_plan_single(GemmDesc g, const LaunchPlan &p0, hipStream_t stream) {
    LaunchPlan p = p0;
    if(p.ksplit > 1) {
        const int64_t need = static_cast<int64_t>(g.M) * g.N * g.batch * p.ksplit;
        if(!g.part || g.part_capacity < need) p.ksplit = 1;
    }
    const pipe::Shape shape = shape_of(p.cfg, g.dtype);
    if(shape != pipe::N_SHAPES) {
        const GemmDesc h = oriented(g);
        Prepared       pr;
        if(prepare_pipelined(h, shape, p.ksplit, pr)) {
            run_pipelined(h, pr, stream);
            return;
        }
    }
    g.ksplit     = 1;
    const int kr = 32; // K extent per slice: a multiple of every configuration's BK
    g.kchunk = (g.K + kr - 1) / kr * kr;
    if(p.ksplit > 1) {
        const int kc = (((g.K + p.ksplit - 1) / p.ksplit) + kr - 1) / kr * kr;
        g.kchunk     = kc;
        g.ksplit     = (g.K + kc - 1) / kc;
    }
    if(g.kchunk <= 0) g.kchunk = 32;
    const bool swap = (g.cm.s0 == 1 && g.cm.c >= 16) && !(g.cn.s0 == 1 && g.cn.c >= 16);
    switch(g.dtype) {
        case DMRG_FP64: launch_typed<double, false>(g, p.cfg, swap, stream); break;
        case DMRG_CX64: launch_typed<double, true>(g, p.cfg, swap, stream); break;
        case DMRG_FP32: launch_typed<float, false>(g, p.cfg, swap, stream); break;
        case DMRG_CX32: launch_typed<float, true>(g, p.cfg, swap, stream); break;
    }
    DMRG_HIP_CHECK(hipGetLastError());
}

// ---------------------------------------------------------------------------------------
// Grouped launches

int grouped_tiles(const GemmDesc &g, TileCfg cfg) {
    const CfgShape sh = cfg_shape(cfg);
    return ((g.M + sh.BM - 1) / sh.BM) * ((g.N + sh.BN - 1) / sh.BN);
}

bool grouped_streams(const GemmDesc &g) { return stream::takes(g); }

// At most four launches (GroupedGemm::Kind), each with its GEMMs' descriptions and their first workgroups, 256-byte aligned.
static size_t    aligned256(size_t b) { return (b + 255) / 256 * 256; }
constexpr size_t GROUP_DESC_MAX = std::max({sizeof(GemmDesc), sizeof(pipe::Desc), sizeof(stream::Desc)});
size_t grouped_store_bytes(size_t ngemm) {
    return aligned256(GROUP_DESC_MAX * ngemm) + aligned256(sizeof(int) * (ngemm + 4)) + 8 * 256;
}

namespace {
// The GEMMs of one launch: descriptions as bytes, and their first workgroups.
struct GroupBuilder {
    std::vector<char> descs;
    std::vector<int>  starts{0};
    int               max_k = 0;
    size_t            lds   = 0;

    template <typename D>
    void add(const D &d, int64_t workgroups, int K, size_t lds_bytes = 0) {
        const int64_t next = static_cast<int64_t>(starts.back()) + workgroups;
        DMRG_REQUIRE(next < (int64_t(1) << 31), DMRG_ERR_DIMS, "grouped GEMM: too many tiles");
        starts.push_back(static_cast<int>(next));
        const char *p = reinterpret_cast<const char *>(&d);
        descs.insert(descs.end(), p, p + sizeof(D));
        max_k = std::max(max_k, K);
        lds   = std::max(lds, lds_bytes);
    }
};
} // namespace

std::vector<GroupedGemm> grouped_prepare(const std::vector<GemmDesc> &gs, TileCfg cfg, void *store, size_t store_bytes) {
    DMRG_REQUIRE(!store || store_bytes >= grouped_store_bytes(gs.size()), DMRG_ERR_ARG, "grouped GEMM: descriptor store too small");
    DMRG_REQUIRE(cfg == TileCfg::T64x64 || cfg == TileCfg::T32x32 || cfg == TileCfg::SMALLK, DMRG_ERR_ARG,
                 "grouped GEMM: tile configuration not available");
    const TileCfg         tiled = cfg == TileCfg::SMALLK ? TileCfg::T32x32 : cfg;
    std::vector<GemmDesc> members;
    int64_t               blocks = 0; // 16-column blocks of the streamed GEMMs
    for(GemmDesc g : gs) {
        if(g.M <= 0 || g.N <= 0) continue;
        DMRG_REQUIRE(g.batch == 1 && !g.accumulate && g.K > 0, DMRG_ERR_ARG, "grouped GEMM: batch 1, K > 0, no accumulation");
        DMRG_REQUIRE(g.dtype == gs[0].dtype, DMRG_ERR_ARG, "grouped GEMM: one dtype per group");
        DMRG_REQUIRE(static_cast<int64_t>(g.M) * g.N < (int64_t(1) << 31), DMRG_ERR_DIMS, "gemm: output too large");
        g.ksplit        = 1;
        g.xcd_remap     = 0;
        g.part          = nullptr;
        g.part_capacity = 0;
        g.ev_after_main = nullptr;
        if(cfg == TileCfg::SMALLK && stream::takes(g)) blocks += (g.N + 15) / 16;
        members.push_back(g);
    }
    // Workgroups start in the order of their numbers: the longest sums first, so that the launch ends evenly.
    std::stable_sort(members.begin(), members.end(), [](const GemmDesc &a, const GemmDesc &b) { return a.K > b.K; });
    const int64_t waves = static_cast<int64_t>(device_cu_count()) * 16;
    GroupBuilder  build[GroupedGemm::N_KINDS];
    for(GemmDesc &g : members) {
        if(cfg == TileCfg::SMALLK && stream::takes(g)) {
            const stream::Desc d = stream::describe(g, std::max<int64_t>(1, waves * ((g.N + 15) / 16) / blocks));
            build[GroupedGemm::STREAMED].add(d, stream::workgroups(d), g.K, stream::lds_bytes(g));
            continue;
        }
        const GemmDesc    h     = oriented(g);
        const pipe::Shape shape = shape_of(tiled, g.dtype);
        pipe::Launch      l;
        if(pipe::describe(h, pipe::shape_info(g.dtype, shape), 1, l, true)) {
            build[GroupedGemm::PIPELINED].add(l.d, grouped_tiles(h, tiled), h.K);
            continue;
        }
        g.a_fast_m      = fast_score(g.am) >= fast_score(g.ak) ? 1 : 0;
        g.b_fast_k      = fast_score(g.bk) >= fast_score(g.bn) ? 1 : 0;
        g.kchunk        = (g.K + 31) / 32 * 32;
        const bool swap = (g.cm.s0 == 1 && g.cm.c >= 16) && !(g.cn.s0 == 1 && g.cn.c >= 16);
        build[swap ? GroupedGemm::STAGED_SWAPPED : GroupedGemm::STAGED].add(g, grouped_tiles(g, TileCfg::T64x64), g.K);
    }
    std::vector<GroupedGemm> out;
    size_t                   store_off = 0;
    for(int k = 0; k < GroupedGemm::N_KINDS; ++k) {
        const GroupBuilder &b = build[k];
        if(b.descs.empty()) continue;
        GroupedGemm gg;
        gg.dtype              = members[0].dtype;
        gg.kind               = static_cast<GroupedGemm::Kind>(k);
        gg.cfg                = tiled;
        gg.ngemm              = static_cast<int>(b.starts.size()) - 1;
        gg.workgroups         = b.starts.back();
        gg.max_k              = b.max_k;
        gg.lds                = b.lds;
        const size_t starts_b = sizeof(int) * b.starts.size();
        if(store) {
            char *base = static_cast<char *>(store);
            gg.owned   = false;
            gg.descs   = base + store_off;
            store_off += aligned256(b.descs.size());
            gg.starts = reinterpret_cast<int *>(base + store_off);
            store_off += aligned256(starts_b);
        } else if(hipMalloc(&gg.descs, b.descs.size()) != hipSuccess || hipMalloc(reinterpret_cast<void **>(&gg.starts), starts_b) != hipSuccess) {
            (void) hipGetLastError();
            out.push_back(gg);
            grouped_free(out);
            throw Error(DMRG_ERR_OOM, "grouped GEMM: descriptor allocation failed");
        }
        out.push_back(gg);
        DMRG_HIP_CHECK(hipMemcpy(gg.descs, b.descs.data(), b.descs.size(), hipMemcpyHostToDevice));
        DMRG_HIP_CHECK(hipMemcpy(gg.starts, b.starts.data(), starts_b, hipMemcpyHostToDevice));
    }
    return out;
}

template <typename R, bool CPLX>
static void grouped_staged(const GroupedGemm &g, hipStream_t s) {
    constexpr int E  = static_cast<int>(sizeof(elem_t<R, CPLX>));
    constexpr int BK = E == 4 ? 32 : 16;
    const dim3    grid(g.workgroups), block(256);
    const auto   *d = static_cast<const GemmDesc *>(g.descs);
    if(g.kind == GroupedGemm::STAGED_SWAPPED)
        hipLaunchKernelGGL((gemm_grouped_kernel<R, CPLX, 64, 64, BK, 2, 2, true>), grid, block, 0, s, d, g.starts, g.ngemm);
    else hipLaunchKernelGGL((gemm_grouped_kernel<R, CPLX, 64, 64, BK, 2, 2, false>), grid, block, 0, s, d, g.starts, g.ngemm);
}

static void grouped_pipelined(const GroupedGemm &g, hipStream_t s) {
    const auto       *d     = static_cast<const pipe::Desc *>(g.descs);
    const pipe::Shape shape = shape_of(g.cfg, g.dtype);
    switch(g.dtype) {
        case DMRG_FP64: pipe::launch_grouped_f64(d, g.starts, g.ngemm, g.workgroups, shape, s); break;
        case DMRG_CX64: pipe::launch_grouped_c128(d, g.starts, g.ngemm, g.workgroups, shape, s); break;
        case DMRG_FP32: pipe::launch_grouped_f32(d, g.starts, g.ngemm, g.workgroups, shape, s); break;
        case DMRG_CX32: pipe::launch_grouped_c64(d, g.starts, g.ngemm, g.workgroups, shape, s); break;
    }
}

void grouped_launch(const GroupedGemm &g, hipStream_t s) {
    if(g.workgroups <= 0) return;
    if(g.kind == GroupedGemm::PIPELINED) grouped_pipelined(g, s);
    else if(g.kind == GroupedGemm::STREAMED)
        stream::launch_grouped(g.dtype, static_cast<const stream::Desc *>(g.descs), g.starts, g.ngemm, g.workgroups, g.max_k, g.lds, s);
    else {
        switch(g.dtype) {
            case DMRG_FP64: grouped_staged<double, false>(g, s); break;
            case DMRG_CX64: grouped_staged<double, true>(g, s); break;
            case DMRG_FP32: grouped_staged<float, false>(g, s); break;
            case DMRG_CX32: grouped_staged<float, true>(g, s); break;
        }
    }
    DMRG_HIP_CHECK(hipGetLastError());
}

void grouped_free(std::vector<GroupedGemm> &gg) {
    for(auto &g : gg) {
        if(g.owned && g.descs) (void) hipFree(g.descs);
        if(g.owned && g.starts) (void) hipFree(g.starts);
        g.descs  = nullptr;
        g.starts = nullptr;
    }
    gg.clear();
}

static std::vector<LaunchPlan> candidates(const GemmDesc &g) {
    std::vector<LaunchPlan> c;
    if(stream::takes(g)) c.push_back({TileCfg::SMALLK, 1});
    if(g.M <= 32) c.push_back({TileCfg::T16x128, 1});
    // The pipelined plans within a third of the cheapest.
    const auto ranked = ranked_plans(g);
    for(const auto &r : ranked)
        if(r.first <= 1.34 * ranked.front().first) c.push_back(r.second);
    // Hybrid plans: as many tile columns as occupy every CU equally without K slicing, the remaining ones sliced over K.
    if(g.part && g.batch == 1 && g.K >= 128) {
        for(TileCfg t : {TileCfg::T64x64, TileCfg::T64x32}) {
            if(shape_of(t, g.dtype) != (t == TileCfg::T64x64 ? pipe::S64x64 : pipe::S64x32)) continue;
            const CfgShape sh = cfg_shape(t);
            const int      tm = (g.M + sh.BM - 1) / sh.BM, tn = (g.N + sh.BN - 1) / sh.BN;
            const int64_t  cus = device_cu_count(), whole = static_cast<int64_t>(tm) * tn / cus * cus / tm;
            if(whole <= 0 || whole >= tn) continue;
            const int nsplit = static_cast<int>(whole * sh.BN);
            for(int ks2 : {2, 3, 4, 8}) {
                if(g.K < 64 * ks2 || g.part_capacity < static_cast<int64_t>(g.M) * (g.N - nsplit) * ks2) continue;
                c.push_back({t, 1, nsplit, ks2});
            }
        }
    }
    return c;
}

static LaunchPlan tune(const GemmDesc &g, hipStream_t stream) {
    const auto cands = candidates(g);
    hipEvent_t e0, e1;
    DMRG_HIP_CHECK(hipEventCreate(&e0));
    DMRG_HIP_CHECK(hipEventCreate(&e1));
    std::vector<float> t(cands.size(), 1e30f);
    try {
        // Two passes over the candidates, the fastest of 3 launches in each: the clocks move by several per cent within
        // one pass.
        for(int pass = 0; pass < 2; ++pass)
            for(size_t c = 0; c < cands.size(); ++c) {
                if(pass == 0) launch_plan(g, cands[c], stream); // warm-up (first-use code load, caches)
                for(int r = 0; r < 3; ++r) {
                    DMRG_HIP_CHECK(hipEventRecord(e0, stream));
                    launch_plan(g, cands[c], stream);
                    DMRG_HIP_CHECK(hipEventRecord(e1, stream));
                    DMRG_HIP_CHECK(hipEventSynchronize(e1));
                    float ms = 0;
                    DMRG_HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
                    t[c] = std::min(t[c], ms);
                }
            }
    } catch(...) {
        (void) hipEventDestroy(e0);
        (void) hipEventDestroy(e1);
        throw;
    }
    // The fastest, but an earlier candidate (they are in the model's order) that is within 2 % of it.
    const float fastest = *std::min_element(t.begin(), t.end());
    LaunchPlan  best    = cands[0];
    for(size_t c = 0; c < cands.size(); ++c)
        if(t[c] <= 1.02f * fastest) {
            best = cands[c];
            break;
        }
    (void) hipEventDestroy(e0);
    (void) hipEventDestroy(e1);
    return best;
}

// Optional persistent cache: with DMRG_TUNE_CACHE=<file>, tuned plans are loaded at first use and each new
// plan is appended, so that separate processes (e.g. profiler passes) launch the same kernels.
static const char *tune_cache_path() {
    static const char *p = std::getenv("DMRG_TUNE_CACHE");
    return (p && *p) ? p : nullptr;
}
static void load_tune_cache_locked() {
    static bool loaded = false;
    if(loaded) return;
    loaded = true;
    const char *path = tune_cache_path();
    if(!path) return;
    FILE *f = std::fopen(path, "r");
    if(!f) return;
    char line[1024];
    while(std::fgets(line, sizeof(line), f)) {
        std::string l(line);
        const size_t sp = l.rfind(' ');
        if(sp == std::string::npos) continue;
        int cfg = 0, ks = 1, nsplit = 0, ks2 = 1;
        if(std::sscanf(l.c_str() + sp + 1, "%d:%d:%d:%d", &cfg, &ks, &nsplit, &ks2) < 2) continue;
        g_tuned[l.substr(0, sp)] = LaunchPlan{static_cast<TileCfg>(cfg), ks, nsplit, ks2};
    }
    std::fclose(f);
}
static void append_tune_cache_locked(const std::string &key, const LaunchPlan &p) {
    const char *path = tune_cache_path();
    if(!path) return;
    if(FILE *f = std::fopen(path, "a")) {
        std::fprintf(f, "%s %d:%d:%d:%d\n", key.c_str(), static_cast<int>(p.cfg), p.ksplit, p.nsplit, p.ksplit2);
        std::fclose(f);
    }
}

void set_autotune(int on) {
    g_autotune = on;
    ++g_plan_state;
}
void set_tune_min_macs(int64_t macs) {
    g_tune_min_macs = macs;
    ++g_plan_state;
}
int  autotune_enabled() { return g_autotune; }
void set_plan_override(int cfg, int ks, int nsplit, int ks2) {
    g_override_cfg    = cfg;
    g_override_ks     = ks;
    g_override_nsplit = nsplit;
    g_override_ks2    = ks2;
    ++g_plan_state;
}
void clear_tuning() {
    std::lock_guard<std::mutex> lock(g_tune_mu);
    g_tuned.clear();
    ++g_plan_state;
}
int tuned_entries() {
    std::lock_guard<std::mutex> lock(g_tune_mu);
    return static_cast<int>(g_tuned.size());
}

static thread_local bool g_tls_no_tune = false;
NoTuneScope::NoTuneScope() : prev_(g_tls_no_tune) { g_tls_no_tune = true; }
NoTuneScope::~NoTuneScope() { g_tls_no_tune = prev_; }

// Plans of GEMMs already met on this thread, by everything but their pointers: planning and describing a GEMM takes
// about 3 us on the host, as much as a launch. An entry is good for one state of the tuner (g_plan_state); at most
// PLAN_CACHE_MAX entries of about 700 bytes are kept, and given back when the thread ends. A full cache gives up one entry at
// random: a stream that cycles through more shapes than it holds keeps hits in proportion (none if the oldest went, or all).
constexpr size_t PLAN_CACHE_MAX = 4096;
struct PlanKey {
    int64_t v[32];
    bool    operator==(const PlanKey &o) const { return std::memcmp(v, o.v, sizeof(v)) == 0; }
};
struct PlanKeyHash {
    size_t operator()(const PlanKey &k) const {
        uint64_t h = 0x9E3779B97F4A7C15ull;
        for(int64_t x : k.v) h = (h ^ static_cast<uint64_t>(x)) * 0xD6E8FEB86659FD93ull, h ^= h >> 32;
        return static_cast<size_t>(h);
    }
};
struct PlanEntry {
    uint64_t   state;
    bool       pipelined; // p is complete; otherwise plan is launched as it stands
    LaunchPlan plan;
    Prepared   p;
};
static PlanKey plan_key(const GemmDesc &g) {
    PlanKey k{};
    int     n = 0;
    auto    add = [&](int64_t x) { k.v[n++] = x; };
    add(static_cast<int64_t>(g.dtype) | static_cast<int64_t>(g.conjA != 0) << 8 | static_cast<int64_t>(g.conjB != 0) << 9 |
        static_cast<int64_t>(g.accumulate != 0) << 10 | static_cast<int64_t>(g.part != nullptr) << 11 |
        static_cast<int64_t>(g.xcd_remap != 0) << 12 | static_cast<int64_t>(reinterpret_cast<uintptr_t>(g.A) & 3) << 16 |
        static_cast<int64_t>(reinterpret_cast<uintptr_t>(g.B) & 3) << 18);
    add(static_cast<int64_t>(g.M) << 32 | static_cast<uint32_t>(g.N));
    add(static_cast<int64_t>(g.K) << 32 | static_cast<uint32_t>(g.batch));
    for(const Idx2 &x : {g.am, g.ak, g.bk, g.bn, g.cm, g.cn}) {
        add(x.s0);
        add(x.s1);
        add(x.c);
    }
    add(g.a_batch), add(g.b_batch), add(g.c_batch), add(g.part_capacity);
    return k;
}

void gemm(const GemmDesc &gin, hipStream_t stream, TileCfg cfg, int ksplit) {
    if(gin.M <= 0 || gin.N <= 0 || gin.batch <= 0) return;
    GemmDesc g = gin;
    // K == 0 is legal: every load is skipped, the K loop is empty and C is written with zeros.
    if(g.K < 0) g.K = 0;
    if(g.K == 0 && g.accumulate) return;
    DMRG_REQUIRE(static_cast<int64_t>(g.M) * g.N < (int64_t(1) << 31), DMRG_ERR_DIMS, "gemm: output too large for 32-bit tile indexing");
    g.a_fast_m = fast_score(g.am) >= fast_score(g.ak) ? 1 : 0;
    g.b_fast_k = fast_score(g.bk) >= fast_score(g.bn) ? 1 : 0;
    if(g_override_cfg >= 0) {
        launch_plan(g, {static_cast<TileCfg>(g_override_cfg), std::max(1, g_override_ks), g_override_nsplit, std::max(1, g_override_ks2)}, stream);
        return;
    }
    if(cfg != TileCfg::AUTO) {
        launch_plan(g, {cfg, std::max(1, ksplit)}, stream);
        return;
    }
    static thread_local std::unordered_map<PlanKey, PlanEntry, PlanKeyHash> cache;
    const uint64_t state = g_plan_state.load(std::memory_order_acquire);
    const PlanKey  ck    = plan_key(g);
    if(ksplit <= 0) {
        const auto it = cache.find(ck);
        if(it != cache.end() && it->second.state == state) {
            PlanEntry &e = it->second;
            if(!e.pipelined) {
                launch_plan(g, e.plan, stream);
                return;
            }
            const GemmDesc h = oriented(g);
            e.p.l.d.a.p  = h.A;
            e.p.l.d.b.p  = h.B;
            e.p.l.d.C    = h.C;
            e.p.l.d.part = h.part;
            run_pipelined(h, e.p, stream);
            return;
        }
    }
    // Tuning needs synchronisation, so it is skipped for accumulating GEMMs (repeated launches would
    // add up) and while the stream is being captured into a graph.
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    DMRG_HIP_CHECK(hipStreamIsCapturing(stream, &cs));
    // Only large GEMMs are timed (at least g_tune_min_macs multiply-adds, or g_tune_min_macs / 16 bytes of
    // operands for the memory-bound ones): a sweep or a request stream meets thousands of small shapes once
    // each, whose tuning (dozens of timed, synchronised launches) costs more than any plan saves.
    const double macs  = static_cast<double>(g.M) * g.N * std::max(g.K, 1) * g.batch;
    const double bytes = (static_cast<double>(g.M) * g.K + static_cast<double>(g.K) * g.N + static_cast<double>(g.M) * g.N) *
                         g.batch * static_cast<double>(dtype_size(g.dtype));
    const bool   large = macs >= static_cast<double>(g_tune_min_macs) || bytes * 16.0 >= static_cast<double>(g_tune_min_macs);
    const bool   tunable  = g_autotune && !g.accumulate && large;
    const bool   can_tune = tunable && cs == hipStreamCaptureStatusNone && !g_tls_no_tune;
    std::string  key;
    LaunchPlan   p;
    bool         found = false;
    {
        std::lock_guard<std::mutex> lock(g_tune_mu);
        load_tune_cache_locked();
        if(can_tune || !g_tuned.empty()) key = tune_key(g);
        auto it = g_tuned.find(key);
        if(it != g_tuned.end()) {
            p     = it->second;
            found = true;
        }
    }
    if(!found) {
        p = can_tune ? tune(g, stream) : heuristic_plan(g);
        if(can_tune) {
            std::lock_guard<std::mutex> lock(g_tune_mu);
            g_tuned[key] = p;
            append_tune_cache_locked(key, p);
        }
    }
    if(ksplit > 0) {
        launch_plan(g, LaunchPlan{p.cfg, ksplit}, stream);
        return;
    }
    // Kept unless a later call may time this GEMM and decide otherwise.
    if(found || can_tune || !tunable) {
        if(cache.size() >= PLAN_CACHE_MAX && cache.find(ck) == cache.end()) {
            static thread_local uint32_t draw = 1;
            size_t                       b    = (draw = draw * 1664525u + 1013904223u) % cache.bucket_count();
            while(cache.bucket_size(b) == 0) b = (b + 1) % cache.bucket_count();
            const PlanKey gone = cache.begin(b)->first;
            cache.erase(gone);
        }
        PlanEntry        e{state, false, p, {}};
        const pipe::Shape shape = shape_of(p.cfg, g.dtype);
        const bool        slices = p.ksplit <= 1 || (g.part && g.part_capacity >= static_cast<int64_t>(g.M) * g.N * g.batch * p.ksplit);
        if(shape != pipe::N_SHAPES && p.nsplit <= 0) e.pipelined = prepare_pipelined(oriented(g), shape, slices ? p.ksplit : 1, e.p);
        cache[ck] = e;
        if(e.pipelined) {
            run_pipelined(oriented(g), e.p, stream);
            return;
        }
    }
    launch_plan(g, p, stream);
}

// ---------------------------------------------------------------------------------------
// Block one-sided Jacobi SVD steps on the matrix cores. Blocks of 16 columns of W (m x npad, ld m) and V
// (n x npad, ld n) are paired by the circle method (round r over nbp players, pair = blockIdx.x, the lower block
// first); a pair's 32 columns are X = [block P, block Q], addressed as one index map with a gap between the two
// blocks. The descriptors are built in the kernel, so a round costs one launch per step and no host work.

namespace {

__device__ inline void bj_block_pair(int nbp, int r, int i, int &P, int &Q) {
    if(i == 0) {
        P = r % (nbp - 1);
        Q = nbp - 1;
    } else {
        P = (r + i) % (nbp - 1);
        Q = (r - i + (nbp - 1)) % (nbp - 1);
    }
    if(P > Q) {
        const int t = P;
        P           = Q;
        Q           = t;
    }
}

constexpr uint32_t BJ_PLAIN = 0x7fffffffu;

// Partial Gram matrices G = X^H X over the row chunks [y rows_per, (y + 1) rows_per): part[(pair ks + y)][i + 32 j].
template <typename R, bool CPLX>
__global__ __launch_bounds__(256) void bj_gram_kernel(int m, int nb, int nbp, int r, const void *W, int ks, int rows_per, void *part) {
    int P, Q;
    bj_block_pair(nbp, r, blockIdx.x, P, Q);
    if(Q >= nb) return; // the padding block of an odd block count
    using E = elem_t<R, CPLX>;
    GemmDesc      g;
    const int64_t gap = static_cast<int64_t>(Q - P) * 16 * m;
    g.M = 32, g.N = 32, g.K = m, g.batch = 1;
    g.A     = static_cast<const E *>(W) + static_cast<int64_t>(P) * 16 * m;
    g.am    = Idx2{m, gap, 16u};
    g.ak    = Idx2{1, 0, BJ_PLAIN};
    g.conjA = CPLX ? 1 : 0;
    g.B = g.A, g.bk = g.ak, g.bn = g.am;
    g.a_fast_m = 0, g.b_fast_k = 1, g.xcd_remap = 0;
    g.ksplit = ks, g.kchunk = rows_per;
    g.part   = static_cast<E *>(part) + static_cast<int64_t>(blockIdx.x) * ks * 32 * 32;
    g.C      = g.part;
    g.cm     = Idx2{1, 0, BJ_PLAIN};
    g.cn     = Idx2{32, 0, BJ_PLAIN};
    gemm_body<R, CPLX, 32, 32, 16, 2, 2, false, false>(g, 0, blockIdx.y, 0);
}

// X <- X Q in place (Q: qbuf[pair], 32 x 32 column-major) for the pairs whose inner solve rotated: row tiles
// [0, tw) of W, then those of V. A workgroup owns its 64 rows of all 32 columns and reads them (both K stages)
// before it writes them.
template <typename R, bool CPLX>
__global__ __launch_bounds__(256) void bj_update_kernel(int m, int n, int nb, int nbp, int r, void *W, void *V, const void *qbuf,
                                                        const int *rotated, int tw) {
    int P, Q;
    bj_block_pair(nbp, r, blockIdx.x, P, Q);
    if(Q >= nb || !rotated[blockIdx.x]) return;
    using E = elem_t<R, CPLX>;
    const bool    on_w = static_cast<int>(blockIdx.y) < tw;
    const int     ld   = on_w ? m : n;
    E            *base = static_cast<E *>(on_w ? W : V) + static_cast<int64_t>(P) * 16 * ld;
    const int64_t gap  = static_cast<int64_t>(Q - P) * 16 * ld;
    GemmDesc      g;
    g.M = ld, g.N = 32, g.K = 32, g.batch = 1;
    g.A  = base;
    g.am = Idx2{1, 0, BJ_PLAIN};
    g.ak = Idx2{ld, gap, 16u};
    g.B  = static_cast<const E *>(qbuf) + static_cast<int64_t>(blockIdx.x) * 32 * 32;
    g.bk = Idx2{1, 0, BJ_PLAIN};
    g.bn = Idx2{32, 0, BJ_PLAIN};
    g.C  = base;
    g.cm = Idx2{1, 0, BJ_PLAIN};
    g.cn = Idx2{ld, gap, 16u};
    g.a_fast_m = 1, g.b_fast_k = 1, g.xcd_remap = 0, g.ksplit = 1, g.kchunk = 32;
    gemm_body<R, CPLX, 64, 32, 16, 2, 2, false, false>(g, on_w ? blockIdx.y : blockIdx.y - tw, 0, 0);
}

} // namespace

void bj_gram_mfma(dmrg_dtype t, int m, int npad, int nbp, int r, const void *W, int ks, int rows_per, void *part, hipStream_t s) {
    const dim3 grid(nbp / 2, ks), block(256);
    const int  nb = npad / 16;
    if(t == DMRG_CX64) hipLaunchKernelGGL((bj_gram_kernel<double, true>), grid, block, 0, s, m, nb, nbp, r, W, ks, rows_per, part);
    else hipLaunchKernelGGL((bj_gram_kernel<double, false>), grid, block, 0, s, m, nb, nbp, r, W, ks, rows_per, part);
}

void bj_update_mfma(dmrg_dtype t, int m, int n, int npad, int nbp, int r, void *W, void *V, const void *qbuf, const int *rotated,
                    hipStream_t s) {
    const int  tw = (m + 63) / 64, tv = (n + 63) / 64, nb = npad / 16;
    const dim3 grid(nbp / 2, tw + tv), block(256);
    if(t == DMRG_CX64)
        hipLaunchKernelGGL((bj_update_kernel<double, true>), grid, block, 0, s, m, n, nb, nbp, r, W, V, qbuf, rotated, tw);
    else hipLaunchKernelGGL((bj_update_kernel<double, false>), grid, block, 0, s, m, n, nb, nbp, r, W, V, qbuf, rotated, tw);
}

} // namespace dmrg
