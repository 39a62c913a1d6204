// Pipelined GEMM body: tiles go from HBM/L2 straight into LDS (buffer loads with an LDS destination), NS stages deep.
//
//   C[b][m,n] (+)= sum_k op(A)[b][m,k] * op(B)[b][k,n], operands addressed through two-level index maps (Idx2).
//
// What bounds it is the matrix core's issue: a vector instruction between the MFMAs of a wavefront does not overlap with
// them on gfx950 (measured on FP64 16x16x4, 64 clocks each: 4 to 5 clocks per instruction and about 9 for the switch, also
// with two wavefronts per SIMD; scalar instructions, barriers and LDS reads at immediate offsets are nearly free). So the
// loop over K has none but the complex sums: loads take no address arithmetic (a uniform base moves from stage to stage),
// no masks (only the last stage of a K chunk is masked) and no register copies on the way to LDS, and conjugation is a sign
// in those sums and the epilogue. Loads and LDS reads are spread between the MFMAs one by one: issued together, all
// wavefronts wait for the same queue with their matrix cores idle (chi = 512 leg 3 of an earlier form: 146 us together, 124 us spread).
//
// The unit of all traffic is 16 bytes: U = 16 / sizeof(element) elements that are consecutive along the operand's
// non-K index (R orientation) or along K (K orientation). A stage holds an operand tile as blocks of 16 units of the
// non-K index; a block is stored k-major or r-major, whichever lets the 64 lanes of a load walk memory in order (the
// choice only changes addresses). An MFMA fragment is one ds_read_b128 per lane; a 16-lane group always covers 256
// contiguous or XOR-spread bytes, so reads are free of bank conflicts in both orders.
//
// Measured (MI355X, microseconds, register-staged kernels -> here): complex FP64 chi = 512, D = 5 leg 1 (1024x2560x512)
// 153 -> 123, leg 3 (1024x512x2560) 148 -> 118, complex FP32 leg 1 92 -> 68, leg 3 80 -> 65 (kernel traces of 200 matvecs;
// the first twenty launches after an idle spell take 15 to 20 % longer); complex 4096x4096x4096 97 TFLOP/s, of 98 that the
// three-product form reaches at the measured MFMA rate; real FP64 2048x1024x5120 380 -> 301 (71 TFLOP/s); real FP32
// 640x301x1505 47 -> 15. No LDS bank conflict is counted on these legs.
#pragma once
#include "common.hpp"

#include <type_traits>

namespace dmrg {
namespace pipe {

constexpr uint32_t OOB = 0x80000000u; // offset past every buffer range below: the load writes zeros to LDS

// One operand as the kernel sees it. All offsets in bytes. K is walked in stages of BK: Kout chunks of Kin consecutive
// values, the last stage of a chunk padded with zeros, so that the step from one stage to the next is one uniform offset.
struct Operand {
    const void *p;
    int64_t     batch;        // bytes between batch entries
    Idx2        r, k;         // the non-K index map; the K map inside one stage
    uint32_t    rmul, rsh;    // i / r.c = umulhi(i, rmul) >> rsh for i < 2^31
    uint32_t    kmul, ksh;    // the same for k.c
    int64_t     kstep, kwrap; // from one stage to the next; added to it at the end of a chunk
    int32_t     R;            // extent of the non-K index
    int32_t     korder;       // 1: consecutive lanes walk K, 0: they walk the non-K index
    int32_t     sep_r;        // the tile origin's offset separates from the in-tile offset
    float       sign;         // -1: conjugate (1 otherwise)
};
struct Desc {
    Operand  a, b;
    void    *C;
    Idx2     cm, cn; // element strides
    int64_t  c_batch;
    void    *part;
    int32_t  M, N;
    int32_t  Kin, stages_per_chunk, stages, stages_per_slice; // stages: Kout chunks of stages_per_chunk
    int32_t  accumulate, ksplit, xcd_remap;
    int32_t  wide; // loads of 16 bytes per lane (else 4); read by grouped launches only
};

// The last i with start[i] <= x.
__device__ __forceinline__ int group_of(const int *start, int n, int x) {
    int lo = 0, hi = n - 1;
    while(lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if(start[mid] <= x) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

template <int N, typename F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr(N > 0) {
        static_for<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

__device__ __forceinline__ uint32_t uni(uint32_t x) { return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(x))); }
__device__ __forceinline__ const char *uni(const char *p) {
    const uint64_t v = reinterpret_cast<uint64_t>(p);
    return reinterpret_cast<const char *>(static_cast<uint64_t>(uni(static_cast<uint32_t>(v))) |
                                          (static_cast<uint64_t>(uni(static_cast<uint32_t>(v >> 32))) << 32));
}

// RO: units run along the non-K index. W: bytes per lane and load (16; 4 where a unit is not contiguous in memory).
template <typename E, int RT, int BK, bool RO, int W, int NW>
struct Loader {
    static constexpr int ES    = static_cast<int>(sizeof(E));
    static constexpr int U     = 16 / ES;
    static constexpr int RN    = RO ? RT / U : RT; // units of the non-K index
    static constexpr int KN    = RO ? BK : BK / U; // units of K
    static constexpr int BYTES = RT * BK * ES;
    static constexpr int SLOTS = BYTES / (64 * W); // loads of one wavefront per stage tile
    static constexpr int L     = SLOTS / NW;
    static_assert(RN % 16 == 0 && SLOTS % NW == 0, "stage does not divide over the wavefronts");
    static_assert((KN & (KN - 1)) == 0, "K units per stage");

    uint32_t    voff[L];
    const char *base; // of the next stage
    uint32_t    wave, lane;

    static __device__ __forceinline__ uint32_t swz(uint32_t rl) { return KN >= 16 ? (rl & (KN - 1)) : ((rl / (16 / (KN < 16 ? KN : 16))) & (KN - 1)); }
    // Unit u of the stage -> its first element's non-K index and K index within the tile.
    static __device__ __forceinline__ void unit(uint32_t u, bool korder, uint32_t &r, uint32_t &k) {
        const uint32_t blk = u / (16 * KN), in = u % (16 * KN);
        uint32_t       rl, kx;
        if(korder) rl = in / KN, kx = (in % KN) ^ swz(rl);
        else rl = in % 16, kx = in / 16;
        r = (blk * 16 + rl) * (RO ? U : 1);
        k = kx * (RO ? 1 : U);
    }
    // Byte offset of unit (rl of a 16-unit block, kx) inside its block.
    static __device__ __forceinline__ int inner(bool korder, uint32_t rl, uint32_t kx) {
        return korder ? (rl * KN + (kx ^ swz(rl))) * 16 : (kx * 16 + rl) * 16;
    }
    // This lane's element (r, k) and byte within it for load e.
    __device__ __forceinline__ void mine(const Operand &o, int e, uint32_t &r, uint32_t &k, uint32_t &byte) const {
        const uint32_t slot = wave + NW * e;
        if constexpr(W == 16) {
            unit(slot * 64 + lane, o.korder, r, k);
            byte = 0;
        } else {
            unit(slot * 16 + lane / 4, o.korder, r, k);
            const uint32_t el = lane % 4 * 4 / ES;
            byte              = lane % 4 * 4 % ES;
            if constexpr(RO) r += el;
            else k += el;
        }
    }
    // Offset of index i, without a division (plain maps have a chunk past every index).
    static __device__ __forceinline__ uint32_t off32(const Idx2 &x, uint32_t mul, uint32_t sh, uint32_t i) {
        const uint32_t d = __umulhi(i, mul) >> sh;
        return (i - d * x.c) * static_cast<uint32_t>(x.s0) + d * static_cast<uint32_t>(x.s1);
    }
    static __device__ __forceinline__ int64_t off64(const Idx2 &x, uint32_t mul, uint32_t sh, uint32_t i) {
        const uint32_t d = __umulhi(i, mul) >> sh;
        return static_cast<int64_t>(i - d * x.c) * x.s0 + static_cast<int64_t>(d) * x.s1;
    }

    // First stage: number st of chunk ch.
    __device__ __forceinline__ void init(const Operand &o, const Desc &g, int64_t b, uint32_t r0, int ch, int st, uint32_t tid) {
        wave = uni(tid >> 6);
        lane = tid & 63;
        base = static_cast<const char *>(o.p) + b * o.batch + st * o.kstep + ch * (g.stages_per_chunk * o.kstep + o.kwrap);
        if(o.sep_r) base += off64(o.r, o.rmul, o.rsh, r0);
        base = uni(base);
        const uint32_t rb = o.sep_r ? 0 : r0;
#pragma unroll
        for(int e = 0; e < L; ++e) {
            uint32_t r, k, byte;
            mine(o, e, r, k, byte);
            const uint32_t v = off32(o.r, o.rmul, o.rsh, rb + r) + off32(o.k, o.kmul, o.ksh, k) + byte;
            voff[e]          = r0 + r < static_cast<uint32_t>(o.R) ? v : OOB;
        }
    }
    // Load e of the next stage. FULL: all of its K values exist, and the load takes no vector instruction besides itself;
    // otherwise the first left values exist and the others become zeros.
    template <int e, bool FULL>
    __device__ __forceinline__ void issue(const Operand &o, char *stage, int left) const {
        const auto rs  = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(base), static_cast<short>(0), 0x7fffffff, 0x00020000);
        auto      *dst = (__attribute__((address_space(3))) void *) (stage + (wave + NW * e) * (64 * W));
        uint32_t   v   = voff[e];
        if constexpr(!FULL) {
            uint32_t r, k, byte;
            mine(o, e, r, k, byte);
            v = static_cast<int>(k) < left ? v : OOB;
        }
        if constexpr(W == 16) __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, dst, 16, static_cast<int>(v), 0, 0, 0);
        else __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, dst, 4, static_cast<int>(v), 0, 0, 0);
    }
    __device__ __forceinline__ void advance(const Operand &o, bool wrap) { base += o.kstep + (wrap ? o.kwrap : 0); }
};

// s_waitcnt vmcnt(vm) lgkmcnt(0); vmcnt counts to 63, so that deeper pipelines wait for a little more than they need.
constexpr int waitcnt(int vm) {
    const int v = vm > 63 ? 63 : vm;
    return (v & 15) | ((v >> 4) << 14) | (7 << 4);
}

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float  v4f __attribute__((ext_vector_type(4)));
template <typename R>
struct mma;
template <>
struct mma<double> {
    using acc                                  = v4d;
    __device__ static inline acc op(double a, double b, acc c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
    __device__ static inline int row(int g, int v) { return g + 4 * v; }
};
template <>
struct mma<float> {
    using acc                                = v4f;
    __device__ static inline acc op(float a, float b, acc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
    __device__ static inline int row(int g, int v) { return 4 * g + v; }
};

template <typename E>
struct alignas(16) Unit {
    E e[16 / sizeof(E)];
};

// stage(i): the LDS memory of stage i (an integral constant), BM BK + BN BK elements.
template <typename R, bool CPLX, int BM, int BN, int BK, int WM, int WN, int NS, bool AR, bool BR, int W, typename Stage>
__device__ __forceinline__ void body(const Desc &g, int bx, int split, int b, Stage &&stage) {
    using E            = std::conditional_t<CPLX, cpx<R>, R>;
    using MM           = mma<R>;
    constexpr int U    = 16 / static_cast<int>(sizeof(E));
    constexpr int NW   = WM * WN;
    constexpr int TM   = BM / (16 * WM), TN = BN / (16 * WN);
    constexpr int NACC = CPLX ? 3 : 1; // complex: sum ar*br, sum ai*bi, sum (ar+ai)*(br+bi)
    using LA           = Loader<E, BM, BK, AR, W, NW>;
    using LB           = Loader<E, BN, BK, BR, W, NW>;
    static_assert(!AR || TM % U == 0, "R orientation needs whole units per wave");
    static_assert(!BR || TN % U == 0, "R orientation needs whole units per wave");
    constexpr int LPS = LA::L + LB::L; // loads per wave and stage
    constexpr int DEP = NS - 1;        // stages in flight
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave % WM, wn = wave / WM;
    const int lg = lane >> 4, ll = lane & 15;

    const int tilesM = (g.M + BM - 1) / BM, tilesN = (g.N + BN - 1) / BN, total = tilesM * tilesN;
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
    const int m0 = mt * BM, n0 = nt * BN;
    const int first = split * g.stages_per_slice;
    const int numK  = min(g.stages, first + g.stages_per_slice) - first;
    int       st    = first % g.stages_per_chunk; // the next stage to load, within its chunk

    LA la;
    LB lb;
    la.init(g.a, g, b, m0, first / g.stages_per_chunk, st, tid);
    lb.init(g.b, g, b, n0, first / g.stages_per_chunk, st, tid);
    // Fragment addresses: per K position of the stage, the lane's offset in a 16-unit block.
    constexpr int NQ = BK / (4 * U);
    int           fa_off[NQ * (AR ? U : 1)], fb_off[NQ * (BR ? U : 1)];
    {
        const int wa = wm * (AR ? TM / U : TM), wb = wn * (BR ? TN / U : TN);
#pragma unroll
        for(int q = 0; q < NQ; ++q) {
            if constexpr(AR && U > 1)
                for(int j = 0; j < U; ++j) fa_off[q * U + j] = wa * LA::KN * 256 + LA::inner(g.a.korder, ll, (q * 4 + lg) * U + j);
            else fa_off[q] = wa * LA::KN * 256 + LA::inner(g.a.korder, ll, q * 4 + lg);
            if constexpr(BR && U > 1)
                for(int j = 0; j < U; ++j) fb_off[q * U + j] = wb * LB::KN * 256 + LB::inner(g.b.korder, ll, (q * 4 + lg) * U + j);
            else fb_off[q] = wb * LB::KN * 256 + LB::inner(g.b.korder, ll, q * 4 + lg);
        }
    }

    typename MM::acc acc[NACC][TM][TN];
#pragma unroll
    for(int c = 0; c < NACC; ++c)
#pragma unroll
        for(int i = 0; i < TM; ++i)
#pragma unroll
            for(int j = 0; j < TN; ++j) acc[c][i][j] = typename MM::acc{0, 0, 0, 0};
    // Single precision: the sums are kept in two levels, of FLUSH rounds of NS stages (128 values of K) and of those,
    // so that the rounding error does not grow with the length of K. Complex matvec at chi = 512, D = 5 against 64 bits:
    // 1.1e-6 in one level, 4.2e-7 in two (7.4e-7 for the register-staged kernels with 8 K slices).
    constexpr bool TWO   = sizeof(R) == 4;
    constexpr int  FLUSH = 128 / (BK * NS) > 0 ? 128 / (BK * NS) : 1;
    typename MM::acc tot[TWO ? NACC : 1][TWO ? TM : 1][TWO ? TN : 1];
    auto             flush = [&](bool clear) {
        if constexpr(TWO) {
#pragma unroll
            for(int c = 0; c < NACC; ++c)
#pragma unroll
                for(int i = 0; i < TM; ++i)
#pragma unroll
                    for(int j = 0; j < TN; ++j) {
                        tot[c][i][j] += acc[c][i][j];
                        acc[c][i][j] = clear ? typename MM::acc{0, 0, 0, 0} : tot[c][i][j];
                    }
        }
    };
    if constexpr(TWO) {
#pragma unroll
        for(int c = 0; c < NACC; ++c)
#pragma unroll
            for(int i = 0; i < TM; ++i)
#pragma unroll
                for(int j = 0; j < TN; ++j) tot[c][i][j] = typename MM::acc{0, 0, 0, 0};
    }

    // Fragments of one K position q of a stage: U consecutive K values of every block of the wave, and for complex
    // elements their re + im.
    struct Frag {
        E a[U][TM], b[U][TN];
    };
    // Read r of the TM + TN that make up position q.
    auto fetch = [&](const char *st, auto q_, auto r_, Frag &f) {
        constexpr int q = decltype(q_)::value, r = decltype(r_)::value;
        if constexpr(r < TM) {
            if constexpr(AR) {
                constexpr int   j = r % U, i = r / U;
                const Unit<E>   u = *reinterpret_cast<const Unit<E> *>(st + fa_off[q * U + j] + i * LA::KN * 256);
#pragma unroll
                for(int x = 0; x < U; ++x) f.a[j][i * U + x] = u.e[x];
            } else {
                const Unit<E> u = *reinterpret_cast<const Unit<E> *>(st + fa_off[q] + r * LA::KN * 256);
#pragma unroll
                for(int x = 0; x < U; ++x) f.a[x][r] = u.e[x];
            }
        } else {
            constexpr int t = r - TM;
            if constexpr(BR) {
                constexpr int   j = t % U, i = t / U;
                const Unit<E>   u = *reinterpret_cast<const Unit<E> *>(st + LA::BYTES + fb_off[q * U + j] + i * LB::KN * 256);
#pragma unroll
                for(int x = 0; x < U; ++x) f.b[j][i * U + x] = u.e[x];
            } else {
                const Unit<E> u = *reinterpret_cast<const Unit<E> *>(st + LA::BYTES + fb_off[q] + t * LB::KN * 256);
#pragma unroll
                for(int x = 0; x < U; ++x) f.b[x][t] = u.e[x];
            }
        }
    };
    auto fetch_all = [&](const char *st, auto q, Frag &f) { static_for<TM + TN>([&](auto r) { fetch(st, q, r, f); }); };
    constexpr int NM = U * TM * TN * NACC; // MFMAs of one K position
    // The MFMAs of one K position with SIDE other operations spread between them: loads and LDS reads are accepted slowly
    // when all waves issue them at once, and an in-order wave that waits there leaves its matrix core idle.
    const R sa = g.a.sign, sb = g.b.sign;
    auto multiply = [&](Frag &f, auto side_n, auto &&side) {
        constexpr int SIDE = decltype(side_n)::value;
        R             xa[U][TM], xb[U][TN];
        static_for<NM>([&](auto m_) {
            constexpr int m = decltype(m_)::value, per = TM * TN * NACC, j = m / per, w = m % per;
            if constexpr(CPLX) {
                // per K value: all ar br, all ai bi, then all sums
                constexpr int c = w / (TM * TN), i = w % (TM * TN) / TN, n = w % TN;
                if constexpr(c == 0) acc[0][i][n] = MM::op(f.b[j][n].re, f.a[j][i].re, acc[0][i][n]);
                else if constexpr(c == 1) acc[1][i][n] = MM::op(f.b[j][n].im, f.a[j][i].im, acc[1][i][n]);
                else acc[2][i][n] = MM::op(xb[j][n], xa[j][i], acc[2][i][n]);
                if constexpr(w == 0) {
#pragma unroll
                    for(int x = 0; x < TM; ++x) xa[j][x] = fma(sa, f.a[j][x].im, f.a[j][x].re);
#pragma unroll
                    for(int x = 0; x < TN; ++x) xb[j][x] = fma(sb, f.b[j][x].im, f.b[j][x].re);
                    // All here: a vector instruction between MFMAs costs the matrix core its own cycles and about nine
                    // more for the switch, so that they are kept together.
#pragma unroll
                    for(int x = 0; x < TM; ++x) asm volatile("" : "+v"(xa[j][x]));
#pragma unroll
                    for(int x = 0; x < TN; ++x) asm volatile("" : "+v"(xb[j][x]));
                }
            } else {
                constexpr int i = w / TN, n = w % TN;
                acc[0][i][n] = MM::op(f.b[j][n], f.a[j][i], acc[0][i][n]);
            }
            __builtin_amdgcn_sched_barrier(0);
            // Operations behind this MFMA: one each from the first MFMA on, so that reads have time to land.
            constexpr int s0 = SIDE <= NM ? (m < SIDE ? m : SIDE) : (m * SIDE + NM - 1) / NM;
            constexpr int s1 = SIDE <= NM ? (m + 1 < SIDE ? m + 1 : SIDE) : ((m + 1) * SIDE + NM - 1) / NM;
            if constexpr(s1 > s0) {
                static_for<s1 - s0>([&](auto x) { side(std::integral_constant<int, s0 + decltype(x)::value>{}); });
                __builtin_amdgcn_sched_barrier(0);
            }
        });
    };

    if(numK > 0) {
        int todo = numK; // stages not yet issued
        // Operation x of refilling a stage; behind the last stage only zeros are loaded, so that the count of loads in
        // flight is the same in every step.
        auto refill = [&](char *p, auto x_, auto full) {
            constexpr int  x = decltype(x_)::value;
            constexpr bool F = decltype(full)::value;
            const int      left = F ? BK : todo > 0 ? g.Kin - st * BK : 0;
            if constexpr(x < LA::L) la.template issue<x, F>(g.a, p, left);
            else lb.template issue<x - LA::L, F>(g.b, p + LA::BYTES, left);
            if constexpr(x == LPS - 1) {
                const bool wrap = st + 1 == g.stages_per_chunk;
                la.advance(g.a, wrap);
                lb.advance(g.b, wrap);
                st = wrap ? 0 : st + 1;
                --todo;
            }
        };
        const int full_stages = g.Kin % BK == 0 ? 0x40000000 : g.Kin / BK; // of a chunk
        static_for<NS>([&](auto s) { static_for<LPS>([&](auto x) { refill(stage(s), x, std::false_type{}); }); });
        // The loads of the next stage have landed for every wave (left: stages that may still be in flight), and every
        // wave has read the last fragments of the current one.
        auto ready = [&](auto left) {
            __builtin_amdgcn_s_waitcnt(waitcnt(decltype(left)::value * LPS));
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        // One stage: the fragments of the next K position are read between the MFMAs of the current one. Behind the last
        // position's barrier come the next stage's first reads and the refill of this stage.
        Frag          f[2];
        constexpr int RD = TM + TN;
        using C0         = std::integral_constant<int, 0>;
        auto positions   = [&](auto s, auto &&last) {
            static_for<NQ>([&](auto q) {
                constexpr int i = decltype(q)::value;
                if constexpr(i + 1 < NQ)
                    multiply(f[i & 1], std::integral_constant<int, RD>{},
                             [&](auto x) { fetch(stage(s), std::integral_constant<int, i + 1>{}, x, f[(i + 1) & 1]); });
                else last(f[i & 1]);
            });
        };
        static_assert(NQ % 2 == 0, "fragment double buffer");
        ready(std::integral_constant<int, NS - 1>{});
        fetch_all(stage(C0{}), C0{}, f[0]);
        auto round = [&](auto full) {
            static_for<NS>([&](auto s) {
                auto next = std::integral_constant<int, (decltype(s)::value + 1) % NS>{};
                positions(s, [&](Frag &cur) {
                    ready(std::integral_constant<int, NS - 2>{});
                    char *p = stage(s);
                    multiply(cur, std::integral_constant<int, RD + LPS>{}, [&](auto x) {
                        constexpr int i = decltype(x)::value;
                        if constexpr(i < RD) fetch(stage(next), C0{}, x, f[0]);
                        else refill(p, std::integral_constant<int, i - RD>{}, full);
                    });
                });
            });
        };
        for(int it = numK / NS; it > 0;) {
            for(; it > 0 && todo >= NS && st + NS <= full_stages; --it) {
                round(std::true_type{});
                if(TWO && it % FLUSH == 0) flush(true);
            }
            if(it > 0) {
                round(std::false_type{});
                if(TWO && it % FLUSH == 0) flush(true);
                --it;
            }
        }
        // The remaining numK % NS stages are in flight already.
        const int rest = numK % NS;
        static_for<DEP>([&](auto s) {
            constexpr int i = decltype(s)::value;
            if(i < rest)
                positions(s, [&](Frag &cur) {
                    if(i + 1 < rest) {
                        ready(std::integral_constant<int, NS - 2 - i>{});
                        multiply(cur, std::integral_constant<int, RD>{},
                                 [&](auto x) { fetch(stage(std::integral_constant<int, i + 1>{}), C0{}, x, f[0]); });
                    } else multiply(cur, C0{}, [](auto) {});
                });
        });
        flush(false);
        __builtin_amdgcn_s_waitcnt(waitcnt(0)); // no load may still be writing LDS when the workgroup ends
        asm volatile("" ::: "memory");
    }

    // Lane l holds column l % 16 of A's block (m) and rows row(l / 16, v) of B's block (n).
    auto mrow = [&](int i) { return AR ? (i / U) * 16 * U + ll * U + i % U : i * 16 + ll; };
    auto nrow = [&](int j, int p) { return BR ? (j / U) * 16 * U + p * U + j % U : j * 16 + p; };
    E   *C    = static_cast<E *>(g.C) + b * g.c_batch;
    E   *P    = g.ksplit > 1 ? static_cast<E *>(g.part) + (static_cast<int64_t>(b) * g.ksplit + split) * g.M * g.N : nullptr;
    const int mb = m0 + wm * TM * 16, nb = n0 + wn * TN * 16;
    int64_t   moff[TM];
    auto      off = [](const Idx2 &x, int i) { return x.c == 0x7fffffffu ? i * x.s0 : idx_off(x, static_cast<uint32_t>(i)); };
#pragma unroll
    for(int i = 0; i < TM; ++i) moff[i] = P ? mb + mrow(i) : off(g.cm, mb + mrow(i));
#pragma unroll
    for(int j = 0; j < TN; ++j)
#pragma unroll
        for(int v = 0; v < 4; ++v) {
            const int gn = nb + nrow(j, MM::row(lg, v));
            if(gn >= g.N) continue;
            E *col = P ? P + static_cast<int64_t>(g.M) * gn : C + off(g.cn, gn);
#pragma unroll
            for(int i = 0; i < TM; ++i) {
                if(mb + mrow(i) >= g.M) continue;
                E val;
                if constexpr(CPLX) {
                    const R p1 = acc[0][i][j][v], p2 = sa * sb * acc[1][i][j][v];
                    val        = E{p1 - p2, acc[2][i][j][v] - p1 - p2};
                } else val = acc[0][i][j][v];
                E *dst = col + moff[i];
                if(!P && g.accumulate) {
                    const E old = *dst;
                    if constexpr(CPLX) val.re += old.re, val.im += old.im;
                    else val += old;
                }
                *dst = val;
            }
        }
}

// One array per stage, so that a fragment read is not taken to alias the loads in flight to the other stages.
#define DMRG_PIPE_STAGES(BYTES, NS)                                                          \
    __shared__ __attribute__((aligned(16))) char S0[(BYTES)];                                \
    __shared__ __attribute__((aligned(16))) char S1[(BYTES)];                                \
    __shared__ __attribute__((aligned(16))) char S2[(NS) > 2 ? (BYTES) : 16];                \
    __shared__ __attribute__((aligned(16))) char S3[(NS) > 3 ? (BYTES) : 16];                \
    static_assert((NS) >= 2 && (NS) <= 4, "number of stages");                               \
    auto stage = [&](auto s) -> char * {                                                     \
        constexpr int i = decltype(s)::value;                                                \
        if constexpr(i == 0) return S0;                                                      \
        else if constexpr(i == 1) return S1;                                                 \
        else if constexpr(i == 2) return S2;                                                 \
        else return S3;                                                                      \
    }

template <typename R, bool CPLX, int BM, int BN, int BK, int WM, int WN, int NS, bool AR, bool BR, int W>
__global__ __launch_bounds__(64 * WM *WN, 2) void kernel(const Desc g) {
    DMRG_PIPE_STAGES((BM + BN) * BK * static_cast<int>(sizeof(R)) * (CPLX ? 2 : 1), NS);
    body<R, CPLX, BM, BN, BK, WM, WN, NS, AR, BR, W>(g, blockIdx.x, blockIdx.y, blockIdx.z, stage);
}

// Several independent GEMMs in one launch: workgroup x belongs to the one whose tile range [start[i], start[i + 1])
// holds x (one K slice and batch entry each). Units run along K or are loaded by 4 bytes, as each GEMM's description says:
// one kernel then serves all members of a leg, where the register-staged tiles needed one launch per (orientation,
// alignment). Bounded by the longest member's chain of K stages: 32 FP64 matvecs of chi 16 to 64, D = 5, take 29 us in three
// launches of about 10 us, against 79 us in six to seven of 10 to 15 us.
template <typename R, bool CPLX, int BM, int BN, int BK, int WM, int WN, int NS>
__global__ __launch_bounds__(64 * WM *WN, 2) void grouped_kernel(const Desc *descs, const int *start, int n) {
    DMRG_PIPE_STAGES((BM + BN) * BK * static_cast<int>(sizeof(R)) * (CPLX ? 2 : 1), NS);
    const int  i = group_of(start, n, blockIdx.x);
    const Desc g = descs[i];
    if(g.wide) body<R, CPLX, BM, BN, BK, WM, WN, NS, false, false, 16>(g, blockIdx.x - start[i], 0, 0, stage);
    else body<R, CPLX, BM, BN, BK, WM, WN, NS, false, false, 4>(g, blockIdx.x - start[i], 0, 0, stage);
}

} // namespace pipe
} // namespace dmrg
