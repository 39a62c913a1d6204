// Block-vector kernels of the eigensolver. Every kernel streams its vectors once from HBM with
// coalesced accesses; reductions go through per-block partials folded in a fixed order.
#include "vecops.hpp"

#include <algorithm>

namespace dmrg {

constexpr int VT_THREADS = 256;

template <typename T>
__device__ inline void ld(const T &v, double &re, double &im) {
    if constexpr(vtraits<T>::cx) {
        re = static_cast<double>(v.re);
        im = static_cast<double>(v.im);
    } else {
        re = static_cast<double>(v);
        im = 0.0;
    }
}
template <typename T>
__device__ inline T mk(double re, double im) {
    using R = typename vtraits<T>::R;
    if constexpr(vtraits<T>::cx) return T{static_cast<R>(re), static_cast<R>(im)};
    else return static_cast<R>(re);
}

__device__ inline double wsum(double v) {
#pragma unroll
    for(int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Block reduction of NV values; results valid in thread 0.
template <int NV>
__device__ inline void bsum(double (&v)[NV], double (*red)[VT_THREADS / 64]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for(int i = 0; i < NV; ++i) v[i] = wsum(v[i]);
    __syncthreads();
    if(lane == 0)
#pragma unroll
        for(int i = 0; i < NV; ++i) red[i][wave] = v[i];
    __syncthreads();
    if(threadIdx.x == 0)
#pragma unroll
        for(int i = 0; i < NV; ++i) {
            double s = 0;
            for(int w = 0; w < VT_THREADS / 64; ++w) s += red[i][w];
            v[i] = s;
        }
}

static int grid_for(int64_t n) {
    return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(VEC_MAX_BLOCKS, (n + VT_THREADS - 1) / VT_THREADS)));
}

// ------------------------------------------------------------------------------------------- fused folds
// A reduction over few workgroups folds its partial sums in its last workgroup instead of a second launch: every
// workgroup stores its partials at device scope (past the XCD's own L2), waits for them and counts itself in; the one that
// counts last reads all partials past the non-coherent caches and sums them in workgroup order (deterministic), then resets
// the counter for the next use.
// The order of partials and count follows from this chip's rules, not from the language: an atomic store at device scope
// (sc1) counts in vmcnt until it has arrived past the L2; every wavefront waits for vmcnt 0 before the barrier in front of
// its workgroup's count, and the count and the loads of the partials are at device scope too. These are the instructions of a
// device-scope release and acquire without the write-back and the invalidation of the L2, which concern plain stores and
// loads; nothing plain passes between the workgroups of one launch. With both (an acquire-release count), a solve at chi = 64
// takes 5.41 ms instead of 5.28, with a fence in every thread 5.76.
#if defined(__HIP_DEVICE_COMPILE__) && !defined(__gfx950__)
#error "the folds' order is written for gfx950"
#endif
// Up to 128 workgroups: every one of them counts itself in at one address, which takes about 10 ns each (n = 122880: 480
// workgroups, update and norm 6.9 us, against 3.3 + 2.6 for the update and a fold of its own).
constexpr int FUSE_MAX_BLOCKS = 128;
constexpr int FUSE_MAX_VALUES = VT_THREADS;

static bool fused(int64_t blocks, int values) { return blocks <= FUSE_MAX_BLOCKS && values <= FUSE_MAX_VALUES; }

static unsigned *scratch_counter(double *scratch) { return reinterpret_cast<unsigned *>(scratch + vec_scratch_doubles() - 8); }

void vec_scratch_init(double *scratch, hipStream_t s) {
    DMRG_HIP_CHECK(hipMemsetAsync(scratch_counter(scratch), 0, 8 * sizeof(double), s));
}

// A partial sum: at device scope where the kernel's last workgroup folds it, else an ordinary store.
__device__ inline void publish(double *p, double v, bool device_scope) {
    if(device_scope) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else *p = v;
}

// What a reduction's last workgroup also writes to pinned host memory: its sums to h_out, and n doubles of d to h.
struct HostCopy {
    double       *h_out = nullptr;
    const double *d     = nullptr;
    double       *h     = nullptr;
    int           n     = 0; // at most VT_THREADS
};

// partial: [row block][nv]; value v goes to out[v], from column v / 2 == j_self on to self_out (when given).
__device__ inline void fold_in_last_block(const double *partial, int nv, double *out, int j_self, double *self_out, unsigned *counter,
                                          const HostCopy &hc = HostCopy{}) {
    __shared__ int last;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // the partials of this wavefront are at device scope
    __syncthreads();
    if(threadIdx.x == 0)
        last = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x * gridDim.y - 1 ? 1 : 0;
    __syncthreads();
    if(!last) return;
    // Thread t sums value t % nv over the row blocks b = t / nv, t / nv + per, ...; then thread v adds the per
    // sums of value v in order. nv <= blockDim.x.
    __shared__ double red[VT_THREADS];
    const int         per = blockDim.x / nv;
    const int         t   = threadIdx.x;
    if(t < per * nv) {
        const int     v  = t % nv;
        const int     nb = static_cast<int>(gridDim.x);
        double        a  = 0.0;
        constexpr int UN = 8;
        for(int b = t / nv; b < nb; b += UN * per) {
            double x[UN];
#pragma unroll
            for(int u = 0; u < UN; ++u)
                x[u] = __hip_atomic_load(partial + static_cast<int64_t>(min(b + u * per, nb - 1)) * nv + v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for(int u = 0; u < UN; ++u)
                if(b + u * per < nb) a += x[u];
        }
        red[t] = a;
    }
    __syncthreads();
    if(t < nv) {
        double acc = 0.0;
        for(int k = 0; k < per; ++k) acc += red[t + k * nv];
        double *o = ((t >> 1) >= j_self && self_out) ? self_out + (t - 2 * j_self) : out + t;
        *o        = acc;
        if(hc.h_out) hc.h_out[t] = acc;
    }
    if(t < hc.n) hc.h[t] = hc.d[t];
    if(t == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ------------------------------------------------------------------------------------------- multidot
// Basis columns per pass (two double accumulators each). Long vectors: 16, so that x is read once per 16 columns. Short
// ones: 4, with the groups of columns in their own workgroups: the rows alone give too few of them, and the reduction
// across a wavefront shrinks from 32 values to 8 (n = 8192, 14 columns: 8 workgroups 14.3 us, 128 workgroups 4.5 us).
constexpr int MD_CH        = 16;
constexpr int MD_CH_SHORT  = 4;
constexpr int64_t MD_SHORT = int64_t(1) << 17; // up to here the basis is read from the caches, and latency is what counts
constexpr int MD_PER_THREAD = 4;  // rows per thread and pass at full grid: amortises the block reduction

// Reduce-scatter of NV values across the 64 lanes of a wavefront: after the call lane l holds in v[0] the
// wave total of value index rs_index<NV>(l) (valid in the lanes whose low bits below the last exchange are
// zero). Halving the set exchanged at each step costs NV - 1 + (6 - log2 NV) shuffles instead of 6 NV.
template <int H, int O, int NV>
__device__ inline void rs_step(double (&v)[NV], int lane) {
    if constexpr(H >= 1) {
        const bool up = (lane & O) != 0;
#pragma unroll
        for(int k = 0; k < H; ++k) {
            const double send = up ? v[k] : v[k + H];
            const double keep = up ? v[k + H] : v[k];
            v[k]              = keep + __shfl_xor(send, O, 64);
        }
        rs_step<H / 2, O / 2, NV>(v, lane);
    } else {
#pragma unroll
        for(int o = O; o >= 1; o >>= 1) v[0] += __shfl_xor(v[0], o, 64); // remaining low lane bits
    }
}
template <int NV>
__device__ inline int rs_index(int lane) {
    int idx = 0;
#pragma unroll
    for(int h = NV / 2, o = 32; h >= 1; h >>= 1, o >>= 1) idx += (lane & o) ? h : 0;
    return idx;
}
template <int NV>
__device__ inline bool rs_owner(int lane) {
    return (lane & (64 / NV - 1)) == 0;
}

// DGKS test evaluated by the projection kernel of a second orthogonalisation pass itself: the pass runs when
// post[0] < eta2 * pre[0] (|t|^2 fell by more than that factor in the first pass); block 0 records the decision
// in flag[0] for the kernels of the pass that follow. pre and post are not written during the kernel, so every
// block reaches the same decision.
struct DgksTest {
    const double *pre  = nullptr;
    const double *post = nullptr;
    double        eta2 = 0.0;
    int          *flag = nullptr;
};

// Columns j < m are V[:, j]; column m (when with_self) is x itself, so x^H x comes out of the same pass. Workgroup
// (b, g) takes the rows of b and the columns [CH g, CH (g + 1)) and then every CH gridDim.y-th group.
template <typename T, int CH, bool FOLD>
__global__ __launch_bounds__(VT_THREADS) void multidot_partial(int64_t n, int m, int mc, const T *V, int64_t ldv, const T *x,
                                                               const int *skip, double *partial, unsigned *counter, double *out,
                                                               int m_out, double *self_out, DgksTest dg, HostCopy hc) {
    if(dg.flag) {
        const bool run = dg.post[0] < dg.eta2 * dg.pre[0];
        if(blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) dg.flag[0] = run ? 1 : 0;
        if(!run) return;
    } else if(skip && *skip == 0) {
        return;
    }
    constexpr int     NV = 2 * CH;
    __shared__ double red[NV][VT_THREADS / 64];
    const int         lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    constexpr bool    SPLIT = CH == MD_CH_SHORT; // long vectors: one workgroup takes all columns of its rows
    for(int j0 = SPLIT ? blockIdx.y * CH : 0; j0 < mc; j0 += SPLIT ? CH * static_cast<int>(gridDim.y) : CH) {
        double acc[NV];
#pragma unroll
        for(int c = 0; c < NV; ++c) acc[c] = 0.0;
        for(int64_t i = blockIdx.x * static_cast<int64_t>(VT_THREADS) + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * VT_THREADS) {
            double xr, xi;
            ld(x[i], xr, xi);
#pragma unroll
            for(int c = 0; c < CH; ++c) {
                if(j0 + c < mc) {
                    double vr, vi;
                    if(j0 + c < m) ld(V[i + (j0 + c) * ldv], vr, vi);
                    else vr = xr, vi = xi;
                    acc[2 * c] += vr * xr + vi * xi; // conj(v) x
                    acc[2 * c + 1] += vr * xi - vi * xr;
                }
            }
        }
        rs_step<NV / 2, 32, NV>(acc, lane);
        if(rs_owner<NV>(lane)) red[rs_index<NV>(lane)][wave] = acc[0];
        __syncthreads();
        if(threadIdx.x < NV) {
            const int c = threadIdx.x >> 1;
            if(j0 + c < mc) {
                double t = 0;
#pragma unroll
                for(int w = 0; w < VT_THREADS / 64; ++w) t += red[threadIdx.x][w];
                publish(partial + 2 * (static_cast<int64_t>(blockIdx.x) * mc + j0 + c) + (threadIdx.x & 1), t, FOLD);
            }
        }
        __syncthreads();
    }
    if constexpr(FOLD) fold_in_last_block(partial, 2 * mc, out, m_out, self_out, counter, hc);
}

static int md_grid(int64_t n) {
    return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(VEC_MAX_BLOCKS, (n + VT_THREADS * MD_PER_THREAD - 1) / (VT_THREADS * MD_PER_THREAD))));
}

// out[j] = sum_b partial[b][j] for j < m (columns from m_out on go to self_out instead, when given): one block
// per column, each thread a fixed strided subset of the partials, then a fixed-order tree (deterministic).
__global__ __launch_bounds__(VT_THREADS) void fold_columns(int nblk, int m, const double *partial, double *out, int m_out,
                                                           double *self_out, const int *skip, HostCopy hc) {
    if(skip && *skip == 0) return;
    __shared__ double red[2][VT_THREADS / 64];
    const int         j   = blockIdx.x;
    double            acc[2] = {0.0, 0.0};
    for(int b = threadIdx.x; b < nblk; b += VT_THREADS) {
        acc[0] += partial[2 * (static_cast<int64_t>(b) * m + j)];
        acc[1] += partial[2 * (static_cast<int64_t>(b) * m + j) + 1];
    }
    bsum<2>(acc, red);
    if(threadIdx.x == 0) {
        double *o = (j >= m_out && self_out) ? self_out + 2 * (j - m_out) : out + 2 * j;
        o[0]      = acc[0];
        o[1]      = acc[1];
        if(hc.h_out) hc.h_out[2 * j] = acc[0], hc.h_out[2 * j + 1] = acc[1];
    }
    if(j == 0 && static_cast<int>(threadIdx.x) < hc.n) hc.h[threadIdx.x] = hc.d[threadIdx.x];
}

template <typename T>
static void multidot_x_impl(int64_t n, int m, const T *V, int64_t ldv, const T *x, double *d_out, double *d_self, const int *skip,
                            const DgksTest &dg, double *scratch, hipStream_t s, const HostCopy &hc = HostCopy{}) {
    const int mc = m + (d_self ? 1 : 0);
    if(mc <= 0) return;
    DMRG_REQUIRE(mc <= VEC_MAX_M, DMRG_ERR_ARG, "multidot: too many columns");
    const int *fskip = dg.flag ? dg.flag : skip; // the fold follows the pass's decision
    if(n <= MD_SHORT) {
        // One row per thread, or two where that lets the last workgroup fold.
        const int groups = (mc + MD_CH_SHORT - 1) / MD_CH_SHORT, most = std::max(1, FUSE_MAX_BLOCKS / groups);
        const int want   = static_cast<int>(std::max<int64_t>(1, (n + VT_THREADS - 1) / VT_THREADS));
        const bool in_last = want <= 2 * most && fused(static_cast<int64_t>(std::min(want, most)) * groups, 2 * mc);
        const int  rows    = in_last ? std::min(want, most) : std::min(want, 256);
        if(in_last) {
            hipLaunchKernelGGL((multidot_partial<T, MD_CH_SHORT, true>), dim3(rows, groups), dim3(VT_THREADS), 0, s, n, m, mc, V, ldv, x, skip, scratch,
                               scratch_counter(scratch), d_out, d_self ? m : -1, d_self, dg, hc);
        } else {
            hipLaunchKernelGGL((multidot_partial<T, MD_CH_SHORT, false>), dim3(rows, groups), dim3(VT_THREADS), 0, s, n, m, mc, V, ldv, x, skip, scratch,
                               nullptr, nullptr, -1, nullptr, dg, HostCopy{});
            hipLaunchKernelGGL(fold_columns, dim3(mc), dim3(VT_THREADS), 0, s, rows, mc, scratch, d_out, d_self ? m : -1, d_self, fskip, hc);
        }
    } else {
        const int g = md_grid(n);
        hipLaunchKernelGGL((multidot_partial<T, MD_CH, false>), dim3(g), dim3(VT_THREADS), 0, s, n, m, mc, V, ldv, x, skip, scratch, nullptr,
                           nullptr, -1, nullptr, dg, HostCopy{});
        hipLaunchKernelGGL(fold_columns, dim3(mc), dim3(VT_THREADS), 0, s, g, mc, scratch, d_out, d_self ? m : -1, d_self, fskip, hc);
    }
    DMRG_HIP_CHECK(hipGetLastError());
}

template <typename T>
void multidot(int64_t n, int m, const T *V, int64_t ldv, const T *x, double *d_out, double *scratch, hipStream_t s) {
    multidot_x_impl<T>(n, m, V, ldv, x, d_out, nullptr, nullptr, DgksTest{}, scratch, s);
}

// The copies to the host ride on the fold of the reduction: a copy of its own is another launch, about 2 us, and its gap.
template <typename T>
void multidot_to_host(int64_t n, int m, const T *V, int64_t ldv, const T *x, double *d_block, double *h_block, int extra, int n_extra,
                      double *scratch, hipStream_t s) {
    HostCopy hc;
    hc.h_out = h_block;
    hc.d     = d_block + extra;
    hc.h     = h_block + extra;
    hc.n     = n_extra;
    multidot_x_impl<T>(n, m, V, ldv, x, d_block, nullptr, nullptr, DgksTest{}, scratch, s, hc);
}

template <typename T>
void multidot_x(int64_t n, int m, const T *V, int64_t ldv, const T *x, double *d_out, double *d_self, const int *skip,
                double *scratch, hipStream_t s) {
    multidot_x_impl<T>(n, m, V, ldv, x, d_out, d_self, skip, DgksTest{}, scratch, s);
}

template <typename T>
void multidot_dgks(int64_t n, int m, const T *V, int64_t ldv, const T *x, double *d_out, const double *d_pre, const double *d_post,
                   double eta2, int *d_flag, double *scratch, hipStream_t s) {
    DgksTest dg;
    dg.pre  = d_pre;
    dg.post = d_post;
    dg.eta2 = eta2;
    dg.flag = d_flag;
    multidot_x_impl<T>(n, m, V, ldv, x, d_out, nullptr, nullptr, dg, scratch, s);
}

// ------------------------------------------------------------------------------------------- gemv
// use(j, load(j)) for j < m in order, in groups of UN loads in flight, then of half as many, and so on. Where two bases are
// read, or one that other CUs have just written, a row waits for its columns' latencies one after another otherwise (a solve of
// four pairs at n = 8192 34.2 -> 33.5 ms, Ritz vector and residual of n = 32768, 13 columns 7.8 -> 7.65 us); a plain update and
// long vectors, bound by bandwidth, are faster one by one with all wavefronts resident (complex n = 524288: update of 8
// columns 14.0 us against 14.6, Ritz vector and residual of 8 27.9 against 28.7, FP64 n = 2097152 of 13 91.6 against 106).
template <typename T, int UN, typename L, typename F>
__device__ __forceinline__ void columns(int m, L &&load, F &&use, int j0 = 0) {
    if constexpr(UN == 1) {
        for(int j = j0; j < m; ++j) use(j, load(j));
    } else {
        for(; j0 + UN <= m; j0 += UN) {
            T v[UN];
#pragma unroll
            for(int u = 0; u < UN; ++u) v[u] = load(j0 + u);
#pragma unroll
            for(int u = 0; u < UN; ++u) use(j0 + u, v[u]);
        }
        columns<T, UN / 2>(m, load, use, j0);
    }
}
constexpr int COL_UN = 8;

// Row i of x = V y and r = W y - theta x.
template <typename T, int UN = COL_UN>
__device__ __forceinline__ void ritz_row(int64_t i, int m, const T *V, const T *W, int64_t ldv, const double *y, double theta, double &xr,
                                         double &xi, double &rr, double &ri) {
    double wr = 0, wi = 0;
    struct VW {
        T v, w;
    };
    xr = xi = 0;
    auto add = [&](int j, const T &v, const T &w) {
        double vr, vi, ur, ui;
        ld(v, vr, vi);
        ld(w, ur, ui);
        const double yr = y[2 * j], yi = y[2 * j + 1];
        xr += vr * yr - vi * yi;
        xi += vr * yi + vi * yr;
        wr += ur * yr - ui * yi;
        wi += ur * yi + ui * yr;
    };
    if constexpr(UN == 1) {
        for(int j = 0; j < m; ++j) add(j, V[i + j * ldv], W[i + j * ldv]);
    } else {
        columns<VW, UN>(m, [&](int j) { return VW{V[i + j * ldv], W[i + j * ldv]}; }, [&](int j, const VW &e) { add(j, e.v, e.w); });
    }
    rr = wr - theta * xr, ri = wi - theta * xi;
}
// Row i of V h.
template <typename T, int UN = COL_UN>
__device__ __forceinline__ void gemv_row(int64_t i, int m, const T *V, int64_t ldv, const double *h, double &ar, double &ai) {
    ar = ai = 0;
    columns<T, UN>(m, [&](int j) { return V[i + j * ldv]; },
               [&](int j, const T &v) {
                   double vr, vi;
                   ld(v, vr, vi);
                   ar += vr * h[2 * j] - vi * h[2 * j + 1];
                   ai += vr * h[2 * j + 1] + vi * h[2 * j];
               });
}

template <typename T>
__global__ __launch_bounds__(VT_THREADS) void gemv_update_kernel(int64_t n, int m, const T *V, int64_t ldv, const double *h,
                                                                 double alpha, double beta, T *x) {
    __shared__ double hs[2 * VEC_MAX_M];
    for(int j = threadIdx.x; j < 2 * m; j += VT_THREADS) hs[j] = h[j];
    __syncthreads();
    for(int64_t i = blockIdx.x * static_cast<int64_t>(VT_THREADS) + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * VT_THREADS) {
        double ar, ai;
        gemv_row<T, 1>(i, m, V, ldv, hs, ar, ai);
        double xr = 0, xi = 0;
        if(beta != 0.0) ld(x[i], xr, xi);
        x[i] = mk<T>(beta * xr + alpha * ar, beta * xi + alpha * ai);
    }
}

// y = beta x + alpha V h (x may alias y) and per-block partials of |y|^2.
template <typename T, bool FOLD>
__global__ __launch_bounds__(VT_THREADS) void gemv_update_norm_kernel(int64_t n, int m, const T *V, int64_t ldv, const double *h,
                                                                      double alpha, double beta, const T *x, T *y,
                                                                      const int *skip, double *partial, unsigned *counter,
                                                                      double *out) {
    if(skip && *skip == 0) return;
    __shared__ double hs[2 * VEC_MAX_M];
    __shared__ double red[2][VT_THREADS / 64];
    for(int j = threadIdx.x; j < 2 * m; j += VT_THREADS) hs[j] = h[j];
    __syncthreads();
    double acc[2] = {0.0, 0.0};
    for(int64_t i = blockIdx.x * static_cast<int64_t>(VT_THREADS) + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * VT_THREADS) {
        double ar, ai;
        gemv_row<T, 1>(i, m, V, ldv, hs, ar, ai);
        double xr = 0, xi = 0;
        if(beta != 0.0) ld(x[i], xr, xi);
        const T yv = mk<T>(beta * xr + alpha * ar, beta * xi + alpha * ai);
        y[i]       = yv;
        double yr, yi;
        ld(yv, yr, yi); // the norm of the stored (possibly FP32-rounded) vector
        acc[0] += yr * yr + yi * yi;
    }
    bsum<2>(acc, red);
    if(threadIdx.x == 0) {
        publish(partial + 2 * blockIdx.x, acc[0], FOLD);
        publish(partial + 2 * blockIdx.x + 1, 0.0, FOLD);
    }
    if constexpr(FOLD) fold_in_last_block(partial, 2, out, -1, nullptr, counter);
}

static int ew_grid(int64_t n) { return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(8192, (n + VT_THREADS - 1) / VT_THREADS))); }

template <typename T>
void gemv_update(int64_t n, int m, const T *V, int64_t ldv, const double *d_h, double alpha, double beta, T *x, hipStream_t s) {
    DMRG_REQUIRE(m <= VEC_MAX_M, DMRG_ERR_ARG, "gemv: too many columns");
    hipLaunchKernelGGL(gemv_update_kernel<T>, dim3(ew_grid(n)), dim3(VT_THREADS), 0, s, n, m, V, ldv, d_h, alpha, beta, x);
    DMRG_HIP_CHECK(hipGetLastError());
}

template <typename T>
void gemv_update_norm(int64_t n, int m, const T *V, int64_t ldv, const double *d_h, double alpha, double beta, const T *x, T *y,
                      double *d_nrm2, const int *skip, double *scratch, hipStream_t s) {
    DMRG_REQUIRE(m <= VEC_MAX_M, DMRG_ERR_ARG, "gemv: too many columns");
    const int g = grid_for(n);
    if(fused(g, 2)) {
        hipLaunchKernelGGL((gemv_update_norm_kernel<T, true>), dim3(g), dim3(VT_THREADS), 0, s, n, m, V, ldv, d_h, alpha, beta, x, y, skip, scratch,
                           scratch_counter(scratch), d_nrm2);
    } else {
        hipLaunchKernelGGL((gemv_update_norm_kernel<T, false>), dim3(g), dim3(VT_THREADS), 0, s, n, m, V, ldv, d_h, alpha, beta, x, y, skip, scratch,
                           nullptr, nullptr);
        hipLaunchKernelGGL(fold_columns, dim3(1), dim3(VT_THREADS), 0, s, g, 1, scratch, d_nrm2, -1, nullptr, skip, HostCopy{});
    }
    DMRG_HIP_CHECK(hipGetLastError());
}

// ------------------------------------------------------------------------------------------- Ritz vector + residual
// The coefficients come with the launch (up to RITZ_ARGS of them) or from device memory (y). With one column at a time, the
// compiler is held to eight wavefronts a SIMD: left alone it unrolls into 86 registers and five.
constexpr int RITZ_ARGS = 32;
struct RitzCoef {
    double y[2 * RITZ_ARGS];
};
template <typename T, int UN, bool FOLD>
__global__ __launch_bounds__(VT_THREADS, UN == 1 ? 8 : 4) void ritz_kernel(int64_t n, int m, const T *V, const T *W, int64_t ldv, const double *y,
                                                          const RitzCoef c, double theta, T *x, T *r, double *partial, unsigned *counter,
                                                          double *out, HostCopy hc) {
    __shared__ double ys[2 * VEC_MAX_M];
    __shared__ double red[2][VT_THREADS / 64];
    if(y) {
        for(int j = threadIdx.x; j < 2 * m; j += VT_THREADS) ys[j] = y[j];
    } else if(threadIdx.x < 2 * m) {
        ys[threadIdx.x] = c.y[threadIdx.x]; // 2 m <= 2 RITZ_ARGS < VT_THREADS
    }
    __syncthreads();
    double acc[2] = {0.0, 0.0};
    for(int64_t i = blockIdx.x * static_cast<int64_t>(VT_THREADS) + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * VT_THREADS) {
        double xr, xi, rr, ri;
        ritz_row<T, UN>(i, m, V, W, ldv, ys, theta, xr, xi, rr, ri);
        x[i] = mk<T>(xr, xi);
        r[i] = mk<T>(rr, ri);
        acc[0] += rr * rr + ri * ri;
        acc[1] += xr * xr + xi * xi;
    }
    bsum<2>(acc, red);
    if(threadIdx.x == 0) {
        publish(partial + 2 * blockIdx.x, acc[0], FOLD);
        publish(partial + 2 * blockIdx.x + 1, acc[1], FOLD);
    }
    if constexpr(FOLD) fold_in_last_block(partial, 2, out, -1, nullptr, counter, hc);
}

template <typename T>
static void ritz_launch(int64_t n, int m, const T *V, const T *W, int64_t ld, const double *d_y, const RitzCoef &c, double theta, T *x, T *r,
                        double *d_out, double *h_out, double *scratch, hipStream_t s) {
    HostCopy hc;
    hc.h_out = h_out;
    DMRG_REQUIRE(m <= VEC_MAX_M, DMRG_ERR_ARG, "ritz: too many columns");
    const int g = grid_for(n);
    if(fused(g, 2)) {
        hipLaunchKernelGGL((ritz_kernel<T, COL_UN, true>), dim3(g), dim3(VT_THREADS), 0, s, n, m, V, W, ld, d_y, c, theta, x, r, scratch,
                           scratch_counter(scratch), d_out, hc);
    } else {
        const auto kernel = n <= MD_SHORT ? ritz_kernel<T, COL_UN, false> : ritz_kernel<T, 1, false>;
        hipLaunchKernelGGL(kernel, dim3(g), dim3(VT_THREADS), 0, s, n, m, V, W, ld, d_y, c, theta, x, r, scratch, nullptr, nullptr, HostCopy{});
        hipLaunchKernelGGL(fold_columns, dim3(1), dim3(VT_THREADS), 0, s, g, 1, scratch, d_out, -1, nullptr, nullptr, hc);
    }
    DMRG_HIP_CHECK(hipGetLastError());
}

template <typename T>
void ritz_residual(int64_t n, int m, const T *V, const T *W, int64_t ld, const double *h_y, double *d_y, double theta, T *x, T *r,
                   double *d_out, double *h_out, double *scratch, hipStream_t s) {
    RitzCoef c{};
    if(m <= RITZ_ARGS) {
        std::copy(h_y, h_y + 2 * m, c.y);
        d_y = nullptr;
    } else {
        DMRG_HIP_CHECK(hipMemcpyAsync(d_y, h_y, 2 * static_cast<size_t>(m) * sizeof(double), hipMemcpyHostToDevice, s));
    }
    ritz_launch<T>(n, m, V, W, ld, d_y, c, theta, x, r, d_out, h_out, scratch, s);
}

// ------------------------------------------------------------------------------------------- expansion of a small basis
// Ritz vector and residual, Gram-Schmidt with the DGKS test, and normalisation of a small problem, in one workgroup with the
// vector in LDS. Bounded by latency: a pass over a basis in the caches takes 1 to 2 us, a launch of its own 4 us and 6 to 9
// of the host's time, and the steps are six launches otherwise (n up to 512, up to 14 columns: 8.2 us against 19 in six, and
// a sweep of L = 16 at chi = 32 takes 194 ms against 273).
constexpr int     EX_THREADS = 1024;
constexpr int     EX_WAVES   = EX_THREADS / 64;
// The vector and, with the Ritz step, the basis elements up to which one CU's loads cost less than the launches. Iterations of
// solves in one workgroup / in three launches, us: FP64 n = 2048 16.5 / 18.5 at 8 columns, 23.1 / 23.8 at 20, 33.5 / 33.2 at 28;
// n = 4096 23.4 / 23.5 at 8, 28.1 / 25.3 at 12, 54.8 / 47.3 at 32; complex n = 2048 28.4 / 28.7 at 20, 32.4 / 32.4 at 24.
constexpr int64_t EX_MAX_BYTES    = 32768;
constexpr int64_t EX_MAX_ELEMENTS = 40960;

template <typename T>
struct ExpandArgs {
    int64_t  n, ldv;
    int      m;
    const T *V, *W, *src; // W null: src is orthogonalised, else the residual
    T       *x, *r, *t;
    double   theta, eta2;
    double  *ritz, *nrm;
};

// Sums over the workgroup, in every thread.
template <int NV>
__device__ inline void all_sum(double (&v)[NV], double (*red)[EX_WAVES]) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for(int i = 0; i < NV; ++i) v[i] = wsum(v[i]);
    __syncthreads();
    if(lane == 0)
#pragma unroll
        for(int i = 0; i < NV; ++i) red[i][wave] = v[i];
    __syncthreads();
#pragma unroll
    for(int i = 0; i < NV; ++i) {
        v[i] = 0;
#pragma unroll
        for(int w = 0; w < EX_WAVES; ++w) v[i] += red[i][w];
    }
}

template <typename T>
__global__ __launch_bounds__(EX_THREADS) void expand_kernel(const ExpandArgs<T> g, const RitzCoef c) {
    extern __shared__ __attribute__((aligned(16))) char expand_lds[];
    T                *tv = reinterpret_cast<T *>(expand_lds);
    __shared__ double hs[2 * RITZ_ARGS], part[2 * RITZ_ARGS][2], red[3][EX_WAVES];
    const int         tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n = static_cast<int>(g.n), m = g.m;
    double            acc[3] = {0.0, 0.0, 0.0};
    if(g.W) {
        if(tid < 2 * m) hs[tid] = c.y[tid];
        __syncthreads();
        for(int i = tid; i < n; i += EX_THREADS) {
            double xr, xi, rr, ri;
            ritz_row<T>(i, m, g.V, g.W, g.ldv, hs, g.theta, xr, xi, rr, ri);
            const T      rv = mk<T>(rr, ri);
            g.x[i]          = mk<T>(xr, xi);
            g.r[i]          = rv;
            tv[i]           = rv;
            double sr, si;
            ld(rv, sr, si);
            acc[0] += rr * rr + ri * ri;
            acc[1] += xr * xr + xi * xi;
            acc[2] += sr * sr + si * si;
        }
    } else {
        for(int i = tid; i < n; i += EX_THREADS) {
            const T v = g.src[i];
            tv[i]     = v;
            double sr, si;
            ld(v, sr, si);
            acc[2] += sr * sr + si * si;
        }
    }
    all_sum<3>(acc, red);
    if(g.W && tid == 0) g.ritz[0] = acc[0], g.ritz[1] = acc[1];
    const double pre = acc[2];
    double       post[1] = {pre};
    // Projections: a wavefront per column and segment of rows, so that few columns also keep all wavefronts reading.
    const int segs = m > 0 ? max(1, EX_WAVES / m) : 1, len = (n + segs - 1) / segs;
    for(int pass = 0; m > 0 && pass < 2; ++pass) {
        for(int task = wave; task < m * segs; task += EX_WAVES) {
            const int j = task % m, i0 = task / m * len, i1 = min(n, i0 + len);
            const T  *v = g.V + j * g.ldv;
            double    ar = 0, ai = 0;
#pragma unroll 8
            for(int i = i0 + lane; i < i1; i += 64) {
                double vr, vi, xr, xi;
                ld(v[i], vr, vi);
                ld(tv[i], xr, xi);
                ar += vr * xr + vi * xi; // conj(v) x
                ai += vr * xi - vi * xr;
            }
            ar = wsum(ar);
            if constexpr(vtraits<T>::cx) ai = wsum(ai);
            if(lane == 0) part[task][0] = ar, part[task][1] = ai;
        }
        __syncthreads();
        if(tid < 2 * m) {
            double h = 0;
            for(int q = 0; q < segs; ++q) h += part[q * m + (tid >> 1)][tid & 1];
            hs[tid] = h;
        }
        __syncthreads();
        post[0] = 0;
        for(int i = tid; i < n; i += EX_THREADS) {
            double ar, ai;
            gemv_row<T>(i, m, g.V, g.ldv, hs, ar, ai);
            double xr, xi;
            ld(tv[i], xr, xi);
            const T y = mk<T>(xr - ar, xi - ai);
            tv[i]     = y;
            double yr, yi;
            ld(y, yr, yi);
            post[0] += yr * yr + yi * yi;
        }
        all_sum<1>(post, red);
        if(!(post[0] < g.eta2 * pre)) break;
    }
    const double a = post[0] > 0.0 ? 1.0 / sqrt(post[0]) : 0.0; // a zero vector stays zero (breakdown tests see it)
    for(int i = tid; i < n; i += EX_THREADS) {
        double re, im;
        ld(tv[i], re, im);
        g.t[i] = mk<T>(a * re, a * im);
    }
    if(tid == 0) g.nrm[0] = pre, g.nrm[1] = 0.0, g.nrm[2] = post[0], g.nrm[3] = 0.0;
}

template <typename T>
bool expand_small(int64_t n, int m, const T *V, const T *W, int64_t ldv, const double *h_y, double theta, T *x, T *r, const T *src, T *t,
                  double eta2, double *d_ritz, double *d_nrm, hipStream_t s) {
    if(n * static_cast<int64_t>(sizeof(T)) > EX_MAX_BYTES || m > RITZ_ARGS || (W && n * m > EX_MAX_ELEMENTS)) return false;
    RitzCoef c{};
    if(W) std::copy(h_y, h_y + 2 * m, c.y);
    const ExpandArgs<T> g{n, ldv, m, V, W, src, x, r, t, theta, eta2, d_ritz, d_nrm};
    hipLaunchKernelGGL(expand_kernel<T>, dim3(1), dim3(EX_THREADS), static_cast<size_t>(n) * sizeof(T), s, g, c);
    DMRG_HIP_CHECK(hipGetLastError());
    return true;
}

// The same for problems of several workgroups, up to MD_SHORT rows: three launches (and a fold after the first two where one
// workgroup per 256 rows is too many to fold in the last of them) instead of six (eleven). Each workgroup projects the rows
// that it has just formed, so that the basis comes from its caches the second time; the second Gram-Schmidt pass's
// projections are taken whether or not its test asks for them, and its norm from |t|^2 - |h|^2. That is no difference of close
// numbers: h holds the rounding errors of the first pass, a few eps |src| with the solver's bases (orthonormal to 4e-15 after
// 3000 steps with restarts in 64 bits, 5e-8 in 32), and a t below 100 eps |src| is dropped as a breakdown; down to that line
// the stored vector's norm is 1 to 2.2e-16 (in 32 bits to 2e-9, as with the norm taken from the vector). Longer vectors come from HBM, where the extra projections cost more than the
// launches. n = 8192, 14 columns: 22 us of kernels either way, but 5.4 ms a solve against 6.9; n = 122880: 13.0 ms against 14.5.

// partial[blockIdx.x][2 j] = this workgroup's rows of conj(V[:, j]) x.
template <typename T>
__device__ __forceinline__ void project_rows(int64_t n, int m, const T *V, int64_t ldv, const T *x, double *partial, int nv, bool device_scope,
                                             double (*red)[VT_THREADS / 64]) {
    constexpr int CH = MD_CH, NV = 2 * CH;
    const int     lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for(int j0 = 0; j0 < m; j0 += CH) {
        double acc[NV];
#pragma unroll
        for(int c = 0; c < NV; ++c) acc[c] = 0.0;
        for(int64_t i = blockIdx.x * static_cast<int64_t>(VT_THREADS) + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * VT_THREADS) {
            double xr, xi;
            ld(x[i], xr, xi);
            T v[CH];
#pragma unroll
            for(int c = 0; c < CH; ++c) v[c] = V[i + min(j0 + c, m - 1) * ldv];
#pragma unroll
            for(int c = 0; c < CH; ++c) {
                double vr, vi;
                ld(v[c], vr, vi);
                acc[2 * c] += vr * xr + vi * xi; // conj(v) x
                acc[2 * c + 1] += vr * xi - vi * xr;
            }
        }
        rs_step<NV / 2, 32, NV>(acc, lane);
        __syncthreads();
        if(rs_owner<NV>(lane)) red[rs_index<NV>(lane)][wave] = acc[0];
        __syncthreads();
        if(threadIdx.x < NV && j0 + static_cast<int>(threadIdx.x >> 1) < m) {
            double t = 0;
#pragma unroll
            for(int w = 0; w < VT_THREADS / 64; ++w) t += red[threadIdx.x][w];
            publish(partial + static_cast<int64_t>(blockIdx.x) * nv + 2 * j0 + threadIdx.x, t, device_scope);
        }
    }
}

// x, r as in ritz_kernel; columns: V^H r, then (|r|^2 as stored, 0), (0, 0), (|r|^2, |x|^2).
template <typename T>
__global__ __launch_bounds__(VT_THREADS) void ritz_project_kernel(int64_t n, int m, const T *V, const T *W, int64_t ldv, const double *y,
                                                                  const RitzCoef c, double theta, T *x, T *r, double *partial,
                                                                  unsigned *counter, double *out, double *tail) {
    __shared__ double ys[2 * VEC_MAX_M];
    __shared__ double red[2 * MD_CH][VT_THREADS / 64];
    const int         nv = 2 * m + 6;
    if(y) {
        for(int j = threadIdx.x; j < 2 * m; j += VT_THREADS) ys[j] = y[j];
    } else if(threadIdx.x < 2 * m) {
        ys[threadIdx.x] = c.y[threadIdx.x]; // 2 m <= 2 RITZ_ARGS < VT_THREADS
    }
    __syncthreads();
    double acc[3] = {0.0, 0.0, 0.0};
    for(int64_t i = blockIdx.x * static_cast<int64_t>(VT_THREADS) + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * VT_THREADS) {
        double xr, xi, rr, ri;
        ritz_row<T>(i, m, V, W, ldv, ys, theta, xr, xi, rr, ri);
        const T rv = mk<T>(rr, ri);
        x[i]       = mk<T>(xr, xi);
        r[i]       = rv;
        double sr, si;
        ld(rv, sr, si);
        acc[0] += sr * sr + si * si;
        acc[1] += rr * rr + ri * ri;
        acc[2] += xr * xr + xi * xi;
    }
    bsum<3>(acc, red);
    if(threadIdx.x == 0) {
        double *p = partial + static_cast<int64_t>(blockIdx.x) * nv + 2 * m;
        const double v[6] = {acc[0], 0.0, 0.0, 0.0, acc[1], acc[2]};
#pragma unroll
        for(int k = 0; k < 6; ++k) publish(p + k, v[k], counter != nullptr);
    }
    project_rows<T>(n, m, V, ldv, r, partial, nv, counter != nullptr, red);
    if(counter) fold_in_last_block(partial, nv, out, m, tail, counter);
}

// t = src - V h; columns: V^H t, then (|t|^2, 0).
template <typename T>
__global__ __launch_bounds__(VT_THREADS) void update_project_kernel(int64_t n, int m, const T *V, int64_t ldv, const double *h, const T *src,
                                                                    T *t, double *partial, unsigned *counter, double *out) {
    __shared__ double hs[2 * VEC_MAX_M];
    __shared__ double red[2 * MD_CH][VT_THREADS / 64];
    const int         nv = 2 * m + 2;
    for(int j = threadIdx.x; j < 2 * m; j += VT_THREADS) hs[j] = h[j];
    __syncthreads();
    double acc[1] = {0.0};
    for(int64_t i = blockIdx.x * static_cast<int64_t>(VT_THREADS) + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * VT_THREADS) {
        double ar, ai, xr, xi;
        gemv_row<T>(i, m, V, ldv, hs, ar, ai);
        ld(src[i], xr, xi);
        const T y = mk<T>(xr - ar, xi - ai);
        t[i]      = y;
        double yr, yi;
        ld(y, yr, yi);
        acc[0] += yr * yr + yi * yi;
    }
    bsum<1>(acc, red);
    if(threadIdx.x == 0) {
        double *p = partial + static_cast<int64_t>(blockIdx.x) * nv + 2 * m;
        publish(p, acc[0], counter != nullptr);
        publish(p + 1, 0.0, counter != nullptr);
    }
    project_rows<T>(n, m, V, ldv, t, partial, nv, counter != nullptr, red);
    if(counter) fold_in_last_block(partial, nv, out, -1, nullptr, counter);
}

// The second pass where |t|^2 (h2[2 m]) fell below eta2 |src|^2 (nrm[0]), and the normalisation; nrm[2] = |t|^2.
template <typename T>
__global__ __launch_bounds__(VT_THREADS) void expand_finish_kernel(int64_t n, int m, const T *V, int64_t ldv, const double *h2, double eta2, T *t,
                                                                   double *nrm) {
    __shared__ double hs[2 * VEC_MAX_M];
    __shared__ double red[1][VT_THREADS / 64];
    __shared__ double total;
    double            post  = h2[2 * m];
    const bool        again = m > 0 && post < eta2 * nrm[0];
    if(again) { // the same in every workgroup
        double acc[1] = {0.0};
        for(int j = threadIdx.x; j < 2 * m; j += VT_THREADS) {
            hs[j] = h2[j];
            acc[0] += hs[j] * hs[j];
        }
        bsum<1>(acc, red);
        if(threadIdx.x == 0) total = acc[0];
        __syncthreads();
        post -= total;
        if(post < 0.0) post = 0.0; // NaN stays NaN
    }
    const double a = post > 0.0 ? 1.0 / sqrt(post) : 0.0; // a zero vector stays zero (breakdown tests see it)
    for(int64_t i = blockIdx.x * static_cast<int64_t>(VT_THREADS) + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * VT_THREADS) {
        double ar = 0, ai = 0, xr, xi;
        if(again) gemv_row<T>(i, m, V, ldv, hs, ar, ai);
        ld(t[i], xr, xi);
        t[i] = mk<T>(a * (xr - ar), a * (xi - ai));
    }
    if(blockIdx.x == 0 && threadIdx.x == 0) nrm[2] = post, nrm[3] = 0.0;
}

static bool expand_fits(int64_t n, int m) { return n <= MD_SHORT && m + 3 <= VEC_MAX_M; }
// One row a thread, or two where that lets the last workgroup fold.
static int expand_grid(int64_t n, int values) {
    const int b = static_cast<int>(std::max<int64_t>(1, (n + VT_THREADS - 1) / VT_THREADS));
    return b > FUSE_MAX_BLOCKS && b <= 2 * FUSE_MAX_BLOCKS && values <= FUSE_MAX_VALUES ? (b + 1) / 2 : b;
}

template <typename T>
bool expand_project(int64_t n, int m, const T *V, const T *W, int64_t ldv, const double *h_y, double *d_y, double theta, T *x, T *r, double *d_out,
                    double *d_tail, double *scratch, hipStream_t s) {
    if(!expand_fits(n, m)) return false;
    RitzCoef c{};
    if(m <= RITZ_ARGS) {
        std::copy(h_y, h_y + 2 * m, c.y);
        d_y = nullptr;
    } else {
        DMRG_HIP_CHECK(hipMemcpyAsync(d_y, h_y, 2 * static_cast<size_t>(m) * sizeof(double), hipMemcpyHostToDevice, s));
    }
    const int  g  = expand_grid(n, 2 * m + 6);
    const bool in = fused(g, 2 * m + 6);
    hipLaunchKernelGGL(ritz_project_kernel<T>, dim3(g), dim3(VT_THREADS), 0, s, n, m, V, W, ldv, d_y, c, theta, x, r, scratch,
                       in ? scratch_counter(scratch) : nullptr, d_out, d_tail);
    if(!in) hipLaunchKernelGGL(fold_columns, dim3(m + 3), dim3(VT_THREADS), 0, s, g, m + 3, scratch, d_out, m, d_tail, nullptr, HostCopy{});
    DMRG_HIP_CHECK(hipGetLastError());
    return true;
}

template <typename T>
bool expand_update(int64_t n, int m, const T *V, int64_t ldv, const double *d_h, const T *src, T *t, double eta2, double *d_h2, double *d_nrm,
                   double *scratch, hipStream_t s) {
    if(!expand_fits(n, m)) return false;
    const int  g  = expand_grid(n, 2 * m + 2);
    const bool in = fused(g, 2 * m + 2);
    hipLaunchKernelGGL(update_project_kernel<T>, dim3(g), dim3(VT_THREADS), 0, s, n, m, V, ldv, d_h, src, t, scratch,
                       in ? scratch_counter(scratch) : nullptr, d_h2);
    if(!in) hipLaunchKernelGGL(fold_columns, dim3(m + 1), dim3(VT_THREADS), 0, s, g, m + 1, scratch, d_h2, -1, nullptr, nullptr, HostCopy{});
    hipLaunchKernelGGL(expand_finish_kernel<T>, dim3(ew_grid(n)), dim3(VT_THREADS), 0, s, n, m, V, ldv, d_h2, eta2, t, d_nrm);
    DMRG_HIP_CHECK(hipGetLastError());
    return true;
}

// ------------------------------------------------------------------------------------------- basis rotation
// B[:, 0:k] <- B[:, 0:m] Q in place for up to two bases: a thread owns a row, reads its m values and writes k, so that a basis
// is read and written once; Q comes with the launch. Bounded by the launch up to about 10^5 rows, by memory beyond. As a
// GEMM with Q's upload, a copy back and a synchronisation per basis, a restart cost about 100 us in a sweep's small solves.
constexpr int ROT_MAX_M = 24;  // a row's values in registers
constexpr int ROT_ARGS  = 448; // doubles of Q (3.5 KiB of kernel arguments)
struct RotationCoef {
    double q[ROT_ARGS];
};
template <typename T>
__global__ __launch_bounds__(VT_THREADS) void rotate_basis_kernel(int64_t n, int m, int k, int64_t ldv, T *B0, T *B1, const RotationCoef c) {
    T            *B = blockIdx.y == 0 ? B0 : B1;
    const int64_t i = blockIdx.x * static_cast<int64_t>(VT_THREADS) + threadIdx.x;
    if(i >= n) return;
    T v[ROT_MAX_M];
#pragma unroll
    for(int a = 0; a < ROT_MAX_M; ++a)
        if(a < m) v[a] = B[i + a * ldv];
    for(int j = 0; j < k; ++j) {
        double re = 0, im = 0;
#pragma unroll
        for(int a = 0; a < ROT_MAX_M; ++a)
            if(a < m) {
                double vr, vi;
                ld(v[a], vr, vi);
                if constexpr(vtraits<T>::cx) {
                    const double qr = c.q[2 * (j * m + a)], qi = c.q[2 * (j * m + a) + 1];
                    re += vr * qr - vi * qi;
                    im += vr * qi + vi * qr;
                } else {
                    re += vr * c.q[j * m + a];
                }
            }
        B[i + j * ldv] = mk<T>(re, im);
    }
}

template <typename T>
bool rotate_basis(int64_t n, int m, int k, int64_t ldv, T *B0, T *B1, const std::complex<double> *Q, hipStream_t s) {
    const int64_t blocks = (n + VT_THREADS - 1) / VT_THREADS;
    if(m > ROT_MAX_M || k > m || m * k * (vtraits<T>::cx ? 2 : 1) > ROT_ARGS || blocks >= (int64_t(1) << 31)) return false;
    RotationCoef c{};
    for(int i = 0; i < m * k; ++i) {
        if constexpr(vtraits<T>::cx) c.q[2 * i] = Q[i].real(), c.q[2 * i + 1] = Q[i].imag();
        else c.q[i] = Q[i].real();
    }
    hipLaunchKernelGGL(rotate_basis_kernel<T>, dim3(static_cast<unsigned>(blocks), B1 ? 2 : 1), dim3(VT_THREADS), 0, s, n, m, k, ldv, B0, B1, c);
    DMRG_HIP_CHECK(hipGetLastError());
    return true;
}

// ------------------------------------------------------------------------------------------- Gram-Schmidt on three vectors
// Modified Gram-Schmidt on the columns of V (n x 3) in one workgroup, a thread owning its rows throughout: a column of norm
// below eps stays as it is and later ones are not projected against it. Column by column from the host, the norms cost three
// synchronisations and twelve launches. Bounded by latency up to the limit (about 1 us per pass), by one CU's loads beyond.
constexpr int64_t GS3_MAX_BYTES = 131072;
template <typename T>
__global__ __launch_bounds__(EX_THREADS) void gram_schmidt3_kernel(int n, T *V, double eps) {
    __shared__ double red[4][EX_WAVES];
    for(int i = 0; i < 3; ++i) {
        T     *vi      = V + static_cast<int64_t>(i) * n;
        double nrm2[1] = {0.0};
        for(int k = threadIdx.x; k < n; k += EX_THREADS) {
            double re, im;
            ld(vi[k], re, im);
            nrm2[0] += re * re + im * im;
        }
        all_sum<1>(nrm2, red);
        const double rii = sqrt(nrm2[0]);
        if(rii < eps) continue; // the same in every thread
        const double a = 1.0 / rii;
        double       h[4] = {0.0, 0.0, 0.0, 0.0};
        for(int k = threadIdx.x; k < n; k += EX_THREADS) {
            double re, im;
            ld(vi[k], re, im);
            const T q = mk<T>(a * re, a * im);
            vi[k]     = q;
            ld(q, re, im);
            for(int j = i + 1; j < 3; ++j) {
                double xr, xi;
                ld(V[static_cast<int64_t>(j) * n + k], xr, xi);
                h[2 * (j - i - 1)] += re * xr + im * xi;
                h[2 * (j - i - 1) + 1] += re * xi - im * xr;
            }
        }
        all_sum<4>(h, red);
        for(int k = threadIdx.x; k < n; k += EX_THREADS) {
            double re, im;
            ld(vi[k], re, im);
            for(int j = i + 1; j < 3; ++j) {
                const double hr = h[2 * (j - i - 1)], hi = h[2 * (j - i - 1) + 1];
                double       xr, xi;
                ld(V[static_cast<int64_t>(j) * n + k], xr, xi);
                V[static_cast<int64_t>(j) * n + k] = mk<T>(xr - (re * hr - im * hi), xi - (re * hi + im * hr));
            }
        }
    }
}
template <typename T>
bool gram_schmidt3(int64_t n, T *V, double eps, hipStream_t s) {
    if(n * static_cast<int64_t>(sizeof(T)) > GS3_MAX_BYTES) return false;
    hipLaunchKernelGGL(gram_schmidt3_kernel<T>, dim3(1), dim3(EX_THREADS), 0, s, static_cast<int>(n), V, eps);
    DMRG_HIP_CHECK(hipGetLastError());
    return true;
}

template <typename T>
__global__ void combine3_kernel(int64_t n, const T *V, double c0, double c1, double c2, T *out) {
    for(int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        double a[3][2];
        for(int j = 0; j < 3; ++j) ld(V[i + j * n], a[j][0], a[j][1]);
        out[i] = mk<T>(c0 * a[0][0] + c1 * a[1][0] + c2 * a[2][0], c0 * a[0][1] + c1 * a[1][1] + c2 * a[2][1]);
    }
}
template <typename T>
void combine3(int64_t n, const T *V, const double *c, T *out, hipStream_t s) {
    hipLaunchKernelGGL(combine3_kernel<T>, dim3(ew_grid(n)), dim3(VT_THREADS), 0, s, n, V, c[0], c[1], c[2], out);
    DMRG_HIP_CHECK(hipGetLastError());
}

// ------------------------------------------------------------------------------------------- elementwise
template <typename T>
__global__ void scale_inv_norm_kernel(int64_t n, T *x, const double *nrm2) {
    const double a = nrm2[0] > 0.0 ? 1.0 / sqrt(nrm2[0]) : 0.0; // a zero vector stays zero (breakdown tests see it)
    for(int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        double re, im;
        ld(x[i], re, im);
        x[i] = mk<T>(a * re, a * im);
    }
}
template <typename T>
void scale_by_inv_norm(int64_t n, T *x, const double *d_nrm2, hipStream_t s) {
    hipLaunchKernelGGL(scale_inv_norm_kernel<T>, dim3(ew_grid(n)), dim3(VT_THREADS), 0, s, n, x, d_nrm2);
    DMRG_HIP_CHECK(hipGetLastError());
}

template <typename T>
__global__ void scale_kernel(int64_t n, T *x, double a) {
    for(int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        double re, im;
        ld(x[i], re, im);
        x[i] = mk<T>(a * re, a * im);
    }
}
template <typename T>
void scale(int64_t n, T *x, double alpha, hipStream_t s) {
    hipLaunchKernelGGL(scale_kernel<T>, dim3(ew_grid(n)), dim3(VT_THREADS), 0, s, n, x, alpha);
    DMRG_HIP_CHECK(hipGetLastError());
}

template <typename T, typename D>
__global__ void jacobi_kernel(int64_t n, const T *r, const D *diag, double theta, double floor, T *t) {
    for(int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        double rr, ri, dr, di;
        ld(r[i], rr, ri);
        ld(diag[i], dr, di);
        double den = dr - theta;
        if(fabs(den) < floor) den = den < 0 ? -floor : floor;
        t[i] = mk<T>(rr / den, ri / den);
    }
}
template <typename T, typename D>
void jacobi_precond(int64_t n, const T *r, const D *diag, double theta, double floor, T *t, hipStream_t s) {
    hipLaunchKernelGGL((jacobi_kernel<T, D>), dim3(ew_grid(n)), dim3(VT_THREADS), 0, s, n, r, diag, theta, floor, t);
    DMRG_HIP_CHECK(hipGetLastError());
}

__device__ inline uint64_t splitmix64(uint64_t z) {
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}
__device__ inline double u11(uint64_t z) { return static_cast<double>(z >> 11) * (2.0 / 9007199254740992.0) - 1.0; }

template <typename T>
__global__ void random_kernel(int64_t n, T *x, uint64_t seed) {
    for(int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const uint64_t h = splitmix64(seed * 0x100000001B3ull + static_cast<uint64_t>(i));
        x[i]             = mk<T>(u11(h), vtraits<T>::cx ? u11(splitmix64(h)) : 0.0);
    }
}
template <typename T>
void random_fill(int64_t n, T *x, uint64_t seed, hipStream_t s) {
    hipLaunchKernelGGL(random_kernel<T>, dim3(ew_grid(n)), dim3(VT_THREADS), 0, s, n, x, seed);
    DMRG_HIP_CHECK(hipGetLastError());
}

template <typename TO, typename TI>
__global__ void convert_kernel(int64_t n, const TI *in, TO *out) {
    for(int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        double re, im;
        ld(in[i], re, im);
        out[i] = mk<TO>(re, im);
    }
}
template <typename TO, typename TI>
void convert(int64_t n, const TI *in, TO *out, hipStream_t s) {
    hipLaunchKernelGGL((convert_kernel<TO, TI>), dim3(ew_grid(n)), dim3(VT_THREADS), 0, s, n, in, out);
    DMRG_HIP_CHECK(hipGetLastError());
}

// ------------------------------------------------------------------------------------------- projected CG
// Kernels of the FP32 correction-equation solver (CG on A = sigma P (H - theta) P, P = I - x x^H). The scalars
// live on the device: dots = {x^H q (2), p^H q (2)}; state as laid out by the CG_* offsets. Every block of a
// kernel derives the same step from the same inputs; only block 0 writes the state, into the slot of the
// next iteration (k + 1) & 1, which no block of the current kernel reads.

template <typename T>
__global__ __launch_bounds__(VT_THREADS) void cg_shift_kernel(int64_t n, const T *p, T *q, double theta, double sigma, const double *state,
                                                              int k) {
    if(state[CG_STOP + (k & 1)] != 0.0) return;
    for(int64_t i = blockIdx.x * static_cast<int64_t>(VT_THREADS) + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * VT_THREADS) {
        double qr, qi, pr, pi;
        ld(q[i], qr, qi);
        ld(p[i], pr, pi);
        q[i] = mk<T>(sigma * (qr - theta * pr), sigma * (qi - theta * pi));
    }
}

// r = -sigma (r - x c) with c = x^H r (dots[0..1]); p = r; t = 0; partial |r|^2 per block.
template <typename T>
__global__ __launch_bounds__(VT_THREADS) void cg_init_kernel(int64_t n, const T *x, const double *c, double sigma, T *r, T *p, T *t,
                                                             double *partial, unsigned *counter, double *out) {
    __shared__ double red[1][VT_THREADS / 64];
    const double      cr = c[0], ci = c[1];
    double            acc[1] = {0.0};
    for(int64_t i = blockIdx.x * static_cast<int64_t>(VT_THREADS) + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * VT_THREADS) {
        double rr, ri, xr, xi;
        ld(r[i], rr, ri);
        ld(x[i], xr, xi);
        const double vr = -sigma * (rr - (xr * cr - xi * ci)), vi = -sigma * (ri - (xr * ci + xi * cr));
        const T      v  = mk<T>(vr, vi);
        r[i]            = v;
        p[i]            = v;
        t[i]            = mk<T>(0.0, 0.0);
        double wr, wi;
        ld(v, wr, wi);
        acc[0] += wr * wr + wi * wi;
    }
    bsum<1>(acc, red);
    if(threadIdx.x == 0) {
        publish(partial + 2 * blockIdx.x, acc[0], counter != nullptr);
        publish(partial + 2 * blockIdx.x + 1, 0.0, counter != nullptr);
    }
    if(counter) fold_in_last_block(partial, 2, out, -1, nullptr, counter);
}

// state <- start of the iteration: rho_0 = |r|^2 (rr[0]); stopped when r = 0.
__global__ void cg_start_kernel(const double *rr, double *state) {
    state[CG_RHO]      = rr[0];
    state[CG_RHO + 1]  = 0.0;
    state[CG_RHO0]     = rr[0];
    state[CG_STOP]     = rr[0] > 0.0 ? 0.0 : 1.0;
    state[CG_STOP + 1] = 0.0;
    state[CG_ITS]      = 0.0;
    state[CG_RR]       = rr[0];
}

// alpha = rho / p^H q; t += alpha p; r -= alpha (q - x (x^H q)); partial |r|^2. No update on a breakdown (p^H q <= 0).
template <typename T>
__global__ __launch_bounds__(VT_THREADS) void cg_update_kernel(int64_t n, const T *x, const T *p, const T *q, const double *dots,
                                                               const double *state, int k, T *t, T *r, double *partial,
                                                               unsigned *counter, double *out) {
    __shared__ double red[1][VT_THREADS / 64];
    const double      pq   = dots[2];
    const bool        live = state[CG_STOP + (k & 1)] == 0.0 && pq > 0.0;
    const double      a    = live ? state[CG_RHO + (k & 1)] / pq : 0.0;
    const double      cr = dots[0], ci = dots[1];
    double            acc[1] = {0.0};
    if(live) {
        for(int64_t i = blockIdx.x * static_cast<int64_t>(VT_THREADS) + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * VT_THREADS) {
            double xr, xi, pr, pi, qr, qi, tr, ti, rr, ri;
            ld(x[i], xr, xi);
            ld(p[i], pr, pi);
            ld(q[i], qr, qi);
            ld(t[i], tr, ti);
            ld(r[i], rr, ri);
            t[i]            = mk<T>(tr + a * pr, ti + a * pi);
            const double yr = qr - (xr * cr - xi * ci), yi = qi - (xr * ci + xi * cr);
            const T      v  = mk<T>(rr - a * yr, ri - a * yi);
            r[i]            = v;
            double wr, wi;
            ld(v, wr, wi);
            acc[0] += wr * wr + wi * wi;
        }
    }
    bsum<1>(acc, red);
    if(threadIdx.x == 0) {
        publish(partial + 2 * blockIdx.x, acc[0], counter != nullptr);
        publish(partial + 2 * blockIdx.x + 1, 0.0, counter != nullptr);
    }
    if(counter) fold_in_last_block(partial, 2, out, -1, nullptr, counter);
}

// beta = |r|^2 / rho; p = r + beta p; block 0 advances the state (rho, stop flag, step count).
template <typename T>
__global__ __launch_bounds__(VT_THREADS) void cg_direction_kernel(int64_t n, const T *r, const double *dots, const double *rr,
                                                                  double *state, int k, double rtol2, T *p) {
    const bool   stopped = state[CG_STOP + (k & 1)] != 0.0;
    const bool   live    = !stopped && dots[2] > 0.0;
    const double rho     = state[CG_RHO + (k & 1)];
    if(blockIdx.x == 0 && threadIdx.x == 0) {
        const int nx          = (k + 1) & 1;
        state[CG_RHO + nx]    = live ? rr[0] : rho;
        state[CG_STOP + nx]   = (!live || rr[0] <= rtol2 * state[CG_RHO0]) ? 1.0 : 0.0;
        state[CG_ITS]         = state[CG_ITS] + (live ? 1.0 : 0.0);
        if(live) state[CG_RR] = rr[0];
    }
    if(!live) return;
    const double b = rr[0] / rho;
    for(int64_t i = blockIdx.x * static_cast<int64_t>(VT_THREADS) + threadIdx.x; i < n; i += static_cast<int64_t>(gridDim.x) * VT_THREADS) {
        double rr_, ri, pr, pi;
        ld(r[i], rr_, ri);
        ld(p[i], pr, pi);
        p[i] = mk<T>(rr_ + b * pr, ri + b * pi);
    }
}

template <typename T>
void cg_init(int64_t n, const T *x, const double *d_c, double sigma, T *r, T *p, T *t, double *d_rr, double *state, double *scratch,
             hipStream_t s) {
    const int g = grid_for(n);
    const bool in_last = fused(g, 2);
    hipLaunchKernelGGL(cg_init_kernel<T>, dim3(g), dim3(VT_THREADS), 0, s, n, x, d_c, sigma, r, p, t, scratch,
                       in_last ? scratch_counter(scratch) : nullptr, d_rr);
    if(!in_last) hipLaunchKernelGGL(fold_columns, dim3(1), dim3(VT_THREADS), 0, s, g, 1, scratch, d_rr, -1, nullptr, nullptr, HostCopy{});
    hipLaunchKernelGGL(cg_start_kernel, dim3(1), dim3(1), 0, s, d_rr, state);
    DMRG_HIP_CHECK(hipGetLastError());
}

template <typename T>
void cg_shift(int64_t n, const T *p, T *q, double theta, double sigma, const double *state, int k, hipStream_t s) {
    hipLaunchKernelGGL(cg_shift_kernel<T>, dim3(grid_for(n)), dim3(VT_THREADS), 0, s, n, p, q, theta, sigma, state, k);
    DMRG_HIP_CHECK(hipGetLastError());
}

template <typename T>
void cg_step(int64_t n, const T *x, T *p, const T *q, const double *d_dots, T *t, T *r, double *d_rr, double *state, int k,
             double rtol2, double *scratch, hipStream_t s) {
    const int g = grid_for(n);
    const bool in_last = fused(g, 2);
    hipLaunchKernelGGL(cg_update_kernel<T>, dim3(g), dim3(VT_THREADS), 0, s, n, x, p, q, d_dots, state, k, t, r, scratch,
                       in_last ? scratch_counter(scratch) : nullptr, d_rr);
    if(!in_last) hipLaunchKernelGGL(fold_columns, dim3(1), dim3(VT_THREADS), 0, s, g, 1, scratch, d_rr, -1, nullptr, nullptr, HostCopy{});
    hipLaunchKernelGGL(cg_direction_kernel<T>, dim3(g), dim3(VT_THREADS), 0, s, n, r, d_dots, d_rr, state, k, rtol2, p);
    DMRG_HIP_CHECK(hipGetLastError());
}

#define DMRG_VEC_INST(T)                                                                                                 \
    template void multidot<T>(int64_t, int, const T *, int64_t, const T *, double *, double *, hipStream_t);          \
    template void gemv_update<T>(int64_t, int, const T *, int64_t, const double *, double, double, T *, hipStream_t); \
    template void ritz_residual<T>(int64_t, int, const T *, const T *, int64_t, const double *, double *, double, T *,  \
                                   T *, double *, double *, double *, hipStream_t);                                    \
    template void multidot_to_host<T>(int64_t, int, const T *, int64_t, const T *, double *, double *, int, int, double *, hipStream_t);\
    template bool expand_small<T>(int64_t, int, const T *, const T *, int64_t, const double *, double, T *, T *, const T *, T *, double,\
                                  double *, double *, hipStream_t);                                                   \
    template bool expand_project<T>(int64_t, int, const T *, const T *, int64_t, const double *, double *, double, T *, T *,\
                                    double *, double *, double *, hipStream_t);                                       \
    template bool expand_update<T>(int64_t, int, const T *, int64_t, const double *, const T *, T *, double, double *, double *,\
                                   double *, hipStream_t);                                                            \
    template bool rotate_basis<T>(int64_t, int, int, int64_t, T *, T *, const std::complex<double> *, hipStream_t);   \
    template bool gram_schmidt3<T>(int64_t, T *, double, hipStream_t);                                                \
    template void combine3<T>(int64_t, const T *, const double *, T *, hipStream_t);                                  \
    template void scale_by_inv_norm<T>(int64_t, T *, const double *, hipStream_t);                                    \
    template void scale<T>(int64_t, T *, double, hipStream_t);                                                         \
    template void random_fill<T>(int64_t, T *, uint64_t, hipStream_t);                                               \
    template void multidot_x<T>(int64_t, int, const T *, int64_t, const T *, double *, double *, const int *, double *,  \
                                hipStream_t);                                                                          \
    template void multidot_dgks<T>(int64_t, int, const T *, int64_t, const T *, double *, const double *, const double *, \
                                   double, int *, double *, hipStream_t);                                              \
    template void gemv_update_norm<T>(int64_t, int, const T *, int64_t, const double *, double, double, const T *, T *,  \
                                      double *, const int *, double *, hipStream_t);
DMRG_VEC_INST(double)
DMRG_VEC_INST(float)
#define DMRG_CG_INST(T)                                                                                                  \
    template void cg_init<T>(int64_t, const T *, const double *, double, T *, T *, T *, double *, double *, double *,     \
                             hipStream_t);                                                                               \
    template void cg_shift<T>(int64_t, const T *, T *, double, double, const double *, int, hipStream_t);               \
    template void cg_step<T>(int64_t, const T *, T *, const T *, const double *, T *, T *, double *, double *, int, double, \
                             double *, hipStream_t);
DMRG_CG_INST(float)
DMRG_CG_INST(cpx<float>)
DMRG_VEC_INST(cpx<double>)
DMRG_VEC_INST(cpx<float>)
template void jacobi_precond<double, double>(int64_t, const double *, const double *, double, double, double *, hipStream_t);
template void jacobi_precond<float, double>(int64_t, const float *, const double *, double, double, float *, hipStream_t);
template void jacobi_precond<cpx<double>, cpx<double>>(int64_t, const cpx<double> *, const cpx<double> *, double, double,
                                                       cpx<double> *, hipStream_t);
template void jacobi_precond<cpx<float>, cpx<double>>(int64_t, const cpx<float> *, const cpx<double> *, double, double,
                                                      cpx<float> *, hipStream_t);
template void convert<float, double>(int64_t, const double *, float *, hipStream_t);
template void convert<double, float>(int64_t, const float *, double *, hipStream_t);
template void convert<cpx<float>, cpx<double>>(int64_t, const cpx<double> *, cpx<float> *, hipStream_t);
template void convert<cpx<double>, cpx<float>>(int64_t, const cpx<float> *, cpx<double> *, hipStream_t);
template void convert<double, double>(int64_t, const double *, double *, hipStream_t);
template void convert<cpx<double>, cpx<double>>(int64_t, const cpx<double> *, cpx<double> *, hipStream_t);

} // namespace dmrg
