// One-sided (Hestenes) Jacobi SVD on the GPU, the method of LAPACK's gesvj that the reference can select
// (svd_lapacke.cpp:193-212). The columns of W (m x n, m >= n) are rotated pairwise until they are mutually
// orthogonal; then S = column norms, U = normalised columns and V = the accumulated rotations. One-sided
// Jacobi keeps high relative accuracy for small singular values.
//
// Each sweep runs the n(n-1)/2 pairs in n-1 rounds of disjoint pairs (circle method). When W and V fit in
// LDS, one workgroup runs every sweep with both matrices resident and a barrier between rounds (up to 128 x 64 the whole
// SVD is that one launch). Others of up to 32 columns launch one kernel per round with one workgroup (1 to 4 wavefronts, by
// column length) per pair; larger ones pair blocks of 16 columns instead (block one-sided Jacobi, three launches per round of block pairs). The
// only host round trip per sweep reads whether any rotation was applied.
#include "svd.hpp"

#include <algorithm>
#include <cmath>

namespace dmrg {

namespace {

template <typename T>
struct jtraits;
template <>
struct jtraits<double> {
    static constexpr bool cx = false;
};
template <>
struct jtraits<cpx<double>> {
    static constexpr bool cx = true;
};

// |gr + i gi| (gi = 0 for real T), the inner product of two columns of squared norms al and be, where they are to be rotated,
// else 0. A column whose squared norm is zero counts as a zero column, also where rounding has left something below 1e-162 in
// it: linearly dependent columns shrink by eps a sweep. Norms of 1e130 or 1e-130 have products and squared products outside
// the range; where al be is well inside, so are the others as far as they matter (|g|^2 <= al be), which one test of al be on
// the serial chain of a round decides (tests of each root cost the block path 3 %).
template <typename T>
__device__ inline double coupling(double gr, double gi, double al, double be, double tol) {
    const double p = al * be, g2 = jtraits<T>::cx ? gr * gr + gi * gi : gr * gr;
    if(__builtin_expect(!(p > 1e-240 && p < 1e240), 0)) {
        const double top = fmax(fabs(gr), fabs(gi)), f = top < 1.0 ? 0x1p+520 : 0x1p-520;
        const double g = jtraits<T>::cx ? sqrt((gr * f) * (gr * f) + (gi * f) * (gi * f)) / f : fabs(gr);
        const double b = sqrt(al) * sqrt(be);
        return g > tol * b && b > 0.0 ? g : 0.0;
    }
    return g2 > (tol * tol) * p ? (jtraits<T>::cx ? sqrt(g2) : fabs(gr)) : 0.0;
}

// The smaller root of t^2 + 2 z t = 1, of z's sign.
__device__ inline double tangent(double z) {
    if(fabs(z) > 1e150) return 0.5 / z; // z^2 leaves the range
    return (z >= 0 ? 1.0 : -1.0) / (fabs(z) + sqrt(1.0 + z * z));
}

__device__ inline double wave_sum(double v) {
#pragma unroll
    for(int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Pair of round r (circle method over np players; player np-1 stays fixed).
__device__ inline void round_pair(int np, int r, int i, int &a, int &b) {
    if(i == 0) {
        a = r % (np - 1);
        b = np - 1;
    } else {
        a = (r + i) % (np - 1);
        b = (r - i + (np - 1)) % (np - 1);
    }
}

// One round: workgroup w of the grid (NT threads, a multiple of 64) handles pair w. flag[0] is raised when a
// rotation is applied. Several wavefronts per pair shorten the dependent walk down long columns.
template <typename T, int NT>
__global__ __launch_bounds__(NT) void jacobi_round(int m, int n, int np, int r, T *W, T *V, double tol, unsigned *flag) {
    int p, q;
    round_pair(np, r, blockIdx.x, p, q);
    if(p >= n || q >= n) return; // padding player (odd n); uniform over the workgroup
    if(p > q) {
        const int t = p;
        p           = q;
        q           = t;
    }
    T        *wp = W + static_cast<int64_t>(p) * m, *wq = W + static_cast<int64_t>(q) * m;
    const int tid = threadIdx.x;
    double    al = 0, be = 0, gr = 0, gi = 0;
#pragma unroll 4
    for(int i = tid; i < m; i += NT) {
        if constexpr(jtraits<T>::cx) {
            const T x = wp[i], y = wq[i];
            al += x.re * x.re + x.im * x.im;
            be += y.re * y.re + y.im * y.im;
            gr += x.re * y.re + x.im * y.im; // conj(x) y
            gi += x.re * y.im - x.im * y.re;
        } else {
            const double x = wp[i], y = wq[i];
            al += x * x;
            be += y * y;
            gr += x * y;
        }
    }
    al = wave_sum(al);
    be = wave_sum(be);
    gr = wave_sum(gr);
    gi = wave_sum(gi);
    if constexpr(NT > 64) {
        __shared__ double red[4][NT / 64];
        const int         w = tid >> 6;
        if((tid & 63) == 0) red[0][w] = al, red[1][w] = be, red[2][w] = gr, red[3][w] = gi;
        __syncthreads();
        al = be = gr = gi = 0;
#pragma unroll
        for(int k = 0; k < NT / 64; ++k) al += red[0][k], be += red[1][k], gr += red[2][k], gi += red[3][k];
    }
    const double g = coupling<T>(gr, gi, al, be, tol);
    if(g == 0.0) return; // same decision in every thread of the workgroup
    // Align the phase of column q so that the off-diagonal is |g|, then a real rotation zeroes it:
    // t = sign(z) / (|z| + sqrt(1 + z^2)), z = (be - al) / (2 |g|); w_p' = c w_p - s w_q^, w_q' = s w_p + c w_q^.
    const double z  = (be - al) / (2.0 * g);
    const double t  = tangent(z);
    const double c  = 1.0 / sqrt(1.0 + t * t), s = c * t;
    const double er = gr / g, ei = -gi / g; // e^{-i phi}
    if(tid == 0) atomicOr(flag, 1u);
    auto rotate = [&](T *x, T *y, int len) {
#pragma unroll 4
        for(int i = tid; i < len; i += NT) {
            if constexpr(jtraits<T>::cx) {
                const T      xv = x[i], yv = y[i];
                const double yr = yv.re * er - yv.im * ei, yi = yv.re * ei + yv.im * er; // e^{-i phi} y
                x[i]            = T{c * xv.re - s * yr, c * xv.im - s * yi};
                y[i]            = T{s * xv.re + c * yr, s * xv.im + c * yi};
            } else {
                const double xv = x[i], yv = y[i] * er;
                x[i]            = c * xv - s * yv;
                y[i]            = s * xv + c * yv;
            }
        }
    };
    rotate(wp, wq, m);
    rotate(V + static_cast<int64_t>(p) * n, V + static_cast<int64_t>(q) * n, n);
}

// ------------------------------------------------------------------------------------------------------------
// Block one-sided Jacobi: columns in blocks of BB = B2 / 2 (W and V padded with zero columns to whole blocks);
// each round pairs the blocks (circle method) and, for every block pair, (1) forms the Gram matrix G = X^H X of
// its B2 columns X on the matrix cores (partial sums over row chunks, bj_gram_mfma), (2) runs cyclic two-sided
// Jacobi on G in LDS, accumulating Q (bj_eig; the 2 x 2 rotation and its threshold are those of jacobi_round,
// computed from the same inner products), (3) rotates X <- X Q and V[:, cols] <- V[:, cols] Q on the matrix cores
// (bj_update_mfma). A sweep meets every column pair, as the scalar sweep does, in n / BB - 1 rounds of 3
// launches instead of n - 1 launches.

template <typename T>
__device__ inline T jconj(const T &a) {
    if constexpr(jtraits<T>::cx) return T{a.re, -a.im};
    else return a;
}
template <typename T>
__device__ inline T jmul(const T &a, const T &b) {
    if constexpr(jtraits<T>::cx) return T{a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
    else return a * b;
}
template <typename T>
__device__ inline T jzero() {
    if constexpr(jtraits<T>::cx) return T{0.0, 0.0};
    else return 0.0;
}
template <typename T>
__device__ inline T jscale(double a, const T &b) {
    if constexpr(jtraits<T>::cx) return T{a * b.re, a * b.im};
    else return a * b;
}
template <typename T>
__device__ inline T jadd(const T &a, const T &b) {
    if constexpr(jtraits<T>::cx) return T{a.re + b.re, a.im + b.im};
    else return a + b;
}
template <typename T>
__device__ inline T jreal(double a) {
    if constexpr(jtraits<T>::cx) return T{a, 0.0};
    else return a;
}
template <typename T>
__device__ inline double jre(const T &a) {
    if constexpr(jtraits<T>::cx) return a.re;
    else return a;
}

constexpr int BJ_THREADS = 256;
constexpr int BJ_ROWS    = 64; // granularity of the Gram kernel's row chunks

// Sums the partial Gram matrices of a pair (fixed order), diagonalises G by cyclic Jacobi sweeps in LDS and
// writes the accumulated rotation Q (B2 x B2, column-major) and whether any rotation was applied.
template <typename T, int B2>
__global__ __launch_bounds__(BJ_THREADS) void bj_eig(int n, int nbp, int r, int ks, const T *part, T *qbuf, int *rotated,
                                                      double tol, int max_inner, unsigned *flag) {
    constexpr int BB = B2 / 2, NP = B2 / 2;
    int           P, Q;
    round_pair(nbp, r, blockIdx.x, P, Q);
    const int tid = threadIdx.x;
    if(P * BB >= n || Q * BB >= n) {
        if(tid == 0) rotated[blockIdx.x] = 0;
        return;
    }
    __shared__ T      G[B2][B2 + 1], Qs[B2][B2 + 1];
    __shared__ double rc[NP], rs[NP];
    __shared__ T      re[NP];
    __shared__ int    rp[NP], rq[NP], ron[NP];
    __shared__ int    any_sweep, any_total;
    const T          *src = part + static_cast<int64_t>(blockIdx.x) * ks * B2 * B2;
    for(int idx = tid; idx < B2 * B2; idx += BJ_THREADS) {
        const int i = idx % B2, j = idx / B2;
        T         a = jzero<T>();
        for(int c = 0; c < ks; ++c) a = jadd(a, src[static_cast<int64_t>(c) * B2 * B2 + idx]);
        G[i][j]  = a;
        Qs[i][j] = jreal<T>(i == j ? 1.0 : 0.0);
    }
    if(tid == 0) any_total = 0;
    __syncthreads();
    // Hermitian: keep the upper triangle, real diagonal.
    for(int idx = tid; idx < B2 * B2; idx += BJ_THREADS) {
        const int i = idx % B2, j = idx / B2;
        if(i > j) G[i][j] = jconj(G[j][i]);
        else if(i == j) G[i][i] = jreal<T>(jre(G[i][i]));
    }
    __syncthreads();
    for(int sw = 0; sw < max_inner; ++sw) {
        if(tid == 0) any_sweep = 0;
        __syncthreads();
        for(int rr = 0; rr < B2 - 1; ++rr) {
            if(tid < NP) {
                int p, q;
                round_pair(B2, rr, tid, p, q);
                if(p > q) {
                    const int t = p;
                    p           = q;
                    q           = t;
                }
                rp[tid]         = p;
                rq[tid]         = q;
                const double al = jre(G[p][p]), be = jre(G[q][q]);
                const T      gm = G[p][q];
                double       gr, gi;
                if constexpr(jtraits<T>::cx) gr = gm.re, gi = gm.im;
                else gr = gm, gi = 0.0;
                const double g  = coupling<T>(gr, gi, al, be, tol);
                const bool   on = g != 0.0;
                ron[tid]        = on ? 1 : 0;
                if(on) {
                    const double z = (be - al) / (2.0 * g);
                    const double t = tangent(z);
                    const double c = 1.0 / sqrt(1.0 + t * t);
                    rc[tid]        = c;
                    rs[tid]        = c * t;
                    if constexpr(jtraits<T>::cx) re[tid] = T{gr / g, -gi / g}; // e^{-i phi}
                    else re[tid] = gr / g;
                    any_sweep = 1;
                }
            }
            __syncthreads();
            // rows p, q of G <- J^H G
            for(int k = tid; k < NP * B2; k += BJ_THREADS) {
                const int u = k / B2, col = k % B2;
                if(!ron[u]) continue;
                const int    p = rp[u], q = rq[u];
                const double c = rc[u], sn = rs[u];
                const T      ec = jconj(re[u]);
                const T      a = G[p][col], b = jmul(ec, G[q][col]);
                G[p][col]      = jadd(jscale(c, a), jscale(-sn, b));
                G[q][col]      = jadd(jscale(sn, a), jscale(c, b));
            }
            __syncthreads();
            // columns p, q of G and Q <- . J
            for(int k = tid; k < 2 * NP * B2; k += BJ_THREADS) {
                const int u = (k / B2) % NP, row = k % B2;
                if(!ron[u]) continue;
                const int    p = rp[u], q = rq[u];
                const double c = rc[u], sn = rs[u];
                const bool onG = k < NP * B2;
                T(*M)[B2 + 1]  = onG ? G : Qs;
                const T a = M[row][p], b = jmul(re[u], M[row][q]);
                const T np_ = jadd(jscale(c, a), jscale(-sn, b)), nq_ = jadd(jscale(sn, a), jscale(c, b));
                // the rotation annihilates G[p][q] and G[q][p]: store the exact zero there
                M[row][p] = (onG && row == q) ? jzero<T>() : np_;
                M[row][q] = (onG && row == p) ? jzero<T>() : nq_;
            }
            __syncthreads();
        }
        const int done = !any_sweep;
        if(tid == 0 && any_sweep) any_total = 1;
        __syncthreads();
        if(done) break;
    }
    if(tid == 0) {
        rotated[blockIdx.x] = any_total;
        if(any_total) atomicOr(flag, 1u);
    }
    if(any_total) {
        T *qo = qbuf + static_cast<int64_t>(blockIdx.x) * B2 * B2;
        for(int idx = tid; idx < B2 * B2; idx += BJ_THREADS) qo[idx] = Qs[idx % B2][idx / B2];
    }
}

// LDS budget of the single-workgroup paths (gfx950 has 160 KiB per CU).
constexpr size_t JACOBI_LDS_BYTES = 152 * 1024;

// Sum over the 16 lanes of a row, in all of them, by data-parallel primitives: a step takes two moves and an addition in
// registers, where a shuffle through LDS takes its latency.
template <int CTRL>
__device__ inline double dpp_move(double v) {
    const auto b  = __builtin_bit_cast(uint64_t, v);
    const int  lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(b), CTRL, 0xf, 0xf, true);
    const int  hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(b >> 32), CTRL, 0xf, 0xf, true);
    return __builtin_bit_cast(double, static_cast<uint64_t>(static_cast<uint32_t>(hi)) << 32 | static_cast<uint32_t>(lo));
}
__device__ inline double row_sum(double v) {
    v += dpp_move<0xb1>(v);  // lane ^ 1
    v += dpp_move<0x4e>(v);  // lane ^ 2
    v += dpp_move<0x141>(v); // 7 - lane within 8
    v += dpp_move<0x140>(v); // 15 - lane within 16
    return v;
}

// The whole SVD in one workgroup, W (n columns of up to 16 E rows) and V (n x n, up to 16 EV rows) resident in LDS: loads A
// (its adjoint where tr), runs all sweeps, sorts and writes U, Vt and S[0:n], and the number of sweeps to S[n]. A row of 16
// lanes has one pair of a round, with its elements of both columns in registers between the inner products and the
// rotation; n <= 64 makes at most 32 pairs, so that every row has one pair a round and a barrier ends the round. A round is
// one serial chain (LDS read, three sums, the rotation's angle, LDS write, barrier), which is what bounds it: hence the
// sums without LDS and an angle of two dependent roots instead of five roots and quotients. Whole SVDs of a graded
// spectrum: FP64 64x64 1.39 ms against 5.4 in rounds of block pairs with three launches each, complex 2.65 against 7.0;
// FP64 32x32 0.31 ms against 1.20 with sums through LDS and the rest in launches of its own.
template <typename T, int E, int EV>
__global__ __launch_bounds__(512) void jacobi_resident(int m, int n, int tr, const T *A, double tol, int max_sweeps, T *U, T *Vt, double *S) {
    constexpr bool cx = jtraits<T>::cx;
    // 16 doubles of padding: neighbouring columns lie in different halves of the banks (complex rows fill all banks).
    constexpr int  SW = 16 * E + (cx || E % 2 ? 0 : 16), SV = 16 * EV + (cx || EV % 2 ? 0 : 16);
    extern __shared__ __attribute__((aligned(16))) unsigned char jacobi_lds_raw[];
    T             *Ws = reinterpret_cast<T *>(jacobi_lds_raw), *Vs = Ws + n * SW;
    __shared__ double nrm[64];
    __shared__ int    perm[64];
    __shared__ int    rotated;
    const int tid = threadIdx.x, lane = tid & 15, grp = tid >> 4, np = n + (n & 1);
    for(int t = tid; t < n * SW; t += blockDim.x) {
        const int j = t / SW, i = t - j * SW;
        T         v = jzero<T>();
        if(i < m) v = tr ? jconj(A[j + static_cast<int64_t>(n) * i]) : A[i + static_cast<int64_t>(m) * j];
        Ws[t] = v;
    }
    for(int t = tid; t < n * SV; t += blockDim.x) Vs[t] = jreal<T>(t / SV == t % SV ? 1.0 : 0.0);
    int sweep = 0;
    for(; sweep < max_sweeps; ++sweep) {
        if(tid == 0) rotated = 0;
        __syncthreads();
        for(int r = 0; r < np - 1; ++r) {
            int p = r, q = np - 1; // round_pair(np, r, grp, p, q), 0 <= r, grp < np - 1
            if(grp > 0) {
                p = r + grp, q = r - grp;
                if(p >= np - 1) p -= np - 1;
                if(q < 0) q += np - 1;
            }
            if(p > q) {
                const int tt = p;
                p            = q;
                q            = tt;
            }
            if(grp < np / 2 && q < n) {
                T *wp = Ws + p * SW + lane, *wq = Ws + q * SW + lane, *vp = Vs + p * SV + lane, *vq = Vs + q * SV + lane;
                T  x[E], y[E], vx[EV], vy[EV];
                double al = 0, be = 0, gr = 0, gi = 0;
#pragma unroll
                for(int e = 0; e < E; ++e) x[e] = wp[16 * e], y[e] = wq[16 * e];
#pragma unroll
                for(int e = 0; e < EV; ++e) vx[e] = vp[16 * e], vy[e] = vq[16 * e];
#pragma unroll
                for(int e = 0; e < E; ++e) {
                    if constexpr(cx) {
                        al += x[e].re * x[e].re + x[e].im * x[e].im;
                        be += y[e].re * y[e].re + y[e].im * y[e].im;
                        gr += x[e].re * y[e].re + x[e].im * y[e].im; // conj(x) y
                        gi += x[e].re * y[e].im - x[e].im * y[e].re;
                    } else {
                        al += x[e] * x[e];
                        be += y[e] * y[e];
                        gr += x[e] * y[e];
                    }
                }
                al = row_sum(al), be = row_sum(be), gr = row_sum(gr);
                if constexpr(cx) gi = row_sum(gi);
                const double g = coupling<T>(gr, gi, al, be, tol);
                if(g != 0.0) {
                    // The rotation of jacobi_round: with d = be - al, h = sqrt(d^2 + (2 g)^2) and u = |d| + h the tangent is
                    // sign(d) 2 g / u. d and g are scaled to about 1 first, so that no square leaves the range.
                    const double d0 = be - al, e2 = fmax(fabs(d0), g);
                    int          ex;
                    (void) frexp(e2, &ex);
                    const double d = ldexp(fabs(d0), -ex), g2 = ldexp(g, 1 - ex);
                    const double u = d + sqrt(d * d + g2 * g2), w = rsqrt(u * u + g2 * g2);
                    const double c = u * w, s = d0 >= 0 ? g2 * w : -(g2 * w);
                    const double er = cx ? gr / g : (gr > 0 ? 1.0 : -1.0), ei = cx ? -gi / g : 0.0;
                    if(lane == 0) rotated = 1;
                    auto rot = [&](T &xv, T &yv) {
                        if constexpr(cx) {
                            const double yr = yv.re * er - yv.im * ei, yi = yv.re * ei + yv.im * er; // e^{-i phi} y
                            const T      x0 = xv;
                            xv              = T{c * x0.re - s * yr, c * x0.im - s * yi};
                            yv              = T{s * x0.re + c * yr, s * x0.im + c * yi};
                        } else {
                            const double x0 = xv, y0 = yv * er;
                            xv              = c * x0 - s * y0;
                            yv              = s * x0 + c * y0;
                        }
                    };
#pragma unroll
                    for(int e = 0; e < E; ++e) {
                        rot(x[e], y[e]);
                        wp[16 * e] = x[e], wq[16 * e] = y[e];
                    }
#pragma unroll
                    for(int e = 0; e < EV; ++e) {
                        rot(vx[e], vy[e]);
                        vp[16 * e] = vx[e], vq[16 * e] = vy[e];
                    }
                }
            }
            __syncthreads();
        }
        const int any = rotated;
        __syncthreads();
        if(any == 0) break;
    }
    for(int j = grp; j < n; j += static_cast<int>(blockDim.x) / 16) {
        double a = 0;
#pragma unroll
        for(int e = 0; e < E; ++e) {
            const T v = Ws[j * SW + lane + 16 * e];
            if constexpr(cx) a += v.re * v.re + v.im * v.im;
            else a += v * v;
        }
        a = row_sum(a);
        if(lane == 0) nrm[j] = sqrt(a), perm[j] = j;
    }
    __syncthreads();
    // Descending, equal ones in their order, NaN before all numbers: a total order, so that every rank is taken once and a
    // column that is not a number stands in S.
    if(tid < n) {
        int rank = 0;
        const double mine = nrm[tid];
        for(int i = 0; i < n; ++i) {
            const double other = nrm[i];
            if(other != other) rank += mine == mine || i < tid ? 1 : 0;
            else rank += other > mine || (other == mine && i < tid) ? 1 : 0;
        }
        perm[rank] = tid;
        S[rank]    = nrm[tid];
    }
    if(tid == 0) S[n] = static_cast<double>(sweep);
    __syncthreads();
    // A = W' diag(S) V^H, W' the normalised columns; the factors of A^H the other way round.
    T *left = tr ? Vt : U, *right = tr ? U : Vt;
    for(int t = tid; t < m * n; t += blockDim.x) {
        const int    k = tr ? t % n : t / m, i = tr ? t / n : t % m;
        const double sk = nrm[perm[k]], f = sk > 0 ? 1.0 / sk : 0.0;
        const T      v = jscale(f, Ws[perm[k] * SW + i]);
        left[t]        = tr ? jconj(v) : v;
    }
    for(int t = tid; t < n * n; t += blockDim.x) {
        const int k = tr ? t / n : t % n, j = tr ? t % n : t / n;
        const T   v = Vs[perm[k] * SV + j];
        right[t]    = tr ? v : jconj(v);
    }
}
template <typename T>
size_t resident_lds(int n, int E, int EV) {
    const bool pad = !jtraits<T>::cx;
    return static_cast<size_t>(n) * (16 * (E + EV) + (pad && E % 2 == 0 ? 16 : 0) + (pad && EV % 2 == 0 ? 16 : 0)) * sizeof(T);
}
template <typename T, int E, int EV>
void launch_resident(int m, int n, int tr, const T *A, double tol, int max_sweeps, T *U, T *Vt, double *S, hipStream_t s) {
    const size_t lds = resident_lds<T>(n, E, EV);
    DMRG_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(&jacobi_resident<T, E, EV>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                       static_cast<int>(JACOBI_LDS_BYTES)));
    const int pairs = (n + 1) / 2;
    hipLaunchKernelGGL((jacobi_resident<T, E, EV>), dim3(1), dim3((16 * pairs + 63) / 64 * 64), lds, s, m, n, tr, A, tol, max_sweeps, U, Vt, S);
    DMRG_HIP_CHECK(hipGetLastError());
}

// Whole Jacobi iteration in one workgroup with W (m x n) and V (n x n) resident in LDS, for small problems
// where a kernel launch per round would dominate. A wavefront handles one pair; the wavefronts take the
// pairs of a round in turn, a barrier separates the rounds, and the sweeps stop after a sweep that applied no
// rotation (at most max_sweeps; the number of sweeps run goes to sweeps_out).
template <typename T>
__global__ __launch_bounds__(1024) void jacobi_lds(int m, int n, int np, T *W, T *V, double tol, int max_sweeps, int *sweeps_out) {
    extern __shared__ unsigned char lds_raw[];
    T            *Ws = reinterpret_cast<T *>(lds_raw);
    T            *Vs = Ws + static_cast<int64_t>(m) * n;
    __shared__ int rotated;
    const int     tid = threadIdx.x, lane = tid & 63, grp = tid >> 6, ngrp = blockDim.x / 64;
    for(int t = tid; t < m * n; t += blockDim.x) Ws[t] = W[t];
    for(int t = tid; t < n * n; t += blockDim.x) {
        const bool d = (t % n) == (t / n);
        if constexpr(jtraits<T>::cx) Vs[t] = T{d ? 1.0 : 0.0, 0.0};
        else Vs[t] = d ? 1.0 : 0.0;
    }
    int sweep = 0;
    for(; sweep < max_sweeps; ++sweep) {
        if(tid == 0) rotated = 0;
        __syncthreads();
        for(int r = 0; r < np - 1; ++r) {
            // every wavefront runs the same trip count
            for(int i0 = 0; i0 < np / 2; i0 += ngrp) {
                const int i = i0 + grp;
                int       p = 0, q = 0;
                bool      live = i < np / 2;
                if(live) {
                    round_pair(np, r, i, p, q);
                    live = p < n && q < n;
                }
                if(p > q) {
                    const int tt = p;
                    p            = q;
                    q            = tt;
                }
                T     *wp = Ws + p * m, *wq = Ws + q * m;
                double al = 0, be = 0, gr = 0, gi = 0;
                if(live) {
                    for(int k = lane; k < m; k += 64) {
                        if constexpr(jtraits<T>::cx) {
                            const T x = wp[k], y = wq[k];
                            al += x.re * x.re + x.im * x.im;
                            be += y.re * y.re + y.im * y.im;
                            gr += x.re * y.re + x.im * y.im;
                            gi += x.re * y.im - x.im * y.re;
                        } else {
                            const double x = wp[k], y = wq[k];
                            al += x * x;
                            be += y * y;
                            gr += x * y;
                        }
                    }
                }
                al = wave_sum(al);
                be = wave_sum(be);
                gr = wave_sum(gr);
                if constexpr(jtraits<T>::cx) gi = wave_sum(gi);
                const double g = coupling<T>(gr, gi, al, be, tol);
                if(!live || g == 0.0) continue;
                const double z  = (be - al) / (2.0 * g);
                const double t  = tangent(z);
                const double c  = 1.0 / sqrt(1.0 + t * t), s = c * t;
                const double er = gr / g, ei = -gi / g;
                if(lane == 0) rotated = 1;
                auto rot = [&](T *x, T *y, int len) {
                    for(int k = lane; k < len; k += 64) {
                        if constexpr(jtraits<T>::cx) {
                            const T      xv = x[k], yv = y[k];
                            const double yr = yv.re * er - yv.im * ei, yi = yv.re * ei + yv.im * er;
                            x[k]            = T{c * xv.re - s * yr, c * xv.im - s * yi};
                            y[k]            = T{s * xv.re + c * yr, s * xv.im + c * yi};
                        } else {
                            const double xv = x[k], yv = y[k] * er;
                            x[k]            = c * xv - s * yv;
                            y[k]            = s * xv + c * yv;
                        }
                    }
                };
                rot(wp, wq, m);
                rot(Vs + p * n, Vs + q * n, n);
            }
            __syncthreads();
        }
        const int any = rotated;
        __syncthreads();
        if(any == 0) break;
    }
    for(int t = tid; t < m * n; t += blockDim.x) W[t] = Ws[t];
    for(int t = tid; t < n * n; t += blockDim.x) V[t] = Vs[t];
    if(tid == 0) sweeps_out[0] = sweep;
}

template <typename T>
__global__ void identity_kernel(int n, T *V) {
    const int64_t total = static_cast<int64_t>(n) * n;
    for(int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < total; t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const bool d = (t % n) == (t / n);
        if constexpr(jtraits<T>::cx) V[t] = T{d ? 1.0 : 0.0, 0.0};
        else V[t] = d ? 1.0 : 0.0;
    }
}

// out[j + n i] = conj(in[i + m j]) (conjugate transpose of an m x n matrix).
template <typename T>
__global__ void adjoint_kernel(int m, int n, const T *in, T *out) {
    const int64_t total = static_cast<int64_t>(m) * n;
    for(int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < total; t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        const int64_t i = t % m, j = t / m;
        T             v = in[t];
        if constexpr(jtraits<T>::cx) v.im = -v.im;
        out[j + static_cast<int64_t>(n) * i] = v;
    }
}

__global__ void column_norms_kernel(int m, int n, const double *W, int cx, double *out) {
    // out[j] = |W[:, j]| (W viewed as doubles; complex columns are 2m doubles long)
    const int j = blockIdx.x;
    if(j >= n) return;
    const int64_t len = static_cast<int64_t>(m) * (cx ? 2 : 1);
    double        acc = 0;
    for(int64_t i = threadIdx.x; i < len; i += 64) {
        const double v = W[j * len + i];
        acc += v * v;
    }
    acc = wave_sum(acc);
    if(threadIdx.x == 0) out[j] = sqrt(acc);
}

// Assemble the outputs in descending order of S: Uo[:, k] = W[:, perm[k]] / S[k] (m x n),
// Vo[k, :] = conj(V[:, perm[k]])^T (n x n, leading dimension n): A = Uo diag(S) Vo.
template <typename T>
__global__ void assemble_kernel(int m, int n, const int *perm, const double *S, const T *W, const T *V, T *Uo, T *Vo) {
    const int64_t tu = static_cast<int64_t>(m) * n, tv = static_cast<int64_t>(n) * n;
    for(int64_t t = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x; t < tu + tv; t += static_cast<int64_t>(gridDim.x) * blockDim.x) {
        if(t < tu) {
            const int64_t i = t % m, k = t / m;
            const double  sk = S[k];
            const double  f  = sk > 0 ? 1.0 / sk : 0.0;
            T             v  = W[i + static_cast<int64_t>(m) * perm[k]];
            if constexpr(jtraits<T>::cx) v = T{v.re * f, v.im * f};
            else v *= f;
            Uo[t] = v;
        } else {
            const int64_t q = t - tu, k = q % n, j = q / n;
            T             v = V[j + static_cast<int64_t>(n) * perm[k]];
            if constexpr(jtraits<T>::cx) v.im = -v.im;
            Vo[q] = v;
        }
    }
}

constexpr int    JACOBI_LDS_MAX_N = 32;
// Block path from this many columns on (measured on gfx950, complex n x n, ms per SVD, per-pair rounds / block
// rounds: 64: 2.86 / 2.4, 128: 7.4 / 5.8, 256: 19.5 / 14.4, 512: 61 / 35, 2048: 1325 / 289); B2 columns (two
// blocks) per inner problem. From 33 columns there are at least 3 blocks, so every round has work.
constexpr int JACOBI_BLOCK_MIN_N = 33;
constexpr int JACOBI_BLOCK_B2    = 32;
// Inner Jacobi sweeps per block pair and round: one sweep leaves the outer sweep count unchanged (the outer
// iteration finishes what an inexact inner solve leaves) at a fraction of the cost of converging each one.
constexpr int JACOBI_BLOCK_INNER = 1;

unsigned grid_of(int64_t total) { return static_cast<unsigned>(std::max<int64_t>(1, std::min<int64_t>((total + 255) / 256, 8192))); }

} // namespace

template <typename T>
void DeviceSvd::jacobi(int m, int n, const T *A, std::vector<double> &S) {
    // Work on W = A (m >= n) or W = A^H (m < n); W has mm >= nn.
    const bool tr = m < n;
    const int  mm = tr ? n : m, nn = tr ? m : n;
    k_            = nn;
    const size_t es = sizeof(T);
    const double tol = std::sqrt(static_cast<double>(mm)) * 2.3e-16; // gesvj's threshold, sqrt(m) eps
    const int    E = mm <= 32 ? 2 : mm <= 64 ? 4 : mm <= 80 ? 5 : 8, EV = nn <= 32 ? 2 : 4;
    // Up to the size that one workgroup's registers, rows of lanes and LDS hold, that is faster than any number of launches
    // (complex 128x64 does not fit: 6.4 ms in rounds of block pairs).
    if(mm <= 128 && nn <= 64 && resident_lds<T>(nn, E, EV) <= JACOBI_LDS_BYTES) {
        u.reserve(static_cast<size_t>(mm) * nn * es);
        vt.reserve(static_cast<size_t>(mm) * nn * es);
        res.reserve(static_cast<size_t>(nn + 1) * sizeof(double));
        auto run = [&](auto e, auto ev) {
            launch_resident<T, decltype(e)::value, decltype(ev)::value>(mm, nn, tr ? 1 : 0, A, tol, 60, u.as<T>(), vt.as<T>(), res.as<double>(), s);
        };
        using std::integral_constant;
        if(EV == 2 && E == 2) run(integral_constant<int, 2>{}, integral_constant<int, 2>{});
        else if(EV == 2 && E == 4) run(integral_constant<int, 4>{}, integral_constant<int, 2>{});
        else if(EV == 2 && E == 5) run(integral_constant<int, 5>{}, integral_constant<int, 2>{});
        else if(EV == 2) run(integral_constant<int, 8>{}, integral_constant<int, 2>{});
        else if(E == 5) run(integral_constant<int, 5>{}, integral_constant<int, 4>{});
        else if(E == 4) run(integral_constant<int, 4>{}, integral_constant<int, 4>{});
        else run(integral_constant<int, 8>{}, integral_constant<int, 4>{});
        S.resize(nn + 1);
        DMRG_HIP_CHECK(hipMemcpyAsync(S.data(), res.p, (nn + 1) * sizeof(double), hipMemcpyDeviceToHost, s));
        DMRG_HIP_CHECK(hipStreamSynchronize(s));
        DMRG_REQUIRE(S[nn] < 60, DMRG_ERR_NOT_CONVERGED, "Jacobi SVD: no convergence in 60 sweeps");
        S.resize(nn);
        return;
    }
    const size_t lds_need = (static_cast<size_t>(mm) * nn + static_cast<size_t>(nn) * nn) * es;
    const bool   resident = nn > 1 && nn <= JACOBI_LDS_MAX_N && lds_need <= JACOBI_LDS_BYTES;
    const bool   blocked  = !resident && nn >= JACOBI_BLOCK_MIN_N;
    const int    npad     = blocked ? (nn + 15) / 16 * 16 : nn; // whole 16-column blocks (zero columns)
    a.reserve(static_cast<size_t>(mm) * npad * es);  // W (m x npad)
    e.reserve(static_cast<size_t>(nn) * npad * es);  // V (n x npad)
    sv.reserve(static_cast<size_t>(nn) * sizeof(double));
    info.reserve(sizeof(unsigned) * 2 + static_cast<size_t>(nn) * sizeof(int));
    res.reserve(static_cast<size_t>(nn) * sizeof(double));
    T *W = a.as<T>(), *V = e.as<T>();
    if(tr) hipLaunchKernelGGL(adjoint_kernel<T>, dim3(grid_of(static_cast<int64_t>(m) * n)), dim3(256), 0, s, m, n, A, W);
    else DMRG_HIP_CHECK(hipMemcpyAsync(W, A, static_cast<size_t>(m) * n * es, hipMemcpyDeviceToDevice, s));
    hipLaunchKernelGGL(identity_kernel<T>, dim3(grid_of(static_cast<int64_t>(nn) * nn)), dim3(256), 0, s, nn, V);
    DMRG_HIP_CHECK(hipGetLastError());
    if(npad > nn) {
        DMRG_HIP_CHECK(hipMemsetAsync(W + static_cast<int64_t>(mm) * nn, 0, static_cast<size_t>(mm) * (npad - nn) * es, s));
        DMRG_HIP_CHECK(hipMemsetAsync(V + static_cast<int64_t>(nn) * nn, 0, static_cast<size_t>(nn) * (npad - nn) * es, s));
    }
    unsigned    *flag = info.as<unsigned>();
    const int    np   = nn + (nn & 1);
    unsigned     hflag = 0;
    int          sweep = 0;
    const size_t lds   = lds_need;
    // A round costs about the same few microseconds inside one workgroup as one launch per round over the
    // whole chip (measured on gfx950), so the resident path pays off only while one workgroup takes a whole
    // round with one wavefront per pair and the launches it saves dominate.
    if(resident) {
        int *dsweeps = reinterpret_cast<int *>(flag + 1);
        // n <= 32: at most 16 pairs a round, one wavefront each
        DMRG_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(&jacobi_lds<T>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                           static_cast<int>(JACOBI_LDS_BYTES)));
        hipLaunchKernelGGL((jacobi_lds<T>), dim3(1), dim3(1024), lds, s, mm, nn, np, W, V, tol, 60, dsweeps);
        DMRG_HIP_CHECK(hipGetLastError());
        int hs = 0;
        DMRG_HIP_CHECK(hipMemcpyAsync(&hs, dsweeps, sizeof(int), hipMemcpyDeviceToHost, s));
        DMRG_HIP_CHECK(hipStreamSynchronize(s));
        DMRG_REQUIRE(hs < 60, DMRG_ERR_NOT_CONVERGED, "Jacobi SVD: no convergence in 60 sweeps");
        sweep = 60; // skip the per-round path below
    }
    // Block path: column blocks of JACOBI_BLOCK_B2 / 2, three launches per round of block pairs.
    if(blocked) {
        constexpr int    B2     = JACOBI_BLOCK_B2;
        static_assert(B2 == 32, "the matrix-core Gram and update kernels take pairs of 16-column blocks");
        const dmrg_dtype dt     = jtraits<T>::cx ? DMRG_CX64 : DMRG_FP64;
        const int        nb     = npad / (B2 / 2);
        const int     nbp    = nb + (nb & 1);
        const int     npairs = nbp / 2;
        const int     ks     = static_cast<int>(std::clamp<int64_t>((512 + npairs - 1) / npairs, 1, std::max(1, mm / BJ_ROWS)));
        const int     rows_per = ((mm + ks - 1) / ks + BJ_ROWS - 1) / BJ_ROWS * BJ_ROWS;
        const int     ksn      = (mm + rows_per - 1) / rows_per; // chunks actually holding rows
        bj_part.reserve(static_cast<size_t>(npairs) * ksn * B2 * B2 * es);
        bj_q.reserve(static_cast<size_t>(npairs) * B2 * B2 * es);
        bj_rot.reserve(static_cast<size_t>(npairs) * sizeof(int));
        T   *part = bj_part.as<T>(), *qb = bj_q.as<T>();
        int *rot  = bj_rot.as<int>();
        for(; sweep < 60; ++sweep) {
            DMRG_HIP_CHECK(hipMemsetAsync(flag, 0, sizeof(unsigned), s));
            for(int r = 0; r < nbp - 1; ++r) {
                bj_gram_mfma(dt, mm, npad, nbp, r, W, ksn, rows_per, part, s);
                hipLaunchKernelGGL((bj_eig<T, B2>), dim3(npairs), dim3(BJ_THREADS), 0, s, npad, nbp, r, ksn, part, qb, rot, tol, JACOBI_BLOCK_INNER, flag);
                bj_update_mfma(dt, mm, nn, npad, nbp, r, W, V, qb, rot, s);
            }
            DMRG_HIP_CHECK(hipGetLastError());
            DMRG_HIP_CHECK(hipMemcpyAsync(&hflag, flag, sizeof(unsigned), hipMemcpyDeviceToHost, s));
            DMRG_HIP_CHECK(hipStreamSynchronize(s));
            if(hflag == 0) break;
        }
        sweep = 60; // skip the per-pair rounds below
    }
    for(; sweep < 60 && nn > 1; ++sweep) {
        DMRG_HIP_CHECK(hipMemsetAsync(flag, 0, sizeof(unsigned), s));
        for(int r = 0; r < np - 1; ++r) {
            if(mm > 256) hipLaunchKernelGGL((jacobi_round<T, 256>), dim3(np / 2), dim3(256), 0, s, mm, nn, np, r, W, V, tol, flag);
            else if(mm > 128) hipLaunchKernelGGL((jacobi_round<T, 128>), dim3(np / 2), dim3(128), 0, s, mm, nn, np, r, W, V, tol, flag);
            else hipLaunchKernelGGL((jacobi_round<T, 64>), dim3(np / 2), dim3(64), 0, s, mm, nn, np, r, W, V, tol, flag);
        }
        DMRG_HIP_CHECK(hipGetLastError());
        DMRG_HIP_CHECK(hipMemcpyAsync(&hflag, flag, sizeof(unsigned), hipMemcpyDeviceToHost, s));
        DMRG_HIP_CHECK(hipStreamSynchronize(s));
        if(hflag == 0) break;
    }
    DMRG_REQUIRE(nn <= 1 || hflag == 0 || resident, DMRG_ERR_NOT_CONVERGED, "Jacobi SVD: no convergence in 60 sweeps");
    hipLaunchKernelGGL(column_norms_kernel, dim3(nn), dim3(64), 0, s, mm, nn, reinterpret_cast<const double *>(W),
                       jtraits<T>::cx ? 1 : 0, res.as<double>());
    std::vector<double> norms(nn);
    DMRG_HIP_CHECK(hipMemcpyAsync(norms.data(), res.p, nn * sizeof(double), hipMemcpyDeviceToHost, s));
    DMRG_HIP_CHECK(hipStreamSynchronize(s));
    std::vector<int> perm(nn);
    for(int i = 0; i < nn; ++i) perm[i] = i;
    std::stable_sort(perm.begin(), perm.end(), [&](int x, int y) { return norms[x] > norms[y]; });
    S.resize(nn);
    for(int i = 0; i < nn; ++i) S[i] = norms[perm[i]];
    int *dperm = reinterpret_cast<int *>(flag + 2);
    DMRG_HIP_CHECK(hipMemcpyAsync(dperm, perm.data(), nn * sizeof(int), hipMemcpyHostToDevice, s));
    DMRG_HIP_CHECK(hipMemcpyAsync(sv.p, S.data(), nn * sizeof(double), hipMemcpyHostToDevice, s));
    // W = Uw S Vw^H. Without transpose: U = Uw (m x k), Vt = Vw^H (k x n). With transpose (A = W^H):
    // U = Vw (m x k) and Vt = Uw^H (k x n).
    u.reserve(static_cast<size_t>(mm) * nn * es);
    vt.reserve(static_cast<size_t>(nn) * nn * es);
    hipLaunchKernelGGL(assemble_kernel<T>, dim3(grid_of(static_cast<int64_t>(mm) * nn + static_cast<int64_t>(nn) * nn)), dim3(256), 0, s, mm,
                       nn, dperm, sv.as<double>(), W, V, u.as<T>(), vt.as<T>());
    DMRG_HIP_CHECK(hipGetLastError());
    if(tr) {
        // U_A (m x k) = Vw[:, perm] = adjoint of vt (k x m); Vt_A (k x n) = Uw^H = adjoint of u (n x k).
        DevBuf t1, t2;
        t1.reserve(static_cast<size_t>(m) * k_ * es);
        t2.reserve(static_cast<size_t>(k_) * n * es);
        hipLaunchKernelGGL(adjoint_kernel<T>, dim3(grid_of(static_cast<int64_t>(k_) * m)), dim3(256), 0, s, k_, m, vt.as<T>(), t1.as<T>());
        hipLaunchKernelGGL(adjoint_kernel<T>, dim3(grid_of(static_cast<int64_t>(n) * k_)), dim3(256), 0, s, n, k_, u.as<T>(), t2.as<T>());
        DMRG_HIP_CHECK(hipGetLastError());
        DMRG_HIP_CHECK(hipStreamSynchronize(s));
        std::swap(u, t1);
        std::swap(vt, t2);
    }
    DMRG_HIP_CHECK(hipStreamSynchronize(s));
}
template void DeviceSvd::jacobi<double>(int, int, const double *, std::vector<double> &);
template void DeviceSvd::jacobi<cpx<double>>(int, int, const cpx<double> *, std::vector<double> &);

} // namespace dmrg
