// Batched Hermitian eigensolver of libwbmi: cyclic two-sided Jacobi.
//
// One workgroup per k-point; the matrix A and the accumulated rotations V stay
// on the chip for the whole solve (LDS; V in registers above nw = 64).  Each
// Jacobi step rotates nw/2 disjoint (p, q) pairs of the round-robin (circle)
// ordering at once.  The complex rotation is
// G = diag(1, e^{-i phi}) R diag(1, e^{i phi}) with a_pq = |a_pq| e^{i phi} and
// R the real symmetric Jacobi rotation (Golub & Van Loan, Matrix Computations,
// sec. 8.5.2).  Sweeps stop when a whole sweep applies no rotation.  Eigenvalues
// are returned ascending with eigenvectors as columns, as np.linalg.eigh does
// (data_K/data_K.py:213).  k_eigh_jacobi (any type, run-time size) serves
// refine = 0; refined solves start from the FP32 kernels below it.
#include <cfloat>

#include <type_traits>

#include "mfma_c64.h"
#include "round_flag.h"
#include "wbmi_common.h"

// update items per lane per batch (loads of a batch are issued together)
#define JB 8

template <typename T>
struct Eps;
template <>
struct Eps<double> {
    static constexpr double v = 2.220446049250313e-16;
};
template <>
struct Eps<float> {
    static constexpr float v = 1.1920929e-07f;
};

// pair i of round r (0 <= i < n/2, 0 <= r < n-1) in the circle ordering of n
// (even) players: i + r - 1 < 2(n-1) and n - 2 - i + r < 2(n-1), so one
// conditional subtraction replaces the modulo.
__device__ inline void rr_pair(int n, int r, int i, int& p, int& q) {
    const int m = n - 1;
    int a = i + r - 1;
    a = a >= m ? a - m : a;
    p = (i == 0) ? 0 : a + 1;
    int b = n - 2 - i + r;
    b = b >= m ? b - m : b;
    q = b + 1;
}

// Items (pair, index) of a round, pair-major, dealt to the 64 lanes:
// lane t starts at item t and steps by 64 items.
struct ItemWalk {
    int pr, i, dp, di;
    __device__ ItemWalk(int n, int tid) : pr(tid / n), i(tid % n), dp(64 / n), di(64 % n) {}
    __device__ inline void next(int n) {
        pr += dp;
        i += di;
        if (i >= n) {
            i -= n;
            ++pr;
        }
    }
};

// T: arithmetic and LDS type; Tin: type of H; TO: type of the stored eigenvectors
template <typename T, typename Tin, typename TO = T>
__global__ void __launch_bounds__(64) k_eigh_jacobi(int nw, const cplx<Tin>* __restrict__ H, int64_t Hstride,
                                                    double* __restrict__ Eout, cplx<TO>* __restrict__ Uout,
                                                    int max_sweeps) {
    extern __shared__ char smem[];
    const int n = nw + (nw & 1);  // padded to even; the dummy index is decoupled
    const int ld = n + 1;         // LDS row stride (one element of padding against bank conflicts)
    const int np = n / 2;
    cplx<T>* A = (cplx<T>*)smem;
    cplx<T>* V = A + n * ld;
    T* prm = (T*)(V + n * ld);  // per pair: c, s*cos(phi), s*sin(phi)
    int* flag = (int*)(prm + 3 * np);
    const int tid = threadIdx.x;
    const int64_t k = blockIdx.x;
    const cplx<Tin>* Hk = H + k * Hstride;

    for (int i = tid; i < n; i += 64)
        for (int j = 0; j < n; ++j) {
            cplx<T> a = mk((T)0, (T)0);
            if (i < nw && j < nw) {
                cplx<Tin> x = Hk[i * nw + j], y = Hk[j * nw + i];
                a = mk((T)(0.5 * (x.re + y.re)), (T)(0.5 * (x.im - y.im)));
            }
            A[i * ld + j] = a;
            V[i * ld + j] = mk((T)(i == j ? 1 : 0), (T)0);
        }
    __syncthreads();

    const T eps = Eps<T>::v;
    for (int sweep = 0; sweep < max_sweeps; ++sweep) {
        if (tid == 0) *flag = 0;
        __syncthreads();
        for (int r = 0; r < n - 1; ++r) {
            bool rot = false;
            if (tid < np) {
                int p, q;
                rr_pair(n, r, tid, p, q);
                cplx<T> apq = A[p * ld + q];
                T g = sqrt(apq.re * apq.re + apq.im * apq.im);
                T app = A[p * ld + p].re, aqq = A[q * ld + q].re;
                T c = 1, sc = 0, ss = 0;
                T scale = fabs(app) > fabs(aqq) ? fabs(app) : fabs(aqq);
                if (g > (T)0.5 * eps * scale && g > (T)(sizeof(T) == 8 ? 1e-300 : 1e-36)) {
                    T tau = (aqq - app) / (2 * g);
                    T t = (tau >= 0 ? (T)1 : (T)-1) / (fabs(tau) + sqrt((T)1 + tau * tau));
                    c = (T)1 / sqrt((T)1 + t * t);
                    T s = t * c;
                    sc = s * apq.re / g;
                    ss = s * apq.im / g;
                    rot = true;
                    *flag = 1;
                }
                prm[3 * tid] = c;
                prm[3 * tid + 1] = sc;
                prm[3 * tid + 2] = ss;
            }
            // the workgroup is one wavefront: __any is uniform over it
            if (!__any(rot)) continue;
            __syncthreads();
            // columns of A and V:  col_p <- c col_p - s e^{-i phi} col_q ; col_q <- s e^{i phi} col_p + c col_q
            // Items of a phase touch disjoint elements: each lane loads JB items, then rotates and stores them.
            for (ItemWalk w(n, tid); w.pr < np;) {
                int ii[JB], pp[JB], qq[JB];
                bool ok[JB];
                T cc[JB];
                cplx<T> se[JB], ap[JB], aq[JB], vp[JB], vq[JB];
#pragma unroll
                for (int u = 0; u < JB; ++u) {
                    ok[u] = w.pr < np;
                    const int pr = ok[u] ? w.pr : 0;
                    rr_pair(n, r, pr, pp[u], qq[u]);
                    ii[u] = w.i;
                    w.next(n);
                    cc[u] = prm[3 * pr];
                    se[u] = mk(prm[3 * pr + 1], prm[3 * pr + 2]);
                    ap[u] = A[ii[u] * ld + pp[u]];
                    aq[u] = A[ii[u] * ld + qq[u]];
                    vp[u] = V[ii[u] * ld + pp[u]];
                    vq[u] = V[ii[u] * ld + qq[u]];
                }
#pragma unroll
                for (int u = 0; u < JB; ++u) {
                    if (!ok[u]) continue;
                    A[ii[u] * ld + pp[u]] = cc[u] * ap[u] - mulc(aq[u], se[u]);
                    A[ii[u] * ld + qq[u]] = se[u] * ap[u] + cc[u] * aq[u];
                    V[ii[u] * ld + pp[u]] = cc[u] * vp[u] - mulc(vq[u], se[u]);
                    V[ii[u] * ld + qq[u]] = se[u] * vp[u] + cc[u] * vq[u];
                }
            }
            __syncthreads();
            // rows of A:  row_p <- c row_p - s e^{i phi} row_q ; row_q <- s e^{-i phi} row_p + c row_q
            for (ItemWalk w(n, tid); w.pr < np;) {
                int jj[JB], pp[JB], qq[JB];
                bool ok[JB];
                T cc[JB];
                cplx<T> se[JB], ap[JB], aq[JB];
#pragma unroll
                for (int u = 0; u < JB; ++u) {
                    ok[u] = w.pr < np;
                    const int pr = ok[u] ? w.pr : 0;
                    rr_pair(n, r, pr, pp[u], qq[u]);
                    jj[u] = w.i;
                    w.next(n);
                    cc[u] = prm[3 * pr];
                    se[u] = mk(prm[3 * pr + 1], prm[3 * pr + 2]);
                    ap[u] = A[pp[u] * ld + jj[u]];
                    aq[u] = A[qq[u] * ld + jj[u]];
                }
#pragma unroll
                for (int u = 0; u < JB; ++u) {
                    if (!ok[u]) continue;
                    A[pp[u] * ld + jj[u]] = cc[u] * ap[u] - se[u] * aq[u];
                    A[qq[u] * ld + jj[u]] = mulc(ap[u], se[u]) + cc[u] * aq[u];
                }
            }
            __syncthreads();
        }
        if (*flag == 0) break;
        __syncthreads();
    }
    // ascending order: rank of each eigenvalue (ties broken by index)
    for (int i = tid; i < nw; i += 64) {
        T ei = A[i * ld + i].re;
        int rank = 0;
        for (int j = 0; j < nw; ++j) {
            T ej = A[j * ld + j].re;
            rank += (ej < ei) || (ej == ei && j < i);
        }
        Eout[k * nw + rank] = (double)ei;
        for (int m = 0; m < nw; ++m) {
            const cplx<T> v = V[m * ld + i];
            Uout[(k * nw + m) * nw + rank] = mk((TO)v.re, (TO)v.im);
        }
    }
}

// Rotation of one FP32 pivot a_pq with diagonal app, aqq: c, s cos(phi), s sin(phi); false (and
// the identity) where |a_pq| is below rounding.  FAST: hardware reciprocal and reciprocal square
// root (1 ulp; c^2 + s^2 = 1 to rounding as with correctly rounded division, in far fewer
// instructions).
template <bool FAST>
__device__ inline bool jacobi_rotation(cplx<float> apq, float app, float aqq, float& c, float& sc, float& ss) {
    typedef float T;
    const T g = sqrt(fmaf(apq.re, apq.re, apq.im * apq.im));
    c = 1;
    sc = 0;
    ss = 0;
    const T scale = fabs(app) > fabs(aqq) ? fabs(app) : fabs(aqq);
    if (!(g > (T)0.5 * Eps<T>::v * scale && g > (T)1e-36)) return false;
    if constexpr (FAST) {
        const T rg = __builtin_amdgcn_rcpf(g);
        const T tau = (aqq - app) * (T)0.5 * rg;
        const T ta = __builtin_amdgcn_rcpf(fabs(tau) + sqrt((T)1 + tau * tau));
        const T t = tau >= 0 ? ta : -ta;
        c = __builtin_amdgcn_rsqf((T)1 + t * t);
        const T s = t * c;
        sc = s * apq.re * rg;
        ss = s * apq.im * rg;
    } else {
        const T tau = (aqq - app) / (2 * g);
        const T t = (tau >= 0 ? (T)1 : (T)-1) / (fabs(tau) + sqrt((T)1 + tau * tau));
        c = (T)1 / sqrt((T)1 + t * t);
        const T s = t * c;
        sc = s * apq.re / g;
        ss = s * apq.im / g;
    }
    return true;
}

// The two updates, each product pair as a multiplication and an explicit fma: complex64 vectors
// are stored in the last bit these give, so it is not left to the compiler's contraction.
// Columns p, q of one row: x_p <- c x_p - s e^{-i phi} x_q, x_q <- s e^{i phi} x_p + c x_q.
// IMRE: the imaginary part of s e^{i phi} x_p starts from the product with x_p's imaginary part.
template <bool IMRE>
__device__ inline void rotate_cols(cplx<float>& xp, cplx<float>& xq, float c, float sc, float ss) {
    const cplx<float> p = xp, q = xq;
    xp.re = fmaf(c, p.re, -fmaf(q.re, sc, q.im * ss));
    xp.im = fmaf(c, p.im, -fmaf(q.im, sc, -(q.re * ss)));
    xq.re = fmaf(c, q.re, fmaf(p.re, sc, -(p.im * ss)));
    xq.im = fmaf(c, q.im, IMRE ? fmaf(ss, p.re, sc * p.im) : fmaf(p.im, sc, p.re * ss));
}
// Rows p, q of one column: x_p <- c x_p - s e^{i phi} x_q, x_q <- s e^{-i phi} x_p + c x_q
__device__ inline void rotate_rows(cplx<float>& xp, cplx<float>& xq, float c, float sc, float ss) {
    const cplx<float> p = xp, q = xq;
    xp.re = fmaf(c, p.re, -fmaf(sc, q.re, -(ss * q.im)));
    xp.im = fmaf(c, p.im, -fmaf(ss, q.re, sc * q.im));
    xq.re = fmaf(c, q.re, fmaf(p.re, sc, p.im * ss));
    xq.im = fmaf(c, q.im, fmaf(p.im, sc, -(p.re * ss)));
}

// ---------------------------------------------------------------------------
// FP32 Jacobi for padded sizes n = N <= 64: the rotations of k_eigh_jacobi, in the same order,
// with the size known at compile time and A and V in LDS.  A round's N/2 pairs cut A into
// (N/2)^2 blocks of rows {p_i, q_i} x columns {p_j, q_j}: a thread loads a block, rotates its
// columns by pair j and its rows by pair i and stores it, so that every element of A is read
// and written once a round (a column phase and a row phase, with a barrier between them, moved
// them twice); V's column pairs are dealt out the same way in the same phase.  Every element
// still sees the column rotation first, so the bits are those of the two phases.
// Bound: VALU issue (about 390 instructions a round and wave at N = 32, 64 LDS operations) and,
// for few k-points, the latency of a round.
// One wave per k for N <= 32, four above (LDS holds four such workgroups a CU at N = 48); few k-points: below.
// The parameters of N = 16, 32 and 64 use the hardware reciprocals (FAST), those of the sizes between correctly rounded
// division: either way the rotations are unitary to FP32 rounding and the refinement removes the rest, but where close
// bands keep a vector from converging further, its complex64 bits depend on it, so each size keeps its formula.
// Measured against k_eigh_jacobi (sizes at run time, two phases): 9.1 -> 2.6 ms for 3898 k-points
// at nw = 48, 1.05 -> 0.62 ms for 6112 at nw = 24, 165 -> 67 us for 1728 at nw = 12.
// ---------------------------------------------------------------------------
// Waves per k: with fewer k-points than fill the GPU, four (N > 16) and sixteen (N > 32): a round's items
// over more SIMDs, the same operations per element.  Diagonalisation and refinement of 50 k-points: nw = 18
// 136 -> 121 us, 32 292 -> 201, 48 574 -> 451, 64 885 -> 697; where the waves no longer fit side by side
// it costs (nw = 32, 1024 k-points 429 -> 453; nw = 48, 640 915 -> 1008).
template <int N>
__host__ __device__ constexpr int jacobi_b_waves(bool few) {
    return N <= 16 ? 1 : N <= 32 ? (few ? 4 : 1) : (few ? 16 : 4);
}
template <int N>
__host__ __device__ constexpr size_t jacobi_b_lds() {
    return sizeof(float4) * (N / 2) + 2 * sizeof(cplx<float>) * N * (N + 1) + sizeof(int) * (N + 2);
}

// U0 (optional, N = 16 and 32): approximate eigenvectors (columns), e.g. those of
// the same k-point index in the neighbouring K-block.  The sweeps then run on
// A = U0^+ H U0 (both products on the FP64 matrix cores, stored in FP32) with
// the rotations accumulated onto V = U0: a nearly diagonal start needs about
// three active sweeps instead of six or seven.  Any unitary U0 gives the same
// eigen-decomposition; a poor one only costs sweeps.
template <int N, int NWAVE, typename Tin, typename TO>
__global__ void __launch_bounds__(64 * NWAVE) k_eigh_jacobi_b(int nw, const cplx<Tin>* __restrict__ H, int64_t Hstride,
                                                             double* __restrict__ Eout, cplx<TO>* Uout, int max_sweeps,
                                                             const cplx<TO>* U0) {
    typedef float T;
    constexpr int NTH = 64 * NWAVE;
    constexpr int n = N, ld = N + 1, np = N / 2;
    constexpr int NB = np * np, NV = np * N;                          // A blocks and V items of a round
    constexpr int IB = (NB + NTH - 1) / NTH, IV = (NV + NTH - 1) / NTH;  // per thread
    constexpr bool FAST = N == 16 || N == 32 || N == 64;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    float4* prm = (float4*)smem;  // per pair: c, s cos(phi), s sin(phi), p | q << 16
    cplx<T>* A = (cplx<T>*)(prm + np);
    cplx<T>* V = A + n * ld;
    int* rank = (int*)(V + n * ld);
    int* flags = rank + n;  // round flag (workgroups of several waves): RoundFlag
    const int tid = threadIdx.x;
    const int64_t k = blockIdx.x;
    const cplx<Tin>* Hk = H + k * Hstride;

    bool warm = false;
    if constexpr (N == 16 || N == 32) warm = U0 != nullptr;
    if (!warm) {
        for (int t = tid; t < n * n; t += NTH) {
            const int i = t / n, j = t % n;
            cplx<T> a = mk((T)0, (T)0);
            if (i < nw && j < nw) {
                cplx<Tin> x = Hk[i * nw + j], y = Hk[j * nw + i];
                a = mk((T)(0.5 * (x.re + y.re)), (T)(0.5 * (x.im - y.im)));
            }
            A[i * ld + j] = a;
            V[i * ld + j] = mk((T)(i == j ? 1 : 0), (T)0);
        }
        __syncthreads();
    } else if constexpr (N == 16 || N == 32) {
        // V = U0 (identity on the padding index of odd nw)
        const cplx<TO>* U0k = U0 + k * nw * nw;
        for (int t = tid; t < n * n; t += NTH) {
            const int i = t / n, j = t % n;
            cplx<T> v = mk((T)(i == j ? 1 : 0), (T)0);
            if (i < nw && j < nw) {
                const cplx<TO> u = U0k[i * nw + j];
                v = mk((T)u.re, (T)u.im);
            }
            V[i * ld + j] = v;
        }
        __syncthreads();
        // T = H U0 into A, then A = U0^+ T (one 32 x 32 block per product, the first wave's)
        MfmaBlock C;
        auto store = [&] {
#pragma unroll
            for (int bi = 0; bi < 2; ++bi)
#pragma unroll
                for (int bj = 0; bj < 2; ++bj)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int r = mfma_row(bi, v), c = mfma_col(bj);
                        if (r < n && c < n) A[r * ld + c] = mk((T)C.re[bi][bj][v], (T)C.im[bi][bj][v]);
                    }
        };
        if (tid < 64) {
            C.zero();
            mfma_block(
                C, n, n, n, 0, 0,
                [&](int r, int m) {
                    if (r >= nw || m >= nw) return mk(0.0, 0.0);
                    const cplx<Tin> x = Hk[r * nw + m], y = Hk[m * nw + r];
                    return mk(0.5 * ((double)x.re + (double)y.re), 0.5 * ((double)x.im - (double)y.im));
                },
                [&](int m, int c) { return mk((double)V[m * ld + c].re, (double)V[m * ld + c].im); });
            store();
        }
        __syncthreads();
        if (tid < 64) {
            C.zero();
            mfma_block(
                C, n, n, n, 0, 0, [&](int r, int m) { return mk((double)V[m * ld + r].re, -(double)V[m * ld + r].im); },
                [&](int m, int c) { return mk((double)A[m * ld + c].re, (double)A[m * ld + c].im); });
            __builtin_amdgcn_wave_barrier();  // every read of T is done (one wave, in order)
            store();
        }
        __syncthreads();
    }

    // the thread's blocks: row pair i, column pair j; its V items: row, pair
    int bij[IB], vij[IV];
#pragma unroll
    for (int u = 0; u < IB; ++u) {
        const int b = tid + NTH * u;
        bij[u] = (b / np) | (b % np) << 16;
    }
#pragma unroll
    for (int u = 0; u < IV; ++u) {
        const int b = tid + NTH * u;
        vij[u] = (b / n) | (b % n) * ld << 16;  // pair, offset of the row
    }
    RoundFlag flag;
    for (int sweep = 0; sweep < max_sweeps; ++sweep) {
        bool swept = false;
        for (int r = 0; r < n - 1; ++r) {
            bool rot = false;
            if (tid < np) {
                int p, q;
                rr_pair(n, r, tid, p, q);
                T c, sc, ss;
                rot = jacobi_rotation<FAST>(A[p * ld + q], A[p * ld + p].re, A[q * ld + q].re, c, sc, ss);
                prm[tid] = make_float4(c, sc, ss, __int_as_float(p | (q << 16)));
            }
            bool any;
            if constexpr (NTH == 64) {
                any = __any(rot);  // the workgroup is one wavefront: uniform over it
                __syncthreads();
            } else {
                // the pairs belong to wave 0
                if (tid < 64) {
                    const bool w = __any(rot);
                    if (tid == 0) flag.put(flags, w);
                }
                __syncthreads();
                any = flag.take(flags) != 0;
            }
            if (!any) continue;
            swept = true;
            constexpr int B = 4;  // items whose loads are issued together
#pragma unroll
            for (int u0 = 0; u0 < IB; u0 += B) {
                int o[B][4];
                cplx<T> x[B][4];
                float4 pi[B], pj[B];
#pragma unroll
                for (int v = 0; v < B; ++v) {
                    const int u = u0 + v;
                    if (u >= IB || (NTH * (u + 1) > NB && tid + NTH * u >= NB)) continue;
                    pi[v] = prm[bij[u] & 0xffff];
                    pj[v] = prm[bij[u] >> 16];
                    const int ri = __float_as_int(pi[v].w), cj = __float_as_int(pj[v].w);
                    const int rp = (ri & 0xffff) * ld, rq = (ri >> 16) * ld, cp = cj & 0xffff, cq = cj >> 16;
                    o[v][0] = rp + cp;
                    o[v][1] = rp + cq;
                    o[v][2] = rq + cp;
                    o[v][3] = rq + cq;
#pragma unroll
                    for (int e = 0; e < 4; ++e) x[v][e] = A[o[v][e]];
                }
#pragma unroll
                for (int v = 0; v < B; ++v) {
                    const int u = u0 + v;
                    if (u >= IB || (NTH * (u + 1) > NB && tid + NTH * u >= NB)) continue;
                    rotate_cols<FAST>(x[v][0], x[v][1], pj[v].x, pj[v].y, pj[v].z);
                    rotate_cols<FAST>(x[v][2], x[v][3], pj[v].x, pj[v].y, pj[v].z);
                    rotate_rows(x[v][0], x[v][2], pi[v].x, pi[v].y, pi[v].z);
                    rotate_rows(x[v][1], x[v][3], pi[v].x, pi[v].y, pi[v].z);
#pragma unroll
                    for (int e = 0; e < 4; ++e) A[o[v][e]] = x[v][e];
                }
            }
#pragma unroll
            for (int u0 = 0; u0 < IV; u0 += 2 * B) {
                int op[2 * B], oq[2 * B];
                cplx<T> xp[2 * B], xq[2 * B];
                float4 P[2 * B];
#pragma unroll
                for (int v = 0; v < 2 * B; ++v) {
                    const int u = u0 + v;
                    if (u >= IV || (NTH * (u + 1) > NV && tid + NTH * u >= NV)) continue;
                    P[v] = prm[vij[u] & 0xffff];
                    const int pq = __float_as_int(P[v].w);
                    op[v] = (vij[u] >> 16) + (pq & 0xffff);
                    oq[v] = (vij[u] >> 16) + (pq >> 16);
                    xp[v] = V[op[v]];
                    xq[v] = V[oq[v]];
                }
#pragma unroll
                for (int v = 0; v < 2 * B; ++v) {
                    const int u = u0 + v;
                    if (u >= IV || (NTH * (u + 1) > NV && tid + NTH * u >= NV)) continue;
                    rotate_cols<true>(xp[v], xq[v], P[v].x, P[v].y, P[v].z);
                    V[op[v]] = xp[v];
                    V[oq[v]] = xq[v];
                }
            }
            __syncthreads();
        }
        if (!swept) break;
    }
    __syncthreads();
    // ascending order: rank of each eigenvalue (ties broken by index)
    for (int i = tid; i < nw; i += NTH) {
        const T ei = A[i * ld + i].re;
        int rk = 0;
        for (int j = 0; j < nw; ++j) {
            const T ej = A[j * ld + j].re;
            rk += (ej < ei) || (ej == ei && j < i);
        }
        rank[i] = rk;
        Eout[k * nw + rk] = (double)ei;
    }
    __syncthreads();
    for (int t = tid; t < nw * nw; t += NTH) {
        const int m = t / nw, i = t % nw;
        const cplx<T> v = V[m * ld + i];
        Uout[(k * nw + m) * nw + rank[i]] = mk((TO)v.re, (TO)v.im);
    }
}

// ---------------------------------------------------------------------------
// 64 < n <= 128: FP32 Jacobi with A in LDS (132 KB at n = 128) and V in registers, one 16-wave
// workgroup per k.  A is updated in blocks of two rows by two columns as in k_eigh_jacobi_b.
// V fills no LDS: lane l of every wave stands for pair position l - (64 - n/2) of the circle
// ordering and holds the elements of that pair's two columns in the wave's rows (rows wave,
// wave + 16, ...).  From one round to the next the first column of pair i + 1 becomes that of
// pair i and the second of pair i - 1 that of pair i (rr_pair), so the columns move by one lane
// (DPP wave shifts; the pairs sit in the top lanes, whose last one takes over its own second
// column), and after the n - 1 rounds of a sweep every column is back in place.
// Bound: VALU issue of the one workgroup that fits a CU (A 3.5k, V 2.5k cycles a round at
// n = 128); keeping V in row chunks of LDS took five workgroups per k, each repeating all of A
// (150 k-points at nw = 128: 29.1 -> 3.2 ms).
// ---------------------------------------------------------------------------
#define JREG_THREADS 1024
#define JREG_WAVES (JREG_THREADS / 64)

__host__ __device__ inline size_t jreg_lds(int n) {
    return sizeof(float4) * (n / 2) + sizeof(cplx<float>) * n * (n + 1) + sizeof(int) * (n + 2);
}

// lane l takes lane l + 1's value (the last lane: `last`) / lane l - 1's
__device__ inline float lane_from_next(float x, float last) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(last), __float_as_int(x), 0x130, 0xf, 0xf, false));
}
__device__ inline float lane_from_prev(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(x), __float_as_int(x), 0x138, 0xf, 0xf, false));
}

template <typename Tin, typename TO>
__global__ void __launch_bounds__(JREG_THREADS) k_eigh_jacobi_reg(int nw, const cplx<Tin>* __restrict__ H,
                                                                  int64_t Hstride, double* __restrict__ Eout,
                                                                  cplx<TO>* __restrict__ Uout, int max_sweeps) {
    typedef float T;
    constexpr int RV = 128 / JREG_WAVES;  // rows of V per wave
    constexpr int IB = 64 * 64 / JREG_THREADS;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int n = nw + (nw & 1), ld = n + 1, np = n / 2, nb = np * np;
    float4* prm = (float4*)smem;
    cplx<T>* A = (cplx<T>*)(prm + np);
    int* rank = (int*)(A + n * ld);
    int* flags = rank + n;  // RoundFlag
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t k = blockIdx.x;
    const cplx<Tin>* Hk = H + k * Hstride;
    for (int t = tid; t < n * n; t += JREG_THREADS) {
        const int i = t / n, j = t % n;
        cplx<T> a = mk((T)0, (T)0);
        if (i < nw && j < nw) {
            const cplx<Tin> x = Hk[i * nw + j], y = Hk[j * nw + i];
            a = mk((T)(0.5 * (x.re + y.re)), (T)(0.5 * (x.im - y.im)));
        }
        A[i * ld + j] = a;
    }
    const int first = 64 - np, pos = lane - first;  // pos < 0: no pair
    int p0 = 0, q0 = 0;
    if (pos >= 0) rr_pair(n, 0, pos, p0, q0);
    cplx<T> vp[RV], vq[RV];
#pragma unroll
    for (int v = 0; v < RV; ++v) {
        const int row = wave + JREG_WAVES * v;
        vp[v] = mk((T)(pos >= 0 && row == p0 ? 1 : 0), (T)0);
        vq[v] = mk((T)(pos >= 0 && row == q0 ? 1 : 0), (T)0);
    }
    int bi[IB], bj[IB];
#pragma unroll
    for (int u = 0; u < IB; ++u) {
        const int b = tid + JREG_THREADS * u;
        bi[u] = b < nb ? b / np : -1;
        bj[u] = b % np;
    }
    __syncthreads();
    RoundFlag flag;
    for (int sweep = 0; sweep < max_sweeps; ++sweep) {
        bool swept = false;
        for (int r = 0; r < n - 1; ++r) {
            if (tid < 64) {
                bool rot = false;
                if (tid < np) {
                    int p, q;
                    rr_pair(n, r, tid, p, q);
                    T c, sc, ss;
                    rot = jacobi_rotation<false>(A[p * ld + q], A[p * ld + p].re, A[q * ld + q].re, c, sc, ss);
                    prm[tid] = make_float4(c, sc, ss, __int_as_float(p | (q << 16)));
                }
                const bool w = __any(rot);
                if (tid == 0) flag.put(flags, w);
            }
            __syncthreads();
            const bool any = flag.take(flags) != 0;
            if (any) {
                swept = true;
#pragma unroll
                for (int u0 = 0; u0 < IB; u0 += 2) {
                    int o[2][4];
                    cplx<T> x[2][4];
                    float4 pi[2], pj[2];
#pragma unroll
                    for (int v = 0; v < 2; ++v) {
                        if (bi[u0 + v] < 0) continue;
                        pi[v] = prm[bi[u0 + v]];
                        pj[v] = prm[bj[u0 + v]];
                        const int ri = __float_as_int(pi[v].w), cj = __float_as_int(pj[v].w);
                        const int rp = (ri & 0xffff) * ld, rq = (ri >> 16) * ld, cp = cj & 0xffff, cq = cj >> 16;
                        o[v][0] = rp + cp;
                        o[v][1] = rp + cq;
                        o[v][2] = rq + cp;
                        o[v][3] = rq + cq;
#pragma unroll
                        for (int e = 0; e < 4; ++e) x[v][e] = A[o[v][e]];
                    }
#pragma unroll
                    for (int v = 0; v < 2; ++v) {
                        if (bi[u0 + v] < 0) continue;
                        rotate_cols<false>(x[v][0], x[v][1], pj[v].x, pj[v].y, pj[v].z);
                        rotate_cols<false>(x[v][2], x[v][3], pj[v].x, pj[v].y, pj[v].z);
                        rotate_rows(x[v][0], x[v][2], pi[v].x, pi[v].y, pi[v].z);
                        rotate_rows(x[v][1], x[v][3], pi[v].x, pi[v].y, pi[v].z);
#pragma unroll
                        for (int e = 0; e < 4; ++e) A[o[v][e]] = x[v][e];
                    }
                }
                const float4 P = prm[pos >= 0 ? pos : 0];
#pragma unroll
                for (int v = 0; v < RV; ++v) rotate_cols<false>(vp[v], vq[v], P.x, P.y, P.z);
            }
            // columns to their pair positions of the next round
#pragma unroll
            for (int v = 0; v < RV; ++v) {
                const cplx<T> tn = mk(lane_from_next(vp[v].re, vq[v].re), lane_from_next(vp[v].im, vq[v].im));
                const cplx<T> bn = mk(lane_from_prev(vq[v].re), lane_from_prev(vq[v].im));
                vq[v] = pos == 0 ? tn : bn;
                vp[v] = pos == 0 ? vp[v] : tn;
            }
            if (any) __syncthreads();
        }
        if (!swept) break;
    }
    __syncthreads();
    // ascending order (ties by index)
    for (int i = tid; i < nw; i += JREG_THREADS) {
        const T ei = A[i * ld + i].re;
        int rk = 0;
        for (int j = 0; j < nw; ++j) {
            const T ej = A[j * ld + j].re;
            rk += (ej < ei) || (ej == ei && j < i);
        }
        rank[i] = rk;
        Eout[k * nw + rk] = (double)ei;
    }
    __syncthreads();  // A is read no more: V goes through it, its columns in order
    if (pos >= 0) {
#pragma unroll
        for (int v = 0; v < RV; ++v) {
            const int row = wave + JREG_WAVES * v;
            if (row < nw && p0 < nw) A[row * ld + rank[p0]] = vp[v];
            if (row < nw && q0 < nw) A[row * ld + rank[q0]] = vq[v];
        }
    }
    __syncthreads();
    for (int t = tid; t < nw * nw; t += JREG_THREADS) {
        const cplx<T> v = A[(t / nw) * ld + t % nw];
        Uout[k * nw * nw + t] = mk((TO)v.re, (TO)v.im);
    }
}

// ---------------------------------------------------------------------------
// FP64 refinement steps of approximate eigenvectors (Ogita & Aishima,
// "Iterative refinement for symmetric eigenvalue decomposition", Japan J.
// Indust. Appl. Math. 35 (2018), Algorithm 1, written for Hermitian matrices):
//   R = I - X^+ X,  S = X^+ A X,  lam_i = S_ii / (1 - R_ii),
//   delta = 2 (||S - diag(lam)|| + max|lam| ||R||)   (Frobenius bounds),
//   E_ij = (S_ij + lam_j R_ij) / (lam_j - lam_i) if |lam_j - lam_i| > delta, else R_ij / 2,
//   X <- X + X E.
// Each step squares the error of the vectors of separated eigenvalues;
// clusters below delta are re-orthogonalised only.
// ---------------------------------------------------------------------------

// stop refining once ||E||_F is below this: complex64 vectors are limited by
// their storage; complex128 vectors after a step with ||E|| < 1e-10 are
// accurate to ~||E||^2 ||H|| / gap, i.e. to FP64 rounding
#define OA_TOL_C64 1e-8
#define OA_TOL_C128 1e-10
// complex64 vectors: a correction with ||E||_F below this is the last one.  The
// step converges quadratically, so the vectors it leaves are accurate to about
// ||E||^2 = 1e-8 (well below complex64 rounding) where the gaps are not small,
// and the cluster pass that follows rotates every pair still mixed by more than
// OA_TOL_C64 (close pairs converge more slowly).
#define OA_LAST_C64 1e-4

// Scratch of cluster_jacobi in LDS: per pair {c, s cos phi, s sin phi} and
// (p, q), plus a round flag pair.
__host__ __device__ inline size_t cj_lds(int n) {
    const int np = (n + 1) / 2;
    return sizeof(double) * 3 * np + sizeof(int) * (2 * np + 4);
}

// Finishes the refinement where it stalls: a pair closer than the
// Ogita-Aishima threshold delta is only re-orthogonalised by the correction
// step, so its two vectors can stay any unitary mix of the pair's
// eigenvectors.  With S = X^+ A X of the refined X (Hermitian, diagonal to
// the refinement's accuracy for separated eigenvalues), cyclic Jacobi sweeps
// (round-robin order, rotations of Golub & Van Loan, sec. 8.5.2, as in
// k_eigh_jacobi) rotate only the pairs with
//   |S_pq| > floor_abs  and  |S_pq| > theta |S_qq - S_pp|,
// i.e. whose mixing angle exceeds theta: none after a converged refinement of
// a separated spectrum, the unresolved pairs (and larger clusters) otherwise.
// The rotations update S (columns and rows) and the columns of X.
// Uniform control flow: the round flag is set by the rotating threads and
// read by every thread after a barrier (double-buffered by round parity).
__device__ inline bool cluster_pair(cplx<double> apq, double app, double aqq, double theta, double floor_abs) {
    const double g = sqrt(apq.re * apq.re + apq.im * apq.im);
    return g > floor_abs && g > theta * fabs(aqq - app);
}

template <int NTH, class FS, class FX>
__device__ void cluster_jacobi(int n, FS S, FX X, char* scratch, double theta, double floor_abs, int max_sweeps) {
    const int ne = n + (n & 1), np = ne / 2;
    double* prm = (double*)scratch;
    int* pq = (int*)(prm + 3 * np);
    int* flags = pq + 2 * np;  // [0] sweep, [1 + (r & 1)] round
    const int tid = threadIdx.x;
    for (int sweep = 0; sweep < max_sweeps; ++sweep) {
        if (tid == 0) flags[0] = flags[1] = flags[2] = 0;
        __syncthreads();
        for (int r = 0; r < ne - 1; ++r) {
            // the next round's flag: its last readers (round r - 1) passed a barrier since, or read 0
            if (tid == 0) flags[1 + ((r + 1) & 1)] = 0;
            if (tid < np) {
                int p, q;
                rr_pair(ne, r, tid, p, q);
                double c = 1.0, sc = 0.0, ss = 0.0;
                if (p < n && q < n) {
                    const cplx<double> apq = S(p, q);
                    const double g = sqrt(apq.re * apq.re + apq.im * apq.im);
                    const double app = S(p, p).re, aqq = S(q, q).re;
                    if (cluster_pair(apq, app, aqq, theta, floor_abs)) {
                        const double tau = (aqq - app) / (2.0 * g);
                        const double t = (tau >= 0 ? 1.0 : -1.0) / (fabs(tau) + sqrt(1.0 + tau * tau));
                        c = 1.0 / sqrt(1.0 + t * t);
                        const double sn = t * c;
                        sc = sn * apq.re / g;
                        ss = sn * apq.im / g;
                        flags[1 + (r & 1)] = 1;
                        flags[0] = 1;
                    }
                }
                prm[3 * tid] = c;
                prm[3 * tid + 1] = sc;
                prm[3 * tid + 2] = ss;
                pq[2 * tid] = p;
                pq[2 * tid + 1] = q;
            }
            __syncthreads();
            if (flags[1 + (r & 1)] == 0) continue;
            // columns of S and X: col_p <- c col_p - s e^{-i phi} col_q ; col_q <- s e^{i phi} col_p + c col_q
            for (int t = tid; t < np * n; t += NTH) {
                const int pr = t / n, i = t % n;
                const int p = pq[2 * pr], q = pq[2 * pr + 1];
                if (p >= n || q >= n) continue;
                const double c = prm[3 * pr];
                const cplx<double> se = mk(prm[3 * pr + 1], prm[3 * pr + 2]);
                if (c == 1.0 && se.re == 0.0 && se.im == 0.0) continue;
                const cplx<double> ap = S(i, p), aq = S(i, q), xp = X(i, p), xq = X(i, q);
                S(i, p) = c * ap - mulc(aq, se);
                S(i, q) = se * ap + c * aq;
                X(i, p) = c * xp - mulc(xq, se);
                X(i, q) = se * xp + c * xq;
            }
            __syncthreads();
            // rows of S: row_p <- c row_p - s e^{i phi} row_q ; row_q <- s e^{-i phi} row_p + c row_q
            for (int t = tid; t < np * n; t += NTH) {
                const int pr = t / n, j = t % n;
                const int p = pq[2 * pr], q = pq[2 * pr + 1];
                if (p >= n || q >= n) continue;
                const double c = prm[3 * pr];
                const cplx<double> se = mk(prm[3 * pr + 1], prm[3 * pr + 2]);
                if (c == 1.0 && se.re == 0.0 && se.im == 0.0) continue;
                const cplx<double> ap = S(p, j), aq = S(q, j);
                S(p, j) = c * ap - se * aq;
                S(q, j) = mulc(ap, se) + c * aq;
            }
            __syncthreads();
        }
        const bool more = flags[0] != 0;
        __syncthreads();
        if (!more) break;
    }
}

// Refinement steps until the correction satisfies ||E||_F < tol (at most
// `iters`), then eigenvalues as Rayleigh quotients of the final vectors.
// Well-separated spectra stop after two steps (||E|| ~ eps32, then ~eps32^2).
// A pair closer than delta of the first step (FP32 vectors mix it) is only
// re-orthogonalised there; the following steps separate it, converging
// quadratically once the mixing angle is small (six to eight steps for a
// relative gap of 4e-6 at nw = 18..40).
//
// One wave per 16 x 16 block of the matrices, NB x NB waves per k-point (nw <= 64): a wave keeps its block
// of S, R and X + X E in registers from the product to the elementwise step that uses it, S and X^+ X
// share their operand, and X, T = A X / E and (NB <= 3) A are the matrices in LDS; at NB = 4 A comes from
// L2.  The chain of dependent products and barriers bounds it, not the matrix cores, so what counts is
// k-points in flight and steps left out: the cluster pass runs only where a pair needs it.
// With four waves per k-point for every size, S and R through LDS and the cluster pass always, against now:
// nw = 32, 4096 k-points: complex128 657 -> 406 us (0.18 ms of matrix instructions), complex64 382 -> 192;
// nw = 12, 1728: 42.5 -> 26.2; nw = 2, 625: 32.9 -> 15.2; through global memory before, nw = 48, 3898
// k-points, complex64: 1509 -> 725; nw = 64, 294: 314 -> 182.
// SPLIT: re re, im im, re im and im re summed apart (complex64 up to nw = 44; above, and for complex128, together: half
// the accumulators).  Neither order is the more accurate; but a last-bit difference in the FP64 vectors
// moves a complex64 element by its rounding now and then, and close bands magnify that (summed together at nw = 32, a
// mixed-form dipole moved by 5e-9), so each size keeps one order.
template <typename TU, int NB, bool SPLIT>
__global__ void __launch_bounds__(64 * NB * NB, NB == 3 ? 5 : NB == 4 ? 4 : 3)
k_eigh_refine(int nw, const cplx<double>* __restrict__ H64, int64_t Hstride, double* __restrict__ Eout,
              cplx<TU>* __restrict__ U, int iters, double tol) {
    constexpr int NTH = 64 * NB * NB;
    constexpr bool ALDS = NB <= 3;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int ld = nw + 1;
    cplx<double>* sX = (cplx<double>*)smem;                 // X (approximate eigenvectors)
    cplx<double>* sT = sX + nw * ld;                        // A X, then E
    cplx<double>* sA = sT + nw * ld;                        // A (for the whole solve)
    double* lam = (double*)(ALDS ? sA + nw * ld : sA);
    double* den = lam + nw;                                 // squared norms of the columns' parts, [NB][nw]
    double* red2 = den + NB * nw;                           // two sets, steps in turn:
    // [0] ||S-D||^2, [1] ||R||^2, [2] max|lam|, [3] ||E||^2
    char* cjs = (char*)(red2 + 8);                          // cluster_jacobi scratch
    int* rank = (int*)(cjs + cj_lds(nw));
    const int tid = threadIdx.x, li = tid & 15, lk = (tid & 63) >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), r0 = 16 * (wave / NB), c0 = 16 * (wave % NB);
    const int64_t k = blockIdx.x;
    const cplx<double>* Hk = H64 + k * Hstride;
    cplx<TU>* Uk = U + k * nw * nw;
    const int c = c0 + li;                                       // the lane's elements: (r0 + lk + 4 v, c)
    const int ra = min(r0 + li, nw - 1), cc = min(c, nw - 1);    // operand row and column
    auto row = [&](int v) { return r0 + lk + 4 * v; };
    auto inside = [&](int v) { return c < nw && row(v) < nw; };
    auto herm = [&](int i, int j) {  // (H + H^+)/2
        const cplx<double> x = Hk[i * nw + j], y = Hk[j * nw + i];
        return mk(0.5 * (x.re + y.re), 0.5 * (x.im - y.im));
    };
    struct Tile {
        wbmi_v4d re, im;
        __device__ inline cplx<double> get(int v) const { return mk(re[v], im[v]); }
    };
    const wbmi_v4d z4 = {0.0, 0.0, 0.0, 0.0};
    struct Sum {
        wbmi_v4d re, im, ii, ir;  // ii, ir: SPLIT only
        __device__ inline void add(cplx<double> a, cplx<double> b) {
            re = __builtin_amdgcn_mfma_f64_16x16x4f64(a.re, b.re, re, 0, 0, 0);
            im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.re, b.im, im, 0, 0, 0);
            if constexpr (SPLIT) {
                ir = __builtin_amdgcn_mfma_f64_16x16x4f64(a.im, b.re, ir, 0, 0, 0);
                ii = __builtin_amdgcn_mfma_f64_16x16x4f64(a.im, b.im, ii, 0, 0, 0);
            } else {
                re = __builtin_amdgcn_mfma_f64_16x16x4f64(-a.im, b.im, re, 0, 0, 0);
                im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.im, b.re, im, 0, 0, 0);
            }
        }
        __device__ inline Tile tile() const {
            if constexpr (SPLIT) return Tile{re - ii, im + ir};
            else return Tile{re, im};
        }
    };
    // the wave's block of P Q, and of P Q and P Q2 together; operand columns / rows from nw on count zero
    auto product = [&](auto P, auto Q) {
        Sum t{z4, z4, z4, z4};
#pragma unroll 2
        for (int k0 = 0; k0 < nw; k0 += 4) {
            const int m = min(k0 + lk, nw - 1);
            const cplx<double> a = P(m);
            cplx<double> b = Q(m);
            if (k0 + lk >= nw) b = mk(0.0, 0.0);
            t.add(a, b);
        }
        return t.tile();
    };
    auto products = [&](auto P, auto Q, auto Q2, Tile& r, Tile& r2) {
        Sum t{z4, z4, z4, z4}, t2 = t;
#pragma unroll 2
        for (int k0 = 0; k0 < nw; k0 += 4) {
            const int m = min(k0 + lk, nw - 1);
            cplx<double> a = P(m);
            const cplx<double> b = Q(m), b2 = Q2(m);
            if (k0 + lk >= nw) a = mk(0.0, 0.0);
            t.add(a, b);
            t2.add(a, b2);
        }
        r = t.tile();
        r2 = t2.tile();
    };
    auto Arow = [&](int m) {
        if constexpr (ALDS) return sA[ra * ld + m];
        else return herm(ra, m);
    };
    auto Xrow = [&](int m) { return sX[ra * ld + m]; };
    auto Xadj = [&](int m) { return conj(sX[m * ld + ra]); };
    auto Xcol = [&](int m) { return sX[m * ld + cc]; };
    auto Tcol = [&](int m) { return sT[m * ld + cc]; };
    auto store = [&](cplx<double>* M, const Tile& t) {
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if (inside(v)) M[row(v) * ld + c] = t.get(v);
    };
    auto add_X_times_T = [&] {  // X <- X + X sT
        Tile t = product(Xrow, Tcol);
#pragma unroll
        for (int v = 0; v < 4; ++v)
            if (inside(v)) {
                const cplx<double> x = sX[row(v) * ld + c];
                t.re[v] += x.re;
                t.im[v] += x.im;
            }
        __syncthreads();
        store(sX, t);
    };
#pragma unroll
    for (int v = 0; v < 4; ++v)
        if (inside(v)) {
            const cplx<TU> u = Uk[row(v) * nw + c];
            sX[row(v) * ld + c] = mk((double)u.re, (double)u.im);
            if constexpr (ALDS) sA[row(v) * ld + c] = herm(row(v), c);
        }
    double scale = 0.0;
    for (int it = 0; it < iters; ++it) {
        double* red = red2 + 4 * (it & 1);
        if (tid < 4) red[tid] = 0.0;
        __syncthreads();
        store(sT, product(Arow, Xcol));
        __syncthreads();
        Tile S, R;
        products(Xadj, Tcol, Xcol, S, R);
        // R = I - X^+ X, the eigenvalues, Frobenius norms and max|lam|
        double s2 = 0.0, r2 = 0.0, lm = 0.0;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            if (!inside(v)) continue;
            const bool diag = row(v) == c;
            R.re[v] = (diag ? 1.0 : 0.0) - R.re[v];
            R.im[v] = -R.im[v];
            cplx<double> sv = S.get(v);
            if (diag) {
                const double l = sv.re / (1.0 - R.re[v]);
                lam[c] = l;
                lm = fabs(l);
                sv.re -= l;
            }
            s2 += sv.re * sv.re + sv.im * sv.im;
            r2 += R.re[v] * R.re[v] + R.im[v] * R.im[v];
        }
        for (int off = 32; off > 0; off >>= 1) {
            s2 += __shfl_down(s2, off);
            r2 += __shfl_down(r2, off);
            lm = fmax(lm, __shfl_down(lm, off));
        }
        if ((tid & 63) == 0) {
            atomicAdd(&red[0], s2);
            atomicAdd(&red[1], r2);
            atomicMax((unsigned long long*)&red[2], (unsigned long long)__double_as_longlong(lm));
        }
        __syncthreads();
        scale = red[2];
        const double delta = 2.0 * (sqrt(red[0]) + scale * sqrt(red[1]));
        // E into sT (A X is no longer read), ||E||^2 into red[3]
        double e2 = 0.0;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            if (!inside(v)) continue;
            const double lc = lam[c], dl = lc - lam[row(v)];
            cplx<double> e;
            if (fabs(dl) > delta)
                e = (1.0 / dl) * mk(S.re[v] + lc * R.re[v], S.im[v] + lc * R.im[v]);
            else
                e = mk(0.5 * R.re[v], 0.5 * R.im[v]);
            sT[row(v) * ld + c] = e;
            e2 += e.re * e.re + e.im * e.im;
        }
        for (int off = 32; off > 0; off >>= 1) e2 += __shfl_down(e2, off);
        if ((tid & 63) == 0) atomicAdd(&red[3], e2);
        __syncthreads();
        // (this set is cleared two steps on, after barriers that follow every thread's reading)
        const bool converged = red[3] < tol * tol || (sizeof(TU) == 4 && red[3] < OA_LAST_C64 * OA_LAST_C64);
        add_X_times_T();
        if (converged) break;
    }
    __syncthreads();
    if (sizeof(TU) == 8) {
        // complex128 output: one Newton-Schulz step X <- X (I + R/2), R = I - X^+ X, so that the
        // basis is orthonormal to rounding also where a close pair leaves the vectors themselves
        // accurate only to ~eps |H| / gap (the correction steps do not preserve orthogonality)
        Tile t = product(Xadj, Xcol);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            t.re[v] = 0.5 * ((row(v) == c ? 1.0 : 0.0) - t.re[v]);
            t.im[v] = -0.5 * t.im[v];
        }
        store(sT, t);
        __syncthreads();
        add_X_times_T();
        __syncthreads();
    }
    // S = X^+ A X of the refined columns; pairs left mixed are rotated apart (scale: max |lam| of the last step)
    store(sT, product(Arow, Xcol));
    __syncthreads();
    const Tile S = product(Xadj, Tcol);
    double x2 = 0.0;
#pragma unroll
    for (int v = 0; v < 4; ++v)
        if (inside(v)) {
            const cplx<double> x = sX[row(v) * ld + c];
            x2 += x.re * x.re + x.im * x.im;
            if (row(v) == c) lam[c] = S.re[v];
        }
    x2 += __shfl_xor(x2, 16);
    x2 += __shfl_xor(x2, 32);
    if (lk == 0 && c < nw) den[r0 / 16 * nw + c] = x2;  // summed in a fixed order: energies repeat bit for bit
    __syncthreads();
    const double theta = tol, floor_abs = 64.0 * DBL_EPSILON * scale;
    int mixed = 0;
#pragma unroll
    for (int v = 0; v < 4; ++v)
        if (inside(v) && row(v) != c) mixed |= cluster_pair(S.get(v), lam[row(v)], lam[c], theta, floor_abs);
    if (__syncthreads_or(mixed)) {
        store(sT, S);
        __syncthreads();
        cluster_jacobi<NTH>(
            nw, [&](int i, int j) -> cplx<double>& { return sT[i * ld + j]; },
            [&](int i, int j) -> cplx<double>& { return sX[i * ld + j]; }, cjs, theta, floor_abs, 10);
        for (int i = tid; i < nw; i += NTH) {
            double d = 0.0;
            for (int m = 0; m < nw; ++m) {
                const cplx<double> x = sX[m * ld + i];
                d += x.re * x.re + x.im * x.im;
            }
            den[i] = d;
            for (int q = 1; q < NB; ++q) den[q * nw + i] = 0.0;
            lam[i] = sT[i * ld + i].re;
        }
        __syncthreads();
    }
    // eigenvalues: Rayleigh quotients x_c^+ A x_c / x_c^+ x_c = S_cc / x_c^+ x_c
    for (int i = tid; i < nw; i += NTH) {
        double d = den[i];
#pragma unroll
        for (int q = 1; q < NB; ++q) d += den[q * nw + i];
        lam[i] /= d;
    }
    __syncthreads();
    // ascending order (ties by index)
    for (int i = tid; i < nw; i += NTH) {
        const double l = lam[i];
        int rk = 0;
        for (int j = 0; j < nw; ++j) rk += (lam[j] < l) || (lam[j] == l && j < i);
        rank[i] = rk;
        Eout[k * nw + rk] = l;
    }
    __syncthreads();
#pragma unroll
    for (int v = 0; v < 4; ++v)
        if (inside(v)) {
            const cplx<double> x = sX[row(v) * ld + c];
            Uk[row(v) * nw + rank[c]] = mk((TU)x.re, (TU)x.im);
        }
}

// ---------------------------------------------------------------------------
// Refinement for 64 < nw <= 128: the same steps with the four nw x nw matrices
// (X, T, S/E, R) in a per-k workspace of global memory and every product as
// 32 x 32 wave tasks on the FP64 matrix cores (operands read through L2).
// ---------------------------------------------------------------------------
#define OAG_THREADS 1024  // one wave per 32 x 32 block; nw = 128, 150 k-points: 1.60 ms in 8 waves, 1.25 in 16
#define OAG_NWMAX 128

// C = P Q (n x n) as wave tasks; out(r, c, value) for r, c < n
template <class FP, class FQ, class FO>
__device__ __attribute__((always_inline)) void wg_gemm(int n, FP P, FQ Q, FO out) {
    const int wave = threadIdx.x >> 6, nwave = OAG_THREADS / 64;
    const int nb = (n + 31) / 32;
    for (int t = wave; t < nb * nb; t += nwave) {
        const int rb = t / nb, cb = t % nb;
        MfmaBlock C;
        C.zero();
        mfma_block(C, n, n, n, rb * 32, cb * 32, P, Q);
#pragma unroll
        for (int bi = 0; bi < 2; ++bi)
#pragma unroll
            for (int bj = 0; bj < 2; ++bj)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int r = rb * 32 + mfma_row(bi, v), c = cb * 32 + mfma_col(bj);
                    if (r < n && c < n) out(r, c, C.get(bi, bj, v));
                }
    }
}

__device__ inline double block_sum_to(double v, double* slot) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off);
    if ((threadIdx.x & 63) == 0) atomicAdd(slot, v);
    return v;
}

template <typename TU>
__global__ void __launch_bounds__(OAG_THREADS) k_eigh_refine_g(int n, const cplx<double>* __restrict__ H64,
                                                              int64_t Hstride, double* __restrict__ Eout,
                                                              cplx<TU>* __restrict__ U, int iters, double tol,
                                                              cplx<double>* __restrict__ work) {
    __shared__ double lam[OAG_NWMAX];
    __shared__ double red[4];  // [0] ||S-D||^2, [1] ||R||^2, [2] max|lam|, [3] ||E||^2
    __shared__ int rank[OAG_NWMAX];
    __shared__ __attribute__((aligned(16))) char cjs[sizeof(double) * 3 * (OAG_NWMAX / 2) +
                                                     sizeof(int) * (OAG_NWMAX + 4)];
    const int tid = threadIdx.x, n2 = n * n;
    const int64_t k = blockIdx.x;
    const cplx<double>* Hk = H64 + k * Hstride;
    cplx<TU>* Uk = U + k * n2;
    cplx<double>* X = work + k * 4 * (int64_t)n2;
    cplx<double>* T = X + n2;
    cplx<double>* S = T + n2;
    cplx<double>* R = S + n2;
    auto Aop = [&](int r, int m) {
        const cplx<double> x = Hk[r * n + m], y = Hk[m * n + r];
        return mk(0.5 * (x.re + y.re), 0.5 * (x.im - y.im));
    };
    for (int t = tid; t < n2; t += OAG_THREADS) {
        const cplx<TU> u = Uk[t];
        X[t] = mk((double)u.re, (double)u.im);
    }
    __syncthreads();
    for (int it = 0; it < iters; ++it) {
        if (tid < 4) red[tid] = 0.0;
        wg_gemm(n, Aop, [&](int m, int c) { return X[m * n + c]; }, [&](int r, int c, cplx<double> v) { T[r * n + c] = v; });
        __syncthreads();
        wg_gemm(n, [&](int r, int m) { return conj(X[m * n + r]); }, [&](int m, int c) { return T[m * n + c]; },
                [&](int r, int c, cplx<double> v) { S[r * n + c] = v; });
        wg_gemm(n, [&](int r, int m) { return conj(X[m * n + r]); }, [&](int m, int c) { return X[m * n + c]; },
                [&](int r, int c, cplx<double> v) { R[r * n + c] = mk((r == c ? 1.0 : 0.0) - v.re, -v.im); });
        __syncthreads();
        for (int i = tid; i < n; i += OAG_THREADS) lam[i] = S[i * n + i].re / (1.0 - R[i * n + i].re);
        __syncthreads();
        double s2 = 0.0, r2 = 0.0, lm = 0.0;
        for (int t = tid; t < n2; t += OAG_THREADS) {
            const int i = t / n, j = t % n;
            cplx<double> sv = S[t];
            if (i == j) sv.re -= lam[i];
            s2 += sv.re * sv.re + sv.im * sv.im;
            r2 += R[t].re * R[t].re + R[t].im * R[t].im;
        }
        for (int i = tid; i < n; i += OAG_THREADS) lm = fmax(lm, fabs(lam[i]));
        for (int off = 32; off > 0; off >>= 1) lm = fmax(lm, __shfl_down(lm, off));
        block_sum_to(s2, &red[0]);
        block_sum_to(r2, &red[1]);
        if ((tid & 63) == 0) atomicMax((unsigned long long*)&red[2], (unsigned long long)__double_as_longlong(lm));
        __syncthreads();
        const double delta = 2.0 * (sqrt(red[0]) + red[2] * sqrt(red[1]));
        double e2 = 0.0;
        for (int t = tid; t < n2; t += OAG_THREADS) {
            const int i = t / n, j = t % n;
            const double dl = lam[j] - lam[i];
            const cplx<double> r = R[t];
            cplx<double> e;
            if (fabs(dl) > delta) {
                const cplx<double> sv = S[t];
                e = (1.0 / dl) * mk(sv.re + lam[j] * r.re, sv.im + lam[j] * r.im);
            } else {
                e = 0.5 * r;
            }
            S[t] = e;
            e2 += e.re * e.re + e.im * e.im;
        }
        block_sum_to(e2, &red[3]);
        __syncthreads();
        // every thread reads red[3] here; it is cleared only after the next barrier
        const bool converged = red[3] < tol * tol || (sizeof(TU) == 4 && red[3] < OA_LAST_C64 * OA_LAST_C64);
        wg_gemm(n, [&](int r, int m) { return X[r * n + m]; }, [&](int m, int c) { return S[m * n + c]; },
                [&](int r, int c, cplx<double> v) { T[r * n + c] = X[r * n + c] + v; });
        __syncthreads();
        cplx<double>* t = X;
        X = T;
        T = t;
        if (converged) break;
    }
    if (sizeof(TU) == 8) {
        // Newton-Schulz orthonormalisation X <- X (I + R/2), R = I - X^+ X
        wg_gemm(n, [&](int r, int m) { return conj(X[m * n + r]); }, [&](int m, int c) { return X[m * n + c]; },
                [&](int r, int c, cplx<double> v) { R[r * n + c] = mk(0.5 * ((r == c ? 1.0 : 0.0) - v.re), -0.5 * v.im); });
        __syncthreads();
        wg_gemm(n, [&](int r, int m) { return X[r * n + m]; }, [&](int m, int c) { return R[m * n + c]; },
                [&](int r, int c, cplx<double> v) { T[r * n + c] = X[r * n + c] + v; });
        __syncthreads();
        cplx<double>* t = X;
        X = T;
        T = t;
    }
    // S = X^+ A X of the refined columns; pairs left mixed are rotated apart
    const double scale = red[2];  // max |lam| of the last step
    wg_gemm(n, Aop, [&](int m, int c) { return X[m * n + c]; }, [&](int r, int c, cplx<double> v) { T[r * n + c] = v; });
    __syncthreads();
    wg_gemm(n, [&](int r, int m) { return conj(X[m * n + r]); }, [&](int m, int c) { return T[m * n + c]; },
            [&](int r, int c, cplx<double> v) { S[r * n + c] = v; });
    __syncthreads();
    for (int i = tid; i < n; i += OAG_THREADS) lam[i] = S[i * n + i].re;
    __syncthreads();
    int mixed = 0;
    for (int t = tid; t < n2; t += OAG_THREADS) {
        const int i = t / n, j = t % n;
        if (i != j) mixed |= cluster_pair(S[t], lam[i], lam[j], tol, 64.0 * DBL_EPSILON * scale);
    }
    if (__syncthreads_or(mixed))
        cluster_jacobi<OAG_THREADS>(
            n, [&](int i, int j) -> cplx<double>& { return S[i * n + j]; },
            [&](int i, int j) -> cplx<double>& { return X[i * n + j]; }, cjs, tol, 64.0 * DBL_EPSILON * scale, 10);
    // Rayleigh quotients x_c^+ A x_c / x_c^+ x_c = S_cc / x_c^+ x_c
    for (int c = tid; c < n; c += OAG_THREADS) {
        double den = 0.0;
        for (int m = 0; m < n; ++m) {
            const cplx<double> x = X[m * n + c];
            den += x.re * x.re + x.im * x.im;
        }
        lam[c] = S[c * n + c].re / den;
    }
    __syncthreads();
    for (int i = tid; i < n; i += OAG_THREADS) {
        int rk = 0;
        for (int j = 0; j < n; ++j) rk += (lam[j] < lam[i]) || (lam[j] == lam[i] && j < i);
        rank[i] = rk;
    }
    __syncthreads();
    for (int t = tid; t < n2; t += OAG_THREADS) {
        const int r = t / n, c = t % n;
        const cplx<double> x = X[t];
        Uk[r * n + rank[c]] = mk((TU)x.re, (TU)x.im);
    }
    for (int i = tid; i < n; i += OAG_THREADS) Eout[k * n + rank[i]] = lam[i];
}

// Scratch of wbmi_eigh_noalloc: the per-k refinement workspace (X, T, S/E, R;
// 64 < nw <= 128) in a file-scope device array, so that callers that cannot allocate
// (graph capture, serving loops) get the refined solver without a workspace.  Each GPU
// holds its own copy for the life of the process; calls on one GPU share it (their
// kernels write every element before reading it, so nothing needs clearing, and
// overlapping calls on one GPU race).  Host code uses the per-device address from
// hipGetSymbolAddress, never the array's name.
#define WBMI_EIGH_SCRATCH_BYTES ((size_t)64 << 20)
static __device__ __align__(256) char scratch[WBMI_EIGH_SCRATCH_BYTES];

int wbmi_eigh_scratch_init(void** ptr) {
    *ptr = nullptr;
    return hipGetSymbolAddress(ptr, HIP_SYMBOL(scratch)) == hipSuccess && *ptr ? 0 : 1;
}

// bytes of global workspace wbmi_eigh needs (refinement for nw > 64: k_eigh_refine_g)
static size_t eigh_work_bytes(int nk, int nw, int refine) {
    return (refine && nw > 64) ? sizeof(cplx<double>) * 4 * (size_t)nw * nw * nk : 0;
}

extern "C" size_t wbmi_eigh_work_bytes(int nk, int nw, int prec, int refine) {
    (void)prec;
    return nk > 0 && nw > 0 ? eigh_work_bytes(nk, nw, refine) : 0;
}

#define JACOBI_SWEEPS 40
#define JACOBI_FEW_1 768  // k-points up to which four waves (N <= 32), sixteen (N > 32) share one
#define JACOBI_FEW_4 512

template <int N, typename TU>
static int launch_jacobi_b(wbmi_ctx* ctx, int nk, int nw, const cplx<double>* H64, int64_t Hstride, double* E,
                           cplx<TU>* U, const cplx<TU>* U0) {
    const size_t lds = jacobi_b_lds<N>();
    auto launch = [&](auto few) -> int {
        constexpr int NWAVE = jacobi_b_waves<N>(decltype(few)::value);
        auto kernel = k_eigh_jacobi_b<N, NWAVE, double, TU>;
        if (lds > 64 * 1024)
            WBMI_HIP_CHECK(ctx, hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(kernel, dim3(nk), dim3(64 * NWAVE), lds, ctx->stream, nw, H64, Hstride, E, U, JACOBI_SWEEPS, U0);
        WBMI_LAUNCH_CHECK(ctx);
        return WBMI_OK;
    };
    return N > 16 && nk <= (N <= 32 ? JACOBI_FEW_1 : JACOBI_FEW_4) ? launch(std::true_type{}) : launch(std::false_type{});
}

// the launcher of padded size n = 2 HALF, searched from HALF down
template <int HALF, typename TU>
static int launch_jacobi_n(wbmi_ctx* ctx, int nk, int nw, const cplx<double>* H64, int64_t Hstride, double* E,
                           cplx<TU>* U, const cplx<TU>* U0) {
    if ((nw + 1) / 2 == HALF) return launch_jacobi_b<2 * HALF, TU>(ctx, nk, nw, H64, Hstride, E, U, U0);
    if constexpr (HALF > 1)
        return launch_jacobi_n<HALF - 1, TU>(ctx, nk, nw, H64, Hstride, E, U, U0);
    else
        return wbmi_fail(ctx, WBMI_ERR_ARG, "wbmi_eigh: nw = %d", nw);
}

// FP32 Jacobi of the FP64 Hamiltonian (eigenvectors stored as TU)
template <typename TU>
static int jacobi_f32_of_f64(wbmi_ctx* ctx, int nk, int nw, const cplx<double>* H64, int64_t Hstride, double* E,
                             cplx<TU>* U, const cplx<TU>* U0 = nullptr) {
    if (nw <= 64) return launch_jacobi_n<32, TU>(ctx, nk, nw, H64, Hstride, E, U, U0);
    const size_t lds = jreg_lds(nw + (nw & 1));
    WBMI_HIP_CHECK(ctx, hipFuncSetAttribute((const void*)k_eigh_jacobi_reg<double, TU>,
                                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL((k_eigh_jacobi_reg<double, TU>), dim3(nk), dim3(JREG_THREADS), lds, ctx->stream, nw, H64,
                       Hstride, E, U, JACOBI_SWEEPS);
    WBMI_LAUNCH_CHECK(ctx);
    return WBMI_OK;
}

template <typename TU, int NB>
static int launch_refine(wbmi_ctx* ctx, int nk, int nw, const cplx<double>* H64, int64_t Hstride, double* E,
                         cplx<TU>* U, int steps, double tol) {
    const size_t lds = (NB <= 3 ? 3 : 2) * sizeof(cplx<double>) * nw * (nw + 1) + sizeof(double) * ((1 + NB) * nw + 8) +
                       cj_lds(nw) + sizeof(int) * nw + 16;
    auto launch = [&](auto split) -> int {
        auto kernel = k_eigh_refine<TU, NB, decltype(split)::value>;
        WBMI_HIP_CHECK(ctx, hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(kernel, dim3(nk), dim3(64 * NB * NB), lds, ctx->stream, nw, H64, Hstride, E, U, steps, tol);
        WBMI_LAUNCH_CHECK(ctx);
        return WBMI_OK;
    };
    if constexpr (sizeof(TU) == 4 && NB < 3)
        return launch(std::true_type{});
    else if constexpr (sizeof(TU) == 4 && NB == 3)
        return nw <= 44 ? launch(std::true_type{}) : launch(std::false_type{});
    else
        return launch(std::false_type{});
}

// FP32 Jacobi of the FP64 Hamiltonian, then FP64 Ogita-Aishima steps; eigenvectors stored as TU
template <typename TU>
static int eigh_refined(wbmi_ctx* ctx, int nk, int nw, const cplx<double>* H64, int64_t Hstride, double* E,
                        cplx<TU>* U, int steps, void* work, size_t work_bytes, const cplx<TU>* U0 = nullptr) {
    const double tol = sizeof(TU) == 4 ? OA_TOL_C64 : OA_TOL_C128;
    if (nw > 64 && (!work || work_bytes < eigh_work_bytes(nk, nw, steps)))
        return wbmi_fail(ctx, WBMI_ERR_ARG, "wbmi_eigh: refinement at nw = %d needs %zu bytes of workspace", nw,
                         eigh_work_bytes(nk, nw, steps));
    int rc = jacobi_f32_of_f64<TU>(ctx, nk, nw, H64, Hstride, E, U, U0);
    if (rc) return rc;
    if (nw > 64) {
        hipLaunchKernelGGL((k_eigh_refine_g<TU>), dim3(nk), dim3(OAG_THREADS), 0, ctx->stream, nw, H64, Hstride, E, U,
                           steps, tol, (cplx<double>*)work);
        WBMI_LAUNCH_CHECK(ctx);
        return WBMI_OK;
    }
    return nw <= 16   ? launch_refine<TU, 1>(ctx, nk, nw, H64, Hstride, E, U, steps, tol)
           : nw <= 32 ? launch_refine<TU, 2>(ctx, nk, nw, H64, Hstride, E, U, steps, tol)
           : nw <= 48 ? launch_refine<TU, 3>(ctx, nk, nw, H64, Hstride, E, U, steps, tol)
                      : launch_refine<TU, 4>(ctx, nk, nw, H64, Hstride, E, U, steps, tol);
}

extern "C" int wbmi_eigh(wbmi_ctx* ctx, int nk, int nw, const void* H_dev, int64_t Hstride, double* E_dev,
                         void* U_dev, int prec, int refine, const void* H64_dev, void* work_dev, size_t work_bytes) {
    if (!ctx) return WBMI_ERR_ARG;
    if (nk <= 0 || nw <= 0 || nw > 128 || !E_dev || !U_dev || Hstride < (int64_t)nw * nw)
        return wbmi_fail(ctx, WBMI_ERR_ARG, "wbmi_eigh: bad arguments (nw <= 128, Hstride >= nw*nw)");
    if (refine < 0 || refine > 16) return wbmi_fail(ctx, WBMI_ERR_ARG, "wbmi_eigh: refine must be 0..16");
    if (prec != WBMI_F64 && prec != WBMI_F32) return wbmi_fail(ctx, WBMI_ERR_ARG, "wbmi_eigh: bad precision");
    if (refine) {
        // the FP64 Hamiltonian: H_dev (complex128) for prec = WBMI_F64, H64_dev for prec = WBMI_F32
        const void* H64 = prec == WBMI_F64 ? H_dev : H64_dev;
        if (!H64) return wbmi_fail(ctx, WBMI_ERR_ARG, "wbmi_eigh: refinement needs the FP64 Hamiltonian");
        if (prec == WBMI_F64)
            return eigh_refined<double>(ctx, nk, nw, (const cplx<double>*)H64, Hstride, E_dev, (cplx<double>*)U_dev,
                                        refine, work_dev, work_bytes);
        return eigh_refined<float>(ctx, nk, nw, (const cplx<double>*)H64, Hstride, E_dev, (cplx<float>*)U_dev, refine,
                                   work_dev, work_bytes);
    }
    if (!H_dev) return wbmi_fail(ctx, WBMI_ERR_ARG, "wbmi_eigh: H_dev is null");
    if (nw > 64) return wbmi_fail(ctx, WBMI_ERR_ARG, "wbmi_eigh: nw > 64 needs refine >= 1");
    const int n = nw + (nw & 1);
    const int sweeps = 40;
    if (prec == WBMI_F64) {
        size_t lds = 2 * sizeof(cplx<double>) * n * (n + 1) + 3 * sizeof(double) * (n / 2) + 16;
        WBMI_HIP_CHECK(ctx, hipFuncSetAttribute((const void*)k_eigh_jacobi<double, double>,
                                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL((k_eigh_jacobi<double, double>), dim3(nk), dim3(64), lds, ctx->stream, nw,
                           (const cplx<double>*)H_dev, Hstride, E_dev, (cplx<double>*)U_dev, sweeps);
    } else {
        size_t lds = 2 * sizeof(cplx<float>) * n * (n + 1) + 3 * sizeof(float) * (n / 2) + 16;
        WBMI_HIP_CHECK(ctx, hipFuncSetAttribute((const void*)k_eigh_jacobi<float, float>,
                                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL((k_eigh_jacobi<float, float>), dim3(nk), dim3(64), lds, ctx->stream, nw,
                           (const cplx<float>*)H_dev, Hstride, E_dev, (cplx<float>*)U_dev, sweeps);
    }
    WBMI_LAUNCH_CHECK(ctx);
    return WBMI_OK;
}

extern "C" size_t wbmi_eigh_noalloc_max_bytes(void) { return WBMI_EIGH_SCRATCH_BYTES; }

extern "C" int wbmi_eigh_noalloc(wbmi_ctx* ctx, int nk, int nw, const void* H_dev, int64_t Hstride, double* E_dev,
                                 void* U_dev, int prec, int refine, const void* H64_dev) {
    if (!ctx) return WBMI_ERR_ARG;
    const size_t need = nk > 0 && nw > 0 ? eigh_work_bytes(nk, nw, refine) : 0;
    if (need > WBMI_EIGH_SCRATCH_BYTES)
        return wbmi_fail(ctx, WBMI_ERR_ARG,
                         "wbmi_eigh_noalloc: %d k-points at nw = %d need %zu bytes of scratch, more than its %zu "
                         "(at most %zu k-points per call at this nw)",
                         nk, nw, need, WBMI_EIGH_SCRATCH_BYTES,
                         WBMI_EIGH_SCRATCH_BYTES / eigh_work_bytes(1, nw, refine));
    if (need > 0 && !ctx->eigh_scratch) return wbmi_fail(ctx, WBMI_ERR_HIP, "wbmi_eigh_noalloc: no scratch address");
    return wbmi_eigh(ctx, nk, nw, H_dev, Hstride, E_dev, U_dev, prec, refine, H64_dev, ctx->eigh_scratch,
                     WBMI_EIGH_SCRATCH_BYTES);
}

extern "C" int wbmi_eigh_guess(wbmi_ctx* ctx, int nk, int nw, const void* H_dev, int64_t Hstride, double* E_dev,
                               void* U_dev, int prec, int refine, const void* H64_dev, const void* U0_dev,
                               void* work_dev, size_t work_bytes) {
    if (!ctx) return WBMI_ERR_ARG;
    if (!U0_dev)
        return wbmi_eigh(ctx, nk, nw, H_dev, Hstride, E_dev, U_dev, prec, refine, H64_dev, work_dev, work_bytes);
    if (nk <= 0 || nw <= 0 || nw > 128 || !E_dev || !U_dev || Hstride < (int64_t)nw * nw)
        return wbmi_fail(ctx, WBMI_ERR_ARG, "wbmi_eigh_guess: bad arguments (nw <= 128, Hstride >= nw*nw)");
    if (refine < 1 || refine > 16) return wbmi_fail(ctx, WBMI_ERR_ARG, "wbmi_eigh_guess: refine must be 1..16");
    if (prec != WBMI_F64 && prec != WBMI_F32) return wbmi_fail(ctx, WBMI_ERR_ARG, "wbmi_eigh_guess: bad precision");
    const void* H64 = prec == WBMI_F64 ? H_dev : H64_dev;
    if (!H64) return wbmi_fail(ctx, WBMI_ERR_ARG, "wbmi_eigh_guess: refinement needs the FP64 Hamiltonian");
    if (prec == WBMI_F64)
        return eigh_refined<double>(ctx, nk, nw, (const cplx<double>*)H64, Hstride, E_dev, (cplx<double>*)U_dev,
                                    refine, work_dev, work_bytes, (const cplx<double>*)U0_dev);
    return eigh_refined<float>(ctx, nk, nw, (const cplx<double>*)H64, Hstride, E_dev, (cplx<float>*)U_dev, refine,
                               work_dev, work_bytes, (const cplx<float>*)U0_dev);
}
