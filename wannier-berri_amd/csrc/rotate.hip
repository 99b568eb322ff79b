// Gauge rotation Xbar = U^+ X U of libwbmi (data_K/data_K.py:130-132).
//
// k_rotate_r (nw <= 32) and k_rotate_s (above) run on the FP64 matrix cores (v_mfma_f64_16x16x4f64, operand
// layout in mfma_c64.h) whatever the storage type, k_rotate_v (complex64 velocity, 32 < nw <= 64) on FP64 FMAs,
// k_rotate_h (complex64, nw <= 32, every channel but the velocity) on the fp16 matrix cores.  In the first two neither
// X nor the product between passes through LDS (k_rotate_r keeps U there): with the summed index
// enumerated as 4 s + lane / 16 for step s,
//   * lane l's U element of step s and column block b, U[4 s + l / 16][16 b + l % 16], is the B
//     operand of T = X U and, conjugated, the A operand of U^+ T for row block b;
//   * register v of T's row block i, T[16 i + l / 16 + 4 v][l % 16], is the B operand of step
//     4 i + v of U^+ T.
// So X goes from memory into the A operand of the first product, T never leaves the accumulators,
// and Xbar is stored from those of the second.
//
// Complex64 storage: channels are rotated with FP64 arithmetic on the
// complex64 operands (only the stored result is rounded).  FP32 accumulation
// would leave a normwise error ~eps32 |X| |U| in every element, which the
// 1/(E_n - E_m)^2 of the Berry curvature amplifies for small elements between
// close bands.
#include <type_traits>

#include "mfma_c64.h"
#include "wbmi_common.h"

__host__ __device__ inline bool bit_of(uint64_t lo, uint64_t hi, int c) { return c < 64 ? (lo >> c) & 1 : (hi >> (c - 64)) & 1; }

// element (r, c) of an nw x nw matrix, 0 outside: loaded at clamped indices and selected, so that no
// branch separates a batch of loads
template <typename T>
__device__ inline cplx<T> rot_load(const cplx<T>* M, int nw, int r, int c) {
    const cplx<T> v = M[min(r, nw - 1) * nw + min(c, nw - 1)];
    const bool ok = r < nw && c < nw;
    return mk(ok ? v.re : (T)0, ok ? v.im : (T)0);
}
template <typename T>
__device__ inline cplx<double> rot_elem(const cplx<T>* M, int nw, int r, int c) {
    const cplx<T> v = rot_load(M, nw, r, c);
    return mk((double)v.re, (double)v.im);
}

// element (r, c) of X, of its Hermitian part when flagged
template <bool HERM, typename T>
__device__ inline cplx<double> rot_x(const cplx<T>* X, int nw, int r, int c) {
    cplx<double> x = rot_elem(X, nw, r, c);
    if constexpr (HERM) {
        const cplx<double> w = rot_elem(X, nw, c, r);
        x = mk(0.5 * (x.re + w.re), 0.5 * (x.im - w.im));
    }
    return x;
}

// the two halves of rot_cmac: between them, other accumulators' products keep the matrix core busy
__device__ inline void rot_cmac_re(wbmi_v4d& re, wbmi_v4d& im, cplx<double> a, cplx<double> b) {
    re = __builtin_amdgcn_mfma_f64_16x16x4f64(a.re, b.re, re, 0, 0, 0);
    im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.re, b.im, im, 0, 0, 0);
}
__device__ inline void rot_cmac_im(wbmi_v4d& re, wbmi_v4d& im, cplx<double> a, cplx<double> b) {
    re = __builtin_amdgcn_mfma_f64_16x16x4f64(-a.im, b.im, re, 0, 0, 0);
    im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.im, b.re, im, 0, 0, 0);
}

__device__ inline void rot_cmac(wbmi_v4d& re, wbmi_v4d& im, cplx<double> a, cplx<double> b) {
    re = __builtin_amdgcn_mfma_f64_16x16x4f64(a.re, b.re, re, 0, 0, 0);
    re = __builtin_amdgcn_mfma_f64_16x16x4f64(-a.im, b.im, re, 0, 0, 0);
    im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.re, b.im, im, 0, 0, 0);
    im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.im, b.re, im, 0, 0, 0);
}

// nw <= 16 NB, NB = 1, 2: a wave rotates whole channels, in turn with the other waves of its k-point;
// U (FP64) in LDS, shared by the waves of a workgroup; steps past nw are left out.
// Bound at nw = 32: the channels' traffic (read and written once) next to the products, which take
// as long.  Measured against one LDS tile per wave (one workgroup of 8 waves a CU): 4096 k-points of 36
// channels at nw = 32 1.72 -> 1.50 ms complex128, 1.57 -> 1.40 complex64; 2500 of 9 at nw = 2 67 -> 19 us.
// (Registers: 8 waves a CU without spills at complex128, 12 at complex64.)
#define ROTR_WAVES 4
template <typename T, int NB>
__global__ void __launch_bounds__(64 * ROTR_WAVES, NB == 1 ? 4 : sizeof(T) == 8 ? 2 : 3) k_rotate_r(int nw, int nch, const cplx<T>* __restrict__ U,
                                                                             cplx<T>* X, uint64_t herm_lo,
                                                                             uint64_t herm_hi, uint64_t skip_lo,
                                                                             uint64_t skip_hi) {
    constexpr int NS = 4 * NB, LD = 16 * NB + 1;  // steps of the summed index, LDS row stride
    // complex64: in the order of the summed index, as above 64 bands, so that one element in 1e8 is not rounded the other
    // way by the kernel a size takes (J = 4 was no faster: 1.44 ms against 1.40 for 36 channels of 4096 k-points, nw = 32)
    constexpr int J = sizeof(T) == 8 ? 2 : 1;
    __shared__ cplx<double> sU[16 * NB * LD];
    const int lane = threadIdx.x & 63, li = lane & 15, g = lane >> 4;
    const int nwave = ROTR_WAVES * (int)gridDim.y, wave = (int)(threadIdx.x >> 6) + ROTR_WAVES * (int)blockIdx.y;
    const int64_t k = blockIdx.x;
    const int nw2 = nw * nw;
    const cplx<T>* Uk = U + k * nw2;
    for (int t = threadIdx.x; t < 256 * NB * NB; t += 64 * ROTR_WAVES)
        sU[t / (16 * NB) * LD + t % (16 * NB)] = rot_elem(Uk, nw, t / (16 * NB), t % (16 * NB));
    __syncthreads();
    int q = -1;
    for (int c = 0; c < nch; ++c) {
        // the wave's channels: those to rotate in turn over the waves of the k-point's workgroups
        if (bit_of(skip_lo, skip_hi, c) || ++q % nwave != wave) continue;
        cplx<T>* Xc = X + (k * nch + c) * nw2;
        const bool herm = bit_of(herm_lo, herm_hi, c);
        wbmi_v4d tr[NB][NB], ti[NB][NB];
#pragma unroll
        for (int bi = 0; bi < NB; ++bi) {
            // 16 rows of X as the A operand (its Hermitian part when flagged): step s of lane group g is
            // k = 4 J (s / J) + J g + s % J, J consecutive elements a lane (complex128: 128 bytes of a row per load group)
            cplx<T> x[NS], w[NS];
            const int r = 16 * bi + li;
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const int m = 4 * J * (s / J) + J * g + s % J;
                x[s] = r < nw && m < nw ? Xc[r * nw + m] : mk((T)0, (T)0);
            }
            if (herm) {
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const int m = 4 * J * (s / J) + J * g + s % J;
                    w[s] = r < nw && m < nw ? Xc[m * nw + r] : mk((T)0, (T)0);
                }
            }
#pragma unroll
            for (int bj = 0; bj < NB; ++bj) {
                tr[bi][bj] = wbmi_v4d{0.0, 0.0, 0.0, 0.0};
                ti[bi][bj] = tr[bi][bj];
            }
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                if (4 * J * (s / J) + s % J >= nw) continue;
                const int m = 4 * J * (s / J) + J * g + s % J;
                cplx<double> a = mk((double)x[s].re, (double)x[s].im);
                if (herm) a = mk(0.5 * (a.re + (double)w[s].re), 0.5 * (a.im - (double)w[s].im));
#pragma unroll
                for (int bj = 0; bj < NB; ++bj) rot_cmac(tr[bi][bj], ti[bi][bj], a, sU[m * LD + 16 * bj + li]);
            }
        }
#pragma unroll
        for (int bo = 0; bo < NB; ++bo)
#pragma unroll
            for (int bj = 0; bj < NB; ++bj) {
                wbmi_v4d re = {0.0, 0.0, 0.0, 0.0}, im = re;
#pragma unroll
                for (int s = 0; s < NS; ++s)
                    if (4 * s < nw)
                        rot_cmac(re, im, conj(sU[(4 * s + g) * LD + 16 * bo + li]), mk(tr[s / 4][bj][s % 4], ti[s / 4][bj][s % 4]));
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int r = 16 * bo + g + 4 * v, cc = 16 * bj + li;
                    if (r < nw && cc < nw) Xc[r * nw + cc] = mk((T)re[v], (T)im[v]);
                }
            }
    }
}

// 16 (NB - 1) < nw <= 16 NB, NB = 3 .. 8: one workgroup per (channel, k), one wave per strip of 16 columns:
// T's strip (16 NB x 16) stays in the wave's accumulators, every wave reads all of X and U (through L1 and L2),
// and a barrier separates the last read of X from the first store over it.
// Bound: the matrix cores (nw = 128: 2.3 ms at peak for 36 channels of 150 k-points) and the latency of
// the operand loads, which are branch-free and issued J steps at a time.  Measured against register tiles
// without matrix cores up to 64 and one workgroup per k-point with T through memory above: 3898 k-points of 9
// channels at nw = 48 4.74 -> 1.41 ms complex128, 3.31 -> 1.32 complex64; 150 of 35 at nw = 128 7.95 -> 4.22
// and 8.69 -> 3.90 ms.
template <typename T, int NB>
__global__ void __launch_bounds__(64 * NB, NB <= 4 ? 3 : 2) k_rotate_s(int nw, int nch, const cplx<T>* __restrict__ U, cplx<T>* X,
                                                       uint64_t herm_lo, uint64_t herm_hi, uint64_t skip_lo,
                                                       uint64_t skip_hi) {
    constexpr int NS = 4 * NB, J = NB > 4 && sizeof(T) == 4 ? 1 : 2;
    const int c = blockIdx.x;
    if (bit_of(skip_lo, skip_hi, c)) return;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, g = lane >> 4;
    const int64_t k = blockIdx.y;
    const int nw2 = nw * nw;
    const cplx<T>* Uk = U + k * nw2;
    cplx<T>* Xc = X + (k * nch + c) * nw2;
    const bool herm = bit_of(herm_lo, herm_hi, c);
    const int col = 16 * wave + li;
    wbmi_v4d tr[NB], ti[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        tr[b] = wbmi_v4d{0.0, 0.0, 0.0, 0.0};
        ti[b] = tr[b];
    }
    // J steps at a time, k = 4 J t + J g + j as in k_rotate_r
    auto first = [&](auto hermitian) {
#pragma unroll 1
        for (int t = 0; t < NS / J; ++t) {
            cplx<double> u[J], x[J][NB];
#pragma unroll
            for (int j = 0; j < J; ++j) {
                const int m = 4 * J * t + J * g + j;
                u[j] = rot_elem(Uk, nw, m, col);
#pragma unroll
                for (int b = 0; b < NB; ++b) x[j][b] = rot_x<decltype(hermitian)::value>(Xc, nw, 16 * b + li, m);
            }
#pragma unroll
            for (int j = 0; j < J; ++j) {
#pragma unroll
                for (int b = 0; b < NB; ++b) rot_cmac_re(tr[b], ti[b], x[j][b], u[j]);
#pragma unroll
                for (int b = 0; b < NB; ++b) rot_cmac_im(tr[b], ti[b], x[j][b], u[j]);
            }
        }
    };
    if (herm)
        first(std::true_type{});
    else
        first(std::false_type{});
    __syncthreads();
    // two row blocks at a time (four accumulators in turn)
    auto second = [&](int bo, auto two) {
        constexpr int NO = decltype(two)::value ? 2 : 1;
        wbmi_v4d re[NO], im[NO];
#pragma unroll
        for (int q = 0; q < NO; ++q) re[q] = im[q] = wbmi_v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            cplx<double> u[NO];
            const cplx<double> t = mk(tr[s / 4][s % 4], ti[s / 4][s % 4]);
#pragma unroll
            for (int q = 0; q < NO; ++q) u[q] = conj(rot_elem(Uk, nw, 4 * s + g, 16 * (bo + q) + li));
#pragma unroll
            for (int q = 0; q < NO; ++q) rot_cmac_re(re[q], im[q], u[q], t);
#pragma unroll
            for (int q = 0; q < NO; ++q) rot_cmac_im(re[q], im[q], u[q], t);
        }
#pragma unroll
        for (int q = 0; q < NO; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = 16 * (bo + q) + g + 4 * v;
                if (r < nw && col < nw) Xc[r * nw + col] = mk((T)re[q][v], (T)im[q][v]);
            }
    };
    for (int bo = 0; bo + 1 < NB; bo += 2) second(bo, std::true_type{});
    if constexpr (NB & 1) second(NB - 1, std::false_type{});
}

// complex64 in FP64 arithmetic at 32 < nw <= 64 (the mixed form's velocity): one 256-thread workgroup per k, U, X and T
// = X U in LDS, 4 x 4 register tiles and one FMA chain per element in the order of the summed index.  Slower than
// the matrix cores (3898 k-points at nw = 48: 356 us a channel against 146) and no more accurate; but the order of the
// sums decides the complex64 rounding of one element in 1e8, and in the velocity between two close bands
// the cut sums of DerMorb show it: with k_rotate_s here the gyrotropic tensor moves by up to 1.7e-9 of itself (more than
// 1e-10 in 6 of 150 models at nw = 64, without it 1).  So these sizes keep the order of this kernel, and those
// above 64 and below 33 that of the matrix cores; the channels that enter with one energy denominator less take k_rotate_s.
#define ROTV_THREADS 256
__device__ inline void rotv_product(int nw, int r0, int c0, cplx<double> (&acc)[4][4], const cplx<double>* sT, const cplx<float>* sU,
                                    const cplx<float>* sX, bool herm, bool second) {
    const int ld = nw + 1;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = mk(0.0, 0.0);
    for (int m = 0; m < nw; ++m) {
        cplx<double> x[4], y[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = min(r0 + i, nw - 1), c = min(c0 + i, nw - 1);
            const cplx<float> a = second ? sU[m * ld + r] : sX[r * ld + m];
            x[i] = mk((double)a.re, (double)a.im);
            if (!second && herm) {
                const cplx<float> w = sX[m * ld + r];
                x[i] = mk(0.5 * (x[i].re + (double)w.re), 0.5 * (x[i].im - (double)w.im));
            }
            if (second) {
                y[i] = sT[m * ld + c];
            } else {
                const cplx<float> u = sU[m * ld + c];
                y[i] = mk((double)u.re, (double)u.im);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (second) cfma_cj(acc[i][j], x[i], y[j]);
                else cfma(acc[i][j], x[i], y[j]);
            }
    }
}
__global__ void __launch_bounds__(ROTV_THREADS) k_rotate_v(int nw, int nch, const cplx<float>* __restrict__ U, cplx<float>* X,
                                                          uint64_t herm_lo, uint64_t herm_hi, uint64_t skip_lo, uint64_t skip_hi) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int ld = nw + 1, nw2 = nw * nw, tid = threadIdx.x;
    cplx<double>* sT = (cplx<double>*)smem;
    cplx<float>* sU = (cplx<float>*)(sT + nw * ld);
    cplx<float>* sX = sU + nw * ld;
    const int64_t k = blockIdx.x;
    const cplx<float>* Uk = U + k * nw2;
    const int r0 = 4 * (tid / 16), c0 = 4 * (tid % 16);
    const bool active = r0 < nw && c0 < nw;
    for (int t = tid; t < nw2; t += ROTV_THREADS) sU[(t / nw) * ld + t % nw] = Uk[t];
    for (int c = 0; c < nch; ++c) {
        if (bit_of(skip_lo, skip_hi, c)) continue;
        const bool herm = bit_of(herm_lo, herm_hi, c);
        cplx<float>* Xc = X + (k * nch + c) * nw2;
        for (int t = tid; t < nw2; t += ROTV_THREADS) sX[(t / nw) * ld + t % nw] = Xc[t];
        __syncthreads();
        cplx<double> acc[4][4];
        if (active) {
            rotv_product(nw, r0, c0, acc, sT, sU, sX, herm, false);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (r0 + i < nw && c0 + j < nw) sT[(r0 + i) * ld + c0 + j] = acc[i][j];
        }
        __syncthreads();
        if (active) {
            rotv_product(nw, r0, c0, acc, sT, sU, sX, herm, true);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (r0 + i < nw && c0 + j < nw) Xc[(r0 + i) * nw + c0 + j] = mk((float)acc[i][j].re, (float)acc[i][j].im);
        }
        __syncthreads();
    }
}

// Split-half rotation (complex64 storage, nw <= 32): Xbar = U^+ X U with both products
// on the fp16 matrix cores (v_mfma_f32_16x16x16_f16).  Each real operand is scaled by a
// power of two and split into two fp16 numbers, x = hi + lo (hi = fp16(x), lo = fp16(x - hi):
// 22 significant bits), and a product is Ah Bh + Ah Bl + Al Bh accumulated in FP32; the
// dropped Al Bl is 2^-22 of the terms.  So a product carries FP32-accumulation rounding,
// eps32 sqrt(nw) |X| |U| per element, where the FP64-arithmetic path carries only the
// rounding of the stored result.  Used for every channel but the velocity dH/dk (whose
// elements between close bands enter the Berry curvature through 1/(E_n - E_m)^2).
//
// One wave per (k, channel), no LDS and no barriers: X is loaded from HBM straight into
// the A-operand registers, U (split once per k) serves as the B operand of T = X U and,
// conjugated, as the A operand of U^+ T, and the accumulators of T are the B operand of
// the second product.  That last step relies on the output layout of the 16 x 16 MFMA:
// lane l, register v holds D[RH_ROW(l / 16, v)][l % 16], so the k index of every operand
// is enumerated in that same order (any order common to A and B gives the same sum).
typedef _Float16 wbmi_h4 __attribute__((ext_vector_type(4)));
typedef float wbmi_f4 __attribute__((ext_vector_type(4)));
#define ROTH_WAVES 4
#define RH_ROW(g, v) (4 * (g) + (v))

struct SplitH {
    wbmi_h4 hi, lo;
};

__device__ inline SplitH split_h(const float* x, float s) {
    SplitH r;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float v = x[j] * s;
        const _Float16 h = (_Float16)v;
        r.hi[j] = h;
        r.lo[j] = (_Float16)(v - (float)h);
    }
    return r;
}

__device__ inline wbmi_h4 neg_h(wbmi_h4 a) { return -a; }

// acc += (Ah + Al)(Bh + Bl) without Al Bl
__device__ inline wbmi_f4 mfma3(const SplitH& a, const SplitH& b, wbmi_f4 acc) {
    acc = __builtin_amdgcn_mfma_f32_16x16x16f16(a.hi, b.hi, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x16f16(a.hi, b.lo, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_16x16x16f16(a.lo, b.hi, acc, 0, 0, 0);
    return acc;
}

__device__ inline SplitH neg_split(const SplitH& a) { return SplitH{neg_h(a.hi), neg_h(a.lo)}; }

// (4 waves per SIMD: the accumulators in VGPRs rather than AGPRs, 128 registers in all)
__global__ void __launch_bounds__(64 * ROTH_WAVES, 4) k_rotate_h(int nw, int nch, const cplx<float>* __restrict__ U,
                                                             cplx<float>* X, uint64_t herm_lo, uint64_t herm_hi,
                                                             uint64_t skip_lo, uint64_t skip_hi) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = lane & 15, g = lane >> 4;
    const int64_t k = blockIdx.x;
    const int nw2 = nw * nw;
    const cplx<float>* Uk = U + k * nw2;
    // U as the B operand of X U: block (ks, bj) holds U[16 ks + RH_ROW(g, j)][16 bj + li]; the same
    // registers are the A operand of U^+ T for output row block bj (conjugated)
    const float su = 16384.f;
    SplitH ur[2][2], ui[2][2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int bj = 0; bj < 2; ++bj) {
            float re[4], im[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int m = 16 * ks + RH_ROW(g, j), c = 16 * bj + li;
                const cplx<float> u = (m < nw && c < nw) ? Uk[m * nw + c] : mk(0.f, 0.f);
                re[j] = u.re;
                im[j] = u.im;
            }
            ur[ks][bj] = split_h(re, su);
            ui[ks][bj] = split_h(im, su);
        }
    // the waves take the channels to rotate in turn (rotation index q = wave, wave + ROTH_WAVES, ...)
    int q = -1;
    for (int ch = 0; ch < nch; ++ch) {
        if (bit_of(skip_lo, skip_hi, ch)) continue;
        if (++q % ROTH_WAVES != wave) continue;
        cplx<float>* Xc = X + (k * nch + ch) * nw2;
        const bool herm = bit_of(herm_lo, herm_hi, ch);
        // X as the A operand: block (bi, ks) holds X[16 bi + li][16 ks + RH_ROW(g, j)], four
        // consecutive elements of a row (at nw = 32 two 16-byte loads: the row offset is a
        // multiple of 4 elements and a channel starts 8 KB-aligned)
        float xre[2][2][4], xim[2][2][4];
#pragma unroll
        for (int bi = 0; bi < 2; ++bi)
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                const int r = 16 * bi + li, m0 = 16 * ks + RH_ROW(g, 0);
                if (nw == 32) {
                    const float4* p = (const float4*)(Xc + r * 32 + m0);
                    const float4 a = p[0], b = p[1];
                    xre[bi][ks][0] = a.x; xim[bi][ks][0] = a.y; xre[bi][ks][1] = a.z; xim[bi][ks][1] = a.w;
                    xre[bi][ks][2] = b.x; xim[bi][ks][2] = b.y; xre[bi][ks][3] = b.z; xim[bi][ks][3] = b.w;
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const cplx<float> x = (r < nw && m0 + j < nw) ? Xc[r * nw + m0 + j] : mk(0.f, 0.f);
                        xre[bi][ks][j] = x.re;
                        xim[bi][ks][j] = x.im;
                    }
                }
                if (herm) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int m = m0 + j;
                        const cplx<float> w = (r < nw && m < nw) ? Xc[m * nw + r] : mk(0.f, 0.f);
                        xre[bi][ks][j] = 0.5f * (xre[bi][ks][j] + w.re);
                        xim[bi][ks][j] = 0.5f * (xim[bi][ks][j] - w.im);
                    }
                }
            }
        float mx = 0.f;
#pragma unroll
        for (int bi = 0; bi < 2; ++bi)
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int j = 0; j < 4; ++j) mx = fmaxf(mx, fmaxf(fabsf(xre[bi][ks][j]), fabsf(xim[bi][ks][j])));
        for (int o = 32; o >= 1; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
        // scale: max |x| s < 2^14 (fp16 holds up to 65504)
        int e = 0;
        frexpf(mx, &e);
        const float sx = mx > 0.f ? ldexpf(1.f, 14 - e) : 1.f;
        SplitH xr[2][2], xi[2][2];
#pragma unroll
        for (int bi = 0; bi < 2; ++bi)
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                xr[bi][ks] = split_h(xre[bi][ks], sx);
                xi[bi][ks] = split_h(xim[bi][ks], sx);
            }
        // T = X U:  Tr = Xr Ur - Xi Ui,  Ti = Xr Ui + Xi Ur   (scaled by sx su)
        wbmi_f4 tr[2][2], ti[2][2];
#pragma unroll
        for (int bi = 0; bi < 2; ++bi)
#pragma unroll
            for (int bj = 0; bj < 2; ++bj) {
                wbmi_f4 ar = {0.f, 0.f, 0.f, 0.f}, ai = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) {
                    ar = mfma3(xr[bi][ks], ur[ks][bj], ar);
                    ar = mfma3(neg_split(xi[bi][ks]), ui[ks][bj], ar);
                    ai = mfma3(xr[bi][ks], ui[ks][bj], ai);
                    ai = mfma3(xi[bi][ks], ur[ks][bj], ai);
                }
                tr[bi][bj] = ar;
                ti[bi][bj] = ai;
            }
        // T as the B operand of U^+ T: block (ks = bi, bj), element j = v; scale st = sx / 8
        // (|T| <= sqrt(nw) max|X| < 8 max|X|), i.e. the accumulators times 1 / (8 su)
        SplitH bre[2][2], bim[2][2];
        const float tsc = 1.f / (8.f * su);
#pragma unroll
        for (int bi = 0; bi < 2; ++bi)
#pragma unroll
            for (int bj = 0; bj < 2; ++bj) {
                float vr[4], vi[4];
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    vr[v] = tr[bi][bj][v];
                    vi[v] = ti[bi][bj][v];
                }
                bre[bi][bj] = split_h(vr, tsc);
                bim[bi][bj] = split_h(vi, tsc);
            }
        // Xbar = U^+ T: rows bo; A = conj(U)^T: Ar = Ur^T, Ai = -Ui^T
        //   Xr = Ur^T Tr + Ui^T Ti,  Xi = Ur^T Ti - Ui^T Tr   (scaled by su sx / 8)
        const float osc = 8.f / (su * sx);
#pragma unroll
        for (int bo = 0; bo < 2; ++bo)
#pragma unroll
            for (int bj = 0; bj < 2; ++bj) {
                wbmi_f4 ar = {0.f, 0.f, 0.f, 0.f}, ai = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < 2; ++ks) {
                    ar = mfma3(ur[ks][bo], bre[ks][bj], ar);
                    ar = mfma3(ui[ks][bo], bim[ks][bj], ar);
                    ai = mfma3(ur[ks][bo], bim[ks][bj], ai);
                    ai = mfma3(neg_split(ui[ks][bo]), bre[ks][bj], ai);
                }
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int r = 16 * bo + RH_ROW(g, v), cc = 16 * bj + li;
                    if (r < nw && cc < nw) Xc[r * nw + cc] = mk(ar[v] * osc, ai[v] * osc);
                }
            }
    }
}

// no kernel of the rotation needs a workspace
extern "C" size_t wbmi_rotate_work_bytes(int nk, int nw, int prec) {
    (void)nk;
    (void)nw;
    (void)prec;
    return 0;
}

template <typename T, int NB>
static int launch_rotate_nb(wbmi_ctx* ctx, int nk, int nw, int nch, const void* U_dev, void* X_dev, const uint64_t* h,
                            const uint64_t* s) {
    if constexpr (NB <= 2) {
        // few k-points: their channels over several workgroups, about four per CU
        int nrot = 0;
        for (int c = 0; c < nch; ++c) nrot += !bit_of(s[0], s[1], c);
        int parts = (nrot + ROTR_WAVES - 1) / ROTR_WAVES;
        parts = nk >= 1024 || parts < 1 ? 1 : parts < 1024 / nk ? parts : 1024 / nk;
        hipLaunchKernelGGL((k_rotate_r<T, NB>), dim3(nk, parts), dim3(64 * ROTR_WAVES), 0, ctx->stream, nw, nch,
                           (const cplx<T>*)U_dev, (cplx<T>*)X_dev, h[0], h[1], s[0], s[1]);
        WBMI_LAUNCH_CHECK(ctx);
    } else {
        // k-points over gridDim.y, at most 65535 per launch
        for (int k0 = 0; k0 < nk; k0 += 65535) {
            const int n = nk - k0 < 65535 ? nk - k0 : 65535;
            hipLaunchKernelGGL((k_rotate_s<T, NB>), dim3(nch, n), dim3(64 * NB), 0, ctx->stream, nw, nch,
                               (const cplx<T>*)U_dev + (int64_t)k0 * nw * nw, (cplx<T>*)X_dev + (int64_t)k0 * nch * nw * nw,
                               h[0], h[1], s[0], s[1]);
            WBMI_LAUNCH_CHECK(ctx);
        }
    }
    return WBMI_OK;
}

template <typename T>
static int launch_rotate(wbmi_ctx* ctx, int nk, int nw, int nch, const void* U_dev, void* X_dev, const uint64_t* h,
                         const uint64_t* s) {
    switch ((nw + 15) / 16) {
        case 1: return launch_rotate_nb<T, 1>(ctx, nk, nw, nch, U_dev, X_dev, h, s);
        case 2: return launch_rotate_nb<T, 2>(ctx, nk, nw, nch, U_dev, X_dev, h, s);
        case 3: return launch_rotate_nb<T, 3>(ctx, nk, nw, nch, U_dev, X_dev, h, s);
        case 4: return launch_rotate_nb<T, 4>(ctx, nk, nw, nch, U_dev, X_dev, h, s);
        case 5: return launch_rotate_nb<T, 5>(ctx, nk, nw, nch, U_dev, X_dev, h, s);
        case 6: return launch_rotate_nb<T, 6>(ctx, nk, nw, nch, U_dev, X_dev, h, s);
        case 7: return launch_rotate_nb<T, 7>(ctx, nk, nw, nch, U_dev, X_dev, h, s);
        default: return launch_rotate_nb<T, 8>(ctx, nk, nw, nch, U_dev, X_dev, h, s);
    }
}

extern "C" int wbmi_rotate(wbmi_ctx* ctx, int nk, int nw, int nch, const void* U_dev, void* X_dev,
                           const int32_t* herm_host, const int32_t* skip_host, int prec, void* work_dev,
                           size_t work_bytes) {
    if (!ctx) return WBMI_ERR_ARG;
    if (nk <= 0 || nw <= 0 || nw > 128 || nch <= 0 || nch > 128 || !U_dev || !X_dev)
        return wbmi_fail(ctx, WBMI_ERR_ARG, "wbmi_rotate: bad arguments (nw <= 128, nch <= 128)");
    (void)work_dev;
    (void)work_bytes;
    uint64_t h[2] = {0, 0}, s[2] = {0, 0};
    for (int c = 0; c < nch; ++c) {
        if (herm_host && herm_host[c]) h[c / 64] |= 1ull << (c % 64);
        if (skip_host && skip_host[c]) s[c / 64] |= 1ull << (c % 64);
    }
    if (prec == WBMI_F64) return launch_rotate<double>(ctx, nk, nw, nch, U_dev, X_dev, h, s);
    if (prec == WBMI_F32 && nw > 32 && nw <= 64) {
        const size_t lds = (sizeof(cplx<double>) + 2 * sizeof(cplx<float>)) * nw * (nw + 1);
        WBMI_HIP_CHECK(ctx, hipFuncSetAttribute((const void*)k_rotate_v, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        hipLaunchKernelGGL(k_rotate_v, dim3(nk), dim3(ROTV_THREADS), lds, ctx->stream, nw, nch, (const cplx<float>*)U_dev,
                           (cplx<float>*)X_dev, h[0], h[1], s[0], s[1]);
        WBMI_LAUNCH_CHECK(ctx);
        return WBMI_OK;
    }
    if (prec == WBMI_F32) return launch_rotate<float>(ctx, nk, nw, nch, U_dev, X_dev, h, s);
    if (prec == WBMI_F32_SPLIT) {
        if (nw > 32)  // above one 32 x 32 block per operand: the FP64-arithmetic path
            return launch_rotate<float>(ctx, nk, nw, nch, U_dev, X_dev, h, s);
        hipLaunchKernelGGL(k_rotate_h, dim3(nk), dim3(64 * ROTH_WAVES), 0, ctx->stream, nw, nch,
                           (const cplx<float>*)U_dev, (cplx<float>*)X_dev, h[0], h[1], s[0], s[1]);
        WBMI_LAUNCH_CHECK(ctx);
        return WBMI_OK;
    }
    return wbmi_fail(ctx, WBMI_ERR_ARG, "wbmi_rotate: bad precision");
}
