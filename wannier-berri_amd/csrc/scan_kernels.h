// Covariant formula traces + Fermi-level scan of libwbmi.
//
// Replaces the per-(k, band group) loop of StaticCalculator.__call__
// (calculators/static.py:60-136).  One workgroup per k-point, several where few
// k-points leave the GPU idle (launch_scan_t), of a size per formula and nw
// (launch_scan); the formula is a template parameter, so every calculator gets
// its own kernel.
//
// Band partition.  The reference evaluates, for every band group G, the
// formula with inn = G and out = all other bands.  Every sum in the formulas
// is then either over l in out (l not in G) or over n' in G, so with a label
// per band (lab[x] = group of x) the traces of ALL groups come from one set
// of per-band values v_n, n in G, using the masks
//     Off(x, y) = lab[x] != lab[y]      (x, y in different groups)
//     On(x, y)  = lab[x] == lab[y]
// and the masked matrices
//     D'^a = -V^a o M,  M = dEinv o Off,  V'' = V o On,  A'' = A o On.
// The Fermi-sea group (all bands below EFmin, data_K.py:178-185) and the
// cumulative cuts [0, c) of non-additive formulas (static.py:109-117) are
// two-set partitions evaluated the same way.
//
// DerOmega.  With G^{bd} = V^b D'^d and K^{bd} = A^b D'^d,
//   dD.ln = X1^{bd} = -M o [W^{bd} + G^{bd} + G^{db} - D'^b V''^d - D'^d V''^b]
//   dD.nl = X2^{ad}, X2^{ad}_nl = -conj(X1^{ad}_ln)   (V, W Hermitian, D' anti-Hermitian)
//   dA.ln = Y1^{bd} = A'^{bd} - D'^d A''^b + K^{bd}
// (formula/elementary.py:63-70, formula/formula.py:108-118).  X1 is symmetric
// in (b, d), so the elementwise terms are folded half-and-half into each
// product: Q1 = G + (W - S)/2, Y1 = K + A' - D'A''.
// The traces use only diagonal elements of D'^a X1, X2 A^b and D'^a Y1, so
// every product element is consumed where it is computed: a wave task forms
// one 16 x 32 block of one of the products on the FP64 matrix cores, adds the
// elementwise terms, multiplies by the consumer weights, reduces over the
// summed index with cross-lane shuffles and adds the result to the per-band
// rows with LDS atomics.  The waves take tasks from an LDS counter.  No
// product is stored and no barrier separates them.
//
// For DerOmega the operands V and A stay in LDS (rows padded by one element)
// when nw <= 32.
// All arithmetic is FP64 (energies, dEinv, traces, histogram); channels may
// be stored in FP32 or FP64.
#pragma once

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "mfma_c64.h"
#include "wbmi_common.h"

#define SC_THREADS 512  // workgroup size of the scan kernels (others: launch_scan)
#define SC_NWMAX 128
#define SC_LDS (160 * 1024)
#define SC_XCD_LOG 3
#define SC_XCD (1 << SC_XCD_LOG)
#define SC_M_NW 64    // dEinv o Off lives in LDS up to this nw (DerOmega / DerMorb: wherever it fits)
#define SC_LDS_NW 32  // V and A live in LDS up to this nw
// DerMorb with internal terms only: kernels of their own, for V and W Hermitian to the rounding of FP64
// sums, and for complex64 channels
#define SC_DERMORB_IN (WBMI_FORMULA_OMEGAHPLUS + 1000)
#define SC_DERMORB_IN32 (SC_DERMORB_IN + 1)
#define SC_DERMORB_EX (SC_DERMORB_IN + 2)  // with external terms, sign = +1, complex128
#define SC_IS_DERMORB_IN(F) ((F) == SC_DERMORB_IN || (F) == SC_DERMORB_IN32)
#define SC_IS_DERMORB_CUTS(F) (SC_IS_DERMORB_IN(F) || (F) == SC_DERMORB_EX)

static __constant__ int c_alpha[3] = {1, 2, 0};  // utility.py:45-46
static __constant__ int c_beta[3] = {2, 0, 1};

struct ScanArgs {
    wbmi_scan_params p;
    int nw, nch, stage_va;
    int nk, parts;  // workgroups per k-point, set at the launch
    double weight;
    // tetrahedron method: `tetra` = number of corners, 8 (parallelepiped: corner ix*4 + iy*2 + iz
    // at k + (2i-1) dK/2, 12 tetrahedra around the centre) or 4 (tetrahedral K-block: the vertices,
    // one tetrahedron); corner energies [tetra][nk][nw], ascending Fermi levels Ef[nEF]; hist holds
    // nEF step rows (prefix-summed later) followed by nEF rows added as they are
    int tetra, nEF;
    const double* Ec;
    int64_t ec_stride;
    const double* Ef;
    // k-resolved scans: k-point k accumulates into hist + k * hist_stride (0: one histogram)
    int64_t hist_stride;
};

// dynamic shared-memory layout
struct Smem {
    char* V;            // [3][nw][ld] staged V (elements as stored)
    char* A;            // [3][nw][ld] staged A (external terms)
    double* acc;        // [nw][9] per-band values of the partition
    double* M;          // [nw][ld] dEinv o Off
    double* E;
    double* cut;        // [nw+1][9]
    double* gw;         // group weights (mean energy)
    int* lab;
    int* gs;
    int* ge;
    int* act;
    int* gb;    // group borders [nw+1]
    int* gin;   // group in range
    int* misc;  // [0] = ngroups, [1], [2] = sea group [lo, hi) (empty: lo == hi)
    int* ch;    // channel slot per role [WBMI_NROLES]
    int* need;  // non-additive formulas: cut to be evaluated [nw+1]
    // tetrahedron method only (empty regions otherwise)
    double* tC;    // [nw][8] corner energies
    double* tEmn;  // [nw] min over centre and corners
    double* tEmx;  // [nw] max over centre and corners
    double* tv;    // [nw+1][9] group values
    int* tg;       // [nw] group of each band
    int* tlo;      // [nw] first Fermi level of the band's partial range
    int* tcnt;     // [nw] length of that range
    int* tpre;     // [nw+1] prefix sums of tcnt
};

__host__ __device__ inline size_t al16(size_t x) { return (x + 15) & ~(size_t)15; }

// byte offsets of the LDS regions and their total size
struct SmemOffsets {
    size_t V, A, acc, M, E, cut, gw, ints, tet, tints, total;
};

// vsz: bytes of one staged V / A element
__host__ __device__ inline SmemOffsets smem_offsets(int nw, bool lm, bool stage_v, bool stage_a, bool tetra, size_t vsz) {
    const size_t ld = nw + 1;
    SmemOffsets o;
    size_t off = 0;
    o.V = off;
    off = al16(off + (stage_v ? vsz * 3 * nw * ld : 0));
    o.A = off;
    off = al16(off + (stage_a ? vsz * 3 * nw * ld : 0));
    o.acc = off;
    off = al16(off + sizeof(double) * nw * 9);
    o.M = off;
    off = al16(off + (lm ? sizeof(double) * nw * ld : 0));
    o.E = off;
    off = al16(off + sizeof(double) * nw);
    o.cut = off;
    off = al16(off + sizeof(double) * (nw + 1) * 9);
    o.gw = off;
    off = al16(off + sizeof(double) * nw);
    o.ints = off;
    off = al16(off + sizeof(int) * (7 * nw + 2 + 4 + WBMI_NROLES));
    o.tet = off;
    off = al16(off + (tetra ? sizeof(double) * (8 * nw + 2 * nw + (nw + 1) * 9) : 0));
    o.tints = off;
    off = al16(off + (tetra ? sizeof(int) * (4 * nw + 1) : 0));
    o.total = off;
    return o;
}

__device__ __attribute__((always_inline)) inline Smem make_smem(char* base, int nw, bool lm, bool stage_v,
                                                                bool stage_a, bool tetra, size_t vsz) {
    const SmemOffsets o = smem_offsets(nw, lm, stage_v, stage_a, tetra, vsz);
    Smem s;
    // LDS addresses even where a region is empty (never read then): no null tests on LDS pointers
    s.V = base + o.V;
    s.A = base + o.A;
    s.acc = (double*)(base + o.acc);
    s.M = (double*)(base + o.M);  // empty region (never read) without LM
    s.E = (double*)(base + o.E);
    s.cut = (double*)(base + o.cut);
    s.gw = (double*)(base + o.gw);
    int* q = (int*)(base + o.ints);
    s.lab = q;
    s.gs = q + nw;
    s.ge = q + 2 * nw;
    s.act = q + 3 * nw;
    s.gb = q + 4 * nw;
    s.gin = q + 5 * nw + 1;
    s.misc = q + 6 * nw + 1;
    s.ch = q + 6 * nw + 5;
    s.need = q + 6 * nw + 5 + WBMI_NROLES;
    double* t = (double*)(base + o.tet);
    s.tC = t;
    s.tEmn = t + 8 * nw;
    s.tEmx = t + 9 * nw;
    s.tv = t + 10 * nw;
    int* ti = (int*)(base + o.tints);
    s.tg = ti;
    s.tlo = ti + nw;
    s.tcnt = ti + 2 * nw;
    s.tpre = ti + 3 * nw;
    return s;
}

// Element access to the channels of one k-point.
// LM: dEinv o Off read from LDS (nw <= SC_M_NW) or formed from E and the labels.
// ST: V read from its LDS copy (DerOmega and DerMorb at nw <= SC_LDS_NW) or from the
// channels; SA: the same for A (staged together with V, and only with external terms, the only
// case that reads it).
// Both are compile-time so that every access is a plain LDS or global load.
template <typename T, bool LM, bool ST, bool SA, int NW = 0>
struct KCtx {
    const cplx<T>* X;  // channels of this k: [nch][nw][nw]
    int nw, ld;  // run-time size (NW = 0); NW > 0 fixes both at compile time
    __device__ inline int n_() const {
        if constexpr (NW > 0) return NW;
        else return nw;
    }
    __device__ inline int ld_() const {
        if constexpr (NW > 0) return NW + 1;
        else return ld;
    }
    const int* ch;
    const double* E;
    const double* M;  // dEinv o Off, row stride ld
    const int* lab;
    const int* gs;
    const int* ge;
    const cplx<T>* sV;  // LDS copies of V and A (ST)
    const cplx<T>* sA;
    const double* bv;    // WBMI_FORMULA_BANDVALUES: this k's caller values [nw][nbv]
    int nbv;
    int part, parts;  // this workgroup's share of the k-point's tasks
    __device__ inline cplx<double> get(int role, int x, int y) const {
        cplx<T> v = X[((int64_t)ch[role] * n_() + x) * n_() + y];
        return mk((double)v.re, (double)v.im);
    }
    // the same for a role that is the same in every lane: one scalar base, one 32-bit offset for all roles
    __device__ inline cplx<double> getu(int role, int x, int y) const {
        const cplx<T>* p = X + (int64_t)__builtin_amdgcn_readfirstlane(ch[role]) * n_() * n_();
        const cplx<T> v = p[(unsigned)(x * n_() + y)];
        return mk((double)v.re, (double)v.im);
    }
    __device__ inline cplx<double> Vu(int a, int x, int y) const {
        if constexpr (ST) return V(a, x, y);
        else return getu(WBMI_ROLE_V + a, x, y);
    }
    __device__ inline cplx<double> Au(int a, int x, int y) const {
        if constexpr (SA) return A(a, x, y);
        else return getu(WBMI_ROLE_A + a, x, y);
    }
    __device__ inline cplx<double> V(int a, int x, int y) const {
        if constexpr (ST) {
            const cplx<T> v = sV[(a * n_() + x) * ld_() + y];
            return mk((double)v.re, (double)v.im);
        } else {
            return get(WBMI_ROLE_V + a, x, y);
        }
    }
    __device__ inline cplx<double> A(int a, int x, int y) const {
        if constexpr (SA) {
            const cplx<T> v = sA[(a * n_() + x) * ld_() + y];
            return mk((double)v.re, (double)v.im);
        } else {
            return get(WBMI_ROLE_A + a, x, y);
        }
    }
    __device__ inline cplx<double> W(int a, int b, int x, int y) const { return get(WBMI_ROLE_W + 3 * a + b, x, y); }
    __device__ inline cplx<double> Ad(int a, int d, int x, int y) const { return get(WBMI_ROLE_AD + 3 * a + d, x, y); }
    __device__ inline cplx<double> O(int c, int x, int y) const { return get(WBMI_ROLE_O + c, x, y); }
    __device__ inline cplx<double> Od(int c, int d, int x, int y) const { return get(WBMI_ROLE_OD + 3 * c + d, x, y); }
    __device__ inline cplx<double> B(int a, int x, int y) const { return get(WBMI_ROLE_B + a, x, y); }
    __device__ inline cplx<double> C(int a, int x, int y) const { return get(WBMI_ROLE_C + a, x, y); }
    __device__ inline cplx<double> Bd(int a, int d, int x, int y) const { return get(WBMI_ROLE_BD + 3 * a + d, x, y); }
    __device__ inline cplx<double> Cd(int c, int d, int x, int y) const { return get(WBMI_ROLE_CD + 3 * c + d, x, y); }
    __device__ inline cplx<double> S(int b, int x, int y) const { return get(WBMI_ROLE_S + b, x, y); }
    __device__ inline cplx<double> Sd(int b, int d, int x, int y) const { return get(WBMI_ROLE_SD + 3 * b + d, x, y); }
    // X o On: elements between bands of the same group
    __device__ inline cplx<double> Ainu(int a, int x, int y) const { return lab[x] == lab[y] ? Au(a, x, y) : mk(0.0, 0.0); }
    __device__ inline cplx<double> Vinu(int a, int x, int y) const { return lab[x] == lab[y] ? Vu(a, x, y) : mk(0.0, 0.0); }
    // dEinv_xy Off(x, y) (data_K.py:290-298): from LDS, or formed from E and the labels
    __device__ inline double m(int x, int y) const {
        if constexpr (LM) {
            return M[x * ld_() + y];
        } else {
            const double de = E[x] - E[y];
            return (lab[x] != lab[y] && fabs(de) >= 1e-7) ? 1.0 / de : 0.0;
        }
    }
    // D'^a_xy = -V^a_xy dEinv_xy Off(x, y)  (branch-free: M = 0 gives an exact zero for finite V)
    __device__ inline cplx<double> Dp(int a, int x, int y) const { return (-m(x, y)) * V(a, x, y); }
    __device__ inline cplx<double> Dpu(int a, int x, int y) const { return (-m(x, y)) * Vu(a, x, y); }
};

// pre-Hermitian Omega summand s^c_xy for x, y in the same group
// (formula/covariant.py:175-200): Omega.nn = s + s^+
template <typename T, bool LM, bool ST, bool SA, int NW>
__device__ __attribute__((always_inline)) cplx<double> omega_s(const KCtx<T, LM, ST, SA, NW>& K, int c, int x, int y, bool internal, bool external) {
    const int al = c_alpha[c], be = c_beta[c];
    cplx<double> s = mk(0.0, 0.0);
    for (int l = 0; l < K.n_(); ++l) {
        if (K.lab[l] == K.lab[x]) continue;
        cplx<double> dxa = K.Dp(al, x, l);
        if (internal) s += times_i(-(dxa * K.Dp(be, l, y)));
        if (external) s += K.Dp(be, x, l) * K.A(al, l, y) - dxa * K.A(be, l, y);
    }
    if (external) {
        for (int m = K.gs[x]; m < K.ge[x]; ++m) s += times_i(-(K.A(al, x, m) * K.A(be, m, y)));
        s += 0.5 * K.O(c, x, y);
    }
    return s;
}

// pre-Hermitian Morb_H summand h^c_xy for x, y in the same group
// (formula/covariant.py:390-414)
template <typename T, bool LM, bool ST, bool SA, int NW>
__device__ __attribute__((always_inline)) cplx<double> morbh_s(const KCtx<T, LM, ST, SA, NW>& K, int c, int x, int y, bool internal, bool external) {
    const int al = c_alpha[c], be = c_beta[c];
    cplx<double> s = mk(0.0, 0.0);
    for (int l = 0; l < K.n_(); ++l) {
        if (K.lab[l] == K.lab[x]) continue;
        cplx<double> dxa = K.Dp(al, x, l);
        if (internal) s += times_i(-(K.E[l] * (dxa * K.Dp(be, l, y))));
        if (external) s += K.Dp(be, x, l) * K.B(al, l, y) - dxa * K.B(be, l, y);
    }
    if (external) {
        for (int m = K.gs[x]; m < K.ge[x]; ++m) s += times_i(-(K.E[m] * (K.A(al, x, m) * K.A(be, m, y))));
        s += 0.5 * K.C(c, x, y);
    }
    return s;
}

// Group block of the inverse effective mass (formula/elementary.py:28-33 through
// formula/formula.py:95-107 with A = V, dA = W): for x, y in one band group,
//   M^{bd}_xy = W^{bd}_xy - sum_{l off} D^d_xl V^b_ly + sum_{l off} V^b_xl D^d_ly
// (D' carries the off-group mask, so the sums run over every l).
template <typename T, bool LM, bool ST, bool SA, int NW>
__device__ __attribute__((always_inline)) cplx<double> mass_xy(const KCtx<T, LM, ST, SA, NW>& K, int b, int d, int x,
                                                               int y) {
    cplx<double> v = K.W(b, d, x, y);
    for (int l = 0; l < K.n_(); ++l) {
        v -= K.Dp(d, x, l) * K.V(b, l, y);
        v += K.V(b, x, l) * K.Dp(d, l, y);
    }
    return v;
}

// Contraction of a rank-4 product X[a][b][c][d] to the Hall tensor [j][i]
// (calculators/static.py:419-423): 0.5 sum over (a, b) = (al_j, be_j) (+), (be_j, al_j) (-)
// and (c, d) = (be_i, al_i) (+), (al_i, be_i) (-).  `term(a, b, c, d)` gives X.
template <typename Fn>
__device__ __attribute__((always_inline)) cplx<double> hall_contract(int j, int i, Fn term) {
    const int aj = c_alpha[j], bj = c_beta[j], ai = c_alpha[i], bi = c_beta[i];
    cplx<double> v = term(aj, bj, bi, ai);
    v -= term(aj, bj, ai, bi);
    v -= term(bj, aj, bi, ai);
    v += term(bj, aj, ai, bi);
    return mk(0.5 * v.re, 0.5 * v.im);
}

template <int F>
__host__ __device__ constexpr int ncomp_of() {
    return F == WBMI_FORMULA_IDENTITY ? 1
           : (F == WBMI_FORMULA_OMEGA || F == WBMI_FORMULA_MORB_HPM || F == WBMI_FORMULA_SPIN) ? 3
                                                                                                : 9;
}

template <int F>
__host__ __device__ constexpr bool uses_A() {
    return F == WBMI_FORMULA_OMEGA || F == WBMI_FORMULA_DEROMEGA || F == WBMI_FORMULA_VELOMEGA ||
           F == WBMI_FORMULA_MORB_HPM || F == WBMI_FORMULA_VELHPLUS || F == WBMI_FORMULA_DERMORB ||
           F == WBMI_FORMULA_OMEGASPIN || F == WBMI_FORMULA_OMEGAOMEGA || F == WBMI_FORMULA_OMEGAHPLUS;
}

// build M = dEinv o Off for the current labels (data_K.py:290-298), or dEinv itself (the cut
// partitions: one matrix for all of them, their sums run over the off-side bands alone)
template <bool MASKED>
__device__ __attribute__((always_inline)) void build_M(const Smem& S, int nw) {
    const int ld = nw + 1;
    for (int t = threadIdx.x; t < nw * nw; t += (int)blockDim.x) {
        int x = t / nw, y = t % nw;
        double m = 0.0;
        if (!MASKED || S.lab[x] != S.lab[y]) {
            double de = S.E[x] - S.E[y];
            if (fabs(de) >= 1e-7) m = 1.0 / de;
        }
        S.M[x * ld + y] = m;
    }
}

// sum of v over the lanes of a wave that differ only in the lane bits of `mask`
__device__ inline double wave_sum(double v, int mask) {
    for (int b = 1; b < 64; b <<= 1)
        if (mask & b) v += __shfl_xor(v, b);
    return v;
}

// Wave tasks.  One wave forms the 16-row x 32-column block (rh, cb) of a dense product
// P = X Y on the matrix cores (FP64 MFMA, mfma_c64.h), adds the elementwise terms of
// each element (x, y) and accumulates the consumers' weighted elements into
// the workgroup's per-band rows acc[band][comp] (LDS FP64 atomic adds, .re) after a
// shuffle reduction over the summed index.  The band of an element is its column y (kind 1 forms its
// product transposed for this).  Kinds (task indices b, d; for kinds 5, 6 b = c):
//   0  Q1^{bd} = V^b D'^d + (W - D'^b V''^d - D'^d V''^b)/2, y in the partition, x off-side, so that
//      X1^{bd} = dD.ln = -M o (Q1^{bd} + Q1^{db}).  V and W Hermitian and D' anti-Hermitian give
//      dD.nl = X2^{ad}_yx = -conj(X1^{ad}_xy), so every term that holds dD, from the left or from
//      the right, is Re q^a_yx X1^{bd}_xy with one weight per partner a:
//        q^a = -i w D'^a_yx - dw conj(A^a_xy) - 2 conj(B^a_xy)
//      (DerOmega T1 and T3; DerMorb s2 in w, s7); DerMorb s1 reads the raw V^b D'^d
//   2  Y1^{bd} = A^b D'^d + A' - D'^d A''^b, x off-side: DerOmega T2;
//      x same-side (DerMorb): s5 terms of A' + A^b D'^d
//   3  YB^{bd} = B^b D'^d + B' - D'^d B''^b, x off-side: DerMorb s6
//   4  DA^{bd} = D'^d A^b, same side: DerMorb s5 (-D'^d A^b) and the Omega block (-D'^al A^be + D'^be A^al)
//   5  DD^c = D'^al D'^be, same side: Omega block, internal term
//   6  AA^c = A''^al A''^be, same side: Omega block, external term
//   7  VA^{d be} = V''^d A''^be, same side: DerMorb s4
// DerOmega contributions carry the band weight dw(n) = 2 (DerOmega) or
// 2 sign E_n (DerMorb's Eav o dOmega term; only cut partitions are summed, so a
// same-side element may be credited to either of its bands).
struct TaskCtx {
    bool in, ex;
    bool s5;      // DerMorb's s5 and T4 are summed: (2 E_l + 2 sign E_n) Im(A^a_nl dA_ln), dA Hermitian, is
                  // odd under l <-> n for sign = +1, so its trace vanishes there (complex64 channels, whose
                  // A is Hermitian to storage rounding only, keep it)
    double sign;
    int cut;      // two-set partition [0, cut); < 0: the groups of the labels
};

// The component c of a term with index pair (alpha_c, beta_c) = (x, y) (sig +1) or (y, x) (-1), x != y
__device__ inline int third_index(int x, int y) { return 3 - x - y; }
__device__ inline double pair_sign(int x, int y) { return y == (x == 2 ? 0 : x + 1) ? 1.0 : -1.0; }

// DerOmega's T4 has no real trace for Hermitian A; complex64 channels, whose A is Hermitian to storage
// rounding only, keep it: groups of up to SC_T4_LOOP bands by a loop per band, larger ones as tasks
#define SC_T4_LOOP 4
template <bool DM, typename T>
__host__ __device__ constexpr bool keep_t4() {
    return !DM && sizeof(T) == 4;
}

// per-lane sums of a task: 0 - 2 one per partner a = 0, 1, 2; kind 0 of DerMorb: [3] = s1; kind 4:
// [3] - [5] the Omega block's components; kinds 5, 6: one per e; kind 7: one
template <int KIND, bool DM>
__host__ __device__ constexpr int task_nt() {
    return KIND == 0 ? (DM ? 4 : 3) : KIND == 4 ? (DM ? 6 : 3) : KIND == 7 ? 1 : 3;
}

// V^a_ln of a weight D'^a_nl = m_ln conj(V^a_ln): complex64 channels, whose triangles now and then differ by their
// rounding at a whole k-point (an element of the transform rounded to either side), read V^a_nl itself
template <typename T, bool LM, bool ST, bool SA, int NW>
__device__ __attribute__((always_inline)) cplx<double> partner_V(const KCtx<T, LM, ST, SA, NW>& K, int a, int l, int n) {
    if constexpr (sizeof(T) == 4) return conj(K.Vu(a, n, l));
    else return K.Vu(a, l, n);
}

template <int KIND, bool DM, typename T, bool LM, bool ST, bool SA, int NW>
__device__ __attribute__((always_inline)) void formula_task(const Smem& S, const KCtx<T, LM, ST, SA, NW>& K, const TaskCtx& tc_,
                                                           double* acc, int b, int d, int rh, int cb) {
    constexpr bool dm = DM;
    const int nw = K.n_(), lane = threadIdx.x & 63;
    const int r0 = rh * 16, c0 = cb * 32;  // a 16 x 32 half block
    const bool in = tc_.in, ex = tc_.ex;
    const double sign = tc_.sign;
    const int cut = tc_.cut;
    const int al = c_alpha[b], be = c_beta[b];  // kinds 5, 6: b = c
    // blocks without an element in use, and the range [k0, k1) of the summed index with D' != 0
    // (kinds 6, 7: with both factors in the partition)
    int k0 = 0, k1 = nw;
    bool act[2], multi = false;  // multi: a column whose group has several bands
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int n = c0 + mfma_col(u);
        act[u] = n < nw && S.act[n];
        multi |= act[u] && S.ge[n] - S.gs[n] > 1;
    }
    if (!__any(act[0] || act[1])) return;
    if (cut >= 0) {
        if constexpr (KIND == 0 || KIND == 3) {
            if (r0 + 16 <= cut) return;
        } else if constexpr (KIND == 2) {
            if (r0 + 16 <= cut && !(dm && tc_.s5)) return;
        } else {
            if (r0 >= cut) return;
        }
        if constexpr (KIND == 6 || KIND == 7)
            k1 = cut;
        else
            k0 = cut;
    }
    MfmaHalf P;
    P.zero();
    if constexpr (KIND == 0)
        mfma_half(P, nw, nw, k0, k1, r0, c0, [&](int r, int m) { return K.Vu(b, r, m); }, [&](int m, int c) { return K.Dpu(d, m, c); });
    else if constexpr (KIND == 2)
        mfma_half(P, nw, nw, k0, k1, r0, c0, [&](int r, int m) { return K.Au(b, r, m); }, [&](int m, int c) { return K.Dpu(d, m, c); });
    else if constexpr (KIND == 3)
        mfma_half(P, nw, nw, k0, k1, r0, c0, [&](int r, int m) { return K.getu(WBMI_ROLE_B + b, r, m); }, [&](int m, int c) { return K.Dpu(d, m, c); });
    else if constexpr (KIND == 4)
        mfma_half(P, nw, nw, k0, k1, r0, c0, [&](int r, int m) { return K.Dpu(d, r, m); }, [&](int m, int c) { return K.Au(b, m, c); });
    else if constexpr (KIND == 5)
        mfma_half(P, nw, nw, k0, k1, r0, c0, [&](int r, int m) { return K.Dpu(al, r, m); }, [&](int m, int c) { return K.Dpu(be, m, c); });
    else if constexpr (KIND == 6)
        mfma_half(P, nw, nw, k0, k1, r0, c0, [&](int r, int m) { return K.Ainu(al, r, m); }, [&](int m, int c) { return K.Ainu(be, m, c); });
    else
        mfma_half(P, nw, nw, k0, k1, r0, c0, [&](int r, int m) { return K.Vinu(b, r, m); }, [&](int m, int c) { return K.Ainu(d, m, c); });
    // kinds 0, 2, 3, the within-group part -D'^d X''^b (X = V, A, B): one term for a group of one
    // band (the epilogue's), else a second product over the bands of the columns' groups.  Kind 0 of
    // DerMorb keeps it apart, as s1 reads the first product alone
    constexpr bool within = KIND == 0 || KIND == 2 || KIND == 3;
    bool big = false;
    MfmaHalf P2;
    MfmaHalf& Pw = (KIND == 0 && DM) ? P2 : P;
    if constexpr (within) {
        big = __any(multi);
        if constexpr (KIND == 0 && DM) P2.zero();
        if (big) {
            int g0 = 0, g1 = cut;
            if (cut < 0) {
                g0 = nw;
                g1 = 0;
#pragma unroll
                for (int u = 0; u < 2; ++u)
                    if (act[u]) {
                        g0 = min(g0, S.gs[c0 + mfma_col(u)]);
                        g1 = max(g1, S.ge[c0 + mfma_col(u)]);
                    }
                for (int o = 8; o >= 1; o >>= 1) {
                    g0 = min(g0, __shfl_xor(g0, o));
                    g1 = max(g1, __shfl_xor(g1, o));
                }
            }
            mfma_half(
                Pw, nw, nw, g0, g1, r0, c0, [&](int r, int m) { return r < cut ? mk(0.0, 0.0) : -K.Dpu(d, r, m); },
                [&](int m, int c) {
                    if (K.lab[m] != K.lab[c]) return mk(0.0, 0.0);
                    if constexpr (KIND == 0) return K.Vu(b, m, c);
                    else if constexpr (KIND == 2) return K.Au(b, m, c);
                    else return K.getu(WBMI_ROLE_B + b, m, c);
                });
        }
    }

    // part[u][w]: u = the lane's band slot, its column bj (the band n is the column y of every element)
    constexpr int NU = 2, NT = task_nt<KIND, DM>();
    double part[NU][NT];
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
        for (int w = 0; w < NT; ++w) part[u][w] = 0.0;
    // s1: the c with beta_c = d, partner alpha_c
    const int s1c = d == 2 ? 0 : d + 1;  // beta_c = c + 2
    {
        // the elementwise channel (W, A', B') of this row half: all loads issued before use
        cplx<double> gz[2][4];
        if constexpr (KIND == 0 || KIND == 2 || KIND == 3) {
#pragma unroll
            for (int bj = 0; bj < 2; ++bj)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int x = r0 + mfma_hrow(v), y = c0 + mfma_col(bj);
                    const bool ok = x < nw && y < nw;
                    const int xx = ok ? x : 0, yy = ok ? y : 0;
                    if constexpr (KIND == 0)
                        gz[bj][v] = K.getu(WBMI_ROLE_W + 3 * (b) + d, xx, yy);  // (l, n)
                    else if constexpr (KIND == 2)
                        gz[bj][v] = ex ? K.getu(WBMI_ROLE_AD + 3 * (b) + d, xx, yy) : mk(0.0, 0.0);
                    else
                        gz[bj][v] = K.getu(WBMI_ROLE_BD + 3 * (b) + d, xx, yy);
                }
        }
#pragma unroll
        for (int bj = 0; bj < 2; ++bj) {
            const int n = c0 + mfma_col(bj);
            if (!act[bj]) continue;
            const double dw = dm ? 2.0 * sign * K.E[n] : 2.0;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int l = r0 + mfma_hrow(v);
                if (l >= nw) continue;
                const cplx<double> pv = P.get(bj, v);
                const bool same = K.lab[l] == K.lab[n];
                if constexpr (KIND == 0) {
                    if (same) continue;
                    // W^{bd}_ln / 2 - (D'^d V''^b)_ln, with D'_xy = -m_xy V_xy and m_nl = -m_ln
                    // (V_nn is real to its rounding only; its imaginary part enters as V_nn - V_ll does, which may be as small)
                    const double mln = K.m(l, n);
                    cplx<double> z = 0.5 * gz[bj][v];
                    if (!big) z += mln * (K.Vu(b, n, n) * K.Vu(d, l, n));
                    if constexpr (DM) z += P2.get(bj, v);
                    const cplx<double> Pm = (-mln) * (pv + z);
                    // -conj dD.nl: its within-group part from V's other triangle, as stored, in groups of up to SC_T4_LOOP bands
                    cplx<double> Pn = Pm;
                    if constexpr (sizeof(T) == 4)
                        if (ex) {
                            if (!big) {
                                Pn = (-mln) * (pv + 0.5 * gz[bj][v] + mln * conj(K.Vu(b, n, n) * K.Vu(d, n, l)));
                            } else if (S.ge[n] - S.gs[n] <= SC_T4_LOOP) {
                                cplx<double> c = mk(0.0, 0.0);
#pragma unroll 1
                                for (int q = S.gs[n]; q < S.ge[n]; ++q)
                                    c += K.m(l, q) * (conj(K.Vu(b, n, q) * K.Vu(d, q, l)) - K.Vu(d, l, q) * K.Vu(b, q, n));
                                Pn = Pm - mln * c;
                            }
                        }
                    const double wD = in ? (dm ? dw + 2.0 * K.E[l] : dw) : 0.0;
#pragma unroll
                    for (int a = 0; a < 3; ++a) {
                        // -i wD D'_nl, D'_nl = m_ln conj(V_ln)
                        const cplx<double> va = partner_V(K, a, l, n);
                        cplx<double> q = (wD * mln) * mk(-va.im, -va.re);
                        if (ex) {
                            const cplx<double> A = K.Au(a, l, n);
                            part[bj][a] -= dw * (A.re * Pn.re + A.im * Pn.im);
                            if (dm) q -= 2.0 * conj(K.getu(WBMI_ROLE_B + a, l, n));
                        }
                        part[bj][a] += q.re * Pm.re - q.im * Pm.im;
                    }
                    if constexpr (DM)
                        if (in) part[bj][3] += ((mln * conj(partner_V(K, c_alpha[s1c], l, n))) * pv).im;  // Re(-i D'^al V^d D'^be)
                } else if constexpr (KIND == 2) {
                    if (!same) {
                        // A'^{bd} - D'^d A''^b
                        const double mln = K.m(l, n);
                        cplx<double> z = gz[bj][v];
                        if (!big) z += mln * (K.Vu(d, l, n) * K.Au(b, n, n));
                        const cplx<double> Y1 = (-dw * mln) * (pv + z);
#pragma unroll
                        for (int a = 0; a < 3; ++a) {
                            const cplx<double> va = partner_V(K, a, l, n);
                            part[bj][a] += va.re * Y1.re + va.im * Y1.im;  // Re conj(V_ln) Y1
                        }
                    } else if (dm ? tc_.s5 : keep_t4<DM, T>() && S.ge[n] - S.gs[n] > SC_T4_LOOP) {
                        // s5 and T4: Re(-i sig (2 E_l + 2 sign E_n) A^a_nl (A' + A^b D'^d)_ln)
                        const cplx<double> dA = pv + K.getu(WBMI_ROLE_AD + 3 * (b) + d, l, n);
                        const double w5 = dm ? dw + 2.0 * K.E[l] : dw;
#pragma unroll
                        for (int a = 0; a < 3; ++a) part[bj][a] += w5 * (K.Au(a, n, l) * dA).im;
                    }
                } else if constexpr (KIND == 3) {
                    if (same) continue;
                    // B'^{bd} - D'^d B''^b
                    cplx<double> z = gz[bj][v];
                    if (!big) z -= K.Dpu(d, l, n) * K.getu(WBMI_ROLE_B + b, n, n);
                    const cplx<double> YB = pv + z;
#pragma unroll
                    for (int a = 0; a < 3; ++a) part[bj][a] -= 2.0 * (K.Dpu(a, n, l) * YB).re;  // s6
                } else if constexpr (KIND == 4) {
                    if (!same) continue;
                    // s5 and T4 with -D'^d A^b in place of dA; Omega block: 2 sign coef Re(DA_ln V^e_nl)
                    if (dm ? tc_.s5 : S.ge[n] - S.gs[n] > SC_T4_LOOP) {
                        const double w5 = dm ? dw + 2.0 * K.E[l] : dw;
#pragma unroll
                        for (int a = 0; a < 3; ++a) part[bj][a] -= w5 * (K.Au(a, n, l) * pv).im;
                    }
                    if constexpr (DM)
#pragma unroll
                        for (int e = 0; e < 3; ++e) part[bj][3 + e] += (pv * K.Vu(e, n, l)).re;
                } else if constexpr (KIND == 5 || KIND == 6) {
                    if (!same) continue;
                    // Omega block term -i P_ln: 2 sign Re(-i P_ln V^e_nl)
#pragma unroll
                    for (int w = 0; w < 3; ++w) part[bj][w] += (pv * K.Vu(w, n, l)).im;
                } else {
                    if (!same) continue;
                    // s4: Re(-2i A^al_np (V''^d A''^be)_pn)
                    part[bj][0] += (K.Au(c_alpha[s1c], n, l) * pv).im;
                }
            }
        }
    }
    // reduce over the summed index l: the rows, lane bits 4-5
    const int mask = 0x30;
    const bool writer = (lane >> 4) == 0;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        const int n = c0 + mfma_col(u);
        double sum[NT];
#pragma unroll
        for (int w = 0; w < NT; ++w) sum[w] = wave_sum(part[u][w], mask);
        if (!writer || n >= nw) continue;
        double* row = acc + n * 9;
        if constexpr (KIND <= 4) {
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                // the component whose index pair holds b and the partner a: column (c, d); X1 is
                // symmetric in its indices, so kind 0 also feeds (c', b) of the pair of d and a
                if (a != b) atomicAdd(&row[third_index(a, b) * 3 + d], pair_sign(a, b) * sum[a]);
                if constexpr (KIND == 0)
                    if (a != d) atomicAdd(&row[third_index(a, d) * 3 + b], pair_sign(a, d) * sum[a]);
            }
        }
        if constexpr (KIND == 0 && DM) {
            if (in) atomicAdd(&row[s1c * 3 + b], 2.0 * sum[3]);
        } else if constexpr (KIND == 4 && DM) {
            // Omega block: D'^d A^b enters s^c with -1 for (al_c, be_c) = (d, b), +1 for (b, d)
            if (b != d && sign != 0.0)
#pragma unroll
                for (int e = 0; e < 3; ++e)
                    atomicAdd(&row[third_index(b, d) * 3 + e], -2.0 * sign * pair_sign(d, b) * sum[3 + e]);
        } else if constexpr (KIND == 5 || KIND == 6) {
#pragma unroll
            for (int e = 0; e < 3; ++e) atomicAdd(&row[b * 3 + e], 2.0 * sign * sum[e]);
        } else if constexpr (KIND == 7) {
            atomicAdd(&row[s1c * 3 + b], 2.0 * sum[0]);
        }
    }
}

// DerOmega's per-band terms where V and A are not in LDS, for the partition of the labels:
//   T5: 0.5 dO.nn = 0.5 [O'^{cd}_nn - (D'^d O^c)_nn + (O^c D'^d)_nn].  O is Hermitian and D' anti-Hermitian, so
//     (D'^d O^c)_nn = -conj((O^c D'^d)_nn) and only the real part, Re O'_nn + 2 Re sum_l conj(O_ln) D'_ln, is used;
//   T4 of the groups of one band where it is kept (keep_t4): 2 Im A^a_nn dA_nn^{bd},
//     dA_nn = A'_nn + sum_l A^b_nl D'^d_ln - D'^d_nl A^b_ln.
// 8 x 8 bands a wave and all components, as in diag_traces (a thread per (n, c, d) read the columns, and for T4
// also rows, nine times: DerOmega of 216 k-points at nw = 128 3.66 -> 3.27 ms complex64, 2.72 -> 2.56 complex128;
// with V in LDS the threads are faster, 4096 at nw = 32 0.73 against 0.79 ms).
template <typename T, bool LM, bool ST, bool SA, int NW>
__device__ __attribute__((always_inline)) void der_diag(const Smem& S, const KCtx<T, LM, ST, SA, NW>& K) {
    constexpr bool T4 = keep_t4<false, T>();
    const int nw = K.n_(), lane = threadIdx.x & 63, nwave = ((int)blockDim.x >> 6) * K.parts;
    const int n8 = (nw + 7) / 8, split = min(max(nwave / n8, 1), n8);
    for (int t = ((int)threadIdx.x >> 6) * K.parts + K.part; t < n8 * split; t += nwave) {
        const int nn = 8 * (t % n8) + (lane >> 3), n = min(nn, nw - 1);
        const bool on = nn < nw && S.act[n], one = on && S.ge[n] - S.gs[n] == 1;
        if (!__any(on)) continue;
        double t5[9];
        cplx<double> y[T4 ? 9 : 1];
#pragma unroll
        for (int q = 0; q < 9; ++q) {
            t5[q] = 0.0;
            if constexpr (T4) y[q] = mk(0.0, 0.0);
        }
        for (int l0 = 8 * (t / n8); l0 < nw; l0 += 8 * split) {
            const int ll = l0 + (lane & 7), l = min(ll, nw - 1);
            const double m = on && ll < nw ? K.m(n, l) : 0.0;
            cplx<double> D[3], O[3];
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                D[a] = m * K.Vu(a, l, n);  // D'_ln = -m_ln V_ln
                O[a] = K.getu(WBMI_ROLE_O + a, l, n);
            }
#pragma unroll
            for (int q = 0; q < 9; ++q) t5[q] += 2.0 * (conj(O[q / 3]) * D[q % 3]).re;
            if constexpr (T4) {
                cplx<double> Dt[3], A[3], At[3];
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    Dt[a] = m * K.Vu(a, n, l);
                    A[a] = K.Au(a, n, l);
                    At[a] = K.Au(a, l, n);
                }
#pragma unroll
                for (int q = 0; q < 9; ++q) y[q] += A[q / 3] * D[q % 3] + Dt[q % 3] * At[q / 3];
            }
        }
        const bool first = t < n8;  // the elementwise terms once
#pragma unroll
        for (int q = 0; q < 9; ++q) {
            t5[q] = wave_sum(t5[q], 7);
            if constexpr (T4) {
                y[q].re = wave_sum(y[q].re, 7);
                y[q].im = wave_sum(y[q].im, 7);
            }
        }
        if ((lane & 7) || !on) continue;
#pragma unroll
        for (int q = 0; q < 9; ++q) {
            const int b = q / 3, d = q % 3;
            if (first) t5[q] += K.getu(WBMI_ROLE_OD + q, n, n).re;
            atomicAdd(&S.acc[n * 9 + q], t5[q]);
            if constexpr (T4) {
                if (!one) continue;
                if (first) y[q] += K.getu(WBMI_ROLE_AD + q, n, n);
#pragma unroll
                for (int a = 0; a < 3; ++a)
                    if (a != b) atomicAdd(&S.acc[n * 9 + third_index(a, b) * 3 + d], 2.0 * pair_sign(a, b) * (K.Au(a, n, n) * y[q]).im);
            }
        }
    }
}

// DerOmega (formula/covariant.py:212-259) or, dm = true, DerMorb
// (formula/covariant.py:463-552) per-band values into S.acc[n][c*3+d], for the partition of the
// labels (cut < 0) or [0, cut) (the labels set likewise).
// DerMorb = DerMorb_H + sign [Eav o dOmega + (Omega V + V Omega)/2] on cut
// partitions; its trace terms (s1 ... s7, the Omega block) are listed at
// formula_task.  DerOmega's term T4, -i sig Tr A^a dA.nn^{bd}, is a real trace of two Hermitian
// matrices times -i: it has no real part and is left out (complex64 channels: keep_t4).
// DM is compile-time so that the DerOmega kernel carries only the kinds it runs (0 and 2): its
// register allocation and code size are not those of the DerMorb kinds.
// The workgroups part = 0, 1, .. of one k share its tasks and per-band terms: each adds up its own,
// and the sums over groups are linear in them.
template <bool DM, typename T, bool LM, bool ST, bool SA, int NW>
__device__ __attribute__((always_inline)) void eval_deromega(const Smem& S, const KCtx<T, LM, ST, SA, NW>& K, bool in, bool ex,
                                                            int sign, int cut) {
    constexpr bool dm = DM;
    const int nw = K.n_(), tid = threadIdx.x;
    const int t0 = tid + (int)blockDim.x * K.part, tstep = (int)blockDim.x * K.parts;  // per-band terms
    const int l0 = cut >= 0 ? cut : 0;  // D' != 0 from here on
    constexpr bool diag = !DM && !ST;  // V and A in LDS: a thread per (n, c, d) and group
    if constexpr (diag) {
        if (ex) der_diag(S, K);
    } else {
        // per-band terms, lanes running over (n, c, d)
        for (int t = t0; t < nw * 9; t += tstep) {
            const int n = t % nw, c = (t / nw) / 3, d = (t / nw) % 3;
            if (!S.act[n] || !ex) continue;
            // T5: 0.5 dO.nn = 0.5 [O'^{cd}_nn - (D'^d O^c)_nn + (O^c D'^d)_nn].  O is Hermitian
            // and D' anti-Hermitian, so (D'^d O^c)_nn = -conj((O^c D'^d)_nn) and only the real part,
            // Re O'_nn + 2 Re sum_l conj(O_ln) D'_ln, is used: column n of O, which consecutive
            // threads (consecutive n) read from consecutive addresses
            double t5 = K.Od(c, d, n, n).re;
#pragma unroll 8
            for (int l = l0; l < nw; ++l) t5 += 2.0 * (conj(K.O(c, l, n)) * K.Dp(d, l, n)).re;
            double v = (dm ? sign * S.E[n] : 1.0) * t5;
            if constexpr (DM) {
                // s3: dH.nn = C'^{cd}_nn - (D'^d C^c)_nn + (C^c D'^d)_nn
                cplx<double> s3 = K.Cd(c, d, n, n);
                for (int l = l0; l < nw; ++l) s3 += K.C(c, n, l) * K.Dp(d, l, n) - K.Dp(d, n, l) * K.C(c, l, n);
                // Omega block, elementwise part: 2 sign Re sum_{l in G} (O^c_nl / 2) V^d_ln
                cplx<double> ov = mk(0.0, 0.0);
                for (int l = S.gs[n]; l < S.ge[n]; ++l) ov += K.O(c, n, l) * K.V(d, l, n);
                v += s3.re + sign * ov.re;
            }
            S.acc[n * 9 + c * 3 + d] = v;
        }
    }
    int t4 = 0;  // tasks for T4: some group is too large for the loop
    if constexpr (keep_t4<DM, T>()) {
        for (int n = tid; n < nw; n += (int)blockDim.x) t4 |= S.act[n] && S.ge[n] - S.gs[n] > SC_T4_LOOP;
        t4 = __syncthreads_or(t4);
        for (int t = t0; t < nw * 9 && ex; t += tstep) {
            const int n = t % nw, b = (t / nw) / 3, d = (t / nw) % 3, g0 = S.gs[n], g1 = S.ge[n];
            if (!S.act[n] || (diag && g1 - g0 == 1) || g1 - g0 > SC_T4_LOOP) continue;
            double v[3] = {0.0, 0.0, 0.0};
            for (int m = g0; m < g1; ++m) {
                cplx<double> y = K.Ad(b, d, m, n);  // dA.nn^{bd}_mn
#pragma unroll 4
                for (int l = 0; l < nw; ++l) y += K.A(b, m, l) * K.Dp(d, l, n) - K.Dp(d, m, l) * K.A(b, l, n);
#pragma unroll
                for (int a = 0; a < 3; ++a) v[a] += (K.A(a, n, m) * y).im;
            }
#pragma unroll
            for (int a = 0; a < 3; ++a)
                if (a != b) atomicAdd(&S.acc[n * 9 + third_index(a, b) * 3 + d], 2.0 * pair_sign(a, b) * v[a]);
        }
    }
    if (tid == 0) S.misc[3] = 0;  // task counter
    __syncthreads();
    // wave tasks (kind, b, d, row block, column block), round-robin over the waves
    const TaskCtx tcx{in, ex, dm && ex && (sign != 1 || sizeof(T) == 4), (double)sign, cut};
    int cnt[8];
    cnt[0] = in || ex ? 9 : 0;
    cnt[1] = 0;
    cnt[2] = ex ? 9 : 0;
    cnt[3] = dm && ex ? 9 : 0;
    cnt[4] = ex && (dm ? tcx.s5 || sign != 0 : t4 != 0) ? 9 : 0;
    cnt[5] = dm && in && sign != 0 ? 3 : 0;
    cnt[6] = dm && ex && sign != 0 ? 3 : 0;
    cnt[7] = dm && ex ? 9 : 0;
    // a task is one 16-row x 32-column half block of one product; the waves take the next
    // task from an LDS counter, kinds in the order above (the heaviest, kind 0, first), so the
    // waves finish together whatever the mix of kinds
    const int nblk = (nw + 31) / 32, nrh = (nw + 15) / 16, nb2 = nrh * nblk;
    int ntask = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) ntask += cnt[q] * nb2;
    const int lane = tid & 63;
    for (;;) {
        int t = 0;
        if (lane == 0) t = atomicAdd(&S.misc[3], 1);
        t = __builtin_amdgcn_readfirstlane(t) * K.parts + K.part;
        if (t >= ntask) break;
        int kind = -1, rem = 0, base = 0;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int nq = cnt[q] * nb2;
            if (kind < 0 && t - base < nq) {
                kind = q;
                rem = t - base;
            }
            base += nq;
        }
        const int idx = rem / nb2, rh = (rem % nb2) / nblk, cb = rem % nblk;
        const int b = kind == 5 || kind == 6 ? idx : idx / 3, d = kind == 5 || kind == 6 ? 0 : idx % 3;
        switch (kind) {
            case 0: formula_task<0, DM>(S, K, tcx, S.acc, b, d, rh, cb); break;
            case 2: formula_task<2, DM>(S, K, tcx, S.acc, b, d, rh, cb); break;
            case 4:
                if constexpr (DM || keep_t4<DM, T>()) formula_task<4, DM>(S, K, tcx, S.acc, b, d, rh, cb);
                break;
            default:
                if constexpr (DM) {
                    switch (kind) {
                        case 3: formula_task<3, DM>(S, K, tcx, S.acc, b, d, rh, cb); break;
                        case 5: formula_task<5, DM>(S, K, tcx, S.acc, b, d, rh, cb); break;
                        case 6: formula_task<6, DM>(S, K, tcx, S.acc, b, d, rh, cb); break;
                        default: formula_task<7, DM>(S, K, tcx, S.acc, b, d, rh, cb); break;
                    }
                }
                break;
        }
    }
}

// ---------------------------------------------------------------------------
// every cut of a non-additive formula at once
// ---------------------------------------------------------------------------
//
// Morb_Hpm and DerMorb are scanned as T(c), the trace over the bands [0, c) with the rest outside, at
// every border c of a group in range: up to nw partitions per k-point.  Evaluated one by one they cost
// O(nw^4) (DerMorb) and O(nw^3) (Morb_Hpm) per k.  Each term of T(c) is a sum over bands of which some
// are below c and some are not, so it belongs to the cuts between its highest band inside and its lowest
// band outside, and
//     T(c) = sum_{n < c <= l} g(n, l) + sum_{x < c} r(x)
// with g(n, l) what remains when the other bands of the term are summed over q <= n or m >= l.  These
// sums are triangular matrix products, formed once for all cuts.  T(c) is added up from its own terms
// only, never as a difference of running sums: bands that no evaluated cut separates may be degenerate
// to 1e-7, and their terms exceed the rest by as much as the inverse cube of that.

// T(c) += sum over n < c <= l of a 16 x 16 tile's values (rows n of block nb, columns l of block lb >= nb;
// the lane's elements (n, l) = (lane / 16 + 4 v, lane % 16), zero where n >= l), component comp.
// The sums over n < c are a product with a triangle of ones (the values already have the operand layout).
__device__ __attribute__((always_inline)) inline void cut_tile_add(const Smem& S, int nw, int nb, int lb, const double (&val)[4],
                                                                  int comp) {
    const int lane = threadIdx.x & 63, g = lane >> 4, j = lane & 15;
    wbmi_v4d L = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int v = 0; v < 4; ++v) L = __builtin_amdgcn_mfma_f64_16x16x4f64(4 * v + g < j ? 1.0 : 0.0, val[v], L, 0, 0, 0);
    // L: (c, l), sum over n < c; rows summed over l, each lane keeping row g + 4 (lane % 4)
    double x[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) x[v] = nb < lb || g + 4 * v <= j ? L[v] : 0.0;
    const double r0 = (lane & 1 ? x[1] : x[0]) + __shfl_xor(lane & 1 ? x[0] : x[1], 1);
    const double r1 = (lane & 1 ? x[3] : x[2]) + __shfl_xor(lane & 1 ? x[2] : x[3], 1);
    double r = (lane & 2 ? r1 : r0) + __shfl_xor(lane & 2 ? r0 : r1, 2);
    r = wave_sum(r, 0xc);
    const int c = 16 * nb + g + 4 * (lane & 3);
    if ((lane & 0xc) == 0 && c < nw) atomicAdd(&S.cut[c * 9 + comp], r);
    if (nb == lb) return;
    // cuts above the rows: the columns l >= c
    double cs = wave_sum((val[0] + val[1]) + (val[2] + val[3]), 0x30);
    for (int o = 1; o < 16; o <<= 1) {
        const double t = __shfl_down(cs, o, 16);
        if (j + o < 16) cs += t;
    }
    const int l0 = 16 * lb, cend = min(l0 + 16, nw);
    const double all = __shfl(cs, 0);
    for (int c0 = 16 * nb + 16; c0 < cend; c0 += 64) {
        const int cc = c0 + lane;
        const double t = __shfl(cs, cc > l0 ? (cc - l0) & 15 : 0);
        if (cc < cend) atomicAdd(&S.cut[cc * 9 + comp], cc <= l0 ? all : t);
    }
}

// Some evaluated cut separates block nb's rows from block lb's columns (one answer per wave)
__device__ inline bool cut_tile_needed(const Smem& S, int nw, int nb, int lb) {
    bool any = false;
    for (int c = 16 * nb + 1 + (int)(threadIdx.x & 63); c < min(16 * lb + 16, nw); c += 64) any |= S.need[c] != 0;
    return __any(any);
}

// Tile pair t of the nb (nb + 1) / 2 pairs rb <= cb, by their distance (the nearest sum over most bands)
__device__ inline void cut_tile_pair(int t, int nblk, int& rb, int& cb) {
    int d = 0;
    while (t >= nblk - d) {
        t -= nblk - d;
        ++d;
    }
    rb = t;
    cb = t + d;
}

// the sums of row v are formed here, not put off to their use with every operand kept in registers
__device__ __attribute__((always_inline)) inline void cut_pin(double (&o)[7][4], int v) {
#pragma unroll
    for (int q = 0; q < 7; ++q) asm volatile("" : "+v"(o[q][v]));
}

// three complex 16 x 16 blocks in the accumulators
struct CutAcc {
    wbmi_v4d re[3], im[3];
    __device__ inline void zero() {
#pragma unroll
        for (int r = 0; r < 3; ++r) re[r] = im[r] = wbmi_v4d{0.0, 0.0, 0.0, 0.0};
    }
    __device__ inline void add(int r, cplx<double> x, cplx<double> y) {
        re[r] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.re, y.re, re[r], 0, 0, 0);
        im[r] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.re, y.im, im[r], 0, 0, 0);
        re[r] = __builtin_amdgcn_mfma_f64_16x16x4f64(-x.im, y.im, re[r], 0, 0, 0);
        im[r] = __builtin_amdgcn_mfma_f64_16x16x4f64(x.im, y.re, im[r], 0, 0, 0);
    }
    __device__ inline cplx<double> get(int r, int v) const { return mk(re[r][v], im[r][v]); }
};

// DerMorb with internal terms only (formula/covariant.py:463-552), every needed cut into S.cut.  With
// P = D' without its mask (anti-Hermitian), Q^a_nl = i (1 / (E_l - E_n)) (2 sign E_n + 2 E_l) P^a_nl and
// n < c <= l, the per-cut terms (formula_task: kinds 0, s1 and 5) are, summed over n and l,
//     Re Q^a_nl F^{bd}_ln  to the pair of a and b, column d, and (X1 symmetric) to that of a and d, column b
//     2 Im P^a_nl H^{bd}_ln  to the pair of a and d, column b
//     F = Y + U + W / 2, H = Y - sign U,  Y_ln = sum_{m >= c} V^b_lm P^d_mn,  U_ln = -sum_{q < c} P^d_lq V^b_qn.
// A term of Y with m > l stays with the pair (n, l); one with m < l belongs to the pair (n, m), where
// Q V (for F) or, because swapping l and m conjugates it, P V again (for H) collects it; m = l counts half
// in both.  U the same with q and n.  So a task, one pair of 16-band blocks and one b, is the products
//     [P; Q] (n, m) V^b (m, l) over m >= l,   V^b (n, q) [P, Q] (q, l) over q <= n
// for three d and three a at once: a V and three P elements per 24 MFMAs, which leaves the matrix cores
// as the bound.  294 k-points at nw = 64, every cut (complex64): 7.5 ms one by one, 0.4 ms together (0.25 with HERM).
// HERM: V and W are Hermitian to the rounding of the sums.  Otherwise (complex64: partner_V, and the rotation in
// FP32 arithmetic, whose two triangles differ by their rounding) every term reads the triangle that
// formula_task reads, 36 MFMAs: P V with both triangles of V, V P with both of P.
template <bool HERM, typename T, bool LM, bool ST, bool SA, int NW>
__device__ __attribute__((always_inline)) void eval_dermorb_in(const Smem& S, const KCtx<T, LM, ST, SA, NW>& K, double sign) {
    constexpr int NS = HERM ? 1 : 2;
    const int nw = K.n_(), lane = threadIdx.x & 63, lk = lane >> 4, li = lane & 15;
    const int nblk = (nw + 15) / 16, ntask = 3 * (nblk * (nblk + 1) / 2);
    for (;;) {
        int t = 0;
        if (lane == 0) t = atomicAdd(&S.misc[3], 1);
        t = __builtin_amdgcn_readfirstlane(t) * K.parts + K.part;
        if (t >= ntask) break;
        const int b = t % 3;
        int nb, lb;
        cut_tile_pair(t / 3, nblk, nb, lb);
        if (!cut_tile_needed(S, nw, nb, lb)) continue;
        int ax[3];  // the indices b, b + 1, b + 2: everything below is relative to b
#pragma unroll
        for (int r = 0; r < 3; ++r) ax[r] = (b + r) % 3;
        // the pairs' values: components (c, d) relative to b, c = 1, 2 in [0, 6), (0, 0) in [6]
        double o[7][4];
#pragma unroll
        for (int q = 0; q < 7; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) o[q][v] = 0.0;
        CutAcc G[NS], Z;  // P V or V P of both kinds of V or P; Q V or V Q
        // FIRST: the sums over m >= l, with f = W / 2 - (P V) = conj(F), h = -(P V) = conj(H); else those
        // over q <= n, with f = (V P), h = -sign (V P)
        auto add_pairs = [&](auto first) {
            constexpr bool FIRST = decltype(first)::value;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                // an opaque row: the operands are loaded anew for each v and call, not kept in registers
                int nn = 16 * nb + lk + 4 * v;
                asm volatile("" : "+v"(nn)::"memory");
                const int ll = 16 * lb + li;
                const bool ok = nn < ll && ll < nw;
                const int x = min(nn, nw - 1), y = min(ll, nw - 1);
                const double m = K.m(x, y), kap = -m * (2.0 * sign * S.E[x] + 2.0 * S.E[y]);
                cplx<double> P[3], Pu[3];
#pragma unroll
                for (int r = 0; r < 3; ++r) {
                    Pu[r] = (-m) * K.Vu(ax[r], x, y);
                    P[r] = HERM ? Pu[r] : (-m) * conj(K.Vu(ax[r], y, x));
                }
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    cplx<double> f = G[0].get(d, v);
                    if constexpr (FIRST) f = (HERM ? 0.5 * K.getu(WBMI_ROLE_W + 3 * b + ax[d], x, y) : 0.5 * conj(K.getu(WBMI_ROLE_W + 3 * b + ax[d], y, x))) - f;
#pragma unroll
                    for (int a = 0; a < 3; ++a) {
                        const double s = -kap * (Pu[a] * conj(f)).im - (Z.get(a, v) * conj(P[d])).re;
                        if (a != 0) {
                            const double e = pair_sign(a, 0) * s;
                            o[(third_index(a, 0) - 1) * 3 + d][v] += ok ? e : 0.0;
                        }
                        if (a != d) {
                            const bool pos = pair_sign(a, d) > 0.0;
                            const cplx<double> h = G[pos ? 0 : NS - 1].get(d, v);
                            const double hw = FIRST ? -2.0 : -2.0 * sign;
                            const double e = pair_sign(a, d) * (s + hw * ((pos ? Pu[a] : P[a]) * conj(h)).im);
                            const int c = third_index(a, d);
                            o[c == 0 ? 6 : (c - 1) * 3][v] += ok ? e : 0.0;
                        }
                    }
                }
                cut_pin(o, v);
            }
        };
        // rows and columns past the end repeat the last one; their results are not read
        const int n = min(16 * nb + li, nw - 1), l = min(16 * lb + li, nw - 1);
        const double En = S.E[n], El = S.E[l];
        Z.zero();
#pragma unroll
        for (int q = 0; q < NS; ++q) G[q].zero();
        for (int k0 = 16 * lb; k0 < nw; k0 += 4) {
            const int m = min(k0 + lk, nw - 1);
            const double w = k0 + lk >= nw || m < l ? 0.0 : m == l ? 0.5 : 1.0;
            const cplx<double> vl = w * K.Vu(b, m, l), vu = HERM ? vl : w * conj(K.Vu(b, l, m));
            const double mm = K.m(n, m), kap = -mm * (2.0 * sign * En + 2.0 * S.E[m]);
#pragma unroll
            for (int r = 0; r < 3; ++r) {
                const cplx<double> P = (-mm) * conj(K.Vu(ax[r], m, n)), Pu = HERM ? P : (-mm) * K.Vu(ax[r], n, m);
                G[0].add(r, P, vu);
                if constexpr (!HERM) G[1].add(r, Pu, vl);
                Z.add(r, mk(-kap * Pu.im, kap * Pu.re), vl);
            }
        }
        add_pairs(std::true_type{});
        Z.zero();
#pragma unroll
        for (int q = 0; q < NS; ++q) G[q].zero();
        for (int k0 = 0; k0 < min(16 * nb + 16, nw); k0 += 4) {
            const int q = min(k0 + lk, nw - 1);
            const double w = k0 + lk >= nw || q > n ? 0.0 : q == n ? 0.5 : 1.0;
            const cplx<double> vl = w * K.Vu(b, n, q), vu = HERM ? vl : w * conj(K.Vu(b, q, n));
            const double mm = K.m(q, l), kap = mm * (2.0 * sign * S.E[q] + 2.0 * El);  // Q enters with -
#pragma unroll
            for (int r = 0; r < 3; ++r) {
                const cplx<double> Pu = (-mm) * K.Vu(ax[r], q, l), P = HERM ? Pu : (-mm) * conj(K.Vu(ax[r], l, q));
                G[0].add(r, vu, P);
                if constexpr (!HERM) G[1].add(r, vl, Pu);
                Z.add(r, vl, mk(-kap * Pu.im, kap * Pu.re));
            }
        }
        add_pairs(std::false_type{});
#pragma unroll
        for (int q = 0; q < 7; ++q) cut_tile_add(S, nw, nb, lb, o[q], q == 6 ? b * 4 : ax[1 + q / 3] * 3 + ax[q % 3]);
    }
}

// DerMorb with external terms for sign = +1 and complex128 channels, every needed cut into S.cut (internal
// terms too when `in`).  Next to eval_dermorb_in (A, V Hermitian; B is not):
//   Q^a_nl also holds (2 E_n conj(A^a_ln) + 2 conj(B^a_ln)) / (E_l - E_n);
//   formula_task's kinds 2 and 3 together are Re -2 P^a_nl (E_n FA + FB)^{bd}_ln to the pair of a and b, with A
//     and B in the place of V and A', B' in that of W / 2;
//   kind 4's Omega block, -2 Re (P^d A^b)_ln V^e_nl over l, n < c, belongs to the pair (n, m) of A^b_mn with
//     (V^e P^d)_nm, and to that of P^d_nm with (V^e A^b)_nm;
//   kinds 6 and 7 cancel, 2 Im tr V^e A^al A^be + 2 Im tr V^e A^be A^al, and the s5 terms vanish;
//   the per-band terms with O and C are pair values and r(max(n, l)).
// A task is a pair of 16-band blocks and one b, in two passes (V, then A and B), or the per-band terms of one c.
// 1287 k-points at nw = 18, a narrow window: 0.94 ms one by one, 0.50 together, 0.39 with V and A in LDS
// and the per-band terms as tasks.
template <typename T, bool LM, bool ST, bool SA, int NW>
__device__ __attribute__((always_inline)) void eval_dermorb_ex(const Smem& S, const KCtx<T, LM, ST, SA, NW>& K, bool in) {
    const int nw = K.n_(), tid = threadIdx.x, lane = tid & 63, lk = lane >> 4, li = lane & 15;
    const int nblk = (nw + 15) / 16, ntask = 6 * (nblk * (nblk + 1) / 2);
    const double win = in ? 1.0 : 0.0;
    for (;;) {
        int t = 0;
        if (lane == 0) t = atomicAdd(&S.misc[3], 1);
        t = __builtin_amdgcn_readfirstlane(t) * K.parts + K.part;
        if (t >= ntask) break;
        const int npair = ntask / 6, b = t / npair;
        int nb, lb;
        cut_tile_pair(t % npair, nblk, nb, lb);
        // the lane's pair (x, y) of a tile, its rows opaque (operands loaded anew, not kept in registers)
        auto pair = [&](int v, int& x, int& y) {
            int nn = 16 * nb + lk + 4 * v;
            asm volatile("" : "+v"(nn)::"memory");
            const int ll = 16 * lb + li;
            x = min(nn, nw - 1);
            y = min(ll, nw - 1);
            return nn < nw && ll < nw ? ll - nn : -1;
        };
        if (b >= 3) {
            const int c = b - 3;
            double g[3][4], r[3] = {0.0, 0.0, 0.0};
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                int x, y;
                const int dist = pair(v, x, y);
                const double m = K.m(x, y), Ex = S.E[x];
                const cplx<double> Oxy = K.getu(WBMI_ROLE_O + c, x, y), Oyx = K.getu(WBMI_ROLE_O + c, y, x);
                const cplx<double> Cxy = K.getu(WBMI_ROLE_C + c, x, y), Cyx = K.getu(WBMI_ROLE_C + c, y, x);
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    const cplx<double> Vxy = K.Vu(d, x, y), Vyx = K.Vu(d, y, x);
                    const double e = 2.0 * Ex * (conj(Oyx) * Vyx).re + (Cxy * Vyx + Vxy * Cyx).re;
                    g[d][v] = dist > 0 ? m * e : 0.0;
                    if (dist > 0) r[d] += (Oxy * Vyx + Oyx * Vxy).re;
                    if (dist == 0)
                        r[d] += (Oxy * Vxy).re + Ex * K.getu(WBMI_ROLE_OD + 3 * c + d, x, x).re + K.getu(WBMI_ROLE_CD + 3 * c + d, x, x).re;
                }
            }
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                cut_tile_add(S, nw, nb, lb, g[d], c * 3 + d);
                r[d] = wave_sum(r[d], 0x30);
                if (lane < 16 && 16 * lb + lane < nw) atomicAdd(&S.acc[(16 * lb + lane) * 9 + c * 3 + d], r[d]);
            }
            continue;
        }
        if (!cut_tile_needed(S, nw, nb, lb)) continue;
        int ax[3];  // the indices b, b + 1, b + 2: everything below is relative to b
#pragma unroll
        for (int r = 0; r < 3; ++r) ax[r] = (b + r) % 3;
        // the pairs' values: components (c, d) relative to b, c = 1, 2 in [0, 6), (0, 0) in [6]
        double o[7][4];
#pragma unroll
        for (int q = 0; q < 7; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) o[q][v] = 0.0;
        const int n = min(16 * nb + li, nw - 1), l = min(16 * lb + li, nw - 1);
        const double En = S.E[n], El = S.E[l];
        // weight of the summed band k0 + lk: beyond the limit counted fully, on it half
        auto above = [&](int k0) { return k0 + lk >= nw || k0 + lk < l ? 0.0 : k0 + lk == l ? 0.5 : 1.0; };
        auto below = [&](int k0) { return k0 + lk >= nw || k0 + lk > n ? 0.0 : k0 + lk == n ? 0.5 : 1.0; };
        const int kmax = min(16 * nb + 16, nw);
        // Q^a_xy, x inside
        auto Qof = [&](int a, int x, int y, double m, double Ex, double Ey, cplx<double> P) {
            const double kap = -win * m * (2.0 * Ex + 2.0 * Ey);
            const cplx<double> A = K.Au(a, y, x), B = K.getu(WBMI_ROLE_B + a, y, x);
            return mk(-kap * P.im - m * (2.0 * Ex * A.re + 2.0 * B.re), kap * P.re + m * (2.0 * Ex * A.im + 2.0 * B.im));
        };
        {
            CutAcc G, Z, D;  // P V or V P; Q V or -V Q; V A
            auto add_pairs = [&](auto first) {
                constexpr bool FIRST = decltype(first)::value;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    int x, y;
                    const bool ok = pair(v, x, y) > 0;
                    const double m = K.m(x, y);
                    cplx<double> P[3], Q[3];
#pragma unroll
                    for (int r = 0; r < 3; ++r) {
                        P[r] = (-m) * K.Vu(ax[r], x, y);
                        Q[r] = Qof(ax[r], x, y, m, S.E[x], S.E[y], P[r]);
                    }
#pragma unroll
                    for (int d = 0; d < 3; ++d) {
                        cplx<double> f = G.get(d, v);
                        const cplx<double> h = f;
                        if constexpr (FIRST) f = 0.5 * K.getu(WBMI_ROLE_W + 3 * b + ax[d], x, y) - f;
                        const cplx<double> A = FIRST ? mk(0.0, 0.0) : K.Au(ax[d], x, y);
#pragma unroll
                        for (int a = 0; a < 3; ++a) {
                            const double s = (Q[a] * conj(f)).re - (Z.get(a, v) * conj(P[d])).re;
                            if (a != 0) {
                                const double e = pair_sign(a, 0) * s;
                                o[(third_index(a, 0) - 1) * 3 + d][v] += ok ? e : 0.0;
                            }
                            if (a != d) {
                                double e = s - 2.0 * win * (P[a] * conj(h)).im;
                                // the Omega block's A^d with (V P^a) and P^a with (V A^d)
                                if constexpr (!FIRST)
                                    e -= 2.0 * ((G.get(a, v) * conj(A)).re + (P[a] * conj(D.get(d, v))).re);
                                e *= pair_sign(a, d);
                                const int c = third_index(a, d);
                                o[c == 0 ? 6 : (c - 1) * 3][v] += ok ? e : 0.0;
                            }
                        }
                    }
                    cut_pin(o, v);
                }
            };
            G.zero();
            Z.zero();
            for (int k0 = 16 * lb; k0 < nw; k0 += 4) {
                const int m = min(k0 + lk, nw - 1);
                const cplx<double> vl = above(k0) * K.Vu(b, m, l);
                const double mm = K.m(n, m), Em = S.E[m];
#pragma unroll
                for (int r = 0; r < 3; ++r) {
                    const cplx<double> P = (-mm) * conj(K.Vu(ax[r], m, n));
                    G.add(r, P, vl);
                    Z.add(r, Qof(ax[r], n, m, mm, En, Em, P), vl);
                }
            }
            add_pairs(std::true_type{});
            G.zero();
            Z.zero();
            D.zero();
            for (int k0 = 0; k0 < kmax; k0 += 4) {
                const int q = min(k0 + lk, nw - 1);
                const cplx<double> vl = below(k0) * K.Vu(b, n, q);
                const double mm = K.m(q, l), Eq = S.E[q];
#pragma unroll
                for (int r = 0; r < 3; ++r) {
                    const cplx<double> P = (-mm) * K.Vu(ax[r], q, l);
                    G.add(r, vl, P);
                    Z.add(r, vl, -Qof(ax[r], q, l, mm, Eq, El, P));
                    D.add(r, vl, K.Au(ax[r], q, l));
                }
            }
            add_pairs(std::false_type{});
        }
        {
            // A and B: f = conj(E_n FA + FB), the weight -2 P
            CutAcc G, H, Z;
            auto add_pairs = [&](auto first) {
                constexpr bool FIRST = decltype(first)::value;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    int x, y;
                    const bool ok = pair(v, x, y) > 0;
                    const double m = K.m(x, y), Ex = S.E[x];
                    cplx<double> P[3];
#pragma unroll
                    for (int r = 0; r < 3; ++r) P[r] = (-m) * K.Vu(ax[r], x, y);
#pragma unroll
                    for (int d = 0; d < 3; ++d) {
                        cplx<double> f = G.get(d, v);
                        if constexpr (FIRST)
                            f = Ex * conj(K.getu(WBMI_ROLE_AD + 3 * b + ax[d], y, x)) + conj(K.getu(WBMI_ROLE_BD + 3 * b + ax[d], y, x)) - Ex * f - H.get(d, v);
#pragma unroll
                        for (int a = 1; a < 3; ++a) {
                            cplx<double> z = Z.get(a, v);
                            if constexpr (FIRST) z += Ex * G.get(a, v);
                            const double s = -2.0 * (P[a] * conj(f)).re + (FIRST ? 2.0 : -2.0) * (z * conj(P[d])).re;
                            const double e = pair_sign(a, 0) * s;
                            o[(third_index(a, 0) - 1) * 3 + d][v] += ok ? e : 0.0;
                        }
                    }
                    cut_pin(o, v);
                }
            };
            // G = P A, H = P conj(B)^T, Z = P B
            G.zero();
            H.zero();
            Z.zero();
            for (int k0 = 16 * lb; k0 < nw; k0 += 4) {
                const int m = min(k0 + lk, nw - 1);
                const double w = above(k0), mm = K.m(n, m);
                const cplx<double> al = w * K.Au(b, m, l), bl = w * K.getu(WBMI_ROLE_B + b, m, l), bu = w * conj(K.getu(WBMI_ROLE_B + b, l, m));
#pragma unroll
                for (int r = 0; r < 3; ++r) {
                    const cplx<double> P = (-mm) * conj(K.Vu(ax[r], m, n));
                    G.add(r, P, al);
                    H.add(r, P, bu);
                    if (r > 0) Z.add(r, P, bl);
                }
            }
            add_pairs(std::true_type{});
            // G = (E_n A + B^+) P, Z = (E A + B) P with the summed band's energy
            G.zero();
            Z.zero();
            for (int k0 = 0; k0 < kmax; k0 += 4) {
                const int q = min(k0 + lk, nw - 1);
                const double w = below(k0), mm = K.m(q, l), Eq = S.E[q];
                const cplx<double> A = K.Au(b, n, q);
                const cplx<double> m1 = w * (En * A + conj(K.getu(WBMI_ROLE_B + b, q, n))), m2 = w * (Eq * A + K.getu(WBMI_ROLE_B + b, n, q));
#pragma unroll
                for (int r = 0; r < 3; ++r) {
                    const cplx<double> P = (-mm) * K.Vu(ax[r], q, l);
                    G.add(r, m1, P);
                    if (r > 0) Z.add(r, m2, P);
                }
            }
            add_pairs(std::false_type{});
        }
#pragma unroll
        for (int q = 0; q < 7; ++q) cut_tile_add(S, nw, nb, lb, o[q], q == 6 ? b * 4 : ax[1 + q / 3] * 3 + ax[q % 3]);
    }
    __syncthreads();
    for (int t = tid; t < nw * 9; t += (int)blockDim.x) {
        double v = S.cut[t + 9];
        for (int x = 0; x <= t / 9; ++x) v += S.acc[x * 9 + t % 9];
        S.cut[t + 9] = v;
    }
}

// Morb_Hpm (formula/covariant.py:390-414), every needed cut into S.cut: the sums over l outside are
// pair values, those over m inside are r(max(n, m)).  One wave per pair of 16-band blocks.
// 294 k-points at nw = 64, every cut: 1.72 ms with a loop over l per cut and band, 0.028 ms.
template <typename T, bool LM, bool ST, bool SA, int NW>
__device__ __attribute__((always_inline)) void eval_morb_cuts(const Smem& S, const KCtx<T, LM, ST, SA, NW>& K, bool in, bool ex,
                                                             double sign) {
    const int nw = K.n_(), tid = threadIdx.x, lane = tid & 63, lk = lane >> 4, li = lane & 15;
    const int nblk = (nw + 15) / 16;
    for (int t = tid >> 6; t < nblk * (nblk + 1) / 2; t += (int)blockDim.x >> 6) {
        int nb, lb;
        cut_tile_pair(t, nblk, nb, lb);
        double o[3][4], r[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int nn = 16 * nb + lk + 4 * v, ll = 16 * lb + li;
            const bool ok = nn < ll && ll < nw, okd = nn == ll && ll < nw;
            const int x = min(nn, nw - 1), y = min(ll, nw - 1);
            const double Ex = sign * S.E[x], Ey = S.E[y];
            cplx<double> D[3], Dt[3], A[3], At[3], B[3];
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                D[a] = K.Dp(a, x, y);
                Dt[a] = in ? K.Dp(a, y, x) : mk(0.0, 0.0);
                A[a] = ex ? K.A(a, x, y) : mk(0.0, 0.0);
                At[a] = ex ? K.A(a, y, x) : mk(0.0, 0.0);
                B[a] = ex ? K.B(a, y, x) : mk(0.0, 0.0);
            }
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const int al = c == 2 ? 0 : c + 1, be = c == 0 ? 2 : c - 1;
                double g = 0.0, w = 0.0;
                if (in) g += 2.0 * (Ey + Ex) * (D[al] * Dt[be]).im;
                if (ex) {
                    g += 2.0 * (D[be] * B[al] - D[al] * B[be]).re + 2.0 * Ex * (D[be] * At[al] - D[al] * At[be]).re;
                    w = 2.0 * (Ey + Ex) * (A[al] * At[be]).im;
                    if (ok) w += 2.0 * (S.E[x] + sign * Ey) * (At[al] * A[be]).im;
                    if (okd) w += K.C(c, x, x).re + Ex * K.O(c, x, x).re;
                }
                o[c][v] = ok ? g : 0.0;
                r[c] += ok || okd ? w : 0.0;
            }
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            cut_tile_add(S, nw, nb, lb, o[c], c);
            const double rs = wave_sum(r[c], 0x30);
            if (lane < 16 && 16 * lb + lane < nw) atomicAdd(&S.acc[(16 * lb + lane) * 9 + c], rs);
        }
    }
    __syncthreads();
    for (int t = tid; t < nw * 3 && ex; t += (int)blockDim.x) {
        const int c = t / 3 + 1, q = t % 3;
        double v = S.cut[c * 9 + q];
        for (int x = 0; x < c; ++x) v += S.acc[x * 9 + q];
        S.cut[c * 9 + q] = v;
    }
}

// Diagonal elements of the band-group blocks of Omega (formula/covariant.py:175-200) or, MORB, of
// Morb_H + sign E o Omega (formula/covariant.py:390-414) for the partition of the labels, added to
// S.acc[n][c], c = 0 .. 2; `single`: only for groups of one band.
// A wave takes 8 bands n by 8 bands l at a time and all three components: rows (n, l) and columns (l, n) of the
// channels are both read in runs of 8 elements, each element once, with no copy of V and A in LDS (which
// held one workgroup a CU at nw = 32) and no element read once per component.  Bound: the channels' bytes
// and the latency of the loads.  Against four lanes
// per (n, c) on LDS copies up to nw = 32 and one thread per (n, c) above: Omega of 4096 k-points at nw = 32
// 255 -> 105 us complex128, 127 -> 100 complex64; 5832 at nw = 24 172 -> 90 and 95 -> 78; 3375 at nw = 48
// 540 -> 201 and 490 -> 193.  Velocity products (one thread per (n, a, b), each Omega or Morb_Hpm element formed
// for every a and both orders) of 1331 k-points at nw = 18: 105 -> 28 (Omega), 186 -> 41 us (Morb_Hpm).
template <bool MORB, typename T, bool LM, bool ST, bool SA, int NW>
__device__ __attribute__((always_inline)) void diag_traces(const Smem& S, const KCtx<T, LM, ST, SA, NW>& K, bool in, bool ex, double sign,
                                                          bool single) {
    const int nw = K.n_(), lane = threadIdx.x & 63, nwave = (int)blockDim.x >> 6;
    const int n8 = (nw + 7) / 8, split = min(max(nwave / n8, 1), n8);  // waves that share 8 rows
    for (int t = threadIdx.x >> 6; t < n8 * split; t += nwave) {
        const int nn = 8 * (t % n8) + (lane >> 3), n = min(nn, nw - 1);
        const bool on = nn < nw && S.act[n] && !(single && S.ge[n] - S.gs[n] > 1);
        if (!__any(on)) continue;
        const int lab = S.lab[n];
        const double En = S.E[n];
        double v[3] = {0.0, 0.0, 0.0};
        for (int l0 = 8 * (t / n8); l0 < nw; l0 += 8 * split) {
            const int ll = l0 + (lane & 7), l = min(ll, nw - 1);
            if (!on || ll >= nw) continue;
            const bool same = S.lab[l] == lab;
            const double m = K.m(n, l), El = S.E[l];  // zero within the group
            // weights of the internal and the A A terms: Omega's and Morb_H's
            const double w = MORB ? El + sign * En : 1.0;
            cplx<double> D[3], Vt[3], At[3], Bt[3];
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                D[a] = K.getu(WBMI_ROLE_V + a, n, l);
                Vt[a] = in ? K.getu(WBMI_ROLE_V + a, l, n) : mk(0.0, 0.0);
                At[a] = ex ? K.getu(WBMI_ROLE_A + a, l, n) : mk(0.0, 0.0);
                if constexpr (MORB) Bt[a] = ex ? K.getu(WBMI_ROLE_B + a, l, n) : mk(0.0, 0.0);
            }
            if (ex && same) {
                // the A A terms, and O and C (D' is zero here)
                cplx<double> A[3];
#pragma unroll
                for (int a = 0; a < 3; ++a) A[a] = K.getu(WBMI_ROLE_A + a, n, l);
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    v[c] += 2.0 * w * (A[c == 2 ? 0 : c + 1] * At[c == 0 ? 2 : c - 1]).im;
                    if (l == n) {
                        const double o = K.getu(WBMI_ROLE_O + c, n, n).re;
                        v[c] += MORB ? K.getu(WBMI_ROLE_C + c, n, n).re + sign * En * o : o;
                    }
                }
            }
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                D[a] = (-m) * D[a];
                Vt[a] = m * Vt[a];  // D'_ln = -m_ln V_ln
                // the external terms' factor of D'_nl: A (Omega) or B + sign E_n A (Morb_Hpm)
                if constexpr (MORB) Bt[a] += (sign * En) * At[a];
                else Bt[a] = At[a];
            }
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const int al = c == 2 ? 0 : c + 1, be = c == 0 ? 2 : c - 1;
                double x = w * (D[al] * Vt[be]).im;
                if (ex) x += (D[be] * Bt[al] - D[al] * Bt[be]).re;
                v[c] += 2.0 * x;
            }
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const double x = wave_sum(v[c], 7);
            if ((lane & 7) == 0 && on) atomicAdd(&S.acc[n * 9 + c], x);
        }
    }
}

// Products with the velocity, acc[n][a][b] = Re sum_{m in G} V^a_nm H^b_mn: groups of one band from their
// diagonal elements H^b_nn in acc[n][b], larger ones from H(b, m, n)
template <typename T, bool LM, bool ST, bool SA, int NW, class FH>
__device__ __attribute__((always_inline)) void vel_times(const Smem& S, const KCtx<T, LM, ST, SA, NW>& K, FH H) {
    const int nw = K.n_(), tid = threadIdx.x;
    __syncthreads();
    for (int n = tid; n < nw; n += (int)blockDim.x) {
        if (!S.act[n] || S.ge[n] - S.gs[n] > 1) continue;
        const double h[3] = {S.acc[n * 9], S.acc[n * 9 + 1], S.acc[n * 9 + 2]};
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const double v = K.getu(WBMI_ROLE_V + a, n, n).re;
#pragma unroll
            for (int b = 0; b < 3; ++b) S.acc[n * 9 + a * 3 + b] = v * h[b];
        }
    }
    for (int t = tid; t < nw * 3; t += (int)blockDim.x) {
        const int n = t / 3, b = t % 3;
        if (!S.act[n] || S.ge[n] - S.gs[n] <= 1) continue;
        double v[3] = {0.0, 0.0, 0.0};
        for (int m = S.gs[n]; m < S.ge[n]; ++m) {
            const cplx<double> h = H(b, m, n);
#pragma unroll
            for (int a = 0; a < 3; ++a) v[a] += (K.V(a, n, m) * h).re;
        }
#pragma unroll
        for (int a = 0; a < 3; ++a) S.acc[n * 9 + a * 3 + b] = v[a];
    }
}

// Per-band values for the current partition (the labels'; cut >= 0: they are those of [0, cut), and M
// holds the unmasked dEinv) into S.acc[n][comp].
template <int F, typename T, bool LM, bool ST, bool SA, int NW>
__device__ __attribute__((always_inline)) void eval_partition(const Smem& S, const KCtx<T, LM, ST, SA, NW>& K, const wbmi_scan_params& p, int cut = -1) {
    const int nw = K.n_();
    const int tid = threadIdx.x;
    const bool in = p.internal_terms, ex = p.external_terms;
    if constexpr (LM)
        if (cut < 0) build_M<true>(S, nw);
    for (int t = tid; t < nw * 9; t += (int)blockDim.x) S.acc[t] = 0.0;
    __syncthreads();
    if (F == WBMI_FORMULA_IDENTITY) {
        for (int n = tid; n < nw; n += (int)blockDim.x)
            if (S.act[n]) S.acc[n * 9] = 1.0;
    } else if (F == WBMI_FORMULA_OMEGA) {
        diag_traces<false>(S, K, in, ex, 0.0, false);
    } else if (F == WBMI_FORMULA_MORB_HPM) {
        diag_traces<true>(S, K, in, ex, (double)p.sign, false);
    } else if (F == WBMI_FORMULA_VELOMEGA) {
        // Re sum_{n' in G} V^a_nn' Omega^b_n'n, Omega = s + s^+ (formula/formula.py:141-148)
        diag_traces<false>(S, K, in, ex, 0.0, true);
        vel_times(S, K, [&](int b, int m, int n) { return omega_s(K, b, m, n, in, ex) + conj(omega_s(K, b, n, m, in, ex)); });
    } else if (F == WBMI_FORMULA_VELHPLUS) {
        // Re sum_{n' in G} V^a_nn' Hpm^b_n'n with the group block of Morb_Hpm,
        // Hpm = Morb_H.nn + sign Eav o Omega.nn (formula/covariant.py:424-449,
        // formula/formula.py:141-148; FormulaProduct is additive)
        diag_traces<true>(S, K, in, ex, (double)p.sign, true);
        vel_times(S, K, [&](int b, int m, int n) {
            cplx<double> h = morbh_s(K, b, m, n, in, ex) + conj(morbh_s(K, b, n, m, in, ex));
            if (p.sign != 0)
                h += (p.sign * 0.5 * (S.E[m] + S.E[n])) * (omega_s(K, b, m, n, in, ex) + conj(omega_s(K, b, n, m, in, ex)));
            return h;
        });
    } else if (F == WBMI_FORMULA_DERSPIN) {
        // generalised derivative of the spin (formula/formula.py:95-107 with A = Xbar('SS'),
        // dA = Xbar('SS', 1)): Re [S'^{bd}_nn - sum_{l off} D^d_nl S^b_ln + sum_{l off} S^b_nl D^d_ln]
        for (int t = tid; t < nw * 9; t += (int)blockDim.x) {
            const int n = t / 9, b = (t % 9) / 3, d = t % 3;
            if (!S.act[n]) continue;
            cplx<double> v = K.Sd(b, d, n, n);
            for (int l = 0; l < nw; ++l) {
                v -= K.Dp(d, n, l) * K.S(b, l, n);
                v += K.S(b, n, l) * K.Dp(d, l, n);
            }
            S.acc[t] = v.re;
        }
    } else if (F == WBMI_FORMULA_SPIN) {
        // Re S^s_nn: the group trace of Xbar('SS') (formula/covariant.py:331-335)
        for (int t = tid; t < nw * 3; t += (int)blockDim.x) {
            const int n = t / 3, sp = t % 3;
            if (S.act[n]) S.acc[n * 9 + sp] = K.S(sp, n, n).re;
        }
    } else if (F == WBMI_FORMULA_VELSPIN) {
        // Re sum_{n' in G} V^a_nn' S^b_n'n (formula/formula.py:121-148, covariant.py:811-814)
        for (int t = tid; t < nw * 9; t += (int)blockDim.x) {
            const int n = t / 9, a = (t % 9) / 3, b = t % 3;
            if (!S.act[n]) continue;
            cplx<double> v = mk(0.0, 0.0);
            for (int m = S.gs[n]; m < S.ge[n]; ++m) v += K.V(a, n, m) * K.S(b, m, n);
            S.acc[t] = v.re;
        }
    } else if (F == WBMI_FORMULA_INVMASS) {
        // inverse effective mass, the generalised derivative of the velocity (formula/elementary.py:28-33,
        // formula/formula.py:95-107 with A = V, dA = W): Re [W^{bd}_nn - sum_{l off} D^d_nl V^b_ln
        // + sum_{l off} V^b_nl D^d_ln]
        for (int t = tid; t < nw * 9; t += (int)blockDim.x) {
            const int n = t / 9, b = (t % 9) / 3, d = t % 3;
            if (!S.act[n]) continue;
            cplx<double> v = K.W(b, d, n, n);
            for (int l = 0; l < nw; ++l) {
                v -= K.Dp(d, n, l) * K.V(b, l, n);
                v += K.V(b, n, l) * K.Dp(d, l, n);
            }
            S.acc[t] = v.re;
        }
    } else if (F == WBMI_FORMULA_VELVEL) {
        // Re sum_{n' in G} V^a_nn' V^b_n'n (FormulaProduct of two velocities, formula/covariant.py:817-820)
        for (int t = tid; t < nw * 9; t += (int)blockDim.x) {
            const int n = t / 9, a = (t % 9) / 3, b = t % 3;
            if (!S.act[n]) continue;
            cplx<double> v = mk(0.0, 0.0);
            for (int m = S.gs[n]; m < S.ge[n]; ++m) v += K.V(a, n, m) * K.V(b, m, n);
            S.acc[t] = v.re;
        }
    } else if (F == WBMI_FORMULA_VELVELVEL) {
        // [a][b][c] = Re sum_{m, l in G} V^a_nm V^b_ml V^c_ln (formula/formula.py:121-148), a = comp_slice
        const int a = p.comp_slice;
        for (int t = tid; t < nw * 9; t += (int)blockDim.x) {
            const int n = t / 9, b = (t % 9) / 3, c = t % 3;
            if (!S.act[n]) continue;
            cplx<double> v = mk(0.0, 0.0);
            for (int m = S.gs[n]; m < S.ge[n]; ++m)
                for (int l = S.gs[n]; l < S.ge[n]; ++l) v += K.V(a, n, m) * K.V(b, m, l) * K.V(c, l, n);
            S.acc[t] = v.re;
        }
    } else if (F == WBMI_FORMULA_MASSVEL) {
        // [a][b][c] = Re sum_{m in G} M^{ab}_nm V^c_mn, a = comp_slice
        const int a = p.comp_slice;
        for (int t = tid; t < nw * 9; t += (int)blockDim.x) {
            const int n = t / 9, b = (t % 9) / 3, c = t % 3;
            if (!S.act[n]) continue;
            cplx<double> v = mk(0.0, 0.0);
            for (int m = S.gs[n]; m < S.ge[n]; ++m) v += mass_xy(K, a, b, n, m) * K.V(c, m, n);
            S.acc[t] = v.re;
        }
    } else if (F == WBMI_FORMULA_HALL_SURF) {
        // VelMassVel X[a][b][c][d] = Re sum_{m, l in G} V^a_nm M^{bc}_ml V^d_ln, contracted
        for (int t = tid; t < nw * 9; t += (int)blockDim.x) {
            const int n = t / 9, j = (t % 9) / 3, i = t % 3;
            if (!S.act[n]) continue;
            const cplx<double> v = hall_contract(j, i, [&](int a, int b, int c, int d) {
                cplx<double> x = mk(0.0, 0.0);
                for (int m = S.gs[n]; m < S.ge[n]; ++m)
                    for (int l = S.gs[n]; l < S.ge[n]; ++l) x += K.V(a, n, m) * mass_xy(K, b, c, m, l) * K.V(d, l, n);
                return x;
            });
            S.acc[t] = v.re;
        }
    } else if (F == WBMI_FORMULA_HALL_SEA) {
        // MassMass X[a][b][c][d] = Re sum_{m in G} M^{ab}_nm M^{cd}_mn, its axes moved as
        // transpose(0, 4, 1, 2, 3) (Y[p][q][r][s] = X[q][r][s][p]), contracted
        for (int t = tid; t < nw * 9; t += (int)blockDim.x) {
            const int n = t / 9, j = (t % 9) / 3, i = t % 3;
            if (!S.act[n]) continue;
            const cplx<double> v = hall_contract(j, i, [&](int p0, int q, int r, int s4) {
                cplx<double> x = mk(0.0, 0.0);
                for (int m = S.gs[n]; m < S.ge[n]; ++m) x += mass_xy(K, q, r, n, m) * mass_xy(K, s4, p0, m, n);
                return x;
            });
            S.acc[t] = v.re;
        }
    } else if (F == WBMI_FORMULA_OMEGASPIN || F == WBMI_FORMULA_OMEGAOMEGA || F == WBMI_FORMULA_OMEGAHPLUS) {
        // Re sum_{n' in G} Omega^a_nn' Y^b_n'n, Omega = s + s^+, Y = S (OmegaS), Omega (OmegaOmega)
        // or Morb_Hpm with sign +1 (OmegaHplus) (formula/formula.py:121-148, covariant.py:849-866)
        for (int t = tid; t < nw * 9; t += (int)blockDim.x) {
            const int n = t / 9, a = (t % 9) / 3, b = t % 3;
            if (!S.act[n]) continue;
            cplx<double> v = mk(0.0, 0.0);
            for (int m = S.gs[n]; m < S.ge[n]; ++m) {
                const cplx<double> om = omega_s(K, a, n, m, in, ex) + conj(omega_s(K, a, m, n, in, ex));
                cplx<double> y;
                if (F == WBMI_FORMULA_OMEGASPIN) {
                    y = K.S(b, m, n);
                } else {
                    const cplx<double> ob = omega_s(K, b, m, n, in, ex) + conj(omega_s(K, b, n, m, in, ex));
                    if (F == WBMI_FORMULA_OMEGAOMEGA)
                        y = ob;
                    else
                        y = morbh_s(K, b, m, n, in, ex) + conj(morbh_s(K, b, n, m, in, ex)) +
                            (0.5 * (S.E[m] + S.E[n])) * ob;
                }
                v += om * y;
            }
            S.acc[t] = v.re;
        }
    } else if (F == WBMI_FORMULA_BANDVALUES) {
        // the caller's per-band shares of the group traces, 9 of them from row comp_slice * 9
        for (int t = tid; t < nw * 9; t += (int)blockDim.x) {
            const int n = t / 9, c = t % 9;
            if (S.act[n]) S.acc[t] = K.bv[n * K.nbv + p.comp_slice * 9 + c];
        }
    } else if (F == WBMI_FORMULA_DEROMEGA) {
        eval_deromega<false>(S, K, in, ex, 0, cut);
    } else if (F == WBMI_FORMULA_DERMORB) {
        eval_deromega<true>(S, K, in, ex, p.sign, cut);
    }
    __syncthreads();
}

// ---------------------------------------------------------------------------
// tetrahedron method (grid/tetrahedron.py:15-128, 269-281)
// ---------------------------------------------------------------------------

#define TETRA_SPLIT 1e-12  // minimum separation of sorted corner energies (tetrahedron.py:17-21)
#define TETRA_PAD 1e-11    // above max + TETRA_PAD every tetrahedron is fully occupied

// Occupied fraction (der 0) of a tetrahedron with linear energy between the corner values,
// or its der-th derivative in the Fermi level.  der 0 evaluates the three cubic pieces as
// products of ratios; der >= 1 differentiates their power-series form, with the
// coefficients grouped as the reference groups them (its rounding where corners nearly
// coincide).  No contraction into FMAs, so that the rounding is that of separate operations.
__device__ inline double tetra_occ(double ef, double a, double b, double c, double d, int der) {
#pragma clang fp contract(off)
    double t;
    if (a > b) { t = a; a = b; b = t; }
    if (c > d) { t = c; c = d; d = t; }
    if (a > c) { t = a; a = c; c = t; }
    if (b > d) { t = b; b = d; d = t; }
    if (b > c) { t = b; b = c; c = t; }
    const double e1 = a;
    const double e2 = b - e1 < TETRA_SPLIT ? e1 + TETRA_SPLIT : b;
    const double e3 = c - e2 < TETRA_SPLIT ? e2 + TETRA_SPLIT : c;
    const double e4 = d - e3 < TETRA_SPLIT ? e3 + TETRA_SPLIT : d;
    if (der == 0) {
        if (ef >= e4) return 1.0;
        if (ef < e1) return 0.0;
        if (ef >= e3) return 1.0 - ((ef - e4) / (e1 - e4)) * ((ef - e4) / (e2 - e4)) * ((ef - e4) / (e3 - e4));
        if (ef >= e2) {
            const double a13 = (ef - e1) / (e3 - e1), a14 = (ef - e1) / (e4 - e1);
            const double a23 = (ef - e2) / (e3 - e2), a24 = (ef - e2) / (e4 - e2);
            return a23 * a24 + a13 * (a14 * (1.0 - a24) + a24 * (1.0 - a23));
        }
        return ((ef - e1) / (e2 - e1)) * ((ef - e1) / (e3 - e1)) * ((ef - e1) / (e4 - e1));
    }
    if (ef >= e4 || ef < e1) return 0.0;
    double c1, c2, c3;
    if (ef >= e3) {
        const double r3 = 1.0 / ((e4 - e1) * (e4 - e2) * (e4 - e3));
        c1 = 3.0 * (e4 * e4) * r3;
        c2 = -3.0 * e4 * r3;
        c3 = r3;
    } else if (ef >= e2) {
        const double r2 = 1.0 / ((e3 - e1) * (e4 - e1) * (e3 - e2) * (e4 - e2));
        c1 = (-2.0 * e1 * ((e3 - e2) * (e4 - e2)) + (2.0 * e2 * e4 + e2 * e2) * (e1 - e3) +
              (e1 * e2 + e2 * e3 + e1 * e3) * (e2 - e4)) * r2;
        c2 = (((e3 - e2) * (e4 - e2)) - (e1 - e3) * (2.0 * e2 + e4) - (e3 + e1 + e2) * (e2 - e4)) * r2;
        c3 = r2 * (e1 + e2 - e3 - e4);
    } else {
        const double r1 = 1.0 / ((e2 - e1) * (e3 - e1) * (e4 - e1));
        c1 = 3.0 * (e1 * e1) * r1;
        c2 = -3.0 * e1 * r1;
        c3 = r1;
    }
    if (der == 1) return c1 + ef * (2.0 * c2 + 3.0 * c3 * ef);
    if (der == 2) return 2.0 * c2 + 6.0 * c3 * ef;
    return 6.0 * c3;
}

// Weight of one band at one k: the mean over the 12 tetrahedra joining the centre to the
// two triangles (F00, F01, F11), (F00, F10, F11) of each face of the parallelepiped, faces
// taken as x = side, y = side, z = side for side 0 then 1.  C[ix*4 + iy*2 + iz].
__device__ inline double tetra_band(double ef, double ec, const double* C, int der, int ncorner) {
    // tetrahedral K-blocks: one tetrahedron, the 4 corners themselves (tetrahedron.py:204-209)
    if (ncorner == 4) return tetra_occ(ef, C[0], C[1], C[2], C[3], der);
    double occ = 0.0;
#pragma unroll
    for (int side = 0; side < 2; ++side) {
        // face x = side: F[a][b] = C[side*4 + a*2 + b]
        occ += tetra_occ(ef, ec, C[side * 4], C[side * 4 + 1], C[side * 4 + 3], der);
        occ += tetra_occ(ef, ec, C[side * 4], C[side * 4 + 2], C[side * 4 + 3], der);
        // face y = side: F[a][b] = C[a*4 + side*2 + b]
        occ += tetra_occ(ef, ec, C[side * 2], C[side * 2 + 1], C[4 + side * 2 + 1], der);
        occ += tetra_occ(ef, ec, C[side * 2], C[4 + side * 2], C[4 + side * 2 + 1], der);
        // face z = side: F[a][b] = C[a*4 + b*2 + side]
        occ += tetra_occ(ef, ec, C[side], C[2 + side], C[6 + side], der);
        occ += tetra_occ(ef, ec, C[side], C[4 + side], C[6 + side], der);
    }
    return occ / 12.0;
}

// first index e with Ef[e] >= x (lower) or Ef[e] > x (upper) in the ascending Ef[0..n)
__device__ inline int ef_bound(const double* __restrict__ Ef, int n, double x, bool upper) {
    int lo = 0, hi = n;
    while (lo < hi) {
        const int m = (lo + hi) >> 1;
        if (upper ? Ef[m] <= x : Ef[m] < x) lo = m + 1;
        else hi = m;
    }
    return lo;
}

// Adds the in-range groups' values S.tv with their tetrahedron weights (static.py:119-125;
// TetraWeights.weights_all_band_groups, tetrahedron.py:212-255): band b of group g adds
// tv[g] / |g| * w_b(Ef).  w_b is 0 below the band's lowest energy over centre and corners
// and (der 0) 1 above its highest: that part is one step row of the histogram; the levels
// in between are evaluated one by one, spread over all threads.
static __device__ void tetra_accumulate(const Smem& S, const ScanArgs& args, int ncomp, double* __restrict__ hist) {
    const int nw = args.nw, nEF = args.nEF, der = args.p.fder, tid = threadIdx.x;
    for (int b = tid; b < nw; b += (int)blockDim.x) {
        const int g = S.tg[b];
        int lo = 0, hi = 0;
        if (g >= 0 && S.gin[g]) {  // g < 0: a band in no group (the odd last band under degen_Kramers)
            lo = ef_bound(args.Ef, nEF, S.tEmn[b], false);
            hi = ef_bound(args.Ef, nEF, S.tEmx[b] + TETRA_PAD, true);
            const double f = args.weight / (S.gb[g + 1] - S.gb[g]);
            if (der == 0 && hi < nEF)
                for (int c = 0; c < ncomp; ++c) unsafeAtomicAdd(hist + (int64_t)hi * ncomp + c, f * S.tv[g * 9 + c]);
            if (der == -1) {
                // 1 - occupation: 1 below the band's span (rows 0 .. hi-1), minus the occupation inside
                for (int c = 0; c < ncomp; ++c) {
                    unsafeAtomicAdd(hist + c, f * S.tv[g * 9 + c]);
                    if (hi < nEF) unsafeAtomicAdd(hist + (int64_t)hi * ncomp + c, -f * S.tv[g * 9 + c]);
                }
            }
        }
        S.tlo[b] = lo;
        S.tcnt[b] = hi - lo;
    }
    __syncthreads();
    if (tid == 0) {
        S.tpre[0] = 0;
        for (int b = 0; b < nw; ++b) S.tpre[b + 1] = S.tpre[b] + S.tcnt[b];
    }
    __syncthreads();
    const int total = S.tpre[nw];
    for (int t = tid; t < total; t += (int)blockDim.x) {
        // band b with tpre[b] <= t < tpre[b + 1]
        int lo = 0, hi = nw;
        while (hi - lo > 1) {
            const int m = (lo + hi) >> 1;
            if (S.tpre[m] <= t) lo = m;
            else hi = m;
        }
        const int b = lo, e = S.tlo[b] + (t - S.tpre[b]), g = S.tg[b];
        const double w = der == -1 ? -tetra_band(args.Ef[e], S.E[b], S.tC + b * 8, 0, args.tetra)
                                   : tetra_band(args.Ef[e], S.E[b], S.tC + b * 8, der, args.tetra);
        const double f = args.weight * w / (S.gb[g + 1] - S.gb[g]);
        for (int c = 0; c < ncomp; ++c)
            unsafeAtomicAdd(hist + (int64_t)(nEF + e) * ncomp + c, f * S.tv[g * 9 + c]);
    }
}

// select_bands share of the group [a, b) (utility.py:398-403): 1 without a selection
__device__ inline double group_selected(const wbmi_scan_params& p, int a, int b) {
    if (!p.band_weight) return 1.0;
    double s = 0.0;
    for (int n = a; n < b; ++n) s += p.band_weight[n];
    return s / (double)(b - a);
}

// Fermi-level bin of a group with mean energy E (static.py:131-136): 0 for
// E < EFmin (added to every level), ceil((E - EFmin)/dEF) up to EFmax, -1 = none.
__device__ inline int fermi_bin(const wbmi_scan_params& p, double E) {
    if (E < p.EFmin) return 0;
    if (E <= p.EFmax) {
        const int bin = (int)ceil((E - p.EFmin) / p.dEF);
        return bin < p.nEF_extra ? bin : -1;
    }
    return -1;
}

// MODE: 0 = Fermi-level bins, 1 = tetrahedron weights, 2 = per-band table (hist is then
// out[nk][nw][ncomp]: each band gets its group's trace / group size, or, for the identity
// formula, the group's mean energy)

// Workgroup sizes of the DerOmega / DerMorb kernels.  The epilogues and the LDS and L2 latencies, not
// the products, bound them, so what counts is waves in flight from workgroups in different phases: four
// waves per SIMD at 128 registers, in as many workgroups as the LDS of a CU holds (staged V, A in their
// storage type).  DerOmega at 4096 k-points, nw = 32: complex64 (two workgroups of 8 waves) 0.78 ms
// against 0.94 for one of 12 waves; complex128 fits one workgroup, 12 waves of 168 registers 0.95 ms
// against 1.01 for 16 of 128.  nw = 18, 1331 k-points: 0.20 ms in 4-wave workgroups, 0.25 in 12-wave ones.
// Within-group sums of large groups (the Fermi sea, the cuts of DerMorb) are a second product of the
// task instead of a loop per element, ranges of the summed index without a term are left out, and the
// sea is one more group of the main partition: DerMorb of 294 k-points at nw = 64, internal terms,
// every cut: 39.7 -> 7.6 ms; with external terms at nw = 18 and a narrow window 2.02 -> 0.92 ms per
// 1287 k-points; DerOmega of 150 k-points at nw = 128 10.4 -> 2.1 ms.
// The tetrahedron variants (MODE 1) keep 8 waves: their weight code is inlined.
__host__ __device__ constexpr int scan_min_waves(bool tasks, int nth) { return !tasks ? 1 : nth == 768 ? 3 : 4; }

// NW > 0: the kernel for nw = NW only, every size and row stride a compile-time constant
template <typename T, int F, bool LM, bool ST, int MODE, int NW, int NTH>
__global__ void __launch_bounds__(NTH, SC_IS_DERMORB_CUTS(F) ? 2 : (scan_min_waves((F == WBMI_FORMULA_DEROMEGA || F == WBMI_FORMULA_DERMORB) && MODE != 1, NTH)))
k_static_scan(ScanArgs args, const double* __restrict__ Eall, const cplx<T>* __restrict__ Xall, double* __restrict__ hist) {
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    const wbmi_scan_params& p = args.p;
    const int nw = NW > 0 ? NW : args.nw, ld = nw + 1;
    // the workgroups of one k-point (args.parts) follow each other on one XCD (workgroups go round the
    // XCDs in turn), so that its channels come from that XCD's L2: 294 k-points at nw = 64, complex64, DerOmega
    // 364 -> 339 us, DerMorb 446 -> 431; at nw = 128 no difference (2.88 -> 2.85 ms)
    const int parts = args.parts, unit = (int)blockIdx.x >> SC_XCD_LOG;
    const int64_t k = parts > 1 ? (int64_t)(unit / parts) * SC_XCD + (blockIdx.x & (SC_XCD - 1)) : blockIdx.x;
    if (parts > 1 && k >= args.nk) return;
    const int tid = threadIdx.x;
    if (MODE != 2) hist += k * args.hist_stride;
    constexpr bool tasks = F == WBMI_FORMULA_DEROMEGA || F == WBMI_FORMULA_DERMORB;
    static_assert(tasks || SC_IS_DERMORB_CUTS(F) || !ST, "V and A are staged for DerOmega and DerMorb");
    constexpr bool SA = ST;
    constexpr bool stage_v = ST;
    const bool stage_a = SA && p.external_terms;
    constexpr bool tetra = MODE == 1;  // compile-time: the Fermi-bin kernels carry no tetrahedron code
    constexpr bool tab = MODE == 2;
    const Smem S = make_smem(smem_raw, nw, LM, stage_v, stage_a, tetra, sizeof(cplx<T>));
    for (int n = tid; n < nw; n += (int)blockDim.x) S.E[n] = Eall[k * nw + n];
    for (int r = tid; r < WBMI_NROLES; r += (int)blockDim.x) S.ch[r] = p.ch[r];
    if (tetra)
        for (int t = tid; t < args.tetra * nw; t += (int)blockDim.x) {
            const int c = t / nw, b = t % nw;
            S.tC[b * 8 + c] = args.Ec[c * args.ec_stride + k * nw + b];
        }
    __syncthreads();
    if (tetra) {
        // band energy range over the centre and the corners (tetrahedron.py:189-193)
        for (int b = tid; b < nw; b += (int)blockDim.x) {
            double mn = S.E[b], mx = S.E[b];
            for (int c = 0; c < args.tetra; ++c) {
                mn = fmin(mn, S.tC[b * 8 + c]);
                mx = fmax(mx, S.tC[b * 8 + c]);
            }
            S.tEmn[b] = mn;
            S.tEmx[b] = mx;
        }
        __syncthreads();
    }
    const cplx<T>* Xk = Xall + k * (int64_t)args.nch * nw * nw;
    if (stage_v) {
        // SB elements per thread and pass, indices clamped into range (a thread past the end
        // rewrites the last element with its own value): no branches, so the scheduler issues all
        // of a pass's loads before its first LDS store
        constexpr int SB = NW > 0 ? (3 * NW * NW + NTH - 1) / NTH : 4;
        const int nw2 = nw * nw, n3 = 3 * nw2;
        const cplx<T>* src[2][3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            src[0][a] = Xk + (int64_t)S.ch[WBMI_ROLE_V + a] * nw2;
            src[1][a] = Xk + (int64_t)(stage_a ? S.ch[WBMI_ROLE_A + a] : 0) * nw2;
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            if (q == 1 && !stage_a) break;
            cplx<T>* dst = (cplx<T>*)(q == 0 ? S.V : S.A);
            for (int t0 = 0; t0 < n3; t0 += SB * NTH) {
                cplx<T> v[SB];
                int lo[SB];
#pragma unroll
                for (int u = 0; u < SB; ++u) {
                    const int t = min(t0 + tid + NTH * u, n3 - 1);
                    const int a = t >= 2 * nw2 ? 2 : t >= nw2 ? 1 : 0, xy = t - a * nw2;
                    const int x = xy / nw;
                    lo[u] = (a * nw + x) * ld + xy - x * nw;
                    v[u] = (a == 0 ? src[q][0] : a == 1 ? src[q][1] : src[q][2])[xy];
                }
#pragma unroll
                for (int u = 0; u < SB; ++u) dst[lo[u]] = v[u];
            }
        }
    }
    constexpr int ncomp = ncomp_of<F>();
    constexpr bool additive = F == WBMI_FORMULA_IDENTITY || F == WBMI_FORMULA_OMEGA ||
                              F == WBMI_FORMULA_DEROMEGA || F == WBMI_FORMULA_VELOMEGA ||
                              F == WBMI_FORMULA_VELHPLUS || F == WBMI_FORMULA_DERSPIN ||
                              F == WBMI_FORMULA_VELSPIN || F == WBMI_FORMULA_SPIN || F == WBMI_FORMULA_INVMASS ||
                              F == WBMI_FORMULA_VELVEL || F == WBMI_FORMULA_VELVELVEL || F == WBMI_FORMULA_MASSVEL ||
                              F == WBMI_FORMULA_HALL_SURF || F == WBMI_FORMULA_HALL_SEA ||
                              F == WBMI_FORMULA_BANDVALUES || F == WBMI_FORMULA_OMEGASPIN ||
                              F == WBMI_FORMULA_OMEGAOMEGA || F == WBMI_FORMULA_OMEGAHPLUS;

    // band groups (grid/tetrahedron.py:132-162, data_K.py:172-186), formed by wave 0: each lane
    // owns bands lane and lane + 64 (nw <= 128); borders from two ballots and popcounts, one
    // lane per group for its range test and mean energy, wave reductions for the sea group
    if (tid < 64) {
        const int lane = tid;
        const double thr = p.degen_thresh;
        auto is_border = [&](int i) {  // i in [0, nw]
            bool b = i == 0 || i == nw || (i < nw && S.E[i] - S.E[i - 1] > thr);
            if (p.degen_Kramers && (i & 1)) b = false;
            return b;
        };
        const bool b0 = lane <= nw && is_border(lane);
        const bool b1 = lane + 64 <= nw && is_border(lane + 64);
        const bool b2 = lane == 0 && nw == 128 && is_border(128);
        const uint64_t m0 = __ballot(b0), m1 = __ballot(b1);
        const uint64_t below = lane ? (~0ull >> (64 - lane)) : 0ull;
        const int n0 = __popcll(m0), n1 = __popcll(m1);
        if (b0) S.gb[__popcll(m0 & below)] = lane;
        if (b1) S.gb[n0 + __popcll(m1 & below)] = lane + 64;
        if (b2) S.gb[n0 + n1] = 128;
        const int nb = n0 + n1 + (nw == 128 && is_border(128) ? 1 : 0);
        const int ng = nb - 1;
        // degen_Kramers keeps only even borders, so with odd nw the last band is in no group
        // (grid/tetrahedron.py:132-136): it is an "out" band of every group and adds nothing itself
        for (int i = lane; i < nw; i += 64) S.tg[i] = -1;
        wave_lds_sync();
        int first_in = nw, last_in = 0;
        for (int g = lane; g < ng; g += 64) {
            const int a = S.gb[g], b = S.gb[g + 1];
            int inr;
            if (tab) {
                inr = 1;  // every group (Tabulator, tabulate.py:25-31)
            } else if (tetra) {
                // range over centre and corners against [Ef[0], Ef[-1]] (tetrahedron.py:140-152)
                double mn = S.tEmn[a], mx = S.tEmx[a];
                for (int i = a; i < b; ++i) {
                    mn = fmin(mn, S.tEmn[i]);
                    mx = fmax(mx, S.tEmx[i]);
                    S.tg[i] = g;
                }
                inr = (mx >= p.EFmin) && (mn <= p.EFmax);
            } else {
                inr = (S.E[b - 1] >= p.EFmin) && (S.E[a] <= p.EFmax);
            }
            S.gin[g] = inr;
            if (inr) {
                first_in = min(first_in, a);
                last_in = max(last_in, b);
            }
            double sum = 0.0;
            for (int i = a; i < b; ++i) sum += S.E[i];
            S.gw[g] = sum / (b - a);
        }
        for (int o = 32; o >= 1; o >>= 1) {
            first_in = min(first_in, __shfl_xor(first_in, o));
            last_in = max(last_in, __shfl_xor(last_in, o));
        }
        int sea_lo = 0, sea_hi = 0;
        if (p.fder == 0 && !tab) {
            // bands below the range, up to the first group in it (data_K.py:178-185;
            // tetra: highest energy over centre and corners below Ef[0], tetrahedron.py:155-162)
            int hi = 0, lo = 0;
            for (int i = lane; i < nw; i += 64) {
                if ((tetra ? S.tEmx[i] : S.E[i]) < p.EFmin) hi = i + 1;
                // tetra with Emin: bands entirely below Emin stay out (tetrahedron.py:246-251)
                if (tetra && p.erange && S.tEmx[i] < p.Emin) lo = i + 1;
            }
            for (int o = 32; o >= 1; o >>= 1) {
                hi = max(hi, __shfl_xor(hi, o));
                lo = max(lo, __shfl_xor(lo, o));
            }
            sea_hi = first_in < hi ? first_in : hi;
            sea_lo = lo < sea_hi ? lo : sea_hi;
        } else if (tetra && p.fder == -1) {
            // hole-like: bands whose lowest energy lies above Ef[-1], from the end of the last
            // group in range on (tetrahedron.py:165-172,246-253)
            int bandmin = nw, bandmax = nw;
            for (int i = lane; i < nw; i += 64) {
                if (S.tEmn[i] > p.EFmax) bandmin = min(bandmin, i);
                // with Emax: bands entirely above Emax stay out (tetrahedron.py:252-258)
                if (p.erange && S.tEmn[i] > p.Emax) bandmax = min(bandmax, i);
            }
            for (int o = 32; o >= 1; o >>= 1) {
                bandmin = min(bandmin, __shfl_xor(bandmin, o));
                bandmax = min(bandmax, __shfl_xor(bandmax, o));
            }
            if (bandmin < last_in) bandmin = last_in;
            if (bandmin < bandmax) {
                sea_lo = bandmin;
                sea_hi = bandmax;
            }
        }
        if (lane == 0) {
            S.misc[0] = ng;
            S.misc[1] = sea_lo;
            S.misc[2] = sea_hi;
        }
    }
    __syncthreads();
    const int ng = S.misc[0];
    const int sea_lo = S.misc[1], sea_hi = S.misc[2];

    KCtx<T, LM, ST, SA, NW> K;
    K.X = Xk;
    K.nw = nw;
    K.ld = ld;
    K.ch = S.ch;
    K.E = S.E;
    K.M = S.M;
    K.lab = S.lab;
    K.gs = S.gs;
    K.ge = S.ge;
    K.sV = (const cplx<T>*)S.V;
    K.sA = (const cplx<T>*)S.A;
    K.bv = (const double*)(const void*)Xall + k * (int64_t)nw * args.nch;
    K.nbv = args.nch;
    K.parts = parts;
    K.part = parts > 1 ? unit % parts : 0;

    if (additive || tab) {
        // main partition: every group at once (each group's trace with inn = the group,
        // out = the rest: the additive scan and the per-band table of any formula); a band in
        // no group (label -1) is an out band of every group
        for (int n = tid; n < nw; n += (int)blockDim.x) {
            S.lab[n] = -1;
            S.gs[n] = n;
            S.ge[n] = n;
            S.act[n] = 0;
        }
        __syncthreads();
        for (int g = 0; g < ng; ++g)
            for (int n = S.gb[g] + tid; n < S.gb[g + 1]; n += (int)blockDim.x) {
                S.lab[n] = g;
                S.gs[n] = S.gb[g];
                S.ge[n] = S.gb[g + 1];
                S.act[n] = S.gin[g];
            }
        __syncthreads();
        // the Fermi-sea group [sea_lo, sea_hi) (hole-like tetra: the bands above) as one more group:
        // it holds whole groups, none of them in range, and a group's values do not depend on how
        // the bands outside it are grouped
        for (int n = sea_lo + tid; n < sea_hi; n += (int)blockDim.x) {
            S.lab[n] = ng;
            S.gs[n] = sea_lo;
            S.ge[n] = sea_hi;
            S.act[n] = 1;
        }
        __syncthreads();
        eval_partition<F>(S, K, p);
        for (int t = tid; t < ng * ncomp; t += (int)blockDim.x) {
            const int g = t / ncomp, c = t % ncomp;
            if (tab) {
                double v;
                if (F == WBMI_FORMULA_IDENTITY) {
                    v = S.gw[g];  // Eavln: mean energy of the group
                } else {
                    v = 0.0;
                    for (int n = S.gb[g]; n < S.gb[g + 1]; ++n) v += S.acc[n * 9 + c];
                    v /= (S.gb[g + 1] - S.gb[g]);
                }
                for (int n = S.gb[g]; n < S.gb[g + 1]; ++n) hist[(k * nw + n) * ncomp + c] = v;
                continue;
            }
            if (tetra) {
                if (!S.gin[g]) continue;
                double s = 0.0;
                for (int n = S.gb[g]; n < S.gb[g + 1]; ++n) s += S.acc[n * 9 + c];
                S.tv[g * 9 + c] = s * group_selected(p, S.gb[g], S.gb[g + 1]);
                continue;
            }
            const int bin = S.gin[g] ? fermi_bin(p, S.gw[g]) : -1;
            if (bin < 0) continue;
            double s = 0.0;
            for (int n = S.gb[g]; n < S.gb[g + 1]; ++n) s += S.acc[n * 9 + c];
            unsafeAtomicAdd(hist + (int64_t)bin * ncomp + c, args.weight * s * group_selected(p, S.gb[g], S.gb[g + 1]));
        }
        __syncthreads();
        if (sea_hi > sea_lo) {
            // the sea's sum at every level (bin 0); one wave per component
            for (int c = tid >> 6; c < ncomp; c += (int)blockDim.x >> 6) {
                double v = 0.0;
                for (int n = sea_lo + (tid & 63); n < sea_hi; n += 64) v += S.acc[n * 9 + c];
                v = wave_sum(v, 63);
                if ((tid & 63) == 0) unsafeAtomicAdd(hist + c, args.weight * v);
            }
            __syncthreads();
        }
    } else {
        // non-additive: traces of the cumulative cuts [0, c) (static.py:109-117) at the borders of
        // the groups in range and of the sea
        constexpr bool all_cuts = SC_IS_DERMORB_CUTS(F) || F == WBMI_FORMULA_MORB_HPM;
        for (int n = tid; n <= nw; n += (int)blockDim.x) S.need[n] = 0;
        if constexpr (all_cuts) {
            for (int t = tid; t < nw * 9; t += (int)blockDim.x) S.acc[t] = S.cut[t + 9] = 0.0;
            for (int n = tid; n < nw; n += (int)blockDim.x) S.lab[n] = n;  // D' unmasked
            if (tid == 0) S.misc[3] = 0;                                  // task counter
        }
        if constexpr (LM) build_M<false>(S, nw);
        __syncthreads();
        for (int g = tid; g < ng; g += (int)blockDim.x)
            if (S.gin[g]) S.need[S.gb[g]] = S.need[S.gb[g + 1]] = 1;
        if (tid == 0 && sea_hi > sea_lo) S.need[sea_lo] = S.need[sea_hi] = 1;
        __syncthreads();
        if constexpr (SC_IS_DERMORB_IN(F)) {
            if (p.internal_terms) eval_dermorb_in<F == SC_DERMORB_IN>(S, K, (double)p.sign);
            __syncthreads();
        } else if constexpr (F == SC_DERMORB_EX) {
            eval_dermorb_ex(S, K, p.internal_terms);
            __syncthreads();
        } else if constexpr (all_cuts) {
            eval_morb_cuts(S, K, p.internal_terms, p.external_terms, (double)p.sign);
            __syncthreads();
        } else {
            for (int cidx = 1; cidx <= nw; ++cidx) {
                if (!S.need[cidx]) continue;
                for (int n = tid; n < nw; n += (int)blockDim.x) {
                    int inn = n < cidx;
                    S.lab[n] = inn ? 0 : 1;
                    S.gs[n] = inn ? 0 : cidx;
                    S.ge[n] = inn ? cidx : nw;
                    S.act[n] = inn;
                }
                __syncthreads();
                eval_partition<F>(S, K, p, cidx);
                for (int c = tid >> 6; c < ncomp; c += (int)blockDim.x >> 6) {
                    double v = 0.0;
                    for (int n = tid & 63; n < cidx; n += 64) v += S.acc[n * 9 + c];
                    v = wave_sum(v, 63);
                    if ((tid & 63) == 0) S.cut[cidx * 9 + c] = v;
                }
                __syncthreads();
            }
        }
        for (int c = tid; c < ncomp; c += (int)blockDim.x) S.cut[c] = 0.0;
        __syncthreads();
        for (int t = tid; t < ng * ncomp; t += (int)blockDim.x) {
            const int g = t / ncomp, c = t % ncomp;
            if (tetra) {
                if (S.gin[g])
                    S.tv[g * 9 + c] = (S.cut[S.gb[g + 1] * 9 + c] - S.cut[S.gb[g] * 9 + c]) *
                                      group_selected(p, S.gb[g], S.gb[g + 1]);
                continue;
            }
            const int bin = S.gin[g] ? fermi_bin(p, S.gw[g]) : -1;
            if (bin < 0) continue;
            const double s = S.cut[S.gb[g + 1] * 9 + c] - S.cut[S.gb[g] * 9 + c];
            unsafeAtomicAdd(hist + (int64_t)bin * ncomp + c, args.weight * s * group_selected(p, S.gb[g], S.gb[g + 1]));
        }
        if (sea_hi > sea_lo)
            for (int c = tid; c < ncomp; c += (int)blockDim.x)
                unsafeAtomicAdd(hist + c, args.weight * (S.cut[sea_hi * 9 + c] - S.cut[sea_lo * 9 + c]));
    }
    if (tetra) {
        __syncthreads();
        tetra_accumulate(S, args, ncomp, hist);
    }
}

template <typename T, int F, bool LM, bool ST, int MODE, int NW = 0, int NTH = SC_THREADS>
static int launch_scan_t(wbmi_ctx* ctx, int nk, const ScanArgs& a, const double* E, const void* X, double* hist) {
    const bool stage_a = ST && a.p.external_terms;
    const size_t lds = smem_offsets(a.nw, LM, ST, stage_a, MODE == 1, sizeof(cplx<T>)).total;
    if (lds > SC_LDS) return wbmi_fail(ctx, WBMI_ERR_ARG, "wbmi_static_scan: %zu bytes of LDS needed", lds);
    // DerOmega / DerMorb of few k-points: several workgroups share a k-point's tasks, so that there are
    // about four per CU (above nw = 32, where a k-point's tasks fill them; two below).  The kernels of all cuts, complex64
    // internal terms, 294 k-points at nw = 64: 446 us with two per CU, 332 with four, 348 with more; complex128
    // external terms at nw = 40 529, 416 and 498; 300 at nw = 18 120, 122 and 171.  Fermi bins only: the
    // other modes use a k-point's sums before they are complete.
    constexpr bool tasks = F == WBMI_FORMULA_DEROMEGA || F == WBMI_FORMULA_DERMORB;
    const int want = a.nw > 32 ? 1024 : 512;
    const int parts = (tasks || SC_IS_DERMORB_CUTS(F)) && MODE == 0 && nk < want ? std::min(8, want / nk) : 1;
    WBMI_HIP_CHECK(ctx, hipFuncSetAttribute((const void*)k_static_scan<T, F, LM, ST, MODE, NW, NTH>,
                                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    ScanArgs args = a;
    args.nk = nk;
    args.parts = parts;
    const int grid = parts > 1 ? (nk + SC_XCD - 1) / SC_XCD * SC_XCD * parts : nk;
    hipLaunchKernelGGL((k_static_scan<T, F, LM, ST, MODE, NW, NTH>), dim3(grid), dim3(NTH), lds, ctx->stream, args, E,
                       (const cplx<T>*)X, hist);
    WBMI_LAUNCH_CHECK(ctx);
    return WBMI_OK;
}

// dEinv o Off in LDS up to SC_M_NW (DerOmega / DerMorb: wherever it fits: an element formed on the fly
// costs a division), else formed on the fly; V and A in LDS up to SC_LDS_NW for the formulas with
// wave tasks.  Sizes: see scan_min_waves
template <typename T, int F, int MODE>
static int launch_scan(wbmi_ctx* ctx, int nk, const ScanArgs& a, const double* E, const void* X, double* hist) {
    constexpr bool tasks = F == WBMI_FORMULA_DEROMEGA || F == WBMI_FORMULA_DERMORB;
    // the kernels of all cuts: Morb_Hpm reads each dEinv once; DerMorb's is bound by its 256 registers,
    // two waves per SIMD
    if constexpr (F == WBMI_FORMULA_MORB_HPM && MODE != 2) {
        return launch_scan_t<T, F, false, false, MODE, 0, 256>(ctx, nk, a, E, X, hist);
    } else if constexpr (SC_IS_DERMORB_CUTS(F)) {
        if (a.stage_va && smem_offsets(a.nw, true, true, a.p.external_terms, MODE == 1, sizeof(cplx<T>)).total <= SC_LDS / 2)
            return launch_scan_t<T, F, true, true, MODE, 0, 256>(ctx, nk, a, E, X, hist);
        if (smem_offsets(a.nw, true, false, false, MODE == 1, sizeof(cplx<T>)).total <= SC_LDS / 2)
            return launch_scan_t<T, F, true, false, MODE, 0, 256>(ctx, nk, a, E, X, hist);
        return launch_scan_t<T, F, MODE == 0, false, MODE, 0, 512>(ctx, nk, a, E, X, hist);
    } else if constexpr (F == WBMI_FORMULA_OMEGA || F == WBMI_FORMULA_VELOMEGA || F == WBMI_FORMULA_VELHPLUS ||
                         F == WBMI_FORMULA_IDENTITY || F == WBMI_FORMULA_MORB_HPM) {
        // as many waves as diag_traces has rows of 8 bands: a workgroup's prologue costs every wave of it (nw = 24,
        // 5832 k-points: 90 us in 3 waves, 121 in 4, 182 in 8); dEinv in LDS only for velocity products, whose
        // groups of several bands read it more than once.  The tetrahedron kernels keep 8 waves for their weights
        // (1728 k-points at nw = 12, 201 levels: 159 us, 200 in 2 waves).
        constexpr bool lm = F == WBMI_FORMULA_VELOMEGA || F == WBMI_FORMULA_VELHPLUS;
        if constexpr (MODE != 1) {
            if (a.nw <= 8) return launch_scan_t<T, F, lm, false, MODE, 0, 64>(ctx, nk, a, E, X, hist);
            if (a.nw <= 16) return launch_scan_t<T, F, lm, false, MODE, 0, 128>(ctx, nk, a, E, X, hist);
            if (a.nw <= 24) return launch_scan_t<T, F, lm, false, MODE, 0, 192>(ctx, nk, a, E, X, hist);
            if (a.nw <= 32) return launch_scan_t<T, F, lm, false, MODE, 0, 256>(ctx, nk, a, E, X, hist);
            if (a.nw <= 48) return launch_scan_t<T, F, lm, false, MODE, 0, 384>(ctx, nk, a, E, X, hist);
        }
        if (a.nw <= SC_M_NW) return launch_scan_t<T, F, lm, false, MODE, 0, 512>(ctx, nk, a, E, X, hist);
        return launch_scan_t<T, F, false, false, MODE, 0, 512>(ctx, nk, a, E, X, hist);
    } else if constexpr (tasks && MODE != 1) {
        if (a.stage_va) {
            if constexpr (MODE == 0 && F == WBMI_FORMULA_DEROMEGA)
                // nw = 32 (a single 32-column block, the spin blocks of the spinor models) has its own
                // Fermi-bin kernels with the size fixed at compile time
                if (a.nw == 32) return launch_scan_t<T, F, true, true, MODE, 32, sizeof(T) == 4 ? 512 : 768>(ctx, nk, a, E, X, hist);
            const size_t lds = smem_offsets(a.nw, true, true, a.p.external_terms, false, sizeof(cplx<T>)).total;
            if (lds <= SC_LDS / 4) return launch_scan_t<T, F, true, true, MODE, 0, 256>(ctx, nk, a, E, X, hist);
            if (lds <= SC_LDS / 2) return launch_scan_t<T, F, true, true, MODE, 0, 512>(ctx, nk, a, E, X, hist);
            return launch_scan_t<T, F, true, true, MODE, 0, 768>(ctx, nk, a, E, X, hist);
        }
        const size_t lds = smem_offsets(a.nw, true, false, false, false, sizeof(cplx<T>)).total;
        if (lds <= SC_LDS / 2) return launch_scan_t<T, F, true, false, MODE, 0, 512>(ctx, nk, a, E, X, hist);
        return launch_scan_t<T, F, true, false, MODE, 0, 1024>(ctx, nk, a, E, X, hist);
    } else {
        if constexpr (tasks)
            if (a.stage_va) return launch_scan_t<T, F, true, true, MODE>(ctx, nk, a, E, X, hist);
        if (a.nw <= SC_M_NW) return launch_scan_t<T, F, true, false, MODE>(ctx, nk, a, E, X, hist);
        return launch_scan_t<T, F, false, false, MODE>(ctx, nk, a, E, X, hist);
    }
}

template <typename T, int MODE>
static int dispatch_scan(wbmi_ctx* ctx, int nk, const ScanArgs& a, const double* E, const void* X, double* hist) {
    switch (a.p.formula) {
        case WBMI_FORMULA_IDENTITY: return launch_scan<T, WBMI_FORMULA_IDENTITY, MODE>(ctx, nk, a, E, X, hist);
        case WBMI_FORMULA_OMEGA: return launch_scan<T, WBMI_FORMULA_OMEGA, MODE>(ctx, nk, a, E, X, hist);
        case WBMI_FORMULA_DEROMEGA: return launch_scan<T, WBMI_FORMULA_DEROMEGA, MODE>(ctx, nk, a, E, X, hist);
        case WBMI_FORMULA_VELOMEGA: return launch_scan<T, WBMI_FORMULA_VELOMEGA, MODE>(ctx, nk, a, E, X, hist);
        case WBMI_FORMULA_MORB_HPM: return launch_scan<T, WBMI_FORMULA_MORB_HPM, MODE>(ctx, nk, a, E, X, hist);
        case WBMI_FORMULA_VELHPLUS: return launch_scan<T, WBMI_FORMULA_VELHPLUS, MODE>(ctx, nk, a, E, X, hist);
        case WBMI_FORMULA_DERMORB:
            if constexpr (MODE != 2)
                if (!a.p.external_terms) {
                    return launch_scan<T, sizeof(T) == 4 ? SC_DERMORB_IN32 : SC_DERMORB_IN, MODE>(ctx, nk, a, E, X, hist);
                }
            if constexpr (MODE != 2 && sizeof(T) == 8)
                if (a.p.sign == 1) return launch_scan<T, SC_DERMORB_EX, MODE>(ctx, nk, a, E, X, hist);
            return launch_scan<T, WBMI_FORMULA_DERMORB, MODE>(ctx, nk, a, E, X, hist);
        case WBMI_FORMULA_DERSPIN: return launch_scan<T, WBMI_FORMULA_DERSPIN, MODE>(ctx, nk, a, E, X, hist);
        case WBMI_FORMULA_VELSPIN: return launch_scan<T, WBMI_FORMULA_VELSPIN, MODE>(ctx, nk, a, E, X, hist);
        case WBMI_FORMULA_SPIN: return launch_scan<T, WBMI_FORMULA_SPIN, MODE>(ctx, nk, a, E, X, hist);
        case WBMI_FORMULA_INVMASS: return launch_scan<T, WBMI_FORMULA_INVMASS, MODE>(ctx, nk, a, E, X, hist);
        case WBMI_FORMULA_VELVEL: return launch_scan<T, WBMI_FORMULA_VELVEL, MODE>(ctx, nk, a, E, X, hist);
        case WBMI_FORMULA_VELVELVEL: return launch_scan<T, WBMI_FORMULA_VELVELVEL, MODE>(ctx, nk, a, E, X, hist);
        case WBMI_FORMULA_MASSVEL: return launch_scan<T, WBMI_FORMULA_MASSVEL, MODE>(ctx, nk, a, E, X, hist);
        case WBMI_FORMULA_HALL_SURF: return launch_scan<T, WBMI_FORMULA_HALL_SURF, MODE>(ctx, nk, a, E, X, hist);
        case WBMI_FORMULA_HALL_SEA: return launch_scan<T, WBMI_FORMULA_HALL_SEA, MODE>(ctx, nk, a, E, X, hist);
        case WBMI_FORMULA_BANDVALUES: return launch_scan<T, WBMI_FORMULA_BANDVALUES, MODE>(ctx, nk, a, E, X, hist);
        case WBMI_FORMULA_OMEGASPIN: return launch_scan<T, WBMI_FORMULA_OMEGASPIN, MODE>(ctx, nk, a, E, X, hist);
        case WBMI_FORMULA_OMEGAOMEGA: return launch_scan<T, WBMI_FORMULA_OMEGAOMEGA, MODE>(ctx, nk, a, E, X, hist);
        case WBMI_FORMULA_OMEGAHPLUS: return launch_scan<T, WBMI_FORMULA_OMEGAHPLUS, MODE>(ctx, nk, a, E, X, hist);
        default: return wbmi_fail(ctx, WBMI_ERR_UNSUPPORTED, "wbmi_static_scan: formula %d", a.p.formula);
    }
}

// one translation unit per (precision, Fermi-bin | tetrahedron) instantiates the kernels
int scan_dispatch_f64(wbmi_ctx* ctx, int nk, const ScanArgs& a, const double* E, const void* X, double* hist);
int scan_dispatch_f32(wbmi_ctx* ctx, int nk, const ScanArgs& a, const double* E, const void* X, double* hist);
int scan_dispatch_tetra_f64(wbmi_ctx* ctx, int nk, const ScanArgs& a, const double* E, const void* X, double* hist);
int scan_dispatch_tetra_f32(wbmi_ctx* ctx, int nk, const ScanArgs& a, const double* E, const void* X, double* hist);
int scan_dispatch_tab_f64(wbmi_ctx* ctx, int nk, const ScanArgs& a, const double* E, const void* X, double* hist);
int scan_dispatch_tab_f32(wbmi_ctx* ctx, int nk, const ScanArgs& a, const double* E, const void* X, double* hist);
