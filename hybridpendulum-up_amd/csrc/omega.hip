// Omega DFTs of the transforms (the unnormalized DFT over the omega axes and
// its inverse with 1/N per axis), on the rows of the compact coefficients:
// k_slab_dft over (k1, k2) of each slab, k_axis_dft_mfma over k3.  FP32 grids with
// XformDev::keep: k_slab_dft_chirp (N <= 32), k_slab_dft_fma (dim 2, N > 32).
#include <algorithm>

#include "drift.h"
#include "kernels_common.h"
#include "mfma.h"

namespace hpup {

// Omega DFTs of the coefficients of a real grid.  Before the omega DFT the
// coefficients satisfy F^l_{-m,-n}(x) = s conj F^l_mn(x), s = (-1)^(m-n)
// (the forward beta stage writes that mirror), so after it
// F^l_{-m,-n}(k) = s conj F^l_mn(-k): the forward DFTs need only the rows
// with n > 0, or n = 0 and m >= 0 (the half list hr: pairs (row, mirror row
// | bit 30 when s = -1)), and the last pass writes the mirror rows.  The
// inverse transform's real output depends on the coefficients only through
// their Hermitian part (F^l_mn(k) + s conj F^l_{-m,-n}(-k)) / 2, which the
// first inverse pass forms on the half rows, so the rest of the inverse runs
// on those rows only.
enum OmegaRows {
    kRowsAll = 0,     // every row
    kRowsHalf = 1,    // the half rows
    kRowsMirror = 2,  // the half rows, output written to the mirror rows too
    kRowsSym = 3      // the half rows, input taken as the Hermitian part
};

struct HalfRow {
    int r, rm;  // row and mirror row
    bool neg;   // s = -1
};
__device__ __forceinline__ HalfRow half_row(const int32_t* hr, int64_t i) {
    const int32_t b = hr[2 * i + 1];
    return {hr[2 * i], b & 0x3fffffff, ((b >> 30) & 1) != 0};
}
// s conj z
template <class T> __device__ __forceinline__ cT<T> sconj(cT<T> z, bool neg) {
    return neg ? cmk<T>(-z.x, z.y) : cmk<T>(z.x, -z.y);
}

// ------------------------------------------------- (k1, k2): k_slab_dft --
//
// 2-D DFT of N x N slabs (N even, at most 64), times `scale`, by real cos/sin
// products of the parts even and odd in a1 and a2 (the folding of the MFMA
// (alpha, gamma) stages): with H = N / 2 and x folded over a1 <-> -a1 and
// a2 <-> -a2 into the complex planes ee, oe, eo, oo (even/odd in a1, then a2),
//   EE = cos ee cos', OE = sin oe cos', EO = cos eo sin', OO = sin oo sin'
// for k1, k2 = 0..H (cos/sin (2 pi k a / N), a = 0..H), and
//   X[+-k1, k2] = EE -+ OO + s i (+-OE + EO),  X[+-k1, -k2] = EE +- OO + s i (+-OE - EO)
// with s = -1 forward, +1 inverse.  That is 8 real products of (N/2 + 1)^2
// tables per axis, against 3 of N^2 for a Toeplitz form on Gauss products, so
// that the slabs' traffic is what bounds the kernel.  A block of four waves
// holds XC slabs in LDS; each wave takes tiles of 16 columns by 16 output
// rows; the first axis' results replace its inputs: row a2 holds EE (k1 =
// 0..H) then OE (0 < k1 < H), row -a2 EO then OO.  Row stride N + 1 (odd):
// the operand reads of a phase fall in distinct banks.  NYQ (H a multiple of 16,
// N = 32 and 64): the row k = H, alone in a tile of its own otherwise, is the
// alternating sum of the cosine operands, formed on the vector units on the way
// to the products (N = 32, FP32, B = 20, 32^2: 65 -> 39 us).
//
// Measured per launch: B = 30, 60^2, FP64 6.1 -> 1.02 ms forward, 0.79 ms inverse
// (direct sums on all rows before; half of the rows now); on half of the rows
// against Toeplitz products: B = 15, 30^3, FP64 0.80 -> 0.65 ms, FP32 0.32 ->
// 0.23 ms; B = 30, 20^3, FP32 1.08 -> 0.64 ms.
//
// N = 32, whose 17 points do not fill the tiles, gains no time in FP32 against the Toeplitz
// products, and keeps this form for its error, half of theirs: B = 20, 2-D, forward /
// inverse 37 / 34 -> 38 / 36 us, B = 30 121 / 121 -> 122 / 114, B = 8, 3-D 58 / 57 -> 64 / 64; relative
// error 2.7e-7 / 3.0e-7 -> 1.3e-7 / 2.0e-7 (B = 12, the whole transform).  FP64, B = 20: 75 / 76 ->
// 75 / 62 us.
//
// Slab sl is row sl / nz at k3 = sl % nz (rows from the half list unless hr is
// null).  In place when in == out: a block's slabs are read whole before any is
// written, and the mirror rows a mirror pass writes are read by no other slab.
constexpr int kSlabMaxXC = 16;

// Elements a thread loads before its first use: a block's slabs in one batch
// (two in FP64 when the mirror slabs are loaded too), one memory round trip.  At the
// largest N of two classes a second batch holds the rest: N = 22 needs 10 and N = 62 16;
// with these they are up to 9 % faster and the other sizes of their classes (16 to 20,
// 56 to 60) 1-4 % slower, by the loads they repeat.
constexpr int slab_batch(int KS, bool NYQ) {
    return NYQ ? (KS == 5 ? 12 : 16) : KS == 1 ? 3 : KS == 2 ? 7 : KS == 3 ? 8 : KS == 4 ? 15 : KS == 5 ? 6 : KS == 6 ? 9 : KS == 7 ? 12 : 15;
}

// (FP32 is compiled for 5 waves per SIMD: without the bound the compiler spreads
// over 100 to 140 registers, 3 or 4 waves, and the slabs wait for their loads.  N = 32,
// B = 20, 2-D, without the mirror slabs' loads: 38 us at 4 waves, 40 at 5; with them 38
// and 36)
template <class T, int KS, int TPW, bool SYM, bool NYQ>
__global__ __launch_bounds__(256, TPW > 1 ? 1 : sizeof(T) == 8 ? 3 : NYQ && !SYM ? 4 : 5) void k_slab_dft(const cT<T>* in, cT<T>* out, const T* __restrict__ tab, int N,
                                                  T scale, T sgn, int nslab, int nz, const int32_t* __restrict__ hr,
                                                  int mirror, int XC) {
    using MF = Mfma<T>;
    using acc_t = typename MF::acc;
    extern __shared__ __align__(16) char smem_sd[];
    cT<T>* sf = reinterpret_cast<cT<T>*>(smem_sd);
    __shared__ int64_t sb[kSlabMaxXC], sm[kSlabMaxXC];  // element offsets of a slab and of its mirror slab
    __shared__ int sneg[kSlabMaxXC], sself[kSlabMaxXC];
    const int H = N / 2, NN = N * N, rs = N + 1, sx = N * rs, H1 = H + 1;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, lr = lane & 15, lq = lane >> 4;
    const int sl0 = (int)blockIdx.x * XC, xn = min(XC, nslab - sl0);
    if (tid < xn) {
        const int sl = sl0 + tid;
        if (hr) {
            const int i = sl / nz, k3 = sl - i * nz;
            const HalfRow h = half_row(hr, i);
            sb[tid] = ((int64_t)h.r * nz + k3) * NN;
            sm[tid] = ((int64_t)h.rm * nz + (k3 == 0 ? 0 : nz - k3)) * NN;
            sneg[tid] = h.neg;
            sself[tid] = h.rm == h.r;
        } else {
            sb[tid] = sm[tid] = (int64_t)sl * NN;
            sneg[tid] = 0;
            sself[tid] = 1;
        }
    }
    __syncthreads();
    const float invN = 1.0f / (float)N, invNN = 1.0f / (float)NN;
    {  // the slabs (SYM: their Hermitian part with the mirror slab at (-a1, -a2))
        const int tot = xn * NN;
        constexpr int NF = slab_batch(KS, NYQ), NL = SYM && sizeof(T) == 8 ? (NF + 1) / 2 : NF;
        for (int i0 = tid; i0 < tot; i0 += 256 * NL) {
            cT<T> v[NL], y[SYM ? NL : 1];
#pragma unroll
            for (int u = 0; u < NL; u++) {
                const int i = i0 + 256 * u < tot ? i0 + 256 * u : i0;
                const int xl = div_small(i, invNN), e = i - xl * NN;
                v[u] = in[sb[xl] + e];
                if constexpr (SYM) {
                    const int a2 = div_small(e, invN), a1 = e - a2 * N;
                    y[u] = in[sm[xl] + (a2 ? N - a2 : 0) * N + (a1 ? N - a1 : 0)];
                }
            }
#pragma unroll
            for (int u = 0; u < NL; u++) {
                const int i = i0 + 256 * u;
                const int xl = div_small(i, invNN), e = i - xl * NN, a2 = div_small(e, invN), a1 = e - a2 * N;
                if (i < tot) {
                    if constexpr (SYM) {
                        const cT<T> c = sconj<T>(y[u], sneg[xl]);
                        v[u] = cmk<T>(T(0.5) * (v[u].x + c.x), T(0.5) * (v[u].y + c.y));
                    }
                    sf[xl * sx + a2 * rs + a1] = v[u];
                }
            }
        }
    }
    // tiles of 16 columns (x, k) by 16 rows; wave w takes the tasks w, w + 4, ...
    // (NYQ: a slab's columns below H in whole tiles, the columns H of all slabs
    // in one more, so that the stores of a row start on its line)
    const int MT = NYQ ? H / 16 : (H1 + 15) / 16, ncol = xn * H1;
    const int ntask = (NYQ ? xn * MT + 1 : (ncol + 15) / 16) * MT;
    const float invH1 = 1.0f / (float)H1, invMT = 1.0f / (float)MT;
    auto task = [&](int t, int& mt, int& xl, int& c, bool& ok) {
        const int id = min(w + 4 * t, ntask - 1), ct = div_small(id, invMT);
        mt = id - ct * MT;
        ok = w + 4 * t < ntask;
        if constexpr (NYQ) {
            const bool last = ct == xn * MT;
            xl = last ? min(lr, xn - 1) : div_small(ct, invMT);
            c = last ? H : 16 * (ct - xl * MT) + lr;
            ok = ok && (!last || lr < xn);
        } else {
            const int col = min(16 * ct + lr, ncol - 1);
            ok = ok && 16 * ct + lr < ncol;
            xl = div_small(col, invH1);
            c = col - xl * H1;
        }
    };
    T tc[KS], ts[KS], th[NYQ ? KS : 1];
    if constexpr (NYQ) {
#pragma unroll
        for (int k = 0; k < KS; k++) th[k] = tab[H * kAgTabK + 4 * k + lq];
    }
    // the sum over a column's four lanes
    auto sum4 = [](T x) {
        x += __shfl_xor(x, 16, 64);
        return x + __shfl_xor(x, 32, 64);
    };
    auto load_tab = [&](int mt) {
#pragma unroll
        for (int k = 0; k < KS; k++) {
            const int i = (16 * mt + lr) * kAgTabK + 4 * k + lq;
            tc[k] = tab[i];
            ts[k] = tab[kAgTabR * kAgTabK + i];
        }
    };
    acc_t a[TPW][8];  // ee, oe, eo, oo: real and imaginary part
    T hy[NYQ ? TPW : 1][4];
    {
        int mt, xl, c;
        bool ok;
        task(0, mt, xl, c, ok);
        load_tab(mt);
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < TPW; t++) {  // axis 1: column (x, a2), K = a1
        int mt, xl, g;
        bool ok;
        task(t, mt, xl, g, ok);
        if (t > 0) load_tab(mt);
        const cT<T>* r0 = sf + xl * sx + g * rs;
        const cT<T>* r1 = sf + xl * sx + (g ? N - g : 0) * rs;
#pragma unroll
        for (int q = 0; q < 8; q++) a[t][q] = MF::zero();
        if constexpr (NYQ) hy[t][0] = hy[t][1] = hy[t][2] = hy[t][3] = T(0);
#pragma unroll
        for (int k = 0; k < KS; k++) {
            const int i = min(4 * k + lq, H), j = i ? N - i : 0;
            const cT<T> p = r0[i], q = r0[j], u = r1[i], v = r1[j];
            const cT<T> e0 = cadd<T>(p, q), o0 = csub<T>(p, q), e1 = cadd<T>(u, v), o1 = csub<T>(u, v);
            a[t][0] = MF::fma(tc[k], e0.x + e1.x, a[t][0]);
            a[t][1] = MF::fma(tc[k], e0.y + e1.y, a[t][1]);
            a[t][2] = MF::fma(ts[k], o0.x + o1.x, a[t][2]);
            a[t][3] = MF::fma(ts[k], o0.y + o1.y, a[t][3]);
            a[t][4] = MF::fma(tc[k], e0.x - e1.x, a[t][4]);
            a[t][5] = MF::fma(tc[k], e0.y - e1.y, a[t][5]);
            a[t][6] = MF::fma(ts[k], o0.x - o1.x, a[t][6]);
            a[t][7] = MF::fma(ts[k], o0.y - o1.y, a[t][7]);
            if constexpr (NYQ) {
                hy[t][0] = fma(th[k], e0.x + e1.x, hy[t][0]);
                hy[t][1] = fma(th[k], e0.y + e1.y, hy[t][1]);
                hy[t][2] = fma(th[k], e0.x - e1.x, hy[t][2]);
                hy[t][3] = fma(th[k], e0.y - e1.y, hy[t][3]);
            }
        }
    }
    __syncthreads();  // every read done: the results replace the inputs
#pragma unroll
    for (int t = 0; t < TPW; t++) {
        int mt, xl, g;
        bool ok;
        task(t, mt, xl, g, ok);
        cT<T>* r0 = sf + xl * sx + g * rs;
        cT<T>* r1 = sf + xl * sx + (g ? N - g : 0) * rs;
        const bool two = g > 0 && g < H;
        if constexpr (NYQ) {
#pragma unroll
            for (int q = 0; q < 4; q++) hy[t][q] = sum4(hy[t][q]);
            if (ok && mt == 0 && lq == 0) {
                r0[H] = cmk<T>(hy[t][0], hy[t][1]);
                if (two) r1[H] = cmk<T>(hy[t][2], hy[t][3]);
            }
        }
        if (ok) {
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int k = 16 * mt + MF::orow(lq, v);
                if (k > H) continue;
                r0[k] = cmk<T>(a[t][0][v], a[t][1][v]);
                if (two) r1[k] = cmk<T>(a[t][4][v], a[t][5][v]);
                if (k > 0 && k < H) {
                    r0[H + k] = cmk<T>(a[t][2][v], a[t][3][v]);
                    if (two) r1[H + k] = cmk<T>(a[t][6][v], a[t][7][v]);
                }
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < TPW; t++) {  // axis 2: column (x, k1), K = a2
        int mt, xl, k1;
        bool ok;
        task(t, mt, xl, k1, ok);
        if (TPW > 1) load_tab(mt);
        const bool two = k1 > 0 && k1 < H;
        const int od = two ? H : 0;  // the odd planes' offset (zeroed where they vanish)
        const cT<T>* c0 = sf + xl * sx + k1;
#pragma unroll
        for (int q = 0; q < 8; q++) a[t][q] = MF::zero();
        if constexpr (NYQ) hy[t][0] = hy[t][1] = hy[t][2] = hy[t][3] = T(0);
#pragma unroll
        for (int k = 0; k < KS; k++) {
            const int g = min(4 * k + lq, H);
            const cT<T>* pe = c0 + g * rs;
            const cT<T>* po = c0 + (g ? N - g : 0) * rs;
            const cT<T> ee = pe[0], eo = po[0];
            cT<T> oe = pe[od], oo = po[od];
            if (!two) oe = oo = czero<T>();
            a[t][0] = MF::fma(tc[k], ee.x, a[t][0]);
            a[t][1] = MF::fma(tc[k], ee.y, a[t][1]);
            a[t][2] = MF::fma(tc[k], oe.x, a[t][2]);
            a[t][3] = MF::fma(tc[k], oe.y, a[t][3]);
            a[t][4] = MF::fma(ts[k], eo.x, a[t][4]);
            a[t][5] = MF::fma(ts[k], eo.y, a[t][5]);
            a[t][6] = MF::fma(ts[k], oo.x, a[t][6]);
            a[t][7] = MF::fma(ts[k], oo.y, a[t][7]);
            if constexpr (NYQ) {
                hy[t][0] = fma(th[k], ee.x, hy[t][0]);
                hy[t][1] = fma(th[k], ee.y, hy[t][1]);
                hy[t][2] = fma(th[k], oe.x, hy[t][2]);
                hy[t][3] = fma(th[k], oe.y, hy[t][3]);
            }
        }
        if constexpr (NYQ) {
#pragma unroll
            for (int q = 0; q < 4; q++) hy[t][q] = sum4(hy[t][q]);
        }
        if (ok) {
            cT<T>* ob = out + sb[xl];
            cT<T>* om = out + sm[xl];
            const bool mir = mirror && !sself[xl];
            const bool neg = sneg[xl];
            auto put = [&](int q1, int q2, T re, T im) {
                const cT<T> z = cmk<T>(re * scale, im * scale);
                ob[q2 * N + q1] = z;
                if (mir) om[(q2 ? N - q2 : 0) * N + (q1 ? N - q1 : 0)] = sconj<T>(z, neg);
            };
            if constexpr (NYQ) {
                if (mt == 0 && lq == 0) {  // k2 = H: EE + s i OE, EE - s i OE at -k1
                    put(k1, H, hy[t][0] - sgn * hy[t][3], hy[t][1] + sgn * hy[t][2]);
                    if (two) put(N - k1, H, hy[t][0] + sgn * hy[t][3], hy[t][1] - sgn * hy[t][2]);
                }
            }
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int k2 = 16 * mt + MF::orow(lq, v);
                if (k2 > H) continue;
                const T eer = a[t][0][v], eei = a[t][1][v], oor = a[t][6][v], ooi = a[t][7][v];
                // s i (OE + EO) and s i (EO - OE)
                const T pr = -sgn * (a[t][3][v] + a[t][5][v]), pi = sgn * (a[t][2][v] + a[t][4][v]);
                const T mr = -sgn * (a[t][5][v] - a[t][3][v]), mi = sgn * (a[t][4][v] - a[t][2][v]);
                put(k1, k2, (eer - oor) + pr, (eei - ooi) + pi);
                if (two) put(N - k1, k2, (eer + oor) + mr, (eei + ooi) + mi);
                if (k2 > 0 && k2 < H) {
                    put(k1, N - k2, (eer + oor) - mr, (eei + ooi) - mi);
                    if (two) put(N - k1, N - k2, (eer - oor) - pr, (eei - ooi) - pi);
                }
            }
        }
    }
}

// ----------------------------------------------------- k3: k_axis_dft_mfma --
//
// The length-N DFT as a chirp-Toeplitz product (Bluestein's identity
// -2 k a = (k - a)^2 - k^2 - a^2):
//   X_k = p_k sum_a c_{k-a} (p_a x_a),  p_k = e^{-+ i pi k^2 / N}, c_d = e^{+- i pi d^2 / N}.
// bs holds c_d at [d + 32] (64 entries) and then p_k (zero for k >= N), 96
// entries; the inverse tables are the conjugates.
template <class T> struct ToepTab {
    cT<T> re_in[64], im_in[64];  // c_d and i c_d (the imaginary input half)
    __device__ __forceinline__ void fill(const cT<T>* bs, int tid) {
        if (tid < 64) {
            const cT<T> c = bs[tid];
            re_in[tid] = c;
            im_in[tid] = cmk<T>(-c.y, c.x);
        }
    }
};

// DFT along the outermost axis: lines of N points at stride `inner`, one per
// (line block L, column j); 64-column chunks as the B operand of the Toeplitz
// GEMM (the k_axis3_mfma layout), times `scale`.  Out of place or in place.
// Line block blockIdx.y is a row (from the half list unless kRowsAll); the
// mirror of column j = k2 N + k1 is (-k2) N + (-k1) (3-D rows, inner = N^2).
template <class T, int MODE>
__global__ __launch_bounds__(256) void k_axis_dft_mfma(const cT<T>* in, cT<T>* out, const cT<T>* __restrict__ bs,
                                                       int N, int64_t inner, T scale, const int32_t* __restrict__ hr) {
    using MF = Mfma<T>;
    using acc_t = typename MF::acc;
    constexpr int CP = 65;
    __shared__ T sre[32 * CP], sim[32 * CP];
    __shared__ ToepTab<T> tab;
    __shared__ cT<T> pk[32];
    int64_t L = blockIdx.y, Lm = L;
    bool neg = false;
    if (MODE != kRowsAll) {
        const HalfRow h = half_row(hr, blockIdx.y);
        L = h.r;
        Lm = h.rm;
        neg = h.neg;
    }
    const int64_t j0 = (int64_t)blockIdx.x * 64;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, lr = lane & 15, lq = lane >> 4;
    // mirror column of j (clamped in range)
    auto mirror_col = [&](int64_t j) {
        const int jj = (int)(j < inner ? j : inner - 1), c2 = jj / N, c1 = jj - c2 * N;
        return (int64_t)(c2 == 0 ? 0 : N - c2) * N + (c1 == 0 ? 0 : N - c1);
    };
    // the chunk's eight elements per thread (row a = w + 4 i, column lane):
    // unconditional clamped loads, all issued before the first use
    cT<T> x[8], y[8];
    {
        const int64_t j = j0 + lane, jm = MODE == kRowsSym ? mirror_col(j) : 0;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int a = w + 4 * i;
            const bool ok = a < N && j < inner;
            x[i] = in[ok ? (L * N + a) * inner + j : 0];
            if (MODE == kRowsSym) y[i] = in[ok ? (Lm * N + (a == 0 ? 0 : N - a)) * inner + jm : 0];
        }
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int a = w + 4 * i;
            if (MODE == kRowsSym) {
                const cT<T> c = sconj<T>(y[i], neg);
                x[i] = cmk<T>(T(0.5) * (x[i].x + c.x), T(0.5) * (x[i].y + c.y));
            }
            if (!(a < N && j < inner)) x[i] = czero<T>();
        }
    }
    tab.fill(bs, tid);
    if (tid < 32) pk[tid] = bs[64 + tid];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int a = w + 4 * i;
        const cT<T> v = a < N ? cmul<T>(x[i], pk[a]) : czero<T>();
        sre[a * CP + lane] = v.x;
        sim[a * CP + lane] = v.y;
    }
    __syncthreads();
    acc_t acc[4];
#pragma unroll
    for (int it = 0; it < 4; it++) acc[it] = MF::zero();
    // K = 4 steps over the rows that hold data (rows a >= N are zero), for the
    // real and then the imaginary half
    const int ks = (N + 3) / 4;
#pragma unroll
    for (int half = 0; half < 2; half++) {
        const T* sp = half == 0 ? sre : sim;
        const cT<T>* t = half == 0 ? tab.re_in : tab.im_in;
#pragma unroll 4
        for (int s = 0; s < ks; s++) {
            const int k = 4 * s + lq;
            const T bv = sp[k * CP + 16 * w + lr];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const cT<T> f = t[16 * h + lr + 32 - k];
                acc[h] = MF::fma(f.x, bv, acc[h]);
                acc[h + 2] = MF::fma(f.y, bv, acc[h + 2]);
            }
        }
    }
    const int64_t j = j0 + 16 * w + lr;
    if (j >= inner) return;
    const int64_t jm = MODE == kRowsMirror ? mirror_col(j) : 0;
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int k = 16 * h + MF::orow(lq, v);
            if (k < N) {
                const cT<T> z = cscale<T>(cmul<T>(cmk<T>(acc[h][v], acc[h + 2][v]), pk[k]), scale);
                out[(L * N + k) * inner + j] = z;
                if (MODE == kRowsMirror && Lm != L) out[(Lm * N + (k == 0 ? 0 : N - k)) * inner + jm] = sconj<T>(z, neg);
            }
        }
}

// ------------------------------------- (k1, k2), FP32 with XformDev::keep --
//
// The (k1, k2) DFTs in the summation orders that FP32 grids behind 64-bit figures
// keep (see the (alpha, gamma) stages of the same name in transform.hip):
// Toeplitz products for N <= 32, direct sums beyond.  k_slab_dft takes 0.7 (N =
// 30) and 0.15 (N = 60) of their time.
constexpr int kPad = 34;

// C X^T products of a 32 x 32 tile with three real products instead of four (Gauss):
// P1 = Re C Re X, P2 = Im C Im X, P3 = (Re C + Im C)(Re X + Im X), and
// C X = P1 - P2 + i (P3 - P1 - P2)
template <class T> struct ToepGauss {
    using MF = Mfma<T>;
    using acc_t = typename MF::acc;
    const ToepTab<T>* c;
    int k2t, k1t, lr, lq, ks;  // ks: K = 4 steps that reach the data
    // along k1: reduction over k = 4 u + lq
    __device__ __forceinline__ void t1(const T* pr, const T* pi, cT<T>* out) const {
        acc_t p1 = MF::zero(), p2 = MF::zero(), p3 = MF::zero();
        const int row = (16 * k2t + lr) * kPad, b = 16 * k1t + lr + 32 - lq;
#pragma unroll 4
        for (int u = 0; u < ks; u++) {
            const T xr = pr[row + 4 * u + lq], xi = pi[row + 4 * u + lq];
            const cT<T> f = c->re_in[b - 4 * u];
            p1 = MF::fma(xr, f.x, p1);
            p2 = MF::fma(xi, f.y, p2);
            p3 = MF::fma(xr + xi, f.x + f.y, p3);
        }
#pragma unroll
        for (int v = 0; v < 4; v++) out[v] = cmk<T>(p1[v] - p2[v], p3[v] - p1[v] - p2[v]);
    }
    // along k2: reduction over k = ks lq + u
    __device__ __forceinline__ void t2(const T* pr, const T* pi, cT<T>* out) const {
        acc_t p1 = MF::zero(), p2 = MF::zero(), p3 = MF::zero();
        const int col = 16 * k1t + lr, r0 = ks * lq, b = 16 * k2t + lr + 32 - ks * lq;
#pragma unroll 4
        for (int u = 0; u < ks; u++) {
            const T xr = pr[(r0 + u) * kPad + col], xi = pi[(r0 + u) * kPad + col];
            const cT<T> f = c->re_in[b - u];
            p1 = MF::fma(f.x, xr, p1);
            p2 = MF::fma(f.y, xi, p2);
            p3 = MF::fma(f.x + f.y, xr + xi, p3);
        }
#pragma unroll
        for (int v = 0; v < 4; v++) out[v] = cmk<T>(p1[v] - p2[v], p3[v] - p1[v] - p2[v]);
    }
};

// 2-D DFT over (k1, k2) of N x N slabs of in, times `scale`, into out (in
// place when they are equal: a slab is read whole before it is written, and
// the mirror rows a kRowsMirror pass writes are read by no other slab).  Slab
// sl is row sl / nz at k3 = sl % nz (rows from the half list).
template <class T, int MODE>
__global__ __launch_bounds__(256) void k_slab_dft_chirp(const cT<T>* in, cT<T>* out, const cT<T>* __restrict__ bs,
                                                       int N, T scale, int nslab, int nz, const int32_t* __restrict__ hr) {
    __shared__ T pa_re[32 * kPad], pa_im[32 * kPad], pb_re[32 * kPad], pb_im[32 * kPad];
    __shared__ ToepTab<T> tab;
    __shared__ cT<T> pk[32];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int k2t = w >> 1, k1t = w & 1, lr = lane & 15, lq = lane >> 4;
    tab.fill(bs, tid);
    if (tid < 32) pk[tid] = bs[64 + tid];
    __syncthreads();
    // reductions trimmed to the N data points (plane A is zero beyond N along
    // k1; plane B's rows k2 >= N are zero through p_k2 = 0)
    ToepGauss<T> gm{&tab, k2t, k1t, lr, lq, (N + 3) / 4};
    const int NN = N * N;
    const int k1 = 16 * k1t + lr;
    const cT<T> p1 = pk[k1];
    // slab sl: its base, and for the mirror modes the mirror slab's (at -k3)
    auto slab = [&](int sl, int64_t& b, int64_t& bm, bool& neg, bool& self) {
        const int i = sl / nz, k3 = sl - i * nz;
        const HalfRow h = half_row(hr, i);
        b = ((int64_t)h.r * nz + k3) * NN;
        bm = ((int64_t)h.rm * nz + (k3 == 0 ? 0 : nz - k3)) * NN;
        neg = h.neg;
        self = h.rm == h.r;
    };
    // the slab's four elements per thread (clamped in-range loads; with the
    // mirror slab's element at (-k2, -k1) for kRowsSym); the next slab's are
    // loaded while this one is transformed
    cT<T> x[4], y[4];
    auto load = [&](int sl) {
        int64_t b, bm;
        bool ng, sf;
        slab(sl, b, bm, ng, sf);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int idx = tid + 256 * i, a2 = idx >> 5, a1 = idx & 31;
            const bool ok = a2 < N && a1 < N;
            x[i] = in[b + (ok ? a2 * N + a1 : 0)];
            if (MODE == kRowsSym) {
                const int m2 = a2 == 0 ? 0 : N - a2, m1 = a1 == 0 ? 0 : N - a1;
                y[i] = in[bm + (ok ? m2 * N + m1 : 0)];
            }
        }
    };
    if ((int)blockIdx.x < nslab) load(blockIdx.x);
    for (int sl = blockIdx.x; sl < nslab; sl += gridDim.x) {
        int64_t b, bm;
        bool neg, self;
        slab(sl, b, bm, neg, self);
#pragma unroll
        for (int i = 0; i < 4; i++) {  // pre-chirp along k1, zero outside the slab
            const int idx = tid + 256 * i, a2 = idx >> 5, a1 = idx & 31;
            cT<T> u = x[i];
            if (MODE == kRowsSym) {
                const cT<T> c = sconj<T>(y[i], neg);
                u = cmk<T>(T(0.5) * (u.x + c.x), T(0.5) * (u.y + c.y));
            }
            const cT<T> v = a2 < N && a1 < N ? cmul<T>(u, pk[a1]) : czero<T>();
            pa_re[a2 * kPad + a1] = v.x;
            pa_im[a2 * kPad + a1] = v.y;
        }
        __syncthreads();  // plane A complete; plane B of the previous slab consumed
        // another slab: no overlap with this slab's output, also in place
        if (sl + (int)gridDim.x < nslab) load(sl + gridDim.x);
        cT<T> R[4];
        gm.t1(pa_re, pa_im, R);
#pragma unroll
        for (int v = 0; v < 4; v++) {  // along k1 done; pre-chirp along k2 (p = 0 in the padding)
            const int k2 = 16 * k2t + Mfma<T>::orow(lq, v);
            const cT<T> yv = cmul<T>(cmul<T>(R[v], p1), pk[k2]);
            pb_re[k2 * kPad + k1] = yv.x;
            pb_im[k2 * kPad + k1] = yv.y;
        }
        __syncthreads();  // plane B complete; plane A consumed
        gm.t2(pb_re, pb_im, R);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int k2 = 16 * k2t + Mfma<T>::orow(lq, v);
            if (k1 < N && k2 < N) {
                const cT<T> z = cscale<T>(cmul<T>(R[v], pk[k2]), scale);
                out[b + k2 * N + k1] = z;
                if (MODE == kRowsMirror && !self)
                    out[bm + (k2 == 0 ? 0 : N - k2) * N + (k1 == 0 ? 0 : N - k1)] = sconj<T>(z, neg);
            }
        }
    }
}

// In-place 2-D DFT over (k1, k2) of every N x N slab, twiddle-indexed.
template <class T>
__global__ __launch_bounds__(1024) void k_slab_dft_fma(cT<T>* __restrict__ F, const cT<T>* __restrict__ twN, int N, T scale) {
    extern __shared__ char smem_raw[];
    const int NN = N * N;
    cT<T>* sA = reinterpret_cast<cT<T>*>(smem_raw);
    cT<T>* sB = sA + NN;
    cT<T>* tw = sB + NN;
    const int64_t base = (int64_t)blockIdx.x * NN;
    for (int e = threadIdx.x; e < NN; e += blockDim.x) sA[e] = F[base + e];
    for (int e = threadIdx.x; e < N; e += blockDim.x) tw[e] = twN[e];
    __syncthreads();
    for (int e = threadIdx.x; e < NN; e += blockDim.x) {
        const int k1 = e % N, k2 = e / N;
        cT<T> acc = czero<T>();
        int t = 0;
        for (int a = 0; a < N; a++) {
            cfma<T>(acc, tw[t], sA[k2 * N + a]);
            t += k1;
            if (t >= N) t -= N;
        }
        sB[e] = acc;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < NN; e += blockDim.x) {
        const int k1 = e % N, k2 = e / N;
        cT<T> acc = czero<T>();
        int t = 0;
        for (int a = 0; a < N; a++) {
            cfma<T>(acc, tw[t], sB[a * N + k1]);
            t += k2;
            if (t >= N) t -= N;
        }
        F[base + e] = cscale<T>(acc, scale);
    }
}

// ---------------------------------------------------------- launchers ---

// (k1, k2) DFT of nslab slabs.  XC slabs per block: as many as fill the four
// waves' tiles of 16 columns once (N <= 32; larger slabs go one by one), two
// tiles per wave at N = 64, whose 33 columns take three.
template <class T, int KS, int TPW, bool NYQ = false>
static void slab_dft_t(const void* in, void* out, int64_t nslab, int N, int nz, const T* tab, T scale, T sgn,
                       const int32_t* hr, bool sym, bool mirror, hipStream_t st) {
    const int H1 = N / 2 + 1, MT = NYQ ? N / 32 : (H1 + 15) / 16;
    const int XC = MT == 1 ? std::min(64 / H1, kSlabMaxXC) : 1;
    const size_t sh = sizeof(cT<T>) * (size_t)XC * N * (N + 1);
    const unsigned grid = (unsigned)((nslab + XC - 1) / XC);
    auto go = [&](auto kern) {
        allow_lds((const void*)kern, sh);
        hipLaunchKernelGGL(kern, dim3(grid), dim3(256), sh, st, (const cT<T>*)in, (cT<T>*)out, tab, N, scale, sgn,
                           (int)nslab, nz, hr, mirror ? 1 : 0, XC);
    };
    if (sym) go(k_slab_dft<T, KS, TPW, true, NYQ>);
    else go(k_slab_dft<T, KS, TPW, false, NYQ>);
}

template <class T>
static void slab_dft(const XformDev<T>& X, const void* in, void* out, int64_t nslab, int nz, bool inverse, T scale,
                     const int32_t* hr, bool sym, bool mirror, hipStream_t st) {
    const int N = X.N;
    HPUP_REQUIRE(N >= 2 && N <= 64 && N % 2 == 0 && X.omT, HPUP_ERR_UNSUPPORTED, "slab DFT needs an even N <= 64");
    HPUP_REQUIRE(nslab < ((int64_t)1 << 30), HPUP_ERR_UNSUPPORTED, "slab DFT: too many slabs");
    if (nslab == 0) return;
    const T sgn = inverse ? T(1) : T(-1);
    if (N == 32) return slab_dft_t<T, 5, 1, true>(in, out, nslab, N, nz, X.omT, scale, sgn, hr, sym, mirror, st);
    switch (N / 8) {  // K = N / 2 + 1 points in steps of 4
    case 0: return slab_dft_t<T, 1, 1>(in, out, nslab, N, nz, X.omT, scale, sgn, hr, sym, mirror, st);
    case 1: return slab_dft_t<T, 2, 1>(in, out, nslab, N, nz, X.omT, scale, sgn, hr, sym, mirror, st);
    case 2: return slab_dft_t<T, 3, 1>(in, out, nslab, N, nz, X.omT, scale, sgn, hr, sym, mirror, st);
    case 3: return slab_dft_t<T, 4, 1>(in, out, nslab, N, nz, X.omT, scale, sgn, hr, sym, mirror, st);
    case 4: return slab_dft_t<T, 5, 1>(in, out, nslab, N, nz, X.omT, scale, sgn, hr, sym, mirror, st);
    case 5: return slab_dft_t<T, 6, 1>(in, out, nslab, N, nz, X.omT, scale, sgn, hr, sym, mirror, st);
    case 6: return slab_dft_t<T, 7, 1>(in, out, nslab, N, nz, X.omT, scale, sgn, hr, sym, mirror, st);
    case 7: return slab_dft_t<T, 8, 1>(in, out, nslab, N, nz, X.omT, scale, sgn, hr, sym, mirror, st);
    default: return slab_dft_t<T, 9, 2, true>(in, out, nslab, N, nz, X.omT, scale, sgn, hr, sym, mirror, st);
    }
}

// k3 DFT on all rows, N <= 32
template <class T>
static void axis_all(const XformDev<T>& X, const void* in, void* out, bool inverse, hipStream_t st) {
    const int64_t inner = (int64_t)X.N * X.N;
    dim3 grid((unsigned)((inner + 63) / 64), (unsigned)X.nrc);
    hipLaunchKernelGGL((k_axis_dft_mfma<T, kRowsAll>), grid, dim3(256), 0, st, (const cT<T>*)in, (cT<T>*)out,
                       inverse ? X.bsI : X.bsF, X.N, inner, inverse ? T(1) / T(X.N) : T(1), nullptr);
}
template <class T, int MODE>
static void axis_half(const XformDev<T>& X, const void* in, void* out, const cT<T>* bs, T scale, hipStream_t st) {
    const int N = X.N;
    const int64_t inner = (int64_t)N * N;
    HPUP_REQUIRE(X.nhalf <= 65535, HPUP_ERR_UNSUPPORTED, "axis DFT: more than 65535 rows");
    dim3 grid((unsigned)((inner + 63) / 64), (unsigned)X.nhalf);
    hipLaunchKernelGGL((k_axis_dft_mfma<T, MODE>), grid, dim3(256), 0, st, (const cT<T>*)in, (cT<T>*)out, bs, N,
                       inner, scale, X.hrows);
}

template <class T, int MODE>
static void slab_keep(const XformDev<T>& X, const void* in, void* out, bool inverse, T scale, hipStream_t st) {
    const int N = X.N, nz = X.dim == 3 ? N : 1;
    const int64_t nslab = X.nhalf * nz;
    HPUP_REQUIRE(nslab < ((int64_t)1 << 31), HPUP_ERR_UNSUPPORTED, "slab DFT: too many slabs");
    const unsigned grid = (unsigned)std::min<int64_t>(nslab, 4096);
    hipLaunchKernelGGL((k_slab_dft_chirp<T, MODE>), dim3(grid), dim3(256), 0, st, (const cT<T>*)in, (cT<T>*)out,
                       inverse ? X.bsI : X.bsF, N, scale, (int)nslab, nz, X.hrows);
}

template <class T>
void launch_omega_half(const XformDev<T>& X, const void* in, void* out, bool inverse, hipStream_t st) {
    HPUP_REQUIRE(omega_half_ok(X), HPUP_ERR_UNSUPPORTED, "half-row omega DFT: dim 2 (N <= 64) or dim 3 (N <= 32)");
    const int N = X.N;
    const T s2 = inverse ? T(1) / T(N * N) : T(1), s3 = inverse ? T(1) / T(N) : T(1);
    const cT<T>* bs = inverse ? X.bsI : X.bsF;
    const int nz = X.dim == 3 ? N : 1;
    const int64_t nslab = X.nhalf * nz;
    if (!inverse) {
        HPUP_REQUIRE(in == out, HPUP_ERR_ARG, "forward half-row omega DFT runs in place");
        if constexpr (sizeof(T) == 4) {
            if (X.keep) {
                if (X.dim == 2) return slab_keep<T, kRowsMirror>(X, in, out, false, s2, st);
                slab_keep<T, kRowsHalf>(X, in, out, false, s2, st);
                return axis_half<T, kRowsMirror>(X, out, out, bs, s3, st);
            }
        }
        slab_dft<T>(X, in, out, nslab, nz, false, s2, X.hrows, false, X.dim == 2, st);
        if (X.dim == 3) axis_half<T, kRowsMirror>(X, out, out, bs, s3, st);
        return;
    }
    HPUP_REQUIRE(in != out, HPUP_ERR_ARG, "inverse half-row omega DFT runs out of place");
    if constexpr (sizeof(T) == 4) {
        if (X.keep) {
            if (X.dim == 2) return slab_keep<T, kRowsSym>(X, in, out, true, s2, st);
            axis_half<T, kRowsSym>(X, in, out, bs, s3, st);
            return slab_keep<T, kRowsHalf>(X, out, out, true, s2, st);
        }
    }
    if (X.dim == 3) {
        axis_half<T, kRowsSym>(X, in, out, bs, s3, st);
        slab_dft<T>(X, out, out, nslab, nz, true, s2, X.hrows, false, false, st);
    } else {
        slab_dft<T>(X, in, out, nslab, nz, true, s2, X.hrows, true, false, st);
    }
}

// out-of-place or in-place omega DFT of every row.  3-D, N <= 32: the k3 pass
// reads in and writes out, then the (k1, k2) pass runs in place on out (DFTs
// along different axes commute); N > 32: the (k1, k2) pass, then the k3
// product with the DFT matrix
template <class T>
void launch_omega_dft(const XformDev<T>& X, const void* in, void* out, bool inverse, hipStream_t st) {
    const int N = X.N;
    if (X.dim == 0) {
        if (in != out)
            HPUP_HIP(hipMemcpyAsync(out, in, sizeof(cT<T>) * (size_t)X.nrc, hipMemcpyDeviceToDevice, st));
        return;
    }
    const T s2 = inverse ? T(1) / T(N * N) : T(1);
    if constexpr (sizeof(T) == 4) {
        if (X.keep && X.dim == 2 && N > 32) {
            const int NN = N * N;
            HPUP_REQUIRE(NN <= 4096, HPUP_ERR_UNSUPPORTED, "omega grid larger than 64 per axis");
            if (in != out)
                HPUP_HIP(hipMemcpyAsync(out, in, sizeof(cT<T>) * (size_t)(X.nrc * X.nx), hipMemcpyDeviceToDevice, st));
            const size_t sh = sizeof(cT<T>) * (2 * (size_t)NN + N);
            allow_lds((const void*)k_slab_dft_fma<T>, sh);
            hipLaunchKernelGGL(k_slab_dft_fma<T>, dim3((unsigned)X.nrc), dim3(1024), sh, st, (cT<T>*)out,
                               inverse ? X.twNi : X.twNf, N, s2);
            return;
        }
    }
    if (X.dim == 3 && N <= 32) {
        axis_all<T>(X, in, out, inverse, st);
        slab_dft<T>(X, out, out, X.nrc * N, N, inverse, s2, nullptr, false, false, st);
        return;
    }
    slab_dft<T>(X, in, out, X.nrc * (X.dim == 3 ? N : 1), X.dim == 3 ? N : 1, inverse, s2, nullptr, false, false, st);
    if (X.dim == 3)
        launch_axis_outer<T>(out, out, inverse ? X.idftN : X.dftN, N, (int64_t)N * N, X.nrc, T(1), st);
}

template void launch_omega_half<float>(const XformDev<float>&, const void*, void*, bool, hipStream_t);
template void launch_omega_half<double>(const XformDev<double>&, const void*, void*, bool, hipStream_t);
template void launch_omega_dft<float>(const XformDev<float>&, const void*, void*, bool, hipStream_t);
template void launch_omega_dft<double>(const XformDev<double>&, const void*, void*, bool, hipStream_t);

}  // namespace hpup
