// Drift kernels of the pendulum models (real circulants, structured mixing):
//   k_drift_fold: omega grids of 18 to 30 points per axis, parity-folded;
//   k_drift_tile: up to 16 points, one wave per slab, forward and adjoint operator;
//   k_drift_fold64: 34 to 62 points, the reduced model in FP64, parity-folded.
//
// k_drift_fold evaluates the derivative of the (r, k3) slabs it visits with the
// integrator epilogue, as k_drift_fused does (see drift_mfma.hip for the terms):
//   dF = T1 V1 + T2 V2 + b1 c1 T1 F + b2 c2 T2 F + W,
//   V1 = -U1 F - a2 c2 Z3 - a3 c3 T2 F,  V2 = -U2 F - a1 c1 Z3,
//   W  = -sum_p c_p CG_p F + D F + (e3 + b3 c3) Z3,   c_p = i kc_p,
// with T_p = c0 1 1^T + i K_p, K_p real and antisymmetric (kappa_p(-d) = -kappa_p(d)).
// A thread owns the four elements (+-i1, +-i2), i1, i2 = 0..H = N/2, so the
// sums and differences over each axis' sign (even and odd parts) are formed in
// its registers.  On those parts K_p maps even to odd and back, and so does a
// multiplication by kc_p: every product is a real (H + 1) x (H + 1) matrix on one
// parity plane, a quarter of the full circulant, and N = 30 fills the 16 x 16
// matrix instruction exactly.  With x' = (x(+) +- x(-)) / 2 per axis and planes
// holding 4 x' (plain sums):
//   (K x)'_e[k] = sum_a (kappa[k-a] - kappa[k+a]) x'_o[a]                  0 < a < H
//   (K x)'_o[k] = sum_a (kappa[k-a] + kappa[k+a]) x'_e[a]  (kappa[k-a] at a = 0, H)
//   (1 1^T x)'_e[k] = sum_a 2 x'_e[a]                       (x'_e at a = 0, H)
//   (kc x)'_e = kc x'_o, (kc x)'_o = kc x'_e.
// Wave w = p1 + 2 p2 produces plane (p1, p2) of everything but W from the LDS
// planes of F, V1 and V2.  The matrices' operands stay in its registers, every
// LDS address is a register plus an immediate, and an axis sum is folded over a
// lane's own points before one matrix instruction adds it: the unfolded kernels
// spend most of their vector instructions on table reads, axis sums, lane
// permutes and addresses.  The matrices come from the host (OpTab), rounded once.
//
// What bounds it: no single unit (B = 15, N = 30, FP32: matrix pipe 27 %, vector
// units 32 %, tag lookups 61 %, HBM 69 % of a copy's rate, waves waiting half of their
// time).  The six gathered source rows cost 0.28 of 1.37 ms, the streams alone 0.83 ms.  Against
// k_drift_fused / k_drift_fused_c (ms per launch, average of a step's four):
//   B = 15, N = 30: FP32 1.63 -> 1.35, FP64 3.00 -> 2.53;  B = 30, N = 20, FP32: 5.54 -> 3.85.
// Tried and not kept: the slab in its natural order with 16-byte loads and the
// folding in LDS (FP64 N = 30: 2.80, FP32 N = 20: 4.63), mixing tables prefetched
// through LDS (FP32 1.57), three waves per SIMD in FP64 (spills, 3.08).
#include "drift.h"
#include "kernels_common.h"
#include "mfma.h"

namespace hpup {

template <class T> using kc_ptr = __attribute__((address_space(4))) const T*;
template <class T> __device__ __forceinline__ kc_ptr<T> as_const(const T* p) { return (kc_ptr<T>)p; }

template <class P> __device__ __forceinline__ P* at_b(P* p, unsigned ob) {
    using C = typename std::conditional<std::is_const<P>::value, const char, char>::type;
    return reinterpret_cast<P*>(reinterpret_cast<C*>(p) + ob);
}
// data touched once per launch: FP64 streams it (FP32 measures the same either way)
template <class T> __device__ __forceinline__ cT<T> ld_once(const cT<T>* p) {
    if constexpr (sizeof(T) == 8) return ld_stream<T>(p);
    else return *p;
}
template <class T> __device__ __forceinline__ void st_once(cT<T>* p, cT<T> v) {
    if constexpr (sizeof(T) == 8) st_stream<T>(p, v);
    else *p = v;
}

// (x0, x1, x2, x3) at signs (+,+), (-,+), (+,-), (-,-) <-> planes ee, oe, eo, oo
// (even/odd in axis 1, then 2): the same sums both ways
template <class T> __device__ __forceinline__ void parity4(const cT<T>* x, cT<T>* y) {
    const cT<T> s0 = cadd<T>(x[0], x[1]), d0 = csub<T>(x[0], x[1]);
    const cT<T> s1 = cadd<T>(x[2], x[3]), d1 = csub<T>(x[2], x[3]);
    y[0] = cadd<T>(s0, s1);
    y[1] = cadd<T>(d0, d1);
    y[2] = csub<T>(s0, s1);
    y[3] = csub<T>(d0, d1);
}

// waves per SIMD: FP32 fits 128 registers, FP64 needs more than three allow
template <class T> constexpr int fold_waves() { return sizeof(T) == 4 ? 4 : 2; }

// XS: slabs (consecutive k3 of one row, which share the mixing sources and
// coefficients) a workgroup visits together; KS: K = 4
// steps over the H + 1 points of an axis
template <class T, int DIM, int KS, int XS>
__global__ __launch_bounds__(256, fold_waves<T>()) void k_drift_fold(DriftDev<T> D, MixDev<T> MX, const cT<T>* Fin,
                                                                     const cT<T>* __restrict__ Z3, const cT<T>* F0,
                                                                     cT<T>* Fout, StageCoef<T> sc,
                                                                     int ngroup) {
    using MF = Mfma<T>;
    using acc_t = typename MF::acc;
    constexpr int NC = DIM + 2;
    // FP64: the next slab's own elements are loaded before this one's products
    // (N = 30: 2.55 -> 2.48 ms; FP32, four waves per SIMD instead of two, gains
    // nothing at N = 30 and loses 14 % at N = 20, which spills)
    constexpr bool AHEAD = sizeof(T) == 8;
    constexpr int MB = 2;  // source rows whose loads are issued together
    extern __shared__ __align__(16) char smem_fold[];
    const int N = D.N, NN = N * N, H = N / 2, H1 = H + 1;
    constexpr int HP = 4 * KS, RS = HP + 1, PL = HP * RS;  // a plane: H1 x H1 points in HP x RS, zero beyond
    const int nz = DIM == 3 ? N : 1;
    cT<T>* pF = reinterpret_cast<cT<T>*>(smem_fold);  // [XS][4][HP][RS]; the result planes in the end
    cT<T>* pV1 = pF + XS * 4 * PL;
    cT<T>* pV2 = pV1 + XS * 4 * PL;
    __shared__ T skc[32], skd[32];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, lr = lane & 15, lq = lane >> 4;
    for (int i = tid; i < 3 * XS * 4 * PL; i += 256) pF[i] = czero<T>();
    if (tid < N) {
        skc[tid] = D.kc[tid];
        skd[tid] = D.kd[tid];
    }

    // ---- this wave's matrices (plane (p1, p2)), entry [out lr][in 4 s + lq]
    const int p1 = w & 1, p2 = w >> 1;
    T m1[KS], m2[KS], d1[KS], d2[KS], rr1, rr2;
    {
        constexpr OpTab ot(30);
#pragma unroll
        for (int s = 0; s < KS; s++) {
            const int i = lr * ot.S + 4 * s + lq;
            m1[s] = D.op[ot.mat(0, 0, p1) + i];  // K into this plane's parity
            m2[s] = D.op[ot.mat(1, 0, p2) + i];
            d1[s] = D.op[ot.mat(0, 1, p1) + i];  // b c (i K): K to the other parity and kc back
            d2[s] = D.op[ot.mat(1, 1, p2) + i];
        }
        rr1 = D.op[ot.vec(0, p1) + lr];
        rr2 = D.op[ot.vec(1, p2) + lr];
    }

    // weights of the axis sums: a half for a = 0 (step 0) and a = H (the last
    // step), one else (zeros lie beyond H)
    const T wa = lq == 0 || lq == H ? T(0.5) : T(1), wb = lq == (H & 3) ? T(0.5) : T(1);
    auto add_w = [&](cT<T>& t, int s, cT<T> x) {
        if (s == 0) t = cscale<T>(x, wa);
        else if (s < KS - 1) t = cadd<T>(t, x);
        else t = cmk<T>(fma(wb, x.x, t.x), fma(wb, x.y, t.y));
    };
    // ---- this thread's elements
    const int HH = H1 * H1, q = tid / HH;
    const bool act = q < XS;
    const int xs = act ? q : 0, e = act ? tid - q * HH : 0, i2 = e / H1, i1 = e - i2 * H1;
    const int pos = xs * 4 * PL + i2 * RS + i1;  // in plane (0, 0)
    const bool self1 = i1 == 0 || i1 == H, self2 = i2 == 0 || i2 == H;
    unsigned ob[4];
    {
        const int n1 = i1 ? N - i1 : 0, n2 = i2 ? N - i2 : 0;
        ob[0] = (unsigned)(xs * NN + i2 * N + i1) * (unsigned)sizeof(cT<T>);
        ob[1] = (unsigned)(xs * NN + i2 * N + n1) * (unsigned)sizeof(cT<T>);
        ob[2] = (unsigned)(xs * NN + n2 * N + i1) * (unsigned)sizeof(cT<T>);
        ob[3] = (unsigned)(xs * NN + n2 * N + n1) * (unsigned)sizeof(cT<T>);
    }
    const T kc1 = D.kc[i1], kc2 = D.kc[i2];  // of the (+, +) element; zero where an axis is its own mirror
    // D(k) = sum_i G_ii kd(k_i) - sum_{i != j} G_ij kc(k_i) kc(k_j)
    const T dde = D.G[0] * D.kd[i1] + D.G[DIM + 1] * D.kd[i2], ddo = -(D.G[1] + D.G[DIM]) * kc1 * kc2;
    const T g22 = DIM == 3 ? D.G[8] : T(0), g02 = DIM == 3 ? (D.G[2] + D.G[6]) * kc1 : T(0),
            g12 = DIM == 3 ? (D.G[5] + D.G[7]) * kc2 : T(0);
    const bool gyro = DIM == 3 && D.has_gyro;
    __syncthreads();

    // LDS reads of the products: T1 takes data rows i2 = lr over a = 4 s + lq,
    // T2 data columns i1 = lr (lr beyond the plane is clamped: not stored).  Each
    // plane's base is a register, the steps are immediate offsets.
    const int lrc = lr < HP ? lr : HP - 1;
    const int orw = lrc * RS + lq, ocl = lq * RS + lrc;
    const cT<T>* bw = pF + w * PL;
    const cT<T>* b1 = pF + (w ^ 1) * PL;
    const cT<T>* b2 = pF + (w ^ 2) * PL;
    constexpr int OV1 = XS * 4 * PL, OV2 = 2 * OV1;

    const int nrc = (int)D.nrc, TS = MX.TS;
    const int nxcd = gridDim.x >= 8 ? 8 : 1;
    const int per = (int)gridDim.x / nxcd;
    const int xcd = (int)blockIdx.x % nxcd;
    const int hi = (int)((int64_t)ngroup * (xcd + 1) / nxcd);
    int sl = (int)((int64_t)ngroup * xcd / nxcd) + (int)blockIdx.x / nxcd;  // group sl: row sl % nrc, k3 group sl / nrc
    const int dr = per % nrc, dk = per / nrc;
    int rp = sl % nrc, kg = sl / nrc;
    const kc_ptr<int32_t> ord = as_const<int32_t>(MX.order);
    int rnext = sl < hi ? ord[rp] : 0;
    cT<T> fo[4], Zv[4];
    auto load_own = [&](int row, int k3g) {
        const int64_t bn = ((int64_t)row * nz + k3g * XS) * NN;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            fo[j] = *at_b(Fin + bn, ob[j]);
            Zv[j] = DIM == 3 ? ld_once<T>(at_b(Z3 + bn, ob[j])) : czero<T>();
        }
    };
    if (AHEAD && sl < hi) load_own(rnext, kg);
    while (sl < hi) {
        // a wave's priority rises through a slab (mixing, products, epilogue), so that
        // workgroups drift apart in phase instead of queueing for one unit: 2-3 %
        __builtin_amdgcn_s_setprio(0);
        const int r = rnext;
        const int k30 = kg * XS;  // the group's first k3
        const int64_t base = ((int64_t)r * nz + k30) * NN;
        int rn = rp + dr, kn = kg + dk;
        if (rn >= nrc) {
            rn -= nrc;
            kn++;
        }
        rnext = ord[rn];
        const cT<T>* Fb = Fin + base;
        const T kc3 = DIM == 3 ? skc[k30 + xs] : T(0), kd3 = DIM == 3 ? skd[k30 + xs] : T(0);
        if (!AHEAD) load_own(r, kg);
        // ---- mixing, as in k_drift_fused: W += (g0 kc1 + i g1 kc2) F_s, V1 += i u1 F_s, V2 += u2 F_s
        const kc_ptr<int32_t> srcT = as_const<int32_t>(MX.src) + (int64_t)r * TS;
        const kc_ptr<T> coefT = as_const<T>((const T*)MX.coef) + 2 * (int64_t)r * TS * NC;
        cT<T> W[4], V1[4], V2[4];
        {
            const T de = DIM == 3 ? dde + g22 * kd3 : dde, a1 = g02 * kc3, a2 = g12 * kc3;
            cT<T> pl[4];
            parity4<T>(fo, pl);
            if (act) {
#pragma unroll
                for (int j = 0; j < 4; j++) pF[pos + j * PL] = pl[j];
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                T dd = (j == 0 || j == 3) ? de + ddo : de - ddo;
                if (DIM == 3) dd -= (j & 1 ? -a1 : a1) + (j & 2 ? -a2 : a2);
                W[j] = cscale<T>(fo[j], dd);
                V1[j] = V2[j] = czero<T>();
            }
        }
        for (int t0 = 0; t0 < TS; t0 += MB) {
            int src[MB];
            cT<T> fv[MB][4];
#pragma unroll
            for (int u = 0; u < MB; u++) src[u] = t0 + u < TS ? srcT[t0 + u] : -1;
#pragma unroll
            for (int u = 0; u < MB; u++) {
                const cT<T>* Fs = Fin + ((int64_t)(src[u] < 0 ? 0 : (src[u] & 0xffffff)) * nz + k30) * NN;
#pragma unroll
                for (int j = 0; j < 4; j++) fv[u][j] = *at_b(Fs, ob[j]);
            }
#pragma unroll
            for (int u = 0; u < MB; u++) {
                if (src[u] < 0) continue;
                const int fl = src[u] >> 24;
                const int64_t cb = (int64_t)(t0 + u) * NC;
                if (fl & 1) {
                    const T a = coefT[2 * cb] * kc1, b = coefT[2 * (cb + 1) + 1] * kc2;
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const T aj = j & 1 ? -a : a, bj = j & 2 ? -b : b;
                        W[j].x = fma(aj, fv[u][j].x, fma(-bj, fv[u][j].y, W[j].x));
                        W[j].y = fma(aj, fv[u][j].y, fma(bj, fv[u][j].x, W[j].y));
                    }
                }
                if (fl & 2) {
                    const T ui = coefT[2 * (cb + DIM) + 1];
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        V1[j].x = fma(-ui, fv[u][j].y, V1[j].x);
                        V1[j].y = fma(ui, fv[u][j].x, V1[j].y);
                    }
                }
                if (fl & 4) {
                    const T ur = coefT[2 * (cb + DIM + 1)];
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        V2[j].x = fma(ur, fv[u][j].x, V2[j].x);
                        V2[j].y = fma(ur, fv[u][j].y, V2[j].y);
                    }
                }
            }
        }
        if (DIM == 3) {
            const kc_ptr<T> e3p = as_const<T>((const T*)D.e3) + 2 * (int64_t)r;
            const T e3r = e3p[0], e3i = e3p[1] + D.b[2] * kc3;
            const T z1 = gyro ? kc2 * D.gyro[1] : T(0), z2 = gyro ? kc1 * D.gyro[0] : T(0);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const T s1 = j & 2 ? -z1 : z1, s2 = j & 1 ? -z2 : z2;
                V1[j].x = fma(s1, Zv[j].y, V1[j].x);
                V1[j].y = fma(-s1, Zv[j].x, V1[j].y);
                V2[j].x = fma(s2, Zv[j].y, V2[j].x);
                V2[j].y = fma(-s2, Zv[j].x, V2[j].y);
                W[j].x = fma(e3r, Zv[j].x, fma(-e3i, Zv[j].y, W[j].x));
                W[j].y = fma(e3r, Zv[j].y, fma(e3i, Zv[j].x, W[j].y));
            }
        }
        {
            cT<T> pl[4];
            parity4<T>(V1, pl);
            if (act) {
#pragma unroll
                for (int j = 0; j < 4; j++) pV1[pos + j * PL] = pl[j];
            }
            parity4<T>(V2, pl);
            if (act) {
#pragma unroll
                for (int j = 0; j < 4; j++) pV2[pos + j * PL] = pl[j];
            }
        }
        cT<T> f0v[4];
        if (sc.read_f0) {
#pragma unroll
            for (int j = 0; j < 4; j++) f0v[j] = ld_once<T>(at_b(F0 + base, ob[j]));
        }
        if (AHEAD && sl + per < hi) load_own(rnext, kn);
        __syncthreads();  // 1: the planes are complete
        __builtin_amdgcn_s_setprio(1);

        // ---- everything but T1 V1
        acc_t cr[XS], ci[XS];
#pragma unroll
        for (int x = 0; x < XS; x++) {
            const cT<T>* frow = bw + orw + x * 4 * PL;                     // own plane
            const cT<T>* fcol = bw + ocl + x * 4 * PL;
            const cT<T>* f1row = b1 + orw + x * 4 * PL;                    // other parity in axis 1
            const cT<T>* f2col = b2 + ocl + x * 4 * PL;                    // other parity in axis 2
            const cT<T>* y2col = p2 ? f2col : fcol + OV2;                  // p2 odd: b2 c2 (c0 1 1^T F); even: c0 1 1^T V2
            acc_t ar = MF::zero(), ai = MF::zero(), gr = MF::zero(), gi = MF::zero();
            cT<T> s1 = czero<T>(), s2 = czero<T>(), s3 = czero<T>();  // axis sums of this lane's a
#pragma unroll
            for (int s = 0; s < KS; s++) {
                const cT<T> x1 = frow[4 * s], x2 = fcol[4 * s * RS];
                ar = MF::fma(x1.x, d1[s], ar);
                ai = MF::fma(x1.y, d1[s], ai);
                ar = MF::fma(d2[s], x2.x, ar);
                ai = MF::fma(d2[s], x2.y, ai);
                const cT<T> v = f2col[OV2 + 4 * s * RS];
                ar = MF::fma(m2[s], -v.y, ar);
                ai = MF::fma(m2[s], v.x, ai);
                const cT<T> y2 = y2col[4 * s * RS];
                add_w(s2, s, y2);
                if (p1) {
                    const cT<T> y1 = f1row[4 * s];
                    add_w(s1, s, y1);
                }
                if (gyro) {  // T2 F
                    const cT<T> z = f2col[4 * s * RS];
                    gr = MF::fma(m2[s], -z.y, gr);
                    gi = MF::fma(m2[s], z.x, gi);
                    add_w(s3, s, x2);
                }
            }
            // p2 odd: times i (b2 kc2 c0 sum F); even: c0 sum V2
            ar = MF::fma(rr2, p2 ? -s2.y : s2.x, ar);
            ai = MF::fma(rr2, p2 ? s2.x : s2.y, ai);
            if (p1) {
                ar = MF::fma(-s1.y, rr1, ar);
                ai = MF::fma(s1.x, rr1, ai);
            }
            if (gyro && !p2) {
                gr = MF::fma(rr2, s3.x, gr);
                gi = MF::fma(rr2, s3.y, gi);
            }
            cr[x] = ar;
            ci[x] = ai;
            if (gyro) {  // V1 -= i a3 kc3 T2 F (planes hold four times the parts)
                const T s = T(4) * skc[k30 + x] * D.gyro[2];
                cT<T>* v1 = pV1 + (x * 4 + w) * PL;
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int o2 = MF::orow(lq, v);
                    if (o2 < H1 && lr < H1) {
                        cT<T> u = v1[o2 * RS + lr];
                        u.x = fma(s, gi[v], u.x);
                        u.y = fma(-s, gr[v], u.y);
                        v1[o2 * RS + lr] = u;
                    }
                }
            }
        }
        __syncthreads();  // 2: V1 complete; F and V2 consumed
#pragma unroll
        for (int x = 0; x < XS; x++) {
            acc_t ar = cr[x], ai = ci[x];
            cT<T> s1 = czero<T>();
#pragma unroll
            for (int s = 0; s < KS; s++) {
                const cT<T> v = b1[OV1 + orw + x * 4 * PL + 4 * s];
                ar = MF::fma(-v.y, m1[s], ar);
                ai = MF::fma(v.x, m1[s], ai);
                if (!p1) {  // c0 1 1^T V1
                    const cT<T> y = bw[OV1 + orw + x * 4 * PL + 4 * s];
                    add_w(s1, s, y);
                }
            }
            if (!p1) {
                ar = MF::fma(s1.x, rr1, ar);
                ai = MF::fma(s1.y, rr1, ai);
            }
            cT<T>* t = pF + (x * 4 + w) * PL;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int o2 = MF::orow(lq, v);
                if (o2 < H1 && lr < H1) t[o2 * RS + lr] = cmk<T>(ar[v], ai[v]);
            }
        }
        __syncthreads();  // 3: the result planes are complete
        __builtin_amdgcn_s_setprio(2);

        // ---- dF = unfolded planes + W, epilogue (as k_drift_fused)
        cT<T> y[4], qv[4];
        {
            cT<T> pl[4];
#pragma unroll
            for (int j = 0; j < 4; j++) pl[j] = pF[pos + j * PL];
            parity4<T>(pl, y);
        }
#pragma unroll
        for (int j = 0; j < 4; j++) qv[j] = cadd<T>(y[j], W[j]);
        const bool st[4] = {act, act && !self1, act && !self2, act && !self1 && !self2};
        if (sc.deriv_only) {
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (st[j]) st_once<T>(at_b(Fout + base, ob[j]), cscale<T>(qv[j], sc.dt));
        } else {
            if (!sc.read_f0) {
#pragma unroll
                for (int j = 0; j < 4; j++) f0v[j] = *at_b(Fb, ob[j]);  // the slab itself, read again (an L2 hit)
            }
            const T h = sc.dt * sc.cd;
#pragma unroll
            for (int j = 0; j < 4; j++) {  // every load is consumed before the first store
                f0v[j].x = fma(h, qv[j].x, f0v[j].x);
                f0v[j].y = fma(h, qv[j].y, f0v[j].y);
                asm volatile("" : "+v"(f0v[j].x), "+v"(f0v[j].y));
            }
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (st[j]) st_once<T>(at_b(Fout + base, ob[j]), f0v[j]);
        }
        sl += per;
        kg = kn;
        rp = rn;
    }
}

// ------------------------------------------------------ N = 34 .. 62 ----
//
// The same folding for the reduced model's larger grids in FP64: planes of up to
// 32 x 32 points, 2 x 2 tiles of the matrix instruction each.  A workgroup of eight
// waves holds one slab; wave (plane, row tile) forms both column tiles.  LDS holds
// two fields of four planes: F and V2, then V1 in F's place, then the result in
// V2's; V1 and W wait in registers (NQ quartets of elements per thread).  The
// axes share their matrices, which leaves room for them in LDS: in registers, as in
// k_drift_fold, they spill 137 registers (B = 30, N = 60: 4.80 ms), axis 1's alone
// in LDS 59 (3.57 ms), both 19 (2.97 ms; k_drift_fused64 5.38 ms).  N <= 42, one quartet a
// thread, spills none: 2.8-3.1x, N = 44 .. 62 1.9-2.2x faster than k_drift_fused64 (B =
// 10).  What bounds it: 17000 matrix cycles of 47000 per slab; one workgroup fits a CU,
// so the mixing's loads and the products take turns.
template <int KS, int NQ>
__global__ __launch_bounds__(512, 2) void k_drift_fold64(DriftDev<double> D, MixDev<double> MX, const cT<double>* Fin,
                                                         const cT<double>* F0, cT<double>* Fout, StageCoef<double> sc,
                                                         int nslab) {
    using T = double;
    using MF = Mfma<T>;
    using acc_t = typename MF::acc;
    constexpr int NC = 4, MB = 2, HP = 4 * KS, RS = HP + 1, PL = HP * RS, OV = 4 * PL;
    extern __shared__ __align__(16) char smem_fold64[];
    const int N = D.N, NN = N * N, H = N / 2, H1 = H + 1, HH = H1 * H1;
    cT<T>* pA = reinterpret_cast<cT<T>*>(smem_fold64);  // [4][HP][RS], zero beyond H1 x H1
    cT<T>* pB = pA + OV;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, lr = lane & 15, lq = lane >> 4;
    const int pl = w & 3, rt = w >> 2, p1 = pl & 1, p2 = pl >> 1;
    for (int i = tid; i < 2 * OV; i += 512) pA[i] = czero<T>();

    // ---- the axes' matrices (the same for both: D.same12) in LDS, [parity][in][out]
    T* sM = reinterpret_cast<T*>(pA + 2 * OV);
    constexpr OpTab ot(62);
    for (int i = tid; i < 2 * HP * HP; i += 512) {
        const int par = i / (HP * HP), e = i - par * HP * HP, a = e / HP, o = e - a * HP;
        sM[i] = D.op[ot.mat(0, 0, par) + o * ot.S + a];
    }
    T rr1[2], k1o[2], rr2, k2o;  // k_o: -b kc of the outputs
    {
        const int o2 = 16 * rt + lr;
        k2o = D.op[ot.vec(1, 2) + o2];
        rr2 = D.op[ot.vec(1, p2) + o2];
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int o1 = 16 * c + lr;
            k1o[c] = D.op[ot.vec(0, 2) + o1];
            rr1[c] = D.op[ot.vec(0, p1) + o1];
        }
    }
    const T wa = lq == 0 || lq == H ? T(0.5) : T(1), wb = lq == (H & 3) ? T(0.5) : T(1);
    auto add_w = [&](cT<T>& t, int s, cT<T> x) {
        if (s == 0) t = cscale<T>(x, wa);
        else if (s < KS - 1) t = cadd<T>(t, x);
        else t = cmk<T>(fma(wb, x.x, t.x), fma(wb, x.y, t.y));
    };
    // LDS reads of the products (rows and columns beyond the plane are clamped: not stored)
    const int row = 16 * rt + lr < HP ? 16 * rt + lr : HP - 1;
    const int orw = row * RS + lq;
    const T* sm2 = sM + p2 * HP * HP + lq * HP + row;
    const T* sd2 = sM + (p2 ^ 1) * HP * HP + lq * HP + row;
    int ocl[2];
    const T *sm1[2], *sd1[2];  // K into this plane's parity along axis 1; the other one
#pragma unroll
    for (int c = 0; c < 2; c++) {
        const int col = 16 * c + lr < HP ? 16 * c + lr : HP - 1;
        ocl[c] = lq * RS + col;
        sm1[c] = sM + p1 * HP * HP + lq * HP + col;
        sd1[c] = sM + (p1 ^ 1) * HP * HP + lq * HP + col;
    }
    const cT<T>* aw = pA + pl * PL;
    const cT<T>* a1 = pA + (pl ^ 1) * PL;
    const cT<T>* a2 = pA + (pl ^ 2) * PL;

    const int nrc = (int)D.nrc, TS = MX.TS;
    const int nxcd = gridDim.x >= 8 ? 8 : 1;
    const int per = (int)gridDim.x / nxcd;
    const int xcd = (int)blockIdx.x % nxcd;
    const int hi = (int)((int64_t)nslab * (xcd + 1) / nxcd);
    const kc_ptr<int32_t> ord = as_const<int32_t>(MX.order);
    __syncthreads();
    for (int sl = (int)((int64_t)nslab * xcd / nxcd) + (int)blockIdx.x / nxcd; sl < hi; sl += per) {
        const int r = ord[sl];
        const int64_t base = (int64_t)r * NN;
        const kc_ptr<int32_t> srcT = as_const<int32_t>(MX.src) + (int64_t)r * TS;
        const kc_ptr<T> coefT = as_const<T>((const T*)MX.coef) + 2 * (int64_t)r * TS * NC;
        // the thread's quartets, their offsets formed anew for each slab (held
        // through the loop they would cost the registers that V1 and W take)
        int zo;
        asm volatile("v_mov_b32 %0, 0" : "=v"(zo));
        cT<T> W[NQ][4], V1[NQ][4];
        auto quartet = [&](int q, bool& act, int& pos, unsigned* ob, int& i1, int& i2) {
            const int e0 = tid + zo + 512 * q;
            act = e0 < HH;
            const int e = act ? e0 : 0;
            i2 = e / H1;
            i1 = e - i2 * H1;
            pos = i2 * RS + i1;
            const int n1 = i1 ? N - i1 : 0, n2 = i2 ? N - i2 : 0;
            ob[0] = (unsigned)(i2 * N + i1) * (unsigned)sizeof(cT<T>);
            ob[1] = (unsigned)(i2 * N + n1) * (unsigned)sizeof(cT<T>);
            ob[2] = (unsigned)(n2 * N + i1) * (unsigned)sizeof(cT<T>);
            ob[3] = (unsigned)(n2 * N + n1) * (unsigned)sizeof(cT<T>);
        };
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            bool act;
            int pos, i1, i2;
            unsigned ob[4];
            quartet(q, act, pos, ob, i1, i2);
            const T kc1 = D.kc[i1], kc2 = D.kc[i2];
            const T dde = D.G[0] * D.kd[i1] + D.G[3] * D.kd[i2], ddo = -(D.G[1] + D.G[2]) * kc1 * kc2;
            cT<T> fo[4], V2[4], pv[4];
#pragma unroll
            for (int j = 0; j < 4; j++) fo[j] = *at_b(Fin + base, ob[j]);
#pragma unroll
            for (int j = 0; j < 4; j++) W[q][j] = V1[q][j] = V2[j] = czero<T>();
            for (int t0 = 0; t0 < TS; t0 += MB) {
                int src[MB];
                cT<T> fv[MB][4];
#pragma unroll
                for (int u = 0; u < MB; u++) src[u] = t0 + u < TS ? srcT[t0 + u] : -1;
#pragma unroll
                for (int u = 0; u < MB; u++) {
                    const cT<T>* Fs = Fin + (int64_t)(src[u] < 0 ? 0 : (src[u] & 0xffffff)) * NN;
#pragma unroll
                    for (int j = 0; j < 4; j++) fv[u][j] = *at_b(Fs, ob[j]);
                }
#pragma unroll
                for (int u = 0; u < MB; u++) {
                    if (src[u] < 0) continue;
                    const int fl = src[u] >> 24;
                    const int64_t cb = (int64_t)(t0 + u) * NC;
                    if (fl & 1) {
                        const T a = coefT[2 * cb] * kc1, b = coefT[2 * (cb + 1) + 1] * kc2;
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            const T aj = j & 1 ? -a : a, bj = j & 2 ? -b : b;
                            W[q][j].x = fma(aj, fv[u][j].x, fma(-bj, fv[u][j].y, W[q][j].x));
                            W[q][j].y = fma(aj, fv[u][j].y, fma(bj, fv[u][j].x, W[q][j].y));
                        }
                    }
                    if (fl & 2) {
                        const T ui = coefT[2 * (cb + 2) + 1];
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            V1[q][j].x = fma(-ui, fv[u][j].y, V1[q][j].x);
                            V1[q][j].y = fma(ui, fv[u][j].x, V1[q][j].y);
                        }
                    }
                    if (fl & 4) {
                        const T ur = coefT[2 * (cb + 3)];
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            V2[j].x = fma(ur, fv[u][j].x, V2[j].x);
                            V2[j].y = fma(ur, fv[u][j].y, V2[j].y);
                        }
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const T dd = (j == 0 || j == 3) ? dde + ddo : dde - ddo;
                W[q][j].x = fma(dd, fo[j].x, W[q][j].x);
                W[q][j].y = fma(dd, fo[j].y, W[q][j].y);
            }
            parity4<T>(fo, pv);
            if (act) {
#pragma unroll
                for (int j = 0; j < 4; j++) pA[pos + j * PL] = pv[j];
            }
            parity4<T>(V2, pv);
            if (act) {
#pragma unroll
                for (int j = 0; j < 4; j++) pB[pos + j * PL] = pv[j];
            }
            __builtin_amdgcn_sched_barrier(0);  // one quartet's registers at a time
        }
        __syncthreads();  // 1: F and V2 complete

        // ---- everything but T1 V1
        acc_t ar[2], ai[2];
#pragma unroll
        for (int c = 0; c < 2; c++) ar[c] = ai[c] = MF::zero();
        {
            cT<T> s1 = czero<T>();  // axis sums of this lane's a
#pragma unroll
            for (int s = 0; s < KS; s++) {
                const cT<T> x1 = aw[orw + 4 * s];
#pragma unroll
                for (int c = 0; c < 2; c++) {  // b1 c1 (i K): K to the other parity and kc back
                    const T d = k1o[c] * sd1[c][4 * s * HP];
                    ar[c] = MF::fma(x1.x, d, ar[c]);
                    ai[c] = MF::fma(x1.y, d, ai[c]);
                }
                if (p1) {
                    const cT<T> y1 = a1[orw + 4 * s];
                    add_w(s1, s, y1);
                }
            }
            if (p1) {
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    ar[c] = MF::fma(-s1.y, rr1[c], ar[c]);
                    ai[c] = MF::fma(s1.x, rr1[c], ai[c]);
                }
            }
        }
        {
            const cT<T>* f = aw;
            const cT<T>* f2 = a2;
            const cT<T>* y2p = p2 ? f2 : f + OV;  // p2 odd: b2 c2 (c0 1 1^T F); even: c0 1 1^T V2
            cT<T> s2[2] = {czero<T>(), czero<T>()};
#pragma unroll
            for (int s = 0; s < KS; s++) {
                const T m = sm2[4 * s * HP], d = k2o * sd2[4 * s * HP];
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    const int o = ocl[c] + 4 * s * RS;
                    const cT<T> x2 = f[o], v = f2[OV + o], y2 = y2p[o];
                    ar[c] = MF::fma(d, x2.x, ar[c]);
                    ai[c] = MF::fma(d, x2.y, ai[c]);
                    ar[c] = MF::fma(m, -v.y, ar[c]);
                    ai[c] = MF::fma(m, v.x, ai[c]);
                    add_w(s2[c], s, y2);
                }
            }
#pragma unroll
            for (int c = 0; c < 2; c++) {
                ar[c] = MF::fma(rr2, p2 ? -s2[c].y : s2[c].x, ar[c]);
                ai[c] = MF::fma(rr2, p2 ? s2[c].x : s2[c].y, ai[c]);
            }
        }
        __syncthreads();  // 2: F and V2 consumed
        cT<T> f0v[NQ][4];
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            bool act;
            int pos, i1, i2;
            unsigned ob[4];
            quartet(q, act, pos, ob, i1, i2);
            cT<T> pv[4];
            parity4<T>(V1[q], pv);
            if (act) {
#pragma unroll
                for (int j = 0; j < 4; j++) pA[pos + j * PL] = pv[j];
            }
            const cT<T>* Fz = (sc.read_f0 ? F0 : Fin) + base;
            if (!sc.deriv_only) {
#pragma unroll
                for (int j = 0; j < 4; j++) f0v[q][j] = ld_once<T>(at_b(Fz, ob[j]));
            }
        }
        __syncthreads();  // 3: V1 complete
        {
            cT<T> s1 = czero<T>();
#pragma unroll
            for (int s = 0; s < KS; s++) {
                const cT<T> v = a1[orw + 4 * s];
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    const T m = sm1[c][4 * s * HP];
                    ar[c] = MF::fma(-v.y, m, ar[c]);
                    ai[c] = MF::fma(v.x, m, ai[c]);
                }
                if (!p1) {  // c0 1 1^T V1
                    const cT<T> y = aw[orw + 4 * s];
                    add_w(s1, s, y);
                }
            }
            if (!p1) {
#pragma unroll
                for (int c = 0; c < 2; c++) {
                    ar[c] = MF::fma(s1.x, rr1[c], ar[c]);
                    ai[c] = MF::fma(s1.y, rr1[c], ai[c]);
                }
            }
        }
#pragma unroll
        for (int c = 0; c < 2; c++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int o2 = 16 * rt + MF::orow(lq, v), o1 = 16 * c + lr;
                if (o2 < H1 && o1 < H1) pB[pl * PL + o2 * RS + o1] = cmk<T>(ar[c][v], ai[c][v]);
            }
        __syncthreads();  // 4: the result planes are complete, V1 consumed

        // ---- dF = unfolded planes + W, epilogue
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            bool act;
            int pos, i1, i2;
            unsigned ob[4];
            quartet(q, act, pos, ob, i1, i2);
            const bool self1 = i1 == 0 || i1 == H, self2 = i2 == 0 || i2 == H;
            const bool st[4] = {act, act && !self1, act && !self2, act && !self1 && !self2};
            cT<T> pv[4], y[4];
#pragma unroll
            for (int j = 0; j < 4; j++) pv[j] = pB[pos + j * PL];
            parity4<T>(pv, y);
            const T h = sc.dt * sc.cd;
#pragma unroll
            for (int j = 0; j < 4; j++) {  // every load is consumed before the first store
                y[j] = cadd<T>(y[j], W[q][j]);
                y[j] = sc.deriv_only ? cscale<T>(y[j], sc.dt)
                                     : cmk<T>(fma(h, y[j].x, f0v[q][j].x), fma(h, y[j].y, f0v[q][j].y));
                asm volatile("" : "+v"(y[j].x), "+v"(y[j].y));
            }
#pragma unroll
            for (int j = 0; j < 4; j++)
                if (st[j]) st_once<T>(at_b(Fout + base, ob[j]), y[j]);
        }
    }
}

// ------------------------------------------------------------ N <= 16 ----
//
// Omega grids of up to 16 points per axis: a slab is one 16 x 16 tile of the matrix
// instruction, unfolded, and one wave holds it whole, four elements a lane in the
// accumulators' layout.  The circulant T_p = c0 1 1^T + i K_p is a real 16 x 16 product
// and an axis sum; results and the mixing stay in registers, F, V2 and then V1 go through
// LDS to become operands.  A workgroup is one wave, so nothing waits for another wave:
// with four waves to a slab and three barriers the same work took two to three times as
// long (k_drift_fused_c; B = 12, N = 16 FP64 485 -> 177 us, FP32 222 -> 98 us; B = 20, 2-D,
// N = 14 FP64 142 -> 43 us, FP32 64 -> 24 us; k_drift_fold 1.2-1.7 times k_drift_fused_c's
// rate at N <= 14).  B = 12, N = 16, FP64: its streams take 120 of the 177 us at a copy's rate,
// the rest is gathered rows and issue at two waves a SIMD (FP32: four).  Two source rows in
// flight; three measured the same to 4 % slower, six 10-20 % slower in 3-D.
//
// ADJ: the adjoint operator, on the transposed tables and circulants of k_drift_fused's: the
// damping joins V1 and V2, and axis 3 comes whole as D.s3.  B = 10, N = 16, FP64, per launch
// (k_drift_fused before): 299 -> 95 us; the forward operator 281 -> 96 us.
template <class T, int DIM, bool ADJ>
__global__ __launch_bounds__(64, fold_waves<T>()) void k_drift_tile(DriftDev<T> D, MixDev<T> MX, const cT<T>* Fin,
                                                                    const cT<T>* __restrict__ Z3, const cT<T>* F0,
                                                                    cT<T>* Fout, StageCoef<T> sc, int nslab) {
    using MF = Mfma<T>;
    using acc_t = typename MF::acc;
    constexpr int NC = DIM + 2, MB = 2, RS = 17;
    __shared__ cT<T> pF[16 * RS], pV[16 * RS];  // F and then V1; V2
    const int N = D.N, NN = N * N, nz = DIM == 3 ? N : 1;
    const int lane = threadIdx.x, lr = lane & 15, lq = lane >> 4;
    for (int i = lane; i < 16 * RS; i += 64) pF[i] = pV[i] = czero<T>();

    // matrices K_1, K_2, entry [out lr][in 4 s + lq]
    T m1[4], m2[4];
    const T c1 = lr < N ? D.c0[0] : T(0), c2 = lr < N ? D.c0[1] : T(0);
#pragma unroll
    for (int s = 0; s < 4; s++) {
        const int a = 4 * s + lq, j = lr - a;
        const bool in = a < N && lr < N;
        m1[s] = in ? D.kap[j < 0 ? j + N : j].y : T(0);
        m2[s] = in ? D.kap[N + (j < 0 ? j + N : j)].y : T(0);
    }
    // the lane's elements (k2, k1 = lr)
    unsigned ob[4];
    bool ok[4];
    int ps[4];
    T kc2[4], dd0[4];
    const T kc1 = lr < N ? D.kc[lr] : T(0);
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int k2 = MF::orow(lq, v);
        ok[v] = lr < N && k2 < N;
        ob[v] = ok[v] ? (unsigned)(k2 * N + lr) * (unsigned)sizeof(cT<T>) : 0u;
        ps[v] = k2 * RS + lr;
        kc2[v] = ok[v] ? D.kc[k2] : T(0);
        // D(k) = sum_i G_ii kd(k_i) - sum_{i != j} G_ij kc(k_i) kc(k_j)
        dd0[v] = ok[v] ? D.G[0] * D.kd[lr] + D.G[DIM + 1] * D.kd[k2] - (D.G[1] + D.G[DIM]) * kc1 * kc2[v] : T(0);
    }
    const T g22 = DIM == 3 ? D.G[8] : T(0), g02 = DIM == 3 ? D.G[2] + D.G[6] : T(0), g12 = DIM == 3 ? D.G[5] + D.G[7] : T(0);
    const bool gyro = DIM == 3 && D.has_gyro;
    const int orw = lr * RS + lq, ocl = lq * RS + lr;
    __syncthreads();

    const int nrc = (int)D.nrc, TS = MX.TS;
    const int nxcd = gridDim.x >= 8 ? 8 : 1;
    const int per = (int)gridDim.x / nxcd;
    const int xcd = (int)blockIdx.x % nxcd;
    const int hi = (int)((int64_t)nslab * (xcd + 1) / nxcd);
    int sl = (int)((int64_t)nslab * xcd / nxcd) + (int)blockIdx.x / nxcd;  // slab sl: row sl % nrc of the walk, k3 = sl / nrc
    const int dr = per % nrc, dk = per / nrc;
    int rp = sl % nrc, k3 = sl / nrc;
    const kc_ptr<int32_t> ord = as_const<int32_t>(MX.order);
    while (sl < hi) {
        const int r = ord[rp];
        const int64_t base = ((int64_t)r * nz + k3) * NN;
        const T kc3 = DIM == 3 ? as_const<T>(D.kc)[k3] : T(0), kd3 = DIM == 3 ? as_const<T>(D.kd)[k3] : T(0);
        cT<T> fo[4], Zv[4], W[4], V1[4], V2[4];
#pragma unroll
        for (int v = 0; v < 4; v++) {
            fo[v] = *at_b(Fin + base, ob[v]);
            Zv[v] = DIM == 3 && (!ADJ || gyro) ? ld_once<T>(at_b(Z3 + base, ob[v])) : czero<T>();
        }
        const kc_ptr<int32_t> srcT = as_const<int32_t>(MX.src) + (int64_t)r * TS;
        const kc_ptr<T> coefT = as_const<T>((const T*)MX.coef) + 2 * (int64_t)r * TS * NC;
#pragma unroll
        for (int v = 0; v < 4; v++) {
            W[v] = ADJ && DIM == 3 ? ld_once<T>(at_b(D.s3 + base, ob[v])) : czero<T>();
            V1[v] = V2[v] = czero<T>();
        }
        for (int t0 = 0; t0 < TS; t0 += MB) {
            int src[MB];
            cT<T> fv[MB][4];
#pragma unroll
            for (int u = 0; u < MB; u++) src[u] = t0 + u < TS ? srcT[t0 + u] : -1;
#pragma unroll
            for (int u = 0; u < MB; u++) {
                const cT<T>* Fs = Fin + ((int64_t)(src[u] < 0 ? 0 : (src[u] & 0xffffff)) * nz + k3) * NN;
#pragma unroll
                for (int v = 0; v < 4; v++) fv[u][v] = *at_b(Fs, ob[v]);
            }
#pragma unroll
            for (int u = 0; u < MB; u++) {
                if (src[u] < 0) continue;
                const int fl = src[u] >> 24;
                const int64_t cb = (int64_t)(t0 + u) * NC;
                if (fl & 1) {
                    const T a = coefT[2 * cb] * kc1, g1 = coefT[2 * (cb + 1) + 1];
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const T b = g1 * kc2[v];
                        W[v].x = fma(a, fv[u][v].x, fma(-b, fv[u][v].y, W[v].x));
                        W[v].y = fma(a, fv[u][v].y, fma(b, fv[u][v].x, W[v].y));
                    }
                }
                if (fl & 2) {
                    const T ui = coefT[2 * (cb + DIM) + 1];
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        V1[v].x = fma(-ui, fv[u][v].y, V1[v].x);
                        V1[v].y = fma(ui, fv[u][v].x, V1[v].y);
                    }
                }
                if (fl & 4) {
                    const T ur = coefT[2 * (cb + DIM + 1)];
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        V2[v].x = fma(ur, fv[u][v].x, V2[v].x);
                        V2[v].y = fma(ur, fv[u][v].y, V2[v].y);
                    }
                }
            }
        }
        T e3r = T(0), e3i = T(0);
        if (DIM == 3 && !ADJ) {
            const kc_ptr<T> e3p = as_const<T>((const T*)D.e3) + 2 * (int64_t)r;
            e3r = e3p[0];
            e3i = e3p[1] + D.b[2] * kc3;
        }
#pragma unroll
        for (int v = 0; v < 4; v++) {
            T dd = dd0[v];
            if (DIM == 3) dd += g22 * kd3 - kc3 * (g02 * kc1 + g12 * kc2[v]);
            W[v].x = fma(dd, fo[v].x, W[v].x);
            W[v].y = fma(dd, fo[v].y, W[v].y);
            if (ADJ) {
                const T a1 = D.b[0] * kc1, a2 = D.b[1] * kc2[v];
                V1[v].x = fma(a1, fo[v].y, V1[v].x);
                V1[v].y = fma(-a1, fo[v].x, V1[v].y);
                V2[v].x = fma(a2, fo[v].y, V2[v].x);
                V2[v].y = fma(-a2, fo[v].x, V2[v].y);
            }
            if (DIM == 3) {
                if (gyro) {
                    const T z1 = kc2[v] * D.gyro[1], z2 = kc1 * D.gyro[0];
                    V1[v].x = fma(z1, Zv[v].y, V1[v].x);
                    V1[v].y = fma(-z1, Zv[v].x, V1[v].y);
                    V2[v].x = fma(z2, Zv[v].y, V2[v].x);
                    V2[v].y = fma(-z2, Zv[v].x, V2[v].y);
                }
                if (!ADJ) {
                    W[v].x = fma(e3r, Zv[v].x, fma(-e3i, Zv[v].y, W[v].x));
                    W[v].y = fma(e3r, Zv[v].y, fma(e3i, Zv[v].x, W[v].y));
                }
            }
            if (ok[v]) {
                pF[ps[v]] = fo[v];
                pV[ps[v]] = V2[v];
            }
        }
        cT<T> f0v[4];
        if (sc.read_f0) {
#pragma unroll
            for (int v = 0; v < 4; v++) f0v[v] = ld_once<T>(at_b(F0 + base, ob[v]));
        } else {
#pragma unroll
            for (int v = 0; v < 4; v++) f0v[v] = fo[v];
        }
        __syncthreads();  // (one wave: orders its LDS accesses)

        // ---- everything but T1 V1: T2 V2, and T_p F for the damping b_p c_p T_p F, c_p = i kc
        // (!ADJ), and the gyroscopic term.  Each has accumulators of its own: its terms
        // alternate in sign, and in one chain every addition would round at the size
        // of all their partial sums; and kc scales the sum, not the matrix, whose
        // entries stay rounded once.  Error of the FP32 derivative, 2-D, N = 8 / 14 / 16: 2.3e-7
        // / 2.7e-7 / 2.8e-7 in one chain, now 2.1e-7 / 2.3e-7 / 2.3e-7 (k_drift_fused_c 1.9e-7 /
        // 2.1e-7 / 2.3e-7); T2 F serves the gyroscopic term too (B = 10, N = 16, FP64: 100 -> 97
        // us).  The axis sums added over lanes by shuffles, not by the matrix instruction:
        // 1.9e-7 / 2.2e-7 / 2.2e-7, but FP32 8-18 % slower.
        {
            acc_t pr = MF::zero(), pi = MF::zero(), qr = MF::zero(), qi = MF::zero(), ar = MF::zero(), ai = MF::zero();
            cT<T> s1 = czero<T>(), s2 = czero<T>(), sv = czero<T>();  // axis sums of F along 1 and 2, of V2 along 2
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const cT<T> x1 = pF[orw + 4 * s], x2 = pF[ocl + 4 * s * RS], v = pV[ocl + 4 * s * RS];
                if (!ADJ) {
                    pr = MF::fma(-x1.y, m1[s], pr);
                    pi = MF::fma(x1.x, m1[s], pi);
                }
                if (!ADJ || gyro) {
                    qr = MF::fma(m2[s], -x2.y, qr);
                    qi = MF::fma(m2[s], x2.x, qi);
                }
                ar = MF::fma(m2[s], -v.y, ar);
                ai = MF::fma(m2[s], v.x, ai);
                s1 = cadd<T>(s1, x1);
                s2 = cadd<T>(s2, x2);
                sv = cadd<T>(sv, v);
            }
            if (!ADJ) {
                pr = MF::fma(s1.x, c1, pr);
                pi = MF::fma(s1.y, c1, pi);
            }
            qr = MF::fma(c2, s2.x, qr);
            qi = MF::fma(c2, s2.y, qi);
            ar = MF::fma(c2, sv.x, ar);
            ai = MF::fma(c2, sv.y, ai);
            const T k1 = D.b[0] * kc1, g3 = gyro ? kc3 * D.gyro[2] : T(0);
#pragma unroll
            for (int v = 0; v < 4; v++) {
                T wr = ar[v], wi = ai[v];
                if (!ADJ) {
                    const T k2 = D.b[1] * kc2[v];
                    wr = fma(-k1, pi[v], fma(-k2, qi[v], wr));
                    wi = fma(k1, pr[v], fma(k2, qr[v], wi));
                }
                W[v].x += wr;
                W[v].y += wi;
                if (gyro) {
                    V1[v].x = fma(g3, qi[v], V1[v].x);
                    V1[v].y = fma(-g3, qr[v], V1[v].y);
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int v = 0; v < 4; v++)
            if (ok[v]) pF[ps[v]] = V1[v];
        __syncthreads();
        acc_t ar = MF::zero(), ai = MF::zero();
        {
            cT<T> s1 = czero<T>();
#pragma unroll
            for (int s = 0; s < 4; s++) {
                const cT<T> v = pF[orw + 4 * s];
                ar = MF::fma(-v.y, m1[s], ar);
                ai = MF::fma(v.x, m1[s], ai);
                s1 = cadd<T>(s1, v);
            }
            ar = MF::fma(s1.x, c1, ar);
            ai = MF::fma(s1.y, c1, ai);
        }
        const T h = sc.dt * sc.cd;
        cT<T> y[4];
#pragma unroll
        for (int v = 0; v < 4; v++) {  // every load is consumed before the first store
            const cT<T> q = cmk<T>(ar[v] + W[v].x, ai[v] + W[v].y);
            y[v] = sc.deriv_only ? cscale<T>(q, sc.dt) : cmk<T>(fma(h, q.x, f0v[v].x), fma(h, q.y, f0v[v].y));
            asm volatile("" : "+v"(y[v].x), "+v"(y[v].y));
        }
#pragma unroll
        for (int v = 0; v < 4; v++)
            if (ok[v]) st_once<T>(at_b(Fout + base, ob[v]), y[v]);
        __syncthreads();  // V1 consumed
        sl += per;
        rp += dr;
        k3 += dk;
        if (rp >= nrc) {
            rp -= nrc;
            k3++;
        }
    }
}

// ---------------------------------------------------------- launcher -----

// N = 18 .. 30 (below, k_drift_tile): 3-D 1.07-1.39x, 2-D 1.2-1.3x in FP64 and 1.03-1.38x in
// FP32 faster than the kernels that serve the others.
template <class T> bool drift_fold_ok(const DriftDev<T>& D) {
    if (!D.ramp || !D.odd || !D.smix || !D.op || D.adj || (sizeof(T) == 4 && D.keep)) return false;
    return D.N % 2 == 0 && D.N >= 18 && D.N <= 30;
}

template <class T, int DIM, bool ADJ>
static void tile_t(const DriftDev<T>& D, const MixDev<T>& MX, const void* Fin, const void* Z3, const void* F0, void* Fout,
                   const StageCoef<T>& sc, hipStream_t st) {
    const int64_t nslab = D.nrc * (DIM == 3 ? D.N : 1);
    auto kern = k_drift_tile<T, DIM, ADJ>;
    const unsigned grid = persistent_blocks((const void*)kern, nslab, 64, 0);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(64), 0, st, D, MX, (const cT<T>*)Fin, (const cT<T>*)Z3, (const cT<T>*)F0,
                       (cT<T>*)Fout, sc, (int)nslab);
}
// Every N up to 16: faster at all of them (from one round of the waves on), even where
// most of the tile is padding (N = 4, B = 20: 1.9x FP32, 2.4x FP64)
template <class T> bool drift_tile_ok(const DriftDev<T>& D) {
    if (!D.ramp || !D.smix || D.gpart || (sizeof(T) == 4 && D.keep)) return false;
    return D.N <= 16;
}
template <class T>
void launch_drift_tile(const DriftDev<T>& D, const MixDev<T>& MX, const void* Fin, const void* Z3, const void* F0,
                       void* Fout, const StageCoef<T>& sc, hipStream_t st) {
    HPUP_REQUIRE(drift_tile_ok<T>(D) && !sc.read_acc && !sc.write_acc, HPUP_ERR_UNSUPPORTED,
                 "one-tile drift: real circulants, structured mixing, N <= 16, no stage sums");
    if (D.adj && D.dim == 3) tile_t<T, 3, true>(D, MX, Fin, Z3, F0, Fout, sc, st);
    else if (D.adj) tile_t<T, 2, true>(D, MX, Fin, Z3, F0, Fout, sc, st);
    else if (D.dim == 3) tile_t<T, 3, false>(D, MX, Fin, Z3, F0, Fout, sc, st);
    else tile_t<T, 2, false>(D, MX, Fin, Z3, F0, Fout, sc, st);
}

template <int KS, int NQ>
static void fold64_t(const DriftDev<double>& D, const MixDev<double>& MX, const void* Fin, const void* F0, void* Fout,
                     const StageCoef<double>& sc, hipStream_t st) {
    const size_t sh = sizeof(cT<double>) * 2 * 4 * (size_t)(4 * KS * (4 * KS + 1)) + sizeof(double) * 2 * (16 * KS * KS);
    auto kern = k_drift_fold64<KS, NQ>;
    allow_lds((const void*)kern, sh);
    const unsigned grid = persistent_blocks((const void*)kern, D.nrc, 512, sh);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(512), sh, st, D, MX, (const cT<double>*)Fin, (const cT<double>*)F0,
                       (cT<double>*)Fout, sc, (int)D.nrc);
}

bool drift_fold64_ok(const DriftDev<double>& D) {
    return D.ramp && D.odd && D.same12 && D.smix && D.op && !D.adj && D.dim == 2 && D.N % 2 == 0 && D.N >= 34 && D.N <= 62;
}
void launch_drift_fold64(const DriftDev<double>& D, const MixDev<double>& MX, const void* Fin, const void* F0, void* Fout,
                         const StageCoef<double>& sc, hipStream_t st) {
    HPUP_REQUIRE(drift_fold64_ok(D) && !sc.read_acc && !sc.write_acc, HPUP_ERR_UNSUPPORTED,
                 "folded drift, N = 34 .. 62: odd real circulants, structured mixing, no stage sums");
    const bool one = (D.N / 2 + 1) * (D.N / 2 + 1) <= 512;  // N <= 42
    switch ((D.N / 2 + 4) / 4) {
    case 5: return fold64_t<5, 1>(D, MX, Fin, F0, Fout, sc, st);
    case 6: return one ? fold64_t<6, 1>(D, MX, Fin, F0, Fout, sc, st) : fold64_t<6, 2>(D, MX, Fin, F0, Fout, sc, st);
    case 7: return fold64_t<7, 2>(D, MX, Fin, F0, Fout, sc, st);
    default: return fold64_t<8, 2>(D, MX, Fin, F0, Fout, sc, st);
    }
}

template <class T, int DIM, int KS, int XS>
static void fold_t(const DriftDev<T>& D, const MixDev<T>& MX, const void* Fin, const void* Z3, const void* F0, void* Fout,
                   const StageCoef<T>& sc, hipStream_t st) {
    const size_t sh = sizeof(cT<T>) * 3 * XS * 4 * (size_t)(4 * KS * (4 * KS + 1));
    HPUP_REQUIRE(DIM == 2 || D.N % XS == 0, HPUP_ERR_UNSUPPORTED, "folded drift: whole slab groups");
    const int nkg = DIM == 3 ? D.N / XS : 1;
    const int64_t ng = D.nrc * nkg;
    auto kern = k_drift_fold<T, DIM, KS, XS>;
    allow_lds((const void*)kern, sh);
    const unsigned grid = persistent_blocks((const void*)kern, ng, 256, sh);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(256), sh, st, D, MX, (const cT<T>*)Fin, (const cT<T>*)Z3, (const cT<T>*)F0,
                       (cT<T>*)Fout, sc, (int)ng);
}

template <class T>
void launch_drift_fold(const DriftDev<T>& D, const MixDev<T>& MX, const void* Fin, const void* Z3, const void* F0,
                       void* Fout, const StageCoef<T>& sc, hipStream_t st) {
    HPUP_REQUIRE(drift_fold_ok<T>(D) && !sc.read_acc && !sc.write_acc,
                 HPUP_ERR_UNSUPPORTED, "folded drift: odd real circulants, structured mixing, no stage sums");
    if (D.dim == 2)
        return D.N <= 22 ? fold_t<T, 2, 3, 1>(D, MX, Fin, Z3, F0, Fout, sc, st)
                         : fold_t<T, 2, 4, 1>(D, MX, Fin, Z3, F0, Fout, sc, st);
    // slabs per workgroup: as many quarter planes as 256 threads hold
    if (D.N <= 20) return fold_t<T, 3, 3, 2>(D, MX, Fin, Z3, F0, Fout, sc, st);  // N = 18, 20
    if (D.N == 22) return fold_t<T, 3, 3, 1>(D, MX, Fin, Z3, F0, Fout, sc, st);
    return fold_t<T, 3, 4, 1>(D, MX, Fin, Z3, F0, Fout, sc, st);  // N = 24 .. 30
}

template bool drift_tile_ok<float>(const DriftDev<float>&);
template bool drift_tile_ok<double>(const DriftDev<double>&);
template void launch_drift_tile<float>(const DriftDev<float>&, const MixDev<float>&, const void*, const void*, const void*,
                                       void*, const StageCoef<float>&, hipStream_t);
template void launch_drift_tile<double>(const DriftDev<double>&, const MixDev<double>&, const void*, const void*,
                                        const void*, void*, const StageCoef<double>&, hipStream_t);
template bool drift_fold_ok<float>(const DriftDev<float>&);
template bool drift_fold_ok<double>(const DriftDev<double>&);
template void launch_drift_fold<float>(const DriftDev<float>&, const MixDev<float>&, const void*, const void*, const void*,
                                       void*, const StageCoef<float>&, hipStream_t);
template void launch_drift_fold<double>(const DriftDev<double>&, const MixDev<double>&, const void*, const void*,
                                        const void*, void*, const StageCoef<double>&, hipStream_t);

}  // namespace hpup
