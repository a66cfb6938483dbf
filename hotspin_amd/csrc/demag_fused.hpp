// demag_fused.hpp -- the demag convolution in three kernels.
//
// The five passes of demag.hip carry the half spectrum through HBM three
// times (X1, then X2 with the padded axis 1, twice).  Where one x-frequency
// column of the mesh fits into LDS, the middle three passes become one:
//   k_frows  rows, R2C along axis 2                      m  -> X
//   k_fmid   per column: FFT along axis 1, convolution along axis 0 with the
//            kernel, inverse FFT along axis 1            X  -> X (in place)
//   k_irows  C2R along axis 2                            X  -> B
// so the spectrum is written twice and read twice and the padded axis 1
// exists in LDS only: 24 N + 48 N0 N1 H2 + 24 N0 (KR/..) bytes instead of
// 24 N + 48 N0 N1 H2 + 96 N0 P1 H2.
//
// X is column-major: [solve][k][c][i][j], k the x frequency, so that a column
// is one contiguous piece and W rows of the row passes (consecutive j) make
// contiguous pieces of 8 W bytes.
//
// Axis 0 is convolved directly: the kernel K~(d; j', k) is the transform of
// the real-space tensor along axes 1 and 2 only, d = i - i' the plane
// distance.  For the few planes of a film this takes fewer operations than a
// zero-padded FFT pair (36 N0 flop against about 10 P0 log2 P0 per output),
// no padding, and any N0.  Its components XX, YY, ZZ and YZ are real and even
// in d; XZ and XY (odd along axis 0) are imaginary and odd, K~ = i kappa.
// With u = i x_x in place of x_x and v = i y_x in place of y_x the tensor is
// real:  v   =  Kxx u - kxy x_y - kxz x_z
//        y_y =  kxy u + Kyy x_y + Kyz x_z
//        y_z =  kxz u + Kyz x_y + Kzz x_z,
// and -d transposes it.  A mirrored row P1 - j' has Kyz and kxy negated.
#pragma once

#include <algorithm>
#include <vector>

#include "fft2.hpp"

namespace fused {

constexpr int kEpt = 24;       // tile elements (complex) per thread of k_fmid, at most
constexpr int kMidMax = 512;   // threads of a k_fmid block
constexpr long kLds = 163840;

// Q = A * B with A even (the zero-padded half of the input rows is then a
// whole number of A-point inputs) and both factors near sqrt(Q)
constexpr Split2 split_even(int L) {
    Split2 best{0, 0};
    for (int a = 2; a <= 32; a += 2) {
        if (L % a) continue;
        const int b = L / a;
        if (!reg_dft_ok(a) || !reg_dft_ok(b) || b > 32) continue;
        const int d0 = best.A ? (best.A > best.B ? best.A - best.B : best.B - best.A) : 1 << 30;
        const int d1 = a > b ? a - b : b - a;
        if (d1 < d0 || (d1 == d0 && a < b)) best = Split2{a, b};
    }
    return best;
}

template <typename T>
struct Mid {
    cpx<T>* X;
    const T* kt;  // [column][d][KR][6]: XX, YY, ZZ, YZ, kappa XZ, kappa XY
    int N0, ncol, CB, nsolve;
    const cpx<T>* tw;  // w_Q^t, t < Q
    const int* live;   // per-solve flags or null
};

// Table rows of K~ for a Q-point axis 1: frequency q = k1 + A k2 sits in slot
// k1 B + k2; rows q and Q - q share |K|, and the slots k1 <= A/2 cover both.
constexpr int table_rows(int Q) { return (split_even(Q).A / 2 + 1) * split_even(Q).B; }

// the tensor at one distance and row (six values from an 8- or 16-byte boundary)
template <typename T>
struct Coef {
    T xx, yy, zz, yz, xz, xy;
    __device__ __forceinline__ void load(const T* p) {
        using V2 = typename std::conditional<sizeof(T) == 4, float2, double2>::type;
        const V2 a = *(const V2*)p, b = *(const V2*)(p + 2), c = *(const V2*)(p + 4);
        xx = a.x, yy = a.y, zz = b.x, yz = b.y, xz = c.x, xy = c.y;
    }
};
__device__ __forceinline__ float fmaT(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fmaT(double a, double b, double c) { return __builtin_fma(a, b, c); }
// axis-0 items per thread: 3 IB values each, at most kEpt in all
constexpr int mid_itm(int IB) { return 8 / IB; }

// One block: CB columns of one solve, 3 N0 pencils of Q points each, held in
// LDS as lds[pencil * A (B+1) + k1 (B+1) + k2] (the odd row pitch keeps both
// phases free of bank conflicts).  blockDim.x = elements / kEpt, rounded up
// to whole waves.
template <typename T, int Q, int IB, bool MULTI>
__global__ void __launch_bounds__(kMidMax) k_fmid(Mid<T> a) {
    constexpr int A = split_even(Q).A, B = split_even(Q).B, BP = B + 1, PL = A * BP, AIN = A / 2;
    constexpr int UA = (kEpt + A - 1) / A, UB = (kEpt + B - 1) / B, ITM = mid_itm(IB);
    constexpr int KR = (A / 2 + 1) * B, N1 = Q / 2;
    static_assert(A * B == Q && A % 2 == 0, "two-level split");
    extern __shared__ __align__(16) unsigned char mid_smem[];
    cpx<T>* tws = reinterpret_cast<cpx<T>*>(mid_smem);
    cpx<T>* lds = tws + Q;
    const int tid = threadIdx.x, NT = blockDim.x;
    const int lb = xcd_swizzle(blockIdx.x, gridDim.x);
    const int tile = lb / a.nsolve, sol = lb % a.nsolve;
    if (a.live && !a.live[sol]) return;
    const int N0 = a.N0, col0 = tile * a.CB, ncb = min(a.CB, a.ncol - col0);
    const int PC = 3 * N0, NP = PC * ncb;
    cpx<T>* X = a.X + ((long)sol * a.ncol + col0) * (long)(PC * N1);
    {  // phase 1: A-point DFTs over n1 of the rows j = B n1 + n2 < N1
        cpx<T> v[UA][A];
#pragma unroll
        for (int u = 0; u < UA; u++) {
            const int e = tid + u * NT;
            const int p = e / B, n2 = e % B;
            const cpx<T>* xp = X + (e < NP * B ? p * N1 + n2 : 0);
#pragma unroll
            for (int n1 = 0; n1 < AIN; n1++) v[u][n1] = xp[B * n1];
        }
        for (int t = tid; t < Q; t += NT) tws[t] = a.tw[t];
        __syncthreads();
#pragma unroll
        for (int u = 0; u < UA; u++) {
            const int e = tid + u * NT;
            const int p = e / B, n2 = e % B;
            if (e < NP * B) {
                if (p % PC < N0) {  // the x component enters as i x
#pragma unroll
                    for (int n1 = 0; n1 < AIN; n1++) v[u][n1] = {-v[u][n1].y, v[u][n1].x};
                }
#pragma unroll
                for (int n1 = AIN; n1 < A; n1++) v[u][n1] = {T(0), T(0)};
                dft_reg<T, A, -1>(v[u]);
#pragma unroll
                for (int k1 = 0; k1 < A; k1++)
                    lds[p * PL + k1 * BP + n2] = k1 ? cmul(v[u][k1], tws[n2 * k1]) : v[u][k1];
            }
        }
    }
    __syncthreads();
    {  // phase 2: B-point DFTs over n2, in place
#pragma unroll
        for (int u = 0; u < UB; u++) {
            const int e = tid + u * NT;
            if (e < NP * A) {
                cpx<T> w[B];
                cpx<T>* q = lds + e * BP;
#pragma unroll
                for (int m = 0; m < B; m++) w[m] = q[m];
                dft_reg<T, B, -1>(w);
#pragma unroll
                for (int m = 0; m < B; m++) q[m] = w[m];
            }
        }
    }
    __syncthreads();
    {  // axis 0: y(i) = sum_i' K~(i - i') x(i'); one item = IB planes of the three components at one slot
        const int NIB = MULTI ? (N0 + IB - 1) / IB : 1, items = ncb * NIB * Q;
        cpx<T> y[ITM][3][IB];
#pragma unroll
        for (int it = 0; it < ITM; it++) {
            const int e = tid + it * NT;
#pragma unroll
            for (int q = 0; q < IB; q++) y[it][0][q] = y[it][1][q] = y[it][2][q] = {T(0), T(0)};
            if (e < items) {
                const int slot = e % Q, r = e / Q, ib = MULTI ? r % NIB : 0, col = MULTI ? r / NIB : r;
                const int k1 = slot / B, k2 = slot % B;
                const bool mir = k1 > A / 2;
                const int row = mir ? (A - k1) * B + (B - 1 - k2) : slot;
                const T sj = mir ? T(-1) : T(1);
                const T* kb = a.kt + ((long)(col0 + col) * N0 * KR + row) * 6;
                const cpx<T>* xs = lds + col * PC * PL + k1 * BP + k2;
                // K~ at plane distance ad >= 0 for this row
                auto coef = [&](int ad, Coef<T>& w) {
                    w.load(kb + (long)ad * (6 * KR));
                    w.xy *= sj;
                    w.yz *= sj;
                };
                auto acc = [&](const Coef<T>& w, bool neg, const cpx<T>& x0, const cpx<T>& x1, const cpx<T>& x2,
                               int q) {
                    const T xy = neg ? -w.xy : w.xy, xz = neg ? -w.xz : w.xz;
                    cpx<T>&a0 = y[it][0][q], &a1 = y[it][1][q], &a2 = y[it][2][q];
                    // chained into the accumulators: three fma each (a sum of products
                    // added afterwards takes a fourth instruction)
                    a0.x = fmaT(-xz, x2.x, fmaT(-xy, x1.x, fmaT(w.xx, x0.x, a0.x)));
                    a0.y = fmaT(-xz, x2.y, fmaT(-xy, x1.y, fmaT(w.xx, x0.y, a0.y)));
                    a1.x = fmaT(w.yz, x2.x, fmaT(w.yy, x1.x, fmaT(xy, x0.x, a1.x)));
                    a1.y = fmaT(w.yz, x2.y, fmaT(w.yy, x1.y, fmaT(xy, x0.y, a1.y)));
                    a2.x = fmaT(w.zz, x2.x, fmaT(w.yz, x1.x, fmaT(xz, x0.x, a2.x)));
                    a2.y = fmaT(w.zz, x2.y, fmaT(w.yz, x1.y, fmaT(xz, x0.y, a2.y)));
                };
                if constexpr (!MULTI) {  // N0 == IB: every distance in registers, signs known at compile time
                    Coef<T> w[IB];
#pragma unroll
                    for (int d = 0; d < IB; d++) coef(d, w[d]);
#pragma unroll
                    for (int i = 0; i < IB; i++) {
                        const cpx<T> x0 = xs[i * PL], x1 = xs[(IB + i) * PL], x2 = xs[(2 * IB + i) * PL];
#pragma unroll
                        for (int q = 0; q < IB; q++) acc(w[q < i ? i - q : q - i], q < i, x0, x1, x2, q);
                    }
                } else {
                    // window w[n] = K~(i0 - ip - 3 + n), n < IB + 3, over the input planes ip .. ip + 3
                    // (the sign of the odd components taken when a distance enters)
                    const int i0 = ib * IB;
                    Coef<T> w[IB + 3];
                    auto enter = [&](int d, Coef<T>& o) {
                        coef(min(d < 0 ? -d : d, N0 - 1), o);
                        if (d < 0) {
                            o.xy = -o.xy;
                            o.xz = -o.xz;
                        }
                    };
#pragma unroll
                    for (int n = 4; n < IB + 3; n++) enter(i0 - 3 + n, w[n - 4]);
                    for (int ip = 0; ip < N0; ip += 4) {
#pragma unroll
                        for (int n = IB + 2; n >= 4; n--) w[n] = w[n - 4];
#pragma unroll
                        for (int n = 0; n < 4; n++) enter(i0 - ip - 3 + n, w[n]);
#pragma unroll
                        for (int r2 = 0; r2 < 4; r2++) {
                            const int i = min(ip + r2, N0 - 1);
                            cpx<T> x0 = xs[i * PL], x1 = xs[(N0 + i) * PL], x2 = xs[(2 * N0 + i) * PL];
                            if (ip + r2 >= N0) x0 = x1 = x2 = {T(0), T(0)};
#pragma unroll
                            for (int q = 0; q < IB; q++) acc(w[q - r2 + 3], false, x0, x1, x2, q);
                        }
                    }
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int it = 0; it < ITM; it++) {
            const int e = tid + it * NT;
            if (e < items) {
                const int slot = e % Q, r = e / Q, ib = MULTI ? r % NIB : 0, col = MULTI ? r / NIB : r;
                cpx<T>* o = lds + (col * PC + ib * IB) * PL + (slot / B) * BP + slot % B;
#pragma unroll
                for (int c = 0; c < 3; c++)
#pragma unroll
                    for (int q = 0; q < IB; q++)
                        if (!MULTI || ib * IB + q < N0) o[(c * N0 + q) * PL] = y[it][c][q];
            }
        }
    }
    __syncthreads();
    {  // inverse phase 2: B-point DFTs over k2 in place, then the twiddle
#pragma unroll
        for (int u = 0; u < UB; u++) {
            const int e = tid + u * NT;
            if (e < NP * A) {
                cpx<T> w[B];
                cpx<T>* q = lds + e * BP;
                const int k1 = e % A;
#pragma unroll
                for (int m = 0; m < B; m++) w[m] = q[m];
                dft_reg<T, B, +1>(w);
#pragma unroll
                for (int m = 0; m < B; m++) {
                    cpx<T> t = tws[m * k1];
                    t.y = -t.y;
                    q[m] = m ? cmul(w[m], t) : w[m];
                }
            }
        }
    }
    __syncthreads();
    {  // inverse phase 1: A-point DFTs over k1, the rows j < N1 stored
#pragma unroll
        for (int u = 0; u < UA; u++) {
            const int e = tid + u * NT;
            if (e < NP * B) {
                const int p = e / B, n2 = e % B;
                cpx<T> v[A];
#pragma unroll
                for (int k1 = 0; k1 < A; k1++) v[k1] = lds[p * PL + k1 * BP + n2];
                dft_reg<T, A, +1>(v);
                cpx<T>* xp = X + p * N1 + n2;
                if (p % PC < N0) {  // y_x = -i v
#pragma unroll
                    for (int n1 = 0; n1 < AIN; n1++) xp[B * n1] = {v[n1].y, -v[n1].x};
                } else {
#pragma unroll
                    for (int n1 = 0; n1 < AIN; n1++) xp[B * n1] = v[n1];
                }
            }
        }
    }
}

// ---- row passes -----------------------------------------------------------
// M = P2/2 points; LDS row pitch of the W spectrum rows: lanes walk the rows
// first (64/W points of each), and this pitch puts those 64 words on distinct
// banks.
template <int M, int W>
constexpr int row_pitch() {
    return M + 1 + ((64 / W - (M + 1)) % 32 + 32) % 32;
}
template <int M, int W>
constexpr int frow_lds() {
    constexpr int A = split2(M).A, B = split2(M).B;
    return (W * A * (B + 1) > W * row_pitch<M, W>()) ? W * A * (B + 1) : W * row_pitch<M, W>();
}

// R2C of rows [row0, row0 + W) of x times 2 half (rows of n2 reals; the mask
// repeats every mrows rows), out column-major: out[(sol (M+1) + k) rows + row].
template <typename T, int M, int W, int NT = W * split2(M).B>
__global__ void __launch_bounds__(NT) k_frows(const T* __restrict__ x, const T* __restrict__ msk, long mrows,
                                              cpx<T>* __restrict__ out, long nrows, int rows, int n2,
                                              T half, const cpx<T>* __restrict__ twM,
                                              const cpx<T>* __restrict__ twP, Live lv) {
    constexpr int A = split2(M).A, B = split2(M).B, BP = B + 1, PM = row_pitch<M, W>();
    static_assert(A * B == M && A <= B, "two-level split");
    __shared__ cpx<T> lds[frow_lds<M, W>()];
    __shared__ cpx<T> tws[M + 1];
    const int tid = threadIdx.x;
    const long row0 = (long)xcd_swizzle(blockIdx.x, gridDim.x) * W;
    if (all_dead(lv, row0, (row0 + W <= nrows ? row0 + W : nrows) - 1)) return;
    constexpr int TA = (M + NT - 1) / NT, TB = (M + 1 + NT - 1) / NT;
    cpx<T> ta[TA], tb[TB];
#pragma unroll
    for (int q = 0; q < TA; q++) ta[q] = twM[tid + q * NT < M ? tid + q * NT : 0];
#pragma unroll
    for (int q = 0; q < TB; q++) tb[q] = twP[tid + q * NT <= M ? tid + q * NT : 0];
    {
        const int nb = tid % B, p = tid / B;
        const long r = row0 + p;
        const bool rin = r < nrows;
        const long rc = rin ? r : row0;
        const T* xr = x + rc * n2;
        const T* mr = msk ? msk + (rc % mrows) * n2 : nullptr;
        cpx<T> v[A];
        if ((n2 & 1) == 0) {  // uniform
            using V2 = typename std::conditional<sizeof(T) == 4, float2, double2>::type;
            V2 q[A];
#pragma unroll
            for (int n1 = 0; n1 < A; n1++) {
                q[n1].x = q[n1].y = T(0);
                if (2 * B * n1 < n2) {  // uniform: some lane's pair is a cell
                    const int n = B * n1 + nb;
                    q[n1] = *(const V2*)(xr + 2 * (2 * n < n2 ? n : 0));
                }
            }
            if (mr) {  // uniform
#pragma unroll
                for (int n1 = 0; n1 < A; n1++)
                    if (2 * B * n1 < n2) {
                        const int n = B * n1 + nb;
                        const V2 w = *(const V2*)(mr + 2 * (2 * n < n2 ? n : 0));
                        q[n1].x *= w.x;
                        q[n1].y *= w.y;
                    }
            }
#pragma unroll
            for (int n1 = 0; n1 < A; n1++) {
                const bool ok = rin && 2 * (B * n1 + nb) < n2;
                v[n1] = {ok ? T(q[n1].x) : T(0), ok ? T(q[n1].y) : T(0)};
            }
        } else {
#pragma unroll
            for (int n1 = 0; n1 < A; n1++) {
                const int n = B * n1 + nb;
                const int i0 = 2 * n < n2 ? 2 * n : 0, i1 = 2 * n + 1 < n2 ? 2 * n + 1 : 0;
                cpx<T> z = {T(0), T(0)};
                if (2 * B * n1 < n2) {  // uniform
                    z = {xr[i0], xr[i1]};
                    if (mr) {
                        z.x *= mr[i0];
                        z.y *= mr[i1];
                    }
                }
                v[n1] = {rin && 2 * n < n2 ? z.x : T(0), rin && 2 * n + 1 < n2 ? z.y : T(0)};
            }
        }
#pragma unroll
        for (int q = 0; q < TA; q++)
            if (tid + q * NT < M) tws[tid + q * NT] = ta[q];
        __syncthreads();
        dft_reg<T, A, -1>(v);
#pragma unroll
        for (int k1 = 0; k1 < A; k1++) lds[(p * A + k1) * BP + nb] = k1 ? cmul(v[k1], tws[nb * k1]) : v[k1];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < TB; q++)
        if (tid + q * NT <= M) tws[tid + q * NT] = tb[q];
    cpx<T> u[B];
    const int k1 = tid % A, p2 = tid / A;
    if (tid < W * A) {
#pragma unroll
        for (int m = 0; m < B; m++) u[m] = lds[(p2 * A + k1) * BP + m];
        dft_reg<T, B, -1>(u);
    }
    __syncthreads();
    if (tid < W * A) {
#pragma unroll
        for (int k2 = 0; k2 < B; k2++) lds[p2 * PM + k1 + A * k2] = u[k2];
    }
    __syncthreads();
    // split X[k] = E + w^k O: lanes walk the W rows first, so that a column's W values leave together
    const int p = tid % W, kk = tid / W;
    const long r = row0 + p;
    if (r < nrows) {
        const long sol = r / rows;
        cpx<T>* o = out + sol * (M + 1) * (long)rows + (r - sol * rows);
        auto split = [&](int k) {
            const cpx<T> zk = lds[p * PM + (k == M ? 0 : k)];
            const cpx<T> zm = lds[p * PM + (k == 0 ? 0 : M - k)];
            const cpx<T> E = {half * (zk.x + zm.x), half * (zk.y - zm.y)};
            const cpx<T> O = {half * (zk.y + zm.y), half * (zm.x - zk.x)};
            o[(long)k * rows] = cadd(E, cmul(tws[k], O));
        };
#pragma unroll
        for (int q = 0; q < A; q++) split(kk + B * q);
        if (kk == 0) split(M);
    }
}

// C2R of rows [row0, row0 + W) from the column-major spectrum.
template <typename T, int M, int W, int NT = W * split2(M).B>
__global__ void __launch_bounds__(NT) k_irows(const cpx<T>* __restrict__ in, T* __restrict__ x, long nrows, int rows,
                                              int n2, const cpx<T>* __restrict__ twM,
                                              const cpx<T>* __restrict__ twP, Live lv) {
    constexpr int A = split2(M).A, B = split2(M).B, BP = B + 1, PM = row_pitch<M, W>();
    static_assert(A * B == M && A <= B, "two-level split");
    __shared__ cpx<T> lds[frow_lds<M, W>()];
    __shared__ cpx<T> tws[M];
    __shared__ cpx<T> twp[M];
    const int tid = threadIdx.x;
    const long row0 = (long)xcd_swizzle(blockIdx.x, gridDim.x) * W;
    if (all_dead(lv, row0, (row0 + W <= nrows ? row0 + W : nrows) - 1)) return;
    {
        const int p = tid % W, kk = tid / W;
        const long r = row0 + p < nrows ? row0 + p : row0;  // a valid row for the lanes past the end
        const long sol = r / rows;
        const cpx<T>* q0 = in + sol * (M + 1) * (long)rows + (r - sol * rows);
        constexpr int TA = (M + NT - 1) / NT;
        cpx<T> g[A], gm, ta[TA], tb[TA];
#pragma unroll
        for (int q = 0; q < A; q++) g[q] = q0[(long)(kk + B * q) * rows];
        gm = q0[(long)M * rows];
#pragma unroll
        for (int q = 0; q < TA; q++) {
            const int e = tid + q * NT;
            ta[q] = twM[e < M ? e : 0];
            tb[q] = twP[e < M ? e : 0];
        }
#pragma unroll
        for (int q = 0; q < A; q++) lds[p * PM + kk + B * q] = g[q];
        if (kk == 0) lds[p * PM + M] = gm;
#pragma unroll
        for (int q = 0; q < TA; q++) {
            const int e = tid + q * NT;
            if (e < M) {
                tws[e] = ta[q];
                twp[e] = tb[q];
            }
        }
    }
    __syncthreads();
    const int nb = tid % B, p = tid / B;
    cpx<T> v[A];
#pragma unroll
    for (int n1 = 0; n1 < A; n1++) {
        const int k = B * n1 + nb;
        cpx<T> a = lds[p * PM + k];
        cpx<T> b = lds[p * PM + (M - k)];
        cpx<T> s = {a.x + b.x, a.y - b.y};
        cpx<T> d = {a.x - b.x, a.y + b.y};
        cpx<T> w = twp[k];
        w.y = -w.y;
        cpx<T> wd = cmul(w, d);
        v[n1] = {s.x - wd.y, s.y + wd.x};
    }
    __syncthreads();
    dft_reg<T, A, +1>(v);
#pragma unroll
    for (int k1 = 0; k1 < A; k1++) {
        cpx<T> w = tws[nb * k1];
        w.y = -w.y;
        lds[(p * A + k1) * BP + nb] = k1 ? cmul(v[k1], w) : v[k1];
    }
    __syncthreads();
    if (tid < W * A) {
        const int k1 = tid % A, p2 = tid / A;
        const long r = row0 + p2;
        cpx<T> u[B];
#pragma unroll
        for (int m = 0; m < B; m++) u[m] = lds[(p2 * A + k1) * BP + m];
        dft_reg<T, B, +1>(u);
        if (r < nrows) {
            using V2 = typename std::conditional<sizeof(T) == 4, float2, double2>::type;
            T* xr = x + r * n2;
#pragma unroll
            for (int k2 = 0; k2 < B; k2++) {
                const int n = k1 + A * k2;
                if (2 * A * k2 < n2) {  // uniform
                    if ((n2 & 1) == 0) {
                        if (2 * n < n2) {
                            V2 q;
                            q.x = u[k2].x;
                            q.y = u[k2].y;
                            *(V2*)(xr + 2 * n) = q;
                        }
                    } else {
                        if (2 * n < n2) xr[2 * n] = u[k2].x;
                        if (2 * n + 1 < n2) xr[2 * n + 1] = u[k2].y;
                    }
                }
            }
        }
    }
}

// ---- launch shapes ------------------------------------------------------------
inline size_t mid_lds(int Q, int A, int B, int N0, int CB, size_t cs) {
    return ((size_t)3 * N0 * CB * A * (B + 1) + Q) * cs;
}
// planes per axis-0 item: all N0 of them up to 8, beyond that the one of 6
// and 8 that pads N0 less
inline int mid_ib(int N0) {
    if (N0 <= 8) return N0;
    return (N0 + 5) / 6 * 6 < (N0 + 7) / 8 * 8 ? 6 : 8;
}
// threads of a block: mid_itm axis-0 items each
inline int mid_nt(int N0, int Q, int CB) {
    const int IB = mid_ib(N0), items = CB * ((N0 + IB - 1) / IB) * Q, itm = mid_itm(IB);
    return ((items + itm - 1) / itm + 63) / 64 * 64;
}
// whether a column of the mesh fits one block
inline bool mid_fits(int N0, int Q, int A, int B, size_t cs) {
    return mid_nt(N0, Q, 1) <= kMidMax && mid_lds(Q, A, B, N0, 1, cs) <= (size_t)kLds;
}
// Columns per block: about 6144 elements (three blocks a CU), fewer while the
// launch would leave CUs idle.  A column's arithmetic does not depend on it.
inline int mid_cb(int N0, int Q, int A, int B, int ncol, int nsolve, size_t cs) {
    int cb = std::max(1, 6144 * 8 / (int)cs / (3 * N0 * Q));
    cb = std::min(cb, ncol);
    while (cb > 1 && ((long)((ncol + cb - 1) / cb) * nsolve < 512 || mid_nt(N0, Q, cb) > kMidMax ||
                      mid_lds(Q, A, B, N0, cb, cs) > (size_t)kLds))
        cb--;
    return cb;
}
// ---- registry ---------------------------------------------------------------
template <typename T>
using frows_t = void (*)(const T*, const T*, long, cpx<T>*, long, int, int, T, const cpx<T>*, const cpx<T>*,
                         hipStream_t, Live);
template <typename T>
using irows_t = void (*)(const cpx<T>*, T*, long, int, int, const cpx<T>*, const cpx<T>*, hipStream_t, Live);
template <typename T>
using mid_t = void (*)(const Mid<T>&, hipStream_t);

template <typename T>
struct Rows {
    frows_t<T> fwd = nullptr;
    irows_t<T> inv = nullptr;
};
template <typename T>
struct Mids {
    mid_t<T> one[9] = {};    // N0 = 1..8 planes
    mid_t<T> multi[9] = {};  // more, in blocks of 6 or 8
    int A = 0, B = 0;
    mid_t<T> pick(int N0) const { return N0 <= 8 ? one[N0] : multi[mid_ib(N0)]; }
};
template <typename T>
Rows<T>& rows_of(int M);  // registries, defined in demag.hip
template <typename T>
Mids<T>& mids_of(int Q);

// Rows per block: full 128-byte pieces of a column (16 rows of 8 bytes) while
// the tile stays near 32 KB.
template <typename T, int M>
constexpr int frow_w() {
    int w = 128 / (int)sizeof(cpx<T>);
    while (w > 2 && ((long)w * M * (long)sizeof(cpx<T>) > 40000 || w * split2(M).B > 1024)) w /= 2;
    while (w < 16 && w * split2(M).B < 64) w *= 2;
    return w;
}
template <typename T, int M>
void launch_frows(const T* x, const T* msk, long mrows, cpx<T>* out, long nrows, int rows, int n2, T half,
                  const cpx<T>* twM, const cpx<T>* twP, hipStream_t st, Live lv) {
    constexpr int W = frow_w<T, M>();
    hipLaunchKernelGGL((k_frows<T, M, W>), dim3((unsigned)((nrows + W - 1) / W)), dim3(W * split2(M).B), 0, st, x, msk,
                       mrows, out, nrows, rows, n2, half, twM, twP, lv);
}
template <typename T, int M>
void launch_irows(const cpx<T>* in, T* x, long nrows, int rows, int n2, const cpx<T>* twM, const cpx<T>* twP,
                  hipStream_t st, Live lv) {
    constexpr int W = frow_w<T, M>();
    hipLaunchKernelGGL((k_irows<T, M, W>), dim3((unsigned)((nrows + W - 1) / W)), dim3(W * split2(M).B), 0, st, in, x,
                       nrows, rows, n2, twM, twP, lv);
}

template <typename T, int Q, int IB, bool MULTI>
void launch_mid(const Mid<T>& m, hipStream_t st) {
    constexpr int A = split_even(Q).A, B = split_even(Q).B;
    const size_t lds = mid_lds(Q, A, B, m.N0, m.CB, sizeof(cpx<T>));
    const int nt = mid_nt(m.N0, Q, m.CB);
    if (lds > 65536)
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&k_fmid<T, Q, IB, MULTI>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    const unsigned g = (unsigned)((m.ncol + m.CB - 1) / m.CB) * (unsigned)m.nsolve;
    hipLaunchKernelGGL((k_fmid<T, Q, IB, MULTI>), dim3(g), dim3(nt), lds, st, m);
}

template <typename T, int M>
void add_rows() {
    if constexpr (two_level_ok(M) && M >= 8) rows_of<T>(M) = {&launch_frows<T, M>, &launch_irows<T, M>};
}
template <typename T, int Q, int IB>
void add_mid_ib(Mids<T>& m) {
    // only what can fit a block (mid_fits): LDS, and items per thread
    constexpr int A = split_even(Q).A, B = split_even(Q).B;
    constexpr long lds = (3L * IB * A * (B + 1) + Q) * (long)sizeof(cpx<T>);
    if constexpr (lds <= kLds && Q <= kMidMax * mid_itm(IB)) m.one[IB] = &launch_mid<T, Q, IB, false>;
    if constexpr ((IB == 6 || IB == 8) && lds * 3 / 2 <= kLds) m.multi[IB] = &launch_mid<T, Q, IB, true>;
}
template <typename T, int Q>
void add_mid() {
    if constexpr (split_even(Q).A > 0) {
        Mids<T>& m = mids_of<T>(Q);
        m.A = split_even(Q).A;
        m.B = split_even(Q).B;
        add_mid_ib<T, Q, 1>(m), add_mid_ib<T, Q, 2>(m), add_mid_ib<T, Q, 3>(m), add_mid_ib<T, Q, 4>(m);
        add_mid_ib<T, Q, 5>(m), add_mid_ib<T, Q, 6>(m), add_mid_ib<T, Q, 7>(m), add_mid_ib<T, Q, 8>(m);
    }
}
template <typename T, int L>
void register_len() {
    add_rows<T, L>();
    add_mid<T, L>();
}
}  // namespace fused
