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
// exists in LDS only.  Bytes a field in FP32: 24 N + 96 N0 N1 H2 and the
// kernel table, instead of 24 N + 96 N0 N1 H2 + 96 N0 P1 H2 and the octant; with
// axis 1 folded (k_frows) 24 N + 96 N0 P1 H2 and the table.
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
// With u = i x_x in place of x_x and v = -i y_x in place of y_x the tensor is
// real and symmetric:
//        v   = -Kxx u + kxy x_y + kxz x_z
//        y_y =  kxy u + Kyy x_y + Kyz x_z
//        y_z =  kxz u + Kyz x_y + Kzz x_z;
// at -d kxy and kxz are negated, in a mirrored row P1 - j' kxy and Kyz.
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
    const T* kt;  // [column][d][KR][6]: -XX, YY, ZZ, YZ, kappa XZ, kappa XY
    int N0, N1, ncol, CB, nsolve, R;
    const cpx<T>* tw;  // w_P1^t, P1 = Q R
    const int* live;   // per-solve flags or null
};

// Table rows of K~ for a Q-point axis 1: frequency q = k1 + A k2 sits in slot
// k1 B + k2; rows q and Q - q share |K|, and the slots k1 <= A/2 cover both.
// A folded column (see k_frows) has all Q rows; its mirror is another column.
constexpr int table_rows(int Q, bool fold) { return fold ? Q : (split_even(Q).A / 2 + 1) * split_even(Q).B; }
// K~ columns per x frequency: 1, or the residues s <= R/2 of a folded axis 1
constexpr int table_cols(int R) { return R > 1 ? R / 2 + 1 : 1; }

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
// Planes per item of unfolded FP32 launches that leave the chip mostly idle (fewer
// than kFewWaves waves with the usual items of 6 or 8, one a thread): twice the
// threads share the N0^2 products.  The sums are formed in the same order, so a
// solve's bits do not depend on it.  One field with the usual items / with four
// planes: 32^3 (132 waves) 25.1 / 21.1 us, 16x16x32 23.9 / 18.2, 64x64x16 22.7 /
// 19.1, 512x8x32 (513) 33.6 / 28.7, 512x32x16 (1026) 33.7 / 30.2, but 256x64x9
// (1028) 23.6 / 24.9 and 512x64x9 (2052) 31.5 / 34.9.
constexpr int kFewIB = 4;
constexpr long kFewWaves = 1024;
// axis-0 items per thread: 3 IB values each, at most 24 in all
constexpr int mid_itm(int IB, bool multi = false) { return multi && IB == kFewIB ? 1 : 8 / IB; }

// Shape of a column's tile.
template <int Q_, bool FOLD>
struct Geom {
    static constexpr int Q = Q_, A = split_even(Q_).A, B = split_even(Q_).B, BP = B + 1, PL = A * BP;
    static constexpr int KR = table_rows(Q_, FOLD);
};

// The table entry (distance 0) of column tc's slot; sj = -1 for a mirrored row.
template <typename T, bool FOLD, typename G>
__device__ __forceinline__ const T* table_row(const Mid<T>& a, const G& g, int tc, int slot, int k1, int k2, T& sj) {
    bool mir;
    int row;
    if constexpr (FOLD) {  // column k R + s: frequencies R q + s, mirrored at R (Q - 1 - q) + R - s
        const int k = tc / a.R, s = tc % a.R;
        mir = 2 * s > a.R;
        row = mir ? g.Q - 1 - slot : slot;
        tc = k * (a.R / 2 + 1) + (mir ? a.R - s : s);
    } else {
        mir = k1 > g.A / 2;
        row = mir ? (g.A - k1) * g.B + (g.B - 1 - k2) : slot;
    }
    sj = mir ? T(-1) : T(1);
    return a.kt + ((long)tc * a.N0 * g.KR + row) * 6;
}

// Axis 0: y(i) = sum_i' K~(i - i') x(i') in place; one item = IB planes of the
// three components at one slot (MULTI: N0 > IB).
template <typename T, int IB, bool MULTI, bool FOLD, typename G>
__device__ __forceinline__ void axis0(const Mid<T>& a, const G& g, cpx<T>* lds, int col0, int ncb) {
    constexpr int ITM = mid_itm(IB, MULTI);
    const int tid = threadIdx.x, NT = blockDim.x, N0 = a.N0, PC = 3 * N0, PL = g.PL;
    const int NIB = MULTI ? (N0 + IB - 1) / IB : 1, items = ncb * NIB * g.Q;
    cpx<T> y[ITM][3][IB];
#pragma unroll
    for (int it = 0; it < ITM; it++) {
        const int e = tid + it * NT;
#pragma unroll
        for (int q = 0; q < IB; q++) y[it][0][q] = y[it][1][q] = y[it][2][q] = {T(0), T(0)};
        if (e < items) {
            const int r = e / g.Q, slot = e - r * g.Q, ib = MULTI ? r % NIB : 0, col = MULTI ? r / NIB : r;
            const int k1 = slot / g.B, k2 = slot - k1 * g.B;
            T sj;
            const T* kb = table_row<T, FOLD>(a, g, col0 + col, slot, k1, k2, sj);
            const cpx<T>* xs = lds + col * PC * PL + k1 * g.BP + k2;
            // K~ at plane distance ad >= 0 for this row
            auto coef = [&](int ad, Coef<T>& w) {
                w.load(kb + (long)ad * (6 * g.KR));
                w.xy *= sj;
                w.yz *= sj;
            };
            auto acc = [&](const Coef<T>& w, bool neg, const cpx<T>& x0, const cpx<T>& x1, const cpx<T>& x2,
                           int q) {
                const T xy = neg ? -w.xy : w.xy, xz = neg ? -w.xz : w.xz;
                cpx<T>&a0 = y[it][0][q], &a1 = y[it][1][q], &a2 = y[it][2][q];
                // chained into the accumulators: three fma each (a sum of products
                // added afterwards takes a fourth instruction)
                a0.x = fmaT(xz, x2.x, fmaT(xy, x1.x, fmaT(w.xx, x0.x, a0.x)));
                a0.y = fmaT(xz, x2.y, fmaT(xy, x1.y, fmaT(w.xx, x0.y, a0.y)));
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
            const int r = e / g.Q, slot = e - r * g.Q, ib = MULTI ? r % NIB : 0, col = MULTI ? r / NIB : r;
            const int k1 = slot / g.B, k2 = slot - k1 * g.B;
            cpx<T>* o = lds + (col * PC + ib * IB) * PL + k1 * g.BP + k2;
#pragma unroll
            for (int c = 0; c < 3; c++)
#pragma unroll
                for (int q = 0; q < IB; q++)
                    if (!MULTI || ib * IB + q < N0) o[(c * N0 + q) * PL] = y[it][c][q];
        }
    }
    __syncthreads();
}

// One block: CB columns of one solve, 3 N0 pencils of Q points each, held in
// LDS as lds[pencil * A (B+1) + k1 (B+1) + k2] (the odd row pitch keeps both
// phases free of bank conflicts).  Axis 0 in items of IB planes (MULTI: N0 >
// IB); blockDim.x gives a thread mid_itm(IB) items, 12 to 24 elements, rounded up
// to whole waves (mid_nt).
template <typename T, int Q, int IB, bool MULTI, bool FOLD>
__global__ void __launch_bounds__(kMidMax) k_fmid(Mid<T> a) {
    using G = Geom<Q, FOLD>;
    constexpr int A = G::A, B = G::B, BP = G::BP, PL = G::PL, AIN = FOLD ? A : A / 2;
    constexpr int UA = (kEpt + A - 1) / A, UB = (kEpt + B - 1) / B;
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
    const int N1 = FOLD ? Q : a.N1;           // rows a column has in X
    const bool half = FOLD || 2 * N1 == Q;    // uniform: they are those of the A-point inputs n1 < AIN
    cpx<T>* X = a.X + ((long)sol * a.ncol + col0) * (long)(PC * N1);
    {  // phase 1: A-point DFTs over n1 of the rows j = B n1 + n2 < N1 (the upper half is padding unless folded)
        cpx<T> v[UA][A];
#pragma unroll
        for (int u = 0; u < UA; u++) {
            const int e = tid + u * NT;
            const int p = e / B, n2 = e % B;
            const cpx<T>* xp = X + (e < NP * B ? p * N1 : 0) + n2;
            if (half) {
#pragma unroll
                for (int n1 = 0; n1 < AIN; n1++) v[u][n1] = xp[B * n1];
            } else {
#pragma unroll
                for (int n1 = 0; n1 < AIN; n1++) v[u][n1] = xp[B * n1 + n2 < N1 ? B * n1 : -n2];
#pragma unroll
                for (int n1 = 0; n1 < AIN; n1++)
                    if (B * n1 + n2 >= N1) v[u][n1] = {T(0), T(0)};
            }
        }
        for (int t = tid; t < Q; t += NT) tws[t] = a.tw[FOLD ? t * a.R : t];
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
    axis0<T, IB, MULTI, FOLD>(a, G{}, lds, col0, ncb);
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
                if (p % PC < N0) {  // y_x = i v
#pragma unroll
                    for (int n1 = 0; n1 < AIN; n1++) v[n1] = {-v[n1].y, v[n1].x};
                }
                if (half) {
#pragma unroll
                    for (int n1 = 0; n1 < AIN; n1++) xp[B * n1] = v[n1];
                } else {
#pragma unroll
                    for (int n1 = 0; n1 < AIN; n1++)
                        if (B * n1 + n2 < N1) xp[B * n1] = v[n1];
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
constexpr int frow_full() {
    constexpr int A = split2(M).A, B = split2(M).B;
    return (W * A * (B + 1) > W * row_pitch<M, W>()) ? W * A * (B + 1) : W * row_pitch<M, W>();
}
// Folded FP32 rows whose tile is larger than 48 KB go through LDS in halves,
// even frequencies (in the exchange: even k1) first, then odd: the pairs k,
// M - k that R2C and C2R need have one parity.  The room goes into more rows a
// block, for longer pieces of a column: at 512x512x16, folded 8 ways, 32 rows
// in halves (64-byte pieces) take 57 us forward and 77 inverse, 16 rows (32-byte
// pieces) whole 73 and 81, in halves 76 and 82; 252 MB at the copy rate take 53.
template <typename T, int M, int W, int R>
constexpr bool row_halves() {
    return sizeof(T) == 4 && R > 1 && split2(M).A % 2 == 0 && split2(M).B % 2 == 0 &&
           (long)frow_full<M, W>() * (long)sizeof(cpx<T>) > 49152;
}
// pitch of a row's half spectrum: 32 / WA lanes of each of WA rows on distinct banks
template <int M, int WA>
constexpr int half_pitch() {
    constexpr int n = M / 2 + 1, want = WA >= 32 ? 1 : 32 / WA;
    return n + ((want - n) % 32 + 32) % 32;
}
template <typename T, int M, int W, int R>
constexpr int frow_lds() {
    constexpr int A = split2(M).A, B = split2(M).B;
    if (!row_halves<T, M, W, R>()) return frow_full<M, W>();
    constexpr int x = W * (A / 2) * (B + 1), y = W * half_pitch<M, (R > 1 ? W / (R / 2) : W)>();
    return x > y ? x : y;
}

// Rows of a block.  R = 1: W consecutive rows.  R > 1 (axis 1 folded by R):
// where a whole column, 3 N0 P1 points, is too large for LDS, the first radix
// R of axis 1 is done here: P1 = R Q, and the block takes the rows j' + Q m,
// m < R/2 (the others are padding), of W / (R/2) consecutive j' of one pencil:
//   x_s[j'] = w_P1^(s j') sum_m w_R^(s m) x[j' + Q m],  s < R,
// whose Q-point transforms are the frequencies R q + s.  The spectrum then has
// R columns per x frequency, [solve][k][s][c][i][j' < Q].
struct RowP {
    int rows, N1, Q, PC;  // rows and pencils (3 N0) of a solve
    int nsolve, n2;
    long mrows;           // rows of the mask
};
template <int W, int R>
struct RowMap {
    static constexpr int RH = R > 1 ? R / 2 : 1, WA = W / RH;
    long row0;      // R = 1: first row; R > 1: first row of the pencil
    int j0, sol, pen;
    __device__ __forceinline__ RowMap(const RowP& g) {
        const int b = xcd_swizzle(blockIdx.x, gridDim.x);
        if constexpr (R == 1) {
            row0 = (long)b * W;
            j0 = sol = pen = 0;
        } else {
            const int ng = (g.Q + WA - 1) / WA;
            row0 = (long)(b / ng) * g.N1;
            j0 = b % ng * WA;
            sol = b / ng / g.PC;
            pen = b / ng - sol * g.PC;
        }
    }
    // row of slot p (p = m WA + a), and whether it exists (a padded axis 1 has N1 < Q R / 2 rows)
    __device__ __forceinline__ long row(const RowP& g, int p, bool& in) const {
        if constexpr (R == 1) {
            in = row0 + p < (long)g.rows * g.nsolve;
            return in ? row0 + p : row0;
        } else {
            const int a = j0 + p % WA, j = a + g.Q * (p / WA);
            in = a < g.Q && j < g.N1;
            return row0 + (in ? j : 0);
        }
    }
    __device__ __forceinline__ bool dead(const RowP& g, const Live& lv) const {
        if constexpr (R == 1) {
            const long last = (long)g.rows * g.nsolve - 1;
            return all_dead(lv, row0, row0 + W - 1 < last ? row0 + W - 1 : last);
        } else {
            return lv.flag && !lv.flag[sol];
        }
    }
};

// R2C of a block's rows of x times 2 half (rows of n2 reals; the mask repeats
// every mrows rows), written column by column.
template <typename T, int M, int W, int R, int NT = W * split2(M).B>
__global__ void __launch_bounds__(NT) k_frows(const T* __restrict__ x, const T* __restrict__ msk,
                                              cpx<T>* __restrict__ out, RowP g, T half,
                                              const cpx<T>* __restrict__ twM, const cpx<T>* __restrict__ twP,
                                              const cpx<T>* __restrict__ tw1, Live lv) {
    constexpr int A = split2(M).A, B = split2(M).B, BP = B + 1, PM = row_pitch<M, W>();
    static_assert(A * B == M && A <= B, "two-level split");
    __shared__ cpx<T> lds[frow_lds<T, M, W, R>()];
    __shared__ cpx<T> tws[M + 1];
    constexpr bool HALVES = row_halves<T, M, W, R>();
    const int tid = threadIdx.x, n2 = g.n2;
    const RowMap<W, R> rm(g);
    if (rm.dead(g, lv)) return;
    cpx<T> u[B];
    const int k1 = tid % A, p2 = tid / A;
    // X[k] = E + w^k O from Z[k] and Z[M - k]
    auto split = [&](const cpx<T>& zk, const cpx<T>& zm, int k) {
        const cpx<T> E = {half * (zk.x + zm.x), half * (zk.y - zm.y)};
        const cpx<T> O = {half * (zk.y + zm.y), half * (zm.x - zk.x)};
        return cadd(E, cmul(tws[k], O));
    };
    constexpr int TA = (M + NT - 1) / NT, TB = (M + 1 + NT - 1) / NT;
    cpx<T> ta[TA], tb[TB];
#pragma unroll
    for (int q = 0; q < TA; q++) ta[q] = twM[tid + q * NT < M ? tid + q * NT : 0];
#pragma unroll
    for (int q = 0; q < TB; q++) tb[q] = twP[tid + q * NT <= M ? tid + q * NT : 0];
    {
        const int nb = tid % B, p = tid / B;
        bool rin;
        const long rc = rm.row(g, p, rin);
        const T* xr = x + rc * n2;
        const T* mr = msk ? msk + (rc % g.mrows) * n2 : nullptr;
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
        if constexpr (HALVES) {
#pragma unroll
            for (int k1 = 1; k1 < A; k1++) v[k1] = cmul(v[k1], tws[nb * k1]);
#pragma unroll
            for (int h = 0; h < 2; h++) {
#pragma unroll
                for (int q = 0; q < A / 2; q++) lds[(p * (A / 2) + q) * BP + nb] = v[2 * q + h];
                __syncthreads();
                if (tid < W * A && k1 % 2 == h) {
#pragma unroll
                    for (int m = 0; m < B; m++) u[m] = lds[(p2 * (A / 2) + k1 / 2) * BP + m];
                }
                __syncthreads();
            }
        } else {
#pragma unroll
            for (int k1 = 0; k1 < A; k1++) lds[(p * A + k1) * BP + nb] = k1 ? cmul(v[k1], tws[nb * k1]) : v[k1];
        }
    }
    if constexpr (!HALVES) __syncthreads();
#pragma unroll
    for (int q = 0; q < TB; q++)
        if (tid + q * NT <= M) tws[tid + q * NT] = tb[q];
    if constexpr (HALVES) {
        constexpr int RH = R / 2, WA = W / RH, KS = NT / WA, PH = half_pitch<M, WA>();
        if (tid < W * A) dft_reg<T, B, -1>(u);
        const int a = tid % WA, kk = tid / WA, j = rm.j0 + a;
        const bool jin = j < g.Q;
        cpx<T> wj[R];
#pragma unroll
        for (int s = 1; s < R; s++) wj[s] = tw1[s * (jin ? j : 0)];
        const long cs = (long)g.PC * g.Q;
        cpx<T>* o = out + rm.sol * (long)(M + 1) * R * cs + (long)rm.pen * g.Q + j;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if (h) __syncthreads();
            if (tid < W * A && k1 % 2 == h) {
#pragma unroll
                for (int k2 = 0; k2 < B; k2++) lds[p2 * PH + (k1 + A * k2) / 2] = u[k2];
            }
            __syncthreads();
            if (jin)
                for (int k = h + 2 * kk; k <= M; k += 2 * KS) {
                    cpx<T> f[R];
#pragma unroll
                    for (int m = 0; m < R; m++) {
                        f[m] = {T(0), T(0)};
                        if (m < RH) {
                            const cpx<T>* z = lds + (m * WA + a) * PH;
                            f[m] = split(z[(k == M ? 0 : k) / 2], z[(k == 0 ? 0 : M - k) / 2], k);
                        }
                    }
                    dft_reg<T, R, -1>(f);
#pragma unroll
                    for (int s = 0; s < R; s++) o[((long)k * R + s) * cs] = s ? cmul(f[s], wj[s]) : f[s];
                }
        }
        return;
    }
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
    auto split_row = [&](int p, int k) {
        return split(lds[p * PM + (k == M ? 0 : k)], lds[p * PM + (k == 0 ? 0 : M - k)], k);
    };
    if constexpr (R == 1) {  // lanes walk the W rows first, so that a column's W values leave together
        const int p = tid % W, kk = tid / W;
        bool in;
        const long r = rm.row(g, p, in);
        if (in) {
            const long sol = r / g.rows;
            cpx<T>* o = out + sol * (M + 1) * (long)g.rows + (r - sol * g.rows);
#pragma unroll
            for (int q = 0; q < A; q++) o[(long)(kk + B * q) * g.rows] = split_row(p, kk + B * q);
            if (kk == 0) o[(long)M * g.rows] = split_row(p, M);
        }
    } else {  // ... the WA values of j' first
        constexpr int RH = R / 2, WA = W / RH, KS = NT / WA;
        const int a = tid % WA, kk = tid / WA, j = rm.j0 + a;
        if (j < g.Q) {
            cpx<T> wj[R];
#pragma unroll
            for (int s = 1; s < R; s++) wj[s] = tw1[s * j];
            const long cs = (long)g.PC * g.Q;
            cpx<T>* o = out + rm.sol * (long)(M + 1) * R * cs + (long)rm.pen * g.Q + j;
            for (int k = kk; k <= M; k += KS) {
                cpx<T> f[R];
#pragma unroll
                for (int m = 0; m < R; m++) f[m] = m < RH ? split_row(m * WA + a, k) : cpx<T>{T(0), T(0)};
                dft_reg<T, R, -1>(f);
#pragma unroll
                for (int s = 0; s < R; s++) o[((long)k * R + s) * cs] = s ? cmul(f[s], wj[s]) : f[s];
            }
        }
    }
}

// C2R of a block's rows from the column-major spectrum; R > 1: the last radix
// of axis 1 first, x[j' + Q m] = sum_s w_R^(-s m) w_P1^(-s j') z_s[j'].
template <typename T, int M, int W, int R, int NT = W * split2(M).B>
__global__ void __launch_bounds__(NT) k_irows(const cpx<T>* __restrict__ in, T* __restrict__ x, RowP g,
                                              const cpx<T>* __restrict__ twM, const cpx<T>* __restrict__ twP,
                                              const cpx<T>* __restrict__ tw1, Live lv) {
    constexpr int A = split2(M).A, B = split2(M).B, BP = B + 1, PM = row_pitch<M, W>();
    static_assert(A * B == M && A <= B, "two-level split");
    __shared__ cpx<T> lds[frow_lds<T, M, W, R>()];
    __shared__ cpx<T> tws[M];
    __shared__ cpx<T> twp[M];
    constexpr bool HALVES = row_halves<T, M, W, R>();
    const int tid = threadIdx.x, n2 = g.n2;
    const RowMap<W, R> rm(g);
    if (rm.dead(g, lv)) return;
    const int nb = tid % B, p = tid / B;
    cpx<T> v[A];
    // Z[k] of C2R from X[k] and X[M - k]
    auto join = [&](const cpx<T>& a, const cpx<T>& b, int k) -> cpx<T> {
        const cpx<T> s = {a.x + b.x, a.y - b.y};
        const cpx<T> d = {a.x - b.x, a.y + b.y};
        cpx<T> w = twp[k];
        w.y = -w.y;
        const cpx<T> wd = cmul(w, d);
        return {s.x - wd.y, s.y + wd.x};
    };
    {
        constexpr int TA = (M + NT - 1) / NT;
        cpx<T> ta[TA], tb[TA];
#pragma unroll
        for (int q = 0; q < TA; q++) {
            const int e = tid + q * NT;
            ta[q] = twM[e < M ? e : 0];
            tb[q] = twP[e < M ? e : 0];
        }
        if constexpr (R == 1) {
            const int p = tid % W, kk = tid / W;
            bool ok;
            const long r = rm.row(g, p, ok);
            const long sol = r / g.rows;
            const cpx<T>* q0 = in + sol * (M + 1) * (long)g.rows + (r - sol * g.rows);
            cpx<T> v[A], vm;
#pragma unroll
            for (int q = 0; q < A; q++) v[q] = q0[(long)(kk + B * q) * g.rows];
            vm = q0[(long)M * g.rows];
#pragma unroll
            for (int q = 0; q < A; q++) lds[p * PM + kk + B * q] = v[q];
            if (kk == 0) lds[p * PM + M] = vm;
        } else if constexpr (HALVES) {
            constexpr int RH = R / 2, WA = W / RH, KS = NT / WA, PH = half_pitch<M, WA>(), U = (M / 2 + KS - 1) / KS;
            const int a = tid % WA, kk = tid / WA, j = rm.j0 + a < g.Q ? rm.j0 + a : 0;
            cpx<T> wj[R];
#pragma unroll
            for (int s = 1; s < R; s++) {
                wj[s] = tw1[s * j];
                wj[s].y = -wj[s].y;
            }
            const long cs = (long)g.PC * g.Q;
            const cpx<T>* q0 = in + rm.sol * (long)(M + 1) * R * cs + (long)rm.pen * g.Q + j;
            // the R columns of frequency k, and their last radix into LDS
            auto fetch = [&](int k, cpx<T>* f) {
#pragma unroll
                for (int s = 0; s < R; s++) f[s] = q0[((long)k * R + s) * cs];
            };
            auto place = [&](int k, cpx<T>* f) {
#pragma unroll
                for (int s = 1; s < R; s++) f[s] = cmul(f[s], wj[s]);
                dft_reg<T, R, +1>(f);
#pragma unroll
                for (int m = 0; m < RH; m++) lds[(m * WA + a) * PH + k / 2] = f[m];
            };
            auto freq = [&](int h, int u) { return h + 2 * (kk + u * KS); };  // < M: one of half h
            cpx<T> f[U][R], fm[R];
#pragma unroll
            for (int u = 0; u < U; u++) fetch(freq(0, u) < M ? freq(0, u) : 0, f[u]);
            if (kk == 0) fetch(M, fm);
#pragma unroll
            for (int q = 0; q < TA; q++) {
                const int e = tid + q * NT;
                if (e < M) {
                    tws[e] = ta[q];
                    twp[e] = tb[q];
                }
            }
#pragma unroll
            for (int h = 0; h < 2; h++) {
#pragma unroll
                for (int u = 0; u < U; u++)
                    if (freq(h, u) < M) place(freq(h, u), f[u]);
                if (h == 0 && kk == 0) place(M, fm);
                __syncthreads();
                if (nb % 2 == h) {
                    const cpx<T>* z = lds + p * PH;
#pragma unroll
                    for (int n1 = 0; n1 < A; n1++) {
                        const int k = B * n1 + nb;
                        v[n1] = join(z[k / 2], z[(M - k) / 2], k);
                    }
                }
                if (h == 0) {
#pragma unroll
                    for (int u = 0; u < U; u++) fetch(freq(1, u) < M ? freq(1, u) : 1, f[u]);
                }
                __syncthreads();
            }
        } else {
            constexpr int RH = R / 2, WA = W / RH, KS = NT / WA, U = 16 / R > 1 ? 16 / R : 1;
            const int a = tid % WA, kk = tid / WA, j = rm.j0 + a < g.Q ? rm.j0 + a : 0;
            cpx<T> wj[R];
#pragma unroll
            for (int s = 1; s < R; s++) {
                wj[s] = tw1[s * j];
                wj[s].y = -wj[s].y;
            }
            const long cs = (long)g.PC * g.Q;
            const cpx<T>* q0 = in + rm.sol * (long)(M + 1) * R * cs + (long)rm.pen * g.Q + j;
            for (int k0 = kk; k0 <= M; k0 += U * KS) {  // U frequencies of R loads in flight
                cpx<T> f[U][R];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const long k = k0 + u * KS <= M ? k0 + u * KS : M;
#pragma unroll
                    for (int s = 0; s < R; s++) f[u][s] = q0[(k * R + s) * cs];
                }
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const int k = k0 + u * KS;
                    if (k <= M) {
#pragma unroll
                        for (int s = 1; s < R; s++) f[u][s] = cmul(f[u][s], wj[s]);
                        dft_reg<T, R, +1>(f[u]);
#pragma unroll
                        for (int m = 0; m < RH; m++) lds[(m * WA + a) * PM + k] = f[u][m];
                    }
                }
            }
        }
        if constexpr (!HALVES) {
#pragma unroll
            for (int q = 0; q < TA; q++) {
                const int e = tid + q * NT;
                if (e < M) {
                    tws[e] = ta[q];
                    twp[e] = tb[q];
                }
            }
        }
    }
    if constexpr (!HALVES) {
        __syncthreads();
#pragma unroll
        for (int n1 = 0; n1 < A; n1++) {
            const int k = B * n1 + nb;
            v[n1] = join(lds[p * PM + k], lds[p * PM + (M - k)], k);
        }
        __syncthreads();
    }
    dft_reg<T, A, +1>(v);
#pragma unroll
    for (int k1 = 1; k1 < A; k1++) {
        cpx<T> w = tws[nb * k1];
        w.y = -w.y;
        v[k1] = cmul(v[k1], w);
    }
    cpx<T> u[B];
    const int k1 = tid % A, p2 = tid / A;
    if constexpr (HALVES) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if (h) __syncthreads();
#pragma unroll
            for (int q = 0; q < A / 2; q++) lds[(p * (A / 2) + q) * BP + nb] = v[2 * q + h];
            __syncthreads();
            if (tid < W * A && k1 % 2 == h) {
#pragma unroll
                for (int m = 0; m < B; m++) u[m] = lds[(p2 * (A / 2) + k1 / 2) * BP + m];
            }
        }
    } else {
#pragma unroll
        for (int k1 = 0; k1 < A; k1++) lds[(p * A + k1) * BP + nb] = v[k1];
        __syncthreads();
    }
    if (tid < W * A) {
        bool rin;
        const long r = rm.row(g, p2, rin);
        if constexpr (!HALVES) {
#pragma unroll
            for (int m = 0; m < B; m++) u[m] = lds[(p2 * A + k1) * BP + m];
        }
        dft_reg<T, B, +1>(u);
        if (rin) {
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
inline int mid_nt(int N0, int Q, int CB, int IB = 0) {
    if (!IB) IB = mid_ib(N0);
    const int items = CB * ((N0 + IB - 1) / IB) * Q, itm = mid_itm(IB, N0 > IB);
    return ((items + itm - 1) / itm + 63) / 64 * 64;
}
// whether a column of the mesh fits one block
inline bool mid_fits(int N0, int Q, int A, int B, size_t cs) {
    return mid_nt(N0, Q, 1) <= kMidMax && mid_lds(Q, A, B, N0, 1, cs) <= (size_t)kLds;
}
// Tile elements (complex) of a block that leave a CU six blocks (half of it,
// three).  Small tiles hide each other's phases: 3072 against 6144 elements
// take 24.7 against 30.8 us at 32 solves of 128x128x2, 13.5 against 14.7 at
// 64x64x4.
constexpr long kTile = 3072;
// The direct convolution's N0^2 products pass the zero-padded FFTs of the five
// passes between 32 planes (three kernels 98 us, five passes 160 at 32 solves
// of 32x32x32) and 64 (54 against 43 us at 64x64x64).
constexpr int kPlanes = 32;
inline long mid_elems(size_t cs) { return kTile * 8 / (long)cs; }
// Fold R of axis 1 for N0 planes and P1 points (fits(R): registered and a
// column fits a block; timed: the plan's five passes would be timed), 0 if
// none.  No folding up to 6144 elements a column (FP64: 3072).  Beyond, a
// column leaves too few blocks a CU, and folding until it has 3072 elements is
// best while the rows still leave in 64-byte pieces (R <= 4: 42.4 us a field at
// 256x256x8 against 45.7 with R = 2 and 48.3 without), else until it has 6144
// (R = 8 at 512x512x16: 298 us, R = 16 with 16-byte pieces 334; five passes
// 317) in blocks of at most 256 threads: five and six waves run badly (R = 4
// with 320 threads against R = 8: 320x320x10 109 us a field against 87, five
// passes 89; 128x128x26 70 against 54, five passes 55).
// FP64 stops at R = 4, with which 256x256x8 leaves the five passes behind
// (73 us against 96); beyond, it has no row kernels.
// More than 16 planes on compiled lengths stay with the five passes rather
// than fold.  One field, folded / five passes: 64x64x24 30.3 / 27.2 us,
// 96x96x24 39.5 / 35.1, 256x64x20 46.0 / 39.2, 128x128x32 62.4 / 52.8; RK4 steps
// of batches are between 0.9 (64x256x20) and 1.14 (512x64x24) times as long.
// Without folding, three kernels up to 32 planes: one field of 32^3 takes 21.1 us
// against 20.3, a step of 64 solves 729 us against 945.  A plan at padded lengths has
// untimed passes, and folds (96x96x30: a step of 8 solves 789 us against 893).
template <typename F>
int mid_fold(int N0, int P1, size_t cs, bool timed, F fits) {
    const long el = kTile;
    if (N0 > kPlanes) return 0;
    auto ok = [&](int R, long most) { return P1 % R == 0 && 3L * N0 * (P1 / R) <= most && fits(R); };
    if (ok(1, cs == 8 ? 2 * el : el)) return 1;
    if (cs == 8 && N0 > kPlanes / 2 && timed) return 0;
    for (int R = 2; R <= 4; R *= 2)
        if (ok(R, el)) return R;
    if (cs == 8)
        for (int R = 2; R <= 8; R *= 2)
            if (mid_nt(N0, P1 / R, 1) <= 256 && ok(R, 2 * el)) return R;
    return ok(1, 1L << 40) ? 1 : 0;
}
// Columns per block: about kTile elements, fewer while the launch would leave
// CUs idle.  A column's arithmetic does not depend on it.
inline int mid_cb(int N0, int Q, int A, int B, int ncol, int nsolve, size_t cs) {
    int cb = (int)std::max(1L, mid_elems(cs) / (3L * N0 * Q));
    cb = std::min(cb, ncol);
    while (cb > 1 && ((long)((ncol + cb - 1) / cb) * nsolve < 512 || mid_nt(N0, Q, cb) > kMidMax ||
                      mid_lds(Q, A, B, N0, cb, cs) > (size_t)kLds))
        cb--;
    return cb;
}
// ---- registry ---------------------------------------------------------------
template <typename T>
using frows_t = void (*)(const T*, const T*, cpx<T>*, const RowP&, T, const cpx<T>*, const cpx<T>*, const cpx<T>*,
                         hipStream_t, Live);
template <typename T>
using irows_t = void (*)(const cpx<T>*, T*, const RowP&, const cpx<T>*, const cpx<T>*, const cpx<T>*, hipStream_t,
                         Live);
template <typename T>
using mid_t = void (*)(const Mid<T>&, hipStream_t);

constexpr int kFolds = 4;  // R = 1, 2, 4, 8
template <typename T>
struct Rows {
    frows_t<T> fwd[kFolds] = {};
    irows_t<T> inv[kFolds] = {};
};
template <typename T>
struct Mids {
    mid_t<T> one[2][9] = {};    // [folded] N0 = 1..8 planes
    mid_t<T> multi[2][9] = {};  // more, in blocks of 6 or 8
    mid_t<T> few = nullptr;     // more, in blocks of kFewIB, unfolded
    int A = 0, B = 0;
    mid_t<T> pick(int N0, bool fold) const {
        return N0 <= 8 ? one[fold][N0] : multi[fold][mid_ib(N0)];
    }
};
inline int fold_index(int R) { return R == 1 ? 0 : (R == 2 ? 1 : (R == 4 ? 2 : 3)); }
inline int table_rows_of(int Q, bool fold) { return table_rows(Q, fold); }
// The kernels of one plan.
template <typename T>
struct Form {
    frows_t<T> fwd = nullptr;
    irows_t<T> inv = nullptr;
    mid_t<T> mid = nullptr;
    mid_t<T> few = nullptr;  // mid for launches of few waves, null where it has none
    int A = 0, B = 0;  // split of the mid kernel's columns
};
// registries (demag.hip): the entry to fill at library load, and the entry of a
// length for reading (an empty one if there is none)
template <typename T>
Rows<T>& add_rows_of(int M);
template <typename T>
Mids<T>& add_mids_of(int Q);
template <typename T>
const Rows<T>& rows_of(int M);
template <typename T>
const Mids<T>& mids_of(int Q);

// Rows per block: full 128-byte pieces of a column (16 rows of 8 bytes) while
// the tile stays near 32 KB; folded, 16 rows or as many as 72 KB hold, and in
// halves (row_halves) 32 or as many as 70 KB and a block's threads hold
// (neighbouring blocks complete the lines in L2).
template <typename T, int M, int R>
constexpr int frow_w() {
    constexpr int cs = (int)sizeof(cpx<T>), rh = R > 1 ? R / 2 : 1;
    const bool halves = row_halves<T, M, 16, R>();
    int w = R == 1 ? 128 / cs : (halves ? 32 : 16);
    if (w < rh) w = rh;
    while (w > 2 && w > rh && ((long)w * M * cs > (R == 1 ? 40000 : (halves ? 140000 : 72000)) || w * split2(M).B > 1024))
        w /= 2;
    while (w < 16 && w * split2(M).B < 64) w *= 2;
    return w;
}
template <int W, int R>
unsigned frow_grid(const RowP& g) {
    constexpr int WA = R > 1 ? W / (R / 2) : W;
    if (R == 1) return (unsigned)(((long)g.rows * g.nsolve + W - 1) / W);
    return (unsigned)((long)g.nsolve * g.PC * ((g.Q + WA - 1) / WA));
}
template <typename T, int M, int R>
void launch_frows(const T* x, const T* msk, cpx<T>* out, const RowP& g, T half, const cpx<T>* twM, const cpx<T>* twP,
                  const cpx<T>* tw1, hipStream_t st, Live lv) {
    constexpr int W = frow_w<T, M, R>();
    hipLaunchKernelGGL((k_frows<T, M, W, R>), dim3(frow_grid<W, R>(g)), dim3(W * split2(M).B), 0, st, x, msk, out,
                       g, half, twM, twP, tw1, lv);
}
template <typename T, int M, int R>
void launch_irows(const cpx<T>* in, T* x, const RowP& g, const cpx<T>* twM, const cpx<T>* twP, const cpx<T>* tw1,
                  hipStream_t st, Live lv) {
    constexpr int W = frow_w<T, M, R>();
    hipLaunchKernelGGL((k_irows<T, M, W, R>), dim3(frow_grid<W, R>(g)), dim3(W * split2(M).B), 0, st, in, x, g,
                       twM, twP, tw1, lv);
}

template <typename T, int Q, int IB, bool MULTI, bool FOLD>
void launch_mid(const Mid<T>& m, hipStream_t st) {
    constexpr int A = split_even(Q).A, B = split_even(Q).B;
    const size_t lds = mid_lds(Q, A, B, m.N0, m.CB, sizeof(cpx<T>));
    const int nt = mid_nt(m.N0, Q, m.CB, IB);
    if (lds > 65536)
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&k_fmid<T, Q, IB, MULTI, FOLD>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    const unsigned g = (unsigned)((m.ncol + m.CB - 1) / m.CB) * (unsigned)m.nsolve;
    hipLaunchKernelGGL((k_fmid<T, Q, IB, MULTI, FOLD>), dim3(g), dim3(nt), lds, st, m);
}

template <typename T, int M, int F>
void add_rows_fold(Rows<T>& r) {
    constexpr int R = 1 << F, W = frow_w<T, M, R>();
    constexpr long lds = ((long)frow_lds<T, M, W, R>() + 2 * M) * (long)sizeof(cpx<T>);
    if constexpr (lds <= kLds && W * split2(M).B <= 1024) {
        r.fwd[F] = &launch_frows<T, M, R>;
        r.inv[F] = &launch_irows<T, M, R>;
    }
}
template <typename T, int M>
void add_rows() {
    if constexpr (two_level_ok(M) && M >= 8) {
        Rows<T>& r = add_rows_of<T>(M);
        add_rows_fold<T, M, 0>(r), add_rows_fold<T, M, 1>(r), add_rows_fold<T, M, 2>(r);
        if constexpr (sizeof(T) == 4) add_rows_fold<T, M, 3>(r);
    }
}
template <typename T, int Q, int IB, bool FOLD>
void add_mid_ib(Mids<T>& m) {
    // only what can fit a block (mid_fits): LDS, and items per thread
    constexpr int A = split_even(Q).A, B = split_even(Q).B;
    constexpr long lds = (3L * IB * A * (B + 1) + Q) * (long)sizeof(cpx<T>);
    if constexpr (lds <= kLds && Q <= kMidMax * mid_itm(IB)) m.one[FOLD][IB] = &launch_mid<T, Q, IB, false, FOLD>;
    if constexpr ((IB == 6 || IB == 8) && lds * 3 / 2 <= kLds)
        m.multi[FOLD][IB] = &launch_mid<T, Q, IB, true, FOLD>;
}
template <typename T, int Q, bool FOLD>
void add_mid_fold(Mids<T>& m) {
    add_mid_ib<T, Q, 1, FOLD>(m), add_mid_ib<T, Q, 2, FOLD>(m), add_mid_ib<T, Q, 3, FOLD>(m);
    add_mid_ib<T, Q, 4, FOLD>(m), add_mid_ib<T, Q, 5, FOLD>(m), add_mid_ib<T, Q, 6, FOLD>(m);
    add_mid_ib<T, Q, 7, FOLD>(m), add_mid_ib<T, Q, 8, FOLD>(m);
}
template <typename T, int Q>
void add_mid() {
    if constexpr (split_even(Q).A > 0) {
        Mids<T>& m = add_mids_of<T>(Q);
        m.A = split_even(Q).A;
        m.B = split_even(Q).B;
        if constexpr (sizeof(T) == 4 && Q <= kMidMax) m.few = &launch_mid<T, Q, kFewIB, true, false>;
        add_mid_fold<T, Q, false>(m);
        add_mid_fold<T, Q, true>(m);
    }
}
// every length of a list
template <typename T, int... L>
void register_rows() {
    (add_rows<T, L>(), ...);
}
template <typename T, int... Q>
void register_mids() {
    (add_mid<T, Q>(), ...);
}
}  // namespace fused
